"""Products of widths that are no multiples of 64: the two kernels' results on
both sides of the rule that chooses between them (generic_by_wave,
bm_kernels.hip), and that few tokens cost about what one does."""
import ctypes as C

import numpy as np
import pytest

import native
from native import bh, same_bits

pytestmark = pytest.mark.gpu
DB = bh.DeviceBuffer

# tokens, width, the rule's bound on M * N there
BOUNDS = [(1, 500, 8192), (1, 700, 3072), (2, 130, 8192), (2, 1003, 4096), (2, 2050, 2048),
          (4, 70, 12288), (3, 1030, 8192), (4, 2050, 5120), (5, 201, 32768), (9, 500, 24576),
          (16, 1001, 16384)]


def check(hip, M, K, N):
    print("generic M=%d K=%d N=%d" % (M, K, N), flush=True)
    r = np.random.default_rng(M * 17 + K + N)
    packed = r.integers(0, 256, (N, (K + 3) // 4)).astype(np.uint8)
    if K % 4:
        packed[:, -1] &= (1 << (2 * (K % 4))) - 1
    x = r.standard_normal((M, K)).astype(np.float32)
    g = (r.standard_normal(K) * 0.02).astype(np.float32)
    dx, dg, dw = DB.from_array(x), DB.from_array(g), DB.from_array(packed)
    do, dq, ds = DB(4 * M * N), DB(M * K), DB(4 * M)
    da = DB(hip.bm_hip_act_bytes(M, K))
    bh.check(hip.bm_hip_bitlinear_dev(dx.ptr, M, K, dg.ptr, dw.ptr, N, 0.02, 0, do.ptr, dq.ptr,
                                      K, ds.ptr, da.ptr, None), "bitlinear")
    hip.bm_hip_synchronize()
    ref, _, _ = native.orc_bitlinear(x, packed, N, K, 0.02, g)
    same_bits(do.download((M, N), np.float32), ref, "out")
    xq = r.integers(-128, 128, (M, K + 3)).astype(np.int8)
    dxq = DB.from_array(xq)
    bh.check(hip.bm_hip_ternary_gemm_i32_dev(dxq.ptr, M, K + 3, dw.ptr, N, K, 0, do.ptr, da.ptr,
                                             None), "int32")
    hip.bm_hip_synchronize()
    want = native.orc_gemm_i32(np.ascontiguousarray(xq[:, :K]), packed, N, K)
    np.testing.assert_array_equal(do.download((M, N), np.int32), want)


@pytest.mark.parametrize("M,K,bound", BOUNDS)
def test_both_sides(hip, M, K, bound):
    for N in (bound // M, bound // M + 1):
        check(hip, M, K, N)


@pytest.mark.parametrize("M,K,N", [(1, 1, 8193), (1, 3, 8207), (1, 4100, 17), (2, 63, 4097),
                                   (2, 1025, 2064), (4, 1023, 2049), (3, 4, 4111), (7, 1025, 2350),
                                   (8, 4100, 2049), (9, 3, 3649), (37, 1000, 450), (41, 2050, 401)])
def test_staged_edges(hip, M, K, N):
    """The staged tiles where they do not fill: rows, tokens, slices, and the
    K % 4 columns after them."""
    check(hip, M, K, N)


def _us_per_call(call, n=50):
    """Fastest of a few replays of a graph of n calls, per call."""
    rt = C.CDLL("libamdhip64.so")
    vp = C.c_void_p
    rt.hipStreamCreateWithFlags.argtypes = [C.POINTER(vp), C.c_uint]
    rt.hipStreamBeginCapture.argtypes = [vp, C.c_int]
    rt.hipStreamEndCapture.argtypes = [vp, C.POINTER(vp)]
    rt.hipGraphInstantiate.argtypes = [C.POINTER(vp), vp, vp, C.c_char_p, C.c_size_t]
    for f in ("hipStreamSynchronize", "hipGraphExecDestroy", "hipGraphDestroy", "hipStreamDestroy"):
        getattr(rt, f).argtypes = [vp]
    rt.hipGraphLaunch.argtypes = [vp, vp]
    L = bh.lib()
    s, g, e = vp(), vp(), vp()
    assert rt.hipStreamCreateWithFlags(C.byref(s), 1) == 0
    assert rt.hipStreamBeginCapture(s, 1) == 0
    rcs = [call(s.value) for _ in range(n)]
    assert rt.hipStreamEndCapture(s, C.byref(g)) == 0 and not any(rcs)
    assert rt.hipGraphInstantiate(C.byref(e), g, None, None, 0) == 0
    e0, e1 = L.bm_hip_event_create(), L.bm_hip_event_create()
    best = 1e9
    for _ in range(8):
        L.bm_hip_event_record(e0, s.value)
        assert rt.hipGraphLaunch(e, s) == 0
        L.bm_hip_event_record(e1, s.value)
        assert rt.hipStreamSynchronize(s) == 0
        best = min(best, L.bm_hip_event_elapsed_ms(e0, e1) * 1000.0 / n)
    L.bm_hip_event_destroy(e0)
    L.bm_hip_event_destroy(e1)
    rt.hipGraphExecDestroy(e)
    rt.hipGraphDestroy(g)
    rt.hipStreamDestroy(s)
    return best


@pytest.mark.parametrize("K", [130, 8190])
def test_few_tokens_cost_about_one(hip, K):
    """128 rows leave the chip idle at one token, so 2 and 8 tokens fit beside
    it: measured 1.0 to 1.4 times one token's time.  The staged tiles of 8
    tokens took 2.1 to 3.6 times; 1.75 lies between."""
    N, M = 128, 8
    r = np.random.default_rng(K)
    dw = DB.from_array(r.integers(0, 256, (N, (K + 3) // 4)).astype(np.uint8))
    dxq = DB.from_array(r.integers(-128, 128, (M, K)).astype(np.int8))
    do, da = DB(4 * M * N), DB(max(hip.bm_hip_i8_act_bytes(M, K), 1))
    us = {}
    for m in (1, 2, M):
        us[m] = _us_per_call(lambda s: hip.bm_hip_ternary_gemm_i32_dev(
            dxq.ptr, m, K, dw.ptr, N, K, 0, do.ptr, da.ptr, s))
        print("K=%d M=%d: %.2f us" % (K, m, us[m]), flush=True)
    assert us[2] < 1.75 * us[1] and us[M] < 1.75 * us[1], us
