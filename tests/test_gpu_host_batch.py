"""The host-pointer batch call: above the zero-copy size, results that leave in
published slices, x read from the pinned stage or copied, and the memory that
the call holds; below it, odd widths."""
import ctypes as C

import numpy as np
import pytest

import native
from native import bh, ptr, same_bits

pytestmark = pytest.mark.gpu


def inputs(M, n, rows, seed):
    r = np.random.default_rng(seed)
    packed = bh.synth_ternary(seed, 1, rows, n, bh.SYNTH_P0_40)
    x = (r.standard_normal((M, n)) * np.exp(r.standard_normal((M, 1)))).astype(np.float32)
    return x, packed, (1.0 + 0.1 * r.standard_normal(n)).astype(np.float32)


def host_call(hip, x, packed, g, rows, stride, norm=True, quant=True, shift=0):
    """The call's results; `out` starts `shift` floats into a buffer."""
    M, n = x.shape
    w, nw = bh.make_tensor(packed, rows, n, 0.02), bh.make_tensor(data=g)
    buf = np.full(M * rows + 2 * shift, np.nan, np.float32)
    out = buf[shift:shift + M * rows].reshape(M, rows)
    xn = np.full(n + 4, 7.0, np.float32)
    xq = np.full((M, stride), 99, np.int8)
    hip.hip_bitlinear_forward_batch(ptr(x), M, n, C.byref(w), C.byref(nw), ptr(out),
                                    ptr(xn) if norm else None, ptr(xq) if quant else None, stride)
    assert np.isnan(buf[:shift]).all() and np.isnan(buf[M * rows + shift:]).all()
    return out, xn, xq


def device_call(hip, x, packed, g, rows):
    """The same product through device buffers."""
    M, n = x.shape
    DB = bh.DeviceBuffer
    dx, dg, dw = DB.from_array(x), DB.from_array(g), DB.from_array(packed)
    do, dq, ds = DB(4 * M * rows), DB(M * n), DB(4 * M)
    da = DB(max(hip.bm_hip_act_bytes(M, n), 1))
    bh.check(hip.bm_hip_bitlinear_dev(dx.ptr, M, n, dg.ptr, dw.ptr, rows, 0.02, 1, do.ptr, dq.ptr, n,
                                      ds.ptr, da.ptr, None), "bitlinear")
    hip.bm_hip_synchronize()
    return do.download((M, rows), np.float32), dq.download((M, n), np.int8)


def check(hip, M, n, rows, stride, norm=True, quant=True, shift=0, tokens=()):
    """The host call against the device product, the oracle's norm of the last
    token (all that x_norm keeps), and the oracle's rows of `tokens`."""
    print("host batch M=%d n=%d rows=%d stride=%d norm=%d quant=%d" % (M, n, rows, stride, norm,
                                                                       quant), flush=True)
    x, packed, g = inputs(M, n, rows, M + n + rows)
    out, xn, xq = host_call(hip, x, packed, g, rows, stride, norm, quant, shift)
    want, q = device_call(hip, x, packed, g, rows)
    same_bits(out, want, "out")
    if norm:
        rn, _, _, _ = native.orc_quantize_rows(x[-1:], g)
        same_bits(xn[:n], rn[0], "x_norm")
    assert (xn[n if norm else 0:] == 7.0).all()
    if quant:
        np.testing.assert_array_equal(xq[:, :n], q)
    assert (xq[:, n if quant else 0:] == 99).all()
    for m in tokens:
        ref, _, rq = native.orc_bitlinear(x[m:m + 1], packed, rows, n, 0.02, g)
        same_bits(out[m], ref[0], "out[%d]" % m)
        if quant:
            np.testing.assert_array_equal(xq[m, :n], rq[0])


@pytest.mark.parametrize("norm,quant", [(True, True), (False, True), (True, False), (False, False)])
@pytest.mark.parametrize("M,n,rows,stride", [
    (256, 1024, 4192, 1024),    # slices of all three parts
    (130, 1003, 517, 1010),     # the last x_norm on no 16 bytes: bytes; the generic product
    (63, 1025, 1, 1025),        # results of a few bytes per token
    (40, 8256, 300, 8300),      # x from a device copy
    (70, 2048, 1024, 2048)])
def test_large_calls(hip, M, n, rows, stride, norm, quant):
    check(hip, M, n, rows, stride, norm, quant, tokens=(0, M // 2, M - 1))


@pytest.mark.parametrize("M", [1, 2, 3])
@pytest.mark.parametrize("n,rows", [(130, 17), (1003, 1003), (2050, 64)])
def test_small_odd_widths(hip, M, n, rows):
    """Zero-copy calls at widths off 64: the product reads its int8 rows from the
    mapped memory, one or two of them staged, more by a wave each."""
    check(hip, M, n, rows, n + 2, tokens=range(M))


def test_large_then_small(hip):
    """Calls of falling and rising size on one stage and one set of words."""
    for M, n, rows in ((512, 1024, 4192), (33, 2048, 1024), (3, 1024, 300), (512, 1024, 4192),
                       (90, 1088, 700), (1, 2048, 70001), (40, 8256, 300), (256, 1024, 512)):
        check(hip, M, n, rows, n + 16, tokens=(0, M - 1))


def test_more_slices_than_words(hip):
    """147 MB of results: slices of 128 KiB."""
    check(hip, 9000, 64, 4096, 64, tokens=(0, 4500, 8999))


@pytest.mark.parametrize("M,n,rows,shift", [(1536, 1024, 4192, 0), (1700, 1024, 4099, 1),
                                            (6, 64, 1100000, 3)])
def test_streamed_results(hip, M, n, rows, shift):
    """Results beyond the caches, to outputs that start on any float."""
    check(hip, M, n, rows, n + 5, shift=shift)


def test_memory_of_large_calls(hip):
    """A call whose x is read from the stage holds no device copy of x."""
    M, n, rows = 4096, 8192, 16
    free0, free1, total = C.c_size_t(), C.c_size_t(), C.c_size_t()
    info = C.CDLL("libamdhip64.so").hipMemGetInfo
    info.argtypes = [C.POINTER(C.c_size_t)] * 2
    x, packed, g = inputs(M, n, rows, 3)
    host_call(hip, x[:2], packed, g, rows, n)
    assert info(C.byref(free0), C.byref(total)) == 0
    print("host batch M=%d n=%d rows=%d" % (M, n, rows), flush=True)
    out, _, _ = host_call(hip, x, packed, g, rows, n)
    assert info(C.byref(free1), C.byref(total)) == 0
    results = M * (4 * rows + 4 * n + n)
    bound = 1.25 * (results + hip.bm_hip_act_bytes(M, n)) + (32 << 20)
    assert bound < results + hip.bm_hip_act_bytes(M, n) + x.nbytes
    assert free0.value - free1.value < bound, (free0.value - free1.value, bound)
    for m in (0, M - 1):
        ref, _, _ = native.orc_bitlinear(x[m:m + 1], packed, rows, n, 0.02, g)
        same_bits(out[m], ref[0], "out[%d]" % m)
