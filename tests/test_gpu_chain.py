"""The wave-parallel running sum of squares (bm_dev.h, chain_wave): rows that
would show any difference from the one-by-one fp32 sum, through every kernel
that uses it, bit-exact against the oracle.  Widths at the edges of the
elements-per-lane classes, padded chains and the largest of each."""
import numpy as np
import pytest

import native
from native import bh, same_bits

pytestmark = pytest.mark.gpu
DB = bh.DeviceBuffer


def rows_for(n, seed):
    r = np.random.default_rng(seed)
    c = (n + 3) // 4
    # sums to 2^24 - 1, then adds of 1/4 that each round away: the sum stays
    # below 2^24 while any sum in another order passes it
    stuck = np.full(c, 0.5)
    stuck[:4] = [4095.0, 90.0, 9.0, 3.0]
    # the same one add later in the chain, inside a lane
    late = np.roll(stuck, min(c - 4, c // 2 + 1))
    late[: min(c - 4, c // 2 + 1)] = 0.0
    rows = [
        r.standard_normal(n) * np.exp(r.standard_normal(n)),
        np.where(r.random(n) < 0.02, 4096.0, 1.0),   # ties at half an ulp
        np.ldexp(1.0, r.integers(-20, 20, n)),
        r.integers(-3, 4, n).astype(np.float64),     # sums that hit powers of two
        r.standard_normal(n) * 1e-23,                # denormal squares
        np.zeros(n),
        np.where(np.arange(n) == n - 1, 3.0, 0.0),
        np.where(np.arange(n) == n // 2, 1e20, r.standard_normal(n)),  # inf from there on
        np.repeat(stuck, 4)[:n],
        np.repeat(late, 4)[:n],
        np.geomspace(1e-6, 1e6, n),                  # a new binade every few adds
    ]
    return np.ascontiguousarray(np.stack(rows).astype(np.float32))


@pytest.mark.parametrize("K", [64, 1024, 1088, 2048, 2112, 4096, 4160, 8192])
def test_one_token_prologue(hip, K):
    """bm_hip_bitlinear_dev at one token: the fused row kernel's prologue."""
    N = 128
    packed = bh.synth_ternary(5, 1, N, K, bh.SYNTH_P0_40)
    g = (np.random.default_rng(K).standard_normal(K) * 0.02).astype(np.float32)
    x = rows_for(K, K)
    dg, dw = DB.from_array(g), DB.from_array(packed)
    for i in range(x.shape[0]):
        print("one token K=%d row %d" % (K, i), flush=True)
        dx, do, dq, ds = DB.from_array(x[i]), DB(4 * N), DB(K), DB(4)
        da = DB(hip.bm_hip_act_bytes(1, K))
        bh.check(hip.bm_hip_bitlinear_dev(dx.ptr, 1, K, dg.ptr, dw.ptr, N, 0.02, 1, do.ptr, dq.ptr,
                                          K, ds.ptr, da.ptr, None), "bitlinear")
        hip.bm_hip_synchronize()
        on, oq, osc, _ = native.orc_quantize_rows(x[i:i + 1], g)
        np.testing.assert_array_equal(dq.download(K, np.int8), oq[0])
        same_bits(ds.download(1, np.float32), osc, "scale row %d" % i)
        ref, _, _ = native.orc_bitlinear(x[i:i + 1], packed, N, K, 0.02, g)
        same_bits(do.download(N, np.float32), ref[0], "out row %d" % i)


@pytest.mark.parametrize("n", [1, 3, 5, 1000, 1024, 1027, 2048, 2052, 4096, 4099, 8190, 8192, 8200])
def test_token_block_quantizer(hip, n):
    """The per-token quantizer at few tokens: 16-byte and scalar loads, every
    elements-per-lane class, the K % 4 tail, int8 rows of any stride."""
    x = rows_for(n, 9 * n) if n >= 16 else rnd_rows(n)
    M = x.shape[0]
    g = (np.random.default_rng(n).standard_normal(n) * 0.02).astype(np.float32)
    on, oq, osc, _ = native.orc_quantize_rows(x, g)
    for stride, qs in ((n, n), (n + 1, n + 3), ((n + 3) // 4 * 4, (n + 15) // 16 * 16)):
        print("quantize n=%d x stride=%d int8 stride=%d" % (n, stride, qs), flush=True)
        xs = np.zeros((M, stride), np.float32)
        xs[:, :n] = x
        dx, dg, dn, ds = DB.from_array(xs), DB.from_array(g), DB(4 * M * n), DB(4 * M)
        dq = DB.from_array(np.full((M, qs), 99, np.int8))
        bh.check(hip.bm_hip_quantize_dev(dx.ptr, M, n, stride, dg.ptr, dn.ptr, dq.ptr, qs, ds.ptr,
                                         None, None), "quantize")
        hip.bm_hip_synchronize()
        same_bits(dn.download((M, n), np.float32), on, "x_norm")
        q = dq.download((M, qs), np.int8)
        np.testing.assert_array_equal(q[:, :n], oq)
        assert (q[:, n:] == 99).all()
        same_bits(ds.download(M, np.float32), osc, "scale")


@pytest.mark.parametrize("n", [1, 2, 3, 4, 7, 8])
@pytest.mark.parametrize("M", [1, 512, 513])
def test_narrow_rows(hip, n, M):
    """Rows of a few values: both quantizers on either side of their rule, from
    which the norm and the int8 rows come."""
    print("quantize M=%d n=%d" % (M, n), flush=True)
    r = np.random.default_rng(100 * n + M)
    x = (r.standard_normal((M, n)) * np.exp(3.0 * r.standard_normal((M, 1)))).astype(np.float32)
    g = (r.standard_normal(n) * 0.02).astype(np.float32)
    dx, dg, dn, dq, ds = DB.from_array(x), DB.from_array(g), DB(4 * M * n), DB(M * n), DB(4 * M)
    bh.check(hip.bm_hip_quantize_dev(dx.ptr, M, n, n, dg.ptr, dn.ptr, dq.ptr, n, ds.ptr, None, None),
             "quantize")
    hip.bm_hip_synchronize()
    on, oq, osc, _ = native.orc_quantize_rows(x, g)
    same_bits(dn.download((M, n), np.float32), on, "x_norm")
    np.testing.assert_array_equal(dq.download((M, n), np.int8), oq)
    same_bits(ds.download(M, np.float32), osc, "scale")


def rnd_rows(n):
    return np.random.default_rng(n).standard_normal((5, n)).astype(np.float32)


@pytest.mark.parametrize("M", [1, 2, 7, 8, 9, 37])
@pytest.mark.parametrize("K", [1, 3, 4, 63, 1000, 1023, 1024 + 4, 1025, 2050, 4100])
def test_generic_product(hip, M, K):
    """Widths that are not multiples of 64: int32 totals and the fp32 epilogue
    with its remainder columns; rows that do not fill a block; code 11."""
    for N in (1, 15, 17, 130):
        print("generic M=%d K=%d N=%d" % (M, K, N), flush=True)
        r = np.random.default_rng(M * 131 + K * 7 + N)
        kb = (K + 3) // 4
        packed = r.integers(0, 256, (N, kb)).astype(np.uint8)
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
        dxq, dt = DB.from_array(xq), DB(4 * M * N)
        bh.check(hip.bm_hip_ternary_gemm_i32_dev(dxq.ptr, M, K + 3, dw.ptr, N, K, 0, dt.ptr, da.ptr,
                                                 None), "int32")
        hip.bm_hip_synchronize()
        want = native.orc_gemm_i32(np.ascontiguousarray(xq[:, :K]), packed, N, K)
        np.testing.assert_array_equal(dt.download((M, N), np.int32), want)
