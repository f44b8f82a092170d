"""The host-pointer batch call above the zero-copy size: results that leave in
published slices, x read from the pinned stage or copied, and the memory that
the call holds."""
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


def host_call(hip, x, packed, g, rows, stride, norm=True, quant=True):
    M, n = x.shape
    w, nw = bh.make_tensor(packed, rows, n, 0.02), bh.make_tensor(data=g)
    out = np.full((M, rows), np.nan, np.float32)
    xn = np.full(n + 4, 7.0, np.float32)
    xq = np.full((M, stride), 99, np.int8)
    hip.hip_bitlinear_forward_batch(ptr(x), M, n, C.byref(w), C.byref(nw), ptr(out),
                                    ptr(xn) if norm else None, ptr(xq) if quant else None, stride)
    return out, xn, xq


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
