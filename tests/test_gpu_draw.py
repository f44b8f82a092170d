"""The draw without top-k (bm_sample.hip, draw_parallel): tokens, scaled logits
and generator states against the oracle where its decisions can go wrong:
one-entry and one-block vocabularies, both sides of the 256-entry heap, small
and very large nuclei, whole vocabularies, tied probabilities, top_k above
256, unaligned workspaces."""
import ctypes as C

import numpy as np
import pytest

import native
from native import bh, same_bits

pytestmark = pytest.mark.gpu
DB = bh.DeviceBuffer


def draw(hip, logits, temp, min_p, top_p, top_k, rng, ws, off=0):
    V = logits.size
    buf = np.zeros((V + 3) // 4 * 4, np.float32)
    buf[:V] = logits
    dl, dr, dt = DB.from_array(buf), DB.from_array(np.array([rng], np.uint64)), DB(4)
    bh.check(hip.bm_hip_sample_advanced(dl.ptr, V, temp, min_p, top_p, top_k, dr.ptr,
                                        ws.ptr + off, dt.ptr, None), "sample_advanced")
    hip.bm_hip_synchronize()
    return (int(dt.download(1, np.int32)[0]), dl.download(V, np.float32),
            int(dr.download(1, np.uint64)[0]))


def check(hip, logits, temp, min_p, top_p, top_k, rng, ws, off=0):
    tok, scaled, state = draw(hip, logits, temp, min_p, top_p, top_k, rng, ws, off)
    ref = logits.copy()
    st = C.c_uint64(rng)
    want = native.oracle().orc_sample(native.ptr(ref), ref.size, temp, min_p, top_p, top_k,
                                      C.byref(st))
    same_bits(scaled, ref, "scaled logits")
    assert (tok, state) == (want, st.value)


@pytest.mark.parametrize("V", [1, 5, 64, 255, 256, 257, 4097, 50257, 256000])
@pytest.mark.parametrize("top_p", [0.3, 0.9, 0.999, 1.0])
def test_draw(hip, V, top_p):
    ws = DB(hip.bm_hip_sample_workspace_bytes(V) + 4)
    r = np.random.default_rng(V)
    for sigma in (0.0, 0.5, 1.5, 4.0, 30.0):
        for min_p, top_k in ((0.0, 0), (0.01, 0), (0.0, 300)):
            print("draw V=%d top_p=%g sigma=%g min_p=%g top_k=%d" % (V, top_p, sigma, min_p, top_k),
                  flush=True)
            logits = (r.standard_normal(V) * sigma).astype(np.float32)
            check(hip, logits, 0.8, min_p, top_p, top_k, int(r.integers(1, 2 ** 63)), ws,
                  4 if top_k else 0)


@pytest.mark.parametrize("step", [0.25, 1.0, 1e-3])
def test_draw_ties(hip, step):
    """Logits on a grid: most probabilities are tied, the heap's order decides."""
    V = 5000
    ws = DB(hip.bm_hip_sample_workspace_bytes(V))
    r = np.random.default_rng(int(step * 1000))
    for top_p in (0.5, 0.95, 1.0):
        for i in range(8):
            print("ties step=%g top_p=%g draw %d" % (step, top_p, i), flush=True)
            logits = (np.round(r.standard_normal(V) * 3.0 / step) * step).astype(np.float32)
            check(hip, logits, 1.0, 0.0, top_p, 0, int(r.integers(1, 2 ** 63)), ws)


def test_draw_nonfinite(hip):
    V = 1000
    ws = DB(hip.bm_hip_sample_workspace_bytes(V))
    r = np.random.default_rng(1)
    base = (r.standard_normal(V) * 2.0).astype(np.float32)
    for name, at in (("-inf", -np.inf), ("nan", np.nan), ("lowest", -3.4e38)):
        for top_p in (0.9, 1.0):
            print("draw with %s top_p=%g" % (name, top_p), flush=True)
            logits = base.copy()
            logits[::3] = at
            check(hip, logits, 1.0, 0.0, top_p, 0, int(r.integers(1, 2 ** 63)), ws)
