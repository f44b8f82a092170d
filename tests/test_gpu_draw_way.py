"""Which way a draw without top-k goes (bm_sample.hip): the parallel draw leaves
the candidates' buffer alone and only lists (index, logit) pairs; the sequential
walk writes probabilities into one or the other.  The workspace is filled with
a pattern before every call, so its contents tell."""
import ctypes as C

import numpy as np
import pytest

import native
from native import bh, ptr, same_bits

pytestmark = pytest.mark.gpu
DB = bh.DeviceBuffer
CAND = np.dtype([("id", np.int32), ("val", np.float32)])


class Sampler:
    def __init__(self, hip, V):
        self.hip, self.V = hip, V
        self.seg = ((V + 63) // 64 + 3) & ~3
        self.ws = DB(hip.bm_hip_sample_workspace_bytes(V))
        assert self.ws.ptr % 16 == 0
        self.pad = (V + 3) // 4 * 4
        self.dl, self.dr, self.dt = DB(4 * self.pad), DB(8), DB(4)

    def draw(self, logits, temp, min_p, top_p, top_k, rng):
        """(token, generator state, True for the sequential way); the token, the
        state and the scaled logits are the oracle's.  self.tried: whether the
        parallel draw's sums were formed at all."""
        V, hip = self.V, self.hip
        buf = np.zeros(self.pad, np.float32)
        buf[:V] = logits
        for b, a in ((self.dl, buf), (self.dr, np.array([rng], np.uint64))):
            bh.check(hip.bm_hip_memcpy_h2d(b.ptr, ptr(a), a.nbytes), "upload")
        n_cand = (V + 1) // 2 * 2 + 64 * self.seg
        sums = 8 * (2 * 64 + 2048) + 4 * 64 * self.seg  # after the candidates: sums and terms
        bh.check(hip.bm_hip_memset(self.ws.ptr, 0xA5, 8 * n_cand + sums), "pattern")
        bh.check(hip.bm_hip_sample_advanced(self.dl.ptr, V, temp, min_p, top_p, top_k, self.dr.ptr,
                                            self.ws.ptr, self.dt.ptr, None), "sample_advanced")
        hip.bm_hip_synchronize()
        tok = int(self.dt.download(1, np.int32)[0])
        state = int(self.dr.download(1, np.uint64)[0])
        scaled = self.dl.download(V, np.float32)
        ref, st = np.array(logits, np.float32), C.c_uint64(rng)
        want = native.oracle().orc_sample(ptr(ref), V, temp, min_p, top_p, top_k, C.byref(st))
        same_bits(scaled, ref, "scaled logits")
        assert (tok, state) == (want, st.value)
        got = self.ws.download(8 * n_cand + sums, np.uint8)
        self.tried = bool((got[8 * n_cand:] != 0xA5).any())
        got = got[:8 * n_cand].view(CAND)
        cand, pre = got[:(V + 1) // 2 * 2], got[(V + 1) // 2 * 2:]
        touched = (cand.view(np.uint64) != 0xA5A5A5A5A5A5A5A5).any()
        pre = pre[pre.view(np.uint64) != 0xA5A5A5A5A5A5A5A5]
        other = (pre["val"].view(np.uint32) != scaled[pre["id"]].view(np.uint32)).any()
        return tok, state, bool(touched or other)


@pytest.mark.parametrize("V,min_p", [(50257, 0.0), (50257, 0.05), (1000, 0.05), (1000, 0.0)])
def test_draws_that_give_up(hip, V, min_p):
    """Of 200 vectors at most 2 go the sequential way.  Expected: sums of up to
    a few hundred terms are exact; 50257 terms of any spread miss a rounding of
    their sum by less than the bound about n 2^-26 = 0.07 % of the time."""
    s = Sampler(hip, V)
    r = np.random.default_rng(V)
    rng, gave_up = 0x853C49E6748FEA9B, 0
    for i in range(200):
        logits = (r.standard_normal(V) * 4.0).astype(np.float32)
        _, rng, seq = s.draw(logits, 0.8, min_p, 0.9, 0, rng)
        gave_up += seq
    print("V=%d min_p=%g: %d of 200 sequential" % (V, min_p, gave_up), flush=True)
    assert gave_up <= 2


@pytest.mark.parametrize("V,top_ps", [(8, (0.125, 0.25, 0.5, 0.875)), (64, (0.25, 0.75)),
                                      (1024, (0.5, 0.75))])
def test_sums_that_hit_top_p(hip, V, top_ps):
    """Equal logits: probabilities 1/V, sums that equal top_p exactly."""
    s = Sampler(hip, V)
    for top_p in top_ps:
        for i in range(8):
            tok, _, seq = s.draw(np.full(V, 1.5, np.float32), 1.0, 0.0, top_p, 0, 977 * i + 5)
            print("V=%d top_p=%g: token %d" % (V, top_p, tok), flush=True)
            assert tok < V * top_p and not seq


def test_sums_at_midpoints(hip):
    """Few candidates whose softmax sum lies halfway between two floats."""
    r = np.random.default_rng(3)
    found = 0
    while found < 24:
        V = int(r.integers(2, 9))
        logits = (r.standard_normal(V)).astype(np.float32)
        d = (logits - logits.max()).astype(np.float32)
        ex = np.empty_like(d)
        native.oracle().orc_expf_array(ptr(d), ptr(ex), V)
        total = float(ex.astype(np.float64).sum())
        f = np.float32(total)
        half = float(np.spacing(f)) / 2
        if abs(total - float(f)) != half:
            continue
        found += 1
        s = Sampler(hip, V)
        print("midpoint V=%d %r" % (V, total), flush=True)
        for top_p in (0.5, 0.9):
            _, _, seq = s.draw(logits, 1.0, 0.0, top_p, 0, int(r.integers(1, 2 ** 62)))
            assert not seq


@pytest.mark.parametrize("V,min_p,top_p,top_k,tried", [
    (95, 0.0, 1.0, 0, False), (96, 0.0, 1.0, 0, True), (5, 0.0, 0.9, 0, True),
    (300, 0.0, 1.0, 299, False), (300, 0.0, 1.0, 300, True), (300, 0.0, 1.0, 301, True),
    (5000, 0.0, 1.0, 257, False), (5000, 0.0, 0.9, 257, True), (5000, 0.05, 1.0, 0, False),
    (1, 0.0, 1.0, 0, False)])
def test_when_it_is_tried(hip, V, min_p, top_p, top_k, tried):
    """Calls that only the sequential way can decide, or decides sooner, do not
    pay for the parallel draw's sums."""
    s = Sampler(hip, V)
    r = np.random.default_rng(V + top_k)
    for i in range(4):
        print("V=%d min_p=%g top_p=%g top_k=%d" % (V, min_p, top_p, top_k), flush=True)
        s.draw((r.standard_normal(V) * 2.0).astype(np.float32), 0.9, min_p, top_p, top_k, 31 * i + 7)
        assert s.tried == tried


def test_positive_infinity(hip):
    """One infinite logit: every probability is NaN or 0 in the reference, and the
    draw goes the sequential way."""
    V = 1000
    s = Sampler(hip, V)
    logits = np.random.default_rng(5).standard_normal(V).astype(np.float32)
    logits[417] = np.inf
    print("+inf", flush=True)
    _, _, seq = s.draw(logits, 1.0, 0.0, 1.0, 0, 12345)
    assert seq
