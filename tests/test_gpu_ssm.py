"""The prefill SSM as one pipeline (bm_model.hip, k_ssm_fused) and in three
phases per 1024-token chunk (head dims that are not multiples of 16): prompts at
the edges of the pipeline's 64-token tiles and of the chunks, carried conv rings
at every position, grids that are and are not multiples of 8 blocks; states and
logits bit-exact against the oracle's token-serial prefill."""
import numpy as np
import pytest

import native
from native import bh, ptr, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d_model,n_heads", [(64, 8), (64, 4), (192, 8), (256, 4), (128, 2), (96, 8),
                                             (64, 1)])
def test_prefill_tiles(hip, d_model, n_heads):
    blob = bh.synth_model(97, d_model, 2, n_heads, 7 * d_model + n_heads, fp_sigma=0.5)
    m = bh.Model(blob)
    O = native.oracle()
    h = O.orc_model_load(ptr(blob), blob.nbytes)
    try:
        for parts in ([1], [2, 1], [3], [62], [63, 1], [64], [65], [2, 64], [66, 67], [128], [129],
                      [191, 3, 1]):
            print("ssm d_model=%d heads=%d parts=%s" % (d_model, n_heads, parts), flush=True)
            m.reset()
            O.orc_model_free(h)
            h = O.orc_model_load(ptr(blob), blob.nbytes)
            toks = bh.synth_prompt(sum(parts) + 3, 97, sum(parts) + 1)
            at = 0
            for n in parts:
                p = toks[at:at + n].copy()
                m.prefill(p)
                O.orc_model_prefill(h, ptr(p), p.size)
                at += n
            for layer in range(m.n_layers):
                cs, ss, pos = m.layer_state(layer)
                ocs = np.empty((3, m.d_inner), np.float32)
                oss = np.empty(m.d_inner, np.float32)
                assert pos == O.orc_model_layer_state(h, layer, ptr(ocs), ptr(oss))
                same_bits(cs, ocs, "conv_state[%d]" % layer)
                same_bits(ss, oss, "ssm_state[%d]" % layer)
            hist = np.array(toks, np.int32)
            a = m.step(int(toks[-1]), hist[-256:], 1.0)
            b = O.orc_model_step(h, int(toks[-1]), ptr(hist[-256:].copy()), min(hist.size, 256), 1.0)
            same_bits(m.logits(), np.ctypeslib.as_array(O.orc_model_logits(h), (m.vocab,)),
                      "logits after %s" % parts)
            assert a == b
    finally:
        O.orc_model_free(h)
        m.free()


@pytest.mark.parametrize("d_model,n_heads", [(96, 8), (64, 16), (120, 8)])
def test_three_phase_chunks(hip, d_model, n_heads):
    """Prompts of several 1024-token chunks at head dims 24, 8 and 30: the conv
    ring and the states handed from chunk to chunk, the planes that hold one
    chunk, a second chunk of a single token."""
    blob = bh.synth_model(97, d_model, 2, n_heads, 3 * d_model + n_heads, fp_sigma=0.5)
    m = bh.Model(blob)
    O = native.oracle()
    for parts in ([1024], [1025], [2050], [7, 1030], [1026, 2, 1100], [3073]):
        print("three-phase d_model=%d heads=%d parts=%s" % (d_model, n_heads, parts), flush=True)
        m.reset()
        h = O.orc_model_load(ptr(blob), blob.nbytes)
        try:
            toks = bh.synth_prompt(sum(parts) + 5, 97, sum(parts) + 1)
            at = 0
            for n in parts:
                p = toks[at:at + n].copy()
                m.prefill(p)
                O.orc_model_prefill(h, ptr(p), p.size)
                at += n
            for layer in range(m.n_layers):
                cs, ss, pos = m.layer_state(layer)
                ocs = np.empty((3, m.d_inner), np.float32)
                oss = np.empty(m.d_inner, np.float32)
                assert pos == O.orc_model_layer_state(h, layer, ptr(ocs), ptr(oss))
                same_bits(cs, ocs, "conv_state[%d]" % layer)
                same_bits(ss, oss, "ssm_state[%d]" % layer)
            hist = np.array(toks[-256:], np.int32)
            a = m.step(int(toks[-1]), hist, 1.0)
            assert a == O.orc_model_step(h, int(toks[-1]), ptr(hist), hist.size, 1.0)
            same_bits(m.logits(), np.ctypeslib.as_array(O.orc_model_logits(h), (m.vocab,)),
                      "logits after %s" % parts)
        finally:
            O.orc_model_free(h)
    m.free()
