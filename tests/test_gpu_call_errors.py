"""Model calls that are refused or fail: what they return, and that nothing of
them is left running or behind on the device."""
import ctypes as C

import numpy as np
import pytest

from native import bh, ptr, same_bits

pytestmark = pytest.mark.gpu


def test_step_refuses_negative_history(hip):
    """A negative history length is an error before anything is enqueued (the
    picked token would land below the token ring's start), and the model goes
    on as if the call had not been made."""
    blob = bh.synth_model(97, 64, 2, 4, 3, fp_sigma=0.5)
    a, b = bh.Model(blob), bh.Model(blob)
    hist = np.array([5, 9], np.int32)
    for m in (a, b):
        m.prefill(hist)
        m.step(9, hist)
    for n in (-1, -257, -2 ** 31):
        print("history length %d" % n, flush=True)
        assert hip.bm_hip_model_step(a.h, 9, ptr(hist), n, 1.3) == -1
        assert "history" in bh.last_error()
    assert a.state_save() == b.state_save()
    assert a.step(9, hist, 1.3) == b.step(9, hist, 1.3)
    same_bits(a.logits(), b.logits(), "logits")
    a.free()
    b.free()


def test_failed_generate_leaves_nothing_running(hip):
    """generate enqueues the prefill and then needs a longer token buffer, whose
    allocation is refused while this thread captures another stream in global
    mode: when the call returns its error the prefill has run to its end (the
    state, read without waiting for the model's stream, is a plain prefill's),
    and the model generates as before."""
    rt = C.CDLL("libamdhip64.so")
    vp = C.c_void_p
    rt.hipStreamCreateWithFlags.argtypes = [C.POINTER(vp), C.c_uint]
    rt.hipStreamBeginCapture.argtypes = [vp, C.c_int]
    rt.hipStreamEndCapture.argtypes = [vp, C.POINTER(vp)]
    rt.hipGraphDestroy.argtypes = [vp]
    rt.hipStreamDestroy.argtypes = [vp]
    blob = bh.synth_model(97, 256, 24, 8, 21, fp_sigma=0.5)
    prompt = bh.synth_prompt(5, 97, 4001)
    m, ref = bh.Model(blob), bh.Model(blob)
    first, _ = m.generate(prompt, 4)
    ref.prefill(prompt[:-1])
    m.reset()
    out = np.empty(5000, np.int32)  # more than the 4096 tokens a first call makes room for
    s, g = vp(), vp()
    assert rt.hipStreamCreateWithFlags(C.byref(s), 1) == 0
    assert rt.hipStreamBeginCapture(s, 0) == 0
    print("generate that fails after its prefill", flush=True)
    rc = hip.bm_hip_model_generate(m.h, ptr(prompt), prompt.size, out.size, 1.0, 0, ptr(out), None)
    why = bh.last_error()
    rt.hipStreamEndCapture(s, C.byref(g))  # invalidated by the refused call
    rt.hipGetLastError()                   # that error is this test's own
    got = m.layer_state(m.n_layers - 1)
    if g:
        rt.hipGraphDestroy(g)
    rt.hipStreamDestroy(s)
    assert rc == -1 and "hipMalloc" in why, (rc, why)
    want = ref.layer_state(m.n_layers - 1)
    same_bits(got[0], want[0], "conv_state")
    same_bits(got[1], want[1], "ssm_state")
    assert got[2] == want[2]
    m.reset()
    again, _ = m.generate(prompt, 4)
    assert list(again) == list(first)
    m.free()
    ref.free()


def test_reset_with_an_error_pending(hip):
    """reset does not fail for an error that the caller's own earlier HIP call
    left in the thread."""
    rt = C.CDLL("libamdhip64.so")
    m = bh.Model(bh.synth_model(97, 64, 2, 4, 3, fp_sigma=0.5))
    fresh = m.state_save()
    m.prefill(np.array([5, 9, 3], np.int32))
    assert m.state_save() != fresh
    print("reset with an error pending", flush=True)
    assert rt.hipMalloc(None, C.c_size_t(16)) != 0  # refused on the host: no pointer to fill
    rc = hip.bm_hip_model_reset(m.h)
    rt.hipGetLastError()
    assert rc == 0, bh.last_error()
    assert m.state_save() == fresh
    m.free()
