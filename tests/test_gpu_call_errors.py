"""Model calls that are refused or fail: what they return, and that nothing of
them is left running or behind on the device."""
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
