"""The work that a user of this library has it do, as cases that can be timed.

Each case goes through the public entry points (include/bm_hip.h, by way of
bitmamba_hip): single BitLinear products on device buffers, int8-input
products, the dispatch-table calls on host buffers, the sampler, and whole
generations on the device-resident model.  Every entry point promises the
bits of the reference's scalar kernels, so every tolerance is "exact".
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "bitmamba.c_amd"))
import bitmamba_hip as bh  # noqa: E402

# The model shapes of bench.py: vocabulary 50257, 24 layers
MODELS = {
    "1b": dict(vocab=50257, d_model=2048, n_layers=24, n_heads=64, seed=1000, dist=bh.SYNTH_P0_40),
    "255m": dict(vocab=50257, d_model=1024, n_layers=24, n_heads=32, seed=255,
                 dist=bh.SYNTH_UNIFORM),
}
_models = {}  # a serving program loads its weights once
_images = {}  # model images registered with bm_hip_set_mmap: they live as long as the program


def listed():
    return [
        # one token through one in_proj-sized product, the smallest call: the
        # in_proj of a 255M-shape layer at decode (bench.py's single BitLinear)
        dict(name="linear_m1", kind="linear", M=1, K=1024, N=4384, canonical=True),
        # a handful of tokens (a short prompt) through the 1B in_proj
        dict(name="linear_few", kind="linear", M=13, K=2048, N=8384, canonical=True),
        # an ordinary prompt through the 1B out_proj, a count that fills no tile
        dict(name="linear_mid", kind="linear", M=300, K=4096, N=2048, canonical=True),
        # a long prompt through the in_proj, the largest fp32 product of bench.py
        dict(name="linear_big", kind="linear", M=2048, K=2048, N=8512, canonical=True),
        # widths of no power of two and no multiple of 64, weights as the
        # caller's file holds them (code 11 allowed)
        dict(name="linear_odd", kind="linear", M=37, K=1000, N=1003, canonical=False),
        # int8 activations that are quantized elsewhere, few and many tokens
        # (bench.py's stress shape)
        dict(name="int8_few", kind="int8", M=16, K=8192, N=8192, canonical=False),
        dict(name="int8_big", kind="int8", M=4096, K=8192, N=8192, canonical=False),
        # the reference engine's own calls through its dispatch table: host
        # buffers, weights of a registered image; one token and a prompt
        dict(name="host_m1", kind="host", M=1, d_model=1024, heads=32, part="in"),
        dict(name="host_batch", kind="host", M=256, d_model=1024, heads=32, part="in"),
        # one token drawn by nucleus sampling over the whole vocabulary
        dict(name="sample_nucleus", kind="sample", V=50257, sigma=4.0, temp=0.8, min_p=0.0,
             top_p=0.9, top_k=0),
        # a chat answer: a short prompt, then greedy decode token by token
        dict(name="decode_1b", kind="generate", model="1b", prompt=9, steps=64, temp=0.0,
             min_p=0.0, top_p=1.0, top_k=0, penalty=1.0, stop=False),
        # the first token after a long prompt
        dict(name="first_token_1b", kind="generate", model="1b", prompt=1025, steps=1, temp=0.0,
             min_p=0.0, top_p=1.0, top_k=0, penalty=1.0, stop=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "int8", "host", "sample", "generate",
                       "generate"])
    if kind in ("linear", "int8"):
        # widths: those of the models, other multiples of 64, and any
        K = rng.choice([1024, 2048, 4096, 64 * _log(rng, 2, 128), _log(rng, 128, 8192)])
        N = rng.choice([2 * K + 96, 4 * K + 192, _log(rng, 128, 12000)])
        M = rng.choice([1, _log(rng, 2, 64), _log(rng, 2, 4096)])
        if K % 64:
            M = min(M, 256)
        while M > 1 and M * N * K > 4096 * 8192 * 8192:
            M //= 2
        return dict(kind=kind, M=M, K=K, N=N, canonical=rng.random() < 0.6)
    if kind == "host":
        heads = rng.choice([4, 8, 16, 32])
        d_model = 32 * heads if rng.random() < 0.7 else 64 * rng.randint(1, 4) * heads // 4
        return dict(kind=kind, M=rng.choice([1, _log(rng, 2, 512)]), d_model=d_model, heads=heads,
                    part=rng.choice(["in", "out"]))
    if kind == "sample":
        return dict(kind=kind, V=_log(rng, 1000, 120000), sigma=rng.uniform(2.0, 6.0),
                    temp=rng.choice([0.7, 0.8, 1.0, 1.3]), min_p=rng.choice([0.0, 0.05]),
                    top_p=rng.choice([0.9, 0.95, 1.0]), top_k=rng.choice([0, 40, 100]))
    long_prompt = rng.random() < 0.5
    sampled = rng.random() < 0.5
    return dict(kind=kind, model=rng.choice(["1b", "255m"]),
                prompt=_log(rng, 40, 1100) if long_prompt else rng.randint(1, 40),
                steps=rng.randint(1, 8) if long_prompt else rng.randint(8, 64),
                temp=0.8 if sampled else 0.0, min_p=0.05 if sampled else 0.0,
                top_p=0.9 if sampled else 1.0, top_k=40 if sampled else 0,
                penalty=rng.choice([1.0, 1.15]), stop=rng.random() < 0.3)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 7919 + 11)
    return g


def _packed(g, N, K, canonical):
    """Packed ternary rows: p(0) = 0.4 and p(+-1) = 0.3; where the weights are not
    declared canonical, half of the +1 are written as code 11."""
    kb = (K + 3) // 4
    u = torch.rand((N, kb, 4), generator=g, device="cuda")
    code = torch.ones((N, kb, 4), dtype=torch.uint8, device="cuda")
    code[u < 0.3] = 0
    code[u >= 0.7] = 2
    if not canonical:
        code[u >= 0.85] = 3
    return (code[..., 0] | (code[..., 1] << 2) | (code[..., 2] << 4) | (code[..., 3] << 6)).contiguous()


def _activations(g, M, K):
    """Residual-stream rows: each token at a scale of its own, a few wide channels."""
    x = torch.randn((M, K), generator=g, device="cuda")
    x *= torch.exp(torch.randn((M, 1), generator=g, device="cuda") * 0.7)
    return x * torch.exp(torch.randn((1, K), generator=g, device="cuda") * 0.3)


def _scale(K):
    return 1.0 / math.sqrt(K)


def _linear_inputs(case, seed):
    g = _generator(seed)
    M, K, N = case["M"], case["K"], case["N"]
    x = _activations(g, M, K)
    gamma = 1.0 + 0.1 * torch.randn(K, generator=g, device="cuda")
    return x, gamma, _packed(g, N, K, case["canonical"])


def _int8_inputs(case, seed):
    g = _generator(seed)
    xq = torch.randn((case["M"], case["K"]), generator=g, device="cuda") * 32.0
    return xq.round().clamp(-127, 127).to(torch.int8), _packed(g, case["N"], case["K"],
                                                              case["canonical"])


def _image(case):
    key = (case["d_model"], case["heads"])
    if key not in _images:
        blob = bh.synth_model(256, case["d_model"], 1, case["heads"], 7, fp_sigma=0.5)
        _images[key] = blob
    # the last image registered counts: a program has one, the cases several
    if not bh.lib().bm_hip_set_mmap(bh.ptr(_images[key]), _images[key].nbytes):
        raise RuntimeError(bh.last_error())
    return _images[key]


def _host_tensors(case):
    blob = _image(case)
    which = (bh.BM_L_IN_PROJ, bh.BM_L_IN_NORM) if case["part"] == "in" else (bh.BM_L_OUT_PROJ,
                                                                            bh.BM_L_OUT_NORM)
    return [bh.image_tensors(blob, 0, w) for w in which]


def _host_x(case, seed, K):
    r = np.random.RandomState(seed % (2 ** 31))
    x = r.standard_normal((case["M"], K)) * np.exp(0.7 * r.standard_normal((case["M"], 1)))
    return x.astype(np.float32)


def _logits(case, seed):
    g = _generator(seed)
    return torch.randn(case["V"], generator=g, device="cuda") * case["sigma"]


def prepare(case, seed):
    if not bh.lib().bm_hip_init():
        raise RuntimeError(bh.last_error())
    L, kind = bh.lib(), case["kind"]
    s = dict(case)
    if kind == "linear":
        M, K, N = case["M"], case["K"], case["N"]
        s["x"], s["gamma"], s["w"] = _linear_inputs(case, seed)
        s["out"] = torch.empty((M, N), device="cuda")
        s["xq"] = torch.empty((M, K), dtype=torch.int8, device="cuda")
        s["sx"] = torch.empty(M, device="cuda")
        s["act"] = torch.empty(L.bm_hip_act_bytes(M, K), dtype=torch.uint8, device="cuda")
    elif kind == "int8":
        M, K, N = case["M"], case["K"], case["N"]
        s["xq"], s["w"] = _int8_inputs(case, seed)
        s["out"] = torch.empty((M, N), dtype=torch.int32, device="cuda")
        s["act"] = torch.empty(L.bm_hip_i8_act_bytes(M, K), dtype=torch.uint8, device="cuda")
    elif kind == "host":
        s["w"], s["nw"] = _host_tensors(case)
        M, K, N = case["M"], s["w"].cols, s["w"].rows
        s["x"] = _host_x(case, seed, K)
        s["out"] = np.empty((M, N), np.float32)
        s["xn"] = np.empty(K, np.float32)
        s["xq"] = np.empty((M, K), np.int8)
    elif kind == "sample":
        pad = -case["V"] % 4
        s["src"] = torch.nn.functional.pad(_logits(case, seed), (0, pad))
        s["logits"] = torch.empty_like(s["src"])
        s["rng"] = torch.tensor([(seed * 0x9E3779B97F4A7C15 + 0x853C49E6748FEA9B) % 2 ** 63],
                                dtype=torch.int64, device="cuda")
        s["token"] = torch.empty(1, dtype=torch.int32, device="cuda")
        s["work"] = torch.zeros(L.bm_hip_sample_workspace_bytes(case["V"]), dtype=torch.uint8,
                                device="cuda")
    else:
        if case["model"] not in _models:
            c = MODELS[case["model"]]
            _models[case["model"]] = bh.Model(
                bh.synth_model(c["vocab"], c["d_model"], c["n_layers"], c["n_heads"], c["seed"],
                               dist=c["dist"]))
        s["m"] = _models[case["model"]]
        r = np.random.RandomState(seed % (2 ** 31))
        s["tokens"] = r.randint(1, 50000, case["prompt"]).astype(np.int32)
        s["seed"] = int(seed) + 1
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    L, kind = bh.lib(), s["kind"]
    if kind == "linear":
        M, K, N = s["M"], s["K"], s["N"]
        bh.check(L.bm_hip_bitlinear_dev(s["x"].data_ptr(), M, K, s["gamma"].data_ptr(),
                                        s["w"].data_ptr(), N, _scale(K), int(s["canonical"]),
                                        s["out"].data_ptr(), s["xq"].data_ptr(), K,
                                        s["sx"].data_ptr(), s["act"].data_ptr(), None))
        return {"out": s["out"], "xq": s["xq"], "scale": s["sx"]}
    if kind == "int8":
        M, K, N = s["M"], s["K"], s["N"]
        bh.check(L.bm_hip_ternary_gemm_i32_dev(s["xq"].data_ptr(), M, K, s["w"].data_ptr(), N, K,
                                               int(s["canonical"]), s["out"].data_ptr(),
                                               s["act"].data_ptr(), None))
        return s["out"]
    if kind == "host":
        K = s["w"].cols
        if s["M"] == 1:
            L.hip_bitlinear_forward(bh.ptr(s["x"]), K, ctypes.byref(s["w"]), ctypes.byref(s["nw"]),
                                    bh.ptr(s["out"]), bh.ptr(s["xn"]), bh.ptr(s["xq"]))
        else:
            L.hip_bitlinear_forward_batch(bh.ptr(s["x"]), s["M"], K, ctypes.byref(s["w"]),
                                          ctypes.byref(s["nw"]), bh.ptr(s["out"]), bh.ptr(s["xn"]),
                                          bh.ptr(s["xq"]), K)
        return {"out": s["out"], "x_norm": s["xn"], "xq": s["xq"]}
    if kind == "sample":
        # the decode leaves new logits for every token: the sampler scales them in place
        bh.check(L.bm_hip_copy_dev(s["logits"].data_ptr(), s["src"].data_ptr(),
                                   4 * s["src"].numel(), None))
        bh.check(L.bm_hip_sample_advanced(s["logits"].data_ptr(), s["V"], s["temp"], s["min_p"],
                                          s["top_p"], s["top_k"], s["rng"].data_ptr(),
                                          s["work"].data_ptr(), s["token"].data_ptr(),
                                          L.bm_hip_stream()))
        return {"logits": s["logits"], "rng": s["rng"], "token": s["token"]}
    m = s["m"]
    m.reset()
    m.set_sampler(s["temp"], s["min_p"], s["top_p"], s["top_k"])
    m.seed(s["seed"])
    tokens, _ = m.generate(s["tokens"], s["steps"], penalty=s["penalty"], stop_on_eos=s["stop"])
    # the logits of the last step and the session as the chat saves it
    return {"logits": m.logits(), "state": np.frombuffer(m.state_save(), np.uint8),
            "tokens": tokens}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _host_shape(case):
    dm, di = case["d_model"], 2 * case["d_model"]
    return (dm, 2 * di + 3 * case["heads"]) if case["part"] == "in" else (di, dm)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, K, N = case["M"], case["K"], case["N"]
        b = 4 * M * K + 4 * K + N * ((K + 3) // 4) + 4 * M * N + M * K + 4 * M
        return {"bytes": b, "flops": 2 * M * N * K}
    if kind == "int8":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": M * K + N * ((K + 3) // 4) + 4 * M * N, "flops": 2 * M * N * K}
    if kind == "host":
        M, (K, N) = case["M"], _host_shape(case)
        return {"bytes": 4 * M * K + 8 * K + N * (K // 4) + 4 * M * N + M * K,
                "flops": 2 * M * N * K}
    if kind == "sample":
        return {"bytes": 8 * case["V"], "flops": 4 * case["V"]}
    c = MODELS[case["model"]]
    dm, di, nh, nl, V = c["d_model"], 2 * c["d_model"], c["n_heads"], c["n_layers"], c["vocab"]
    layer = (2 * di + 3 * nh) * dm + dm * di  # ternary weights of a layer
    state = 4 * 4 * di                        # conv ring and state, fp32
    n = case["prompt"] - 1
    per_layer = layer // 4 + 4 * (dm + di) + 4 * 7 * di + 2 * state
    byt = (nl * per_layer + 4 * n * dm if n else 0) + case["steps"] * (
        nl * per_layer + V * dm // 4 + 4 * V + 4 * dm)
    return {"bytes": byt,
            "flops": 2 * n * nl * layer + case["steps"] * 2 * (nl * layer + V * dm)}


def tolerance(case):
    # int32 totals, int8 values and the fp32 epilogue follow the reference's
    # scalar kernels operation by operation; so do the sampler and the model
    return "exact"


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _decode(packed, K):
    sh = torch.tensor([0, 2, 4, 6], device=packed.device, dtype=torch.uint8)
    w = ((packed.unsqueeze(-1) >> sh) & 3).to(torch.int8).reshape(packed.shape[0], -1)[:, :K]
    return (w - 1).clamp(max=1).to(torch.float64)


def _exact_linear(x, gamma, packed, K, w_scale):
    x, gamma = x.double(), gamma.double()
    xn = x * torch.rsqrt(x.square().mean(1, keepdim=True) + 1e-6) * gamma
    scale = 127.0 / (xn.abs().amax(1, keepdim=True) + 1e-5)
    q = torch.trunc(xn * scale + torch.copysign(torch.full_like(xn, 0.5), xn)).clamp(-128, 127)
    return q @ _decode(packed, K).T / (scale * w_scale), xn, q, scale[:, 0]


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        K = case["K"]
        x, gamma, w = _linear_inputs(case, seed)
        out, _, q, scale = _exact_linear(x, gamma, w, K, float(np.float32(_scale(K))))
        return {"out": out, "xq": q.to(torch.int8), "scale": scale}
    if kind == "int8":
        xq, w = _int8_inputs(case, seed)
        return (xq.double() @ _decode(w, case["K"]).T).to(torch.int32)
    if kind == "host":
        # the weights are those of the image, read out of it here
        w, nw = _host_tensors(case)
        K, N = w.cols, w.rows
        packed = np.ctypeslib.as_array(w.packed_data, (N, K // 4)).copy()
        gamma = np.ctypeslib.as_array(nw.data, (K,)).copy()
        out, xn, q, _ = _exact_linear(torch.from_numpy(_host_x(case, seed, K)),
                                      torch.from_numpy(gamma), torch.from_numpy(packed), K,
                                      float(w.scale))
        return {"out": out, "x_norm": xn[-1], "xq": q.to(torch.int8)}
    if kind == "sample":
        pad = -case["V"] % 4
        lg = _logits(case, seed).double() / float(np.float32(case["temp"]))
        # the drawn token and the generator's state have no 64-bit value; the
        # padding past the vocabulary is not scaled (it is zero)
        return {"logits": torch.nn.functional.pad(lg, (0, pad)), "rng": None, "token": None}
    return None  # a whole model on the CPU in 64 bits takes minutes
