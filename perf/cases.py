"""The work this library is measured on: what a program that serves mixture-of-experts layers
has it do, through the entry points of ``coalsack_amd.capi`` (the C ABI of
``include/coalsack_moe.h``).

A case is a dict of plain values.  ``kind`` says which calls it makes:

  stack   a decode step through several resident layers, each with RMSNorm in front and the
          residual added (csk_moe_forward for the first, csk_moe_stack_forward for the rest)
  layer   one resident layer over a batch in device memory (csk_moe_forward)
  frame   the same layer called by an engine whose activations live in host memory
          (csk_moe_forward_host)
  linear  a linear projection with resident weights, activations in host memory
          (csk_matmul_transpose_f16)
  ffn     the shared expert's dense FFN, activations in host memory (csk_dense_ffn_f16)
  load    the experts of a layer from the checkpoint's own bytes in host memory into HBM
          (csk_layer_set_expert, or csk_layer_set_expert_matrix for K-quants), and the first
          tokens through them

``format`` is how the expert weights are stored: "mxfp4", "f16", or for ``load`` also "q4_k" and
"q6_k".  Sizes are the 20b- and 120b-shaped layers of the benchmark (hidden = intermediate =
2880, top-4 of 32 or of 128 experts, eight of them hot) and generic ones beside them.
"""
import ctypes as C
import math
import weakref

import numpy as np
import torch

from coalsack_amd import capi, synth

_DEFAULTS = dict(layers=1, k=4, format="mxfp4", hot=0, sigmoid=False, standard=False, weight_first=False, bias=True)


def _case(**kw):
    return {**_DEFAULTS, **kw}


def listed():
    shape20 = dict(E=32, k=4, H=2880, F=2880)
    shape120 = dict(E=128, k=4, H=2880, F=2880, hot=8)
    return [
        # one user's next token through a stack of large layers: the latency of a small call
        _case(name="stack_1", kind="stack", layers=8, T=1, **shape120),
        # a batch of sixteen users' next tokens
        _case(name="stack_16", kind="stack", layers=8, T=16, **shape120),
        # a fuller batch on a layer of many small experts
        _case(name="stack_small_50", kind="stack", layers=8, T=50, E=64, k=8, H=2048, F=768),
        # a short prompt, or decode and prompt tokens mixed
        _case(name="layer_300", kind="layer", T=300, **shape120),
        # long prompts
        _case(name="prefill_2048", kind="layer", T=2048, **shape20),
        _case(name="prefill_4096", kind="layer", T=4096, **shape120),
        # a few tokens on few, wide experts; the other router and activation
        _case(name="wide_6", kind="layer", T=6, E=16, k=2, H=4096, F=6144, sigmoid=True, standard=True, bias=False),
        # fp16 experts (F16 or K-quant checkpoints): decode with the llama4 options, and a prompt
        _case(name="f16_decode_8", kind="layer", T=8, E=16, k=1, H=5120, F=8192, format="f16", sigmoid=True,
              standard=True, weight_first=True, bias=False),
        _case(name="f16_prefill_1000", kind="layer", T=1000, format="f16", **shape20),
        # an engine on the host calls the layer for a couple of tokens
        _case(name="frame_2", kind="frame", T=2, **shape20),
        # an attention projection over a prompt
        _case(name="linear_200", kind="linear", T=200, H=2880, F=4096, format="f16"),
        # loading a checkpoint's experts
        _case(name="load_mxfp4", kind="load", T=1, E=8, k=4, H=2880, F=2880),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, lo, hi):
    return 32 * _log_int(rng, lo // 32, hi // 32)


def draw(rng):
    """One more case of the same ranges; none costs more than the largest listed one."""
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["stack"] * 4 + ["layer"] * 7 + ["frame"] * 2 + ["linear", "ffn"] + ["load"] * 2)
        c = _case(kind=kind)
        if kind in ("linear", "ffn"):
            c.update(T=_log_int(rng, 1, 1024), H=_log_int(rng, 1024, 5120), F=_log_int(rng, 1024, 8192), format="f16",
                     bias=rng.random() < 0.5)
            return {k: v for k, v in c.items() if k != "k"}
        c["E"] = rng.choice([8, 16, 32, 64, 128])
        c["k"] = rng.choice([1, 2, 4, 4, 8])
        wide = c["E"] <= 16 and rng.random() < 0.5
        if rng.random() < 0.4 and not wide:
            c["H"] = c["F"] = 2880
        else:
            c["H"] = _dim(rng, 1024, 6144 if wide else 3072)
            c["F"] = _dim(rng, 512, 8192 if wide else 3072)
        c["format"] = "f16" if rng.random() < 0.25 else "mxfp4"
        c["hot"] = 8 if c["E"] == 128 and rng.random() < 0.5 else 0
        c["sigmoid"] = rng.random() < 0.2
        c["standard"] = c["sigmoid"] or rng.random() < 0.2
        c["weight_first"] = c["sigmoid"] and rng.random() < 0.5
        c["bias"] = rng.random() < 0.7
        if kind == "stack":
            c["layers"] = rng.randint(4, 8)
            c["T"] = _log_int(rng, 1, 64)
        elif kind == "layer":
            c["T"] = _log_int(rng, 1, 4096)
        elif kind == "frame":
            c["T"] = _log_int(rng, 1, 256)
        else:
            c.update(E=rng.choice([4, 8]), k=rng.choice([2, 4]), T=rng.randint(1, 4), hot=0)
            if c["format"] == "f16":
                c["format"] = rng.choice(["f16", "q4_k", "q6_k"])
                c["H"], c["F"] = 256 * max(4, c["H"] // 256), 256 * max(2, c["F"] // 256)
        held = c["layers"] * c["E"] * 3 * _matrix_bytes(c)
        if held <= 16e9 and _cost(c) <= most and (kind != "load" or held <= 0.2e9):
            return c


# ------------------------------------------------------------------ preparation
_keep_lib = None


def _library():
    global _keep_lib
    if _keep_lib is None:
        _keep_lib = capi.load(0)
    return _keep_lib


class _State(dict):
    """What a program keeps between calls; gives the library's handles back when it is dropped."""

    def gives_back(self, *closers):
        for close in closers:
            weakref.finalize(self, close)
        return self


def _options(layer, case):
    layer.set_options(sigmoid=case["sigmoid"],
                      act=capi.ACT_STANDARD_SWIGLU if case["standard"] else capi.ACT_MODIFIED_SWIGLU,
                      weight_before_ffn=case["weight_first"])


def _bias_rows(L, e, case):
    return (L.b_up[e], L.b_gate[e], L.b_down[e]) if case["bias"] else (None, None, None)


def _resident_layer(lib, case, seed, index):
    """A layer with weights, router, biases and norm in HBM; weights are generated on the GPU."""
    L = synth.LayerInputs(case["E"], case["k"], case["H"], case["F"], seed=seed, layer=index,
                          hot_experts=case["hot"], with_norm=True)
    f16 = case["format"] == "f16"
    layer = lib.layer(L.E, L.k, L.H, L.F, f16=f16)
    _options(layer, case)
    layer.set_router(L.gate_w, L.gate_b)
    layer.fill_synthetic(seed, index)
    if case["bias"]:
        put = layer.set_expert_f16 if f16 else layer.set_expert
        for e in range(L.E):
            put(e, None, None, None, *_bias_rows(L, e, case))
    layer.set_norm(L.norm_w, 1e-5)
    return layer


def _hidden(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn((case["T"], case["H"]), generator=g, device="cuda", dtype=torch.float32)


def _halves(rng, rows, cols):
    """A weight matrix as a checkpoint holds it: normal with a deviation of 1 / sqrt(columns)."""
    return (rng.standard_normal((rows, cols), np.float32) / np.float32(math.sqrt(cols))).astype(np.float16)


def _checkpoint_bytes(rng, fmt, rows, cols):
    """One expert matrix in the checkpoint's own format (bytes of random weights of ordinary size)."""
    n = rows * cols
    if fmt == "mxfp4":
        b = rng.integers(0, 256, (n // 32, 17), dtype=np.uint8)
        b[:, 0] = 117 + b[:, 0] % 5
    elif fmt == "q4_k":
        b = rng.integers(0, 256, (n // 256, 144), dtype=np.uint8)
        b[:, 0:4] = np.array([1e-4, 7.5e-4], np.float16).view(np.uint8)
    elif fmt == "q6_k":
        b = rng.integers(0, 256, (n // 256, 210), dtype=np.uint8)
        b[:, 208:210] = np.array([2e-5], np.float16).view(np.uint8)
    else:
        return _halves(rng, rows, cols)
    return b.reshape(-1)


def prepare(case, seed):
    lib = _library()
    kind = case["kind"]
    rng = np.random.default_rng([seed, 11])
    if kind in ("stack", "layer", "frame"):
        layers = [_resident_layer(lib, case, seed, i) for i in range(case["layers"])]
        s = _State(lib=lib, case=case, layers=layers)
        s.gives_back(*(layer.close for layer in layers))
        if kind == "frame":
            s["hidden"] = rng.standard_normal((case["T"], case["H"]), np.float32)
        else:
            s["hidden"] = _hidden(case, seed)
            s["out"] = torch.empty_like(s["hidden"])
        return s
    if kind == "linear":
        w = lib.f16_upload(_halves(rng, case["F"], case["H"]))
        s = _State(lib=lib, case=case, w=w, x=rng.standard_normal((case["T"], case["H"]), np.float32),
                   out=np.empty((case["T"], case["F"]), np.float32))
        return s.gives_back(lambda: lib.f16_free(w))
    if kind == "ffn":
        H, F = case["H"], case["F"]
        w = [lib.f16_upload(_halves(rng, r, c)) for r, c in ((F, H), (F, H), (H, F))]
        b = [rng.normal(0.0, 0.01, n).astype(np.float32) if case["bias"] else None for n in (F, F, H)]
        s = _State(lib=lib, case=case, w=w, b=b, x=rng.standard_normal((case["T"], H), np.float32),
                   out=np.empty((case["T"], H), np.float32))
        return s.gives_back(*(lambda h=h: lib.f16_free(h) for h in w))
    # load: the checkpoint's bytes on the host, a layer to fill
    L = synth.LayerInputs(case["E"], case["k"], case["H"], case["F"], seed=seed)
    layer = lib.layer(L.E, L.k, L.H, L.F, f16=case["format"] != "mxfp4")
    _options(layer, case)
    shapes = {capi.W_UP: (L.F, L.H), capi.W_GATE: (L.F, L.H), capi.W_DOWN: (L.H, L.F)}
    weights = [{w: _checkpoint_bytes(rng, case["format"], *shapes[w]) for w in shapes} for _ in range(L.E)]
    s = _State(lib=lib, case=case, layer=layer, inputs=L, weights=weights, hidden=_hidden(case, seed))
    s["out"] = torch.empty_like(s["hidden"])
    return s.gives_back(layer.close)


# ------------------------------------------------------------------------- a pass
_GGML = {"q4_k": 12, "q6_k": 14}


def _ptr(a):
    return None if a is None else a.ctypes.data_as(C.c_void_p)


def run(s):
    lib, case = s["lib"], s["case"]
    kind, T = case["kind"], case["T"]
    if kind == "layer":
        s["layers"][0].forward_device(s["hidden"].data_ptr(), T, s["out"].data_ptr())
        return s["out"]
    if kind == "stack":
        out = s["out"].data_ptr()
        s["layers"][0].forward_device(s["hidden"].data_ptr(), T, out, capi.FWD_RMSNORM | capi.FWD_RESIDUAL)
        capi.stack_forward(lib, s["layers"][1:], out, T)
        return s["out"]
    if kind == "frame":
        return s["layers"][0].forward(s["hidden"], want_pairs=True)
    if kind == "linear":
        lib.check(lib.dll.csk_matmul_transpose_f16(_ptr(s["x"]), T, case["H"], s["w"], _ptr(s["out"])))
        return s["out"]
    if kind == "ffn":
        lib.check(lib.dll.csk_dense_ffn_f16(_ptr(s["x"]), T, case["H"], case["F"], *s["w"], *map(_ptr, s["b"]),
                                            _ptr(s["out"])))
        return s["out"]
    layer, L = s["layer"], s["inputs"]
    layer.set_router(L.gate_w, L.gate_b)
    for e, w in enumerate(s["weights"]):
        bias = _bias_rows(L, e, case)
        if case["format"] == "mxfp4":
            layer.set_expert(e, w[capi.W_UP], w[capi.W_GATE], w[capi.W_DOWN], *bias)
        elif case["format"] == "f16":
            layer.set_expert_f16(e, w[capi.W_UP], w[capi.W_GATE], w[capi.W_DOWN], *bias)
        else:
            for which, data in w.items():
                layer.set_expert_matrix(e, which, _GGML[case["format"]], data)
            layer.set_expert_f16(e, None, None, None, *bias)
    layer.forward_device(s["hidden"].data_ptr(), T, s["out"].data_ptr())
    return s["out"]


# ------------------------------------------------------------ what a pass has to do
_BYTES_PER_WEIGHT = {"mxfp4": 17 / 32, "f16": 2.0, "q4_k": 144 / 256, "q6_k": 210 / 256}


def _matrix_bytes(case):
    return case["H"] * case["F"] * _BYTES_PER_WEIGHT[case["format"]]


def _experts_used(case):
    """Experts that at least one of T tokens is expected to select."""
    E, k, T, hot = case["E"], case["k"], case["T"], case["hot"]
    if not hot:
        return E * (1.0 - (1.0 - k / E) ** T)
    p_hot, p_cold = min(1.0, 0.5 * k / hot), 0.5 * k / (E - hot)  # the hot ones take about half of the assignments
    return hot * (1.0 - (1.0 - p_hot) ** T) + (E - hot) * (1.0 - (1.0 - p_cold) ** T)


def work(case):
    H, F, T = case["H"], case["F"], case["T"]
    if case["kind"] == "linear":
        return {"bytes": 2.0 * H * F + 4.0 * T * (H + F), "flops": 2.0 * T * H * F}
    if case["kind"] == "ffn":
        return {"bytes": 6.0 * H * F + 8.0 * T * H + (4.0 * (2 * F + H) if case["bias"] else 0.0), "flops": 6.0 * T * H * F}
    E, k, n = case["E"], case["k"], case["layers"]
    expert = 3.0 * _matrix_bytes(case) + (4.0 * (2 * F + H) if case["bias"] else 0.0)
    flops = n * T * (k * 6.0 * H * F + 2.0 * E * H)
    if case["kind"] == "load":
        return {"bytes": 2.0 * E * expert + 4.0 * E * (H + 1) + 8.0 * T * H, "flops": flops}
    moved = _experts_used(case) * expert + 4.0 * E * (H + 1) + 8.0 * T * H
    return {"bytes": n * moved, "flops": flops}


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50.0)


def tolerance(case):
    """Four times the distance (2-norm, relative) from the same path in float64, measured on
    these shapes: 3.0e-5 to 4.4e-5 for one MXFP4 layer, whose activations the kernels carry as
    three FP6 terms; 9.4e-5 after eight layers with their residual sums; 4.5e-7 to 6.4e-7 with
    fp16 weights (activations as two fp16 terms, fp32 sums)."""
    if case["format"] != "mxfp4":
        return {"rel": 3e-6}
    return {"rel": 4e-4 if case["kind"] == "stack" else 1.8e-4}
