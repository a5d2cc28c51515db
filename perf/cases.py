"""Timed cases of the decode path, through the package's public entry points.

A decode engine for a Qwen3-4B-shaped model (hidden 2560, intermediate 9728, 32 query and 8 KV
heads of 128, vocabulary 151936) spends its time here: weights are quantized and prepared once,
then every step runs the projections, norms and attention of its layers for 1 to 64 tokens
(greedy decoding, small batches, speculative verification), captured in a HIP graph as an engine
captures its decode step, or as one executor launch. The kinds of case:

* ``linear``    one projection, called eagerly: the smallest call a program makes.
* ``layers``    the single calls of a decode layer around attention (residual + RMSNorm, qkv, o,
                residual + RMSNorm, gate_up + SwiGLU, down), for a few layers with weights of their
                own, in one captured graph. Attention's output and the second norm's addend are
                given, so that an FP8 activation code next to a rounding step does not decide what
                the following calls are compared on.
* ``mlp``       gate_up + SwiGLU, then down, likewise.
* ``head``      the output projection over the vocabulary, in a captured graph.
* ``attention`` head norm + RoPE + cache write and decode attention, for a few layers' caches, in
                one captured graph.
* ``segments``  the executor's launch between two attention calls (o, residual + RMSNorm,
                gate_up + SwiGLU, down, residual + RMSNorm, the next qkv), one launch a layer.
* ``step``      a whole decode step as one executor launch, attention included; returns logits.
* ``pack``      quantize a bf16 weight and relay it into the layout the kernels consume.

Weight formats: ``w4a16``, ``w8a16``, ``fp8`` (W8A8, activations quantized per token), and the
engine's default INT8 / INT4 with an fp16 scale per 64 values (``int8g64``, ``int4g64``).
"""

import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dryft-flash-infer_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from kernels import DecodeAttention, add_rms_norm, cuda_fp8, qkv_norm_rope_to_cache  # noqa: E402
from kernels.decode_stack import DecodeStack  # noqa: E402

EPS = 1e-6
HEAD = 128
GROUP = 4  # query heads per KV head
FORMATS = ("w4a16", "w8a16", "fp8", "int8g64", "int4g64")
STACK_FORMATS = ("w4a16", "w8a16")  # the executor's chains whose results can be compared closely
BF16 = torch.bfloat16


def listed():
    qwen = {"hidden": 2560, "inter": 9728, "kv_heads": 8}
    return [
        # One W8A16 down projection of one token, as a program without a graph calls it.
        {"name": "linear_w8a16_m1", "kind": "linear", "fmt": "w8a16", "m": 1, "n": 2560, "k": 9728},
        # Greedy decoding at batch 1: the executor between two attention calls. (In FP8 W8A8 such a
        # chain's last results differ by 4 % between correct implementations: activation codes flip.)
        {"name": "segments_w8a16_m1", "kind": "segments", "fmt": "w8a16", "m": 1, "layers": 4, **qwen},
        # Greedy decoding at batch 1 as one launch per token, at the end of a 512-token prompt.
        {"name": "step_w4a16", "kind": "step", "fmt": "w4a16", "layers": 4, "keys": 513, "vocab": 151936, **qwen},
        # Batch 8 in FP8 W8A8.
        {"name": "layers_fp8_m8", "kind": "layers", "fmt": "fp8", "m": 8, "layers": 4, **qwen},
        # An odd number of rows: a batch with some sequences finished.
        {"name": "layers_w8a16_m23", "kind": "layers", "fmt": "w8a16", "m": 23, "layers": 4, **qwen},
        # The engine's default weight format at batch 32.
        {"name": "layers_int8g64_m32", "kind": "layers", "fmt": "int8g64", "m": 32, "layers": 4, **qwen},
        # Speculative verification at batch 1: a confirmed token and four drafts.
        {"name": "layers_int4g64_m5", "kind": "layers", "fmt": "int4g64", "m": 5, "layers": 4, **qwen},
        # The widest pass of the linears: 64 rows of verification over 4-bit weights.
        {"name": "mlp_w4a16_m64", "kind": "mlp", "fmt": "w4a16", "m": 64, "layers": 4, **qwen},
        # The vocabulary projection of a small batch.
        {"name": "head_w4a16_m16", "kind": "head", "fmt": "w4a16", "m": 16, "n": 151936, "k": 2560},
        # One long conversation.
        {"name": "attention_b1_32k", "kind": "attention", "batch": 1, "tokens": 1, "keys": 32768, "int8": False,
         "layers": 4, "kv_heads": 8},
        # Batch 32 with two tokens a sequence over an INT8 cache, an odd context.
        {"name": "attention_b32_t2_int8", "kind": "attention", "batch": 32, "tokens": 2, "keys": 577, "int8": True,
         "layers": 4, "kv_heads": 8},
        # Loading: the largest weight of the model, the tied embedding.
        {"name": "pack_w4a16_embedding", "kind": "pack", "fmt": "w4a16", "n": 151936, "k": 2560},
    ]


def _log(rng, lo, hi):
    """A whole number in lo..hi, spread over its logarithm."""
    return min(hi, max(lo, int(lo * (hi / lo) ** rng.random() + 0.5)))


def draw(rng):
    kind = rng.choice(("linear", "layers", "layers", "layers", "mlp", "mlp", "head", "attention", "attention",
                       "segments", "step", "pack"))
    shape = {"hidden": 256 * rng.randint(4, 20), "inter": 256 * rng.randint(10, 54), "kv_heads": rng.choice((4, 8, 10))}
    if kind == "linear":
        return {"kind": kind, "fmt": rng.choice(FORMATS), "m": _log(rng, 1, 64), "n": 16 * _log(rng, 64, 1216),
                "k": 256 * rng.randint(4, 38)}
    if kind in ("layers", "mlp"):
        return {"kind": kind, "fmt": rng.choice(FORMATS), "m": _log(rng, 1, 64), "layers": rng.randint(2, 4), **shape}
    if kind == "head":
        return {"kind": kind, "fmt": rng.choice(FORMATS), "m": _log(rng, 1, 64), "n": 16 * _log(rng, 1000, 9496),
                "k": 256 * rng.randint(4, 16)}
    if kind == "attention":
        batch = _log(rng, 1, 32)
        return {"kind": kind, "batch": batch, "tokens": rng.choice((1, 1, 1, 2, 3, 5)),
                "keys": _log(rng, 33, 65536 // batch), "int8": rng.random() < 0.4, "layers": 4, "kv_heads": 8}
    if kind == "segments":
        return {"kind": kind, "fmt": rng.choice(STACK_FORMATS), "m": rng.randint(1, 4), "layers": rng.randint(2, 4), **shape}
    if kind == "step":
        return {"kind": kind, "fmt": rng.choice(STACK_FORMATS), "layers": rng.randint(1, 4),
                "keys": _log(rng, 1, 4096), "vocab": 16 * _log(rng, 2000, 9496), **shape}
    return {"kind": kind, "fmt": rng.choice(FORMATS), "n": 16 * _log(rng, 64, 9496), "k": 256 * rng.randint(4, 16)}


# ---- inputs -----------------------------------------------------------------------------------

class _Inputs:
    """Tensors from a seed, in a fixed order of draws."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed) + 1)

    def normal(self, *shape, std=1.0, mean=0.0):
        t = torch.randn(*shape, generator=self.gen, device="cuda")
        return t.mul_(std).add_(mean).to(BF16)

    def weight(self, n, k):
        """A projection's bf16 weight, at the scale of a trained or freshly initialised model."""
        return torch.randn(n, k, generator=self.gen, device="cuda", dtype=BF16).mul_(0.02)

    def norm_weight(self, n):
        return self.normal(n, std=0.1, mean=1.0)


def _pack(w, fmt):
    if fmt.endswith("g64"):
        return cuda_fp8.prepare(cuda_fp8.quantize(w, bits=4 if fmt == "int4g64" else 8, fmt="ref"))
    return cuda_fp8.prepare(cuda_fp8.quantize(w, bits=4 if fmt == "w4a16" else 8, fmt=fmt))


def _shapes(case):
    """(n, k) of a layer's projections."""
    h, i, kv = case["hidden"], case["inter"], case["kv_heads"]
    return {"qkv": ((GROUP + 2) * kv * HEAD, h), "o": (h, GROUP * kv * HEAD), "gate_up": (2 * i, h), "down": (h, i)}


def _layer_inputs(case, seed, names, keep):
    """Per layer the bf16 weights (handed to ``keep`` one at a time) and the layer's other inputs."""
    src = _Inputs(seed)
    m, h = case.get("m", 1), case["hidden"]
    layers = []
    for _ in range(case["layers"]):
        layer = {name: keep(src.weight(*_shapes(case)[name])) for name in names}
        layer["norm_in"], layer["norm_post"] = src.norm_weight(h), src.norm_weight(h)
        layer["h"] = src.normal(m, h)
        layer["delta"], layer["delta_post"] = src.normal(m, h, std=0.5), src.normal(m, h, std=0.5)
        layer["attn"] = src.normal(m, GROUP * case["kv_heads"] * HEAD, std=0.3)
        layers.append(layer)
    return layers


def _captured(step):
    """``step`` as a HIP graph and the tensors its replays write."""
    step()  # what the first call creates must exist before the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return {"graph": graph, "out": out}


def _attention_inputs(case, seed):
    src = _Inputs(seed)
    batch, tokens, keys, kv = case["batch"], case["tokens"], case["keys"], case["kv_heads"]
    capacity = keys + 64
    angles = torch.randn(capacity, HEAD, generator=src.gen, device="cuda")
    t = {"cos": angles.cos().to(BF16), "sin": angles.sin().to(BF16), "capacity": capacity,
         "first": max(0, keys - tokens), "layers": []}
    for _ in range(case["layers"]):
        layer = {"qkv": src.normal(batch * tokens, (GROUP + 2) * kv * HEAD), "qn": src.norm_weight(HEAD),
                 "kn": src.norm_weight(HEAD)}
        for name in ("k", "v"):
            if case["int8"]:
                layer[name] = torch.randint(-127, 128, (batch, kv, capacity, HEAD), generator=src.gen, device="cuda",
                                            dtype=torch.int8)
                layer[name + "s"] = torch.rand(batch, kv, capacity, generator=src.gen, device="cuda").add_(0.5).div_(64)
            else:
                layer[name] = torch.randn(batch, kv, capacity, HEAD, generator=src.gen, device="cuda", dtype=BF16)
                layer[name + "s"] = None
        t["layers"].append(layer)
    return t


def _step_inputs(case, seed, keep):
    src = _Inputs(seed)
    h, kv, keys = case["hidden"], case["kv_heads"], case["keys"]
    capacity = keys + 64
    angles = torch.randn(capacity, HEAD, generator=src.gen, device="cuda")
    t = {"cos": angles.cos().to(BF16), "sin": angles.sin().to(BF16), "h": src.normal(1, h),
         "norm_out": src.norm_weight(h), "head": keep(src.weight(case["vocab"], h)), "layers": []}
    for _ in range(case["layers"]):
        layer = {name: keep(src.weight(*nk)) for name, nk in _shapes(case).items()}
        layer.update(norm_in=src.norm_weight(h), norm_post=src.norm_weight(h), qn=src.norm_weight(HEAD),
                     kn=src.norm_weight(HEAD), k=src.normal(1, kv, capacity, HEAD), v=src.normal(1, kv, capacity, HEAD))
        t["layers"].append(layer)
    return t


# ---- the framework's side -----------------------------------------------------------------------

def _prepare_linear(case, seed):
    src = _Inputs(seed)
    w = _pack(src.weight(case["n"], case["k"]), case["fmt"])
    return {"w": w, "x": src.normal(case["m"], case["k"])}


def _prepare_layers(case, seed):
    fmt = case["fmt"]
    layers = _layer_inputs(case, seed, ("qkv", "o", "gate_up", "down"), lambda w: _pack(w, fmt))

    def step():
        outs = []
        for L in layers:
            r, x = add_rms_norm(L["h"], L["delta"], L["norm_in"], EPS)
            qkv = cuda_fp8.matmul(x, L["qkv"])
            o = cuda_fp8.matmul(L["attn"], L["o"])
            r, x = add_rms_norm(r, L["delta_post"], L["norm_post"], EPS)
            act = cuda_fp8.gate_up_swiglu(x, L["gate_up"])
            outs.append([qkv, o, r, act, cuda_fp8.matmul(act, L["down"])])
        return outs
    return dict(_captured(step), inputs=layers)


def _prepare_mlp(case, seed):
    fmt = case["fmt"]
    layers = _layer_inputs(case, seed, ("gate_up", "down"), lambda w: _pack(w, fmt))

    def step():
        outs = []
        for L in layers:
            act = cuda_fp8.gate_up_swiglu(L["h"], L["gate_up"])
            outs.append([act, cuda_fp8.matmul(act, L["down"])])
        return outs
    return dict(_captured(step), inputs=layers)


def _prepare_head(case, seed):
    state = _prepare_linear(case, seed)
    return dict(_captured(lambda: cuda_fp8.matmul(state["x"], state["w"])), inputs=state)


def _prepare_attention(case, seed):
    t = _attention_inputs(case, seed)
    batch, tokens, kv = case["batch"], case["tokens"], case["kv_heads"]
    # positions of the pass's tokens, the same for every sequence (as an engine's lockstep batch)
    positions = torch.arange(t["first"], t["first"] + tokens, dtype=torch.int32, device="cuda")
    attends = [DecodeAttention(batch, kv, GROUP, HEAD, t["capacity"], "cuda", tokens=tokens, quant=case["int8"])
               for _ in t["layers"]]

    def step():
        outs = []
        for L, attend in zip(t["layers"], attends):
            q = qkv_norm_rope_to_cache(L["qkv"], GROUP * kv, kv, L["qn"], L["kn"], t["cos"], t["sin"], positions,
                                       tokens, L["k"], L["v"], EPS, k_scale=L["ks"], v_scale=L["vs"])
            outs.append([q, attend(q, L["k"], L["v"], positions, L["ks"], L["vs"])])
        return outs
    return dict(_captured(step), inputs=t, attends=attends, positions=positions)


def _prepare_segments(case, seed):
    fmt, m, h = case["fmt"], case["m"], case["hidden"]
    layers = _layer_inputs(case, seed, ("o", "gate_up", "down", "qkv"), lambda w: _pack(w, fmt).tiles)
    new = lambda n: torch.empty(m, n, dtype=BF16, device="cuda")  # noqa: E731
    chains, outs = [], []
    for L in layers:
        o, act, down, r1, r2 = new(h), new(case["inter"]), new(h), new(h), new(h)
        qkv = new((GROUP + 2) * case["kv_heads"] * HEAD)
        chain = DecodeStack(fmt, m)
        chain.add(L["o"], L["attn"], o)
        chain.add_normed(L["gate_up"], L["h"], act, L["norm_post"], EPS, delta=o, resid_out=r1, swiglu=True)
        chain.add(L["down"], act, down)
        chain.add_normed(L["qkv"], r1, qkv, L["norm_in"], EPS, delta=down, resid_out=r2)
        chains.append(chain.build())
        outs.append([r1, act, down, r2, qkv])
    return {"chains": chains, "out": outs, "inputs": layers}


def _prepare_step(case, seed):
    fmt, h, kv, inter = case["fmt"], case["hidden"], case["kv_heads"], case["inter"]
    t = _step_inputs(case, seed, lambda w: _pack(w, fmt).tiles)
    new = lambda n: torch.empty(1, n, dtype=BF16, device="cuda")  # noqa: E731
    positions = torch.tensor([case["keys"] - 1], dtype=torch.int32, device="cuda")
    chain = DecodeStack(fmt, 1)
    width = (GROUP + 2) * kv * HEAD
    qkv, resid = new(width), new(h)
    chain.add_normed(t["layers"][0]["qkv"], t["h"], qkv, t["layers"][0]["norm_in"], EPS, resid_out=resid)
    logits = new(case["vocab"])
    keep = [qkv, resid]
    for i, L in enumerate(t["layers"]):
        att, o, act, down, r1, r2 = new(GROUP * kv * HEAD), new(h), new(inter), new(h), new(h), new(h)
        chain.add_attention(qkv, GROUP * kv, kv, L["qn"], L["kn"], t["cos"], t["sin"], positions, L["k"], L["v"], att,
                            EPS)
        chain.add(L["o"], att, o)
        chain.add_normed(L["gate_up"], resid, act, L["norm_post"], EPS, delta=o, resid_out=r1, swiglu=True)
        chain.add(L["down"], act, down)
        if i + 1 < len(t["layers"]):
            after = t["layers"][i + 1]
            qkv = new(width)
            chain.add_normed(after["qkv"], r1, qkv, after["norm_in"], EPS, delta=down, resid_out=r2)
        else:
            chain.add_normed(t["head"], r1, logits, t["norm_out"], EPS, delta=down, resid_out=r2)
        keep += [att, o, act, down, r1, r2, qkv]
        resid = r2
    return {"chains": [chain.build()], "out": [resid, logits], "inputs": t, "keep": keep, "positions": positions}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        state = _prepare_linear(case, seed)
    elif kind == "pack":
        state = {"weight": _Inputs(seed).weight(case["n"], case["k"]), "fmt": case["fmt"]}
    else:
        state = {"layers": _prepare_layers, "mlp": _prepare_mlp, "head": _prepare_head, "attention": _prepare_attention,
                 "segments": _prepare_segments, "step": _prepare_step}[kind](case, seed)
    state["kind"] = kind
    return state


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return cuda_fp8.matmul(state["x"], state["w"])
    if kind == "pack":
        p = _pack(state["weight"], state["fmt"])
        return {"weight": p.weight.view(torch.uint8), "scale": p.scale}
    if kind in ("segments", "step"):
        for chain in state["chains"]:
            chain.run()
    else:
        state["graph"].replay()
    return state["out"]


# ---- work and tolerances ----------------------------------------------------------------------------

_CODE = {"w4a16": 0.5, "int4g64": 0.5, "w8a16": 1.0, "int8g64": 1.0, "fp8": 1.0}
_PER_SCALE = {"w4a16": 128, "int4g64": 64, "int8g64": 64}


def _weight_bytes(fmt, n, k):
    return n * k * _CODE[fmt] + 2 * n * (k // _PER_SCALE.get(fmt, k))


def _linear_work(fmt, m, n, k, n_out):
    return _weight_bytes(fmt, n, k) + 2 * m * (k + n_out), 2 * m * n * k


def _attention_work(batch, tokens, keys, kv, value_bytes):
    rows = batch * tokens
    read = 2 * batch * kv * keys * (HEAD * value_bytes + (4 if value_bytes == 1 else 0))
    return (read + 2 * rows * HEAD * ((GROUP + 2) * kv + 2 * GROUP * kv),  # qkv in, q and the output out
            4 * rows * GROUP * kv * keys * HEAD)


def work(case):
    kind, m = case["kind"], case.get("m", 1)
    parts = []
    if kind in ("linear", "head"):
        parts.append(_linear_work(case["fmt"], m, case["n"], case["k"], case["n"]))
    elif kind == "pack":
        parts.append((2 * case["n"] * case["k"] + _weight_bytes(case["fmt"], case["n"], case["k"]), 0))
    elif kind == "attention":
        one = _attention_work(case["batch"], case["tokens"], case["keys"], case["kv_heads"], 1 if case["int8"] else 2)
        parts += [one] * case["layers"]
    else:
        shapes = _shapes(case)
        names = ("gate_up", "down") if kind == "mlp" else tuple(shapes)
        for name in names:
            n, k = shapes[name]
            b, f = _linear_work(case["fmt"], m, n, k, n // 2 if name == "gate_up" else n)
            parts.append((b * case["layers"], f * case["layers"]))
        if kind in ("layers", "segments"):
            parts.append((case["layers"] * m * case["hidden"] * 2 * 4, 0))  # the residual stream around the two norms
        if kind == "step":
            parts += [_attention_work(1, 1, case["keys"], case["kv_heads"], 2)] * case["layers"]
            parts.append(_linear_work(case["fmt"], 1, case["vocab"], case["hidden"], case["vocab"]))
    return {"bytes": float(sum(p[0] for p in parts)), "flops": float(sum(p[1] for p in parts))}


def tolerance(case):
    """Against another correct implementation at the same precision (bf16 results of 32-bit sums)."""
    kind = case["kind"]
    if kind == "pack":
        return "exact"
    if kind == "step":  # bf16 roundings of a layer travel through the next ones
        return {"rel": 3e-2, "max": 0.3}
    if kind == "segments":
        return {"rel": 1e-2, "max": 0.1}
    if kind == "attention":  # bf16 probabilities
        return {"rel": 1e-2, "max": 0.1}
    if case["fmt"] == "fp8" and kind in ("layers", "mlp"):
        # an act value one bf16 step away can move its e4m3 code by one (6 to 12 %) before down
        return {"rel": 3e-2, "max": 0.3}
    return {"rel": 6e-3, "max": 0.06}


# ---- the same in 64 bits -------------------------------------------------------------------------

def _quantized64(w, fmt):
    """The values a quantized weight stands for, exactly."""
    n, k = w.shape
    if fmt == "fp8":
        s = (w.float().abs().amax(1, keepdim=True) / 448).clamp_min(1e-12)
        code = (w.float() / s).clamp(-448, 448).to(torch.float8_e4m3fn)
        return code.double() * s.to(BF16).double()
    limit = 7 if _CODE[fmt] < 1 else 127
    g = w.float().view(n, -1, _PER_SCALE.get(fmt, k))
    s = (g.abs().amax(2, keepdim=True) / limit).clamp_min(1e-12) * (1.0 + 2.0 ** -10)
    s = s.to(torch.float16 if fmt.endswith("g64") else BF16)
    q = (g / s.float()).round().clamp(-limit, limit)
    return (q.double() * s.double()).view(n, k)


def _bf(x):
    """Rounded to the bf16 that the entry points hand on."""
    return x.to(BF16).double()


def _linear64(x, w64, fmt):
    if fmt == "fp8":  # the activation as its per-token e4m3 codes
        s = (x.float().abs().amax(1, keepdim=True) / 448).clamp_min(1e-12)
        x = (x.float() / s).clamp(-448, 448).to(torch.float8_e4m3fn).double() * s.double()
    return x.double() @ w64.T


def _swiglu64(gu):
    """silu(gate) * up of the bf16 gate and up values, silu rounded to bf16 as the entry point states."""
    g, u = _bf(gu).chunk(2, 1)
    return _bf(torch.nn.functional.silu(g)) * u


def _norm64(x, w):
    """RMSNorm, its normalised value rounded to bf16 before the gain (the model's own cast)."""
    return _bf(x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)) * w.double()


def _rope64(x, w, cos, sin):
    """Head norm and rotation of [rows, heads, 128] at cos/sin [rows, 128]."""
    y = _bf(_norm64(x, w))
    half = torch.cat((-y[..., HEAD // 2:], y[..., :HEAD // 2]), -1)
    return y * cos.double()[:, None] + half * sin.double()[:, None]


def _attend64(q, k, v, first):
    """q [batch, tokens, heads, 128] over k, v [batch, kv_heads, keys, 128]; token t sees keys
    0 .. first + t."""
    batch, tokens, heads, _ = q.shape
    kv = k.shape[1]
    out = torch.empty_like(q)
    for b in range(batch):
        qb = q[b].view(tokens, kv, heads // kv, HEAD)
        s = torch.einsum("tkgd,knd->tkgn", qb, k[b]) * HEAD ** -0.5
        seen = torch.arange(k.shape[2], device=k.device)[None] <= first + torch.arange(tokens, device=k.device)[:, None]
        p = s.masked_fill(~seen[:, None, None], float("-inf")).softmax(-1)
        out[b] = torch.einsum("tkgn,knd->tkgd", p, v[b]).reshape(tokens, heads, HEAD)
    return out


def exact(case, seed):
    kind, fmt = case["kind"], case.get("fmt")
    if kind == "pack":
        w = _Inputs(seed).weight(case["n"], case["k"])
        if fmt == "fp8":
            s = (w.float().abs().amax(1).double() / 448).clamp_min(1e-12)
        else:
            limit = 7 if _CODE[fmt] < 1 else 127
            g = w.view(case["n"], -1, _PER_SCALE.get(fmt, case["k"]))
            s = (g.abs().amax(2).double() / limit).clamp_min(1e-12) * (1.0 + 2.0 ** -10)
            s = s.view(-1) if fmt == "w8a16" else s
        return {"weight": None, "scale": s}
    if kind in ("linear", "head"):
        src = _Inputs(seed)
        w64 = _quantized64(src.weight(case["n"], case["k"]), fmt)
        return _linear64(src.normal(case["m"], case["k"]), w64, fmt)
    if kind in ("layers", "mlp", "segments"):
        names = {"layers": ("qkv", "o", "gate_up", "down"), "mlp": ("gate_up", "down"),
                 "segments": ("o", "gate_up", "down", "qkv")}[kind]
        outs = []
        for L in _layer_inputs(case, seed, names, lambda w: w):
            lin = lambda x, name: _linear64(x, _quantized64(L[name], fmt), fmt)  # noqa: E731
            if kind == "mlp":
                act = _swiglu64(lin(L["h"], "gate_up"))
                outs.append([act, lin(_bf(act), "down")])
                continue
            h = L["h"].double()
            if kind == "layers":
                h = _bf(h + L["delta"].double())
                qkv = lin(_bf(_norm64(h, L["norm_in"])), "qkv")
            o = lin(L["attn"], "o")
            r = h + (L["delta_post"].double() if kind == "layers" else _bf(o))
            act = _swiglu64(lin(_bf(_norm64(_bf(r), L["norm_post"])), "gate_up"))
            down = lin(_bf(act), "down")
            if kind == "layers":
                outs.append([qkv, o, r, act, down])
            else:
                r2 = _bf(r) + _bf(down)
                outs.append([r, act, down, r2, lin(_bf(_norm64(_bf(r2), L["norm_in"])), "qkv")])
        return outs
    if kind == "attention":
        t = _attention_inputs(case, seed)
        batch, tokens, kv, first = case["batch"], case["tokens"], case["kv_heads"], t["first"]
        at = torch.arange(first, first + tokens, device="cuda")
        cos, sin = t["cos"][at].repeat(batch, 1), t["sin"][at].repeat(batch, 1)
        outs = []
        for L in t["layers"]:
            x = L["qkv"].double().view(batch * tokens, -1, HEAD)
            q = _rope64(x[:, :GROUP * kv], L["qn"], cos, sin)
            k_new = _bf(_rope64(x[:, GROUP * kv:(GROUP + 1) * kv], L["kn"], cos, sin))
            cache = []
            for name, new in (("k", k_new), ("v", x[:, (GROUP + 1) * kv:])):
                new = new.view(batch, tokens, kv, HEAD).transpose(1, 2)
                old = L[name][:, :, :first + tokens].double()
                if case["int8"]:
                    old = old * L[name + "s"][:, :, :first + tokens, None].double()
                    s = new.abs().amax(-1, keepdim=True).clamp_min(1e-12) / 127
                    new = torch.floor(new / s + 0.5).clamp(-127, 127) * s
                old[:, :, first:] = new
                cache.append(old)
            a = _attend64(_bf(q).view(batch, tokens, GROUP * kv, HEAD), *cache, first)
            outs.append([q.reshape(batch * tokens, -1), a.reshape(batch * tokens, -1)])
            del cache
        return outs
    t = _step_inputs(case, seed, lambda w: w)
    kv, at = case["kv_heads"], case["keys"] - 1
    cos, sin = t["cos"][at:at + 1], t["sin"][at:at + 1]
    r = t["h"].double()
    for L in t["layers"]:
        lin = lambda x, name: _linear64(x, _quantized64(L[name], fmt), fmt)  # noqa: E731
        x = _bf(lin(_bf(_norm64(r, L["norm_in"])), "qkv")).view(1, -1, HEAD)
        q = _bf(_rope64(x[:, :GROUP * kv], L["qn"], cos, sin))
        k, v = L["k"][:, :, :at + 1].double(), L["v"][:, :, :at + 1].double()
        k[:, :, at] = _bf(_rope64(x[:, GROUP * kv:(GROUP + 1) * kv], L["kn"], cos, sin))
        v[:, :, at] = x[:, (GROUP + 1) * kv:]
        att = _attend64(q.view(1, 1, GROUP * kv, HEAD), k, v, at).view(1, -1)
        r = _bf(r + _bf(lin(_bf(att), "o")))
        act = _swiglu64(lin(_bf(_norm64(r, L["norm_post"])), "gate_up"))
        r = _bf(r + _bf(lin(_bf(act), "down")))
    return [r, _linear64(_bf(_norm64(r, t["norm_out"])), _quantized64(t["head"], fmt), fmt)]
