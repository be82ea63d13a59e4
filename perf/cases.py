"""The work that a program on fp8lin has it do, as cases to time and compare.

Every case goes through the public entry points (fp8lin.LinearEngine and the
operators of fp8lin) with the inputs that such a program holds:

  layers  two layers of one tensor-parallel rank, full attention then the
          gated-delta one, from the hidden state to the next: norms, fused
          projections, Q/K epilogue, output projections and MLPs.  Up to 32
          rows they are replayed as one captured graph, as the decode loop
          of an engine does; more rows (a prefill chunk) run eagerly.
  mlp     gate/up, SwiGLU and down of one layer, eagerly.
  linear  one projection, eagerly: FP8 with block or row scales, BF16, the
          decoded-weight cache, or dequantize-then-GEMM.
  vision  the three BF16 projections with bias of a vision block (QKV, fc1,
          fc2), whose widths are not multiples of 256.
  head    the output head's logits and greedy candidates.

Layer sizes are one rank's of the shipped configuration (hidden 5120,
intermediate 17408, 24/4 heads of 256 and 16/48 delta heads of 128 over two
ranks, vocabulary 248320); the others are generic.
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "a100-vision-infer_amd"))
import fp8lin  # noqa: E402

EPS = 1e-6
ROPE = {"partial_rotary_factor": 0.25, "mrope_section": [11, 11, 10], "rope_theta": 10000000}
GRAPH_ROWS = 32  # decode and batched decode replay a graph
L0, L1 = "model.language_model.layers.0", "model.language_model.layers.1"
RANK = {"hidden": 5120, "inter": 8704, "heads": 12, "kv_heads": 2, "head_dim": 256, "delta_in": 8192, "delta_gates": 48,
        "delta_out": 3072}


def listed():
    return [
        # one token of one request: the decode loop
        {"name": "decode_1", "kind": "layers", "m": 1, **RANK},
        # three drafted tokens and the last accepted one: verification of a speculative step
        {"name": "verify_4", "kind": "layers", "m": 4, **RANK},
        # a batched decode step, an odd number of requests
        {"name": "batch_27", "kind": "layers", "m": 27, **RANK},
        # the smallest call: one square projection for two rows, where the call itself counts
        {"name": "square_2", "kind": "linear", "m": 2, "n": 4096, "k": 4096, "weight": "fp8", "bias": False},
        # a short prompt, or the tail chunk of a longer one
        {"name": "short_prompt_93", "kind": "mlp", "m": 93, "hidden": 5120, "inter": 8704},
        # a prefill chunk
        {"name": "chunk_512", "kind": "layers", "m": 512, **RANK},
        # a prompt of text and image tokens in one piece, the largest call
        {"name": "prompt_3913", "kind": "mlp", "m": 3913, "hidden": 5120, "inter": 8704},
        # vocabulary shard of the head at a verification step
        {"name": "head_4", "kind": "head", "m": 4, "n": 75968, "k": 5120},
        # one image's patches through a vision block's projections
        {"name": "vision_1036", "kind": "vision", "m": 1036, "hidden": 1152, "inter": 4304},
        # a small prefill against weights of the decoded cache
        {"name": "cached_40", "kind": "linear", "m": 40, "n": 7168, "k": 5120, "weight": "cached", "bias": False},
        # a prefill chunk under the dequantize-then-GEMM option
        {"name": "dequant_640", "kind": "linear", "m": 640, "n": 17408, "k": 5120, "weight": "dequant", "bias": False},
        # row-scaled codes of ragged sizes
        {"name": "row_scales_77", "kind": "linear", "m": 77, "n": 4100, "k": 2880, "weight": "fp8_row", "bias": True},
    ]


def _log_int(rng, lo, hi, step=1):
    """A multiple of step in [lo, hi], its logarithm uniform."""
    v = lo * (hi / lo) ** rng.random()
    return max(lo, min(hi, int(v / step + 0.5) * step))


def draw(rng):
    most = max(work(c)["flops"] for c in listed())
    while True:
        kind = rng.choice(["layers", "layers", "mlp", "mlp", "linear", "linear", "linear", "vision", "head"])
        hidden = rng.choice([2048, 2560, 3072, 4096, 5120])
        if kind == "layers":
            kv = rng.choice([1, 2, 4])
            c = {"kind": kind, "m": _log_int(rng, 1, 1024), "hidden": hidden, "inter": _log_int(rng, 2048, 8704, 128),
                 "heads": kv * rng.randint(2, 6), "kv_heads": kv, "head_dim": rng.choice([128, 256]),
                 "delta_in": _log_int(rng, 2048, 8192, 128), "delta_gates": rng.choice([16, 32, 48]),
                 "delta_out": _log_int(rng, 1024, 4096, 128)}
        elif kind == "mlp":
            c = {"kind": kind, "m": _log_int(rng, 9, 3913), "hidden": hidden, "inter": _log_int(rng, 2048, 8704, 128)}
        elif kind == "linear":
            weight = rng.choice(["fp8", "fp8", "fp8_row", "bf16", "cached", "dequant"])
            c = {"kind": kind, "m": _log_int(rng, 1, 2048), "n": _log_int(rng, 256, 17408, 4),
                 "k": _log_int(rng, 512, 8704, rng.choice([16, 64, 128])), "weight": weight, "bias": rng.random() < 0.5}
        elif kind == "vision":
            c = {"kind": kind, "m": _log_int(rng, 64, 4096), "hidden": _log_int(rng, 768, 1664, 16),
                 "inter": _log_int(rng, 3072, 6656, 16)}
        else:
            c = {"kind": kind, "m": rng.randint(1, 8), "n": _log_int(rng, 16000, 124160, 16), "k": hidden}
        if work(c)["flops"] <= most:
            return c


# ---- inputs, in plain torch -------------------------------------------------


class _Inputs:
    """Seeded tensors: weights N(0, 0.02^2), activations N(0, 1)."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.gen, device="cuda")

    def acts(self, *shape):
        return self.normal(*shape).to(torch.bfloat16)

    def norm_weight(self, n):
        return (0.1 * self.normal(n)).to(torch.bfloat16)

    def bf16(self, n, k):
        return (0.02 * self.normal(n, k)).to(torch.bfloat16)

    def bias(self, n):
        return (0.1 * self.normal(n)).to(torch.bfloat16)

    def fp8(self, n, k):
        """E4M3 codes with one scale per 128 x 128 block, expanded along rows."""
        w = 0.02 * self.normal(n, k)
        rows, cols = -(-n // 128), -(-k // 128)
        full = torch.zeros(rows * 128, cols * 128, device="cuda")
        full[:n, :k] = w
        block = full.view(rows, 128, cols, 128).abs().amax(dim=(1, 3)).clamp_min(1e-12) / 448
        scales = block.repeat_interleave(128, 0)[:n].contiguous()
        codes = (w / scales.repeat_interleave(128, 1)[:, :k]).to(torch.float8_e4m3fn).view(torch.uint8)
        return codes.contiguous(), scales

    def fp8_row(self, n, k):
        """E4M3 codes with one scale per row."""
        w = 0.02 * self.normal(n, k)
        scales = w.abs().amax(1).clamp_min(1e-12) / 448
        return (w / scales[:, None]).to(torch.float8_e4m3fn).view(torch.uint8).contiguous(), scales


def _inputs(case, seed):
    """The case's tensors: {"x": ..., weights by name as (data, scale) or (data, None), ...}."""
    r, m, kind = _Inputs(seed), case["m"], case["kind"]
    if kind == "layers":
        h, inter, d = case["hidden"], case["inter"], case["head_dim"]
        qkv, o = 2 * (case["heads"] + case["kv_heads"]) * d, case["heads"] * d
        t = {"x": r.acts(m, h), "core0": r.acts(m, o), "core1": r.acts(m, case["delta_out"]),
             "positions": torch.randint(0, 4096, (3, m), generator=r.gen, device="cuda"),
             "q_norm": r.norm_weight(d), "k_norm": r.norm_weight(d)}
        for i in range(4):
            t["norm%d" % i] = r.norm_weight(h)
        w = {L0 + ".self_attn.qkv_gate": r.fp8(qkv, h), L0 + ".self_attn.o_proj": r.fp8(h, o),
             L1 + ".linear_attn.in_proj_qkvz": r.fp8(case["delta_in"], h),
             L1 + ".linear_attn.in_proj_ba": (r.bf16(case["delta_gates"], h), None),
             L1 + ".linear_attn.out_proj": r.fp8(h, case["delta_out"])}
        for layer in (L0, L1):
            w[layer + ".mlp.gate_up"] = r.fp8(2 * inter, h)
            w[layer + ".mlp.down_proj"] = r.fp8(h, inter)
        return {**t, "weights": w, "biases": {}}
    if kind == "mlp":
        h, inter = case["hidden"], case["inter"]
        w = {L0 + ".mlp.gate_up": r.fp8(2 * inter, h), L0 + ".mlp.down_proj": r.fp8(h, inter)}
        return {"x": r.acts(m, h), "weights": w, "biases": {}}
    if kind == "vision":
        h, inter = case["hidden"], case["inter"]
        sizes = {"model.visual.blocks.0.attn.qkv": (3 * h, h), "model.visual.blocks.0.mlp.linear_fc1": (inter, h),
                 "model.visual.blocks.0.mlp.linear_fc2": (h, inter)}
        return {"x": r.acts(m, h), "hid": r.acts(m, inter), "weights": {n: (r.bf16(*s), None) for n, s in sizes.items()},
                "biases": {n: r.bias(s[0]) for n, s in sizes.items()}}
    n, k = case["n"], case["k"]
    if kind == "head":
        codes, scales = r.fp8(n, k)
        # A trained head's rows have a clear winner: lean each hidden state towards one vocabulary row.
        ids = torch.randint(0, n, (m,), generator=r.gen, device="cuda")
        lean = codes[ids].view(torch.float8_e4m3fn).float() * scales[ids].repeat_interleave(128, 1)[:, :k]
        x = (r.normal(m, k) + 0.3 * lean / 0.02).to(torch.bfloat16)
        return {"x": x, "weights": {"lm_head": (codes, scales)}, "biases": {}}
    make = {"bf16": lambda: (r.bf16(n, k), None), "fp8_row": lambda: r.fp8_row(n, k)}.get(case["weight"], lambda: r.fp8(n, k))
    name = L0 + ".proj"
    return {"x": r.acts(m, k), "weights": {name: make()}, "biases": {name: r.bias(n)} if case["bias"] else {}}


# ---- the framework ----------------------------------------------------------


def prepare(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    weight = case.get("weight")
    eng = fp8lin.LinearEngine(fp8lin.LinearOptions(cublas_prefill=weight == "dequant"),
                              weight_cache_bytes=1 << 40 if weight == "cached" else 0)
    for name, (data, scale) in t["weights"].items():
        eng.add(name + ".weight", data, scale)
    for name, b in t["biases"].items():
        eng.add(name + ".bias", b)
    if kind == "layers":
        p = L1 + ".linear_attn."
        eng.fuse_weights(p + "in_proj_all", [p + "in_proj_qkvz", p + "in_proj_ba"])
    if weight == "cached":
        eng.build_cache()
    state = {"case": case, "engine": eng, **{k: v for k, v in t.items() if k not in ("weights", "biases")}}
    if kind == "layers" and case["m"] <= GRAPH_ROWS:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _layers(state)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outputs = _layers(state)
        state["graph"], state["outputs"] = graph, outputs
    return state


def _layers(s):
    c, eng = s["case"], s["engine"]
    n = fp8lin.fused_rms(s["x"], s["norm0"], EPS, True)
    q, gate, k, v = eng.full_attention_inputs(n, L0 + ".self_attn", s["positions"], s["q_norm"], s["k_norm"], c["heads"],
                                              c["kv_heads"], c["head_dim"], ROPE, EPS)
    o = eng.linear(s["core0"], L0 + ".self_attn.o_proj")
    r, n = fp8lin.residual_rms(s["x"], o, s["norm1"], EPS)
    r, n = fp8lin.residual_rms(r, eng.mlp(n, L0 + ".mlp"), s["norm2"], EPS)
    p = eng.linear(n, L1 + ".linear_attn.in_proj_all")
    o = eng.linear(s["core1"], L1 + ".linear_attn.out_proj")
    r, n = fp8lin.residual_rms(r, o, s["norm3"], EPS)
    return {"q": q, "gate": gate, "k": k, "v": v, "proj": p, "residual": r, "mlp": eng.mlp(n, L1 + ".mlp")}


def run(state):
    c, eng = state["case"], state["engine"]
    kind = c["kind"]
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    if kind == "layers":
        return _layers(state)
    if kind == "mlp":
        return eng.mlp(state["x"], L0 + ".mlp")
    if kind == "linear":
        return eng.linear(state["x"], L0 + ".proj")
    if kind == "vision":
        b = "model.visual.blocks.0."
        return {"qkv": eng.linear(state["x"], b + "attn.qkv"), "fc1": eng.linear(state["x"], b + "mlp.linear_fc1"),
                "fc2": eng.linear(state["hid"], b + "mlp.linear_fc2")}
    logits = eng.linear(state["x"], "lm_head")
    return {"logits": logits, "candidates": fp8lin.vocabulary_candidates(logits)}


# ---- what a pass cannot do without ------------------------------------------


def _gemm(m, n, k, weight="fp8"):
    """(weight bytes, flops) of one projection."""
    scales = {"bf16": 0, "cached": 0, "fp8_row": 4 * n}.get(weight, 4 * n * -(-k // 128))
    return n * k * (2 if weight in ("bf16", "cached") else 1) + scales, 2.0 * m * n * k


def work(case):
    m, kind = case["m"], case["kind"]
    if kind == "layers":
        h, inter, d = case["hidden"], case["inter"], case["head_dim"]
        qkv, o, din, g, dout = 2 * (case["heads"] + case["kv_heads"]) * d, case["heads"] * d, case["delta_in"], case["delta_gates"], case["delta_out"]
        parts = [_gemm(m, qkv, h), _gemm(m, h, o), _gemm(m, din, h), _gemm(m, g, h, "bf16"), _gemm(m, h, dout)]
        parts += 2 * [_gemm(m, 2 * inter, h), _gemm(m, h, inter)]
        # x, the two attention cores; q, gate, k, v, the delta projection, residual and the last MLP's output
        values = m * (h + o + dout) + m * (2 * o + 2 * case["kv_heads"] * d + din + g + 2 * h)
    elif kind == "mlp":
        h, inter = case["hidden"], case["inter"]
        parts, values = [_gemm(m, 2 * inter, h), _gemm(m, h, inter)], 2 * m * h
    elif kind == "vision":
        h, inter = case["hidden"], case["inter"]
        parts = [_gemm(m, 3 * h, h, "bf16"), _gemm(m, inter, h, "bf16"), _gemm(m, h, inter, "bf16")]
        values = m * (h + inter) + m * (3 * h + inter + h)
    else:
        n, k = case["n"], case["k"]
        parts, values = [_gemm(m, n, k, case.get("weight", "fp8"))], m * (n + k)
    return {"bytes": sum(p[0] for p in parts) + 2 * values, "flops": sum(p[1] for p in parts)}


def tolerance(case):
    return _TOLERANCE[case["kind"]]


# BF16 outputs of sums in FP32.  One projection is 1.7e-3 off its 64-bit value (the output's rounding); another order
# of its sum moves a rounding here and there.  Two layers pass their roundings on.
_TOLERANCE = {"linear": {"rel": 7e-3, "max": 0.04}, "vision": {"rel": 7e-3, "max": 0.04}, "head": {"rel": 7e-3, "max": 0.04},
              "mlp": {"rel": 1.4e-2, "max": 0.1}, "layers": {"rel": 2.8e-2, "max": 0.2}}


# ---- the same in 64 bits ----------------------------------------------------


def _weight64(data, scale):
    """The weight that the layer is defined with: bf16(code * scale), or the BF16 matrix itself."""
    if scale is None:
        return data.double()
    w = data.view(torch.float8_e4m3fn).float()
    s = scale[:, None] if scale.dim() == 1 else scale.repeat_interleave(128, 1)[:, :data.size(1)]
    return (w * s).to(torch.bfloat16).double()


def _rms64(x, weight):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (1 + weight.double())


def _rope64(x, positions):
    """Interleaved multi-axis rotary embedding of x [T, H, D]."""
    rotary = int(x.size(-1) * ROPE["partial_rotary_factor"])
    half = rotary // 2
    inv = ROPE["rope_theta"] ** (-2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / rotary)
    freqs = positions.double()[:, :, None] * inv
    f = freqs[0].clone()
    for axis in (1, 2):
        f[:, axis:ROPE["mrope_section"][axis] * 3:3] = freqs[axis][:, axis:ROPE["mrope_section"][axis] * 3:3]
    cos, sin = f.cos()[:, None], f.sin()[:, None]
    a, b = x[..., :half], x[..., half:rotary]
    return torch.cat([a * cos - b * sin, b * cos + a * sin, x[..., rotary:]], -1)


def _mlp64(x, w, prefix):
    gate, up = torch.mm(x, _weight64(*w[prefix + ".gate_up"]).t()).chunk(2, -1)
    return torch.mm(gate * torch.sigmoid(gate) * up, _weight64(*w[prefix + ".down_proj"]).t())


def exact(case, seed):
    t, kind, m = _inputs(case, seed), case["kind"], case["m"]
    w, x = t["weights"], t["x"].double()

    def linear(v, name):
        y = torch.mm(v, _weight64(*w[name]).t())
        return y + t["biases"][name].double() if name in t["biases"] else y

    if kind == "mlp":
        return _mlp64(x, w, L0 + ".mlp")
    if kind == "linear":
        return linear(x, L0 + ".proj")
    if kind == "vision":
        b = "model.visual.blocks.0."
        return {"qkv": linear(x, b + "attn.qkv"), "fc1": linear(x, b + "mlp.linear_fc1"),
                "fc2": linear(t["hid"].double(), b + "mlp.linear_fc2")}
    if kind == "head":
        logits = linear(x, "lm_head")
        return {"logits": logits, "candidates": torch.stack([v.double() for v in logits.max(-1)], -1)}
    heads, kv, d = case["heads"], case["kv_heads"], case["head_dim"]
    n = _rms64(x, t["norm0"])
    p = linear(n, L0 + ".self_attn.qkv_gate")
    qg = p[:, :heads * 2 * d].reshape(m, heads, 2 * d)
    k, v = p[:, heads * 2 * d:].reshape(m, 2, kv, d).unbind(1)
    q = _rope64(_rms64(qg[..., :d], t["q_norm"]), t["positions"])
    r = x + linear(t["core0"].double(), L0 + ".self_attn.o_proj")
    r = r + _mlp64(_rms64(r, t["norm1"]), w, L0 + ".mlp")
    n = _rms64(r, t["norm2"])
    delta = L1 + ".linear_attn."
    proj = torch.cat([linear(n, delta + "in_proj_qkvz"), linear(n, delta + "in_proj_ba")], -1)
    r = r + linear(t["core1"].double(), delta + "out_proj")
    return {"q": q, "gate": qg[..., d:].reshape(m, heads * d), "k": _rope64(_rms64(k, t["k_norm"]), t["positions"]), "v": v,
            "proj": proj, "residual": r, "mlp": _mlp64(_rms64(r, t["norm3"]), w, L1 + ".mlp")}
