"""Workloads of the quantized-linear path through pulsarlm_amd.ops, for timing one version of
the library against another: the linears of decoder layers at decode batch sizes (captured
once in a HIP graph and replayed, as a serving loop does), single GEMMs at prefill sizes
(eager calls, their row count changes from call to call) and MoE blocks from router logits.

``listed()`` gives fixed cases, ``draw(rng)`` more of the same ranges; ``prepare`` makes inputs
and repacked weights from a seed, ``run`` is one pass, ``work`` its unavoidable bytes and
operations, ``tolerance`` the allowed relative error and ``exact`` the same outputs in float64
by plain torch.
"""

from __future__ import annotations

import math

import torch

from pulsarlm_amd import ops

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# Largest drawn GEMM and MoE block (flop): the largest listed ones.
_MAX_GEMM_FLOPS = 2.0 * 4096 * 24576 * 4096
_MAX_MOE_FLOPS = 2.0 * 4096 * 8 * 3 * 2048 * 768
# Weights one captured decode pass reads: past the 256 MB Infinity Cache, as a whole model's are.
_DECODE_BYTES = 320e6


def _layer(name, fmt, m, layers, hidden, qkv, inter, dtype="bf16", group=128, scale="fp16"):
    return {"name": name, "kind": "layer", "fmt": fmt, "m": m, "layers": layers, "hidden": hidden, "qkv": qkv,
            "inter": inter, "dtype": dtype, "group": group, "scale": scale}


def _gemm(name, fmt, m, n, k, dtype="bf16", group=128, scale="fp16"):
    return {"name": name, "kind": "gemm", "fmt": fmt, "m": m, "n": n, "k": k, "dtype": dtype, "group": group,
            "scale": scale}


def _moe(name, tokens, graph, experts=128, top_k=8, hidden=2048, inter=768, dtype="bf16", group=128):
    return {"name": name, "kind": "moe", "tokens": tokens, "graph": graph, "experts": experts, "top_k": top_k,
            "hidden": hidden, "inter": inter, "dtype": dtype, "group": group}


def listed():
    return [
        # One user's token: batch-1 decode of four Qwen3-8B layers, int4 weights.
        _layer("layer_int4_m1", "int4", 1, 4, 4096, 6144, 12288),
        # A small server's decode batch, not a power of two.
        _layer("layer_int4_m12", "int4", 12, 4, 4096, 6144, 12288),
        # A busy server's decode batch (continuous batching).
        _layer("layer_int4_m48", "int4", 48, 4, 4096, 6144, 12288),
        # Decode of a block-scaled fp8 checkpoint, Qwen3-27B-like layer, bf16 activations.
        _layer("layer_fp8_m4", "fp8", 4, 1, 5120, 7168, 17408, scale="fp32"),
        # The smallest call: one eager batch-1 projection.
        _gemm("gemm_int4_m1_small", "int4", 1, 1024, 2048),
        # A short prompt: a ragged prefill of the qkv projection.
        _gemm("gemm_int4_m333_qkv", "int4", 333, 6144, 4096),
        # A full prefill chunk through the widest projection.
        _gemm("gemm_int4_m4096_gate_up", "int4", 4096, 24576, 4096),
        # A checkpoint with 32-wide groups and fp16 activations; N and K off the tile sizes.
        _gemm("gemm_int4_g32_m200", "int4", 200, 5000, 4128, dtype="fp16", group=32),
        # Prefill of a block-scaled fp8 checkpoint with bf16 activations, ragged.
        _gemm("gemm_fp8_m1000_qkv", "fp8", 1000, 7168, 5120, scale="fp32"),
        # Prefill with per-token e4m3 activations on the fp8 matrix instructions.
        _gemm("gemm_w8a8_m2048_down", "w8a8", 2048, 5120, 17408, scale="fp32"),
        # Decode of a mixture-of-experts block (Qwen3-30B-A3B-like), a small batch.
        _moe("moe_t8", 8, True),
        # Its prefill.
        _moe("moe_t4096", 4096, False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "gemm", "gemm", "moe"])
    if kind == "layer":
        fmt = rng.choice(["int4", "int4", "fp8", "w8a8"])
        hidden = 128 * rng.randint(16, 40)
        qkv = 128 * (hidden * rng.randint(9, 12) // 8 // 128)
        inter = 128 * (hidden * rng.randint(16, 28) // 8 // 128)
        per_layer = (hidden * (qkv + hidden + 3 * inter)) // (2 if fmt == "int4" else 1)
        c = _layer("", fmt, _log_int(rng, 1, 64), max(1, min(6, math.ceil(_DECODE_BYTES / per_layer))), hidden, qkv,
                   inter, dtype=rng.choice(["bf16", "bf16", "fp16"]),
                   group=rng.choice([128, 128, 64, 32]) if fmt == "int4" else 128,
                   scale=rng.choice(["fp16", "bf16"]) if fmt == "int4" else "fp32")
    elif kind == "gemm":
        fmt = rng.choice(["int4", "int4", "fp8", "w8a8"])
        group = rng.choice([128, 128, 64, 32]) if fmt == "int4" else 128
        while True:
            m, n = _log_int(rng, 65, 4096), _log_int(rng, 1000, 24576)
            k = group * max(1, _log_int(rng, 1024, 17408) // group)
            if 2.0 * m * n * k <= _MAX_GEMM_FLOPS:
                break
        c = _gemm("", fmt, m, n, k, dtype=rng.choice(["bf16", "bf16", "fp16"]), group=group,
                  scale=rng.choice(["fp16", "bf16", "fp32"]) if fmt == "int4" else "fp32")
    else:
        while True:
            c = _moe("", _log_int(rng, 1, 4096), False, experts=rng.choice([32, 64, 128]),
                     top_k=rng.choice([2, 4, 8]), hidden=128 * rng.randint(8, 32), inter=128 * rng.randint(3, 12),
                     dtype=rng.choice(["bf16", "bf16", "fp16"]), group=rng.choice([128, 128, 64]))
            weights = c["experts"] * 3 * c["hidden"] * c["inter"] / 2
            if c["inter"] % c["group"] == 0 and weights <= 400e6 and work(c)["flops"] <= _MAX_MOE_FLOPS:
                break
        c["graph"] = c["tokens"] <= 64
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# Inputs (all from a seeded generator on the GPU, in a fixed order)
# ---------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _raw_weight(g, fmt, n, k, group, scale):
    """Checkpoint form: (int32 [N, K/8], scales [N, K/g]) or (e4m3 [N, K], fp32 128 x 128 block scales)."""
    if fmt == "int4":
        packed = torch.randint(-2**31, 2**31, (n, k // 8), generator=g, device="cuda").to(torch.int32)
        return packed, (_randn(g, n, k // group).mul_(0.02).abs_().add_(1e-3)).to(_DTYPES[scale])
    rows = -(-n // 128)
    w = _randn(g, rows * 128, k).mul_(0.02)
    s = w.view(rows, 128, k // 128, 128).abs().amax(dim=(1, 3)).div_(448.0)
    codes = (w.view(rows, 128, k // 128, 128) / s[:, None, :, None]).view(rows * 128, k)[:n]
    return codes.to(torch.float8_e4m3fn).contiguous(), s


def _block_n(fmt):
    return 1 if fmt == "int4" else 128


def _repack(fmt, raw, group):
    if fmt == "int4":
        return ops.repack_int4_marlin_cuda(raw[0], raw[1], 1, group)
    return ops.repack_fp8_marlin_cuda(raw[0], raw[1], 128, 128)


def _linear(fmt, x, weight, n, group):
    if fmt == "int4":
        return ops.gemm_int4_marlin_cuda(x, weight[0], weight[1], n, 1, group)
    if fmt == "fp8":
        return ops.gemm_fp8_marlin_cuda(x, weight[0], weight[1], n, 128, 128)
    return ops.gemm_fp8_w8a8_cuda(x, weight[0], weight[1], n, 128, 128)


def _layer_inputs(case, seed):
    """Yields per layer ({name: (raw weight, N)}, {name: x})."""
    g = _gen(seed)
    dt = _DTYPES[case["dtype"]]
    h, qkv, inter, m = case["hidden"], case["qkv"], case["inter"], case["m"]
    for _ in range(case["layers"]):
        raw = {}
        for name, n, k in (("qkv", qkv, h), ("o", h, h), ("gate_up", 2 * inter, h), ("down", h, inter)):
            raw[name] = (_raw_weight(g, case["fmt"], n, k, case["group"], case["scale"]), n)
        yield raw, {name: _randn(g, m, h).to(dt) for name in ("qkv", "o", "gate_up")}


def _moe_inputs(case, seed):
    """(raw gate_up, raw down, h, logits): logits whose top-k follow a Zipf(1.2) popularity."""
    g = _gen(seed)
    e, h, inter, t = case["experts"], case["hidden"], case["inter"], case["tokens"]

    def experts(n, k):
        packed = torch.randint(-2**31, 2**31, (e, n, k // 8), generator=g, device="cuda").to(torch.int32)
        return packed, (_randn(g, e, n, k // case["group"]).mul_(0.02).abs_().add_(1e-3)).to(torch.float16)

    gate_up, down = experts(2 * inter, h), experts(h, inter)
    x = _randn(g, t, h).to(_DTYPES[case["dtype"]])
    order = torch.randperm(e, generator=g, device="cuda")
    popularity = -1.2 * torch.log(1.0 + order.float())
    u = torch.rand(t, e, generator=g, device="cuda").clamp_(1e-6, 1 - 1e-6)
    return gate_up, down, x, (popularity - torch.log(-torch.log(u))).to(torch.bfloat16)


_capture_stream = None


def _captured(step):
    """A HIP graph of step() and its outputs, captured after one eager pass on the capture stream."""
    global _capture_stream
    if _capture_stream is None:
        _capture_stream = torch.cuda.Stream()
    _capture_stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(_capture_stream):
        step()
    _capture_stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=_capture_stream):
        out = step()
    return graph, out


def prepare(case, seed):
    state = {"case": case}
    group = case["group"]
    if case["kind"] == "layer":
        layers = []
        for raw, x in _layer_inputs(case, seed):
            weights = {name: (_repack(case["fmt"], r, group), n) for name, (r, n) in raw.items()}
            layers.append((weights, x))
            del raw

        def linear(x, weight):
            return _linear(case["fmt"], x, weight[0], weight[1], group)

        def step():
            out = []
            for w, x in layers:
                gate_up = linear(x["gate_up"], w["gate_up"])
                act = ops.silu_mul_cuda(gate_up)
                out.append({"qkv": linear(x["qkv"], w["qkv"]), "o": linear(x["o"], w["o"]), "gate_up": gate_up,
                            "act": act, "down": linear(act, w["down"])})
            return out

        state["keep"] = layers
        state["graph"], state["out"] = _captured(step)
    elif case["kind"] == "gemm":
        g = _gen(seed)
        state["w"] = _repack(case["fmt"], _raw_weight(g, case["fmt"], case["n"], case["k"], group, case["scale"]), group)
        state["x"] = _randn(g, case["m"], case["k"]).to(_DTYPES[case["dtype"]])
    else:
        gate_up, down, x, logits = _moe_inputs(case, seed)
        gu, dn = (ops.repack_int4_experts(p, s, group) for p, s in (gate_up, down))

        def block():
            return ops.moe_block_int4_cuda(x, logits, case["top_k"], gu, dn, case["inter"], group)

        state["block"] = block
        if case["graph"]:
            state["graph"], state["out"] = _captured(block)
    return state


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    case = state["case"]
    if case["kind"] == "gemm":
        return _linear(case["fmt"], state["x"], state["w"], case["n"], case["group"])
    return state["block"]()


# ---------------------------------------------------------------------------
# Work, tolerance
# ---------------------------------------------------------------------------


def _gemm_bytes(fmt, m, n, k, group, scale):
    if fmt == "int4":
        return n * k / 2 + n * (k / group) * (4 if scale == "fp32" else 2) + 2 * m * k + 2 * m * n
    return n * k + -(-n // 128) * (k // 128) * 4 + 2 * m * k + 2 * m * n


def work(case):
    if case["kind"] == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _gemm_bytes(case["fmt"], m, n, k, case["group"], case["scale"]), "flops": 2.0 * m * n * k}
    if case["kind"] == "layer":
        h, qkv, inter, m = case["hidden"], case["qkv"], case["inter"], case["m"]
        b = f = 0.0
        for n, k in ((qkv, h), (h, h), (2 * inter, h), (h, inter)):
            b += _gemm_bytes(case["fmt"], m, n, k, case["group"], case["scale"])
            f += 2.0 * m * n * k
        return {"bytes": case["layers"] * (b + 6 * m * inter), "flops": case["layers"] * f}
    t, top_k, e, h, inter = case["tokens"], case["top_k"], case["experts"], case["hidden"], case["inter"]
    rows = t * top_k
    # Experts hit: the expected number under the router's popularity (drawn without replacement,
    # taken as independent draws).
    p = [(1.0 + i) ** -1.2 for i in range(e)]
    hit = sum(1.0 - (1.0 - min(1.0, v / sum(p))) ** rows for v in p)
    hit = max(float(min(top_k, e)), hit)
    per_expert = sum(n * k / 2 + n * k / case["group"] * 2 for n, k in ((2 * inter, h), (h, inter)))
    return {"bytes": hit * per_expert + 4 * t * h + 2 * t * e + 8 * rows, "flops": 2.0 * rows * 3 * h * inter}


def tolerance(case):
    # One rounding of the output to 16 bits is 1.7e-3 (bf16) or 2.1e-4 (fp16) of its norm; four
    # times that, and about twice as much where a rounded activation feeds a second GEMM.
    half = case["dtype"] == "fp16"
    if case["kind"] == "gemm":
        if case["fmt"] == "w8a8":
            return {"rel": 7e-3}
        return {"rel": 1e-3 if half else 7e-3}
    if case["kind"] == "layer" and case["fmt"] == "w8a8":
        return {"rel": 2e-2}  # a flipped rounding of the activation may flip its e4m3 code
    return {"rel": 2e-3 if half else 1.2e-2}


# ---------------------------------------------------------------------------
# Float64 restatement
# ---------------------------------------------------------------------------


def _dense(fmt, raw, group, dtype):
    """The dequantized weight round(q * round(s)) in ``dtype``, as float64 (W8A8: q * s unrounded)."""
    w, s = raw
    if fmt == "int4":
        q = torch.stack([(w << (28 - 4 * j)) >> 28 for j in range(8)], dim=-1).flatten(-2)
        sd = s.to(dtype).to(torch.float64).repeat_interleave(group, dim=-1)
        return (q.to(torch.float64) * sd).to(dtype).to(torch.float64)
    n, k = w.shape
    sd = s if fmt == "w8a8" else s.to(dtype)
    sd = sd.to(torch.float64).repeat_interleave(128, dim=0)[:n].repeat_interleave(128, dim=1)[:, :k]
    dense = w.to(torch.float32).to(torch.float64) * sd
    return dense if fmt == "w8a8" else dense.to(dtype).to(torch.float64)


def _exact_linear(fmt, x, raw, group, dtype):
    """x in ``dtype`` (W8A8: rounded per row to e4m3 with scale max(amax, 1e-12) / 448)."""
    if fmt == "w8a8":
        xf = x.to(torch.float32)
        sx = xf.abs().amax(dim=1, keepdim=True).clamp_min(1e-12) / 448.0
        xd = (xf / sx).to(torch.float8_e4m3fn).to(torch.float32).to(torch.float64) * sx.to(torch.float64)
    else:
        xd = x.to(torch.float64)
    return xd @ _dense(fmt, raw, group, dtype).t()


def exact(case, seed):
    dt, group = _DTYPES[case["dtype"]], case["group"]
    if case["kind"] == "gemm":
        g = _gen(seed)
        raw = _raw_weight(g, case["fmt"], case["n"], case["k"], group, case["scale"])
        return _exact_linear(case["fmt"], _randn(g, case["m"], case["k"]).to(dt), raw, group, dt)
    if case["kind"] == "layer":
        inter, out = case["inter"], []
        for raw, x in _layer_inputs(case, seed):
            y = {name: _exact_linear(case["fmt"], x[name], raw[name][0], group, dt) for name in x}
            # The W8A8 quantizer sees the activation in its own 16-bit type.
            gate_up = y["gate_up"].to(dt).to(torch.float64) if case["fmt"] == "w8a8" else y["gate_up"]
            act = torch.nn.functional.silu(gate_up[:, :inter])
            if case["fmt"] == "w8a8":
                act = act.to(dt).to(torch.float64)
            act = act * gate_up[:, inter:]
            y["act"] = act
            if case["fmt"] == "w8a8":
                act = act.to(dt)
            y["down"] = _exact_linear(case["fmt"], act, raw["down"][0], group, dt)
            out.append({name: y[name] for name in ("qkv", "o", "gate_up", "act", "down")})
        return out
    gate_up, down, x, logits = _moe_inputs(case, seed)
    inter, top_k = case["inter"], case["top_k"]
    prob = torch.softmax(logits.to(torch.float64), dim=1)
    value, chosen = torch.sort(prob, dim=1, descending=True, stable=True)
    value, chosen = value[:, :top_k], chosen[:, :top_k]
    weights = value / value.sum(dim=1, keepdim=True)
    out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    xd = x.to(torch.float64)
    for e in range(case["experts"]):
        token, slot = torch.nonzero(chosen == e, as_tuple=True)
        if token.numel() == 0:
            continue
        gu = xd[token] @ _dense("int4", (gate_up[0][e], gate_up[1][e]), group, dt).t()
        act = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
        y = act @ _dense("int4", (down[0][e], down[1][e]), group, dt).t()
        out.index_add_(0, token, y * weights[token, slot][:, None])
    return out, None, weights, None
