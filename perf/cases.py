"""Performance cases: what users of the grouped-GEMM library have it do, through its public entry points.

Nine kinds of work.  Each has one or two listed cases and a range of sizes and options that ``draw`` samples:

  gemm       one ``m_grouped_gemm``: every projection of an expert layer, forward (``trans_b``) or activation gradient
  layer      an expert feed-forward layer: route, gate/up projection, SwiGLU, down projection, weighted combine; as one
             decode step without gradients, or as a training step that returns the gradients of everything
  route      the token movement of such a layer alone (permute, unpermute and their gradients)
  masked     ``m_grouped_gemm_masked``: decode with a fixed number of row slots per expert
  wgrad      ``k_grouped_gemm``: the weight gradient of one projection
  fp8_block  activations quantised 1x128 on the GPU, then the block-scaled FP8 GEMM
  fp8_channel, fp8_wgrad   the per-channel scaled FP8 GEMMs, forward and weight gradient
  quantize   the transposing 128x128 quantizer that feeds FP8 weight gradients

Shapes are those of the repository's benchmark and tests (128 experts; N x K of 1536 x 2048, 2048 x 768, 3072 x 4096
and 4096 x 1536; 655360 rows at the top, a few hundred rows at the bottom) and generic ones between them.  Group sizes
are drawn from the seed the way the benchmark draws them: a Dirichlet(1) vector over the experts and a multinomial
draw of rows (or of blocks of 128 rows where a contract asks for padded experts), so experts are unequal and some are
empty.  Activations are N(0, 1), weights N(0, 1) / sqrt(K).
"""
import math

import torch
import torch.nn.functional as F

from triton_grouped_gemm_amd import ops
from triton_grouped_gemm_amd.gemm.BF16.k_grouped_gemm import k_grouped_gemm
from triton_grouped_gemm_amd.gemm.BF16.m_grouped_gemm import m_grouped_gemm
from triton_grouped_gemm_amd.gemm.BF16.m_grouped_gemm_masked_TMA import m_grouped_gemm_masked
from triton_grouped_gemm_amd.gemm.FP8.k_grouped_gemm_channel_expert import matmul as fp8_k_grouped
from triton_grouped_gemm_amd.gemm.FP8.m_grouped_gemm_channel_expert import gmm_fp8_act_per_channel_w_per_expert
from triton_grouped_gemm_amd.gemm.deep_gemm_ops import m_grouped_fp8_nt_contiguous
from triton_grouped_gemm_amd.quant.fp8_cast import per_block_cast_to_fp8, per_token_cast_to_fp8
from triton_grouped_gemm_amd.quant.trans_per_block_quant_expand_128x import trans_per_block_quant_expand_128x

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32,
          "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
ELEMENT_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4, "e4m3": 1, "e5m2": 1}

# A pass never costs more than the largest listed case.
MOST_FLOPS = 4.1e12
MOST_BYTES = 5.5e9


def listed():
    return [
        # The smallest call: the four ragged groups of the repository's smallest configuration.  Launch and host time.
        {"name": "gemm_tiny", "kind": "gemm", "dtype": "bf16", "trans_b": True, "groups": 4, "rows": 320, "n": 512,
         "k": 256, "align": 1},
        # An ordinary forward projection in half precision, [K, N] weights, no size a multiple of a tile.
        {"name": "gemm_ragged_nn", "kind": "gemm", "dtype": "fp16", "trans_b": False, "groups": 64, "rows": 20011,
         "n": 1416, "k": 2056, "align": 1},
        # The largest call: the gate/up projection of a prefill or training batch, the repository's headline.
        {"name": "gemm_prefill", "kind": "gemm", "dtype": "bf16", "trans_b": True, "groups": 128, "rows": 655360,
         "n": 1536, "k": 2048, "align": 128},
        # One decode step of a small batch: a row or two per expert, the layer streams weights.
        {"name": "layer_decode", "kind": "layer", "train": False, "dtype": "bf16", "tokens": 24, "topk": 8,
         "experts": 128, "hidden": 2048, "ffn": 768},
        # One training step of the layer on a micro-batch: both projections forward and backward, weight gradients,
        # and the token movement either side.
        {"name": "layer_train", "kind": "layer", "train": True, "dtype": "bf16", "tokens": 4096, "topk": 8,
         "experts": 128, "hidden": 2048, "ffn": 768},
        # Token movement of an ordinary batch, forward and backward.
        {"name": "route_train", "kind": "route", "dtype": "bf16", "tokens": 8192, "topk": 8, "experts": 128,
         "hidden": 2048},
        # Decode with 512 row slots per expert, filled at random (the repository's decode configuration).
        {"name": "masked_decode", "kind": "masked", "dtype": "bf16", "groups": 128, "slots": 512, "fill": 1.0,
         "n": 4096, "k": 1536},
        # Weight gradient of the gate/up projection of a micro-batch: a few hundred ragged tokens per expert.
        {"name": "wgrad", "kind": "wgrad", "dtype": "bf16", "groups": 128, "rows": 32771, "m": 2048, "n": 1536},
        # FP8 prefill with 128-padded experts: 1x128 quantisation of the activations and the block-scaled GEMM.
        {"name": "fp8_block_prefill", "kind": "fp8_block", "groups": 128, "rows": 65536, "n": 3072, "k": 4096,
         "mn_major": True},
        # FP8 forward of a moderate batch, e5m2 activations and e4m3 weights with per-token and per-channel scales.
        {"name": "fp8_channel", "kind": "fp8_channel", "groups": 32, "rows": 8192, "n": 3072, "k": 4096, "act": "e5m2",
         "out": "fp16"},
        # FP8 weight gradient, every expert's tokens padded to 128.
        {"name": "fp8_wgrad", "kind": "fp8_wgrad", "groups": 32, "rows": 32768, "m": 3072, "n": 4096, "act": "e4m3"},
        # The quantizer in front of it, on ragged experts.
        {"name": "quantize", "kind": "quantize", "groups": 64, "rows": 33001, "n": 4096, "dtype": "e4m3"},
    ]


# ---- further cases of the same ranges --------------------------------------------------------------------------

WIDTHS = (512, 768, 1024, 1408, 1536, 2048, 2816, 3072, 4096)


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _width(rng, step):
    """A layer width: mostly one in use, one time in three any multiple of ``step``."""
    if rng.random() < 2 / 3:
        return rng.choice(WIDTHS)
    return step * _log_int(rng, 256 // step, 4096 // step)


def _draw_once(rng):
    kind = rng.choice(["gemm", "gemm", "layer", "layer", "route", "masked", "wgrad", "fp8_block", "fp8_channel",
                       "fp8_wgrad", "quantize"])
    groups = rng.choice([4, 8, 16, 32, 64, 128, _log_int(rng, 4, 256)])
    if kind == "gemm":
        align = rng.choice([1, 1, 128])
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "fp16"]), "trans_b": rng.random() < 0.5,
                "groups": groups, "rows": align * _log_int(rng, 256 // align, 655360 // align), "n": _width(rng, 8),
                "k": _width(rng, 8), "align": align}
    if kind == "layer":
        train = rng.random() < 0.5
        experts = rng.choice([8, 16, 32, 64, 128])
        return {"kind": kind, "train": train, "dtype": rng.choice(["bf16", "bf16", "fp16"]),
                "tokens": _log_int(rng, 256, 16384) if train else _log_int(rng, 1, 512),
                "topk": rng.choice([1, 2, 4, 8]), "experts": experts, "hidden": rng.choice([1024, 2048, 2880, 4096]),
                "ffn": rng.choice([512, 768, 1024, 1408, 1536])}
    if kind == "route":
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"]), "tokens": _log_int(rng, 16, 81920),
                "topk": rng.choice([1, 2, 4, 6, 8]), "experts": max(8, groups),
                "hidden": rng.choice([1024, 2048, 2880, 4096])}
    if kind == "masked":
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "fp16"]), "groups": groups,
                "slots": rng.choice([128, 256, 512]), "fill": rng.choice([0.05, 0.25, 1.0]), "n": _width(rng, 8),
                "k": _width(rng, 8)}
    if kind == "wgrad":
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "fp16"]), "groups": groups,
                "rows": _log_int(rng, 256, 262144), "m": _width(rng, 8), "n": _width(rng, 8)}
    if kind == "fp8_block":
        return {"kind": kind, "groups": groups, "rows": 128 * _log_int(rng, 4, 2048), "n": _width(rng, 128),
                "k": _width(rng, 128), "mn_major": rng.random() < 0.5}
    if kind == "fp8_channel":
        return {"kind": kind, "groups": groups, "rows": _log_int(rng, 128, 262144), "n": _width(rng, 16),
                "k": _width(rng, 16), "act": rng.choice(["e4m3", "e5m2"]), "out": rng.choice(["bf16", "fp16"])}
    if kind == "fp8_wgrad":
        return {"kind": kind, "groups": groups, "rows": 128 * _log_int(rng, 4, 2048), "m": _width(rng, 16),
                "n": _width(rng, 16), "act": rng.choice(["e4m3", "e5m2"])}
    return {"kind": kind, "groups": groups, "rows": _log_int(rng, 512, 262144), "n": _width(rng, 128),
            "dtype": rng.choice(["e4m3", "e4m3", "e5m2"])}


def draw(rng):
    while True:
        case = _draw_once(rng)
        w = work(case)
        if w["flops"] <= MOST_FLOPS and w["bytes"] <= MOST_BYTES:
            return case


# ---- inputs ----------------------------------------------------------------------------------------------------

def _expert_rows(groups, rows, align, gen):
    """int32 ``[groups]`` on the CPU, summing to ``rows`` exactly: Dirichlet(1) shares, multinomial blocks of ``align``."""
    shares = torch._standard_gamma(torch.ones(groups, dtype=torch.float64), generator=gen)
    blocks = torch.multinomial(shares / shares.sum(), rows // align, replacement=True, generator=gen)
    return (torch.bincount(blocks, minlength=groups) * align).to(torch.int32)


class _Source:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.cpu = torch.Generator().manual_seed(seed)
        self.gpu = torch.Generator(device="cuda").manual_seed(seed)

    def randn(self, *shape, dtype, scale=1.0):
        out = torch.empty(shape, device="cuda", dtype=dtype)
        flat = out.view(-1)
        step = 1 << 28
        for at in range(0, flat.numel(), step):
            part = flat[at:at + step]
            part.copy_(torch.randn(part.numel(), device="cuda", generator=self.gpu).mul_(scale))
        return out

    def codes(self, *shape, dtype):
        """FP8 codes as a quantizer leaves them: a normal variable whose largest values reach the type's range."""
        out = torch.empty(shape, device="cuda", dtype=dtype)
        flat = out.view(-1)
        top = torch.finfo(dtype).max
        step = 1 << 28
        for at in range(0, flat.numel(), step):
            part = flat[at:at + step]
            part.copy_(torch.randn(part.numel(), device="cuda", generator=self.gpu).mul_(top / 4.5).clamp_(-top, top))
        return out

    def scales(self, *shape, dtype):
        """The scales that belong to such codes: largest absolute value over the type's range."""
        top = torch.finfo(dtype).max
        return torch.rand(shape, device="cuda", generator=self.gpu).add_(3.5).div_(top)

    def sizes(self, groups, rows, align):
        return _expert_rows(groups, rows, align, self.cpu).cuda()

    def routing(self, tokens, experts, topk):
        """Top-k of router logits with a preference for some experts: int32 assignment and fp32 probabilities."""
        logits = torch.randn(tokens, experts, device="cuda", generator=self.gpu)
        logits += 0.5 * torch.randn(experts, device="cuda", generator=self.gpu)
        probs, idx = torch.softmax(logits, -1).topk(topk, dim=-1)
        return idx.to(torch.int32), probs.contiguous()


def prepare(case, seed):
    src = _Source(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind in ("gemm", "masked"):
        dt, g, n, k = DTYPES[case["dtype"]], case["groups"], case["n"], case["k"]
        trans_b = case.get("trans_b", True)
        s["b"] = src.randn(*((g, n, k) if trans_b else (g, k, n)), dtype=dt, scale=k ** -0.5)
        if kind == "gemm":
            s["a"] = src.randn(case["rows"], k, dtype=dt)
            s["sizes"] = src.sizes(g, case["rows"], case["align"])
        else:
            slots = case["slots"]
            most = max(1, int(slots * case["fill"]))
            s["a"] = src.randn(g * slots, k, dtype=dt)
            s["out"] = torch.zeros(g * slots, n, device="cuda", dtype=dt)
            s["sizes"] = torch.randint(0, most + 1, (g,), generator=src.cpu, dtype=torch.int32).cuda()
    elif kind == "layer":
        dt, h, f, e = DTYPES[case["dtype"]], case["hidden"], case["ffn"], case["experts"]
        s["x"] = src.randn(case["tokens"], h, dtype=dt)
        s["w1"] = src.randn(e, 2 * f, h, dtype=dt, scale=h ** -0.5)
        s["w2"] = src.randn(e, h, f, dtype=dt, scale=f ** -0.5)
        s["idx"], s["probs"] = src.routing(case["tokens"], e, case["topk"])
        if case["train"]:
            s["grad"] = src.randn(case["tokens"], h, dtype=dt)
            for name in ("x", "w1", "w2", "probs"):
                s[name].requires_grad_(True)
    elif kind == "route":
        dt, h = DTYPES[case["dtype"]], case["hidden"]
        s["x"] = src.randn(case["tokens"], h, dtype=dt).requires_grad_(True)
        s["idx"], probs = src.routing(case["tokens"], case["experts"], case["topk"])
        s["probs"] = probs.requires_grad_(True)
        s["grad"] = src.randn(case["tokens"], h, dtype=dt)
    elif kind == "wgrad":
        dt = DTYPES[case["dtype"]]
        s["a"] = src.randn(case["rows"], case["m"], dtype=dt)
        s["b"] = src.randn(case["rows"], case["n"], dtype=dt)
        s["sizes"] = src.sizes(case["groups"], case["rows"], 1)
    elif kind == "fp8_block":
        g, n, k = case["groups"], case["n"], case["k"]
        s["x"] = src.randn(case["rows"], k, dtype=torch.bfloat16)
        s["sizes"] = src.sizes(g, case["rows"], 128)
        s["w"] = per_block_cast_to_fp8(src.randn(g, n, k, dtype=torch.bfloat16, scale=k ** -0.5))
    elif kind == "fp8_channel":
        g, m, n, k = case["groups"], case["rows"], case["n"], case["k"]
        act = DTYPES[case["act"]]
        s["a"], s["a_scale"] = src.codes(m, k, dtype=act), src.scales(m, 1, dtype=act)
        s["b"] = src.codes(g, n, k, dtype=torch.float8_e4m3fn)
        s["b_scale"] = src.scales(g, n, dtype=torch.float8_e4m3fn) * k ** -0.5
        s["sizes"] = src.sizes(g, m, 1)
    elif kind == "fp8_wgrad":
        g, t, m, n = case["groups"], case["rows"], case["m"], case["n"]
        act = DTYPES[case["act"]]
        s["x"], s["x_scale"] = src.codes(m, t, dtype=act), src.scales(g, m, dtype=act).t()
        s["y"] = src.codes(n, t, dtype=torch.float8_e4m3fn)
        s["y_scale"] = src.scales(g, n, dtype=torch.float8_e4m3fn).t()
        s["sizes"] = src.sizes(g, t, 128)
    else:
        s["x"] = src.randn(case["rows"], case["n"], dtype=torch.bfloat16)
        s["sizes"] = src.sizes(case["groups"], case["rows"], 1)
    return s


# ---- one pass --------------------------------------------------------------------------------------------------

def _layer(s):
    case = s["case"]
    rows, row_id_map = ops.permute(s["x"], s["idx"], num_experts=case["experts"])
    _, sizes = ops.permute_map(s["idx"], num_experts=case["experts"])
    gate, up = ops.gmm(rows, s["w1"], sizes, trans_b=True).chunk(2, dim=-1)
    y = ops.gmm(F.silu(gate) * up, s["w2"], sizes, trans_b=True)
    return ops.unpermute(y, row_id_map, s["probs"])


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "gemm":
        return m_grouped_gemm(s["a"], s["b"], s["sizes"], case["trans_b"])
    if kind == "layer":
        if not case["train"]:
            with torch.no_grad():
                return _layer(s)
        out = _layer(s)
        return (out.detach(), *torch.autograd.grad(out, (s["x"], s["w1"], s["w2"], s["probs"]), s["grad"]))
    if kind == "route":
        rows, row_id_map = ops.permute(s["x"], s["idx"], num_experts=case["experts"])
        out = ops.unpermute(rows, row_id_map, s["probs"])
        grads = torch.autograd.grad(out, (s["x"], s["probs"]), s["grad"])
        return (rows.detach(), row_id_map, out.detach(), *grads)
    if kind == "masked":
        m_grouped_gemm_masked(s["a"], s["b"], s["out"], s["sizes"], case["slots"])
        return s["out"]
    if kind == "wgrad":
        return k_grouped_gemm(s["a"], s["b"], s["sizes"])
    if kind == "fp8_block":
        x = per_token_cast_to_fp8(s["x"], scales_mn_major=case["mn_major"])
        return m_grouped_fp8_nt_contiguous(x, s["w"], s["sizes"])
    if kind == "fp8_channel":
        return gmm_fp8_act_per_channel_w_per_expert(s["a"], s["a_scale"], s["b"], s["b_scale"], s["sizes"],
                                                    DTYPES[case["out"]])
    if kind == "fp8_wgrad":
        return fp8_k_grouped(s["x"], s["x_scale"], s["y"], s["y_scale"], s["sizes"], case["m"], case["n"], case["rows"],
                             case["groups"], 1 if case["act"] == "e4m3" else 2, 1)
    return trans_per_block_quant_expand_128x(s["x"], s["sizes"], dtype=DTYPES[case["dtype"]])


# ---- what a pass cannot do without -----------------------------------------------------------------------------

def _used(groups, rows, align=1):
    """Expected number of experts with rows under Dirichlet(1) shares and ``rows / align`` multinomial draws."""
    draws = rows // align
    return groups * draws / (draws + groups - 1)


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        e, m, n, k = ELEMENT_BYTES[case["dtype"]], case["rows"], case["n"], case["k"]
        weights = _used(case["groups"], m, case["align"]) * n * k
        return {"bytes": e * (m * k + weights + m * n), "flops": 2 * m * n * k}
    if kind == "masked":
        e, n, k = ELEMENT_BYTES[case["dtype"]], case["n"], case["k"]
        most = max(1, int(case["slots"] * case["fill"]))
        m = case["groups"] * most / 2
        weights = case["groups"] * most / (most + 1) * n * k
        return {"bytes": e * (m * k + weights + m * n), "flops": 2 * m * n * k}
    if kind == "layer":
        e, t, h, f = ELEMENT_BYTES[case["dtype"]], case["tokens"], case["hidden"], case["ffn"]
        used = case["experts"] * (1 - (1 - case["topk"] / case["experts"]) ** t)
        m = t * case["topk"]
        # token rows in and out, permuted rows, both projections' results and the activation, each written and read
        forward = 2 * t * h + 2 * m * (h + 2 * f + f + h) + used * 3 * f * h
        if not case["train"]:
            return {"bytes": e * forward, "flops": 6 * m * f * h}
        # backward: the gradient of each of those rows, the saved rows and weights read again, two weight gradients
        backward = 2 * t * h + 2 * m * (h + 2 * f + f + h) + m * (h + 2 * f + f + h) + used * 3 * f * h
        return {"bytes": e * (forward + backward + case["experts"] * 3 * f * h), "flops": 18 * m * f * h}
    if kind == "route":
        e, t, h, k = ELEMENT_BYTES[case["dtype"]], case["tokens"], case["hidden"], case["topk"]
        return {"bytes": e * h * (4 * t + 5 * t * k) + 16 * t * k, "flops": 6 * t * k * h}
    if kind == "wgrad":
        e, t, m, n = ELEMENT_BYTES[case["dtype"]], case["rows"], case["m"], case["n"]
        return {"bytes": e * (t * (m + n) + case["groups"] * m * n), "flops": 2 * t * m * n}
    if kind == "fp8_block":
        m, n, k = case["rows"], case["n"], case["k"]
        weights = _used(case["groups"], m, 128) * n * k
        return {"bytes": 2 * m * k + 2 * m * k * (1 + 4 / 128) + weights + 2 * m * n, "flops": 2 * m * n * k}
    if kind == "fp8_channel":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": m * k + _used(case["groups"], m) * n * k + 2 * m * n, "flops": 2 * m * n * k}
    if kind == "fp8_wgrad":
        t, m, n = case["rows"], case["m"], case["n"]
        return {"bytes": t * (m + n) + 2 * case["groups"] * m * n, "flops": 2 * t * m * n}
    m, n = case["rows"], case["n"]
    return {"bytes": 2 * m * n + n * (m + 128 * case["groups"] - m % 128), "flops": 4 * m * n}


def tolerance(case):
    """Relative error (2-norm) that another correct implementation at the same precision shows: four times the largest
    that these paths show against 64-bit arithmetic (one rounding to bf16 1.7e-3, two in the routed row movers 2.0e-3,
    a layer's chain of them 4.5e-3; fp16 an eighth of that; fp32 row movers 1e-7)."""
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    kept = case["out"] if kind == "fp8_channel" else case.get("dtype", "bf16")
    if kind == "layer":
        return {"rel": 1.8e-2 if kept == "bf16" else 2.2e-3}
    return {"rel": {"bf16": 8e-3, "fp16": 1e-3, "fp32": 5e-7}[kept]}
