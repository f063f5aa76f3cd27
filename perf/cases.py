"""Performance cases of the MoE hot path: what a user of this package has it do, at the sizes it is used at.

Seven kinds of work, each through public entry points.  The operators that the reference library also has are called
as torch.ops.umdk_cam_op_lib.*, the ones that only this package has as functions of umdk_original_amd:

  layer       fused_deep_moe: a whole w8a8 MoE layer (routing plan, permute + int8 quantisation, gate/up GEMM, SwiGLU,
              re-quantisation, down GEMM, combine), bf16 or fp16 tokens, with or without a mask of active tokens
  layer_fp8   fused_deep_moe_fp8: the same layer with block-scaled FP8 weights and activations
  exchange    moe_dispatch_fused, then moe_combine_gather with the dispatch's map: the two halves around a caller's own
              experts; copied, int8 or FP8 rows out, 16-bit or int8 wire rows back, with or without a shared expert
  normal      get_dispatch_layout, moe_dispatch_prefill and moe_combine_prefill: the prefill operators in a row
  shmem       moe_dispatch_shmem, then moe_combine_shmem: the decode pair
  experts     grouped_matmul_swiglu_quant, then grouped_matmul_dequant: the two expert GEMMs alone, with the rows per
              expert skewed

Inputs are N(0,1) activations, sigmoid routing scores with a Zipf-skewed expert bias (few experts or top-1 and top-2:
softmax scores without a bias; no expert id occurs twice for a token), weights N(0, 1/K) quantised per output channel
(int8) or per 128 x 128 block (FP8).
"""
import math

import torch

import umdk_original_amd as cam
from umdk_original_amd import synth

OPS = torch.ops.umdk_cam_op_lib
MAX_BYTES = 2.6e9   # of a drawn case, about the largest listed one
MAX_FLOPS = 2.45e12


def listed():
    return [
        # One user's next token: 8 of 128 experts are read and nothing else; launches and latency count.
        dict(name="layer_one_token", kind="layer", tokens=1, hidden=4096, experts=128, top_k=8, inter=1536,
             dtype="bf16", active=1.0),
        # A small model's layer (the golden configuration of the tests): launches count, little work in each.
        dict(name="layer_small", kind="layer", tokens=128, hidden=1024, experts=8, top_k=2, inter=512,
             dtype="bf16", active=1.0),
        # One rank's share of a wide layer, as the fused operator's unit tests call it: few tokens, every expert hit.
        dict(name="layer_rank_share", kind="layer", tokens=16, hidden=7168, experts=16, top_k=8, inter=2048,
             dtype="bf16", active=1.0),
        # A full decode batch: all weights streamed once.
        dict(name="layer_decode", kind="layer", tokens=128, hidden=4096, experts=128, top_k=8, inter=1536,
             dtype="bf16", active=1.0),
        # A chunk of a prompt, ragged, fp16 tokens, an intermediate size that is no multiple of 512.
        dict(name="layer_chunk_fp16", kind="layer", tokens=1021, hidden=2048, experts=64, top_k=6, inter=1408,
             dtype="fp16", active=1.0),
        # A long prompt: matrix bound, the largest case.
        dict(name="layer_prefill", kind="layer", tokens=8192, hidden=4096, experts=128, top_k=8, inter=1536,
             dtype="bf16", active=1.0),
        # A decode batch padded to 64 slots of which 48 are in use, block-scaled FP8.
        dict(name="fp8_decode", kind="layer_fp8", tokens=64, hidden=4096, experts=128, top_k=8, inter=1536,
             dtype="bf16", active=0.75),
        # A prompt in block-scaled FP8, odd token count.
        dict(name="fp8_prefill", kind="layer_fp8", tokens=4093, hidden=4096, experts=128, top_k=8, inter=1536,
             dtype="bf16", active=1.0),
        # Dispatch and combine of the benchmark: 4096 tokens x 7168 to 256 experts and back.
        dict(name="exchange_prefill", kind="exchange", tokens=4096, hidden=7168, experts=256, top_k=8, dtype="bf16",
             quant=2, wire=False, shared=False),
        # The prefill operators as a model calls them one after the other, unquantised rows, odd token count.
        dict(name="normal_prefill", kind="normal", tokens=1999, hidden=4096, experts=64, top_k=6, dtype="bf16"),
        # The decode pair: int8 rows out, bf16 rows back.
        dict(name="shmem_decode", kind="shmem", tokens=128, hidden=7168, experts=256, top_k=8, dtype="bf16", quant=2,
             smooth=False),
        # The expert GEMMs of one rank's 32 experts over 8192 rows, three experts empty.
        dict(name="experts_skewed", kind="experts", rows=8192, hidden=7168, experts=32, inter=2048),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer_fp8", "layer_fp8", "exchange", "normal", "shmem", "experts"])
    if kind in ("layer", "layer_fp8"):
        experts = _log(rng, 4, 256)
        case = dict(kind=kind, tokens=_log(rng, 1, 8192), hidden=128 * rng.randint(8, 56), experts=experts,
                    top_k=rng.randint(1, min(8, experts)), inter=128 * rng.randint(4, 24),
                    dtype="bf16" if kind == "layer_fp8" else rng.choice(["bf16", "bf16", "fp16"]), active=1.0)
        if case["tokens"] <= 256 and rng.random() < 0.25:
            case["active"] = round(rng.uniform(0.5, 1.0), 2)
    elif kind == "experts":
        case = dict(kind=kind, rows=_log(rng, 64, 16384), hidden=128 * rng.randint(8, 56), experts=_log(rng, 4, 64),
                    inter=128 * rng.randint(4, 24))
    else:
        experts = _log(rng, 8, 512)
        hidden = 8 * rng.randint(128, 896)
        case = dict(kind=kind, tokens=_log(rng, 1, 8000 if kind != "shmem" else 512), hidden=hidden, experts=experts,
                    top_k=rng.randint(1, min(8, experts)), dtype=rng.choice(["bf16", "bf16", "fp16"]))
        if kind == "exchange":
            case["quant"] = rng.choice([0, 2, 2, 4])
            case["wire"] = rng.random() < 0.25
            case["shared"] = rng.random() < 0.25
            if case["quant"] == 4:
                case["dtype"], case["hidden"] = "bf16", (hidden + 127) // 128 * 128
        if kind == "shmem":
            case["quant"] = rng.choice([0, 2, 2])
            case["smooth"] = case["quant"] == 2 and rng.random() < 0.5
    # no dearer than the dearest listed case: fewer tokens (rows), then fewer experts
    while True:
        w = work(case)
        if w["bytes"] <= MAX_BYTES and w["flops"] <= MAX_FLOPS:
            return case
        size = "rows" if kind == "experts" else "tokens"
        if w["flops"] > MAX_FLOPS or "inter" not in case:
            case[size] = max(1, case[size] * 3 // 4)
        else:
            case["experts"] = max(4, case["experts"] * 3 // 4)
            if "top_k" in case:
                case["top_k"] = min(case["top_k"], case["experts"])


# ---------------------------------------------------------------------------------------------- inputs
def _dtype(case):
    return torch.float16 if case["dtype"] == "fp16" else torch.bfloat16


def _routing(case, gen, dev):
    """[T,K] int32 ids and fp32 gate weights that sum to 1."""
    t, e, k = case["tokens"], case["experts"], case["top_k"]
    logits = torch.randn(t, e, generator=gen, device=dev)
    if e <= 8 or k <= 2:
        scores = torch.softmax(logits, dim=-1)
        ids = torch.topk(scores, k, dim=-1).indices
    else:
        scores = torch.sigmoid(logits)
        bias = torch.arange(1, e + 1, dtype=torch.float32, device=dev).pow(-1.1)
        bias = bias[torch.randperm(e, generator=gen, device=dev)]
        ids = torch.topk(scores + bias, k, dim=-1).indices
    w = torch.gather(scores, 1, ids)
    return ids.to(torch.int32).contiguous(), (w / w.sum(dim=-1, keepdim=True)).contiguous()


def _int8_weight(g, kd, n, gate_up, gen, dev):
    """Packed int8 weights [g,kd,n] and fp32 channel scales [g,n]."""
    q = torch.empty((g, kd, n), dtype=torch.int8, device=dev)
    scale = torch.empty((g, n), dtype=torch.float32, device=dev)
    for i in range(g):
        w = torch.randn(kd, n, generator=gen, device=dev)
        top = torch.maximum(w.amax(dim=0), -w.amin(dim=0))
        scale[i] = top * (kd ** -0.5 / 127.0)
        q[i] = w.mul_(127.0 / top).round_().to(torch.int8)
    return cam.prepack_weight(q, gate_up), scale


def _fp8_weight(g, kd, n, gate_up, gen, dev):
    """Packed E4M3 weights [g,kd,n] and E8M0 block scales [g,kd/128,n/128]."""
    q = torch.empty((g, kd, n), dtype=torch.float8_e4m3fn, device=dev)
    for i in range(g):
        q[i] = torch.randn(kd, n, generator=gen, device=dev).mul_(64.0).to(torch.float8_e4m3fn)
    exp = 127 - 6 - round(math.log2(kd) / 2)
    scale = torch.randint(exp - 1, exp + 2, (g, kd // 128, n // 128), generator=gen, dtype=torch.uint8, device=dev)
    return cam.prepack_weight(q, gate_up), scale


def prepare(case, seed):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    kind, s = case["kind"], dict(case)
    h = case["hidden"]
    if kind in ("layer", "layer_fp8", "experts"):
        g, i = case["experts"], case["inter"]
        make = _fp8_weight if kind == "layer_fp8" else _int8_weight
        s["w1"], s["w1s"] = make(g, h, 2 * i, True, gen, dev)
        s["w2"], s["w2s"] = make(g, i, h, False, gen, dev)
    if kind == "experts":
        rows = case["rows"]
        sizes = synth.zipf_group_sizes(g, rows, int(seed), num_empty=min(3, g // 4))
        s["group_list"] = torch.cumsum(sizes, 0).to(dev)
        s["x"] = torch.randn(rows, h, generator=gen, device=dev).mul_(32.0).round_().clamp_(-127, 127).to(torch.int8)
        s["x_scale"] = torch.rand(rows, generator=gen, device=dev) * 0.02 + 0.02
        return s
    t, k, e = case["tokens"], case["top_k"], case["experts"]
    s["x"] = torch.randn(t, h, generator=gen, device=dev).to(_dtype(case))
    s["ids"], s["gates"] = _routing(case, gen, dev)
    if kind in ("layer", "layer_fp8"):
        s["mask"] = None
        if case["active"] < 1.0:
            s["mask"] = torch.arange(t, device=dev) < max(1, int(t * case["active"]))
    elif kind in ("exchange", "shmem"):
        # what the experts give back, in dispatch order
        y = torch.randn(t * k, h, generator=gen, device=dev).to(_dtype(case))
        if case.get("wire"):
            blocks = torch.randint(-127, 128, (t * k, h), generator=gen, dtype=torch.int8, device=dev)
            scales = (torch.rand((t * k, h // 8), generator=gen, device=dev) * 0.02 + 0.001).to(torch.bfloat16)
            y = torch.cat([blocks, scales.view(torch.int8)], dim=1).contiguous()
        s["y"] = y
        s["shared_x"] = None
        if case.get("shared"):
            rows = torch.randn(t, h, generator=gen, device=dev)
            s["shared_x"] = rows.to(torch.bfloat16 if case.get("wire") else _dtype(case))
        s["smooth_scales"] = None
        if case.get("smooth"):
            s["smooth_scales"] = torch.rand(e, h, generator=gen, device=dev) * 1.5 + 0.5
    return s


# ---------------------------------------------------------------------------------------------- one pass
def run(s):
    kind = s["kind"]
    if kind == "layer":
        return OPS.fused_deep_moe(s["x"], s["ids"], [s["w1"]], [s["w1s"]], [s["w2"]], [s["w2s"]], s["gates"], None,
                                  s["mask"], "", 1, 0, s["experts"], 1, 0, 0, 0)
    if kind == "layer_fp8":
        return cam.fused_deep_moe_fp8(s["x"], s["ids"], s["w1"], s["w1s"], s["w2"], s["w2s"], s["gates"], s["mask"])
    if kind == "exchange":
        d = cam.moe_dispatch_fused(s["x"], s["ids"], s["experts"], quant_mode=s["quant"])
        out = cam.moe_combine_gather(s["y"], None, d["slot_row"], s["gates"], shared_x=s["shared_x"])
        if s["quant"] == 0:
            del d["recv_x_scales"]  # not written
        return d, out
    if kind == "normal":
        per_rank, per_expert, in_rank = OPS.get_dispatch_layout(s["ids"], s["experts"], 1)
        rows, expand_idx, recv_count, received = OPS.moe_dispatch_prefill(
            s["x"], s["ids"], s["gates"], per_rank, in_rank, per_expert, 0, "", 0, 1)
        out = OPS.moe_combine_prefill(rows, s["ids"], s["gates"], expand_idx, recv_count, "", 0, 1)
        return per_rank, per_expert, in_rank, rows, expand_idx, recv_count, received, out
    if kind == "shmem":
        d = OPS.moe_dispatch_shmem(s["x"], s["ids"], s["smooth_scales"], None, 1, 0, s["experts"], 1, 0, 0, 1, 0,
                                   s["quant"], 0, 1, 0)
        out = OPS.moe_combine_shmem(s["y"], s["ids"], d[2], d[4], s["gates"], None, None, None, None, None, None, 1, 0,
                                    s["experts"], 1, 0, 0, 1, 0, 0, 0, 0, 0, 0)
        # the scales are written for quantised rows only, d[5] for two tensor-parallel ranks only
        return [d[0], d[1], d[2], d[3], d[4], out] if s["quant"] else [d[0], d[2], d[3], d[4], out]
    y, y_scale = cam.grouped_matmul_swiglu_quant(s["x"], s["x_scale"], s["w1"], s["w1s"], s["group_list"])
    return y, y_scale, cam.grouped_matmul_dequant(y, y_scale, s["w2"], s["w2s"], s["group_list"])


def work(case):
    """Bytes read and written once, and multiply-adds of the GEMMs.  An expert's weights count when a token reaches it:
    as many experts as uniform routing would reach."""
    kind, h = case["kind"], case["hidden"]
    if kind == "experts":
        rows, i, g = case["rows"], case["inter"], case["experts"]
        live = int((synth.zipf_group_sizes(g, rows, 0, num_empty=min(3, g // 4)) > 0).sum())
        return dict(bytes=live * (3 * h * i + 4 * (2 * i + h)) + rows * (h + 4 + i + 4 + 2 * h), flops=6 * rows * h * i)
    t, k, e = case["tokens"], case["top_k"], case["experts"]
    rows = t * k
    if kind in ("layer", "layer_fp8"):
        i = case["inter"]
        active = t if case["active"] >= 1.0 else max(1, int(t * case["active"]))
        live = e * (1.0 - (1.0 - k / e) ** active)
        scales = 3 * h * i // 16384 if kind == "layer_fp8" else 4 * (2 * i + h)
        return dict(bytes=live * (3 * h * i + scales) + active * 2 * h + t * (2 * h + 8 * k) + 8 * e,
                    flops=6 * active * k * h * i)
    if kind == "normal":
        out = rows * 2 * h
    else:
        out = {0: 2 * rows * h, 2: rows * (h + 4), 4: rows * (h + h // 128)}[case["quant"]]
    back = rows * (h + h // 4) if case.get("wire") else rows * 2 * h
    moved = t * 2 * h + out + back + t * 2 * h          # x, rows out, rows back, tokens
    moved += rows * (4 + 4 + 4 + 4)                     # ids, gate weights, place in the expert, row map
    if kind != "shmem":
        moved += rows * 12                              # (rank, token, k) triples
    if case.get("shared"):
        moved += t * 2 * h
    if case.get("smooth"):
        moved += min(e, rows) * 4 * h
    return dict(bytes=moved, flops=2 * rows * h)


def tolerance(case):
    # Layers: 16-bit results behind one re-quantisation to 8 bits, where a sum in another order can round the other way.
    if case["kind"] in ("layer", "layer_fp8"):
        return {"rel": 1e-2}
    # int8 products of a SiLU that another exponential may round differently; bf16 rows behind them.
    if case["kind"] == "experts":
        return {"rel": 1e-2, "differ": 1e-3}
    # One 16-bit rounding of an fp32 sum; whole numbers are the same.
    return {"rel": 4e-3, "max": 0.02}
