"""The work this library is used for, as timed cases: what an inference engine has a quantized Mixture-of-Experts layer do.

Every case goes through the public operator objects of flyingfish_amd.ops with weights, scratch and output buffers that a
program keeps from call to call, and takes a batch of token rows from activations to the layer's output (or one linear
from activations to its output). Weights are N(0, 0.02) under the library's own absmax quantizers, the router gate is
N(0, 0.02) in BF16, activations are N(0, 1) in BF16.

Kinds of work:
  layer    a decode step of a noaux_tc layer with a shared expert: FP32 logits, top-k, experts, combine (NativeMoe)
  softmax  a decode step of a small softmax-routed layer without a shared expert
  prefill  a prompt chunk: FP32 logits, top-k, token-sorted grouped GEMMs, combine; expert popularity is Zipf-like (s = 1.1)
  e8m0     a decode step of the E2M1/E8M0 contract in exact arithmetic
  form     a decode step in the summation orders of the CPU expert path (layers that split experts between CPU and GPU)
  linear   a standalone projection
"""
import math

import torch

from flyingfish_amd import capi, synth
from flyingfish_amd.ops import (CombineOps, DecodeOps, E8m0DecodeOps, ExpertTable, Fp8Ops, NativeMoe, NvFp4Ops, PrefillOps,
                                RouteOps)

_FORMATS = {"fp8": capi.FMT_FP8_BLOCK128, "nvfp4": capi.FMT_NVFP4, "bf16": capi.FMT_BF16, "fp8_channel": capi.FMT_FP8_CHANNEL,
            "e2m1": capi.FMT_E2M1_E8M0, "e4m3": capi.FMT_E4M3_E8M0_32}
_SHARED = {"fp8": "fp8", "nvfp4": "bf16", "bf16": "bf16", "fp8_channel": "fp8_channel", "e2m1": "e4m3"}
_ZIPF = 1.1


def _layer(name, kind, fmt, rows, shape, **more):
    hidden, inter, experts, top_k, groups, keep = shape
    case = {"kind": kind, "format": fmt, "rows": rows, "hidden": hidden, "inter": inter, "experts": experts, "top_k": top_k,
            "n_group": groups, "topk_group": keep, **more}
    return {"name": name, **case} if name else case


def _linear(name, fmt, act, m, k, n):
    case = {"kind": "linear", "format": fmt, "act": act, "m": m, "k": k, "n": n}
    return {"name": name, **case} if name else case


_DSV3 = (7168, 2048, 256, 8, 8, 4)       # hidden, intermediate, experts, top-k, groups, groups kept
_DSV3_FLAT = (7168, 2048, 256, 8, 1, 1)  # the same layer routed without groups
_MEDIUM = (4096, 1536, 64, 6, 1, 1)
_SMALL = (2048, 1408, 64, 4, 1, 1)


def listed():
    return [
        # one user, small model: a layer call is a few launches on weights that mostly stay in the caches
        _layer("softmax_small_1", "softmax", "fp8", 1, _SMALL),
        # one user, large model: every token streams nine experts from HBM
        _layer("fp8_1", "layer", "fp8", 1, _DSV3),
        # a few users at once
        _layer("fp8_8", "layer", "fp8", 8, _DSV3),
        # a busy decode server: most experts are touched, several rows each
        _layer("fp8_64", "layer", "fp8", 64, _DSV3),
        # the same layer with 4-bit routed experts and a BF16 shared expert
        _layer("nvfp4_32", "layer", "nvfp4", 32, _DSV3),
        # a full prompt chunk on the FP8 matrix cores (W8A8)
        _layer("prefill_fp8_4096", "prefill", "fp8", 4096, _DSV3_FLAT),
        # a shorter, ragged prompt with 4-bit experts (W4A16)
        _layer("prefill_nvfp4_1021", "prefill", "nvfp4", 1021, _DSV3_FLAT),
        # a ragged prompt in the E2M1/E8M0 contract (W4A8, MX matrix cores)
        _layer("prefill_e8m0_1500", "prefill", "e2m1", 1500, _DSV3_FLAT),
        # one user, E2M1/E8M0 experts in exact arithmetic
        _layer("e8m0_1", "e8m0", "e2m1", 1, _DSV3_FLAT),
        # a few users on per-channel FP8 experts, bit-equal to the experts that stay on the CPU
        _layer("form_fp8_channel_4", "form", "fp8_channel", 4, _MEDIUM, form=16),
        # an attention projection at a decode batch of 16 (W8A16) and over a prompt chunk (W8A8)
        _linear("linear_fp8_16", "fp8", "bf16", 16, 7168, 2048),
        _linear("linear_w8a8_2048", "fp8", "fp8", 2048, 2048, 7168),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["softmax", "layer", "layer", "layer", "prefill", "prefill", "e8m0", "form", "linear", "linear"])
    if kind == "linear":
        fmt, act = rng.choice([("fp8", "bf16"), ("fp8", "fp8"), ("nvfp4", "bf16")])
        m = _log_int(rng, 1, 2048) if act == "fp8" else _log_int(rng, 1, 64)
        return _linear(None, fmt, act, m, 128 * rng.randint(12, 56), 128 * rng.randint(12, 56))
    if kind == "softmax":
        return _layer(None, kind, "fp8", _log_int(rng, 1, 16), (128 * rng.randint(8, 24), 128 * rng.randint(5, 16), 64, rng.randint(2, 8), 1, 1))
    hidden, inter = 256 * rng.randint(8, 28), 128 * rng.randint(6, 16)
    experts = rng.choice([64, 128, 256])
    top_k = rng.randint(4, 8)
    groups, keep = rng.choice([(1, 1), (8, 4)])
    if kind == "layer":
        return _layer(None, kind, rng.choice(["fp8", "nvfp4"]), _log_int(rng, 1, 64), (hidden, inter, experts, top_k, groups, keep))
    if kind == "prefill":
        fmt = rng.choice(["fp8", "fp8", "nvfp4", "e2m1"])
        rows = _log_int(rng, 65, {"fp8": 4096, "nvfp4": 1500, "e2m1": 3000}[fmt])
        return _layer(None, kind, fmt, rows, (hidden, inter, experts, top_k, 1, 1))
    if kind == "e8m0":
        return _layer(None, kind, "e2m1", _log_int(rng, 1, 16), (hidden, inter, 64, top_k, 1, 1))
    return _layer(None, kind, rng.choice(["fp8_channel", "bf16"]), _log_int(rng, 1, 32), (hidden, inter, 64, top_k, 1, 1), form=rng.choice([16, 8]))


# ---- inputs ------------------------------------------------------------------------------------------------------------

def _fill_expert(table, e, seed):
    """Seeded N(0, 0.02) weights of one expert, quantized into its slot."""
    hidden, inter, fmt = table.hidden, table.inter, table.format
    v = table.expert_views(e)
    for i, shape in enumerate([(inter, hidden), (inter, hidden), (hidden, inter)]):
        w = synth.normal(shape, 0.02, seed + i, device="cuda")
        if fmt == capi.FMT_BF16:
            v[2 * i].copy_(w)
            continue
        if fmt == capi.FMT_NVFP4:
            codes, scales, g = synth.quant_nvfp4(w)
            table.global_scales[e, i] = g
        else:
            codes, scales = {capi.FMT_FP8_BLOCK128: synth.quant_fp8_block, capi.FMT_FP8_CHANNEL: synth.quant_fp8_channel,
                             capi.FMT_E2M1_E8M0: synth.quant_e2m1_e8m0, capi.FMT_E4M3_E8M0_32: synth.quant_e4m3_e8m0_block32}[fmt](w)
        v[2 * i].copy_(codes)
        v[2 * i + 1].copy_(scales)


def _experts(case, seed):
    """(table of the routed experts, table that holds the shared expert, its descriptor)."""
    fmt, shared_fmt = case["format"], _SHARED[case["format"]]
    n = case["experts"]
    table = ExpertTable.allocate(_FORMATS[fmt], n, case["hidden"], case["inter"])
    for e in range(n):
        _fill_expert(table, e, seed * 1000003 + 3 * e)
    if case["kind"] == "softmax":
        return table, None, None
    shared_table = ExpertTable.allocate(_FORMATS[shared_fmt], 1, case["hidden"], case["inter"])
    _fill_expert(shared_table, 0, seed * 1000003 + 3 * n)
    return table, shared_table, shared_table.shared_struct(0)


def _router_and_tokens(case, seed):
    """Router gate and token rows. A prompt chunk's popularity is skewed: the tokens share a common component and the
    gate rows carry the experts' log-popularity along it, so logit = log popularity + noise."""
    rows, hidden, experts = case["rows"], case["hidden"], case["experts"]
    router = synth.normal((experts, hidden), 0.02, seed * 1000003 + 900001, device="cuda")
    x = synth.normal((rows, hidden), 1.0, seed * 1000003 + 900002, device="cuda")
    if case["kind"] == "prefill":
        common = 0.1 * torch.sign(synth.normal((hidden,), 1.0, seed * 1000003 + 900003, device="cuda"))
        pop = synth.zipf_popularity(experts, _ZIPF, seed * 1000003 + 900004).cuda()
        router += pop[:, None] * common[None, :] / (0.01 * hidden)
        x += common[None, :]
    return router.to(torch.bfloat16), x.to(torch.bfloat16)


def prepare(case, seed):
    if case["kind"] == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        w = synth.normal((n, k), 0.02, seed * 1000003 + 1, device="cuda")
        s = {"case": case, "x": synth.normal((m, k), 1.0, seed * 1000003 + 2, device="cuda", dtype=torch.bfloat16),
             "y": torch.empty((m, n), dtype=torch.bfloat16, device="cuda")}
        if case["format"] == "nvfp4":
            s["codes"], s["scales"], g = synth.quant_nvfp4(w)
            s["global"] = torch.tensor([g], dtype=torch.float32, device="cuda")
        else:
            s["codes"], s["scales"] = synth.quant_fp8_block(w)
        return s
    rows, top_k, hidden = case["rows"], case["top_k"], case["hidden"]
    table, shared_table, shared = _experts(case, seed)
    router, x = _router_and_tokens(case, seed)
    s = {"case": case, "table": table, "shared_table": shared_table, "router": router, "x": x}
    if case["kind"] == "layer":
        s["bias"] = torch.zeros(case["experts"], dtype=torch.float32, device="cuda")
        s["layer"] = NativeMoe(table, shared, router, s["bias"], rows, top_k, routed_scaling=2.5, n_group=case["n_group"],
                               topk_group=case["topk_group"], swiglu=capi.SWIGLU_TWICE,
                               routed_weight=capi.WEIGHT_AFTER_DOWN_BF16, combine_mode=capi.COMBINE_UNGATED)
        return s
    softmax = case["kind"] == "softmax"
    s["ids"] = torch.empty((rows, top_k), dtype=torch.int32, device="cuda")
    s["weights"] = torch.empty((rows, top_k), dtype=torch.bfloat16 if softmax else torch.float32, device="cuda")
    s["logits"] = torch.empty((rows, case["experts"]), dtype=torch.bfloat16 if softmax else torch.float32, device="cuda")
    s["y"] = torch.empty((rows, hidden), dtype=torch.bfloat16, device="cuda")
    s["status"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    if softmax:
        s["decode"] = DecodeOps(table, None, rows, top_k, capi.ACT_BF16, capi.SWIGLU_TWICE, 0.0, capi.WEIGHT_AFTER_DOWN_BF16, False)
        return s
    s["bias"] = torch.zeros(case["experts"], dtype=torch.float32, device="cuda")
    if case["kind"] == "prefill":
        if case["format"] == "e2m1":
            s["prefill"] = PrefillOps(table, rows, top_k, swiglu=capi.SWIGLU_CLAMPED_ONCE, swiglu_limit=7.0, shared=shared,
                                      routed_weight=capi.WEIGHT_BEFORE_DOWN_F32, act_mode=capi.ACT_E4M3_E8M0_32)
        else:
            s["prefill"] = PrefillOps(table, rows, top_k, shared=shared,
                                      act_mode=capi.ACT_FP8_BLOCK128 if case["format"] == "fp8" else capi.ACT_BF16)
    elif case["kind"] == "e8m0":
        s["decode"] = E8m0DecodeOps(table, shared, rows, top_k, 7.0)
    else:
        s["decode"] = DecodeOps(table, shared, rows, top_k, weights_f32=True)
    return s


# ---- one pass ----------------------------------------------------------------------------------------------------------

def _softmax_step(s):
    case, dec, x = s["case"], s["decode"], s["x"]
    ids, weights, _ = RouteOps.route(x, s["router"], case["top_k"], capi.SCORE_SOFTMAX, logits=s["logits"], ids=s["ids"], weights=s["weights"])
    if case["rows"] == 1:
        dec.contribute(x, ids, weights, stage=0)
        if dec.finish(x, ids, weights, capi.COMBINE_ROUTED, s["y"], status=s["status"]):
            return s["y"]
        contributions, _ = dec.contribute(x, ids, weights, stage=1)
        return CombineOps.combine(contributions, None, ids, capi.COMBINE_ROUTED, status=s["status"], out=s["y"])
    dec.done.zero_()
    contributions, _ = dec.contribute(x, ids, weights)
    return CombineOps.combine(contributions, None, ids, capi.COMBINE_ROUTED, done=dec.done, status=s["status"], out=s["y"])


def run(state):
    s, case = state, state["case"]
    if case["kind"] == "linear":
        if case["format"] == "nvfp4":
            return NvFp4Ops.gemm(s["codes"], s["scales"], s["global"], s["x"], out=s["y"])
        return Fp8Ops.linear(s["codes"], s["scales"], s["x"], capi.ACT_FP8_BLOCK128 if case["act"] == "fp8" else capi.ACT_BF16, out=s["y"])
    if case["kind"] == "layer":
        y = s["layer"].run(s["x"])
        return {"y": y, "ids": s["layer"].ids, "weights": s["layer"].weights}
    if case["kind"] == "softmax":
        return {"y": _softmax_step(s), "ids": s["ids"], "weights": s["weights"]}
    x = s["x"]
    op = s["prefill"] if case["kind"] == "prefill" else s["decode"]
    score = capi.NOAUX_SQRTSOFTPLUS if case["format"] == "e2m1" else capi.NOAUX_SIGMOID
    ids, weights = RouteOps.route_noaux(x, s["router"], s["bias"], case["top_k"], s["logits"], s["ids"], s["weights"], done=op.done,
                                        score_mode=score, routed_scaling=2.5)
    if case["kind"] == "prefill":
        contributions, shared_out = op.contribute(x, ids, weights), op.shared_out
    elif case["kind"] == "e8m0":
        contributions, shared_out = op.contribute(x, ids, weights)
    else:
        contributions, shared_out = op.contribute(x, ids, weights, form=capi.FORM_LANE16 if case["form"] == 16 else capi.FORM_LANE8)
    y = CombineOps.combine(contributions, shared_out, ids, capi.COMBINE_UNGATED, done=op.done, status=s["status"], out=s["y"])
    out = {"y": y, "ids": ids, "weights": weights}
    if case["kind"] == "form":  # an engine that adds experts of its own takes the contributions
        out["contributions"], out["shared"] = contributions, shared_out
    return out


# ---- what a pass cannot do without -------------------------------------------------------------------------------------

def _weight_bytes(fmt, hidden, inter):
    return 3 * hidden * inter * {"fp8": 1 + 4 / 128 ** 2, "nvfp4": 0.5 + 1 / 16, "bf16": 2, "fp8_channel": 1,
                                 "e2m1": 0.5 + 1 / 32, "e4m3": 1 + 1 / 32 ** 2}[fmt]


def _experts_touched(case):
    """Expected number of distinct experts among rows x top_k choices."""
    n, k, rows = case["experts"], case["top_k"], case["rows"]
    if case["kind"] == "prefill":
        pop = [(r + 1.0) ** -_ZIPF for r in range(n)]
        share = [p / sum(pop) for p in pop]
    else:
        share = [1.0 / n] * n
    return sum(1.0 - (1.0 - p) ** (rows * k) for p in share) if case["kind"] == "prefill" else n * (1.0 - (1.0 - k / n) ** rows)


def work(case):
    if case["kind"] == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": n * k * (1 + 4 / 128 ** 2 if case["format"] == "fp8" else 0.5 + 1 / 16) + 2.0 * m * (k + n), "flops": 2.0 * m * k * n}
    rows, hidden, inter, k, n = case["rows"], case["hidden"], case["inter"], case["top_k"], case["experts"]
    shared = 0 if case["kind"] == "softmax" else 1
    nbytes = _experts_touched(case) * _weight_bytes(case["format"], hidden, inter)
    if shared:
        nbytes += _weight_bytes(_SHARED[case["format"]], hidden, inter)
    nbytes += n * hidden * 2 + rows * hidden * 2 * 2 + rows * k * 8
    if case["kind"] == "form":
        nbytes += rows * (k + 1) * hidden * 2
    return {"bytes": nbytes, "flops": rows * (6.0 * hidden * inter * (k + shared) + 2.0 * hidden * n)}


def tolerance(case):
    """Four times what another order of the sums changes: a batch against its rows one at a time for decode, an FP64
    restatement with the same roundings for the linears and prompt chunks, the exact entry for E2M1/E8M0 chunks. Where the
    activations are quantized again between the stages one flipped BF16 step moves a whole 128-group. ids are whole
    numbers and their summation order is pinned: none may differ."""
    kind, fmt = case["kind"], case["format"]
    if kind in ("e8m0", "form"):  # exact integer dots, pinned summation orders: the bits are the contract
        return "exact"
    if kind == "linear":
        return {"rel": 1e-3, "max": 0.03} if case["act"] == "fp8" else {"rel": 1e-4, "max": 0.03}
    if kind == "prefill":
        return {"fp8": {"rel": 1e-2, "max": 0.12}, "nvfp4": {"rel": 1.6e-3, "max": 0.06}, "e2m1": {"rel": 8e-3, "max": 0.16}}[fmt]
    return {"rel": 1e-3, "max": 0.03} if kind == "softmax" else {"rel": 2.5e-3, "max": 0.06}
