"""Performance cases of the library: the calls a program that serves or tests MXFP4 / MXFP8 models makes, over the
range of sizes it makes them at.

Four kinds of call:

* ``gemm``   - the drop-in call, ``mxfp4_gemm`` on operands that are already quantised, scales in one of the three
               layouts, B row-major or preshuffled, bf16 or f32 result.
* ``linear`` - one linear layer of a served model: bf16 activations are quantised (scales straight into the MFMA32
               order) and multiplied with resident weights whose scales were converted once.
* ``moe``    - one mixture-of-experts MLP: routing table -> alignment by expert -> gathered quantiser -> gate/up GEMM
               with the gated activation -> down GEMM, the result per (token, expert) pair, rows sorted by expert.
* ``mxfp8``  - ``mxfp8_gemm``: 8-bit activations against 8-bit or packed 4-bit weights.

``gemm`` operands are uniform nibbles with scales of a few binades, as in the repository's benchmark configurations;
the weights of the other kinds are normal variates put through the library's quantiser, as a converted checkpoint's are.
"""

import math

import torch

import wave_amd
from wave_amd import _lib as L

_OUT = {"bf16": torch.bfloat16, "f32": torch.float32}
_SCALES = {"row": L.SCALE_ROW_MAJOR, "e8m0": L.SCALE_E8M0_SHUFFLE, "mfma32": L.SCALE_MFMA32}
_FP8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}


def listed():
    return [
        # The size of most of the library's examples and tests, all layouts row-major: launch-bound.
        {"name": "gemm_1024_f32", "kind": "gemm", "m": 1024, "n": 1024, "k": 1024, "out": "f32", "scales": "row", "b": "row"},
        # One token through an attention projection: the smallest call of a decode loop.
        {"name": "linear_m1", "kind": "linear", "m": 1, "n": 8192, "k": 4096, "out": "bf16", "b": "row"},
        # A decode batch against a wide MLP projection, scales as a drop-in caller hands them over.
        {"name": "gemm_m16_decode", "kind": "gemm", "m": 16, "n": 28672, "k": 8192, "out": "bf16", "scales": "row", "b": "row"},
        # A large decode batch (or a speculative one) through the same projection, weights prepared once.
        {"name": "linear_m128", "kind": "linear", "m": 128, "n": 28672, "k": 8192, "out": "bf16", "b": "row"},
        # A short prefill in the reference's preshuffled-scales-and-B format.
        {"name": "gemm_m256_preshuffled", "kind": "gemm", "m": 256, "n": 28672, "k": 8192, "out": "bf16", "scales": "e8m0",
         "b": "preshuffle"},
        # A ragged prefill chunk through a projection of middle width.
        {"name": "linear_m1000", "kind": "linear", "m": 1000, "n": 7168, "k": 4096, "out": "bf16", "b": "row"},
        # A prefill chunk through a down projection: narrow output, long K.
        {"name": "linear_m2048_down", "kind": "linear", "m": 2048, "n": 4096, "k": 14336, "out": "bf16", "b": "row"},
        # No dimension but K in whole tiles, f32 result, scales in e8m0_shuffle order over a wide range.
        {"name": "gemm_ragged_f32", "kind": "gemm", "m": 4093, "n": 6144, "k": 7168, "out": "f32", "scales": "e8m0", "b": "row"},
        # The headline size: a long prefill, compute-bound.
        {"name": "gemm_8192", "kind": "gemm", "m": 8192, "n": 8192, "k": 8192, "out": "bf16", "scales": "row", "b": "row"},
        # An expert MLP at a serving batch: bound by reading every expert's weights.
        {"name": "moe_64_tokens", "kind": "moe", "tokens": 64, "topk": 2, "experts": 8, "hidden": 4096, "inter": 14336},
        # The same layer at a prefill batch: the largest case.
        {"name": "moe_4096_tokens", "kind": "moe", "tokens": 4096, "topk": 2, "experts": 8, "hidden": 4096, "inter": 14336},
        # 8-bit operands at a prefill batch.
        {"name": "mxfp8_4096", "kind": "mxfp8", "m": 4096, "n": 8192, "k": 8192, "out": "bf16", "a_fmt": "e4m3", "b_fmt": "e4m3"},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "linear", "linear", "linear", "moe", "mxfp8"])
    if kind == "moe":
        # (32 experts, hidden = intermediate = 2880: the sizes of the expert-batch tests whose K is not in whole tiles)
        experts, topk, hidden, inter = rng.choice([(8, 2, 4096, 14336), (16, 2, 4096, 4096), (32, 4, 2880, 2880)])
        return {"kind": kind, "tokens": round(_log(rng, 16, 4096)), "topk": topk, "experts": experts, "hidden": hidden,
                "inter": inter}
    while True:
        m = round(_log(rng, 32 if kind == "mxfp8" else 1, 8192))
        n = 32 * round(_log(rng, 1024, 28672) / 32)
        if rng.random() < 0.5:
            n = max(1024, 256 * round(n / 256))
        k = 256 * round(_log(rng, 1024, 16384) / 256)
        if 2.0 * m * n * k <= (0.5e12 if kind == "mxfp8" else 1.1e12):
            break
    case = {"kind": kind, "m": m, "n": n, "k": k, "out": rng.choice(["bf16", "bf16", "bf16", "f32"])}
    if kind == "mxfp8":
        case["a_fmt"] = rng.choice(["e4m3", "e5m2"])
        case["b_fmt"] = rng.choice(["e4m3", "e5m2", "e2m1"])
        return case
    case["b"] = rng.choice(["row", "row", "preshuffle"])
    if kind == "gemm":
        case["scales"] = rng.choice(["row", "row", "e8m0", "mfma32"])
    if case["b"] == "row" and rng.random() < 0.2:
        case["k"] = k - 32 * rng.randint(1, 7)  # a partial last K tile
    return case


def _normal_weight(rows, k, gen):
    return torch.randn(rows, k, device="cuda", generator=gen, dtype=torch.bfloat16) * k ** -0.5


def _scales(lo, hi, rows, k, layout, gen):
    s = torch.randint(lo, hi + 1, (rows, k // 32), dtype=torch.uint8, device="cuda", generator=gen)
    return s if layout == L.SCALE_ROW_MAJOR else wave_amd.scale_convert(s, rows, k // 32, L.SCALE_ROW_MAJOR, layout)


def _fp8_operand(rows, k, fmt, gen):
    """Normal variates as 8-bit floats (or packed e2m1) with one e8m0 scale per 32 elements, row-major."""
    x = torch.randn(rows, k, device="cuda", generator=gen, dtype=torch.bfloat16)
    if fmt == "e2m1":
        return wave_amd.quantize_mxfp4(x)
    # the OCP MX rule: the scale is the group's largest power of two less the format's largest exponent
    emax = 8 if fmt == "e4m3" else 15
    top = 448.0 if fmt == "e4m3" else 57344.0
    g = x.view(rows, k // 32, 32)
    e = torch.floor(torch.log2(g.abs().amax(dim=2).float().clamp_min(2.0 ** -100))) - emax
    q = (g.float() * torch.exp2(-e).unsqueeze(2)).clamp_(-top, top).to(_FP8[fmt])
    return q.view(rows, k), (e + 127).to(torch.uint8)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    state = {"kind": kind}
    if kind == "moe":
        tokens, topk, experts = case["tokens"], case["topk"], case["experts"]
        hidden, inter = case["hidden"], case["inter"]
        rows = tokens * topk
        state.update(topk=topk, experts=experts, inter=inter, rows=rows)
        state["x"] = torch.randn(tokens, hidden, device="cuda", generator=gen, dtype=torch.bfloat16)
        logits = torch.rand(tokens, experts, device="cuda", generator=gen)
        state["topk_ids"] = logits.topk(topk, dim=1).indices.to(torch.int32)
        i32 = {"dtype": torch.int32, "device": "cuda"}
        state["sorted_ids"] = torch.empty(rows, **i32)
        state["expert_ids"] = torch.empty(rows, **i32)
        state["total"] = torch.empty(1, **i32)
        state["offsets"] = torch.empty(experts + 1, **i32)

        def resident(pairs):
            w = torch.stack([p[0] for p in pairs])
            s = torch.stack([p[1] for p in pairs])
            e, n, ks = s.shape
            native = [wave_amd.scale_convert(s[i], n, ks, L.SCALE_ROW_MAJOR, L.SCALE_MFMA32) for i in range(e)]
            return w, torch.stack(native)

        w1 = [wave_amd.quantize_mxfp4(_normal_weight(2 * inter, hidden, gen)) for _ in range(experts)]
        # The fused first GEMM takes gate and up rows interleaved; a hidden size it does not serve runs the two calls.
        state["fused"] = hidden % 256 == 0 and inter % 128 == 0
        state["w1"], state["w1s"] = resident(w1)
        if state["fused"]:
            state["w1_il"], state["w1s_il"] = resident([tuple(wave_amd.interleave_gate_up(t) for t in p) for p in w1])
        del w1
        state["w2"], state["w2s"] = resident([wave_amd.quantize_mxfp4(_normal_weight(hidden, inter, gen)) for _ in range(experts)])
        state["h"] = torch.empty(rows, 2 * inter, device="cuda", dtype=torch.bfloat16)
        state["out"] = torch.empty(rows, hidden, device="cuda", dtype=torch.bfloat16)
        return state

    m, n, k = case["m"], case["n"], case["k"]
    state["out"] = torch.empty(m, n, device="cuda", dtype=_OUT[case["out"]])
    if kind == "mxfp8":
        state["x"], state["xs"] = _fp8_operand(m, k, case["a_fmt"], gen)
        state["w"], state["ws"] = _fp8_operand(n, k, case["b_fmt"], gen)
        state["fmt"] = (None, L.MXFP8_E2M1) if case["b_fmt"] == "e2m1" else None
        return state
    b_layout = L.B_PRESHUFFLE if case["b"] == "preshuffle" else L.B_ROW_MAJOR
    if kind == "linear":
        state["x"] = torch.randn(m, k, device="cuda", generator=gen, dtype=torch.bfloat16)
        w, ws = wave_amd.quantize_mxfp4(_normal_weight(n, k, gen), scale_layout=L.SCALE_MFMA32)
        state["opts"] = {"a_scale_layout": L.SCALE_MFMA32, "b_scale_layout": L.SCALE_MFMA32, "b_layout": b_layout}
    else:
        layout = _SCALES[case["scales"]]
        lo, hi = (100, 154) if case["scales"] == "e8m0" else (124, 130)
        state["x"] = torch.randint(0, 256, (m, k // 2), dtype=torch.uint8, device="cuda", generator=gen)
        state["xs"] = _scales(lo, hi, m, k, layout, gen)
        w = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device="cuda", generator=gen)
        ws = _scales(lo, hi, n, k, layout, gen)
        state["opts"] = {"a_scale_layout": layout, "b_scale_layout": layout, "b_layout": b_layout}
    state["w"] = wave_amd.b_preshuffle(w) if b_layout == L.B_PRESHUFFLE else w
    state["ws"] = ws
    return state


def run(state):
    kind, out = state["kind"], state["out"]
    if kind == "gemm":
        wave_amd.mxfp4_gemm(state["x"], state["xs"], state["w"], state["ws"], out, **state["opts"])
        return out
    if kind == "linear":
        xq, xs = wave_amd.quantize_mxfp4(state["x"], scale_layout=L.SCALE_MFMA32)
        wave_amd.mxfp4_gemm(xq, xs, state["w"], state["ws"], out, **state["opts"])
        return out
    if kind == "mxfp8":
        wave_amd.mxfp8_gemm(state["x"], state["xs"], state["w"], state["ws"], out, elem_format=state["fmt"])
        return out
    native = {"a_scale_layout": L.SCALE_MFMA32, "b_scale_layout": L.SCALE_MFMA32}
    offsets, inter = state["offsets"], state["inter"]
    wave_amd.moe_align_block_size(state["topk_ids"], state["experts"], 1, state["sorted_ids"], state["expert_ids"],
                                  state["total"], offsets)
    xq, xs = wave_amd.quantize_mxfp4_rows(state["x"], state["sorted_ids"], state["topk"], scale_layout=L.SCALE_MFMA32)
    act = None
    if state["fused"]:
        try:
            act = wave_amd.mxfp4_gemm_gated_quantize(xq, xs, state["w1_il"], state["w1s_il"], offsets, **native)
        except ValueError:  # a batch between the fused kernels' ranges
            pass
    if act is None:
        h = state["h"]
        wave_amd.mxfp4_gemm_grouped(xq, xs, state["w1"], state["w1s"], offsets, h, **native)
        act = wave_amd.silu_and_mul_quantize(h[:, :inter], h[:, inter:], scale_layout=L.SCALE_MFMA32)
    wave_amd.mxfp4_gemm_grouped(act[0], act[1], state["w2"], state["w2s"], offsets, out, **native)
    return out, offsets, state["sorted_ids"]


def work(case):
    def mx4(rows, k):
        return rows * (k // 2 + k // 32)

    if case["kind"] == "moe":
        tokens, topk, experts = case["tokens"], case["topk"], case["experts"]
        hidden, inter = case["hidden"], case["inter"]
        rows = tokens * topk
        touched = experts * (1.0 - (1.0 - topk / experts) ** tokens)  # experts a random batch reaches
        return {"bytes": int(touched * (mx4(2 * inter, hidden) + mx4(hidden, inter))) + tokens * hidden * 2 + rows * (4 + hidden * 2),
                "flops": 2.0 * rows * hidden * inter * 3}
    m, n, k = case["m"], case["n"], case["k"]
    out = m * n * (2 if case["out"] == "bf16" else 4)
    if case["kind"] == "mxfp8":
        b = mx4(n, k) if case["b_fmt"] == "e2m1" else n * (k + k // 32)
        return {"bytes": m * (k + k // 32) + b + out, "flops": 2.0 * m * n * k}
    a = m * k * 2 if case["kind"] == "linear" else mx4(m, k)
    return {"bytes": a + mx4(n, k) + out, "flops": 2.0 * m * n * k}


def tolerance(case):
    # About four times what the path was seen to differ by from its own operands multiplied in float64 (relative, and
    # the largest difference): one rounding of a bf16 result 1.7e-3 / 3.9e-3, also at the end of the expert MLP; the
    # order of the f32 sums 7e-8 / 1.6e-6; with 8-bit operands the matrix core's own alignment of the products of one
    # instruction 1.4e-5 / 8e-5.
    if case["kind"] == "moe" or case["out"] == "bf16":
        return {"rel": 7e-3, "max": 2e-2}
    if case["kind"] == "mxfp8":
        return {"rel": 6e-5, "max": 4e-4}
    return {"rel": 4e-7, "max": 1e-5}
