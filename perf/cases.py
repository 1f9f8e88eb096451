"""What the blockwise-FP8 path is timed on: twelve calls of a serving program.

Each case is one layer, or one block, of a DeepSeek-style FP8 model as a
program on this library runs it: the routing, the linear layers at decode and
prefill sizes, the expert layers in both layouts, the producers fused with the
quantizer, and the codec in both directions.  ``listed()`` holds the sizes the
repository's own benchmark and tests use; ``draw()`` spreads over the ranges
they stand for (any row count, ragged widths, every dtype the calls take).
"""
from __future__ import annotations

import math

import torch

import inferop_amd as ia

DEV = "cuda"
TORCH_DT = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
DT_BYTES = {"fp32": 4, "fp16": 2, "bf16": 2}
DT_CODE = {"fp32": ia.dtype.fp32, "fp16": ia.dtype.fp16, "bf16": ia.dtype.bf16}


def listed():
    return [
        # MoE router of one decode batch: the smallest call a step makes.
        {"name": "route_decode", "kind": "topk", "tokens": 64, "experts": 256, "topk": 8},
        # One linear layer of a single sequence's decode step, the quantizer
        # and the GEMM in one call.
        {"name": "linear_decode_m1", "kind": "fused_linear", "m": 1, "n": 2112, "k": 7168,
         "dt": "bf16", "out": "bf16"},
        # The same layer kind for a small batch through the two tensor-level
        # calls (quantize, gemm).
        {"name": "linear_decode_m16", "kind": "linear", "m": 16, "n": 7168, "k": 2048,
         "dt": "bf16", "out": "bf16"},
        # The GEMM alone at a full decode batch (the activations come quantized
        # from a fused producer).
        {"name": "gemm_decode_m64", "kind": "gemm", "m": 64, "n": 4096, "k": 7168, "out": "bf16"},
        # A ragged batch over a ragged width, fp16 model.
        {"name": "gemm_ragged_m77", "kind": "gemm", "m": 77, "n": 4672, "k": 7168, "out": "fp16"},
        # A chunk of prefill through a short-K layer.
        {"name": "linear_chunk_m512", "kind": "linear", "m": 512, "n": 7168, "k": 2048,
         "dt": "bf16", "out": "bf16"},
        # Prefill of a 4096-token prompt, the long-K down projection: the
        # largest call of a step.
        {"name": "gemm_prefill_m4096", "kind": "gemm", "m": 4096, "n": 7168, "k": 16384,
         "out": "bf16"},
        # Expert layer of a decode step: fixed rows per expert, counts on the
        # device (the layout a captured step uses).
        {"name": "moe_decode_masked", "kind": "moe_masked", "experts": 32, "max_m": 16, "rows": 64,
         "n": 4096, "k": 7168, "out": "bf16"},
        # Expert layer of a prefill: rows sorted by expert.
        {"name": "moe_prefill", "kind": "moe", "experts": 32, "rows": 4096, "n": 4096, "k": 7168,
         "out": "bf16"},
        # Activation of the MLP at prefill, fused with the quantizer.
        {"name": "silu_quant_prefill", "kind": "silu", "rows": 4096, "cols": 18432, "dt": "bf16"},
        # Residual add, RMSNorm and quantizer before a block at prefill.
        {"name": "norm_quant_prefill", "kind": "norm", "rows": 4096, "cols": 7168, "dt": "bf16"},
        # Encode and decode of a prompt's activations (quantize, dequantize).
        {"name": "codec_prefill", "kind": "codec", "rows": 4096, "cols": 7168, "dt": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _k(rng, lo, hi):
    """A K (or row width): whole 128-wide scale groups, even and odd counts."""
    return 128 * _log(rng, lo // 128, hi // 128)


def draw(rng):
    kind = rng.choice(["topk", "fused_linear", "linear", "gemm", "gemm", "moe_masked", "moe",
                       "silu", "norm", "codec"])
    dt = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    out = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if kind == "topk":
        e = rng.choice([8, 64, 128, 160, 256, 384])
        return {"kind": kind, "tokens": _log(rng, 1, 4096), "experts": e,
                "topk": min(e, rng.choice([1, 2, 4, 6, 8]))}
    if kind == "fused_linear":
        return {"kind": kind, "m": rng.randint(1, 32), "n": _log(rng, 512, 16384),
                "k": _k(rng, 512, 8192), "dt": dt, "out": out}
    if kind in ("linear", "gemm"):
        # the whole range of a serving program, kept below the largest listed
        # product
        while True:
            m, n, k = _log(rng, 1, 4096), _log(rng, 512, 36864), _k(rng, 512, 18432)
            if m * n * k <= 4096 * 7168 * 16384 and n * k <= 7168 * 18432 and m * n <= 4096 * 18432:
                break
        case = {"kind": kind, "m": m, "n": n, "k": k, "out": out}
        if kind == "linear":
            case["dt"] = dt
        return case
    if kind in ("moe_masked", "moe"):
        e = rng.choice([8, 16, 32])
        n, k = rng.choice([(4096, 7168), (7168, 2048), (_log(rng, 512, 4096), _k(rng, 512, 7168))])
        if kind == "moe":
            return {"kind": kind, "experts": e, "rows": _log(rng, 16, 4096), "n": n, "k": k,
                    "out": out}
        max_m = rng.choice([8, 16, 32, 64, 128])
        return {"kind": kind, "experts": e, "max_m": max_m,
                "rows": _log(rng, 8, max(8, e * max_m // 2)), "n": n, "k": k, "out": out}
    rows = _log(rng, 1, 4096)
    cols = _k(rng, 512, 18432)
    return {"kind": kind, "rows": rows, "cols": cols, "dt": dt}


# ---- inputs -------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _acts(g, rows, cols, dt, std=1.0):
    """Activations: normal, one value in a thousand an outlier of 20 sigma."""
    x = torch.randn((rows, cols), generator=g, device=DEV)
    big = torch.rand((rows, cols), generator=g, device=DEV) < 1e-3
    x = torch.where(big, x * 20.0, x) * std
    return x.to(TORCH_DT[dt])


def _quant_rows(x):
    """The stored form of activations: E4M3 bytes and a scale per 128 columns."""
    rows, cols = x.shape
    v = x.float().view(rows, cols // 128, 128)
    s = v.abs().amax(-1) * torch.tensor(1.0 / 448.0, dtype=torch.float32, device=x.device)
    s = torch.where(s == 0, torch.ones_like(s), s)
    q = (v / s[..., None]).to(torch.float8_e4m3fn).view(torch.uint8).view(rows, cols)
    return q, s


def _weight(g, n, k):
    """A layer's weight as a checkpoint stores it: N(0, 0.02) in E4M3 bytes
    with a scale per 128 x 128 block."""
    nb = -(-n // 128)
    w = torch.zeros((nb * 128, k), device=DEV)
    w[:n] = torch.randn((n, k), generator=g, device=DEV) * 0.02
    v = w.view(nb, 128, k // 128, 128)
    s = v.abs().amax((1, 3)) * (1.0 / 448.0)
    q = (v / s[:, None, :, None]).to(torch.float8_e4m3fn).view(torch.uint8)
    return q.view(nb * 128, k)[:n].contiguous(), s.contiguous()


def _counts(case, seed):
    """Rows per expert: a uniform multinomial routing."""
    g = torch.Generator()
    g.manual_seed(seed)
    pick = torch.randint(0, case["experts"], (case["rows"],), generator=g)
    return torch.bincount(pick, minlength=case["experts"])


def _masked_counts(case, seed):
    return torch.clamp(_counts(case, seed), max=case["max_m"])


def _inputs(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "topk":
        return {"logits": torch.randn((case["tokens"], case["experts"]), generator=g,
                                      device=DEV) * 2.0}
    if kind in ("fused_linear", "linear"):
        x = _acts(g, case["m"], case["k"], case["dt"])
        bq, bs = _weight(g, case["n"], case["k"])
        return {"x": x, "bq": bq, "bs": bs}
    if kind == "gemm":
        aq, as_ = _quant_rows(_acts(g, case["m"], case["k"], "bf16"))
        bq, bs = _weight(g, case["n"], case["k"])
        return {"aq": aq, "as": as_, "bq": bq, "bs": bs}
    if kind in ("moe_masked", "moe"):
        e, n, k = case["experts"], case["n"], case["k"]
        rows = case["rows"] if kind == "moe" else e * case["max_m"]
        aq, as_ = _quant_rows(_acts(g, rows, k, "bf16"))
        bq = torch.empty((e, n, k), dtype=torch.uint8, device=DEV)
        bs = torch.empty((e, -(-n // 128), k // 128), device=DEV)
        for i in range(e):
            bq[i], bs[i] = _weight(g, n, k)
        return {"aq": aq, "as": as_, "bq": bq, "bs": bs}
    if kind == "silu":
        return {"gate_up": _acts(g, case["rows"], 2 * case["cols"], case["dt"])}
    if kind == "norm":
        return {"residual": _acts(g, case["rows"], case["cols"], case["dt"]),
                "x": _acts(g, case["rows"], case["cols"], case["dt"], 0.1),
                "weight": (1.0 + 0.1 * torch.randn((case["cols"],), generator=g, device=DEV)
                           ).to(TORCH_DT[case["dt"]])}
    return {"x": _acts(g, case["rows"], case["cols"], case["dt"])}


def prepare(case, seed):
    """The inputs in hand before the call, and the buffers a serving program
    keeps for the outputs of the raw calls."""
    st = _inputs(case, seed)
    st["case"] = case
    kind = case["kind"]

    def u8(*shape):
        return torch.empty(shape, dtype=torch.uint8, device=DEV)

    def f32(*shape):
        return torch.empty(shape, dtype=torch.float32, device=DEV)

    if kind == "topk":
        st["ids"] = torch.empty((case["tokens"], case["topk"]), dtype=torch.int32, device=DEV)
        st["weights"] = f32(case["tokens"], case["topk"])
    elif kind == "fused_linear":
        st["q"], st["s"] = u8(case["m"], case["k"]), f32(case["m"], case["k"] // 128)
        st["c"] = torch.empty((case["m"], case["n"]), dtype=TORCH_DT[case["out"]], device=DEV)
    elif kind == "moe":
        off = torch.zeros(case["experts"] + 1, dtype=torch.int32)
        off[1:] = torch.cumsum(_counts(case, seed), 0)
        st["offsets"] = off.to(DEV)
        st["c"] = torch.empty((case["rows"], case["n"]), dtype=TORCH_DT[case["out"]], device=DEV)
    elif kind == "moe_masked":
        st["masked_m"] = _masked_counts(case, seed).to(torch.int32).to(DEV)
        st["expected_m"] = -(-case["rows"] // case["experts"])
        # rows past an expert's count are never written
        st["c"] = torch.zeros((case["experts"], case["max_m"], case["n"]),
                              dtype=TORCH_DT[case["out"]], device=DEV)
    elif kind in ("silu", "norm"):
        st["q"], st["s"] = u8(case["rows"], case["cols"]), f32(case["rows"], case["cols"] // 128)
    return st


def _ok(status):
    if status != ia.Status.OK:
        raise ia.InferopError(status, "perf case")


def run(state):
    """One call (or one layer's calls) as a serving program makes them."""
    case = state["case"]
    kind = case["kind"]
    if kind == "topk":
        _ok(ia.topk_softmax(state["ids"], state["weights"], state["logits"], case["tokens"],
                            case["experts"], case["topk"]))
        return [state["ids"], state["weights"]]
    if kind == "fused_linear":
        _ok(ia.quant_w8a8_block_fp8_gemm(state["c"], state["q"], state["s"], state["x"],
                                         DT_CODE[case["dt"]], state["bq"], state["bs"], case["m"],
                                         case["n"], case["k"], out_dt=DT_CODE[case["out"]]))
        return [state["q"], state["s"], state["c"]]
    if kind == "linear":
        q, s = ia.quantize(state["x"])
        return [q, s, ia.gemm(q, s, state["bq"], state["bs"], TORCH_DT[case["out"]])]
    if kind == "gemm":
        return ia.gemm(state["aq"], state["as"], state["bq"], state["bs"], TORCH_DT[case["out"]])
    if kind == "moe":
        _ok(ia.w8a8_block_fp8_grouped_gemm(state["c"], state["aq"], state["as"], state["bq"],
                                           state["bs"], state["offsets"], case["rows"], case["n"],
                                           case["k"], case["experts"],
                                           out_dt=DT_CODE[case["out"]]))
        return state["c"]
    if kind == "moe_masked":
        _ok(ia.w8a8_block_fp8_grouped_gemm_masked(
            state["c"], state["aq"], state["as"], state["bq"], state["bs"], state["masked_m"],
            case["max_m"], case["n"], case["k"], case["experts"], state["expected_m"],
            out_dt=DT_CODE[case["out"]]))
        return state["c"]
    if kind == "silu":
        _ok(ia.silu_and_mul_quant_fp8(state["q"], state["s"], state["gate_up"],
                                      DT_CODE[case["dt"]], case["rows"], case["cols"]))
        return [state["q"], state["s"]]
    if kind == "norm":
        _ok(ia.fused_add_rmsnorm_quant_fp8(state["residual"], state["q"], state["s"], state["x"],
                                           state["weight"], DT_CODE[case["dt"]], case["rows"],
                                           case["cols"]))
        return [state["residual"], state["q"], state["s"]]
    q, s = ia.quantize(state["x"])
    return [q, s, ia.dequantize(q, s, TORCH_DT[case["dt"]])]


# ---- what a pass cannot do without ----------------------------------------------
def _row_bytes(m, k):
    return m * k + 4 * m * (k // 128)


def _weight_bytes(n, k):
    return n * k + 4 * (-(-n // 128)) * (k // 128)


def work(case):
    kind = case["kind"]
    if kind == "topk":
        t = case["tokens"]
        return {"bytes": 4 * t * case["experts"] + 8 * t * case["topk"],
                "flops": 4 * t * case["experts"]}
    if kind in ("fused_linear", "linear", "gemm"):
        m, n, k = case["m"], case["n"], case["k"]
        b = _row_bytes(m, k) + _weight_bytes(n, k) + m * n * DT_BYTES[case["out"]]
        if kind != "gemm":
            b += m * k * DT_BYTES[case["dt"]]
        return {"bytes": b, "flops": 2 * m * n * k}
    if kind in ("moe", "moe_masked"):
        # the weights of the experts a uniform routing reaches, once
        e, n, k, rows = case["experts"], case["n"], case["k"], case["rows"]
        hit = e * (1.0 - (1.0 - 1.0 / e) ** rows)
        return {"bytes": int(hit * _weight_bytes(n, k)) + _row_bytes(rows, k)
                + rows * n * DT_BYTES[case["out"]], "flops": 2 * rows * n * k}
    rows, cols, b = case["rows"], case["cols"], DT_BYTES[case["dt"]]
    el = rows * cols
    if kind == "silu":
        return {"bytes": 2 * el * b + _row_bytes(rows, cols), "flops": 6 * el}
    if kind == "norm":
        return {"bytes": 3 * el * b + cols * b + _row_bytes(rows, cols), "flops": 6 * el}
    return {"bytes": 2 * el * b + 2 * _row_bytes(rows, cols), "flops": 3 * el}


def tolerance(case):
    kind = case["kind"]
    if kind == "codec":
        # every byte and scale is defined to the last bit
        return "exact"
    if kind == "topk":
        # fp32 exponentials and a sum over at most 384 experts
        return {"rel": 4e-7, "max": 3e-6, "differ": 1e-3}
    if kind in ("silu", "norm"):
        # the quantized value is rounded to the model's dtype first: a last-bit
        # change of the fp32 value moves few of the 16-bit values, by one step
        # each
        step = {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11, "fp32": 2.0 ** -20}[case["dt"]]
        return {"rel": max(0.05 * step, 2e-6), "max": 4.0 * step, "differ": 2e-4}
    # The matrix cores' own sum of a 128-wide group and the fp32 sums over K lie
    # 2.2e-5 (2-norm; largest 2.8e-4) from the 64-bit result; against that
    # result rounded to the output's dtype a bf16 output differs by 2.8e-4 and an
    # fp16 one by 9.8e-5, each value by one step at most.  Four times that.
    return {"bf16": {"rel": 1.1e-3, "max": 2.0 ** -6, "differ": 0.0},
            "fp16": {"rel": 4e-4, "max": 2.0 ** -8, "differ": 0.0},
            "fp32": {"rel": 9e-5, "max": 1.2e-3, "differ": 0.0}}[case["out"]]


# ---- the same in 64 bits, in plain torch ----------------------------------------
def _values(q):
    return q.view(torch.float8_e4m3fn).to(torch.float64)


def _gemm64(aq, as_, bq, bs):
    a = _values(aq) * as_.double().repeat_interleave(128, 1)
    b = _values(bq) * bs.double().repeat_interleave(128, 0)[:bq.shape[0]].repeat_interleave(128, 1)
    return a @ b.t().contiguous()


def exact(case, seed):
    st = _inputs(case, seed)
    kind = case["kind"]
    if kind == "topk":
        p = torch.softmax(st["logits"].double(), -1)
        w, ids = torch.topk(p, case["topk"], dim=-1)
        return [ids.to(torch.int32), w / w.sum(-1, keepdim=True)]
    if kind in ("fused_linear", "linear"):
        q, s = _quant_rows(st["x"])
        s64 = st["x"].double().view(s.shape[0], s.shape[1], 128).abs().amax(-1) / 448.0
        return [None, s64, _gemm64(q, s, st["bq"], st["bs"])]
    if kind == "gemm":
        return _gemm64(st["aq"], st["as"], st["bq"], st["bs"])
    if kind == "moe":
        out = torch.empty((case["rows"], case["n"]), dtype=torch.float64, device=DEV)
        lo = 0
        for e, cnt in enumerate(_counts(case, seed).tolist()):
            if cnt:
                out[lo:lo + cnt] = _gemm64(st["aq"][lo:lo + cnt], st["as"][lo:lo + cnt],
                                           st["bq"][e], st["bs"][e])
            lo += cnt
        return out
    if kind == "moe_masked":
        mm = case["max_m"]
        out = torch.zeros((case["experts"], mm, case["n"]), dtype=torch.float64, device=DEV)
        for e, cnt in enumerate(_masked_counts(case, seed).tolist()):
            if cnt:
                out[e, :cnt] = _gemm64(st["aq"][e * mm:e * mm + cnt], st["as"][e * mm:e * mm + cnt],
                                       st["bq"][e], st["bs"][e])
        return out
    rows, cols = case["rows"], case["cols"]
    if kind == "silu":
        g = st["gate_up"].double()
        y = torch.nn.functional.silu(g[:, :cols]) * g[:, cols:]
        return [None, y.view(rows, cols // 128, 128).abs().amax(-1) / 448.0]
    if kind == "norm":
        r = st["residual"].double() + st["x"].double()
        y = r * torch.rsqrt((r * r).mean(-1, keepdim=True) + 1e-6) * st["weight"].double()
        return [r, None, y.view(rows, cols // 128, 128).abs().amax(-1) / 448.0]
    q, s = _quant_rows(st["x"])
    s64 = st["x"].double().view(rows, cols // 128, 128).abs().amax(-1) / 448.0
    return [None, s64, _values(q) * s.double().repeat_interleave(128, 1)]
