"""Performance cases of the quantized-inference path, through its Plan surface.

A case is a dict of plain values; `kind` names the call a serving program makes
and the other keys its sizes and options.  `listed()` holds the fixed cases,
`draw()` more of the same ranges, `prepare()` what the program holds before
the call, `run()` one pass, `work()` the bytes and operations a pass cannot do
without, `tolerance()` how far another correct implementation may be, and
`exact()` the result in 64-bit arithmetic.
"""
from __future__ import annotations

import math

import torch

from baracuda_amd import plans as P

DEV = "cuda:0"

_VOCAB = 32000      # rows of a decode step's embedding table


def listed():
    return [
        # One new token of one stream: embedding row, then the four linears of a
        # decoder layer (qkv, attention output, gate + up, down), captured once
        # and replayed, as decode loops are run.
        {"name": "step_b1", "kind": "step", "b": 1, "hidden": 4096, "ffn": 14336},
        # The same step for a batch of 24 streams and an MLP width that is not a
        # multiple of 512.
        {"name": "step_b24", "kind": "step", "b": 24, "hidden": 4096, "ffn": 11008},
        # A long prompt through a square projection: per-token quantization and
        # the W8A8 GEMM (4096 tokens, N = K = 4096).
        {"name": "linear_prefill", "kind": "linear", "dtype": "bf16", "m": 4096, "n": 4096, "k": 4096},
        # A chunk of a prompt, an odd number of tokens, float32 activations and
        # output.
        {"name": "linear_chunk", "kind": "linear", "dtype": "f32", "m": 777, "n": 11008, "k": 4096},
        # An encoder MLP's first half on int8 activations: bias and GELU in the
        # epilogue, a hidden size that is a multiple of 64 only.
        {"name": "int8_gelu", "kind": "int8", "element": "s8", "layout": "rcr", "epilogue": "bias_gelu",
         "m": 1500, "n": 5120, "k": 2880},
        # MLP up-projection of a long prompt in FP8: delayed-scaling cast of the
        # activations, then the GEMM to bf16.
        {"name": "fp8_linear", "kind": "fp8_linear", "m": 2048, "n": 14336, "k": 4096},
        # FP8 in and out with bias and SiLU for a batch of a few hundred rows.
        {"name": "fp8_silu", "kind": "fp8", "element": "e4m3", "layout": "rcr", "epilogue": "bias_silu",
         "m": 200, "n": 11008, "k": 4096},
        # Weight-only int8 decode of one token (m = 1).
        {"name": "gemv_s8w", "kind": "gemv_s8w", "n": 14336, "k": 4096},
        # Dense m = 1 decode in bf16, with the workspace the plan asks for.
        {"name": "gemv_dense", "kind": "gemv_dense", "dtype": "bf16", "n": 4096, "k": 4096, "batch": 1},
        # Mixture of experts, a long prompt: 4096 tokens, 2 of 8 experts, Zipf
        # routing, W8A8.
        {"name": "moe_prefill", "kind": "moe_s8", "tokens": 4096, "experts": 8, "topk": 2, "n": 14336, "k": 4096},
        # The same experts in bf16 for a serving batch of 192 tokens.
        {"name": "moe_batch", "kind": "moe_float", "dtype": "bf16", "tokens": 192, "experts": 8, "topk": 2,
         "n": 14336, "k": 4096},
        # Many small experts: 512 tokens, 6 of 64, W8A8.
        {"name": "moe_fine", "kind": "moe_s8", "tokens": 512, "experts": 64, "topk": 6, "n": 1408, "k": 2048},
    ]


_MAX_FLOPS = 2.0 * 8192 * 14336 * 4096      # of the largest listed case


def _log(rng, lo, hi, step=1):
    """An integer of [lo, hi], even over the logarithm, a multiple of `step`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def draw(rng):
    kind = rng.choice(["step", "linear", "linear", "int8", "fp8_linear", "fp8", "gemv_s8w", "gemv_dense",
                       "moe_s8", "moe_float"])
    if kind == "step":
        # batches of 1 to 64 streams, widths in multiples of 128
        return {"kind": kind, "b": _log(rng, 1, 64), "hidden": _log(rng, 1024, 5120, 128),
                "ffn": _log(rng, 2816, 14336, 128)}
    if kind in ("linear", "int8", "fp8_linear", "fp8"):
        # 16 to 4096 tokens (odd counts among them), widths in multiples of 16, depths of 64
        m, n, k = _log(rng, 16, 4096), _log(rng, 1024, 14336, 16), _log(rng, 1024, 14336, 64)
        m = max(16, min(m, int(_MAX_FLOPS / (2.0 * n * k))))
        case = {"kind": kind, "m": m, "n": n, "k": k}
        if kind == "linear":
            case["dtype"] = rng.choice(["bf16", "bf16", "f32"])
        elif kind == "int8":
            case["element"] = rng.choice(["s8", "s8", "u8"])
            case["layout"] = rng.choice(["rcr", "rcr", "rrr"])
            case["epilogue"] = rng.choice(["identity", "bias_relu", "bias_gelu", "bias_silu"])
        elif kind == "fp8":
            case["element"] = rng.choice(["e4m3", "e4m3", "e5m2"])
            case["layout"] = rng.choice(["rcr", "rcr", "rrr"])
            case["epilogue"] = rng.choice(["identity", "bias", "bias_gelu", "bias_silu"])
        return case
    if kind == "gemv_s8w":
        return {"kind": kind, "n": _log(rng, 1024, 65536), "k": _log(rng, 1024, 14336, 64)}
    if kind == "gemv_dense":
        return {"kind": kind, "dtype": rng.choice(["bf16", "f16", "f32"]), "n": _log(rng, 1024, 32000, 8),
                "k": _log(rng, 1024, 8192), "batch": rng.choice([1, 1, 1, 4])}
    experts = rng.choice([8, 16, 64])
    case = {"kind": kind, "tokens": _log(rng, 1, 4096), "experts": experts, "topk": rng.choice([1, 2, 4, 6]),
            "n": _log(rng, 768, 14336 if experts < 64 else 2048, 64), "k": _log(rng, 1024, 4096, 64)}
    most = _MAX_FLOPS / (2 if kind == "moe_s8" else 4)
    case["tokens"] = max(1, min(case["tokens"], int(most / (2.0 * case["topk"] * case["n"] * case["k"]))))
    if kind == "moe_float":
        case["dtype"] = rng.choice(["bf16", "f16"])
    return case


# ---- inputs -----------------------------------------------------------------
_TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32,
          "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2, "s8": torch.int8, "u8": torch.uint8}
_FP8_MAX = {"e4m3": 448.0, "e5m2": 57344.0}
_EPI = {"identity": P.EpilogueKind.Identity, "bias": P.EpilogueKind.Bias, "bias_relu": P.EpilogueKind.BiasRelu,
        "bias_gelu": P.EpilogueKind.BiasGelu, "bias_silu": P.EpilogueKind.BiasSilu}
_LAYOUT = {"rcr": P.LayoutSku.Rcr, "rrr": P.LayoutSku.Rrr}


class _Rand:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def s8(self, *shape):
        return torch.randint(-127, 128, shape, dtype=torch.int8, device=DEV, generator=self.g)

    def u8(self, *shape):
        return torch.randint(0, 256, shape, dtype=torch.uint8, device=DEV, generator=self.g)

    def normal(self, *shape, dtype=torch.float32, std=1.0):
        return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=self.g)

    def uniform(self, lo, hi, *shape):
        return torch.empty(shape, dtype=torch.float32, device=DEV).uniform_(lo, hi, generator=self.g)

    def fp8(self, element, *shape):
        """N(0, 1) scaled so that the largest magnitude maps to the format's
        largest value, and the scale that undoes it.  An e5m2 operand keeps its
        products within float32 and half of the format's range."""
        x = self.normal(*shape)
        s = _FP8_MAX[element] / float(x.abs().max())
        if element == "e5m2":
            s /= 256.0
        return (x * s).to(_TORCH[element]), 1.0 / s


def _linear(r, m, n, k, dtype):
    """What a W8A8 linear layer keeps and is given."""
    t = _TORCH[dtype]
    return {"plan": P.QuantizedLinearPlan.select(P.QuantizedLinearDescriptor(m, n, k)),
            "x": r.normal(m, k, dtype=t), "w": r.s8(n, k), "sw": r.uniform(0.001, 0.01, n),
            "out": torch.empty((m, n), dtype=t, device=DEV),
            "q": torch.empty((m, k), dtype=torch.int8, device=DEV),
            "sa": torch.empty(m, dtype=torch.float32, device=DEV)}


def _run_linear(s):
    s["plan"].run(s["x"], s["w"], s["sw"], s["out"], s["q"], s["sa"])


def _routing(case, seed):
    """Zipf(1.1) top-k routing: pair ids grouped by expert, and their experts."""
    g = torch.Generator()
    g.manual_seed(seed)
    e, topk, tokens = case["experts"], case["topk"], case["tokens"]
    p = 1.0 / torch.arange(1, e + 1, dtype=torch.float64) ** 1.1
    p = p[torch.randperm(e, generator=g)]
    chosen = torch.multinomial(p.expand(tokens, e), topk, replacement=False, generator=g).reshape(-1)
    order = torch.argsort(chosen, stable=True)
    return order.to(torch.int32).to(DEV), chosen[order].to(torch.int32).to(DEV)


def prepare(case, seed):
    r, kind = _Rand(seed), case["kind"]
    if kind == "step":
        b, h, f = case["b"], case["hidden"], case["ffn"]
        shapes = [("qkv", h + h // 2, h), ("o", h, h), ("gate_up", 2 * f, h), ("down", h, f)]
        lin = {name: _linear(r, b, n, k, "bf16") for name, n, k in shapes}
        s = {"kind": kind, "table": r.normal(_VOCAB, h, dtype=torch.bfloat16, std=0.02), "lin": lin,
             "idx": torch.randint(0, _VOCAB, (b,), dtype=torch.int32, device=DEV, generator=r.g).view(torch.uint32)}

        def step():
            P.gather_rows(lin["qkv"]["x"], s["table"], s["idx"])
            for v in lin.values():
                _run_linear(v)

        step()      # loads the code before the capture
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            step()
        return s
    if kind == "linear":
        return dict(_linear(r, case["m"], case["n"], case["k"], case["dtype"]), kind=kind)
    if kind == "int8":
        m, n, k, el = case["m"], case["n"], case["k"], case["element"]
        e = {"s8": P.ElementKind.S8, "u8": P.ElementKind.U8}[el]
        plan = P.IntGemmPlan.select(P.IntGemmDescriptor(m, n, k, layout=_LAYOUT[case["layout"]],
                                                        epilogue=_EPI[case["epilogue"]], output=e, element=e))
        rand = r.s8 if el == "s8" else r.u8
        ws = plan.workspace_size()
        return {"kind": kind, "plan": plan, "a": rand(m, k), "b": rand(n, k) if case["layout"] == "rcr" else rand(k, n),
                "d": torch.empty((m, n), dtype=_TORCH[el], device=DEV), "alpha": _int8_alpha(case),
                "bias": None if case["epilogue"] == "identity" else r.normal(n, std=20.0),
                "ws": torch.empty(ws, dtype=torch.uint8, device=DEV) if ws else None}
    if kind == "fp8_linear":
        m, n, k = case["m"], case["n"], case["k"]
        b, sb = r.fp8("e4m3", n, k)
        x = r.normal(m, k, dtype=torch.bfloat16)
        a = torch.empty((m, k), dtype=torch.float8_e4m3fn, device=DEV)
        recipe = P.Fp8Recipe(P.Fp8Format.E4M3, 16)
        cast = P.Fp8CastPlan.select()
        cast.run(x, a, recipe)              # the step before: its amax sets this step's scale
        recipe.update_after_pass()
        plan = P.Fp8GemmPlan.select(P.Fp8GemmDescriptor(m, n, k, output=P.ElementKind.Bf16))
        return {"kind": kind, "plan": plan, "cast": cast, "recipe": recipe, "x": x, "a": a, "b": b,
                "sa": recipe.scale_inv_host(), "sb": sb, "d": torch.empty((m, n), dtype=torch.bfloat16, device=DEV)}
    if kind == "fp8":
        m, n, k, el = case["m"], case["n"], case["k"], case["element"]
        e = {"e4m3": P.ElementKind.Fp8E4M3, "e5m2": P.ElementKind.Fp8E5M2}[el]
        a, sa = r.fp8(el, m, k)
        b, sb = r.fp8(el, *((n, k) if case["layout"] == "rcr" else (k, n)))
        plan = P.Fp8GemmPlan.select(P.Fp8GemmDescriptor(m, n, k, layout=_LAYOUT[case["layout"]],
                                                        epilogue=_EPI[case["epilogue"]], output=e, element=e))
        return {"kind": kind, "plan": plan, "a": a, "b": b, "alpha": sa * sb / math.sqrt(k),
                "bias": None if case["epilogue"] == "identity" else r.normal(n, std=0.5),
                "d": torch.empty((m, n), dtype=_TORCH[el], device=DEV)}
    if kind == "gemv_s8w":
        n, k = case["n"], case["k"]
        return {"kind": kind, "plan": P.GemvS8wPlan.select(n, k), "x": r.normal(k, dtype=torch.bfloat16),
                "w": r.s8(n, k), "scale": r.uniform(0.001, 0.01, n),
                "d": torch.empty(n, dtype=torch.bfloat16, device=DEV)}
    if kind == "gemv_dense":
        n, k, batch, t = case["n"], case["k"], case["batch"], _TORCH[case["dtype"]]
        plan = P.GemvDensePlan.select(P.GemvDenseDescriptor(n, k, batch), t)
        ws = plan.workspace_size()
        return {"kind": kind, "plan": plan, "a": r.normal(batch, k, dtype=t),
                "b": r.normal(batch, k, n, dtype=t, std=1.0 / math.sqrt(k)),
                "d": torch.empty((batch, n), dtype=t, device=DEV),
                "ws": torch.empty(ws, dtype=torch.uint8, device=DEV) if ws else None}
    # moe_s8 / moe_float
    e, topk, tokens, n, k = (case[x] for x in ("experts", "topk", "tokens", "n", "k"))
    ids, experts = _routing(case, seed)
    s = {"kind": kind, "ids": ids, "experts": experts,
         "counts": torch.empty(e, dtype=torch.int32, device=DEV),
         "offsets": torch.empty(e + 1, dtype=torch.int32, device=DEV)}
    if kind == "moe_s8":
        s.update(plan=P.MoeS8GroupedPlan.select(e, topk, tokens * topk, n, k), x=r.s8(tokens, k), w=r.s8(e, n, k),
                 sa=r.uniform(0.005, 0.02, tokens), sw=r.uniform(0.001, 0.01, e * n),
                 out=torch.empty((tokens * topk, n), dtype=torch.bfloat16, device=DEV))
    else:
        t = _TORCH[case["dtype"]]
        el = P.ElementKind.Bf16 if case["dtype"] == "bf16" else P.ElementKind.F16
        s.update(plan=P.MoePlan.select(P.MoeDescriptor(tokens, e, topk, k, n, element=el)),
                 x=r.normal(tokens, k, dtype=t), w=r.normal(e, n, k, dtype=t, std=1.0 / math.sqrt(k)),
                 out=torch.empty((tokens * topk, n), dtype=t, device=DEV))
    return s


def _int8_alpha(case):
    """Scale that spreads the outputs over the 8-bit range."""
    if case["element"] == "s8":
        return 40.0 / (127.0 * 127.0 / 3.0 * math.sqrt(case["k"]))
    return 128.0 / (127.5 * 127.5 * case["k"])


# ---- one pass ----------------------------------------------------------------
def run(s):
    kind, plan = s["kind"], s.get("plan")
    if kind == "step":
        s["graph"].replay()
        return {name: v["out"] for name, v in s["lin"].items()}
    if kind == "linear":
        _run_linear(s)
        return s["out"]
    if kind == "int8":
        plan.run(s["a"], s["b"], s["d"], alpha=s["alpha"], beta=0.0, bias=s["bias"], workspace=s["ws"])
        return s["d"]
    if kind == "fp8_linear":
        s["cast"].run(s["x"], s["a"], s["recipe"])
        plan.run(s["a"], s["b"], s["d"], scale_a=s["sa"], scale_b=s["sb"])
        return {"out": s["d"], "amax": s["recipe"].amax_history}
    if kind == "fp8":
        plan.run(s["a"], s["b"], s["d"], alpha=s["alpha"], bias=s["bias"])
        return s["d"]
    if kind == "gemv_s8w":
        plan.run(s["x"], s["w"], s["scale"], s["d"])
        return s["d"]
    if kind == "gemv_dense":
        n, k = s["d"].shape[1], s["a"].shape[1]
        plan.run(s["a"], s["b"], s["d"], lda=k, stride_a=k, ldb=n, stride_b=k * n, ldd=n, stride_d=n,
                 workspace=s["ws"])
        return s["d"]
    if kind == "moe_s8":
        plan.run(s["x"], s["w"], s["ids"], s["experts"], s["out"], s["counts"], s["offsets"], s["sa"], s["sw"])
        return s["out"]
    plan.run(s["x"], s["w"], s["ids"], s["experts"], s["out"], s["counts"], s["offsets"])
    return s["out"]


# ---- what a pass cannot do without -------------------------------------------
_BYTES = {"bf16": 2, "f16": 2, "f32": 4}


def work(case):
    kind = case["kind"]
    if kind == "step":
        b, h, f = case["b"], case["hidden"], case["ffn"]
        shapes = [(h + h // 2, h), (h, h), (2 * f, h), (h, f)]
        return {"bytes": sum(n * k + 2 * b * (n + k) + 4 * n for n, k in shapes),
                "flops": sum(2.0 * b * n * k for n, k in shapes)}
    if kind == "gemv_s8w":
        n, k = case["n"], case["k"]
        return {"bytes": n * k + 2 * k + 6 * n, "flops": 2.0 * n * k}
    if kind == "gemv_dense":
        n, k, z, b = case["n"], case["k"], _BYTES[case["dtype"]], case["batch"]
        return {"bytes": b * z * (n * k + n + k), "flops": 2.0 * b * n * k}
    if kind in ("moe_s8", "moe_float"):
        t, e, topk, n, k = (case[x] for x in ("tokens", "experts", "topk", "n", "k"))
        z = 1 if kind == "moe_s8" else 2
        # experts that get a token: all of them but for a few tokens
        touched = min(e, t * topk)
        return {"bytes": z * (t * k + touched * n * k) + 2 * t * topk * n, "flops": 2.0 * t * topk * n * k}
    m, n, k = case["m"], case["n"], case["k"]
    z_in, z_out = 1, 1
    if kind == "linear":
        z_in = z_out = _BYTES[case["dtype"]]
    elif kind == "fp8_linear":
        z_in = z_out = 2
    return {"bytes": z_in * m * k + n * k + z_out * m * n, "flops": 2.0 * m * n * k}


def tolerance(case):
    kind = case["kind"]
    if kind == "int8":
        # integer sums, one float32 epilogue; GELU and SiLU go through
        # approximate exponentials, so a value at a rounding tie may differ
        return {"differ": 1e-3}
    if kind == "fp8":
        # float32 sums in another order move a value across a rounding tie of
        # the 8-bit output: a step is an eighth (e4m3) or a quarter (e5m2)
        return {"rel": 1e-2, "max": 0.3}
    if case.get("dtype") == "f32":
        if kind == "linear":
            # a rounding tie of the quantizer moves a whole int8 step
            return {"rel": 4e-4, "max": 2e-2}
        return {"rel": 1e-5, "max": 1e-4}
    if case.get("dtype") == "f16":
        return {"rel": 1e-3, "max": 4e-3}
    # one rounding to bf16 (2^-9 each way)
    return {"rel": 7e-3, "max": 2e-2}


# ---- the same in 64 bits -------------------------------------------------------
def _fake(x, k):
    """Per-token symmetric int8 quantization in 64 bits: codes and scales."""
    x = x.double()
    s = x.abs().amax(dim=1, keepdim=True) / 127.0
    s = torch.where(s == 0, torch.ones_like(s), s)
    return torch.clamp(torch.round(x / s), -127, 127), s


def _exact_linear(x, w, sw):
    q, s = _fake(x, x.shape[1])
    return (q @ w.double().t()) * s * sw.double()


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    if kind == "step":
        lin = s["lin"]
        x = {name: v["x"] for name, v in lin.items()}
        x["qkv"] = s["table"][s["idx"].view(torch.int32).long()]
        return {name: _exact_linear(x[name], v["w"], v["sw"]) for name, v in lin.items()}
    if kind == "linear":
        return _exact_linear(s["x"], s["w"], s["sw"])
    if kind == "int8":
        return None
    if kind == "fp8_linear":
        a = (s["x"].double() / s["sa"]).float().to(torch.float8_e4m3fn)
        out = (a.double() @ s["b"].double().t()) * (s["sa"] * s["sb"])
        amax = torch.zeros(16, dtype=torch.float64, device=DEV)
        amax[1] = s["x"].double().abs().max()
        return {"out": out, "amax": amax}
    if kind == "fp8":
        b = s["b"].double().t() if case["layout"] == "rcr" else s["b"].double()
        v = (s["a"].double() @ b) * s["alpha"]
        if s["bias"] is not None:
            v = v + s["bias"].double()
        if case["epilogue"] == "bias_gelu":
            v = torch.nn.functional.gelu(v)
        elif case["epilogue"] == "bias_silu":
            v = torch.nn.functional.silu(v)
        return v
    if kind == "gemv_s8w":
        return (s["w"].double() @ s["x"].double()) * s["scale"].double()
    if kind == "gemv_dense":
        return torch.stack([a.double() @ b.double() for a, b in zip(s["a"], s["b"])])
    n, k, topk = case["n"], case["k"], case["topk"]
    out = torch.empty((case["tokens"] * topk, n), dtype=torch.float64, device=DEV)
    w = s["w"]
    for e in range(case["experts"]):
        rows = s["ids"][s["experts"] == e].long()
        if rows.numel() == 0:
            continue
        v = s["x"][rows // topk].double() @ w[e].double().t()
        if kind == "moe_s8":
            v = v * s["sa"][rows // topk].double()[:, None] * s["sw"][e * n:(e + 1) * n].double()
        out[rows] = v
    return out
