"""The work that programs have this framework do, as cases that can be timed.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw()`
others of the same ranges; `prepare()` builds what a program holds before the
call, `run()` makes the call through the public entry points, `work()` prices
it, and `exact()` gives the same outputs from plain torch in 64 bits.

Kinds of case, by "op":
  weights   serving with MXFP4 weights kept packed and unquantized
            activations: `mxfp4_linear_w` (decode, prefill; bf16, fp16, fp32)
  dual      two activation batches against one packed weight: `dual_mxfp4`
  infer     `MXFP4Linear` without gradients: activations and the layer's own
            weight quantized in the call
  step      `MXFP4Linear` forward and backward, straight-through or with the
            backward in MXFP4
  packed    quantize operands and multiply them (`mxfp4_gemm_packed`), with
            the fused quantizer or through the reference's call sequence
  fp8       `mxfp4_gemm_fp8` on E4M3 operands and fp32 block scales
  dense     the dense GEMMs of `dual_gemm` (one product, two, or two in one
            accumulator)
"""

import math

import torch

from lockstep_amd import dual_gemm, fp4, mxfp4_gemm
from lockstep_amd.fp4_linear import MXFP4Linear

_DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one token through the up projection of a served MLP (hidden 4096,
        # ffn 14336): the smallest call, where latency counts
        {"name": "decode_1", "op": "weights", "dtype": "bf16", "M": 1, "N": 14336, "K": 4096},
        # twenty requests decoded together, the down projection
        {"name": "decode_20", "op": "weights", "dtype": "bf16", "M": 20, "N": 4096, "K": 14336},
        # a prompt of odd length
        {"name": "prefill_600", "op": "weights", "dtype": "bf16", "M": 600, "N": 14336, "K": 4096},
        # fp32 activations against a packed weight: a fake-quant evaluation
        {"name": "weights_f32_256", "op": "weights", "dtype": "f32", "M": 256, "N": 1024, "K": 1024},
        # two batches that share one weight
        {"name": "dual_2048", "op": "dual", "dtype": "bf16", "M": 2048, "N": 4096, "K": 4096},
        # a small evaluation batch through a layer that keeps plain weights
        {"name": "infer_200", "op": "infer", "dtype": "bf16", "M": 200, "N": 8192, "K": 2048},
        # training under autocast, the layer's default backward, ragged tokens
        {"name": "step_3000", "op": "step", "quantized": False, "M": 3000, "N": 2048, "K": 8192},
        # training under autocast with all three products in MXFP4
        {"name": "step_q_4096", "op": "step", "quantized": True, "M": 4096, "N": 8192, "K": 2048},
        # the large square product, both operands quantized on the fly
        {"name": "packed_8192", "op": "packed", "spelling": "fused", "dtype": "f32", "M": 8192, "N": 8192,
         "K": 8192},
        # the reference's call sequence (codes, fp32 scales, pack) at odd sizes
        {"name": "packed_ref_1111", "op": "packed", "spelling": "reference", "dtype": "bf16", "M": 1111,
         "N": 3000, "K": 2176},
        # E4M3 operands with fp32 block scales, B as [K, N]
        {"name": "fp8_1500", "op": "fp8", "dtype": "bf16", "M": 1500, "N": 4096, "K": 4096},
        # two dense products in one launch, few output tiles
        {"name": "dense_1024", "op": "dense", "form": "separate", "dtype": "bf16", "M": 1024, "N": 1024,
         "K": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, m):
    return max(lo, _log(rng, lo, hi) // m * m)


def _width(rng, lo, hi):
    """An output width: mostly a multiple of 64, sometimes of 8, sometimes any."""
    return _mult(rng, lo, hi, rng.choice((64, 64, 8, 1)))


def draw(rng):
    op = rng.choice(("weights", "weights", "weights", "dual", "infer", "step", "step", "packed", "packed", "fp8",
                     "dense"))
    while True:
        c = {"op": op}
        if op == "weights":
            c["dtype"] = rng.choice(("bf16", "bf16", "bf16", "f16", "f32"))
            c.update(M=_log(rng, 1, 4096), N=_width(rng, 512, 16384), K=_mult(rng, 512, 14336, 128))
            most = 3e11 if c["dtype"] == "bf16" else 1e11
        elif op == "dual":
            c.update(dtype="bf16", M=_log(rng, 1, 2048), N=_width(rng, 512, 16384), K=_mult(rng, 512, 8192, 128))
            most = 1.5e11
        elif op == "infer":
            c["dtype"] = rng.choice(("bf16", "f16", "f32"))
            c.update(M=_log(rng, 1, 4096), N=_width(rng, 512, 8192), K=_mult(rng, 512, 8192, 128))
            most = 3e11
        elif op == "step":
            c["quantized"] = rng.choice((False, True))
            m = 128 if c["quantized"] else 1
            c.update(M=_mult(rng, 128, 8192, m), N=_mult(rng, 512, 8192, 128), K=_mult(rng, 512, 8192, 128))
            most = 1.5e11
        elif op == "packed":
            c["spelling"] = rng.choice(("fused", "reference"))
            c["dtype"] = rng.choice(("bf16", "f32"))
            c.update(M=_log(rng, 64, 8192), N=_width(rng, 256, 8192), K=_mult(rng, 512, 8192, 128))
            most = 5e11
        elif op == "fp8":
            c.update(dtype="bf16", M=_log(rng, 64, 4096), N=_mult(rng, 256, 8192, 16), K=_mult(rng, 512, 8192, 128))
            most = 1.5e11
        else:
            c["form"] = rng.choice(("gemm", "separate", "packed"))
            c["dtype"] = rng.choice(("bf16", "f16"))
            c.update(M=_log(rng, 64, 4096), N=_mult(rng, 256, 4096, 8), K=_mult(rng, 512, 8192, 64))
            most = 6e10
        if 2.0 * c["M"] * c["N"] * c["K"] <= most:
            return c


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _acts(g, M, K, dt):
    """Activations: normal, with channels of different size."""
    s = torch.exp(0.7 * torch.randn((1, K), generator=g, device="cuda"))
    return (torch.randn((M, K), generator=g, device="cuda") * s).to(dt)


def _weight(g, N, K):
    return torch.randn((N, K), generator=g, device="cuda") * (1.0 / math.sqrt(K))


def _grid(g, shape, dt):
    """Twice the E2M1 values: the integer grid of the dual-accumulator GEMMs."""
    q = torch.tensor([0, 1, 2, 3, 4, 6, 8, 12, -1, -2, -3, -4, -6, -8, -12], device="cuda", dtype=torch.float32)
    return q[torch.randint(0, 15, shape, generator=g, device="cuda")].to(dt)


def _inputs(case, seed):
    """The plain tensors that both prepare() and exact() start from."""
    g = _gen(seed)
    op, M, N, K = case["op"], case["M"], case["N"], case["K"]
    dt = _DT[case.get("dtype", "bf16")]
    if op == "weights":
        return {"a": _acts(g, M, K, dt), "w": _weight(g, N, K)}
    if op == "dual":
        return {"a0": _acts(g, M, K, dt), "a1": _acts(g, M, K, dt), "w": _weight(g, N, K)}
    if op == "infer":
        return {"a": _acts(g, M, K, dt), "w": _weight(g, N, K).to(dt)}
    if op == "step":
        return {"x": _acts(g, M, K, dt), "w": _weight(g, N, K),
                "gy": (torch.randn((M, N), generator=g, device="cuda") / math.sqrt(N)).to(dt)}
    if op == "packed":
        return {"a": _acts(g, M, K, dt), "w": _weight(g, N, K).to(dt)}
    if op == "fp8":
        return {"a": _acts(g, M, K, torch.float32), "w": _weight(g, N, K)}
    grid = case["form"] == "packed"
    mk = (lambda s: _grid(g, s, dt)) if grid else (lambda s: torch.randn(s, generator=g, device="cuda").to(dt))
    return {"a1": mk((M, K)), "b1": mk((K, N)), "a2": mk((M, K)), "b2": mk((K, N))}


def prepare(case, seed):
    t = _inputs(case, seed)
    op = case["op"]
    if op in ("weights", "dual"):
        # the weight is quantized once, when it is loaded
        t["w_pk"], t["w_scale"] = fp4.quantize_pack_mxfp4(t.pop("w"))
    elif op in ("infer", "step"):
        w = t.pop("w")
        layer = MXFP4Linear(case["K"], case["N"], quantized_backward=case.get("quantized", False))
        layer.weight = torch.nn.Parameter(w)
        t["layer"] = layer
        if op == "step":
            t["x"].requires_grad_(True)
    elif op == "fp8":
        # operands as a program holds them: E4M3 bytes, B as [K, N], fp32 scales
        a_codes, t["a_scale"] = fp4.quantize_mxfp4(t.pop("a"))
        w_codes, w_scale = fp4.quantize_mxfp4(t.pop("w"))
        t["a8"] = fp4.codes_to_e4m3(a_codes)
        t["b8"] = fp4.codes_to_e4m3(w_codes.t().contiguous())
        t["b_scale"] = w_scale.t().contiguous()
    elif op == "dense" and case["form"] == "packed":
        t["a2"] = t["a2"] * 2.0  # the second product's slot, exact in the operand type
    t["case"] = case
    return t


# ------------------------------------------------------------------ one pass
def run(t):
    case = t["case"]
    op = case["op"]
    if op == "weights":
        return mxfp4_gemm.mxfp4_linear_w(t["a"], t["w_pk"], t["w_scale"])
    if op == "dual":
        return dual_gemm.dual_mxfp4(t["a0"], t["a1"], t["w_pk"], t["w_scale"])
    if op == "infer":
        with torch.no_grad():
            return t["layer"](t["a"])
    if op == "step":
        layer, x = t["layer"], t["x"]
        x.grad = layer.weight.grad = None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = layer(x)
        y.backward(t["gy"])
        return {"y": y.detach(), "dx": x.grad, "dw": layer.weight.grad}
    if op == "packed":
        a, w = t["a"], t["w"]
        if case["spelling"] == "fused":
            (ap, asc), (wp, wsc) = fp4.quantize_pack_mxfp4_many([a, w], scale_layout="kmajor")
        else:
            ac, asc = fp4.quantize_mxfp4(a)
            wc, wsc = fp4.quantize_mxfp4(w)
            ap, wp = fp4.pack_fp4(ac), fp4.pack_fp4(wc)
        c = mxfp4_gemm.mxfp4_gemm_packed(ap, wp, asc, wsc)
        return {"a_pk": ap, "a_scale": asc, "w_pk": wp, "w_scale": wsc, "c": c}
    if op == "fp8":
        return mxfp4_gemm.mxfp4_gemm_fp8(t["a8"], t["b8"], t["a_scale"], t["b_scale"])
    if case["form"] == "gemm":
        return dual_gemm.gemm(t["a1"], t["b1"])
    f = dual_gemm.dual_separate if case["form"] == "separate" else dual_gemm.dual_packed
    return f(t["a1"], t["a2"], t["b1"], t["b2"])


# ------------------------------------------------------------------ its price
def work(case):
    """Bytes read and written once, and multiply-adds times two."""
    op, M, N, K = case["op"], case["M"], case["N"], case["K"]
    size = {"bf16": 2, "f16": 2, "f32": 4}[case.get("dtype", "bf16")]
    mx = 0.5 + 1 / 32  # a packed element and its share of an E8M0 scale
    flops = 2.0 * M * N * K
    if op == "weights":
        return {"bytes": size * M * K + mx * N * K + size * M * N, "flops": flops}
    if op == "dual":
        return {"bytes": 2 * size * M * K + mx * N * K + 2 * size * M * N, "flops": 2 * flops}
    if op == "infer":
        return {"bytes": size * (M * K + N * K + M * N), "flops": flops}
    if op == "step":  # x, w (fp32) and gy in, y, dx and dw (fp32) out
        return {"bytes": 2.0 * M * K + 4 * N * K + 2 * M * N + 2 * M * N + 2 * M * K + 4 * N * K, "flops": 3 * flops}
    if op == "packed":
        out = mx if case["spelling"] == "fused" else 0.5 + 4 / 32
        return {"bytes": (size + out) * (M + N) * K + 2 * M * N, "flops": flops}
    if op == "fp8":
        return {"bytes": (1 + 4 / 32) * (M + N) * K + 2 * M * N, "flops": flops}
    two = case["form"] != "gemm"
    outs = 2 if case["form"] == "separate" else 1
    return {"bytes": (2 if two else 1) * size * (M + N) * K + 4 * outs * M * N, "flops": flops * (2 if two else 1)}


def tolerance(case):
    """Codes and scales are compared exactly.  Products accumulate in fp32, so
    two correct orders of summation differ by about 1e-7 to 1e-6 before the
    output is rounded; the rounding of a 16-bit output decides the rest."""
    dt = "f32" if case["op"] == "dense" else case.get("dtype", "bf16")
    if case["op"] == "packed":
        dt = "bf16"  # the product's output type, whatever the operands were
    return {"bf16": {"rel": 7e-3, "max": 1.6e-2}, "f16": {"rel": 8e-4, "max": 2e-3},
            "f32": {"rel": 1e-5, "max": 1e-4}}[dt]


# ------------------------------------------------------------------ in 64 bits
def _quant64(x):
    """x quantized to MXFP4 along its last axis and taken back to float64
    values: blocks of 32, scale 2^(floor(log2(amax)) - 2) with the logarithm
    rounded to float32, elements to the nearest of {0, .5, 1, 1.5, 2, 3, 4, 6},
    ties to the smaller."""
    R, K = x.shape
    b = x.double().reshape(R, K // 32, 32)
    amax = b.abs().amax(-1, keepdim=True)
    e = torch.log2(amax.clamp_min(1e-30)).float().double().floor() - 2
    s = torch.where(amax == 0, torch.ones_like(e), torch.exp2(e.clamp(-127, 127)))
    mids = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=x.device, dtype=torch.float64)
    mags = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], device=x.device, dtype=torch.float64)
    q = b / s
    v = mags[torch.bucketize(q.abs(), mids)] * torch.sign(q)
    return (v * s).reshape(R, K)


def exact(case, seed):
    t = _inputs(case, seed)
    op = case["op"]
    if op == "weights":
        return t["a"].double() @ _quant64(t["w"]).t()
    if op == "dual":
        w = _quant64(t["w"]).t()
        return t["a0"].double() @ w, t["a1"].double() @ w
    if op == "infer":
        return _quant64(t["a"]) @ _quant64(t["w"]).t()
    if op == "step":
        x, w, gy = t["x"], t["w"], t["gy"]
        y = _quant64(x) @ _quant64(w).t()
        if case["quantized"]:
            dx = _quant64(gy) @ _quant64(w.t().contiguous()).t()
            dw = _quant64(gy.t().contiguous()) @ _quant64(x.t().contiguous()).t()
        else:
            dx = gy.double() @ w.to(gy.dtype).double()
            dw = gy.double().t() @ x.double()
        return {"y": y, "dx": dx, "dw": dw}
    if op == "packed":
        return {"a_pk": None, "a_scale": None, "w_pk": None, "w_scale": None,
                "c": _quant64(t["a"]) @ _quant64(t["w"]).t()}
    if op == "fp8":
        return _quant64(t["a"]) @ _quant64(t["w"]).t()
    c1 = t["a1"].double() @ t["b1"].double()
    if case["form"] == "gemm":
        return c1
    if case["form"] == "separate":
        return c1, t["a2"].double() @ t["b2"].double()
    return c1 + (2.0 * t["a2"].double()) @ t["b2"].double()
