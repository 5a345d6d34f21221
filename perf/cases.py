"""The work of the post-training-quantization path that its speed is judged by.

Seven kinds of work, each through the public entry points of
``tokenvector.inference_amd`` (device buffers are torch tensors here, handed
over by address, as a program that shares memory with the library does):

  linear     ``QuantizedLinear.forward``: the activation's calibrate +
             quantize, the GEMM and the dequant + bias epilogue.  Weight
             formats INT8, FP8 (reference products), FP8 full rate and GGUF
             Q8_0; activations per tensor or per token; 1 to 32 rows is
             decoding, more is prefill.
  layer      the four INT8 linears of one transformer block in turn, the unit
             that a forward pass repeats.
  int4       the grouped-INT4 GEMM on f32 activations, decoding and prefill,
             with and without the act-order column permutation.
  qlinear    QLinearMatMul on int8 codes: int8 in, int8 out, zero points.
  node       the QuantizedGemm graph node on host lists of int32 codes, the
             call that the graph runtime makes.
  calibrate  the per-tensor calibrators on an activation tensor.
  quantize   the streaming quantizers of activations and weights.

Layer sizes are the GPT-2-124M linears (768, 2304, 3072) that the benchmark
runs and other sizes between 256 and 4096, output widths odd ones among them;
rows go from 1 to 32768.
"""
import math

import numpy as np
import torch

from tokenvector.inference_amd import device as D
from tokenvector.inference_amd import session as S

# qkv, attn_out, mlp_up, mlp_down of one block: (N, K)
BLOCK = ((2304, 768), (768, 768), (3072, 768), (768, 3072))

_CTX = None


def _ctx():
    """One context for the program, as its stream and workspaces are meant."""
    global _CTX
    if _CTX is None:
        _CTX = D.Context(0)
    return _CTX


def listed():
    return [
        # one token through the widest attention projection: the smallest call
        {"name": "decode-int8-m1", "kind": "linear", "fmt": "int8", "act": "token",
         "m": 1, "n": 2304, "k": 768},
        # a decode batch on 4-bit weights, the long reduction of the MLP
        {"name": "decode-int4-m32", "kind": "int4", "m": 32, "n": 768, "k": 3072, "gs": 128,
         "perm": False},
        # a small decode batch on GGUF Q8_0 weights
        {"name": "decode-q8-m8", "kind": "linear", "fmt": "q8_0", "act": "token",
         "m": 8, "n": 3072, "k": 768},
        # the benchmark's unit: one block's linears at 8 x 1024 tokens
        {"name": "prefill-int8-layer", "kind": "layer", "act": "tensor", "m": 8192},
        # the largest: 32 x 1024 tokens through the MLP's first linear, full-rate FP8
        {"name": "prefill-fp8-m32768", "kind": "linear", "fmt": "fp8_fast", "act": "tensor",
         "m": 32768, "n": 3072, "k": 768},
        # the drop-in FP8 (the reference decoder's products) on a 2048-token prompt
        {"name": "prefill-fp8ref-m2048", "kind": "linear", "fmt": "fp8", "act": "tensor",
         "m": 2048, "n": 768, "k": 3072},
        # Q8_0 weights on a prompt of an odd length
        {"name": "prefill-q8-m1531", "kind": "linear", "fmt": "q8_0", "act": "token",
         "m": 1531, "n": 3072, "k": 768},
        # 4-bit weights on a 2048-token prompt
        {"name": "prefill-int4-m2048", "kind": "int4", "m": 2048, "n": 2304, "k": 768, "gs": 128,
         "perm": False},
        # the quantized-operator model: int8 in and out, an odd number of rows
        {"name": "qlinear-m3001", "kind": "qlinear", "m": 3001, "n": 768, "k": 3072},
        # the graph runtime's own call on host lists
        {"name": "node-m256", "kind": "node", "m": 256, "n": 2304, "k": 768},
        # a calibration set's activation through every calibrator
        {"name": "calibrate-m8192", "kind": "calibrate", "how": "all", "rows": 8192, "cols": 768},
        # the quantize stream at the largest activation
        {"name": "quantize-m65536", "kind": "quantize", "how": "row", "rows": 65536, "cols": 768},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _nk(rng):
    """Half of the time one of the block's linears, else other sizes of that range."""
    if rng.random() < 0.5:
        return rng.choice(BLOCK)
    return _log(rng, 256, 4096), 128 * _log(rng, 2, 32)


def _rows(rng, lo, hi, n, k, most):
    """Rows between lo and hi, as many as `most` multiply-adds allow."""
    return _log(rng, lo, max(lo, min(hi, int(most // (n * k)))))


def draw(rng):
    most = 32768.0 * 3072 * 768
    kind = rng.choice(("decode", "decode", "linear", "linear", "layer", "int4", "int4", "qlinear",
                       "node", "calibrate", "quantize"))
    if kind == "decode":
        n, k = _nk(rng)
        m = rng.randint(1, 32)
        how = rng.choice(("int8", "q8_0", "int4"))
        if how == "int4":
            return {"kind": "int4", "m": m, "n": n, "k": k, "gs": rng.choice((32, 64, 128)),
                    "perm": False}
        return {"kind": "linear", "fmt": how, "act": "token", "m": m, "n": n, "k": k}
    if kind == "linear":
        n, k = _nk(rng)
        fmt = rng.choice(("int8", "fp8", "fp8_fast", "q8_0"))
        act = "tensor" if fmt.startswith("fp8") else rng.choice(("tensor", "token"))
        return {"kind": "linear", "fmt": fmt, "act": act,
                "m": _rows(rng, 33, 32768, n, k, most / 2), "n": n, "k": k}
    if kind == "layer":
        return {"kind": "layer", "act": rng.choice(("tensor", "token")), "m": _log(rng, 1, 10240)}
    if kind == "int4":
        n, k = _nk(rng)
        return {"kind": "int4", "m": _rows(rng, 33, 8192, n, k, most / 4), "n": n, "k": k,
                "gs": rng.choice((32, 64, 128, 128)), "perm": rng.random() < 0.25}
    if kind == "qlinear":
        n, k = _nk(rng)
        return {"kind": "qlinear", "m": _rows(rng, 33, 16384, n, k, most / 2), "n": n, "k": k}
    if kind == "node":
        n, k = _nk(rng)
        return {"kind": "node", "m": _rows(rng, 16, 1024, n, k, 2.0e9), "n": n, "k": k}
    if kind == "calibrate":
        return {"kind": "calibrate", "how": rng.choice(("minmax", "kl", "percentile", "mse", "all")),
                "rows": _log(rng, 64, 16384), "cols": rng.choice((768, 3072, _log(rng, 256, 4096)))}
    how = rng.choice(("row", "tensor", "channel", "fp8", "int4"))
    cols = rng.choice((768, 3072)) if rng.random() < 0.5 else 128 * _log(rng, 2, 32)
    rows = _log(rng, 256, 4096) if how in ("channel", "int4") else _log(rng, 64, 16384)
    return {"kind": "quantize", "how": how, "rows": rows, "cols": cols}


# ---- inputs ---------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _acts(g, rows, cols):
    """Activations: Gaussian, channels of different gains, a few of them
    outliers, as the inputs of a transformer's linears have."""
    gain = torch.exp(0.25 * torch.randn(cols, generator=g, device="cuda"))
    gain = torch.where(torch.rand(cols, generator=g, device="cuda") < 0.005, gain * 10.0, gain)
    return torch.randn(rows, cols, generator=g, device="cuda") * gain


def _weights(g, n, k):
    return torch.randn(n, k, generator=g, device="cuda") * 0.02


def _bias(g, n):
    return torch.randn(n, generator=g, device="cuda") * 0.01


def _q8_blocks(w):
    """GGUF Q8_0 blocks of w: per 32 weights an f16 d and 32 int8 codes."""
    n, k = w.shape
    b = w.view(n, k // 32, 32)
    d = (b.abs().amax(-1) / 127.0).half()
    q = torch.clamp(torch.round(b / d.float().clamp_min(1e-8)[..., None]), -127, 127).to(torch.int8)
    raw = torch.cat([d[..., None].view(torch.uint8).reshape(n, k // 32, 2), q.view(torch.uint8)], -1)
    return raw.contiguous(), d, q


def _int4_pack(w, gs):
    """Grouped INT4: packed bytes (low nibble = even column), scales, codes."""
    n, k = w.shape
    b = w.view(n, k // gs, gs)
    sc = (b.abs().amax(-1).double().clamp_min(1e-8) / 7.0).float()
    q = torch.clamp(torch.round(b.double() * (1.0 / sc.double())[..., None]), -8, 7).to(torch.int64)
    q = q.view(n, k)
    packed = ((q[:, 0::2] + 8) | ((q[:, 1::2] + 8) << 4)).to(torch.uint8).contiguous()
    return packed, sc, q


_FMT = {"int8": D.WEIGHT_INT8, "fp8": D.WEIGHT_FP8, "fp8_fast": D.WEIGHT_FP8_FAST}
_ACT = {"tensor": D.ACT_PER_TENSOR, "token": D.ACT_PER_TOKEN}


def _linear_inputs(seed, m, n, k):
    g = _gen(seed)
    return _acts(g, m, k), _weights(g, n, k), _bias(g, n)


def _linear(x, w, b, fmt):
    (m, k), n = x.shape, w.shape[0]
    if fmt == "q8_0":
        raw = _q8_blocks(w)[0]
        torch.cuda.synchronize()
        lin = D.QuantizedLinear.from_gguf_q8_0(_ctx(), raw.data_ptr(), n, k, b.data_ptr())
    else:
        torch.cuda.synchronize()
        lin = D.QuantizedLinear.from_float(_ctx(), w.data_ptr(), n, k, b.data_ptr(), _FMT[fmt])
    return {"x": x, "m": m, "lin": lin, "y": torch.empty(m, n, device="cuda")}


def _params():
    return torch.zeros(8, dtype=torch.int32, device="cuda")


def _qlinear_inputs(case, seed):
    m, n, k = case["m"], case["n"], case["k"]
    g = _gen(seed)
    a = torch.clamp(torch.round(_acts(g, m, k) * 25.0) - 3, -128, 127).to(torch.int8)
    w = torch.clamp(torch.round(torch.randn(n, k, generator=g, device="cuda") * 32.0), -127, 127)
    # an output scale that puts most outputs inside the int8 range
    sy = float(np.float32(math.sqrt(k) * 32.0 * 32.0 * 0.02 * 0.003 / 40.0))
    return a, w.to(torch.int8), sy


def _node_inputs(case, seed):
    m, n, k = case["m"], case["n"], case["k"]
    r = np.random.default_rng(seed)
    a = np.clip(np.rint(r.standard_normal(m * k, np.float32) * 30.0), -127, 127).astype(np.int32)
    w = np.clip(np.rint(r.standard_normal(n * k, np.float32) * 32.0), -127, 127).astype(np.int32)
    bias = r.standard_normal(n, np.float32) * np.float32(0.01)
    scales = (r.random(n, np.float32) * np.float32(1e-4) + np.float32(6e-4)).astype(np.float32)
    return a, w, bias, scales, np.float32(0.031)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": dict(case), "ctx": _ctx()}
    if kind == "linear":
        s.update(_linear(*_linear_inputs(seed, case["m"], case["n"], case["k"]), case["fmt"]))
        s["act"] = _ACT[case["act"]]
    elif kind == "layer":
        s["linears"] = [_linear(*_linear_inputs(seed * 4 + i, case["m"], n, k), "int8")
                        for i, (n, k) in enumerate(BLOCK)]
        s["act"] = _ACT[case["act"]]
    elif kind == "int4":
        m, n, k = case["m"], case["n"], case["k"]
        s["x"], w, s["bias"] = _linear_inputs(seed, m, n, k)
        s["packed"], s["scales"], _ = _int4_pack(w, case["gs"])
        s["perm"] = torch.randperm(k, generator=_gen(seed + 1), device="cuda") if case["perm"] else None
        s["y"] = torch.empty(m, n, device="cuda")
    elif kind == "qlinear":
        s["a"], s["w"], s["sy"] = _qlinear_inputs(case, seed)
        s["y"] = torch.empty(case["m"], case["n"], dtype=torch.int8, device="cuda")
    elif kind == "node":
        s["a"], s["w"], s["bias"], scales, sa = _node_inputs(case, seed)
        s["node"] = S.new_node("linear", S.OperatorType_QuantizedGemm)
        s["node"].scale_a, s["node"].scales_w = sa, scales
    elif kind == "calibrate":
        s["x"] = _acts(_gen(seed), case["rows"], case["cols"])
        s["p"] = {h: _params() for h in _calibrators(case["how"])}
    else:
        rows, cols, how = case["rows"], case["cols"], case["how"]
        g = _gen(seed)
        s["x"] = _weights(g, rows, cols) if how in ("channel", "int4") else _acts(g, rows, cols)
        s["p"] = _params()
        if how == "int4":
            s["q"] = torch.empty(rows, cols // 2, dtype=torch.uint8, device="cuda")
            s["scales"] = torch.empty(rows, cols // 128, device="cuda")
        else:
            s["q"] = torch.empty(rows, cols, dtype=torch.uint8 if how == "fp8" else torch.int8,
                                 device="cuda")
            s["scales"] = torch.empty(rows, device="cuda")
    torch.cuda.synchronize()  # the library's stream starts after torch's
    return s


def _calibrators(how):
    return ("minmax", "kl", "percentile", "mse") if how == "all" else (how,)


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "linear":
        s["lin"].forward(s["x"].data_ptr(), s["m"], s["y"].data_ptr(), s["act"])
        return s["y"]
    if kind == "layer":
        for t in s["linears"]:
            t["lin"].forward(t["x"].data_ptr(), t["m"], t["y"].data_ptr(), s["act"])
        return [t["y"] for t in s["linears"]]
    if kind == "int4":
        perm = s["perm"].data_ptr() if s["perm"] is not None else None
        D.matmul_int4_grouped(ctx, s["x"].data_ptr(), s["packed"].data_ptr(), s["scales"].data_ptr(),
                              s["bias"].data_ptr(), perm, s["y"].data_ptr(), case["m"], case["n"],
                              case["k"], case["gs"])
        return s["y"]
    if kind == "qlinear":
        D.qlinear_matmul(ctx, s["a"].data_ptr(), 0.02, -3, s["w"].data_ptr(), 0.003, 0, s["sy"], 7,
                         s["y"].data_ptr(), case["m"], case["n"], case["k"])
        return s["y"]
    if kind == "node":
        m, n, k = case["m"], case["n"], case["k"]
        return s["node"].execute([(s["a"], (m, k)), (s["w"], (n, k)), (s["bias"], (n,))], [(m, n)])[0]
    n = case["rows"] * case["cols"]
    if kind == "calibrate":
        for how, p in s["p"].items():
            if how == "minmax":
                D.calibrate_minmax(ctx, s["x"].data_ptr(), n, 1, p.data_ptr())
            elif how == "kl":
                D.calibrate_kl(ctx, s["x"].data_ptr(), n, p.data_ptr())
            elif how == "percentile":
                D.calibrate_percentile(ctx, s["x"].data_ptr(), n, p.data_ptr())
            else:
                D.calibrate_mse(ctx, s["x"].data_ptr(), n, p.data_ptr())
        return {h: {"range": p.view(torch.float32)[:3], "zero_point": p[3:4]}
                for h, p in s["p"].items()}
    how, x, q, sc = case["how"], s["x"].data_ptr(), s["q"].data_ptr(), s["scales"].data_ptr()
    if how == "row":
        D.quantize_dynamic_int8_rowwise(ctx, x, case["rows"], case["cols"], q, sc)
        return {"codes": s["q"], "scales": s["scales"]}
    if how == "channel":
        D.calibrate_rows(ctx, x, case["rows"], case["cols"], sc)
        D.quantize_int8_per_channel(ctx, x, case["rows"], case["cols"], sc, q)
        return {"codes": s["q"], "scales": s["scales"]}
    if how == "int4":
        D.quantize_int4_grouped(ctx, x, case["rows"], case["cols"], 128, q, sc)
        return {"codes": s["q"], "scales": s["scales"]}
    if how == "tensor":
        D.quantize_int8_dynamic_tensor(ctx, x, n, q, s["p"].data_ptr())
    else:
        D.quantize_fp8_e4m3_dynamic_tensor(ctx, x, n, q, s["p"].data_ptr())
    return {"codes": s["q"], "scale": s["p"].view(torch.float32)[:1]}


# ---- what a pass cannot do without -----------------------------------------

def _linear_work(m, n, k, weight_bytes):
    return {"bytes": 4 * m * k + weight_bytes + 8 * n + 4 * m * n, "flops": 2 * m * n * k}


def work(case):
    kind = case["kind"]
    if kind == "layer":
        parts = [_linear_work(case["m"], n, k, n * k) for n, k in BLOCK]
        return {u: sum(p[u] for p in parts) for u in ("bytes", "flops")}
    if kind in ("linear", "int4", "qlinear", "node"):
        m, n, k = case["m"], case["n"], case["k"]
        if kind == "linear":
            return _linear_work(m, n, k, n * k // 32 * 34 if case["fmt"] == "q8_0" else n * k)
        if kind == "int4":
            w = _linear_work(m, n, k, n * k // 2 + 4 * n * k // case["gs"])
            return {"bytes": w["bytes"] - 4 * n + (8 * k if case["perm"] else 0), "flops": w["flops"]}
        if kind == "qlinear":
            return {"bytes": m * k + n * k + m * n, "flops": 2 * m * n * k}
        return {"bytes": 4 * (m * k + n * k + m * n + 2 * n), "flops": 2 * m * n * k}
    n = case["rows"] * case["cols"]
    if kind == "calibrate":  # x is in hand once for each calibrator that is asked for
        return {"bytes": 4 * n * len(_calibrators(case["how"])), "flops": 0}
    codes = n // 2 if case["how"] == "int4" else n
    scales = 4 * n // 128 if case["how"] == "int4" else 4 * case["rows"]
    return {"bytes": 4 * n + codes + (scales if case["how"] in ("row", "channel", "int4") else 4),
            "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind in ("qlinear", "quantize", "calibrate"):
        return "exact"  # codes, and scales formed by one f64 division rounded to f32
    if kind == "linear" and case["fmt"] == "fp8_fast":
        return {"rel": 1e-4, "max": 1e-3}  # the FP8 matrix unit's own accumulation
    if kind == "linear" and case["fmt"] in ("fp8", "q8_0"):
        return {"rel": 6e-7, "max": 6e-6}  # f32 sums over K
    return {"rel": 1e-7, "max": 6e-7}      # exact sums, one rounding to f32


# ---- the same in 64 bits ----------------------------------------------------

def _sym_codes(x, scale):
    """int8 codes of x for an f32 scale whose f32 reciprocal multiplies."""
    inv = (torch.ones_like(scale) / scale).double()
    return torch.clamp(torch.round(x.double() * inv), -127, 127)


def _e4m3(v, reference_decode):
    """Values of the e4m3 codes of v (|v| <= 240): nearest even, a subnormal
    that would round up to the first normal staying the last subnormal; the
    reference decoder reads subnormal codes at half their value."""
    c = torch.where(v.abs() < 2.0 ** -6, torch.clamp(v, -7 * 2.0 ** -9, 7 * 2.0 ** -9), v)
    d = c.to(torch.float8_e4m3fn).double()
    return torch.where(d.abs() < 2.0 ** -6, d / 2, d) if reference_decode else d


def _fp8_scale(x, dim=None):
    am = x.abs().amax() if dim is None else x.abs().amax(dim)
    return (am.double().clamp_min(1e-8) / 240.0).float()


def _exact_linear(x, w, b, fmt, act):
    if fmt.startswith("fp8"):
        sa, sw = _fp8_scale(x), _fp8_scale(w, 1)
        a = _e4m3(x * (1.0 / sa), fmt == "fp8")
        c = _e4m3(w * (1.0 / sw)[:, None], fmt == "fp8")
        return (a @ c.t()) * sa.double() * sw.double() + b.double()
    if act == "token":
        am = x.abs().amax(1).double().clamp_min(1e-8) / 127.0
        a, sa = torch.clamp(torch.round(x.double() * (1.0 / am)[:, None]), -127, 127), am.float().double()[:, None]
    else:
        s = (x.abs().amax().double().clamp_min(1e-8) / 127.0).float()
        a, sa = _sym_codes(x, s), s.double()
    if fmt == "q8_0":
        _, d, q = _q8_blocks(w)
        return (a @ (q.double() * d.double()[..., None]).view(w.shape).t()) * sa + b.double()
    sw = (w.abs().amax(1).double().clamp_min(1e-8) / 127.0).float().double()
    c = torch.clamp(torch.round(w.double() * (1.0 / sw.clamp_min(1e-8))[:, None]), -127, 127)
    return (a @ c.t()) * sa * sw + b.double()


def _range(thr):
    return {"range": torch.tensor([thr / 127.0, -thr, thr], dtype=torch.float64), "zero_point": None}


def _exact_kl(x, bins=2048, target=128):
    bw = float(x.abs().max()) / bins
    b = torch.clamp((x.double().abs() / bw).long(), max=bins - 1).reshape(-1)
    hist = torch.bincount(b, minlength=bins).cpu().numpy().astype(np.float64)
    best, best_kl = bins, 1e45
    for th in range(target, bins + 1, 16):
        p = hist[:th].copy()
        p[th - 1] += hist[th:].sum()
        p /= hist.sum()
        per = th // target
        edge = [i * per for i in range(target)] + [th]
        q = np.concatenate([np.full(edge[i + 1] - edge[i], p[edge[i]:edge[i + 1]].sum() / (edge[i + 1] - edge[i]))
                            for i in range(target)])
        ok = (p > 1e-12) & (q > 1e-12)
        kl = float(np.sum(p[ok] * np.log(p[ok] / q[ok])))
        if kl < best_kl:
            best, best_kl = th, kl
    return best * bw


def _exact_mse(x, candidates=50):
    am = float(x.abs().max())
    best, best_mse = am, 1e45
    parts = x.reshape(-1).split(1 << 24)
    for c in range(1, candidates + 1):
        thr = am * c / candidates
        scale = thr / 127.0
        mse = 0.0
        for p in parts:
            d = p.double()
            q = torch.clamp(torch.round(torch.clamp(d, -thr, thr) * (1.0 / scale)), -127, 127)
            mse += float(((d - q * scale) ** 2).sum())
        if mse < best_mse:
            best, best_mse = thr, mse
    return best


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, w, b = _linear_inputs(seed, case["m"], case["n"], case["k"])
        return _exact_linear(x, w, b, case["fmt"], case["act"])
    if kind == "layer":
        return [_exact_linear(*_linear_inputs(seed * 4 + i, case["m"], n, k), "int8", case["act"])
                for i, (n, k) in enumerate(BLOCK)]
    if kind == "int4":
        x, w, b = _linear_inputs(seed, case["m"], case["n"], case["k"])
        _, sc, q = _int4_pack(w, case["gs"])
        if case["perm"]:
            x = x[:, torch.randperm(case["k"], generator=_gen(seed + 1), device="cuda")]
        wd = q.double() * sc.double().repeat_interleave(case["gs"], 1)
        return x.double() @ wd.t() + b.double()
    if kind == "node":
        a, w, bias, scales, sa = _node_inputs(case, seed)
        m, n, k = case["m"], case["n"], case["k"]
        acc = a.reshape(m, k).astype(np.float64) @ w.reshape(n, k).astype(np.float64).T
        return acc * float(sa) * scales.astype(np.float64) + bias.astype(np.float64)
    if kind == "calibrate":
        x, out = _acts(_gen(seed), case["rows"], case["cols"]), {}
        for how in _calibrators(case["how"]):
            if how == "minmax":
                out[how] = _range(max(float(x.abs().max()), 1e-8))
            elif how == "kl":
                out[how] = _range(_exact_kl(x))
            elif how == "percentile":
                a = x.abs().reshape(-1)
                i = int(min(a.numel() - 1, float(np.float32(99.99)) / 100.0 * a.numel()))
                out[how] = _range(max(float(a.sort().values[i]), 1e-8))
            else:
                out[how] = _range(_exact_mse(x))
        return out
    if kind == "quantize":
        rows, cols, how = case["rows"], case["cols"], case["how"]
        g = _gen(seed)
        x = _weights(g, rows, cols) if how in ("channel", "int4") else _acts(g, rows, cols)
        if how == "int4":
            am = x.view(rows, cols // 128, 128).abs().amax(-1)
            return {"codes": None, "scales": am.double().clamp_min(1e-8) / 7.0}
        if how in ("row", "channel"):
            return {"codes": None, "scales": x.abs().amax(1).double().clamp_min(1e-8) / 127.0}
        return {"codes": None, "scale": (x.abs().amax().double().clamp_min(1e-8)
                                         / (240.0 if how == "fp8" else 127.0)).reshape(1)}
    return None  # qlinear: whole numbers
