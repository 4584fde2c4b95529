"""The workloads this library is timed on, through its public entry points.

A case is a plain dict. `op` says what a pass does:

  gemm   C = alpha*A*B + beta*C of one operand kind, by itself or with the fused steps of a layer (bias, activation, an
         8-bit copy of the result in place of C); `count` of them one after another, on operands of their own
  f4     E4M3 activations times 4-bit weights (`scaled`: with one E8M0 scale per 32 values)
  k4     int8 product on the K-packed weights of the dot-product entry point
  packed pack A and B into panels of 64, multiply the panels, unpack C
  cvt    quantise an array to OCP fp8 (saturating, scaled) and read it back as bf16

`layout` of a gemm: "nn" A and B row-major, "nt" A row-major and B with K contiguous (a linear layer's [out][in] weight),
"tn" A column-major and B row-major.
"""
import math

import torch

import skl_amd
from skl_amd import Epilogue

_TORCH = {"i8": torch.int8, "bf16": torch.bfloat16, "f16": torch.float16, "e4m3": torch.uint8, "e5m2": torch.uint8, "f32": torch.float32}
_NAME = {"i8": "i8", "bf16": "bf16", "f16": "f16", "e4m3": "f8e4m3", "e5m2": "f8e5m2", "f32": "f32"}
_ACT = {"none": Epilogue.ACT_NONE, "relu": Epilogue.ACT_RELU, "silu": Epilogue.ACT_SILU, "gelu": Epilogue.ACT_GELU}
_FP8_EXACT_MAX_K = 2304  # longer fp8 products run on the fp8 matrix-core instructions


def _gemm(name, kind, layout, m, n, k, beta=0, bias=False, act="none", out="c", count=1):
    return {"name": name, "op": "gemm", "count": count, "kind": kind, "layout": layout, "m": m, "n": n, "k": k, "beta": beta, "bias": bias, "act": act, "out": out}


def listed():
    return [
        # The smallest calls: products of the size of SKL's vector kernels' benchmarks, four in a row as the heads or
        # experts of a layer are. Latency and launches.
        _gemm("bf16 four 64x128x128", "bf16", "nn", 64, 128, 128, count=4),
        # A small square product, too small to fill the chip.
        _gemm("i8 512^3", "i8", "nn", 512, 512, 512),
        # One token through a quantised layer: a stream over the weights.
        _gemm("i8 decode 1x4096x11008", "i8", "nn", 1, 11008, 4096),
        # A decode batch through a bf16 linear layer (weights [out][in]) with bias and activation.
        _gemm("bf16 decode 16x4096x11008 silu", "bf16", "nt", 16, 11008, 4096, bias=True, act="silu"),
        # The same with 4-bit block-scaled weights.
        {"name": "mxfp4 decode 16x4096x11008", "op": "f4", "scaled": True, "m": 16, "n": 11008, "k": 4096},
        # An ordinary dense product accumulating into C.
        _gemm("bf16 2048x4096x4096 accum", "bf16", "nn", 2048, 4096, 4096, beta=1),
        # No size a multiple of a tile.
        _gemm("bf16 3000x5000x7000", "bf16", "nn", 3000, 5000, 7000),
        # Prefill through an fp8 layer that feeds the next fp8 layer: bias, activation, E4M3 output only.
        _gemm("e4m3 layer 2048x2048x8192", "e4m3", "nt", 2048, 8192, 2048, bias=True, act="gelu", out="q8"),
        # The largest product: fp8, column-major A as SKL's matrix kernels take it.
        _gemm("e4m3 8192^3", "e4m3", "tn", 8192, 8192, 8192),
        # The packed path end to end.
        {"name": "f16 packed 4096x4096x14336", "op": "packed", "kind": "f16", "m": 4096, "n": 14336, "k": 4096},
        # Quantisation of a large tensor and the way back.
        {"name": "cvt f32 e4m3 8192x8192", "op": "cvt", "src": "f32", "fmt": "e4m3", "count": 1 << 26},
        # Single precision, every sum in the order of SKL's loops.
        _gemm("f32 2048^3", "f32", "nn", 2048, 2048, 2048),
    ]


_MOST_FLOPS = 2 * 4096 * 4096 * 8192  # so that no drawn product takes longer than the largest listed one


def _size(rng, low, high):
    """Log-uniform in [low, high]; two of three whole multiples of 64 (or 16, below 128), the others as they fall."""
    v = round(math.exp(rng.uniform(math.log(low), math.log(high))))
    if rng.random() < 2 / 3:
        step = 64 if v >= 128 else 16 if v >= 16 else 1
        v = max(step, v // step * step)
    return min(max(v, low), high)


def _draw_steps(rng, kind):
    """The fused steps of a layer."""
    act = rng.choice(("none", "relu") if kind == "i8" else ("none", "relu", "silu", "gelu"))
    return {"bias": True, "act": act, "out": rng.choice(("c", "q8"))}


def draw(rng):
    family = rng.choice(("small", "decode", "decode", "f4", "k4", "gemm", "gemm", "layer", "layer", "packed", "cvt", "f32"))
    if family == "f4":
        return {"op": "f4", "scaled": rng.random() < 0.5, "m": round(math.exp(rng.uniform(0, math.log(512)))),
                "n": _size(rng, 1024, 16384), "k": 32 * rng.randint(32, 448)}
    if family == "k4":
        return {"op": "k4", "m": round(math.exp(rng.uniform(0, math.log(512)))), "n": _size(rng, 128, 16384), "k": 4 * _size(rng, 64, 3584)}
    if family == "packed":
        return {"op": "packed", "kind": rng.choice(("i8", "bf16", "f16", "e4m3")), "m": _size(rng, 128, 4096), "n": _size(rng, 128, 14336), "k": _size(rng, 128, 4096)}
    if family == "cvt":
        return {"op": "cvt", "src": rng.choice(("f32", "bf16")), "fmt": rng.choice(("e4m3", "e5m2")), "count": _size(rng, 1 << 16, 1 << 26)}
    if family == "f32":
        return {"op": "gemm", "count": 1, "kind": "f32", "layout": rng.choice(("nn", "nt", "tn")), "m": _size(rng, 64, 2048), "n": _size(rng, 64, 2048),
                "k": _size(rng, 64, 2048), "beta": rng.randint(0, 1), "bias": False, "act": "none", "out": "c"}
    kind = rng.choice(("i8", "bf16", "f16", "e4m3", "e5m2"))
    c = {"op": "gemm", "kind": kind, "layout": rng.choice(("nn", "nt", "tn")), "count": 1, "beta": 0, "bias": False, "act": "none", "out": "c"}
    if family == "small":
        c.update(count=4, m=_size(rng, 16, 1024), n=_size(rng, 64, 1024), k=_size(rng, 64, 2048), beta=rng.randint(0, 1))
    elif family == "decode":
        c.update(layout=rng.choice(("nn", "nt")), m=round(math.exp(rng.uniform(0, math.log(128)))), n=_size(rng, 1024, 16384), k=_size(rng, 1024, 14336))
        if rng.random() < 0.5:
            c.update(_draw_steps(rng, kind))
    else:
        while True:
            m, n, k = _size(rng, 128, 8192), _size(rng, 512, 16384), _size(rng, 512, 14336)
            if 2 * m * n * k <= _MOST_FLOPS:
                break
        c.update(m=m, n=n, k=k)
        if family == "layer":
            c.update(layout="nt", **_draw_steps(rng, kind))
        else:
            c.update(beta=rng.randint(0, 1))
    return c


_ready = None


def _library():
    """The library, bound to torch's stream; every buffer is device memory, so no pointer needs to be looked up."""
    global _ready
    if _ready is None:
        lib = skl_amd.load()
        if lib.skl_hip_init(torch.cuda.current_device()) != 0:
            skl_amd.check_error()
        lib.skl_hip_set_pointer_mode(1)
        lib.skl_hip_set_stream(torch.cuda.current_stream().cuda_stream)
        _ready = lib
    return _ready


def _normal(gen, shape, scale=1.0):
    return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, scale, generator=gen)


def _to_fp8(lib, x, fmt):
    q = torch.empty(x.shape, dtype=torch.uint8, device="cuda")
    getattr(lib, f"skl_cvt_sat_f32_{_NAME[fmt]}_gfx950")(q.data_ptr(), x.data_ptr(), 1.0, x.numel())
    return q


def _operand(lib, gen, kind, shape, weight):
    """int8 uniform; bf16 N(0, 1) activations and N(0, 0.02^2) weights; f16 U(-1, 1); fp8 and f32 N(0, 1)."""
    if kind == "i8":
        return torch.randint(-128, 128, shape, dtype=torch.int8, device="cuda", generator=gen)
    if kind == "f16":
        return torch.empty(shape, dtype=torch.float32, device="cuda").uniform_(-1.0, 1.0, generator=gen).half()
    x = _normal(gen, shape, 0.02 if kind == "bf16" and weight else 1.0)
    if kind in ("e4m3", "e5m2"):
        return _to_fp8(lib, x, kind)
    return x.to(_TORCH[kind])


def _output(gen, kind, m, n, beta):
    dtype = torch.int32 if kind == "i8" else torch.float32
    if not beta:
        return torch.empty((m, n), dtype=dtype, device="cuda")
    return torch.randint(-1000, 1000, (m, n), dtype=dtype, device="cuda", generator=gen) if kind == "i8" else _normal(gen, (m, n))


def _prepare_gemm(lib, gen, case):
    if case["count"] > 1:
        each = [_prepare_gemm(lib, gen, dict(case, count=1)) for _ in range(case["count"])]
        return {"calls": sum((e["calls"] for e in each), []), "out": [e["out"] for e in each], "keep": each}
    m, n, k, kind = case["m"], case["n"], case["k"], case["kind"]
    a = _operand(lib, gen, kind, (k, m) if case["layout"] == "tn" else (m, k), False)
    b = _operand(lib, gen, kind, (n, k) if case["layout"] == "nt" else (k, n), True)
    rsa, csa = (1, m) if case["layout"] == "tn" else (k, 1)
    rsb, csb = (1, k) if case["layout"] == "nt" else (n, 1)
    scalar = int if kind == "i8" else float
    fused = case["bias"] or case["act"] != "none" or case["out"] == "q8"
    q8 = case["out"] == "q8"
    keep, ep = [a, b], ()
    if fused:
        # the accumulated products' spread, which an int8 layer's bias and scales are made for
        spread = math.sqrt(k) * {"i8": 5461.0, "bf16": 0.02, "f16": 1 / 3}.get(kind, 1.0)
        bias = _normal(gen, (n,), spread if kind == "i8" else 1.0)
        bias = bias.to(torch.int32) if kind == "i8" else bias
        out = torch.empty((m, n), dtype=torch.int8 if kind == "i8" else torch.uint8, device="cuda") if q8 else None
        scales = torch.empty((n,), device="cuda").uniform_(0.5, 1.5, generator=gen) * ((40.0 if kind == "i8" else 1.0) / spread) if q8 else None
        fmt = Epilogue.Q_INT8 if kind == "i8" else Epilogue.Q_F8E4M3_SAT
        ep = (Epilogue(bias=bias.data_ptr(), activation=_ACT[case["act"]], q=out.data_ptr() if q8 else None, rsq=n, csq=1,
                       q_scale=scales.data_ptr() if q8 else None, q_scale_per_column=True, q_only=q8, q_format=fmt),)
        keep += [bias, scales]
    if not fused or not q8:
        out = _output(gen, kind, m, n, case["beta"])
    c = torch.empty((4,), dtype=torch.int32, device="cuda") if q8 else out  # not touched by a call that writes only the copy
    keep.append(c)
    t, acc = _NAME[kind], "i32" if kind == "i8" else "f32"
    alpha, beta = scalar(1), scalar(case["beta"])
    if fused:
        entry = getattr(lib, f"skl_gemm_fused_{t}rc_{t}rc_{acc}rc_gfx950")
        args = (m, n, k, alpha, a.data_ptr(), rsa, csa, b.data_ptr(), rsb, csb, beta, c.data_ptr(), n, 1) + ep
    elif case["layout"] == "nn" and kind not in ("e4m3", "e5m2"):
        entry = getattr(lib, f"skl_gemm_{t}_{t}_{acc}_gfx950")
        args = (m, n, k, alpha, a.data_ptr(), k, b.data_ptr(), n, beta, c.data_ptr(), n)
    elif case["layout"] == "tn":
        entry = getattr(lib, f"skl_gemm_{t}c_{t}_{acc}_gfx950")
        args = (m, n, k, alpha, a.data_ptr(), m, b.data_ptr(), n, beta, c.data_ptr(), n)
    else:
        entry = getattr(lib, f"skl_gemm_{t}rc_{t}rc_{acc}rc_gfx950")
        args = (m, n, k, alpha, a.data_ptr(), rsa, csa, b.data_ptr(), rsb, csb, beta, c.data_ptr(), n, 1)
    return {"calls": [(entry, args)], "out": out, "keep": keep}


def _prepare_f4(lib, gen, case):
    m, n, k = case["m"], case["n"], case["k"]
    a = _operand(lib, gen, "e4m3", (m, k), False)
    b = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device="cuda", generator=gen)
    out = torch.empty((m, n), dtype=torch.float32, device="cuda")
    keep = [a, b]
    if case["scaled"]:  # E8M0: 2^-7 to 2^0
        scales = torch.randint(120, 128, (n, k // 32), dtype=torch.uint8, device="cuda", generator=gen)
        keep.append(scales)
        entry = lib.skl_gemm_f8e4m3rc_mxf4e2m1c_f32rc_gfx950
        args = (m, n, k, 1.0, a.data_ptr(), k, 1, b.data_ptr(), k, scales.data_ptr(), k // 32, 0.0, out.data_ptr(), n, 1)
    else:
        entry = lib.skl_gemm_f8e4m3rc_f4e2m1c_f32rc_gfx950
        args = (m, n, k, 1.0, a.data_ptr(), k, 1, b.data_ptr(), k, 0.0, out.data_ptr(), n, 1)
    return {"calls": [(entry, args)], "out": out, "keep": keep}


def _prepare_k4(lib, gen, case):
    m, n, k = case["m"], case["n"], case["k"]
    a = _operand(lib, gen, "i8", (m, k), False)
    b = _operand(lib, gen, "i8", (k // 4, n, 4), True)
    out = torch.empty((m, n), dtype=torch.int32, device="cuda")
    args = (m, n, k // 4, 1, a.data_ptr(), k, 4, b.data_ptr(), 4 * n, 0, out.data_ptr(), n)
    return {"calls": [(lib.skl_gemm_i8rcp1x4_i8p4x1c_i32_gfx950, args)], "out": out, "keep": [a, b]}


def _prepare_packed(lib, gen, case):
    m, n, k, kind = case["m"], case["n"], case["k"], case["kind"]
    te = lib.skl_hip_te()
    m1, n1 = -(-m // te), -(-n // te)
    w = 8 if kind in ("i8", "e4m3") else 16
    t, acc = _NAME[kind], "i32" if kind == "i8" else "f32"
    scalar = int if kind == "i8" else float
    a = _operand(lib, gen, kind, (m, k), False)
    b = _operand(lib, gen, kind, (k, n), True)
    ap = torch.empty((m1, k, te), dtype=a.dtype, device="cuda")
    bp = torch.empty((n1, k, te), dtype=b.dtype, device="cuda")
    cp = torch.empty((m1, n1, te, te), dtype=torch.int32 if kind == "i8" else torch.float32, device="cuda")
    out = torch.empty((m, n), dtype=cp.dtype, device="cuda")
    calls = [
        (getattr(lib, f"skl_pack_e{w}_e{w}rcptex1c_gfx950"), (m, k, a.data_ptr(), k, ap.data_ptr(), k * te, te, 0)),
        (getattr(lib, f"skl_pack_e{w}rc_e{w}rcprc_gfx950"), (k, n, b.data_ptr(), n, 1, 1, te, bp.data_ptr(), te, 1, te, k * te, 0)),
        (getattr(lib, f"skl_gemm_{t}rcptex1c_{t}rcp1xte_{acc}rcptexterc_gfx950"),
         (m1, n1, k, scalar(1), ap.data_ptr(), k * te, te, bp.data_ptr(), te, k * te, scalar(0), cp.data_ptr(), te, 1, n1 * te * te, te * te)),
        (lib.skl_unpack_e32rcprc_e32rc_gfx950, (te, te, cp.data_ptr(), te, 1, n1 * te * te, te * te, m, n, out.data_ptr(), n, 1)),
    ]
    return {"calls": calls, "out": out, "keep": [a, b, ap, bp, cp]}


def _prepare_cvt(lib, gen, case):
    n, fmt = case["count"], case["fmt"]
    src = _normal(gen, (n,)).to(torch.float32 if case["src"] == "f32" else torch.bfloat16)
    q = torch.empty((n,), dtype=torch.uint8, device="cuda")
    back = torch.empty((n,), dtype=torch.bfloat16, device="cuda")
    calls = [(getattr(lib, f"skl_cvt_sat_{case['src']}_{_NAME[fmt]}_gfx950"), (q.data_ptr(), src.data_ptr(), 1.5, n)),
             (getattr(lib, f"skl_cvt_{_NAME[fmt]}_bf16_gfx950"), (back.data_ptr(), q.data_ptr(), n))]
    return {"calls": calls, "out": (q, back), "keep": [src]}


def prepare(case, seed):
    lib = _library()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    make = {"gemm": _prepare_gemm, "f4": _prepare_f4, "k4": _prepare_k4, "packed": _prepare_packed, "cvt": _prepare_cvt}
    return make[case["op"]](lib, gen, case)


def run(state):
    for entry, args in state["calls"]:
        entry(*args)
    return state["out"]


def work(case):
    if case["op"] == "cvt":
        src = 4 if case["src"] == "f32" else 2
        return {"bytes": case["count"] * (src + 1 + 1 + 2), "flops": 0}
    m, n, k = case["m"], case["n"], case["k"]
    flops = 2 * m * n * k
    if case["op"] == "f4":
        return {"bytes": m * k + n * k // 2 + (n * k // 32 if case["scaled"] else 0) + 4 * m * n, "flops": flops}
    if case["op"] == "k4":
        return {"bytes": m * k + n * k + 4 * m * n, "flops": flops}
    es = {"bf16": 2, "f16": 2, "f32": 4}.get(case["kind"], 1)
    operands = (m * k + k * n) * es
    if case["op"] == "packed":  # each of the four calls reads its inputs and writes its outputs once
        return {"bytes": 3 * operands + 3 * 4 * m * n, "flops": flops}
    c = m * n * (1 if case["out"] == "q8" else 8 if case["beta"] else 4)
    return {"bytes": case["count"] * (operands + c + (4 * n if case["bias"] else 0)), "flops": case["count"] * flops}


def tolerance(case):
    """About four times what the results were seen to differ from the same product in 64 bits."""
    kind = "e4m3" if case["op"] == "f4" else case.get("kind", "i8")
    if kind == "i8":
        return "exact"
    # the fp8 instructions align the products of one instruction: 1.3e-5 (largest 9e-5) at any K; sums in fp32 of exact
    # products, or of f32's rounded ones: up to 8e-7 (largest 6e-6)
    aligned = kind in ("e4m3", "e5m2") and case["k"] > _FP8_EXACT_MAX_K
    if case.get("out") == "q8":  # a sum next to a rounding boundary: 4e-4 of the bytes, and 6e-6
        return {"differ": 2e-3 if aligned else 3e-5}
    return {"rel": 5e-5, "max": 4e-4} if aligned else {"rel": 3e-6, "max": 2.5e-5}


def _in_64_bits(x, kind):
    """A stored operand as float64."""
    if kind in ("e4m3", "e5m2"):
        x = x.view(torch.float8_e4m3fn if kind == "e4m3" else torch.float8_e5m2).float()
    return x.double()


def exact(case, seed):
    """The result in 64 bits; the 8-bit outputs, and what a conversion writes, have no other value than the one they are compared with."""
    if case["op"] == "cvt" or case.get("out") == "q8":
        return None
    state = prepare(case, seed)
    if case.get("count", 1) > 1:
        return [_exact_gemm(case, one["keep"][0], one["keep"][1], one["out"], one["keep"][2]) for one in state["keep"]]
    m, n, k = case["m"], case["n"], case["k"]
    a, b = state["keep"][0], state["keep"][1]
    if case["op"] == "f4":
        values = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64, device="cuda")
        w = values[torch.stack((b & 15, b >> 4), dim=-1).long()].reshape(n, k)
        if case["scaled"]:
            w *= torch.exp2(state["keep"][2].double() - 127).repeat_interleave(32, dim=1)
        return (_in_64_bits(a, "e4m3") @ w.t())
    if case["op"] == "k4":
        return (a.double() @ b.permute(0, 2, 1).reshape(k, n).double()).round()
    if case["op"] == "packed":
        return _in_64_bits(a, case["kind"]) @ _in_64_bits(b, case["kind"])
    return _exact_gemm(case, a, b, state["out"], state["keep"][2])


def _exact_gemm(case, a, b, c, bias):
    a, b = _in_64_bits(a, case["kind"]), _in_64_bits(b, case["kind"])
    v = (a.t() if case["layout"] == "tn" else a) @ (b.t() if case["layout"] == "nt" else b)
    if case["beta"]:
        v += case["beta"] * c.double()
    if case["bias"]:
        v += bias.double()
    if case["act"] == "relu":
        v = torch.relu(v)
    elif case["act"] == "silu":
        v = v * torch.sigmoid(v)
    elif case["act"] == "gelu":
        v = 0.5 * v * (1 + torch.erf(v / math.sqrt(2)))
    return v
