"""Workloads of the library as its users run them, with their inputs, the work
each cannot do without and the accuracy it owes.

A case is one call of a public entry point: a dense GEMM (the ``matmul`` of a
dtype's module), a grouped (MoE) GEMM, the flash-attention forward, or an
operand quantizer.  ``listed()`` holds the named ones; ``draw(rng)`` gives
others of the same kinds and ranges.  Inputs are made on the GPU from the seed
alone: activations of unit variance, weights scaled by 1/sqrt(K), BF8 and
MXFP4 operands quantized from such values.
"""

import torch

from gfx950_gluon_tutorials_amd import quant
from gfx950_gluon_tutorials_amd.attention import MetaData, fmha_v3, fmha_v4
from gfx950_gluon_tutorials_amd.gemm.inter_wave import a4w4 as a4w4_8w, a8w8 as a8w8_8w, a16w16 as a16w16_8w
from gfx950_gluon_tutorials_amd.gemm.intra_wave import a4w4, a8w8, a16w16
from gfx950_gluon_tutorials_amd.gemm.moe import moe_matmul, moe_matmul_a4w4, moe_matmul_a8w8

MODULES = {4: {"f16": a16w16, "bf16": a16w16, "bf8": a8w8, "mxfp4": a4w4},
           8: {"f16": a16w16_8w, "bf16": a16w16_8w, "bf8": a8w8_8w, "mxfp4": a4w4_8w}}
TORCH = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
K_STEP = {"f16": 8, "bf16": 8, "bf8": 16, "mxfp4": 256}          # dense K granularity
MOE_K_STEP = {"f16": 64, "bf16": 64, "bf8": 128, "mxfp4": 256}   # grouped K granularity
E5M2_MAX = 57344.0


def _gemm(name, dtype, M, N, K, schedule="dp", waves=4, scales="row"):
    return {"name": name, "kind": "gemm", "dtype": dtype, "M": M, "N": N, "K": K, "schedule": schedule,
            "waves": waves, "scales": scales}


def _moe(name, dtype, T, E, N, K):
    return {"name": name, "kind": "moe", "dtype": dtype, "T": T, "E": E, "N": N, "K": K}


def _attn(name, dtype, B, HQ, HK, S, D, layout="bhsd", variant=4):
    return {"name": name, "kind": "attn", "dtype": dtype, "B": B, "HQ": HQ, "HK": HK, "S": S, "D": D,
            "layout": layout, "variant": variant}


def _quant(name, to, dtype, R, K):
    return {"name": name, "kind": "quant", "to": to, "dtype": dtype, "R": R, "K": K}


def listed():
    return [
        # The smallest call: one output tile, where launch and latency are everything.
        _gemm("gemm_f16_256x256x512", "f16", 256, 256, 512),
        # Decoding: a batch of 16 tokens through one weight matrix.
        _gemm("gemm_bf16_16x4096x8192", "bf16", 16, 4096, 8192),
        # One GPU's share of an 8-way row split of the 4096 x 4096 x 8192 GEMM,
        # with the schedule the library recommends for few rows.
        _gemm("gemm_f16_512x4096x8192_splitk", "f16", 512, 4096, 8192, schedule="splitk"),
        # A ragged batch of prompt tokens: edges in M and N, a K tail.
        _gemm("gemm_bf16_1000x3000x2056", "bf16", 1000, 3000, 2056),
        # The benchmark's headline GEMM.
        _gemm("gemm_f16_4096x4096x8192", "f16", 4096, 4096, 8192),
        # Prefill of 1024 tokens in BF8 with per-tensor scales.
        _gemm("gemm_bf8_1024x4096x7168", "bf8", 1024, 4096, 7168),
        # Decoding of 64 sequences with MXFP4 weights and activations.
        _gemm("gemm_mxfp4_64x8192x8192", "mxfp4", 64, 8192, 8192),
        # The activations of an MXFP4 layer quantized on the way to its GEMM.
        _quant("quant_mxfp4_bf16_4096x7168", "mxfp4", "bf16", 4096, 7168),
        # Decoding through 32 experts: 16 sequences, 8 experts each.
        _moe("moe_bf16_t128", "bf16", 128, 32, 4096, 7168),
        # The grouped benchmark's prefill.
        _moe("moe_mxfp4_t32768", "mxfp4", 32768, 32, 4096, 7168),
        # Long-sequence attention, one point of the sequence-length sweep.
        _attn("attn_bf16_h64_s8192_d128", "bf16", 1, 64, 64, 8192, 128),
        # A short ragged prompt with grouped K/V heads in the (batch, seq, head, dim) layout.
        _attn("attn_f16_b2_h16k4_s1088_d64", "f16", 2, 16, 4, 1088, 64, layout="bshd"),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = lo * (hi / lo) ** rng.random()
    return max(step, min(hi // step * step, round(v / step) * step))


def draw(rng):
    kind = rng.choice(["gemm"] * 6 + ["moe"] * 2 + ["attn"] * 2 + ["quant"])
    while True:
        if kind == "gemm":
            dtype = rng.choice(["f16", "bf16", "bf8", "mxfp4"])
            case = _gemm("", dtype, _log(rng, 1, 8192), _log(rng, 256, 8192, rng.choice([1, 8, 128])),
                         _log(rng, 512, 32768, K_STEP[dtype]), schedule=rng.choice(["dp", "dp", "dp", "auto", "splitk"]),
                         waves=rng.choice([4, 4, 4, 8]), scales=rng.choice(["row", "kmajor"]))
        elif kind == "moe":
            dtype = rng.choice(["f16", "bf16", "bf8", "mxfp4"])
            case = _moe("", dtype, _log(rng, 16, 32768), _log(rng, 4, 64), _log(rng, 512, 4096, 8),
                        _log(rng, 512, 7168, MOE_K_STEP[dtype]))
        elif kind == "attn":
            hk = _log(rng, 1, 32)
            case = _attn("", rng.choice(["f16", "bf16"]), _log(rng, 1, 8), hk * rng.choice([1, 2, 4]), hk,
                         _log(rng, 64, 8192, 64), rng.choice([64, 128]), layout=rng.choice(["bhsd", "bshd"]),
                         variant=rng.choice([3, 4, 4]))
        else:
            case = _quant("", rng.choice(["mxfp4", "e5m2"]), rng.choice(["bf16", "f16", "f32"]), _log(rng, 1, 8192),
                          _log(rng, 512, 16384, 32))
        w = work(case)
        if w["flops"] <= 1.1e12 and w["bytes"] <= 1.9e9:
            del case["name"]
            return case


# --- inputs ---------------------------------------------------------------

def _e5m2(x):
    """Per-tensor BF8: codes of x / scale with the largest magnitude on the largest code."""
    scale = (x.abs().amax() / E5M2_MAX).float().reshape(1)
    return (x / scale).to(torch.float8_e5m2), scale


def _mxfp4(x):
    """MXFP4 along the last axis: packed e2m1 codes (even k in the low nibble)
    and one E8M0 exponent byte per 32 values."""
    g = x.reshape(-1, 32)
    e = torch.floor(torch.log2(g.abs().amax(dim=1, keepdim=True))) - 2
    y = g * torch.exp2(-e)
    mids = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=x.device)
    code = torch.bucketize(y.abs(), mids, out_int32=True).to(torch.uint8) | ((y < 0).to(torch.uint8) << 3)
    code = code.reshape(x.shape)
    return code[..., 0::2] | (code[..., 1::2] << 4), (e + 127).to(torch.uint8).reshape(*x.shape[:-1], -1)


def _rand(gen, *shape, scale=1.0, dtype=torch.float32):
    x = torch.randn(*shape, generator=gen, device="cuda", dtype=dtype)
    return x.mul_(scale) if scale != 1.0 else x


def _operand(gen, dtype, rows, K, scale=1.0):
    """One K-contiguous operand: (values,) or (codes, scales)."""
    if dtype in ("f16", "bf16"):
        return (_rand(gen, rows, K, scale=scale, dtype=TORCH[dtype]),)
    x = _rand(gen, rows, K, scale=scale)
    return _e5m2(x) if dtype == "bf8" else _mxfp4(x)


def _kmajor(s):
    """The (rows, groups) view of scales stored group by group; rows padded to 4 bytes."""
    rows, groups = s.shape
    buf = torch.empty(groups, -(-rows // 4) * 4, dtype=torch.uint8, device=s.device)
    buf[:, :rows] = s.t()
    return buf.t()[:rows]


def _inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, dtype = case["kind"], case["dtype"]
    if kind == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        a, b = _operand(gen, dtype, M, K), _operand(gen, dtype, N, K, scale=K ** -0.5)
        if dtype == "mxfp4" and case["scales"] == "kmajor":
            a, b = (a[0], _kmajor(a[1])), (b[0], _kmajor(b[1]))
        return {"a": a, "b": b}
    if kind == "moe":
        T, E, N, K = case["T"], case["E"], case["N"], case["K"]
        share = -torch.log(torch.rand(E, 5, generator=gen, device="cuda")).sum(dim=1)  # Gamma(5): Dirichlet(5) shares
        owner = torch.multinomial(share, T, replacement=True, generator=gen)
        off = torch.zeros(E + 1, dtype=torch.int32, device="cuda")
        off[1:] = torch.cumsum(torch.bincount(owner, minlength=E), dim=0)
        a = _operand(gen, dtype, T, K)
        if dtype in ("f16", "bf16"):
            b = (_rand(gen, E, N, K, scale=K ** -0.5, dtype=TORCH[dtype]),)
        else:
            first = _operand(gen, dtype, N, K, scale=K ** -0.5)
            b = tuple(torch.empty(E, *t.shape, dtype=t.dtype, device="cuda") for t in first)
            for e in range(E):
                for dst, src in zip(b, first if e == 0 else _operand(gen, dtype, N, K, scale=K ** -0.5)):
                    dst[e] = src
            if dtype == "bf8":
                b = (b[0], b[1].reshape(E))
        return {"a": a, "b": b, "off": off}
    if kind == "attn":
        B, HQ, HK, S, D = (case[k] for k in ("B", "HQ", "HK", "S", "D"))
        shape = (lambda h: (B, h, S, D)) if case["layout"] == "bhsd" else (lambda h: (B, S, h, D))
        return dict(zip("qkv", (_rand(gen, *shape(h), dtype=TORCH[dtype]) for h in (HQ, HK, HK))))
    return {"x": _rand(gen, case["R"], case["K"], dtype=TORCH[dtype])}


def prepare(case, seed):
    state = _inputs(case, seed)
    state["case"] = case
    if case["kind"] == "gemm":
        state["fn"] = MODULES[case["waves"]][case["dtype"]].matmul
    elif case["kind"] == "attn":
        state["o"] = torch.empty_like(state["q"])
        md = MetaData(sm_scale=case["D"] ** -0.5)
        md.layout = case["layout"]
        md.max_seqlens_q = md.max_seqlens_k = case["S"]
        state["md"] = md
        state["fn"] = (fmha_v3 if case["variant"] == 3 else fmha_v4).run_gluon_attention
    return state


def run(state):
    case = state["case"]
    kind, dtype = case["kind"], case["dtype"]
    if kind == "gemm":
        a, b, sched = state["a"], state["b"], case["schedule"]
        if dtype == "mxfp4":
            return state["fn"](a[0], b[0], a[1], b[1], schedule=sched)
        if dtype == "bf8":
            return state["fn"](a[0], b[0].T, a_scale=a[1], b_scale=b[1], out_dtype=torch.bfloat16, schedule=sched)
        return state["fn"](a[0], b[0].T, schedule=sched)
    if kind == "moe":
        a, b, off = state["a"], state["b"], state["off"]
        if dtype == "mxfp4":
            return moe_matmul_a4w4(a[0], b[0], a[1], b[1], off)
        if dtype == "bf8":
            return moe_matmul_a8w8(a[0], b[0], off, a_scale=a[1], b_scales=b[1])
        return moe_matmul(a[0], b[0], off)
    if kind == "attn":
        state["fn"](state["q"], state["k"], state["v"], state["o"], state["md"])
        return state["o"]
    if case["to"] == "mxfp4":
        return list(quant.quantize_mxfp4(state["x"]))
    codes, scale = quant.quantize_e5m2(state["x"])
    return [codes.view(torch.uint8), scale]


# --- work and accuracy ----------------------------------------------------

def work(case):
    kind, dtype = case["kind"], case["dtype"]
    if kind == "quant":
        n = case["R"] * case["K"]
        out = n / 2 + n / 32 if case["to"] == "mxfp4" else n + 4
        return {"bytes": n * (4 if dtype == "f32" else 2) + out, "flops": 0}
    if kind == "attn":
        B, HQ, HK, S, D = (case[k] for k in ("B", "HQ", "HK", "S", "D"))
        return {"bytes": 2 * B * S * D * (2 * HQ + 2 * HK), "flops": 4 * B * HQ * S * S * D}
    N, K = case["N"], case["K"]
    M = case["M"] if kind == "gemm" else case["T"]
    weights = 1 if kind == "gemm" else min(case["E"], case["T"])  # an expert without tokens is not read
    per_k = {"f16": 2, "bf16": 2, "bf8": 1, "mxfp4": 0.5 + 1 / 32}[dtype]
    return {"bytes": (M + weights * N) * K * per_k + 2 * M * N, "flops": 2 * M * N * K}


def tolerance(case):
    """Relative errors of correct results against 64-bit ones: one rounding to
    the 16-bit output (f16 about 2e-4, bf16 about 1.7e-3; attention also
    rounds the probabilities), four times over.  Quantizers are exact."""
    if case["kind"] == "quant":
        return "exact"
    if case["kind"] == "attn":
        return {"rel": 1.6e-3 if case["dtype"] == "f16" else 1.2e-2}
    return {"rel": 8e-4 if case["dtype"] == "f16" else 7e-3}


def _dequant(t, dtype):
    """A K-contiguous operand (codes or values, scales) in 64 bits."""
    if dtype in ("f16", "bf16"):
        return t[0].double()
    if dtype == "bf8":
        return t[0].float().double() * t[1].double()
    table = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device="cuda")
    code = torch.stack([t[0] & 15, t[0] >> 4], dim=-1).reshape(*t[0].shape[:-1], -1).int()
    v = table[code & 7] * (1 - 2 * (code >> 3))
    return v * torch.exp2(t[1].double() - 127).repeat_interleave(32, dim=-1)


def exact(case, seed):
    kind, dtype = case["kind"], case["dtype"]
    x = _inputs(case, seed)
    if kind == "gemm":
        return _dequant(x["a"], dtype) @ _dequant(x["b"], dtype).T
    if kind == "moe":
        off = x["off"].tolist()
        out = torch.empty(case["T"], case["N"], dtype=torch.float64, device="cuda")
        for e in range(case["E"]):
            rows = slice(off[e], off[e + 1])
            if off[e + 1] > off[e]:
                a = tuple(t if dtype == "bf8" and i else t[rows] for i, t in enumerate(x["a"]))
                out[rows] = _dequant(a, dtype) @ _dequant(tuple(t[e] for t in x["b"]), dtype).T
        return out
    if kind == "attn":
        order = (0, 1, 2, 3) if case["layout"] == "bhsd" else (0, 2, 1, 3)
        q, k, v = (x[n].permute(order) for n in "qkv")
        out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
        group = case["HQ"] // case["HK"]
        for b in range(case["B"]):
            for h in range(case["HQ"]):
                s = q[b, h].double() @ k[b, h // group].double().T * case["D"] ** -0.5
                out[b, h] = torch.softmax(s, dim=1) @ v[b, h // group].double()
        return out.permute(order).contiguous()
    if case["to"] == "mxfp4":
        return None
    return [None, x["x"].double().abs().amax().reshape(1) / E5M2_MAX]
