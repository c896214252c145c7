"""The work this package is timed on: what a serving engine has it do.

Every case goes through a public module's ``forward``, as a model calls it:

  linear    Fp8Linear: bf16 activations through a block-scaled FP8 weight
            (1x128 activation quant and GEMM), buffers installed as the
            engine's warmup installs them
  silu      SiluMulQuantFp8: SiLU*Mul and 1x128 quant between the two MLP GEMMs
  norm      RMSNormFP8Quant, or FusedAddRMSNormFP8Quant with ``add``: the norm
            in front of a quantized linear
  experts   FusedExperts (contiguous layout, prefill) or VllmFusedExperts
            (sorted-token layout, decode) with 128x128-block-scaled weights

Token counts go from one decoding sequence to a prefill chunk of 4096 (silu
8192) tokens; weight shapes are those of the benchmark's configurations and
their tensor-parallel shards.  Inputs are drawn on the GPU from the seed:
activations ~N(0, 1), weight codes as a ~N(0, 0.02) weight quantizes to, block
scales powers of two (a requantized checkpoint) or as given (a checkpoint's
own), routing by the top-k of seeded softmax logits.
"""
import torch

from kb_nano_amd import (Fp8Linear, FusedAddRMSNormFP8Quant, FusedExperts, RMSNormFP8Quant, SiluMulQuantFp8,
                         VllmFusedExperts)

FP8 = torch.float8_e4m3fn
F64 = torch.float64

# (N, K) of the dense layers: the benchmark's prefill and decode layers, their shards over
# eight GPUs, and the smallest configuration
DENSE = [(24576, 1536), (36864, 7168), (7168, 18432), (7168, 16384), (10240, 8192), (8192, 8192), (57344, 8192),
         (8192, 28672), (3072, 1536), (4608, 7168), (7168, 2048), (7168, 2304), (2048, 2048)]
# (experts, hidden, intermediate, top-k)
MOE = [(256, 7168, 2048, 8), (128, 4096, 1536, 8)]
# intermediate sizes of the gated MLPs (whole and sharded) and hidden sizes of the norms
GLU = [18432, 2304, 2048, 3584, 14336]
HIDDEN = [7168, 8192, 4096, 2048]


def listed():
    return [
        # the smallest layer at a decode batch of 64: launches and latency
        {"name": "linear_64_2048x2048", "kind": "linear", "M": 64, "N": 2048, "K": 2048},
        # a decode step of 8 sequences, attention's input projection: streams the weight
        {"name": "linear_8_10240x8192", "kind": "linear", "M": 8, "N": 10240, "K": 8192},
        # a decode step of 200 sequences, attention's output projection: between streaming and compute
        {"name": "linear_200_8192x8192", "kind": "linear", "M": 200, "N": 8192, "K": 8192},
        # a mixed batch (a prefill chunk's ragged end plus decoding sequences) on one of eight shards
        {"name": "linear_777_4608x7168", "kind": "linear", "M": 777, "N": 4608, "K": 7168},
        # a full prefill chunk through the widest layer: matrix-core bound
        {"name": "linear_4096_36864x7168", "kind": "linear", "M": 4096, "N": 36864, "K": 7168},
        # the MLP's activation over a large prefill: bandwidth bound
        {"name": "silu_8192x18432", "kind": "silu", "M": 8192, "I": 18432},
        # the same for one 128-row block on one of eight shards
        {"name": "silu_128x2304", "kind": "silu", "M": 128, "I": 2304},
        # the norm between layers over a prefill chunk, residual updated in place
        {"name": "add_norm_4096x7168", "kind": "norm", "M": 4096, "H": 7168, "add": True},
        # the first norm of a decode step
        {"name": "norm_61x8192", "kind": "norm", "M": 61, "H": 8192, "add": False},
        # a prefill chunk through 256 experts: streams every expert's weights, 128 rows an expert
        {"name": "experts_4096_of_256", "kind": "experts", "layout": "contiguous", "T": 4096, "E": 256, "H": 7168,
         "I": 2048, "topk": 8, "pow2": True},
        # a short prefill through 128 experts with a checkpoint's own scales: about 32 rows an expert
        {"name": "experts_515_of_128", "kind": "experts", "layout": "contiguous", "T": 515, "E": 128, "H": 4096,
         "I": 1536, "topk": 8, "pow2": False},
        # a decode step of 64 sequences through 256 experts: two rows an expert
        {"name": "experts_64_of_256", "kind": "experts", "layout": "sorted", "T": 64, "E": 256, "H": 7168, "I": 2048,
         "topk": 8, "pow2": False},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["silu"] * 2 + ["norm"] * 2 + ["experts"] * 3)
    if kind == "linear":
        N, K = rng.choice(DENSE)
        return {"kind": kind, "M": _log_int(rng, 1, 4096), "N": N, "K": K}
    if kind == "silu":
        return {"kind": kind, "M": 128 * _log_int(rng, 1, 64), "I": rng.choice(GLU)}   # whole 128-row blocks only
    if kind == "norm":
        return {"kind": kind, "M": _log_int(rng, 1, 4096), "H": rng.choice(HIDDEN), "add": rng.random() < 0.5}
    E, H, I, topk = rng.choice(MOE)
    layout = rng.choice(["contiguous", "sorted"])
    T = _log_int(rng, 128, 4096) if layout == "contiguous" else _log_int(rng, 1, 1024)
    return {"kind": kind, "layout": layout, "T": T, "E": E, "H": H, "I": I, "topk": topk, "pow2": rng.random() < 0.5}


# ------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(shape, g, std=1.0):
    return (torch.randn(shape, device="cuda", generator=g) * std).bfloat16()


def _weight(N, K, g, pow2=True, experts=0):
    """Codes and 128x128 block scales of ~N(0, 0.02) weights [(experts,) N, K]: a block's largest
    magnitude is about 4.1 deviations, so the codes' deviation is 448 / 4.1 (scales as given) or
    0.02 / 2^-12 (scales rounded up to a power of two)."""
    shape = (experts, N, K) if experts else (N, K)
    w = torch.empty(shape, dtype=FP8, device="cuda")
    rows, step = w.view(-1, K), max(1, (1 << 27) // K)
    for r in range(0, rows.shape[0], step):
        part = rows[r:r + step]
        x = torch.randn(part.shape, device="cuda", generator=g)
        part.copy_(x.mul_(82.0 if pow2 else 109.0).clamp_(-448.0, 448.0))
    blocks = shape[:-2] + (-(-N // 128), -(-K // 128))
    u = torch.rand(blocks, device="cuda", generator=g)
    s = torch.exp2(-12.0 + (u < 0.1).float() - (u > 0.9).float()) if pow2 else 1.83e-4 * (0.75 + 0.5 * u)
    return w, s.contiguous()


def _routing(T, E, topk, g):
    p = torch.softmax(torch.randn(T, E, device="cuda", generator=g), dim=-1)
    w, ids = torch.topk(p, topk, dim=-1)
    return ids.contiguous(), (w / w.sum(dim=-1, keepdim=True)).contiguous()


def _inputs(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "linear":
        w, s = _weight(case["N"], case["K"], g)
        return {"x": _normal((case["M"], case["K"]), g), "w": w, "s": s}
    if kind == "silu":
        x = torch.randn((case["M"], 2 * case["I"]), device="cuda", generator=g)
        big = torch.rand(x.shape, device="cuda", generator=g) < 1e-3   # a few large activations, as models have
        return {"x": torch.where(big, x * 50.0, x).bfloat16()}
    if kind == "norm":
        d = {"x": _normal((case["M"], case["H"]), g), "w": _normal((case["H"],), g, 0.1) + 1.0}
        if case["add"]:
            d["r"] = _normal((case["M"], case["H"]), g, 2.0)
        return d
    E, H, I = case["E"], case["H"], case["I"]
    d = {"x": _normal((case["T"], H), g)}
    d["w13"], d["s13"] = _weight(2 * I, H, g, case["pow2"], E)
    d["w2"], d["s2"] = _weight(H, I, g, case["pow2"], E)
    d["ids"], d["tw"] = _routing(case["T"], E, case["topk"], g)
    return d


def prepare(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        d["op"] = Fp8Linear()
        d["op"]._ensure_buffers(case["M"], case["K"], case["N"], d["x"].device)   # as the engine's warmup does
    elif kind == "silu":
        d["op"] = SiluMulQuantFp8()
    elif kind == "norm":
        d["op"] = FusedAddRMSNormFP8Quant() if case["add"] else RMSNormFP8Quant()
    elif case["layout"] == "contiguous":
        d["op"] = FusedExperts()
    else:
        d["op"] = VllmFusedExperts()
    d["case"] = dict(case)
    return d


def run(state):
    case, op, x = state["case"], state["op"], state["x"]
    kind = case["kind"]
    if kind == "linear":
        return op(x, state["w"], state["s"])
    if kind == "silu":
        return op(x)
    if kind == "norm":
        if case["add"]:
            q, s, r = op(x, state["r"], state["w"])
            return q, s, r, x
        return op(x, state["w"])
    if case["layout"] == "contiguous":
        return op(x, state["w13"], state["w2"], state["tw"], state["ids"], case["E"], w13_scale=state["s13"],
                  w2_scale=state["s2"], use_fp8_w8a8=True, block_shape=[128, 128])
    return op(x, state["w13"], state["w2"], state["tw"], state["ids"], case["E"], state["s13"], state["s2"],
              [128, 128])


# ---------------------------------------------------------- what it must do

def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2 * M * K + N * K + 4 * (-(-N // 128)) * (K // 128) + 2 * M * N, "flops": 2 * M * N * K}
    if kind == "silu":
        n = case["M"] * case["I"]
        return {"bytes": 4 * n + n + n // 32, "flops": 8 * n}
    if kind == "norm":
        n = case["M"] * case["H"]
        return {"bytes": (2 + 1) * n + n // 32 + (6 * n if case["add"] else 0), "flops": 8 * n}
    T, E, H, I, k = case["T"], case["E"], case["H"], case["I"], case["topk"]
    active = E * (1.0 - (1.0 - k / E) ** T)   # experts that some token is routed to
    return {"bytes": active * 3 * H * I * (1 + 4 / 16384) + 4 * T * H + 12 * T * k, "flops": 2 * T * k * 3 * H * I}


def tolerance(case):
    kind = case["kind"]
    if kind == "silu":
        return "exact"                     # codes and scales are bytes
    if kind == "norm":
        # a row's sum in another order moves a few codes to their neighbour: 1.6e-4 against 64 bits
        return {"rel": 7e-4, "max": 0.2}
    if kind == "linear":
        # fp32 sums in another order, rounded to bf16: 2.3e-4, largest 0.0078 (one rounding step)
        return {"rel": 1e-3, "max": 0.03}
    # the same through an e4m3 intermediate: 2.2e-3 to 3.5e-3, largest 0.076
    return {"rel": 1e-2, "max": 0.3}


# ------------------------------------------------------------------ 64 bits

def _quant64(v):
    """1x128 e4m3 codes (as float64) and power-of-two scales of v [M, K] (float64), per group
    scale = amax / 448 rounded up to a power of two."""
    M, K = v.shape
    g = v.view(M, K // 128, 128)
    s = torch.exp2(torch.ceil(torch.log2((g.abs().amax(-1).clamp_min(1e-10) / 448.0))))
    q = (g / s[..., None]).float().to(FP8).to(F64)
    return q.view(M, K), s


def _deq64(w, s):
    N, K = w.shape
    full = s.to(F64).repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)[:, :K]
    return w.to(torch.float32).to(F64).mul_(full)


def _times(v, w, s):
    """quantize-dequantize v [M, K] and multiply by the dequantized weight's transpose, in chunks of rows of w."""
    q, sc = _quant64(v)
    a = q * sc.repeat_interleave(128, 1)
    return torch.cat([a @ _deq64(w[n:n + 8192], s[n // 128:(n + 8192) // 128]).t().contiguous()
                      for n in range(0, w.shape[0], 8192)], 1)


def _bf16(v):
    """Rounded to bf16, as float64."""
    return v.float().bfloat16().to(F64)


def _silu_mul64(gate, up):
    return _bf16(_bf16(gate / (1.0 + torch.exp(-gate))) * up)


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    x = d["x"].to(F64)
    if kind == "linear":
        return _times(x, d["w"], d["s"])
    if kind == "silu":
        rows = [_quant64(_silu_mul64(p[:, :case["I"]], p[:, case["I"]:])) for p in x.split(1024)]
        return torch.cat([q for q, _ in rows]), torch.cat([s for _, s in rows])
    if kind == "norm":
        a = x + d["r"].to(F64) if case["add"] else x
        base = _bf16(a) if case["add"] else a
        v = base / torch.sqrt((a * a).mean(-1, keepdim=True) + 1e-6) * d["w"].to(F64)
        q, s = _quant64(v)
        return (q, s, a, v) if case["add"] else (q, s)
    out = torch.zeros(x.shape, dtype=F64, device=x.device)
    I = case["I"]
    for e in range(case["E"]):
        t, slot = torch.nonzero(d["ids"] == e, as_tuple=True)
        if t.numel():
            gu = _bf16(_times(x[t], d["w13"][e], d["s13"][e]))
            y = _times(_silu_mul64(gu[:, :I], gu[:, I:]), d["w2"][e], d["s2"][e])
            out.index_add_(0, t, y * d["tw"][t, slot].to(F64)[:, None])
    return out
