"""The products that users of this library have it compute, as cases to time: what a case is (`listed`, `draw`), what a
program holds before the call (`prepare`), the call itself (`run`: one launch of C = alpha * A.B + beta * C through
`Context.gemm_bf16` on the null stream), what it cannot do without (`work`) and how far another correct implementation
may be from it (`tolerance`).

A case: m, n, k, batch, nt (B stored N x K), in_type (bf16, f16, e4m3, e5m2, f32, f64), out (same: the operands' type,
bf16 for 8-bit operands; f32), alpha, beta, dist (uniform: [-1, 1); normal: activations ~ N(0, 1) against weights
~ N(0, 0.02); scaled: both ~ N(0, 1 / K)).
"""
import math

import torch

import maize_amd as mz

# operand type -> (torch type, library type, bytes per element, torch type of C for out == "same")
TYPES = {
    "bf16": (torch.bfloat16, mz.IN_BF16, 2, torch.bfloat16),
    "f16": (torch.float16, mz.IN_F16, 2, torch.float16),
    "e4m3": (torch.float8_e4m3fn, mz.IN_E4M3, 1, torch.bfloat16),
    "e5m2": (torch.float8_e5m2, mz.IN_E5M2, 1, torch.bfloat16),
    "f32": (torch.float32, mz.IN_F32, 4, torch.float32),
    "f64": (torch.float64, mz.IN_F64, 8, torch.float64),
}
# What a multiply-add of each type costs beside one of bf16 on the matrix cores (dense peaks: 2500, 5000, 157 and 79 TFLOP/s):
# bounds the size of drawn cases.
COST = {"bf16": 1.0, "f16": 1.0, "e4m3": 0.5, "e5m2": 0.5, "f32": 16.0, "f64": 32.0}


def case(name, m, n, k, nt=False, in_type="bf16", batch=1, out="same", alpha=1.0, beta=0.0, dist="uniform"):
    c = dict(m=m, n=n, k=k, nt=nt, in_type=in_type, batch=batch, out=out, alpha=alpha, beta=beta, dist=dist)
    return dict(c, name=name) if name else c


def listed():
    return [
        # The smallest call: one block of a caller's own tiling, bound by the launch.
        case("block_64", 64, 64, 64),
        # A small product whose extents the caller does not choose (ragged samples against a small layer): no row of any operand
        # is 16-byte material.
        case("ragged_small", 150, 201, 333),
        # Decoding: 16 tokens against a K x N projection of a 4096-wide model.
        case("decode", 16, 14336, 4096, dist="normal"),
        # The last projection of a small decoder: seven tokens against a vocabulary of odd size, weights stored N x K.
        case("vocabulary", 7, 50257, 768, nt=True, dist="normal"),
        # Decoding against 8-bit weights.
        case("decode_e4m3", 16, 14336, 4096, nt=True, in_type="e4m3"),
        # Prefill: 1024 tokens against a square projection, weights stored N x K.
        case("prefill", 1024, 4096, 4096, nt=True, dist="normal"),
        # Gradients summed into an fp32 buffer over a ragged batch of tokens: the token count is K and it is odd.
        case("accumulate_ragged", 1024, 3072, 1999, out="f32", beta=1.0, dist="normal"),
        # The reference's example product, the headline figure.
        case("square_4096", 4096, 4096, 4096),
        # The same with every extent off the tile.
        case("ragged_4000", 4000, 4104, 4032),
        # Many independent products in one launch.
        case("batched_2048", 2048, 2048, 2048, batch=32),
        # A large product on weights stored N x K.
        case("large_8192", 8192, 8192, 8192, nt=True, dist="scaled"),
        # Full precision (the catalogue's tf32 entry runs on fp32 matrix instructions), a size that no tile divides.
        case("single_2000", 2000, 2000, 2000, in_type="f32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extent(rng, lo, hi, grain):
    """An extent in [lo, hi], spread over its logarithm: a multiple of `grain` (1: any)."""
    return max(lo, min(hi, _log(rng, lo, hi) // grain * grain or grain))


def draw(rng):
    """One more case: few rows against weights, a single product, a batch of products or a small block, of any operand type,
    layout and epilogue; a third of them with extents that are no multiple of anything."""
    largest = 8192.0 ** 3
    while True:
        kind = rng.choice(["small", "rows", "rows", "product", "product", "batched"])
        in_type = rng.choice(["bf16"] * 6 + ["f16", "f16", "e4m3", "e4m3", "e5m2", "f32", "f64"])
        grain = 1 if rng.random() < 1.0 / 3.0 else rng.choice([8, 16, 64])
        batch = 1
        if kind == "small":
            m, n, k = (_extent(rng, 16, 384, grain) for _ in range(3))
        elif kind == "rows":
            m, n, k = _extent(rng, 1, 64, 1), _extent(rng, 1024, 65536, grain), _extent(rng, 512, 16384, grain)
        elif kind == "product":
            m, n, k = (_extent(rng, 128, 8192, grain) for _ in range(3))
        else:
            m, n, k = (_extent(rng, 32, 2048, grain) for _ in range(3))
            batch = _extent(rng, 2, 128, 1)
        elems = batch * (m * k + k * n + m * n)
        if batch * m * n * k * COST[in_type] > 0.5 * largest or elems * 8 > 2 ** 32:
            continue
        out, alpha, beta = "same", 1.0, 0.0
        r = rng.random()
        if in_type not in ("f32", "f64") and r < 0.15:
            out, beta = "f32", rng.choice([0.0, 1.0])
        elif r > 0.9:
            alpha, beta = 0.5, 0.5
        dist = "normal" if kind == "rows" else rng.choice(["uniform", "scaled"])
        return case(None, m, n, k, rng.random() < 0.5, in_type, batch, out, alpha, beta, dist)


_context = None


def context():
    """The device context that a program keeps for its life (loads the code object)."""
    global _context
    if _context is None:
        torch.cuda.init()
        _context = mz.Context(0)
    return _context


def _values(gen, shape, kind, sigma):
    x = torch.empty(shape, device="cuda", dtype=torch.float64 if kind == torch.float64 else torch.float32)
    x = x.uniform_(-1.0, 1.0, generator=gen) if sigma is None else x.normal_(0.0, sigma, generator=gen)
    return x.to(kind)


def prepare(c, seed):
    kind, in_type, _, same = TYPES[c["in_type"]]
    b, m, n, k = c["batch"], c["m"], c["n"], c["k"]
    sigma_a, sigma_b = {"uniform": (None, None), "normal": (1.0, 0.02), "scaled": (k ** -0.5, k ** -0.5)}[c["dist"]]
    if c["in_type"] in ("e4m3", "e5m2") and sigma_a is not None:
        sigma_a = sigma_b = 1.0        # 8-bit operands carry their scale apart: the values themselves fill the format's range
    gen = torch.Generator("cuda").manual_seed(int(seed))
    bs = (n, k) if c["nt"] else (k, n)
    a = _values(gen, (b, m, k), kind, sigma_a)
    w = _values(gen, (b,) + bs, kind, sigma_b)
    out_kind = torch.float32 if c["out"] == "f32" else same
    out = _values(gen, (b, m, n), out_kind, None) if c["beta"] else torch.zeros((b, m, n), device="cuda", dtype=out_kind)
    views = [mz.GlobalMatrix(a.data_ptr(), m, k), mz.GlobalMatrix(w.data_ptr(), *bs), mz.GlobalMatrix(out.data_ptr(), m, n)]
    how = dict(layout=mz.LAYOUT_NT if c["nt"] else mz.LAYOUT_NN, batch=b)
    if b > 1:
        how.update(stride_a=m * k, stride_b=k * n, stride_c=m * n)
    if c["in_type"] == "bf16" and c["out"] == "same" and (c["alpha"], c["beta"]) == (1.0, 0.0):
        desc = mz.gemm_desc(*views, **how)
    else:
        desc = mz.gemm_ex_desc(*views, in_type=in_type, out_type=mz.OUT_F32 if c["out"] == "f32" else mz.OUT_SAME,
                               alpha=c["alpha"], beta=c["beta"], **how)
    return context(), desc, out, (a, w)


def run(state):
    ctx, desc, out, _ = state
    ctx.gemm_bf16(desc)
    return out


def work(c):
    _, _, size, same = TYPES[c["in_type"]]
    b, m, n, k = c["batch"], c["m"], c["n"], c["k"]
    c_bytes = (4 if c["out"] == "f32" else torch.empty(0, dtype=same).element_size()) * m * n * (2 if c["beta"] else 1)
    return {"bytes": b * (size * (m * k + k * n) + c_bytes), "flops": 2.0 * b * m * n * k}


def tolerance(c):
    """About four times what the library shows against sums in fp64 on 72 products of these ranges: a rounding to bf16 is
    1.7e-3 of the result's norm (3.9e-3 at most of a value), one to half an eighth of it; sums in the operands' precision
    grow with the square root of their length (fp32 matrix instructions: 1.3e-6 at k = 5168, 5.2e-7 at 840; bf16 products
    summed in fp32: 2.3e-7 at 2000; fp64: 4.0e-16 at 128); 8-bit products left unrounded show what the matrix instruction
    drops when it aligns them (1.3e-5 at k = 15296)."""
    grow = math.sqrt(c["k"])
    if c["in_type"] == "f64":
        return {"rel": 1.4e-16 * grow, "max": 1.2e-15 * grow}
    if c["in_type"] == "f32":
        return {"rel": 8e-8 * grow, "max": 6e-7 * grow}
    if c["out"] == "f32":
        return {"rel": 6e-5, "max": 3e-4} if c["in_type"] in ("e4m3", "e5m2") else {"rel": 1e-7 + 2e-8 * grow, "max": 1e-6 + 2e-7 * grow}
    return {"rel": 8.5e-4, "max": 2e-3} if c["in_type"] == "f16" else {"rel": 6.8e-3, "max": 1.6e-2}
