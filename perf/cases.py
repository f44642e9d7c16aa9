"""The calls a user of this framework makes, for timing.

Every case is one call of an ``@eas.kernel`` on torch GPU tensors: the kernels are the ones
the framework exists for (elementwise add and fma, the naive matmul, the threadgroup-tile
fp32 matmul and the simdgroup-MMA matmul with 16-bit or fp32 operands), written here as a
user writes them.  A case is a dict of plain values; ``kind`` names the kernel, ``dtype`` the
type of its operands and ``out`` the type of a matmul's result.

``listed()`` holds the standing cases, ``draw(rng)`` gives another one of the same ranges.
"""

from __future__ import annotations

import math

import torch

import eas
from eas import mk

# -- the kernels ---------------------------------------------------------------


@eas.kernel
def add_kernel(a, b, c, N, BLOCK: eas.constexpr):
    offs = mk.program_id(0) * BLOCK + mk.arange(0, BLOCK)
    mask = offs < N
    mk.store(c, offs, mk.load(a, offs, mask) + mk.load(b, offs, mask), mask)


@eas.kernel
def fma_kernel(a, b, c, d, N, BLOCK: eas.constexpr):
    offs = mk.program_id(0) * BLOCK + mk.tid(0, BLOCK)
    mask = offs < N
    mk.store(d, offs, mk.load(a, offs, mask) * mk.load(b, offs, mask) + mk.load(c, offs, mask), mask)


@eas.kernel
def matmul_kernel(a, b, c, M, N, BLOCK: eas.constexpr, K: eas.constexpr):
    """One thread per output, k unrolled while tracing."""
    row = mk.program_id(0)
    col = mk.program_id(1) * BLOCK + mk.tid(0, BLOCK)
    mask = mk.where(row < M, col < N, False)
    acc = 0.0
    for k in range(K):
        acc = acc + mk.load(a, row * K + k, mask) * mk.load(b, k * N + col, mask)
    mk.store(c, row * N + col, acc, mask)


@eas.kernel
def matmul_tiled_kernel(a, b, c, M, N, BM: eas.constexpr, BN: eas.constexpr, BK: eas.constexpr,
                        K: eas.constexpr, NT: eas.constexpr):
    """fp32 through padded threadgroup tiles, four outputs per thread."""
    tid = mk.tid(0, NT)
    ng = BN // 4
    lda, ldb = BK + 1, BN + 1
    rm, cg = tid // ng, tid % ng
    tile_n, tile_m = mk.program_id(0) * BN, mk.program_id(1) * BM
    row, col = tile_m + rm, tile_n + cg * 4
    As = mk.alloc_tg(BM * lda)
    Bs = mk.alloc_tg(BK * ldb)
    acc = [0.0, 0.0, 0.0, 0.0]
    for k0 in range(0, K, BK):
        for i in range(0, BM * BK, NT):
            e = tid + i
            r, q = e // BK, e % BK
            inside = e < BM * BK
            mk.store(As, r * lda + q,
                     mk.load(a, (tile_m + r) * K + k0 + q, inside & (tile_m + r < M) & (k0 + q < K)), inside)
        for i in range(0, BK * BN, NT):
            e = tid + i
            r, q = e // BN, e % BN
            inside = e < BK * BN
            mk.store(Bs, r * ldb + q,
                     mk.load(b, (k0 + r) * N + tile_n + q, inside & (k0 + r < K) & (tile_n + q < N)), inside)
        mk.barrier()
        for j in range(4):
            acc[j] = acc[j] + mk.dot(As, rm * lda, 1, Bs, cg * 4 + j, ldb, BK)
        mk.barrier()
    for j in range(4):
        mk.store(c, row * N + col + j, acc[j], (row < M) & (col + j < N))


def _mma_body(a, b, c, M, N, BM, BN, BK, K, NT, tile, rounded, finish):
    """The simdgroup-MMA matmul: operands rounded to 16 bits in threadgroup tiles, f32 sums."""
    tid = mk.tid(0, NT)
    sg = mk.sg_id()
    base_n, base_m = mk.program_id(0) * BN, mk.program_id(1) * BM
    sg_m, sg_n = sg // (BN // 8), sg % (BN // 8)
    lda, ldb, ldc = BK + 1, BN + 1, BN + 1
    As, Bs, Cs = tile(BM * lda), tile(BK * ldb), mk.alloc_tg(BM * ldc)
    acc = mk.mma_zero()
    for k0 in range(0, K, BK):
        for i in range(0, BM * BK, NT):
            e = tid + i
            r, q = e // BK, e % BK
            inside = e < BM * BK
            ok = mk.where(inside, mk.where(base_m + r < M, k0 + q < K, False), False)
            mk.store(As, r * lda + q, rounded(mk.load(a, (base_m + r) * K + k0 + q, ok)), inside)
        for i in range(0, BK * BN, NT):
            e = tid + i
            r, q = e // BN, e % BN
            inside = e < BK * BN
            ok = mk.where(inside, mk.where(k0 + r < K, base_n + q < N, False), False)
            mk.store(Bs, r * ldb + q, rounded(mk.load(b, (k0 + r) * N + base_n + q, ok)), inside)
        mk.barrier()
        for kk in range(0, BK, 8):
            acc = mk.mma(As, sg_m * 8 * lda + kk, lda, Bs, kk * ldb + sg_n * 8, ldb, acc)
        mk.barrier()
    mk.mma_store(Cs, sg_m * 8 * ldc + sg_n * 8, ldc, acc)
    mk.barrier()
    for i in range(0, BM * BN, NT):
        e = tid + i
        r, q = e // BN, e % BN
        row, col = base_m + r, base_n + q
        mk.store(c, row * N + col, finish(mk.load(Cs, r * ldc + q, True)), mk.where(row < M, col < N, False))


@eas.kernel
def matmul_mma_kernel(a, b, c, M, N, BM: eas.constexpr, BN: eas.constexpr, BK: eas.constexpr,
                      K: eas.constexpr, NT: eas.constexpr):
    _mma_body(a, b, c, M, N, BM, BN, BK, K, NT, mk.alloc_tg_f16, mk.to_f16, lambda v: v)


@eas.kernel
def matmul_mma_f16out_kernel(a, b, c, M, N, BM: eas.constexpr, BN: eas.constexpr, BK: eas.constexpr,
                             K: eas.constexpr, NT: eas.constexpr):
    _mma_body(a, b, c, M, N, BM, BN, BK, K, NT, mk.alloc_tg_f16, mk.to_f16, mk.to_f16)


@eas.kernel
def matmul_mma_bf16_kernel(a, b, c, M, N, BM: eas.constexpr, BN: eas.constexpr, BK: eas.constexpr,
                           K: eas.constexpr, NT: eas.constexpr):
    _mma_body(a, b, c, M, N, BM, BN, BK, K, NT, mk.alloc_tg_bf16, mk.to_bf16, lambda v: v)


@eas.kernel
def matmul_mma_bf16out_kernel(a, b, c, M, N, BM: eas.constexpr, BN: eas.constexpr, BK: eas.constexpr,
                              K: eas.constexpr, NT: eas.constexpr):
    _mma_body(a, b, c, M, N, BM, BN, BK, K, NT, mk.alloc_tg_bf16, mk.to_bf16, mk.to_bf16)


_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2}


def _cdiv(a, b):
    return -(-a // b)


# -- the cases -----------------------------------------------------------------


def listed():
    return [
        # The smallest call: a vector that fits one CU, where a launch is all there is.
        {"name": "add_f32_1031", "kind": "add", "dtype": "f32", "N": 1031, "BLOCK": 256},
        # The elementwise headline: three 1 GiB streams.
        {"name": "add_f32_2e28", "kind": "add", "dtype": "f32", "N": 1 << 28, "BLOCK": 256},
        # A thread-per-element kernel on an ordinary vector of odd length.
        {"name": "fma_f32_odd", "kind": "fma", "dtype": "f32", "N": 9_999_991, "BLOCK": 256},
        # The first matmul a user writes, one thread per output.
        {"name": "naive_f32", "kind": "naive", "dtype": "f32", "M": 1000, "N": 1500, "K": 256, "BLOCK": 256},
        # fp32 matmul with threadgroup tiles, at its usual size.
        {"name": "tiled_f32_1024", "kind": "tiled", "dtype": "f32", "M": 1024, "N": 1024, "K": 1024},
        # The same on a shape whose rows have no alignment (feature counts are what the data has).
        {"name": "tiled_f32_odd", "kind": "tiled", "dtype": "f32", "M": 1021, "N": 1531, "K": 771},
        # The matmul headline: f16 operands, f32 result.
        {"name": "mma_f16_4096", "kind": "mma", "dtype": "f16", "out": "f32", "M": 4096, "N": 4096, "K": 4096},
        # 16-bit operands whose rows start at odd addresses: a vocabulary or feature count as it comes.
        {"name": "mma_f16_odd", "kind": "mma", "dtype": "f16", "out": "f32", "M": 1531, "N": 2047, "K": 1023},
        # fp32 tensors multiplied on the 16-bit matrix cores (the kernel rounds while loading).
        {"name": "mma_f32in", "kind": "mma", "dtype": "f32", "out": "f32", "M": 1024, "N": 2048, "K": 2048},
        # A linear layer on a chunk of a prompt, in bf16.
        {"name": "chunk_bf16", "kind": "mma", "dtype": "bf16", "out": "bf16", "M": 512, "N": 14336, "K": 4096},
        # A linear layer on one decode step of 16 sequences: the weights are read once.
        {"name": "decode_f16", "kind": "mma", "dtype": "f16", "out": "f16", "M": 16, "N": 14336, "K": 4096},
        # The largest: a square linear layer on a whole prompt.
        {"name": "prefill_f16", "kind": "mma", "dtype": "f16", "out": "f16", "M": 8192, "N": 8192, "K": 8192},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extent(rng, lo, hi, steps=(1, 1, 2, 8, 64)):
    """An extent of [lo, hi], log-uniform; as it comes, or rounded to a multiple."""
    step = rng.choice(steps)
    return max(lo, _cdiv(_log_int(rng, lo, hi), step) * step)


def draw(rng):
    kind = rng.choice(["add", "fma", "naive", "tiled", "tiled", "mma", "mma", "mma", "linear", "linear"])
    if kind in ("add", "fma"):
        dtype = "f32" if kind == "fma" else rng.choice(["f32", "f16", "bf16"])
        return {"kind": kind, "dtype": dtype, "N": _extent(rng, 1000, 1 << 27, (1, 1, 64)),
                "BLOCK": rng.choice([256, 1024])}
    if kind == "naive":
        return {"kind": "naive", "dtype": "f32", "M": _extent(rng, 32, 2000), "N": _extent(rng, 32, 2000),
                "K": _extent(rng, 16, 512), "BLOCK": rng.choice([64, 256])}
    if kind == "tiled":
        return {"kind": "tiled", "dtype": "f32", "M": _extent(rng, 48, 2048), "N": _extent(rng, 48, 2048),
                "K": _extent(rng, 32, 2048)}
    dtype = rng.choice(["f16", "f16", "bf16", "f32"])
    if kind == "mma":  # any matmul, f32 result
        return {"kind": "mma", "dtype": dtype, "out": "f32", "M": _extent(rng, 130, 3000),
                "N": _extent(rng, 64, 3000), "K": _extent(rng, 32, 3000)}
    # a linear layer: few or many rows, its widths multiples of 64 more often than not
    dtype = "f16" if dtype == "f32" else dtype
    steps = (1, 8, 64, 64, 64)
    return {"kind": "mma", "dtype": dtype, "out": dtype, "M": _extent(rng, 1, 1024, (1,)),
            "N": _extent(rng, 512, 14336, steps), "K": _extent(rng, 512, 4096, steps)}


def _inputs(case, seed):
    """The operands, made from the seed alone: N(0, 1) vectors, N(0, 1/K) fp32 matrices, U(-1, 1)
    matrices for the MMA, and N(0, 1) activations with N(0, 0.02) weights for a linear layer."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    dt = _TORCH[case["dtype"]]

    def normal(n, scale):
        return torch.empty(n, device="cuda").normal_(0.0, scale, generator=g).to(dt)

    if case["kind"] in ("add", "fma"):
        return [normal(case["N"], 1.0) for _ in range(2 if case["kind"] == "add" else 3)]
    m, n, k = case["M"], case["N"], case["K"]
    if case["kind"] in ("naive", "tiled"):
        return [normal(m * k, k ** -0.5), normal(k * n, k ** -0.5)]
    if case["out"] == "f32":
        return [torch.empty(s, device="cuda").uniform_(-1.0, 1.0, generator=g).to(dt) for s in (m * k, k * n)]
    return [normal(m * k, 1.0), normal(k * n, 0.02)]


def prepare(case, seed):
    """The tensors in hand before the call, and the call's kernel and options."""
    ins = _inputs(case, seed)
    kind, dt = case["kind"], _TORCH[case["dtype"]]
    if kind in ("add", "fma"):
        out = torch.empty(case["N"], device="cuda", dtype=dt)
        kernel = add_kernel if kind == "add" else fma_kernel
        return {"kernel": kernel, "args": (*ins, out, case["N"]), "opts": {"BLOCK": case["BLOCK"]}, "out": out}
    m, n, k = case["M"], case["N"], case["K"]
    out = torch.empty(m * n, device="cuda", dtype=_TORCH[case.get("out", "f32")])
    if kind == "naive":
        kernel, opts = matmul_kernel, {"BLOCK": case["BLOCK"], "K": k, "_grid": (m, _cdiv(n, case["BLOCK"]))}
    elif kind == "tiled":
        kernel = matmul_tiled_kernel
        opts = {"BM": 32, "BN": 32, "BK": 32, "K": k, "NT": 256, "_grid": (_cdiv(n, 32), _cdiv(m, 32))}
    else:
        kernel = {("f16", "f32"): matmul_mma_kernel, ("f32", "f32"): matmul_mma_kernel,
                  ("f16", "f16"): matmul_mma_f16out_kernel, ("bf16", "f32"): matmul_mma_bf16_kernel,
                  ("bf16", "bf16"): matmul_mma_bf16out_kernel}[case["dtype"], case["out"]]
        opts = {"BM": 32, "BN": 32, "BK": 32, "K": k, "NT": 512, "_grid": (_cdiv(n, 32), _cdiv(m, 32))}
    args = (*ins, out, m, n)
    kernel.compile(*args, **opts)
    return {"kernel": kernel, "args": args, "opts": opts, "out": out}


def run(state):
    """One call, on torch's current stream and without waiting for it."""
    state["kernel"](*state["args"], **state["opts"], _sync=False)
    return state["out"]


def work(case):
    size = _BYTES[case["dtype"]]
    if case["kind"] == "add":
        return {"bytes": 3 * size * case["N"], "flops": case["N"]}
    if case["kind"] == "fma":
        return {"bytes": 4 * size * case["N"], "flops": 2 * case["N"]}
    m, n, k = case["M"], case["N"], case["K"]
    return {"bytes": size * (m * k + k * n) + _BYTES[case.get("out", "f32")] * m * n, "flops": 2 * m * n * k}


def tolerance(case):
    if case["kind"] in ("add", "fma"):
        return "exact"
    # about four times the distance from 64 bits that was measured
    if case["kind"] in ("naive", "tiled"):
        return {"rel": 3e-6}  # f32 products and sums over up to 2048 terms (5.7e-7 at 1024)
    if case["out"] == "f32":
        return {"rel": 2e-6}  # exact products of 16-bit operands, f32 sums (4.1e-7 at 4096 terms)
    # the f32 sum rounded once to f16 (2.1e-4) or bf16 (1.7e-3)
    return {"rel": 8e-4 if case["out"] == "f16" else 7e-3}


def exact(case, seed):
    ins = _inputs(case, seed)
    if case["kind"] == "add":
        return ins[0].double() + ins[1].double()
    if case["kind"] == "fma":
        return ins[0].double() * ins[1].double() + ins[2].double()
    m, n, k = case["M"], case["N"], case["K"]
    a, b = ins[0].view(m, k), ins[1].view(k, n)
    if case["kind"] == "mma" and case["dtype"] == "f32":  # the kernel multiplies f16 values
        a, b = a.half(), b.half()
    return (a.double() @ b.double()).view(-1)
