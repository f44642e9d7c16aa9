"""The one-thread-per-output matmul (examples/matmul.py:23-43) on its ordered fp32 GEMM: which kernels are lifted,
which launches take it, and every output bit for bit against the fma chain over ascending k (a NaN has to stay a
NaN), with subnormals, underflow to -0, infinities and NaN among the operands."""

from __future__ import annotations

import numpy as np
import pytest

import eas
import kernels as K
from eas import mk
from easy_as_amd.codegen.gemm_lift import Unsupported, analyze_chain
from easy_as_amd.runtime.hip import plan_launch
from oracle import ops


@eas.kernel
def chain_variant_kernel(a, b, c, M, N, BLOCK: eas.constexpr, K: eas.constexpr, VARIANT: eas.constexpr):
    """K.matmul_kernel with one change; 0, 8 and 9 are the same matmul, 1-7 are not."""
    V = VARIANT
    row = mk.program_id(1 if V == 8 else 0)
    col = mk.program_id(0 if V == 8 else 1) * BLOCK + mk.tid(0, BLOCK)
    mask = mk.where(row < M, col < N, False)
    if V == 1:
        mask = row < M
    if V == 2:
        mask = mk.where(row < N, col < M, False)
    acc = mk.load(c, 0, mask) if V == 3 else (1.0 if V == 4 else 0.0)
    for k in reversed(range(K)) if V == 5 else range(K):
        x, y = mk.load(a, row * K + k, mask), mk.load(b, k * (M if V == 6 else N) + col, mask)
        acc = acc + (y * x if V == 9 else x * y)
    mk.store(c, col * N + row if V == 7 else row * N + col, acc, mask)


@pytest.mark.parametrize("variant", range(10))
def test_which_kernels_are_lifted(variant):
    f = np.zeros(8, np.float32)
    ck = chain_variant_kernel.compile(f, f, f, 8, 8, BLOCK=64, K=5, VARIANT=variant)
    lifted = variant in (0, 8, 9)
    assert ("gemm" in ck.geometry.params) == lifted and ck.geometry.kind == "thread"
    if lifted:
        spec = analyze_chain(ck.ir, 64)
        assert (spec.a, spec.b, spec.c, spec.m_sym, spec.n_sym) == ("a", "b", "c", "M", "N")
        assert spec.ordered and spec.K == 5 and (spec.TM, spec.TN) == (1, 64) and spec.row_axis == (variant == 8)
    else:
        with pytest.raises(Unsupported):
            analyze_chain(ck.ir, 64)


def test_which_launches_take_the_gemm():
    f = np.zeros(64, np.float32)
    ck = K.matmul_kernel.compile(f, f, f, 8, 8, BLOCK=64, K=5)
    buf = {"a": np.zeros(500 * 5, np.float32), "b": np.zeros(5 * 300, np.float32), "c": np.zeros(500 * 300, np.float32)}
    plan = plan_launch(ck, {**buf, "M": 500, "N": 300}, grid=(500, 5, 1))
    assert plan.entry == "matmul_kernel__mm" and plan.hidden == (0, 500, 0, 300) and plan.grid == (8 * 5, 1, 1)
    plan = plan_launch(ck, {**buf, "M": 500, "N": 300}, grid=(7, 2, 1))  # 7 rows, 128 columns
    assert plan.entry == "matmul_kernel__mm" and plan.hidden == (0, 7, 0, 128)
    with pytest.raises(ValueError):  # a two-dimensional kernel without a grid, as ever
        plan_launch(ck, {**buf, "M": 500, "N": 300}, nthreads=300)
    # a buffer the matrices do not fit, indices past 2^32: the kernel's own threads
    plan = plan_launch(ck, {**buf, "M": 501, "N": 300}, grid=(501, 5, 1))
    assert plan.entry is None and plan.grid == (501, 5, 1) and plan.hidden == (501 * 64,)
    plan = plan_launch(ck, {"M": 1 << 31, "N": 300}, grid=(1 << 22, 5, 1))
    assert plan.entry == "matmul_kernel__mm"
    plan = plan_launch(ck, {"M": 1 << 31, "N": 300}, grid=(1 << 25, 5, 1))
    assert plan.entry is None
    assert plan_launch(ck, {**buf, "M": 0, "N": 300}, grid=(4, 5, 1)) is None


def _chain(a, b):
    s = np.zeros((a.shape[0], b.shape[1]), np.float32)
    for k in range(a.shape[1]):
        s = ops.fmaf(np.ascontiguousarray(np.broadcast_to(a[:, k:k + 1], s.shape)).reshape(-1),
                     np.ascontiguousarray(np.broadcast_to(b[k:k + 1], s.shape)).reshape(-1), s.reshape(-1)).reshape(s.shape)
    return s


@pytest.mark.gpu
@pytest.mark.parametrize("entry", ["auto", "tile128"])
@pytest.mark.parametrize("mnk", [(1, 1, 1), (3, 65, 2), (37, 130, 5), (65, 64, 31), (130, 131, 32), (64, 63, 33),
                                 (129, 257, 64), (200, 70, 100), (33, 129, 131)])
@pytest.mark.parametrize("values", ["normal", "tiny", "special"])
def test_bit_exact(gpu_runtime, monkeypatch, mnk, entry, values):
    import torch

    monkeypatch.setenv("EAS_HIP_GEMM_ENTRY", entry)
    m, n, k = mnk
    rng = np.random.default_rng(m + n + k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    if values == "tiny":  # products around the smallest subnormal: many round to +-0
        a, b = (np.ldexp(x, rng.integers(-77, -70, x.shape)).astype(np.float32) for x in (a, b))
    if values == "special":
        for x in (a, b):
            u = rng.integers(0, 60, x.shape)
            for i, v in enumerate((np.inf, -np.inf, -0.0, 3e38, 1e-42, np.nan)):
                x[u == i] = v
    ta, tb = (torch.full((x.size + 4,), float("nan"), device="cuda") for x in (a, b))
    ta[:a.size], tb[:b.size] = torch.from_numpy(a.reshape(-1)).cuda(), torch.from_numpy(b.reshape(-1)).cuda()
    tc = torch.full((m * n + 64,), -7.0, device="cuda")
    K.matmul_kernel(ta[:a.size], tb[:b.size], tc, m, n, BLOCK=64, K=k, _grid=(m, K.cdiv(n, 64)))
    c = tc.cpu().numpy()
    assert (c[m * n:] == -7.0).all()
    got, want = c[:m * n].reshape(m, n), _chain(a, b)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.array_equal(got[ok].view(np.uint32), want[ok].view(np.uint32))
    if values == "tiny" and m * n > 1000 and k < 3:
        assert np.signbit(want[want == 0]).any()


@pytest.mark.gpu
def test_native_launches_and_a_thread_count(gpu_runtime):
    """The reference's launch(pipeline, argv, writable, threads, threadgroup): whole threadgroups run the GEMM, any
    other thread count the kernel's own threads; both the same bits."""
    import struct

    import torch

    hip = gpu_runtime._mod()
    m, n, k = 40, 100, 33
    rng = np.random.default_rng(3)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    ta, tb = torch.from_numpy(a.reshape(-1)).cuda(), torch.from_numpy(b.reshape(-1)).cuda()
    ck = K.matmul_kernel.compile(ta, tb, ta, m, n, BLOCK=64, K=k)
    kern = hip.compile(ck.src, "matmul_kernel")
    want = _chain(a, b)
    for threads, rows in ((m * 64, m), (m * 64 - 1, m - 1)):
        tc = torch.full((m * n,), float("nan"), device="cuda")
        argv = [hip.wrap_pointer(t.data_ptr(), t.numel() * 4) for t in (ta, tb, tc)]
        torch.cuda.synchronize()
        hip.launch(kern, argv + [struct.pack("<I", m), struct.pack("<I", n)], [False, False, True, False, False],
                   (threads, 2, 1), (64, 1, 1))
        torch.cuda.synchronize()
        got = tc.cpu().numpy().reshape(m, n)
        assert np.array_equal(got[:rows].view(np.uint32), want[:rows].view(np.uint32))
    # the last thread of the last row's threadgroups was left out
    assert np.isnan(got[m - 1, 63]) and np.array_equal(got[m - 1, :63], want[m - 1, :63])


@pytest.mark.gpu
@pytest.mark.parametrize("mnk", [(65, 64, 31), (130, 131, 32), (64, 63, 33), (37, 130, 46), (129, 70, 9)])
@pytest.mark.parametrize("values", ["normal", "tiny", "special"])
def test_bit_exact_on_64_tiles_with_a_short_k(gpu_runtime, monkeypatch, mnk, values):
    """K of 8 to 48 on a small output runs on the kernel's threads unless an entry is named; here the 64 x 64 tiles."""
    m, n, k = mnk
    f = np.zeros(8, np.float32)
    ck = K.matmul_kernel.compile(f, f, f, m, n, BLOCK=64, K=k)
    assert plan_launch(ck, {"M": m, "N": n}, grid=(m, K.cdiv(n, 64), 1)).entry is None
    monkeypatch.setenv("EAS_HIP_GEMM_ENTRY", "4wave")
    assert plan_launch(ck, {"M": m, "N": n}, grid=(m, K.cdiv(n, 64), 1)).entry == "matmul_kernel__mm"
    test_bit_exact(gpu_runtime, monkeypatch, mnk, "4wave", values)


@pytest.mark.gpu
@pytest.mark.parametrize("mnk", [(130, 131, 257), (70, 300, 259), (129, 257, 290), (200, 70, 287), (65, 129, 319)])
@pytest.mark.parametrize("values", ["normal", "tiny", "special"])
def test_bit_exact_on_128_tiles_with_a_k_tail(gpu_runtime, monkeypatch, mnk, values):
    """K off a multiple of 4: the chunk of A that straddles K, with 9 and with 10 stages."""
    m, n, k = mnk
    f = np.zeros(8, np.float32)
    ck = K.matmul_kernel.compile(f, f, f, m, n, BLOCK=64, K=k)
    monkeypatch.setenv("EAS_HIP_GEMM_ENTRY", "tile128")
    plan = plan_launch(ck, {"M": m, "N": n}, grid=(m, K.cdiv(n, 64), 1))
    assert plan.entry == "matmul_kernel__mm__t128" and plan.grid == (K.cdiv(m, 128) * K.cdiv(n, 128), 1, 1)
    test_bit_exact(gpu_runtime, monkeypatch, mnk, "tile128", values)
