"""GEMM launches whose operands the DMA cannot take (odd K, odd row stride, odd addresses, f32 inputs) on the
register bodies of the main entry: every tile, the ends of rows and of the buffers, K below and around a
stage.  Each output against float64 of the rounded operands (max|C - R| <= 1e-5 sqrt(K) max|R|: f16 products
are exact in f32); a row of NaN past the rectangle, a NaN column beside it and a sentinel after C must not be
read into, or written by, the launch.
"""

from __future__ import annotations

import math
import struct

import numpy as np
import pytest

import kernels as K
from easy_as_amd.codegen.gemm_lift import REGISTER_TILES, _register_tiles
from easy_as_amd.runtime.hip import plan_launch


def test_register_tile_rule():
    # the tile with the least rounds x time per round, the larger of equals
    for m, n, cus in ((1531, 2047, 256), (300, 700, 256), (700, 1501, 256), (2999, 2999, 256), (4095, 4095, 80),
                      (129, 1, 256), (1 << 20, 3, 256)):
        cost = {-(-m // bm) * -(-n // bn): -(-(-(-m // bm) * -(-n // bn)) // cus) * w for bm, bn, w in REGISTER_TILES}
        assert cost[_register_tiles(m, n, cus)] == min(cost.values())
    assert _register_tiles(1531, 2047, 256) == 12 * 16  # 128 x 128
    assert _register_tiles(300, 700, 256) == 5 * 11     # 64 x 64
    assert _register_tiles(700, 1501, 256) == 6 * 24    # 128 x 64
    assert _register_tiles(2999, 2999, 256) == 12 * 12  # 256 x 256


def _run(rt, m, n, k, dtype, grid=None, pad=0):
    """C of an m x n x k launch on its plan's grid (or `grid` workgroups), with B's rows `pad` wider than the
    launch: the rectangle then ends before its rows do."""
    import torch

    rng = np.random.default_rng(m * 7 + n * 3 + k)
    a = rng.uniform(-1, 1, (m, k)).astype(np.float16).astype(np.float32)
    b = rng.uniform(-1, 1, (k, n + pad)).astype(np.float16).astype(np.float32)
    td = {"f16": torch.float16, "f32": torch.float32, "bf16": torch.bfloat16}[dtype]
    if dtype == "bf16":
        a = torch.from_numpy(a).to(td).float().numpy()
        b = torch.from_numpy(b).to(td).float().numpy()
    if pad:
        b[:, n:] = np.nan
    # a NaN right after the last element of each operand: what lies past the end never reaches C
    ta = torch.full((m * k + 8,), float("nan"), dtype=td, device="cuda")
    tb = torch.full((k * (n + pad) + 8,), float("nan"), dtype=td, device="cuda")
    ta[:m * k] = torch.from_numpy(a.reshape(-1)).to("cuda", td)
    tb[:k * (n + pad)] = torch.from_numpy(b.reshape(-1)).to("cuda", td)
    tc = torch.full((m * (n + pad) + 64,), -7.0, device="cuda")
    kern = K.matmul_mma_bf16_kernel if dtype == "bf16" else K.matmul_mma_kernel
    ck = kern.compile(ta, tb, tc, m, n + pad, BM=32, BN=32, BK=8, K=k, NT=512)
    assert ck.geometry.kind == "gemm"
    args = {"a": ta[:m * k], "b": tb[:k * (n + pad)], "c": tc, "M": m, "N": n + pad}
    plan = plan_launch(ck, args, grid=(K.cdiv(n, 32), K.cdiv(m, 32), 1))
    assert plan.entry is None and plan.block == (256, 1, 1)
    n_hi = min(n + pad, K.cdiv(n, 32) * 32)
    assert plan.hidden == (0, m, 0, n_hi)
    argv, writable, _, stream = rt.build_argv(ck.ir, args, ck.writes)
    argv += [struct.pack("<I", h) for h in plan.hidden]
    rt._mod().launch_groups(rt.kernel_handle(ck, None), argv, writable + [False] * 4,
                            (grid, 1, 1) if grid else plan.grid, plan.block, stream=stream)
    torch.cuda.synchronize()
    c = tc.cpu().numpy()
    assert (c[m * (n + pad):] == -7.0).all()
    c = c[:m * (n + pad)].reshape(m, n + pad)
    assert (c[:, n_hi:] == -7.0).all()
    r = a.astype(np.float64) @ b[:, :n].astype(np.float64)
    assert np.abs(c[:, :n] - r).max() <= 1e-5 * math.sqrt(k) * np.abs(r).max()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [(bm, bn) for bm, bn, _ in REGISTER_TILES], ids=lambda t: f"{t[0]}x{t[1]}")
@pytest.mark.parametrize("mnk,dtype", [((129, 65, 8), "f32"), ((257, 9, 9), "f16"), ((130, 255, 31), "f16"),
                                       ((131, 257, 63), "bf16"), ((200, 130, 64), "f32"), ((259, 129, 65), "f16"),
                                       ((300, 301, 127), "bf16"), ((513, 519, 129), "f16"), ((140, 66, 515), "f32"),
                                       ((140, 67, 514), "f16")])
def test_register_tiles_every_output(gpu_runtime, tile, mnk, dtype):
    m, n, k = mnk
    _run(gpu_runtime, m, n, k, dtype, grid=K.cdiv(m, tile[0]) * K.cdiv(n, tile[1]))


@pytest.mark.gpu
@pytest.mark.parametrize("mnk,dtype", [((1, 9, 8), "f32"), ((7, 101, 33), "f16"), ((16, 63, 1023), "f16"),
                                       ((17, 65, 129), "bf16"), ((33, 130, 257), "f32"), ((64, 129, 97), "f16"),
                                       # above 64 rows: 64 x 64 tiles
                                       ((65, 130, 257), "f32"), ((128, 129, 97), "f16"), ((100, 1001, 65), "bf16"),
                                       # rows below 8 elements: one f32 dot product per output
                                       ((5, 7, 64), "f16"), ((40, 9, 7), "f32"), ((130, 5, 33), "f16"),
                                       ((130, 30, 3), "f32")])
def test_few_rows_and_short_rows(gpu_runtime, mnk, dtype):
    _run(gpu_runtime, *mnk, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("mnk,dtype", [((140, 96, 65), "f16"), ((20, 64, 70), "f32"), ((300, 160, 64), "f32")])
def test_a_rectangle_that_ends_inside_its_rows(gpu_runtime, mnk, dtype):
    _run(gpu_runtime, *mnk, dtype, pad=3)


@pytest.mark.gpu
@pytest.mark.parametrize("mnk,dtype", [((100, 129, 65), "f16"), ((65, 200, 72), "f32"), ((128, 130, 48), "bf16")])
def test_guard_of_a_few_row_grid_above_64_rows(gpu_runtime, mnk, dtype):
    # one workgroup per 64 columns for operands the DMA cannot take: the plan launches tiles instead
    _run(gpu_runtime, *mnk, dtype, grid=K.cdiv(mnk[1], 64), pad=mnk[1] == 130)


@pytest.mark.gpu
@pytest.mark.parametrize("mnk,dtype", [((29, 130, 1023), "f16"), ((55, 200, 1000), "f32"), ((40, 131, 771), "bf16"),
                                       ((9, 129, 1541), "bf16"), ((14, 96, 776), "f32"), ((61, 67, 1031), "f16"),
                                       ((20, 72, 1030), "f16"),
                                       # over 256 groups of 64 columns: two of them, in turn, on the same LDS
                                       ((20, 16451, 771), "f16"), ((50, 16450, 1000), "f32"), ((7, 16391, 1023), "bf16")])
def test_few_rows_steady_loop(gpu_runtime, mnk, dtype):
    # K above 512: each of the four waves has more than the 4 stages of 32 k that the loop without a branch needs
    _run(gpu_runtime, *mnk, dtype)
