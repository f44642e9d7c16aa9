"""Launches of 17-128 rows by the alignment of their rows: 16 bytes the skinny path; above 64 rows 4 bytes a DMA entry's
tile (64 x 64, 128 x 64, 128 x 128: the smallest of one round of CUs) and any others 64 x 64 register tiles.  The
Python and the C planner alike, and on the GPU each output against float64."""

from __future__ import annotations

import math

import numpy as np
import pytest

import kernels as K
from easy_as_amd.runtime import hip_ext
from easy_as_amd.runtime.hip import pack_scalar, plan_launch


class _Buf:
    def __init__(self, numel, ptr):
        self.n, self.ptr = numel, ptr

    def numel(self):
        return self.n

    def data_ptr(self):
        return self.ptr


def _plans(m, n, k, off=(0, 0), choice="auto"):
    """(Python plan, C plan) as (grid, block, hidden, entry's suffix); off: bytes A and B lie past a 256-byte boundary."""
    hip = hip_ext.load_hip_ext(require=True)
    f16, f32 = np.zeros(1, np.float16), np.zeros(1, np.float32)
    ck = K.matmul_mma_kernel.compile(f16, f16, f32, m, n, BM=32, BN=32, BK=8, K=k, NT=512)
    args = {"a": _Buf(m * k, (1 << 30) + off[0]), "b": _Buf(k * n, (2 << 30) + off[1]), "c": _Buf(m * n, 3 << 30),
            "M": m, "N": n}
    groups = (K.cdiv(n, 32), K.cdiv(m, 32), 1)
    p = plan_launch(ck, args, grid=groups, compute_units=256)
    size = {"a": 2, "b": 2, "c": 4}
    argv = [hip.wrap_pointer(args[a.name].ptr, args[a.name].n * size[a.name]) if a.kind == "buffer"
            else pack_scalar(a.dtype, args[a.name]) for a in ck.ir.args]
    c = hip.plan_dispatch(ck.src, groups, (512, 1, 1), True, argv=argv, compute_units=256, entry_choice=choice)
    suffix = lambda e: None if e is None else e[len("matmul_mma_kernel"):]  # noqa: E731
    return (p.grid, p.block, p.hidden, suffix(p.entry)), (*c[:3], suffix(c[3]))


@pytest.mark.parametrize("m,n,k,off,entry,grid", [
    # rows at 16 bytes: the skinny path
    (100, 4096, 1024, (0, 0), None, 64), (65, 4096, 1024, (16, 32), None, 64),
    # at 4 bytes: the smallest tile of one round of CUs
    (100, 4098, 1022, (0, 0), "__t64x64", 130), (100, 4096, 1022, (0, 0), "__t64x64", 128),
    (100, 4098, 1024, (0, 0), "__t64x64", 130), (100, 4096, 1024, (8, 0), "__t64x64", 128),
    (65, 4096, 1024, (0, 4), "__t64x64", 128), (128, 8192, 1022, (0, 0), "__t64x64", 256),
    (128, 8194, 1022, (0, 0), "__t128x64", 129), (128, 16384, 1022, (0, 0), "__t128x64", 256),
    (128, 16390, 1000, (0, 0), "__t128", 129), (128, 40962, 1000, (0, 0), "__t128", 321),
    # odd rows or addresses: register tiles
    (100, 4097, 1023, (0, 0), None, 130), (100, 4096, 1024, (2, 0), None, 128), (100, 4098, 1022, (0, 2), None, 130),
    # up to 64 rows every operand takes the skinny grid
    (64, 4098, 1022, (0, 0), None, 65), (17, 4097, 1023, (0, 0), None, 65), (64, 4096, 1024, (2, 0), None, 64)])
def test_few_rows_by_alignment(m, n, k, off, entry, grid):
    py, c = _plans(m, n, k, off)
    assert py == c and py[3] == entry and py[0] == (grid, 1, 1)


@pytest.mark.parametrize("choice", ["8wave", "tile128", "tile128x256", "tile128x64", "tile64", "4wave"])
def test_a_named_entry(monkeypatch, choice):
    monkeypatch.setenv("EAS_HIP_GEMM_ENTRY", choice)
    for m, n, k in ((100, 4098, 1022), (100, 4097, 1023), (100, 4096, 1024), (40, 4098, 1022)):
        py, c = _plans(m, n, k, choice=choice)
        assert py == c
        if choice == "4wave":  # 64 x 64 register tiles, but for what the skinny path takes
            assert py[3] is None and py[0][0] == (64 if n == 4096 else 65 if m == 40 else 130)


@pytest.mark.gpu
@pytest.mark.parametrize("mnk,off", [((100, 4098, 1022), 0), ((65, 130, 258), 0), ((128, 8194, 130), 0),
                                     ((127, 16390, 66), 0), ((100, 264, 520), 4), ((100, 264, 520), 8),
                                     ((100, 264, 520), 1)])
@pytest.mark.parametrize("eas_tensor", [False, True])
def test_outputs(gpu_runtime, mnk, off, eas_tensor):
    """A and B start `off` elements into their allocations; an eas.Tensor of such memory is planned by its address too."""
    import torch

    import eas

    m, n, k = mnk
    rng = np.random.default_rng(m + n + k)
    a, b = (rng.uniform(-1, 1, s).astype(np.float16) for s in ((m, k), (k, n)))
    ta, tb = (torch.full((x.size + off + 8,), float("nan"), dtype=torch.float16, device="cuda") for x in (a, b))
    for t, x in ((ta, a), (tb, b)):
        t[off:off + x.size] = torch.from_numpy(x.reshape(-1)).cuda()
    ta, tb = ta[off:off + a.size], tb[off:off + b.size]
    tc = torch.full((m * n + 64,), -7.0, device="cuda")
    args = [eas.tensor(t, device="hip") if eas_tensor else t for t in (ta, tb)]
    ck = K.matmul_mma_kernel.compile(*args, tc, m, n, BM=32, BN=32, BK=8, K=k, NT=512)
    grid = (K.cdiv(n, 32), K.cdiv(m, 32), 1)
    plan = plan_launch(ck, {"a": args[0], "b": args[1], "c": tc, "M": m, "N": n}, grid=grid, compute_units=256)
    tiles = [(K.cdiv(m, bm) * K.cdiv(n, bn), e) for bm, bn, e in ((64, 64, "__t64x64"), (128, 64, "__t128x64"),
                                                                  (128, 128, "__t128"))]
    want = (K.cdiv(n, 64), None) if off == 8 else (tiles[0][0], None) if off == 1 else \
        next((t for t in tiles if t[0] <= 256), tiles[2])
    assert plan.grid == (want[0], 1, 1) and plan.entry == (want[1] and "matmul_mma_kernel" + want[1])
    K.matmul_mma_kernel(*args, tc, m, n, BM=32, BN=32, BK=8, K=k, NT=512, _grid=grid)
    torch.cuda.synchronize()
    c = tc.cpu().numpy()
    assert (c[m * n:] == -7.0).all()
    r = a.astype(np.float64) @ b.astype(np.float64)
    assert np.abs(c[:m * n].reshape(m, n) - r).max() <= 1e-5 * math.sqrt(k) * np.abs(r).max()
