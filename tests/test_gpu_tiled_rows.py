"""The fp32 tiled matmul on rows of any length (K, N not multiples of 4) through the DMA entries: the chunk that
straddles the end of a row of A, the one that straddles N, K below and around a stage, both entries.  Each output
against float64 (max|C - R| <= 1e-5 sqrt(K) max|R|); a NaN right after each operand must not reach C, and nothing
is written past it."""

from __future__ import annotations

import math

import numpy as np
import pytest

import kernels as K
from easy_as_amd.runtime.hip import plan_launch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entry", ["auto", "tile128"])
@pytest.mark.parametrize("mnk", [(1, 1, 1), (3, 5, 3), (65, 67, 31), (64, 66, 33), (130, 129, 62), (129, 131, 64),
                                 (70, 333, 127), (257, 63, 130), (33, 259, 771), (200, 301, 100), (128, 126, 2),
                                 (130, 129, 257), (129, 131, 290), (70, 333, 287), (257, 63, 319)])
def test_rows_of_any_length(gpu_runtime, monkeypatch, mnk, entry):
    import torch

    monkeypatch.setenv("EAS_HIP_GEMM_ENTRY", entry)
    m, n, k = mnk
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    ta, tb = (torch.full((x.size + 4,), float("nan"), device="cuda") for x in (a, b))
    ta[:m * k] = torch.from_numpy(a.reshape(-1)).cuda()
    tb[:k * n] = torch.from_numpy(b.reshape(-1)).cuda()
    tc = torch.full((m * n + 64,), -7.0, device="cuda")
    kern, args = K.matmul_tiled_kernel, (ta[:m * k], tb[:k * n], tc, m, n, 0, 0)
    grid = (K.cdiv(n, 32), K.cdiv(m, 32), 1)
    opts = dict(BM=32, BN=32, BK=32, K=k, NT=256)
    ck = kern.compile(*args, **opts)
    plan = plan_launch(ck, dict(zip((x.name for x in ck.ir.args), args)), grid=grid)
    assert plan.entry == ("matmul_tiled_kernel__t128" if entry == "tile128" and (k % 4 == 0 or k >= 256) else None)
    kern(*args, **opts, _grid=grid)
    c = tc.cpu().numpy()
    assert (c[m * n:] == -7.0).all()
    r = a.astype(np.float64) @ b
    assert np.abs(c[:m * n].reshape(m, n) - r).max() <= 1e-5 * math.sqrt(k) * np.abs(r).max()
