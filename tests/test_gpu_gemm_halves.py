"""The f16 smaller-tile entries' stages of two halves of 32 k: K of one half, one stage, an odd number of halves, tails
of 2 to 8; N whose 8-column chunk straddles the edge, rows of under 8 columns.  Each output against float64
(<= 1e-5 sqrt(K) max|R|); a NaN right after each operand must not reach C, and nothing is written past it."""

from __future__ import annotations

import math

import numpy as np
import pytest

import kernels as K
from easy_as_amd.runtime.hip import plan_launch

pytestmark = pytest.mark.gpu

_ENTRIES = {"tile64": "__t64x64", "tile128x64": "__t128x64", "tile128": "__t128", "tile128x256": "__t128x256"}


@pytest.mark.parametrize("choice", list(_ENTRIES))
@pytest.mark.parametrize("mnk", [(129, 66, 2), (130, 64, 30), (131, 130, 32), (193, 258, 34), (129, 262, 62),
                                 (257, 132, 64), (140, 126, 66), (150, 300, 96), (129, 6, 98), (200, 190, 100),
                                 (129, 2, 160), (300, 520, 258)])
def test_halves(gpu_runtime, monkeypatch, mnk, choice):
    import torch

    monkeypatch.setenv("EAS_HIP_GEMM_ENTRY", choice)
    m, n, k = mnk
    rng = np.random.default_rng(m + n + k)
    a, b = (rng.uniform(-1, 1, s).astype(np.float16) for s in ((m, k), (k, n)))
    ta, tb = (torch.full((x.size + 8,), float("nan"), dtype=torch.float16, device="cuda") for x in (a, b))
    ta[:a.size], tb[:b.size] = torch.from_numpy(a.reshape(-1)).cuda(), torch.from_numpy(b.reshape(-1)).cuda()
    tc = torch.full((m * n + 64,), -7.0, device="cuda")
    args, opts = (ta[:a.size], tb[:b.size], tc, m, n), dict(BM=32, BN=32, BK=8, K=k, NT=512)
    grid = (K.cdiv(n, 32), K.cdiv(m, 32), 1)
    ck = K.matmul_mma_kernel.compile(*args, **opts)
    plan = plan_launch(ck, dict(zip((x.name for x in ck.ir.args), args)), grid=grid)
    assert plan.entry == "matmul_mma_kernel" + _ENTRIES[choice]
    K.matmul_mma_kernel(*args, **opts, _grid=grid)
    c = tc.cpu().numpy()
    assert (c[m * n:] == -7.0).all()
    r = a.astype(np.float64) @ b.astype(np.float64)
    assert np.abs(c[:m * n].reshape(m, n) - r).max() <= 1e-5 * math.sqrt(k) * np.abs(r).max()
