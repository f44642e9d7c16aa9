"""16-bit GEMMs with rows of under 8 elements (K or N), one f32 dot product per output: below and above 64 and 128 rows,
rectangles inside wider rows, tiles past the edge.  Each output against float64 (<= 1e-5 sqrt(K) max|R|); NaN right
after the operands and a sentinel after C stay out of it.  And that no thread goes to a place outside C: a launch of N
columns takes as many turns as it has outputs for its threads."""

from __future__ import annotations

import math
import re

import numpy as np
import pytest

import kernels as K


def test_the_loop_runs_over_outputs():
    f16, f32 = np.zeros(1, np.float16), np.zeros(1, np.float32)
    src = K.matmul_mma_kernel.compile(f16, f16, f32, 8, 8, BM=32, BN=32, BK=8, K=63, NT=512).src
    body = re.search(r"void eas_gemm_elementwise\(.*?\n}\n", src, re.S).group(0)
    assert "min(TM, M - m0)" in body and "e < h * w" in body and "continue" not in body


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("mnk,pad", [((1, 1, 1023), 0), ((16, 1, 64), 0), ((64, 7, 130), 0), ((65, 5, 33), 0), ((128, 1, 257), 0),
                                     ((130, 1, 1024), 0), ((300, 7, 100), 0), ((1000, 3, 64), 0), ((16, 300, 2), 0),
                                     ((64, 513, 7), 0), ((100, 70, 5), 0), ((257, 129, 3), 0), ((5, 17000, 6), 0),
                                     ((40, 64, 7), 3), ((200, 32, 5), 9)])
def test_narrow(gpu_runtime, mnk, pad, dtype):
    import torch

    m, n, k = mnk
    td = torch.float16 if dtype == "f16" else torch.float32
    rng = np.random.default_rng(m + n + k)
    a, b = (rng.uniform(-1, 1, s).astype(np.float16) for s in ((m, k), (k, n + pad)))
    ta, tb = (torch.full((x.size + 8,), float("nan"), dtype=td, device="cuda") for x in (a, b))
    for t, x in ((ta, a), (tb, b)):
        t[:x.size] = torch.from_numpy(x.reshape(-1)).to("cuda", td)
    tc = torch.full((m * (n + pad) + 64,), -7.0, device="cuda")
    K.matmul_mma_kernel(ta[:a.size], tb[:b.size], tc, m, n + pad, BM=32, BN=32, BK=8, K=k, NT=512,
                        _grid=(K.cdiv(n, 32), K.cdiv(m, 32)))
    torch.cuda.synchronize()
    c = tc.cpu().numpy()
    assert (c[m * (n + pad):] == -7.0).all()
    c = c[:m * (n + pad)].reshape(m, n + pad)
    n_hi = min(n + pad, K.cdiv(n, 32) * 32)
    assert (c[:, n_hi:] == -7.0).all()
    r = a.astype(np.float64) @ b.astype(np.float64)[:, :n_hi]
    assert np.abs(c[:, :n_hi] - r).max() <= 1e-5 * math.sqrt(k) * np.abs(r).max()


@pytest.mark.gpu
@pytest.mark.parametrize("mnk,dtype", [((64, 7, 4095), "f16"), ((300, 7, 1023), "f16"), ((1000, 3, 4095), "f16"), ((40, 3, 4096), "f32")])
def test_part_sums(gpu_runtime, mnk, dtype):
    """Eight part sums of K / 8 terms: 2-norm error about 0.3 u sqrt(K / 8) (u = 2^-24), a single chain of K terms about
    0.27 u sqrt(K), which is past the bound of 0.5 u sqrt(K / 8)."""
    import torch

    m, n, k = mnk
    td = torch.float16 if dtype == "f16" else torch.float32
    g = torch.Generator(device="cuda").manual_seed(7)
    a, b = (torch.empty(s, device="cuda").uniform_(-1, 1, generator=g).half().to(td) for s in (m * k, k * n))
    c = torch.full((m * n,), float("nan"), device="cuda")
    K.matmul_mma_kernel(a, b, c, m, n, BM=32, BN=32, BK=8, K=k, NT=512, _grid=(K.cdiv(n, 32), K.cdiv(m, 32)))
    torch.cuda.synchronize()
    want = a.view(m, k).double() @ b.view(k, n).double()
    err = ((c.view(m, n).double() - want).norm() / want.norm()).item()
    assert err <= 0.5 * 2.0 ** -24 * math.sqrt(k / 8)
