"""Which of the 64 x 64 and 128 x 64 tiles the GEMM plan takes where even 128 x 128 ones would fill at most half of the
CUs: 64 x 64 for one round of CUs, up to 1.75 rounds for K <= 256.  The Python and the C planner alike."""

from __future__ import annotations

import numpy as np
import pytest

import kernels as K
from easy_as_amd.runtime import hip_ext
from easy_as_amd.runtime.hip import pack_scalar, plan_launch


@pytest.mark.parametrize("m,n,k,entry,grid", [
    (1024, 1024, 258, "__t64x64", 256), (1024, 1026, 258, "__t128x64", 136), (1280, 1280, 256, "__t64x64", 400),
    (1280, 1280, 258, "__t128x64", 200), (1792, 1024, 256, "__t64x64", 448), (1856, 1024, 256, "__t128x64", 240),
    (193, 64, 4096, "__t64x64", 4)])
def test_small_tiles(m, n, k, entry, grid):
    hip = hip_ext.load_hip_ext(require=True)
    f16, f32 = np.zeros(1, np.float16), np.zeros(1, np.float32)
    ck = K.matmul_mma_kernel.compile(f16, f16, f32, m, n, BM=32, BN=32, BK=8, K=k, NT=512)
    groups = (K.cdiv(n, 32), K.cdiv(m, 32), 1)
    plan = plan_launch(ck, {"M": m, "N": n}, grid=groups, compute_units=256)
    assert plan.entry == "matmul_mma_kernel" + entry and plan.grid == (grid, 1, 1)
    sizes, base, argv = {"a": 2 * m * k, "b": 2 * k * n, "c": 4 * m * n}, 1 << 30, []
    for a in ck.ir.args:
        if a.kind == "buffer":
            argv.append(hip.wrap_pointer(base, sizes[a.name]))
            base += 1 << 30
        else:
            argv.append(pack_scalar(a.dtype, m if a.name == "M" else n))
    assert hip.plan_dispatch(ck.src, groups, (512, 1, 1), True, argv=argv, compute_units=256, entry_choice="auto") == \
        (plan.grid, plan.block, plan.hidden, plan.entry)
