"""Which launches of the one-thread-per-output matmul run on its own threads, in the Python and the C planner: a short K
on a small output, and rows of B of under 4 columns.  Either way gives the same bits (tests/test_gpu_chain_matmul.py)."""

from __future__ import annotations

import ctypes
import struct

import numpy as np
import pytest

import kernels as K
from easy_as_amd import build
from easy_as_amd.runtime import hip_ext
from easy_as_amd.runtime.hip import plan_launch

EAS_HIP_OK = 0


def _c_takes_gemm(src, m, n, k, block) -> bool:
    hip_ext.load_hip_ext(require=True)  # shares the process's HIP runtime
    lib = ctypes.CDLL(str(build.LIB))
    shape, gemm, plan = (ctypes.create_string_buffer(4096) for _ in range(3))
    assert lib.eas_hip_launch_shape_parse(src.encode(), shape) == EAS_HIP_OK
    assert lib.eas_hip_gemm_shape_parse(src.encode(), gemm) == EAS_HIP_OK
    args = struct.pack("<QQQII", 1 << 30, 2 << 30, 3 << 30, m, n)
    lengths = (ctypes.c_uint64 * 5)(4 * m * k, 4 * k * n, 4 * m * n, 0, 0)
    size, tptg = (ctypes.c_uint64 * 3)(m, -(-n // block), 1), (ctypes.c_uint32 * 3)(0, 0, 0)
    return lib.eas_hip_plan_gemm(shape, gemm, args, ctypes.c_size_t(len(args)), lengths, 5, 1, size, tptg, 256, None,
                                 plan) == EAS_HIP_OK


@pytest.mark.parametrize("k", [7, 8, 30, 48, 49, 64])
def test_threads_or_gemm(k):
    f = np.zeros(8, np.float32)
    ck = K.matmul_kernel.compile(f, f, f, 8, 8, BLOCK=64, K=k)
    for m, n in ((1, 1), (7, 128), (512, 576), (512, 577), (1000, 1000), (300, 960), (300, 961), (4608, 4), (4609, 4), (1 << 17, 4),
                 (1000, 1), (1 << 17, 3)):
        plan = plan_launch(ck, {"M": m, "N": n}, grid=(m, K.cdiv(n, 64), 1))
        threads = n < 4 or (8 <= k <= 48 and m * K.cdiv(n, 64) * 64 <= 288 << 10)
        assert (plan.entry is None) == threads, (m, n)
        assert _c_takes_gemm(ck.src, m, n, k, 64) != threads, (m, n)
        if threads:
            assert plan.grid == (m, K.cdiv(n, 64), 1) and plan.hidden == (m * 64,)


@pytest.mark.parametrize("choice,suffix", [("4wave", ""), ("tile128", "__t128")])
def test_a_named_entry_is_the_gemm(monkeypatch, choice, suffix):
    f = np.zeros(8, np.float32)
    ck = K.matmul_kernel.compile(f, f, f, 8, 8, BLOCK=64, K=32)
    monkeypatch.setenv("EAS_HIP_GEMM_ENTRY", choice)
    assert plan_launch(ck, {"M": 100, "N": 130}, grid=(100, 3, 1)).entry == "matmul_kernel__mm" + suffix
    assert _c_takes_gemm(ck.src, 100, 130, 32, 64)
