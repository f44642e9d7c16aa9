"""The compiled main entry of a 16-bit GEMM, which many bodies share."""

from __future__ import annotations

import re
import subprocess
from pathlib import Path

import numpy as np
import pytest

import kernels as K
from easy_as_amd.runtime import hip_ext
from easy_as_amd.runtime.hip import COMPILE_OPTIONS

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")


def _code(k, dtype=np.float16) -> bytes:
    a, c = np.zeros(1, dtype), np.zeros(1, np.float32)
    ck = K.matmul_mma_kernel.compile(a, a, c, 8, 8, BM=32, BN=32, BK=8, K=k, NT=512)
    return hip_ext.load_hip_ext(require=True).compile_to_code(ck.src, "k.hip", list(COMPILE_OPTIONS))


@pytest.mark.skipif(not OBJDUMP.exists(), reason="needs llvm-objdump")
def test_few_row_bodies_have_no_checks_that_always_pass(tmp_path):
    # 1174 compares with a thread index of unknown range, 794 with 0 <= tid < 256 known
    path = tmp_path / "k.co"
    path.write_bytes(_code(4096))
    asm = subprocess.run([str(OBJDUMP), "-d", "--mcpu=gfx950", str(path)], check=True, capture_output=True, text=True).stdout
    main = re.search(r"<matmul_mma_kernel>:\n(.*?)\n\n", asm, re.S).group(1)
    assert len(re.findall(r"\tv_cmpx?_", main)) < 1000


@pytest.mark.parametrize("k,dtype,limit", [(1023, np.float16, 105_000), (2048, np.float32, 120_000), (1022, np.float16, 190_000)])
def test_no_bodies_that_no_launch_reaches(k, dtype, limit):
    # with the few-row DMA body for K off a multiple of 8 and the register body for 65-128 rows:
    # 110, 127 and 193 KB; without 96, 109 and 179
    assert len(_code(k, dtype)) < limit
