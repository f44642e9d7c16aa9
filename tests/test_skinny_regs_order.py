"""The few-row register body hands operands from lane to lane through a wave's own LDS slot, without a barrier: in the
compiled code every read of a stage has to come after all of its writes, and every write after the reads of the stage
before (the compiler sees one lane, to which a write at another address looks free to move)."""

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


def _wave_loops(asm: str) -> list[list[str]]:
    """Bodies of the branch-free loops that hold MFMAs and LDS writes and no barrier."""
    ins = [(int(m.group(2), 16), m.group(1).strip()) for m in re.finditer(r"^\t(\S.*?)// ([0-9A-F]{12}):", asm, re.M)]
    at = {a: i for i, (a, _) in enumerate(ins)}
    loops = []
    for i, (a, text) in enumerate(ins):
        m = re.match(r"s_cbranch\S*\s+(\d+)", text)
        if m and int(m.group(1)) > 32767:
            body = [t for _, t in ins[at[a + 4 + 4 * (int(m.group(1)) - 65536)]:i]]
            text = " ".join(body)
            if "v_mfma" in text and "ds_write" in text and "s_barrier" not in text and "branch" not in text:
                loops.append(body)
    return loops


@pytest.mark.skipif(not OBJDUMP.exists(), reason="needs llvm-objdump")
@pytest.mark.parametrize("dtype,k", [(np.float16, 1023), (np.float32, 2048)])
def test_reads_of_a_stage_follow_its_writes(tmp_path, dtype, k):
    hip = hip_ext.load_hip_ext(require=True)
    a, c = np.zeros(1, dtype), np.zeros(1, np.float32)
    ck = K.matmul_mma_kernel.compile(a, a, c, 8, 8, BM=32, BN=32, BK=8, K=k, NT=512)
    path = tmp_path / "k.co"
    path.write_bytes(hip.compile_to_code(ck.src, "k.hip", list(COMPILE_OPTIONS)))
    asm = subprocess.run([str(OBJDUMP), "-d", "--mcpu=gfx950", str(path)], check=True, capture_output=True, text=True).stdout
    loops = _wave_loops(asm)
    assert len(loops) >= 3  # 1, 2 and 4 row tiles
    for body in loops:
        order = "".join("W" if t.startswith("ds_write") else "r" if t.startswith("ds_read") else "" for t in body)
        order = order[order.index("rW") + 1:] + order[:order.index("rW") + 1] if "rW" in order else order
        runs = {len(w) for w in re.findall("W+", order)}
        # one or two stages a loop, each all of its writes and then all of its reads
        assert len(runs) == 1 and len(re.findall("W+r+", order)) <= 2, order
