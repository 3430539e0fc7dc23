"""The order in which gemm_quad_kernel's waves fill, read and refill the operand ring in LDS
(flashqwen_amd/csrc/fqa_quad_schedule.h), run on the host by tests/cpp/quad_schedule.cpp with
operations that record it, for every tile and for fewer, as many and more k steps than the
ring has: no read before every wave's DMA has landed, no refill before every wave's reads
have ended."""
from __future__ import annotations

import subprocess
from pathlib import Path

import pytest

from flashqwen_amd import build as fb

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.skipif(not Path(fb.HIPCC).exists(), reason="hipcc not present")
def test_every_refill_follows_every_read(tmp_path):
    exe = tmp_path / "quad_schedule"
    # the schedule is a host and device template; only its host side is compiled here
    subprocess.run([fb.HIPCC, "-O1", "-std=c++17", "-Wall", "-x", "hip", "--offload-host-only",
                    str(ROOT / "tests" / "cpp" / "quad_schedule.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0]) > 100_000
