"""fqa_gemm where its tile kernels can go wrong: numbers of k steps around a pipeline's
depth, ragged last row tiles, row strides that allow no 16-byte stores, each output form.
The bounds are test_gpu_gemm's: one bf16 rounding (2^-8 relative) or 1e-5 relative for fp32,
plus 1e-6 sqrt(K) for fp32 accumulation."""
from __future__ import annotations

import pytest

from tests.test_gpu_gemm import _run_case


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,kw", [
    (1025, 512, 64, {}),                    # one k step, one row in the last tile
    (1280, 1024, 128, {}),                  # two steps
    (1500, 512, 192, {"ldy_pad": 4}),       # three; rows of y on 8 bytes only
    (2047, 256, 320, {"ldy_pad": 8}),       # five; the last row clamped
    (1300, 512, 256, {"out_f32": True}),    # fp32 out
    (1100, 256, 1024, {}),                  # split K (partials)
    (1100, 256, 1024, {"out_f32": True}),
    (5000, 2304, 128, {"ldx_pad": 8}),      # several tiles per workgroup slot
])
def test_gemm_256_tile(gpu, M, N, K, kw):
    _run_case(gpu, M, N, K, seed=M + K, **kw)
