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
    (2300, 2304, 128, {"ldx_pad": 8}),      # several tiles per workgroup slot
    (384, 24576, 64, {}),                   # 192 x 256 tiles, full rows
    (300, 24576, 128, {"ldy_pad": 4}),      # ... ragged
    (500, 24576, 192, {}),                  # 256 x 192 tiles
    (400, 24576, 64, {"out_f32": True}),
    (1500, 4096, 12288, {}),                # 192 x 256 with K split
])
def test_gemm_256_tile(gpu, M, N, K, kw):
    _run_case(gpu, M, N, K, seed=M + K, **kw)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,kw", [
    # unsplit, rows below, at and past a slab's and a 16-row block's edge; as many k steps as
    # waves, fewer (idle waves) and ring depths crossed
    (1, 128, 128, {}),
    (7, 1024, 192, {"ldy_pad": 4}),
    (9, 512, 1984, {"ldx_pad": 8}),
    (1, 6144, 128, {}),                     # 24 columns: half a block
    (35, 1536, 320, {}),
    (17, 4096, 448, {"out_f32": True}),
    (34, 3072, 192, {"ldy_pad": 12}),
    (65, 2048, 704, {}),
    (66, 3072, 64 * 9, {"out_f32": True}),
    (129, 3072, 128, {}),
    (130, 4096, 192, {}),
    (130, 6144, 256, {}),
    (193, 6144, 128, {"ldx_pad": 16}),
    (257, 4096, 128, {}),
    (387, 2048, 320, {}),
    (61, 2048, 8192, {}),                   # slabs with K split: partials and reduction
    (61, 2048, 8192, {"out_f32": True}),
    # 128- and 256-row tiles of one row tile (rotated k steps), split and not
    (250, 24576, 64, {}),
    (130, 20480, 192, {"out_f32": True}),
    (100, 20480, 320, {}),
    (160, 2048, 12288, {}),
    # 32- and 64-row tiles: k steps below and past the ring
    (20, 20480, 64, {}),
    (33, 20480, 64 * 7, {}),
    (64, 20480, 64 * 6, {"out_f32": True}),
])
def test_gemm_few_rows(gpu, M, N, K, kw):
    _run_case(gpu, M, N, K, seed=M + N + K, **kw)


@pytest.mark.gpu
def test_gemm_smaller_workspace(gpu):
    """A workspace of the least size that the shape ever needed is still enough (fewer K
    splits are used); one byte less is refused."""
    import torch

    from flashqwen_amd._lib import FqaError
    from flashqwen_amd.gemm import gemm, workspace_bytes

    M, N, K = 700, 4096, 12288
    least = 2 * M * N * 4
    assert workspace_bytes(M, N, K) >= least
    g = torch.Generator(device=gpu)
    g.manual_seed(5)
    x = torch.empty(M, K, dtype=torch.bfloat16, device=gpu).normal_(generator=g)
    w = torch.empty(N, K, dtype=torch.bfloat16, device=gpu).normal_(0.0, 0.02, generator=g)
    ws = torch.empty(workspace_bytes(M, N, K), dtype=torch.uint8, device=gpu)
    ref = x.float() @ w.float().T
    for n in (ws.numel(), least):
        y = gemm(x, w, workspace=ws[:n]).float()
        # one bf16 rounding, and fp32 sums of 12288 products in two orders
        assert torch.all((y - ref).abs() <= 2.0 ** -8 * ref.abs() + 2e-6 * K ** 0.5)
    with pytest.raises(FqaError):
        gemm(x, w, workspace=ws[:least - 16])


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,write_k,rows", [
    (40, 64, 1, None),      # one k step: the 128-row tile's append epilogue
    (100, 64, 1, None),
    (129, 1024, 0, None),   # a slab's fp32 sums through the append kernel
    (300, 1024, 0, None),   # 128 x 128 tiles
    (345, 1024, 0, None),
    (448, 1024, 1, 440),    # ... with the row count inside the last one
    (450, 1024, 1, 440),    # two planes of 256 x 128 tiles through the append kernel
    (700, 512, 1, 690),     # 256 x 128 tiles
    (1500, 256, 0, 1490),   # 192 x 256 tiles
])
def test_qkv_fused_tiles(gpu, M, K, write_k, rows):
    from tests.test_gpu_qkv_fused import _case

    _case(gpu, M, K, write_k, seed=M + 3 * K, rows=rows)
