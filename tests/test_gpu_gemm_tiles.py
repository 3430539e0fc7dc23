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
@pytest.mark.parametrize("M,N,K", [
    (61, 2048, 8192),       # slabs with K split
    (700, 4096, 12288),     # 256 x 256 tiles, K split
    (160, 2048, 12288),
    (100, 6144, 4096),
    (480, 6144, 4096),
])
def test_gemm_larger_workspace(gpu, M, N, K):
    """A workspace larger than fqa_gemm_workspace_bytes asks for changes no bit."""
    import torch

    from flashqwen_amd.gemm import gemm, workspace_bytes

    n = workspace_bytes(M, N, K)
    assert n > 0
    g = torch.Generator(device=gpu)
    g.manual_seed(M)
    x = torch.empty(M, K, dtype=torch.bfloat16, device=gpu).normal_(generator=g)
    w = torch.empty(N, K, dtype=torch.bfloat16, device=gpu).normal_(0.0, 0.02, generator=g)
    ws = torch.empty(max(16 * M * N * 4, 2 * n), dtype=torch.uint8, device=gpu)
    want = gemm(x, w, out_f32=True, workspace=ws[:n])
    for size in (n + 16, ws.numel()):
        assert torch.equal(gemm(x, w, out_f32=True, workspace=ws[:size]), want)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (300, 16640, 64),       # 192 x 256 tiles, ragged
    (300, 16512, 64),       # 256 x 192
    (385, 22016, 64),       # 256 x 256
    (130, 16512, 64),       # 256 x 128, one row tile
    (1025, 256, 64),        # past 1024 rows the workspace holds a pair per 256 columns, where
    (1025, 3840, 64),       # the plan's own tiles are 128 columns wide: 256 x 256 instead
    (1100, 2048, 256),      # ... and fqa_gemm splits K
])
def test_argmax_tiles(gpu, M, N, K):
    """fqa_gemm_argmax on each tile, within an exactly sized workspace, against the fp32
    logits of fqa_gemm (the same values where it needs no workspace, else float64 products
    within fp32 rounding)."""
    import torch

    from flashqwen_amd import _lib
    from flashqwen_amd.gemm import gemm, gemm_argmax, workspace_bytes

    print(f"[argmax_tiles] M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device=gpu)
    g.manual_seed(M + N)
    x = torch.empty(M, K, dtype=torch.bfloat16, device=gpu).normal_(generator=g)
    w = torch.empty(N, K, dtype=torch.bfloat16, device=gpu).normal_(0.0, 0.5, generator=g)
    x[-1] = w[-1] * 8  # the last row peaks in the last column
    n = int(_lib.load().fqa_gemm_argmax_workspace_bytes(M, N, K))
    ws = torch.full((n + 4096,), 0x5A, dtype=torch.uint8, device=gpu)
    got = gemm_argmax(x, w, workspace=ws[:n]).long()
    assert torch.all(ws[n:] == 0x5A)
    if workspace_bytes(M, N, K) == 0:
        logits, tol = gemm(x, w, out_f32=True), 0.0
    else:
        logits, tol = x.double() @ w.double().T, 1e-4
    assert torch.all(logits.gather(1, got[:, None])[:, 0] >= logits.max(1).values - tol)
    assert int(got[-1]) == N - 1


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,write_k,rows", [
    (40, 64, 1, None),      # one k step: the 128-row tile's append epilogue
    (100, 64, 1, None),
    (129, 1024, 0, None),   # a slab's fp32 sums through the append kernel
    (300, 1024, 0, None),   # 128 x 128 tiles
    (345, 1024, 0, None),
    (448, 1024, 1, 440),    # ... with the row count inside the last one
    (450, 1024, 1, 440),
    (488, 4096, 0, None),
    (489, 4096, 1, 480),    # two planes of 256 x 128 tiles through the append kernel
    (512, 4032, 0, None),   # ... which take 4096 k or more
    (700, 512, 1, 690),     # 256 x 128 tiles
    (1500, 256, 0, 1490),   # 192 x 256 tiles
])
def test_qkv_fused_tiles(gpu, M, K, write_k, rows):
    from tests.test_gpu_qkv_fused import _case

    _case(gpu, M, K, write_k, seed=M + 3 * K, rows=rows)
