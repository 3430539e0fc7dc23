"""fqa_sample's top-p rows where the select can go wrong, against the fp64 oracle as
tests/test_gpu_sample.py checks it: a boundary among a few large weights, in a broad body,
likely tokens all at one end of the vocabulary, flat rows (the boundary bin does not fit the
LDS copy), one dominant token; vocabularies below, at and above the copy's capacity and
around a chunk of the row; rows that start on 4 bytes only."""
from __future__ import annotations

import numpy as np
import pytest

from tests.test_gpu_sample import _check_sampled, _run


def _rows(rng, B, vocab):
    lg = rng.standard_normal((B, vocab)) * 2.0
    kind = np.arange(B) % 6
    for b in range(B):
        if kind[b] == 1 and vocab > 64:    # a few large weights
            lg[b, rng.integers(0, vocab, 20)] += 12.0
        elif kind[b] == 2:                 # likely tokens first
            lg[b, : vocab // 20 + 1] += 6.0
        elif kind[b] == 3:                 # ... and last, on few values
            lg[b, -(vocab // 50 + 1):] = 9.0
        elif kind[b] == 4:
            lg[b] *= 0.01
        elif kind[b] == 5:                 # one dominant token
            lg[b, rng.integers(vocab)] = 40.0
    return lg.astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("vocab", [1023, 1025, 16384, 16385, 17408 + 1, 50257, 151936])
def test_top_p_rows(gpu, vocab):
    rng = np.random.default_rng(vocab)
    B = 24
    lg = _rows(rng, B, vocab)
    it = rng.choice([0.7, 1.0, 1.6], size=B).astype(np.float32)
    tp = rng.choice([0.999, 0.95, 0.9, 0.5, 0.05], size=B).astype(np.float32)
    u = rng.random(B).astype(np.float32)
    got = _run(lg, it, tp, u)
    exact = _check_sampled(lg, it, tp, u, got)
    # the same allowance for fp32 draws at a cumulative boundary as the other sampled rows
    assert exact >= B - 2
    assert np.array_equal(_run(lg, it, tp, u), got)


@pytest.mark.gpu
@pytest.mark.parametrize("vocab", [4097, 151936])
def test_top_p_near_one(gpu, vocab):
    """The boundary far down the row's tail, and past what fp32 sums resolve."""
    rng = np.random.default_rng(vocab + 2)
    B = 24
    lg = _rows(rng, B, vocab)
    tp = rng.choice([0.9995, 0.9999, 0.99999, 0.999999], size=B).astype(np.float32)
    it, u = np.ones(B, np.float32), rng.random(B).astype(np.float32)
    exact = _check_sampled(lg, it, tp, u, _run(lg, it, tp, u))
    assert exact >= B - 2


@pytest.mark.gpu
def test_rows_on_four_bytes(gpu):
    """A row stride that is odd in elements: the 16-byte loads start on any 4 bytes."""
    import torch

    from flashqwen_amd.sample import sample

    rng = np.random.default_rng(5)
    B, vocab = 12, 20001
    lg = _rows(rng, B, vocab)
    it = np.where(np.arange(B) % 3 == 0, 0.0, 1.1).astype(np.float32)
    tp = np.where(np.arange(B) % 2 == 0, 0.9, 1.0).astype(np.float32)
    u = rng.random(B).astype(np.float32)
    want = _run(lg, it, tp, u)
    wide = torch.full((B, vocab + 4), 99.0, device=gpu)
    for off in (1, 2, 3):
        x = wide[:, off:off + vocab]
        x.copy_(torch.from_numpy(lg))
        got = sample(x, *(torch.from_numpy(v).to(gpu) for v in (it, tp, u)))
        assert np.array_equal(got.cpu().numpy(), want)
        wide.fill_(99.0)


@pytest.mark.gpu
def test_bin_cut_by_the_smallest_counted_weight(gpu):
    """top_p so close to 1 that the boundary bin is the one the smallest counted weight cuts:
    more of its weights lie in the bin than its histogram counts (tests/test_sample_select.py),
    and the row is read again instead of copied."""
    from tests.test_sample_select import close_to_one, cut_bin_row

    tp = close_to_one()
    lg = np.tile(cut_bin_row(), (len(tp), 1))
    rng = np.random.default_rng(9)
    it, u = np.ones(len(tp), np.float32), rng.random(len(tp)).astype(np.float32)
    got = _run(lg, it, tp, u)
    # equal weights side by side: a draw within fp32 rounding of the total (1e-5 of 150000
    # tokens) falls on a neighbour, which _check_sampled allows
    _check_sampled(lg, it, tp, u, got)
    assert np.array_equal(_run(lg, it, tp, u), got)


@pytest.mark.gpu
@pytest.mark.parametrize("vocab", [1025, 151936])
def test_rows_with_nan_and_inf(gpu, vocab):
    """Rows with NaN or infinite logits give some token of the vocabulary and leave the rows
    beside them alone."""
    rng = np.random.default_rng(vocab + 1)
    B = 16
    lg = _rows(rng, B, vocab)
    it = np.where(np.arange(B) % 5 == 4, 0.0, 1.0).astype(np.float32)
    tp = rng.choice([1.0, 0.95, 0.5], size=B).astype(np.float32)
    tp[:8:2] = 0.9
    u = rng.random(B).astype(np.float32)
    want = _run(lg, it, tp, u)
    bad = lg.copy()
    bad[0, vocab // 2] = np.nan
    bad[2, [3, vocab // 3]] = np.inf
    bad[4, :] = np.nan
    bad[6, :] = np.inf
    bad[8, ::3] = np.nan
    bad[9, 7] = np.nan
    got = _run(bad, it, tp, u)
    assert np.all((got >= 0) & (got < vocab))
    ordinary = [b for b in range(B) if b not in (0, 2, 4, 6, 8, 9)]
    assert np.array_equal(got[ordinary], want[ordinary])
