"""fqa_sample's rules for what it counts and copies in LDS (flashqwen_amd/csrc/
fqa_sample_select.h), run on the host by tests/cpp/sample_select.cpp.  copy_fits, behind a
restatement of the sums and the histogram before it: where the boundary bin may be copied,
every weight of the bin fits the copy's 16384 places.  in_columns: a weight counted in a
level-1 column has one, NaNs too."""
from __future__ import annotations

import subprocess
from pathlib import Path

import numpy as np
import pytest

from flashqwen_amd import build as fb

ROOT = Path(__file__).resolve().parents[1]
VOCAB, CAP = 151936, 16384


def cut_bin_row():
    """A row whose fp32 total comes out 1.7e-6 too large (every lane of the kernel adds 112
    weights that round up each time), with a tail in the 1/8-octave bin that x_min cuts for
    top_p at 1 - 1.6e-6: a quarter of the tail at or above x_min, the rest below."""
    i = np.arange(VOCAB)
    nth = (i % 9728) // 256 * 4 + i % 4  # the element's place in its lane's part of the row
    body, tail = 0.5112514323816543, nth > 112
    lg = np.full(VOCAB, np.log(body), np.float32)
    lg[nth == 0] = 0.0
    total = 1024 + body * np.count_nonzero(~tail)
    x_min = 1.6172804649938755e-06 / 2 * total / VOCAB
    lo = 2.0 ** np.floor(np.log2(x_min))
    lo *= 1 + np.floor((x_min / lo - 1) * 8) / 8
    hi = lo + 2.0 ** np.floor(np.log2(lo)) / 8
    part = np.random.default_rng(0).random(np.count_nonzero(tail)) < 0.25
    lg[tail] = np.log(np.where(part, (x_min + hi) / 2, (x_min + lo) / 2)).astype(np.float32)
    return lg


def close_to_one():
    """The 100 largest values of top_p below 1."""
    return (1 - np.arange(1, 101) * 2.0 ** -24).astype(np.float32)


@pytest.fixture(scope="module")
def select(tmp_path_factory):
    if not Path(fb.HIPCC).exists():
        pytest.skip("hipcc not present")
    exe = tmp_path_factory.mktemp("select") / "sample_select"
    # no contraction: the kernel rounds each product and sum (fmaf is written where it is
    # meant); no NaN semantics, as the library is built
    subprocess.run([fb.HIPCC, "-O1", "-std=c++17", "-Wall", "-ffp-contract=off",
                    "-fno-honor-nans", "-x", "hip",
                    "--offload-host-only", str(ROOT / "tests" / "cpp" / "sample_select.cpp"),
                    "-o", str(exe)], check=True, capture_output=True, text=True)

    def run(lg, top_p=()):
        if lg is None:
            return subprocess.run([str(exe), "columns"], capture_output=True, text=True)
        r = subprocess.run([str(exe), str(len(lg)), *(repr(float(t)) for t in top_p)],
                           input=lg.astype(np.float32).tobytes(), capture_output=True, check=True)
        return [tuple(map(int, line.split())) for line in r.stdout.decode().splitlines()]

    return run


def test_bin_cut_by_the_smallest_counted_weight(select):
    got = select(cut_bin_row(), close_to_one())
    assert all(in_bin <= CAP for _, _, _, in_bin, fits in got if fits), got
    # the row does meet the case: few enough weights counted, too many in the bin
    assert any(b == cut and counted <= CAP < in_bin for b, cut, counted, in_bin, _ in got)


@pytest.mark.parametrize("vocab", [1023, 16385, 151936])
def test_copied_bins_fit(select, vocab):
    rng = np.random.default_rng(vocab)
    copied = 0
    for scale in (0.01, 0.1, 2.0, 6.0):
        lg = rng.standard_normal(vocab).astype(np.float32) * np.float32(scale)
        for b, cut, counted, in_bin, fits in select(lg, [0.0, 0.3, 0.9, 0.99, 0.9999, 0.999999]):
            assert not fits or in_bin <= CAP
            # away from the cut the count is a bound, and the bin is copied where it fits
            assert b > cut and (in_bin <= counted)
            assert fits == (counted <= CAP)
            copied += fits
    assert copied > 0


def test_counted_weights_have_a_column(select):
    r = select(None)
    assert r.returncode == 0, r.stdout
