"""The exact DP on histograms that strain its bound on the starts it looks at (equal
counts and their many equal costs, spikes beside single counts, fractional and
extreme counts, gaps), bit for bit against the oracle, which tries every start."""

import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _histogram(kind, bins, rng):
    x = (np.arange(bins) + 0.5) / bins * 2 - 1
    if kind == "uniform":
        return np.full(bins, 1000.0)
    if kind == "one_count":
        return np.ones(bins)
    if kind == "spikes":  # nearly all the mass in a few bins
        c = np.ones(bins)
        c[rng.integers(0, bins, 5)] = 2.0 ** 40
        return c
    if kind == "centre":  # a narrow peak: costs far below the total weight
        return np.round(1e9 * np.exp(-(x / 0.004) ** 2)) + (rng.random(bins) < 0.5)
    if kind == "fractions":
        return rng.random(bins) * 10.0 ** rng.integers(-6, 7, bins)
    if kind == "huge":
        return rng.random(bins) * 1e30
    if kind == "tiny":
        return rng.random(bins) * 1e-30
    if kind == "gaps":
        c = np.zeros(bins)
        at = rng.choice(bins, bins // 3, replace=False)
        c[at] = rng.integers(1, 50, at.size)
        return c
    c = np.round(1e7 * np.exp(-0.5 * (x / 0.25) ** 2))  # gradients over their block maxima
    c[0] += 40000
    c[-1] += 40000
    return c


@pytest.mark.parametrize("kind", ["uniform", "one_count", "spikes", "centre", "fractions", "huge", "tiny", "gaps",
                                  "normal"])
@pytest.mark.parametrize("bins,k,force", [(1024, 256, True), (1024, 37, False), (512, 16, True), (256, 17, True),
                                          (64, 2, True), (64, 1, False), (64, 1, True)])
def test_codebook_equals_the_oracle(kind, bins, k, force):
    from gefen_amd.quantization import exact_dp_from_counts

    counts = _histogram(kind, bins, np.random.default_rng(bins + k)).astype(np.float32)
    got = exact_dp_from_counts(torch.from_numpy(counts).to("cuda:0"), k, force).cpu().numpy()
    ref = orc.exact_dp(counts, k, force)
    np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("decades", [9, 14, 15, 17, 25])
@pytest.mark.parametrize("bins,k", [(1024, 4), (1024, 16), (512, 64), (512, 200)])
def test_counts_over_many_decades(bins, k, decades):
    """Log-uniform counts.  Over 9 decades starts are left out; from 14 on none are, and from
    about 15 on none may be: the rounding of the prefix sums exceeds the smallest counts, so
    that a segment's computed cost no longer grows with the segment."""
    from gefen_amd.quantization import exact_dp_from_counts

    for seed in range(4):
        rng = np.random.default_rng(seed * 1000 + k + bins)
        counts = (10.0 ** (rng.random(bins) * decades - decades / 2)).astype(np.float32)
        got = exact_dp_from_counts(torch.from_numpy(counts).to("cuda:0"), k, True).cpu().numpy()
        ref = orc.exact_dp(counts, k, True)
        # codewords of segments whose weights cancel are infinite or NaN, in an order of their own
        np.testing.assert_array_equal(np.sort(got), np.sort(ref), err_msg="seed {}".format(seed))
