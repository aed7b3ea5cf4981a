"""Draws spread over the device against the oracle: logits whose sums, cuts
and thresholds sit where the ordered-sum scan, the bucket sort and the
candidate gathering change paths (ties and half-way adds, equal values,
sums in many binades, infinities, zero thresholds, crowded buckets)."""
import numpy as np
import pytest

from test_gpu_sampling import _check_draws, _put, samp_eng  # noqa: F401

pytestmark = pytest.mark.gpu

V = 40000


def _logits(kind, rng, V):
    if kind == "normal":
        return rng.standard_normal(V) * 2.0
    if kind == "equal":                                  # every add ties or doubles; one bucket, all ties at the cut
        return np.zeros(V)
    if kind == "steps":                                  # powers of two: half-way adds in every binade
        return np.log(2.0) * rng.integers(-24, 1, V)
    if kind == "late":                                   # tiny terms first, the large ones last
        return np.linspace(-60.0, 0.0, V)
    if kind == "inf":
        x = rng.standard_normal(V)
        x[rng.integers(0, V, V // 2)] = -np.inf
        return x
    if kind == "zeros":                                  # the K-th largest is a zero of either sign
        x = np.where(rng.random(V) < 0.5, 0.0, -0.0)
        x[:7] = 1.0
        x[100:200] = -1.0
        return x
    raise ValueError(kind)


@pytest.mark.parametrize("kind", ["normal", "equal", "steps", "late", "inf", "zeros"])
@pytest.mark.parametrize("case", [(1.0, 0.9, 0, 1.1), (0.7, 1.0, 0, 1.0), (1.0, 0.95, 50, 1.1), (2.0, 0.5, 600, 1.0)])
def test_device_draws_match_oracle(samp_eng, oracle, case, kind):  # noqa: F811
    rng = np.random.default_rng(len(kind))
    _check_draws(samp_eng, oracle, case, V, 2, lambda s: _logits(kind, rng, V).astype(np.float32))
    samp_eng.set_sampling(0.0, 1.0, 0, 1.0, 1)


def test_crowded_bucket(samp_eng, oracle):  # noqa: F811
    """More different values in one bucket than a workgroup sorts. All
    probabilities are within 1e-3 of 1 / V, so the device expf's last ulp moves
    the cut: two running sums of terms an ulp apart differ by at most V 2^-23
    relative (an ulp of the sum per add), that is V^2 2^-23 entries; the kept
    values themselves agree to 2^-23 V for the two sums they are divided by."""
    import torch
    x = np.random.default_rng(2).uniform(0.0, 1e-3, V).astype(np.float32)
    samp_eng.set_sampling(1.0, 0.9, 0, 1.0, 5)
    st, ref = oracle.sampler(1.0, 0.9, 0, 1.0, 5), x.copy()
    oracle.sample_logits(st, ref)
    dev = samp_eng.empty(V, torch.float32)
    _put(samp_eng, dev, x)
    samp_eng.sample_logits(dev, V)
    got = samp_eng.to_host(dev)
    samp_eng.set_sampling(0.0, 1.0, 0, 1.0, 1)
    assert np.count_nonzero((got == 0) != (ref == 0)) <= V * V * 2.0 ** -23
    both = (got != 0) & (ref != 0)
    assert np.max(np.abs(got[both] / ref[both] - 1)) <= 2 * V * 2.0 ** -23
    # descending order: nothing kept lies below anything dropped, but where
    # expf (an ulp off, 2^-23 near 1) and the division (2^-24) give one value
    assert x[got != 0].min() >= x[got == 0].max() - 2.0 ** -22


@pytest.mark.parametrize("case", [(1.0, 1.0, 0, 1.0), (1.0, 0.9, 0, 1.0)], ids=["draw", "top-p"])
@pytest.mark.parametrize("size", [16384, 33281, 524801, 2200003])
def test_ordered_sum_runs(samp_eng, oracle, case, size):  # noqa: F811
    """Runs of the ordered sum at their edges: whole, one entry over, more than
    1024 of them, two passes per run. Equal logits: exp(0) = 1, so the device's
    expf is exact."""
    _check_draws(samp_eng, oracle, case, size, 2, lambda s: np.zeros(size, np.float32))
    samp_eng.set_sampling(0.0, 1.0, 0, 1.0, 1)


@pytest.mark.parametrize("kind", ["normal", "equal", "late", "inf"])
@pytest.mark.parametrize("case", [(1.0, 1.0, 0, 1.0), (1.0, 0.9, 0, 1.0), (1.0, 1.0, 4500, 1.0)],
                         ids=["draw", "top-p", "top-k"])
@pytest.mark.parametrize("size", [4097, 5003, 12001])
def test_one_workgroup_ordered_sums(samp_eng, oracle, size, case, kind):  # noqa: F811
    """Ordered sums of one workgroup: picks and cuts in the part that one thread
    adds, at its end and in the scan after it. (Not "steps": where every add is
    half way, an ulp of the device's expf in each of n terms moves the sum by up
    to n 2^-24 relative, past the 4e-6 that the arrays are held to.)"""
    rng = np.random.default_rng(size)
    _check_draws(samp_eng, oracle, case, size, 12, lambda s: _logits(kind, rng, size).astype(np.float32))
    samp_eng.set_sampling(0.0, 1.0, 0, 1.0, 1)
