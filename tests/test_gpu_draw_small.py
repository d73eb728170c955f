"""Nucleus draws whose kept values end inside the first chunk (the total's turns stop at its last value) and whose nuclei lie
on both sides of what one wave sorts, against the oracle's draw: the token, for random numbers over the whole range."""
import numpy as np
import pytest

import gpu_lib as gl
import oracle_lib as ol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 33, 65, 1091, 2047, 2049, 5000])
@pytest.mark.parametrize("spread", [0.02, 0.6, 3.0])
def test_small_nucleus_draws(n, spread):
    rng = np.random.default_rng(n)
    logits = (rng.standard_normal(n) * spread).astype(np.float32)
    logits[n // 2] = logits.max()  # an equal pair: the smaller index first
    for topp in (0.05, 0.5, 0.95):
        for random in (0.0, 0.3, 0.77, 0.999999):
            assert gl.sample(logits, 0.8, topp, random) == ol.sample(logits, 0.8, topp, random), (topp, random)


@pytest.mark.parametrize("n", [4, 8, 64, 2052])
def test_nothing_kept(n):
    """equal logits at a temperature whose reciprocal is past float32: 0 * infinity, no probability to sort. Declined: the
    caller takes the step (the reference's own loop reads before its list here, so there is no token to compare)"""
    assert gl.sample(np.full(n, 3.0, np.float32), 1e-40, 0.5, 0.3) == -2


@pytest.mark.parametrize("n", [1600, 2048, 2100, 8000])
@pytest.mark.parametrize("at,peak", [(0, 14.0), (5, 9.0), (31, 20.0), (33, 14.0), (1500, 14.0)])
def test_likely_token_near_the_front(n, at, peak):
    """a first chunk whose sum is put in its binade by a value of the first lane (then the rest in one pass, to its end or to a
    crossing far behind), or by one after it"""
    rng = np.random.default_rng(n)
    logits = (rng.standard_normal(n) * 2).astype(np.float32)
    logits[at] = peak
    for spread in (1.0, 0.05):
        values = logits * np.float32(spread)
        values[at] = logits[at]
        for topp in (0.5, 0.95, 0.9999):
            for random in (0.0, 0.5, 0.99, 0.999999):
                assert gl.sample(values, 0.8, topp, random) == ol.sample(values, 0.8, topp, random), (spread, topp, random)


@pytest.mark.parametrize("n", [1600, 2047, 2048])
@pytest.mark.parametrize("first,last", [(1.0, 0.0), (1.0, 1e-3), (1.0, 0.9e-3), (0.4, 3e-4), (1e-6, 1e-9)])
def test_total_behind_a_large_first_value(n, first, last):
    """the total itself, to the bit, for values that cross the first value's binade never, at the very end, or on the way"""
    rng = np.random.default_rng(n)
    p = (rng.random(n) * last).astype(np.float32)
    p[3] = first
    total, checkpoints = gl.ordered_sum(p, True)
    sums = np.concatenate([[0.0], np.cumsum(p.astype(np.float64))])
    assert total == sums[-1]
    assert np.array_equal(checkpoints, sums[:-1:256])
