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
