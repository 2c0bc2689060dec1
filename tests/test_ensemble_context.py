"""The generator of an ensemble context is made on first use, with the same
stream as one made from the seed at once, and can be replaced."""
import numpy as np
import pytest

from odemi.api import EnsembleContext, _Seed


@pytest.mark.parametrize("seed", [[0, 1], [7, 3], [7, 3, 2]])
def test_context_rng_is_the_seeds(seed):
    ctx = EnsembleContext(seed[1], 1, _Seed(seed))
    a, b = ctx.rng.random(5), ctx.rng.random(5)
    assert np.array_equal(np.concatenate([a, b]), np.random.default_rng(seed).random(10))
    ctx.rng = None
    assert ctx.rng is None and ctx.i == seed[1]
    assert EnsembleContext(1, 2, None).rng is None
