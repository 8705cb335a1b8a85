"""The multiplier from which on the bisection's rates are all at rate_min."""
import math

import pytest

from sktopt_amd.core.optimizers.oc import _saturating_multiplier


@pytest.mark.parametrize("largest,rate_min,eta", [(1.0, 0.7, 0.5), (3e-5, 0.2, 2.0), (0.0, 0.7, 0.5),
                                                  (2.0, 0.999, 1e-3), (1.0, 1e-9, 1e3)])
def test_rates_are_at_their_minimum_from_it_on(largest, rate_min, eta):
    lam = _saturating_multiplier(largest, rate_min, eta)
    for f in (1.0, 1.5, 1e6):
        assert (largest / (f * lam + 1e-12)) ** eta <= rate_min


@pytest.mark.parametrize("largest,rate_min,eta", [
    (1.0, 0.1, 1e-3), (0.0, 0.1, 1e-3), (1.0, 1e-300, 0.5),  # beyond float64
    (1.0, 0.0, 0.5), (1.0, -1.0, 0.5), (math.inf, 0.7, 0.5), (math.nan, 0.7, 0.5),
    (1.0, 0.7, 1e-4), (1.0, 0.7, 2e3)])
def test_none(largest, rate_min, eta):
    assert _saturating_multiplier(largest, rate_min, eta) == math.inf
