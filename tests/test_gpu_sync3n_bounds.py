"""pairs_probabilities at the bounds of its product form: a small c_a = (1 - P2) A
under a high power of 1 - score, and the direct form with a negative A.

Rotations exact to 1e-15 give scores within a few 2^-53 of 1.
With P2 = 0 the two models are one function, log A + a log(1 - score), so the
two sums agree: 1e-12 relative, and finite wherever 1 - score is not 0 (the
powers alone are down to 1e-356, below the smallest double).  With A < 0 the
logarithm is NaN, as the oracle has it."""
import numpy as np
import pytest

from aspire_amd import sim
from aspire_amd.sync3n import pairs_probabilities_mex
from tests.test_sync3n_oracle import noisy, rel_rotations

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A,a,b", [(1e-90, 18.0, 2.0), (1e-40, 17.5, 1.5), (1e-30, 18.0, 2.0), (1.0, 18.0, 2.0),
                                   (1e-90, 2.0, 18.0), (1e-100, 3.0, 3.0)])
def test_one_model(A, a, b):
    print("case sync3n-bounds", A, a, b, flush=True)
    rng = np.random.default_rng(11)
    R, _ = rel_rotations(sim.rand_rots(rng, 24))
    R = R + 1e-15 * rng.standard_normal(R.shape)
    ind, arb, _ = pairs_probabilities_mex(R, 0.0, A, a, 1.0, b, 0.78)
    assert np.array_equal(np.isfinite(ind), np.isfinite(arb))
    f = np.isfinite(arb)
    assert f.any()
    assert np.allclose(ind[f], arb[f], rtol=1e-12, atol=0)


@pytest.mark.parametrize("prm", [(0.0, -1.0, 2.2, 1.0, 2.5, 0.78), (0.5, -1.0, 2.2, 1.0, 2.5, 0.78),
                                 (0.0, 1.0, 4.5, 1.0, 1.5, 0.78)])
def test_direct_form_and_no_indicative_model(oracle, prm):
    print("case sync3n-direct", prm, flush=True)
    R, _ = noisy(30, 77)
    ind, arb, _ = pairs_probabilities_mex(R, *prm)
    io, ao = oracle.pairs_probabilities(R, *prm)
    for g, o in ((ind, io), (arb, ao)):
        assert np.array_equal(np.isnan(g), np.isnan(o)) and np.array_equal(np.isneginf(g), np.isneginf(o))
        f = np.isfinite(o)
        assert np.allclose(g[f], o[f], rtol=1e-12, atol=0)
