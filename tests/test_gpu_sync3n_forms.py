"""The likelihood sums of pairs_probabilities in every form the parameters
choose (products of likelihoods: b above, equal to and below a; a logarithm per
score: P2 = 1, x0 above 1, a far from b; the direct form: P2 = 0 with A < 0), and
the pair kernels at sizes where a third image's stage lies before, between,
after and among the pair's blocks, against the one-thread oracle.

Log-likelihoods: 1e-12 relative (sums of 2(N-2) terms and of their
logarithms, each within a few units in the last place); scores, counts and
signs products exactly."""
import numpy as np
import pytest

from aspire_amd.sync3n import pairs_probabilities_mex, signs_times_v_mex, triangles_scores_mex
from tests.test_sync3n_oracle import noisy, rel_rotations
from aspire_amd import sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prm", [(0.5, 1.0, 2.2, 1.0, 2.5, 0.78), (0.3, 2.0, 3.0, 0.7, 3.0, 0.6),
                                 (0.6, 0.8, 4.5, 1.3, 1.5, 0.9), (1.0, 1.0, 2.2, 1.0, 2.5, 0.78),
                                 (0.5, 1.0, 2.2, 1.0, 2.5, 1.5), (0.2, 1.0, 0.5, 1.0, 20.0, 0.5),
                                 (0.9, 1.0, 1.0, 1.0, 6.0, 0.999)])
@pytest.mark.parametrize("N", [5, 33, 50])
def test_probabilities(oracle, N, prm):
    print("case", N, prm, flush=True)
    R, _ = noisy(N, 300 + N)
    ind, arb, _ = pairs_probabilities_mex(R, *prm)
    io, ao = oracle.pairs_probabilities(R, *prm)
    assert np.allclose(ind, io, rtol=1e-12, atol=0) and np.allclose(arb, ao, rtol=1e-12, atol=0)


def test_probabilities_of_perfect_scores(oracle):
    # rotations of the cube: products are exact, so mismatches are exactly 0
    # (scores of 1, logarithms of 0) and some alternatives too (0/0)
    rng = np.random.default_rng(2)
    rots = np.zeros((3, 3, 20))
    for k in range(20):
        m = np.eye(3)[rng.permutation(3)] * rng.choice([-1.0, 1.0], 3)
        rots[:, :, k] = m if np.linalg.det(m) > 0 else -m
    R, _ = rel_rotations(rots)
    ind, arb, _ = pairs_probabilities_mex(R, 0.5, 1.0, 2.2, 1.0, 2.5, 0.78)
    io, ao = oracle.pairs_probabilities(R, 0.5, 1.0, 2.2, 1.0, 2.5, 0.78)
    for a, b in ((ind, io), (arb, ao)):
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isneginf(a), np.isneginf(b))
        f = np.isfinite(b)
        assert np.allclose(a[f], b[f], rtol=1e-12, atol=0)


@pytest.mark.parametrize("N", [16, 31, 49, 97])
def test_scores_and_signs(oracle, N):
    R, _ = noisy(N, 400 + N)
    c, h, _ = triangles_scores_mex(R, 64)
    co, ho = oracle.triangles_scores(R, 64)
    assert np.array_equal(h, ho) and np.array_equal(c, co)
    rng = np.random.default_rng(N)
    P = N * (N - 1) // 2
    v, w = rng.standard_normal((P, 5)), rng.random(P)
    for entries in (0, 1, 2):
        ps = w if entries == 2 else None
        assert np.array_equal(signs_times_v_mex(R, v, entries, ps)[0], oracle.signs_times_v(R, v, entries, ps))
