"""The vote's histogram on the matrix cores at its edges: every block equal to
the oracle's, whose peak is found term by term.

K around one and several 64-triangle chunks, one triangle per pair (K = 3,
whose angle often lies halfway between two points: the ties that the
term-by-term path decides), stacks of one axis of symmetry (exact ties in
every pair), missing lines, tables too large for LDS, and angles at 0 and 180
degrees.  The sums of a block differ from the oracle's by rounding in at most
K terms of magnitude 1, so blocks agree to K 2^-52 times a small factor: 1e-10.
"""
import numpy as np
import pytest

from aspire_amd import sim
from aspire_amd.vote import cryo_syncmatrix_vote
from oracle import clm_oracle as co

pytestmark = pytest.mark.gpu


def lines(K, T, seed, kind):
    rng = np.random.default_rng(seed)
    if kind == "random":
        cl = np.zeros((K, K))
        i, j = np.triu_indices(K, 1)
        cl[i, j] = rng.integers(0, T // 2 + 1, i.size)  # 0: no common line
        cl[j, i] = np.where(cl[i, j] > 0, rng.integers(1, T + 1, i.size), 0)
        return cl
    cl = sim.clmatrix_cheat(sim.rand_rots(rng, K), T)
    if kind == "quarter":  # lines on multiples of 45 degrees: angles at 0, 45, 90, 180
        step = T // 8
        cl = np.where(cl > 0, (np.round((cl - 1) / step) * step) % T + 1, 0)
        np.fill_diagonal(cl, 0)
    return cl


@pytest.mark.parametrize("K,T,kind", [(2, 360, "true"), (3, 360, "true"), (3, 360, "quarter"), (9, 360, "quarter"),
                                      (63, 72, "random"), (64, 150, "true"), (65, 360, "random"),
                                      (130, 360, "quarter"), (40, 600, "random"), (129, 512, "true")])
def test_blocks_equal_the_oracle(K, T, kind):
    print("case", K, T, kind, flush=True)
    cl = lines(K, T, 31 * K + T, kind)
    S, ref = cryo_syncmatrix_vote(cl, T), co.syncmatrix_vote(cl, T)
    assert np.array_equal(S, S.T)
    k1, k2 = np.triu_indices(K, 1)
    worst = max(np.abs(S[2 * a:2 * a + 2, 2 * b:2 * b + 2] - ref[2 * a:2 * a + 2, 2 * b:2 * b + 2]).max()
                for a, b in zip(k1, k2))
    assert worst <= 1e-10, worst
