"""The folded exact polar transform at its edges, against the oracle: sides 1
and 2, odd and even sides around a block of four folded columns and around a
staging block, ray counts whose mirror rays coincide (n_theta = 2, 4, odd
halves), and image counts that take every tile and leave partial ones.

Bar: 1e-12 of the largest value in double (the sums of n^2 terms differ by
their rounding, below n^2 2^-53), 1e-6 in single; the conjugate half exact."""
import numpy as np
import pytest

from aspire_amd.pft import cryo_pft
from oracle import clm_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_r,n_theta,K,dtype", [
    (1, 3, 2, 1, np.float64), (2, 2, 4, 2, np.float64), (3, 5, 6, 15, np.float64), (8, 17, 10, 16, np.float32),
    (9, 16, 36, 17, np.float64), (31, 33, 150, 1, np.float64), (64, 20, 72, 63, np.float64),
    (63, 33, 360, 65, np.float32), (66, 33, 30, 130, np.float64), (130, 40, 360, 200, np.float32)])
def test_folded_transform_matches_the_oracle(n, n_r, n_theta, K, dtype):
    print("case", n, n_r, n_theta, K, dtype, flush=True)
    p = np.random.default_rng(n + K).standard_normal((n, n, K)).astype(dtype)
    pf, _ = cryo_pft(p, n_r, n_theta)
    ref = clm_oracle.cryo_pft(p.astype(np.float64), n_r, n_theta)
    L = n_theta // 2
    assert np.array_equal(pf[:, L:], np.conj(pf[:, :L]))
    bar = 1e-12 if dtype == np.float64 else 1e-6
    assert np.abs(pf - ref).max() <= bar * np.abs(ref).max()
