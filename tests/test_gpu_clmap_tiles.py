"""The filtered search on the matrix cores: records bit-identical to the
oracle's at the edges of its tiles (line counts around a tile's outputs, whole
wraps of small maps inside a halo, the largest radius), with a pair's work in
one workgroup and split over several, and with exact ties and NaN rays, whose
pairs the entry-by-entry kernel decides."""
import numpy as np
import pytest

from aspire_amd.clmatrix import clmatrix_records
from oracle import clm_oracle

pytestmark = pytest.mark.gpu


def check(pf, max_shift, step, d):
    rec, _ = clmatrix_records(np.asfortranarray(pf), max_shift, step, map_filter_radius=d)
    P, _ = clm_oracle.preprocess(pf)
    ora = clm_oracle.pairs(P, max_shift, step, map_filter_radius=d)
    for key, ref in (("cl1", "cl1"), ("cl2", "cl2"), ("j", "j"), ("corr", "best"), ("shift", "shift")):
        assert np.array_equal(rec[key], ora[ref]), key


def rays(n_r, n_theta, K, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((n_r, n_theta, K)) + 1j * rng.standard_normal((n_r, n_theta, K))


@pytest.mark.parametrize("n_r,n_theta,K,max_shift,step,d", [
    (5, 6, 3, 1, 1, 2), (10, 22, 3, 0, 1, 10), (18, 122, 3, 1, 1, 1), (17, 124, 2, 0, 1, 1), (33, 126, 2, 1, 0.3, 1),
    (20, 88, 3, 0, 1, 10), (20, 90, 2, 1, 1, 10), (9, 20, 70, 0, 1, 2), (66, 150, 2, 0, 1, 3)])
def test_records_equal_the_oracle(n_r, n_theta, K, max_shift, step, d):
    print("case", n_r, n_theta, K, max_shift, step, d, flush=True)
    check(rays(n_r, n_theta, K, n_r * n_theta), max_shift, step, d)


@pytest.mark.parametrize("d", [1, 3])
def test_exact_ties_and_nan_rays(d):
    pf = rays(15, 36, 6, 5)
    pf[:, :, 0] = pf[:, :1, 0].real
    pf[:, :, 1] = pf[:, :1, 1].real
    pf[:, :, 2] = 0
    pf[:, 4, 3] = np.nan
    pf[:, 22, 3] = np.nan
    check(pf, 1, 1, d)
