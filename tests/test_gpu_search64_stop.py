"""FP64 search of pairs that are ties everywhere, where a wave stops once its list
has overflowed for good: the records are the oracle's first ties, for radially
symmetric images, for lines that repeat (225 ties, more than a list and fewer than
a wave stops at), beside images without ties, over one sweep of the columns and
several, with few pairs (whose shifts and row blocks are split over workgroups)
and many, of maps with and without the filter."""
import numpy as np
import pytest

from aspire_amd.clmatrix import clmatrix_records
from tests.gpu_helpers import oracle_records

pytestmark = pytest.mark.gpu


def stack(K, n_r, n_theta, seed):
    rng = np.random.default_rng(seed)
    pf = rng.standard_normal((n_r, n_theta, K)) + 1j * rng.standard_normal((n_r, n_theta, K))
    for k in range(0, K, 3):
        pf[:, :, k] = np.abs(pf[:, :1, k])
    for k in range(1, K, 3):
        pf[:, :, k] = pf[:, np.arange(n_theta) % (n_theta // 30), k]
    return pf


@pytest.mark.parametrize("K,n_r,n_theta,ms", [(5, 12, 60, 1), (9, 17, 300, 2), (40, 13, 120, 1), (7, 9, 480, 1)])
def test_ties(oracle, K, n_r, n_theta, ms):
    print("case search64-stop", K, n_r, n_theta, flush=True)
    pf = stack(K, n_r, n_theta, K)
    k1, k2 = oracle.all_pairs(K)
    _, ora = oracle_records(oracle, pf, ms, 1, k1, k2)
    rec, _ = clmatrix_records(pf, ms, 1, precision="fp64")
    for a, b in (("cl1", "cl1"), ("cl2", "cl2"), ("j", "j"), ("corr", "best"), ("shift", "shift")):
        assert np.array_equal(rec[a], ora[b]), a


@pytest.mark.parametrize("K,n_r,n_theta,d", [(5, 12, 60, 1), (6, 9, 150, 3), (60, 9, 60, 2)])
def test_filtered_ties(oracle, K, n_r, n_theta, d):
    print("case clmap64-stop", K, n_r, n_theta, d, flush=True)
    pf = stack(K, n_r, n_theta, K)
    rec, _ = clmatrix_records(pf, 0, 1, precision="fp64", map_filter_radius=d)
    k1, k2 = oracle.all_pairs(K)
    P, _ = oracle.preprocess(pf)
    ora = oracle.pairs(P, 0, 1, k1, k2, map_filter_radius=d)
    for a, b in (("cl1", "cl1"), ("cl2", "cl2"), ("j", "j"), ("corr", "best"), ("shift", "shift")):
        assert np.array_equal(rec[a], ora[b]), a
