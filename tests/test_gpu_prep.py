"""The ray preparation (prep_kernel) at the edges of its line blocks: ray
lengths on both sides of the change from 16 to 8 lines per workgroup, the
shortest and the longest, and line counts that leave a partial block or a
block of padding lines.  The FP64 search is bit-identical to the oracle's
only if every prepared ray is, so its records are compared exactly."""
import numpy as np
import pytest

from aspire_amd.clmatrix import clmatrix_records
from oracle import clm_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_r,n_theta,dtype", [(5, 6, np.complex128), (17, 34, np.complex64), (66, 32, np.complex128),
                                               (67, 18, np.complex128), (97, 50, np.complex64),
                                               (129, 66, np.complex128)])
def test_fp64_records_equal_the_oracle(n_r, n_theta, dtype):
    rng = np.random.default_rng(n_r)
    K = 4
    pf = (rng.standard_normal((n_r, n_theta, K)) + 1j * rng.standard_normal((n_r, n_theta, K))).astype(dtype)
    print("case", n_r, n_theta, dtype, flush=True)
    rec, _ = clmatrix_records(np.asfortranarray(pf), 2, 1, precision="fp64")
    P, _ = clm_oracle.preprocess(pf)
    ora = clm_oracle.pairs(P, 2, 1, *clm_oracle.all_pairs(K))
    for key, ref in (("cl1", "cl1"), ("cl2", "cl2"), ("j", "j"), ("corr", "best")):
        assert np.array_equal(rec[key], ora[ref]), key
