"""The re-score by a workgroup per pair (few pairs) against a wave per pair.

The same pairs are searched in a stack of K images, whose pairs are few enough for
a workgroup each, and inside a stack of 60 (1770 pairs: a wave each); the records
must be the same bits.  Noise-free images keep many cells and near-ties a pair,
noise keeps few; one pair, and pairs with no line (zero images), are the edges.
"""
import numpy as np
import pytest

from aspire_amd import sim
from aspire_amd.clmatrix import clmatrix_records

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("snr", [None, 0.5])
@pytest.mark.parametrize("K", [2, 5, 17, 45])
def test_team_matches_waves(prec, snr, K):
    print("case rescore-team", prec, snr, K, flush=True)
    pf = sim.make_stack(K=60, n=33, n_r=17, n_theta=72, snr=snr, max_shift_2d=1, shift_kind="int", seed=11).pf.copy()
    pf[:, :, 1] = 0.0
    few, _ = clmatrix_records(np.asfortranarray(pf[:, :, :K]), 2, 1, precision=prec)
    many, _ = clmatrix_records(pf, 2, 1, precision=prec)
    k1, k2 = np.triu_indices(60, 1)
    inside = k2 < K
    for key in few:
        assert np.array_equal(np.asarray(few[key]), np.asarray(many[key])[inside]), key
