"""Lines and 1-D shifts of known rotations at the edges of their kernel, equal
to the oracle's exactly: shift counts around one column tile, one group of
three and several groups, one shift, ray lengths up to the longest, selections
that leave a wave with none, one, 15, 16, 17 or all of its 64 pairs, and images
whose maximum ties or is NaN (equal real rays, no rays), which are decided term
by term."""
import numpy as np
import pytest

from aspire_amd import sim
from aspire_amd.shifts import common_lines_from_rotations
from oracle import clm_oracle, shifts_oracle

pytestmark = pytest.mark.gpu


def check(pf, rots, max_shift, step, sel=None):
    K, n_theta = pf.shape[2], pf.shape[1]
    cl1, cl2, s = (t.cpu().numpy() for t in common_lines_from_rotations(np.asfortranarray(pf), rots, max_shift, step, sel))
    k1, k2 = clm_oracle.all_pairs(K)
    on = np.ones(k1.size, bool) if sel is None else sel != 0
    P, _ = clm_oracle.preprocess(pf)
    ref = shifts_oracle.rotation_pairs(P, rots, n_theta, max_shift, step, k1[on], k2[on])
    assert np.array_equal(cl1[on], ref["cl1"]) and np.array_equal(cl2[on], ref["cl2"])
    assert np.array_equal(s[on], ref["shift"])
    assert np.all(cl1[~on] == -1) and np.all(cl2[~on] == -1) and np.all(s[~on] == 0)


def stack(n_r, n_theta, K, seed):
    rng = np.random.default_rng(seed)
    pf = rng.standard_normal((n_r, n_theta, K)) + 1j * rng.standard_normal((n_r, n_theta, K))
    return pf, sim.rand_rots(rng, K)


@pytest.mark.parametrize("n_r,n_theta,K,max_shift,step", [
    (5, 36, 9, 0, 1), (18, 72, 12, 7.5, 1), (18, 72, 12, 8, 1), (33, 150, 11, 23.5, 1), (34, 150, 8, 24, 1),
    (66, 72, 6, 10, 0.3), (129, 360, 5, 60, 1)])
def test_lines_and_shifts_equal_the_oracle(n_r, n_theta, K, max_shift, step):
    print("case", n_r, n_theta, K, max_shift, step, flush=True)
    check(*stack(n_r, n_theta, K, n_r), max_shift, step)


def test_selections():
    pf, rots = stack(9, 36, 30, 3)  # 435 pairs: 6 whole waves and a part
    sel = np.zeros(435, np.uint8)
    for wave, n in enumerate((0, 1, 15, 16, 17, 64, 51)):
        at = np.random.default_rng(wave).permutation(min(64, 435 - 64 * wave))[:n]
        sel[64 * wave + at] = 1
    check(pf, rots, 3, 1, sel)


def test_ties_and_missing_rays():
    pf, rots = stack(17, 36, 8, 4)
    pf[:, :, 0] = pf[:, :1, 0].real
    pf[:, :, 1] = pf[:, :1, 0].real
    pf[:, :, 2] = 0
    pf[:, 5, 3] = np.nan
    pf[:, 23, 3] = np.nan
    check(pf, rots, 4, 0.5)
