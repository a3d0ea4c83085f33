"""A pair's columns taken one group after another by one wave (variant ids with
50 added to the waves), against the waves side by side and the oracle.

Shapes where the split leaves remainders: column tiles that do not divide
(300, 180 and 72 rays), pair counts that leave a workgroup's last waves idle,
one pair, and every padded ray length the loop is built for.  The records are
certified, so both forms give the same bits.
"""
import numpy as np
import pytest

from aspire_amd import sim
from aspire_amd.clmatrix import clmatrix_records
from tests.gpu_helpers import assert_parity, compare, oracle_records

pytestmark = pytest.mark.gpu

CASES = [
    # K, n_r, n_theta, precision, side by side, one after another
    (9, 13, 300, "fp32", 105, 154),
    (2, 30, 300, "fp32", 105, 154),
    (6, 44, 300, "fp32", 105, 154),
    (7, 30, 360, "fp32", 206, 254),
    (7, 60, 180, "fp32", 106, 154),
    (6, 90, 72, "fp32", 104, 154),
    (6, 120, 360, "fp32", 106, 154),
    (10, 90, 360, "fp16", 206, 258),
    (7, 90, 300, "bf16", 105, 158),
    (5, 120, 180, "bf16", 106, 158),
]


@pytest.mark.parametrize("K,n_r,n_theta,prec,side,one", CASES)
def test_passes_agree(oracle, K, n_r, n_theta, prec, side, one):
    print("case pair-passes", K, n_r, n_theta, prec, one, flush=True)
    pf = sim.make_stack(K=K, n=2 * n_r - 1, n_r=n_r, n_theta=n_theta, snr=1.0, max_shift_2d=1, shift_kind="int",
                        seed=K + n_r).pf
    a, sa = clmatrix_records(pf, 2, 1, precision=prec, variant=side)
    b, sb = clmatrix_records(pf, 2, 1, precision=prec, variant=one)
    assert sa["variant"] == side and sb["variant"] == one
    for key in a:
        assert np.array_equal(a[key], b[key]), key
    k1, k2 = oracle.all_pairs(K)
    P, ora = oracle_records(oracle, pf, 2, 1, k1, k2)
    assert_parity(compare(oracle, P, ora, b, 2, 1, k1, k2))


def test_even_loads_are_chosen():
    # 300 rays are five column tiles: never five waves on four SIMDs once the pairs are many
    pf = sim.make_stack(K=60, n=25, n_r=13, n_theta=300, snr=1.0, max_shift_2d=1, shift_kind="int", seed=5).pf
    for prec in ("fp32", "fp16"):
        rec, st = clmatrix_records(pf, 1, 1, precision=prec)
        ref, sr = clmatrix_records(pf, 1, 1, precision=prec, variant=105)
        assert st["variant"] != sr["variant"] == 105
        for key in rec:
            assert np.array_equal(rec[key], ref[key]), key
