"""The second pass after a first pass that took a pair's column groups one after
another, and selected pairs of the same shape: FP32, 300 rays, lines that repeat
every 10, so that each pair has 225 exact ties, in more cells than the 58 a
record holds and fewer than the 1024 candidates of a list.

The ties' values are the same products in the same order, so both forms of the
first pass give the same records, and the first tie is the oracle's."""
import numpy as np
import pytest

from aspire_amd.clmatrix import clmatrix_records
from tests.gpu_helpers import assert_parity, compare, oracle_records

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_r", [13, 44, 90])
def test_second_pass(oracle, n_r):
    K, n_theta = 8, 300
    rng = np.random.default_rng(n_r)
    f = rng.standard_normal((n_r, 10, K)) + 1j * rng.standard_normal((n_r, 10, K))
    pf = f[:, np.arange(n_theta) % 10]
    a, sa = clmatrix_records(pf, 2, 1, precision="fp32", variant=105)
    b, sb = clmatrix_records(pf, 2, 1, precision="fp32", variant=154)
    print("case second-after-passes", n_r, sb, flush=True)
    assert sb["variant"] == 154 and sb["uncertain_pairs"] == K * (K - 1) // 2 and sb["emitted"] > 0
    assert sb["fallback_pairs"] == 0
    sel = (np.arange(K * (K - 1) // 2) % 3 != 0).astype(np.uint8)
    c, sc = clmatrix_records(pf, 2, 1, precision="fp32", variant=154, sel=sel)
    assert sc["emitted"] > 0
    for key in a:
        assert np.array_equal(a[key], b[key]), key
        assert np.array_equal(a[key][sel != 0], c[key][sel != 0]), key
    k1, k2 = oracle.all_pairs(K)
    P, ora = oracle_records(oracle, pf, 2, 1, k1, k2)
    assert_parity(compare(oracle, P, ora, b, 2, 1, k1, k2))
