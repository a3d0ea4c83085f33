"""Images with infinities and NaN through the exact polar transform, against the
oracle: every value that such a pixel reaches is an infinity of its weight's sign
or NaN, as in the sums as written, on the axes, at the middle (where all but one
of the folded planes vanish) and off them; the other images of the stack keep
their bits.

Signs are compared where the oracle's value is infinite: the weights there are
cosines of phases that both sides form alike."""
import numpy as np
import pytest

from aspire_amd.pft import cryo_pft

pytestmark = pytest.mark.gpu


def kinds(a):
    return np.where(np.isnan(a), 2.0, np.where(np.isinf(a), np.sign(a), 0.0))


@pytest.mark.parametrize("n,n_r,n_theta", [(9, 5, 12), (16, 9, 10), (40, 21, 36)])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_non_finite_pixels(oracle, n, n_r, n_theta, dt):
    print("case pft-non-finite", n, n_r, n_theta, dt, flush=True)
    c = n // 2
    p = np.random.default_rng(n).standard_normal((n, n, 20)).astype(dt)
    want, _ = cryo_pft(p, n_r, n_theta)
    bad = p.copy()
    bad[c, c, 0] = np.nan
    bad[c, c, 1] = np.inf
    bad[c, 1, 3] = -np.inf
    bad[2, c, 4] = np.nan
    bad[0, n - 1, 7] = np.inf
    bad[[1, n - 1], [n - 1, 0], 16] = np.inf, -np.inf
    bad[..., 18] = np.inf
    hit = [0, 1, 3, 4, 7, 16, 18]
    got, _ = cryo_pft(bad, n_r, n_theta)
    with np.errstate(invalid="ignore"):
        ref = oracle.cryo_pft(bad.astype(np.float64), n_r, n_theta)
    for i in range(20):
        if i in hit:
            for part in ("real", "imag"):
                g, r = kinds(getattr(got[..., i], part)), kinds(getattr(ref[..., i], part))
                assert np.array_equal(g, r), (i, part, (g != r).sum())
        else:
            assert np.array_equal(got[..., i], want[..., i]), i
