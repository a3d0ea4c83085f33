"""The exact polar transform is evaluated at the reference's rounded frequencies
(cryo_pft.m:49-58) for every ray, the mirror rays that share their products
included: against sums of extended precision at those frequencies.

Bar in double: 4e-15 of the image's largest |pf|.  A weight is off by three
roundings of values up to 1 and its image's share of 2^-9 of the mirror ray's
3e-14; sums of some thousand such terms of white noise stay near 1e-15.  (The
sums as written, with phases rounded to a double, are 1.5e-14 off, and with the
mean frequency for both rays 1.2e-14.)  Scaling an image by a power of two
scales every value, whatever the other images' sizes."""
import numpy as np
import pytest

from aspire_amd.pft import cryo_pft
from tests.test_gpu_pft_own_grid import extended

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_r,n_theta,K", [(129, 65, 360, 2), (129, 65, 360, 70), (64, 32, 150, 17), (33, 40, 6, 65),
                                             (20, 9, 10, 3), (15, 8, 72, 64)])
def test_rounded_frequencies(n, n_r, n_theta, K):
    p = np.random.default_rng(n + K).standard_normal((n, n, K))
    got, _ = cryo_pft(p, n_r, n_theta)
    L = n_theta // 2
    rng = np.random.default_rng(5)
    ks, js = rng.integers(0, n_r, 400), rng.integers(0, L, 400)
    ks[:L], js[:L] = n_r - 1, np.arange(L)[:400]
    for i in sorted({0, K // 2, K - 1}):
        ref = extended(p[..., i], n_r, n_theta, ks, js)
        e = np.abs(got[ks, js, i] - ref) / np.abs(got[..., i]).max()
        print("case pft-frequencies", n, n_r, n_theta, K, "image", i, "error", e.max(), "rms",
              np.sqrt((e ** 2).mean()), flush=True)
        assert e.max() <= 4e-15
    assert np.array_equal(got[:, L:], np.conj(got[:, :L]))


@pytest.mark.parametrize("K", [5, 66])
def test_powers_of_two(K):
    print("case pft-powers", K, flush=True)
    p = np.random.default_rng(K).standard_normal((24, 24, K))
    p[..., 1] = 0.0
    s = np.ldexp(1.0, np.random.default_rng(1).integers(-900, 900, K))
    want, _ = cryo_pft(p, 12, 36)
    got, _ = cryo_pft(p * s, 12, 36)
    assert np.array_equal(got, want * s) and not got[..., 1].any()
