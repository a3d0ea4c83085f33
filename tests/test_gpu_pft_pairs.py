"""Images share the NUFFT's grids two by two: an image's transform must not
depend on what its partner holds.

Each image is held to 1e-13 of its own largest |pf| (the method's bound)
whatever the norms of its neighbours, from 1e-200 to 1e200, whose squares leave the
range of a double; a lone image (odd counts) and one beside zeros give the
same; an image with a NaN or an infinity is non-finite at its own points and
leaves its partner as it was.
"""
import numpy as np
import pytest

from aspire_amd import pft as gpft

pytestmark = pytest.mark.gpu


def dev(p):
    import torch

    return torch.as_tensor(np.ascontiguousarray(p.transpose(2, 1, 0))).cuda().permute(2, 1, 0)


@pytest.mark.parametrize("n,K", [(9, 1), (9, 2), (24, 5), (185, 6), (33, 9)])
def test_images_of_unlike_norms(oracle, n, K):
    print("case nufft-pairs", n, K, flush=True)
    n_r, n_theta = n // 2 + 1, 12
    rng = np.random.default_rng(31 * n + K)
    p = rng.standard_normal((n, n, K))
    ref = oracle.cryo_pft(p, n_r, n_theta)
    # powers of two: the references scale exactly
    e = np.array([0, 660, -660, 30, -30, 0, 1, 700, 0])[:K]
    s = np.ldexp(1.0, e)
    p[..., K - 1] = 0.0  # zeros beside, or as, the last image
    got, _ = gpft.cryo_pft(dev(p * s), n_r, n_theta, method="nufft")
    got = got.cpu().numpy()
    assert not got[..., K - 1].any()
    for i in range(K - 1):
        err = np.abs(got[..., i] / s[i] - ref[..., i]).max()
        print("image", i, "error", err / np.abs(ref[..., i]).max(), flush=True)
        assert err <= 1e-13 * np.abs(ref[..., i]).max()


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_partner_of_a_non_finite_image(dt, bad):
    print("case nufft-bad", dt, bad, flush=True)
    rng = np.random.default_rng(7)
    p = rng.standard_normal((20, 20, 5)).astype(dt)
    clean = p.copy()
    p[3, 4, 1] = bad
    p[0, 0, 2] = bad
    p[5, 5, 4] = bad
    clean[..., [1, 2, 4]] = 0.0
    got = gpft.cryo_pft(dev(p), 11, 12, method="nufft")[0].cpu().numpy()
    want = gpft.cryo_pft(dev(clean), 11, 12, method="nufft")[0].cpu().numpy()
    for i in (1, 2, 4):
        assert not np.isfinite(got[..., i]).any()
    for i in (0, 3):
        assert np.array_equal(got[..., i], want[..., i])
