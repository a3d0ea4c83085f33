"""The NUFFT method gives each image a grid of its own: what stands beside it in
the stack, and how many images there are, leaves its transform's bits as they
are, and its error stays the method's where its neighbours' spectra are
concentrated (a constant, a smooth blob) and its own is flat (a point, noise).

Grid sides: even and odd ones (45, 75), windows across both ends of the columns
kept (n_theta = 2 has fx = 0 alone), boxed and direct interpolation.  Error:
1e-13 of the image's own largest |pf|, the method's bound, against sums of
extended precision at a sample of the points."""
import numpy as np
import pytest

from aspire_amd import pft as gpft

pytestmark = pytest.mark.gpu


def dev(p):
    import torch

    return torch.as_tensor(np.ascontiguousarray(p.transpose(2, 1, 0))).cuda().permute(2, 1, 0)


def images(n, seed):
    rng = np.random.default_rng(seed)
    t = np.arange(n) - n // 2
    point = np.zeros((n, n))
    point[n // 3, n // 2] = 1.0
    blob = np.exp(-(t[:, None] ** 2 + t[None, :] ** 2) / (2 * (n / 6) ** 2))
    return np.stack([point, np.ones((n, n)), rng.standard_normal((n, n)), blob, point.T], axis=2)


def extended(p, n_r, n_theta, ks, js):
    """pf at the points (ks, js) in extended precision, at the rounded frequencies."""
    n = p.shape[0]
    fr = gpft.pft_freqs(n_r, n_theta).astype(np.longdouble)
    f = fr[js * n_r + ks]
    g = np.ceil(np.arange(n) - n / 2).astype(np.longdouble)
    ax, ay = f[:, :1] * g, f[:, 1:] * g
    cx, sx, cy, sy = np.cos(ax), np.sin(ax), np.cos(ay), np.sin(ay)
    q = p.astype(np.longdouble)
    tc, ts = cx @ q, sx @ q
    return (tc * cy - ts * sy).sum(1).astype(np.float64) + 1j * (tc * sy + ts * cy).sum(1).astype(np.float64)


@pytest.mark.parametrize("n,n_r,n_theta", [(20, 11, 12), (22, 11, 2), (37, 7, 36), (129, 65, 60), (185, 20, 10)])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_bits_do_not_depend_on_the_neighbours(n, n_r, n_theta, dt):
    print("case pft-own-grid", n, n_r, n_theta, dt, flush=True)
    p = images(n, n).astype(dt)
    whole = gpft.cryo_pft(dev(p), n_r, n_theta, method="nufft")[0].cpu().numpy()
    other = gpft.cryo_pft(dev(p[..., [3, 0, 4, 2]]), n_r, n_theta, method="nufft")[0].cpu().numpy()
    for at, i in enumerate([3, 0, 4, 2]):
        assert np.array_equal(whole[..., i], other[..., at]), i
    for i in range(5):
        alone = gpft.cryo_pft(dev(p[..., i:i + 1]), n_r, n_theta, method="nufft")[0].cpu().numpy()
        assert np.array_equal(whole[..., i], alone[..., 0]), i


@pytest.mark.parametrize("n,n_r,n_theta", [(22, 12, 2), (37, 19, 12), (359, 180, 6), (700, 350, 6), (700, 60, 10)])
def test_error_beside_concentrated_spectra(n, n_r, n_theta):
    p = images(n, n + 1)
    got = gpft.cryo_pft(dev(p), n_r, n_theta, method="nufft")[0].cpu().numpy()
    rng = np.random.default_rng(3)
    m = min(150, n_r * (n_theta // 2))
    at = rng.choice(n_r * (n_theta // 2), m, replace=False)
    ks, js = at % n_r, at // n_r
    for i in range(p.shape[2]):
        ref = extended(p[..., i], n_r, n_theta, ks, js)
        err = np.abs(got[ks, js, i] - ref).max() / np.abs(got[..., i]).max()
        print("case pft-own-grid-error", n, n_r, "image", i, "error", err, flush=True)
        assert err <= 1e-13
