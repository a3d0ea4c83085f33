"""LSQR's tiles of 32 x 256 pairs, the sums over rows of 16 lanes and the scalar
step in the last workgroup, at the sizes where they leave remainders: one
pair, one image past a row block, past a column block, and vectors that just
fill and just pass the workgroups of 64 entries.  Two solves in a row on one
context give the same bits.  1e-10 of the largest entry, as the iterates of
the other sizes: a few hundred ulps of sums whose order differs.
"""
import numpy as np
import pytest

from aspire_amd.shifts import estimate_shifts
from oracle import shifts_oracle as so

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,iters", [(2, 1), (3, 1), (32, 6), (33, 6), (64, 6), (65, 6), (256, 8), (257, 8), (289, 8)])
@pytest.mark.parametrize("damp", [0.0, 0.5])
def test_tiles(K, iters, damp):
    import torch

    print("case lsqr-row-tiles", K, iters, damp, flush=True)
    n_theta = 72
    rng = np.random.default_rng(K)
    P = K * (K - 1) // 2
    cl1 = rng.integers(1, n_theta // 2 + 1, size=P).astype(np.int32)
    cl2 = rng.integers(1, n_theta + 1, size=P).astype(np.int32)
    b = rng.normal(0, 2.0, size=P)
    A, _ = so.system(K, n_theta, cl1, cl2, b)
    xo, io = so.lsqr(A, b, tol=0.0, maxit=iters, damp=damp)
    args = [torch.as_tensor(a).cuda() for a in (cl1, cl2, b)]
    x, st = estimate_shifts(*args, K, n_theta, tol=0.0, maxit=iters, damp=damp)
    again, _ = estimate_shifts(*args, K, n_theta, tol=0.0, maxit=iters, damp=damp)
    assert torch.equal(x, again)
    assert st["iterations"] == io["iterations"]
    np.testing.assert_allclose(x.cpu().numpy().ravel(), xo, rtol=0, atol=1e-10 * np.abs(xo).max())
    assert abs(st["norm_a"] - io.get("norm_a", st["norm_a"])) <= 1e-9 * st["norm_a"]
