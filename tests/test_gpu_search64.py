"""The FP64 search on the matrix cores: records bit-identical to the oracle's
at the edges of its tiles (line counts around 16, 64 and one sweep of columns,
ray lengths around each padded k-step count), on symmetric and asymmetric
shift grids, few and many pairs (a pair's work split over workgroups or not),
and where many candidates tie exactly (equal rays, zero images) or are NaN, so
that the exhaustive kernel decides."""
import numpy as np
import pytest

from aspire_amd.clmatrix import clmatrix_grouped, clmatrix_records
from oracle import clm_oracle

pytestmark = pytest.mark.gpu


def rays(n_r, n_theta, K, seed):
    rng = np.random.default_rng(seed)
    pf = rng.standard_normal((n_r, n_theta, K)) + 1j * rng.standard_normal((n_r, n_theta, K))
    return np.asfortranarray(pf)


def check(pf, max_shift, step, rec=None):
    if rec is None:
        rec, _ = clmatrix_records(pf, max_shift, step, precision="fp64")
    P, _ = clm_oracle.preprocess(pf)
    ora = clm_oracle.pairs(P, max_shift, step, *clm_oracle.all_pairs(pf.shape[2]))
    for key, ref in (("cl1", "cl1"), ("cl2", "cl2"), ("j", "j"), ("corr", "best"), ("shift", "shift")):
        assert np.array_equal(rec[key], ora[ref]), key


@pytest.mark.parametrize("n_r,n_theta,K,max_shift,step", [
    (4, 6, 3, 0, 1), (17, 32, 5, 2, 1), (18, 34, 4, 2, 0.3), (33, 128, 3, 3, 1), (34, 130, 3, 1, 0.5),
    (50, 72, 4, 0, 1), (66, 384, 2, 1, 1), (66, 386, 2, 1, 0.7), (98, 150, 3, 2, 1), (129, 300, 2, 1, 1),
    (20, 24, 70, 1, 1)])
def test_records_equal_the_oracle(n_r, n_theta, K, max_shift, step):
    print("case", n_r, n_theta, K, max_shift, step, flush=True)
    check(rays(n_r, n_theta, K, n_r + n_theta), max_shift, step)


@pytest.mark.parametrize("step", [1, 0.3])
def test_exact_ties_and_missing_rays(step):
    pf = rays(21, 40, 6, 9)
    pf[:, :, 0] = pf[:, :1, 0].real     # every ray equal and real: all candidates of a shift tie
    pf[:, :, 1] = pf[:, :1, 0].real
    pf[:, :, 2] = 0                     # no norm: NaN rays
    pf[:, 3, 3] = np.nan
    pf[:, 23, 3] = np.nan
    pf[:, :20, 4] = np.repeat(pf[:, :5, 4], 4, axis=1)  # each ray four times
    pf[:, 20:, 4] = np.conj(pf[:, :20, 4])
    check(pf, 2, step)


def test_grouped_stacks_of_different_shapes():
    import torch

    pfs = [rays(17, 30, 9, 1), rays(40, 72, 12, 2), rays(17, 30, 2, 3)]
    dev = [torch.as_tensor(np.ascontiguousarray(p.transpose(2, 1, 0)), device="cuda").permute(2, 1, 0) for p in pfs]
    out = None
    for _ in range(3):
        out, _ = clmatrix_grouped(dev, [1, 2, 1], [1, 0.3, 1], "fp64", out=out)
        torch.cuda.synchronize()
    for p, o, ms, ss in zip(pfs, out, [1, 2, 1], [1, 0.3, 1]):
        check(p, ms, ss, {k: v.cpu().numpy() for k, v in o.items()})
