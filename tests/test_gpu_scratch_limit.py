"""The allocation-free call at the images that only the split of least padding
leaves room for: the same records as the allocating call, which takes another
split there."""
import numpy as np
import pytest

from aspire_amd import _lib
from tests.test_zz_no_alloc import run, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,n_r,n_theta,ms,prec", [(510, 90, 300, 0.0, "fp16"), (187, 45, 300, 6.0, "fp16")])
def test_at_the_limit(K, n_r, n_theta, ms, prec):
    import torch

    print("case scratch-limit", K, n_r, n_theta, flush=True)
    g = torch.Generator(device="cuda").manual_seed(K)
    pf = torch.randn((K, n_theta, n_r), generator=g, dtype=torch.complex128, device="cuda").permute(2, 1, 0)
    got, sg, rc = run(_lib.Context(0), "clm_clmatrix_device_noalloc", pf, ms, 0.5, prec)
    assert rc == 0
    ref, sr, rc = run(_lib.context(0), "clm_clmatrix_device", pf, ms, 0.5, prec)
    assert rc == 0 and sg["variant"] != sr["variant"]
    assert same(got, ref)
