"""The shapes that fit the allocation-free call's scratch array (CPU: the HIP
runtime replaced by a stand-in): where the split with the most even loads pads
the columns past the array, the split of least padding is taken, so the call
takes as many images as that one leaves room for.  One image more is refused
with the sizes, before any kernel, and the context goes on."""
import pytest

from tests import hip_stub

# n_r, n_theta, max_shift (step 0.5), precision, images that fit with the least padding
CASES = [(120, 150, 0.0, "fp16", 643), (120, 180, 6.0, "bf16", 127), (90, 180, 0.0, "fp16", 739),
         (65, 420, 0.0, "bf16", 527), (45, 300, 6.0, "fp16", 187), (17, 420, 6.0, "fp16", 333),
         (17, 300, 0.0, "fp32", 1353), (65, 360, 0.0, "fp32", 693),
         (17, 300, 0.0, "fp32", 1376), (17, 420, 6.0, "fp32", 467)]


@pytest.mark.parametrize("n_r,n_theta,ms,prec,K", CASES)
def test_scratch_holds(n_r, n_theta, ms, prec, K, tmp_path):
    out = hip_stub.run(f"""
h = context()
def go(K, entry="clm_clmatrix_device_noalloc"):
    stub.stub_reset()
    rc, st = search(h, params(K, {n_r}, {n_theta}, {prec!r}, max_shift={ms}, step=0.5), entry)
    return rc, st.variant, stub.stub_launches(), L.clm_last_error(h).decode()
print(json.dumps(dict(fits=go({K}), more=go(2 * {K}), small=go({K} // 2), device=go({K} // 2, "clm_clmatrix_device"))))
""", tmp_path)
    assert out["fits"][0] == 0 and out["fits"][2] > 0, out
    assert out["more"][0] == -4 and out["more"][2] == 0 and "scratch" in out["more"][3]
    # where there is room the call is the allocating one's
    assert out["small"][0] == 0 and out["small"][1] == out["device"][1]
