"""What the host launches the pair kernels with (CPU: the HIP runtime replaced by
a stand-in that records launches).

The lagged schedule puts a second wave on each SIMD one tile behind the first: it
is for an even number of waves side by side, whatever the first pass did before,
and it stays off where the caller turns it off.  300 rays are five column tiles;
with pairs enough a wave takes them one after another (four or eight waves), the
second pass and selected pairs five waves side by side."""
import pytest

from tests import hip_stub

SHAPES = [(60, 17, 300, "fp32"), (60, 90, 300, "fp16"), (60, 90, 300, "bf16"), (60, 17, 360, "fp32"),
          (60, 45, 360, "fp16"), (60, 17, 300, "fp16")]


@pytest.mark.parametrize("K,n_r,n_theta,prec", SHAPES)
def test_lagged_schedule(K, n_r, n_theta, prec, tmp_path):
    out = hip_stub.run(f"""
h = context()
r = {{}}
for off in (0, 1):
    p = params({K}, {n_r}, {n_theta}, {prec!r}, reserved=off)
    io = _lib.ClmStackIO(*[PTR.value] * 6)
    stub.stub_reset()
    assert L.clm_clmatrix_grouped(h, 1, ctypes.byref(p), ctypes.byref(io), 1, None) == 0  # captured: both passes
    r["both%d" % off] = [pair_arg(i) for i in launches("pair_kernel")]
    stub.stub_reset()
    stub.stub_int(5)
    assert L.clm_clmatrix_subset_device(h, ctypes.byref(p), *[PTR] * 7, None) == 0
    stub.stub_int(0)
    r["subset%d" % off] = [pair_arg(i) for i in launches("pair_kernel")]
print(json.dumps(r))
""", tmp_path)
    for form in ("both0", "subset0"):
        assert out[form]
        for a in out[form]:
            assert a["lag"] == (a["waves"] % 2 == 0 or a["passes"] > 1), (form, a)
    # the first pass obeys the caller's switch (a refinement by FP32 twins has its own)
    assert out["both1"][0]["lag"] == 0 and out["subset1"][0]["lag"] == 0
    if n_theta == 300 and not (prec == "fp16" and n_r == 17):
        assert out["both0"][0]["passes"] > 1 and out["subset0"][0]["passes"] == 1


# (precision, rays, points, images) of five shifts -> the first pass's variant, any
# within 3% of the fastest measured: column tiles per wave * 100 + waves, + 50 for
# waves that take the column groups in turn
CHOICES = [
    # the least padding, where splits of more even loads are slower
    (("fp32", 420, 120, 90), {107}), (("fp16", 150, 120, 90), {106}), (("bf16", 180, 120, 90), {106}),
    (("fp32", 120, 17, 45), {204}), (("fp16", 360, 17, 45), {308}),
    # more even loads, where they are faster
    (("fp32", 300, 44, 251), {154}), (("fp16", 300, 45, 500), {308}), (("bf16", 360, 91, 400), {258}),
    (("bf16", 300, 91, 300), {258}), (("fp32", 300, 17, 90), {154}),
    # few pairs a compute unit
    (("bf16", 420, 90, 80), {208, 258}), (("fp16", 300, 90, 65), {206}), (("fp32", 360, 33, 12), {106}),
    (("fp32", 300, 45, 40), {154}),
]


def test_split_of_the_first_pass(tmp_path):
    out = hip_stub.run(f"""
h = context()
r = []
for prec, n_theta, n_r, K in {[c[0] for c in CHOICES]!r}:
    rc, st = search(h, params(K, n_r, n_theta, prec))
    r.append([rc, st.variant])
print(json.dumps(r))
""", tmp_path)
    for (shape, want), (rc, got) in zip(CHOICES, out):
        assert rc == 0 and got in want, (shape, got)
