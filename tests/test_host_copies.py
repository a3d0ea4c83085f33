"""Copies to the device that the host does not wait for read memory that is still
there when the stream gets to them (CPU: the HIP runtime replaced by a stand-in
that reads a copy's source when the stream is waited for).

Every form of the search, with tiles built and found in the cache, with and
without pairs, selected pairs among them; the polar transform's and the other
callers' own uploads are waited for on the spot."""
import pytest

from tests import hip_stub

FORMS = {
    "search": "r = [search(h, params(K, 17, 36, prec))[0] for prec in ('fp64', 'fp32', 'fp16', 'bf16') for K in (0, 1, 2, 9, 9)]",
    "noalloc": "r = [search(h, params(9, 17, 36, prec), 'clm_clmatrix_device_noalloc')[0] for prec in ('fp64', 'fp16') for _ in range(2)]",
    "filtered": """r = []
for _ in range(2):
    p = params(9, 17, 36, 'fp64')
    r.append(L.clm_clmatrix_filtered_device(h, ctypes.byref(p), 2, PTR, PTR, PTR, PTR, PTR, PTR, None))""",
    "grouped": """r = []
for flags in (0, 1, 1):
    ps = (_lib.ClmParams * 3)(params(5, 17, 36, 'fp64'), params(6, 17, 36, 'fp16'), params(0, 17, 36, 'fp32'))
    ios = (_lib.ClmStackIO * 3)(*[_lib.ClmStackIO(*[PTR.value] * 6) for _ in range(3)])
    r.append(L.clm_clmatrix_grouped(h, 3, ps, ios, flags, None))""",
    "subset": """r = []
for n in (0, 3):
    stub.stub_int(n)
    for prec in ('fp64', 'fp16'):
        p = params(9, 17, 36, prec)
        r.append(L.clm_clmatrix_subset_device(h, ctypes.byref(p), PTR, PTR, PTR, PTR, PTR, PTR, PTR, None))""",
    "rotations": """r = []
p = params(9, 17, 36, 'fp64')
for _ in range(2):
    r.append(L.clm_common_lines_from_rotations(h, ctypes.byref(p), PTR, PTR, None, PTR, PTR, PTR))""",
    "windowed": """r = []
p = params(9, 17, 36, 'fp16')
for _ in range(2):
    r.append(L.clm_clmatrix_windowed(h, ctypes.byref(p), PTR, PTR, 1.0, 0.1, PTR, PTR, PTR, PTR, PTR, PTR, None))""",
    "autotune": """r = []
p = params(9, 17, 36, 'fp16')
n = ctypes.c_int32(0)
r.append(L.clm_autotune(h, ctypes.byref(p), PTR, 0, None, 0, ctypes.byref(n)))""",
}


@pytest.mark.parametrize("form", sorted(FORMS))
def test_sources_outlive_their_copies(form, tmp_path):
    out = hip_stub.run("h = context()\n" + FORMS[form] + """
L.clm_destroy(h)
print(json.dumps(dict(rc=r, launches=stub.stub_launches(), lost=stub.stub_lost())))
""", tmp_path)
    assert not any(out["rc"]) and out["launches"] > 0, out
    assert out["lost"] == 0, out
