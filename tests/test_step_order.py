"""LSQR's step publishes a workgroup's partial norm before it raises the count of
workgroups that are through, by the order of the instructions (CPU: the device
code as it is compiled): a store past the caches, a wait until it is there, the
count; and the last workgroup's loads of the partial norms go past its caches."""
import os
import re
import subprocess

from aspire_amd import build

SRC = os.path.join(build.CSRC, "shifts.hip")


def test_partial_norm_before_count(tmp_path):
    out = str(tmp_path / "shifts.s")
    subprocess.run([build.hipcc(), *build.HIPCC_FLAGS, "-I", os.path.join(build.ROOT, "include"), "-I", build.CSRC,
                    "--offload-device-only", "-S", "-o", out, SRC], check=True, capture_output=True)
    text = open(out).read()
    bodies = re.findall(r"^(_ZN3lsq11step_kernel\S+):.*?\n(.*?)^\.Lfunc_end", text, flags=re.S | re.M)
    assert len(bodies) == 2
    for name, body in bodies:
        code = re.sub(r"\s*;.*", "", body)
        at = code.index("global_atomic_add ")
        before = code[:at]
        stores = [m.start() for m in re.finditer(r"global_store_dwordx2 .*sc1", before)]
        assert stores, name
        assert re.search(r"s_waitcnt vmcnt\(0\)", before[stores[-1]:]), name
        assert len(re.findall(r"global_load_dwordx2 .*sc1", code[at:])) >= 8, name
