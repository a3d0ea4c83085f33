"""Runs a script against libclm's host code with the HIP runtime replaced by
hip_stub.c: build it, load it ahead of libclm.so in a process of its own, and
return what the script prints (one JSON line)."""
import json
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))

PRELUDE = """
import ctypes, json, struct, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_name.restype = ctypes.c_char_p
stub.stub_arg.restype = ctypes.c_void_p
stub.stub_lost.restype = ctypes.c_long
from aspire_amd import _lib
L = _lib.load()

def context():
    err = ctypes.c_int(0)
    h = L.clm_create(0, ctypes.byref(err))
    assert h and not err.value, err.value
    return h

def params(K, n_r, n_theta, precision, max_shift=2.0, step=1.0, variant=0, reserved=0):
    p = _lib.default_params()
    p.K, p.n_r, p.n_theta, p.pf_dtype = K, n_r, n_theta, _lib.CLM_C128
    p.max_shift, p.shift_step, p.precision, p.variant, p.reserved = max_shift, step, _lib.PRECISIONS[precision], variant, reserved
    return p

BUF = ctypes.create_string_buffer(1 << 16)  # stands for device pointers (nothing reads them)
PTR = ctypes.cast(BUF, ctypes.c_void_p)

def search(h, p, entry="clm_clmatrix_device"):
    st = _lib.ClmStats()
    rc = getattr(L, entry)(h, ctypes.byref(p), PTR, PTR, PTR, PTR, PTR, PTR, ctypes.byref(st))
    return rc, st

def launches(part):
    return [i for i in range(stub.stub_launches()) if part in stub.stub_name(i).decode()]

# fields of the pair kernels' argument, by byte offset
def pair_arg(i):
    a = ctypes.string_at(stub.stub_arg(i), 96)
    cpp, passes, lag, prio = struct.unpack_from("<4i", a, 72)
    return dict(name=stub.stub_name(i).decode(), waves=stub.stub_block(i) // 64, cpp=cpp, passes=passes, lag=lag)
"""


def run(script, tmp_path):
    so = os.path.join(str(tmp_path), "libhip_stub.so")
    subprocess.run(["gcc", "-O1", "-std=c11", "-Wall", "-Wextra", "-Werror", "-fPIC", "-shared",
                    os.path.join(HERE, "hip_stub.c"), "-o", so], check=True)
    # freed memory is filled at once and stays mapped, so that a copy from it shows
    env = dict(os.environ, MALLOC_PERTURB_="165", MALLOC_MMAP_THRESHOLD_=str(1 << 30),
               MALLOC_TRIM_THRESHOLD_=str(1 << 40), PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", PRELUDE + script, so], env=env, cwd=ROOT, capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stderr
    return json.loads(r.stdout.strip().splitlines()[-1])
