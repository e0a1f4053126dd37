"""Runs host-side checks of the library against tests/fake_hip.cpp, a HIP runtime
without a GPU: `run(body)` executes the source text `body` in a process of its own,
where `hk` is the package's binding, `fake` the stand-in, `log()` its record, and
`small(nanl)` makes a plan of the 2-atom cell."""

import functools
import os
import subprocess
import sys
import tempfile

from tests.conftest import ROOT

_PRELUDE = """
import ctypes as C, os, sys
sys.path.insert(0, {root!r})
fake = C.CDLL({fake!r}, mode=C.RTLD_GLOBAL)
fake.fake_log.restype = C.c_char_p
fake.fake_cost.argtypes = [C.c_char_p, C.c_double, C.c_double, C.c_long]
fake.fake_fail_host_malloc.argtypes = [C.c_long]
fake.fake_live.restype = C.c_long
import numpy as np
from cpw2000_amd import hk_psi as hk, synth

def log():
    return fake.fake_log().decode().split("\\n")

def device_array(n):
    p = C.c_void_p()
    assert fake.hipMalloc(C.byref(p), C.c_size_t(n)) == 0
    return p

def small(nanl=0, seed=0, **kw):
    d = synth.make_config(0, nbands=2, **kw)
    if nanl:
        rng = np.random.default_rng(seed)
        m = d["mtxd"]
        d["anlga"] = np.asfortranarray(rng.standard_normal((m, nanl)) + 1j * rng.standard_normal((m, nanl)))
        d["xnlkb"], d["nanl"], d["mxdanl"], d["mxddim"] = np.ones(nanl), nanl, nanl, m
    return d, hk.Plan.from_inputs(d)
"""


@functools.lru_cache(maxsize=None)
def _library():
    out = os.path.join(tempfile.mkdtemp(prefix="fake_hip"), "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I/opt/rocm/include", "-o", out,
                    os.path.join(ROOT, "tests", "fake_hip.cpp")], check=True)
    return out


def run(body):
    code = _PRELUDE.format(root=ROOT, fake=_library()) + body
    env = {k: v for k, v in os.environ.items() if k != "CPWGPU_TUNE_CACHE"}
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT, timeout=300, env=env)
    assert p.returncode == 0, p.stdout + p.stderr
    return p.stdout
