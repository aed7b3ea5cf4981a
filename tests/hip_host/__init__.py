"""The library's host side without a device (host_hip.cpp): `run` executes a
piece of Python in a process of its own, in which libpicchio_hip.so's HIP
calls land in that stand-in. The piece sees `pa` (picchio_amd), `L` (the
library), `hh` (the stand-in's test side) and the helpers of PRELUDE."""
import functools
import os
import subprocess
import sys
import tempfile
import textwrap

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))

PRELUDE = """
import ctypes as C, sys
import numpy as np
hh = C.CDLL({shim!r}, mode=C.RTLD_GLOBAL)
sys.path.insert(0, {root!r})
import picchio_amd as pa
L = pa.lib()
hh.hh_name.restype = C.c_char_p
hh.hh_in_use.restype = hh.hh_peak.restype = hh.hh_groups.restype = C.c_int64
hh.hh_budget.argtypes = [C.c_int64]
vp = C.c_void_p

def small(**kw):
    d = dict(hidden=128, n_layers=2, n_heads=4, n_kv_heads=2, head_dim=64, n_experts=8, topk=4, moe_inter=256,
             vocab=20000, ctx_len=1024)
    d.update(kw)
    return pa.gptoss_cfg(**d)

def engine(cfg, synthetic=True):
    h = vp()
    pa.check(L.pk_engine_create(C.byref(cfg), 0, C.byref(h)))
    if synthetic:
        pa.check(L.pk_engine_build_synthetic(h, 7, 7, 1))
    return h

def dev(n, dtype=np.float32):
    p = vp()
    assert hh.hipMalloc(C.byref(p), C.c_size_t(int(n) * np.dtype(dtype).itemsize)) == 0
    return p

def prompt(h, n, seq=None):
    ids = (np.arange(n) % 50).astype(np.int32)
    return L.pk_prefill_tokens(h, pa.ptr(ids), n, 0, None)

def launches():
    n = [hh.hh_name(i).decode() for i in range(hh.hh_launches())]
    hh.hh_clear()
    return n
"""


@functools.lru_cache(None)
def _shim():
    out = os.path.join(tempfile.mkdtemp(prefix="host_hip_"), "libhost_hip.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__",
                           "-I/opt/rocm/include", "-I", os.path.join(ROOT, "picchio_amd", "csrc"),
                           "-I", os.path.join(ROOT, "include"), os.path.join(HERE, "host_hip.cpp"), "-o", out])
    return out


def run(code, env=None):
    src = PRELUDE.format(shim=_shim(), root=ROOT) + textwrap.dedent(code)
    r = subprocess.run([sys.executable, "-c", src], capture_output=True, text=True, timeout=300,
                       env={**os.environ, **(env or {})})
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
