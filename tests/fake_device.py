"""A copy of libdgv_amd.so on a stand-in HIP runtime (fake_hip.cpp), and scripts run in a child process
on it: host-side tests of launch shapes and of what follows a call of the runtime that fails.  No kernel runs."""
import glob
import os
import subprocess
import sys

from dgv0d3v_direct_collision_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PRELUDE = """
import ctypes as C
import numpy as np
import dgv0d3v_direct_collision_amd as dgv
L = dgv.load()
L.fake_launched.restype = C.c_char_p
L.fake_widest_launch.restype = C.c_uint64
L.fake_largest_malloc.restype = C.c_int64
L.fake_live_bytes.restype = C.c_int64
L.fake_fail_malloc_above.argtypes = [C.c_int64]
def launched(): return L.fake_launched().decode()
def fail_kernel(part): L.fake_fail_kernel(part.encode())
"""


def library(outdir):
    """Links the build's objects (built first where they are missing or older than a source)."""
    sources = glob.glob(os.path.join(build.CSRC, "*"))
    objs = [os.path.join(build.HERE, "_build", os.path.basename(s) + ".o") for s in sources if not s.endswith(".h")]
    newest = max(map(os.path.getmtime, sources))
    if not all(os.path.exists(o) and os.path.getmtime(o) >= newest for o in objs):
        build.build()
    fake = os.path.join(outdir, "fake_hip.o")
    subprocess.run(["g++", "-O1", "-fPIC", "-c", os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", fake], check=True)
    lib = os.path.join(outdir, "libdgv_fake.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-o", lib, fake, *objs, "-Wl,-Bsymbolic"], check=True)
    return lib


def run(lib, script):
    env = dict(os.environ, DGV_LIB_PATH=lib)
    r = subprocess.run([sys.executable, "-c", PRELUDE + script], cwd=ROOT, env=env, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    return r.stdout
