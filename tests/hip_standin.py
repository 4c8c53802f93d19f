"""Runs host code of the library on the CPU, in a child process that preloads a
stand-in for the HIP runtime (hip_standin.cpp)."""
import os
import subprocess
import sys
import textwrap
from pathlib import Path

HERE = Path(__file__).resolve().parent

PRELUDE = """
import ctypes as C
import sys
sys.path[:0] = [{root!r}, {here!r}]
from abm_amd import _lib as L
lib = L.load()
sim = C.CDLL({so!r})
sim.standin_log.restype = C.c_char_p
sim.standin_bytes.restype = C.c_size_t

def log():
    "The calls since the last log(), one string each."
    out = sim.standin_log().decode().split("\\n")[:-1]
    sim.standin_clear()
    return out

def fail(call, which=1):
    sim.standin_fail(call.encode(), which)

def held():
    s = C.c_uint64()
    return sim.standin_bytes(C.byref(s)), s.value

def replica(n, rays=64, **kw):
    kw = dict(dict(tau=10, fov0=-3.2, fov1=3.2, width=500.0, height=500.0, window_pad=30.0, vision_range=2000.0), **kw)
    return L.ForageReplica(n_agents=n, n_rays=rays, **kw)

def forage_batch(*reps):
    h = C.c_void_p()
    L.check(lib.abm_forage_batch_create((L.ForageReplica * len(reps))(*reps), len(reps), C.byref(h)))
    return h

def forage_state():
    one = C.c_void_p(4096)   # never read: kernels do nothing
    return L.ForageState(*[one] * len(L.ForageState._fields_))

def forage_step(h, stream=None, st=forage_state()):
    one = C.c_void_p(4096)
    return lib.abm_forage_step_f64(h, C.byref(st), one, one, one, one, None, C.c_void_p(stream))

def kernels(lines):
    return [ln.split()[1] for ln in lines if ln.startswith("launch ")]
"""


def build(folder) -> Path:
    so = Path(folder) / "hip_standin.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(HERE / "hip_standin.cpp"), "-o", str(so)], check=True)
    return so


def run(so, code):
    """Runs the code after PRELUDE; its assertions fail the caller."""
    prelude = PRELUDE.format(root=str(HERE.parent), here=str(HERE), so=str(so))
    p = subprocess.run([sys.executable, "-c", prelude + textwrap.dedent(code)], capture_output=True, text=True,
                       env=dict(os.environ, LD_PRELOAD=str(so)), timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr
