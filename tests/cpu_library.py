"""The library built for the host: the same sources compiled as C++ against
cpu_hip/, whose runtime runs a kernel one workgroup at a time with bounds
checks and guard pages (cpu_hip/emu.cpp).  For what must not be tried on a GPU."""
import fcntl
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "eom-imsrg_full_amd", "csrc")
CPU = os.path.join(HERE, "cpu_hip")
OUT = os.path.join(ROOT, "_build", "cpu_hip")
CXX = "/opt/rocm/llvm/bin/clang++"
FLAGS = ["-std=c++17", "-O1", "-g1", "-fPIC", "-fno-strict-aliasing", "-fsanitize=bounds", "-fsanitize-trap=bounds",
         "-I" + CPU, "-Wno-everything"]


def build():
    """path of the host library, built anew where a source is younger"""
    os.makedirs(OUT, exist_ok=True)
    with open(os.path.join(OUT, "lock"), "w") as lock:  # one builder at a time
        fcntl.flock(lock, fcntl.LOCK_EX)
        return _build()


def _build():
    lib = os.path.join(OUT, "libimsrg_cpu.so")
    src = [os.path.join(CSRC, f) for f in ("kernels.hip", "ozaki.hip", "adjoint.hip", "hf.hip", "engine.hip", "layout.cpp",
                                           "interaction_io.cpp")]
    src += [os.path.join(CPU, f) for f in ("tensor_cpu.cpp", "emu.cpp")]
    deps = [os.path.join(d, f) for d, _, fs in list(os.walk(CSRC)) + list(os.walk(CPU)) for f in fs]
    deps.append(os.path.join(ROOT, "include", "imsrg_mi355x.h"))
    if os.path.exists(lib) and os.path.getmtime(lib) > max(map(os.path.getmtime, deps)):
        return lib
    objs = [os.path.join(OUT, os.path.basename(f) + ".o") for f in src]
    jobs = [subprocess.Popen([CXX, *FLAGS, "-x", "c++", "-c", f, "-o", o]) for f, o in zip(src, objs)]
    assert all(j.wait() == 0 for j in jobs)
    subprocess.run([CXX, "-shared", "-o", lib + ".tmp", *objs, "-lz", "-lpthread"], check=True)
    os.replace(lib + ".tmp", lib)
    return lib


PRELUDE = """
import ctypes
import numpy as np
from imsrg_mi355x import Basis, random_operator, synthetic_hamiltonian
from imsrg_mi355x import engine as E
"""


def run(code, **env):
    """`code` in a process of its own on the host library; its output.  A read or
    write out of bounds ends it by a signal, a barrier left behind with status 3."""
    e = dict(os.environ, IMSRG_MI355X_LIB=build(), **{k: str(v) for k, v in env.items()})
    e["PYTHONPATH"] = os.pathsep.join([os.path.join(ROOT, "eom-imsrg_full_amd"), ROOT, HERE])
    r = subprocess.run([sys.executable, "-c", PRELUDE + code], env=e, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, f"status {r.returncode}\n{r.stdout}\n{r.stderr[-2000:]}"
    return r.stdout
