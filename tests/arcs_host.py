"""The reverse mode's boundary arcs built for the host (arcs_host.cpp)."""
import ctypes
import os
import subprocess

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
_dp = ctypes.POINTER(ctypes.c_double)


def load(tmp):
    """Compile arcs_host.cpp into the folder `tmp` and load it."""
    so = os.path.join(str(tmp), "arcs_host.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", so, os.path.join(_HERE, "arcs_host.cpp")], check=True)
    lib = ctypes.CDLL(so)
    lib.forward_area.restype = ctypes.c_double
    for f in (lib.arcs_grad, lib.forward_area):
        f.argtypes = [_dp, ctypes.c_int, _dp, ctypes.c_int] + ([_dp, _dp] if f is lib.arcs_grad else [])
    return lib


def _p(a):
    return a.ctypes.data_as(_dp)


def grad(lib, subj, clip):
    """(d/d subject, d/d clip) of the pair's area, or None where the arcs decline it."""
    s, c = np.ascontiguousarray(subj), np.ascontiguousarray(clip)
    gc, gs = np.zeros_like(c), np.zeros_like(s)
    return (gs, gc) if lib.arcs_grad(_p(c), len(c), _p(s), len(s), _p(gc), _p(gs)) else None


def area(lib, subj, clip):
    s, c = np.ascontiguousarray(subj), np.ascontiguousarray(clip)
    return lib.forward_area(_p(c), len(c), _p(s), len(s))
