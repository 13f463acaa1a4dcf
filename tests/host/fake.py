"""Runs a piece of Python against libvmx.so on a HIP runtime that computes nothing (fakehip.cpp), in a
process of its own, for tests of the library's host logic without a GPU."""
import os
import subprocess
import sys
import textwrap

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))

# what the piece of Python finds: `hip` (the runtime's test side), `log` and `launches`
PRELUDE = """
import ctypes, re, sys
import numpy as np
sys.path[:0] = [{root!r}, {tests!r}]
hip = ctypes.CDLL({lib!r}, mode=ctypes.RTLD_GLOBAL)      # before libvmx.so, whose HIP calls it takes
hip.fake_text.restype = ctypes.c_char_p
hip.fake_used.restype = hip.fake_peak.restype = ctypes.c_size_t
hip.fake_capacity.argtypes = [ctypes.c_size_t]
from vampire_amd import _lib as L, system as S
from vampire_amd.context import FP32, FP64, FUSED, PLAIN, Context
import refcases as RC


def log(call):
    '''The lines that call() leaves in the runtime's log.'''
    hip.fake_log(1)
    call()
    lines = hip.fake_text().decode().splitlines()
    hip.fake_log(0)
    return lines


class Launch:
    def __init__(self, line):
        _, name, *v = line.split()
        self.name = re.sub(r'^_ZN3vmx(?:12_GLOBAL__N_1)?\\d+', '', name)
        self.grid, self.block, self.shared = tuple(map(int, v[:3])), int(v[3]), int(v[4])
        self.watched = [int(x) for x in v[5:]]


def launches(lines, part=''):
    return [Launch(x) for x in lines if x.startswith('launch ') and part in x.split()[1]]


"""


def build(folder) -> str:
    lib = os.path.join(str(folder), "libfakehip.so")
    if not os.path.exists(lib):
        subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", lib, os.path.join(HERE, "fakehip.cpp")],
                       check=True, timeout=120)
    return lib


def run(lib: str, code: str) -> None:
    """Runs the code; an assertion that fails in it fails here, with its output."""
    head = PRELUDE.format(root=ROOT, tests=os.path.join(ROOT, "tests"), lib=lib)
    p = subprocess.run([sys.executable, "-c", head + textwrap.dedent(code)], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr
