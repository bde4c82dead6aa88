"""Runs a piece of Python against libspns.so on the host-only runtime of
tests/host_hip.cpp, in a process of its own (no GPU, no torch)."""
import os
import subprocess
import sys

TESTS = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(TESTS)
LIB = os.path.join(ROOT, "spns_amd", "libspns.so")

PRELUDE = """
import ctypes, re, sys
sys.path.insert(0, %r)
hip = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
hip.host_hip_log.restype = ctypes.c_char_p
hip.host_hip_fail_alloc.argtypes = [ctypes.c_long]
import numpy as np
import spns_amd

def log():
    s = hip.host_hip_log().decode()
    hip.host_hip_clear()
    return s.splitlines()

def kernels(lines):
    # names of the kernels launched, without their template arguments
    out = []
    for l in lines:
        if l.startswith("kernel "):
            n, rest = re.match(r"_ZN(?:4spnsL?)?(?:12_GLOBAL__N_1)?(\\d+)(\\w+)", l.split()[1]).groups()
            out.append(rest[:int(n)])
    return out
"""


def build(tmp):
    so = os.path.join(str(tmp), "host_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(TESTS, "host_hip.cpp"), "-o", so], check=True)
    return so


def run(tmp, code, timeout=120, **env):
    r = subprocess.run([sys.executable, "-c", PRELUDE % (ROOT, build(tmp)) + code], capture_output=True, text=True,
                       timeout=timeout, env=dict(os.environ, **env))
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    return r.stdout
