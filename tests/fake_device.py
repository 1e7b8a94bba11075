"""Runs a script in a fresh Python process in which the host code of libcloudsc_hip.so meets the HIP runtime of
tests/hip/fake_hip.cpp: no device, kernels do not run, any call can be made to fail."""
import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PRELUDE = """
import ctypes, json, sys
sys.path.insert(0, {root!r})
fake = ctypes.CDLL({lib!r}, ctypes.RTLD_GLOBAL)  # ahead of the library under test
fake.fake_log.restype = ctypes.c_char_p
fake.fake_pending.restype = ctypes.c_long
fake.fake_pending.argtypes = [ctypes.c_void_p]
import numpy as np
from openifs_amd import cloudsc as C

def arm(name="", nth=0):
    fake.fake_arm(name.encode(), nth)

def calls(name):
    return fake.fake_calls(name.encode())

def log():
    return fake.fake_log().decode().splitlines()
"""


def build(folder):
    lib = os.path.join(folder, "libfake_hip.so")
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-shared", "-fPIC", "-I/opt/rocm/include", "-o",
                    lib, os.path.join(ROOT, "tests", "hip", "fake_hip.cpp")], check=True)
    return lib


def run(lib, script):
    """The JSON value that the script prints last."""
    code = PRELUDE.format(root=ROOT, lib=lib) + script
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stderr
    return json.loads(r.stdout.splitlines()[-1])
