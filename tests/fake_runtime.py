"""Runs a Python script against libglasma.so with tests/fake_hip.cpp in the place of the HIP runtime: the library's host
code on a machine without a GPU, with launches refused and memory limited as the script asks."""
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
PREAMBLE = """
import ctypes, sys
fake = ctypes.CDLL({lib!r}, mode=ctypes.RTLD_GLOBAL)
for f in ("launches", "launches_of", "streams", "pins", "copies"):
    getattr(fake, "fake_" + f).restype = ctypes.c_long
for f in ("used", "pinned"):
    getattr(fake, "fake_" + f).restype = ctypes.c_size_t
fake.fake_refuse_launch.argtypes = [ctypes.c_long]
fake.fake_limit.argtypes = fake.fake_show.argtypes = fake.fake_pin_limit.argtypes = [ctypes.c_size_t]
sys.path.insert(0, {root!r})
import numpy as np
from soerenpragya3dglasma_amd import Glasma, GlasmaBatch, GlasmaError, _lib
"""


def run(script: str) -> str:
    """The script's standard output; fails with all it printed when it does not end normally."""
    with tempfile.TemporaryDirectory() as d:
        so = os.path.join(d, "libfake_hip.so")
        subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        os.path.join(HERE, "fake_hip.cpp"), "-o", so], check=True)
        r = subprocess.run([sys.executable, "-c", PREAMBLE.format(lib=so, root=os.path.dirname(HERE)) + script],
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    return r.stdout
