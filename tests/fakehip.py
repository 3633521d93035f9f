"""Runs a piece of Python against the library with the HIP runtime of
fake_hip.cpp in place of the real one, in a process of its own."""
from __future__ import annotations

import os
import subprocess
import sys
import textwrap

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PREAMBLE = """
import ctypes, os, sys, time
fake = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_launches.restype = ctypes.c_char_p
fake.fake_direct_copies.restype = fake.fake_syncs.restype = ctypes.c_long
sys.path.insert(0, {pkg!r})
import numpy as np
import hydrogen as hg
def launched():
    names = fake.fake_launches().decode().split()
    fake.fake_clear()
    return names
"""


def build(folder) -> str:
    so = os.path.join(str(folder), "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-pthread", "-o", so,
                    os.path.join(HERE, "fake_hip.cpp")], check=True)
    return so


def run(so: str, code: str) -> str:
    """What `code` prints; it fails the caller if it raises."""
    text = PREAMBLE.format(so=so, pkg=os.path.join(ROOT, "hydro-gen_amd")) + textwrap.dedent(code)
    p = subprocess.run([sys.executable, "-c", text], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stderr[-3000:]
    return p.stdout
