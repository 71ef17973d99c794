"""Runs a snippet in a fresh interpreter whose library is bound to the HIP
stand-in of fakehip.c: the host side of the library, on the CPU."""
import os
import subprocess
import sys
import textwrap

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))

PROLOGUE = """
import ctypes, os, sys
import numpy as np
fake = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)   # before the library, whose HIP symbols it provides
fake.fake_log.restype = ctypes.c_char_p
def log():
    lines = fake.fake_log().decode().split("\\n")[:-1]
    fake.fake_log_clear()
    return lines
def knob(name, kind=ctypes.c_size_t):
    return kind.in_dll(fake, name)
from lb3d_amd.gpu import *
from lb3d_amd.gpu import lib
"""


def compile_fake(folder):
    so = os.path.join(str(folder), "libfakehip.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", so, os.path.join(HERE, "fakehip.c")], check=True)
    return so


def run(so, body):
    """The snippet's output; a failed assertion or an error in it fails the caller."""
    r = subprocess.run([sys.executable, "-c", PROLOGUE.format(so=so) + textwrap.dedent(body)], cwd=ROOT,
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr[-3000:]
    return r.stdout
