"""Runs a piece of Python with libsassena_amd.so on the host-side HIP of
fake_hip.c, in a process of its own (no GPU is touched, no kernel runs)."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, sys
sys.path.insert(0, {root!r})
fake = ctypes.CDLL({lib!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_memory.argtypes = [ctypes.c_size_t]
fake.fake_used.restype = ctypes.c_size_t
fake.fake_name.restype = ctypes.c_char_p
fake.fake_arg.restype = ctypes.c_void_p
import numpy as np
import sassena_amd
from sassena_amd import ScatterDevice, SxError

def launches():
    "Names of the kernels launched since the last call."
    names = [fake.fake_name(i).decode() for i in range(fake.fake_launches())]
    fake.fake_forget()
    return names

def ran(names, kernel):
    return any(kernel in n for n in names)
"""


@pytest.fixture(scope="module")
def fake_run(tmp_path_factory):
    if not shutil.which("gcc"):
        pytest.skip("gcc not available")
    lib = str(tmp_path_factory.mktemp("fakehip") / "libfakehip.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O2", "-Wall", "-o", lib, os.path.join(HERE, "fake_hip.c")], check=True)

    def run(code):
        # freed memory is overwritten at once and stays mapped
        env = dict(os.environ, MALLOC_PERTURB_="165", MALLOC_MMAP_THRESHOLD_=str(1 << 30),
                   MALLOC_TRIM_THRESHOLD_=str(1 << 40))
        src = PRELUDE.format(root=ROOT, lib=lib) + textwrap.dedent(code)
        r = subprocess.run([sys.executable, "-c", src], env=env, capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
        return r.stdout

    return run
