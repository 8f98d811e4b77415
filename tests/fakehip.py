"""Run a piece of Python against the library's host code with the HIP runtime
of fake_hip.cpp in place of the real one: a child process, since the library
of this process has the real one.  Returns the log's lines, split."""
import atexit
import functools
import os
import shutil
import subprocess
import sys
import tempfile

from conftest import ROOT

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import sys
sys.path[:0] = [{tests!r}, {root!r}]
import numpy as np
from conftest import load_package
pkg = load_package()
import flowcase as fc
"""


@functools.lru_cache(None)
def runtime():
    d = tempfile.mkdtemp()
    atexit.register(shutil.rmtree, d)
    so = os.path.join(d, "libfakehip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", os.path.join(HERE, "fake_hip.cpp"), "-o", so],
                   check=True)
    return so


def run(code, elapsed=""):
    so = runtime()
    with tempfile.TemporaryDirectory() as d:
        log = os.path.join(d, "log")
        pre = [so] + [p for p in os.environ.get("LD_PRELOAD", "").split(":") if p]
        env = dict(os.environ, LD_PRELOAD=":".join(pre), FAKE_HIP_LOG=log, FAKE_HIP_ELAPSED=elapsed)
        r = subprocess.run([sys.executable, "-c", PRELUDE.format(tests=HERE, root=ROOT) + code], env=env,
                           capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr[-4000:]
        return [ln.split() for ln in open(log)]
