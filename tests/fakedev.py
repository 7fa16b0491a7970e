"""Runs a function of a test module in a child process on the stand-in runtime of
fakehip.cpp: no GPU, no kernels, every HIP call and launch under the test's control."""
import ctypes as C
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def run_child(tmp_path, module, func):
    so = str(tmp_path / "fakehip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-o", so, os.path.join(HERE, "fakehip.cpp")],
                   check=True)
    code = "import sys; sys.path[:0] = [%r, %r]; import fakedev; fakedev.load(%r); import %s as m; m.%s()" % (
        ROOT, HERE, so, module, func)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300, cwd=ROOT)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]


fake = None


def load(so):
    global fake
    fake = C.CDLL(so, mode=C.RTLD_GLOBAL)
    fake.fake_journal.restype = C.c_char_p
    fake.fake_device_alloc.restype = C.c_void_p
    fake.fake_pinned_alloc.restype = C.c_void_p
    fake.fake_is_device.argtypes = [C.c_void_p]
    fake.fake_fail_after.argtypes = [C.c_long]


def launches(prefix=""):
    """(kernel, grid, first argument, second argument) of the launches since clear()"""
    out = []
    for ln in fake.fake_journal().decode().splitlines():
        name, a, b, c = ln.split("\t")
        if name.startswith(prefix):
            out.append((name, int(a), int(b), int(c)))
    return out


def clear():
    fake.fake_clear()
