"""Runs test functions in a process of their own whose HIP runtime is the
stand-in of tests/native/fake_hip.cpp, so that the library's host code (memory,
waits, the choice of kernels) is tested without a GPU.

    hostrun.call(f, *args)   f(*args) in that process; f is a module's function
"""
import ctypes
import multiprocessing
import os
import sys
import traceback

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
FAKE = os.path.join(HERE, "native", os.environ.get("THRML_NATIVE_BUILD", "build"), "libfakehip.so")

fake = None
_pool = None


def _start():
    global fake
    sys.modules["torch"] = None  # the library binds to the stand-in, not to torch's runtime
    fake = ctypes.CDLL(FAKE, mode=ctypes.RTLD_GLOBAL)
    for name in ("fake_live_bytes", "fake_mallocs", "fake_pending_host", "fake_launches"):
        getattr(fake, name).restype = ctypes.c_uint64
    for name in ("fake_set_capacity", "fake_fail_malloc"):
        getattr(fake, name).argtypes = [ctypes.c_uint64]
    fake.fake_launches.argtypes = [ctypes.c_char_p, ctypes.c_uint64]


def _run(f, args):
    fake.fake_reset()
    try:
        return True, f(*args)
    except BaseException:
        return False, traceback.format_exc()


def call(f, *args):
    global _pool
    if not os.path.exists(FAKE):
        pytest.fail(f"{FAKE} is not built (run __graft_entry__.build())")
    if _pool is None:
        _pool = multiprocessing.get_context("spawn").Pool(1, _start)
    ok, r = _pool.apply_async(_run, (f, args)).get(timeout=120)
    if not ok:
        pytest.fail(r)
    return r


# ---- in the test process
def launches():
    """{kernel: launches} since clear_launches()."""
    n = fake.fake_launches(None, 0)
    buf = ctypes.create_string_buffer(n)
    fake.fake_launches(buf, n)
    return {k: int(v) for k, v in (line.rsplit(" ", 1) for line in buf.value.decode().splitlines())}


def clear_launches():
    fake.fake_clear_launches()
