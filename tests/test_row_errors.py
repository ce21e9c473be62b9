"""A single-row call (cbx_sample_row_ex) whose launch or copy fails: its
kernels may be running already, on the handle's pinned buffers that the next
call writes, so it waits for them before it returns.  The library runs over a
stand-in HIP runtime (tests/native/fake_hip.cpp), without a GPU."""
import os
import subprocess
import sys

import pytest

import pkg

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = pkg.load().LIB_PATH

CHILD = r"""
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
fake.fake_events.restype = ctypes.c_char_p
lib.cbx_sample_row_ex.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_int32, ctypes.c_void_p,
    ctypes.c_int32, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int32, ctypes.c_int32,
    ctypes.c_double] + [ctypes.c_void_p] * 3
V = 6563
class P(ctypes.Structure):
    _fields_ = [("top_k", ctypes.c_int32), ("top_p", ctypes.c_float), ("temp", ctypes.c_float),
                ("repeat_penalty", ctypes.c_float), ("min_p", ctypes.c_float),
                ("cfg_weight", ctypes.c_float), ("pad", ctypes.c_int32 * 8)]
s = ctypes.c_void_p()
assert lib.cbx_sampler_create(ctypes.byref(s), 0, V, 16) == 0
assert lib.cbx_sampler_set_latency_rows(s, ctypes.c_int64(0)) == 0  # a redo launch follows the first
x, probs, tok = (ctypes.c_float * V)(), (ctypes.c_float * V)(), ctypes.c_int32()
p = P(50, 0.95, 0.8, 1.2, 0.0, 0.0)
for launch, copy, want_probs in ((0, 0, 0), (0, 0, 1), (1, 0, 0), (2, 0, 0), (2, 0, 1), (0, 1, 1)):
    fake.fake_fail(launch, copy)
    rc = lib.cbx_sample_row_ex(s, x, None, V, None, 0, ctypes.byref(p), None, 0, 0, 0.5,
                               ctypes.byref(tok), None, probs if want_probs else None)
    print(launch, copy, want_probs, rc, fake.fake_events().decode())
"""


@pytest.fixture(scope="module")
def lines(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-w", f"-I{rocm}/include",
                    "-o", out, os.path.join(HERE, "native", "fake_hip.cpp")], check=True)
    r = subprocess.run([sys.executable, "-c", CHILD, out, LIB], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr
    return [x.split() for x in r.stdout.splitlines()]


def test_a_failed_call_waits_for_its_kernels(lines):
    assert len(lines) == 6
    for launch, copy, want_probs, rc, events in lines:
        failed = launch != "0" or copy != "0"
        assert (rc != "0") == failed
        assert events.endswith("S") and events.count("S") == 1, (launch, copy, events)
        assert events.count("L") == (1 if launch == "1" else 2)
        assert events.count("C") == (1 if want_probs == "1" and launch == "0" else 0)
