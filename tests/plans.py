"""The work-sharing rules of csrc/plans.h, compiled with the host compiler: which
kernel form a shape takes on a card of `cus` compute units."""
import ctypes
import os
import subprocess
import tempfile
from collections import namedtuple

_CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                     "vestra-engine_amd", "csrc")
_SHIM = """
#include "plans.h"
extern "C" void linear_form(long long cus, int m, int k, int n, long long* out) {
  const int provided = vk::linear_slices_to_provide(cus, m, n, k);
  const vk::LinearPlan p = vk::linear_plan(cus, m, n, k, provided);
  out[0] = p.tm; out[1] = p.tn; out[2] = p.splits; out[3] = provided; out[4] = p.tiles;
}
extern "C" void attention_form(int cus, unsigned long long s, unsigned long long n, int* out) {
  const int provided = vk::attention_splits_to_provide(cus, s, n);
  const vk::AttentionPlan p = vk::attention_plan(cus, s, n, provided);
  out[0] = p.waves; out[1] = p.splits; out[2] = provided;
}
extern "C" long long max_partial_floats() { return vk::kMaxPartialFloats; }
"""
LinearForm = namedtuple("LinearForm", "tm tn splits provided tiles")
AttentionForm = namedtuple("AttentionForm", "waves splits provided")


def _load():
    with tempfile.TemporaryDirectory() as d:
        src, lib = os.path.join(d, "plans.cpp"), os.path.join(d, "libplans.so")
        with open(src, "w") as f:
            f.write(_SHIM)
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC",
                        "-I", _CSRC, src, "-o", lib], check=True)
        return ctypes.CDLL(lib)


_lib = _load()
_lib.linear_form.argtypes = [ctypes.c_longlong] + [ctypes.c_int] * 3 + [ctypes.c_void_p]
_lib.attention_form.argtypes = [ctypes.c_int, ctypes.c_ulonglong, ctypes.c_ulonglong,
                                ctypes.c_void_p]
_lib.max_partial_floats.restype = ctypes.c_longlong
MAX_PARTIAL_FLOATS = _lib.max_partial_floats()


def linear_form(m, k, n, cus=256):
    out = (ctypes.c_longlong * 5)()
    _lib.linear_form(cus, m, k, n, out)
    return LinearForm(*out)


def attention_form(sequences, n, cus=256):
    out = (ctypes.c_int * 3)()
    _lib.attention_form(cus, sequences, n, out)
    return AttentionForm(*out)
