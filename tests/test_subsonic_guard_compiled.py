"""The sampler's certainty test as compiled from hfv_physics.hpp (for the host) makes the decisions of the restatement
that test_subsonic_guard.py checks against the computed roots and powers."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from hydro_rs_amd import build
from tests.test_subsonic_guard import surely_below

SOURCE = """
#include "hfv_physics.hpp"
#define LOOP(T, NAME) extern "C" void NAME(long n, const T* v, const T* a, const T* num, const T* den, uint8_t* out) { \\
  for (long i = 0; i < n; ++i) out[i] = hfv::surely_below(v[i], a[i], num[i], den[i]); }
LOOP(double, below_f64)
LOOP(float, below_f32)
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("guard")
    (d / "guard.hip").write_text(SOURCE)
    subprocess.check_call([build.HIPCC, "-O2", "-std=c++17", "--cuda-host-only", "-fPIC", "-shared", "-ffp-contract=off",
                           "-Wno-unused-function", "-I", build.CSRC, "-o", str(d / "guard.so"), str(d / "guard.hip")])
    return C.CDLL(str(d / "guard.so"))


@pytest.mark.parametrize("dtype, fn", [(np.float64, "below_f64"), (np.float32, "below_f32")])
def test_compiled_equals_restated(lib, dtype, fn):
    rng = np.random.default_rng(5)
    n = 400_000
    span = 200.0 if dtype == np.float64 else 45.0
    edges = np.array([0.0, -0.0, 1.0, -1.0, 1e-30, 1e30, np.inf, -np.inf, np.nan, np.finfo(dtype).max, np.finfo(dtype).tiny])

    def draw():
        x = np.exp(rng.uniform(-span, span, n)) * rng.choice([-1.0, 1.0], n)
        pick = rng.random(n) < 0.1
        return np.ascontiguousarray(np.where(pick, rng.choice(edges, n), x), dtype=dtype)

    v, a, num, den = (draw() for _ in range(4))
    k = n // 2  # half of them next to the decision
    with np.errstate(all="ignore"):
        v[:k] = (np.abs(a[:k]) * num[:k] / den[:k] * 0.9999 * (1.0 + rng.uniform(-1e-6, 1e-6, k))).astype(dtype)
        want = surely_below(v, a, num, den)
    got = np.zeros(n, np.uint8)
    getattr(lib, fn)(C.c_long(n), *[x.ctypes.data_as(C.c_void_p) for x in (v, a, num, den, got)])
    assert 0.05 < want.mean() < 0.95
    assert np.array_equal(got.astype(bool), want)
