"""The marcher's section list (csrc/sections.h, built for the host by
tests/cpp/build.py) against the restatement of the reference's insertion
(oracle_march.hpp): after every insertion of a random sequence both lists and
both ends are equal, bit for bit.  Sequences over a few grid positions make
sections touch, start and end together and cover each other exactly; a few
step sizes make equal steps meet; empty sections, infinities and NaN come as a
degenerate Gaussian leaves them."""
import ctypes
import os

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "cpp", "_build", "libsection_check.so")


def _lib():
    if not os.path.exists(LIB):
        import subprocess
        import sys
        subprocess.run([sys.executable, os.path.join(HERE, "cpp", "build.py")], check=True, stdout=subprocess.DEVNULL)
    L = ctypes.CDLL(LIB)
    P = ctypes.c_void_p
    L.section_compare_f32.argtypes = [ctypes.c_int, P, ctypes.c_float, P, P]
    L.section_compare_f64.argtypes = [ctypes.c_int, P, ctypes.c_double, P, P]
    return L


def _sequence(rng, kind, n):
    lo, width = rng.uniform(-1.0, 6.0, n), rng.exponential(0.6, n) + 1e-3
    dt = rng.uniform(0.01, 1.0, n)
    if kind in ("grid", "grid_equal_steps"):
        lo, width = rng.integers(-2, 40, n).astype(float), rng.integers(1, 6, n).astype(float)
        dt = rng.permutation(n) + 1.0 if kind == "grid" else rng.integers(1, 4, n).astype(float)
    if kind == "ascending":  # as the depth-ordered Gaussians of a tile come
        lo = np.sort(lo)
        dt = width * 6 / 31
    sec = np.stack([lo, lo + width, dt], axis=1)
    if kind == "degenerate":
        pick = rng.random(n)
        sec[pick < 0.1, 1] = sec[pick < 0.1, 0]
        sec[(pick > 0.1) & (pick < 0.15), 1] = np.inf
        sec[(pick > 0.15) & (pick < 0.2), 0] = -np.inf
        sec[(pick > 0.2) & (pick < 0.23), 2] = np.nan
        sec[(pick > 0.23) & (pick < 0.26), 1] = np.nan
    return sec


@pytest.mark.parametrize("kind", ["spread", "ascending", "grid", "grid_equal_steps", "degenerate"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_list_equals_the_reference_insertion(kind, dtype):
    lib = _lib()
    compare = lib.section_compare_f32 if dtype is np.float32 else lib.section_compare_f64
    rng = np.random.default_rng(5)
    filled = 0
    for trial in range(4000):
        n = int(rng.integers(1, 60))
        sec = np.ascontiguousarray(_sequence(rng, kind, n).astype(dtype))
        start = float(rng.choice([0.0, 1.0, 2.5]))
        size, out = ctypes.c_int(0), np.zeros(3 * 17, dtype)
        at = compare(n, sec.ctypes.data, start, ctypes.byref(size), out.ctypes.data)
        assert at == n, (trial, at, sec[:at + 1], out[:3 * size.value].reshape(-1, 3))
        filled += size.value == 16
    assert kind == "grid_equal_steps" or filled > 100
