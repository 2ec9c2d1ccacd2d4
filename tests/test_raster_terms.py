"""The rasteriser's scalar terms (csrc/raster_terms.h, built for the host by
tests/cpp/build.py) against double: they are weights of the image or decide
which slots merge, so they hold the rounding of the plain float expressions."""
import ctypes
import os

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "cpp", "_build", "libraster_check.so")


def _lib():
    if not os.path.exists(LIB):
        import subprocess
        import sys
        subprocess.run([sys.executable, os.path.join(HERE, "cpp", "build.py")], check=True, stdout=subprocess.DEVNULL)
    return ctypes.CDLL(LIB)


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def test_slot_transmittance_holds_float_rounding():
    """exp(-m) over the masses of a frame and up to where it leaves float's
    normal range: within one rounding and a half of the exact value, whatever
    the exponent (a product with log2 e rounded to float is off by m 2^-24)."""
    m = np.concatenate([np.random.default_rng(1).lognormal(-1.0, 1.5, 100_000), np.linspace(0.0, 86.0, 20_001)]).astype(np.float32)
    out = np.empty_like(m)
    _lib().transmittance_batch(m.size, _ptr(m), _ptr(out))
    keep = m <= 86.0
    err = np.abs(out.astype(np.float64) / np.exp(-m.astype(np.float64)) - 1.0)[keep]
    assert err.max() <= 1.5 * 2.0 ** -24 + 2.0 ** -26, err.max()
