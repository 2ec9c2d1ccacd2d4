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


def test_border_density_is_no_further_off_than_the_plain_expression():
    """exp(-d^2 / (2 var)) from the centre out to 9 standard deviations, over
    the variances of near and far Gaussians: rms and largest relative error at
    most those of expf(-d^2 / 2 / var) in float."""
    rng = np.random.default_rng(2)
    n = 200_000
    var = np.exp(rng.normal(-6.0, 2.0, n)).astype(np.float32)
    d = (rng.uniform(-9.0, 9.0, n) * np.sqrt(var)).astype(np.float32)
    out, plain = np.empty_like(d), np.empty_like(d)
    _lib().density_batch(n, _ptr(d), _ptr(var), _ptr(out), _ptr(plain))
    exact = np.exp(-0.5 * d.astype(np.float64) ** 2 / var.astype(np.float64))
    e, p = out / exact - 1.0, plain / exact - 1.0
    rms = lambda x: np.sqrt((x * x).mean())
    print(f"rms {rms(e):.3g} (plain {rms(p):.3g}), largest {np.abs(e).max():.3g} ({np.abs(p).max():.3g})")
    assert rms(e) <= rms(p)
    assert np.abs(e).max() <= np.abs(p).max()
    # at the centre 1; where the square or the exponent overflows 0, as the plain expression
    edge = np.array([[0.0, 1e-3], [1e3, 1e-3], [1e20, 1e-3], [1e5, 1e-30], [3e19, 1e30]], np.float32)
    o, q = np.empty(5, np.float32), np.empty(5, np.float32)
    _lib().density_batch(5, _ptr(np.ascontiguousarray(edge[:, 0])), _ptr(np.ascontiguousarray(edge[:, 1])), _ptr(o), _ptr(q))
    np.testing.assert_array_equal(o, [1.0, 0.0, 0.0, 0.0, 0.0])
    np.testing.assert_array_equal(o, q)
