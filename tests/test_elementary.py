"""Errors of the step kernels' own FP64 logarithm, sine and cosine.

Rounding of the result is half a unit in the last place. What the terms below
it add at the ends of the reduced ranges, in the same unit:

- logarithm (result 0.35, series' term s (f^2/2 + R) = 0.018 with s = 0.17):
  s 0.036, the square and the sum in parentheses 0.021 each, their product
  0.031, the polynomial 0.016: 0.125;
- sine and cosine (result 0.7, cubic term 0.07): the cube 0.07, its product
  0.07, the small terms 0.07, the square in the fifth-order term 0.01: 0.24.

The host's functions differ from the device's in the split into mantissa and
exponent and in the reciprocal (a quotient on the host; on the device an
approximation and two Newton steps, whose error enters below the last place
of a term of a 20th of the result), so the same limits hold for both.
"""

import os
import shutil
import subprocess

import numpy as np
import pytest

import celeritas_amd as amd_pkg

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LOG, ANGLE = 0.5 + 0.125, 0.5 + 0.24
RANGES = [
    ("log", 1e-307, 1e308, LOG), ("log", 0, 1, LOG), ("log", 0.5, 2, LOG),
    ("log", 0.7071, 0.7072, LOG), ("log", 1.4142, 1.4143, LOG),
    ("log", 1 - 1e-9, 1 + 1e-9, LOG), ("log", 5e-324, 1e-300, LOG),
    ("sin", 0, 6.2831853071795864, ANGLE), ("cos", 0, 6.2831853071795864, ANGLE),
    ("sin", -10, 10, ANGLE), ("cos", -10, 10, ANGLE), ("sin", 3.14159, 3.1416, ANGLE),
    ("cos", 1.57079, 1.5708, ANGLE), ("sin", 1e-12, 1, ANGLE), ("cos", -1e6, 1e6, ANGLE),
]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    out = tmp_path_factory.mktemp("elementary") / "elementary"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", f"-I{os.path.join(ROOT, 'celeritas_amd', 'csrc')}",
                    os.path.join(ROOT, "tests", "native", "elementary.cc"), "-o", str(out)],
                   check=True, capture_output=True, timeout=300)
    return out


@pytest.mark.parametrize("fn, low, high, limit", RANGES)
def test_error(exe, fn, low, high, limit):
    r = subprocess.run([str(exe), fn, repr(float(low)), repr(float(high)), "1000000"], check=True,
                       capture_output=True, text=True, timeout=100)
    worst, at, special = r.stdout.split()
    assert float(worst) <= limit, f"{worst} at {at}"
    assert special == "1"


@pytest.mark.gpu
@pytest.mark.parametrize("fn, low, high, limit", RANGES)
def test_error_on_device(amd, fn, low, high, limit):
    u = np.random.default_rng(5).random(1_000_001)
    # A positive range over decades is sampled by its logarithm
    ratio = np.longdouble(high) / (low or 1)
    x = (low * ratio ** u).astype(float) if low > 0 and ratio > 1e3 else low + (high - low) * u
    x = x[x != 0] if fn == "log" else x
    got = dict(zip(("log", "sin", "cos"), amd_pkg.verify_elementary(x)))[fn]
    want = getattr(np, fn)(x.astype(np.longdouble))
    unit = np.ldexp(np.longdouble(1), np.frexp(want.astype(np.float64))[1] - 53)
    err = np.abs((got - want) / unit)[want != 0].astype(np.float64)
    print(fn, low, high, "largest error", err.max(), "mean", err.mean())
    assert err.max() <= limit, x[want != 0][err.argmax()]


@pytest.mark.gpu
def test_special_values_on_device(amd):
    log, _, _ = amd_pkg.verify_elementary([0.0, -0.0, np.inf, -1.0, -np.inf, np.nan, 1.0])
    np.testing.assert_array_equal(log, [-np.inf, -np.inf, np.inf, np.nan, np.nan, np.nan, 0.0])
    _, sine, cosine = amd_pkg.verify_elementary([0.0, np.nan])
    np.testing.assert_array_equal(sine, [0.0, np.nan])
    np.testing.assert_array_equal(cosine, [1.0, np.nan])
