"""Errors of the step kernels' own FP64 logarithm, sine and cosine.

Rounding of the result is half a unit in the last place. What the terms below
it add at the ends of the reduced ranges, in the same unit:

- logarithm (result 0.35, series' term s (f^2/2 + R) = 0.018 with s = 0.17):
  s 0.036, the square and the sum in parentheses 0.021 each, their product
  0.031, the polynomial 0.016: 0.125;
- sine and cosine (result 0.7, cubic term 0.07): the cube 0.07, its product
  0.07, the small terms 0.07, the square in the fifth-order term 0.01: 0.24.
"""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LOG, ANGLE = 0.5 + 0.125, 0.5 + 0.24


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


@pytest.mark.parametrize("fn, low, high, limit", [
    ("log", 1e-307, 1e308, LOG), ("log", 0, 1, LOG), ("log", 0.5, 2, LOG),
    ("log", 0.7071, 0.7072, LOG), ("log", 1.4142, 1.4143, LOG),
    ("log", 1 - 1e-9, 1 + 1e-9, LOG), ("log", 5e-324, 1e-300, LOG),
    ("sin", 0, 6.2831853071795864, ANGLE), ("cos", 0, 6.2831853071795864, ANGLE),
    ("sin", -10, 10, ANGLE), ("cos", -10, 10, ANGLE), ("sin", 3.14159, 3.1416, ANGLE),
    ("cos", 1.57079, 1.5708, ANGLE), ("sin", 1e-12, 1, ANGLE), ("cos", -1e6, 1e6, ANGLE),
])
def test_error(exe, fn, low, high, limit):
    r = subprocess.run([str(exe), fn, repr(float(low)), repr(float(high)), "1000000"], check=True,
                       capture_output=True, text=True, timeout=100)
    worst, at, special = r.stdout.split()
    assert float(worst) <= limit, f"{worst} at {at}"
    assert special == "1"
