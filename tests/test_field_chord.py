"""The start of the field driver's chord search on the CPU (no GPU).

field::first_chord_trial passes over the trials whose sagitta is known to
shrink them by the full factor; tests/native/chord_trials.cc runs the serial
search beside it over momenta, fields, directions (also along the field),
step lengths up to infinity and driver options, and requires the same trial
at the same count.
"""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("seed", [1, 2])
def test_first_trial_is_the_search_s(tmp_path, seed):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    exe = tmp_path / "chord_trials"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off",
                    f"-I{os.path.join(ROOT, 'celeritas_amd', 'csrc')}",
                    f"-I{os.path.join(ROOT, 'include')}",
                    os.path.join(ROOT, "tests", "native", "chord_trials.cc"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([str(exe), "100000", str(seed)], capture_output=True, text=True,
                       timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    # The rule is used: over a third of the draws start past their first trial
    assert int(r.stdout.split(" from")[0].split()[-1]) < 67_000
