"""Which tables the step kernels stage in LDS, for TestEm3 with more layers
and finer physics grids than the usual ones (host rules, on the CPU)."""

import json
import os
import shutil
import subprocess

import pytest

import celeritas_amd as amd
from celeritas_amd import workloads as wl

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "celeritas_amd", "csrc")
NATIVE = os.path.join(ROOT, "tests", "native")
FLAGS = ["-std=c++17", "-O1", "-pthread", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
         "-I/opt/rocm/include", f"-I{CSRC}", f"-I{os.path.join(ROOT, 'include')}"]
LDS = 160 * 1024


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    out = tmp_path_factory.mktemp("staging") / "staging"
    srcs = []
    for dirpath, _, files in os.walk(CSRC):
        if os.path.basename(dirpath) != "capi":
            srcs += [os.path.join(dirpath, f) for f in files if f.endswith(".cc")]
    subprocess.run(["g++", *FLAGS, os.path.join(NATIVE, "staging.cc"),
                    os.path.join(NATIVE, "hip_host_stubs.cc"), *sorted(srcs),
                    "-Wl,--unresolved-symbols=ignore-all", "-o", str(out)],
                   check=True, capture_output=True, timeout=900)
    return out


# Physics, distances, all geometry, both: the first seven are the sizes at
# which each kernel staged its tables when these held no grid energies and no
# copies of surfaces
@pytest.mark.parametrize("layers, bins, want", [
    (50, 7, (True, True, True, True)),
    (54, 7, (True, True, True, True)),
    (60, 7, (True, True, True, True)),
    (66, 7, (True, True, True, True)),
    (70, 7, (True, True, True, True)),
    (50, 8, (True, True, True, True)),
    (86, 7, (True, True, True, False)),
    (50, 12, (True, True, True, False)),
    (50, 14, (False, True, True, False)),
])
def test_staged_tables(exe, tmp_path, monkeypatch, layers, bins, want):
    monkeypatch.setattr(wl, "TESTEM3_LAYERS", layers)
    monkeypatch.setattr(wl, "TESTEM3_CALO_HALF", 0.4 * layers)
    monkeypatch.setattr(wl, "TESTEM3_WORLD_HALF", 0.4 * layers + 4)
    spec = wl.testem3_physics_spec()
    spec["options"]["bins_per_decade"] = bins
    problem = wl.testem3_problem(physics=amd.generate_physics(spec), init_capacity=1024,
                                 max_events=16)
    (tmp_path / "p.json").write_text(json.dumps(problem))
    out = subprocess.run([str(exe), str(tmp_path / "p.json")], check=True, capture_output=True,
                         text=True, timeout=300).stdout
    physics, distances, geometry, *staged = (int(w) for w in out.split())
    print(out)
    # A region is staged whole or not at all
    for n, region in zip(staged, (physics, distances, geometry, physics + distances)):
        assert n in (0, region)
    assert tuple(n > 0 for n in staged) == want
    # The workgroups that fit a CU beside each other
    assert 3 * max(staged[0], staged[1], staged[3]) <= LDS and 4 * staged[2] <= LDS
