"""Short forms of the tracker (convex cells, axis planes) against the general
ones on the CPU, exactly."""

import json
import os
import shutil
import subprocess

import pytest

import celeritas_amd as amd
from celeritas_amd import workloads as wl
from tests import problems

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "celeritas_amd", "csrc")
NATIVE = os.path.join(ROOT, "tests", "native")
FLAGS = ["-std=c++17", "-O2", "-pthread", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
         "-I/opt/rocm/include", f"-I{CSRC}", f"-I{os.path.join(ROOT, 'include')}"]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    out = tmp_path_factory.mktemp("georules") / "geo_rules"
    srcs = []
    for dirpath, _, files in os.walk(CSRC):
        if os.path.basename(dirpath) != "capi":
            srcs += [os.path.join(dirpath, f) for f in files if f.endswith(".cc")]
    subprocess.run(["g++", *FLAGS, os.path.join(NATIVE, "geo_rules.cc"),
                    os.path.join(NATIVE, "hip_host_stubs.cc"), *sorted(srcs),
                    "-Wl,--unresolved-symbols=ignore-all", "-o", str(out)],
                   check=True, capture_output=True, timeout=900)
    return out


@pytest.mark.parametrize("name", ["simple-cms", "testem3", "barrel"])
def test_short_forms(exe, tmp_path, name):
    if name == "simple-cms":
        prob = problems.geometry_only("simple-cms.org.json")
    elif name == "testem3":
        prob = wl.testem3_problem(physics=amd.generate_physics(wl.testem3_physics_spec()))
    else:
        prob = wl.cylinder_problem(physics=amd.generate_physics(wl.cylinder_physics_spec()))
    (tmp_path / "p.json").write_text(json.dumps(prob))
    out = subprocess.run([str(exe), str(tmp_path / "p.json"), "200"], check=True,
                         capture_output=True, text=True, timeout=300).stdout
    conjunctions, compared, differ = (int(w) for w in out.split())
    assert conjunctions > 0 and compared > 1000
    assert differ == 0
