"""The resident CG's partition (build_cg_plan) on the CPU, plainly and under AddressSanitizer and
UndefinedBehaviorSanitizer: tests/cpp/cg_plan_check.cpp.  Bars of cubes, and of cells up to 20 times as
long as wide, whose workgroups have about twice as many ghosts as those of cubes."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "phybs_amd", "csrc")
SAN = ["-fsanitize=address,undefined", "-fno-sanitize-recover=undefined", "-fno-omit-frame-pointer"]


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
@pytest.mark.parametrize("sanitize", [False, True])
def test_cg_plan(tmp_path, sanitize):
    exe = str(tmp_path / "cg_plan_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-I" + CSRC, os.path.join(HERE, "cpp", "cg_plan_check.cpp"),
                    os.path.join(CSRC, "pbs_cg_plan.cpp"), os.path.join(CSRC, "pbs_tiles.cpp"), "-o", exe]
                   + (SAN if sanitize else []), check=True, capture_output=True)
    r = subprocess.run([exe] + (["quick"] if sanitize else []), capture_output=True, text=True, timeout=600,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    print(r.stdout[-3000:], r.stderr[-3000:])
    assert r.returncode == 0 and "cg_plan_check: all passed" in r.stdout
