"""Rules by which a call takes one kernel or another, checked on the host over all sizes (tests/cpp/host_rules.cpp, built with the
inspector's sources): what a GPU run could only show where two workgroups happen to meet."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "tile-fusion_amd", "csrc")


@pytest.fixture(scope="module")
def host_rules(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    exe = str(tmp_path_factory.mktemp("rules") / "host_rules")
    cmd = ["g++", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-o", exe,
           os.path.join(ROOT, "tests", "cpp", "host_rules.cpp"), os.path.join(CSRC, "tf_inspector.cpp"), os.path.join(CSRC, "tf_march.cpp")]
    b = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert b.returncode == 0, b.stderr[-2000:]
    return exe


@pytest.mark.parametrize("check", ["column_owners", "sweep_columns", "one_launch_fits", "partial_sums", "hubs_and_columns", "streamed_entries"])
def test_rule(host_rules, check):
    r = subprocess.run([host_rules, check], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:]
