"""Rules by which a call takes one kernel or another, checked on the host over all sizes (tests/cpp/host_rules.cpp, built with the
inspector's sources): what a GPU run could only show where two workgroups happen to meet."""
import glob
import os
import re
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


@pytest.mark.parametrize("check", ["column_owners", "sweep_columns", "one_launch_fits", "partial_sums", "hubs_and_columns", "streamed_entries", "even_reads", "rows_with_neighbours"])
def test_rule(host_rules, check):
    r = subprocess.run([host_rules, check], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:]


def test_memory_instructions_written_out_wait():
    """The compiler counts no wait states inside inline assembly.  A store of more than eight bytes: one before its data registers are written again.  A load
    from an address in scalar registers: five after a vector instruction may have written them; one after m0, which is named as overwritten."""
    seen = 0
    for path in glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h")):
        for at in re.finditer(r'asm(?: volatile)?\(((?:"[^"]*"\s*)+)([^;]*)\);', open(path).read()):
            text = "".join(re.findall(r'"([^"]*)"', at.group(1)))
            lines = [t.strip() for t in re.split(r"\\n\\t|\\n", text) if t.strip()]
            for k, line in enumerate(lines):
                if re.match(r"(global|flat|buffer)_store_dwordx[34]", line):
                    seen += 1
                    assert re.match(r"s_nop \d", lines[k + 1] if k + 1 < len(lines) else ""), (path, text)
                if re.match(r"(global|buffer)_load", line):
                    seen += 1
                    states = sum(1 + int(t.split()[1]) if t.startswith("s_nop") else 1 for t in lines[:k])
                    assert states >= 5 and lines[k - 1].startswith("s_nop"), (path, text)
                if re.match(r"s_mov_b32 m0,", line):
                    assert '"m0"' in at.group(2).rsplit(":", 1)[-1], (path, text)
    assert seen >= 4
