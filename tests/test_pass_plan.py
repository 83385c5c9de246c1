"""Circuit passes on the CPU: tests/pass_check.cpp lowers and plans random circuits over the
whole gate table with the library and runs the resulting programs with an interpreter written
from the operations' definitions, against the gates' matrices applied one by one."""
import os
import shutil
import subprocess

import pytest

from conftest import REPO

CSRC = REPO / "rqs-svg_amd" / "csrc"
LIB = REPO / "rqs-svg_amd" / "lib" / "libqcs.so"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def pass_check(tmp_path_factory):
    if not LIB.exists():
        pytest.skip("libqcs.so not built")
    if not shutil.which(HIPCC) and not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    exe = tmp_path_factory.mktemp("pass") / "pass_check"
    subprocess.run([HIPCC, "-O1", "-std=c++17", f"-I{REPO / 'include'}", f"-I{CSRC}", str(REPO / "tests" / "pass_check.cpp"),
                    f"-L{LIB.parent}", "-lqcs", f"-Wl,-rpath,{LIB.parent}", "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    return exe


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_pass_programs_match_the_gates(pass_check, seed):
    p = subprocess.run([str(pass_check), "48", str(seed)], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-2000:]
    assert p.stdout.strip().endswith("ok")
