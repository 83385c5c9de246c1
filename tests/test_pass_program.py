"""Pass programs on the CPU: how they are laid out for the device, how they
go there in parts, and what planning them takes (the programs tests/pass_*_check.cpp)."""
import os
import shutil
import subprocess

import pytest

from conftest import REPO

CSRC = REPO / "rqs-svg_amd" / "csrc"
LIB = REPO / "rqs-svg_amd" / "lib" / "libqcs.so"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def check(source, folder, *args):
    """Builds tests/<source> against the library and runs it; it prints ok at the end."""
    if not LIB.exists():
        pytest.skip("libqcs.so not built")
    if not shutil.which(HIPCC) and not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    exe = folder / "check"
    subprocess.run([HIPCC, "-O1", "-std=c++17", f"-I{REPO / 'include'}", f"-I{CSRC}", str(REPO / "tests" / source),
                    f"-L{LIB.parent}", "-lqcs", f"-Wl,-rpath,{LIB.parent}", "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    p = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0 and p.stdout.strip().endswith("ok"), p.stdout[-2000:] + p.stderr[-2000:]


def test_misaligned_programs_are_refused(tmp_path):
    check("pass_align_check.cpp", tmp_path)


@pytest.mark.parametrize("seed", [1, 2])
def test_programs_in_parts(tmp_path, seed):
    check("pass_parts_check.cpp", tmp_path, seed)


def test_planning_time_grows_with_the_circuit(tmp_path):
    check("pass_time_check.cpp", tmp_path)
