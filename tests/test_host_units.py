"""Host-side checks of what the step kernel reads, compiled from the library's host
sources with g++ under AddressSanitizer and UBSan."""
import os
import shutil
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")
SRC = os.path.join(os.path.dirname(os.path.dirname(CPP)), "bsim_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
@pytest.mark.parametrize("prog", ["unit_table_check", "sim_layout_check"])
def test_host_program(prog, tmp_path):
    exe = str(tmp_path / prog)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fopenmp", "-fsanitize=address,undefined",
                    "-fno-omit-frame-pointer", "-fno-sanitize-recover=undefined", "-ffp-contract=off", "-Wall",
                    "-o", exe, os.path.join(CPP, prog + ".cpp"), os.path.join(SRC, "network.cpp"),
                    os.path.join(SRC, "gen.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0 and f"{prog} ok" in r.stdout, r.stdout + r.stderr
