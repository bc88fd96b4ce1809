"""The eight-wavefront step kernels as compiled for gfx950 use no private (scratch)
memory, as the other kernels' test has it for theirs."""
import os
import re
import subprocess

from bsim_amd import build

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bsim_amd", "csrc", "step_many.hip")


def test_kernels_use_no_scratch(tmp_path):
    out = tmp_path / "step_many.s"
    cmd = [build.hipcc(), *[f for f in build.flags() if f not in ("-fopenmp", "-fPIC")],
           "--offload-device-only", "-S", SRC, "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True)
    asm = out.read_text()
    names = re.findall(r"^\s+\.name:\s+(\S*bsim_step_kernel_many\S*)", asm, flags=re.M)
    priv = [int(x) for x in re.findall(r"^\s+\.private_segment_fixed_size:\s+(\d+)", asm, flags=re.M)]
    assert len(names) == 3 and priv == [0, 0, 0]
