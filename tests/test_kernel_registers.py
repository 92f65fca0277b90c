"""The compiler's register report, for kernels whose time hangs on the waves per SIMD that they leave room for."""
import importlib.util
import re
import shutil
import subprocess
from pathlib import Path

import pytest

PKG = Path(__file__).resolve().parents[1] / "kernel-rsi_amd"


def waves_per_simd(source):
    """{mangled kernel name: waves per SIMD} of one kernel source, compiled as the library is."""
    spec = importlib.util.spec_from_file_location("krsi_build", PKG / "build.py")
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    cmd = [build._hipcc(), *build.HIP_FLAGS, *build.EXTRA_FLAGS.get(source, []), f"-I{build.INCLUDE}",
           f"-I{build.CSRC}", "-Rpass-analysis=kernel-resource-usage", "--offload-device-only", "-c",
           str(build.CSRC / source), "-o", "/dev/null"]
    report = subprocess.run(cmd, capture_output=True, text=True, check=True).stderr
    return {m[1]: int(m[2]) for m in re.finditer(r"Function Name: (\S+).*?Occupancy[^:]*: (\d+)", report, re.S)}


@pytest.mark.skipif(not (Path("/opt/rocm/bin/hipcc").is_file() or shutil.which("hipcc")), reason="no hipcc")
def test_rmsnorm_backward_of_aligned_rows():
    """A backward wave keeps a row's w, dw and two rows of g and x in registers. fp32 rows of 4097 to 8192 columns
    use exactly the 256 that leave two waves per SIMD: a few more leave one ([4096, 8192] 77.3 us with two, 87.0
    with one)."""
    waves = waves_per_simd("rmsnorm.hip")
    assert [v for k, v in waves.items() if "rms_bwd_vecILi2ELi4ELi8ELb0E" in k] == [2]
