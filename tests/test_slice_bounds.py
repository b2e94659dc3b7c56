"""The unguarded loads of the plain SGEMM k loops stay inside their operands: a
host program (tests/cpp/test_slice_bounds.cpp) walks the kernels' own bounds for
operands of few lines, at every K near a boundary of accumulation blocks."""
import os
import shutil
import subprocess

import helpers

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def test_unguarded_loads_stay_inside(tmp_path):
    exe = str(tmp_path / "test_slice_bounds")
    subprocess.run([HIPCC, "-std=c++17", "-O2", "-Wall", "-Werror", "--offload-arch=gfx950",
                    "-I" + os.path.join(helpers.ROOT, "include"),
                    "-I" + os.path.join(helpers.ROOT, "openmp-blas_amd", "csrc"),
                    os.path.join(helpers.ROOT, "tests", "cpp", "test_slice_bounds.cpp"),
                    "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.startswith("ok ") and int(out.stdout.split()[1]) > 10000, out.stdout
