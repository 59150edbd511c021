"""Launch rules shared by the host and the kernels (kernel_geometry.h), checked
on the CPU against the memory that the kernels' rows really cover."""
import os
import subprocess

from support import ROOT


def test_softmax_row_windows_fit_their_launch(tmp_path):
    exe = str(tmp_path / "geometry_check")
    subprocess.run(["gcc", "-O2", "-Wall", "-Werror", "-Wno-unused-function", "-I", os.path.join(ROOT, "dataflow_lib_amd", "csrc", "kernels"),
                    os.path.join(ROOT, "tests", "geometry_check.c"), "-o", exe], check=True)
    res = subprocess.run([exe], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout
