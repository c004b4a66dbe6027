"""The 32-bit offsets of the kernels' row accesses, on the host: grids whose levels span more than 2^32 bytes (an x-z
slice of 2^29 elements or more per field is accepted, up to 2^31), which no test could hold in full."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def test_base_state_offsets(tmp_path):
    exe = tmp_path / "offsets_check"
    # the host pass only: the accessors of the kernels' header, compiled for the CPU
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O1", "-std=c++20", "-o", str(exe),
                    os.path.join(HERE, "native", "offsets_check.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("real,ns", [("double", "mi_fp64"), ("float", "mi_fp32")])
def test_substep_form(tmp_path, real, ns):
    lib = os.path.join(os.path.dirname(HERE), "cppwrf_amd")
    exe = tmp_path / "substep_form_check"
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O1", "-std=c++20", f"-DMI_REAL={real}", f"-DMI_NS={ns}", "-o",
                    str(exe), os.path.join(HERE, "native", "substep_form_check.cpp"), "-L" + lib, "-l:libcppwrf_amd.so",
                    "-Wl,-rpath," + lib], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
