"""Wave schedules of the forward projector, on the CPU: with one workgroup per CU
(bands of which two do not fit the LDS, or a prefetching projector, whatever its
bands) no exchange of two pairs between waves lowers the bands' busiest waves any
more."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBDIR = os.path.join(ROOT, "aretomo3_amd")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.exists(os.path.join(LIBDIR, "libatr_recon.so")):
        pytest.skip("no compiler, or library not built")
    exe = str(tmp_path_factory.mktemp("schedule") / "schedule_check")
    cmd = ["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
           "-I" + os.path.join(LIBDIR, "csrc"), "-I" + os.path.join(ROOT, "include"),
           os.path.join(ROOT, "tests", "schedule_check.cpp"), "-o", exe, "-L", LIBDIR, "-latr_recon",
           "-Wl,-rpath," + LIBDIR]
    build = subprocess.run(cmd, capture_output=True, text=True)
    assert build.returncode == 0, build.stderr
    return exe


@pytest.mark.parametrize("vol_x,vol_z,rows,staging", [
    (1024, 256, 17, 0), (512, 128, 16, 1), (512, 128, 8, 1), (768, 96, 8, 1), (1024, 128, 8, 1),
    (1024, 128, 8, 2), (1024, 256, 17, 2)])
def test_no_exchange_is_left(check, vol_x, vol_z, rows, staging):
    out = subprocess.run([check, str(vol_x), str(vol_z), str(rows), str(staging)], capture_output=True,
                         text=True, timeout=60)
    assert out.returncode == 0, out.stderr
    groups = [tuple(map(float, ln.split())) for ln in out.stdout.splitlines()]
    assert groups
    for now, gain in groups:
        assert now > 0 and gain < 1e-6 * now
