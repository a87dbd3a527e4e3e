"""The host threads and the loop over half buffers that frames are copied with, built
without a device: a failed allocation or call neither ends the process nor leaves a
buffer that a kernel still writes."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_copiers_and_halves_under_failures(tmp_path):
    exe = str(tmp_path / "frame_copy")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror",
                    "-Wno-mismatched-new-delete", "-pthread",
                    "-I", os.path.join(ROOT, "platelet_fiber_gpu_amd", "csrc"),
                    os.path.join(ROOT, "tests", "frames", "frame_copy.cpp"), "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert (r.returncode, r.stdout) == (0, "ok\n"), r.stdout + r.stderr
