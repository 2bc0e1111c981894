"""Source bounds of the wide prefill tiles' LDS copies, on the CPU: a host program walks
every copied lane of the kernels' own offset functions (csrc/copy_bounds.h), with the
copies that run ahead of the last K step and tiles of one weight row."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_copies_stay_inside_the_weights(tmp_path):
    walk = str(tmp_path / "walk")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "kunlunk200_lib_amd", "csrc"),
                    os.path.join(ROOT, "tests", "copy_bounds_walk.cpp"), "-o", walk], check=True)
    proc = subprocess.run([walk], capture_output=True, text=True, timeout=100)
    assert proc.returncode == 0, proc.stdout
