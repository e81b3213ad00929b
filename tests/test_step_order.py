"""The order of what a K-step of the tiles of 256 columns does to LDS, replayed on the CPU for every form of the kernel (tests/cpp/wreg_step.cc)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_read_and_copy_of_a_step_is_behind_the_barrier_it_needs(tmp_path):
    exe = str(tmp_path / "wreg_step")
    subprocess.run(["g++", "-std=c++17", "-O1", os.path.join(ROOT, "tests", "cpp", "wreg_step.cc"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "all steps in order" in r.stdout, r.stdout
