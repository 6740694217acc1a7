"""How many sort slots a sampler takes (pz_slots.h): one per CU where there is
memory for them, fewer on a nearly full device or where an allocation fails,
and never none while one fits."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "native", "slots_check.cpp")
INC = os.path.join(ROOT, "project-zero_amd", "csrc")


def test_slots_fall_back_to_what_fits(tmp_path):
    exe = tmp_path / "slots_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", INC, SRC, "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    print(out.stdout)
    assert out.returncode == 0, out.stdout
