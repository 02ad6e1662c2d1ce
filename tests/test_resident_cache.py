"""The remembered occupancy of persistent launches (csrc/resident_cache.h, compiled by tests/resident_cache.cpp):
a verify loop over several shapes and row counts asks the runtime once per combination."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_a_verify_loop_asks_once_per_key(tmp_path):
    exe = str(tmp_path / "resident_cache")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", os.path.join(HERE, "..", "x100-gemm_amd", "csrc"),
                           os.path.join(HERE, "resident_cache.cpp"), "-o", exe])
    loop, many, wrong = map(int, subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split())
    assert loop == 40 and many and wrong == 0
