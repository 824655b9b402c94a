"""A device allocation that fails leaves no buffer that a later, smaller call
takes for allocated: the library's host code on a HIP runtime without a device
(alloc_fail_check.cpp)."""
import os
import subprocess

import ripples_amd as R

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_DIR = os.path.dirname(R.LIB_PATH)


def test_failed_allocations_claim_no_room(tmp_path):
    exe = str(tmp_path / "alloc_fail_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-rdynamic", "-I", os.path.join(HERE, "..", "include"),
                    os.path.join(HERE, "alloc_fail_check.cpp"), "-o", exe, "-L", LIB_DIR,
                    "-lripples_amd", "-Wl,-rpath," + LIB_DIR, "-Wl,--allow-shlib-undefined"],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
