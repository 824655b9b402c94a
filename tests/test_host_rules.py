"""What the library does around its kernels, on a HIP runtime without a device
(host_rules_check.cpp)."""
import os
import subprocess

import pytest

import ripples_amd as R

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_DIR = os.path.dirname(R.LIB_PATH)


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host") / "host_rules_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-rdynamic", "-I", os.path.join(HERE, "..", "include"),
                    os.path.join(HERE, "host_rules_check.cpp"), "-o", out, "-L", LIB_DIR,
                    "-lripples_amd", "-Wl,-rpath," + LIB_DIR, "-Wl,--allow-shlib-undefined"],
                   check=True, capture_output=True, timeout=300)
    return out


@pytest.mark.parametrize("name", [
    "grid_scratch_after_failure",
    "lds_limit_is_kept",
    "scratch_fits_little_memory",
    "counts_fit_little_memory",
    "long_sets_fill_the_chip",
    "long_lists_go_wide",
    "poor_passes_end",
    "graphs_stay_bounded",
    "spread_fills_its_cus",
    "tuned_settings_part_at_the_team_line",
    "staged_settings_differ",
    "idle_memory_is_given_back",
])
def test_host_rules(exe, name):
    r = subprocess.run([exe, name], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
