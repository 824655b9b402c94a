"""The last workgroup of a selection kernel reads what the others wrote, on other
XCDs too: after it has counted them it must drop the lines its own caches hold.
Read from the kernels' assembly, as no run shows reliably that this is missing."""
import os
import re
import subprocess

from ripples_amd import build

KERNELS = ("top_hist_kernel", "top_tiles_kernel", "top_pick_kernel", "top_rounds_kernel")


def test_last_block_acquires(tmp_path):
    out = str(tmp_path / "select_top.s")
    subprocess.run([build.HIPCC] + build.COMMON + build.HIP_FLAGS +
                   ["--offload-device-only", "-S", os.path.join(build.CSRC, "select_top.hip"), "-o", out],
                   check=True, capture_output=True, timeout=300)
    text = open(out).read()
    for kernel in KERNELS:
        body = re.search(r"^_Z\w*%s\w*:[^\n]*$(.*?)^\.Lfunc_end" % kernel, text, re.M | re.S).group(1)
        # the count of finished blocks is the one 32-bit add in memory whose
        # old value is used
        counts = [m.end() for m in re.finditer(r"global_atomic_add v\d+, .*\bsc0$", body, re.M)]
        assert len(counts) == 1, kernel
        until = body.index("s_barrier", counts[0])
        assert "buffer_inv sc1" in body[counts[0]:until], kernel
