"""What a wave waits for before a bare barrier, read off the assembly of this repository's own source: where the barrier
gives an LDS stage free for other waves' loads, the wave's own reads of that stage have to have returned, wherever the
compiler puts the instructions that use them."""
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which(HIPCC)), reason="no hipcc")
def test_small_hessian_tiles_wait_for_their_reads_before_the_barrier(tmp_path):
    out = tmp_path / "hessian.s"
    subprocess.check_call([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++20", "-ffp-contract=off", "-Xclang",
                           "-target-feature", "-Xclang", "-packed-fp32-ops", "--offload-device-only", "-S", "-o", str(out),
                           os.path.join(ROOT, "behemoth-qtip_amd", "csrc", "hessian.hip")], stderr=subprocess.DEVNULL)
    text = out.read_text()
    kernel = re.search(r"^_ZN\w*syrk_img_small_kernel\w*:.*?s_endpgm", text, re.M | re.S).group(0)
    before = kernel[:kernel.index("s_barrier")]
    waits = re.findall(r"s_waitcnt (.*)", before[before.rindex("v_mfma"):])
    assert len(waits) == 7, waits                       # one per number of stages in flight
    assert all("lgkmcnt(0)" in w for w in waits), waits
