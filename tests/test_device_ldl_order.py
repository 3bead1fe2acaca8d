"""The diagonal-block factorization of the device LDL on the CPU, its waves run in different orders between the barriers of
the workgroup (tests/cpp/diag_block_emulation.cpp): the factor must not depend on which wave comes first, and must equal
the host factorization's, word for word."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "behemoth-qtip_amd", "csrc")


@pytest.fixture(scope="module")
def emulation(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("emulation") / "diag_block_emulation")
    subprocess.check_call(["g++", "-O1", "-std=c++20", "-ffp-contract=off", "-mfma", "-Wno-unknown-pragmas",
                           os.path.join(ROOT, "tests", "cpp", "diag_block_emulation.cpp"),
                           os.path.join(CSRC, "host_ldl_diag.cpp"), "-o", exe])
    return exe


@pytest.mark.parametrize("order", ["0123", "3210", "1230"])
@pytest.mark.parametrize("kb", [16, 48, 256])
def test_diagonal_block_does_not_depend_on_the_order_of_the_waves(emulation, kb, order):
    run = subprocess.run([emulation, str(kb), order], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout
