"""The search for the closed path on the CPU (tests/cpp/close_path_emulation.cpp): where it settles a tile, the states are those of
the cheapest closed path by the plain recursion, whichever wave comes first; each way in which a search can end is taken by some kind
of inputs."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def emulation(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("emulation") / "close_path_emulation")
    subprocess.check_call(["g++", "-O2", "-std=c++20", "-ffp-contract=off", "-mfma", "-mf16c", "-Wno-unknown-pragmas",
                           os.path.join(ROOT, "tests", "cpp", "close_path_emulation.cpp"), "-o", exe])
    return exe


def _run(exe, kind, threads, order, tiles):
    run = subprocess.run([exe, kind, str(threads), order, str(tiles)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout
    words = run.stdout.split()
    return dict(zip(words[0::2], map(int, words[1::2])))


@pytest.mark.parametrize("kind,ends", [("gauss", {"early": 6, "step0": 6, "second": 1, "lowered": 1}),
                                       ("join", {"early": 6, "step0": 6, "lowered": 6}),
                                       ("flat", {"early": 3, "step0": 6}),
                                       ("alike", {"early": 3, "full": 1, "gave_up": 3}),
                                       ("mirror", {"gave_up": 6}),
                                       # costs that leave no room for a limit
                                       ("coarse", {"early": 3, "step0": 3, "refused": 3})])
def test_search_finds_the_cheapest_closed_path(emulation, kind, ends):
    got = _run(emulation, kind, 256, "3210", 24)
    assert all(got[end] >= least for end, least in ends.items()), got


@pytest.mark.parametrize("kind", ["gauss", "alike"])
@pytest.mark.parametrize("order", ["0123", "1032", "2301"])
def test_search_does_not_depend_on_the_order_of_the_waves(emulation, kind, order):
    """The first wave writes the states that the search has found; the others are still to come."""
    assert _run(emulation, kind, 256, order, 24)["early"] >= 3


@pytest.mark.parametrize("order", ["01234567", "76543210"])
def test_search_by_512_threads(emulation, order):
    got = _run(emulation, "gauss", 512, order, 12)
    assert got["early"] + got["step0"] == 12, got
