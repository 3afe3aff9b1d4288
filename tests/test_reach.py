"""The broad phase's arithmetic itself, built for the host from the library's
header and run on the CPU (tests/cpp/reach.cpp)."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="session")
def reach(tmp_path_factory):
    from prrtc_amd.build import HIPCC
    exe = str(tmp_path_factory.mktemp("reach") / "reach")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1",
                    os.path.join(ROOT, "tests", "cpp", "reach.cpp"), "-o", exe], check=True)
    return lambda *a: subprocess.run([exe, *a], capture_output=True, text=True, timeout=120)


def test_scene_lds(reach):
    """A workgroup asks for the LDS its scene takes and no more."""
    assert reach("lds").returncode == 0


@pytest.mark.parametrize("lo, hi, sign", [(-2, 0.5, 1), (-2, 0.5, -1), (2, 4, 1), (5, 7, 1)])
def test_out_of_reach_hits_nothing(reach, lo, hi, sign):
    """An obstacle of each kind brought along the tightest direction to the
    first place where its ball is out of the wave's reach: every exact test is
    positive there, and the surfaces keep the pads (1 mm, and half of 2^-16).  A sphere or
    capsule of negative radius reaches as far as one of the positive (the tests
    square the sum of the radii), and positions far from the origin (up to 10^7
    m) are rounded to more than the 1 mm."""
    res = reach("reach", str(lo), str(hi), str(sign))
    assert res.returncode == 0, res.stdout
    kinds = [line.split() for line in res.stdout.splitlines()]
    assert len(kinds) == 5
    for kind, used, spare in kinds:
        assert int(used) == 4000 and float(spare) >= 0, kind
