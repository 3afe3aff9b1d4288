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
