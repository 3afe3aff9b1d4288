"""The wait of a hand-over is one that the compiler may not move a store
across (planner_device.h, stores_done): read from what it makes of a kernel
with a store on either side."""
import os
import re
import subprocess

from conftest import ROOT


def _compiled(*flags):
    from prrtc_amd.build import FLAGS, HIPCC
    res = subprocess.run([HIPCC, *FLAGS, "--offload-device-only", *flags, os.path.join(ROOT, "tests", "cpp", "stores.hip"),
                          "-o", "-"], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stderr[-2000:]
    return res.stdout


def test_stores_stay_before_the_wait():
    ir = _compiled("-S", "-emit-llvm")
    body = ir[ir.index("@two_stores("):]
    body = body[:body.index("\n}")]
    wait = re.findall(r"asm sideeffect \"s_waitcnt vmcnt\(0\)\", \"([^\"]*)\"", body)
    assert len(wait) == 1 and "~{memory}" in wait[0]
    asm = _compiled("-S")
    asm = asm[asm.index("two_stores:"):asm.index(".Lfunc_end0")]
    steps = re.findall(r"global_store|s_waitcnt vmcnt\(0\)", asm)
    first, wait = steps.index("global_store"), steps.index("s_waitcnt vmcnt(0)")
    assert first < wait < len(steps) - 1 - steps[::-1].index("global_store")
