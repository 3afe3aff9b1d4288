"""The buffers a thread's host-buffer calls keep (host_call.h), over a stand-in
for the HIP runtime on the CPU: reuse, growth, a change of device, failures,
and a device reset between calls, after which nothing of the old set is used
or freed."""
import os
import subprocess

from conftest import ROOT


def test_kept_buffers(tmp_path):
    exe = str(tmp_path / "host_call")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "cpp", "host_call.cpp"), "-o", exe], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
