"""Kernels that need the whole chip run one after the other: the host code that sees to it, against a record of its runtime calls."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_order_of_resident_launches(tmp_path):
    """Whatever streams, threads and devices; streams that are being captured; launches that fail.  No call names another
    stream than the caller's (it may be in the middle of a capture, or gone), no event is a packet of its own."""
    exe = str(tmp_path / "resident_order")
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include", os.path.join(HERE, "resident_order.cpp"), "-o", exe, "-pthread"]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout[-3000:]
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, r.stdout[-3000:]
