"""The read-back slots of the write call (lq_readpool.h) built for the host
against stand-ins of the HIP calls they make: two devices, more callers at once
than slots are kept."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_readpool_host(tmp_path):
    exe = tmp_path / "readpool_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "tests", "host", "readpool"),
                    "-I", os.path.join(ROOT, "latticequant_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "readpool_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
