"""Staged host transfers (hostio.hip) from several threads, on the CPU: built with
the host compiler against host copies in place of the HIP calls.  One transfer
uses the staging pool at a time; the others do not wait for it, however long it
holds it, and every byte arrives."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.mark.skipif(not shutil.which("g++") or not os.path.isdir(os.path.join(ROCM, "include", "hip")),
                    reason="needs g++ and the HIP headers")
def test_transfers_of_other_threads_go_through(tmp_path):
    exe = str(tmp_path / "hostio_stub")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                    "-x", "c++", os.path.join(ROOT, "midapack_amd", "csrc", "hostio.hip"),
                    os.path.join(ROOT, "tests", "hostio_stub.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    bad = [ln for ln in r.stdout.splitlines() if ln.startswith("FAIL")]
    assert r.returncode == 0 and not bad, bad
