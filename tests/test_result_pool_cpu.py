"""Result buffers of a batch (csrc/result_pool.h) taken and released by several threads at once."""
import subprocess
from pathlib import Path

HERE = Path(__file__).resolve().parent


def test_threads(tmp_path):
    exe = tmp_path / "check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", str(HERE.parent / "viscoplastic-lbm_amd" / "csrc"),
                    str(HERE / "host_stub" / "result_pool_check.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, f"exit {res.returncode} {res.stdout}"
