"""Host loops over threads (csrc/parallel.hpp), compiled for the CPU."""
import subprocess
from pathlib import Path

HERE = Path(__file__).resolve().parent


def test_parallel_for_survives_exceptions_and_missing_threads(tmp_path):
    exe = tmp_path / "parallel_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", str(HERE / "parallel_check.cpp"), "-o", str(exe),
                    "-ldl"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
