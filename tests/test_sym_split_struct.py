"""SymSplit itself (utc_amd/csrc/sym_split.h), compiled for the host with
overflow checks: its ranges, records and wave lookup over small and the largest
systems (tests/host/sym_split_sweep.cpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_every_chunk_once_and_every_record_found(tmp_path):
    exe = tmp_path / "sym_split_sweep"
    b = subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                        "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{ROOT / 'utc_amd' / 'csrc'}",
                        str(ROOT / "tests" / "host" / "sym_split_sweep.cpp"), "-o", str(exe)],
                       capture_output=True, text=True)
    assert b.returncode == 0, b.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout + r.stderr
