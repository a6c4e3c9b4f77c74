"""The step planner's work-item order for entries that share cache rows, on the CPU (tests/kv_share_check.cpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_kv_share_order(tmp_path):
    exe = tmp_path / "kv_share_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    str(ROOT / "tests" / "kv_share_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
    _, steps, shared, kept = out.stdout.split()
    assert int(shared) > int(steps) // 2
    assert int(steps) // 4 < int(kept) < int(shared) - int(steps) // 40  # both sides of the rule
