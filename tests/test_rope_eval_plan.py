"""The step planner's tables where the kernel evaluates the RoPE factors, as g4_attn_step_prepare plans them, on the CPU
under AddressSanitizer and UndefinedBehaviorSanitizer (tests/rope_eval_check.cpp)."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_rope_eval_plans(tmp_path):
    exe = tmp_path / "rope_eval_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    str(ROOT / "tests" / "rope_eval_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
    _, steps, evaluated = out.stdout.split()
    assert int(steps) // 4 < int(evaluated) < 3 * int(steps) // 4
    # the check plans with the library's own threshold
    sets = re.search(r"constexpr uint32_t kSets = (\d+);", (ROOT / "tests" / "rope_eval_check.cpp").read_text())[1]
    assert f"kStepRopeEvalSets = {sets};" in (ROOT / "gemma4-webgpu_amd" / "csrc" / "step.hip").read_text()
