"""The launch rules of gemma4-webgpu_amd/csrc/launch_rules.h on the CPU, at sizes measured on both sides of each line."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not installed")
    exe = tmp_path_factory.mktemp("rules") / "launch_rules_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    str(ROOT / "tests" / "launch_rules_check.cpp"), "-o", str(exe)], check=True)

    def evaluate(name, *args):
        out = subprocess.run([str(exe)], input=" ".join(map(str, (name, *args))), capture_output=True, text=True, check=True)
        return int(out.stdout)

    return evaluate


@pytest.mark.parametrize("tokens", [1, 2, 3, 4, 5, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128])
def test_token_merge_columns(rule, tokens):
    """The columns cover the largest tile's tokens, and fewer than twice as many are launched."""
    columns = 1 << rule("token_merge_shift", tokens)
    assert tokens <= columns < 2 * tokens
