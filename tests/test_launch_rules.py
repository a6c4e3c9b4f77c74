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


@pytest.mark.parametrize("heads,seq,form", [
    # the loop form, measured the faster one
    (8, 1, 0), (8, 64, 0), (8, 256, 0), (64, 512, 0), (512, 64, 0), (512, 300, 0), (512, 1024, 0), (1024, 100, 0),
    (1024, 2048, 0), (2048, 100, 0), (2048, 2048, 0), (2048, 4096, 0), (1024, 5000, 0), (2048, 5000, 0), (8, 16385, 0),
    # the register form, measured the faster one
    (1, 513, 4), (8, 600, 4), (8, 1000, 4), (8, 4096, 4), (256, 1024, 4), (512, 1500, 4), (512, 2048, 4), (1024, 3000, 4), (1024, 4096, 4), (8, 4097, 16),
    (8, 16384, 16), (512, 8192, 16), (1024, 7000, 16)])
def test_softmax_form(rule, heads, seq, form):
    assert rule("softmax_scores_per_thread", heads, seq) == form
    if form:  # the register form holds the scores
        assert seq <= 1024 * form


def test_softmax_form_at_the_limits(rule):
    for heads in (1, 256, 257, 2**31, 2**32 - 1):
        for seq in (1, 512, 513, 4096, 4097, 16384, 16385, 2**32 - 1):
            form = rule("softmax_scores_per_thread", heads, seq)
            assert form in (0, 4, 16) and (not form or 512 < seq <= 1024 * form)


@pytest.mark.parametrize("workgroups,seq,chain", [
    # the general form, measured the faster one
    (4, 1, 0), (32, 1, 0), (32, 4, 0), (64, 12, 0), (1, 8, 0), (512, 16, 0), (1024, 1, 0), (1024, 48, 0), (2048, 128, 0),
    (4096, 512, 0), (8192, 768, 0),
    # the chain form, measured the faster one
    (1, 16, 1), (32, 16, 1), (64, 64, 1), (64, 2048, 1), (256, 24, 1), (512, 64, 1), (1024, 96, 1), (2048, 256, 1),
    (4096, 768, 1), (8192, 1024, 1), (8192, 2048, 1)])
def test_attn_output_form(rule, workgroups, seq, chain):
    assert rule("attn_output_chain", workgroups, seq, 256) == chain


def test_attn_output_form_at_the_limits(rule):
    for workgroups in (1, 65535 * 8, 2**32 - 1):
        assert rule("attn_output_chain", workgroups, 0, 256) == 0
        assert rule("attn_output_chain", workgroups, 2**30 - 1, 1) == 1


@pytest.mark.parametrize("size,small", [(0, 1), (1, 1), (255, 1), (4096, 0), (262144, 0), (2**32 - 1, 0)])
def test_argmax_form(rule, size, small):
    assert rule("argmax_small", size) == small
