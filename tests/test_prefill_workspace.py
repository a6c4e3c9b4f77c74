"""One prefill workspace for prompts of several lengths: what the longest one needs is accepted for every shorter one
over the same cached rows, where a short prompt alone would take more (its key parts are shorter and so more). On the
CPU: prepare either refuses for want of workspace or goes on to the upload, which fails without a GPU. On the GPU: the
short prompt in the smaller workspace attends as in its own, against the oracle."""
import ctypes as C

import pytest
import torch

from conftest import announce
from g4attn import abi, ops

LENGTHS = [  # (head_dim, cached rows, longest prompt): the shortest prompts that keep parts of 256 keys, and longer ones
    (256, 300, 497), (256, 1000, 273), (256, 1000, 600), (256, 1500, 193), (256, 2000, 145), (256, 3000, 97),
    (256, 3000, 288), (256, 8000, 33), (512, 0, 465), (512, 300, 289), (512, 1000, 129), (512, 1500, 97),
    (512, 2000, 81), (512, 3000, 49), (512, 8000, 17)]


def _entry(start, tokens):
    e = abi.PrefillEntry()  # addresses that are never read: the upload is the first use of the GPU
    e.q, e.k_cache, e.v_cache, e.out = 1 << 20, 2 << 20, 3 << 20, 4 << 20
    e.n_tokens, e.start, e.scale = tokens, start, 1.0
    return e


@pytest.mark.skipif(torch.cuda.is_available(), reason="made-up addresses: for a machine without a GPU")
@pytest.mark.parametrize("hd,start,longest", LENGTHS)
def test_shorter_prompts_fit_the_longest_ones_workspace(hd, start, longest):
    lib = abi.load()
    need = C.c_size_t()
    e = _entry(start, longest)
    assert lib.g4_attn_prefill_workspace_size(C.byref(e), 1, 8, 1, hd, C.byref(need)) == abi.G4_OK
    plan, larger = abi.DecodePlan(), 0
    for tokens in range(1, longest):
        e, own = _entry(start, tokens), C.c_size_t()
        assert lib.g4_attn_prefill_workspace_size(C.byref(e), 1, 8, 1, hd, C.byref(own)) == abi.G4_OK
        larger += own.value > need.value
        st = lib.g4_attn_prefill_prepare(C.byref(e), 1, 8, 1, hd, 1 << 30, need.value, C.byref(plan), None)
        assert st != abi.G4_ENOSPC, f"{tokens} tokens: {lib.g4_last_error().decode()}"
    st = lib.g4_attn_prefill_prepare(C.byref(e), 1, 8, 1, hd, 1 << 30, 4096, C.byref(plan), None)
    assert st == abi.G4_ENOSPC
    print(f"hd={hd} start={start}: {larger} of {longest - 1} shorter prompts would take more than the longest")


@pytest.mark.gpu
@pytest.mark.parametrize("hd,start,tokens,longest", [(256, 3000, 96, 97), (512, 1500, 90, 97), (256, 1000, 40, 300)])
def test_short_prompt_in_a_longer_ones_workspace(dev, hd, start, tokens, longest):
    from test_gpu_prefill import Chunk, check

    announce(f"attnPrefill hd={hd} start={start} tokens={tokens} in the workspace of {longest}")
    long_one = ops.make_prefill_entries([Chunk(dev, 5, start, longest, 0, hd=hd).entry()], 8, 1, hd)
    need = ops.prefill_workspace_bytes(long_one, 8, 1, hd)
    c = Chunk(dev, 7 * start + tokens, start, tokens, 0, hd=hd)
    arr = ops.make_prefill_entries([c.entry()], 8, 1, hd)
    sizes = [need, ops.prefill_workspace_bytes(arr, 8, 1, hd)]
    for size in sizes:
        guarded = torch.full((size + 4096,), 0x5A, dtype=torch.uint8, device=dev)
        c.out.fill_(float("nan"))
        ops.attn_prefill_run(ops.attn_prefill_prepare(arr, 8, 1, hd, guarded[:size]))
        torch.cuda.synchronize()
        check(c, f"workspace of {size}")
        assert bool((guarded[size:] == 0x5A).all())
    assert (sizes[0] < sizes[1]) == ((hd, tokens) != (256, 40)), sizes
