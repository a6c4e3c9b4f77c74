"""GPU parity of the prefill's per-token merge where its table of query tiles ends: the last tile of an entry with
one token, one short of a full tile, and exactly full, each cut into few parts (the small merge) and into more than
eight; groups of 8, 4, 2 and 1 query heads (16 to 128 tokens per tile), and a whole entry beside a split one. Every
token against the oracle's chain at its own seq_len, and attnOut past an entry's tokens stays untouched."""
import pytest
import torch

from conftest import announce
from test_gpu_prefill import Chunk, check, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nqh,nkh,hd,tokens,start", [
    (8, 1, 256, 1, 900), (8, 1, 256, 15, 900), (8, 1, 256, 16, 5000), (8, 1, 256, 17, 5000), (4, 1, 256, 31, 700),
    (4, 1, 256, 33, 3500), (2, 1, 256, 65, 1500), (2, 2, 256, 127, 1300), (8, 2, 256, 17, 2500), (8, 1, 512, 15, 700),
    (8, 1, 512, 17, 4000), (4, 1, 512, 33, 600)])
def test_prefill_token_merge(dev, nqh, nkh, hd, tokens, start):
    announce(f"prefill token merge nqh={nqh} nkh={nkh} hd={hd} tokens={tokens} start={start}")
    chunks = [Chunk(dev, 3 * start + tokens, start, tokens, 0, nqh=nqh, nkh=nkh, hd=hd),
              Chunk(dev, 7 * start + tokens, 0, 5, 0, nqh=nqh, nkh=nkh, hd=hd)]
    for c in chunks:  # a row's worth of guard behind the outputs
        guarded = torch.full((c.out.numel() + nqh * hd,), 7.0, device=dev)
        c.guard, c.out = guarded[c.out.numel():], guarded[:c.out.numel()]
    run(dev, chunks, nqh=nqh, nkh=nkh, hd=hd)
    for i, c in enumerate(chunks):
        check(c, f"entry {i}")
        assert bool((c.guard == 7.0).all())
