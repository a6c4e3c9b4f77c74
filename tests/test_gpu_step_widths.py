"""GPU parity of the head_dim-512 step where its combine reads the states of 2, 4, 6 or 8 waves: a part's rows over
16-row tiles of eight waves, rounded up to an even count. One entry over a whole GPU's workgroups (256) has parts of
one 32-row tile up to 8192 rows (2 waves), of two up to 16384 (4), of three up to 24576 (6) and of more above (8); its
last part is shorter. Beside that, entries of every width in one plan, and a plan advanced across the edge of a tile."""
import pytest
import torch

from conftest import announce
from g4attn import ops
from test_gpu_step import Layer, check, run_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seq,nqh,nkh", [
    (2000, 8, 1), (8192, 8, 1), (8193, 8, 1), (12300, 8, 1), (16384, 8, 1), (16385, 8, 1), (20011, 8, 1), (24576, 8, 1),
    (24577, 8, 1), (31000, 8, 1), (9000, 8, 2), (5000, 4, 4)])
def test_combine_widths(dev, seq, nqh, nkh):
    announce(f"attnStep hd=512 combine widths seq={seq} nqh={nqh} nkh={nkh}")
    L = Layer(dev, 40 + seq, seq, 0, 1e6, 1, nqh=nqh, nkh=nkh, hd=512)
    want, kb, vb = L.expected()
    run_step(dev, [L.entry(inv_freq=True)], nqh=nqh, nkh=nkh, hd=512)
    check(L, want, kb, vb, f"seq={seq}")


def test_combine_widths_in_one_plan(dev):
    seqs = [1, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 79, 80, 81, 95, 96, 97, 112, 113, 127, 128, 129, 200, 257]
    announce(f"attnStep hd=512 {8 * len(seqs) + 60} entries, parts of 1 to 257 rows")
    # more entries than workgroups fit: every entry is one part, whole
    layers = [Layer(dev, 3000 + i, s, 0, 1e6, 1, hd=512) for i, s in enumerate(seqs * 8 + [5] * 60)]
    run_step(dev, [L.entry(inv_freq=True) for L in layers], hd=512)
    for i, L in enumerate(layers):
        want, kb, vb = L.expected()
        check(L, want, kb, vb, f"entry {i} of {L.seq} rows")


@pytest.mark.parametrize("seq,window", [(16380, 0), (24570, 0), (700, 80), (300, 64)])
def test_combine_widths_advanced(dev, seq, window):
    """Advanced plans: the last part grows past its width, a window's parts move over tile edges."""
    announce(f"attnStep hd=512 advanced seq={seq} window={window}")
    tokens = 20
    L = Layer(dev, 90 + seq, seq + tokens, window, 1e6, 1, hd=512)
    want, kb, vb = L.expected()
    for name, cache in (("k", L.kc), ("v", L.vc)):  # the rows that the earlier tokens would have stored stay in place
        assert cache.shape[0] == seq + tokens, name
    e = dict(L.entry(inv_freq=True), seq_len=seq, position=seq - 1)
    arr = ops.make_step_entries([e], 8, 1, 512)
    ws = torch.empty(ops.step_workspace_bytes(1, 8, 1, 512), dtype=torch.uint8, device=dev)
    plan = ops.attn_step_prepare(arr, 8, 1, 512, ws)
    ops.attn_step_advance(plan, tokens)
    ops.attn_step_run(plan)
    torch.cuda.synchronize()
    check(L, want, kb, vb, f"seq={seq} advanced by {tokens}")
