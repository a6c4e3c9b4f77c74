"""A step whose entries sit at positions of their own (a batch of sequences): from four RoPE factor sets on, the plan
carries the inverse frequencies and the kernel evaluates the factors. The same entries planned as one layer of
attn_step_prepare_layers keep the host's factors on the same partition, so attnOut and the stored rows must be equal
bit for bit, as prepared and after both plans advance a token; three sets (below the rule) and entries that share one
set or bring no table are planned beside them."""
import numpy as np
import pytest
import torch

from conftest import announce
from g4attn import ops
from test_gpu_step import NKH, NQH, ROPE, Layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd", [256, 512])
@pytest.mark.parametrize("seqs", [(2, 40, 700), (3, 41, 701, 1500), (1, 2, 513, 2048, 4097, 9001), (77, 77, 77, 77, 300),
                                  (5, 600, None, 1200, 1900)])
def test_rope_factors_in_the_kernel(dev, hd, seqs):
    announce(f"attnStep RoPE evaluated in the kernel hd={hd} seqs={seqs}")
    tables = {w: ops.rope_inv_freq_host(1e4 if w else 1e6, hd, 0 if w else 1, ROPE) for w in (0, 512)}
    kinds = {}
    for kind in ("step", "layer"):
        layers, entries = [], []
        for i, seq in enumerate(seqs):
            w = 512 * (i % 2)
            L = Layer(dev, 60 + 9 * i, (seq or 333) + 1, 0, theta=1e4 if w else 1e6, divisor=0 if w else 1, hd=hd)
            L.kc[L.pos] = L.vc[L.pos] = 0  # one more row than the first token reads: the advanced token's
            e = dict(L.entry(), seq_len=L.seq - 1, position=L.pos - 1, sliding_window=w)
            if seq:
                e["rope_inv_freq_host"] = tables[w]
            layers.append(L)
            entries.append(e)
        arr = ops.make_step_entries(entries, NQH, NKH, hd)
        if kind == "step":
            ws = torch.empty(ops.step_workspace_bytes(len(entries), NQH, NKH, hd), dtype=torch.uint8, device=dev)
            plan = ops.attn_step_prepare(arr, NQH, NKH, hd, ws)
        else:
            ws = torch.empty(2 * ops.step_workspace_bytes(len(entries), NQH, NKH, hd), dtype=torch.uint8, device=dev)
            plan = ops.attn_step_prepare_layers(arr, NQH, NKH, hd, ws, entries_per_layer=len(entries))[0]
        got = []
        for token in range(2):
            ops.attn_step_run(plan)
            torch.cuda.synchronize()
            got += [t.cpu().numpy().copy() for L in layers for t in (L.out, L.kc[L.pos - 1 + token], L.vc[L.pos - 1 + token])]
            ops.attn_step_advance(plan)
        kinds[kind] = got
    for i, (a, b) in enumerate(zip(kinds["step"], kinds["layer"])):
        assert np.isfinite(a.astype(np.float64)).all()
        np.testing.assert_array_equal(a.view(np.uint8), b.view(np.uint8), err_msg=f"value {i}")
