"""Steps whose entries read the same cache rows (KV-sharing layers): a plan of a few sharing entries in a larger step
streams the rows, one where an eighth of the tiles or more are read again keeps them in the caches, and a pair launch
takes each plan's own form. The same entries on copies of the caches, where nothing is shared, have the same
partition, so attnOut must be equal bit for bit; the oracle's chain checks each entry of the smaller steps."""
import numpy as np
import pytest
import torch

from conftest import announce
from g4attn import ops
from test_gpu_step import Layer, check

pytestmark = pytest.mark.gpu


def layers_of(dev, seed, hd, entries):
    """entries: (seq, window, producer's index or None); a consumer reads its producer's caches and raw k and v."""
    out = []
    for i, (seq, window, p) in enumerate(entries):
        L = Layer(dev, seed + 7 * i, seq, window, hd=hd, cache=None if p is None else (out[p].kc, out[p].vc))
        L.producer = None if p is None else out[p]
        out.append(L)
    return out


def entry(L, own_caches):
    P = L.producer
    e = L.entry(inv_freq=True) if P is None else dict(
        L.entry(store=False, raw_kv=(P.d["k"], P.d["v"]), inv_freq=True), k_weight=P.dkw)
    if own_caches and P is not None:
        e.update(k_cache=P.kc.clone(), v_cache=P.vc.clone())
    return e


def plan_of(dev, layers, hd, own_caches):
    items = [entry(L, own_caches) for L in layers]
    arr = ops.make_step_entries(items, 8, 1, hd)
    ws = torch.empty(ops.step_workspace_bytes(len(items), 8, 1, hd), dtype=torch.uint8, device=dev)
    return ops.attn_step_prepare(arr, 8, 1, hd, ws), (items, arr, ws)


def outputs(layers):
    torch.cuda.synchronize()
    got = [L.out.cpu().numpy().copy() for L in layers]
    for L in layers:
        L.out.fill_(float("nan"))
    return got


def same_bits(a, b):
    for i, (x, y) in enumerate(zip(a, b)):
        assert np.isfinite(x).all()
        np.testing.assert_array_equal(x.view(np.uint32), y.view(np.uint32), err_msg=f"entry {i}")


STEPS = {
    "one small pair": [(3000, 0, None)] * 5 + [(600, 0, None), (600, 0, 5)],
    "an eighth": [(1024, 0, None)] * 7 + [(1024, 0, 2)],
    "most": [(2000, 0, None), (513, 512, None)] + [(2000, 0, 0), (513, 512, 1)] * 4,
    "one cache, other rows": [(900, 0, None), (900, 128, 0), (900, 0, 0), (900, 128, 0)],
    "large batch, one twice": [(700 + 131 * i, 0, None) for i in range(40)] + [(700 + 131 * 9, 0, 9)],
    "large batch, half": [(2000 + 150 * i, 0, None) for i in range(24)] + [(2000 + 150 * i, 0, i) for i in range(24)],
}


@pytest.mark.parametrize("hd", [256, 512])
@pytest.mark.parametrize("name", list(STEPS))
def test_shared_rows(dev, hd, name):
    announce(f"attnStep shared rows hd={hd} {name}")
    layers = layers_of(dev, 500 + hd, hd, STEPS[name])
    plan, keep = plan_of(dev, layers, hd, False)
    ops.attn_step_run(plan)
    torch.cuda.synchronize()
    if sum(L.seq for L in layers) <= 40000:
        for i, L in enumerate(layers):
            want, kb, vb = L.expected(kv_from=L.producer)
            check(L, want, kb, vb, f"{name}: entry {i}")
    shared = outputs(layers)
    plan, keep = plan_of(dev, layers, hd, True)
    ops.attn_step_run(plan)
    same_bits(shared, outputs(layers))


@pytest.mark.parametrize("a", ["one small pair", "most"])
@pytest.mark.parametrize("b", ["one small pair", "most"])
def test_shared_rows_in_a_pair(dev, a, b):
    announce(f"attnStep pair, shared rows: head_dim 512 {a}, 256 {b}")
    la, lb = layers_of(dev, 100, 512, STEPS[a]), layers_of(dev, 900, 256, STEPS[b])
    got = []
    for own in (False, True):
        (pa, ka), (pb, kb) = plan_of(dev, la, 512, own), plan_of(dev, lb, 256, own)
        ops.attn_step_run_pair(pa, pb)
        got.append(outputs(la + lb))
    same_bits(*got)
