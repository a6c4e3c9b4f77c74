"""GPU parity of the engine's own dispatches where their fast forms begin and end: the matmuls'
row form and argmax's batches. Every form evaluates the reference's f32 operations in the reference's
order, so the bar is bit equality with the oracle, which also covers the general forms on the other side of each rule.
"""
import numpy as np
import pytest
import torch

from conftest import announce
from g4attn import ops
from oracle import closed_form as cf
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def up(a, dev, offset=0):
    """On the GPU as the ops take it, `offset` elements past an aligned address."""
    a = np.ascontiguousarray(a)
    t = torch.from_numpy(a.view({2: np.int16, 4: np.int32}[a.itemsize] if a.dtype.kind == "u" else a.dtype).ravel())
    buf = torch.empty(t.numel() + offset, dtype=t.dtype, device=dev)
    buf[offset:] = t
    return buf[offset:]


def bits(t):
    return t.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("fmt", ["f16", "q8", "q4k"])
@pytest.mark.parametrize("M,N,offset", [(1, 1024, 0), (7, 1536, 0), (2049, 1536, 0), (33, 4096, 0), (9, 2560, 1),
                                        (5, 768, 0), (5, 4352, 0)])
def test_matmul_forms(dev, fmt, M, N, offset):
    """offset: the weight (f16, q8) one element past an aligned address, which the row form does not take."""
    announce(f"matmul {fmt} M={M} N={N} offset={offset}")
    rng = np.random.default_rng(M + N)
    x = rng.standard_normal(N, dtype=np.float32)
    out = torch.full((M + 1,), 7.0, device=dev)
    if fmt == "f16":
        w = rng.standard_normal((M, N), dtype=np.float32).astype(np.float16).view(np.uint16)
        want = orc.matmul_quant(x, w, M, N)
        ops.matmul_quant_f16(up(x, dev), up(w, dev, offset), out, M, N)
    elif fmt == "q8":
        q = rng.integers(-128, 128, size=(M, N)).astype(np.int8)
        sc = (rng.random((M, N // 32)) * 0.002).astype(np.float16).view(np.uint16)
        want = orc.matmul_q8(x, q, sc, M, N)
        ops.matmul_q8(up(x, dev), up(q, dev, offset), up(sc, dev), out, M, N)
    else:
        words = rng.integers(0, 2**32, size=M * N // 8, dtype=np.uint64).astype(np.uint32)
        meta = rng.standard_normal((M, N // 256, 16)).astype(np.float16).view(np.uint16)
        want = orc.matmul_q4k(x, words, meta, M, N)
        ops.matmul_q4k(up(x, dev), up(words, dev), up(meta, dev), out, M, N)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(bits(out)[:M], want.view(np.uint32))
    assert float(out[M]) == 7.0


@pytest.mark.parametrize("size,offset", [(1, 0), (3, 1), (4095, 0), (32768, 0), (32769, 0), (40000, 1), (70001, 2)])
def test_argmax_forms(dev, size, offset):
    announce(f"argmax size={size} offset={offset}")
    rng = np.random.default_rng(size)
    x = rng.integers(-3, 9, size=size).astype(np.float32)  # many ties
    x[rng.integers(0, size, size=size // 5)] = np.nan
    res = torch.full((1,), -1, dtype=torch.int32, device=dev)
    ops.argmax(up(x, dev, offset), res, size)
    torch.cuda.synchronize()
    assert int(res.item()) == orc.argmax(x) == cf.argmax_rule(x)
