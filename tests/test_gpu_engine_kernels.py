"""GPU parity of the engine's own dispatches where their fast forms begin and end: attnScore's 64-row tiles,
softmax's register forms, attnOutput's 32-row blocks and 224-row rounds (blocks of zero products are skipped),
the matmuls' row form and argmax's batches. Every form evaluates the reference's f32 operations in the reference's
order, so the bar is bit equality with the oracle, which also covers the general forms on the other side of each rule.
"""
import numpy as np
import pytest
import torch

from conftest import announce
from g4attn import ops
from helpers import cache_f16
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


@pytest.mark.parametrize("nqh,nkh,hd,seq,win,offset", [
    (8, 1, 256, 1, 0, 0), (8, 1, 256, 63, 0, 0), (8, 1, 512, 64, 64, 0), (8, 1, 512, 65, 64, 0), (8, 1, 256, 200, 72, 0),
    (8, 1, 256, 200, 73, 0), (6, 2, 256, 130, 0, 0), (5, 1, 512, 193, 1, 0), (4, 4, 512, 100, 0, 0),
    (8, 1, 512, 2047, 0, 0), (8, 1, 256, 90, 40, 1), (8, 1, 320, 90, 40, 0)])
def test_attn_score_forms(dev, nqh, nkh, hd, seq, win, offset):
    announce(f"attnScore nqh={nqh} nkh={nkh} hd={hd} seq={seq} win={win} offset={offset}")
    kc = cache_f16(hd + seq, seq, nkh, hd)
    kc.reshape(-1)[::97] = np.resize(np.array([0x0001, 0x8000, 0x83FF, 0x0000], np.uint16), kc.reshape(-1)[::97].size)
    q = np.random.default_rng(seq).standard_normal(nqh * hd, dtype=np.float32) * 2
    q[::61] = np.resize(np.array([0.0, -0.0, 1e-40, -3e-39], np.float32), q[::61].size)
    want = orc.attn_score(q, orc.f16_bits_to_f32(kc), nqh, nkh, hd, seq, 0.5, win)
    sc = torch.full((nqh * seq,), float("nan"), device=dev)
    ops.attn_score(up(q, dev), up(kc, dev, offset), sc, nqh, nkh, hd, seq, 0.5, win)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(bits(sc), want.view(np.uint32))


@pytest.mark.parametrize("nh,seq", [(1, 1), (3, 255), (2, 257), (8, 1024), (8, 1025), (2, 4096), (2, 4097), (1, 16384),
                                    (2, 16385)])
def test_softmax_forms(dev, nh, seq):
    announce(f"softmax nh={nh} seq={seq}")
    x = np.random.default_rng(seq).standard_normal((nh, seq), dtype=np.float32) * 4
    x[:, : seq // 3] = -1e30  # rows before a window
    want = orc.softmax(x.ravel(), nh, seq)
    d = up(x, dev)
    ops.softmax(d, nh, seq)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(bits(d), want.view(np.uint32))


@pytest.mark.parametrize("nqh,nkh,hd,seq,zeros,special", [
    (8, 1, 256, 1, 0, False), (8, 1, 256, 31, 0, False), (2, 1, 64, 32, 0, False), (4, 2, 128, 33, 0, False),
    (8, 1, 512, 223, 100, False), (8, 1, 512, 224, 224, False), (8, 1, 512, 225, 224, False), (8, 1, 256, 449, 300, True),
    (8, 2, 256, 700, 650, True), (8, 1, 512, 2047, 0, False), (3, 1, 96, 300, 10, False)])
def test_attn_output_forms(dev, nqh, nkh, hd, seq, zeros, special):
    """`zeros` leading probabilities are 0 (whole blocks of zero products); special: V rows there hold infinities."""
    announce(f"attnOutput nqh={nqh} nkh={nkh} hd={hd} seq={seq} zeros={zeros} special={special}")
    rng = np.random.default_rng(seq + hd)
    vc = cache_f16(7 * seq + hd, seq, nkh, hd)
    p = rng.random((nqh, seq), dtype=np.float32) / seq
    p[:, :zeros] = 0.0
    p[:, seq // 2] = 0.0
    if special:
        vc[5, :, 3] = 0x7C00   # inf * 0 is NaN: the column's sum stays NaN
        vc[zeros - 1, :, 9] = 0xFC00
    with np.errstate(invalid="ignore"):
        want = orc.attn_output(p.ravel(), orc.f16_bits_to_f32(vc), nqh, nkh, hd, seq)
    out = torch.full((nqh * hd,), 7.0, device=dev)
    ops.attn_output(up(p, dev), up(vc, dev), out, nqh, nkh, hd, seq)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    nan = np.isnan(want)
    assert nan.any() == special and np.array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


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
