"""GPU parity of the engine's dispatches on both sides of the launch rules (gemma4-webgpu_amd/csrc/launch_rules.h): every
form evaluates the reference's f32 operations in the reference's order, so the bar is bit equality with the oracle."""
import numpy as np
import pytest
import torch

from conftest import announce
from g4attn import ops
from helpers import cache_f16
from oracle import closed_form as cf
from oracle import oracle as orc
from test_gpu_engine_kernels import bits, up

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,seq", [(8, 512), (8, 513), (256, 513), (257, 600), (257, 706), (257, 707), (300, 100),
                                    (683, 4097), (682, 4097)])
def test_softmax_rule(dev, nh, seq):
    announce(f"softmax nh={nh} seq={seq}")
    x = np.random.default_rng(nh + seq).standard_normal((nh, seq), dtype=np.float32) * 4
    x[:, : seq // 5] = -1e30
    want = orc.softmax(x.ravel(), nh, seq)
    d = up(x, dev)
    ops.softmax(d, nh, seq)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(bits(d), want.view(np.uint32))


@pytest.mark.parametrize("nqh,nkh,hd,seq", [(8, 1, 256, 15), (8, 1, 256, 16), (8, 1, 512, 15), (8, 1, 512, 17), (1, 1, 64, 16),
                                            (264, 8, 256, 53), (264, 8, 256, 61), (264, 8, 512, 289), (264, 8, 512, 287)])
def test_attn_output_rule(dev, nqh, nkh, hd, seq):
    announce(f"attnOutput nqh={nqh} nkh={nkh} hd={hd} seq={seq}")
    vc = cache_f16(seq + hd, seq, nkh, hd)
    p = np.random.default_rng(seq).random((nqh, seq), dtype=np.float32) / seq
    p[:, : seq // 4] = 0.0
    want = orc.attn_output(p.ravel(), orc.f16_bits_to_f32(vc), nqh, nkh, hd, seq)
    out = torch.full((nqh * hd + 1,), 7.0, device=dev)
    ops.attn_output(up(p, dev), up(vc, dev), out, nqh, nkh, hd, seq)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(bits(out)[:-1], want.view(np.uint32))
    assert float(out[-1]) == 7.0


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("size", [1, 255, 256, 257, 511, 767, 768, 769])
def test_argmax_rule(dev, size, offset):
    announce(f"argmax size={size} offset={offset}")
    rng = np.random.default_rng(size)
    for trial in range(4):
        x = rng.integers(-2, 3, size=size).astype(np.float32)  # many ties
        if trial == 1:
            x[rng.integers(0, size, size=max(1, size // 3))] = np.nan
        if trial == 2:
            x[:] = -np.inf  # no candidate: index 0
        if trial == 3:
            x = np.where(x > 0, np.float32(0.0), np.float32(-0.0))  # zeros of both signs compare equal
        res = torch.full((1,), -1, dtype=torch.int32, device=dev)
        ops.argmax(up(x, dev, offset), res, size)
        torch.cuda.synchronize()
        assert int(res.item()) == orc.argmax(x) == cf.argmax_rule(x), (size, offset, trial)
