"""GPU parity of the engine's dispatches on both sides of the launch rules (gemma4-webgpu_amd/csrc/launch_rules.h): every
form evaluates the reference's f32 operations in the reference's order, so the bar is bit equality with the oracle."""
import numpy as np
import pytest
import torch

from conftest import announce
from g4attn import ops
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
