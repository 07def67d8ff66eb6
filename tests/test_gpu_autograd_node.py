"""The autograd node of the native host path (csrc/host_ext.cpp) where a program does more than call backward: it must do what
the Python function that it stands in for does."""
import pytest
import torch
import torch.autograd.forward_ad as forward_ad

import acsr_helpers as A
from r_attention import RegularAttention, attention_with_grad

pytestmark = pytest.mark.gpu

B, H, L, D = 1, 2, 300, 64


def _module(dev, dtype=torch.bfloat16, scale=D ** -0.5):
    return RegularAttention(B, L, H, D, A.causal_windowed_pattern(L, 70), 16, 16, dev, dtype, scale=scale)


def _operands(dev, dtype=torch.bfloat16):
    g = torch.Generator(device="cpu").manual_seed(5)
    return [torch.randn(B, H, L, D, generator=g).to(dtype).to(dev).requires_grad_(True) for _ in range(3)]


@pytest.mark.parametrize("which", [0, 1, 2])
def test_a_tangent_is_refused_and_not_dropped(dev, which):
    attn, x = _module(dev), _operands(dev)
    with forward_ad.dual_level():
        x[which] = forward_ad.make_dual(x[which], torch.ones_like(x[which]))
        with pytest.raises(NotImplementedError, match="jvp"):
            attention_with_grad(*x, attn)
    with forward_ad.dual_level():  # the level alone is nothing to refuse
        assert attention_with_grad(*_operands(dev), attn).grad_fn.name() == "AttendBackward"
