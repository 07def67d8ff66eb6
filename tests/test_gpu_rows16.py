"""The 16-bit forward of 16 rows a wavefront (launches of few row blocks) against float64 where its tiles can go wrong, and the
two sides of the line at which the dispatch changes kernels against each other."""
import pytest
import torch

import acsr_helpers as A
from r_attention import RegularAttention

pytestmark = pytest.mark.gpu

MASKS = {
    "diagonal": lambda L: [A.causal_windowed_pattern(L, 0)],
    "causal": lambda L: [A.causal_windowed_pattern(L, 16)],
    "windowed": lambda L: [A.windowed_pattern(L, 70)],
    "dilated": lambda L: [A.dilated_pattern(L, 40, 3)],
    "strided": lambda L: A.strided_patterns(L, 9, 7),
    "far only": lambda L: A.strided_patterns(L, 9, 7)[1:],  # the first rows hold nothing
}


def want(q, k, v, masks, dev):
    live = sum(m.device_mask(dev) for m in masks).cpu() > 0
    s = (q.double() @ k.double().transpose(2, 3) * q.shape[-1] ** -0.5).masked_fill(~live, float("-inf"))
    p = torch.where(live.any(1)[:, None], torch.softmax(s, -1), torch.zeros_like(s))
    return p @ v.double()


@pytest.mark.parametrize("name", MASKS)
@pytest.mark.parametrize("L", [17, 64, 65, 129, 200, 520])
@pytest.mark.parametrize("dtype,d", [(torch.float16, 64), (torch.bfloat16, 128)])
def test_against_float64(dev, name, L, dtype, d):
    masks, B, H = MASKS[name](L), 2, 2
    g = torch.Generator().manual_seed(L + d)
    q, k, v = (torch.randn(B, H, L, d, generator=g).to(dtype) for _ in range(3))
    ref = want(q, k, v, masks, dev)
    attn = RegularAttention(B, L, H, d, masks, 16, 16, dev, dtype, scale=d ** -0.5)
    for kT in (k.to(dev).transpose(2, 3), k.to(dev).transpose(2, 3).contiguous()):
        got = attn([q.to(dev), kT, v.to(dev)]).double().cpu()
        assert float((got - ref).norm() / ref.norm()) <= (1.5e-3 if dtype == torch.float16 else 8e-3)
        assert float((got - ref).abs().max()) <= (8e-3 if dtype == torch.float16 else 4e-2)


@pytest.mark.parametrize("d,most", [(64, 384), (128, 192)])
def test_both_sides_of_the_line(dev, d, most):
    """`most` heads of one row block go to this kernel, one head more to the other: the shared heads agree."""
    L, dtype = 128, torch.bfloat16
    g = torch.Generator(device=dev).manual_seed(d)
    q, k, v = (torch.randn(1, most + 1, L, d, generator=g, device=dev).to(dtype) for _ in range(3))
    outs = []
    for H in (most, most + 1):
        attn = RegularAttention(1, L, H, d, A.windowed_pattern(L, 20), 16, 16, dev, dtype, scale=d ** -0.5)
        outs.append(attn([q[:, :H], k[:, :H].transpose(2, 3), v[:, :H]]).float())
    assert float((outs[0] - outs[1][:, :most]).norm() / outs[0].norm()) <= 4e-3
