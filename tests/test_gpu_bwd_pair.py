"""The backward's keys' side by pairs of wavefronts against float64 where its halves, stages and exchange can go wrong, and that a head's
gradients do not depend on how many others there are."""
import pytest
import torch

import acsr_helpers as A
from r_attention import RegularAttention, attention_with_grad

pytestmark = pytest.mark.gpu

MASKS = {
    "diagonal": lambda L: [A.causal_windowed_pattern(L, 0)],
    "causal": lambda L: [A.causal_windowed_pattern(L, 16)],
    "windowed": lambda L: [A.windowed_pattern(L, min(L - 1, 70))],
    "dilated": lambda L: [A.dilated_pattern(L, 5, 3)],
    "strided": lambda L: A.strided_patterns(L, 9, 7),
    "everything": lambda L: [A.causal_windowed_pattern(L, L - 1)],
}


def step(masks, q, k, v, grad, dev, dtype):
    B, H, L, d = q.shape
    q, k, v = (t.detach().clone().requires_grad_(True) for t in (q, k, v))
    attn = RegularAttention(B, L, H, d, masks, 16, 16, dev, dtype, scale=d ** -0.5)
    return torch.autograd.grad(attention_with_grad(q, k, v, attn), (q, k, v), grad)


@pytest.mark.parametrize("name", MASKS)
@pytest.mark.parametrize("L", [17, 33, 64, 65, 129, 200, 520])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [128, 64])
def test_against_float64(dev, name, L, dtype, d):
    masks, B, H = MASKS[name](L), 1, 2
    g = torch.Generator().manual_seed(L)
    q, k, v, grad = (torch.randn(B, H, L, d, generator=g).to(dtype) for _ in range(4))
    live = sum(m.device_mask(dev) for m in masks).cpu() > 0
    q64, k64, v64 = (t.double().requires_grad_(True) for t in (q, k, v))
    s = (q64 @ k64.transpose(2, 3) * d ** -0.5).masked_fill(~live, -1e300)
    out = torch.softmax(s, -1) * live.any(1)[:, None] @ v64
    want = torch.autograd.grad(out, (q64, k64, v64), grad.double())
    got = step(masks, q.to(dev), k.to(dev), v.to(dev), grad.to(dev), dev, dtype)
    # P and dS are rounded to the type once between the products, the sums are float32
    rel = {torch.float16: 2e-3, torch.bfloat16: 1e-2}[dtype]
    scale = max(float(w.norm()) for w in want)  # (a diagonal mask has dq = dk = 0)
    for a, w in zip(got, want):
        assert float((a.double().cpu() - w).norm()) <= rel * max(float(w.norm()), 0.1 * scale)


def test_a_head_s_bits_do_not_depend_on_the_launch(dev):
    """1024 heads of one row block, and one head more: the same bits for the heads that both have."""
    most, L, d, dtype = 1024, 128, 128, torch.bfloat16
    g = torch.Generator(device=dev).manual_seed(5)
    q, k, v, grad = (torch.randn(1, most + 1, L, d, generator=g, device=dev).to(dtype) for _ in range(4))
    masks = [A.windowed_pattern(L, 20)]
    a = step(masks, *(t[:, :most].contiguous() for t in (q, k, v, grad)), dev, dtype)
    b = step(masks, q, k, v, grad, dev, dtype)
    for x, y in zip(a, b):
        assert torch.equal(x, y[:, :most])
