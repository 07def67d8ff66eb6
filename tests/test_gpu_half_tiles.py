"""Wavefronts of 32 rows whose spans begin or end inside a tile of 64 positions, in launches that fill the chip: the forward and the
gradients against float64 where one half of a tile is left out, the other one, neither, and where a row has nothing at all."""
import pytest
import torch

import acsr_helpers as A
from r_attention import RegularAttention, attention_with_grad

pytestmark = pytest.mark.gpu

MASKS = {
    "one half": lambda L: [A.causal_windowed_pattern(L, 0)],
    "a half and a column": lambda L: [A.causal_windowed_pattern(L, 32)],
    "to the tile's end": lambda L: [A.windowed_pattern(L, 16)],
    "over the tile's end": lambda L: [A.causal_windowed_pattern(L, 65)],
    "dilated": lambda L: [A.dilated_pattern(L, 33, 3)],
    "whole halves": lambda L: [A.blocked_pattern(L, 32)],
    "far only": lambda L: A.strided_patterns(L, 9, 7)[1:],  # the first rows hold nothing
    "strided": lambda L: A.strided_patterns(L, 40, 5),
}


@pytest.mark.parametrize("name", MASKS)
@pytest.mark.parametrize("L", [137, 200])
@pytest.mark.parametrize("dtype,d", [(torch.float16, 64), (torch.bfloat16, 64), (torch.bfloat16, 128)])
def test_against_float64(dev, name, L, dtype, d):
    masks, H, few = MASKS[name](L), 520, 2  # two row blocks a head: more than 1024, the kernels of large launches
    g = torch.Generator(device=dev).manual_seed(L + d)
    q, k, v, grad = (torch.randn(1, H, L, d, generator=g, device=dev).to(dtype) for _ in range(4))
    attn = RegularAttention(1, L, H, d, masks, 16, 16, dev, dtype, scale=d ** -0.5)
    leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
    out = attention_with_grad(*leaves, attn)
    got = [out, *torch.autograd.grad(out, leaves, grad)]
    keys = attn([q, k.transpose(2, 3).contiguous(), v])  # K^T with the keys contiguous: tiles read by columns
    live = sum(m.device_mask(dev) for m in masks).cpu() > 0
    refs = [t[:, :few].cpu().double().requires_grad_(True) for t in (q, k, v)]
    s = (refs[0] @ refs[1].transpose(2, 3) * d ** -0.5).masked_fill(~live, -1e300)
    ref = torch.softmax(s, -1) * live.any(1)[:, None] @ refs[2]
    want = [ref.detach(), *torch.autograd.grad(ref, refs, grad[:, :few].cpu().double())]
    # P and dS are rounded to the type once between the products, the sums are float32
    rel = {torch.float16: 2e-3, torch.bfloat16: 1e-2}[dtype]
    scale = max(float(w.norm()) for w in want)  # (a diagonal mask has dq = dk = 0)
    for a, w in zip([*got, keys], [*want, ref.detach()]):
        assert float((a[:, :few].double().cpu() - w).norm()) <= rel * max(float(w.norm()), 0.1 * scale)
