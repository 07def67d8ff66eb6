"""The forwards whose wavefronts share the keys of their rows (launches of few row blocks), against float64 around the numbers of tiles
at which its wavefronts run out of work, get a second tile, or leave the end to fewer of them; with a plan and without."""
import pytest
import torch

import acsr_helpers as A
from r_attention import RegularAttention, attention_launcher

pytestmark = pytest.mark.gpu


# 16-bit types: probabilities are rounded to the type once, half an ulp of it (2^-11, 2^-8), relative.  float32: products are off by
# less than 2^-24 of theirs, and so is every addition; four times what five of them in a row leave
BOUNDS = {torch.float16: 5e-4, torch.bfloat16: 4e-3, torch.float32: 1.2e-6}


def band(L, lo, hi, dev):
    back = torch.arange(L)[:, None] - torch.arange(L)[None, :]
    return ((back >= lo) & (back <= hi)).to(torch.uint8).to(dev)


# 32 rows of a causal window of w see w + 31 positions, of which the walk may begin 7 early: 1, 2, 3, 4, 5, 8, 9, 16, 17 tiles of 32
MASKS = {f"causal {w}": (lambda w: lambda L, dev: [A.causal_windowed_pattern(L, w - 1)])(w) for w in (1, 2, 34, 65, 90, 98, 130, 218, 226, 474, 490)}
MASKS |= {
    "dilated": lambda L, dev: [A.dilated_pattern(L, 50, 3)],
    "strided": lambda L, dev: A.strided_patterns(L, 40, 16),             # a second segment of periodic columns
    "bands": lambda L, dev: [band(L, 0, 40, dev), band(L, 200, 330, dev)],  # a second segment that begins with rows of nothing
    "far only": lambda L, dev: A.strided_patterns(L, 9, 7)[1:],           # the first rows hold nothing
}


@pytest.mark.parametrize("name", MASKS)
@pytest.mark.parametrize("few", [True, False])  # eight and four wavefronts of 32 rows (16-bit types), four of 16 and of 32 (float32)
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("L", [1000, 1001])  # (K^T is read where it lies: by pieces, and, in the native call, from rows that start anywhere)
@pytest.mark.parametrize("dtype", BOUNDS)
def test_against_float64(dev, name, few, dtype, d, L):
    B = 1
    H = 3 if few else 6 if dtype == torch.float32 else 12
    masks = MASKS[name](L, dev)
    g = torch.Generator().manual_seed(d + H)
    q, k, v = (torch.randn(B, H, L, d, generator=g).to(dtype).to(dev) for _ in range(3))
    live = sum(m if torch.is_tensor(m) else m.device_mask(dev) for m in masks) > 0
    s = (q.double() @ k.double().transpose(2, 3) * d ** -0.5).masked_fill(~live, float("-inf"))
    p = torch.where(live.any(1)[:, None], torch.softmax(s, -1), torch.zeros_like(s))
    ref = p @ v.double()
    attn = RegularAttention(B, L, H, d, masks, 16, 16, dev, dtype, scale=d ** -0.5)
    first = attn([q, k.transpose(2, 3), v]).clone()
    for kT in (k.transpose(2, 3), k.transpose(2, 3).contiguous()):
        got, lse = attn.forward_with_stats([q, kT, v])
        assert float((got.double() - ref).norm() / ref.norm()) <= BOUNDS[dtype]
        assert torch.allclose(lse.double().view(B, H, L), torch.logsumexp(s, -1).nan_to_num(neginf=float("inf")), atol=2e-6 * d, rtol=1e-6)
        assert float((attn([q, kT, v]).double() - ref).norm() / ref.norm()) <= BOUNDS[dtype]
    # without a plan the workgroups find the same walks (the hint chooses the kernel in either)
    bare = attention_launcher(q, k.transpose(2, 3), v, torch.empty_like(q), attn.segments, attn.scale, live_percent=attn._live_percent)
    assert torch.equal(bare, first)


@pytest.mark.parametrize("dtype,d", [(torch.float16, 64), (torch.bfloat16, 128), (torch.float32, 64), (torch.float32, 128)])
def test_values_that_no_row_sees_do_not_matter(dev, dtype, d):
    """A cache that is filled up to row n, NaN behind: the rows up to there are what they are without it."""
    L, n, B, H = 512, 320, 1, 2
    g = torch.Generator(device=dev).manual_seed(d)
    q, k, v = (torch.randn(B, H, L, d, generator=g, device=dev).to(dtype) for _ in range(3))
    attn = RegularAttention(B, L, H, d, A.causal_windowed_pattern(L, 99), 16, 16, dev, dtype, scale=d ** -0.5)
    want = attn([q, k.transpose(2, 3), v])[:, :, :n].clone()
    k[:, :, n:], v[:, :, n:] = float("nan"), float("nan")
    assert torch.equal(attn([q, k.transpose(2, 3), v])[:, :, :n], want)


@pytest.mark.parametrize("H,kt,same", [(224, False, True), (225, False, False), (192, True, True), (193, True, False)])
def test_the_line_at_d64(dev, H, kt, same):
    """Launches of 129 row blocks and more come here where some of the walk is dead; equal bits say which kernel ran."""
    L, d, dtype = 128, 64, torch.bfloat16
    g = torch.Generator(device=dev).manual_seed(H)
    q, k, v = (torch.randn(1, H, L, d, generator=g, device=dev).to(dtype) for _ in range(3))
    attn = RegularAttention(1, L, H, d, A.causal_windowed_pattern(L, 99), 16, 16, dev, dtype, scale=d ** -0.5)
    whole = attn([q, k.transpose(2, 3).contiguous() if kt else k.transpose(2, 3), v]).clone()
    few = RegularAttention(1, L, 100, d, A.causal_windowed_pattern(L, 99), 16, 16, dev, dtype, scale=d ** -0.5)
    part = few([q[:, :100], k[:, :100].transpose(2, 3), v[:, :100]])
    assert torch.equal(whole[:, :100], part) == same
    assert float((whole[:, :100].float() - part.float()).norm() / part.float().norm()) <= 4e-3


@pytest.mark.parametrize("kt", [False, True])
@pytest.mark.parametrize("d", [64, 128])
def test_float32_scores_have_the_bits_of_larger_launches(dev, d, kt):
    """The statistic of a row of one key is its score (the scale makes the exponents' factor 1: no other rounding), which the backward
    takes again: the same bits whichever kernel computed it."""
    L, H, ln2 = 300, 70, 0.6931471824645996
    g = torch.Generator(device=dev).manual_seed(d)
    q, k, v = (torch.randn(1, H, L, d, generator=g, device=dev) for _ in range(3))

    def statistic(heads):
        attn = RegularAttention(1, L, heads, d, A.causal_windowed_pattern(L, 0), 16, 16, dev, torch.float32, scale=ln2)
        kT = k[:, :heads].transpose(2, 3)
        return attn.forward_with_stats([q[:, :heads], kT.contiguous() if kt else kT, v[:, :heads]])[1].clone()
    want = statistic(H)  # (210 row blocks; then 9 and 36: workgroups of 16 and of 32 rows)
    assert torch.equal(statistic(3), want[:, :3]) and torch.equal(statistic(12), want[:, :12])
