"""The 16-bit forward of launches that leave the chip part idle (wavefronts that share the keys of 32 rows, and, of more row blocks, 16 rows a
wavefront) against float64 where its tiles can go wrong, and the two sides of the lines at which the dispatch changes kernels against each other."""
import pytest
import torch

import _splat_hip as hip
import acsr_helpers as A
from r_attention import RegularAttention, attention_launcher

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


def copies(masks, L, heads, d, dev):
    segs = A.create_acsr_segments(masks, 16, dev)
    of_head = hip.lib().splat_attention_plan_bytes(segs.seg_array(L), len(segs), L) // (2 * len(segs) * (5 + 128) * 16)
    n = (310 if d == 64 else 190) // (of_head * heads)
    assert (224 if d == 64 else 128) < n * of_head * heads <= (320 if d == 64 else 192)
    return n


@pytest.mark.parametrize("name", MASKS)
@pytest.mark.parametrize("L", [17, 64, 65, 129, 200, 520])
@pytest.mark.parametrize("dtype,d", [(torch.float16, 64), (torch.bfloat16, 128)])
@pytest.mark.parametrize("blocks", ["few", "more"])
def test_against_float64(dev, name, L, dtype, d, blocks):
    """`more`: as many copies of the heads as take the launch between the lines of the two kernels' (225 to 320 row blocks; 129 to 192 at d = 128)."""
    masks, B, H = MASKS[name](L), 2, 2
    g = torch.Generator().manual_seed(L + d)
    q, k, v = (torch.randn(B, H, L, d, generator=g).to(dtype) for _ in range(3))
    ref = want(q, k, v, masks, dev)
    n = copies(masks, L, B * H, d, dev) if blocks == "more" else 1
    attn = RegularAttention(B, L, H * n, d, masks, 16, 16, dev, dtype, scale=d ** -0.5)
    q, k, v = (t.repeat(1, n, 1, 1).to(dev) for t in (q, k, v))
    for kT in (k.transpose(2, 3), k.transpose(2, 3).contiguous()):
        got = attn([q, kT, v])
        assert blocks == "few" or 0 < attn._live_percent <= 75
        parts = got.chunk(n, 1)
        assert all(torch.equal(parts[0], x) for x in parts[1:])
        got = parts[0].double().cpu()
        assert float((got - ref).norm() / ref.norm()) <= (1.5e-3 if dtype == torch.float16 else 8e-3)
        assert float((got - ref).abs().max()) <= (8e-3 if dtype == torch.float16 else 4e-2)


@pytest.mark.parametrize("d,most,mask,percent", [(64, 320, A.windowed_pattern(128, 20), 30), (128, 192, A.windowed_pattern(128, 20), 30),
                                                 (64, 128, A.blocked_pattern(128, 128), 100), (128, 128, A.blocked_pattern(128, 128), 100)])
def test_both_sides_of_the_line(dev, d, most, mask, percent):
    """`most` heads of one row block go to one kernel, one head more to the next (16 rows a wavefront up to 320 or 192, shared keys up to 128
    where the walk is live throughout): the shared heads agree.  The line depends on how much of the walk is live; the module's first call (the launcher) and the next (native) take the same side."""
    L, dtype = 128, torch.bfloat16
    g = torch.Generator(device=dev).manual_seed(d)
    q, k, v = (torch.randn(1, most + 1, L, d, generator=g, device=dev).to(dtype) for _ in range(3))
    outs = []
    for H in (most, most + 1):
        attn = RegularAttention(1, L, H, d, mask, 16, 16, dev, dtype, scale=d ** -0.5)
        x = [q[:, :H], k[:, :H].transpose(2, 3), v[:, :H]]
        first = attn(x).clone()
        assert attn._live_percent == percent
        # the kernels differ in the order of their additions: equal bits say which one ran
        kinds = [attention_launcher(*x, torch.empty_like(first), attn.segments, attn.scale, attn._plan, live_percent=p) for p in (1, 100)]
        assert torch.equal(first, attn(x)) and torch.equal(first, attn.forward_with_stats(x)[0])
        assert torch.equal(first, kinds[0] if percent <= 75 else kinds[1])
        assert torch.equal(*kinds) == (H <= 128 or H > (320 if d == 64 else 192))
        outs.append(first.float())
    assert float((outs[0] - outs[1][:, :most]).norm() / outs[0].norm()) <= 4e-3
    assert not torch.equal(outs[0], outs[1][:, :most])


@pytest.mark.parametrize("L,masks", [(700, lambda L: [A.causal_windowed_pattern(L, 199)]), (300, lambda L: [A.dilated_pattern(L, 40, 3)]),
                                     (640, lambda L: [A.blocked_pattern(L, 128)]), (777, lambda L: A.strided_patterns(L, 64, 32))])
def test_live_percent_is_what_the_masks_say(dev, L, masks):
    """Live entries over the positions of the tiles that each block of 128 rows walks (64 positions each; dense runs start on a
    multiple of 64, gathered ones at the block's first column), rounded up."""
    segs = A.create_acsr_segments(masks(L), 16, dev)
    assert segs.live_percent(L, dev) == 0
    segs.plan(L, dev)
    rs = {int(t[3].splat_row_stride) for t in segs.tuples}
    rs = rs.pop() if len(rs) == 1 else 1
    live = walked = 0
    for m, t in zip(masks(L), segs.tuples):
        dm, step = m.device_mask(dev).cpu() > 0, int(t[3].splat_max_step)
        live += int(dm.sum())
        for b in range(-(-L // (128 * rs)) * rs):
            r0 = b // rs * 128 * rs + b % rs
            cols = torch.nonzero(dm[r0:r0 + 128 * rs:rs].any(0)).flatten()
            if cols.numel():
                c0 = int(cols[0]) if step > 1 else int(cols[0]) // 64 * 64
                walked += -(-((int(cols[-1]) - c0) // step + 1) // 64) * 64 * 128
    assert segs.live_percent(L, dev) == -(-100 * live // walked)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("layout", ["rows", "keys"])
def test_rows_too_far_apart_for_32_bit_offsets(dev, dtype, layout):
    """A few rows of V (and K) 16 MB apart: the kernels of shared keys, whose offsets do not reach, leave such launches to the others."""
    L, d = 150, 64
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(1, 1, L, d, generator=g).to(dtype) for _ in range(3))
    masks = [A.causal_windowed_pattern(L, 40)]
    ref = want(q, k, v, masks, dev)
    step = (1 << 24) // torch.finfo(dtype).bits * 8

    def apart(t):
        far = torch.empty((L - 1) * step + d, dtype=dtype, device=dev).as_strided((1, 1, L, d), (0, 0, step, 1))
        return far.copy_(t)
    attn = RegularAttention(1, L, 1, d, masks, 16, 16, dev, dtype, scale=d ** -0.5)
    kT = k.to(dev).transpose(2, 3).contiguous() if layout == "keys" else apart(k).transpose(2, 3)
    far_v = apart(v)
    for _ in range(2):  # (the launcher, the native call)
        got = attn([q.to(dev), kT, far_v]).double().cpu()
        assert float((got - ref).norm() / ref.norm()) <= (8e-3 if dtype == torch.bfloat16 else 1e-6)
