"""K^T with the keys contiguous whose rows start anywhere, read where it lies: bit for bit what rows of the same keys give, at lengths
around the edges of pieces and tiles, at odd strides and addresses, and up to the last byte of its memory."""
import ctypes

import pytest
import torch

import _splat_hip as hip
import acsr_helpers as A
from r_attention import RegularAttention

pytestmark = pytest.mark.gpu

TYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def heads(more, dtype, d, L):
    """Three, or as many as 16 rows a wavefront take in 16-bit types (193 to 320 row blocks in two batches, 129 to 192 at d = 128) and more than the
    64 row blocks of the float32 kernel of shared keys."""
    return 3 if not more else (155 if d == 64 and dtype != "f32" else 94) // -(-L // 128)


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("L", [8, 9, 15, 63, 65, 130, 201, 519])
@pytest.mark.parametrize("more", [False, True])
def test_equals_rows_of_keys(dev, dtype, d, L, more):
    B, H, dt = 2, heads(more, dtype, d, L), TYPES[dtype]
    masks = [A.causal_windowed_pattern(L, 33)] if L % 2 else [A.windowed_pattern(L, 70)]
    attn = RegularAttention(B, L, H, d, masks, 16, 16, dev, dt, scale=d ** -0.5)
    g = torch.Generator(device=dev).manual_seed(L + d)
    q, k, v = (torch.randn(B, H, L, d, generator=g, device=dev).to(dt) for _ in range(3))
    first = attn([q, k.transpose(2, 3), v]).clone()
    want = attn([q, k.transpose(2, 3), v]).clone()
    assert torch.equal(first, want) and 0 < attn._live_percent <= 75
    # as it is stored by a contiguous copy: the last row ends where its memory ends
    whole = torch.empty(B * H * d * L, dtype=dt, device=dev)
    exact = whole.view(B, H, d, L)
    exact.copy_(k.transpose(2, 3))
    assert torch.equal(attn([q, exact, v]), want)
    # a part of longer rows, from an odd element on; what lies around it must not matter
    long = torch.full((B, H, d, L + 7), float("nan"), dtype=dt, device=dev)
    part = long[..., 3:3 + L]
    part.copy_(k.transpose(2, 3))
    assert torch.equal(attn([q, part, v]), want)


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("L", [201, 519])
@pytest.mark.parametrize("more", [False, True])
def test_two_segments(dev, dtype, d, L, more):
    """A window and a band 60 to 80 keys before it: walks that change segments, the second of which begins with rows of nothing."""
    B, H, dt = 2, heads(more, dtype, d, L), TYPES[dtype]
    at = torch.arange(L)
    back = at[:, None] - at[None, :]
    masks = [((back >= lo) & (back <= hi)).to(torch.uint8).to(dev) for lo, hi in ((0, 33), (60, 80))]
    attn = RegularAttention(B, L, H, d, masks, 16, 16, dev, dt, scale=d ** -0.5)
    g = torch.Generator(device=dev).manual_seed(L + d)
    q, k, v = (torch.randn(B, H, L, d, generator=g, device=dev).to(dt) for _ in range(3))
    want = attn([q, k.transpose(2, 3), v]).clone()
    live = sum(masks).cpu() > 0
    s = (q[:, :3].double() @ k[:, :3].double().transpose(2, 3) * d ** -0.5).cpu().masked_fill(~live, float("-inf"))
    assert float((want[:, :3].double().cpu() - torch.softmax(s, -1) @ v[:, :3].double().cpu()).abs().max()) <= (1e-5 if dt == torch.float32 else 0.04)
    assert torch.equal(attn([q, k.transpose(2, 3).contiguous(), v]), want)
    long = torch.full((B, H, d, L + 7), float("nan"), dtype=dt, device=dev)
    part = long[..., 3:3 + L]
    part.copy_(k.transpose(2, 3))
    assert torch.equal(attn([q, part, v]), want)


@pytest.mark.parametrize("blocks,ran", [(128, True), (129, False)])
def test_launches_that_copy_whole_pieces_refuse(dev, blocks, ran):
    L, d, dt = 121, 64, torch.bfloat16
    attn = RegularAttention(1, L, blocks, d, A.windowed_pattern(L, L), 16, 16, dev, dt, scale=1.0)
    q, v = (torch.randn(1, blocks, L, d, device=dev).to(dt) for _ in range(2))
    kT = torch.randn(1, blocks, d, L, device=dev).to(dt)
    want = attn([q, kT.transpose(2, 3).contiguous().transpose(2, 3), v]).clone()
    assert torch.equal(attn([q, kT, v]), want)  # through the transposing copy where the kernel refuses
    out, arr, plan = torch.zeros_like(q), attn.segments.seg_array(L), attn._plan
    rc = hip.lib().splat_attention_fwd_keys(q.data_ptr(), *q.stride()[:3], kT.data_ptr(), *kT.stride()[:3], v.data_ptr(), *v.stride()[:3],
                                            out.data_ptr(), *out.stride()[:3], arr, 1, 1, blocks, L, d, ctypes.c_float(1.0),
                                            hip.dtype_code(dt), plan.data_ptr(), plan.numel() * plan.element_size(), None, 0,
                                            hip.stream_ptr(dev))
    torch.cuda.synchronize()
    assert (rc == 0) == ran and bool((out == 0).all()) != ran
    assert not ran or torch.equal(out, want)
