"""Rows that step by n and whose first column less the row index has one residue modulo n, whichever it is, are grouped by phase."""
import pytest
import torch

import acsr_helpers as A
from r_attention import RegularAttention, attention_with_grad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,w,s,stride", [(300, 40, 2, 2), (300, 41, 2, 2), (257, 17, 4, 4), (300, 33, 3, 3), (64, 9, 6, 1), (64, 8, 6, 6), (70, 9, 2, 2), (64, 9, 2, 1)])
def test_the_builders_report_the_stride(dev, L, w, s, stride):
    pat = A.dilated_pattern(L, w, s)
    dense = pat.device_mask(dev)
    for mask in (pat, dense, dense.cpu().numpy().tolist()):
        got = A.create_acsr(mask, 16, dev)
        assert int(got[3].splat_row_stride) == stride and int(got[3].splat_max_step) == s
    shifted = dense.clone()
    shifted[L // 2] = dense[L // 2 - 1]  # one row of another phase
    assert int(A.create_acsr(shifted, 16, dev)[3].splat_row_stride) == 1


def reference(q, k, v, grad, live):
    q, k, v = (t.double().cpu().requires_grad_(True) for t in (q, k, v))
    s = (q @ k.transpose(2, 3) * q.shape[-1] ** -0.5).masked_fill(~live, float("-inf"))
    out = torch.softmax(s, -1) @ v
    return [out.detach(), *torch.autograd.grad(out, (q, k, v), grad.double().cpu())]


# what the types give: probabilities and score gradients rounded once to 11 or 8 bits, sums in float32
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 5e-6), (torch.float16, 4e-3), (torch.bfloat16, 3e-2)])
@pytest.mark.parametrize("d,fused", [(64, True), (128, True), (80, False), (64, False)])
@pytest.mark.parametrize("L,w,s", [(300, 41, 2), (517, 17, 4), (300, 33, 3)])
def test_forward_and_gradients_of_odd_dilated_windows(dev, L, w, s, d, fused, dtype, tol):
    pat = A.dilated_pattern(L, w, s)
    g = torch.Generator().manual_seed(L + d)
    q, k, v, grad = (torch.randn(1, 2, L, d, generator=g).to(dtype).to(dev) for _ in range(4))
    want = reference(q, k, v, grad, pat.device_mask(dev).cpu() > 0)
    attn = RegularAttention(1, L, 2, d, [pat], 16, 16, dev, dtype, scale=d ** -0.5, fused=fused)
    if not fused:
        got = [attn([q, k.transpose(2, 3), v])]
    else:
        for t in (q, k, v):
            t.requires_grad_(True)
        out = attention_with_grad(q, k, v, attn)
        got = [out.detach(), *torch.autograd.grad(out, (q, k, v), grad)]
    for a, b in zip(got, want):
        assert float((a.double().cpu() - b).norm() / b.norm()) <= tol


def test_a_forward_without_a_plan_buffer_takes_masks_that_fit_only_ungrouped(dev):
    """985 row blocks fill the library's own buffer; grouped by phase the mask would need 988."""
    import _splat_hip as hip
    from r_attention import attention_plan
    from test_zz_no_alloc import forward_args
    L, d = 985 * 128, 64
    segs = A.create_acsr_segments([A.dilated_pattern(L, 9, 4)], 16, dev)
    arr = hip.seg_array(segs.seg_args(), L)
    assert arr[0].row_stride_hint == 4 and hip.lib().splat_attention_plan_bytes(arr, 1, L) > hip.STATIC_PLAN_BYTES
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(1, 1, L, d, generator=g).half().to(dev) for _ in range(3))
    got, want = torch.empty_like(q), torch.empty_like(q)
    args = lambda out: forward_args(q, k.transpose(2, 3), v, out, arr, 1, d ** -0.5)
    hip.check(hip.lib().splat_attention_fwd_noalloc(*args(got), hip.stream_ptr(dev)), "splat_attention_fwd_noalloc")
    plan = attention_plan(segs, L, dev)
    hip.check(hip.lib().splat_attention_fwd_planned(*args(want), plan.data_ptr(), plan.numel(), hip.stream_ptr(dev)), "splat_attention_fwd_planned")
    # (float16 probabilities of the two walks are rounded against different references: 2^-11 each)
    assert float((got.double() - want.double()).norm() / want.double().norm()) <= 1e-3
