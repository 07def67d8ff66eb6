"""The operators' kernels for head dimensions that pad their tiles and for rows of the compressed matrix that start anywhere,
against float64: 16-bit types, d in whole 16-byte pieces, odd row lengths, few and many row blocks."""
import pytest
import torch

import acsr_helpers as A
import r_sddmm
import r_spmm
from r_attention import RegularAttention

pytestmark = pytest.mark.gpu

SENTINEL = -77.0
MASKS = {
    "one": lambda L: [A.causal_windowed_pattern(L, 0)],
    "causal17": lambda L: [A.causal_windowed_pattern(L, 16)],
    "windowed129": lambda L: [A.windowed_pattern(L, 64)],
    "windowed301": lambda L: [A.windowed_pattern(L, 150)],
    "dilated": lambda L: [A.dilated_pattern(L, 41, 3)],
    "strided": lambda L: A.strided_patterns(L, 13, 7),
}
HALF_ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}  # of a value, rounded once from float32


def case(dev, name, B, H, L, d, dtype):
    masks = MASKS[name](L)
    g = torch.Generator().manual_seed(L + d)
    q, k, v = (torch.randn(B, H, L, d, generator=g).to(dtype) for _ in range(3))
    attn = RegularAttention(B, L, H, d, masks, 16, 16, dev, dtype, scale=d ** -0.5, fused=False)
    return masks, attn, q, k, v


def slots(attn, L):
    """(columns [L, T], live [L, T]) of the compressed rows."""
    cols, live = zip(*(r_sddmm.live_slot_columns(t[2].cpu(), t[3].cpu(), t[4].cpu(), int(t[5]), None if fc is None else fc.cpu())
                       for t, fc in zip(attn.segments.tuples, attn.segments.first_cols)))
    return torch.cat(cols, 1).clamp(0, L - 1), torch.cat(live, 1)


@pytest.mark.parametrize("name", MASKS)
@pytest.mark.parametrize("B,H,L", [(1, 2, 130), (1, 3, 333), (4, 16, 530)])
@pytest.mark.parametrize("dtype,d", [(torch.float16, 8), (torch.bfloat16, 24), (torch.float16, 32), (torch.float16, 64),
                                     (torch.bfloat16, 72), (torch.float16, 80), (torch.bfloat16, 96), (torch.bfloat16, 120),
                                     (torch.float16, 128)])
def test_operators_against_float64(dev, name, B, H, L, d, dtype):
    masks, attn, q, k, v = case(dev, name, B, H, L, d, dtype)
    T = attn.acsr_trailing_dim if len(masks) == 1 else attn.segments.T
    cols, live = slots(attn, L)
    scores = q.double() @ k.double().transpose(2, 3) * d ** -0.5
    want = scores.gather(3, cols.expand(B, H, L, T))
    lse = torch.logsumexp(scores.masked_fill(~(sum(m.device_mask(dev) for m in masks).cpu() > 0), float("-inf")), -1)
    qd, kd, vd = q.to(dev), k.to(dev).transpose(2, 3), v.to(dev)
    none = [None] * 4

    def sddmm(**kw):
        out = torch.full((B, H, L, T), SENTINEL, dtype=dtype, device=dev)
        r_sddmm.rsddmm_launcher(qd, kd, out, *none, T, None, None, None, None, 16, 16, scale=d ** -0.5, segments=attn.segments, **kw)
        return out
    got = sddmm()
    assert torch.all(got.cpu()[..., ~live] == SENTINEL), "dead slots must not be written"
    # float32 sums of d products of 16-bit values, then one rounding
    err = (got.double().cpu() - want).abs()[..., live]
    assert bool((err <= 1.01 * HALF_ULP[dtype] * want.abs()[..., live] + 1e-5).all())
    assert torch.equal(got, sddmm(plan=False))
    probs = sddmm(lse=lse.float().to(dev).contiguous())
    pw = torch.exp(want - lse[..., None])
    perr = (probs.double().cpu() - pw).abs()[..., live]
    assert bool((perr <= 1.01 * HALF_ULP[dtype] * pw[..., live] + 1e-5).all())
    # the product of the stored probabilities; dead slots hold anything
    given = torch.where(live.to(dev), probs, torch.full_like(probs, float("nan")))
    dense = torch.zeros(B, H, L, L, dtype=torch.float64)
    dense.scatter_add_(3, cols.expand(B, H, L, T), torch.where(live, probs.double().cpu(), torch.zeros(()).double()))
    ref = dense @ v.double()
    out = torch.full((B, H, L, d), SENTINEL, dtype=dtype, device=dev)
    r_spmm.rspmm_launcher(given, vd, out, *none, None, None, T, None, None, 16, 16, segments=attn.segments)
    oerr = (out.double().cpu() - ref).abs()
    assert bool((oerr <= 1.01 * HALF_ULP[dtype] * ref.abs() + 1e-5).all())


@pytest.mark.parametrize("d", [24, 80])
def test_padding_meets_no_infinity(dev, d):
    """An infinite key gives infinite scores at its column and leaves every other one finite: the padded part of the tiles
    multiplies nothing of it."""
    B, H, L = 1, 2, 200
    masks, attn, q, k, v = case(dev, "windowed129", B, H, L, d, torch.float16)
    k[:, :, 60] = float("inf")
    T = attn.acsr_trailing_dim
    cols, live = slots(attn, L)
    out = torch.zeros(B, H, L, T, dtype=torch.float16, device=dev)
    r_sddmm.rsddmm_launcher(q.abs().to(dev) + 1, k.to(dev).transpose(2, 3), out, *[None] * 4, T, None, None, None, None, 16, 16,
                            segments=attn.segments)
    got = out.cpu()
    hit = (cols == 60) & live
    assert bool((got[..., hit] == float("inf")).all()) and bool(torch.isfinite(got[..., live & ~hit]).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("L,d", [(1, 8), (63, 64), (64, 80), (65, 33), (131, 128)])
@pytest.mark.parametrize("lead", [0, 1, 3])
def test_transposed_keys_from_any_alignment(dev, L, d, lead, dtype):
    """K^T whose rows start ``lead`` elements into longer ones, whole pieces and remainders: the copy holds the same bits."""
    kT = torch.randn(2, 3, d, L + lead, generator=torch.Generator().manual_seed(L + d)).to(dtype).to(dev)[..., lead:]
    assert torch.equal(A.transpose_keys(kT), kT.transpose(2, 3).contiguous())


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("in_dt,out_dt", [(torch.float16, torch.float16), (torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16),
                                          (torch.float32, torch.float32)])
@pytest.mark.parametrize("L,T", [(1, 3), (5, 3), (21, 7), (16, 7), (21, 9), (13, 11), (40, 15), (100, 33), (65, 111), (67, 113), (203, 129), (259, 239), (300, 241)])
def test_softmax_of_rows_at_every_alignment(dev, L, T, in_dt, out_dt, in_place):
    """Rows of every chunk alignment up to the end of the buffer (the tensors fill their allocation's last chunk or not), with live rows, short ones, empty ones and one that is the type's
    lowest value throughout, against float64; dead slots keep what they held."""
    import r_softmax
    if in_place and in_dt != out_dt:
        pytest.skip("in place: one type")
    B, H = 1, 3
    g = torch.Generator().manual_seed(L + T)
    counts = torch.full((L,), float(T))
    counts[torch.rand(L, generator=g) < 0.3] = float(T // 2)
    counts[3::8], counts[5::11] = 0.0, 1.0
    x = (2 * torch.randn(B, H, L, T, generator=g)).to(in_dt)
    x[:, 1, 4 % L] = torch.finfo(in_dt).min
    live = torch.arange(T)[None, :] < counts[:, None]
    x = torch.where(live, x, torch.full_like(x, 55.0))
    want = torch.softmax(x.double().masked_fill(~live, float("-inf")), -1)
    cnt = counts.to(dev)
    xd = x.to(dev)
    out = xd if in_place else torch.full((B, H, L, T), 55.0, dtype=out_dt, device=dev)
    z = torch.zeros(L, device=dev)
    r_softmax.rsoftmax_launcher(xd, out, z, z, z, z, T, 256, cnt, (1, 1), 16)
    got = out.double().cpu()
    assert torch.all(got[..., ~live] == 55.0)
    keep = live.expand(B, H, L, T).clone()
    if in_dt != torch.float16:
        keep[:, 1, 4 % L] = False  # (a row below the kernel's -1e30 has no defined result; its neighbours do)
    tol = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 0.0}[out_dt] * 1.01
    bad = keep & ~((got - want).abs() <= tol * want + 1e-6)
    assert not bool(bad.any()), [(*i, float(got[tuple(i)]), float(want[tuple(i)])) for i in bad.nonzero().tolist()[:8]]


@pytest.mark.parametrize("d", [8, 64, 80, 96])
@pytest.mark.parametrize("B,H,L", [(1, 2, 130), (4, 16, 131), (2, 16, 256)])
def test_operators_with_the_keys_contiguous(dev, d, B, H, L):
    """K^T stored along the keys, on both sides of the lines at which it is turned first: as with K's rows contiguous, up to the
    order of the float32 additions (one ulp of the 16-bit scores)."""
    masks, attn, q, k, v = case(dev, "windowed129", B, H, L, d, torch.float16)
    outs = []
    for kT in (k.to(dev).transpose(2, 3), k.to(dev).transpose(2, 3).contiguous()):
        out = torch.full((B, H, L, attn.acsr_trailing_dim), SENTINEL, dtype=torch.float16, device=dev)
        r_sddmm.rsddmm_launcher(q.to(dev), kT, out, *[None] * 4, attn.acsr_trailing_dim, None, None, None, None, 16, 16, scale=d ** -0.5,
                                segments=attn.segments)
        outs.append(out.double().cpu())
    assert bool(((outs[0] - outs[1]).abs() <= 2.02 * HALF_ULP[torch.float16] * outs[0].abs() + 1e-5).all())
