"""The 16-bit SDDMM of launches of few row blocks.  Operands are -1, 0 and 1, so that scores are whole numbers that bfloat16 holds, and
results are compared for equality: K as rows and along the keys, with the plan table and without, up to and beyond the launch sizes it takes."""
import pytest
import torch

from oracle import splat_oracle as O
import acsr_helpers as A
import r_sddmm
from test_gpu_operators import SENTINEL, acsr_pair, live
from test_gpu_operators_f32 import MASKS

pytestmark = pytest.mark.gpu


def signs(shape, seed, dtype):
    return torch.randint(-1, 2, shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("layout", ["rows", "keys", "keys_anywhere"])
@pytest.mark.parametrize("d", [8, 32, 40, 64, 96, 104, 128])
@pytest.mark.parametrize("name", list(MASKS))
def test_scores(dev, name, d, layout, dtype):
    mask = MASKS[name]()
    L = mask.shape[0]
    q, k = signs((1, 2, L, d), L + d, dtype), signs((1, 2, L, d), L + d + 1, dtype)
    acsr, acsr_np = acsr_pair(mask, 16, dev)
    want = O.sddmm(q.float(), k.float().transpose(2, 3), acsr_np, first_col=O.row_extents(mask)[0])
    kT = k.to(dev).transpose(2, 3)
    if layout == "keys":
        kT = kT.contiguous()
    elif layout == "keys_anywhere":
        kT = torch.cat([kT, kT[..., :1]], -1).contiguous()[..., :L]
    lv = live(acsr_np)
    for plan in (None, False, A.ACSRSegments.single(acsr[0], acsr[1], acsr[2], acsr[3], acsr[4], acsr[5]).plan(L, dev)):
        out = torch.full((1, 2, L, acsr[5]), SENTINEL, dtype=dtype, device=dev)
        r_sddmm.rsddmm_launcher(q.to(dev), kT, out, acsr[0], acsr[1], acsr[2], acsr[3], acsr[5], acsr[4], (1, 1), None, None, 16, 16, plan=plan)
        got = out.float().cpu()
        assert torch.equal(got[..., lv], want[..., lv])
        assert torch.all(got[..., ~lv] == SENTINEL)


# 4 half row blocks a head; 512 of them (K along the keys; 1024 where 64 < d <= 96), 640 and, d > 96, 256 (rows, with the plan table), 1024 to 4096 (the same, 70 or 55 slots): both sides of the lines, two segments too
@pytest.mark.parametrize("layout,heads", [("keys", 128), ("keys", 129), ("keys", 256), ("keys", 257), ("rows", 64), ("rows", 65), ("rows", 160), ("rows", 161), ("rows", 256), ("rows", 257), ("rows", 1024), ("rows", 1025)])
@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("d", [64, 80, 128])
def test_launch_sizes(dev, d, two, layout, heads):
    L = 250
    pats = A.strided_patterns(L, 40, 16) if two else [A.causal_windowed_pattern(L, 69)]
    segs = A.create_acsr_segments(pats, 16, dev)
    q, k = signs((1, heads, L, d), heads, torch.bfloat16), signs((1, heads, L, d), d, torch.bfloat16)
    kT = k.to(dev).transpose(2, 3)
    out = torch.full((1, heads, L, segs.T), SENTINEL, dtype=torch.bfloat16, device=dev)
    r_sddmm.rsddmm_launcher(q.to(dev), kT.contiguous() if layout == "keys" else kT, out, None, None, None, None, segs.T, None, None, None,
                            None, 16, 16, segments=segs)
    dense = q.float() @ k.float().transpose(2, 3)
    masks = O.create_strided_segment_masks(L, 40, 16) if two else [O.create_causal_windowed_mask(L, 69)]
    want = torch.cat([O.compress(dense, O.create_acsr(m, 16), first_col=O.row_extents(m)[0], fill=SENTINEL) for m in masks], -1)
    assert torch.equal(out.float().cpu(), want)


@pytest.mark.parametrize("width", [17, 40, 41])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_short_rows_in_launches_that_fill_the_chip(dev, d, width):
    L, heads = 250, 300
    acsr, acsr_np = acsr_pair(O.create_causal_windowed_mask(L, width - 1), 16, dev)
    q, k = signs((1, heads, L, d), heads, torch.float16), signs((1, heads, L, d), d, torch.float16)
    out = torch.full((1, heads, L, acsr[5]), SENTINEL, dtype=torch.float16, device=dev)
    r_sddmm.rsddmm_launcher(q.to(dev), k.to(dev).transpose(2, 3), out, acsr[0], acsr[1], acsr[2], acsr[3], acsr[5], acsr[4], (1, 1), None, None, 16, 16)
    want, lv, got = O.sddmm(q.float(), k.float().transpose(2, 3), acsr_np, first_col=[0] * L), live(acsr_np), out.float().cpu()
    assert torch.equal(got[..., lv], want[..., lv]) and torch.all(got[..., ~lv] == SENTINEL)


# half row blocks on both sides of every line of the launcher: rows of up to 256 slots, 300 (512 of one segment) and 450 (128 at d = 64, 256, 512 of two segments)
@pytest.mark.parametrize("probabilities", [False, True])
@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("d", [64, 96, 128])
@pytest.mark.parametrize("width,heads", [(39, 3), (39, 40), (70, 12), (70, 30), (70, 75), (70, 82), (300, 10), (300, 17), (300, 37), (300, 64), (300, 65),
                                         (450, 15), (450, 17), (450, 37), (450, 65)])
def test_the_plan_table_changes_no_bit(dev, width, heads, d, two, probabilities):
    """Rows of K, operands whose sums round, scores and probabilities."""
    L = 500
    pats = A.strided_patterns(L, width - 20, 32) if two else [A.causal_windowed_pattern(L, width - 1)]
    segs = A.create_acsr_segments(pats, 16, dev)
    g = torch.Generator(device=dev).manual_seed(width + heads)
    q, k = (torch.randn(1, heads, L, d, generator=g, device=dev).to(torch.bfloat16) for _ in range(2))
    lse = torch.randn(1, heads, L, generator=g, device=dev) + 20.0 if probabilities else None
    got = []
    for plan in (segs.plan(L, dev), False, None):
        out = torch.full((1, heads, L, segs.T), SENTINEL, dtype=torch.bfloat16, device=dev)
        r_sddmm.rsddmm_launcher(q, k.transpose(2, 3), out, None, None, None, None, segs.T, None, None, None, None, 16, 16, scale=0.3, segments=segs,
                                lse=lse, plan=plan)
        got.append(out)
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
