"""The float32 SDDMM and SpMM of up to 128 inner values or columns.  Operands are small whole numbers, so that every sum is exact whatever
its order, and results are compared for equality."""
import pytest
import torch

from oracle import splat_oracle as O
import acsr_helpers as A
import r_sddmm
import r_spmm
from test_gpu_operators import SENTINEL, _random_rows_mask, acsr_pair, live

pytestmark = pytest.mark.gpu

# row blocks of 64, tiles of 32 positions, subtiles of 16; rows that step differently, rows grouped by phase, empty rows
MASKS = {
    "one_row": lambda: O.create_causal_windowed_mask(1, 0),
    "block_64": lambda: O.create_causal_windowed_mask(64, 31),
    "block_65": lambda: O.create_windowed_mask(65, 16),
    "window_301": lambda: O.create_windowed_mask(333, 150),
    "blocked": lambda: O.create_blocked_mask(200, 33),
    "dilated_2": lambda: O.create_dilated_mask(300, 40, 2),
    "dilated_4_odd": lambda: O.create_dilated_mask(257, 17, 4),
    "ragged": lambda: _random_rows_mask(260, 5, [1], 70),
    "steps": lambda: _random_rows_mask(260, 6, [1, 2, 3], 50),
}


def whole(shape, seed):
    return torch.randint(-8, 9, shape, generator=torch.Generator().manual_seed(seed)).float()


@pytest.mark.parametrize("layout", ["rows", "keys", "keys_anywhere", "rows_anywhere"])
@pytest.mark.parametrize("d", [1, 32, 33, 64, 80, 96, 127, 128])
@pytest.mark.parametrize("name", list(MASKS))
def test_sddmm(dev, name, d, layout):
    mask = MASKS[name]()
    L = mask.shape[0]
    q, k = whole((2, 2, L, d), L + d), whole((2, 2, L, d), L + d + 1)
    acsr, acsr_np = acsr_pair(mask, 16, dev)
    want = O.sddmm(q, k.transpose(2, 3), acsr_np, first_col=O.row_extents(mask)[0])
    kT = k.to(dev).transpose(2, 3)
    if layout == "keys":
        kT = kT.contiguous()
    elif layout == "keys_anywhere":  # rows of K^T that start on any word
        kT = torch.cat([kT, kT[..., :1]], -1).contiguous()[..., :L]
    elif layout == "rows_anywhere":
        kT = torch.cat([k, k[..., :1]], -1).to(dev)[..., :d].transpose(2, 3)
    out = torch.full((2, 2, L, acsr[5]), SENTINEL, device=dev)
    r_sddmm.rsddmm_launcher(q.to(dev), kT, out, acsr[0], acsr[1], acsr[2], acsr[3], acsr[5], acsr[4], (1, 1), None, None, 16, 16)
    got, lv = out.cpu(), live(acsr_np)
    assert torch.equal(got[..., lv], want[..., lv])
    assert torch.all(got[..., ~lv] == SENTINEL)


@pytest.mark.parametrize("n_out", [1, 32, 33, 64, 80, 95, 128])
@pytest.mark.parametrize("name", list(MASKS))
def test_spmm(dev, name, n_out):
    mask = MASKS[name]()
    L = mask.shape[0]
    acsr, acsr_np = acsr_pair(mask, 16, dev)
    T, lv = acsr[5], live(acsr_np)
    p, v = whole((2, 2, L, T), L + n_out), whole((2, 2, L, n_out), L + n_out + 1)
    want = O.spmm(torch.where(lv, p, torch.zeros(())), v, acsr_np, first_col=O.row_extents(mask)[0])
    p = torch.where(lv, p, torch.full((), float("nan")))  # dead slots hold garbage
    for vd in (v.to(dev), torch.cat([v, v[..., :1]], -1).to(dev)[..., :n_out]):  # rows of V on 16-byte boundaries and anywhere
        out = torch.full((2, 2, L, n_out), float("nan"), device=dev)
        r_spmm.rspmm_launcher(p.to(dev), vd, out, acsr[0], acsr[1], acsr[2], acsr[3], acsr[6], acsr[7], T, acsr[4], (1, 1, 1), 16, 16)
        assert torch.equal(out.cpu(), want)


def test_two_segments_in_launches_that_share_tiles_out_and_ones_that_do_not(dev):
    L, d = 640, 48
    pats = A.strided_patterns(L, 48, 32)
    segs = A.create_acsr_segments(pats, 16, dev)
    union = torch.from_numpy(sum(O.create_strided_segment_masks(L, 48, 32)) > 0)
    q, k, v = (whole((1, 1, L, d), s) for s in (1, 2, 3))
    want = torch.where(union, (q @ k.transpose(2, 3)).remainder(7.0), torch.zeros(())) @ v  # (sums that float32 holds)
    for B, H in ((1, 1), (8, 16)):
        qd, kd, vd = (t.to(dev).expand(B, H, L, d).contiguous() for t in (q, k, v))
        out = torch.zeros(B, H, L, segs.T, device=dev)
        r_sddmm.rsddmm_launcher(qd, kd.transpose(2, 3), out, None, None, None, None, segs.T, None, None, None, None, 16, 16, segments=segs)
        res = torch.empty(B, H, L, d, device=dev)
        r_spmm.rspmm_launcher(out.remainder(7.0), vd, res, None, None, None, None, None, None, segs.T, None, None, 16, 16, segments=segs)
        assert torch.equal(res.cpu(), want.expand(B, H, L, d))


# 1024 row blocks of 64 rows of more than 600 slots at d <= 64 (450 for 33 to 56 values) go to the general kernel: both sides of each line
@pytest.mark.parametrize("layout", ["rows", "keys"])
@pytest.mark.parametrize("d,width,heads", [(32, 600, 64), (32, 601, 64), (64, 601, 63), (40, 450, 64), (40, 451, 64), (56, 451, 64), (57, 451, 64), (80, 601, 64)])
@pytest.mark.parametrize("step", [1, 2])
def test_sddmm_on_both_sides_of_the_general_kernel(dev, step, d, width, heads, layout):
    """Through the launcher's own path, which turns K along the keys for gathered masks where the general kernel runs."""
    L = 1024
    mask = O.create_dilated_mask(L, width, 2) if step == 2 else O.create_causal_windowed_mask(L, width - 1)
    acsr, acsr_np = acsr_pair(mask, 16, dev)
    q, k = whole((1, heads, L, d), heads).to(dev), whole((1, heads, L, d), d).to(dev)
    out = torch.full((1, heads, L, acsr[5]), SENTINEL, device=dev)
    kT = k.transpose(2, 3)
    r_sddmm.rsddmm_launcher(q, kT.contiguous() if layout == "keys" else kT, out, acsr[0], acsr[1], acsr[2], acsr[3], acsr[5], acsr[4], (1, 1), None, None, 16, 16)
    lv = live(acsr_np)
    for h in (0, heads // 2, heads - 1):
        want = O.sddmm(q[:, h:h + 1].cpu(), k[:, h:h + 1].cpu().transpose(2, 3), acsr_np, first_col=O.row_extents(mask)[0])
        got = out[:, h:h + 1].cpu()
        assert torch.equal(got[..., lv], want[..., lv]) and torch.all(got[..., ~lv] == SENTINEL)
