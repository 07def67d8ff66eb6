"""The three operators in one launch (splat_operators) against the three calls, bit for bit where those add in its order, and against float64: rows at the edges of what a row of
LDS holds, row blocks that interleave, two segments, rows whose steps differ, heads that are padded, K along the keys, sequences that end
inside a workgroup and inside a wavefront's rows."""
import ctypes

import pytest
import torch

import acsr_helpers as A
import _splat_hip as hip
from r_sddmm import live_slot_columns
from test_gpu_operators import SENTINEL

pytestmark = pytest.mark.gpu


def _steps_differ(L):
    """Rows of 0 to 9 slots whose steps are 1, 2 and 3 in turns: no walk in which positions are slots."""
    mask = torch.zeros(L, L, dtype=torch.uint8)
    for i in range(L):
        n, step = i % 10, 1 + i % 3
        for t in range(n):
            if i + step * t < L:
                mask[i, i + step * t] = 1
    return mask


MASKS = {"1": lambda L: A.causal_windowed_pattern(L, 0), "7": lambda L: A.causal_windowed_pattern(L, 6),
         **{str(w): (lambda w: lambda L: A.causal_windowed_pattern(L, w - 1))(w) for w in (33, 64, 65, 128, 129, 200, 256, 257, 509, 512)},
         "windowed 257": lambda L: A.windowed_pattern(L, 128), "blocked 64": lambda L: A.blocked_pattern(L, 64),
         "blocked 512": lambda L: A.blocked_pattern(L, 256), "dilated 77 by 3": lambda L: A.dilated_pattern(L, 77, 3),
         "dilated 300 by 2": lambda L: A.dilated_pattern(L, min(300, L // 2), 2), "strided": lambda L: A.strided_patterns(L, 20, 40),
         "strided 7": lambda L: A.strided_patterns(L, 7, L // 50), "strided 100": lambda L: A.strided_patterns(L, 100, 16),
         "strided 200": lambda L: A.strided_patterns(L, 200, 7), "steps differ": _steps_differ}


def _operands(dev, dtype, heads, L, d, layout, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed + L + d)
    if layout == "tokens":
        q, k, v = (torch.randn(1, L, heads, d, generator=g, device=dev).to(dtype).transpose(1, 2) for _ in range(3))
    else:
        q, k, v = (torch.randn(1, heads, L, d, generator=g, device=dev).to(dtype) for _ in range(3))
    kT = k.transpose(2, 3)
    return q, kT.contiguous() if layout == "keys" else kT, v


def _one_launch(segs, q, kT, v, scale, buffers, T=None):
    heads, L, d = q.shape[1:]
    T = T or segs.T
    arr, plan = segs.seg_array(L, T), segs.plan(L, q.device)
    return hip.lib().splat_operators(q.data_ptr(), *q.stride()[:3], kT.data_ptr(), *kT.stride()[:4], v.data_ptr(), *v.stride()[:3],
                                     *(b.data_ptr() for b in buffers), arr, len(segs), 1, heads, L, v.shape[2], d, T, ctypes.c_float(scale),
                                     hip.dtype_code(q.dtype), plan.data_ptr(), plan.numel() * plan.element_size(), segs.one_step(L, q.device), hip.stream_ptr(q.device))


def _segments(mask, dev):
    if not isinstance(mask, list):
        mask = [mask]
    return A.create_acsr_segments(mask, 16, dev)


@pytest.mark.parametrize("dtype,d,layout", [(torch.bfloat16, 64, "rows"), (torch.float16, 128, "tokens"), (torch.bfloat16, 80, "keys"),
                                            (torch.float16, 32, "keys"), (torch.bfloat16, 104, "rows")])
@pytest.mark.parametrize("L,heads", [(600, 3), (1037, 8), (600, 54), (700, 140)])  # (eight wavefronts a workgroup and, from 512 workgroups on, four)
@pytest.mark.parametrize("mask", list(MASKS))
def test_equals_the_three_calls(dev, mask, L, heads, dtype, d, layout):
    segs = _segments(MASKS[mask](L), dev)
    T = segs.T
    q, kT, v = _operands(dev, dtype, heads, L, d, layout)
    arr, code, stream, plan = segs.seg_array(L, T), hip.dtype_code(dtype), hip.stream_ptr(dev), segs.plan(L, dev)
    sizes = [heads * L * T + 8, heads * L * T + 8, heads * L * d + 8]
    want, got = ([torch.full((n,), SENTINEL, dtype=dtype, device=dev) for n in sizes] for _ in range(2))
    rc = _one_launch(segs, q, kT, v, 0.2, got)
    if mask == "steps differ":
        assert rc == -5
    elif T > 256 and len(segs) > 1:  # (left to the separate calls in many and in few workgroups, with K along the keys and more than 64 values in some more)
        assert (rc == 0) == (heads == 8 and not (layout == "keys" and d > 64))
    else:
        assert rc == 0
    if rc:
        assert rc == -5 and all(torch.all(b == SENTINEL) for b in got)
        return
    table = (plan.data_ptr(), plan.numel() * plan.element_size())
    rows = kT if layout != "keys" else kT.transpose(2, 3).contiguous().transpose(2, 3)
    hip.check(hip.lib().splat_sddmm_planned(q.data_ptr(), *q.stride()[:3], rows.data_ptr(), *rows.stride()[:4], want[0].data_ptr(), arr, len(segs), 1, heads,
                                            L, L, d, T, ctypes.c_float(0.2), code, code, None, *table, stream), "splat_sddmm_planned")
    hip.check(hip.lib().splat_softmax(want[0].data_ptr(), want[1].data_ptr(), arr, len(segs), heads, L, T, code, code, stream), "splat_softmax")
    hip.check(hip.lib().splat_spmm_planned(want[1].data_ptr(), v.data_ptr(), *v.stride()[:3], want[2].data_ptr(), arr, len(segs), 1, heads, L, L, d, T, code,
                                           code, *table, stream), "splat_spmm_planned")
    scores = [b[0][:-8].double() for b in (want, got)]
    eps = torch.finfo(dtype).eps
    if T > 256 and not torch.equal(*scores):
        # (the general kernel, which takes some launches of longer rows, adds in another order: a float32 sum of d products of a size of 5 apart, rounded)
        assert float((scores[0] - scores[1]).abs().max()) <= 8 * eps
    else:
        assert torch.equal(want[0], got[0]) and torch.equal(want[1], got[1])
        if T >= 8 and len(segs) == 1:  # (shorter rows and segments are the general kernel's)
            assert torch.equal(want[2], got[2])
    # dead slots and what lies behind the buffers stay as they were
    for b in got:
        assert torch.all(b[-8:] == SENTINEL)
    few = slice(0, 3)
    out = torch.zeros(heads, L, d, dtype=torch.float64, device=dev)[few]
    live_rows = torch.zeros(L, device=dev)
    for t, fc, off in zip(segs.tuples, segs.first_cols, segs.offsets):
        cols, live = live_slot_columns(t[2], t[3], t[4], int(t[5]), fc)
        part = got[1][:-8].view(heads, L, T)[few, :, off:off + int(t[5])].double()
        assert torch.all(part[:, ~live] == SENTINEL) and torch.all(got[0][:-8].view(heads, L, T)[few, :, off:off + int(t[5])].double()[:, ~live] == SENTINEL)
        dense = torch.zeros(len(out), L, L, dtype=torch.float64, device=dev)
        dense.scatter_add_(2, cols.clamp(0, L - 1).expand(len(out), L, -1), torch.where(live, part, 0.0))
        out += dense @ v[0, few].double()
        live_rows += t[4]
    # (probabilities that sum to 1 times values of at most 6: the float32 sum of up to 512 of them, and one rounding to the type)
    err = (got[2][:-8].view(heads, L, d)[few].double() - out).abs()
    assert float((err - out.abs() * eps / 2 * 1.01).max()) <= 512 * 6 * 2.0 ** -24
    rows_sum = torch.where(got[1][:-8].view(heads, L, T).double() == SENTINEL, 0.0, got[1][:-8].view(heads, L, T).double()).sum(-1)
    assert float((rows_sum - (live_rows > 0).double()).abs().max()) <= eps + 512 * 2.0 ** -24


@pytest.mark.parametrize("T", [104, 128, 256, 416, 512])
def test_large_matrices_equal_their_halves(dev, T):
    """Scores and probabilities that the caches do not hold are stored around them: the same bits."""
    L, d, dtype, heads = 2048, 32, torch.bfloat16, 2 * -(-(84 << 20) // (4 * 2048 * T))
    segs = _segments(A.causal_windowed_pattern(L, T - 1), dev)
    q, kT, v = _operands(dev, dtype, heads, L, d, "rows")

    def both(h0, n):
        bufs = [torch.full((n, L, w), SENTINEL, dtype=dtype, device=dev) for w in (T, T, d)]
        hip.check(_one_launch(segs, q[:, h0:h0 + n], kT[:, h0:h0 + n], v[:, h0:h0 + n], 0.2, bufs), "splat_operators")
        return bufs
    whole, parts = both(0, heads), [both(0, heads // 2), both(heads // 2, heads // 2)]
    for i in range(3):
        assert torch.equal(whole[i], torch.cat([x[i] for x in parts]))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("mask", ["33", "512", "strided"])
def test_infinities_and_not_a_number(dev, dtype, mask):
    """Scores of minus infinity weigh nothing, rows of nothing but them give zeros, NaN stays in the rows that see it: as the three calls."""
    L, d, heads = 600, 64, 2
    segs = _segments(MASKS[mask](L), dev)
    T = segs.T
    q, kT, v = _operands(dev, dtype, heads, L, d, "rows")
    q, kT = q.clone(), kT.transpose(2, 3).clone().transpose(2, 3)
    q[:, 0, 40:80] = 1.0
    kT[:, 0, :, 30:60] = float("-inf")
    kT[:, 1, 3, 100] = float("nan")
    arr, code, stream, plan = segs.seg_array(L, T), hip.dtype_code(dtype), hip.stream_ptr(dev), segs.plan(L, dev)
    want, got = ([torch.full((heads, L, w), SENTINEL, dtype=dtype, device=dev) for w in (T, T, d)] for _ in range(2))
    hip.check(_one_launch(segs, q, kT, v, 1.0, got), "splat_operators")
    table = (plan.data_ptr(), plan.numel() * plan.element_size())
    hip.check(hip.lib().splat_sddmm_planned(q.data_ptr(), *q.stride()[:3], kT.data_ptr(), *kT.stride()[:4], want[0].data_ptr(), arr, len(segs), 1, heads,
                                            L, L, d, T, ctypes.c_float(1.0), code, code, None, *table, stream), "splat_sddmm_planned")
    hip.check(hip.lib().splat_softmax(want[0].data_ptr(), want[1].data_ptr(), arr, len(segs), heads, L, T, code, code, stream), "splat_softmax")
    hip.check(hip.lib().splat_spmm_planned(want[1].data_ptr(), v.data_ptr(), *v.stride()[:3], want[2].data_ptr(), arr, len(segs), 1, heads, L, L, d, T, code,
                                           code, *table, stream), "splat_spmm_planned")
    for a, b in zip(got[:2], want[:2]):
        assert torch.allclose(a.float(), b.float(), rtol=torch.finfo(dtype).eps, atol=8 * torch.finfo(dtype).eps, equal_nan=True)
    assert torch.equal(torch.isnan(got[2]), torch.isnan(want[2]))
    assert torch.allclose(got[2].float(), want[2].float(), rtol=0, atol=4 * torch.finfo(dtype).eps, equal_nan=True)


def test_what_it_does_not_take(dev):
    """Other types, dimensions, rows and addresses are left to the separate calls, before anything is written."""
    L, heads = 300, 2
    segs = _segments(A.causal_windowed_pattern(L, 19), dev)

    def code(dtype=torch.bfloat16, d=64, segs=segs, shift=0):
        q, kT, v = _operands(dev, dtype, heads, L, d, "rows")
        bufs = [torch.full((heads * L * w + 8,), 7.0, dtype=dtype, device=dev) for w in (segs.T, segs.T, d)]
        rc = _one_launch(segs, q, kT, v, 1.0, [bufs[0], bufs[1], bufs[2][shift:]])
        torch.cuda.synchronize()
        assert rc == 0 or all(bool(torch.all(b == 7.0)) for b in bufs)
        return rc
    assert code() == 0
    assert code(dtype=torch.float32) == code(d=12) == code(d=136) == code(shift=1) == -5
    L = 600
    assert code(segs=_segments(_steps_differ(L), dev)) == -5
    assert code(segs=_segments(A.causal_windowed_pattern(L, 512), dev)) == -5


def _three_calls(segs, q, kT, v, scale, buffers, T=None):
    """The same through splat_sddmm_planned, splat_softmax and splat_spmm_planned."""
    heads, L, d = q.shape[1:]
    T = T or segs.T
    arr, plan, code, stream = segs.seg_array(L, T), segs.plan(L, q.device), hip.dtype_code(q.dtype), hip.stream_ptr(q.device)
    table = (plan.data_ptr(), plan.numel() * plan.element_size())
    s, p, o = buffers
    hip.check(hip.lib().splat_sddmm_planned(q.data_ptr(), *q.stride()[:3], kT.data_ptr(), *kT.stride()[:4], s.data_ptr(), arr, len(segs), 1, heads, L, kT.shape[3],
                                            d, T, ctypes.c_float(scale), code, code, None, *table, stream), "splat_sddmm_planned")
    hip.check(hip.lib().splat_softmax(s.data_ptr(), p.data_ptr(), arr, len(segs), heads, L, T, code, code, stream), "splat_softmax")
    hip.check(hip.lib().splat_spmm_planned(p.data_ptr(), v.data_ptr(), *v.stride()[:3], o.data_ptr(), arr, len(segs), 1, heads, L, v.shape[2], d, T, code, code,
                                           *table, stream), "splat_spmm_planned")


@pytest.mark.parametrize("layout", ["rows", "keys"])
@pytest.mark.parametrize("heads", [2, 80])  # (eight wavefronts a workgroup and four)
@pytest.mark.parametrize("mask,d", [("33", 64), ("200", 128), ("strided", 64)])
def test_columns_before_the_first_stand_for_it(dev, mask, d, heads, layout):
    """Metadata made by hand, whose first rows begin before column 0: nothing is read in front of K and V, as with the separate calls, where such columns
    have the first one's key and value."""
    L = 600
    segs = _segments(MASKS[mask](L), dev)
    T, t = segs.T, segs.tuples[0]
    n = int(t[5])
    first = torch.arange(L, device=dev) - (n - 1)
    t[2].fill_(1.0), t[3].copy_(first.to(t[3].dtype)), t[4].fill_(n), segs.first_cols[0].copy_(first)
    q, kT, v = _operands(dev, torch.bfloat16, heads, L, d, layout)
    want, got = ([torch.full((heads, L, w), SENTINEL, dtype=torch.bfloat16, device=dev) for w in (T, T, d)] for _ in range(2))
    hip.check(_one_launch(segs, q, kT, v, 0.2, got), "splat_operators")
    _three_calls(segs, q, kT.transpose(2, 3).contiguous().transpose(2, 3), v, 0.2, want)
    for a, b in zip(got[:2], want[:2]):
        assert torch.equal(a, b) and torch.all(a[:, :, :n] != SENTINEL)
    columns = (first[:, None] + torch.arange(n, device=dev)).clamp(min=0)
    q8, k8, v8 = q[0, 0].double(), kT[0, 0].double(), v[0, 0].double()
    s = (q8 @ k8).gather(1, columns) * 0.2
    # (one rounding of a sum of d products to the type)
    assert float((got[0][0, :, :n].double() - s).abs().max()) <= float(s.abs().max()) * torch.finfo(torch.bfloat16).eps
    if len(segs) == 1:
        out = (got[1][0].double()[:, :, None] * v8[columns]).sum(1)
        err = (got[2][0].double() - out).abs()
        assert float((err - out.abs() * torch.finfo(torch.bfloat16).eps / 2 * 1.01).max()) <= T * 6 * 2.0 ** -24
        assert torch.equal(got[2], want[2])
    else:
        assert torch.allclose(got[2].float(), want[2].float(), rtol=2 * torch.finfo(torch.bfloat16).eps, atol=1e-4)


@pytest.mark.parametrize("layout", ["rows", "keys"])
@pytest.mark.parametrize("L,heads", [(600, 2), (600, 80)])
@pytest.mark.parametrize("mask,T,d", [("128", 64, 64), ("128", 40, 128), ("200", 64, 80), ("512", 256, 64), ("512", 129, 128), ("dilated 77 by 3", 33, 64), ("windowed 257", 128, 64),
                                      ("blocked 512", 200, 128), ("strided 100", 110, 64), ("strided 7", 30, 64)])
def test_rows_longer_than_the_buffers_rows(dev, mask, T, d, L, heads, layout):
    """Rows of more live columns than a compressed row has slots end with the last slot, in all three results, as with the separate calls."""
    segs = _segments(MASKS[mask](L), dev)
    assert segs.T > T
    q, kT, v = _operands(dev, torch.bfloat16, heads, L, d, layout)
    want, got = ([torch.full((heads * L * w + 8,), SENTINEL, dtype=torch.bfloat16, device=dev) for w in (T, T, d)] for _ in range(2))
    hip.check(_one_launch(segs, q, kT, v, 0.2, got, T), "splat_operators")
    _three_calls(segs, q, kT.transpose(2, 3).contiguous().transpose(2, 3), v, 0.2, want, T)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    if len(segs) == 1:
        assert torch.equal(got[2], want[2])
    else:
        assert torch.allclose(got[2].float(), want[2].float(), rtol=2 * torch.finfo(torch.bfloat16).eps, atol=1e-4)


def test_results_that_share_memory_with_operands_are_left_to_the_separate_calls(dev):
    """No launch in which one workgroup stores what another still reads: results over an operand, from its first byte to its last one, over each other, or
    over rows between an operand's; neighbours in memory are taken."""
    heads, L, d, dtype = 2, 256, 64, torch.bfloat16
    segs = _segments(A.causal_windowed_pattern(L, d - 1), dev)
    n = heads * L * d
    assert segs.T == d  # (so that all six have one size)
    for operand in range(3):
        for result in range(3):
            for shift, taken in ((0, False), (8, False), (-8, False), (n - 8, False), (8 - n, False), (n, True), (-n, True)):
                pool = torch.full((10 * n,), SENTINEL, dtype=dtype, device=dev)
                at = 3 * n + operand * n  # the operand is where it is, the result around it, the others further on
                ops = [pool[at:at + n] if i == operand else torch.randn(n, device=dev).to(dtype) for i in range(3)]
                ops[operand].copy_(torch.randn(n, device=dev))
                bufs = [pool[at + shift:at + shift + n] if i == result else torch.empty(n, dtype=dtype, device=dev) for i in range(3)]
                q, k, v = (t.view(1, heads, L, d) for t in ops)
                rc = _one_launch(segs, q, k.transpose(2, 3), v, 0.2, bufs)
                assert rc == (0 if taken else -5), (operand, result, shift)
    pool = torch.randn(8 * n, device=dev).to(dtype)
    q, k, v, s, p, o = (pool[i * n:(i + 1) * n] for i in range(6))
    x = (q.view(1, heads, L, d), k.view(1, heads, L, d).transpose(2, 3), v.view(1, heads, L, d))
    assert _one_launch(segs, *x, 0.2, [s, p, o]) == 0
    for bufs in ([s, pool[3 * n + 8:4 * n + 8], o], [s, p, s], [s, p, p]):
        assert _one_launch(segs, *x, 0.2, bufs) == -5
    wide = torch.randn(1, heads, L, 2 * d, device=dev).to(dtype)  # rows of K with room between them
    assert _one_launch(segs, x[0], wide[..., :d].transpose(2, 3), x[2], 0.2, [s, p, wide.view(-1)[d:d + n]]) == -5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("layout", ["rows", "keys"])
@pytest.mark.parametrize("which", ["q", "k", "probabilities as k"])
def test_a_modules_own_buffers_as_operands(dev, which, layout, dtype):
    """The output of the call before (the module's buffer) as q or K of the next call, or its probabilities where a row has as many slots as a head has
    values: as with a copy."""
    from r_attention import RegularAttention
    heads, L, d = 24, 512, 64
    g = torch.Generator(device=dev).manual_seed(3)
    q, k, v, w = (torch.randn(1, heads, L, d, generator=g, device=dev).to(dtype) for _ in range(4))
    attn, other = (RegularAttention(1, L, heads, d, A.causal_windowed_pattern(L, d - 1), 16, 16, dev, dtype, scale=0.125, fused=False) for _ in range(2))
    attn.rsoftmax_output.zero_()  # (dead slots)
    first = attn([q, k.transpose(2, 3), v])
    if which == "probabilities as k":
        first = attn.rsoftmax_output
    if layout == "keys" and which != "q":
        x = lambda t: [q, t.view(1, heads, d, L), w]  # noqa: E731
    else:
        x = lambda t: [t, k.transpose(2, 3), w] if which == "q" else [q, t.transpose(2, 3), w]  # noqa: E731
    want = other(x(first.clone()))
    got = attn(x(first))
    assert torch.equal(got, want)


@pytest.mark.parametrize("T,d,layout,blocks,taken", [
    (257, 32, "rows", 80, True), (257, 32, "rows", 78, False), (257, 32, "rows", 448, True), (257, 32, "rows", 450, False), (300, 64, "rows", 512, True),
    (300, 64, "rows", 514, False), (300, 64, "keys", 126, False), (300, 64, "keys", 128, True), (300, 128, "rows", 128, True), (300, 128, "rows", 126, False),
    (300, 72, "keys", 190, False), (300, 72, "keys", 192, True), (300, 128, "rows", 256, True), (300, 128, "rows", 258, False), (129, 64, "rows", 2048, True),
    (129, 64, "rows", 2050, False), (256, 128, "rows", 768, True), (256, 104, "rows", 770, False), (200, 128, "rows", 1536, False), (200, 128, "rows", 1538, True),
    (200, 96, "rows", 1000, True), (128, 128, "rows", 1000, True), (128, 32, "keys", 2050, True)])
def test_which_launches_of_two_segments_are_one(dev, T, d, layout, blocks, taken):
    """Both sides of every line of the rule, by slots, head dimension, layout of K and workgroups of 64 rows (heads of 128 rows)."""
    L, heads = 128, blocks // 2
    near = A.causal_windowed_pattern(L, 15)
    segs = _segments([near, A.strided_patterns(L, 16, 16)[1]], dev)
    arr, plan = segs.seg_array(L, T), segs.plan(L, dev)
    q, kT, v = _operands(dev, torch.bfloat16, heads, L, d, layout)
    bufs = [torch.full((heads, L, w), SENTINEL, dtype=torch.bfloat16, device=dev) for w in (T, T, d)]
    assert _one_launch(segs, q, kT, v, 0.2, bufs, T) == (0 if taken else -5)
    if taken:
        want = [torch.full((heads, L, w), SENTINEL, dtype=torch.bfloat16, device=dev) for w in (T, T, d)]
        _three_calls(segs, q, kT.transpose(2, 3).contiguous().transpose(2, 3), v, 0.2, want, T)
        eps = torch.finfo(torch.bfloat16).eps
        for a, b in zip(bufs, want):  # (long rows may be added in another order: one rounding apart)
            assert torch.equal(a == SENTINEL, b == SENTINEL)
            assert float(((a.float() - b.float()).abs() - eps * b.float().abs()).max()) <= 1e-4


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("mask,d", [("dilated 60 by 5", 64), ("dilated 40 by 8", 96), ("dilated 300 by 2", 128), ("dilated 300 by 2", 64), ("dilated 77 by 3", 128), ("512", 128)])
def test_keys_that_are_turned_before_and_inside(dev, mask, d, dtype):
    """A module's forward in many workgroups with K along the keys, on both sides of the rule for turning it first, is the one with rows of K, bit for bit;
    two sequences whose heads lie between each other's in memory."""
    from r_attention import RegularAttention
    B, H, L = 2, 36, 640
    pattern = {"dilated 60 by 5": lambda L: A.dilated_pattern(L, 60, 5), "dilated 40 by 8": lambda L: A.dilated_pattern(L, 40, 8), **MASKS}[mask](L)
    g = torch.Generator(device=dev).manual_seed(d)
    q, k, v = (torch.randn(H, B, L, d, generator=g, device=dev).to(dtype).transpose(0, 1) for _ in range(3))
    attn = RegularAttention(B, L, H, d, pattern, 16, 16, dev, dtype, scale=0.2, fused=False)
    dead = [b.fill_(SENTINEL) for b in (attn.rsddmm_output, attn.rsoftmax_output)]
    want = [t.clone() for t in (attn([q, k.transpose(2, 3), v]), *dead)]
    along = k.transpose(2, 3).contiguous()
    got = attn([q, along, v])
    for a, b in zip((got, *dead), want):
        assert torch.equal(a, b)
    each = RegularAttention(1, L, H, d, pattern, 16, 16, dev, dtype, scale=0.2, fused=False)  # one sequence after the other
    for i in range(B):
        one = each([q[i:i + 1], k[i:i + 1].transpose(2, 3), v[i:i + 1]])
        assert torch.equal(one[0], want[0][i])


@pytest.mark.parametrize("mask", ["33", "64", "200", "512", "blocked 512", "dilated 77 by 3", "dilated 300 by 2", "strided", "strided 100"])
@pytest.mark.parametrize("heads", [2, 54])
def test_infinities_and_not_a_number_in_values(dev, mask, heads):
    """Rows that see a value of infinity or NaN have it; no row that the three calls leave finite is any other here, nor any other column."""
    L, d, dtype = 600, 64, torch.bfloat16
    segs = _segments(MASKS[mask](L), dev)
    q, kT, v = _operands(dev, dtype, heads, L, d, "rows")
    v = v.clone()
    rows, columns = [0, 100, 333, L - 1], [3, 5, 6, 7]
    for r, c, x in zip(rows, columns, (float("inf"), float("nan"), float("-inf"), float("nan"))):
        v[:, 0, r, c] = x
    want, got = ([torch.full((heads, L, w), SENTINEL, dtype=dtype, device=dev) for w in (segs.T, segs.T, d)] for _ in range(2))
    hip.check(_one_launch(segs, q, kT, v, 0.2, got), "splat_operators")
    _three_calls(segs, q, kT, v, 0.2, want)
    finite = torch.isfinite(got[2])
    assert torch.all(finite | ~torch.isfinite(want[2])) and torch.all(finite[1:])
    for r, c in zip(rows, columns):
        sees = torch.zeros(L, dtype=torch.bool, device=dev)
        for t, fc in zip(segs.tuples, segs.first_cols):
            cols, live = live_slot_columns(t[2], t[3], t[4], int(t[5]), fc)
            sees |= ((cols == r) & live).any(1)
        assert not torch.any(finite[0, sees, c])
    assert torch.all(finite[0][:, [c for c in range(d) if c not in columns]])
    both = finite & torch.isfinite(want[2])
    assert torch.allclose(got[2][both].float(), want[2][both].float(), rtol=2 * torch.finfo(dtype).eps, atol=1e-4)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L,heads", [(600, 8), (1037, 40)])
@pytest.mark.parametrize("mask", ["257", "509", "512", "blocked 512", "dilated 300 by 2", "strided 200"])
def test_probabilities_of_long_rows_are_the_softmax_of_their_scores(dev, mask, L, heads, dtype):
    """Rows of more than 256 slots, whose scores some separate launches add in another order: the probabilities are splat_softmax's of the scores that are
    stored beside them, bit for bit."""
    segs = _segments(MASKS[mask](L), dev)
    d, T = 64, segs.T
    assert T > 256
    q, kT, v = _operands(dev, dtype, heads, L, d, "rows")
    got = [torch.full((heads, L, w), SENTINEL, dtype=dtype, device=dev) for w in (T, T, d)]
    rc = _one_launch(segs, q, kT, v, 0.2, got)
    assert rc == 0 or (rc == -5 and len(segs) > 1 and heads == 40)
    if rc == 0:
        again = torch.full_like(got[1], SENTINEL)
        hip.check(hip.lib().splat_softmax(got[0].data_ptr(), again.data_ptr(), segs.seg_array(L, T), len(segs), heads, L, T, hip.dtype_code(dtype),
                                          hip.dtype_code(dtype), hip.stream_ptr(dev)), "splat_softmax")
        assert torch.equal(got[1], again)
