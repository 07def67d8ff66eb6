"""The sampled product and the softmax of its rows in one call against the two calls, bit for bit: rows at the edges of the softmax's splits and
beyond the longest that the sampled product takes along, masks whose row blocks interleave, two segments, with the plan table and
without, launches on both sides of the line from which a workgroup owns whole rows."""
import ctypes

import pytest
import torch

import acsr_helpers as A
import _splat_hip as hip
from test_gpu_operators import SENTINEL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.float16, 104), (torch.float32, 40), (torch.float32, 128)])
@pytest.mark.parametrize("heads", [1, 64, 100])  # (4 half row blocks a head; few, the line's, and what the line-wise kernel takes of the widest)
@pytest.mark.parametrize("pattern", [lambda L: A.causal_windowed_pattern(L, 5), lambda L: A.causal_windowed_pattern(L, 128),
                                     lambda L: A.causal_windowed_pattern(L, 129), lambda L: A.dilated_pattern(L, 77, 3),
                                     lambda L: A.strided_patterns(L, 40, 16), lambda L: A.causal_windowed_pattern(L, 201),
                                     lambda L: A.blocked_pattern(L, 200), lambda L: A.causal_windowed_pattern(L + 51, 257),
                                     *((lambda w: lambda L: A.causal_windowed_pattern(L + 51, w - 1))(w) for w in (32, 33, 64, 65, 256))],
                         ids=["5", "128", "129", "dilated 77", "strided", "201", "blocked 200", "257", "edge 32", "edge 33", "edge 64", "edge 65",
                              "edge 256"])
@pytest.mark.parametrize("layout", ["rows", "keys"])
def test_equals_the_two_calls(dev, layout, pattern, heads, dtype, d):
    L = 250
    masks = pattern(L)
    segs = A.create_acsr_segments(masks if isinstance(masks, list) else [masks], 16, dev)
    L, T = segs.tuples[0][0].shape[0], segs.T
    g = torch.Generator(device=dev).manual_seed(T + d)
    q, k = (torch.randn(1, heads, L, d, generator=g, device=dev).to(dtype) for _ in range(2))
    kT = k.transpose(2, 3)
    if layout == "keys":
        kT = kT.contiguous()
    arr, code, stream = segs.seg_array(L, T), hip.dtype_code(dtype), hip.stream_ptr(dev)
    plan = segs.plan(L, dev)
    for table, nbytes in ((plan.data_ptr(), plan.numel() * plan.element_size()), (None, 0)):
        buffers = [torch.full((heads * L * T + 8,), SENTINEL, dtype=dtype, device=dev) for _ in range(4)]
        want, want_p, got, got_p = (b.data_ptr() for b in buffers)
        x = (q.data_ptr(), *q.stride()[:3], kT.data_ptr(), *kT.stride()[:4])
        shape = (arr, len(segs), 1, heads, L, L, d, T, ctypes.c_float(0.2), code, code)
        if table is None:
            hip.check(hip.lib().splat_sddmm(*x, want, *shape, stream), "splat_sddmm")
        else:
            hip.check(hip.lib().splat_sddmm_planned(*x, want, *shape, None, table, nbytes, stream), "splat_sddmm_planned")
        hip.check(hip.lib().splat_softmax(want, want_p, arr, len(segs), heads, L, T, code, code, stream), "splat_softmax")
        hip.check(hip.lib().splat_sddmm_softmax(*x, got, got_p, *shape, table, nbytes, stream), "splat_sddmm_softmax")
        assert torch.equal(buffers[0], buffers[2]) and torch.equal(buffers[1], buffers[3])
        rows = buffers[3][:-8].view(heads, L, T).double()
        sums = torch.where(rows == SENTINEL, 0.0, rows).sum(-1)
        # (a row of n slots sums to 1 within the roundings of its entries, at most half a unit of the type each, and of its float32 sum)
        assert float((sums - 1).abs().max()) <= torch.finfo(dtype).eps + 256 * 2.0 ** -24


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows", [300, 41000, 140000])  # (as many row groups a wavefront as the chip has room for, and more)
@pytest.mark.parametrize("T", [7, 9, 128, 136, 249, 256, 257, 504, 511, 1023])
def test_softmax_of_few_and_many_rows(dev, T, rows, dtype):
    """Every row's live slots against float64, a float32 evaluation of an exponential and a quotient apart, then rounded."""
    g = torch.Generator(device=dev).manual_seed(T)
    L = 50
    nnz = torch.randint(0, T + 1, (L,), generator=g, device=dev).float()
    nnz[::2] = T
    zeros = torch.zeros(L, device=dev)
    seg = (hip.AcsrSeg * 1)()
    seg[0].sTod_lin, seg[0].sTod_trans, seg[0].nnz, seg[0].slot_offset = zeros.data_ptr(), zeros.data_ptr(), nnz.data_ptr(), 0
    BH = rows // L
    x = (torch.randn(BH, L, T, generator=g, device=dev) * 3).to(dtype)
    buf = torch.full((BH * L * T + 9,), SENTINEL, dtype=dtype, device=dev)
    for shift in (0, 1):  # (a buffer that starts anywhere, too)
        buf.fill_(SENTINEL)
        out = buf[shift:shift + BH * L * T]
        hip.check(hip.lib().splat_softmax(x.data_ptr(), out.data_ptr(), seg, 1, BH, L, T, hip.dtype_code(dtype), hip.dtype_code(dtype),
                                          hip.stream_ptr(dev)), "splat_softmax")
        live = torch.arange(T, device=dev)[None] < nnz[:, None]
        want = torch.softmax(x[:64].double().masked_fill(~live, float("-inf")), -1)
        for part, ref in ((out.view(BH, L, T)[:64], want), (out.view(BH, L, T)[-1:], torch.softmax(x[-1:].double().masked_fill(~live, float("-inf")), -1))):
            err = (part.double() - ref).abs() / ref.clamp_min(1e-30)
            # (exp2 of a float32 product of up to 40: 40 * 2^-24 of it; the sum and the quotient a few units; one rounding to the type)
            assert float(torch.where(live & (ref > 1e-4), err, 0.0).max()) <= 128 * 2.0 ** -24 + torch.finfo(dtype).eps / 2 * 1.01
            assert torch.all(part.double()[~live.expand_as(part)] == SENTINEL)
        assert torch.all(buf[:shift] == SENTINEL) and torch.all(buf[shift + BH * L * T:] == SENTINEL)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [104, 128, 200, 256, 304, 320, 456, 512])
@pytest.mark.parametrize("planned", [True, False])
def test_large_matrices_equal_their_halves(dev, planned, T, dtype):
    """Scores and probabilities that the caches do not hold are stored around them; the halves of the same heads are not: the same bits."""
    L, d, heads = 2048, 32, 2 * -(-(84 << 20) // (4 * 2048 * T))
    segs = A.create_acsr_segments([A.causal_windowed_pattern(L, T - 1)], 16, dev)
    assert segs.T == T
    g = torch.Generator(device=dev).manual_seed(T)
    q, k = (torch.randn(1, heads, L, d, generator=g, device=dev).to(dtype) for _ in range(2))
    arr, code, stream, plan = segs.seg_array(L, T), hip.dtype_code(dtype), hip.stream_ptr(dev), segs.plan(L, dev)

    def both(h0, n):
        s, p = (torch.full((n, L, T), SENTINEL, dtype=dtype, device=dev) for _ in range(2))
        a, b = q[:, h0:h0 + n], k[:, h0:h0 + n].transpose(2, 3)
        table = (None, plan.data_ptr(), plan.numel() * plan.element_size()) if planned else ()
        hip.check((hip.lib().splat_sddmm_planned if planned else hip.lib().splat_sddmm)(
            a.data_ptr(), *a.stride()[:3], b.data_ptr(), *b.stride()[:4], s.data_ptr(), arr, 1, 1, n, L, L, d, T, ctypes.c_float(0.2), code,
            code, *table, stream), "splat_sddmm")
        hip.check(hip.lib().splat_softmax(s.data_ptr(), p.data_ptr(), arr, 1, n, L, T, code, code, stream), "splat_softmax")
        return s, p
    whole, parts = both(0, heads), [both(0, heads // 2), both(heads // 2, heads // 2)]
    for i in range(2):
        assert torch.equal(whole[i], torch.cat([x[i] for x in parts]))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows", [300, 140000, 450000])  # (small, and beyond what the caches hold)
@pytest.mark.parametrize("T", [9, 31, 32, 33, 48, 49, 63, 64, 65, 104, 112, 113, 127, 128, 130, 192, 264, 376, 384, 385, 392, 440, 448, 449, 456, 505, 512])
def test_softmax_rows_over_lanes(dev, T, rows, dtype):
    """Edges of the splits of a row over lanes, two segments with dead slots between and after them, in place, against float64."""
    g = torch.Generator(device=dev).manual_seed(T)
    L, off = 50, T * 2 // 3 - 1
    cnt = [torch.randint(0, n + 1, (L,), generator=g, device=dev).float() for n in (off, T - off)]
    cnt[0][::3], cnt[1][::3] = off, T - off
    cnt[0][1], cnt[1][1] = 0, 0
    seg = (hip.AcsrSeg * 2)()
    for k in range(2):
        seg[k].sTod_lin = seg[k].sTod_trans = seg[k].nnz = cnt[k].data_ptr()
        seg[k].slot_offset = (0, off)[k]
    BH = rows // L
    x = (torch.randn(BH, L, T, generator=g, device=dev) * 3).to(dtype)
    slot = torch.arange(T, device=dev)[None]
    live = (slot < cnt[0][:, None]) | ((slot >= off) & (slot < off + cnt[1][:, None]))
    want = torch.softmax(torch.cat([x[:32], x[-1:]]).double().masked_fill(~live, float("-inf")), -1)
    dead = torch.cat([x[:32], x[-1:]])
    hip.check(hip.lib().splat_softmax(x.data_ptr(), x.data_ptr(), seg, 2, BH, L, T, hip.dtype_code(dtype), hip.dtype_code(dtype),
                                      hip.stream_ptr(dev)), "splat_softmax")
    got = torch.cat([x[:32], x[-1:]])
    err = (got.double() - want).abs() / want.clamp_min(1e-30)
    # (as above; probabilities above 1e-4 are normal numbers of both types)
    assert float(torch.where(live & (want > 1e-4), err, 0.0).max()) <= 128 * 2.0 ** -24 + torch.finfo(dtype).eps / 2 * 1.01
    assert torch.equal(got[~live.expand_as(got)], dead[~live.expand_as(got)])


@pytest.mark.parametrize("T", [264, 301, 384, 385, 392, 441, 512, 513])
@pytest.mark.parametrize("heads", [30, 60, 110])  # (half row blocks; a round of row blocks that is not full; one more, of which little is left)
@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.float16, 128)])
def test_long_rows_equal_the_two_calls(dev, dtype, d, heads, T):
    """Rows of more than 256 slots, to the longest that the sampled product takes along and beyond."""
    test_equals_the_two_calls(dev, "rows", lambda L: A.causal_windowed_pattern(520, T - 1), heads, dtype, d)


def test_long_rows_of_two_segments_equal_the_two_calls(dev):
    test_equals_the_two_calls(dev, "rows", lambda L: A.strided_patterns(700, 256, 16), 50, torch.bfloat16, 64)


@pytest.mark.parametrize("din,dout", [(torch.bfloat16, torch.float32), (torch.float16, torch.float16), (torch.float32, torch.float32)])
@pytest.mark.parametrize("T", [7, 20, 32, 33, 40, 48, 49, 64, 65, 72, 104, 112, 113, 128, 129, 136, 200, 255, 256, 257, 301, 384, 385, 448, 456, 504, 511, 512, 1000])
def test_a_row_s_bits_do_not_depend_on_the_call(dev, T, din, dout):
    """A few rows, the same rows among as many as the caches do not hold, and in a buffer that starts off every boundary: one sum."""
    g = torch.Generator(device=dev).manual_seed(T)
    L, off = 64, T // 3
    cnt = [torch.randint(0, n + 1, (L,), generator=g, device=dev).float() for n in (off, T - off)]
    cnt[0][::2], cnt[1][::2] = off, T - off
    seg = (hip.AcsrSeg * 2)()
    for k in range(2):
        seg[k].sTod_lin = seg[k].sTod_trans = seg[k].nnz = cnt[k].data_ptr()
        seg[k].slot_offset = (0, off)[k]
    x = (torch.randn(1, L, T, generator=g, device=dev) * 3).to(din)

    def softmax(x, shift):
        n = x.shape[0]
        src = torch.empty(x.numel() + shift, dtype=din, device=dev)[shift:].view(x.shape)
        src.copy_(x)
        dst = torch.full((x.numel() + shift,), 7.0, dtype=dout, device=dev)[shift:].view(x.shape)
        hip.check(hip.lib().splat_softmax(src.data_ptr(), dst.data_ptr(), seg, 2, n, L, T, hip.dtype_code(din), hip.dtype_code(dout),
                                          hip.stream_ptr(dev)), "splat_softmax")
        return dst
    want = softmax(x, 0)
    assert torch.equal(softmax(x, 1), want)
    many = (90 << 20) // (L * T * x.element_size())
    for n in (20000 // L, many):
        assert torch.equal(softmax(x.expand(n, L, T), 0), want.expand(n, L, T))
