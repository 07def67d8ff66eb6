"""The float32 forward and backward on split operands against float64: what the parts hold, and what they do not (taken again in
float32 arithmetic).  Forwards in launches of few, some and many row blocks, which three kernels take."""
import pytest
import torch

import acsr_helpers as A
from r_attention import RegularAttention, attention_launcher, attention_with_grad
from test_gpu_f32_tiles import alike, copies

pytestmark = pytest.mark.gpu


LAUNCHES = pytest.mark.parametrize("launch", ["few", "some", "many"])


def case(dev, masks, B, H, L, d, seed, scale_q=1.0, scale_k=1.0, scale_v=1.0, launch="few"):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(B, H, L, d, generator=g) * s for s in (scale_q, scale_k, scale_v))
    live = sum(m.device_mask(dev) for m in masks).cpu() > 0
    s = (q.double() @ k.double().transpose(2, 3) * d ** -0.5).masked_fill(~live, float("-inf"))
    want = torch.softmax(s, -1) @ v.double()
    n = copies(launch, B * H, L)
    attn = RegularAttention(B, L, H * n, d, masks, 16, 16, dev, torch.float32, scale=d ** -0.5)
    q, k, v = (t.repeat(1, n, 1, 1).to(dev) for t in (q, k, v))
    return attn, [q, k.transpose(2, 3), v], want, live


def error(got, want):
    got = alike(got, got.shape[1] // want.shape[1])
    return float((got.double().cpu() - want).norm() / want.norm())


# scores of N(0, 1) operands are rounded to 2^-24 of up to 5 or so, the sums behind them as often as they have terms: 1e-6 is three
# times what that comes to, and far below what an operand's missing part would give (2^-17)
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("q,k,v", [(1, 1, 1), (1, 1, 1e-30), (1, 1, 1e-36), (1, 1, 1e36), (1e-20, 1e20, 1), (1e-35, 1e35, 1), (1e35, 1e-35, 1), (1e-36, 1, 1)])
@LAUNCHES
def test_scales_of_the_operands(dev, d, q, k, v, launch):
    attn, x, want, _ = case(dev, [A.causal_windowed_pattern(401, 149)], 1, 2, 401, d, d, q, k, v, launch)
    assert error(attn(x), want) <= 1e-6


@pytest.mark.parametrize("d", [64, 128])
@LAUNCHES
def test_scores_that_rise_along_the_walk(dev, d, launch):
    """Later keys outrun the references of the first tiles by far more than an exponential holds."""
    attn, x, want, _ = case(dev, [A.causal_windowed_pattern(300, 199)], 1, 2, 300, d, 3 * d, launch=launch)
    x[1].mul_(torch.linspace(0.1, 60.0, 300, device=dev))
    s = (x[0][:, :2].double() @ x[1][:, :2].double() * d ** -0.5).cpu()
    live = A.causal_windowed_pattern(300, 199).device_mask(dev).cpu() > 0
    want = torch.softmax(s.masked_fill(~live, float("-inf")), -1) @ x[2][:, :2].double().cpu()
    assert error(attn(x), want) <= 1e-6 * float(s.abs().max())  # a score's rounding is relative to it


@pytest.mark.parametrize("keys_along", [False, True])
@pytest.mark.parametrize("L,d", [(400, 64), (400, 128), (96, 64)])
@LAUNCHES
def test_values_that_are_not_finite_reach_the_rows_that_see_them(dev, L, d, keys_along, launch):
    w = 40
    attn, x, want, live = case(dev, [A.causal_windowed_pattern(L, w - 1)], 1, 2, L, d, L + d, launch=launch)
    clean = attn(x).clone()
    x[2][:, :, 50, 3] = float("inf")
    x[2][:, :, 50, 7] = 3.4e38  # above what a bfloat16 holds
    x[1][:, 1, :, 9] = float("nan")
    x[0][:, 0, 70, 2] = float("inf")
    if keys_along:
        x[1] = x[1].contiguous()
    got = attn(x)
    sees_v, sees_k = live[:, 50].to(dev), live[:, 9].to(dev)
    assert bool(torch.isnan(got[:, 1, sees_k]).all()) and bool(torch.isnan(got[:, 0, 70]).all())
    ok = sees_v.clone()
    ok[70] = False
    assert bool((got[:, 0, ok, 3] == float("inf")).all()) and bool((got[:, 0, ok, 7] > 1e35).all())
    rest = torch.ones_like(got, dtype=torch.bool)
    rest[:, 1, sees_k] = False
    rest[:, 0, 70] = False
    rest[:, :, sees_v, 3] = False
    rest[:, :, sees_v, 7] = False
    assert bool(torch.isfinite(got[rest]).all()) and float((got[rest] - clean[rest]).abs().max()) <= 1e-5


def gradients(dev, d, L, scale_q, scale_k, scale_v, scale_g, seed=0, change=None):
    masks = [A.causal_windowed_pattern(L, 69)]
    g = torch.Generator().manual_seed(seed + d)
    q, k, v, go = (torch.randn(1, 2, L, d, generator=g) * s for s in (scale_q, scale_k, scale_v, scale_g))
    if change is not None:
        change(q, k, v, go)
    live = masks[0].device_mask(dev).cpu() > 0
    wide = [t.double().requires_grad_(True) for t in (q, k, v)]
    p = torch.softmax((wide[0] @ wide[1].transpose(2, 3) * d ** -0.5).masked_fill(~live, float("-inf")), -1)
    want = torch.autograd.grad(p @ wide[2], wide, go.double())
    attn = RegularAttention(1, L, 2, d, masks, 16, 16, dev, torch.float32, scale=d ** -0.5)
    on = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
    got = torch.autograd.grad(attention_with_grad(*on, attn), on, go.to(dev))
    return got, want, live


# as above, through one more product and a difference that may cancel
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("q,k,v,g", [(1, 1, 1, 1), (1, 1, 1, 1e-30), (1, 1, 1, 1e-36), (1, 1, 1e-34, 1), (1, 1, 1e-20, 1e20),
                                     (1e-34, 1, 1, 1), (1, 1e-34, 1, 1), (1e30, 1e-30, 1, 1), (1, 1, 1e15, 1e15)])
def test_gradients_at_scales_of_the_operands(dev, d, q, k, v, g):
    got, want, _ = gradients(dev, d, 211, q, k, v, g)
    for a, b in zip(got, want):
        if float(b.abs().max()) > 1e-35:  # (below, float32 itself is subnormal)
            assert error(a, b) <= 3e-6


@pytest.mark.parametrize("d", [64, 128])
def test_gradients_that_are_not_finite_stay_where_they_belong(dev, d):
    def spoil(q, k, v, go):
        go[0, 0, 100, 5] = float("inf")
        v[0, 1, 20, 3] = float("nan")
    clean, _, live = gradients(dev, d, 211, 1, 1, 1, 1)
    got, _, _ = gradients(dev, d, 211, 1, 1, 1, 1, change=spoil)
    sees, seen = live[:, 20].to(dev), live[100].to(dev)  # the rows that see key 20, the keys that row 100 sees
    assert not bool(torch.isfinite(got[0][0, 0, 100]).any()) and not bool(torch.isfinite(got[2][0, 0, seen, 5]).any())
    assert not bool(torch.isfinite(got[0][0, 1, sees]).any())
    rows = torch.arange(211, device=dev) != 100
    assert torch.allclose(got[0][0, 0, rows], clean[0][0, 0, rows], rtol=0, atol=1e-5)
    assert torch.allclose(got[0][0, 1, ~sees], clean[0][0, 1, ~sees], rtol=0, atol=1e-5)
    for i in (1, 2) if d == 64 else ():  # (at d = 128 dK and dV are float32 products, where 0 * inf of a tile's masked positions is NaN)
        assert torch.allclose(got[i][0, 0, ~seen], clean[i][0, 0, ~seen], rtol=0, atol=1e-5)


def small(at):
    """Column 5 of one operand far below the others."""
    def change(*x):
        x[at][..., 5] *= 1e-36
    return change


def column_error(got, want):
    got = alike(got, got.shape[1] // want.shape[1])
    return float((got[..., 5].double().cpu() - want[..., 5]).norm() / want[..., 5].norm())


# what the kernel splits itself, dS, is small where dO and V are so together, and Q or K may make up for it.  (The bounds here are those of
# test_gradients_at_scales_of_the_operands: nothing below is smaller than float32's normal values.)
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("q,k,v,g", [(1, 1, 1e-16, 1e-17), (1, 1, 1e-17, 1e-17), (1e-20, 1e20, 1e-17, 1e-18), (1e20, 1e-20, 1e-18, 1e-17), (1, 1, 1e-19, 1e-17)])
def test_gradients_of_small_inner_values(dev, d, q, k, v, g):
    got, want, _ = gradients(dev, d, 211, q, k, v, g)
    for a, b in zip(got, want):
        if float(b.abs().max()) > 1e-36:
            assert error(a, b) <= 3e-6


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("operand,gradient", [(1, 0), (0, 1), (3, 2)])  # K and dQ, Q and dK, dO and dV
def test_gradients_of_a_small_column(dev, d, operand, gradient):
    got, want, _ = gradients(dev, d, 211, 1, 1, 1, 1, change=small(operand))
    assert column_error(got[gradient], want[gradient]) <= 3e-6


def unlikely_key(q, k, *_):
    """Key 30 scores -80 with every row: probabilities of about 2^-122.  The rounding of such a score, 2^-25 of it a term or so, is one of its
    probability 80 times as large: 2e-5 is four times that."""
    q[..., 0] = 8.0
    k[..., 0] = 0.0
    k[..., 30, :] = 0.0
    k[..., 30, 0] = -80.0 / 8.0 * q.shape[-1] ** 0.5


@pytest.mark.parametrize("d", [64, 128])
def test_gradients_of_an_unlikely_key(dev, d):
    got, want, _ = gradients(dev, d, 211, 1, 1, 1, 1, change=unlikely_key)
    for i in (1, 2):
        a, b = got[i][:, :, 30].double().cpu(), want[i][:, :, 30]
        assert float(b.abs().max()) > 1e-37
        assert float((a - b).norm() / b.norm()) <= 2e-5


@pytest.mark.parametrize("keys_along", [False, True])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("unlikely", [False, True])
@LAUNCHES
def test_forward_of_a_small_column(dev, d, unlikely, keys_along, launch):
    """A column of V that is small, or that only an unlikely key has."""
    L, masks = 211, [A.causal_windowed_pattern(211, 69)]
    g = torch.Generator().manual_seed(d)
    q, k, v = (torch.randn(1, 2, L, d, generator=g) for _ in range(3))
    if unlikely:
        unlikely_key(q, k)
        v[..., 5] = 0.0
        v[..., 30, 5] = 1.0
    else:
        small(2)(q, k, v)
    live = masks[0].device_mask(dev).cpu() > 0
    want = torch.softmax((q.double() @ k.double().transpose(2, 3) * d ** -0.5).masked_fill(~live, float("-inf")), -1) @ v.double()
    n = copies(launch, 2, L)
    attn = RegularAttention(1, L, 2 * n, d, masks, 16, 16, dev, torch.float32, scale=d ** -0.5)
    q, k, v = (t.repeat(1, n, 1, 1).to(dev) for t in (q, k, v))
    kT = k.transpose(2, 3)
    got = attn([q, kT.contiguous() if keys_along else kT, v])
    assert error(got, want) <= 1e-6 * (20 if unlikely else 1)
    rows = live[:, 30] if unlikely else torch.ones(L, dtype=torch.bool)
    assert column_error(got[:, :, rows.to(dev)], want[:, :, rows]) <= (2e-5 if unlikely else 1e-6)


WALKS = {"windowed": lambda L: [A.windowed_pattern(L, 23)], "gathered": lambda L: [A.dilated_pattern(L, 11, 3)],
         "two segments": lambda L: A.strided_patterns(L, 20, 18), "steps on dense columns": lambda L: A.strided_patterns(L, 30, 7)[1:]}


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("L", [130, 257])
@pytest.mark.parametrize("name", list(WALKS))
@LAUNCHES
def test_rows_taken_again_on_every_walk(dev, name, L, d, launch):
    """Column 0 of Q and V beyond what the parts hold, of K and dO zero: the same scores, every row in float32 arithmetic."""
    masks, B, H = WALKS[name](L), 1, 2
    g = torch.Generator().manual_seed(L + d)
    q, k, v, go = (torch.randn(B, H, L, d, generator=g) for _ in range(4))
    q[..., 0] = v[..., 0] = 2.0 ** 90
    k[..., 0] = go[..., 0] = 0.0
    live = sum(m.device_mask(dev) for m in masks).cpu() > 0
    wide = [t.double().requires_grad_(True) for t in (q, k, v)]
    s = (wide[0] @ wide[1].transpose(2, 3) * d ** -0.5).masked_fill(~live, float("-inf"))
    p = torch.where(live.any(1)[:, None], torch.softmax(s, -1), torch.zeros_like(s)).masked_fill(~live, 0.0)
    want = p @ wide[2]
    grads = [torch.nan_to_num(t) for t in torch.autograd.grad(want, wide, go.double())]
    want = want.detach()

    n = copies(launch, B * H, L)

    def close(got, want):  # N(0, 1) columns, and column 0, which may be 2^90 times as large
        got = alike(got, n)
        for part in (slice(0, 1), slice(1, None)):
            a, b = got[..., part].double().cpu(), want[..., part]
            assert float((a - b).abs().max()) <= 2e-5 * max(1.0, float(b.abs().max()))

    attn = RegularAttention(B, L, H * n, d, masks, 16, 16, dev, torch.float32, scale=d ** -0.5)
    on = [t.repeat(1, n, 1, 1).to(dev) for t in (q, k, v)]
    for kT in (on[1].transpose(2, 3), on[1].transpose(2, 3).contiguous()):
        close(attn([on[0], kT, on[2]]), want)
        out = torch.empty_like(on[0])  # without a plan table
        attention_launcher(on[0], kT, on[2], out, attn.segments, d ** -0.5, live_percent=attn._live_percent)
        close(out, want)
    on = [t.requires_grad_(True) for t in on]
    for a, b in zip(torch.autograd.grad(attention_with_grad(*on, attn), on, go.repeat(1, n, 1, 1).to(dev)), grads):
        close(a, b)


@pytest.mark.parametrize("d", [64, 128])
def test_listed_rows_taken_again(dev, d):
    B, H, L = 1, 2, 700
    attn = RegularAttention(B, L, H, d, A.strided_patterns(L, 64, 50), 16, 16, dev, torch.float32, scale=d ** -0.5)
    g = torch.Generator(device=dev).manual_seed(d)
    q, k, v, go = (torch.randn(B, H, L, d, generator=g, device=dev) for _ in range(4))
    k[..., 0] = go[..., 0] = 0.0
    far = [t.clone() for t in (q, v)]
    for t in far:
        t[..., 0] = 2.0 ** 90
    clean = attn.backward_pass([q, k.transpose(2, 3), v], go, sparse_rows=True)
    again = attn.backward_pass([far[0], k.transpose(2, 3), far[1]], go, sparse_rows=True)
    for a, b in zip(again, clean):
        assert float((a - b)[..., 1:].abs().max()) <= 2e-5 * float(b.abs().max())


@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("L", [64, 130, 257])
@pytest.mark.parametrize("masks", [lambda L: A.causal_windowed_pattern(L, 39), lambda L: A.dilated_pattern(L, 20, 3), lambda L: A.strided_patterns(L, 24, 16)],
                         ids=["causal", "dilated", "strided"])
def test_gradients_of_keys_in_many_workgroups_are_those_of_few(dev, masks, L, large):
    """dK and dV at d = 64 in a launch beyond two workgroups a CU, whose kernel is another one, against the same heads in a launch of few: the same
    operations in the same order, so the same bits; ``large``: rows that the split operands do not hold, one of them infinite."""
    g = torch.Generator(device=dev).manual_seed(L)
    x = [torch.randn(1, 2, L, 64, generator=g, device=dev) for _ in range(4)]
    if large:
        x[1][0, 0, L // 2] *= 1e30
        x[3][0, 1, L // 3, 5] = float("inf")
    times = 513 // (2 * ((L + 127) // 128) * 2) + 1
    one, other = (RegularAttention(1, L, 2 * n, 64, masks(L), 16, 16, dev, torch.float32, scale=0.125) for n in (1, times))
    out, lse = (t.clone() for t in one.forward_with_stats([x[0], x[1].transpose(2, 3), x[2]]))
    few = one.backward_pass([x[0], x[1].transpose(2, 3), x[2]], x[3], lse, out)
    q, k, v, go, out = (t.repeat(1, times, 1, 1) for t in (*x, out))
    many = other.backward_pass([q, k.transpose(2, 3), v], go, lse.repeat(1, times, 1), out)
    for nm, a, b in zip(("dq", "dk", "dv"), few, many):
        assert large or bool(torch.isfinite(a).all()), nm
        assert torch.equal(torch.nan_to_num(a.repeat(1, times, 1, 1), nan=7e37), torch.nan_to_num(b, nan=7e37)), nm
