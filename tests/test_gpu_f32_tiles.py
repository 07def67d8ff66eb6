"""The float32 attention kernels (16 rows a wavefront, 64 a workgroup, tiles of 32 or 16 positions; in launches of up to 32 and of up to 64 row
blocks wavefronts that share the keys of 16 and of 32 rows) against float64 where their tiles can go wrong: lengths around the edges of
rows, workgroups and row blocks, windows that begin and end inside a subtile, gathered and two-segment walks, rows without entries,
K stored either way."""
import pytest
import torch

import acsr_helpers as A
from r_attention import RegularAttention, attention_launcher, attention_with_grad

pytestmark = pytest.mark.gpu

def copies(launch, heads, L):
    """How often `heads` heads of L rows have to be there for a launch of up to 32 row blocks, of 33 to 64, or of more."""
    return {"few": 1, "some": -(-33 // (heads * -(-L // 128))), "many": -(-66 // (heads * -(-L // 128)))}[launch]


def alike(t, n):
    """The first of n equal copies of some heads (dimension 1)."""
    parts = t.detach().contiguous().view(torch.int32).chunk(n, 1)
    assert all(torch.equal(parts[0], x) for x in parts[1:])
    return t.detach().chunk(n, 1)[0]


MASKS = {
    "diagonal": lambda L: [A.causal_windowed_pattern(L, 0)],
    "causal": lambda L: [A.causal_windowed_pattern(L, 16)],
    "windowed": lambda L: [A.windowed_pattern(L, 23)],
    "dilated": lambda L: [A.dilated_pattern(L, 11, 3)],
    "strided": lambda L: A.strided_patterns(L, 9, 7),
    "far only": lambda L: A.strided_patterns(L, 9, 7)[1:],  # the first rows hold nothing
}
CASES = [(m, L, d) for m in MASKS for L in (17, 64, 257) for d in (64, 128)] + \
    [("causal", L, 64) for L in (1, 15, 16, 63, 65, 127, 128, 129, 700)] + [("dilated", L, 128) for L in (33, 130, 700)]


@pytest.mark.parametrize("launch", ["few", "many"])
@pytest.mark.parametrize("name,L,d", CASES)
def test_forward_and_gradients_against_float64(dev, name, L, d, launch):
    masks = MASKS[name](L)
    if L < 8 and name == "far only":
        pytest.skip("no entries")
    B, H = 2, 2
    g = torch.Generator().manual_seed(L + d)
    q, k, v, go = (torch.randn(B, H, L, d, generator=g) for _ in range(4))
    live = sum(m.device_mask(dev) for m in masks).cpu() > 0
    wide = [t.double().requires_grad_(True) for t in (q, k, v)]
    s = (wide[0] @ wide[1].transpose(2, 3) * d ** -0.5).masked_fill(~live, float("-inf"))
    p = torch.where(live.any(1)[:, None], torch.softmax(s, -1), torch.zeros_like(s)).masked_fill(~live, 0.0)
    want = p @ wide[2]
    grads = torch.autograd.grad(want, wide, go.double())
    n = copies(launch, B * H, L)
    attn = RegularAttention(B, L, H * n, d, masks, 16, 16, dev, torch.float32, scale=d ** -0.5)
    on = [t.repeat(1, n, 1, 1).to(dev) for t in (q, k, v)]
    for kT in (on[1].transpose(2, 3), on[1].transpose(2, 3).contiguous()):
        got = alike(attn([on[0], kT, on[2]]), n).cpu()
        assert float((got - want).detach().abs().max()) <= 1e-5
    on = [t.requires_grad_(True) for t in on]
    out = attention_with_grad(*on, attn)
    assert float((alike(out, n).cpu() - want).detach().abs().max()) <= 1e-5
    for a, b in zip(torch.autograd.grad(out, on, go.repeat(1, n, 1, 1).to(dev)), grads):
        b = torch.nan_to_num(b)
        assert float((alike(a, n).cpu() - b).abs().max()) <= 2e-5 * max(1.0, float(b.abs().max()))


# windows that start at, before and behind the middle of a tile of the row block's walk, and save the workgroup's own one or not
STARTS = {"16 to both sides": lambda L: [A.windowed_pattern(L, 16)], "17": lambda L: [A.windowed_pattern(L, 17)],
          "3": lambda L: [A.windowed_pattern(L, 3)], "40": lambda L: [A.windowed_pattern(L, 40)],
          "gathered": lambda L: [A.dilated_pattern(L, 17, 2)], "residue": lambda L: [A.dilated_pattern(L, 21, 3)],
          "two segments": lambda L: A.strided_patterns(L, 20, 18), "steps on dense columns": lambda L: A.strided_patterns(L, 30, 7)[1:]}


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("L", [130, 515])
@pytest.mark.parametrize("name", STARTS)
@pytest.mark.parametrize("launch", ["few", "some", "many"])
def test_walks_that_start_inside_a_tile(dev, name, L, d, launch):
    masks, B, H = STARTS[name](L), 1, 2
    g = torch.Generator().manual_seed(L + d)
    q, k, v = (torch.randn(B, H, L, d, generator=g) for _ in range(3))
    live = sum(m.device_mask(dev) for m in masks).cpu() > 0
    s = (q.double() @ k.double().transpose(2, 3) * d ** -0.5).masked_fill(~live, float("-inf"))
    want = torch.where(live.any(1)[:, None], torch.softmax(s, -1), torch.zeros_like(s)) @ v.double()
    n = copies(launch, B * H, L)
    attn = RegularAttention(B, L, H * n, d, masks, 16, 16, dev, torch.float32, scale=d ** -0.5)
    on = [t.repeat(1, n, 1, 1).to(dev) for t in (q, k, v)]
    got = attn([on[0], on[1].transpose(2, 3), on[2]]).clone()
    assert float((alike(got, n).cpu() - want).abs().max()) <= 1e-5
    assert torch.equal(attn([on[0], on[1].transpose(2, 3).contiguous(), on[2]]), got)
    out = torch.empty_like(got)  # without a plan table
    attention_launcher(on[0], on[1].transpose(2, 3), on[2], out, attn.segments, d ** -0.5, live_percent=attn._live_percent)
    assert torch.equal(out, got)


@pytest.mark.parametrize("d", [64, 128])
def test_listed_rows_of_the_transposed_mask(dev, d):
    """The keys of a strided far field row by row (rows cut into stretches of queries, their shares added up) against the walk
    by blocks of keys."""
    B, H, L = 1, 2, 1500
    attn = RegularAttention(B, L, H, d, A.strided_patterns(L, 64, 50), 16, 16, dev, torch.float32, scale=d ** -0.5)
    g = torch.Generator(device=dev).manual_seed(d)
    q, k, v, go = (torch.randn(B, H, L, d, generator=g, device=dev) for _ in range(4))
    x = [q, k.transpose(2, 3), v]
    one = attn.backward_pass(x, go, sparse_rows=False)
    two = attn.backward_pass(x, go, sparse_rows=True)
    for a, b in zip(one, two):
        assert float((a - b).abs().max()) <= 2e-5 * float(b.abs().max())
