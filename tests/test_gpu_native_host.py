"""The native host path (csrc/host_ext.cpp) against the Python launchers it stands in for: the same kernels on the same
operands, so the same bits, in every layout it takes; and it leaves the operands it does not take to them."""
import pytest
import torch

import acsr_helpers as A
import _splat_hip as hip
import r_attention
from r_attention import RegularAttention, _AttentionFunction, attention_launcher, attention_with_grad

pytestmark = pytest.mark.gpu


def _operands(dev, B, H, L, d, dtype, layout):
    g = torch.Generator(device="cpu").manual_seed(L + d)

    def one():
        if layout == "tokens":
            return torch.randn(B, L, H, d, generator=g).to(dtype).to(dev).transpose(1, 2)
        if layout == "odd rows":  # rows that do not start on 16-byte boundaries: not an ordinary case
            return torch.randn(B, H, L, d + 1, generator=g).to(dtype).to(dev)[..., :d]
        return torch.randn(B, H, L, d, generator=g).to(dtype).to(dev)
    q, k, v = one(), one(), one()
    kT = k.transpose(2, 3)
    return q, k, (kT.contiguous() if layout == "keys" else kT), v


@pytest.mark.parametrize("layout", ["rows", "tokens", "keys", "odd rows"])
@pytest.mark.parametrize("L,masks", [(520, lambda L: A.causal_windowed_pattern(L, 99)), (333, lambda L: A.windowed_pattern(L, 40)),
                                     (384, lambda L: A.strided_patterns(L, 32, 16))])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_native_forward_equals_the_launcher(dev, layout, L, masks, dtype):
    B, H, d = 2, 3, 64
    attn = RegularAttention(B, L, H, d, masks(L), 16, 16, dev, dtype, scale=d ** -0.5)
    q, _, kT, v = _operands(dev, B, H, L, d, dtype, layout)
    first = attn([q, kT, v]).clone()   # builds the plan: the launcher
    taken = hip.host().forward(attn._native, q, kT, v, attn.rspmm_output.zero_(), attn.scale)
    assert taken == (layout != "odd rows")
    again = attn([q, kT, v])
    want = attention_launcher(q, kT, v, torch.empty_like(first), attn.segments, attn.scale, attn._plan)
    assert torch.equal(first, want) and torch.equal(again, want)


@pytest.mark.parametrize("layout", ["rows", "tokens", "odd rows"])
@pytest.mark.parametrize("L,masks", [(520, lambda L: A.causal_windowed_pattern(L, 99)), (8192, lambda L: A.strided_patterns(L, 64, 64))])
@pytest.mark.parametrize("dtype,d", [(torch.float16, 64), (torch.bfloat16, 128)])
def test_native_gradients_equal_the_python_function(dev, layout, L, masks, dtype, d):
    B, H = 2, 2
    attn = RegularAttention(B, L, H, d, masks(L), 16, 16, dev, dtype, scale=d ** -0.5)
    q, k, _, v = (t.requires_grad_(True) for t in _operands(dev, B, H, L, d, dtype, layout))
    go = torch.randn(B, H, L, d, device=dev).to(dtype)
    out = attention_with_grad(q, k, v, attn)
    got = torch.autograd.grad(out, (q, k, v), go)
    ref = _AttentionFunction.apply(q, k, v, attn)
    want = torch.autograd.grad(ref, (q, k, v), go)
    assert torch.equal(out, ref) and all(torch.equal(a, b) for a, b in zip(got, want))
    with torch.no_grad():
        assert torch.equal(attention_with_grad(q, k, v, attn), ref)


def test_native_operators_refuse_what_the_launchers_check(dev):
    """Operands of the wrong shape or type fall through to the launchers and their messages."""
    L, d = 256, 64
    attn = RegularAttention(1, L, 2, d, A.causal_windowed_pattern(L, 31), 16, 16, dev, torch.bfloat16, scale=1.0)
    q = torch.randn(1, 2, L, d, device=dev).to(torch.bfloat16)
    attn([q, q.transpose(2, 3), q])
    with pytest.raises(hip.SplatError):
        attn([q[:, :, :128], q[:, :, :128].transpose(2, 3), q[:, :, :128]])
    assert not hip.host().forward(attn._native, q, q.float().transpose(2, 3), q, attn.rspmm_output, 1.0)
    assert not hip.host().softmax(attn.segments.native(L, dev, False), q, q[:, :1])


def test_running_out_of_memory_is_the_error_a_program_catches(dev):
    """Allocations of the native path that the device's limit refuses raise what torch.empty raises, in the forward and in the
    backward, and the call works again with room."""
    L, H, d = 8192, 16, 128  # an output of 32 MB
    attn = RegularAttention(1, L, H, d, A.causal_windowed_pattern(L, 31), 16, 16, dev, torch.bfloat16, scale=d ** -0.5)
    x = [torch.randn(1, H, L, d, device=dev).to(torch.bfloat16).requires_grad_(True) for _ in range(3)]
    want = torch.autograd.grad(attention_with_grad(*x, attn).sum(), x)
    out = attention_with_grad(*x, attn)
    up = torch.ones_like(out)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = torch.cuda.get_device_properties(dev).total_memory
    fits = []
    try:
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved(dev) / room, dev)
        with pytest.raises(torch.OutOfMemoryError):
            for _ in range(64):  # what is reserved and free
                fits.append(attention_with_grad(*x, attn))
        with pytest.raises(torch.OutOfMemoryError):
            torch.autograd.grad(out, x, up, retain_graph=True)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
    got = torch.autograd.grad(out, x, up)
    assert all(torch.equal(a, b) for a, b in zip(got, want)) and len(fits) < 64


@pytest.mark.parametrize("layout", ["rows", "tokens", "keys", "odd rows"])
@pytest.mark.parametrize("L,masks", [(520, lambda L: A.causal_windowed_pattern(L, 99)), (384, lambda L: A.strided_patterns(L, 32, 16)),
                                     (301, lambda L: A.dilated_pattern(L, 20, 3))])
@pytest.mark.parametrize("dtype,d", [(torch.float32, 64), (torch.bfloat16, 64), (torch.float16, 80)])
def test_native_operators_equal_the_launchers(dev, layout, L, masks, dtype, d):
    """A forward through the three launchers, and through the one native call, which the module's forwards make; the masks of a layout that
    comes later are chosen by its first forward, and other types are the launchers' to refuse."""
    B, H = 2, 3
    attn = RegularAttention(B, L, H, d, masks(L), 16, 16, dev, dtype, scale=d ** -0.5, fused=False)
    q, _, kT, v = _operands(dev, B, H, L, d, dtype, layout)
    attn._choose_operators = lambda *_: None
    want = [t.clone() for t in (attn([q, kT, v]), attn.rsddmm_output, attn.rsoftmax_output)]
    del attn._choose_operators
    assert attn._operator_masks is None and torch.equal(attn([q, kT, v]), want[0])
    kept = attn._operator_masks
    taken = hip.host().operators(*kept, q, kT, v, attn._rsddmm_output, attn._rsoftmax_output, attn.rspmm_output.zero_(), attn.scale)
    assert taken and torch.equal(attn.rspmm_output, want[0])
    live = (torch.arange(attn.acsr_trailing_dim, device=dev) < sum(t[4] for t in attn.segments.tuples)[:, None]) if len(attn.segments) == 1 else None
    assert torch.equal(attn([q, kT, v]), want[0])
    if live is not None:
        for got, w in zip((attn.rsddmm_output, attn.rsoftmax_output), want[1:]):
            assert torch.equal(got[:, :, live], w[:, :, live])
    other = kT.contiguous() if layout != "keys" else kT.transpose(2, 3).contiguous().transpose(2, 3)
    assert None in attn._operator_masks[:2]
    assert float((attn([q, other, v]).float() - want[0].float()).abs().max()) <= 0.04
    assert None not in attn._operator_masks[:2] and torch.equal(attn([q, kT, v]), want[0])
    with pytest.raises(hip.SplatError):
        attn([q.double(), kT.double(), v.double()])


def test_the_operators_follow_the_module_s_segments(dev):
    """Another mask put in a module's place after a forward is what the next forward computes, in both layouts of K."""
    L, d, dtype = 300, 64, torch.bfloat16
    first, other = A.causal_windowed_pattern(L, 20), A.dilated_pattern(L, 21, 2)  # (rows of 21 slots, both)
    attn, want = (RegularAttention(1, L, 2, d, m, 16, 16, dev, dtype, scale=d ** -0.5, fused=False) for m in (first, other))
    q, _, kT, v = _operands(dev, 1, 2, L, d, dtype, "rows")
    for keys in (kT, kT.contiguous()):
        attn([q, keys, v])
        attn([q, keys, v])
    attn.segments = want.segments
    for keys in (kT, kT.contiguous()):
        for _ in range(2):
            assert torch.equal(attn([q, keys, v]), want([q, keys, v]))


@pytest.mark.parametrize("kind", ["along the keys", "of another type", "on the host"])
def test_the_operators_refuse_before_they_launch(dev, kind):
    """A V that is not an ordinary one leaves the native call with nothing done: the launchers run each operator, once."""
    L, d, dtype = 300, 80, torch.float16
    attn = RegularAttention(1, L, 2, d, A.causal_windowed_pattern(L, 20), 16, 16, dev, dtype, scale=d ** -0.5, fused=False)
    q, _, kT, v = _operands(dev, 1, 2, L, d, dtype, "rows")
    want = attn([q, kT, v]).clone()
    odd = {"along the keys": v.transpose(2, 3).contiguous().transpose(2, 3), "of another type": v.float(), "on the host": v.cpu()}[kind]
    attn._rsddmm_output.fill_(7.0)
    attn._rsoftmax_output.fill_(7.0)
    assert not hip.host().operators(*attn._operator_masks, q, kT, odd, attn._rsddmm_output, attn._rsoftmax_output, attn.rspmm_output, attn.scale)
    assert torch.all(attn._rsddmm_output == 7.0) and torch.all(attn._rsoftmax_output == 7.0)
    if kind == "along the keys":
        assert torch.equal(attn([q, kT, odd]), want)
    else:
        with pytest.raises(hip.SplatError):
            attn([q, kT, odd])


@pytest.mark.parametrize("layout", ["rows", "keys"])
@pytest.mark.parametrize("dtype,d", [(torch.float16, 80), (torch.float32, 64)])
def test_the_first_forward_makes_the_one_call(dev, layout, dtype, d, monkeypatch):
    """A module's first forward makes the native call of the three operators, not the launchers'; the same under stream capture where
    a forward has been before it."""
    L, B, H = 700, 2, 9
    attn, other = (RegularAttention(B, L, H, d, A.causal_windowed_pattern(L, 60), 16, 16, dev, dtype, scale=d ** -0.5, fused=False) for _ in range(2))
    q, _, kT, v = _operands(dev, B, H, L, d, dtype, layout)
    other._choose_operators = lambda *_: None
    want = other([q, kT, v]).clone()

    def launcher(*args, **kwargs):
        raise AssertionError("a launcher")
    for name in ("rsddmm_launcher", "rsoftmax_launcher", "rspmm_launcher"):
        monkeypatch.setattr(r_attention, name, launcher)
    assert torch.equal(attn([q, kT, v]), want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        attn([q, kT, v])
    for _ in range(3):
        attn.rspmm_output.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(attn.rspmm_output, want)
