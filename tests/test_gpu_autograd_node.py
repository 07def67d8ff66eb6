"""The autograd node of the native host path (csrc/host_ext.cpp) where a program does more than call backward: it must do what
the Python function that it stands in for does."""
import gc
import threading

import pytest
import torch
import torch.autograd.forward_ad as forward_ad

import acsr_helpers as A
import _splat_hip as hip
from r_attention import RegularAttention, _AttentionFunction, attention_with_grad

pytestmark = pytest.mark.gpu

B, H, L, D = 1, 2, 300, 64


def _module(dev, dtype=torch.bfloat16, scale=D ** -0.5):
    return RegularAttention(B, L, H, D, A.causal_windowed_pattern(L, 70), 16, 16, dev, dtype, scale=scale)


def _operands(dev, dtype=torch.bfloat16):
    g = torch.Generator(device="cpu").manual_seed(5)
    return [torch.randn(B, H, L, D, generator=g).to(dtype).to(dev).requires_grad_(True) for _ in range(3)]


@pytest.mark.parametrize("which", [0, 1, 2])
def test_a_tangent_is_refused_and_not_dropped(dev, which):
    attn, x = _module(dev), _operands(dev)
    with forward_ad.dual_level():
        x[which] = forward_ad.make_dual(x[which], torch.ones_like(x[which]))
        with pytest.raises(NotImplementedError, match="jvp"):
            attention_with_grad(*x, attn)
    with forward_ad.dual_level():  # the level alone is nothing to refuse
        assert attention_with_grad(*_operands(dev), attn).grad_fn.name() == "AttendBackward"


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning", "ignore::DeprecationWarning")
def test_a_trace_follows_its_inputs(dev):
    attn = _module(dev)
    attention_with_grad(*_operands(dev), attn)  # (the plan's kernels are not for the trace)
    traced = torch.jit.trace(lambda q, k, v: attention_with_grad(q, k, v, attn), tuple(_operands(dev)), check_trace=False)
    other = [(2 * t).detach().requires_grad_(True) for t in _operands(dev)]
    assert torch.equal(traced(*other), attention_with_grad(*other, attn))


def test_functorch_transforms_get_the_message_that_names_them(dev):
    attn = _module(dev)
    q, k, v = _operands(dev)
    with pytest.raises(RuntimeError, match="functorch transforms"):
        torch.vmap(lambda a: attention_with_grad(a, k, v, attn))(q[None])
    with pytest.raises(RuntimeError, match="functorch transforms"):
        torch.func.grad(lambda a: attention_with_grad(a, k, v, attn).float().sum())(q.detach())


def test_a_scale_the_kernels_refuse_is_a_splat_error(dev):
    attn = _module(dev, scale=-1.0)
    with pytest.raises(hip.SplatError, match=r"^splat_attention_fwd_hinted failed \(code -5\): .*scale must be > 0"):
        attention_with_grad(*_operands(dev), attn)


def _gradients(f, x):
    out = f(*x)
    return [out, *torch.autograd.grad(out, x, torch.linspace(-1, 1, out.numel(), device=out.device).view(out.shape).to(out.dtype))]


def test_saved_tensor_hooks_see_what_the_python_function_saves(dev):
    """The same tensors in the same order go through the hooks, and what they hand back is what the backward reads."""
    attn, x = _module(dev), _operands(dev)
    want = _gradients(lambda q, k, v: attention_with_grad(q, k, v, attn), x)
    seen = {}
    for name, f in (("node", attention_with_grad), ("function", _AttentionFunction.apply)):
        packed = seen[name] = []

        def pack(t):
            packed.append((t.dtype, tuple(t.shape)))
            return t.cpu()
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(dev)):
            got = _gradients(lambda q, k, v: f(q, k, v, attn), x)
        assert all(torch.equal(a, b) for a, b in zip(got, want)), name
    assert seen["node"] == seen["function"] and len(seen["node"]) == 5


@pytest.mark.parametrize("swap", [lambda t: t.float() if t.dim() == 4 else t, lambda t: t[:, :, :-1], lambda t: t.cpu(),
                                  lambda t: t.double() if t.dim() == 3 else t])
def test_a_saved_tensor_that_came_back_as_another_is_refused(dev, swap):
    attn, x = _module(dev), _operands(dev)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, swap):
        out = attention_with_grad(*x, attn)
        with pytest.raises(hip.SplatError, match="came back with another type, shape or device"):
            torch.autograd.grad(out.sum(), x)


def test_a_saved_tensor_that_came_back_on_odd_rows_is_copied(dev):
    attn, x = _module(dev), _operands(dev)
    want = _gradients(lambda q, k, v: attention_with_grad(q, k, v, attn), x)

    def odd(t):
        wide = torch.empty(*t.shape[:-1], t.shape[-1] + 1, dtype=t.dtype, device=t.device)[..., 1:]
        return wide.copy_(t)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, odd):
        got = _gradients(lambda q, k, v: attention_with_grad(q, k, v, attn), x)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, grad):
        return None


def test_zeros_where_no_gradient_arrives(dev):
    attn, x = _module(dev), _operands(dev)
    got = torch.autograd.grad(_NoGradient.apply(attention_with_grad(*x, attn)).sum(), x)
    assert all(g.shape == t.shape and not g.any() for g, t in zip(got, x))


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.float16, 128), (torch.float32, 64), (torch.bfloat16, 80)])
@pytest.mark.parametrize("dims", [(2,), (0, 1), (0, 1, 2), (3,)])
def test_gradients_of_sums_arrive_with_strides_of_zero(dev, dtype, d, dims):
    """The gradient of a sum is one tensor expanded along the summed dimensions: the same as its copy in memory."""
    attn = RegularAttention(B, L, H, d, A.causal_windowed_pattern(L, 70), 16, 16, dev, dtype, scale=d ** -0.5)
    g = torch.Generator(device="cpu").manual_seed(6)
    x = [torch.randn(B, H, L, d, generator=g).to(dtype).to(dev).requires_grad_(True) for _ in range(3)]
    up = torch.randn(B, H, L, d, generator=g).to(dtype).to(dev).sum(dim=dims, keepdim=True)
    for f in (attention_with_grad, _AttentionFunction.apply):
        out = f(*x, attn)
        got = torch.autograd.grad(out.sum(dim=dims, keepdim=True), x, up, retain_graph=True)
        want = torch.autograd.grad(out, x, up.expand_as(out).contiguous())
        assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("reentrant", [False, True])
def test_checkpointing_gives_the_same_gradients(dev, reentrant):
    from torch.utils.checkpoint import checkpoint
    attn, x = _module(dev), _operands(dev)
    want = _gradients(lambda q, k, v: attention_with_grad(q, k, v, attn), x)
    up = torch.linspace(-1, 1, want[0].numel(), device=dev).view(want[0].shape).to(want[0].dtype)
    out = checkpoint(lambda q, k, v: attention_with_grad(q, k, v, attn), *x, use_reentrant=reentrant)
    out.backward(up)
    assert torch.equal(out, want[0]) and all(torch.equal(t.grad, g) for t, g in zip(x, want[1:]))


def test_the_backward_outlives_the_module(dev):
    """What the backward reads of the mask belongs to the node: metadata and plans of a module that is gone, with their memory
    written over by whatever is allocated next."""
    x = _operands(dev)
    want = _gradients(lambda q, k, v: attention_with_grad(q, k, v, _module(dev)), x)
    attn = _module(dev)
    out = attention_with_grad(*x, attn)
    del attn
    gc.collect()
    rubbish = [torch.full((n,), -1, dtype=torch.int32, device=dev) for n in (64, 128, 256, 320, 512, 1024, 4096, 16384) for _ in range(32)]
    got = torch.autograd.grad(out, x, torch.linspace(-1, 1, out.numel(), device=dev).view(out.shape).to(out.dtype))
    assert all(torch.equal(a, b) for a, b in zip(got, want[1:])) and len(rubbish) == 256


def test_the_graph_is_freed_kept_and_guarded_as_usual(dev):
    attn, x = _module(dev), _operands(dev)
    out = attention_with_grad(*x, attn)
    first = torch.autograd.grad(out.sum(), x, retain_graph=True)
    again = torch.autograd.grad(out.sum(), x)
    assert all(torch.equal(a, b) for a, b in zip(first, again))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out.sum(), x)
    out = attention_with_grad(*x, attn)
    with torch.no_grad():
        x[1].mul_(2)
    with pytest.raises(RuntimeError, match="inplace operation"):
        torch.autograd.grad(out.sum(), x)


@pytest.mark.parametrize("which", [0, 1, 2])
def test_hooks_and_inputs_that_need_no_gradient(dev, which):
    attn, x = _module(dev), _operands(dev)
    want = torch.autograd.grad(attention_with_grad(*x, attn).sum(), x)[which]
    alone = [t if i == which else t.detach() for i, t in enumerate(x)]
    out = attention_with_grad(*alone, attn)
    seen = []
    out.grad_fn.register_hook(lambda grads_in, grads_out: seen.append((len(grads_in), len(grads_out))))
    x[which].register_hook(lambda g: 2 * g)
    got, = torch.autograd.grad(out.sum(), alone[which])
    assert torch.equal(got, 2 * want) and seen == [(3, 1)]


def test_threads_with_streams_of_their_own(dev):
    """Forward and backward of one module from two threads at once, each on its stream: every call has tensors of its own."""
    attn = _module(dev)
    want = _gradients(lambda q, k, v: attention_with_grad(q, k, v, attn), _operands(dev))
    torch.cuda.synchronize()
    found, failed = [], []

    def work():
        try:
            with torch.cuda.stream(torch.cuda.Stream(device=dev)):
                x = _operands(dev)
                for _ in range(20):
                    found.append(_gradients(lambda q, k, v: attention_with_grad(q, k, v, attn), x))
                torch.cuda.current_stream(dev).synchronize()
        except Exception as e:  # noqa: BLE001
            failed.append(e)
    threads = [threading.Thread(target=work) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not failed and len(found) == 40
    assert all(torch.equal(a, b) for got in found for a, b in zip(got, want))
