"""Ordinary eager calls run the kernels without the registered op; everything that watches or
replaces operators still sees it (``jvp_attention._eager_call``)."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import dmad_amd
from dmad_amd import jvp_attention as ja


class _Names(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def test_only_plain_eager_calls_skip_the_op():
    x = torch.zeros(2)
    assert ja._eager_call(x, None, torch.nn.Parameter(x))
    with _Names():
        assert not ja._eager_call(x)
    with torch.overrides.BaseTorchFunctionMode():
        assert not ja._eager_call(x)
    with torch.autograd.forward_ad.dual_level():
        assert not ja._eager_call(x)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]):
        assert not ja._eager_call(x)
    seen = []
    torch.func.vmap(lambda t: seen.append(ja._eager_call(t)) or t)(torch.zeros(3, 2))
    torch.func.jvp(lambda t: seen.append(ja._eager_call(t)) or t, (x,), (x,))
    torch.jit.trace(lambda t: seen.append(ja._eager_call(t)) or t + 1, (x,), check_trace=False)
    assert seen and not any(seen)
    assert not ja._eager_call(x.as_subclass(type("Sub", (torch.Tensor,), {})))


def _mock_kernels(monkeypatch):
    """Stand-ins in plain torch for the forward and backward launches, which (like the kernels) read
    the memory of their operands and so take dense CPU tensors with data of their own only."""
    def forward(q, k, v, tq, tk, tv, sm_scale, need_mu=True, out=None):
        for t in (q, k, v, tq, tk, tv):
            assert t is None or (t.data_ptr() and not t.is_neg()), "a tensor whose memory does not hold its values"
        p = torch.softmax(q @ k.transpose(-1, -2) * sm_scale, -1)
        o = p @ v
        lse = torch.logsumexp(q @ k.transpose(-1, -2) * sm_scale, -1)
        if tq is None:
            return o, None, lse, None
        return o, torch.cat([tq, tq], -1)[..., :o.shape[-1]] + o, lse, lse.clone()

    def backward(q, k, v, tq, tk, tv, o, to, lse, mu, dout, dto, sm_scale, want_tangent_grads):
        for t in (q, k, v, tq, tk, tv, o, to, lse, mu, dout, dto):
            assert t is None or (t.data_ptr() and not t.is_neg())
        p = torch.softmax(q @ k.transpose(-1, -2) * sm_scale, -1)
        ds = p * (dout @ v.transpose(-1, -2) - (dout * o).sum(-1, keepdim=True)) * sm_scale
        grads = ds @ k, ds.transpose(-1, -2) @ q, p.transpose(-1, -2) @ dout
        tgrads = tuple(g * 2 for g in grads) if dto is not None and want_tangent_grads else (None,) * 3
        return (*grads, *tgrads)

    monkeypatch.setattr(ja, "jvp_attention_forward", forward)
    monkeypatch.setattr(ja, "jvp_attention_backward", backward)


def _call(what, xs):
    if what == "plain":
        return dmad_amd.plain_attention(*xs[:3])
    if what == "sdpa":
        from dmad_amd.sdpa import attention

        return attention(*(x.transpose(1, 2) for x in xs[:3])).transpose(1, 2)
    return dmad_amd.attention(*xs[:3], *(x if what == "full" else x.detach() for x in xs[3:]))


def _cpu_inputs(device="cpu"):
    g = torch.Generator().manual_seed(6)
    return [torch.randn((1, 2, L, 16), generator=g).to(device, torch.bfloat16).requires_grad_(True) for L in (5, 7, 7, 5, 7, 7)]


@pytest.mark.parametrize("what", ["plain", "sdpa", "jvp", "full"])
def test_meta_tensors_give_shapes(what):
    """Shapes of outputs and gradients without a GPU, through the ops' fakes."""
    xs = _cpu_inputs("meta")
    outs = _call(what, xs)
    outs = outs if isinstance(outs, tuple) else (outs,)
    for o in outs:
        assert o.is_meta and o.shape == (1, 2, 5, 16)
    leaves = xs if what == "full" else xs[:3]
    for x, g in zip(leaves, torch.autograd.grad(sum(o.sum() for o in outs), leaves)):
        assert g.is_meta and g.shape == x.shape
    with torch.no_grad():
        assert _call(what, xs)[0].is_meta


@pytest.mark.parametrize("what", ["plain", "sdpa", "jvp", "full"])
def test_batched_cotangents(monkeypatch, what):
    """is_grads_batched hands the backward one tensor of cotangents with a batch dimension that its
    shape does not show: the same gradients as one call per cotangent."""
    _mock_kernels(monkeypatch)
    xs = _cpu_inputs()
    outs = _call(what, xs)
    outs = outs[:1 if what == "jvp" else 2] if isinstance(outs, tuple) else (outs,)
    leaves = xs if what == "full" else xs[:3]
    cts = [torch.randn((3, *o.shape)).bfloat16() for o in outs]
    got = torch.autograd.grad(outs, leaves, cts, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        one = torch.autograd.grad(outs, leaves, [c[i] for c in cts], retain_graph=True)
        for a, b in zip(got, one):
            torch.testing.assert_close(a[i], b)


@pytest.mark.parametrize("what", ["plain", "jvp"])
def test_tensors_whose_memory_is_not_their_value(monkeypatch, what):
    """A negated view and a zero tensor without memory reach the kernels as ordinary tensors."""
    _mock_kernels(monkeypatch)
    with torch.no_grad():
        xs = [x.detach() for x in _cpu_inputs()]
        first = lambda o: o if isinstance(o, torch.Tensor) else o[0]  # noqa: E731
        odd = [torch._neg_view(xs[0]), xs[1], torch._efficientzerotensor(xs[2].shape, dtype=xs[2].dtype), *xs[3:]]
        same = [-xs[0], xs[1], torch.zeros_like(xs[2]), *xs[3:]]
        torch.testing.assert_close(first(_call(what, odd)), first(_call(what, same)))


def _inputs(dev, grad):
    g = torch.Generator().manual_seed(2)
    return [torch.randn((1, 2, 150, 64), generator=g).to(torch.bfloat16).to(dev).requires_grad_(grad) for _ in range(6)]


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["jvp", "plain", "full"])
def test_op_and_direct_calls_agree_bitwise(gpu, what):
    def step():
        xs = _inputs(gpu, True)
        if what == "plain":
            xs = xs[:3]
            out = (dmad_amd.plain_attention(*xs),)
        else:
            if what == "jvp":
                xs = xs[:3] + [t.detach() for t in xs[3:]]
            out = dmad_amd.attention(*xs)
        loss = sum((o.float() * (i + 1)).square().sum() for i, o in enumerate(out))
        return [*out, *torch.autograd.grad(loss, xs[:6 if what == "full" else 3])]

    direct = step()
    with _Names() as m:
        watched = step()
    ops = [n for n in m.names if "dmad" in n]
    assert len(ops) == 2 and "fwd" in ops[0] and "bwd" in ops[1], ops
    torch.cuda.synchronize()
    for a, b in zip(direct, watched):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("plain", [False, True])
def test_second_derivatives_are_still_refused(gpu, plain):
    """The gradients are kernels' outputs: differentiating them raises rather than giving zeros."""
    xs = _inputs(gpu, True)
    o = dmad_amd.plain_attention(*xs[:3]) if plain else dmad_amd.attention(*xs[:3], *(t.detach() for t in xs[3:]))[0]
    (gq,) = torch.autograd.grad(o.float().square().sum(), xs[:1], create_graph=True)
    with pytest.raises((RuntimeError, NotImplementedError)):
        torch.autograd.grad(gq.float().sum(), xs[:1])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("Lq,Lk,H", [(1, 3, 1), (130, 257, 3), (200, 4000, 2)])  # the last one splits
def test_sdpa_writes_its_layout_without_a_copy(gpu, Lq, Lk, H, dtype):
    """Without a backward the kernel writes BSHD; the values are those of the copied output."""
    from dmad_amd.sdpa import attention

    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn((2, L, H, 64), generator=g).to(dtype).to(gpu) for L in (Lq, Lk, Lk))
    with torch.no_grad():
        o = attention(q, k, v)
    ref = attention(q.requires_grad_(True), k, v)
    torch.cuda.synchronize()
    assert o.is_contiguous() and o.shape == (2, Lq, H, 64) and torch.equal(o, ref)
    if Lq > 1 and H > 1:  # else both layouts are one
        ref.mul_(2.0).sum().backward()  # the tracked output is the caller's own to change
