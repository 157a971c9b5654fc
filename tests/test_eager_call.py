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
