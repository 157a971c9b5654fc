"""The kernels that read transposed copies (16-, 32-, 256-wide heads and the full derivative of
64-wide ones), at lengths around the copies' tiles: 64 rows (wide heads) or 128 (up to 32), rows
in pairs, zero rows up to a multiple of 64. Against the float64 oracle; strided views as the
models pass them. Rounded P and outputs put 16-bit results within 1e-2 of it; a row or column of
a copy in the wrong place is off by order 1."""
import pytest
import torch

from oracle import attention as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,full", [(16, False), (32, False), (256, False), (16, True), (32, True), (64, True)])
@pytest.mark.parametrize("Lq,Lk", [(1, 1), (63, 65), (64, 128), (129, 127), (191, 257)])
def test_lengths_around_the_tiles(gpu, D, full, Lq, Lk):
    from dmad_amd.jvp_attention import jvp_attention_backward, jvp_attention_forward

    print(f"case copies D={D} full={full} {Lq} {Lk}", flush=True)
    g = torch.Generator().manual_seed(Lq + D)

    def r(L, std=1.0):
        return (torch.randn((2, L, 3, D), generator=g, dtype=torch.float64) * std).to(torch.bfloat16).transpose(1, 2)

    xs = [r(Lq), r(Lk), r(Lk), r(Lq, 0.1), r(Lk, 0.1), r(Lk, 0.1), r(Lq), r(Lq, 0.1)]
    q, k, v, tq, tk, tv, do, dto = (x.to(gpu) for x in xs)
    s = D ** -0.5
    o, to, lse, mu = jvp_attention_forward(q, k, v, tq, tk, tv, s)
    got = jvp_attention_backward(q, k, v, tq, tk, tv, o, to, lse, mu, do, dto if full else None, s, full)
    torch.cuda.synchronize()
    x64 = [x.double() for x in xs]
    ro, rto, _, _ = orc.jvp_closed_form(*x64[:6])
    ref = orc.grads_full(*x64) if full else orc.grads_dout_only(*x64[:3], x64[6])
    if Lk == 1:  # one key: O = V, and the gradients of Q and K vanish up to rounding
        assert orc.rel_l2(o.cpu(), ro) <= 1e-2 and orc.rel_l2(got[2].cpu(), ref[2]) <= 1e-2
        return
    assert orc.rel_l2(o.cpu(), ro) <= 1e-2 and orc.rel_l2(to.cpu(), rto) <= 1e-2
    for name, a, b in zip(("dq", "dk", "dv", "dtq", "dtk", "dtv"), got, ref):
        assert orc.rel_l2(a.cpu(), b) <= 1e-2, name
