"""Passes and norms as autograd nodes of their own (plain eager calls) against the registered custom
ops, which transforms and dispatch modes still see."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from test_gpu_1_pass import dev, randn

pytestmark = pytest.mark.gpu


def _pass_inputs(dtype=torch.bfloat16):
    ts = [randn((1, 2, 70, 64), dtype, s).to(dev()).requires_grad_() for s in (1, 2, 3, 4)]
    return ts + [randn((1, 2, 70), torch.float32, 5).to(dev()).requires_grad_()]


def test_pass_node_equals_op():
    from poly_attention import _ops

    do, dl = randn((1, 2, 70, 64), torch.bfloat16, 6).to(dev()), randn((1, 2, 70), torch.float32, 7).to(dev())
    got = []
    for op in (_ops._PassNode.apply, _ops.pass_fwd_op):
        ts = _pass_inputs()
        out, lse = op(*ts, None, None, True, 0.0, 0.125, False)
        torch.autograd.backward((out, lse), (do, dl))
        got.append([out, lse, *[t.grad for t in ts]])
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("angles", (False, True))
def test_rms_node_equals_op(angles):
    from poly_attention import _ops

    ang = randn((9, 64), torch.float32, 3).to(dev()) if angles else None
    got = []
    for op in (_ops._RmsNode.apply, lambda *a: _ops.rms_norm_op(*a)[0]):
        x = randn((2, 3, 9, 64), torch.bfloat16, 1).to(dev()).requires_grad_()
        w = randn((64,), torch.bfloat16, 2).to(dev()).requires_grad_()
        y = op(x, w, 1e-6, ang)
        y.backward(torch.ones_like(y))
        got.append([y, x.grad, w.grad])
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_dispatch_modes_see_the_ops():
    from poly_attention import _ops

    class Names(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.seen = set()

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.seen.add(str(func))
            return func(*args, **(kwargs or {}))

    q, k, v, vmul, bias = _pass_inputs()
    w = torch.ones(64, device=dev(), dtype=torch.bfloat16, requires_grad=True)
    with Names() as names:
        _ops.attn_pass(q, k, v, bias=bias, causal=True)
        _ops.rms_norm(q, w, None)
    assert "polyattn.pass_fwd.default" in names.seen and "polyattn.rms_norm.default" in names.seen


def test_no_silent_second_derivative():
    from poly_attention import _ops

    q, k, v, vmul, bias = _pass_inputs()
    out, _ = _ops.attn_pass(q, k, v, causal=True)
    (dq,) = torch.autograd.grad(out.float().sum(), q, create_graph=True)
    with pytest.raises(RuntimeError):
        dq.float().sum().backward()


def test_batched_grads():
    """is_grads_batched: each gradient of the batch as by itself, through a pass, a norm and the norms
    of a layer."""
    from poly_attention import _ops

    q, k, v, vmul, bias = _pass_inputs()
    w = torch.ones(64, device=dev(), dtype=torch.bfloat16, requires_grad=True)
    out, _ = _ops.attn_pass(q, k, v, bias=bias, causal=True)
    normed = _ops.rms_norm(q, w, None)
    layer = _ops.rms_norm_layer([q, k], [w, w], [None, None])[1]
    for y, xs in ((out, (q, k, v, bias)), (normed, (q, w)), (layer, (k, w))):
        dys = randn((3, *y.shape), torch.bfloat16, 8).to(dev())
        got = torch.autograd.grad(y, xs, dys, retain_graph=True, is_grads_batched=True, allow_unused=True)
        for i in range(3):
            want = torch.autograd.grad(y, xs, dys[i], retain_graph=True, allow_unused=True)
            for a, b in zip(got, want):
                assert torch.equal(a[i], b)


def _layer(order):
    from poly_attention import NPolyAttention, PolyAttention

    torch.manual_seed(0)
    kw = dict(dim=128, dim_head=64, heads=2, causal=True)
    layer = PolyAttention(**kw) if order == 2 else NPolyAttention(order=order, **kw)
    layer = layer.to(dev()).to(torch.bfloat16)
    x = randn((2, 40, 128), torch.bfloat16, 9).to(dev()).requires_grad_()
    return x, layer(x), [x, *(p for p in layer.parameters() if p.requires_grad)]


def test_batched_grads_of_a_layer():
    """A whole order-3 layer, whose passes and norms write their gradients into the head-split
    projection's: each gradient of the batch as by itself (to the rounding of a batched product
    in torch), and an ordinary backward afterwards as before."""
    x, y, xs = _layer(3)
    dys = randn((3, *y.shape), torch.bfloat16, 10).to(dev())
    want = [torch.autograd.grad(y, xs, dys[i], retain_graph=True) for i in range(3)]
    got = torch.autograd.grad(y, xs, dys, retain_graph=True, is_grads_batched=True)
    for i in range(3):
        for a, b in zip(got, want[i]):
            assert (a[i].float() - b.float()).norm() <= 1e-2 * b.float().norm()
    again = torch.autograd.grad(y, xs, dys[0])
    for a, b in zip(again, want[0]):
        assert torch.equal(a, b)


def test_batched_grads_of_the_order2_chain_are_refused():
    """One node for the chain: a clear error, and the graph stays usable."""
    x, y, xs = _layer(2)
    dy = randn(tuple(y.shape), torch.bfloat16, 10).to(dev())
    want = torch.autograd.grad(y, xs, dy, retain_graph=True)
    with pytest.raises(RuntimeError, match="one gradient at a time"):
        torch.autograd.grad(y, xs, torch.stack([dy, dy]), retain_graph=True, is_grads_batched=True)
    for a, b in zip(torch.autograd.grad(y, xs, dy), want):
        assert torch.equal(a, b)
