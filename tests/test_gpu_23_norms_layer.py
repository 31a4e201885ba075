"""The q/k norms of a layer in one launch each way (pa_rmsnorm_many) against the single norms: the same
bits in y and dx; dweight is the same rows in another fixed order of partial sums."""

import pytest
import torch

from test_gpu_1_pass import dev, randn

pytestmark = pytest.mark.gpu
param = pytest.mark.parametrize


def _inputs(dtype, wdtype, count, n, d, heads=5):
    proj = randn((2, n, count * heads * d), dtype, 1).to(dev())
    xs = [p.detach() for p in proj.view(2, n, count, heads, d).permute(2, 0, 3, 1, 4)]
    if count > 2:  # another head count and storage order
        xs[1] = xs[1][:, :2].contiguous()
    ws = [(1 + 0.1 * randn((d,), torch.float32, 10 + k)).to(wdtype).to(dev()) for k in range(count)]
    return [x.requires_grad_() for x in xs], [w.requires_grad_() for w in ws]


@param("dtype,wdtype", ((torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32),
                        (torch.float32, torch.float32)))
@param("count", (1, 3, 4))
@param("n,d,rot", ((1, 64, 64), (130, 64, None), (77, 128, 32), (5, 8, 8), (33, 256, None)))
def test_norms_of_a_layer_match_single_norms(dtype, wdtype, count, n, d, rot):
    from poly_attention import _ops

    ang = None if rot is None else torch.rand(n, rot, device=dev()) * 50
    eps = [None, 1e-6, 1e-5, None][:count]
    xs, ws = _inputs(dtype, wdtype, count, n, d)
    dys = [randn(tuple(x.shape), dtype, 20 + k).to(dev()) for k, x in enumerate(xs)]
    many = _ops.rms_norm_layer(xs, ws, eps, ang)
    got = torch.autograd.grad(many, xs + ws, dys)
    with torch.no_grad():
        assert all(torch.equal(a, b) for a, b in zip(many, _ops.rms_norm_layer(xs, ws, eps, ang)))
    for k in range(count):
        one = _ops.rms_norm(xs[k], ws[k], eps[k], ang)
        dx, dw = torch.autograd.grad(one, (xs[k], ws[k]), dys[k])
        assert torch.equal(many[k], one) and torch.equal(got[k], dx)
        # one rounding to the weight's dtype, and the fp32 sum of the rows in another order: each term
        # is at most |dy| |x| rstd <= max|dy| sqrt(d), and a sum of m terms moves by m eps of their size
        rows = xs[k].numel() // d
        terms = float(dys[k].float().abs().max()) * d ** 0.5 * rows
        bound = torch.finfo(wdtype).eps * dw.float().abs() + 2 ** -23 * terms
        assert bool(((got[count + k].float() - dw.float()).abs() <= bound).all())


def test_unused_norm_and_refusals():
    from poly_attention import _ops

    xs, ws = _inputs(torch.bfloat16, torch.bfloat16, 3, 9, 64)
    ys = _ops.rms_norm_layer(xs, ws, [None] * 3)
    got = torch.autograd.grad((ys[0].float().sum() + ys[2].float().sum()), xs + ws, allow_unused=True)
    assert got[1] is None and got[4] is None
    one = _ops.rms_norm(xs[2], ws[2], None)
    assert torch.equal(got[2], torch.autograd.grad(one.float().sum(), xs[2])[0])
    assert _ops.rms_norm_layer(xs * 2, ws * 2, [None] * 6) is None  # more than one launch holds
    assert _ops.rms_norm_layer([xs[0], xs[1].float()], ws[:2], [None] * 2) is None  # two dtypes
