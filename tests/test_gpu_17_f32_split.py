"""The fp32 passes on the bf16 matrix cores (three-way operand split): every workgroup shape of the
dispatch (row blocks per workgroup x waves per row block) at the edges of its tiles, against the
oracle at 1e-4, the split's accuracy against 64 bits, and infinite inputs."""

import pytest
import torch

import oracle.poly_oracle as O
from test_gpu_1_pass import check, dev, randn, run_pass

pytestmark = pytest.mark.gpu
param = pytest.mark.parametrize


@param("n", (1, 31, 33, 64, 65, 129))
@param("d", (64, 128))
def test_small_grids(n, d):
    """Two row blocks and (d = 64) four or (d = 128) two waves each; up to one row past a tile, a
    row block and a stage; causal, GQA, key bias and value multiplier."""
    q = randn((1, 4, n, d), torch.float32, 1)
    k, v, vmul = (randn((1, 2, n, d), torch.float32, s) for s in (2, 3, 4))
    bias = randn((1, 2, n), torch.float32, 5)
    check(run_pass(q, k, v, vmul=vmul, bias=bias, causal=True), torch.float32, f"n={n} d={d}")


@param("units,n,d,causal", ((128, 130, 64, False), (256, 130, 64, True), (256, 257, 64, True),
                            (128, 130, 128, False), (256, 129, 128, True)))
def test_large_grids(units, n, d, causal):
    """Four and eight row blocks per workgroup, the last one partly empty."""
    q, k, v = (randn((units // 16, 16, n, d), torch.float32, s) for s in (6, 7, 8))
    check(run_pass(q, k, v, causal=causal), torch.float32, f"units={units} n={n} d={d}")


def _pass64(q, k, v, do):
    ts = [t.double().requires_grad_() for t in (q, k, v)]
    out, _ = O.attn_pass(*ts, causal=True)
    return [out.detach(), *torch.autograd.grad(out, ts, do.double())]


@param("scale", (1.0, 1e-6, 1e4))
def test_accuracy_against_64_bits(scale):
    """Values of every magnitude split alike: relative error (2-norm) at most 2e-6, four times the
    largest that fp32 products showed at this size (the sums are 300 terms of fp32)."""
    from poly_attention import _ops

    q, k, v, do = (randn((1, 4, 300, 64), torch.float32, s) for s in (9, 10, 11, 12))
    v, do = v * scale, do / scale
    ts = [t.to(dev()).requires_grad_() for t in (q, k, v)]
    out, _ = _ops.attn_pass(*ts, causal=True)
    got = [out.detach(), *torch.autograd.grad(out, ts, do.to(dev()))]
    for a, b in zip(got, _pass64(q, k, v, do)):
        assert ((a.double().cpu() - b).norm() / b.norm()).item() < 2e-6


@param("d", (64, 128))
def test_infinite_and_huge_values(d):
    """An infinite value element reaches every row that attends its key as +-inf in that feature and
    nowhere else, as with fp32 products; a finite value above bf16's largest number stays finite."""
    from poly_attention import _ops

    n = 70
    q, k, v = (randn((1, 2, n, d), torch.float32, s) for s in (13, 14, 15))
    v[0, 0, 40, 5] = float("inf")
    v[0, 1, 40, 9] = 3.4e38
    out, lse = _ops.attn_pass(*(t.to(dev()) for t in (q, k, v)), causal=False)
    ref, ref_lse = O.attn_pass(q.double(), k.double(), v.double(), causal=False)
    out = out.cpu().double()
    inf = torch.isinf(ref)
    assert inf.any() and torch.equal(torch.isinf(out), inf) and (out[inf] > 0).all()
    assert torch.isfinite(out[~inf]).all()
    assert ((out[~inf] - ref[~inf]).abs() <= 1e-4 + 1e-5 * ref[~inf].abs()).all()
    assert torch.allclose(lse.cpu().double(), ref_lse, atol=1e-4)
    # causal: the rows before the key, in the features without an infinity (in feature 5 the eager
    # reference multiplies it by the masked probability 0)
    out, _ = _ops.attn_pass(*(t.to(dev()) for t in (q, k, v)), causal=True)
    ref, _ = O.attn_pass(q.double(), k.double(), v.double(), causal=True)
    rows, feats = slice(0, 32), [f for f in range(d) if f != 5]
    assert ((out[0, 0, rows, feats].cpu().double() - ref[0, 0, rows, feats]).abs() <= 1e-4).all()


def _grads(run, q, k, v, bias, do):
    ts = [t.requires_grad_() for t in (q, k, v, bias)]
    out = run(*ts)
    return [out.detach(), *torch.autograd.grad(out, ts, do)]


@param("d", (64, 128))
@param("causal", (False, True))
@param("where", ("q", "k", "v", "do"))
def test_backward_of_huge_values(d, causal, where):
    """A finite element that bf16 cannot hold sends dQ or dK/dV (whichever has it as an operand) over
    its tiles again, from zero accumulators, dbias and the first head and stage (GQA: two query
    heads per key head, several stages).  Its feature is zero in the tensor it is multiplied with,
    so every score and dP stays ordinary, and its own products are finite: every result against 64
    bits, the element's feature by itself, at test_accuracy_against_64_bits's 2e-6."""
    from poly_attention import _ops

    n, f = 300, 9
    q, do = (randn((1, 4, n, d), torch.float32, s) for s in (16, 17))
    k, v = (randn((1, 2, n, d), torch.float32, s) for s in (18, 19))
    bias = randn((1, 2, n), torch.float32, 20)
    ts = {"q": q, "k": k, "v": v, "do": do}
    ts[{"q": "k", "k": "q", "v": "do", "do": "v"}[where]][..., f] = 0.0
    ts[where][0, 1, 150, f] = 3.39e38
    got = _grads(lambda *a: _ops.attn_pass(*a[:3], bias=a[3], causal=causal)[0],
                 *(t.to(dev()) for t in (q, k, v, bias)), do.to(dev()))
    ref = _grads(lambda *a: O.attn_pass(*a[:3], bias=a[3], causal=causal)[0],
                 *(t.double() for t in (q, k, v, bias)), do.double())
    rest = [i for i in range(d) if i != f]
    for name, a, b in zip(("out", "dq", "dk", "dv", "dbias"), got, ref):
        a = a.cpu().double()
        for part in ((rest, [f]) if a.dim() == 4 else (None,)):
            x, y = (a, b) if part is None else (a[..., part], b[..., part])
            assert torch.isfinite(x).all(), f"{name} {part}"
            assert (x - y).norm() <= 2e-6 * y.norm(), f"{name} of a huge {where} element, {part}"


@param("d", (64, 128))
def test_backward_of_an_infinite_gradient(d):
    """An infinite element of dout: its row's dP and D are infinite, so dq of the row and every dk of
    its key head are not finite; dv of its feature is infinite, and every other dq row, dk and dv
    is as in 64 bits."""
    from poly_attention import _ops

    n, f, i = 100, 5, 40
    q, do = (randn((1, 4, n, d), torch.float32, s) for s in (21, 22))
    k, v = (randn((1, 2, n, d), torch.float32, s) for s in (23, 24))
    bias = randn((1, 2, n), torch.float32, 25)
    do[0, 3, i, f] = float("inf")
    got = _grads(lambda *a: _ops.attn_pass(*a[:3], bias=a[3])[0], *(t.to(dev()) for t in (q, k, v, bias)),
                 do.to(dev()))
    ref = _grads(lambda *a: O.attn_pass(*a[:3], bias=a[3])[0], *(t.double() for t in (q, k, v, bias)),
                 do.double())
    for name, a, b in zip(("out", "dq", "dk", "dv", "dbias"), got, ref):
        a, fin = a.cpu().double(), torch.isfinite(b)
        assert torch.equal(torch.isfinite(a), fin), name
        if name == "dv":
            assert torch.equal(a[~fin], b[~fin]) and (~fin).sum() == n
        assert (a[fin] - b[fin]).norm() <= 2e-6 * b[fin].norm(), name


@param("scale", (1e-30, 2.0 ** -100, 1e30))
def test_accuracy_of_extreme_magnitudes(scale):
    """The three parts hold all 24 bits down to 2^-110 (the third is then bf16's smallest number,
    2^-133) and up to the largest; as test_accuracy_against_64_bits."""
    from poly_attention import _ops

    q, k, v, do = (randn((1, 4, 300, 64), torch.float32, s) for s in (26, 27, 28, 29))
    v = v * scale
    ts = [t.to(dev()).requires_grad_() for t in (q, k, v)]
    out, _ = _ops.attn_pass(*ts, causal=True)
    got = [out.detach(), *torch.autograd.grad(out, ts, do.to(dev()))]
    for a, b in zip(got, _pass64(q, k, v, do)):
        assert ((a.double().cpu() - b).norm() / b.norm()).item() < 2e-6


@param("n", (225, 256, 257, 300))
@param("causal", (False, True))
@param("vmul", (False, True))
def test_one_block_per_workgroup(n, causal, vmul):
    """Head dim 128 in small grids of eight tiles or more (forward and dQ: four waves of a workgroup on
    one row block): one row past a tile, waves with two and with three tiles, and causal blocks
    that leave waves without any; GQA, key bias."""
    q = randn((1, 4, n, 128), torch.float32, 30)
    k, v, m = (randn((1, 2, n, 128), torch.float32, s) for s in (31, 32, 33))
    bias = randn((1, 2, n), torch.float32, 34)
    check(run_pass(q, k, v, vmul=m if vmul else None, bias=bias, causal=causal), torch.float32,
          f"one block n={n} causal={causal} vmul={vmul}")


@param("causal", (False, True))
def test_one_block_masks_and_softclamp(causal):
    n = 270
    q, k, v = (randn((2, 2, n, 128), torch.float32, s) for s in (35, 36, 37))
    km = torch.ones(2, n, dtype=torch.bool)
    km[0, :70] = False
    km[1, 200:] = False
    check(run_pass(q, k, v, key_mask=km, causal=causal), torch.float32, f"one block masked causal={causal}")
    check(run_pass(q, k, v, causal=causal, softclamp=2.0), torch.float32, f"one block softclamp causal={causal}")


def test_one_block_accuracy():
    """test_accuracy_against_64_bits at head dim 128 and as many blocks as CUs."""
    from poly_attention import _ops

    q, k, v, do = (randn((1, 8, 1024, 128), torch.float32, s) for s in (38, 39, 40, 41))
    ts = [t.to(dev()).requires_grad_() for t in (q, k, v)]
    out, _ = _ops.attn_pass(*ts, causal=True)
    got = [out.detach(), *torch.autograd.grad(out, ts, do.to(dev()))]
    for a, b in zip(got, _pass64(q, k, v, do)):
        assert ((a.double().cpu() - b).norm() / b.norm()).item() < 2e-6
