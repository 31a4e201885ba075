"""Value multipliers (the middle levels of an order-n chain) on the direct-to-LDS kernels (bf16 / f16,
head dims 64 and 128): the multiplier is folded into the values by a kernel of its own, and the dK/dV
kernel forms dv and dvmul from the effective value's gradient."""

import pytest
import torch

from parity import assert_parity
from test_gpu_1_pass import check, dev, randn, run_pass

pytestmark = pytest.mark.gpu
param = pytest.mark.parametrize


@param("dtype,d", ((torch.bfloat16, 64), (torch.float16, 64), (torch.bfloat16, 128)))
@param("n", (1, 63, 130, 257))
@param("gqa", (False, True))
def test_value_multiplier(dtype, d, n, gqa):
    """Causal with a key bias; one row past a tile and a workgroup, and lengths that leave the last
    elements of the product's grid ragged."""
    hk = 2 if gqa else 4
    q = randn((2, 4, n, d), dtype, 1)
    k, v, vmul = (randn((2, hk, n, d), dtype, s) for s in (2, 3, 4))
    bias = randn((2, hk, n), torch.float32, 5)
    check(run_pass(q, k, v, vmul=vmul, bias=bias, causal=True), dtype, f"vmul {dtype} d={d} n={n} gqa={gqa}")


@param("causal", (False, True))
def test_value_multiplier_masked(causal):
    """With a key mask (the fix-ups add the fully-masked rows' part to dv and dvmul)."""
    dtype, n = torch.bfloat16, 200
    q, k, v, vmul = (randn((2, 4, n, 64), dtype, s) for s in (6, 7, 8, 9))
    bias = randn((2, 4, n), torch.float32, 10)
    km = torch.ones(2, n, dtype=torch.bool)
    km[0, :70] = False
    km[1, 150:] = False
    check(run_pass(q, k, v, vmul=vmul, bias=bias, key_mask=km, causal=causal), dtype,
          f"vmul masked causal={causal}")


@param("hv,hm", ((2, 4), (4, 2), (1, 4)))
def test_value_multiplier_head_counts(hv, hm):
    """Forward with values and multipliers of different head counts, and of strided layouts
    ([batch, n, heads, dim] storage), against the same call on expanded contiguous tensors."""
    from poly_attention import _ops

    n, d, dtype = 130, 64, torch.bfloat16
    q, k = (randn((2, 4, n, d), dtype, s).to(dev()) for s in (11, 12))
    v = randn((2, n, hv, d), dtype, 13).to(dev()).transpose(1, 2)
    m = randn((2, n, hm, d), dtype, 14).to(dev()).transpose(1, 2)
    out, lse = _ops.attn_pass(q, k, v, vmul=m, causal=True)
    full = (v.repeat_interleave(4 // hv, 1).float() * m.repeat_interleave(4 // hm, 1).float()).to(dtype)
    ref, ref_lse = _ops.attn_pass(q, k, full.contiguous(), causal=True)
    assert_parity(out, ref.cpu(), dtype, f"head counts {hv} {hm}", tol=0.0, roundings=0)
    assert torch.equal(lse, ref_lse)


@param("dtype,d", ((torch.bfloat16, 64), (torch.float16, 64), (torch.bfloat16, 128)))
@param("n,padded", ((4, False), (132, False), (260, False), (63, True), (130, True), (257, True)))
def test_value_multiplier_folded(dtype, d, n, padded):
    """The lengths that take the folded value: a multiple of four (the bias rows of the lengths above
    are not readable in whole 16-byte chunks, so their backward stays register-staged), or a bias
    in padded rows, as a chain's deeper level gives it.  GQA, causal, two wave groups at d = 64."""
    import oracle.poly_oracle as O
    from poly_attention import _ops

    q = randn((2, 4, n, d), dtype, 1)
    k, v, vmul = (randn((2, 2, n, d), dtype, s) for s in (2, 3, 4))
    bias = randn((2, 2, n), torch.float32, 5)
    do, dl = randn((2, 4, n, d), dtype, 6), randn((2, 4, n), torch.float32, 7)
    gb = torch.full((2, 2, n + (-n % 4 if padded else 0)), float("nan"), device=dev())[..., :n]
    gb.copy_(bias)
    assert bool(_ops._bias_flags(gb)) == padded
    g = [t.to(dev()).requires_grad_() for t in (q, k, v, vmul)] + [gb.detach().requires_grad_()]
    out, lse = _ops.attn_pass(*g, causal=True)
    res = [out, *torch.autograd.grad((out, lse), g, (do.to(dev()), dl.to(dev())))]
    refs = []
    for dt in (torch.float32, dtype):
        o = [t.to(dt).requires_grad_() for t in (q, k, v, vmul, bias)]
        ro, rl = O.attn_pass(*o, causal=True)
        refs.append([ro, *torch.autograd.grad((ro, rl), o, (do.to(ro.dtype), dl.to(rl.dtype)))])
    for name, a, b, c in zip(("out", "dq", "dk", "dv", "dvmul", "dbias"), res, *refs):
        assert_parity(a, b, dtype, f"vmul folded {dtype} d={d} n={n} {name}", grad=name != "out", ref_lp=c)


@param("dtype", (torch.bfloat16, torch.float16))
@param("causal", (False, True))
@param("softclamp", (None, 30.0))
def test_value_multiplier_large_grids(dtype, causal, softclamp):
    """Enough heads for one group of waves per workgroup in the backward (1024 workgroups, past the
    threshold of 512 causal, 128 not), where dv and dvmul are formed without a merge."""
    n = 132
    q, k, v, vmul = (randn((8, 64, n, 64), dtype, s) for s in (15, 16, 17, 18))
    bias = randn((8, 64, n), torch.float32, 19)
    check(run_pass(q, k, v, vmul=vmul, bias=bias, causal=causal, softclamp=softclamp), dtype,
          f"vmul large grid {dtype} causal={causal} softclamp={softclamp}")
