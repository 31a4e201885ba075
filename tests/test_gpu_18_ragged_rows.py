"""Lengths that are not a multiple of four on the direct-to-LDS kernels (bf16 / f16): the backward's
per-row values sit in padded rows, and a key bias whose rows may be read to the next multiple of
four takes the same kernels.  Against the oracle; the padding holds NaN, which must not reach any
result."""

import pytest
import torch

import oracle.poly_oracle as O
from parity import TOL, assert_parity
from test_gpu_1_pass import dev, randn

pytestmark = pytest.mark.gpu
param = pytest.mark.parametrize


def _run(n, d, dtype, padded, causal=True, softclamp=None, key_mask=None, hk=2, nq=None):
    from poly_attention import _ops

    nq = n if nq is None else nq
    q = randn((2, 4, nq, d), dtype, 1)
    k, v = (randn((2, hk, n, d), dtype, s) for s in (2, 3))
    bias = randn((2, hk, n), torch.float32, 4)
    do, dl = randn((2, 4, nq, d), dtype, 5), randn((2, 4, nq), torch.float32, 6)
    g = [t.to(dev()).requires_grad_() for t in (q, k, v)]
    base = torch.full((2, hk, n + (-n % 4 if padded else 0)), float("nan"), device=dev())
    gb = base[..., :n]
    gb.copy_(bias)
    assert bool(_ops._bias_flags(gb)) == (padded and n % 4 != 0)
    gb = gb.detach().requires_grad_()
    km = key_mask.to(dev()) if key_mask is not None else None
    out, lse = _ops.attn_pass(*g, bias=gb, key_mask=km, causal=causal, softclamp=softclamp)
    torch.autograd.backward((out, lse), (do.to(dev()), dl.to(dev())))
    res = [out, *[t.grad for t in (*g, gb)]]
    refs = []
    for dt in (torch.float32, dtype):
        o = [t.to(dt).requires_grad_() for t in (q, k, v)]
        ob = bias.clone().to(dt).requires_grad_()
        ro, rl = O.attn_pass(*o, bias=ob, key_mask=key_mask, causal=causal, softclamp_value=softclamp)
        torch.autograd.backward((ro, rl), (do.to(ro.dtype), dl.to(rl.dtype)))
        refs.append([ro, *[t.grad for t in (*o, ob)]])
    for name, a, b, c in zip(("out", "dq", "dk", "dv", "dbias"), res, *refs):
        assert_parity(a, b, dtype, f"ragged n={n} d={d} {dtype} {name}", tol=TOL[dtype],
                      grad=name != "out", ref_lp=c)


@param("dtype,d", ((torch.bfloat16, 64), (torch.float16, 64), (torch.bfloat16, 128)))
@param("n", (65, 127, 130, 259))
@param("padded", (False, True))
def test_ragged_lengths(n, d, dtype, padded):
    _run(n, d, dtype, padded)


@param("n", (67, 190))
@param("causal", (False, True))
@param("softclamp", (None, 20.0))
def test_ragged_masks_and_softclamp(n, causal, softclamp):
    """A key mask replaces the bias by the key term (padded workspace rows)."""
    km = torch.ones(2, n, dtype=torch.bool)
    km[1, n // 2:] = False
    _run(n, 64, torch.bfloat16, True, causal=causal, softclamp=softclamp, key_mask=km)
    _run(n, 64, torch.bfloat16, True, causal=causal, softclamp=softclamp)


def test_ragged_cross_lengths():
    _run(133, 64, torch.bfloat16, True, causal=False, nq=71)
