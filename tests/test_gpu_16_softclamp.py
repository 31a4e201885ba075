"""The soft clamp's two branches in the MFMA kernels (bf16 / f16): the polynomial, taken by a wave
whose scores all lie in |s * scale| <= 0.35 softclamp, and tanhf for a block with any score beyond,
against the fp32 oracle at the bounds of tests/parity.py (the polynomial's own error, 1.3e-7 of
the score, is far below them)."""

import pytest
import torch

from test_gpu_1_pass import check, dev, randn, run_pass

pytestmark = pytest.mark.gpu
param = pytest.mark.parametrize


@param("dtype,d", ((torch.bfloat16, 64), (torch.float16, 64), (torch.bfloat16, 128),
                   (torch.bfloat16, 256)))
@param("causal", (False, True))
@param("softclamp", (0.05, 2.0, 8.0, 50.0))
def test_softclamp_ranges(dtype, d, causal, softclamp):
    """Scores of about unit variance with one large negative score per head (-2.5 |k|^2 scale: -20 at
    d = 64, -40 at 256): at 50 all but those two blocks take the polynomial, at 8 most blocks, at
    2 few, at 0.05 none.  One row past a 128-query workgroup and a ragged last key tile; a key bias.

    The outlier is negative because a row dominated by one key tests something else: there
    dS = P (dP - D) cancels, and D = rowsum(dO * O) with the stored O rounded to bf16 is off by up to
    2^-9 sqrt(d) |O| |dO|, 0.06 at d = 256, which an outlier query of 5 sigma (|q| scale about 1)
    carries into dK whatever the clamp."""
    n = 129
    q, k, v = (randn((1, 2, n, d), dtype, s) for s in (1, 2, 3))
    q[0, 0, 40] = -2.5 * k[0, 0, 7]
    q[0, 1, 100] = -2.5 * k[0, 1, 70]
    bias = randn((1, 2, n), torch.float32, 4)
    check(run_pass(q, k, v, bias=bias, causal=causal, softclamp=softclamp), dtype,
          f"softclamp {softclamp} {dtype} d={d} causal={causal}")


@param("left", (False, True))
def test_softclamp_masked_keys(left):
    """Masked keys and causal rows beside the polynomial: a masked entry's probability is 0 and its
    clamp factor finite."""
    dtype, n = torch.bfloat16, 200
    q, k, v = (randn((2, 4, n, 64), dtype, s) for s in (5, 6, 7))
    km = torch.ones(2, n, dtype=torch.bool)
    km[1, :90] = not left
    km[1, 110:] = left
    check(run_pass(q, k, v, key_mask=km, causal=True, softclamp=30.0), dtype,
          f"softclamp masked left={left}")


@param("scale_softclamp", ((0.125, 30.0), (0.125, 0.05), (1.0, 2.0)))
@param("n", (31, 64))
def test_softclamp_short_passes(scale_softclamp, n):
    """The short-pass kernel (n <= 64, not causal) takes the same clamp."""
    softclamp = scale_softclamp[1]
    q, k, v = (randn((2, 2, n, 64), torch.bfloat16, s) for s in (8, 9, 10))
    q = (q.float() * (scale_softclamp[0] * 8.0)).to(torch.bfloat16)
    check(run_pass(q, k, v, softclamp=softclamp), torch.bfloat16, f"softclamp short {softclamp}")


@param("dtype,d,units", ((torch.bfloat16, 64, (2, 2)), (torch.bfloat16, 64, (8, 64)),
                         (torch.float16, 128, (1, 2))))
@param("n", (130, 132, 516))
def test_softclamp_key_bias_of_minus_1e9(dtype, d, units, n):
    """A finite key bias of -1e9 on the first key, causal: the first row's lse is -1e9 while the keys
    after its own have biases around 0.  Their probability in the backward is 0 whatever the bias
    and lse, and the first key's is 1, though fp32 holds no score beside 1e9.  (One such key: of
    several, it cannot hold log n either.)  The register-staged kernels (n = 130, a bias without
    padded rows) and the direct-to-LDS ones, with one and with two groups of waves (n = 132, 516)."""
    if n > 300 and units[1] > 2:
        units = (1, 8)
    q, k, v = (randn((*units, n, d), dtype, s) for s in (21, 22, 23))
    bias = randn((*units, n), torch.float32, 24)
    bias[..., 0] = -1e9
    check(run_pass(q, k, v, bias=bias, causal=True, softclamp=30.0), dtype,
          f"softclamp bias -1e9 {dtype} d={d} {units} n={n}")


@param("dtype", (torch.bfloat16, torch.float16))
@param("causal", (False, True))
@param("biased", (False, True))
@param("softclamp", (2.0, 30.0))
def test_softclamp_large_grids(dtype, causal, biased, softclamp):
    """Enough heads for one group of waves per workgroup in both directions (1024 workgroups in the
    backward, 512 of 256 queries in the forward), two query and three key tiles, the last of four
    keys; both branches of the clamp."""
    n = 132
    q, k, v = (randn((8, 64, n, 64), dtype, s) for s in (25, 26, 27))
    bias = randn((8, 64, n), torch.float32, 28) if biased else None
    check(run_pass(q, k, v, bias=bias, causal=causal, softclamp=softclamp), dtype,
          f"softclamp {softclamp} large grid {dtype} causal={causal} biased={biased}")


@param("causal", (False, True))
def test_softclamp_at_scale_zero(causal):
    """A scale of 0: every visible key has the same probability, and dq and dk are 0 (a clamp held as a
    multiple of the raw score would be 0 * inf)."""
    from poly_attention import _ops

    q, k, v, do = (randn((1, 2, 132, 64), torch.bfloat16, s).to(dev()) for s in (31, 32, 33, 34))
    ts = [t.requires_grad_() for t in (q, k, v)]
    out, _ = _ops.attn_pass(*ts, causal=causal, softclamp=20.0, scale=0.0)
    dq, dk, dv = torch.autograd.grad(out, ts, do)
    seen = torch.ones(132, 132, device=dev()).tril() if causal else torch.ones(132, 132, device=dev())
    p = seen / seen.sum(-1, keepdim=True)
    assert (out.float() - p @ v.detach().float()).abs().max() <= 2e-2
    assert not dq.any() and not dk.any()
    # P in bf16: each of up to 132 terms off by 2^-9 of itself
    bound = 2.0 ** -8 * (p.t() @ do.float().abs()) + 2.0 ** -8 * dv.float().abs() + 1e-6
    assert ((dv.float() - p.t() @ do.float()).abs() <= bound).all()
