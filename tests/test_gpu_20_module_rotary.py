"""Rotary in the norm kernels: the cos / sin table of runs of rows that walk heads fastest against the
per-row evaluation (same bits), and the modules' own rotary embedding applied there against the
eager modules."""

import pytest
import torch

from parity import assert_drift
from test_gpu_1_pass import dev, randn

pytestmark = pytest.mark.gpu
param = pytest.mark.parametrize


@param("dtype", (torch.bfloat16, torch.float32))
@param("heads,d,rot", ((4, 64, 64), (16, 64, 32), (5, 128, 128), (8, 32, 32), (3, 64, 64), (64, 8, 8)))
@param("n", (1, 7, 130))
def test_trig_table_same_bits(dtype, heads, d, rot, n):
    """[B, n, heads, d] storage takes the table (4 heads and more), the contiguous copy of the same
    rows does not: out, dx and dweight agree bit for bit.  Runs that start inside a token, wrap into
    the next batch row and end past the last row."""
    from poly_attention import _ops

    x = randn((3, n, heads, d), dtype, 1).to(dev()).transpose(1, 2)
    dy = randn((3, n, heads, d), dtype, 2).to(dev()).transpose(1, 2)
    w = (1 + 0.1 * randn((d,), torch.float32, 3)).to(dtype).to(dev())
    ang = (torch.arange(n, device=dev()).float()[:, None] * randn((rot,), torch.float32, 4).to(dev()).abs())
    got = []
    for xi, di in ((x, dy), (x.contiguous(), dy.contiguous())):
        y, rstd = _ops._rms_fwd_raw(xi, w, 1e-6, ang)
        dx, _ = _ops._rms_bwd_raw(di, xi, w, rstd, 1e-6, ang)
        got.append((y, dx))
    for a, b in zip(*got):
        assert torch.equal(a, b)


def _modules(order, dtype, **kw):
    from poly_attention import NPolyAttention, PolyAttention

    cls = PolyAttention if order == 2 else NPolyAttention
    if order != 2:
        kw["order"] = order
    torch.manual_seed(0)
    fused = cls(dim=128, dim_head=64, use_rotary_embed=True, causal=True, **kw)
    eager = cls(dim=128, dim_head=64, use_rotary_embed=True, causal=True, use_flash_kernel=False, **kw)
    eager.load_state_dict(fused.state_dict())
    rot = fused.rotary_emb
    fused, eager = fused.to(dev()), eager.to(dev())
    for m in (fused, eager):  # the frequencies stay fp32
        keep, m.rotary_emb = m.rotary_emb, None
        m.to(dtype)
        m.rotary_emb = keep
    return fused, eager


@param("order", (2, 3))
@param("dtype", (torch.bfloat16, torch.float32))
@param("kw", ({"heads": 4}, {"heads": 4, "kv_heads": 2},
              {"heads": 4, "multiply_root_value": True, "attn_gate": True}))
def test_module_rotary_training(order, dtype, kw):
    """Output, input gradient and every parameter gradient against the eager module in fp32 on the
    same weights; a bf16 result is held to the eager bf16 module's own drift."""
    fused, eager = _modules(order, dtype, **kw)
    x = randn((2, 70, 128), dtype, 5).to(dev())
    dy = randn((2, 70, 128), dtype, 6).to(dev())
    res = []
    for m, dt in ((fused, dtype), (eager, torch.float32), (eager, dtype)):
        keep, m.rotary_emb = m.rotary_emb, None
        m.to(dt)
        m.rotary_emb = keep
        xi = x.to(dt).requires_grad_()
        names = [k for k, p in m.named_parameters() if p.requires_grad]
        ps = [dict(m.named_parameters())[k] for k in names]
        out = m(xi)
        res.append([out, *torch.autograd.grad(out, [xi, *ps], dy.to(dt))])
        if dt == torch.float32 and m is eager and dtype != dt:
            m.rotary_emb = keep
    for name, a, b, c in zip(["out", "dx", *names], *res):
        if dtype == torch.float32:
            assert (a - b).abs().max().item() <= 1e-4 * max(1.0, b.abs().max().item()), name
        else:
            assert_drift(a, b, c, f"module rotary order {order} {name}")


@param("order", (2, 3))
def test_module_rotary_prefill_cache(order):
    """With return_cache the keys of the cache stay unrotated, and a cached step continues from it."""
    fused, eager = _modules(order, torch.float32, heads=4)
    x = randn((2, 33, 128), torch.float32, 7).to(dev())
    with torch.no_grad():
        (a, ca), (b, cb) = (m(x[:, :32], return_cache=True) for m in (fused, eager))
        assert (a - b).abs().max().item() <= 1e-4
        flat = lambda c: [t for e in c for t in (e if isinstance(e, tuple) else (e,))]  # noqa: E731
        for s, t in zip(flat(ca), flat(cb)):
            assert (s - t).abs().max().item() <= 1e-4
        (a, _), (b, _) = (m(x[:, 32:], cache=c, return_cache=True) for m, c in ((fused, ca), (eager, cb)))
        assert (a - b).abs().max().item() <= 1e-4


@param("order", (2, 3))
@param("dtype", (torch.bfloat16, torch.float16))
@param("freqs_too", (True, False))
def test_prefill_rotates_keys_as_the_module(order, dtype, freqs_too, monkeypatch):
    """The rotated keys of a prefill (what the passes get) are the module's rotation of the cached,
    unrotated ones, as a cached step rotates them: the same bits where the layer is cast whole, its
    frequencies with it; with fp32 frequencies to one rounding (a fused product and sum)."""
    from poly_attention import NPolyAttention, PolyAttention, _ops

    kw = dict(dim=128, dim_head=64, heads=4, use_rotary_embed=True, causal=True)
    torch.manual_seed(0)
    layer = PolyAttention(**kw) if order == 2 else NPolyAttention(order=order, **kw)
    freqs = layer.rotary_emb.freqs.data.clone()
    layer = layer.to(dev()).to(dtype)
    if not freqs_too:
        layer.rotary_emb.freqs.data = freqs.to(dev())
    seen = []
    chain = _ops.poly_chain
    monkeypatch.setattr(_ops, "poly_chain", lambda ql, qr, *a, **k: (seen.append(qr), chain(ql, qr, *a, **k))[1])
    with torch.no_grad():
        _, cache = layer(randn((2, 70, 128), dtype, 8).to(dev()), return_cache=True)
        keys = cache[:2] if order == 2 else cache[0]
        for got, raw in zip(seen[0], keys):
            want = layer.rotary_emb.rotate_queries_or_keys(raw)
            if freqs_too:
                assert torch.equal(got, want)
            else:
                err = (got.float() - want.float()).abs()
                assert (err <= torch.finfo(dtype).eps * want.float().abs() + 1e-6).all()


@param("dtype", (torch.bfloat16, torch.float32))
@param("heads", ((4, 8), (2, 3), (8, 2)))
def test_layer_norms_with_and_without_a_table(dtype, heads):
    """The norms of a layer in one launch where every tensor has the cos / sin table (4 heads and more),
    none has, and one has (kv heads): the same bits as one by one, forward and backward."""
    from poly_attention import _ops

    n, d = 37, 64
    ang = torch.arange(n, device=dev()).float()[:, None] * randn((d,), torch.float32, 1).to(dev()).abs()
    xs = [randn((2, n, h, d), dtype, 2 + h).to(dev()).transpose(1, 2) for h in heads]
    ws = [(1 + 0.1 * randn((d,), torch.float32, 20 + h)).to(dtype).to(dev()) for h in heads]
    dys = [randn((2, n, h, d), dtype, 40 + h).to(dev()).transpose(1, 2) for h in heads]
    got = []
    for layer in (True, False):
        ins = [t.detach().requires_grad_() for t in (*xs, *ws)]
        x, w = ins[:2], ins[2:]
        ys = (_ops.rms_norm_layer(x, w, [1e-6] * 2, ang) if layer else
              [_ops.rms_norm(a, b, 1e-6, ang) for a, b in zip(x, w)])
        got.append([*ys, *torch.autograd.grad(ys, x, dys)])
    for a, b in zip(*got):
        assert torch.equal(a, b)
