"""pa_linear_rows: up to 64 rows on the matrix cores against the fp32 product (fp32 sums, one rounding:
the tolerance of the streamed projections), and a step of a larger batch through a module."""

import pytest
import torch

from test_gpu_6_linear import TOL, assert_close, dev, fp32_linear

pytestmark = pytest.mark.gpu
param = pytest.mark.parametrize


@param("dtype", (torch.bfloat16, torch.float16))
@param("rows", (1, 16, 17, 32, 33, 64))
@param("k,outs", ((8, (1,)), (72, (33, 8)), (1024, (257, 1024, 40)), (520, (16,)), (4096, (4096, 2050, 2048)),
                  (2056, (8192,))))
def test_linear_rows_match_fp32(dtype, rows, k, outs):
    from poly_attention import _ops

    g = torch.Generator().manual_seed(rows + k)
    wide = torch.randn(rows, k + 8, generator=g).to(dev(), dtype)
    for x in (wide[:, :k], wide[:, 8:].reshape(rows, 1, k)):
        specs = [((torch.randn(n, k, generator=g) * k ** -0.5).to(dev(), dtype),
                  torch.randn(n, generator=g).to(dev(), dtype) if i % 2 else None) for i, n in enumerate(outs)]
        assert all(_ops.linear_rows_supported(x, *s) for s in specs)
        for y, (w, b) in zip(_ops.linear_rows_group(x, specs), specs):
            assert y.shape == (*x.shape[:-1], w.shape[0]) and y.dtype == dtype
            assert_close(y, fp32_linear(x, w, b), TOL[dtype], f"rows={rows} k={k} n={w.shape[0]}")


def test_linear_rows_leaves_other_calls():
    from poly_attention import _ops

    w = torch.randn(64, 128, device=dev()).bfloat16()
    x = torch.randn(20, 128, device=dev()).bfloat16()
    assert _ops.linear_rows_supported(x, w)
    assert not _ops.linear_rows_supported(torch.randn(65, 128, device=dev()).bfloat16(), w)
    assert not _ops.linear_rows_supported(x.float(), w.float())
    assert not _ops.linear_rows_supported(x.clone().requires_grad_(), w)
    assert not _ops.linear_rows_supported(x[:, :124], w[:, :124])
    with torch.autocast("cuda", torch.float16):
        assert not _ops.linear_rows_supported(x, w)


def test_decode_steps_of_a_larger_batch_equal_parallel():
    from poly_attention import PolyAttention

    torch.manual_seed(3)
    m = PolyAttention(dim=256, heads=4, dim_head=64, causal=True).to(dev(), torch.float16).eval()
    x = torch.randn(24, 6, 256, device=dev(), dtype=torch.float16)
    with torch.no_grad():
        ref = m(x)
        out, cache = m(x[:, :3], return_cache=True)
        outs = [out]
        for i in range(3, 6):
            out, cache = m(x[:, i:i + 1], cache=cache, return_cache=True)
            outs.append(out)
    assert_close(torch.cat(outs, dim=1), ref, 1e-2, "stepwise")
