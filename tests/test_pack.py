"""The packed form of the hot structs (poly_attention._lib.PACK_*) field by field against their ctypes
declarations, the bias padding rule and the one-operation head view (no GPU needed)."""

import ctypes

import pytest
import torch

from poly_attention import _lib, _ops


def _flat(obj, prefix=""):
    for name, typ in obj._fields_:
        value = getattr(obj, name)
        if isinstance(value, ctypes.Structure):
            yield from _flat(value, f"{prefix}{name}.")
        else:
            yield prefix + name, value or 0


@pytest.mark.parametrize("pack,cls", ((_lib.PACK_PASS, _lib.PaPass),
                                      (_lib.PACK_PASS_GRAD, _lib.PaPassGrad),
                                      (_lib.PACK_RMS, _lib.PaRmsNorm)))
def test_packed_fields_in_declaration_order(pack, cls):
    names = [n for n, _ in _flat(cls())]
    values = list(range(1, len(names) + 1))
    got = dict(_flat(cls.from_buffer_copy(pack.pack(*values))))
    assert got == dict(zip(names, values))


@pytest.mark.parametrize("n", (1, 2, 3, 4, 5, 64, 127))
def test_bias_flags(n):
    like = torch.zeros(1)
    own = _ops._empty_lse(2, 3, n, like)
    assert own.shape == (2, 3, n) and own.stride(1) % 4 == 0
    assert bool(_ops._bias_flags(own)) == (n % 4 != 0)
    assert _ops._bias_flags(torch.zeros(2, 3, n)) == 0          # no room after the last row
    assert _ops._bias_flags(own.half()) == 0
    assert _ops._bias_flags(torch.zeros(2, n, 3).transpose(1, 2)) == 0 or n == 1
    # the last row of a longer storage ends inside it, the last row of this view does not
    base = torch.zeros(2 * 3 * n + 3)
    view = base[3:].view(2, 3, n)
    assert _ops._bias_flags(view) == 0
    assert bool(_ops._bias_flags(base[:-3].view(2, 3, n))) == (n % 4 != 0)


def test_head_view():
    t = torch.arange(2 * 5 * 24.0).view(2, 5, 24)
    for x in (t, t[:, 1:], torch.arange(5 * 2 * 24.0).view(5, 2, 24).transpose(0, 1)):
        want = x[..., 4:20].unflatten(-1, (4, 4)).transpose(1, 2)
        got = _ops._head_view(x, 4, 4, 4)
        assert torch.equal(got, want) and got.stride() == want.stride()
        assert got.data_ptr() == want.data_ptr()
