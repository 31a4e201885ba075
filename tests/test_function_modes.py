"""Torch function modes and the plain eager nodes: a mode that has to see the registered custom ops
keeps calls on them; a default device (a mode of torch's own) does not."""

import torch
from torch.overrides import TorchFunctionMode

from poly_attention import _ops


class _Seen(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_function_modes_keep_the_custom_ops():
    t = torch.ones(1)
    assert _ops._plain_eager(t)
    with _Seen():
        assert not _ops._plain_eager(t)
        with torch.device("cpu"):
            assert not _ops._plain_eager(t)
    assert _ops._plain_eager(t)


def test_default_device_is_no_such_mode():
    t = torch.ones(1)
    with torch.device("cpu"):
        assert _ops._plain_eager(t)
        with _Seen():
            assert not _ops._plain_eager(t)
