"""A norm row is held by one wave: 64 lanes of 16 bytes, 512 features in 16 bits and 256 in fp32.  Longer
rows are refused (the modules then take torch.nn.RMSNorm), never half computed."""

import ctypes

import pytest
import torch

from poly_attention import _lib, _ops


@pytest.mark.parametrize("dtype,limit", ((torch.bfloat16, 512), (torch.float16, 512), (torch.float32, 256)))
def test_norm_rows_longer_than_a_wave_are_refused(dtype, limit):
    lib = _lib.load()
    assert _ops.rms_layout_supported(torch.empty(1, 1, 2, limit, dtype=dtype), None)
    assert not _ops.rms_layout_supported(torch.empty(1, 1, 2, limit + 8, dtype=dtype), None)
    r = _lib.PaRmsNorm()
    r.batch = r.heads = r.n = 1
    r.x.dtype, r.x.heads = _lib.DTYPE_CODE[dtype], 1
    for dim, want in ((limit, _lib.PA_EINVAL), (limit + 8, _lib.PA_EUNSUPPORTED)):  # EINVAL: no pointers
        r.dim = dim
        assert lib.pa_rmsnorm_fwd(ctypes.byref(r), None) == want
        assert lib.pa_rmsnorm_bwd(ctypes.byref(r), None) == want
