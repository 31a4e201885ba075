"""The direct-to-LDS kernels with two groups of waves per workgroup (head dim 128, and small grids at
head dim 64): tiles alternate between the groups, whose partial results are merged.  Tile counts of
one, two and an odd number per workgroup, a last tile of one key, groups without a tile, masked
tiles that only one group sees, against the oracle."""

import pytest
import torch

from test_gpu_1_pass import check, randn, run_pass

pytestmark = pytest.mark.gpu
param = pytest.mark.parametrize


@param("dtype,d", ((torch.bfloat16, 64), (torch.float16, 64), (torch.bfloat16, 128), (torch.float16, 128)))
@param("n", (33, 65, 128, 193, 321))
@param("causal", (False, True))
def test_tile_counts(dtype, d, n, causal):
    q, k, v = (randn((1, 2, n, d), dtype, s) for s in (1, 2, 3))
    bias = randn((1, 2, n), torch.float32, 4)
    check(run_pass(q, k, v, bias=bias, causal=causal), dtype, f"groups {dtype} d={d} n={n} causal={causal}")


@param("d", (64, 128))
@param("nq,nk", ((5, 300), (300, 5), (130, 64)))
def test_cross_lengths_and_gqa(d, nq, nk):
    q = randn((1, 4, nq, d), torch.bfloat16, 5)
    k, v = (randn((1, 2, nk, d), torch.bfloat16, s) for s in (6, 7))
    check(run_pass(q, k, v), torch.bfloat16, f"groups cross {nq}x{nk} d={d}")


@param("d", (64, 128))
@param("causal", (False, True))
@param("dead", ((0, 64), (64, 128), (0, 128), (128, 256), (200, 256)))
def test_masked_tiles_of_one_group(d, causal, dead):
    """A run of masked keys that covers tiles of one group only, of both, the first tiles of a group
    (its softmax state then starts late) and the end; the live key range starts at any tile."""
    n = 256
    q, k, v = (randn((2, 2, n, d), torch.bfloat16, s) for s in (8, 9, 10))
    km = torch.ones(2, n, dtype=torch.bool)
    km[1, dead[0]:dead[1]] = False
    check(run_pass(q, k, v, key_mask=km, causal=causal), torch.bfloat16,
          f"groups masked {dead} d={d} causal={causal}")


@param("softclamp", (None, 20.0))
def test_rising_scores(softclamp):
    """Scores that rise along the keys, so that the two groups' running maxima differ widely."""
    n, d = 320, 64
    q, k, v = (randn((1, 2, n, d), torch.bfloat16, s) for s in (11, 12, 13))
    bias = torch.linspace(-200.0, 30.0, n)[None, None].repeat(1, 2, 1)
    check(run_pass(q, k, v, bias=bias, softclamp=softclamp), torch.bfloat16, f"rising scores {softclamp}")


# The lengths above take two groups in the forward at head dim 64 only; these take them in every kernel
# that has them (pa_order.h, two_wave_groups: at 64 from 448 causal, 576 not; at 128 from 384).


@param("dtype,d", ((torch.bfloat16, 64), (torch.float16, 64), (torch.bfloat16, 128), (torch.float16, 128)))
@param("n", (513, 577, 769, 833))
@param("causal", (False, True))
def test_long_tile_counts(dtype, d, n, causal):
    q, k, v = (randn((1, 2, n, d), dtype, s) for s in (21, 22, 23))
    check(run_pass(q, k, v, causal=causal), dtype, f"long groups {dtype} d={d} n={n} causal={causal}")
    n -= 1  # the bias is read in whole chunks
    q, k, v = (t[:, :, :n].contiguous() for t in (q, k, v))
    bias = randn((1, 2, n), torch.float32, 24)
    check(run_pass(q, k, v, bias=bias, causal=causal), dtype, f"long groups {dtype} d={d} n={n} causal={causal} bias")


@param("d", (64, 128))
@param("nq,nk", ((5, 900), (900, 5), (130, 770), (770, 130)))
def test_long_cross_lengths_and_gqa(d, nq, nk):
    q = randn((1, 4, nq, d), torch.bfloat16, 25)
    k, v = (randn((1, 2, nk, d), torch.bfloat16, s) for s in (26, 27))
    check(run_pass(q, k, v), torch.bfloat16, f"long groups cross {nq}x{nk} d={d}")


@param("d", (64, 128))
@param("causal", (False, True))
@param("dead", ((0, 64), (64, 128), (0, 128), (128, 256), (700, 832)))
def test_long_masked_tiles_of_one_group(d, causal, dead):
    n = 832
    q, k, v = (randn((2, 2, n, d), torch.bfloat16, s) for s in (28, 29, 30))
    km = torch.ones(2, n, dtype=torch.bool)
    km[1, dead[0]:dead[1]] = False
    check(run_pass(q, k, v, key_mask=km, causal=causal), torch.bfloat16,
          f"long groups masked {dead} d={d} causal={causal}")


@param("d", (64, 128))
@param("softclamp", (None, 20.0))
def test_long_rising_scores(d, softclamp):
    n = 832
    q, k, v = (randn((1, 2, n, d), torch.bfloat16, s) for s in (31, 32, 33))
    bias = torch.linspace(-200.0, 30.0, n)[None, None].repeat(1, 2, 1)
    check(run_pass(q, k, v, bias=bias, softclamp=softclamp), torch.bfloat16, f"long rising scores d={d} {softclamp}")
