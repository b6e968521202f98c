"""Prefill -> decode rows around the lengths where the mask is compacted in one pass, in several, and
where a workgroup's share of rows has remainders; every pair of types (GPU, bit-exact)."""

import itertools

import pytest
import torch

from test_gpu_prefill_state import _run

pytestmark = pytest.mark.gpu

DTYPES = (torch.bfloat16, torch.float16, torch.float32)


@pytest.mark.parametrize("T", [1, 255, 257, 2047, 2048, 2049, 4097])
@pytest.mark.parametrize("window", [0, 1, 64])
def test_mask_chunks(T, window):
    g = torch.Generator().manual_seed(T)
    mask = torch.rand(3, T, generator=g) < torch.tensor([[1.1], [0.5], [0.01]])  # all, half, few of the tokens
    _run(3, T, 2, 64, window, torch.bfloat16, torch.bfloat16, mask, 1, 0, seed=T)


@pytest.mark.parametrize("in_dtype,cache_dtype", list(itertools.product(DTYPES, DTYPES)))
@pytest.mark.parametrize("D", [8, 24, 256])
def test_types(in_dtype, cache_dtype, D):
    g = torch.Generator().manual_seed(D)
    _run(2, 300, 3, D, 16, in_dtype, cache_dtype, torch.rand(2, 300, generator=g) < 0.9, 0, 1, seed=D, strided=True,
         len_dtype=torch.int32)
