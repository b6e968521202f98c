"""The two-wave dK/dV kernel (head dims 128 and 256) at the edges of its tiles, against the float64
oracle (GPU): sequences of one chunk and of one more or less than a chunk, a key tile and the three
staged chunks; every family, the masks that leave waves idle, arbitrary ids. Bounds as in
test_gpu_attention."""

import numpy as np
import pytest
import torch

from test_gpu_attention import _check, _packed_docs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("n", [2, 32, 34, 64, 96, 98, 126, 128, 130, 258, 514])
def test_dkdv_tile_edges(d, n):
    rng = np.random.default_rng(100 * d + n)
    for family, window, pkw, kind in (("full", 0, None, "none"), ("sps", 5, None, "packed"),
                                      ("reverse_sps", n, 3, "none"), ("sps", 0, 0, "any")):
        tokens = n if family == "full" else n // 2
        docs = (None if kind == "none" else _packed_docs(rng, 2, tokens, family) if kind == "packed"
                else rng.integers(0, 3, size=(2, n)).astype(np.int64))
        _check(family, 2, 1, n, d, window=window, docs=docs, pkw=pkw, seed=n,
               dtype=torch.float16 if family == "sps" else torch.bfloat16, layout="bnhd")


@pytest.mark.parametrize("d", [128, 256])
def test_dkdv_more_chunks_than_mask_words(d):
    # 4200 positions: 132 query chunks for the first keys, past the 128 whose classes are precomputed.
    _check("full", 1, 1, 4200, d, seed=d)
