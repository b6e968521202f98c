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


@pytest.mark.parametrize("n", [2, 34, 126, 128, 130, 258, 514, 1090])
@pytest.mark.parametrize("family,window,pkw,kind", [("full", 0, None, "none"), ("full", 0, None, "any"),
                                                    ("sps", 5, None, "packed"), ("reverse_sps", 200, 3, "packed"),
                                                    ("sps", 0, 0, "any")])
def test_dq_forms_agree(n, family, window, pkw, kind):
    # The two-wave dQ form of large grids gives the bits of the one-wave form of small ones: two heads
    # repeated until the grid is past 512 tiles, against the two on their own (which the oracle tests
    # cover).
    from test_gpu_attention import FAMILY
    from sps_amd import attention as A

    rng = np.random.default_rng(n)
    tokens = n if family == "full" else n // 2
    docs = (None if kind == "none" else _packed_docs(rng, 1, tokens, family) if kind == "packed"
            else rng.integers(0, 3, size=(1, n)).astype(np.int64))
    docs = None if docs is None else torch.tensor(docs, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(n)
    dtype = torch.float16 if family == "sps" else torch.bfloat16
    q, k, v, do = (torch.randn(1, 2, n, 128, generator=g, device="cuda").to(dtype) for _ in range(4))
    copies = 514 // (2 * ((n + 127) // 128)) + 1
    fam = FAMILY[family]

    def grads(x, y, z, w):
        o, lse, x, y, z, ws = A.attention_forward(x, y, z, 0.1, fam, window, docs, pkw, keep_layout=True)
        return A.attention_backward(w, x, y, z, o, lse, 0.1, fam, window, docs, pkw, layout_workspace=ws)

    small = grads(q, k, v, do)
    large = grads(*(t.repeat(1, copies, 1, 1) for t in (q, k, v, do)))
    for a, b in zip(small, large):
        assert torch.equal(a.repeat(1, copies, 1, 1), b)
