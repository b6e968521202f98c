"""The document prepass at the lengths where its form changes (2, 4 or 8 ids a thread, ids not held in
registers), with aligned and misaligned ids of both types and lengths that no store width divides:
masks of both schedules bit-exact against the oracle (GPU)."""

import numpy as np
import pytest
import torch

from oracle import mask as M
from sps_amd import _native as N
from sps_amd import attention as SA

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 2047, 2048, 2049, 2050, 4095, 4096, 4098, 8192, 8194])
@pytest.mark.parametrize("dtype,offset", [(torch.int64, 0), (torch.int64, 1), (torch.int32, 0), (torch.int32, 1),
                                          (torch.int32, 3)])
def test_runs_and_plans(n, dtype, offset):
    rng = np.random.default_rng(10 * n + offset)
    rows = 2
    # One row of runs (single positions and long ones), one whose ids decrease now and then.
    ids = np.stack([np.cumsum(rng.random(n) < 0.01), np.cumsum(rng.random(n) < 0.02) % 3])
    flat = torch.empty(rows * n + offset, dtype=dtype, device="cuda")
    docs = flat[offset:].view(rows, n)
    docs.copy_(torch.from_numpy(ids))
    families = [(N.FAMILY_FULL, 0)] + ([(N.FAMILY_SPS, 7)] if n % 2 == 0 else [])
    for family, window in families:
        want = torch.from_numpy(np.stack([M.mask_c(family, n, r, window) for r in ids])).cuda()
        for schedule in (0, 1):
            assert torch.equal(SA.attention_mask(family, n, docs, window=window, schedule=schedule), want)


@pytest.mark.parametrize("n", [2051, 4097, 4101, 6001, 6002, 8189, 8190, 8191])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_rows_no_store_divides(n, dtype):
    # Run bounds stored from LDS, and ids loaded in pieces from rows that start at any id.
    test_runs_and_plans(n, dtype, 0)
