"""Decode at the edges of its chunk sizes and merge forms, against the float64 oracle (GPU): grids just
below and above the limit that picks the chunk of 8 or 16 loads, 64 and 65 chunks (all records loaded
ahead of the lengths, or rounds of live chunks), and queries whose type differs from the extras'."""

import numpy as np
import pytest
import torch

from oracle import decode as Dc
from sps_amd import decode_attention as DA

pytestmark = pytest.mark.gpu


def _check(b, h, d, nq, kv, q_dtype, e_dtype, storages, n_extra, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(s, generator=g)  # noqa: E731
    q = r(b, nq, h, d).to(q_dtype).cuda()
    segs = []
    for i, s in enumerate(storages):
        # Lengths over the whole range, the ends among them; a chunk edge and one past it.
        shape = (b, h) if i % 2 else (b,)
        ln = torch.randint(0, s + 1, shape, generator=g)
        ln.view(-1)[0], ln.view(-1)[-1] = s, (s // 2) // 8 * 8 + 1
        segs.append(DA.KVSegment(r(b, h, s, d).to(kv).cuda(), r(b, h, s, d).to(kv).cuda(),
                                 ln.to(torch.int64 if i else torch.int32).cuda()))
    extras = [(r(b, h, d).to(e_dtype).cuda(), r(b, h, d).to(e_dtype).cuda()) for _ in range(n_extra)]
    masks = ([0b11, 0b10] if nq == 2 else [1, 1])[:n_extra]
    out = torch.full((b, nq, h, d), float("nan"), device="cuda")
    DA._run_decode(q, nq, segs, extras, masks, out)
    n64 = lambda t: t.double().cpu().numpy()  # noqa: E731
    want = Dc.attend(n64(q), [(n64(s.k), n64(s.v), s.lengths.cpu().numpy(), None) for s in segs],
                     [(n64(k), n64(v)) for k, v in extras], masks, nq)
    # fp32 rounding: a score is a sum of D products (error D 2^-24 sum |q k| <= D 2^-24 |q| |k|), its
    # error moves the weights by twice as much relatively, and the weighted sum of n values adds n 2^-24.
    norm = lambda t: float(t.double().norm(dim=-1).max()) if t.numel() else 0.0  # noqa: E731
    keys = [s.k for s in segs] + [k for k, _ in extras]
    vals = [s.v for s in segs] + [v for _, v in extras]
    score = d * 2.0 ** -24 * norm(q) * max(norm(k) for k in keys) / d ** 0.5
    bound = (2 * score + (sum(storages) + 2) * 2.0 ** -24) * max(float(v.abs().max()) for v in vals)
    assert np.abs(out.double().cpu().numpy() - want).max() <= bound


# D = 64 in 16 bits: 512 keys a chunk of 16 loads; 2048 workgroups of those is the limit.
@pytest.mark.parametrize("b,h,storage", [(1, 1, 1), (1, 1, 255), (1, 2, 257), (4, 64, 512 * 8), (4, 64, 512 * 8 + 1),
                                         (1, 1, 256 * 64), (1, 1, 256 * 64 + 1)])
@pytest.mark.parametrize("nq", [1, 2])
def test_chunk_sizes(b, h, storage, nq):
    _check(b, h, 64, nq, torch.bfloat16, torch.bfloat16, torch.bfloat16, [storage], 2 if nq == 2 else 1, storage)


@pytest.mark.parametrize("d", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("kv,q_dtype,e_dtype", [(torch.float32, torch.float32, torch.float32),
                                                (torch.float16, torch.float32, torch.float16),
                                                (torch.bfloat16, torch.bfloat16, torch.float32),
                                                (torch.bfloat16, torch.float16, torch.bfloat16)])
def test_types_and_segments(d, kv, q_dtype, e_dtype):
    for nq in (1, 2):
        # Three segments (q = 1) over few chunks, and enough keys for more than 64 of them at D = 256.
        _check(2, 3, d, nq, kv, q_dtype, e_dtype, [33, 700, 64] if nq == 1 else [40, 2300], 2, d + nq)
    _check(2, 2, d, 1, kv, q_dtype, e_dtype, [90], 0, d)


# The rows that end the half-size chunks: as many as the merge loads ahead (24; 16 at D = 256) and one more,
# on a grid of one workgroup per CU and a larger one, and two batches of 8 past them (one at D = 256).
@pytest.mark.parametrize("d,b,h,storage", [(64, 2, 8, 256 * 24), (64, 2, 8, 256 * 24 + 1), (64, 1, 2, 256 * 40),
                                           (64, 1, 2, 256 * 40 + 1), (256, 2, 16, 64 * 16), (256, 2, 16, 64 * 16 + 1),
                                           (256, 1, 3, 64 * 24), (256, 1, 3, 64 * 24 + 1)])
@pytest.mark.parametrize("nq", [1, 2])
def test_rows_at_the_merge_limits(d, b, h, storage, nq):
    _check(b, h, d, nq, torch.bfloat16, torch.bfloat16, torch.bfloat16, [storage], 2 if nq == 2 else 1, storage)


@pytest.mark.parametrize("nq", [1, 2])
def test_workspace_of_a_larger_call(nq, monkeypatch):
    # A workspace sized for 2049 workgroups of full chunks, then a call of half as many, which would take
    # half-size chunks if the workspace held their records.
    b, h, storage = 3, 683, 300
    need = DA._decode_ws_bytes(False, b, h, 64, nq, 0, (storage,))
    small = DA._decode_ws_bytes(False, b, 512, 64, nq, 0, (storage,))
    assert need < small
    monkeypatch.setattr(DA, "_decode_ws_bytes", lambda *a: need)
    _check(b, 512, 64, nq, torch.bfloat16, torch.bfloat16, torch.bfloat16, [storage], 1, 3)
