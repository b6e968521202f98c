"""Performance cases of sps_amd: the calls a program makes, over the sizes it makes them at.

Three kinds of work, each through the package's public entry points:

* ``train`` / ``forward``: one attention layer on [B, H, N, D] views of [B, N, H, D] projections,
  with autograd (output and the three input gradients) or without (prefill, evaluation);
* ``block`` / ``prefill``: the attention path around it: RoPE and casts of fp32 projections, attention
  and their gradients; or a prompt's prefill over a few layers (document ids from token ids, then RoPE,
  attention and the decode caches of each layer);
* ``decode`` / ``generate``: one token of segmented decode attention over a layer's caches; or of a
  generation step over every layer, each with its KV-cache update.

``listed()`` holds the named cases, ``draw()`` others of the same ranges.
"""

from __future__ import annotations

import math

import torch

import sps_amd
from sps_amd import workloads

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
EOS, PAD, VOCAB = 1, 0, 32000
MAX_FLOPS = 1.2e12  # no drawn case costs more than the largest listed one
MAX_BYTES = 2.0e9
MAX_EXACT = 4.5e9   # B * H * N^2 up to which exact() builds dense float64 scores


def _attn(name, kind, family, batch, heads, head_dim, tokens, window=0, pkw=None, docs=True, dtype="bf16"):
    return {"name": name, "kind": kind, "family": family, "batch": batch, "heads": heads, "head_dim": head_dim,
            "tokens": tokens, "window": window, "pkw": pkw, "docs": docs, "dtype": dtype}


def _decode(name, kind, layers, batch, heads, head_dim, nq, len_lo, len_hi, storage, ring, dtype="bf16"):
    return {"name": name, "kind": kind, "layers": layers, "batch": batch, "heads": heads, "head_dim": head_dim,
            "nq": nq, "len_lo": len_lo, "len_hi": len_hi, "storage": storage, "ring": ring, "dtype": dtype}


def listed():
    return [
        # Evaluation of short rows, one document each: the smallest call, where the launch counts.
        _attn("forward short", "forward", "sps", 2, 8, 64, 512, window=64, docs=False),
        # Training of the Standard model on packed documents.
        _attn("train standard", "train", "full", 8, 12, 64, 2048),
        # Training of the SPS model with a 64-token window: the benchmark's headline.
        _attn("train sps w64", "train", "sps", 4, 16, 64, 2048, window=64),
        # Training with the window as wide as the context (the doubled-memory variant), wide heads.
        _attn("train sps wide", "train", "sps", 2, 16, 128, 2048, window=4096),
        # Training of the Reverse-SPS model at an odd length, both key windows set, float16.
        _attn("train reverse ragged", "train", "reverse_sps", 3, 10, 128, 1531, window=128, pkw=512, dtype="f16"),
        # The widest head dim that the entry points take.
        _attn("train d256", "train", "reverse_sps", 2, 8, 256, 1024, window=256),
        # The whole attention path of a small training batch, from the fp32 projections and back to them.
        _attn("block small", "block", "sps", 4, 12, 64, 1024, window=64),
        # Long-context prefill of one sequence, dense causal: the largest.
        _attn("forward long", "forward", "full", 1, 16, 128, 16384, docs=False),
        # Prefill of a generation batch: prompts of up to 1024 tokens, left padded, over four layers.
        dict(_attn("prefill prompts", "prefill", "reverse_sps", 16, 12, 64, 1024, window=64), layers=4),
        # Decode of a full serving batch: one query per sequence, ragged lengths.
        _decode("decode batch 64", "decode", 1, 64, 16, 64, 1, 512, 4096, 4096, 64),
        # One generation step of a 12-layer model, 16 sequences, input and <predict> query, caches updated.
        _decode("generate batch 16", "generate", 12, 16, 12, 64, 2, 1024, 4000, 4096, 64),
        # The same for one interactive sequence.
        _decode("generate single", "generate", 12, 1, 12, 64, 2, 512, 4000, 4096, 64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["train", "train", "train", "forward", "forward", "block", "prefill", "decode", "generate"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16"])
        head_dim = rng.choice([32, 64, 64, 64, 128, 128, 256])
        heads = max(2, _log_int(rng, 512, 2048) // head_dim)
        if kind in ("decode", "generate"):
            storage = 8 * _log_int(rng, 64, 1024)
            lo = rng.randint(storage // 16, storage // 2)
            case = _decode("", kind, 1 if kind == "decode" else rng.choice([4, 8, 12]), _log_int(rng, 1, 64), heads,
                           min(head_dim, 128), rng.choice([1, 2]), lo, rng.randint(lo, storage - 8), storage,
                           rng.choice([16, 64, 128]), rng.choice([dtype, dtype, dtype, "f32"]))
        else:
            family = rng.choice(["full", "sps", "sps", "reverse_sps"])
            tokens = _log_int(rng, 128, 4096 if kind != "forward" else 8192)
            if family == "full":
                window = 0
            else:
                window = rng.choice([16, 64, 64, 128, 512, 4096])
            pkw = _log_int(rng, 64, 1024) if family != "full" and rng.random() < 0.2 else None
            docs = kind != "forward" or rng.random() < 0.6
            case = _attn("", kind, family, _log_int(rng, 1, 16), heads, head_dim, tokens, window, pkw, docs, dtype)
            if kind == "prefill":
                case.update(family=rng.choice(["sps", "reverse_sps"]), window=rng.choice([16, 64, 128]), pkw=None,
                            layers=rng.choice([2, 4]))
        del case["name"]
        w = work(case)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return case


# Inputs -------------------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _positions(case):
    return case["tokens"] * (1 if case["family"] == "full" else 2)


def _doc_lengths(case, seed):
    """Token lengths of each row's documents."""
    if case["kind"] == "prefill":
        # A prompt is one document behind its left pads (each pad is a document of its own).
        g = torch.Generator().manual_seed(seed)
        t = case["tokens"]
        n = torch.randint(t // 2, t + 1, (case["batch"],), generator=g).tolist()
        return [[1] * (t - x) + [x] for x in n]
    if not case["docs"]:
        return [[case["tokens"]]] * case["batch"]
    return workloads.packed_doc_lengths(case["batch"], case["tokens"], seed)


def _docs(case, seed):
    if not case["docs"]:
        return None
    ids = torch.from_numpy(workloads.doc_ids_from_lengths(_doc_lengths(case, seed), case["tokens"]))
    if case["family"] != "full":
        ids = ids.repeat_interleave(2, dim=1)
    return ids.cuda()


def _freqs(n, head_dim, interleaved):
    """Complex frequencies of positions 0 .. n - 1 (each token's two positions share one when interleaved)."""
    inv = 10000.0 ** (-torch.arange(0, head_dim, 2, device="cuda").float() / head_dim)
    t = torch.arange(n // 2 if interleaved else n, device="cuda").float()
    f = torch.outer(t, inv)
    f = torch.polar(torch.ones_like(f), f)
    return f.repeat_interleave(2, dim=0).contiguous() if interleaved else f


def _attention(case, q, k, v, docs):
    scale = case["head_dim"] ** -0.5
    if case["family"] == "full":
        return sps_amd.full_attention(q, k, v, scale, documents_idx_BxT=docs)
    fn = sps_amd.sps_sliding_attention if case["family"] == "sps" else sps_amd.reverse_sps_sliding_attention
    return fn(q, k, v, scale, case["window"], documents_idx_BxT=docs, persistent_key_window=case["pkw"])


def prepare(case, seed):
    return {"train": _prepare_attention, "forward": _prepare_attention, "block": _prepare_block,
            "prefill": _prepare_prefill, "decode": _prepare_decode, "generate": _prepare_decode}[case["kind"]](case, seed)


def run(state):
    return {"train": _run_train, "forward": _run_forward, "block": _run_block, "prefill": _run_prefill,
            "decode": _run_decode, "generate": _run_generate}[state["case"]["kind"]](state)


def exact(case, seed):
    if case["kind"] in ("decode", "generate"):
        return _exact_decode(case, seed)
    if case["batch"] * case["heads"] * _positions(case) ** 2 * case.get("layers", 1) > MAX_EXACT:
        return None
    return {"train": _exact_train, "forward": _exact_forward, "block": _exact_block,
            "prefill": _exact_prefill}[case["kind"]](case, seed)


def _prepare_attention(case, seed):
    g, n = _gen(seed), _positions(case)
    shape, dtype = (case["batch"], n, case["heads"], case["head_dim"]), DTYPES[case["dtype"]]
    train = case["kind"] == "train"
    qkv = [_randn(g, *shape, dtype=dtype).transpose(1, 2).requires_grad_(train) for _ in range(3)]
    state = {"case": case, "qkv": qkv, "docs": _docs(case, seed)}
    if train:
        state["do"] = _randn(g, *shape, dtype=dtype).transpose(1, 2)
    return state


def _run_forward(s):
    with torch.no_grad():
        return _attention(s["case"], *s["qkv"], s["docs"])


def _run_train(s):
    o = _attention(s["case"], *s["qkv"], s["docs"])
    return [o.detach(), *torch.autograd.grad(o, s["qkv"], s["do"])]


def _prepare_block(case, seed):
    g, n = _gen(seed), _positions(case)
    b, h, d = case["batch"], case["heads"], case["head_dim"]
    proj = _randn(g, b, n, 3, h, d)
    return {"case": case, "qkv": [proj[:, :, i].requires_grad_() for i in range(3)], "docs": _docs(case, seed),
            "freqs": _freqs(n, d, case["family"] != "full"),
            "do": _randn(g, b, n, h, d, dtype=DTYPES[case["dtype"]]).transpose(1, 2)}


def _run_block(s):
    q, k, v = sps_amd.rope_qkv_for_attention(*s["qkv"], s["freqs"], DTYPES[s["case"]["dtype"]])
    o = _attention(s["case"], q, k, v, s["docs"])
    return [o.detach(), *torch.autograd.grad(o, s["qkv"], s["do"])]


def _prepare_prefill(case, seed):
    g, t, n = _gen(seed), case["tokens"], 2 * case["tokens"]
    b, h, d, layers, w = case["batch"], case["heads"], case["head_dim"], case["layers"], case["window"]
    dtype = DTYPES[case["dtype"]]
    tokens = torch.randint(2, VOCAB, (b, t), generator=g, device="cuda")
    lengths = torch.tensor([x[-1] for x in _doc_lengths(case, seed)], device="cuda")
    current = torch.arange(t, device="cuda")[None] >= t - lengths[:, None]
    tokens = torch.where(current, tokens, PAD)
    zeros = lambda *shape: torch.zeros(shape, dtype=dtype, device="cuda")  # noqa: E731
    ints = lambda *shape: torch.zeros(shape, dtype=torch.int64, device="cuda")  # noqa: E731
    return {"case": case, "tokens": tokens, "current": current, "freqs": _freqs(n, d, True),
            "proj": [_randn(g, b, n, 3, h, d) for _ in range(layers)],
            "nw_k": zeros(layers, b, h, w, d), "nw_v": zeros(layers, b, h, w, d),
            "nw_len": ints(layers, b), "nw_pos": ints(layers, b),
            "br_k": zeros(layers, b, h, t, d), "br_v": zeros(layers, b, h, t, d), "br_len": ints(layers, b, h)}


def _slots(case):
    """(ring, retained) slot of a token's two positions: the persistent key is the retained one."""
    return (1, 0) if case["family"] == "sps" else (0, 1)


def _run_prefill(s):
    case, outs = s["case"], []
    window_slot, retained_slot = _slots(case)
    with torch.no_grad():
        docs = sps_amd.document_ids(s["tokens"], eos_token_id=EOS, pad_token_id=PAD)
        for i, proj in enumerate(s["proj"]):
            q, k, v = sps_amd.rope_qkv_for_attention(*proj.unbind(2), s["freqs"], DTYPES[case["dtype"]])
            outs.append(_attention(case, q, k, v, docs))
            sps_amd.prefill_to_decode(
                k.transpose(1, 2), v.transpose(1, 2), s["current"], window_slot=window_slot,
                retained_slot=retained_slot, nw_k=s["nw_k"][i], nw_v=s["nw_v"][i], nw_len=s["nw_len"][i],
                nw_pos=s["nw_pos"][i], br_k=s["br_k"][i], br_v=s["br_v"][i], br_len=s["br_len"][i],
                window_tokens=case["window"])
    return [docs, outs, *(s[x] for x in ("nw_k", "nw_v", "nw_len", "nw_pos", "br_k", "br_v", "br_len"))]


def _prepare_decode(case, seed):
    g, layers, b, h, d = _gen(seed), case["layers"], case["batch"], case["heads"], case["head_dim"]
    dtype, nq = DTYPES[case["dtype"]], case["nq"]
    row = lambda: _randn(g, layers, b, h, d, dtype=dtype)  # noqa: E731
    lengths = torch.randint(case["len_lo"], case["len_hi"] + 1, (b,), generator=g, device="cuda")
    lengths = lengths[None, :, None].expand(layers, b, h).contiguous()
    return {"case": case, "q": _randn(g, layers, b, nq, h, d, dtype=dtype),
            "nw_k": _randn(g, layers, b, h, case["ring"], d, dtype=dtype),
            "nw_v": _randn(g, layers, b, h, case["ring"], d, dtype=dtype),
            "nw_len": torch.full((layers, b), case["ring"], dtype=torch.int64, device="cuda"),
            "nw_pos": torch.randint(0, case["ring"], (1, b), generator=g, device="cuda").repeat(layers, 1),
            "br_k": _randn(g, layers, b, h, case["storage"], d, dtype=dtype),
            "br_v": _randn(g, layers, b, h, case["storage"], d, dtype=dtype),
            "br_len": lengths.clone(), "start": lengths,
            "normal_k": row(), "normal_v": row(), "predict_k": row(), "predict_v": row(),
            "active": torch.ones(b, dtype=torch.bool, device="cuda")}


def _segments(s, i):
    case = s["case"]
    return [sps_amd.KVSegment(s["nw_k"][i], s["nw_v"][i], s["nw_len"][i], max_len_cap=case["ring"]),
            sps_amd.KVSegment(s["br_k"][i], s["br_v"][i], s["br_len"][i], max_len_cap=case["len_hi"])]


def _current(s, i):
    return {f"current_{x}_{y}_BxHxD": s[f"{x}_{y}"][i] for x in ("normal", "predict") for y in ("k", "v")}


def _extra(s, i):
    return [(s["normal_k"][i], s["normal_v"][i]), (s["predict_k"][i], s["predict_v"][i])]


def _run_decode(s):
    dtype = DTYPES[s["case"]["dtype"]]
    if s["case"]["nq"] == 2:
        return sps_amd.triton_segmented_q2_attention(s["q"][0], _segments(s, 0), **_current(s, 0), attn_dtype=dtype)
    return sps_amd.masked_kv_attention(s["q"][0][:, 0], _segments(s, 0), extra_kv=_extra(s, 0), attn_dtype=dtype)


def _run_generate(s):
    case, outs = s["case"], []
    dtype = DTYPES[case["dtype"]]
    s["br_len"].copy_(s["start"])  # every pass takes the step from the same lengths
    for i in range(case["layers"]):
        update = dict(nw_k=s["nw_k"][i], nw_v=s["nw_v"][i], nw_len=s["nw_len"][i], nw_pos=s["nw_pos"][i],
                      br_k=s["br_k"][i], br_v=s["br_v"][i], br_len=s["br_len"][i],
                      k_window_BxHxD=s["predict_k"][i], v_window_BxHxD=s["predict_v"][i],
                      k_retained_BxHxD=s["normal_k"][i], v_retained_BxHxD=s["normal_v"][i],
                      active_mask_B=s["active"], window_tokens=case["ring"])
        if case["nq"] == 2:
            outs.append(sps_amd.segmented_q2_attention_with_kv_update(
                s["q"][i], _segments(s, i), **_current(s, i), attn_dtype=dtype, **update))
        else:
            outs.append(sps_amd.segmented_q1_attention_with_kv_update(
                s["q"][i][:, 0], _segments(s, i), extra_kv=_extra(s, i), attn_dtype=dtype, **update))
    return [outs, *(s[x] for x in ("nw_k", "nw_v", "nw_len", "nw_pos", "br_k", "br_v", "br_len"))]


# Work and tolerances ------------------------------------------------------------------------------------


def _pairs(case):
    """Visible (query, key) pairs of one head over the batch, for the documents of seed 0 (a persistent-key
    window takes its share off the persistent keys)."""
    cfg = workloads.AttnConfig("", case["family"], case["batch"], case["heads"], case["head_dim"], case["tokens"],
                               case["window"], case["docs"], DTYPES[case["dtype"]])
    lengths = _doc_lengths(case, 0)
    pairs = workloads.visible_pairs(cfg, lengths)
    if case["pkw"] is not None:
        for row in lengths:
            for n in row:
                m = max(0, n - 1 - case["pkw"])
                pairs -= m * (m + 1)  # two queries of each token lose the persistent keys beyond the window
    return pairs


def work(case):
    if case["kind"] in ("decode", "generate"):
        rows = case["layers"] * case["batch"] * case["heads"]
        size = {"bf16": 2, "f16": 2, "f32": 4}[case["dtype"]]
        keys = rows * ((case["len_lo"] + case["len_hi"]) / 2 + case["ring"] + 2)
        d, nq = case["head_dim"], case["nq"]
        moved = keys * d * 2 * size + rows * nq * d * (size + 4)
        if case["kind"] == "generate":
            moved += rows * 4 * d * size  # the new rows' writes
        return {"bytes": moved, "flops": 4.0 * d * nq * keys}
    elems = case["batch"] * _positions(case) * case["heads"] * case["head_dim"]
    pairs = float(_pairs(case) * case["heads"] * case["head_dim"])
    layers = case.get("layers", 1)
    if case["kind"] == "train":
        return {"bytes": 8 * 2 * elems, "flops": 14 * pairs}
    if case["kind"] == "block":
        return {"bytes": (3 * 4 + 2 + 2 + 3 * 4) * elems, "flops": 14 * pairs}
    if case["kind"] == "forward":
        return {"bytes": 4 * 2 * elems, "flops": 4 * pairs}
    cached = sum(row[-1] for row in _doc_lengths(case, 0)) + case["batch"] * case["window"]
    cached *= case["heads"] * case["head_dim"] * 2 * 2
    return {"bytes": layers * ((3 * 4 + 2) * elems + cached), "flops": 4 * pairs * layers}


def tolerance(case):
    # Measured against exact(): outputs and gradients of N(0, 1) inputs carry the rounding of P and dS
    # to the input type and of the result itself; decode keeps fp32 from the cache on.
    if case["kind"] in ("decode", "generate"):
        return {"rel": 1e-5, "max": 1e-4}
    if case["dtype"] == "f16":
        return {"rel": 2e-3, "max": 5e-2}
    return {"rel": 1e-2, "max": 2e-1}


# 64-bit results -----------------------------------------------------------------------------------------


def _visible(case, docs_row, q0, q1, n):
    """[q1 - q0, n] bool: which keys the queries q0 .. q1 - 1 of a row see."""
    q = torch.arange(q0, q1, device="cuda")[:, None]
    k = torch.arange(n, device="cuda")[None]
    see = k <= q
    if docs_row is not None:
        see &= docs_row[q0:q1, None] == docs_row[None]
    if case["family"] != "full":
        dist = q // 2 - k // 2
        persistent = (k % 2) == (0 if case["family"] == "sps" else 1)
        near = torch.where(persistent, True if case["pkw"] is None else dist <= case["pkw"], dist <= case["window"])
        see &= near | (persistent & (k == q))
    return see


def _exact_attention(case, q, k, v, docs, do=None):
    """Output, and with `do` the gradients, of dense attention in float64, [B, H, N, D] each."""
    b, h, n, d = q.shape
    scale = d ** -0.5
    o = torch.empty(b, h, n, d, dtype=torch.float64, device="cuda")
    grads = [torch.zeros_like(o) for _ in range(3)] if do is not None else []
    for i in range(b):
        for q0 in range(0, n, 4096):
            q1 = min(n, q0 + 4096)
            hidden = ~_visible(case, None if docs is None else docs[i], q0, q1, n)[:, :q1]
            for j in range(h):
                qj, kj, vj = q[i, j, q0:q1].double(), k[i, j, :q1].double(), v[i, j, :q1].double()
                p = (qj @ kj.T).mul_(scale).masked_fill_(hidden, -math.inf)
                p = torch.softmax(p, dim=-1)
                o[i, j, q0:q1] = p @ vj
                if do is None:
                    continue
                dj = do[i, j, q0:q1].double()
                dp = dj @ vj.T
                ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * scale
                grads[0][i, j, q0:q1] = ds @ kj
                grads[1][i, j, :q1] += ds.T @ qj
                grads[2][i, j, :q1] += p.T @ dj
    return [o, *grads]


def _exact_forward(case, seed):
    s = _prepare_attention(case, seed)
    return _exact_attention(case, *s["qkv"], s["docs"])[0]


def _exact_train(case, seed):
    s = _prepare_attention(case, seed)
    return _exact_attention(case, *(t.detach() for t in s["qkv"]), s["docs"], s["do"])


def _rotate(x, freqs):
    """RoPE of [B, N, H, D] in float64."""
    z = torch.view_as_complex(x.double().unflatten(-1, (-1, 2)).contiguous())
    return torch.view_as_real(z * freqs.to(torch.complex128)[None, :, None]).flatten(-2)


def _exact_block(case, seed):
    s = _prepare_block(case, seed)
    q, k, v = (t.detach() for t in s["qkv"])
    q, k, v = (t.transpose(1, 2) for t in (_rotate(q, s["freqs"]), _rotate(k, s["freqs"]), v))
    o, dq, dk, dv = _exact_attention(case, q, k, v, s["docs"], s["do"])
    dq, dk, dv = (t.transpose(1, 2) for t in (dq, dk, dv))
    return [o, _rotate(dq, s["freqs"].conj()), _rotate(dk, s["freqs"].conj()), dv]


def _exact_prefill(case, seed):
    s = _prepare_prefill(case, seed)
    docs = _docs(case, seed)
    outs = []
    for proj in s["proj"]:
        q, k, v = proj.unbind(2)
        q, k, v = (t.transpose(1, 2) for t in (_rotate(q, s["freqs"]), _rotate(k, s["freqs"]), v))
        outs.append(_exact_attention(case, q, k, v, docs)[0])
    return [docs, outs, None, None, None, None, None, None, None]


def _exact_decode(case, seed):
    s = _prepare_decode(case, seed)
    d, nq = case["head_dim"], case["nq"]
    outs = []
    for i in range(case["layers"]):
        out = torch.empty(case["batch"], nq, case["heads"], d, dtype=torch.float64, device="cuda")
        for b in range(case["batch"]):
            n = int(s["br_len"][i, b, 0])
            ks, vs = ([s["nw_" + x][i, b].double(), s["br_" + x][i, b, :, :min(n, case["len_hi"])].double(),
                       s["normal_" + x][i, b, :, None].double(), s["predict_" + x][i, b, :, None].double()]
                      for x in ("k", "v"))
            kk, vv = torch.cat(ks, dim=1), torch.cat(vs, dim=1)  # [H, T, D]
            for t in range(nq):
                p = (kk * s["q"][i, b, t, :, None].double()).sum(-1) * d ** -0.5
                if nq == 2 and t == 0:
                    p[:, -1] = -math.inf  # the input query does not see the <predict> key
                p = torch.softmax(p, dim=-1)
                out[b, t] = (p[..., None] * vv).sum(1)
        outs.append(out if nq == 2 else out[:, 0])
    if case["kind"] == "decode":
        return outs[0]
    return [outs, None, None, None, None, None, None, None]
