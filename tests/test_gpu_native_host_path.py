"""The native host path of the entry points against their general path (GPU): the same call with the
binding switched off has to give the same bits, gradients and cache updates over the forms both take,
and everything the binding does not take (tracing, transforms, hooks that change layouts, copies,
errors) has to come out of the general path as before."""

import contextlib

import pytest
import torch
import torch.utils.checkpoint
from torch.autograd import forward_ad

import sps_amd
from sps_amd import _native as N

pytestmark = pytest.mark.gpu


class _Off:
    attention = rope = decode = staticmethod(lambda *a: None)
    kv_update = staticmethod(lambda a: False)


@contextlib.contextmanager
def _general_path():
    real = N.binding()
    N._binding = _Off
    try:
        yield
    finally:
        N._binding = real


class _Counting:
    """The binding, with the number of calls it took."""

    def __init__(self):
        self.real, self.taken = N.binding(), 0

    def __getattr__(self, name):
        def call(*args):
            r = getattr(self.real, name)(*args)
            self.taken += r is not None and r is not False
            return r
        return call

    def __enter__(self):
        N._binding = self
        return self

    def __exit__(self, *exc):
        N._binding = self.real


def _qkv(b=2, h=3, n=96, d=64, dtype=torch.bfloat16, layout="bnhd", seed=0):
    g = torch.Generator().manual_seed(seed)
    shape = (b, n, h, d) if layout != "bhnd" else (b, h, n, d)
    ts = [torch.randn(shape, generator=g).to(dtype).cuda() for _ in range(4)]
    if layout == "bnhd":
        ts = [t.transpose(1, 2) for t in ts]
    elif layout == "packed":  # slices of one projection: strided, not dense
        p = torch.randn((b, n, 3, h, d), generator=g).to(dtype).cuda()
        ts = [p[:, :, i].transpose(1, 2) for i in range(3)] + [ts[3].transpose(1, 2)]
    elif layout == "odd":  # rows not 16-byte aligned
        ts = [torch.randn((b, h, n, d + 1), generator=g).to(dtype).cuda()[..., :d] for _ in range(4)]
    return ts


def _docs(b, n, dtype=torch.int64):
    return (torch.arange(n, device="cuda") // 40).to(dtype).expand(b, n).contiguous()


FNS = {
    "full": lambda q, k, v, docs: sps_amd.full_attention(q, k, v, 0.125, documents_idx_BxT=docs),
    "sps": lambda q, k, v, docs: sps_amd.sps_sliding_attention(q, k, v, 0.125, 7, documents_idx_BxT=docs),
    "reverse": lambda q, k, v, docs: sps_amd.reverse_sps_sliding_attention(
        q, k, v, 0.125, 9, documents_idx_BxT=docs, persistent_key_window=11),
}


@pytest.mark.parametrize("layout,native", [("bnhd", True), ("bhnd", True), ("packed", False), ("odd", False)])
@pytest.mark.parametrize("docs", [None, torch.int32, torch.int64])
@pytest.mark.parametrize("name", list(FNS))
def test_attention_matches_the_general_path(name, docs, layout, native):
    def both():
        q, k, v, do = _qkv(layout=layout, dtype=torch.float16 if name == "sps" else torch.bfloat16)
        ids = None if docs is None else _docs(2, 96, docs)
        leaves = [t.detach().requires_grad_() for t in (q, k, v)]
        out = FNS[name](*leaves, ids)
        grads = torch.autograd.grad(out, leaves, do, retain_graph=True)
        again = torch.autograd.grad(out, leaves, do)
        with torch.no_grad():
            plain = FNS[name](*leaves, ids)
        with torch.inference_mode():
            inf = FNS[name](q, k, v, ids)
        return [out, *grads, *again, plain, inf.clone()]

    with _Counting() as c:
        got = both()
        assert c.taken == (3 if native else 2 if layout == "packed" else 0)
    with _general_path():
        want = both()
    for x, y in zip(got, want):
        assert torch.equal(x, y) and x.stride() == y.stride()


def test_partial_gradients_and_missing_ones():
    q, k, v, do = _qkv()
    for wrt in ((0,), (1,), (2,), (0, 2)):
        res = []
        for ctx in (contextlib.nullcontext, _general_path):
            with ctx():
                ts = [t.detach().requires_grad_(i in wrt) for i, t in enumerate((q, k, v))]
                res.append(torch.autograd.grad(FNS["sps"](*ts, None), [ts[i] for i in wrt], do))
        assert all(torch.equal(a, b) for a, b in zip(*res))


def test_hooks_checkpoint_and_other_streams():
    q, k, v, do = _qkv()
    ids = _docs(2, 96)

    def grads(run):
        ts = [t.detach().requires_grad_() for t in (q, k, v)]
        return torch.autograd.grad(run(*ts), ts, do)

    want = grads(lambda *t: FNS["sps"](*t, ids))
    seen = []
    pack = lambda t: (seen.append(tuple(t.shape)), t)[1]  # noqa: E731

    def hooked(*t):
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
            return FNS["sps"](*t, ids)

    def offloaded(*t):
        with torch.autograd.graph.save_on_cpu():
            return FNS["sps"](*t, ids)

    def relaid(*t):  # the hooks hand back rows that the kernels cannot read in place
        def odd(x):
            if x.dim() != 4:
                return x
            buf = x.new_empty(*x.shape[:-1], x.shape[-1] + 1)[..., :-1]
            return buf.copy_(x)
        with torch.autograd.graph.saved_tensors_hooks(odd, lambda x: x):
            return FNS["sps"](*t, ids)

    runs = [hooked, offloaded, lambda *t: torch.utils.checkpoint.checkpoint(
        lambda *x: FNS["sps"](*x, ids), *t, use_reentrant=False)]
    side = torch.cuda.Stream()

    def on_stream(*t):
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            o = FNS["sps"](*t, ids)
        torch.cuda.current_stream().wait_stream(side)
        o.record_stream(torch.cuda.current_stream())
        return o

    for run in (*runs, on_stream):
        got = grads(run)
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert seen
    with pytest.raises(N.NativeError):  # O itself misaligned: refused by the library, on either path
        grads(relaid)


def test_transforms_keep_the_registered_ops():
    q, k, v, do = _qkv(b=1, h=2, n=64)
    loss = lambda a, b, c: (FNS["sps"](a, b, c, None) * do).float().sum()  # noqa: E731
    res = []
    for ctx in (contextlib.nullcontext, _general_path):
        with ctx():
            # A batch of output gradients, a second differentiation, forward-mode, a traced call.
            ts = [t.detach().requires_grad_() for t in (q, k, v)]
            out = FNS["full"](*ts, None)
            kinds = []
            for f in (lambda: torch.func.grad(loss, argnums=(0, 1, 2))(q, k, v),
                      lambda: torch.autograd.grad(out, ts, torch.stack([do, do * 2]), is_grads_batched=True,
                                                  retain_graph=True),
                      lambda: torch.autograd.grad(torch.autograd.grad(out, ts, do, create_graph=True)[0].float().sum(),
                                                  ts, retain_graph=True),
                      lambda: torch.vmap(lambda x: FNS["full"](x, x, x, None))(torch.stack([q, k])),
                      lambda: _jvp(q, k, v)):
                try:
                    r = f()
                    kinds.append([t.clone() for t in (r if isinstance(r, tuple) else (r,))])
                except (RuntimeError, NotImplementedError) as e:
                    kinds.append(type(e).__name__)
            res.append(kinds)
    for a, b in zip(*res):
        if isinstance(a, str) or isinstance(b, str):
            assert a == b
        else:
            assert all(torch.equal(x, y) for x, y in zip(a, b))


def _jvp(q, k, v):
    with forward_ad.dual_level():
        d = forward_ad.make_dual(q, torch.ones_like(q))
        out = forward_ad.unpack_dual(FNS["sps"](d, k, v, None))
        return out.primal.clone(), torch.tensor(out.tangent is None)


def test_refused_calls_stay_refused():
    q, k, v, _ = _qkv()
    bad = [lambda: FNS["sps"](q[:, :, :95], k[:, :, :95], v[:, :, :95], None), lambda: FNS["sps"](q, k[..., :32], v, None),
           lambda: FNS["sps"](q.float(), k.float(), v.float(), None), lambda: FNS["sps"](q, k.half(), v, None),
           lambda: FNS["sps"](q, k, v, _docs(2, 96).float()), lambda: FNS["sps"](q, k, v, _docs(2, 94)),
           lambda: FNS["sps"](q.cpu(), k.cpu(), v.cpu(), None),
           lambda: sps_amd.full_attention(q, k, v, float("nan")), lambda: sps_amd.full_attention(q, k, v, 1e300),
           lambda: sps_amd.sps_sliding_attention(q, k, v, 0.1, "x")]
    for f in bad:
        errors = []
        for ctx in (contextlib.nullcontext, _general_path):
            with ctx():
                with pytest.raises(Exception) as e:
                    f()
                errors.append((e.type, str(e.value)))
        assert errors[0] == errors[1]
    assert sps_amd.sps_sliding_attention(q, k, v, 0.1, 1 << 40).shape == q.shape  # any window, as before


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("in_dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("batched", [False, True])
def test_rope_matches_the_general_path(in_dtype, out_dtype, batched):
    g = torch.Generator().manual_seed(3)
    proj = torch.randn((2, 40, 3, 4, 32), generator=g).to(in_dtype).cuda()
    f = torch.polar(torch.ones(2, 40, 16), torch.randn((2, 40, 16), generator=g)).cuda()
    f = f if batched else f[0].contiguous()
    gs = [torch.randn((2, 4, 40, 32), generator=g).to(out_dtype).cuda() for _ in range(3)]

    def both():
        ts = [proj[:, :, i].detach().requires_grad_() for i in range(3)]
        outs = sps_amd.rope_qkv_for_attention(*ts, f, out_dtype)
        grads = torch.autograd.grad(outs, ts, gs)
        some = torch.autograd.grad(sps_amd.rope_qkv_for_attention(*ts, f, out_dtype)[1], ts[1], gs[1])
        pair = sps_amd.apply_rotary_emb(ts[0], ts[1], f)
        pg = torch.autograd.grad(pair, ts[:2], [x.transpose(1, 2).to(in_dtype) for x in gs[:2]])
        with torch.no_grad():
            plain = sps_amd.rope_qkv_for_attention(*ts, f, out_dtype)
        return [*outs, *grads, *some, *pair, *pg, *plain]

    with _Counting() as c:
        got = both()
        assert c.taken == 4
    with _general_path():
        want = both()
    for x, y in zip(got, want):
        assert torch.equal(x, y) and x.stride() == y.stride()


def _decode_state(b=3, h=2, d=64, storage=80, ring=16, dtype=torch.bfloat16, len_dtype=torch.int64, seed=0):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(s, generator=g).to(dtype).cuda()  # noqa: E731
    return dict(q=r(b, 2, h, d), nw_k=r(b, h, ring, d), nw_v=r(b, h, ring, d), br_k=r(b, h, storage, d),
                br_v=r(b, h, storage, d), rows=[r(b, h, d) for _ in range(4)],
                nw_len=torch.tensor([ring, 3, 0], dtype=len_dtype).cuda(),
                nw_pos=torch.tensor([5, 0, 0], dtype=len_dtype).cuda(),
                br_len=torch.randint(0, storage + 1, (b, h), generator=g).to(len_dtype).cuda(),
                active=torch.tensor([True, False, True]).cuda())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("len_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("window,cap", [(16, None), (16, 50), (0, 200)])
def test_decode_and_update_match_the_general_path(dtype, len_dtype, window, cap):
    def both(native):
        outs = []
        for nq in (1, 2):
            for fold in (False, True):
                s = _decode_state(dtype=dtype, len_dtype=len_dtype)
                nk, nv, pk, pv = s["rows"]
                segs = [sps_amd.KVSegment(s["br_k"], s["br_v"], s["br_len"], cap)]
                if window:
                    segs.insert(0, sps_amd.KVSegment(s["nw_k"], s["nw_v"], s["nw_len"], window))
                upd = dict(k_window_BxHxD=pk, v_window_BxHxD=pv, k_retained_BxHxD=nk, v_retained_BxHxD=nv,
                           active_mask_B=s["active"], window_tokens=window,
                           **{x: s[x] for x in ("nw_k", "nw_v", "nw_len", "nw_pos", "br_k", "br_v", "br_len")})
                cur = dict(current_normal_k_BxHxD=nk, current_normal_v_BxHxD=nv, current_predict_k_BxHxD=pk,
                           current_predict_v_BxHxD=pv)
                if nq == 2 and fold:
                    o = sps_amd.segmented_q2_attention_with_kv_update(s["q"], segs, **cur, attn_dtype=dtype, **upd)
                elif nq == 2:
                    o = sps_amd.triton_segmented_q2_attention(s["q"], segs, **cur, attn_dtype=dtype)
                    sps_amd.fused_sps_kv_update(**upd)
                elif fold:
                    o = sps_amd.segmented_q1_attention_with_kv_update(
                        s["q"][:, 1], segs, extra_kv=[(nk, nv), (pk, pv)], attn_dtype=dtype, **upd)
                else:
                    o = sps_amd.masked_kv_attention(s["q"][:, 1], segs, extra_kv=[(pk, pv)], attn_dtype=dtype)
                    sps_amd.fused_sps_kv_update(**upd)
                outs += [o, *(s[x] for x in ("nw_k", "nw_v", "nw_len", "nw_pos", "br_k", "br_v", "br_len"))]
        return outs

    with _Counting() as c:
        got = both(True)
        assert c.taken == 6
    with _general_path():
        want = both(False)
    for x, y in zip(got, want):
        assert torch.equal(x, y) and x.stride() == y.stride()


def test_decode_calls_that_need_the_general_path():
    s = _decode_state()
    nk, nv, pk, pv = s["rows"]
    seg = sps_amd.KVSegment(s["br_k"], s["br_v"], s["br_len"])
    calls = [
        lambda: sps_amd.masked_kv_attention(s["q"][:, 0], [], extra_kv=[(nk, nv)], attn_dtype=torch.bfloat16),
        lambda: sps_amd.masked_kv_attention(s["q"][:, 0], (seg,), attn_dtype=torch.bfloat16),
        lambda: sps_amd.masked_kv_attention(s["q"][:, 0], [seg], extra_kv=[(nk.float(), nv)], attn_dtype=torch.float32),
        lambda: sps_amd.masked_kv_attention(s["q"][:, 0], [seg], extra_kv=[(nk, nv[:1])], attn_dtype=torch.bfloat16),
        lambda: sps_amd.masked_kv_attention(s["q"][:, 0], [sps_amd.KVSegment(s["br_k"], s["br_v"], s["br_len"], -1)],
                                            attn_dtype=torch.bfloat16),
        lambda: sps_amd.masked_kv_attention(s["q"][:, 0], [sps_amd.KVSegment(s["br_k"], s["br_v"].half(), s["br_len"])],
                                            attn_dtype=torch.bfloat16),
        lambda: sps_amd.triton_segmented_q2_attention(
            s["q"][:, :1], [seg], current_normal_k_BxHxD=nk, current_normal_v_BxHxD=nv, current_predict_k_BxHxD=pk,
            current_predict_v_BxHxD=pv, attn_dtype=torch.bfloat16),
        lambda: sps_amd.triton_segmented_q1_attention(s["q"][:, 0], [seg] * 4, attn_dtype=torch.bfloat16),
    ]
    for f in calls:
        res = []
        for ctx in (contextlib.nullcontext, _general_path):
            with ctx():
                try:
                    r = f()
                    res.append(r if r is None else r.clone())
                except Exception as e:  # noqa: BLE001
                    res.append((type(e), str(e)))
        a, b = res
        assert torch.equal(a, b) if isinstance(a, torch.Tensor) else a == b


def test_graph_capture_of_native_calls():
    q, k, v, do = _qkv()
    ids = _docs(2, 96)
    leaves = [t.detach().requires_grad_() for t in (q, k, v)]

    def step():
        o = FNS["sps"](*leaves, ids)
        return [o, *torch.autograd.grad(o, leaves, do)]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = step()
    for seed in range(3):
        fresh = _qkv(seed=seed + 1)
        with torch.no_grad():
            for t, x in zip((*leaves, do), fresh):
                t.copy_(x)
        graph.replay()
        got = [t.clone() for t in outs]
        want = step()
        assert all(torch.equal(a, b) for a, b in zip(got, want))

