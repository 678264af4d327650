"""Attention calls that read K and V where they are (head dim 128, few query rows): the same bits as the same kernels on the re-tiled image (without
tangents), and parity with the oracle (with all tangents), where what lies behind the last row is not a number."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(g, B, L, H, dtype, scale, layout):
    """[B, H, L, 128] view of memory whose rows behind the last one are not numbers."""
    shape = (B, L + 70, H, 128) if layout == "blhd" else (B, H, L + 70, 128)
    m = torch.full(shape, float("nan"), device="cuda", dtype=dtype)
    x = (torch.randn(B, H, L, 128, device="cuda", generator=g) * scale).to(dtype)
    view = m[:, :L].transpose(1, 2) if layout == "blhd" else m[:, :, :L]
    view.copy_(x)
    return view


# keys: one, a tile's edge, a step's edge, ragged; the same workgroup shape (128 rows and two key groups, 256 rows) on both sides, no cut, no stream
@pytest.mark.parametrize("dtype, layout", [(torch.bfloat16, "blhd"), (torch.float16, "bhld")])
@pytest.mark.parametrize("rows", [128, 256])
@pytest.mark.parametrize("B, H, Lq, Lkv, causal, lens", [
    (1, 2, 1, 1, False, None), (2, 3, 129, 32, False, None), (1, 2, 300, 33, False, None), (1, 16, 255, 255, False, None), (2, 16, 520, 520, True, None),
    (1, 40, 1000, 1000, False, None), (1, 40, 1100, 65, False, None), (2, 16, 513, 700, False, (1, 411)),
])
def test_forward_gives_the_bits_of_the_re_tiled_image(pkg, stream_override, forward_override, rows, B, H, Lq, Lkv, causal, lens, dtype, layout):
    ops = pkg.ops
    stream_override(chunk=1)
    forward_override(rows, 1)
    g = torch.Generator(device="cuda").manual_seed(Lq + Lkv)
    q = _rows(g, B, Lq, H, dtype, 1.0, layout)
    k, v = _rows(g, B, Lkv, H, dtype, 2.0, layout), _rows(g, B, Lkv, H, dtype, 1.0, layout)
    lens = None if lens is None else torch.tensor(lens, dtype=torch.int32, device="cuda")
    lib, packed = pkg._lib.load_library(), ops.pack_kv(k, v)
    results = []
    for in_place in (True, False):
        o, lse = torch.full((B, H, Lq, 128), float("nan"), device="cuda", dtype=dtype), torch.full((B, H, Lq), float("nan"), device="cuda")
        d = ops._packed_desc(B, H, Lq, Lkv, 128, 128, dtype, 128 ** -0.5)
        d.causal, d.q, d.k, d.v, d.o, d.lse = int(causal), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr()
        d.key_lens = None if lens is None else lens.data_ptr()
        d.q_stride, d.k_stride, d.v_stride, d.o_stride = (ops._strides3(t) for t in (q, k, v, o))
        stream = torch.cuda.current_stream().cuda_stream
        assert (lib.cosmos_attn_fwd_in_place(ctypes.byref(d), stream) if in_place
                else lib.cosmos_attn_run(ctypes.byref(d), packed.image.data_ptr(), packed.image.numel(), stream)) == 0
        results.append((o, lse))
    (o, lse), (want, want_lse) = results
    assert torch.isfinite(o).all() and torch.isfinite(lse).all()
    assert torch.equal(lse, want_lse) and torch.equal(o, want)


@pytest.mark.parametrize("dtype, layout", [(torch.bfloat16, "blhd"), (torch.float16, "bhld")])
@pytest.mark.parametrize("B, H, Lq, Lkv, causal, lens", [
    (1, 2, 1, 1, False, None), (2, 3, 129, 32, False, None), (1, 2, 300, 33, False, None), (1, 16, 255, 255, False, None), (2, 16, 520, 520, True, None),
    (1, 40, 1000, 1000, False, None), (1, 40, 1100, 65, False, None), (2, 16, 513, 700, False, (1, 411)),
])
def test_forward_by_the_library_s_choice(pkg, B, H, Lq, Lkv, causal, lens, dtype, layout):
    """Whichever kernels the two ways take: parity in 64 bits."""
    ops = pkg.ops
    g = torch.Generator(device="cuda").manual_seed(Lq + Lkv)
    q = _rows(g, B, Lq, H, dtype, 1.0, layout)
    k, v = _rows(g, B, Lkv, H, dtype, 2.0, layout), _rows(g, B, Lkv, H, dtype, 1.0, layout)
    lens = None if lens is None else torch.tensor(lens, dtype=torch.int32, device="cuda")
    o, _, lse = ops.fwd_jvp(q, k, v, causal=causal, key_lens=lens)
    s = (q.double() @ k.double().transpose(-1, -2)) * 128 ** -0.5
    if causal:
        s.masked_fill_(torch.ones(Lq, Lkv, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    if lens is not None:
        s.masked_fill_(torch.arange(Lkv, device="cuda")[None, None, None] >= lens[:, None, None, None], float("-inf"))
    want = s.softmax(-1) @ v.double()
    # limits of the parity tests; fp16 rounds 8 times finer
    assert (o.double() - want).norm() / want.norm() < (5e-3 if dtype == torch.bfloat16 else 5e-3 / 8) and (lse - s.logsumexp(-1)).abs().max() < 2e-3


@pytest.mark.parametrize("dtype, layout", [(torch.bfloat16, "blhd"), (torch.float16, "bhld")])
@pytest.mark.parametrize("B, H, Lq, Lkv, lens", [(1, 2, 1, 1, None), (1, 3, 127, 33, None), (2, 2, 300, 256, None), (1, 16, 255, 255, None), (2, 4, 385, 1100, (3, 1100))])
def test_all_tangents(pkg, B, H, Lq, Lkv, lens, dtype, layout):
    ops = pkg.ops
    g = torch.Generator(device="cuda").manual_seed(Lq + Lkv)
    mk = lambda L, scale: _rows(g, B, L, H, dtype, scale, layout)
    q, k, v, tq, tk, tv = mk(Lq, 1.0), mk(Lkv, 1.0), mk(Lkv, 1.0), mk(Lq, 0.1), mk(Lkv, 0.1), mk(Lkv, 0.1)
    dev = None if lens is None else torch.tensor(lens, dtype=torch.int32, device="cuda")
    o, to, _ = ops.fwd_jvp(q, k, v, tq, tk, tv, key_lens=dev)
    assert torch.isfinite(o).all() and torch.isfinite(to).all()
    d = lambda x: x.double()
    s, ds = d(q) @ d(k).transpose(-1, -2) * 128 ** -0.5, (d(tq) @ d(k).transpose(-1, -2) + d(q) @ d(tk).transpose(-1, -2)) * 128 ** -0.5
    if lens is not None:
        out = torch.arange(Lkv, device="cuda")[None, None, None] >= dev[:, None, None, None]
        s = s.masked_fill(out, float("-inf"))
    p = s.softmax(-1)
    want = p @ d(v)
    twant = (p * ds) @ d(v) - (p * ds).sum(-1, keepdim=True) * want + p @ d(tv)
    limit = 5e-3 if dtype == torch.bfloat16 else 5e-3 / 8                 # limit of the parity tests; fp16 rounds 8 times finer
    assert (d(o) - want).norm() / want.norm() < limit and (d(to) - twant).norm() / twant.norm() < limit


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B, S, H, Lkv, causal, scale, how", [
    (2, 255, 16, 255, False, None, "dense"), (1, 300, 3, 300, True, 0.2, "heads first"), (1, 6144, 1, 64, False, None, "dense"), (1, 6145, 1, 64, False, None, "dense"),
    (1, 130, 2, 77, False, 1.0, "unaligned"), (1, 130, 2, 77, False, None, "strided"), (1, 64, 2, 64, False, None, "expanded"), (1, 256, 4, 2000, False, None, "dense"),
    (1, 1024, 16, 1024, False, None, "dense"), (1, 1560, 16, 512, False, None, "dense"), (1, 3520, 40, 3520, False, 0.1, "heads first"), (1, 1560, 16, 77, False, None, "dense"),
])
def test_attention_is_the_general_call(pkg, monkeypatch, B, S, H, Lkv, causal, scale, how, dtype):
    """``attention`` takes a shorter way on the host for these calls: the same bits as ``fwd_jvp`` for every layout, its refusals for what it refuses."""
    g = torch.Generator(device="cuda").manual_seed(S)

    def make(L):
        x = torch.randn(B, L, H, 128, device="cuda", generator=g).to(dtype)
        if how == "heads first":
            return x.transpose(1, 2).contiguous().transpose(1, 2)
        if how == "unaligned":
            return torch.empty(x.numel() + 4, device="cuda", dtype=dtype)[4:].view(x.shape).copy_(x)
        if how == "strided":
            return torch.empty(B, L, H, 256, device="cuda", dtype=dtype)[..., ::2].copy_(x)
        if how == "expanded":
            return x[:, :1].expand(B, L, H, 128)
        return x

    q, k, v = make(S), make(Lkv), make(Lkv)
    t = lambda x: x.transpose(1, 2)
    general, calls = pkg.ops.fwd_jvp, []
    monkeypatch.setattr(pkg.ops, "fwd_jvp", lambda *a, **kw: calls.append(1) or general(*a, **kw))
    with torch.no_grad():
        got = pkg.attention_forward(q, k, v, softmax_scale=scale, causal=causal, dtype=dtype)
    # (a call that is looked over twice, as the last four were, waits 4 us longer than by either way alone)
    assert len(calls) == (1 if S > pkg.ops._ONE_DESCRIPTOR_ROWS or how in ("unaligned", "strided") else 0)
    want = general(t(q), t(k), t(v), causal=causal, sm_scale=scale, out_layout="blhd", need_lse=False)[0].transpose(1, 2)
    assert got.is_contiguous() and got.dtype == dtype and torch.equal(got, want)
    with torch.no_grad(), pytest.raises(AssertionError):
        pkg.attention_forward(q, k[:, :-1], v, dtype=dtype)
    with torch.no_grad(), pytest.raises((RuntimeError, NotImplementedError)):
        pkg.attention_forward(q.cpu(), k.cpu(), v.cpu(), dtype=dtype)


@pytest.mark.parametrize("how", ["expanded", "dense"])
def test_infinite_values_stay_what_they_are(pkg, how):
    """A value that is infinite in every row gives infinity and not NaN, also where rows behind the last one are formed (40 keys of a step of 64)."""
    q = torch.randn(1, 70, 2, 128, device="cuda").bfloat16()
    k, v = (torch.randn(1, 1, 2, 128, device="cuda").bfloat16() for _ in range(2))
    v[..., 5] = float("inf")
    k, v = (x.expand(1, 40, 2, 128) if how == "expanded" else x.repeat(1, 40, 1, 1) for x in (k, v))
    with torch.no_grad():
        o = pkg.attention_forward(q, k, v, dtype=torch.bfloat16)
    assert torch.isposinf(o[..., 5]).all() and torch.isfinite(o[..., :5]).all() and torch.isfinite(o[..., 6:]).all()
