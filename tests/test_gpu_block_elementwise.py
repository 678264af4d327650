"""GPU parity of the fused elementwise steps of the DiT block (LayerNorm + modulation, gated residual, GELU; each with
its tangent), called through the C ABI, against the CPU oracle (library layer_norm / gelu under torch.func.jvp, fp32,
pinned in tests/test_oracle_dit_block.py).

Tolerance: one 16-bit rounding of an fp32 result, with a quarter of slack for the fp32 arithmetic itself:
|got - want| <= 1.25 * 2^-8 |want| + 1e-3 elementwise for bf16 (1.25 * 2^-11 |want| + 2e-4 for fp16; the absolute term
covers cancellation near zero), and
relative-L2 <= 3e-3 (bf16) / 5e-4 (fp16).
"""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

REL = {torch.bfloat16: (1.25 * 2.0 ** -8, 1e-3, 3e-3), torch.float16: (1.25 * 2.0 ** -11, 2e-4, 5e-4)}


def check(name, got, want, dtype, more=0.0):
    got, want = got.float().cpu().double(), want.double()
    rel, ab, l2 = REL[dtype]
    err = (got - want).abs()
    worst = float((err / (rel * want.abs() + ab + more)).max())
    rl = float((got - want).norm() / want.norm().clamp_min(1e-30))
    print(f"  {name}: worst/tol={worst:.2f} rel_l2={rl:.3e}", flush=True)
    assert math.isfinite(worst) and worst <= 1.0, f"{name}: {worst} x the elementwise bound"
    assert rl <= l2, f"{name}: rel-L2 {rl} > {l2}"


def rnd(g, dtype, *shape, std=1.0, mean=0.0):
    return (torch.randn(*shape, generator=g) * std + mean).to(dtype)


@pytest.mark.parametrize("D", [8, 64, 256, 520, 2048, 5120, 8192])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_ln_modulate_widths(pkg, block_oracle, gpu, D, dtype):
    g = torch.Generator().manual_seed(D)
    rows, rpg = 24, 4
    x, tx = rnd(g, dtype, rows, D, std=2.0, mean=0.5), rnd(g, dtype, rows, D, std=0.5)
    sh, sc, tsh, tsc = (rnd(g, dtype, rows // rpg, D, std=s) for s in (1.0, 0.3, 0.3, 0.1))
    print(f"ln_modulate D={D} {dtype}", flush=True)
    d = lambda t: t.to(gpu)
    y, ty = pkg.ln_modulate(d(x), d(sh), d(sc), d(tx), d(tsh), d(tsc))
    want, twant = block_oracle.ln_modulate_torch(x, sh, sc, tx, tsh, tsc, rows_per_group=rpg)
    check("y", y, want, dtype)
    check("ty", ty, twant, dtype)
    # values only, and a tangent with a modulation that does not move
    y2, none = pkg.ln_modulate(d(x), d(sh), d(sc))
    assert none is None
    check("y (values only)", y2, want, dtype)      # another instantiation of the kernel: same bar, not the same bits
    y3, ty3 = pkg.ln_modulate(d(x), d(sh), d(sc), d(tx))
    _, twant3 = block_oracle.ln_modulate_torch(x, sh, sc, tx, rows_per_group=rpg)
    check("y (fixed modulation)", y3, want, dtype)
    check("ty (fixed modulation)", ty3, twant3, dtype)


def test_ln_modulate_video_shape_and_stacked_output(pkg, block_oracle, gpu):
    g = torch.Generator().manual_seed(1)
    B, T, Hh, W, D = 2, 3, 4, 5, 256
    x, tx = rnd(g, torch.bfloat16, B, T, Hh, W, D), rnd(g, torch.bfloat16, B, T, Hh, W, D)
    sh, sc = rnd(g, torch.bfloat16, B * T, D), rnd(g, torch.bfloat16, B * T, D, std=0.3)
    y, ty = pkg.ops.stacked_pair(x.shape, x.dtype, gpu)
    pkg.ln_modulate(x.to(gpu), sh.to(gpu), sc.to(gpu), tx.to(gpu), out=y, tout=ty)
    both = pkg.ops.as_stacked(y.reshape(B, -1, D), ty.reshape(B, -1, D))
    assert both is not None and both.shape == (2 * B, T * Hh * W, D) and both.data_ptr() == y.data_ptr()
    assert pkg.ops.as_stacked(y.clone(), ty.clone()) is None
    want, twant = block_oracle.ln_modulate_torch(x, sh, sc, tx, rows_per_group=Hh * W)
    check("y", y, want, torch.bfloat16)
    check("ty", ty, twant, torch.bfloat16)


def test_ln_modulate_large_mean(pkg, block_oracle, gpu):
    """Rows whose mean is far larger than their spread: the variance is taken around the mean, not from raw moments."""
    g = torch.Generator().manual_seed(2)
    x = rnd(g, torch.bfloat16, 8, 2048, std=0.5, mean=60.0)
    sh, sc = torch.zeros(1, 2048).bfloat16(), torch.zeros(1, 2048).bfloat16()
    y, _ = pkg.ln_modulate(x.to(gpu), sh.to(gpu), sc.to(gpu))
    want, _ = block_oracle.ln_modulate_torch(x, sh, sc, rows_per_group=8)
    check("y", y, want, torch.bfloat16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,D,rpg", [(1, 8, 1), (30, 264, 5), (64, 2048, 16)])
def test_gated_residual(pkg, block_oracle, gpu, dtype, rows, D, rpg):
    g = torch.Generator().manual_seed(rows + D)
    x, res, tx, tres = (rnd(g, dtype, rows, D) for _ in range(4))
    gate, tgate = rnd(g, dtype, rows // rpg, D), rnd(g, dtype, rows // rpg, D, std=0.3)
    d = lambda t: t.to(gpu)
    out, tout = pkg.gated_residual(d(x), d(res), d(gate), d(tx), d(tres), d(tgate))
    want, twant = block_oracle.gated_residual_torch(x, res, gate, tx, tres, tgate, rows_per_group=rpg)
    check("out", out, want, dtype)
    check("tout", tout, twant, dtype)
    o2, none = pkg.gated_residual(d(x), d(res), d(gate))
    assert none is None
    check("out (values only)", o2, want, dtype)
    xd, txd = d(x), d(tx)
    o3, t3 = pkg.gated_residual(xd, d(res), d(gate), txd, d(tres), None, inplace=True)
    assert o3.data_ptr() == xd.data_ptr() and t3.data_ptr() == txd.data_ptr() and torch.equal(o3, out)
    _, twant3 = block_oracle.gated_residual_torch(x, res, gate, tx, tres, None, rows_per_group=rpg)
    check("tout (fixed gate, in place)", t3, twant3, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,D,rpg", [(1, 8, 1), (30, 264, 5), (9, 520, 3), (64, 2048, 16), (7, 5120, 7), (10, 5128, 5), (6, 8192, 2)])
def test_gated_residual_ln_modulate(pkg, block_oracle, gpu, dtype, rows, D, rpg):
    """One pass against the two it stands for, and the LayerNorm against the oracle of the residual that was stored."""
    g = torch.Generator().manual_seed(rows + D)
    x, res, tx, tres = (rnd(g, dtype, rows, D) for _ in range(4))
    gate, sc, sh, tgate, tsc, tsh = (rnd(g, dtype, rows // rpg, D, std=s) for s in (1.0, 0.3, 1.0, 0.3, 0.1, 0.3))
    d = lambda *ts: [t.to(gpu) for t in ts]
    for moving in (None, False, True):       # values only; a tangent with a modulation that does not move; one that does
        t, mt = ((tx, tres) if moving is not None else (None, None)), ((tgate, tsh, tsc) if moving else (None, None, None))
        dt, dmt = [None if v is None else v.to(gpu) for v in t], [None if v is None else v.to(gpu) for v in mt]
        (dx, dres, dg, dsh, dsc) = d(x, res, gate, sh, sc)
        out, tout, y, ty = pkg.ops.gated_residual_ln_modulate(dx, dres, dg, dsh, dsc, *dt, *dmt)
        ref = pkg.gated_residual(dx, dres, dg, *dt, dmt[0])
        assert torch.equal(out, ref[0]) and (tout is None) == (ref[1] is None) == (moving is None)
        assert torch.equal(dx.cpu(), x) and (tout is None or torch.equal(tout, ref[1]))
        want, twant = block_oracle.ln_modulate_torch(out.cpu(), sh, sc, None if tout is None else tout.cpu(), mt[1], mt[2], rows_per_group=rpg)
        check(f"y ({moving})", y, want, dtype)
        if moving is None:
            assert ty is None
        elif rows * D > 8:                    # (rows of 8 elements: the tangent of n is a difference of near-equal terms)
            check(f"ty ({moving})", ty, twant, dtype)
    # modulations of different groups go through the two passes
    out, _, y, _ = pkg.ops.gated_residual_ln_modulate(dx, dres, dg[:1], dsh, dsc)
    ref, _ = pkg.gated_residual(dx, dres, dg[:1])
    assert torch.equal(out, ref) and torch.equal(y, pkg.ln_modulate(ref, dsh, dsc)[0])


@pytest.mark.parametrize("rows,D,rpg", [(30, 264, 5), (64, 2048, 16), (7, 5120, 7), (10, 5128, 5)])      # (the last: two launches)
def test_gated_residual_ln_modulate_into_its_inputs(pkg, gpu, rows, D, rpg):
    """Outputs that are inputs of the same call: the same bits as into buffers of their own."""
    g = torch.Generator().manual_seed(rows + D)
    big = [rnd(g, torch.bfloat16, rows, D).to(gpu) for _ in range(4)]                             # x, res, tx, tres
    mod = [rnd(g, torch.bfloat16, rows // rpg, D, std=0.3).to(gpu) for _ in range(6)]             # gate, shift, scale and their tangents
    call = lambda x, res, tx, tres, **outs: pkg.ops.gated_residual_ln_modulate(x, res, *mod[:3], tx, tres, *mod[3:], **outs)
    want = call(*big)
    for y, ty in ((0, 2), (1, 3), (3, 0)):
        ins = [t.clone() for t in big]
        assert all(torch.equal(a, b) for a, b in zip(call(*ins, y=ins[y], ty=ins[ty]), want))


@pytest.mark.parametrize("rows,rpg,D", [(24, 4, 8), (17, 17, 264), (66, 33, 2048), (8, 1, 2056), (90, 45, 4104), (40, 40, 5120), (21, 21, 8192),
                                        (9000, 4500, 64)])      # (the last: rows enough for runs longer than the shortest)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_reverse_mode(pkg, gpu, rows, rpg, D, dtype):
    """Groups of one run and of several, ragged ones among them; columns that fill the 256 threads' chunks of 8 once to four
    times, with and without a remainder; against torch's own reverse mode in 64 bits.  Bounds: one rounding of each result, as
    above; a sum over n rows of products of size one is off by sqrt(n) 2^-24 more."""
    g = torch.Generator().manual_seed(rows + D)
    x, res, dy, dskip = rnd(g, dtype, rows, D, std=2.0, mean=0.5), *(rnd(g, dtype, rows, D) for _ in range(3))
    sc, gate = rnd(g, dtype, rows // rpg, D, std=0.3), rnd(g, dtype, rows // rpg, D)
    rep = lambda m: m.repeat_interleave(rpg, dim=0)
    xr, scr, shr, rr, gr = (t.double().requires_grad_(True) for t in (x, sc, torch.zeros_like(sc), res, gate))
    y = torch.nn.functional.layer_norm(xr, (D,), eps=1e-6) * (1 + rep(scr)) + rep(shr)
    dx, dsc, dsh = torch.autograd.grad(y, (xr, scr, shr), dy.double())
    d = lambda t: t.to(gpu)
    for skip in (None, dskip):
        got = pkg.ops.ln_modulate_bwd(d(x), d(sc), d(dy), None if skip is None else d(skip))
        check("dx", got[0], dx if skip is None else dx + skip.double(), dtype)
        check("dshift", got[1], dsh, dtype)
        check("dscale", got[2], dsc, dtype)
    dres, dgate = torch.autograd.grad(rep(gr) * rr, (rr, gr), dy.double())
    got = pkg.ops.gated_residual_bwd(d(res), d(gate), d(dy))
    check("dres", got[0], dres, dtype)
    check("dgate", got[1], dgate, dtype)


@pytest.mark.parametrize("rows,rpg,D", [(17, 17, 264), (66, 33, 2048), (5, 1, 64), (34, 17, 2056), (33, 33, 4104)])
def test_reverse_mode_without_eps(pkg, gpu, rows, rpg, D):
    """eps = 0, runs that end inside the rows that are in flight together (four up to 2048 columns, two up to 4096): the rows past
    the end, which have no variance, stay out of the column sums.  Bounds as in test_reverse_mode."""
    dtype, g = torch.bfloat16, torch.Generator().manual_seed(rows + D)
    x, dy, sc = rnd(g, dtype, rows, D, std=2.0, mean=0.5), rnd(g, dtype, rows, D), rnd(g, dtype, rows // rpg, D, std=0.3)
    rep = lambda m: m.repeat_interleave(rpg, dim=0)
    xr, scr, shr = (t.double().requires_grad_(True) for t in (x, sc, torch.zeros_like(sc)))
    y = torch.nn.functional.layer_norm(xr, (D,), eps=0.0) * (1 + rep(scr)) + rep(shr)
    want = torch.autograd.grad(y, (xr, shr, scr), dy.double())
    for name, got, ref in zip(("dx", "dshift", "dscale"), pkg.ops.ln_modulate_bwd(x.to(gpu), sc.to(gpu), dy.to(gpu), eps=0.0), want):
        check(name, got, ref, dtype)


@pytest.mark.parametrize("rows,K,hidden,D", [(1, 32, 32, 16), (3, 2048, 256, 2048), (8, 256, 64, 48), (16, 288, 32, 80), (17, 5120, 256, 128), (40, 96, 96, 32)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_modulation(pkg, gpu, rows, K, hidden, D, dtype):
    """One row to several tiles of 16, k shorter than the sixteen wavefronts that share it and with a remainder, vectors that end
    inside a workgroup; in 64 bits with the two intermediate roundings that the library's layers have as well."""
    g = torch.Generator().manual_seed(rows + K)
    emb, temb = rnd(g, dtype, rows, K), rnd(g, dtype, rows, K, std=0.3)
    lora, tlora = rnd(g, dtype, rows, 3 * D, std=0.3), rnd(g, dtype, rows, 3 * D, std=0.1)
    w1, w2 = [[rnd(g, dtype, *s, std=s[1] ** -0.5) for _ in range(3)] for s in ((hidden, K), (3 * D, hidden))]
    r = lambda t: t.to(dtype).double()
    act, tact = torch.func.jvp(torch.nn.functional.silu, (emb.double(),), (temb.double(),))
    layers = lambda a, i: r(r(a) @ w1[i].double().T) @ w2[i].double().T
    # a first-layer output that lies so near a rounding boundary that fp32 sums take it across moves by one unit of its last place
    most = lambda a: max(float((r(a) @ w1[i].double().T).abs().max()) * float(w2[i].abs().max()) for i in range(3))
    flip = (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10) * max(most(act), most(tact))
    cut = lambda m: m.reshape(rows, 3, D).transpose(0, 1)
    want = torch.stack([cut(layers(act, i) + lora.double()) for i in range(3)])
    d = lambda t: t.to(gpu)
    args = (d(emb), d(lora), [d(w) for w in w1], [d(w) for w in w2])
    out, none = pkg.ops.modulation(*args)
    assert none is None
    check("out", out, want, dtype, flip)
    for te, tl in ((temb, tlora), (temb, None), (None, tlora), (None, None)):
        out, tout = pkg.ops.modulation(*args, None if te is None else d(te), None if tl is None else d(tl), tangent=True)
        check("out", out, want, dtype, flip)
        twant = torch.stack([cut(layers(tact if te is not None else 0 * tact, i) + (0 if tl is None else tl.double())) for i in range(3)])
        check("tout", tout, twant, dtype, flip)


@pytest.mark.parametrize("value", [float("inf"), float("nan"), -3.0e38])
def test_modulation_of_an_embedding_that_does_not_move(pkg, gpu, value):
    """Its tangent is the added vectors' own, whatever the embedding's values are: no 0 times infinity."""
    rn = lambda *s: torch.randn(*s, device=gpu).bfloat16()
    emb, lora, tlora = rn(3, 64), rn(3, 48), rn(3, 48)
    w1, w2 = [rn(32, 64) for _ in range(3)], [rn(48, 32) for _ in range(3)]
    emb[1, 5] = value
    _, tout = pkg.ops.modulation(emb, lora, w1, w2, tlora=tlora, tangent=True)
    assert torch.equal(tout, tlora.reshape(3, 3, 16).transpose(0, 1).expand(3, 3, 3, 16))


@pytest.mark.parametrize("rows,K,hidden,D", [(1, 32, 32, 16), (24, 256, 64, 48), (40, 96, 96, 32)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_modulation_reverse_mode(pkg, gpu, rows, K, hidden, D, dtype):
    """Gradients of emb, lora and the six weights, and the gradients of a penalty on emb's, against 64 bits.  Bound: a gradient goes
    through at most four 16-bit roundings of relative size 2^-9 (bf16) / 2^-12 (fp16), the penalty's through twice as many."""
    from importlib import import_module
    fn = import_module(pkg.__name__ + ".dit_block")._ModulationFn
    g = torch.Generator().manual_seed(rows)
    ins = [rnd(g, dtype, rows, K), rnd(g, dtype, rows, 3 * D, std=0.3)]
    for s in ((hidden, K), (3 * D, hidden)):
        ins += [rnd(g, dtype, *s, std=s[1] ** -0.5) for _ in range(3)]
    dout, v = rnd(g, dtype, 3, 3, rows, D), rnd(g, dtype, rows, K)

    def grads(f, to):
        leaves = [to(t).requires_grad_(True) for t in ins]
        first = torch.autograd.grad(f(*leaves), leaves, to(dout), create_graph=True)
        return *first, *torch.autograd.grad((first[0] * to(v)).sum(), (leaves[0], leaves[2], leaves[5]))

    def ref(emb, lora, *w):
        a = torch.nn.functional.silu(emb)
        return torch.stack([(a @ w[i].T @ w[3 + i].T + lora).reshape(rows, 3, D).transpose(0, 1) for i in range(3)])

    unit = 2.0 ** (-9 if dtype == torch.bfloat16 else -12)
    got, want = grads(fn.apply, lambda t: t.to(gpu)), grads(ref, lambda t: t.double())
    for i, (a, b) in enumerate(zip(got, want)):
        rel = float((a.detach().double().cpu() - b.detach()).norm() / b.detach().norm())
        print(f"  gradient {i}: rel_l2={rel:.2e}", flush=True)
        assert a.dtype == dtype and rel <= (4 if i < 8 else 8) * unit, i


def off16(t):
    """t's values, contiguous, but one element past a 16-byte boundary (a slice of a larger buffer)."""
    v = torch.empty(t.numel() + 1, device=t.device, dtype=t.dtype)[1:].view(t.shape).copy_(t)
    assert v.is_contiguous() and v.data_ptr() % 16 == t.element_size()
    return v


def test_inputs_that_start_off_16_bytes(pkg, gpu):
    """Gradients, embeddings and weights that are contiguous slices of larger buffers: the same bits as from aligned ones.  Weights
    like that go to the modules (the fused call would copy them every time)."""
    g = torch.Generator().manual_seed(3)
    x, dy, dskip, res = (rnd(g, torch.bfloat16, 12, 264).to(gpu) for _ in range(4))
    sc = rnd(g, torch.bfloat16, 3, 264, std=0.3).to(gpu)
    same = lambda a, b: all(p is None and q is None or torch.equal(p, q) for p, q in zip(a, b))
    assert same(pkg.ops.ln_modulate_bwd(off16(x), off16(sc), off16(dy), off16(dskip)), pkg.ops.ln_modulate_bwd(x, sc, dy, dskip))
    assert same(pkg.ops.gated_residual_bwd(off16(res), off16(sc), off16(dy)), pkg.ops.gated_residual_bwd(res, sc, dy))

    torch.manual_seed(0)
    m = pkg.Block(256, 64, 2, use_adaln_lora=True, adaln_lora_dim=32).to(gpu, torch.bfloat16).eval()
    for p in m.parameters():
        torch.nn.init.normal_(p, std=p.shape[-1] ** -0.5)
    x, emb, lora, ctx = (torch.randn(*s, device=gpu).bfloat16() for s in ((1, 2, 2, 4, 256), (1, 2, 256), (1, 2, 768), (1, 8, 64)))
    temb, tlora = torch.randn_like(emb), torch.randn_like(lora)
    run = lambda e, l, te, tl: (m(x, e, ctx, None, l), *m.forward_jvp(x, x, e, te, ctx, None, l, tl))
    with torch.no_grad():
        want = run(emb, lora, temb, tlora)
        assert same(run(off16(emb), off16(lora), off16(temb), off16(tlora)), want)
        for layer in (m.adaln_modulation_mlp[1], m.adaln_modulation_mlp[2]):
            layer.weight = torch.nn.Parameter(off16(layer.weight.detach()))
            assert m._fused_modulations(emb, lora, x) is None
        for a, b in zip(run(emb, lora, temb, tlora), want):      # the modules round the modulation vectors once more
            assert float((a.float() - b.float()).norm()) <= 1e-2 * float(b.float().norm())


def test_modulation_dispatch(pkg, gpu):
    """The block takes the fused call only for the plain MLPs of one 16-bit type; otherwise the modules themselves, which agree."""
    torch.manual_seed(0)
    m = pkg.Block(256, 64, 2, use_adaln_lora=True, adaln_lora_dim=32).to(gpu, torch.bfloat16).eval()
    for p in m.parameters():
        torch.nn.init.normal_(p, std=p.shape[-1] ** -0.5)
    emb, lora = (torch.randn(2, 3, n, device=gpu).bfloat16() for n in (256, 768))
    x = torch.randn(2, 3, 2, 2, 256, device=gpu).bfloat16()
    assert m._fused_modulations(emb, lora, x)[0].requires_grad
    with torch.no_grad():
        got, _ = m._fused_modulations(emb, lora, x)
        for i, name in enumerate(("self_attn", "cross_attn", "mlp")):
            for a, b in zip(got[i].unbind(0), m._modulation(getattr(m, "adaln_modulation_" + name), emb, lora, x)):
                assert float((a.float() - b.reshape(6, 256).float()).abs().max()) <= 2.0 ** -6 * float(b.float().abs().max())
        assert m._fused_modulations(emb.float(), lora, x) is None                                     # another type
        assert m._fused_modulations(emb, lora[:, :1], x) is None                                      # a term that is broadcast
        assert m._fused_modulations(emb[:, :1].expand(2, 65, 256), lora[:, :1].expand(2, 65, 768), x) is None     # many rows
        with torch.autocast("cuda", dtype=torch.float16):
            assert m._fused_modulations(emb, lora, x) is None
        handle = m.adaln_modulation_mlp[1].register_forward_hook(lambda mod, a, out: out * 2)
        assert m._fused_modulations(emb, lora, x) is None
        handle.remove()
        handle = torch.nn.modules.module.register_module_forward_hook(lambda mod, a, out: None)
        assert m._fused_modulations(emb, lora, x) is None
        handle.remove()
        assert m._fused_modulations(emb, lora, x) is not None
        m.adaln_modulation_mlp[0] = torch.nn.GELU()
        assert m._fused_modulations(emb, lora, x) is None


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [8, 1000, 1 << 20])
def test_gelu(pkg, block_oracle, gpu, dtype, n):
    g = torch.Generator().manual_seed(n)
    h, th = rnd(g, dtype, n, std=2.5), rnd(g, dtype, n)
    a, ta = pkg.gelu(h.to(gpu), th.to(gpu))
    want, twant = block_oracle.gelu_torch(h, th)
    check("a", a, want, dtype)
    check("ta", ta, twant, dtype)
    a2, none = pkg.gelu(h.to(gpu))
    assert none is None
    check("a (values only)", a2, want, dtype)
    hd, thd = h.to(gpu), th.to(gpu)
    a3, ta3 = pkg.gelu(hd, thd, inplace=True)
    assert a3.data_ptr() == hd.data_ptr() and torch.equal(a3, a) and torch.equal(ta3, ta)


def test_gelu_tails(pkg, block_oracle, gpu):
    h = torch.tensor([-40.0, -12.0, -6.0, -1e-3, 0.0, 1e-3, 6.0, 12.0], dtype=torch.bfloat16)
    a, ta = pkg.gelu(h.to(gpu), torch.ones_like(h).to(gpu))
    want, twant = block_oracle.gelu_torch(h, torch.ones_like(h))
    check("a", a, want, torch.bfloat16)
    check("ta", ta, twant, torch.bfloat16)
    assert torch.isfinite(a.float()).all() and torch.isfinite(ta.float()).all()


def test_more_than_2_31_elements(pkg, block_oracle, gpu):
    """Offsets beyond 32 bits in the three elementwise kernels: 2.4e9-element tensors, checked at both ends."""
    rows, D, rpg = 1179648, 2048, 4096
    assert rows * D > 2 ** 31
    g = torch.Generator(device=gpu).manual_seed(4)
    x = torch.empty(rows, D, device=gpu, dtype=torch.bfloat16)
    for i in range(0, rows, 131072):
        x[i:i + 131072] = torch.randn(131072, D, generator=g, device=gpu).bfloat16()
    mod = torch.randn(3, rows // rpg, D, generator=g, device=gpu).bfloat16()
    ends = torch.cat([torch.arange(0, 8), torch.arange(rows - 8, rows)]).to(gpu)
    grp = (ends // rpg)
    y, _ = pkg.ln_modulate(x, mod[0], mod[1])
    want, _ = block_oracle.ln_modulate_torch(x[ends].cpu(), mod[0][grp].cpu(), mod[1][grp].cpu())
    check("ln_modulate ends", y[ends], want, torch.bfloat16)
    out, _ = pkg.gated_residual(x, y, mod[2])
    want, _ = block_oracle.gated_residual_torch(x[ends].cpu(), y[ends].cpu(), mod[2][grp].cpu())
    check("gated_residual ends", out[ends], want, torch.bfloat16)
    del out
    a, _ = pkg.gelu(x)
    want, _ = block_oracle.gelu_torch(x[ends].cpu())
    check("gelu ends", a[ends], want, torch.bfloat16)
