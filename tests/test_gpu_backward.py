"""GPU parity of the HIP backward (dq, dk, dv), called through the C ABI, against the CPU oracle.

Oracle: fp64 closed form pinned to torch autograd of math SDPA (tests/test_oracle.py).  Inputs of the GPU call:
q, k, v rounded to 16 bit, and the forward's own o and lse from the HIP forward kernel (as in training).
Tolerances for 16-bit tensors: max-abs <= 2e-2 * max(1, max|want|) (gradients are sums over rows and can be large; a
bf16 result carries a relative rounding of 2^-9) and relative-L2 <= 1e-2 per gradient (the reference's procedure,
flash_attention_jvp_triton.py:567-607, uses atol 1e-2 with rtol 1e-2 / 2e-2 against a 16-bit-rounded naive attention).
"""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

MAX_ABS, REL_L2 = 2e-2, 1e-2


def check(oracle, name, got, want, max_abs=MAX_ABS, rel_l2=REL_L2):
    ma, rl = oracle.error_metrics(got.float().cpu(), want)
    max_abs = max_abs * max(1.0, float(abs(want).max()))
    print(f"  {name}: max_abs={ma:.3e} (limit {max_abs:.3e}) rel_l2={rl:.3e}", flush=True)
    assert math.isfinite(ma) and ma <= max_abs, f"{name}: max-abs {ma} > {max_abs}"
    assert rl <= rel_l2, f"{name}: rel-L2 {rl} > {rel_l2}"


def run_bwd(pkg, oracle, gpu, shape_q, shape_kv=None, causal=False, sm_scale=None, seed=0, dtype=torch.bfloat16,
            primal_std=1.0, dout_std=1.0):
    q, k, v, _, _, _ = oracle.make_inputs(shape_q, shape_kv, seed=seed, primal_std=primal_std, dtype=dtype)
    g = torch.Generator().manual_seed(seed + 1000)
    dout = (torch.randn(q.shape, generator=g) * dout_std).to(dtype)
    print(f"bwd case q={tuple(q.shape)} kv={tuple(k.shape)} causal={causal} dtype={dtype} seed={seed}", flush=True)
    qd, kd, vd, dd = (x.to(gpu) for x in (q, k, v, dout))
    o, _, lse = pkg.attention_with_lse(qd, kd, vd, causal=causal, sm_scale=sm_scale)
    dq, dk, dv = pkg.ops.bwd(qd, kd, vd, o, lse, dd, causal=causal, sm_scale=sm_scale)
    torch.cuda.synchronize()
    rq, rk, rv = oracle.grads_closed_form(q, k, v, dout, sm_scale=sm_scale, causal=causal)
    check(oracle, "dq", dq, rq)
    check(oracle, "dk", dk, rk)
    check(oracle, "dv", dv, rv)
    return dq, dk, dv


def test_bwd_smallest(pkg, oracle, gpu):
    run_bwd(pkg, oracle, gpu, (1, 1, 64, 128))


@pytest.mark.parametrize("Lq,Lkv", [(1, 1), (50, 37), (31, 33), (129, 1), (5, 300), (96, 160)])
def test_bwd_ragged_small(pkg, oracle, gpu, Lq, Lkv):
    run_bwd(pkg, oracle, gpu, (1, 2, Lq, 128), (1, 2, Lkv, 128), seed=Lq + Lkv)


@pytest.mark.parametrize("Lq", [1, 31, 32, 33, 63, 165])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_bwd_query_stream_layouts(pkg, oracle, gpu, Lq, dtype):
    """The fused re-tiling of q, dout and the row sums dout . o: full, ragged and single-row tiles, with the three tensors in three
    different layouts, with dS kept and with the dQ kernel that reads the row sums from memory (same tolerances as above)."""
    q, k, v, _, _, _ = oracle.make_inputs((2, 3, Lq, 128), (2, 3, 70, 128), seed=Lq, dtype=dtype)
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(Lq)).to(dtype)
    want = oracle.grads_closed_form(q, k, v, dout)
    qd, kd, vd = q.transpose(1, 2).contiguous().to(gpu).transpose(1, 2), k.to(gpu), v.to(gpu)
    wide = torch.zeros(2, 3, Lq, 136, dtype=dtype, device=gpu)
    wide[..., :128] = dout.to(gpu)
    o, _, lse = pkg.fwd_jvp(qd, kd, vd)
    for max_ds_mib in (None, -1):
        for name, got, ref in zip(("dq", "dk", "dv"), pkg.ops.bwd(qd, kd, vd, o, lse, wide[..., :128], max_ds_mib=max_ds_mib), want):
            check(oracle, name, got, ref)


@pytest.mark.parametrize("Lkv", [1, 33, 96, 128, 130, 260])
def test_bwd_key_stream_tiles(pkg, oracle, gpu, Lkv):
    """Runs of four re-tiled K^T tiles: fewer than one, one and several, ragged last tiles and last runs."""
    run_bwd(pkg, oracle, gpu, (1, 2, 70, 128), (1, 2, Lkv, 128), seed=Lkv)


@pytest.mark.parametrize("L", [128, 999, 1024])
def test_bwd_self_attention_d128(pkg, oracle, gpu, L):
    run_bwd(pkg, oracle, gpu, (1, 2, L, 128), seed=L)


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_bwd_head_dims(pkg, oracle, gpu, d, dtype):
    run_bwd(pkg, oracle, gpu, (2, 2, 200, d), (2, 2, 333, d), seed=d, dtype=dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_bwd_head_dim_256(pkg, oracle, gpu, dtype):
    """Head dim 256 runs kernels of its own: ragged lengths, several stream tiles, causal, through autograd."""
    run_bwd(pkg, oracle, gpu, (1, 2, 150, 256), (1, 2, 77, 256), dtype=dtype, seed=1)
    run_bwd(pkg, oracle, gpu, (2, 1, 33, 256), (2, 1, 300, 256), dtype=dtype, seed=2)
    run_bwd(pkg, oracle, gpu, (1, 2, 200, 256), causal=True, dtype=dtype, seed=3)
    run_bwd(pkg, oracle, gpu, (1, 2, 1024, 256), dtype=dtype, seed=4, primal_std=0.5, sm_scale=0.5)
    q, k, v, tq, tk, tv = (x.to(gpu) for x in oracle.make_inputs((1, 2, 100, 256), seed=5, dtype=dtype))
    qg = q.clone().requires_grad_(True)
    o, to = pkg.attention_jvp(qg, k, v, tq, tk, tv)
    o.float().sum().backward()
    assert qg.grad is not None and torch.isfinite(qg.grad.float()).all()


@pytest.mark.parametrize("L", [1, 33, 128, 200, 515])
def test_bwd_causal(pkg, oracle, gpu, L):
    run_bwd(pkg, oracle, gpu, (1, 2, L, 64), causal=True, seed=L)


def test_bwd_causal_d128(pkg, oracle, gpu):
    run_bwd(pkg, oracle, gpu, (1, 2, 700, 128), causal=True, seed=4)


# the reference's own procedure: shapes, seed-independent distribution N(0, 0.5), sm_scale 0.5 (…jvp_triton.py:567-607, :717-762)
@pytest.mark.parametrize("shape", [(1, 2, 1024, 64), (1, 2, 999, 64)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_bwd_reference_shapes(pkg, oracle, gpu, shape, causal, dtype):
    run_bwd(pkg, oracle, gpu, shape, causal=causal, sm_scale=0.5, seed=20, dtype=dtype, primal_std=0.5)


@pytest.mark.parametrize("shape", [(1, 2, 256, 1024, 128), (1, 2, 1024, 256, 128), (1, 2, 1024, 512, 64), (1, 2, 1000, 515, 64)])
def test_bwd_reference_cross_attention_shapes(pkg, oracle, gpu, shape):
    Z, H, Lq, Lkv, d = shape
    run_bwd(pkg, oracle, gpu, (Z, H, Lq, d), (Z, H, Lkv, d), sm_scale=0.5, seed=20, primal_std=0.5)


def test_bwd_many_workgroups(pkg, oracle, gpu):
    run_bwd(pkg, oracle, gpu, (2, 4, 1024, 128), (2, 4, 1500, 128), seed=11)


@pytest.mark.parametrize("Lkv", [1, 33, 70, 160, 200, 515])
def test_bwd_several_query_blocks_per_workgroup(pkg, oracle, gpu, Lkv):
    """The kept-dS dQ pass with more query blocks (of 256) than compute units: its loads run 5 key tiles ahead over the ends of blocks.  One key tile,
    fewer than 5, 5 and more, ragged; the last block of a head has wavefronts with a whole, a partly filled and no query tile (same tolerances)."""
    run_bwd(pkg, oracle, gpu, (5, 13, 1070, 128), (5, 13, Lkv, 128), seed=Lkv)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Lq, Lkv, causal", [(15, 17, False), (16, 16, True), (17, 113, False), (48, 81, False), (113, 113, True), (145, 63, False)])
def test_bwd_at_the_edges_of_16(pkg, oracle, gpu, Lq, Lkv, causal, dtype):
    """The dK/dV kernel's results come in 16 queries x 16 keys: both on either side of a multiple, a query half and a key group without a row, the diagonal in each
    (same tolerances)."""
    run_bwd(pkg, oracle, gpu, (2, 3, Lq, 128), (2, 3, Lkv, 128), causal=causal, seed=Lq, dtype=dtype)


@pytest.mark.parametrize("Lkv", [4097, 6144, 6145, 8191])
@pytest.mark.parametrize("Lq", [1, 33, 230])
def test_bwd_workgroups_of_192_and_256_keys(pkg, oracle, gpu, Lkv, Lq):
    """Workgroups of 192 keys (8 heads, up to 6144 keys) and of 256 (more): one query tile, two, and more than the seven that LDS holds; last workgroups that are
    filled, that hold one key, and that lack one (same tolerances)."""
    run_bwd(pkg, oracle, gpu, (1, 8, Lq, 128), (1, 8, Lkv, 128), seed=Lq + Lkv, dtype=torch.float16 if Lq == 33 else torch.bfloat16)


@pytest.mark.parametrize("shape, keys, causal", [((2, 40, 700, 128), 700, True), ((1, 64, 760, 128), 760, True), ((1, 16, 20000, 128), 510, False), ((1, 16, 8000, 128), 192, False)])
@pytest.mark.parametrize("max_ds_mib", [None, -1])
def test_bwd_heads_of_larger_calls(pkg, oracle, gpu, shape, keys, causal, max_ds_mib):
    """Workgroups of 256, 192, 256 and 192 keys: the diagonal through them, and queries cut into ranges; dS kept and not.  The first, the last and one other head against the
    oracle (heads are independent; same tolerances)."""
    q, k, v, _, _, _ = oracle.make_inputs(shape, (*shape[:2], keys, 128), seed=9)
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(10)).to(torch.bfloat16)
    qd, kd, vd, dd = (x.to(gpu) for x in (q, k, v, dout))
    o, _, lse = pkg.attention_with_lse(qd, kd, vd, causal=causal)
    got = pkg.ops.bwd(qd, kd, vd, o, lse, dd, causal=causal, max_ds_mib=max_ds_mib)
    for h in (0, 7, shape[1] - 1):
        one = lambda x: x[-1:, h:h + 1]
        for name, a, ref in zip(("dq", "dk", "dv"), got, oracle.grads_closed_form(one(q), one(k), one(v), one(dout), causal=causal)):
            check(oracle, f"head {h} {name}", one(a), ref)


@pytest.mark.parametrize("Lq", [1, 32, 45, 300])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("which", ["q", "dout", "far"])
def test_bwd_query_rows_the_kernel_does_not_address(pkg, oracle, gpu, Lq, dtype, which):
    """Rows that lie less than a row's bytes apart (one row for all queries), or so far apart that a head's rows span 2 GiB, are copied first: the gradients are
    those of the same values in ordinary rows, byte for byte, and within the tolerances above."""
    q, k, v, _, _, _ = oracle.make_inputs((2, 3, Lq, 128), (2, 3, 70, 128), seed=Lq, dtype=dtype)
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(Lq)).to(dtype)
    if which == "q":
        q = q[:, :, :1].expand(q.shape)
    elif which == "dout":
        dout = dout[:, :, :1].expand(q.shape)
    qd, dd, kd, vd = q.to(gpu), dout.to(gpu), k.to(gpu), v.to(gpu)
    if which == "q":
        qd = qd[:, :, :1].expand(q.shape)
    elif which == "dout":
        dd = dd[:, :, :1].expand(q.shape)
    else:
        stride = max(2 ** 30 // (32 * ((Lq + 31) // 32)), 6 * 128)
        qd = torch.empty(Lq * stride, dtype=dtype, device=gpu).as_strided((2, 3, Lq, 128), (3 * 128, 128, stride, 1)).copy_(qd)
    o, _, lse = pkg.fwd_jvp(q.to(gpu).contiguous(), kd, vd)
    got = pkg.ops.bwd(qd, kd, vd, o, lse, dd)
    same = pkg.ops.bwd(qd.contiguous(), kd, vd, o, lse, dd.contiguous())
    for name, a, b, ref in zip(("dq", "dk", "dv"), got, same, oracle.grads_closed_form(q, k, v, dout)):
        assert torch.equal(a, b), name
        check(oracle, name, a, ref)


def test_bwd_through_autograd_function(pkg, oracle, gpu):
    """`attention(q, k, v, tq, tk, tv, causal, sm_scale)[0].backward(dout)` like the reference's procedure."""
    q, k, v, tq, tk, tv = oracle.make_inputs((1, 2, 300, 64), (1, 2, 300, 64), seed=3, primal_std=0.5)
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(7)).to(torch.bfloat16)
    dev = [x.to(gpu) for x in (q, k, v, tq, tk, tv)]
    for x in dev[:3]:
        x.requires_grad_(True)
    o, to = pkg.flash_attention_jvp.attention(*dev, True, 0.5)
    assert not to.requires_grad
    o.backward(dout.to(gpu))
    rq, rk, rv = oracle.grads_closed_form(q, k, v, dout, sm_scale=0.5, causal=True)
    check(oracle, "dq", dev[0].grad, rq)
    check(oracle, "dk", dev[1].grad, rk)
    check(oracle, "dv", dev[2].grad, rv)


def test_bwd_strided_inputs_and_determinism(pkg, oracle, gpu):
    """[B, S, H, D] storage passed as transposed views; two calls give bitwise identical results (no atomics)."""
    B, S, H, D = 2, 257, 3, 64
    g = torch.Generator().manual_seed(5)
    mk = lambda: (torch.randn((B, S, H, D), generator=g) * 0.7).to(torch.bfloat16)
    q, k, v, dout = mk(), mk(), mk(), mk()
    tr = lambda x: x.to(gpu).transpose(1, 2)
    o, _, lse = pkg.attention_with_lse(tr(q), tr(k), tr(v))
    a = pkg.ops.bwd(tr(q), tr(k), tr(v), o, lse, tr(dout))
    b = pkg.ops.bwd(tr(q), tr(k), tr(v), o, lse, tr(dout))
    torch.cuda.synchronize()
    for x, y in zip(a, b):
        assert torch.equal(x, y)
    rq, rk, rv = oracle.grads_closed_form(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), dout.transpose(1, 2))
    check(oracle, "dq", a[0], rq)
    check(oracle, "dk", a[1], rk)
    check(oracle, "dv", a[2], rv)


def test_bwd_config3_shape_sampled(pkg, oracle, gpu):
    """2B 720p shape (one head pair): gradients of sampled 128-row blocks against the fp32 oracle restricted to
    the rows / keys they depend on is not possible for dk, dv (they sum over all queries), so this checks dq on sampled
    query blocks and an invariant for dk, dv: sum_k dv = sum_q dout P summed over keys = sum_q dout  (rows of P sum to 1)."""
    B, H, L, d = 1, 2, 84480, 128
    g = torch.Generator(device=gpu).manual_seed(0)
    rn = lambda std: (torch.randn((B, H, L, d), generator=g, device=gpu) * std).to(torch.bfloat16)
    q, k, v, dout = rn(1.0), rn(1.0), rn(1.0), rn(1.0)
    o, _, lse = pkg.attention_with_lse(q, k, v)
    dq, dk, dv = pkg.ops.bwd(q, k, v, o, lse, dout)
    torch.cuda.synchronize()
    assert torch.isfinite(dq.float()).all() and torch.isfinite(dk.float()).all() and torch.isfinite(dv.float()).all()
    got = dv.float().sum(dim=2)
    want = dout.float().sum(dim=2)
    assert ((got - want).abs().max() / want.abs().max()).item() < 2e-2
    # dq rows depend on all keys but only on their own query row: oracle on sampled rows
    kc, vc = k.cpu().float(), v.cpu().float()
    for r0 in (0, 40000, L - 128):
        qs, ds = q[:, :, r0:r0 + 128].cpu().float(), dout[:, :, r0:r0 + 128].cpu().float()
        s = torch.einsum("bhqd,bhkd->bhqk", qs, kc) * d ** -0.5
        p = torch.softmax(s, dim=-1)
        osmp = torch.einsum("bhqk,bhkd->bhqd", p, vc)
        dp = torch.einsum("bhqd,bhkd->bhqk", ds, vc)
        dsm = p * (dp - (ds * osmp).sum(-1, keepdim=True))
        ref = torch.einsum("bhqk,bhkd->bhqd", dsm, kc) * d ** -0.5
        check(oracle, f"dq rows {r0}", dq[:, :, r0:r0 + 128], ref.double().numpy())


@pytest.mark.parametrize("chunk", range(2))
def test_bwd_random_shapes(pkg, oracle, gpu, chunk):
    """16 seeded random cases: batch, heads, lengths, head dim, dtype, causal drawn at random (workgroup counts on either
    side of the thresholds at which the last round is cut along the stream)."""
    import numpy as np

    rng = np.random.default_rng(2000 + chunk)
    for _ in range(8):
        B, H = int(rng.integers(1, 4)), int(rng.integers(1, 13))
        Lq, Lkv = int(rng.integers(1, 900)), int(rng.integers(1, 1200))
        d = int(rng.choice([16, 32, 64, 128]))
        causal = rng.random() < 0.2
        if causal:
            Lkv = Lq
        dtype = torch.float16 if rng.random() < 0.3 else torch.bfloat16
        run_bwd(pkg, oracle, gpu, (B, H, Lq, d), (B, H, Lkv, d), causal=causal, seed=int(rng.integers(0, 10000)), dtype=dtype)


def test_bwd_more_than_2_31_elements(pkg, oracle, gpu):
    """Offsets beyond 32 bits in the backward: tensors of 2.2e9 elements (B=4, H=128, L=32896, d=128) generated on the
    GPU; the last (batch, head) against the closed-form oracle restricted to that head (heads are independent)."""
    B, H, L, d = 4, 128, 32896, 128
    assert B * H * L * d > 2 ** 31
    g = torch.Generator(device=gpu).manual_seed(1)

    def rn():
        x = torch.empty(B, H, L, d, device=gpu, dtype=torch.bfloat16)
        for b in range(B):
            x[b] = torch.randn(H, L, d, generator=g, device=gpu).bfloat16()
        return x

    q, k, v, dout = rn(), rn(), rn(), rn()
    o, _, lse = pkg.fwd_jvp(q, k, v)
    dq, dk, dv = pkg.bwd(q, k, v, o, lse, dout)
    torch.cuda.synchronize()
    # fp64 closed form of one head at L = 32896 needs the L x L matrix (8.7 GB): check a row block of dq through the
    # row-independent part instead, and dk / dv through the adjoint identity against the forward-mode kernel's oracle
    for b, h in ((0, 0), (B - 1, H - 1)):
        qh, kh, vh, gh = (x[b, h].float() for x in (q, k, v, dout))
        rows = slice(L - 128, L)
        s = (qh[rows] @ kh.T) * d ** -0.5
        p = torch.softmax(s, dim=-1)
        dp = gh[rows] @ vh.T
        ds = p * (dp - (dp * p).sum(-1, keepdim=True))
        want_dq = (ds @ kh) * d ** -0.5
        check(oracle, f"dq rows of (b={b}, h={h})", dq[b, h, rows], want_dq.cpu())
        # dv = P^T dout, dk = dS^T q s for a block of 128 keys needs all query rows: do it in slabs on the GPU in fp32
        keys = slice(L - 128, L)
        want_dv = torch.zeros(128, d, device=gpu)
        want_dk = torch.zeros(128, d, device=gpu)
        lse_h = lse[b, h]
        for r0 in range(0, L, 4096):
            rr = slice(r0, min(r0 + 4096, L))
            s_blk = (qh[rr] @ kh[keys].T) * d ** -0.5
            p_blk = torch.exp(s_blk - lse_h[rr, None])
            dp_blk = gh[rr] @ vh[keys].T
            delta = (gh[rr] * o[b, h, rr].float()).sum(-1, keepdim=True)
            ds_blk = p_blk * (dp_blk - delta)
            want_dv += p_blk.T @ gh[rr]
            want_dk += (ds_blk.T @ qh[rr]) * d ** -0.5
        check(oracle, f"dv keys of (b={b}, h={h})", dv[b, h, keys], want_dv.cpu())
        check(oracle, f"dk keys of (b={b}, h={h})", dk[b, h, keys], want_dk.cpu())


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("shape", [((2, 5, 700, 128), None), ((1, 3, 333, 128), (1, 3, 517, 128)), ((1, 7, 1100, 128), (1, 7, 90, 128))])
def test_bwd_kept_ds_groups_of_heads_match_the_recomputing_path(pkg, oracle, gpu, shape, causal):
    """At head dim 128 the dK/dV kernel keeps its 16-bit dS tiles and dq comes from them in a second pass, heads served in groups
    that fit ``max_ds_mib``.  A budget of a few MiB forces several groups (with a smaller last one); a negative one the path
    that computes the scores twice.  All meet the oracle, agree with each other to rounding, and repeat bit for bit."""
    shape_q, shape_kv = shape
    if causal and shape_kv is not None:
        pytest.skip("causal needs equal lengths")
    q, k, v, _, _, _ = oracle.make_inputs(shape_q, shape_kv, seed=31)
    g = torch.Generator().manual_seed(32)
    dout = torch.randn(q.shape, generator=g).to(torch.bfloat16)
    qd, kd, vd, dd = (x.to(gpu) for x in (q, k, v, dout))
    o, _, lse = pkg.attention_with_lse(qd, kd, vd, causal=causal)
    want = oracle.grads_closed_form(q, k, v, dout, causal=causal)
    n_qt, n_kb = (q.shape[2] + 31) // 32, (k.shape[2] + 127) // 128
    head_mib = n_qt * 4 * n_kb * 2048 / 2 ** 20
    results = {}
    for name, budget in (("recompute", -1), ("groups of 2", max(1, int(2 * head_mib + 0.999))), ("one group", 1024)):
        print(f"  {name}: max_ds_mib={budget} (a head's dS: {head_mib:.2f} MiB)", flush=True)
        got = pkg.ops.bwd(qd, kd, vd, o, lse, dd, causal=causal, max_ds_mib=budget)
        again = pkg.ops.bwd(qd, kd, vd, o, lse, dd, causal=causal, max_ds_mib=budget)
        torch.cuda.synchronize()
        for nm, a, b, w in zip(("dq", "dk", "dv"), got, again, want):
            assert torch.equal(a, b), f"{name}: {nm} differs between two calls"
            check(oracle, f"{name} {nm}", a, w)
        results[name] = got
    # (the paths cut a thin last round of workgroups along the stream at different places, so their sums round differently:
    # equal to rounding, not bit for bit)
    for other in ("groups of 2", "one group"):
        for a, b in zip(results[other], results["recompute"]):
            assert (a.float() - b.float()).abs().max().item() <= 2e-2 * max(1.0, b.float().abs().max().item())
