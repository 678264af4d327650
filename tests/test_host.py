"""Host-side checks that need no GPU: the C-ABI library loads and exports what the header declares, descriptor
validation returns the documented status codes (validation happens before anything touches the device), and the
Python operators raise the same exception types as the reference for the same misuse."""
import ctypes
import math
import os
import random
import re
import struct

import msgpack
import pytest
import torch

import __graft_entry__ as entry

HEADER = os.path.join(entry.REPO_ROOT, "include", "cosmos_attn_hip.h")


def declared_symbols():
    text = open(HEADER).read()
    return re.findall(r"COSMOS_ATTN_API\s+[\w\s\*]+?\b(cosmos_(?:attn|norm|ln|gated|gelu)\w*)\s*\(", text)


def test_header_and_binding_agree(pkg):
    syms = declared_symbols()
    assert len(syms) >= 9
    assert sorted(syms) == sorted(pkg._lib.EXPORTS)


def test_library_exports_every_declared_symbol(pkg):
    lib = ctypes.CDLL(pkg._lib.LIB_PATH)
    for name in declared_symbols():
        assert hasattr(lib, name), name
    assert pkg._lib.load_library().cosmos_attn_abi_version() == pkg._lib.ABI_VERSION
    m = re.search(r"#define COSMOS_ATTN_ABI_VERSION (\d+)", open(HEADER).read())
    assert int(m.group(1)) == pkg._lib.ABI_VERSION


def test_desc_struct_layout_matches_header(pkg):
    # 10 x int32/float, 6 pointers, 9 int64, 2 pointers, 3 int64, 2 pointers
    assert ctypes.sizeof(pkg._lib.AttnDesc) == 40 + 6 * 8 + 9 * 8 + 2 * 8 + 3 * 8 + 2 * 8
    assert pkg._lib.AttnDesc.q.offset == 40 and pkg._lib.AttnDesc.key_lens.offset == 208


def good_desc(pkg, **over):
    D = pkg._lib.AttnDesc()
    D.abi_version, D.dtype = pkg._lib.ABI_VERSION, pkg._lib.DTYPE_BF16
    D.B, D.H, D.Lq, D.Lkv, D.d_qk, D.d_v, D.causal, D.sm_scale = 1, 2, 100, 70, 128, 64, 0, 0.1
    fake = 0x7F0000000000  # never dereferenced: validation only looks at values
    D.q, D.k, D.v, D.o = fake, fake + 4096, fake + 8192, fake + 12288
    D.tq = D.tk = D.tv = D.to = None
    for name, sl in (("q_stride", (2 * 100 * 128, 100 * 128, 128)), ("k_stride", (2 * 70 * 128, 70 * 128, 128)),
                     ("v_stride", (2 * 70 * 64, 70 * 64, 64)), ("o_stride", (2 * 100 * 64, 100 * 64, 64))):
        setattr(D, name, (ctypes.c_int64 * 3)(*sl))
    for key, val in over.items():
        setattr(D, key, val)
    return D


def test_status_codes_for_bad_descriptors(pkg):
    L, lib = pkg._lib, pkg._lib.load_library()
    ws = lambda D: lib.cosmos_attn_workspace_bytes(ctypes.byref(D))
    run = lambda D: lib.cosmos_attn_fwd_jvp(ctypes.byref(D), None, 0, None)
    D = good_desc(pkg)
    # forward only: tiles of 32 keys, K part 8 KB + V part (64 -> 2 row blocks) 4 KB
    assert ws(D) == 1 * 2 * 3 * (8 + 4) * 1024
    assert run(D) == L.ST_WORKSPACE          # valid descriptor, no workspace: refused before any launch
    fake = 0x7F0000100000
    assert ws(good_desc(pkg, tq=fake, tk=fake, tv=fake, to=fake)) == 1 * 2 * 3 * 2 * (8 + 4) * 1024
    cases = [
        (dict(abi_version=99), L.ST_BAD_ARG),
        (dict(Lq=0), L.ST_BAD_ARG),
        (dict(q=None), L.ST_BAD_ARG),
        (dict(tk=fake), L.ST_BAD_ARG),                 # tangent on k without q, v
        (dict(tq=fake), L.ST_BAD_ARG),                 # tangents given but no `to`
        (dict(dtype=7), L.ST_UNSUPPORTED),
        (dict(d_qk=512), L.ST_BAD_SHAPE),
        (dict(d_v=48), L.ST_BAD_SHAPE),
        (dict(causal=1), L.ST_BAD_SHAPE),              # causal needs Lq == Lkv
        (dict(q=0x7F0000000008), L.ST_BAD_STRIDE),     # 8-byte aligned base
        (dict(k_stride=(ctypes.c_int64 * 3)(70 * 132, 70 * 132, 132)), L.ST_BAD_STRIDE),
    ]
    for over, want in cases:
        D = good_desc(pkg, **over)
        assert ws(D) == 0, over
        assert run(D) == want, (over, run(D))
        assert lib.cosmos_attn_pack_kv(ctypes.byref(D), None, 0, None) == want
        assert lib.cosmos_attn_run(ctypes.byref(D), None, 0, None) == want
    for st in range(7):
        assert len(L.status_string(st)) > 0
    assert L.status_string(0) == "ok"


def plan_of(pkg, D, workspace_bytes=ctypes.c_size_t(-1).value):
    """(query rows, key groups, whole pairs, cut pairs, key ranges) of the launch; "streamed" where the query blocks are streamed."""
    plan = pkg._lib.AttnPlan()
    assert pkg._lib.load_library().cosmos_attn_launch_plan(ctypes.byref(D), workspace_bytes, ctypes.byref(plan)) == pkg._lib.ST_OK
    if plan.streaming_workgroups:
        return "streamed"
    return plan.query_rows, plan.key_groups, plan.whole_pairs, plan.cut_pairs, plan.key_ranges


def partial_result_bytes(plan, d_v, tangents):
    """What the key ranges of a plan leave: fp32 accumulators (two with tangents), then 16 bytes of statistics per row."""
    rows, _, _, cut, ranges = plan
    up = lambda n: (n + 255) // 256 * 256
    return 0 if ranges == 1 else up(cut * ranges * rows * d_v * (2 if tangents else 1) * 4) + up(cut * ranges * rows * 16)


@pytest.mark.parametrize("H,L,tangents,plan", [
    (16, 1560, True, (128, 1, 208, 0, 1)),      # 208 pairs in one round: a cut would only add partial results
    (16, 2600, True, (128, 1, 256, 80, 3)),     # 336 pairs: 80 of a second round, 3 ranges each
    (16, 7040, True, (128, 1, 768, 112, 2)),    # 880 pairs: 112 of a fourth round, 2 ranges each
    (2, 2048, True, (128, 1, 0, 32, 6)),        # 32 pairs, 64 steps: six ranges are as fast as the eight that fill the chip, with less to merge
    (16, 3520, False, (256, 1, 224, 0, 1)),     # forward only: 224 pairs of 256 rows in one round, of 384 rows 160
    (16, 2000, False, (128, 2, 256, 0, 1)),     # a whole round of pairs of 128 rows and 2 key groups
    (16, 37440, False, (384, 1, 1536, 32, 8)),  # 1568 pairs: 32 of a seventh round, 8 ranges each
    (4, 4623, False, (256, 1, 0, 76, 3)),       # 76 pairs, 73 steps
    (2, 1000, False, (128, 2, 0, 16, 4)),       # 16 pairs, 16 steps
    (1, 100, False, (128, 2, 1, 0, 1)),         # 2 steps: too short to cut
])
def test_key_range_plan(pkg, H, L, tangents, plan):
    """What workgroups a call is dealt out to, how many key ranges the pairs of a partly filled last round are cut into, and that the
    workspace asked for has room for their partial results and nothing else."""
    lib = pkg._lib.load_library()
    t = 0x8000000 if tangents else None
    D = good_desc(pkg, B=1, H=H, Lq=L, Lkv=L, d_v=128, tq=t, tk=t, tv=t, to=t)
    assert plan_of(pkg, D) == plan
    extra = lib.cosmos_attn_workspace_bytes(ctypes.byref(D)) - lib.cosmos_attn_packed_bytes(ctypes.byref(D))
    assert extra == partial_result_bytes(plan, 128, tangents)


@pytest.mark.parametrize("d,H,L,plan", [
    (16, 16, 700, (128, 2, 96, 0, 1)),          # forward only
    (16, 40, 1100, (256, 1, 200, 0, 1)),
    (32, 40, 9000, (384, 1, 768, 192, 4)),      # 960 pairs: 192 of a fourth round
    (32, 1, 4000, (128, 2, 0, 32, 8)),          # 32 pairs, 63 steps
    (64, 16, 5000, (384, 1, 224, 0, 1)),        # 224 pairs in one round
    (64, 16, 2660, (384, 1, 0, 112, 2)),        # 112 pairs in halves 52.1 us, 176 pairs of 256 rows 54.3
    (64, 40, 1100, (256, 1, 200, 0, 1)),        # 33.4 us; 120 pairs of 384 rows in halves 37.6
])
def test_key_range_plan_below_head_dim_128(pkg, d, H, L, plan):
    """As above, forward only: a step costs more than its share of matrix instructions there, so that more calls are worth cutting."""
    lib = pkg._lib.load_library()
    D = good_desc(pkg, B=1, H=H, Lq=L, Lkv=L, d_qk=d, d_v=d)
    assert plan_of(pkg, D) == plan
    extra = lib.cosmos_attn_workspace_bytes(ctypes.byref(D)) - lib.cosmos_attn_packed_bytes(ctypes.byref(D))
    assert extra == partial_result_bytes(plan, d, False)


@pytest.mark.parametrize("tangents", [False, True])
@pytest.mark.parametrize("d", [16, 32, 64, 128])
def test_workspace_holds_the_plan_that_runs_and_no_more(pkg, d, tangents):
    """Over sizes, every length of the query against every length of the keys: the bytes asked for are those of the plan that runs, that
    plan is still the one chosen where there is no more room than that, and without room no keys are cut."""
    lib = pkg._lib.load_library()
    t = 0x8000000 if tangents else None
    shapes = set()
    for H in (1, 5, 16, 40):
        for Lq in (1, 129, 226, 700, 993, 1560, 2000, 3520, 4623, 5000, 7040, 16100, 37440):
            for Lkv in (1, 226, 449, 513, 1000, 2049, 4000, 9000):
                D = good_desc(pkg, B=1, H=H, Lq=Lq, Lkv=Lkv, d_qk=d, d_v=d, tq=t, tk=t, tv=t, to=t)
                plan, packed = plan_of(pkg, D), lib.cosmos_attn_packed_bytes(ctypes.byref(D))
                bytes_ = lib.cosmos_attn_workspace_bytes(ctypes.byref(D))
                assert plan_of(pkg, D, bytes_) == plan, (H, Lq, Lkv)
                if plan == "streamed":      # (the size covers the launch that is not streamed as well)
                    continue
                assert bytes_ == packed + partial_result_bytes(plan, d, tangents), (H, Lq, Lkv)
                shapes.add(plan[:2])
                uncut = plan_of(pkg, D, packed)
                assert uncut == "streamed" or uncut[3:] == (0, 1), (H, Lq, Lkv)
    assert shapes == ({(128, 1)} if tangents else {(128, 2), (256, 1), (384, 1)})


def dense_desc(pkg, H, Lq, Lkv, tangents, **over):
    """bf16 at head dim 128, rows one behind the other; tangents None, "q" or "full"."""
    t = {None: (None, None), "q": (0x7F0000000000, None), "full": (0x7F0000000000, 0x7F0000000000)}[tangents]
    rows = lambda L: (ctypes.c_int64 * 3)(H * L * 128, L * 128, 128)
    return good_desc(pkg, H=H, Lq=Lq, Lkv=Lkv, d_v=128, tq=t[0], to=t[0], tk=t[1], tv=t[1], q_stride=rows(Lq), o_stride=rows(Lq), k_stride=rows(Lkv), v_stride=rows(Lkv), **over)


@pytest.mark.parametrize("H, L, tangents, rows", [(12, 6183, "full", 128), (20, 3328, "full", 128), (80, 6144, "q", 128), (40, 2953, "q", 128), (80, 4300, "q", 192), (80, 3557, "q", 192)])
def test_causal_calls_with_tangents_take_the_workgroups_that_end_first(pkg, H, L, tangents, rows):
    """(The other size was measured 9 to 27 % slower.)"""
    assert plan_of(pkg, dense_desc(pkg, H, L, L, tangents, causal=1))[0] == rows


@pytest.mark.parametrize("H, Lq, Lkv, tangents", [(16, 37440, 1600, "q"), (20, 11241, 1910, "q"), (16, 37440, 1024, "full"), (12, 24356, 886, "full")])
def test_padded_calls_are_streamed(pkg, H, Lq, Lkv, tangents):
    """A block of the other kernel costs as much beside its keys as sixteen tiles of them, and the host does not know how many are valid."""
    assert plan_of(pkg, dense_desc(pkg, H, Lq, Lkv, tangents, key_lens=0x7F0000000000)) == "streamed"
    assert plan_of(pkg, dense_desc(pkg, H, Lq, Lkv, tangents))[0] == 192


@pytest.mark.parametrize("tangents", [None, "q", "full"])
def test_forms_of_a_call_that_is_not_cut_take_the_same_kernel(pkg, tangents):
    """What runs without room for partial results (the two-stage run, the in-place call) is what the one-call form runs wherever that cuts no keys: the same results, bit for bit.
    Drawn sizes, and sizes where they parted."""
    lib, rng = pkg._lib.load_library(), random.Random(3)
    log = lambda lo, hi: int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    calls = [(40, 1741, 1741, None), (80, 807, 1623, None), (20, 1845, 1855, None), (16, 2197, 2197, "causal"), (8, 4277, 303, "lens")]
    while len(calls) < 6000:
        Lq, how = log(100, 12000), rng.choice([None, None, "causal", "lens"])
        calls.append((rng.choice([1, 2, 8, 12, 16, 20, 24, 32, 40, 64, 80]), Lq, Lq if how == "causal" or rng.random() < 0.5 else log(20, 5000), how))
    uncut = 0
    for H, Lq, Lkv, how in calls:
        D = dense_desc(pkg, H, Lq, Lkv, tangents, causal=int(how == "causal"), key_lens=0x7F0000000000 if how == "lens" else None)
        plan = plan_of(pkg, D)
        if plan != "streamed" and plan[4] > 1:
            continue
        uncut += 1
        assert plan_of(pkg, D, lib.cosmos_attn_packed_bytes(ctypes.byref(D))) == plan, (H, Lq, Lkv, how)
    assert uncut > 2000


@pytest.mark.parametrize("H, Lq, Lkv, how", [(16, 2197, 2197, "causal"), (16, 3000, 3000, "causal"), (64, 2196, 2196, "lens"), (40, 1129, 4403, "lens"), (80, 2411, 2411, None), (8, 345, 345, None)])
def test_calls_with_all_tangents_that_are_read_in_place(pkg, H, Lq, Lkv, how):
    if torch.cuda.is_available():
        pytest.skip("an accepted call would be launched")
    D = dense_desc(pkg, H, Lq, Lkv, "full", causal=int(how == "causal"), key_lens=0x7F0000000000 if how == "lens" else None)
    assert pkg._lib.load_library().cosmos_attn_fwd_in_place(ctypes.byref(D), None) not in (pkg._lib.ST_WORKSPACE, 0)
    assert plan_of(pkg, D)[0] == 128


def test_forward_override_steers_plan_and_workspace(pkg, forward_override, forward_plan):
    lib = pkg._lib.load_library()
    for rows, ranges in ((64, 0), (-128, 0), (129, 0), (0, -1)):
        assert lib.cosmos_attn_set_forward_override(rows, ranges) == pkg._lib.ST_BAD_ARG
    default = forward_plan((1, 3, 300, 128), 520)
    for rows, groups in ((128, 2), (256, 1), (384, 1)):
        pairs = (300 + rows - 1) // rows * 3
        for ranges, want in ((1, (pairs, 0, 1)), (2, (0, pairs, 2)), (9, (0, pairs, 2))):      # 9 steps of 64 keys: two ranges at most
            forward_override(rows, ranges)
            assert forward_plan((1, 3, 300, 128), 520) == (rows, groups, *want)
            D = good_desc(pkg, H=3, Lq=300, Lkv=520, d_v=128)
            extra = lib.cosmos_attn_workspace_bytes(ctypes.byref(D)) - lib.cosmos_attn_packed_bytes(ctypes.byref(D))
            assert extra == partial_result_bytes((rows, groups, *want), 128, False)
        assert forward_plan((1, 3, 300, 128), 300, causal=True) == (rows, groups, pairs, 0, 1)      # equal work only: never cut
        assert forward_plan((1, 3, 300, 128), 520, padded=True) == (rows, groups, pairs, 0, 1)
    forward_override()
    assert forward_plan((1, 3, 300, 128), 520) == default


@pytest.mark.parametrize("H, Lq, Lkv", [(16, 3520, 3520), (40, 1000, 3000), (3, 300, 520)])
def test_forward_override_for_tangents_leaves_other_calls_alone(pkg, forward_override, H, Lq, Lkv):
    other = [dense_desc(pkg, H, Lq, Lkv, None)] + [dense_desc(pkg, H, Lq, Lkv, t, dtype=pkg._lib.DTYPE_FP16) for t in ("q", "full")]
    want = [plan_of(pkg, D) for D in other]
    forward_override(192, 3)
    assert [plan_of(pkg, D) for D in other] == want
    plan = plan_of(pkg, dense_desc(pkg, H, Lq, Lkv, "full"))
    assert plan[0] == 192 and plan[4] == 3


def built_kernels(path):
    """name -> metadata of every kernel in the library's code objects (ELF images for AMDGPU, machine 224; an ELF note each, in msgpack)."""
    data, at, kernels = open(path, "rb").read(), 0, {}
    while (at := data.find(b"\x7fELF", at + 1)) >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] != 224:
            continue
        sections, (count,) = at + struct.unpack_from("<Q", data, at + 40)[0], struct.unpack_from("<H", data, at + 60)
        for header in range(sections, sections + 64 * count, 64):
            if struct.unpack_from("<I", data, header + 4)[0] != 7:      # SHT_NOTE
                continue
            note = at + struct.unpack_from("<Q", data, header + 24)[0]
            name_size, size, _ = struct.unpack_from("<III", data, note)
            body = note + 12 + (name_size + 3) // 4 * 4
            kernels.update((k[".name"], k) for k in msgpack.unpackb(data[body:body + size], strict_map_key=False)["amdhsa.kernels"])
    return kernels


def test_kernels_of_lone_wavefronts_keep_their_registers(pkg):
    """One wavefront per SIMD with up to 512 registers: what does not fit waits for memory in front of everything that is under way."""
    kernels = built_kernels(pkg._lib.LIB_PATH)
    for name, variants in (("attn_dkdv_kernel", 24), ("attn_jvp_rows_kernel", 2)):
        found = {k: v for k, v in kernels.items() if name in k}
        assert len(found) == variants
        assert not [k for k, v in found.items() if v[".private_segment_fixed_size"] or v[".vgpr_spill_count"] or v[".sgpr_spill_count"]]


def good_bwd_desc(pkg, **over):
    D = pkg._lib.AttnBwdDesc()
    D.abi_version, D.dtype = pkg._lib.ABI_VERSION, pkg._lib.DTYPE_BF16
    D.B, D.H, D.Lq, D.Lkv, D.d, D.causal, D.sm_scale, D.max_ds_mib = 1, 2, 100, 70, 64, 0, 0.1, 0
    fake = 0x7F0000000000  # never dereferenced: validation only looks at values
    for i, name in enumerate(("q", "k", "v", "o", "dout", "lse", "dq", "dk", "dv")):
        setattr(D, name, fake + 4096 * i)
    for name, L in (("q", 100), ("k", 70), ("v", 70), ("o", 100), ("dout", 100), ("dq", 100), ("dk", 70), ("dv", 70)):
        setattr(D, name + "_stride", (ctypes.c_int64 * 3)(2 * L * 64, L * 64, 64))
    for key, val in over.items():
        setattr(D, key, val)
    return D


@pytest.mark.parametrize("H, L", [(12, 2752), (20, 1550), (12, 9052)])
def test_causal_bwd_with_few_blocks_takes_the_small_ones(pkg, H, L):
    """Some 250 to 900 blocks of 128 keys, as many steps as the longest of them has on a unit alone: larger ones leave units idle (measured 8 to 12 % slower).  dS says which."""
    lib, rows = pkg._lib.load_library(), (ctypes.c_int64 * 3)(H * L * 128, L * 128, 128)
    D = good_bwd_desc(pkg, H=H, Lq=L, Lkv=L, d=128, causal=1, **{f"{name}_stride": rows for name in ("q", "k", "v", "o", "dout", "dq", "dk", "dv")})
    tiles, kept = (L + 31) // 32, lib.cosmos_attn_bwd_workspace_bytes(ctypes.byref(D))
    D.max_ds_mib = -1                                   # (without dS the key stream holds the rows of K and V as well: 16 KB a tile)
    ds = kept - (lib.cosmos_attn_bwd_workspace_bytes(ctypes.byref(D)) - H * tiles * 16 * 1024)
    assert ds == H * tiles * 4 * ((L + 127) // 128) * 2048


def test_bwd_desc_layout_and_status_codes(pkg):
    L, lib = pkg._lib, pkg._lib.load_library()
    # 10 x int32/float, 9 pointers, 8 x 3 int64
    assert ctypes.sizeof(L.AttnBwdDesc) == 40 + 9 * 8 + 8 * 3 * 8
    assert L.AttnBwdDesc.q.offset == 40 and L.AttnBwdDesc.dv_stride.offset == 40 + 9 * 8 + 7 * 3 * 8
    ws = lambda D: lib.cosmos_attn_bwd_workspace_bytes(ctypes.byref(D))
    run = lambda D: lib.cosmos_attn_bwd(ctypes.byref(D), None, 0, None)
    D = good_bwd_desc(pkg)
    # statistics (2 floats per query, rounded up to 1 KB) + query stream (4 tiles of 2*4 + 4*2 + 1 fragments)
    # + key stream (3 tiles of 2*4 + 2*2 fragments), per (b, h)
    assert ws(D) == 2048 + 2 * 4 * 17 * 1024 + 2 * 3 * 12 * 1024
    assert run(D) == L.ST_WORKSPACE
    cases = [
        (dict(abi_version=1), L.ST_BAD_ARG),
        (dict(Lkv=0), L.ST_BAD_ARG),
        (dict(lse=None), L.ST_BAD_ARG),
        (dict(dk=None), L.ST_BAD_ARG),
        (dict(dtype=5), L.ST_UNSUPPORTED),
        (dict(d=512), L.ST_BAD_SHAPE),
        (dict(d=48), L.ST_BAD_SHAPE),
        (dict(causal=1), L.ST_BAD_SHAPE),
        (dict(dout=0x7F0000000004), L.ST_BAD_STRIDE),
        (dict(dq_stride=(ctypes.c_int64 * 3)(100 * 66, 100 * 66, 66)), L.ST_BAD_STRIDE),
    ]
    for over, want in cases:
        D = good_bwd_desc(pkg, **over)
        assert ws(D) == 0, over
        assert run(D) == want, (over, run(D))


def test_backward_argument_checks_mirror_reference(pkg):
    q = torch.zeros(1, 2, 8, 64, dtype=torch.bfloat16)
    lse = torch.zeros(1, 2, 8)
    with pytest.raises(AssertionError, match="different headdim"):   # …jvp_triton.py:507-509
        pkg.bwd(q, q, q[..., :32], q, lse, q)
    with pytest.raises(RuntimeError, match="GPU"):                   # no CPU path, no fallback
        pkg.bwd(q, q, q, q, lse, q)
    with pytest.raises(AssertionError, match="Causal cross-attention"):
        pkg.bwd(q, q[:, :, :4], q[:, :, :4], q, lse, q, causal=True)


def test_norm_rope_desc_layout_and_status_codes(pkg):
    L, lib = pkg._lib, pkg._lib.load_library()
    # 8 x int32/float, 6 pointers, 2 x 3 int64
    assert ctypes.sizeof(L.NormRopeDesc) == 32 + 6 * 8 + 2 * 3 * 8
    assert L.NormRopeDesc.x.offset == 32 and L.NormRopeDesc.y_stride.offset == 32 + 6 * 8 + 3 * 8

    def desc(**over):
        D = L.NormRopeDesc()
        D.abi_version, D.dtype, D.B, D.S, D.H, D.D, D.eps = L.ABI_VERSION, L.DTYPE_BF16, 1, 4, 2, 64, 1e-6
        D.x, D.y = 0x7F0000000000, 0x7F0000100000   # never dereferenced: every case below is rejected on the host
        D.x_stride = D.y_stride = (ctypes.c_int64 * 3)(4 * 2 * 64, 2 * 64, 64)
        for k, v in over.items():
            setattr(D, k, v)
        return D

    cases = [
        (dict(abi_version=1), L.ST_BAD_ARG),
        (dict(S=0), L.ST_BAD_ARG),
        (dict(y=None), L.ST_BAD_ARG),
        (dict(tx=0x7F0000200000), L.ST_BAD_ARG),          # a tangent in without a tangent out
        (dict(eps=-1.0), L.ST_BAD_ARG),
        (dict(dtype=5), L.ST_UNSUPPORTED),
        (dict(dtype=5 | L.NORM_ROPE_WEIGHT_16), L.ST_UNSUPPORTED),
        (dict(reserved=7, weight=0x7F0000300004, D=48), L.ST_BAD_SHAPE),      # what the field holds is not looked at
        (dict(reserved=7, weight=0x7F0000300004, y_stride=(ctypes.c_int64 * 3)(4 * 2 * 66, 2 * 66, 66)), L.ST_BAD_STRIDE),
        (dict(dtype=L.DTYPE_FP16 | L.NORM_ROPE_WEIGHT_16, weight=0x7F0000300004), L.ST_BAD_STRIDE),      # a 16-bit weight: 8 bytes
        (dict(D=512), L.ST_BAD_SHAPE),
        (dict(D=48), L.ST_BAD_SHAPE),
        (dict(x=0x7F0000000004), L.ST_BAD_STRIDE),
        (dict(angles=0x7F0000300008), L.ST_BAD_STRIDE),
        (dict(y_stride=(ctypes.c_int64 * 3)(4 * 2 * 66, 2 * 66, 66)), L.ST_BAD_STRIDE),
    ]
    for over, want in cases:
        got = lib.cosmos_norm_rope(ctypes.byref(desc(**over)), None)
        assert got == want, (over, got)


def test_norm_rope_bwd_desc_layout_and_status_codes(pkg):
    L, lib = pkg._lib, pkg._lib.load_library()
    # 8 x int32/float, 6 pointers, 3 x 3 int64
    assert ctypes.sizeof(L.NormRopeBwdDesc) == 32 + 6 * 8 + 3 * 3 * 8
    assert L.NormRopeBwdDesc.x.offset == 32 and L.NormRopeBwdDesc.dx_stride.offset == 32 + 6 * 8 + 2 * 3 * 8

    def desc(**over):
        D = L.NormRopeBwdDesc()
        D.abi_version, D.dtype, D.B, D.S, D.H, D.D, D.eps = L.ABI_VERSION, L.DTYPE_BF16, 2, 100, 6, 64, 1e-6
        D.x, D.dy, D.dx, D.dweight = 0x7F0000000000, 0x7F0000100000, 0x7F0000200000, 0x7F0000300000   # never dereferenced
        D.x_stride = D.dy_stride = D.dx_stride = (ctypes.c_int64 * 3)(100 * 6 * 64, 6 * 64, 64)
        for k, v in over.items():
            setattr(D, k, v)
        return D

    ws = lambda D: lib.cosmos_norm_rope_bwd_workspace_bytes(ctypes.byref(D))
    run = lambda D: lib.cosmos_norm_rope_bwd(ctypes.byref(D), None, 0, None)
    # 2 x 100 positions x 2 groups of 4 heads = 400 thread groups, 32 per block (8 threads per row of 64) -> 13 blocks x 64 floats
    assert ws(desc()) == 13 * 64 * 4
    assert ws(desc(dweight=None)) == 0
    assert run(desc()) == L.ST_WORKSPACE
    for held in (1, 7, -1):      # what the reserved field holds is not looked at: the weight is fp32, and needs no more than its own alignment
        assert run(desc(reserved=held, weight=0x7F0000400004)) == L.ST_WORKSPACE, held
    assert run(desc(dtype=L.DTYPE_BF16 | L.NORM_ROPE_WEIGHT_16, weight=0x7F0000400008)) == L.ST_WORKSPACE
    cases = [
        (dict(abi_version=1), L.ST_BAD_ARG),
        (dict(dtype=L.DTYPE_BF16 | L.NORM_ROPE_WEIGHT_16, weight=0x7F0000400004), L.ST_BAD_STRIDE),
        (dict(H=0), L.ST_BAD_ARG),
        (dict(dy=None), L.ST_BAD_ARG),
        (dict(dtype=5), L.ST_UNSUPPORTED),
        (dict(D=512), L.ST_BAD_SHAPE),
        (dict(D=24), L.ST_BAD_SHAPE),
        (dict(dx=0x7F0000200008), L.ST_BAD_STRIDE),
        (dict(dy_stride=(ctypes.c_int64 * 3)(100 * 6 * 66, 6 * 66, 66)), L.ST_BAD_STRIDE),
    ]
    for over, want in cases:
        D = desc(**over)
        assert ws(D) == 0, over
        assert run(D) == want, (over, run(D))


def test_norm_rope_argument_checks(pkg):
    x = torch.zeros(1, 8, 2, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="GPU"):                   # no CPU path, no fallback
        pkg.norm_rope(x)
    with pytest.raises(AssertionError):
        pkg.norm_rope(x[0])
    with pytest.raises(AssertionError):
        pkg.norm_rope(x, weight=torch.ones(32))
    with pytest.raises(AssertionError, match="one angle per"):
        pkg.norm_rope(x, rope_emb=torch.zeros(4, 1, 1, 64))
    with pytest.raises(AssertionError):                              # head dim outside {16, 32, 64, 128, 256}
        pkg.norm_rope(torch.zeros(1, 8, 2, 48, dtype=torch.bfloat16))


def test_dit_attention_module_mirrors_reference_surface(pkg):
    """Constructor arguments, sub-module / parameter names (a reference state dict must load) and refusals."""
    m = pkg.Attention(64, None, n_heads=2, head_dim=16)
    assert m.is_selfattn and m.backend == "hip"
    # parameter names of cosmos_predict2/_src/predict2/networks/minimal_v4_dit.py:349-359 (te RMSNorm holds `weight`)
    assert sorted(m.state_dict()) == ["k_norm.weight", "k_proj.weight", "output_proj.weight", "q_norm.weight",
                                      "q_proj.weight", "v_proj.weight"]
    assert m.q_proj.weight.shape == (32, 64) and m.output_proj.weight.shape == (64, 32) and m.q_norm.weight.shape == (16,)
    c = pkg.Attention(64, 48, n_heads=2, head_dim=16)
    assert not c.is_selfattn and c.k_proj.weight.shape == (32, 48)
    m.init_weights()
    assert float(m.q_proj.weight.abs().max()) <= 3 / 8 + 1e-6 and torch.equal(m.q_norm.weight, torch.ones(16))
    for name in ("compute_qkv", "compute_attention", "forward", "set_context_parallel_group", "init_weights", "forward_jvp"):
        assert callable(getattr(m, name))
    with pytest.raises(AssertionError, match="Invalid backend"):
        pkg.Attention(64, backend="transformer_engine")
    assert isinstance(pkg.Attention(64, backend="minimal_a2a").attn_op, pkg.HipAttnOp)    # the reference's name for this op protocol
    assert pkg.Attention(64, use_wan_fp32_strategy=True).use_wan_fp32_strategy
    with pytest.raises(RuntimeError, match="GPU"):          # no CPU path
        with torch.no_grad():
            m.bfloat16()(torch.zeros(1, 4, 64, dtype=torch.bfloat16))


def test_block_elementwise_desc_layouts_and_status_codes(pkg):
    L, lib = pkg._lib, pkg._lib.load_library()
    assert ctypes.sizeof(L.LnModulateDesc) == 24 + 8 + 8 * 8 and L.LnModulateDesc.x.offset == 32
    assert ctypes.sizeof(L.GatedResidualDesc) == 16 + 8 + 8 * 8 and L.GatedResidualDesc.x.offset == 24
    assert ctypes.sizeof(L.GeluDesc) == 8 + 8 + 4 * 8 and L.GeluDesc.h.offset == 16
    P = 0x7F0000000000   # never dereferenced: every case below is rejected on the host

    def ln(**over):
        D = L.LnModulateDesc()
        D.abi_version, D.dtype, D.D, D.rows_per_group, D.eps, D.rows = L.ABI_VERSION, L.DTYPE_BF16, 256, 4, 1e-6, 16
        D.x, D.shift, D.scale, D.y = P, P + 0x10000, P + 0x20000, P + 0x30000
        for k, v in over.items():
            setattr(D, k, v)
        return D

    for over, want in [(dict(abi_version=1), L.ST_BAD_ARG), (dict(rows=0), L.ST_BAD_ARG), (dict(scale=None), L.ST_BAD_ARG),
                       (dict(tx=P + 0x40000), L.ST_BAD_ARG), (dict(tshift=P + 0x40000), L.ST_BAD_ARG), (dict(dtype=7), L.ST_UNSUPPORTED),
                       (dict(D=8200), L.ST_UNSUPPORTED), (dict(D=252), L.ST_BAD_SHAPE), (dict(rows_per_group=5), L.ST_BAD_SHAPE),
                       (dict(y=P + 0x30002), L.ST_BAD_STRIDE)]:
        assert lib.cosmos_ln_modulate(ctypes.byref(ln(**over)), None) == want, over

    def gr(**over):
        D = L.GatedResidualDesc()
        D.abi_version, D.dtype, D.D, D.rows_per_group, D.rows = L.ABI_VERSION, L.DTYPE_FP16, 64, 2, 8
        D.x, D.res, D.gate, D.out = P, P + 0x10000, P + 0x20000, P
        for k, v in over.items():
            setattr(D, k, v)
        return D

    for over, want in [(dict(abi_version=0), L.ST_BAD_ARG), (dict(gate=None), L.ST_BAD_ARG), (dict(tx=P + 0x40000), L.ST_BAD_ARG),
                       (dict(tgate=P + 0x40000), L.ST_BAD_ARG), (dict(dtype=3), L.ST_UNSUPPORTED), (dict(D=60), L.ST_BAD_SHAPE),
                       (dict(rows=7), L.ST_BAD_SHAPE), (dict(res=P + 8), L.ST_BAD_STRIDE)]:
        assert lib.cosmos_gated_residual(ctypes.byref(gr(**over)), None) == want, over

    def ge(**over):
        D = L.GeluDesc()
        D.abi_version, D.dtype, D.n, D.h, D.a = L.ABI_VERSION, L.DTYPE_BF16, 64, P, P
        for k, v in over.items():
            setattr(D, k, v)
        return D

    for over, want in [(dict(abi_version=0), L.ST_BAD_ARG), (dict(n=0), L.ST_BAD_ARG), (dict(th=P + 0x100), L.ST_BAD_ARG),
                       (dict(dtype=9), L.ST_UNSUPPORTED), (dict(n=12), L.ST_BAD_SHAPE), (dict(a=P + 4), L.ST_BAD_STRIDE)]:
        assert lib.cosmos_gelu(ctypes.byref(ge(**over)), None) == want, over
    with pytest.raises(RuntimeError, match="GPU"):       # no CPU path
        pkg.gelu(torch.zeros(8, dtype=torch.bfloat16))


def test_gated_residual_ln_modulate_desc_layout_and_status_codes(pkg):
    L, lib = pkg._lib, pkg._lib.load_library()
    assert ctypes.sizeof(L.GatedResidualLnModulateDesc) == 24 + 8 + 14 * 8 and L.GatedResidualLnModulateDesc.x.offset == 32
    P = 0x7F0000000000   # never dereferenced: every case below is rejected on the host
    for over, want in [(dict(abi_version=1), L.ST_BAD_ARG), (dict(rows=0), L.ST_BAD_ARG), (dict(gate=None), L.ST_BAD_ARG), (dict(out=None), L.ST_BAD_ARG),
                       (dict(eps=-1.0), L.ST_BAD_ARG), (dict(tx=P), L.ST_BAD_ARG), (dict(tx=P, tres=P, tout=P), L.ST_BAD_ARG), (dict(tgate=P), L.ST_BAD_ARG),
                       (dict(dtype=7), L.ST_UNSUPPORTED), (dict(D=8200), L.ST_UNSUPPORTED), (dict(D=252), L.ST_BAD_SHAPE),
                       (dict(rows_per_group=5), L.ST_BAD_SHAPE), (dict(res=P + 2), L.ST_BAD_STRIDE), (dict(out=P + 8), L.ST_BAD_STRIDE)]:
        d = L.GatedResidualLnModulateDesc()
        d.abi_version, d.dtype, d.D, d.rows_per_group, d.eps, d.rows = L.ABI_VERSION, L.DTYPE_BF16, 256, 4, 1e-6, 16
        d.x, d.res, d.gate, d.shift, d.scale, d.out, d.y = (P + 0x10000 * i for i in range(7))
        for k, v in over.items():
            setattr(d, k, v)
        assert lib.cosmos_gated_residual_ln_modulate(ctypes.byref(d), None) == want, over


@pytest.mark.parametrize("wrong", [dict(dtype=torch.int8), dict(dtype=torch.float32), dict(dtype=torch.float16), dict(device="meta")])
@pytest.mark.parametrize("which", ["y", "ty"])
def test_given_outputs_of_another_type_or_device_are_refused(pkg, monkeypatch, wrong, which):
    """A preallocated output is written as x's type on x's device: of a narrower type, the kernel would write past its end."""
    launched = []
    monkeypatch.setattr(pkg.ops, "_check_elementwise", lambda x: None)      # (nothing is launched: CPU tensors do)
    monkeypatch.setattr(pkg.ops, "_launch", lambda name, desc, device: launched.append(name))
    x, res, tx, tres = (torch.zeros(4, 16, dtype=torch.bfloat16) for _ in range(4))
    m = torch.zeros(2, 16, dtype=torch.bfloat16)
    good, bad = torch.empty_like(x), torch.empty(4, 16, **{"dtype": x.dtype, **wrong})
    out = {"y": good, "ty": good.clone(), which: bad}
    with pytest.raises(AssertionError):
        pkg.ops.gated_residual_ln_modulate(x, res, m, m, m, tx, tres, **out)
    with pytest.raises(AssertionError):
        pkg.ops.ln_modulate(x, m, m, tx, out=out["y"], tout=out["ty"])
    assert not launched
    out[which] = good.clone()
    pkg.ops.gated_residual_ln_modulate(x, res, m, m, m, tx, tres, **out)
    pkg.ops.ln_modulate(x, m, m, tx, out=out["y"], tout=out["ty"])
    assert launched == ["cosmos_gated_residual_ln_modulate", "cosmos_ln_modulate"]


def test_block_reverse_mode_desc_layouts_and_status_codes(pkg):
    L, lib = pkg._lib, pkg._lib.load_library()
    assert ctypes.sizeof(L.LnModulateBwdDesc) == 24 + 8 + 7 * 8 and L.LnModulateBwdDesc.x.offset == 32
    assert ctypes.sizeof(L.GatedResidualBwdDesc) == 16 + 8 + 5 * 8 and L.GatedResidualBwdDesc.dy.offset == 24
    P = 0x7F0000000000   # never dereferenced: every case below is rejected on the host

    def desc(cls, names, **over):
        D = cls()
        D.abi_version, D.dtype, D.D, D.rows_per_group, D.rows = L.ABI_VERSION, L.DTYPE_BF16, 256, 40, 80
        for i, n in enumerate(names):
            setattr(D, n, P + 0x10000 * i)
        for k, v in over.items():
            setattr(D, k, v)
        return D

    for fn, cls, names, vectors in (("cosmos_ln_modulate_bwd", L.LnModulateBwdDesc, ("x", "scale", "dy", "dskip", "dx", "dshift", "dscale"), 2),
                                    ("cosmos_gated_residual_bwd", L.GatedResidualBwdDesc, ("dy", "res", "gate", "dres", "dgate"), 1)):
        for over, want in [(dict(abi_version=1), L.ST_BAD_ARG), (dict(rows=0), L.ST_BAD_ARG), (dict(dy=None), L.ST_BAD_ARG),
                           (dict(dtype=7), L.ST_UNSUPPORTED), (dict(D=252), L.ST_BAD_SHAPE), (dict(rows_per_group=33), L.ST_BAD_SHAPE),
                           (dict(dy=P + 2), L.ST_BAD_STRIDE), ({}, L.ST_WORKSPACE)]:
            assert getattr(lib, fn)(ctypes.byref(desc(cls, names, **over)), None, 0, None) == want, (fn, over)
        need = getattr(lib, fn + "_workspace_bytes")
        assert need(ctypes.byref(desc(cls, names))) == 2 * 5 * vectors * 256 * 4            # two groups of five runs of eight rows
        assert need(ctypes.byref(desc(cls, names, rows_per_group=16))) == 0                # short groups are one run


def test_modulation_desc_layout_and_status_codes(pkg):
    L, lib = pkg._lib, pkg._lib.load_library()
    assert ctypes.sizeof(L.ModulationDesc) == 24 + 12 * 8 and L.ModulationDesc.emb.offset == 24 and L.ModulationDesc.out.offset == 24 + 10 * 8
    P = 0x7F0000000000   # never dereferenced: every case below is rejected on the host

    def desc(**over):
        D = L.ModulationDesc()
        D.abi_version, D.dtype, D.rows, D.K, D.hidden, D.D = L.ABI_VERSION, L.DTYPE_BF16, 5, 256, 64, 256
        D.emb, D.lora, D.out = P, P + 0x10000, P + 0x20000
        for i in range(3):
            D.w1[i], D.w2[i] = P + 0x30000, P + 0x40000
        for k, v in over.items():
            setattr(D, k, v)
        return D

    none3 = (ctypes.c_void_p * 3)(P, None, P)
    for over, want in [(dict(abi_version=1), L.ST_BAD_ARG), (dict(rows=0), L.ST_BAD_ARG), (dict(lora=None), L.ST_BAD_ARG), (dict(temb=P), L.ST_BAD_ARG),
                       (dict(w1=none3), L.ST_BAD_ARG), (dict(dtype=7), L.ST_UNSUPPORTED), (dict(K=40), L.ST_BAD_SHAPE), (dict(hidden=48), L.ST_BAD_SHAPE),
                       (dict(D=24), L.ST_BAD_SHAPE), (dict(emb=P + 2), L.ST_BAD_STRIDE), ({}, L.ST_WORKSPACE)]:
        assert lib.cosmos_ln_modulation(ctypes.byref(desc(**over)), None, 0, None) == want, over
    assert lib.cosmos_ln_modulation_workspace_bytes(ctypes.byref(desc())) == 3 * 5 * 64 * 2
    assert lib.cosmos_ln_modulation_workspace_bytes(ctypes.byref(desc(tout=P))) == 2 * 3 * 5 * 64 * 2


def test_dit_block_mirrors_reference_surface(pkg):
    m = pkg.Block(64, 48, 2, mlp_ratio=4.0, use_adaln_lora=True, adaln_lora_dim=8)
    names = sorted(m.state_dict())
    # parameter names of cosmos_predict2/_src/predict2/networks/minimal_v4_dit.py:1029-1082 (LayerNorms carry none)
    assert names == sorted(
        [f"{a}.{p}.weight" for a in ("self_attn", "cross_attn") for p in ("q_proj", "k_proj", "v_proj", "output_proj", "q_norm", "k_norm")]
        + ["mlp.layer1.weight", "mlp.layer2.weight"]
        + [f"adaln_modulation_{n}.{i}.weight" for n in ("self_attn", "cross_attn", "mlp") for i in (1, 2)])
    assert m.mlp.layer1.weight.shape == (256, 64) and m.adaln_modulation_mlp[2].weight.shape == (192, 8)
    assert m.cross_attn.k_proj.weight.shape == (64, 48) and m.self_attn.is_selfattn and not m.cross_attn.is_selfattn
    m.init_weights()
    assert float(m.adaln_modulation_mlp[2].weight.abs().max()) == 0.0       # the block starts as the identity
    plain = pkg.Block(64, 48, 2)
    assert sorted(k for k in plain.state_dict() if k.startswith("adaln")) == [f"adaln_modulation_{n}.1.weight" for n in ("cross_attn", "mlp", "self_attn")]
    for name in ("forward", "forward_jvp", "init_weights", "reset_parameters", "set_context_parallel_group"):
        assert callable(getattr(m, name))
    i2v = pkg.Block(64, 48, 2, image_context_dim=32)
    assert isinstance(i2v.cross_attn, pkg.I2VCrossAttention) and i2v.cross_attn.k_img.weight.shape == (64, 32)
    assert {"cross_attn.k_img.weight", "cross_attn.v_img.weight", "cross_attn.k_img_norm.weight"} <= set(i2v.state_dict())
    fp32 = pkg.Block(64, 48, 2, use_wan_fp32_strategy=True)
    assert fp32.use_wan_fp32_strategy and fp32.self_attn.use_wan_fp32_strategy and fp32.cross_attn.use_wan_fp32_strategy


def test_dit_network_mirrors_reference_surface(pkg):
    """State-dict names of the reference's network (minimal_v4_dit.py:1338-1432) and its host-side pieces, on the CPU."""
    import numpy as np
    from einops import rearrange

    net = pkg.MiniTrainDIT(max_img_h=16, max_img_w=16, max_frames=8, in_channels=3, out_channels=5, patch_spatial=2, patch_temporal=1,
                           model_channels=64, num_blocks=2, num_heads=2, crossattn_emb_channels=48, use_adaln_lora=True, adaln_lora_dim=8,
                           extra_per_block_abs_pos_emb=True, use_crossattn_projection=True, crossattn_proj_in_channels=40,
                           extra_image_context_dim=24)
    keys = set(net.state_dict())
    for k in ("x_embedder.proj.1.weight", "pos_embedder.seq", "pos_embedder.dim_spatial_range", "pos_embedder.dim_temporal_range",
              "extra_pos_embedder.pos_emb_h", "extra_pos_embedder.pos_emb_w", "extra_pos_embedder.pos_emb_t",
              "t_embedder.1.linear_1.weight", "t_embedder.1.linear_2.weight", "t_embedding_norm.weight",
              "blocks.0.self_attn.q_proj.weight", "blocks.1.cross_attn.k_img_norm.weight", "blocks.1.adaln_modulation_mlp.2.weight",
              "final_layer.linear.weight", "final_layer.adaln_modulation.1.weight", "final_layer.adaln_modulation.2.weight",
              "crossattn_proj.0.weight", "crossattn_proj.0.bias", "img_context_proj.0.weight", "img_context_proj.0.bias"):
        assert k in keys, k
    assert "t_embedder.1.linear_1.bias" not in keys                      # bias only without adaLN-LoRA (:755)
    assert net.x_embedder.proj[1].weight.shape == (64, (3 + 1) * 2 * 2 * 1)    # one more channel for the padding mask
    assert net.t_embedder[1].linear_2.weight.shape == (3 * 64, 64)
    assert net.final_layer.linear.weight.shape == (2 * 2 * 1 * 5, 64)
    assert net.blocks[0].cross_attn.k_img.weight.shape == (64, 64)       # image context is projected to model_channels first
    assert float(net.final_layer.adaln_modulation[2].weight.detach().abs().max()) == 0.0   # init_weights: modulation starts at zero
    plain = pkg.MiniTrainDIT(max_img_h=16, max_img_w=16, max_frames=8, in_channels=3, out_channels=3, patch_spatial=2, patch_temporal=1,
                             model_channels=64, num_blocks=1, num_heads=2, concat_padding_mask=False)
    assert "t_embedder.1.linear_1.bias" in plain.state_dict() and "final_layer.adaln_modulation.2.weight" not in plain.state_dict()
    for kw in (dict(n_dense_blocks=2), dict(natten_parameters={})):
        with pytest.raises(NotImplementedError):
            pkg.MiniTrainDIT(16, 16, 8, 3, 3, 2, 1, model_channels=64, num_blocks=1, num_heads=2, **kw)

    assert not net.is_context_parallel_enabled
    net.enable_context_parallel(None)
    assert net.is_context_parallel_enabled
    net.disable_context_parallel()
    assert not net.is_context_parallel_enabled
    with pytest.raises(NotImplementedError):
        net.fully_shard(None)

    # host-side pieces against einops with the reference's pattern strings / explicit numpy
    x = torch.randn(2, 4, 4, 6, 8)
    pe = pkg.PatchEmbed(2, 2, in_channels=4, out_channels=16)
    want = rearrange(x, "b c (t r) (h m) (w n) -> b t h w (c r m n)", r=2, m=2, n=2) @ pe.proj[1].weight.T
    assert torch.allclose(pe(x), want, atol=1e-6)
    y = torch.randn(2, 3, 4, 4, 2 * 2 * 1 * 5)
    assert torch.equal(net.unpatchify(y), rearrange(y, "B T H W (p1 p2 t C) -> B C (T t) (H p1) (W p2)", p1=2, p2=2, t=1))
    ts = torch.tensor([[0.5, 2.0], [7.0, 0.1]])
    ang = ts.numpy()[..., None].astype(np.float64) * 10000.0 ** (-np.arange(32) / 32)
    assert np.allclose(pkg.Timesteps(64)(ts).numpy(), np.concatenate([np.cos(ang), np.sin(ang)], -1), atol=1e-5)
    emb, lora = net.t_embedder(ts)
    assert emb.shape == (2, 2, 64) and lora.shape == (2, 2, 192) and torch.equal(emb, pkg.Timesteps(64)(ts))
    e = net.extra_pos_embedder(torch.zeros(2, 3, 4, 5, 64))
    raw = (net.extra_pos_embedder.pos_emb_t[:3, None, None] + net.extra_pos_embedder.pos_emb_h[None, :4, None]
           + net.extra_pos_embedder.pos_emb_w[None, None, :5]).detach().double().numpy()
    want = raw / (1e-6 + np.sqrt((raw ** 2).sum(-1, keepdims=True)) / 8.0)
    assert e.shape == (2, 3, 4, 5, 64) and np.allclose(e[1].detach().numpy(), want, atol=1e-5)
    pm = torch.zeros(2, 1, 4, 4)
    pm[:, :, :2] = 1
    xin = net._with_padding_mask(torch.zeros(2, 3, 2, 8, 8), pm)
    assert xin.shape == (2, 4, 2, 8, 8) and float(xin[:, 3, :, :4].min()) == 1.0 and float(xin[:, 3, :, 4:].max()) == 0.0


def test_rope_position_table_mirrors_reference(pkg, nr_oracle):
    """VideoRopePosition3DEmb (cosmos_predict2/_src/predict2/networks/minimal_v4_dit.py:534-661): layout, fps and NTK rules."""
    import numpy as np

    T, H, W, D = 3, 4, 5, 128
    pe = pkg.VideoRopePosition3DEmb(head_dim=D, len_h=8, len_w=8, len_t=8)
    assert sorted(pe.state_dict()) == ["dim_spatial_range", "dim_temporal_range", "seq"] and pe.seq_dim == 0
    x = torch.zeros(1, T, H, W, 16)
    e = pe(x, fps=torch.tensor([24.0]))
    assert e.shape == (T * H * W, 1, 1, D) and e.dtype == torch.float32
    # at the base frame rate the table is the plain 3-D one (the oracle's construction, pinned on its own)
    np.testing.assert_allclose(e.reshape(-1, D).numpy(), nr_oracle.rope_angles_3d(T, H, W, D), rtol=1e-6, atol=1e-6)
    # half the frame rate: the temporal angles double (frame index / fps * base_fps), the spatial ones stay
    e12 = pe(x, fps=torch.tensor([12.0])).reshape(T, H, W, D)
    e24 = e.reshape(T, H, W, D)
    dim_h = D // 6 * 2
    dim_t = D - 2 * dim_h
    assert torch.allclose(e12[..., : dim_t // 2], 2 * e24[..., : dim_t // 2]) and torch.equal(e12[..., dim_t // 2: D // 2], e24[..., dim_t // 2: D // 2])
    # image batch: no fps, one frame
    assert pe(torch.zeros(2, 1, H, W, 16)).shape == (H * W, 1, 1, D)
    with pytest.raises(AssertionError, match="T should be 1"):
        pe(x)
    with pytest.raises(AssertionError, match="exceed the maximum"):
        pe(torch.zeros(1, 1, 9, 2, 16))
    # NTK extrapolation: ratio r stretches the base to 10000 * r ** (dim / (dim - 2)) on that axis only
    pe2 = pkg.VideoRopePosition3DEmb(head_dim=D, len_h=8, len_w=8, len_t=8, h_extrapolation_ratio=2.0, enable_fps_modulation=False)
    e2 = pe2(x).reshape(T, H, W, D)
    j = 3                                   # some channel of the h block
    want = 2.0 / (10000.0 * 2.0 ** (dim_h / (dim_h - 2))) ** (2 * j / dim_h)     # position h = 2
    assert abs(float(e2[0, 2, 0, dim_t // 2 + j]) - want) < 1e-6 * want + 1e-9
    assert torch.equal(e2[..., dim_t // 2 + dim_h // 2: D // 2], e24[..., dim_t // 2 + dim_h // 2: D // 2])   # w block untouched
    assert torch.allclose(e2[..., : dim_t // 2], e24[..., : dim_t // 2])            # fps modulation off = base frame rate


def test_status_to_exception_mapping(pkg):
    L = pkg._lib
    L.raise_for_status(L.ST_OK)
    for st, exc in ((L.ST_BAD_SHAPE, AssertionError), (L.ST_BAD_STRIDE, AssertionError), (L.ST_UNSUPPORTED, NotImplementedError),
                    (L.ST_BAD_ARG, ValueError), (L.ST_WORKSPACE, RuntimeError), (L.ST_LAUNCH, RuntimeError)):
        with pytest.raises(exc):
            L.raise_for_status(st)


def test_python_argument_checks_mirror_reference(pkg):
    q = torch.zeros(1, 2, 8, 128, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="GPU"):          # no CPU path, no fallback
        pkg.fwd_jvp(q, q, q)
    with pytest.raises(AssertionError):                     # shape checks of _attention.forward (…jvp_triton.py:439-440)
        pkg.fwd_jvp(q, q[:, :1], q)
    with pytest.raises(AssertionError):
        pkg.fwd_jvp(q, q, q[:, :, :4])
    with pytest.raises(AssertionError):                     # head dim outside {16,32,64,128,256} (:444-445)
        pkg.fwd_jvp(q[..., :48], q[..., :48], q)
    with pytest.raises(RuntimeError, match="GPU"):          # 256 is built for the forward paths: the call gets as far as the device check
        pkg.fwd_jvp(torch.zeros(1, 1, 8, 256, dtype=torch.bfloat16), torch.zeros(1, 1, 8, 256, dtype=torch.bfloat16),
                    torch.zeros(1, 1, 8, 256, dtype=torch.bfloat16))
    with pytest.raises(AssertionError, match="Causal cross-attention"):   # :446
        pkg.fwd_jvp(q, q[:, :, :4], q[:, :, :4], causal=True)
    with pytest.raises(AssertionError):                     # tangent shape / stride must match the primal (:447-448)
        pkg.attention_jvp(q, q, q, q[:, :, :4], q, q)
    with pytest.raises(AssertionError):
        pkg.attention_jvp(q, q, q, q.transpose(1, 2).contiguous().transpose(1, 2), q, q)
    with pytest.raises(NotImplementedError):                # attention(): dtype not in the supported list (attention.py:107-108)
        pkg.attention_forward(q.transpose(1, 2), q.transpose(1, 2), q.transpose(1, 2), dtype=torch.float64)
    with pytest.raises(NotImplementedError):                # float32 is on the reference's list (SDPA, :145-148) but not built here
        pkg.attention_forward(q.transpose(1, 2), q.transpose(1, 2), q.transpose(1, 2), dtype=torch.float32)


def test_attn_op_refuses_multi_gpu_group(pkg):
    op = pkg.HipAttnOp()
    op.set_context_parallel_group(None, None, None)   # single GPU: accepted, as a2a_cp.py:189-193
    assert op.pg is None


def test_bench_refuses_more_than_one_gpu():
    import subprocess
    import sys

    r = subprocess.run([sys.executable, os.path.join(entry.REPO_ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert r.returncode != 0 and "one GPU" in r.stderr


def test_checkpoint_configuration_and_kept_attention_results_bookkeeping(pkg):
    """sac_config parsing (object, dict, enum-valued mode) and the record / replay contexts of attention results: state is
    per thread, restored on exit, and a recomputation that makes fewer attention calls than were recorded is an error."""
    import enum
    import threading
    from types import SimpleNamespace

    class Mode(enum.Enum):
        NONE = "none"
        BLOCK_WISE = "block_wise"

    every = pkg.dit_network._checkpoint_every
    assert every(None) == 0 and every(dict(mode="none")) == 0 and every(SimpleNamespace(mode=Mode.NONE, every_n_blocks=3)) == 0
    assert every(dict(mode="predict2_2b_720_aggressive")) == 1 and every(SimpleNamespace(mode=Mode.BLOCK_WISE, every_n_blocks=2)) == 2
    att = pkg.attention
    store = []
    with att.record_attention_results(store):
        assert att._kept.record is store
        seen = []
        t = threading.Thread(target=lambda: seen.append(att._kept.record))
        t.start(); t.join()
        assert seen == [None]                      # another thread does not record into this one's list
        with att.record_attention_results([]) as inner:
            assert att._kept.record is inner
        assert att._kept.record is store
    assert att._kept.record is None
    with att.replay_attention_results([]):
        assert att._kept.replay == []
    assert att._kept.replay is None
    with pytest.raises(AssertionError, match="fewer attention calls"):
        with att.replay_attention_results([("o", "lse")]):
            pass
    assert att._kept.replay is None


@pytest.mark.parametrize("first", [0, 1, 4, 8])
def test_dense16_copies_what_starts_off_16_bytes(pkg, first):
    """A contiguous slice of a larger buffer is contiguous wherever it starts; the elementwise kernels need it to start at 16 bytes."""
    buf = torch.arange(64, dtype=torch.float32).bfloat16()
    assert buf.data_ptr() % 16 == 0
    t = buf[first:first + 48].view(6, 8)
    got = pkg.ops._dense16(t)
    assert got.is_contiguous() and got.data_ptr() % 16 == 0 and torch.equal(got, t)
    assert (got is t) == (first % 8 == 0)
    assert torch.equal(pkg.ops._dense16(t.t()), t.t()) and pkg.ops._dense16(t.t()).is_contiguous()


@pytest.mark.parametrize("cols, depth", [(64, 64), (2048, 2048), (8192, 2048), (2048, 8192), (20480, 5120)])
@pytest.mark.parametrize("count", [1, 2, 3])
def test_rows_below_which_no_layer_asks_are_below_the_rule(pkg, cols, depth, count):
    """linear.linear does not ask cosmos_attn_gemm_preferred below these rows; its answer there is no."""
    from sys import modules
    L, lin = pkg._lib, modules[pkg.__name__ + ".linear"]
    D = L.GemmDesc()
    D.abi_version, D.dtype, D.count = L.ABI_VERSION, L.DTYPE_BF16, count
    for i in range(3):
        D.a[i] = D.b[i] = D.c[i] = 16
    for order, rows, c, d in ((L.GEMM_XWT, lin.FEWEST_ROWS - 1, cols, depth), (L.GEMM_XW, lin.FEWEST_ROWS_BACKWARD - 1, depth, cols),
                              (L.GEMM_XTX, cols, depth, lin.FEWEST_ROWS_BACKWARD - 1)):
        D.order, D.flags, D.rows, D.cols, D.depth = order, (L.GEMM_SUM if order == L.GEMM_XW else 0), rows, c, d
        D.lda, D.ldb, D.ldc = max(rows + -rows % 8 if order == L.GEMM_XTX else d, 256), max(d if order == L.GEMM_XWT else c, 256), c
        assert L.load_library().cosmos_attn_gemm_preferred(ctypes.byref(D)) == 0
    D.order, D.flags, D.rows, D.cols, D.depth, D.lda, D.ldb, D.ldc = L.GEMM_XWT, 0, lin.FEWEST_ROWS, 2048, 2048, 2048, 2048, 2048
    assert L.load_library().cosmos_attn_gemm_preferred(ctypes.byref(D)) == 1


@pytest.mark.parametrize("order, rows, cols, depth, own", [
    # y: the library's time here, us, and this one's, measured
    ("xwt", 10920, 2048, 8192, False),      # 279 / 305
    ("xwt", 12480, 2048, 8192, False),      # 289 / 328
    ("xwt", 4680, 2048, 2048, False),       # 35 / 41
    ("xwt", 28160, 2048, 2048, False),      # 170 / 186
    ("xwt", 1024, 1024, 4096, False),       # 19 / 29
    ("xwt", 37440, 2048, 2048, True),       # 285 / 233
    ("xwt", 17600, 2048, 8192, True),       # 594 / 485
    ("xwt", 10920, 8192, 2048, True),       # 305 / 263
    ("xwt", 3520, 2048, 2048, True),        # 29 / 27
    ("xw", 9360, 2048, 8192, False),        # 258 / 296
    ("xw", 4680, 2048, 8192, False),        # 130 / 142
    ("xw", 37440, 2048, 2048, True),        # 290 / 230
    ("xtx", 512, 512, 30000, False),        # 119 / 186
    ("xtx", 2048, 1024, 30000, False),      # 223 / 287
    ("xtx", 2048, 2048, 28160, False),      # 235 / 282
    ("xtx", 3072, 3072, 30000, False),      # 554 / 592
    ("xtx", 2048, 2048, 10920, True),       # 121 / 84
    ("xtx", 8192, 2048, 84480, True),
])
def test_products_are_preferred_where_they_are_the_faster_ones(pkg, order, rows, cols, depth, own):
    L = pkg._lib
    D = L.GemmDesc()
    D.abi_version, D.dtype, D.count, D.order = L.ABI_VERSION, L.DTYPE_BF16, 1, pkg.ops.GEMM_ORDERS[order]
    D.a[0] = D.b[0] = D.c[0] = 16
    D.rows, D.cols, D.depth, D.ldc = rows, cols, depth, cols
    D.lda, D.ldb = rows if order == "xtx" else depth, depth if order == "xwt" else cols
    assert L.load_library().cosmos_attn_gemm_preferred(ctypes.byref(D)) == own


def _by_address(t, lines, width, ld):
    """What a launch would read of t: its memory, and nothing else that belongs to it."""
    n = (lines - 1) * ld + width
    return torch.frombuffer(bytearray(ctypes.string_at(t.data_ptr(), n * t.element_size())), dtype=t.dtype).as_strided((lines, width), (ld, 1))


@pytest.fixture
def gemm_by_address(pkg, monkeypatch):
    """The layers' own products on the CPU, formed of what a launch would find at its operands' addresses; always preferred."""
    from torch.utils._python_dispatch import _disable_current_modes

    def launch(order, rows, cols, depth, lda, ldb, a, b, total=False, shape=0, lead=None):
        with _disable_current_modes():         # (no mode sees a launch)
            a = [_by_address(x, *((depth, rows) if order == "xtx" else (rows, depth)), lda) for x in a]
            b = [_by_address(y, *((cols, depth) if order == "xwt" else (depth, cols)), ldb) for y in b]
            out = [(x.t() if order == "xtx" else x) @ (y.t() if order == "xwt" else y) for x, y in zip(a, b)]
            out = [y.reshape(*(lead or (rows,)), cols) for y in ([sum(out)] if total else out)]
            return out[0] if total else out
    monkeypatch.setattr(pkg.ops, "launch_gemm", launch)
    monkeypatch.setattr(pkg.ops, "gemm_preferred", lambda *a, **kw: True)


def _layer_inputs(n=2, rows=6, depth=8, cols=16):
    g = torch.Generator().manual_seed(5)
    rn = lambda *s: torch.randn(*s, generator=g).bfloat16()
    return rn(rows, depth).requires_grad_(True), [torch.nn.Parameter(rn(cols, depth)) for _ in range(n)], [rn(rows, cols) for _ in range(n)], [rn(rows, cols) for _ in range(n)]


@pytest.mark.parametrize("cotangent", ["dual", "batched"])
def test_layer_gradients_of_cotangents_that_are_more_than_memory(pkg, gemm_by_address, cotangent):
    """A gradient that is a dual tensor keeps its tangent, one that is a batch is taken whole: as in nn.Linear's backward pass."""
    from sys import modules
    from torch.autograd import forward_ad as fwad
    linear_fn = modules[pkg.__name__ + ".linear"]._LinearFn
    x, w, dy, tdy = _layer_inputs()
    ys, wants = linear_fn.apply(None, x, *w), [torch.nn.functional.linear(x, v) for v in w]
    if cotangent == "dual":
        with fwad.dual_level():
            def grads(out):
                g = torch.autograd.grad(out, [x, *w], [fwad.make_dual(d, t) for d, t in zip(dy, tdy)])
                return [part for t in g for part in fwad.unpack_dual(t)]
            got, want = grads(ys), grads(wants)
    else:
        batch = [torch.stack([d, t]) for d, t in zip(dy, tdy)]
        got, want = (torch.autograd.grad(out, [x, *w], batch, is_grads_batched=True) for out in (ys, wants))
    for a, b in zip(got, want):
        assert a is not None and a.shape == b.shape
        assert (a.double() - b.double()).norm() <= 3 * 2e-3 * b.double().norm()      # (dx: the products' order and their roundings, three at most)


def test_layer_gradients_are_seen_by_a_mode_that_watches_operators(pkg, gemm_by_address):
    from sys import modules
    from torch.utils.flop_counter import FlopCounterMode
    linear_fn = modules[pkg.__name__ + ".linear"]._LinearFn
    x, w, dy, _ = _layer_inputs()
    ys = linear_fn.apply(None, x, *w)
    with FlopCounterMode(display=False) as counter:
        torch.autograd.grad(ys, [x, *w], dy)
    assert counter.get_total_flops() == 2 * 2 * 2 * 6 * 8 * 16        # per layer dx and dw


@pytest.mark.parametrize("frozen", ["weights", "input"])
def test_layer_keeps_only_what_its_gradients_need(pkg, gemm_by_address, frozen):
    """Frozen weights need no x, a frozen x no weights: written over between the passes, or freed, they change nothing (as for nn.Linear)."""
    from sys import modules
    linear_fn = modules[pkg.__name__ + ".linear"]._LinearFn
    x, w, dy, _ = _layer_inputs()
    for t in (w if frozen == "weights" else [x]):
        t.requires_grad_(False)
    saved = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: saved.append(t) or t, lambda t: t):
        ys = linear_fn.apply(None, x, *w)
    assert sum(t.numel() for t in saved) == (sum(v.numel() for v in w) if frozen == "weights" else x.numel())
    wrt = [x] if frozen == "weights" else w
    want = torch.autograd.grad(ys, wrt, dy, retain_graph=True)
    with torch.no_grad():
        for t in ([x] if frozen == "weights" else w):
            t.zero_()
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(ys, wrt, dy), want))


def test_layer_gradients_of_saved_tensors_that_come_back_in_another_layout(pkg, gemm_by_address):
    from sys import modules
    linear_fn = modules[pkg.__name__ + ".linear"]._LinearFn
    x, w, dy, _ = _layer_inputs()
    want = torch.autograd.grad(linear_fn.apply(None, x, *w), [x, *w], dy)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach().t().contiguous(), lambda t: t.t()):
        ys = linear_fn.apply(None, x, *w)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(ys, [x, *w], dy), want))


@pytest.mark.parametrize("what", ["rows", "columns", "dtype"])
def test_layer_gradients_of_saved_tensors_that_come_back_as_others_are_torch_s_errors(pkg, gemm_by_address, what):
    """Nothing is launched with the sizes of tensors that are not there."""
    from sys import modules
    linear_fn = modules[pkg.__name__ + ".linear"]._LinearFn
    x, w, dy, _ = _layer_inputs()
    other = {"rows": lambda t: t[:-1], "columns": lambda t: t[:, :-1], "dtype": lambda t: t.float()}[what]
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach(), other):
        ys = linear_fn.apply(None, x, *w)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(ys, [x, *w], dy)


def test_products_that_are_only_asked_for_if_preferred_are_not_refused(pkg, monkeypatch):
    """A column of rows is contiguous with any stride between its single elements: None, for the caller's own product, and no error."""
    monkeypatch.setattr(pkg.ops, "_check_elementwise", lambda x: None)      # (nothing is launched: CPU tensors do)
    x, w = torch.zeros(1, 2048, dtype=torch.bfloat16).t(), torch.zeros(64, 1, dtype=torch.bfloat16)
    assert x.is_contiguous() and x.stride(1) != 1
    for order, a, b in (("xwt", [x], [w]), ("xtx", [x], [x.float()]), ("xtx", [x, x[:1024]], [x, x])):
        assert pkg.ops.gemm(order, a, b, if_preferred=True) is None
        with pytest.raises(ValueError):
            pkg.ops.gemm(order, a, b)


@pytest.mark.parametrize("stride, status", [(0, "ST_WORKSPACE"), (64, "ST_WORKSPACE"), (120, "ST_WORKSPACE"), (128, None)])
def test_overlapping_rows_are_not_read_in_place(pkg, stride, status):
    L = pkg._lib
    desc = lambda s: pkg.ops._ATTN_DESC.pack(L.ABI_VERSION, L.DTYPE_BF16, 1, 2, 70, 40, 128, 128, 0, 0.1, 16, 16, 16, 0, 0, 0,
                                             70 * 256, 128, 256, 40 * 256, 40 * 128, 128, 40 * 256, 40 * 128, s, 16, 0, 70 * 256, 128, 256, 0, 0)
    if status is not None:
        assert L.load_library().cosmos_attn_fwd_in_place(desc(stride), None) == getattr(L, status)
    elif not torch.cuda.is_available():      # (accepted: nothing of these sizes is refused before the device is looked at)
        assert L.load_library().cosmos_attn_fwd_in_place(desc(stride), None) not in (L.ST_WORKSPACE, 0)
