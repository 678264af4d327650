// dK/dV kernel of the backward for head dim 128, four wavefront roles ("quad").  Included inside the anonymous namespace of
// attn_bwd_gfx950.hip (uses BwdParams, kRows, kBlock, kBwdThreads, kBwdSweepStagger and attn_common_gfx950.h).
//
// Same mathematics as attn_bwd_kernel<T, D, KIND_DKDV> (a workgroup owns 128 keys and streams 32-query tiles, there
// [Q | dO | dO^T | Q^T | LSE log2e, D]), other division of labour and a stream half the size.  There every MFMA takes a fresh 1 KB A fragment from LDS
// and the four wavefront pairs of a workgroup each read the whole stream tile: 1.13 KB of LDS operand per MFMA.  Here a group of
// four wavefronts serves 64 keys, so that every stream fragment feeds four MFMAs (of half the size), and each wavefront has one job:
//   S1  S = Q k^T for its 64 keys (K rows are register-resident B operands), U = P = exp2(S c - LSE') rounded to 16 bit,
//       handed over through LDS;
//   S2  dP = dO v^T (V rows register-resident), W = dS = U * (dP - D) rounded to 16 bit, handed over through LDS and,
//       when dS is kept, stored to memory;
//   O1  dV^T += dO^T U   (accumulators for 64 keys x 128 channels);
//   O2  dK^T += Q^T W.
// 32 MFMAs per wavefront and step for all four; the elementwise work is split between S1 and S2; 0.34 KB of LDS operand per
// MFMA.  Two such groups per workgroup (8 wavefronts, two per SIMD: one of S1 / S2 and one of O1 / O2).  W is formed from the
// ROUNDED P (the hand-over holds 16-bit values); the reference's kernel multiplies before rounding, the difference is one more
// relative rounding of 2^-9 (bf16) on dS.
//
// v_mfma_f32_16x16x32: less energy a product than 32x32x16, which this kernel is bound by, and a lane of S1 / S2 holds 8 queries of 4 keys instead of 16 of 2, so
// that it reads half the row statistics; the rows' -D start the sums of dP, which takes the subtraction out of S2 (with 16 x 16 results they are 8 registers).
// Lane (i = lane % 16, g = lane / 16) of an operand has the contraction's elements 8 g .. + 7 of row or column i; of a result column i and rows 4 g .. + 3.  A
// 32 x 64 tile of S or dP is [16 keys][query half]; its registers, both query halves of 16 keys, are as they are the B operand of dV^T and dK^T, with queries 4 g .. + 3
// and 16 + 4 g .. + 3 as elements 0 .. 3 and 4 .. 7, and the unit that is stored of dS.
// Backward, us, 32x32x16 / this / with -D in front / with fragments 4 instead of 2 groups ahead in the O roles, bf16, 16 heads: 24640 queries and keys 14000 / 13820 / 13720 / 13690, 10920
// 2830 / 2765 / 2738 / 2734, 3520 340 / 336 / 335 / 329, 37440 x 512 583 / 575 / 571 / 570.
//
// Pipeline, step s (tile = sweep position):   S1: MFMAs S(s+1) | U(s)      S2: MFMAs dP(s) | W(s-1)
//                                             O1: tile s-1                 O2: tile s-2
//
// One copy of the stream.  A part of a tile in LDS is 32 rows x 128 channels as 16-byte units (row r, chunk C of 8 channels).  S1 / S2
// read them as MFMA A operands with ds_read_b128 (lane = row); O1 / O2 need the transposed operands (lane = channel, 2 x 4 rows per
// lane) and get them from the SAME units with the transposing read ds_read_b64_tr_b16 (within 16 lanes, lane i passes the address
// of 8 bytes -- row i of a 16 x 4 matrix M of 16-bit values -- and receives M[i/4 + 4k][i%4], k = 0..3): no second, transposed copy
// of the tile in memory, in the fills or in LDS.  The unit (r, C) lies at
//     slot(r, C) = 64 (r/4) + 16 (C/4) + 4 (r%4) + (C%4 XOR quad_swizzle(r/4)), the swizzle 0, 2, 3, 1 for r/4 = 0 .. 3:
// the lanes that a ds_read_b128 serves together (0 .. 3, 12 .. 15 and 20 .. 27, or the rest of 32: rows of two chunks; with the swizzle 0, 2, 1, 3, right for 16 consecutive lanes,
// SQ_LDS_BANK_CONFLICT was 7 % of the cycles, the time the same within 0.3 %, now it is 0) and the 32 lanes of a transposing pass (two runs of 4 rows x 2 chunks, both
// 8-byte halves of each unit) touch 256 consecutive-bank bytes each, and a direct-to-LDS load of 64 units is four whole rows, so
// that the fills read Q and dO rows where they are (or in the copy that is made of rows which they cannot address).
// LDS: rings of the two stream parts (Q 7 deep: fetched three steps before S1 uses it, kept until O2 has used it three steps
// later; dO 5 deep), U and W hand-over (two stages each), statistics ring (6).  All fills are issued by the O wavefronts (five
// 1 KB loads per wavefront and step); one s_barrier per step.  The O wavefronts' LDS reads are written as asm (the compiler
// would put vmcnt(0) in front of the transposing-read builtin: it takes it for an access that may alias the fills in flight),
// with their own lgkmcnt waits, each tied to the registers it makes valid.

template <int D>
struct QuadCfg {
    static_assert(D == 128, "built for head dim 128");
    static constexpr int NQ = D / 32, NF = D / 16;            // 32- and 16-channel chunks
    static constexpr int KP_BYTES = NF * kFragBytes;          // Q part, dO part of a tile
    static constexpr int RQ = 7, RDO = 5, RST = 6;
    static constexpr int HO_BYTES = 4 * kFragBytes;           // hand-over of one group and stage: 64 keys x 32 queries, 16 bit
    static constexpr int Q_OFF = 0;
    static constexpr int DO_OFF = Q_OFF + RQ * KP_BYTES;
    static constexpr int U_OFF = DO_OFF + RDO * KP_BYTES;     // [2 stages][2 groups]
    static constexpr int W_OFF = U_OFF + 4 * HO_BYTES;
    static constexpr int ST_OFF = W_OFF + 4 * HO_BYTES;
    static constexpr int LDS_BYTES = ST_OFF + RST * kFragBytes;
    static constexpr int LOADS = 5;                           // per O wavefront and step: 4 rows twice of each part + the statistics
    static constexpr int IN_FLIGHT = 2 * LOADS;               // at the top of a step: all but the loads of the last two steps must have landed
};

typedef short quad_s16x4 __attribute__((ext_vector_type(4)));

template <typename T, int D, bool SPILL>
__global__ void __attribute__((amdgpu_flat_work_group_size(kBwdThreads, kBwdThreads), amdgpu_waves_per_eu(2, 2)))
attn_dkdv_quad_kernel(const BwdParams p) {
    typedef QuadCfg<D> C;
    typedef typename VecOf<T>::v8 V8;
    typedef typename VecOf<T>::v4 V4;
    constexpr int NQ = C::NQ, NF = C::NF, NG = 4;      // 32-channel chunks; 16-channel chunks = fragments of a part, (chunk f / 2, query half f % 2); groups of 16 keys
    constexpr int PD = 2;      // S roles: LDS operand fetches run this many fragments ahead of use (4: 0.6 % slower); 4 in the O roles, written out below
    constexpr int WAIT_FILLS = (C::IN_FLIGHT & 15) | ((C::IN_FLIGHT >> 4) << 14) | 0x0F70;

    const int bid = blockIdx.x;
    const bool partial = bid >= p.n_full && p.splits > 1;
    const int pair = partial ? p.n_full + (bid - p.n_full) / p.splits : bid;
    const int split = partial ? (bid - p.n_full) % p.splits : 0;
    const int blk = pair % p.n_blk, bhl = pair / p.n_blk, bh = p.bh0 + bhl, b = bh / p.H, h = bh % p.H;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool s_role = wave < 4;                 // waves 0..3: S1, S2 of group 0, S1, S2 of group 1; waves 4..7: O1, O2, O1, O2
    const bool second = (wave & 1) != 0;          // S2 / O2
    const int grp = (wave >> 1) & 1;
    const int ow = wave & 3;                      // O wavefronts: which quarter of each stream part this one copies
    const int l16 = lane & 15, g = lane >> 4;
    const int row0 = blk * kBlock + grp * 64;     // first key of this group
    const bool causal = p.causal != 0;

    int t_lo = 0, t_hi = p.n_tiles;
    if (causal) t_lo = (blk * kBlock) / kRows;    // query tiles before the block's first key see none of its keys
    if (partial) {
        t_lo = (int)((int64_t)split * p.n_tiles / p.splits);
        t_hi = (int)((int64_t)(split + 1) * p.n_tiles / p.splits);
    }
    const int n = t_hi > t_lo ? t_hi - t_lo : 0;
    const int n_sweep = n > 0 ? n : 1;
    const int shift = (((pair >> 3) & 31) * kBwdSweepStagger) % n_sweep;
    auto tile_at = [&](int u) { return __builtin_amdgcn_readfirstlane(t_lo + (u + shift) % n_sweep); };
    auto wrap_inc = [&](int t) { ++t; return t >= t_lo + n_sweep ? t - n_sweep : t; };

    auto rows_of = [&](const QuadRows& r) {   // a head's rows; behind the last one zeros are read
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(r.ptr) + (int64_t)b * r.sb + (int64_t)h * r.sh, 0, (p.L_stream - 1) * r.row + 2 * D, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rsrc_q = rows_of(p.rows_q), rsrc_do = rows_of(p.rows_do);
    const __amdgpu_buffer_rsrc_t rsrc_st = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(p.stream) + (size_t)bh * p.n_tiles * kQuadStatBytes, 0, p.n_tiles * kQuadStatBytes, 0x00020000);
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    auto frag = [&](const char* base, int f) { return *reinterpret_cast<const V8*>(base + f * kFragBytes + lane * 16); };
    // A fragment f of a stream part (lane = row 16 (f % 2) + l16, channels 32 (f / 2) + 8 g .. + 7)
    const int a_off = 16 * quad_unit_slot(l16, g);
    auto afrag = [&](const char* part, int f) { return *reinterpret_cast<const V8*>(part + 4096 * (f & 1) + 256 * (f >> 1) + a_off); };

    // ---- fills (O wavefronts): this wavefront's eight rows 8 ow .. + 7 of a part of tile t into ring slot u, four rows a load
    int off_q[2], off_do[2];                      // what this lane reads of them
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = 8 * ow + 4 * i + ((lane >> 2) & 3), unit = 4 * (lane >> 4) + ((lane & 3) ^ quad_swizzle(2 * ow + i));
        off_q[i] = r * p.rows_q.row + 16 * unit;
        off_do[i] = r * p.rows_do.row + 16 * unit;
    }
    auto fill_part = [&](__amdgpu_buffer_rsrc_t rsrc, const int* off, int row, int part, int t) {
        char* dst = smem + part + 2 * ow * kFragBytes;
        lds_load<0>(rsrc, dst, off[0] + t * (kRows * row), 0);
        lds_load<0>(rsrc, dst + kFragBytes, off[1] + t * (kRows * row), 0);
    };
    auto fill_q = [&](int t, int u) {
        fill_part(rsrc_q, off_q, p.rows_q.row, C::Q_OFF + (u % C::RQ) * C::KP_BYTES, t);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_st, (__attribute__((address_space(3))) void*)(smem + C::ST_OFF + (u % C::RST) * kFragBytes), 4, lane * 4,
                                                 t * kQuadStatBytes, 0, 0);
    };
    auto fill_do = [&](int t, int u) { fill_part(rsrc_do, off_do, p.rows_do.row, C::DO_OFF + (u % C::RDO) * C::KP_BYTES, t); };
    if (!s_role) {   // what the steps before step 0 would have issued
        fill_q(tile_at(0), 0);
#pragma unroll
        for (int u = 0; u < 3; ++u) { fill_do(tile_at(u), u); fill_q(tile_at(u + 1), u + 1); }
    }

    const unsigned u_base = C::U_OFF + grp * C::HO_BYTES, w_base = C::W_OFF + grp * C::HO_BYTES;   // + stage * 2 * HO_BYTES

    if (s_role) {
        // ------------------------------------------------------------------------------------------ S1 / S2
        V8 breg[NG][NQ];            // stationary rows as B operands: K (S1) or V (S2) of keys row0 + 16 kg + l16
        {
            const void* st = second ? p.st2 : p.st1;
            const int64_t sb = second ? p.s2_sb : p.s1_sb, sh = second ? p.s2_sh : p.s1_sh, sl = second ? p.s2_sl : p.s1_sl;
#pragma unroll
            for (int kg = 0; kg < NG; ++kg) {
                const int row = row0 + 16 * kg + l16;
                const T* ptr = reinterpret_cast<const T*>(st) + (int64_t)b * sb + (int64_t)h * sh + (int64_t)row * sl + 8 * g;
                const bool live = row < p.L_stat;
#pragma unroll
                for (int c = 0; c < NQ; ++c) {
                    const V8 z = {0, 0, 0, 0, 0, 0, 0, 0};
                    breg[kg][c] = live ? *reinterpret_cast<const V8*>(ptr + 32 * c) : z;
                }
            }
        }
        // S (S1) or dP (S2) of two tiles, swapping roles every step: [16 keys][query half], register r: key 16 kg + l16, query 16 m + 4 g + r
        f32x4 x0[NG][2], x1[NG][2];
        typedef f32x4 (*tile_t)[2];
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        // the 8 values of this lane's queries
        auto load_rows = [&](const char* stats, float* v) {
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const float4 a = *reinterpret_cast<const float4*>(stats + 16 * g + 64 * m);
                v[4 * m] = a.x; v[4 * m + 1] = a.y; v[4 * m + 2] = a.z; v[4 * m + 3] = a.w;
            }
        };
        __builtin_amdgcn_s_waitcnt(0x0F70);   // the stationary rows are here
        __builtin_amdgcn_s_barrier();         // ... and so are the first stream tiles
        asm volatile("" ::: "memory");

        if (!second) {
            // ---------------------------------------------------------------- S1
            // causal: key (stationary) > query (streamed) possible iff last key of the group > first query of the tile
            auto need_mask = [&](int t) { return causal && row0 + 63 > t * kRows; };
            auto mask = [&](tile_t x, int t) {
#pragma unroll
                for (int kg = 0; kg < NG; ++kg) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const int qrow = t * kRows + 16 * (e >> 2) + 4 * g + (e & 3);
                        x[kg][e >> 2][e & 3] = (row0 + 16 * kg + l16 <= qrow) ? x[kg][e >> 2][e & 3] : -INFINITY;
                    }
                }
            };
            // scores of the first tile
#pragma unroll
            for (int kg = 0; kg < NG; ++kg) x0[kg][0] = x0[kg][1] = zero;
            if (n > 0) {
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    const V8 fa = afrag(smem + C::Q_OFF, f);
#pragma unroll
                    for (int kg = 0; kg < NG; ++kg) x0[kg][f & 1] = mfma16(fa, breg[kg][f >> 1], x0[kg][f & 1]);
                }
                if (need_mask(tile_at(0))) mask(x0, tile_at(0));
            }
            int t_next = tile_at(1);      // tile whose scores the step computes
            // one step: MFMAs of S(s+1) into xn (if NEXT) interleaved with U(s) from x (if CUR)
            float l2v[8];
            auto step = [&](auto NEXT, auto CUR, tile_t x, tile_t xn, int s) {
                constexpr bool next = decltype(NEXT)::value, cur = decltype(CUR)::value;
                const char* qpart = smem + C::Q_OFF + ((s + 1) % C::RQ) * C::KP_BYTES;
                V8 uf[NG];
                V8 fa[NF];
                if (next) {
#pragma unroll
                    for (int i = 0; i < PD; ++i) fa[i] = afrag(qpart, i);
                }
                if (cur) load_rows(smem + C::ST_OFF + (s % C::RST) * kFragBytes, l2v);
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    SCHED_FENCE();
                    if (next && f + PD < NF) fa[f + PD] = afrag(qpart, f + PD);
                    SCHED_FENCE();
#pragma unroll
                    for (int kg = 0; kg < NG; ++kg) {
                        if (next) xn[kg][f & 1] = mfma16(fa[f], breg[kg][f >> 1], f < 2 ? zero : xn[kg][f & 1]);
                        if (cur) {   // an element of these 16 keys behind each MFMA
                            const float pe = __builtin_amdgcn_exp2f(__builtin_fmaf(x[kg][f >> 2][f & 3], p.scale_log2, -l2v[f]));
                            uf[kg][f] = (T)pe;
                        }
                        SCHED_FENCE();
                    }
                }
                if (cur) {
                    const unsigned ua = lds0 + u_base + (s & 1) * 2 * C::HO_BYTES + 16 * lane;
                    asm volatile("ds_write_b128 %0, %1" ::"v"(ua), "v"(uf[0]) : "memory");
                    asm volatile("ds_write_b128 %0, %1 offset:1024" ::"v"(ua), "v"(uf[1]) : "memory");
                    asm volatile("ds_write_b128 %0, %1 offset:2048" ::"v"(ua), "v"(uf[2]) : "memory");
                    asm volatile("ds_write_b128 %0, %1 offset:3072" ::"v"(ua), "v"(uf[3]) : "memory");
                }
            };
            auto body = [&](int s, tile_t cur, tile_t nxt) {
                __builtin_amdgcn_s_waitcnt(0xC07F);   // own hand-over stores of the step before are done
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                if (s + 1 < n) {
                    step(std::true_type(), std::true_type(), cur, nxt, s);
                    if (need_mask(t_next)) mask(nxt, t_next);
                } else if (s < n) {
                    step(std::false_type(), std::true_type(), cur, nxt, s);
                }
                t_next = wrap_inc(t_next);
            };
            for (int s = 0; s <= n + 1; s += 2) {
                body(s, x0, x1);
                if (s + 1 <= n + 1) body(s + 1, x1, x0);
            }
        } else {
            // ---------------------------------------------------------------- S2
            // Inside a 2 KB tile the 16-byte unit (key, g) sits at slot 16 (key / 4) + 4 g + key % 4: the order in which the transposing
            // reads of attn_dq_from_ds_kernel touch 256 consecutive bytes per pass (no bank conflicts).  A store is 1 KB in a row.
            char* const ds_lane = SPILL ? p.ds + (int64_t)bhl * p.ds_head_bytes + ((int64_t)(4 * blk + 2 * grp) * 2 * kFragBytes + 16 * (16 * (l16 >> 2) + 4 * g + (l16 & 3))) : nullptr;
            const int64_t ds_row = (int64_t)p.n_kt_pad * 2 * kFragBytes;
            int t_prev = tile_at(0);      // tile whose W the step forms (sweep position s - 1)
            // one step: MFMAs of dP(s) - D into xc (if CUR) interleaved with W(s-1) = U(s-1) * (dP(s-1) - D) from xp (if PREV).  -D are the sums' first terms:
            // no subtraction per element, whose rows D has.
            auto step = [&](auto CUR, auto PREV, tile_t xc, tile_t xp, int s) {
                constexpr bool cur = decltype(CUR)::value, prev = decltype(PREV)::value;
                const char* dopart = smem + C::DO_OFF + (s % C::RDO) * C::KP_BYTES;
                const char* uin = smem + u_base + ((s + 1) & 1) * 2 * C::HO_BYTES;
                V8 ui[NG], wf[NG];
                V8 fb[NF];
                if (prev) {
#pragma unroll
                    for (int kg = 0; kg < NG; ++kg) ui[kg] = frag(uin, kg);
                }
                f32x4 minus_d[2];
                if (cur) {
#pragma unroll
                    for (int m = 0; m < 2; ++m) minus_d[m] = *reinterpret_cast<const f32x4*>(smem + C::ST_OFF + (s % C::RST) * kFragBytes + 128 + 16 * g + 64 * m);
#pragma unroll
                    for (int i = 0; i < PD; ++i) fb[i] = afrag(dopart, i);
                }
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    SCHED_FENCE();
                    if (cur && f + PD < NF) fb[f + PD] = afrag(dopart, f + PD);
                    SCHED_FENCE();
#pragma unroll
                    for (int kg = 0; kg < NG; ++kg) {
                        if (cur) xc[kg][f & 1] = mfma16(fb[f], breg[kg][f >> 1], f < 2 ? minus_d[f] : xc[kg][f & 1]);
                        if (prev) {
                            const float we = (float)ui[kg][f] * xp[kg][f >> 2][f & 3];
                            wf[kg][f] = (T)we;
                        }
                        SCHED_FENCE();
                    }
                }
                if (prev) {
                    const unsigned wa = lds0 + w_base + ((s + 1) & 1) * 2 * C::HO_BYTES + 16 * lane;
                    asm volatile("ds_write_b128 %0, %1" ::"v"(wa), "v"(wf[0]) : "memory");
                    asm volatile("ds_write_b128 %0, %1 offset:1024" ::"v"(wa), "v"(wf[1]) : "memory");
                    asm volatile("ds_write_b128 %0, %1 offset:2048" ::"v"(wa), "v"(wf[2]) : "memory");
                    asm volatile("ds_write_b128 %0, %1 offset:3072" ::"v"(wa), "v"(wf[3]) : "memory");
                    if (SPILL) {   // the two 32-key tiles of dS of this group, [stream tile][4 blk + 2 grp + kg / 2]: 16 keys a store
                        char* dst = ds_lane + t_prev * ds_row;
#pragma unroll
                        for (int kg = 0; kg < NG; ++kg) __builtin_nontemporal_store(wf[kg], reinterpret_cast<V8*>(dst + kg * kFragBytes));
                    }
                }
            };
            auto body = [&](int s, tile_t cur, tile_t prv) {
                __builtin_amdgcn_s_waitcnt(0xC07F);
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                if (s >= 1 && s < n) step(std::true_type(), std::true_type(), cur, prv, s);
                else if (s < n) step(std::true_type(), std::false_type(), cur, prv, s);
                else if (s >= 1 && s == n) step(std::false_type(), std::true_type(), cur, prv, s);
                if (s >= 1 && s <= n) t_prev = wrap_inc(t_prev);
            };
            for (int s = 0; s <= n + 1; s += 2) {
                body(s, x0, x1);
                if (s + 1 <= n + 1) body(s + 1, x1, x0);
            }
        }
        __builtin_amdgcn_s_waitcnt(0x0070);
    } else {
        // ------------------------------------------------------------------------------------------ O1 / O2
        f32x4 acc[NG][NF];          // dV^T (O1) or dK^T (O2): [16 keys][16 channels], register r: key 16 kg + l16, channel 16 f + 4 g + r
#pragma unroll
        for (int kg = 0; kg < NG; ++kg) {
#pragma unroll
            for (int f = 0; f < NF; ++f) acc[kg][f] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        int t_do = tile_at(3), t_q = tile_at(4);
        const int lag = second ? 2 : 1;                       // O1 accumulates tile s-1, O2 tile s-2
        // Transposing reads.  Lane (g, l16) of the MFMA A operand f is channel 16 f + l16 and queries 4 g .. + 3 (read t = 0), 16 + 4 g .. + 3
        // (t = 1); as a supplier of addresses it passes the 8 bytes of row 16 t + 4 g + l16/4, channels 16 f + 4 (l16%4) .. + 3: unit
        // (row, C = 2 f + (l16%4)/2), its second half when l16 is odd.  Byte offset in the part = 4096 t + 256 (f / 2) + tr_off[f % 2].
        unsigned tr_off[2];
#pragma unroll
        for (int o = 0; o < 2; ++o) tr_off[o] = (unsigned)(16 * quad_unit_slot(4 * g + (l16 >> 2), 2 * o + ((l16 & 3) >> 1)) + 8 * (l16 & 1));
// one MFMA group's A operand: fragment f = two transposing reads (t = 0, 1)
#define QUAD_TR_PAIR(f) asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%3\n\tds_read_b64_tr_b16 %1, %2 offset:%4" \
                                     : "=&v"(lo[f]), "=&v"(hi[f]) : "v"((f) & 1 ? ta1 : ta0), "n"(256 * ((f) / 2)), "n"(256 * ((f) / 2) + 4096) : "memory")
// wait until at most N of this wavefront's LDS reads are outstanding; ties the registers the wait makes valid
#define QUAD_WAIT(N, f) asm volatile("s_waitcnt lgkmcnt(" #N ")" : "+v"(lo[f]), "+v"(hi[f]), "+v"(bf[0]), "+v"(bf[1]), "+v"(bf[2]), "+v"(bf[3]) :: "memory")
#define QUAD_GROUP(f) do { \
            const V8 fa = __builtin_shufflevector(__builtin_bit_cast(V4, lo[f]), __builtin_bit_cast(V4, hi[f]), 0, 1, 2, 3, 4, 5, 6, 7); \
            acc[0][f] = mfma16(fa, bf[0], acc[0][f]); \
            acc[1][f] = mfma16(fa, bf[1], acc[1][f]); \
            acc[2][f] = mfma16(fa, bf[2], acc[2][f]); \
            acc[3][f] = mfma16(fa, bf[3], acc[3][f]); } while (0)
        static_assert(NF == 8, "the MFMA groups below are written out for head dim 128");
        auto turn = [&](auto ACTIVE, int s) __attribute__((always_inline)) {
            constexpr bool active = decltype(ACTIVE)::value;
            __builtin_amdgcn_s_waitcnt(WAIT_FILLS);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            const int u = s - lag;                             // sweep position accumulated in this step
            // O1: dO part of tile u; O2: Q part of tile u
            const unsigned part = lds0 + (second ? C::Q_OFF + ((u + C::RQ) % C::RQ) * C::KP_BYTES : C::DO_OFF + ((u + C::RDO) % C::RDO) * C::KP_BYTES);
            const unsigned ta0 = part + tr_off[0], ta1 = part + tr_off[1];
            // U(u) was written in step u (stage u & 1), W(u) in step u + 1 (stage u & 1 as well)
            const unsigned hin = lds0 + (second ? w_base : u_base) + (u & 1) * 2 * C::HO_BYTES + 16 * lane;
            V8 bf[NG];
            quad_s16x4 lo[NF], hi[NF];
            if (active) {
                asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:1024\n\tds_read_b128 %2, %4 offset:2048\n\tds_read_b128 %3, %4 offset:3072"
                             : "=&v"(bf[0]), "=&v"(bf[1]), "=&v"(bf[2]), "=&v"(bf[3]) : "v"(hin) : "memory");
                QUAD_TR_PAIR(0); QUAD_TR_PAIR(1); QUAD_TR_PAIR(2); QUAD_TR_PAIR(3);
            }
            SCHED_FENCE();
            // dO(s+3), Q(s+4) + statistics(s+4): into slots that were read for the last time in step s-1 or before
            fill_do(t_do, s + 3); fill_q(t_q, s + 4);
            t_do = wrap_inc(t_do); t_q = wrap_inc(t_q);
            SCHED_FENCE();
            if (active) {
                QUAD_TR_PAIR(4); QUAD_WAIT(8, 0); QUAD_GROUP(0);
                QUAD_TR_PAIR(5); QUAD_WAIT(8, 1); QUAD_GROUP(1);
                QUAD_TR_PAIR(6); QUAD_WAIT(8, 2); QUAD_GROUP(2);
                QUAD_TR_PAIR(7); QUAD_WAIT(8, 3); QUAD_GROUP(3);
                QUAD_WAIT(6, 4); QUAD_GROUP(4);
                QUAD_WAIT(4, 5); QUAD_GROUP(5);
                QUAD_WAIT(2, 6); QUAD_GROUP(6);
                QUAD_WAIT(0, 7); QUAD_GROUP(7);
            }
            SCHED_FENCE();
        };
        // (three loops: a step's products under a condition have the compiler keep the accumulators twice)
        int s = 0;
        for (; s < lag; ++s) turn(std::false_type(), s);
        for (; s < lag + n; ++s) turn(std::true_type(), s);
        for (; s <= n + 1; ++s) turn(std::false_type(), s);
#undef QUAD_TR_PAIR
#undef QUAD_WAIT
#undef QUAD_GROUP
        __builtin_amdgcn_s_waitcnt(0x0F70);   // drain the (unused) trailing fills before the LDS is released
        // ---- epilogue: dV = dV^T (O1), dK = s dK^T (O2)
        const float sc = second ? p.sm_scale : 1.0f;
#pragma unroll
        for (int kg = 0; kg < NG; ++kg) {
            const int wrow = grp * 64 + 16 * kg + l16, row = blk * kBlock + wrow;
            if (partial) {   // a range of the stream only: leave the sums for bwd_combine_kernel ([row][dV | dK])
                const int64_t slot = (int64_t)(pair - p.n_full) * p.splits + split;
                float* pa = p.part + (slot * kBlock + wrow) * (2 * D) + (second ? D : 0) + 4 * g;
#pragma unroll
                for (int f = 0; f < NF; ++f) *reinterpret_cast<float4*>(pa + 16 * f) = make_float4(acc[kg][f][0], acc[kg][f][1], acc[kg][f][2], acc[kg][f][3]);
            } else if (row < p.L_stat) {
                T* out = (second ? reinterpret_cast<T*>(p.out2) + (int64_t)b * p.o2_sb + (int64_t)h * p.o2_sh + (int64_t)row * p.o2_sl
                                 : reinterpret_cast<T*>(p.out1) + (int64_t)b * p.o1_sb + (int64_t)h * p.o1_sh + (int64_t)row * p.o1_sl) + 4 * g;
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    V4 v;
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = (T)(acc[kg][f][r] * sc);
                    *reinterpret_cast<V4*>(out + 16 * f) = v;
                }
            }
        }
    }
}
