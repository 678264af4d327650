// dK/dV kernel of the backward for head dim 128.  Included inside the anonymous namespace of attn_bwd_gfx950.hip (uses BwdParams, kRows, kBwdSweepStagger,
// part_unit_slot and attn_common_gfx950.h).
//
// A workgroup of four wavefronts, one per SIMD, owns 64 NG keys and streams 32-query tiles (Q, dO, LSE log2 e, -D).  A wavefront does all of it for its own 16 NG keys:
//     S = Q k^T,  P = exp2(S c - LSE'),  dP - D = dO v^T - D,  dS = P (dP - D),  dV^T += dO^T P,  dK^T += Q^T dS,
// with K and V rows as stationary B operands (128 registers at NG = 4), dV^T and dK^T in all 256 accumulation registers, and P and dS from registers to registers: rounded,
// they are the B operands of the last two products as they lie.  Every stream operand read from LDS feeds NG products.
//
// What bounds it: the part's power limit; with 512 registers a wavefront there is no second one on a SIMD to fill gaps, so the step is written in slots, a product
// and what is issued beside it.  Measured of a wavefront that has its SIMD to itself, per v_mfma_f32_16x16x32 of 16 cycles: with two other instructions 18 cycles, three 22,
// four 26 (an exponential counts twice).  A step has 32 NG products and, at NG = 4, 2.3 others to a product, spread evenly (fixed(), room(), exp_before(), ds_before());
// placed where they are needed first, with all LDS reads of a group in one slot, a step took 3100 cycles instead of 2810.
// The kernel before this one handed P and dS from wavefronts that formed them to wavefronts that held the accumulators, through LDS, 128 keys a workgroup.  At 2 heads x
// 84480 queries and keys, dS kept: 26.2 -> 19.0 million cycles, clock 1.91 -> 1.73 GHz, 13.7 -> 11.0 ms; the backward, us, 16 heads, 24640 13 870 -> 12 160, 10920 2750 -> 2465,
// 5000 (40 heads) 1578 -> 1398, 3520 330 -> 294, 37440 x 512 571 -> 526, 37440 x 300 468 -> 422.
//
// v_mfma_f32_16x16x32: lane (i = lane % 16, g = lane / 16) of an operand has the contraction's elements 8 g .. + 7 of row or column i; of a result column i and rows 4 g .. + 3.
// A tile of S or dP is [16 keys][query half]; its registers, both query halves of 16 keys, are as they are the B operand of dV^T and dK^T, with queries 4 g .. + 3
// and 16 + 4 g .. + 3 as elements 0 .. 3 and 4 .. 7, and the unit that is stored of dS.
//
// A step: S of tile s | dK of tile s - 1 | dP of tile s | dV of tile s.  P is formed from behind the first half of S up to dP's end, dS from dP's end into the next step's
// S, whose results go where P was: each half only once it has been used.
//
// One copy of the stream.  A part of a tile in LDS is 32 rows x 128 channels as 16-byte units (row r, chunk C of 8 channels).  S and dP read them with ds_read_b128
// (lane = row); dV and dK need the transposed operands (lane = channel, 2 x 4 rows) and get them from the SAME units with the transposing read
// ds_read_b64_tr_b16 (within 16 lanes, lane i passes the address of 8 bytes -- row i of a 16 x 4 matrix M of 16-bit values -- and receives M[i/4 + 4k][i%4], k = 0..3).
// The unit (r, C) lies at
//     slot(r, C) = 64 (r/4) + 16 (C/4) + 4 (r%4) + (C%4 XOR part_swizzle(r/4)), the swizzle 0, 2, 3, 1 for r/4 = 0 .. 3:
// the lanes that a ds_read_b128 serves together and the 32 lanes of a transposing pass touch 256 consecutive-bank bytes each (SQ_LDS_BANK_CONFLICT = 0), and a direct-to-LDS
// load of 64 units is four whole rows, so that the loads read Q and dO rows where they are (or in the copy that is made of rows which they cannot address).
// Products, LDS reads and their waits are asm: neither their order nor a wait is the compiler's (which would put vmcnt(0) in front of LDS reads, for the loads in flight).

typedef unsigned bwd_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned bwd_u32x2 __attribute__((ext_vector_type(2)));

constexpr int kDkdvThreads = 256;
template <int NG>
struct DkdvCfg {
    static constexpr int D = 128, NQ = D / 32, NF = D / 16;   // 32- and 16-channel chunks
    static constexpr int KEYS = 4 * 16 * NG;                  // of a workgroup
    static constexpr int PART_BYTES = NF * kFragBytes;        // Q part, dO part of a tile
    static constexpr int STAT_OFF = 2 * PART_BYTES, SLOT_BYTES = STAT_OFF + kTileStatBytes;
    static constexpr int AHEAD = 5, RING = AHEAD + 2;         // tiles: loads run that many steps ahead; Q of the tile before is read for one step more
    static constexpr int LDS_BYTES = RING * SLOT_BYTES;
    static constexpr int LOADS = 5;                           // per wavefront and step: 4 rows twice of each part + the statistics
};
constexpr int kDkdvLdsBytes = DkdvCfg<4>::LDS_BYTES;

#define DKDV_MFMA(OP)                                                                                                                                \
    static __device__ __forceinline__ void first(f32x4& c, bwd_u32x4 a, bwd_u32x4 b) { asm volatile(OP " %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b)); }  \
    static __device__ __forceinline__ void from(f32x4& c, bwd_u32x4 a, bwd_u32x4 b, f32x4 s) { asm volatile(OP " %0, %1, %2, %3" : "=&v"(c) : "v"(a), "v"(b), "v"(s)); } \
    static __device__ __forceinline__ void more(f32x4& c, bwd_u32x4 a, bwd_u32x4 b) { asm volatile(OP " %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b)); }  \
    static __device__ __forceinline__ void sum(f32x4& c, bwd_u32x4 a, bwd_u32x4 b) { asm volatile(OP " %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b)); }
template <typename T> struct DkdvMfma;
template <> struct DkdvMfma<__bf16> { DKDV_MFMA("v_mfma_f32_16x16x32_bf16") };
template <> struct DkdvMfma<_Float16> { DKDV_MFMA("v_mfma_f32_16x16x32_f16") };
#undef DKDV_MFMA

template <int OFF> __device__ __forceinline__ void lds_read(bwd_u32x4& v, unsigned a) { asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF)); }
template <int OFF> __device__ __forceinline__ void lds_read(f32x4& v, unsigned a) { asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF)); }
template <int OFF> __device__ __forceinline__ void lds_read_transposed(bwd_u32x2& v, unsigned a) { asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF)); }
// registers that a wait has made valid
template <typename V> __device__ __forceinline__ void landed(V& a) { asm volatile("" : "+v"(a)); }

template <typename T, int NG, bool SPILL, bool CAUSAL>
__global__ void __attribute__((amdgpu_flat_work_group_size(kDkdvThreads, kDkdvThreads), amdgpu_waves_per_eu(1, 1)))
attn_dkdv_kernel(const BwdParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef DkdvCfg<NG> C;
    typedef DkdvMfma<T> M;
    typedef typename VecOf<T>::v4 V4;
    typedef T V2 __attribute__((ext_vector_type(2)));
    constexpr int D = C::D, NQ = C::NQ, NF = C::NF;

    const int bid = blockIdx.x;
    const bool partial = bid >= p.n_full && p.splits > 1;
    const int pair = partial ? p.n_full + (bid - p.n_full) / p.splits : bid;
    const int split = partial ? (bid - p.n_full) % p.splits : 0;
    const int blk = pair % p.n_blk, bhl = pair / p.n_blk, bh = p.bh0 + bhl, b = bh / p.H, h = bh % p.H;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    const int row0 = blk * C::KEYS + wave * 16 * NG;     // first key of this wavefront

    int t_lo = 0, t_hi = p.n_tiles;
    if (CAUSAL) t_lo = (blk * C::KEYS) / kRows;          // query tiles before the block's first key see none of its keys
    if (partial) {
        t_lo = (int)((int64_t)split * p.n_tiles / p.splits);
        t_hi = (int)((int64_t)(split + 1) * p.n_tiles / p.splits);
    }
    const int n = t_hi > t_lo ? t_hi - t_lo : 0;
    const int n_sweep = n > 0 ? n : 1;
    const int shift = (((pair >> 3) & 31) * kBwdSweepStagger) % n_sweep;
    auto tile_at = [&](int u) { return __builtin_amdgcn_readfirstlane(t_lo + (u + shift) % n_sweep); };
    auto wrap_inc = [&](int t) { ++t; return t >= t_lo + n_sweep ? t - n_sweep : t; };

    auto rows_of = [&](const StreamRows& r) {   // a head's rows; behind the last one zeros are read
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(r.ptr) + (int64_t)b * r.sb + (int64_t)h * r.sh, 0, (p.L_stream - 1) * r.row + 2 * D, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rsrc_q = rows_of(p.rows_q), rsrc_do = rows_of(p.rows_do);
    const __amdgpu_buffer_rsrc_t rsrc_st = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(p.stream) + (size_t)bh * p.n_tiles * kTileStatBytes, 0, p.n_tiles * kTileStatBytes, 0x00020000);
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem;

    // ---- loads: this wavefront's eight rows 8 wave .. + 7 of a part of tile t into a ring slot, four rows a load
    int off_q[2], off_do[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = 8 * wave + 4 * i + ((lane >> 2) & 3), unit = 4 * (lane >> 4) + ((lane & 3) ^ part_swizzle(2 * wave + i));
        off_q[i] = r * p.rows_q.row + 16 * unit;
        off_do[i] = r * p.rows_do.row + 16 * unit;
    }
    auto load = [&](auto which, int t, unsigned slot) __attribute__((always_inline)) {
        constexpr int W = decltype(which)::value;
        char* dst = smem + slot;
        if constexpr (W < 2) lds_load<0>(rsrc_q, dst + (2 * wave + W) * kFragBytes, off_q[W] + t * (kRows * p.rows_q.row), 0);
        else if constexpr (W < 4) lds_load<0>(rsrc_do, dst + C::PART_BYTES + (2 * wave + W - 2) * kFragBytes, off_do[W - 2] + t * (kRows * p.rows_do.row), 0);
        else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_st, (__attribute__((address_space(3))) void*)(dst + C::STAT_OFF), 4, lane * 4, t * kTileStatBytes, 0, 0);
    };
    for (int u = 0; u < C::AHEAD; ++u) {
        const int t = tile_at(u);
        for_each<C::LOADS>([&](auto w) { load(w, t, u * C::SLOT_BYTES); });
    }

    // ---- this wavefront's K and V rows as B operands: key row0 + 16 kg + l16, channels 32 c + 8 g .. + 7
    bwd_u32x4 kb[NG][NQ], vb[NG][NQ];
#pragma unroll
    for (int kg = 0; kg < NG; ++kg) {
        const int row = row0 + 16 * kg + l16;
        const bool live = row < p.L_stat;
        const T* kp = reinterpret_cast<const T*>(p.st1) + (int64_t)b * p.s1_sb + (int64_t)h * p.s1_sh + (int64_t)row * p.s1_sl + 8 * g;
        const T* vp = reinterpret_cast<const T*>(p.st2) + (int64_t)b * p.s2_sb + (int64_t)h * p.s2_sh + (int64_t)row * p.s2_sl + 8 * g;
#pragma unroll
        for (int c = 0; c < NQ; ++c) {
            const bwd_u32x4 z = {0, 0, 0, 0};
            kb[kg][c] = live ? *reinterpret_cast<const bwd_u32x4*>(kp + 32 * c) : z;
            vb[kg][c] = live ? *reinterpret_cast<const bwd_u32x4*>(vp + 32 * c) : z;
        }
    }

    // ---- state: [16 keys][query half], register r: key 16 kg + l16, query 16 m + 4 g + r
    f32x4 x[NG][2], y[NG][2];                  // S, then P | dP - D, then dS
    bwd_u32x4 u[NG], w[NG];                    // P, dS rounded: B operands (queries 4 g .. + 3, 16 + 4 g .. + 3 of 16 keys)
    f32x4 adv[NG][NF], adk[NG][NF];            // dV^T, dK^T: [16 keys][16 channels], register r: key 16 kg + l16, channel 16 f + 4 g + r
#pragma unroll
    for (int kg = 0; kg < NG; ++kg) {
#pragma unroll
        for (int f = 0; f < NF; ++f) { adv[kg][f] = f32x4{0.f, 0.f, 0.f, 0.f}; adk[kg][f] = f32x4{0.f, 0.f, 0.f, 0.f}; }
        // (the first step adds a dK of nothing)
        x[kg][0] = x[kg][1] = y[kg][0] = y[kg][1] = f32x4{0.f, 0.f, 0.f, 0.f};
        w[kg] = bwd_u32x4{0, 0, 0, 0};
    }
    f32x4 l2[2], md[2];                        // LSE log2 e and -D of this lane's queries

    // ---- LDS reads
    bwd_u32x4 fa[4];                           // A operands of the groups under way: one read, or two transposing ones
    bwd_u32x2 lo[4], hi[4];
    const unsigned a_off = lds0 + 16 * part_unit_slot(l16, g);
    unsigned tr_off[2];
#pragma unroll
    for (int o = 0; o < 2; ++o) tr_off[o] = lds0 + (unsigned)(16 * part_unit_slot(4 * g + (l16 >> 2), 2 * o + ((l16 & 3) >> 1)) + 8 * (l16 & 1));
    const unsigned st_off = lds0 + C::STAT_OFF + 16 * g;
    unsigned s_prev = 0, s_cur = 0, s_load = C::AHEAD * C::SLOT_BYTES;      // ring slots: of the tile before, of this step's, of the one that is loaded
    auto next_slot = [](unsigned s) { return s + C::SLOT_BYTES < C::RING * C::SLOT_BYTES ? s + C::SLOT_BYTES : 0u; };

    // The step's products in 32 groups of NG, one A operand each: S (query half G / 4, channels 32 (G % 4)), dK of the tile before (16 channels G % 8), dP, dV.
    // (half 1: the second read of an operand that takes two)
    auto read_group = [&](auto gi, auto half) __attribute__((always_inline)) {
        constexpr int G = decltype(gi)::value % 32, SEC = G / 8, I = G % 8, H = decltype(half)::value;
        const unsigned part = (SEC == 1 ? s_prev : s_cur) + (SEC >= 2 ? C::PART_BYTES : 0);
        if constexpr (SEC % 2 == 0) {
            if constexpr (H == 0) lds_read<4096 * (I / 4) + 256 * (I % 4)>(fa[G % 4], part + a_off);
        } else {
            lds_read_transposed<256 * (I / 2) + 4096 * H>(H ? hi[G % 4] : lo[G % 4], part + tr_off[I % 2]);
        }
    };
    auto group_landed = [&](auto gi) __attribute__((always_inline)) {
        constexpr int G = decltype(gi)::value;
        if constexpr (G / 8 % 2 == 0) landed(fa[G % 4]);
        else { landed(lo[G % 4]); landed(hi[G % 4]); }
    };
    auto operand = [&](auto gi) __attribute__((always_inline)) {
        constexpr int G = decltype(gi)::value;
        if constexpr (G / 8 % 2 == 0) return fa[G % 4];
        else return bwd_u32x4{lo[G % 4].x, lo[G % 4].y, hi[G % 4].x, hi[G % 4].y};
    };
    // statistics of this step's tile: in front of the reads of groups L2_AT and MD_AT
    constexpr int L2_AT = 4, MD_AT = 15;
    auto read_rows = [&](f32x4* v, auto at) __attribute__((always_inline)) {
        lds_read<decltype(at)::value>(v[0], st_off + s_cur);
        lds_read<decltype(at)::value + 64>(v[1], st_off + s_cur);
    };
    // LDS instructions from there up to and with those of group G's read
    constexpr auto reads_of = [](int G) { return (G == L2_AT || G == MD_AT ? 2 : 0) + 1 + G / 8 % 2; };

    // ---- the elements' arithmetic, in single instructions: elements are numbered [query half][16 keys][r], in pairs
    // P: per pair two products with the scale, two exponentials, one rounding (of the pair before: an exponential's result is not to be used right behind it)
    constexpr int PAIRS = 4 * NG;
    auto exp_op = [&](auto oi) __attribute__((always_inline)) {
        constexpr int O = decltype(oi)::value, P = O / 5, K = O % 5, ROUND = P - (K == 2);
        if constexpr (P < PAIRS && K != 2) {
            constexpr int E = 2 * P + (K == 1 || K == 4), m = E / (4 * NG), kg = E / 4 % NG, r = E % 4;
            if constexpr (K < 2) x[kg][m][r] = __builtin_fmaf(x[kg][m][r], p.scale_log2, -l2[m][r]);
            else x[kg][m][r] = __builtin_amdgcn_exp2f(x[kg][m][r]);
        }
        if constexpr (K == 2 && ROUND >= 0 && ROUND < PAIRS) {
            constexpr int E = 2 * ROUND, m = E / (4 * NG), kg = E / 4 % NG, r = E % 4;
            const V2 two = {(T)x[kg][m][r], (T)x[kg][m][r + 1]};
            u[kg][2 * m + r / 2] = __builtin_bit_cast(unsigned, two);
        }
    };
    // dS: per pair two products, one rounding
    auto ds_op = [&](auto oi) __attribute__((always_inline)) {
        constexpr int O = decltype(oi)::value, E = 2 * (O / 3) + (O % 3 == 1), m = E / (4 * NG), kg = E / 4 % NG, r = E % 4;
        if constexpr (O % 3 < 2) {
            y[kg][m][r] *= x[kg][m][r];
        } else {
            const V2 two = {(T)y[kg][m][r], (T)y[kg][m][r + 1]};
            w[kg][2 * m + r / 2] = __builtin_bit_cast(unsigned, two);
        }
    };
    auto mask = [&](int t) {
        if (row0 + 16 * NG - 1 <= t * kRows) return;
        // (key <= query, what a lane adds to either on one side: rows of keys, one register each, are not to be had with NG = 4, where dS is kept)
        const int lane_part = l16 - 4 * g;
#pragma unroll
        for (int kg = 0; kg < NG; ++kg) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                x[kg][e >> 2][e & 3] = lane_part <= t * kRows + 16 * (e >> 2) + (e & 3) - row0 - 16 * kg ? x[kg][e >> 2][e & 3] : -INFINITY;
        }
    };

    // ---- what a slot holds beside its MFMA
    constexpr int SLOTS = 32 * NG, LOAD_G = 9, STORE_G = 4, MISC = NG > 2 ? 2 : 1;
    constexpr auto fixed = [](int q) {
        const int G = q / NG % 32, kg = q % NG, target = (G + 3) % 32;
        int c = 0;
        if (kg == 0) c += 1 + (target == L2_AT || target == MD_AT ? 2 : 0);
        if (kg == 1) c += target / 8 % 2;
        if (kg == NG - 1) c += 1;
        if (kg == MISC && SPILL && G >= STORE_G && G < STORE_G + NG) c += 1;
        if (kg == MISC && G >= LOAD_G && G < LOAD_G + C::LOADS) c += 4;
        return c;
    };
    // room for the elements' work in slots q0 .. q - 1
    constexpr auto room = [fixed](int q0, int q) {
        int c = 0;
        for (int i = q0; i < q; ++i) c += fixed(i) < 3 ? 3 - fixed(i) : 0;
        return c;
    };
    // P: from S of the first query half on, up to dV.  dS: from dP on, up to the next step's S of the second query half
    constexpr int EXP0 = (CAUSAL ? 9 : 5) * NG, EXP1 = 20 * NG, EXP_WORK = 7 * PAIRS + 1;
    constexpr int DS0 = 24 * NG + 2, DS1 = 35 * NG, DS_OPS = 3 * PAIRS;
    // operations done before slot q
    constexpr auto exp_before = [room](int q) {
        if (q <= EXP0) return 0;
        if (q >= EXP1) return 5 * PAIRS + 3;
        const int done = EXP_WORK * room(EXP0, q) / room(EXP0, EXP1);      // of 1 1 1 2 2 a pair
        constexpr int at[7] = {0, 1, 2, 3, 3, 4, 4};
        return 5 * (done / 7) + at[done % 7];
    };
    constexpr auto ds_before = [room](int q) { return q <= DS0 ? 0 : q >= DS1 ? DS_OPS : DS_OPS * room(DS0, q) / room(DS0, DS1); };
    static_assert(ds_before(SLOTS) >= DS_OPS / 2, "the next S is written where the first half of P was");

    // ---- dS of the tile before, to memory: [query tile][16 keys] of 1 KB; inside of 32 x 32 the unit (key, g) sits at slot 16 (key / 4) + 4 g + key % 4, the order
    // in which the transposing reads of attn_dq_from_ds_kernel touch 256 consecutive bytes per pass
    const int64_t ds_row = (int64_t)p.n_kt_pad * 2 * kFragBytes;
    const char* const ds_head = SPILL ? p.ds + (int64_t)bhl * p.ds_head_bytes : nullptr;
    const unsigned ds_lane = (unsigned)(row0 / 16) * kFragBytes + 16 * (16 * (l16 >> 2) + 4 * g + (l16 & 3));
    int t_prev = -1;
    auto store_ds = [&](auto ki) __attribute__((always_inline)) {
        constexpr int kg = decltype(ki)::value;
        const int t = __builtin_amdgcn_readfirstlane(t_prev);
        // (t < 0: there is none yet; stores past the end of a buffer are dropped)
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(ds_head) + (int64_t)(t < 0 ? 0 : t) * ds_row, 0, t < 0 ? 0u : (unsigned)ds_row, 0x00020000);
        __builtin_amdgcn_raw_buffer_store_b128(w[kg], rsrc, ds_lane + kg * kFragBytes, 0, 2);
    };

    int t_cur = tile_at(0), t_load = tile_at(C::AHEAD);
    auto slot = [&](auto qi) __attribute__((always_inline)) {
        constexpr int Q = decltype(qi)::value, G = Q / NG, kg = Q % NG, SEC = G / 8, I = G % 8;
        SCHED_FENCE();
        if constexpr (SEC == 0) {
            constexpr int m = I / 4, c = I % 4;
            if constexpr (c == 0) M::first(x[kg][m], operand(Int<G>{}), kb[kg][c]);
            else M::more(x[kg][m], operand(Int<G>{}), kb[kg][c]);
        } else if constexpr (SEC == 1) {
            M::sum(adk[kg][I], operand(Int<G>{}), w[kg]);
        } else if constexpr (SEC == 2) {
            constexpr int m = I / 4, c = I % 4;
            if constexpr (c == 0) M::from(y[kg][m], operand(Int<G>{}), vb[kg][c], md[m]);
            else M::more(y[kg][m], operand(Int<G>{}), vb[kg][c]);
        } else {
            M::sum(adv[kg][I], operand(Int<G>{}), u[kg]);
        }
        if constexpr (kg == 0) {
            if constexpr (G + 3 == 32) {       // the reads go on to the next tile
                s_prev = s_cur;
                s_cur = next_slot(s_cur);
            }
            if constexpr (G + 3 == L2_AT) read_rows(l2, Int<0>{});
            if constexpr (G + 3 == MD_AT) read_rows(md, Int<128>{});
            read_group(Int<G + 3>{}, Int<0>{});
        }
        if constexpr (kg == 1) read_group(Int<G + 3>{}, Int<1>{});
        if constexpr (kg == NG - 1) {          // the next group's operand is here
            wait_lds<reads_of((G + 2) % 32) + reads_of((G + 3) % 32)>();
            group_landed(Int<(G + 1) % 32>{});
            if constexpr (G + 1 == L2_AT) { landed(l2[0]); landed(l2[1]); }
            if constexpr (G + 1 == MD_AT) { landed(md[0]); landed(md[1]); }
        }
        if constexpr (CAUSAL && Q == 9 * NG - 1) mask(t_cur);
        for_each<exp_before(Q + 1) - exp_before(Q)>([&](auto i) { exp_op(Int<exp_before(Q) + decltype(i)::value>{}); });
        constexpr int DQ = Q >= 24 * NG ? Q : Q + SLOTS;
        for_each<ds_before(DQ + 1) - ds_before(DQ)>([&](auto i) { ds_op(Int<ds_before(DQ) + decltype(i)::value>{}); });
        // dS of the tile before, and behind that (as counted below) the loads
        if constexpr (SPILL && kg == MISC && G >= STORE_G && G < STORE_G + NG) store_ds(Int<G - STORE_G>{});
        if constexpr (kg == MISC && G >= LOAD_G && G < LOAD_G + C::LOADS) load(Int<G - LOAD_G>{}, t_load, s_load);
        if constexpr (Q == (LOAD_G + C::LOADS) * NG) { s_load = next_slot(s_load); t_load = wrap_inc(t_load); }
        if constexpr (Q == (LOAD_G + C::LOADS) * NG + 1) { t_prev = t_cur; t_cur = wrap_inc(t_cur); }
        SCHED_FENCE();
    };
    // vector memory operations (they retire in the order of issue) behind the loads of the next step's tile, AHEAD - 1 steps ago: then that tile is here
    constexpr int NEWER = (C::AHEAD - 2) * (C::LOADS + (SPILL ? NG : 0));
    static_assert(NEWER < 64, "vmcnt");
    auto step = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NEWER) : "memory");
        __builtin_amdgcn_s_barrier();          // ... everybody's loads of it, and everybody is done with the tile two before
        for_each<SLOTS>([&](auto q) { slot(q); });
    };

    __builtin_amdgcn_s_waitcnt(0x0070);        // K, V and the first tiles are here
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (n > 0) {
        for_each<3>([&](auto i) { read_group(i, Int<0>{}); });
        wait_lds<2>();
        group_landed(Int<0>{});
        int s = 0;
#pragma clang loop unroll(disable)
        do step(); while (++s < n);
        // what is left of the last tile: its dS, dK.  (What was read ahead is not used, but its registers are not anybody's before it is here.)
        wait_lds<0>();
        for_each<3>([&](auto i) { group_landed(i); });
        for_each<DS_OPS - ds_before(SLOTS)>([&](auto i) { ds_op(Int<ds_before(SLOTS) + decltype(i)::value>{}); });
        if constexpr (SPILL) for_each<NG>([&](auto i) { store_ds(i); });
        SCHED_FENCE();
        for_each<8>([&](auto f) {
            constexpr int G = 8 + decltype(f)::value;
            read_group(Int<G>{}, Int<0>{});
            read_group(Int<G>{}, Int<1>{});
            wait_lds<0>();
            group_landed(Int<G>{});
            for_each<NG>([&](auto k) { M::sum(adk[decltype(k)::value][decltype(f)::value], operand(Int<G>{}), w[decltype(k)::value]); });
        });
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");      // the last products (written as asm: no hazard checks) are in their registers
    __builtin_amdgcn_s_waitcnt(0x0F70);                     // drain the (unused) trailing loads before the LDS is released

    // ---- epilogue: dV = dV^T, dK = s dK^T.  (The lane's part is counted anew: kept over the loop it takes registers that NG = 4, causal, dS kept, does not have)
    const int lane_now = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0)), l16_now = lane_now & 15, g_now = lane_now >> 4;
#pragma unroll
    for (int kg = 0; kg < NG; ++kg) {
        const int row = row0 + 16 * kg + l16_now;
        if (partial) {   // a range of the stream only: leave the sums for bwd_combine_kernel ([row][dV | dK])
            const int64_t at = ((int64_t)(pair - p.n_full) * p.splits + split) * C::KEYS + row - blk * C::KEYS;
            float* pa = p.part + at * (2 * D) + 4 * g_now;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                asm volatile("" : "+a"(adv[kg][f]), "+a"(adk[kg][f]));
                *reinterpret_cast<f32x4*>(pa + 16 * f) = adv[kg][f];
                *reinterpret_cast<f32x4*>(pa + D + 16 * f) = adk[kg][f];
                SCHED_FENCE();
            }
        } else if (row < p.L_stat) {
            T* dv = reinterpret_cast<T*>(p.out1) + (int64_t)b * p.o1_sb + (int64_t)h * p.o1_sh + (int64_t)row * p.o1_sl + 4 * g_now;
            T* dk = reinterpret_cast<T*>(p.out2) + (int64_t)b * p.o2_sb + (int64_t)h * p.o2_sh + (int64_t)row * p.o2_sl + 4 * g_now;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                asm volatile("" : "+a"(adv[kg][f]), "+a"(adk[kg][f]));
                V4 a, c;
#pragma unroll
                for (int r = 0; r < 4; ++r) { a[r] = (T)adv[kg][f][r]; c[r] = (T)(adk[kg][f][r] * p.sm_scale); }
                *reinterpret_cast<V4*>(dv + 16 * f) = a;
                *reinterpret_cast<V4*>(dk + 16 * f) = c;
                SCHED_FENCE();
            }
        }
    }
#endif
}
