// Forward + JVP at head dim 128, bf16, from about a round of workgroups on.  Included inside the anonymous namespace of attn_fwd_jvp_gfx950.hip, behind attn_mfma16_gfx950.h
// (same image of K and V, same arithmetic and rounding as ScoreWave16 / OutputWave16, but for the sums that outputs are divided by).
//
// A workgroup of four wavefronts, one per SIMD, owns 64 NG query rows; a wavefront does all of it for its own 16 NG: Q in vector registers and dQ in accumulation registers as B operands, S and dS,
// the softmax, P and H, which rounded are the B operands of the outputs' products as they lie, O^T and T^T in accumulation registers.  Nothing is handed over through LDS, a K or V
// operand read from there feeds 2 NG products (dK, dV: NG), and the loads of a tile serve 192 rows instead of 128.  (NG = 4 does not fit: 16 registers too many.)
//
// What bounds it: the part's power limit and, next to that, instruction issue.  A wavefront alone on its SIMD hides two other instructions behind a v_mfma_f32_16x16x32 of
// 16 cycles (measured: with two 18 cycles, three 22, four 26; an exponential counts twice), so a step is written in slots, a product and what is issued beside it, with the elements'
// work spread by the room that LDS reads, waits and loads leave (fixed(), room(), args_before(), exps_before()).  A step is 150 products with all tangents, 102 with one on q alone.
// 16 heads x 33000 positions, all tangents, attn_fwd_jvp_kernel / this: LDS-active cycles 1085 / 364 million, 34.3 / 35.4 million cycles, 1.69 / 1.95 GHz, 20.36 / 18.18 ms; tangent on q
// 15.06 / 12.71 ms (further sizes beside kRowsWhole).
//
// A step: S of tile t, key half 0, then 1 | outputs of tile t - 1.  Arguments of the exponentials and their max behind S; P and H up to the next step's S of half 1, whose results go
// where theirs were: each half only once it has been used.  The loop turns between the arguments and the exponentials (settle()), where masks and a max that moves are looked at:
// what is rare is outside of the loop's one straight block, which the compiler would otherwise fill with copies.  Its products, LDS reads and waits are asm: an operand is here when
// landed() says so, and a read whose result nobody uses is not issued (its registers would be somebody else's by the time it arrives).
// fp16, whose range needs the exact running max, stays with the other kernel.

template <int MODE, int NG>
struct RowsCfg {
    typedef AttnCfg<128, 128, MODE> A;
    static constexpr bool FULL = MODE == MODE_JVP_FULL;
    static constexpr int ROWS = 4 * 16 * NG, NC = 4, NF = 8;                  // of a workgroup; chunks of 32 channels; groups of 16
    static constexpr int KRING = 5, VRING = 4;                                // parts of K and of V in LDS
    static constexpr int KRING_OFF = 0, VRING_OFF = KRING * A::KP_BYTES, SPARE_OFF = VRING_OFF + VRING * A::VP_BYTES;
    static constexpr int LDS_BYTES = SPARE_OFF + 4 * 4 * kFragBytes;          // and 4 KB for each wavefront
    static constexpr int K_LOADS = A::KP_FR / 4, V_LOADS = A::VP_FR / 4;      // per wavefront and step
};
constexpr int kRowsThreads = 256;
// How far an argument of the exponentials may lie above the max that they refer to, in powers of two.  Moving the max costs a wavefront some 2 us here, and 192 rows wait for each other: with kMaxSlack, whose
// 6 keep p in fp16's range, scores of a standard deviation of 4 had it in most steps.  bf16 and fp32 have the range (sums stay below 2^40 times their terms).  What an exact max has is that the
// largest p, 1, is not rounded; so outputs are divided by sums of p as it is rounded, which a row's largest p has its error in as well: six products a step, for the 24 additions of the sum of H.
// us, 6 / 40 (attn_fwd_jvp_kernel), 16 heads, scores of standard deviation 4: all tangents 3072 x 2000 256 / 128 (160), 20000 x 2000 1590 / 780 (851), tangent on q 6144 897 / 478 (584), 37440 x 2048 2570 / 1110;
// 8: 280 / 135 (164), 1760 / 778 (876), 1030 / 480 (591); 1: 128 / 127 (153), 777 / 774 (800), 473 / 476 (559).
// Error against 64 bits, o (dO of a tangent on q), 1000 keys: 1: 2.359e-3 / 2.353e-3 (2.369 / 2.365); 4: 2.02 / 1.88 (3.97 / 2.75); 8: 1.92 / 1.74 (5.19 / 2.95); attn_fwd_jvp_kernel 2.33 (2.37); 1.83 (3.87); 1.65 (4.72).
constexpr float kRowsSlack = 40.f;

typedef unsigned rows_u32x4 __attribute__((ext_vector_type(4)));
// (PAUSE: in front of the loop and behind it, where the compiler may copy an operand just before its use; of the wait that this takes it does not know, asm being asm)
#define ROWS_MFMA(OP)                                                                                                                                 \
    template <bool PAUSE, bool TAN> static __device__ __forceinline__ void first(f32x4& c, rows_u32x4 a, rows_u32x4 b) {                              \
        if constexpr (PAUSE) asm volatile("s_nop 3\n\t" OP " %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));                                            \
        else if constexpr (TAN) asm volatile(OP " %0, %1, %2, 0" : "=&v"(c) : "v"(a), "a"(b));                                                        \
        else asm volatile(OP " %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));                                                                           \
    }                                                                                                                                                 \
    template <bool PAUSE, bool TAN> static __device__ __forceinline__ void more(f32x4& c, rows_u32x4 a, rows_u32x4 b) {                               \
        if constexpr (PAUSE) asm volatile("s_nop 3\n\t" OP " %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));                                            \
        else if constexpr (TAN) asm volatile(OP " %0, %1, %2, %0" : "+v"(c) : "v"(a), "a"(b));                                                        \
        else asm volatile(OP " %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));                                                                           \
    }                                                                                                                                                 \
    template <bool PAUSE> static __device__ __forceinline__ void sum(f32x4& c, rows_u32x4 a, rows_u32x4 b) {                                          \
        if constexpr (PAUSE) asm volatile("s_nop 3\n\t" OP " %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));                                            \
        else asm volatile(OP " %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));                                                                           \
    }
template <typename T> struct RowsMfma;
template <> struct RowsMfma<__bf16> { ROWS_MFMA("v_mfma_f32_16x16x32_bf16") };
#undef ROWS_MFMA
template <int OFF> __device__ __forceinline__ void lds_read(rows_u32x4& v, unsigned a) { asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF)); }
template <int OFF> __device__ __forceinline__ void lds_read(f32x4& v, unsigned a) { asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF)); }
template <int OFF> __device__ __forceinline__ void lds_read_acc(f32x4& v, unsigned a) { asm volatile("ds_read_b128 %0, %1 offset:%2" : "=a"(v) : "v"(a), "n"(OFF)); }
template <int OFF> __device__ __forceinline__ void lds_write_acc(unsigned a, f32x4 v) { asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(a), "a"(v), "n"(OFF) : "memory"); }
template <int OFF> __device__ __forceinline__ void lds_write(unsigned a, rows_u32x4 v) { asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(a), "v"(v), "n"(OFF) : "memory"); }
// registers that a wait has made valid
template <typename V> __device__ __forceinline__ void landed(V& a) { asm volatile("" : "+v"(a)); }

template <typename T, int MODE, int NG>
__global__ void __attribute__((amdgpu_flat_work_group_size(kRowsThreads, kRowsThreads), amdgpu_waves_per_eu(1, 1)))
attn_jvp_rows_kernel(const AttnParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef RowsCfg<MODE, NG> C;
    typedef typename C::A A;
    typedef RowsMfma<T> M;
    typedef typename VecOf<T>::v4 V4;
    typedef T V2 __attribute__((ext_vector_type(2)));
    constexpr bool FULL = C::FULL;
    constexpr int NC = C::NC, NF = C::NF, TILE_BYTES = A::TILE_BYTES, KP_BYTES = A::KP_BYTES, VP_BYTES = A::VP_BYTES;

    // 1-D grid: block id -> (pair, key range); pair = query block + n_qt * (batch * H + head)
    const int bid = blockIdx.x;
    const bool partial = bid >= p.n_full && p.splits > 1;
    const int pair = partial ? p.n_full + (bid - p.n_full) / p.splits : bid;
    const int split = partial ? (bid - p.n_full) % p.splits : 0;
    const int qt = pair % p.n_qt, bh = pair / p.n_qt, b = bh / p.H, h = bh % p.H;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    const int row0 = qt * C::ROWS + wave * 16 * NG;      // first query row of this wavefront

    int kv_len = p.Lkv;
    if (p.key_lens) { const int kl = __builtin_amdgcn_readfirstlane(p.key_lens[b]); kv_len = kl < kv_len ? (kl < 0 ? 0 : kl) : kv_len; }
    int n_tiles_all = (kv_len + kBlockN - 1) / kBlockN;
    if (p.causal) { const int lim = (qt * C::ROWS + C::ROWS + kBlockN - 1) / kBlockN; n_tiles_all = n_tiles_all < lim ? n_tiles_all : lim; }
    const int u_lo = partial ? (int)((int64_t)split * n_tiles_all / p.splits) : 0;
    // (two at least: a second tile that is not there is masked, and zeros.  A loop that may be left at once takes the compiler copies and scratch inside of it)
    static_assert(kMinStepsPerSplit >= 2, "a range of one tile");
    const int n = partial ? (int)((int64_t)(split + 1) * n_tiles_all / p.splits) - u_lo : n_tiles_all == 1 ? 2 : n_tiles_all;

    const __amdgpu_buffer_rsrc_t kv_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(p.kv) + (size_t)bh * p.n_tiles * TILE_BYTES, 0, n_tiles_all * TILE_BYTES, 0x00020000);
    // sweep order: see attn_fwd_jvp_kernel
    const int n_sweep = n_tiles_all > 1 ? n_tiles_all : 2;
    const int shift = p.causal || n_tiles_all < 2 ? 0 : (((pair >> 3) & 31) * COSMOS_ATTN_SWEEP_STAGGER) % n_sweep;
    auto tile_at = [&](int u) { return __builtin_amdgcn_readfirstlane((u_lo + u + shift) % n_sweep); };
    auto wrap_inc = [&](int t) { ++t; return t >= n_sweep ? t - n_sweep : t; };
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem;

    // ---- loads: this wavefront's quarter of a K part or a V part
    const int k_lane = k_fill_lane(lane) * 16, v_lane = lane * 16;
    const int k_run = wave * C::K_LOADS * kFragBytes, v_run = wave * C::V_LOADS * kFragBytes;
    // (`checked`: bytes of the tile's place in the lanes' offset, which the buffer's bounds hold for; the scalar offset's are nobody's to rely on)
    auto load_k = [&](int t, unsigned slot, int checked = 0) __attribute__((always_inline)) { issue_part<C::K_LOADS>(kv_rsrc, smem + C::KRING_OFF + slot + k_run, k_lane + checked, t * TILE_BYTES + k_run); };
    auto load_v = [&](int t, unsigned slot, int checked = 0) __attribute__((always_inline)) { issue_part<C::V_LOADS>(kv_rsrc, smem + C::VRING_OFF + slot + v_run, v_lane + checked, t * TILE_BYTES + KP_BYTES + v_run); };
    // ---- this wavefront's Q and dQ rows as B operands: row 16 j + l16, channels 32 c + 8 g .. + 7
    rows_u32x4 qb[NG][NC], tb[NG][NC];
#pragma unroll
    for (int j = 0; j < NG; ++j) {
        const int row = row0 + 16 * j + l16;
        const bool live = row < p.Lq;
        const int64_t off = (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)row * p.q_sl + 8 * g;
        const T* qp = reinterpret_cast<const T*>(p.q) + off;
        const T* tp = reinterpret_cast<const T*>(p.tq) + off;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const rows_u32x4 z = {0, 0, 0, 0};
            qb[j][c] = live ? *reinterpret_cast<const rows_u32x4*>(qp + 32 * c) : z;
            tb[j][c] = live ? *reinterpret_cast<const rows_u32x4*>(tp + 32 * c) : z;
        }
    }

    // step t forms S of tile t and adds tile t - 1 to the outputs; it loads K of tile t + KRING - 1 and V of tile t + VRING - 2.  Here in the order in which the first steps wait for them,
    // behind Q: the first S wants nothing but that and K
    static_assert(C::KRING == 5 && C::VRING == 4, "the order");
    load_k(0, 0, tile_at(0) * TILE_BYTES);
#pragma unroll
    for (int u = 0; u < C::VRING; ++u) {
        load_k(0, (u + 1) * KP_BYTES, tile_at(u + 1) * TILE_BYTES);
        if (u < C::VRING - 1) load_v(0, u * VP_BYTES, tile_at(u) * TILE_BYTES);
    }

    // ---- state.  S^T of 16 keys x 16 rows: [16 rows][key half], register r: row 16 j + l16, key lane_key(lane) + 8 m + r of the tile
    f32x4 x[NG][2], y[NG][2];                   // S, then S c - max, then P | dS, then H
    rows_u32x4 pw[NG], hw[NG];                  // P, H rounded: B operands
    f32x4 acc[NF][NG], act[NF][NG];             // O^T, T^T: channels 16 f + 4 g + r of row 16 j + l16
    float m_run[NG], l_run[NG];                 // running max; this lane's keys' share of the row sum of P
    f32x4 psum[NG], hsum[NG];                   // row sums of P and H as rounded (of row 16 j + l16, in every register): what outputs are divided by has then the same errors as what is divided
    rows_u32x4 ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
    landed(ones);                               // (in registers, not formed again in the loop)
#pragma unroll
    for (int j = 0; j < NG; ++j) {
#pragma unroll
        for (int f = 0; f < NF; ++f) { acc[f][j] = f32x4{0.f, 0.f, 0.f, 0.f}; act[f][j] = f32x4{0.f, 0.f, 0.f, 0.f}; }
        m_run[j] = l_run[j] = 0.f;
        psum[j] = hsum[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        pw[j] = hw[j] = rows_u32x4{0, 0, 0, 0};
    }

    // ---- the step's products, in 16 groups of one operand A of K or V and, with tangents on k and v, one of dK or dV:
    // 0 .. 7: S, key half G / 4, channels 32 (G % 4); 8 .. 15: outputs, channels 16 (G % 8)
    constexpr int PER = (FULL ? 3 : 2) * NG, SLOTS = 16 * PER;
    constexpr int CHECK = 10 * PER;             // where the max is looked at
    constexpr int AHEAD = FULL ? 1 : 2;         // groups that LDS reads run ahead
    rows_u32x4 fa[AHEAD + 1 == 2 ? 2 : 4], fb[2];
    const unsigned frag_lane = lds0 + frag_offset(lane);
    unsigned k_slot = 0, v_slot = 0, k_load = 0, v_load = (C::VRING - 1) * VP_BYTES;      // ring positions: read by the next reads, loaded next
    auto next_k = [](unsigned s) { return s + KP_BYTES < C::KRING * KP_BYTES ? s + KP_BYTES : 0u; };
    auto next_v = [](unsigned s) { return s + VP_BYTES < C::VRING * VP_BYTES ? s + VP_BYTES : 0u; };
    constexpr int NFA = AHEAD + 1 == 2 ? 2 : 4;
    auto read_a = [&](auto gi) __attribute__((always_inline)) {
        constexpr int G = decltype(gi)::value % 16;
        if constexpr (G < 8) lds_read<C::KRING_OFF + 2048 * (G % 4) + 256 * (G / 4)>(fa[G % NFA], frag_lane + k_slot);
        else lds_read<2048 * (G % 8 / 2) + 256 * (G % 2)>(fa[G % NFA], frag_lane + C::VRING_OFF + v_slot);
    };
    auto read_b = [&](auto gi) __attribute__((always_inline)) {
        constexpr int G = decltype(gi)::value % 16;
        if constexpr (G < 8) lds_read<A::DK_OFF + 2048 * (G % 4) + 256 * (G / 4)>(fb[G % 2], frag_lane + k_slot);
        else lds_read<A::DVT_OFF + 2048 * (G % 8 / 2) + 256 * (G % 2)>(fb[G % 2], frag_lane + C::VRING_OFF + v_slot);
    };
    auto product = [&](auto gi, auto ki, auto pause) __attribute__((always_inline)) {
        constexpr bool PAUSE = decltype(pause)::value;
        constexpr int G = decltype(gi)::value, K = decltype(ki)::value / NG, j = decltype(ki)::value % NG;
        if constexpr (G < 8) {
            constexpr int m = G / 4, c = G % 4;
            if constexpr (K == 0) {
                if constexpr (c == 0) M::template first<PAUSE, true>(y[j][m], fa[G % NFA], tb[j][c]);
                else M::template more<PAUSE, true>(y[j][m], fa[G % NFA], tb[j][c]);
            } else if constexpr (K == 1) {
                if constexpr (c == 0) M::template first<PAUSE, false>(x[j][m], fa[G % NFA], qb[j][c]);
                else M::template more<PAUSE, false>(x[j][m], fa[G % NFA], qb[j][c]);
            } else {
                M::template more<PAUSE, false>(y[j][m], fb[G % 2], qb[j][c]);
            }
        } else {
            constexpr int f = G % 8;
            if constexpr (K == 0) M::template sum<PAUSE>(act[f][j], fa[G % NFA], hw[j]);
            else if constexpr (K == 1) M::template sum<PAUSE>(acc[f][j], fa[G % NFA], pw[j]);
            else M::template sum<PAUSE>(act[f][j], fb[G % 2], pw[j]);
        }
    };

    // The sums' products, beside those of a group of outputs: the first behind the check (beside the third 0.7 % slower, tangent on q; spread over three groups as well).  All tangents take 0.8 % longer
    // than with a max that moves at 2^6 and no such sums, tangent on q 0.3 (17600 and 84480 positions, 16 heads, scores of standard deviation 1).
    constexpr int SUMS_AT = 10;
    static_assert(SUMS_AT * PER >= CHECK && SUMS_AT < 15, "sums that have the tile before only behind the check, of H before it is formed anew");
    auto sums = [&](auto ki, auto pause) __attribute__((always_inline)) {
        constexpr int K = decltype(ki)::value;
        if constexpr (K < NG) M::template more<decltype(pause)::value, false>(hsum[K], ones, hw[K]);
        else M::template more<decltype(pause)::value, false>(psum[K - NG], ones, pw[K - NG]);
    };

    // ---- the elements' arithmetic, in single instructions, pairs (r even, odd) numbered [key half][16 rows][r / 2]
    constexpr int PAIRS = 4 * NG;
    float top = -INFINITY;                      // of all arguments of the exponentials of this lane
    // arguments: per pair two products with the scale, one max
    auto arg_op = [&](auto oi) __attribute__((always_inline)) {
        constexpr int O = decltype(oi)::value, P = O / 3, K = O % 3, m = P / (2 * NG), j = P / 2 % NG, r = 2 * (P % 2);
        if constexpr (K < 2) x[j][m][r + K] = __builtin_fmaf(x[j][m][r + K], p.scale_log2, -m_run[j]);
        else { top = __builtin_fmaxf(__builtin_fmaxf(top, x[j][m][r]), x[j][m][r + 1]); landed(top); }      // (kept here: the compiler would form it at the loop's end)
    };
    // P and H: per pair two exponentials, two products with the scale, two products, two sums
    auto exp_op = [&](auto oi) __attribute__((always_inline)) {
        constexpr int O = decltype(oi)::value, P = O / 8, K = O % 8, m = P / (2 * NG), j = P / 2 % NG, r = 2 * (P % 2) + K % 2;
        if constexpr (K < 2) x[j][m][r] = __builtin_amdgcn_exp2f(x[j][m][r]);
        else if constexpr (K < 4) y[j][m][r] *= p.sm_scale;
        else if constexpr (K < 6) y[j][m][r] *= x[j][m][r];
        else l_run[j] += x[j][m][r];
        if constexpr (K == 7) landed(l_run[j]);      // (kept here: the compiler would form the sums at the loop's end)
    };
    // rounding: a pair's word of P or H
    auto round_p = [&](auto pi) __attribute__((always_inline)) {
        constexpr int P = decltype(pi)::value, m = P / (2 * NG), j = P / 2 % NG, r = 2 * (P % 2);
        const V2 two = {(T)x[j][m][r], (T)x[j][m][r + 1]};
        pw[j][2 * m + P % 2] = __builtin_bit_cast(unsigned, two);
    };
    auto round_h = [&](auto pi) __attribute__((always_inline)) {
        constexpr int P = decltype(pi)::value, m = P / (2 * NG), j = P / 2 % NG, r = 2 * (P % 2);
        const V2 two = {(T)y[j][m][r], (T)y[j][m][r + 1]};
        hw[j][2 * m + P % 2] = __builtin_bit_cast(unsigned, two);
    };
    const bool causal = p.causal != 0;
    // masked keys (>= kv_len, or above the diagonal when causal): arguments of -inf, hence P = 0 and H = 0
    auto need_mask = [&](int t) { return t * kBlockN + kBlockN > kv_len || (causal && t * kBlockN + kBlockN - 1 > row0); };
    auto mask = [&](int t) {
        top = -INFINITY;
#pragma unroll
        for (int j = 0; j < NG; ++j) {
            const int row = row0 + 16 * j + l16, end = (causal && row + 1 < kv_len ? row + 1 : kv_len) - t * kBlockN - lane_key(lane);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                x[j][e >> 2][e & 3] = 8 * (e >> 2) + (e & 3) < end ? x[j][e >> 2][e & 3] : -INFINITY;
                top = fmaxf(top, x[j][e >> 2][e & 3]);
            }
        }
    };
    // The max that the exponentials refer to moves to a row's own where an argument of that row is larger than kRowsSlack.  The sums formed already are scaled in fp32: at once those that hold
    // the tile before, the others one step later, when its outputs, of P and H as they were rounded, are among them.
    constexpr int SUMMED = CHECK / PER - 8;     // groups of channels that hold the tile before when the max is looked at
    bool late = false;                          // the others are still to be scaled, by
    float factor[NG];
#pragma unroll
    for (int j = 0; j < NG; ++j) factor[j] = 1.f;
    auto row_top = [&](int j) {
        float v = fmaxf(fmaxf(fmaxf(x[j][0][0], x[j][0][1]), fmaxf(x[j][0][2], x[j][0][3])), fmaxf(fmaxf(x[j][1][0], x[j][1][1]), fmaxf(x[j][1][2], x[j][1][3])));
        v = fmaxf(v, __shfl_xor(v, 16));
        return fmaxf(v, __shfl_xor(v, 32));
    };
    // (through LDS, in which a wavefront's instructions keep their order: accumulation registers go there as they are, and a copy that the compiler makes in this branch would have it keep
    // them elsewhere.  Four results are under way.)
    const unsigned spare = lds0 + C::SPARE_OFF + wave * 4 * kFragBytes + 16 * lane;
    auto scale = [&](auto first, auto end, const float* alpha) __attribute__((always_inline)) {
        constexpr int F0 = decltype(first)::value, N = decltype(end)::value - F0, COUNT = 2 * N * NG;
        f32x4 v[4];
        auto result = [&](auto i) __attribute__((always_inline)) -> f32x4& {
            constexpr int I = decltype(i)::value, f = F0 + I / 2 % N, j = I / (2 * N);
            if constexpr (I % 2) return act[f][j];
            else return acc[f][j];
        };
        auto fetch = [&](auto i) __attribute__((always_inline)) {
            constexpr int I = decltype(i)::value;
            lds_write_acc<I % 4 * kFragBytes>(spare, result(i));
            lds_read<I % 4 * kFragBytes>(v[I % 4], spare);
        };
        for_each<4>(fetch);
        for_each<COUNT>([&](auto i) {
            constexpr int I = decltype(i)::value;
            // LDS instructions behind the fetch of this one: three more fetches, and what the steps since have written and read back
            constexpr int fetched = COUNT - 1 - I < 3 ? COUNT - 1 - I : 3, steps = I < 3 ? I : 3;
            wait_lds<2 * fetched + 2 * steps>();
            landed(v[I % 4]);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[I % 4][r] = alpha[I / (2 * N)] > 0.f ? alpha[I / (2 * N)] * v[I % 4][r] : 0.f;
            lds_write<I % 4 * kFragBytes>(spare, __builtin_bit_cast(rows_u32x4, v[I % 4]));
            lds_read_acc<I % 4 * kFragBytes>(result(i), spare);
            if constexpr (I + 4 < COUNT) fetch(Int<I + 4>{});
        });
        wait_lds<0>();
    };
    auto scale_late = [&]() __attribute__((always_inline)) {
        scale(Int<SUMMED>{}, Int<NF>{}, factor);
#pragma unroll
        for (int j = 0; j < NG; ++j) { psum[j] *= factor[j]; hsum[j] *= factor[j]; }
    };
    auto raise = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NG; ++j) {
            const float top_j = row_top(j), by = top_j > kRowsSlack ? top_j : 0.f, alpha = __builtin_amdgcn_exp2f(-by);
            m_run[j] += by;
            l_run[j] *= alpha;
#pragma unroll
            for (int e = 0; e < 8; ++e) x[j][e >> 2][e & 3] -= by;
            factor[j] = alpha;
        }
        scale(Int<0>{}, Int<SUMMED>{}, factor);
    };

    // ---- what a slot holds beside its product
    constexpr int LOAD_AT = 2;                  // groups at which the two parts are loaded
    constexpr auto fixed = [](int q) {
        q %= SLOTS;
        const int G = q / PER, k = q % PER;
        return (k == 0) + (FULL && k == 1) + (k == PER - 1) + (k == 2 && G == LOAD_AT ? C::K_LOADS : 0) + (k == 2 && G == LOAD_AT + 2 ? C::V_LOADS : 0);
    };
    constexpr auto room = [fixed](int q0, int q) {
        int c = 0;
        for (int i = q0; i < q; ++i) c += fixed(i) < 3 ? 3 - fixed(i) : 0;
        return c;
    };
    constexpr auto share = [room](int n, int q0, int q1, int q) { return q <= q0 ? 0 : q >= q1 ? n : n * room(q0, q) / room(q0, q1); };
    // arguments: of key half 0 behind its products, in the time of half 1's; of half 1 in the first output groups; then the max is looked at
    constexpr int ARG_OPS = 3 * 2 * NG;
    constexpr auto args_before = [share](int q) { return share(ARG_OPS, 4 * PER + NG, 8 * PER, q) + share(ARG_OPS, 8 * PER + NG, CHECK, q); };
    // P and H: of half 0 up to the last output group, of half 1 into the next step's S of half 0
    constexpr int EXP_HALF = 8 * 2 * NG, E0 = CHECK + 1, E1 = SLOTS + 4 * PER - NG;
    constexpr auto exps_before = [room](int q) {
        if (q <= E0) return 0;
        if (q >= E1) return 2 * EXP_HALF;
        const int done = 10 * PAIRS * room(E0, q) / room(E0, E1);              // 2 2 1 1 1 1 1 1 a pair
        const int rest = done % 10;
        return 8 * (done / 10) + (rest < 2 ? 0 : rest < 4 ? 1 : rest - 2);
    };
    static_assert(exps_before(15 * PER + NG) >= EXP_HALF, "the first half is rounded behind its last operand's last use");
    int t_kload = n_tiles_all < 2 ? 0 : tile_at(C::KRING), t_vload = n_tiles_all < 2 ? 0 : tile_at(C::VRING - 1);      // (one tile: one step, whose loads nobody reads)
    auto elements = [&](auto qi) __attribute__((always_inline)) {
        constexpr int Q = decltype(qi)::value;                                  // (of the step's own tile; the next step's slots follow)
        for_each<args_before(Q + 1) - args_before(Q)>([&](auto i) { arg_op(Int<args_before(Q) + decltype(i)::value>{}); });
        for_each<exps_before(Q + 1) - exps_before(Q)>([&](auto i) { exp_op(Int<exps_before(Q) + decltype(i)::value>{}); });
        // half 0: H behind its last use in the last group, P in front of the next S; half 1: in the next S of half 0, when they are formed
        if constexpr (Q >= 15 * PER + NG && Q < 15 * PER + 2 * NG) for_each<2>([&](auto i) { round_h(Int<2 * (Q - 15 * PER - NG) + decltype(i)::value>{}); });
        if constexpr (Q >= SLOTS && Q < SLOTS + NG) for_each<2>([&](auto i) { round_p(Int<2 * (Q - SLOTS) + decltype(i)::value>{}); });
        if constexpr (Q >= SLOTS && Q < SLOTS + 4 * PER) {
            // pairs of half 1 that are complete, one slot later; those complete before this step at NG
            constexpr auto pairs_before = [exps_before](int q) {
                if (q <= SLOTS + NG) return 0;
                if (q >= SLOTS + 4 * PER - 1) return 2 * NG;
                const int e = exps_before(q - 1) / 8 - 2 * NG;
                return e < 0 ? 0 : e;
            };
            for_each<pairs_before(Q + 1) - pairs_before(Q)>([&](auto i) {
                constexpr int P = 2 * NG + pairs_before(Q) + decltype(i)::value;
                round_p(Int<P>{});
                round_h(Int<P>{});
            });
        }
    };
    // LAST: of the last tile, behind which nothing is read ahead (a read whose registers nobody waits for would arrive in whatever they hold by then)
    auto slot = [&](auto qi, auto last) __attribute__((always_inline)) {
        constexpr int Q = decltype(qi)::value, G = Q / PER, K = Q % PER;
        constexpr bool LAST = decltype(last)::value;
        SCHED_FENCE();
        product(Int<G>{}, Int<K>{}, Int<0>{});
        if constexpr (G == SUMS_AT && K < 2 * NG) sums(Int<K>{}, Int<0>{});
        if constexpr (K == 0) {
            if constexpr (G + AHEAD == 16) k_slot = next_k(k_slot);             // the reads go on to the next K, or V
            if constexpr (G + AHEAD == 8) v_slot = next_v(v_slot);
            if constexpr (!LAST || G + AHEAD < 16) read_a(Int<G + AHEAD>{});
        }
        if constexpr (FULL && K == 1 && (!LAST || G < 15)) read_b(Int<G + 1>{});
        if constexpr (K == PER - 1 && (!LAST || G < 15)) {
            wait_lds<LAST ? 0 : AHEAD - 1>();                                   // the next group's operands are here
            landed(fa[(G + 1) % NFA]);
            if constexpr (FULL) landed(fb[(G + 1) % 2]);
        }
        elements(Int<Q>{});                                                     // of this tile
        elements(Int<Q + SLOTS>{});                                             // of the one before
        if constexpr (K == 2 && G == LOAD_AT) { load_k(t_kload, k_load); k_load = next_k(k_load); t_kload = wrap_inc(t_kload); }
        if constexpr (K == 2 && G == LOAD_AT + 2) { load_v(t_vload, v_load); v_load = next_v(v_load); t_vload = wrap_inc(t_vload); }
        SCHED_FENCE();
    };
    // loads (they retire in the order of issue) of the last two steps may be under way: K of the next step's tile and V of the one before are older
    constexpr int NEWER = 2 * (C::K_LOADS + C::V_LOADS);
    // Between the arguments of a tile and its exponentials: masks, and a max that has to move.  The loop turns here: what is rare is not inside of its body.
    auto settle = [&](int t) __attribute__((always_inline)) {
        if (need_mask(t)) mask(t);
        const bool move = __any(top > kRowsSlack);
        if (late || move) {
            asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");       // (products are asm: their results are in the registers now)
            wait_lds<0>();                                            // (and the operands that are read ahead)
            if (late) scale_late();
            if (move) raise();
            late = move;
            asm volatile("s_nop 7" ::: "memory");
        }
        top = -INFINITY;
    };
    // the rest of a step: outputs of the tile before, exponentials of this one
    auto finish = [&](auto last) __attribute__((always_inline)) { for_each<SLOTS - CHECK>([&](auto q) { slot(Int<CHECK + decltype(q)::value>{}, last); }); };
    auto start = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NEWER) : "memory");
        __builtin_amdgcn_s_barrier();          // ... everybody's loads, and everybody is done with the K and V before
        for_each<CHECK>([&](auto q) { slot(q, Int<0>{}); });
    };

    // (the outputs of no tile, with which the first step begins: nothing times the V part that is not loaded yet)
    {
        const unsigned at = lds0 + C::VRING_OFF + (C::VRING - 1) * VP_BYTES + 16 * lane + wave * C::V_LOADS * kFragBytes;
        const rows_u32x4 z = {0, 0, 0, 0};
        for_each<C::V_LOADS>([&](auto i) { lds_write<decltype(i)::value * kFragBytes>(at, z); });
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(3 * C::K_LOADS + 3 * C::V_LOADS) : "memory");       // Q, dQ and K of two tiles are here (the first step reads ahead)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (n > 0) {
        auto group_now = [&](auto gi) __attribute__((always_inline)) {
            read_a(gi);
            if constexpr (FULL) read_b(gi);
            wait_lds<0>();
            landed(fa[decltype(gi)::value % NFA]);
            if constexpr (FULL) landed(fb[decltype(gi)::value % 2]);
            for_each<PER>([&](auto k) { product(gi, k, Int<1>{}); });
        };
        // the first tile: S and its max
        for_each<8>([&](auto gi) { group_now(gi); });
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        int t_cur = tile_at(0);
        if (need_mask(t_cur)) mask(t_cur);
#pragma unroll
        for (int j = 0; j < NG; ++j) m_run[j] = row_top(j) * p.scale_log2;
        top = -INFINITY;
        for_each<2 * ARG_OPS>([&](auto i) { arg_op(i); });
        top = -INFINITY;
        v_slot = (C::VRING - 1) * VP_BYTES;
        for_each<AHEAD>([&](auto i) { read_a(Int<CHECK / PER + decltype(i)::value>{}); });
        if constexpr (FULL) read_b(Int<CHECK / PER>{});
        wait_lds<AHEAD - 1>();
        landed(fa[CHECK / PER % NFA]);
        if constexpr (FULL) landed(fb[CHECK / PER % 2]);
        int s = 1;
#pragma clang loop unroll(disable)
        do {
            finish(Int<0>{});
            start();
            t_cur = wrap_inc(t_cur);
            settle(t_cur);
        } while (++s < n);
        // the last tile (its V may still be under way)
        finish(Int<1>{});
        __builtin_amdgcn_s_waitcnt(0x0070);
        __builtin_amdgcn_s_barrier();
        for_each<CHECK>([&](auto q) { elements(Int<decltype(q)::value + SLOTS>{}); });
        v_slot = next_v(v_slot);
        SCHED_FENCE();
        if (late) {
            asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
            scale_late();
        }
        for_each<8>([&](auto gi) { group_now(Int<8 + decltype(gi)::value>{}); });
        for_each<2 * NG>([&](auto k) { sums(k, Int<1>{}); });
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");      // the last products are in their registers
#pragma unroll
    for (int j = 0; j < NG; ++j) { landed(psum[j]); landed(hsum[j]); }      // (all of them: what nobody reads is nobody else's register before)
    __builtin_amdgcn_s_waitcnt(0x0F70);                     // drain the (unused) trailing loads before the LDS is released

    // ---- epilogue: O = acc / l ; dO = (T - (r / l) acc) / l ; LSE = (m + log2 l) ln 2
#pragma unroll
    for (int j = 0; j < NG; ++j) {
        auto total = [](float v) { v += __shfl_xor(v, 16); return v + __shfl_xor(v, 32); };
        const float l = total(l_run[j]), p_sum = psum[j][0], h_sum = hsum[j][0];
        const int row = row0 + 16 * j + l16;
        if (partial) {   // a key range only: leave accumulators and statistics for attn_combine_kernel
            const int64_t at = ((int64_t)(pair - p.n_full) * p.splits + split) * C::ROWS + wave * 16 * NG + 16 * j + l16;
            if (g == 0) p.part_stat[at] = make_float4(m_run[j], l, h_sum, p_sum);
            float* pa = p.part_acc + at * 256 + 4 * g;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                asm volatile("" : "+a"(acc[f][j]), "+a"(act[f][j]));
                *reinterpret_cast<f32x4*>(pa + 16 * f) = acc[f][j];
                *reinterpret_cast<f32x4*>(pa + 128 + 16 * f) = act[f][j];
                SCHED_FENCE();
            }
        } else if (row < p.Lq) {
            const float inv_l = 1.0f / p_sum, r_over_l = h_sum * inv_l;
            const int64_t off = (int64_t)b * p.o_sb + (int64_t)h * p.o_sh + (int64_t)row * p.o_sl + 4 * g;
            T* op = reinterpret_cast<T*>(p.o) + off;
            T* tp = reinterpret_cast<T*>(p.to) + off;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                asm volatile("" : "+a"(acc[f][j]), "+a"(act[f][j]));
                V4 ov, tv;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    ov[e] = (T)(acc[f][j][e] * inv_l);
                    tv[e] = (T)((act[f][j][e] - r_over_l * acc[f][j][e]) * inv_l);
                }
                *reinterpret_cast<V4*>(op + 16 * f) = ov;
                *reinterpret_cast<V4*>(tp + 16 * f) = tv;
                SCHED_FENCE();
            }
            if (p.lse && g == 0) p.lse[(int64_t)bh * p.Lq + row] = (m_run[j] + __builtin_log2f(l)) * 0.6931471805599453f;
        }
    }
#endif
}
