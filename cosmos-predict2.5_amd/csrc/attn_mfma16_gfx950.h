// The wavefronts of the attention kernels with v_mfma_f32_16x16x32, head dim 128: ScoreWave16 / OutputWave16 for attn_qstream_kernel, SymWave16 for the 384-row
// workgroups of attn_fwd_sym_kernel.  Included inside the anonymous namespace of attn_fwd_jvp_gfx950.hip, behind ScoreWave and OutputWave;
// like these and SymWave (same image of K and V, same rings, hand-over and arithmetic).
//
// Why, and where.  A product is issued in half the cycles, two of them in the place of one v_mfma_f32_32x32x16: the VALU work between them comes in smaller
// pieces, and accumulators are read and written half as often.  It pays where three wavefronts share a SIMD or steps are long, and costs the issue of the second
// product (4 cycles in 32) where that is what bounds.  Measured in turn on one card, us, 32x32x16 / 16x16x32, 16 heads: forward only, 384 rows a workgroup,
// 37440 positions 8832 / 8699 (two runs of one side differ by 1.2 %), 24640 3864 / 3795, 17600 2002 / 1945, 8800 543 / 528, 40 heads 9360 1491 / 1476; stream with all tangents, 512 keys, 37440
// queries 519 / 486, 17600 247 / 231, 8800 139 / 132, 3520 66.7 / 66.6.  Not here, as it was no faster:
// the stream forward only (37440 213 / 222, 8800 61 / 63) and with a tangent on q (338 / 366), attn_fwd_jvp_kernel (37440 25950 / 25750, 17600 5830 / 5820, 704, K and V
// in place, 32.5 / 34.5), forward only with 128 and 256 rows a workgroup (1560 40.2 / 42.1), head dims below 128 (fewer products to a softmax).
//
// Layout.  Lane (i = lane % 16, g = lane / 16) of an operand holds row (or column) i and the contraction's elements 8 g .. 8 g + 7, of a result column i and rows
// 4 g .. 4 g + 3.  S^T = K Q^T of 32 keys x 32 queries is four results, [query half n][key half m]: row i of key half m is key tile_key(i) + 8 m of the tile, column i
// of query half n query 16 n + i.  So a lane holds, of two queries, the eight keys lane_key(lane) + 8 m + r, in this order those of a 16-byte unit of a V^T fragment: as
// the B operand of O^T = V^T P^T, element 4 m + r, P^T needs no shuffle, and a V^T fragment of 16 channels is one ds_read_b128 per lane of the 32-channel fragments of the
// image.  A K fragment (32 channels of a key half) is one as well, at the same lane address: the fills of the K ring put the keys of a half together (k_fill_lane: the runs of
// eight keys 0, 2, 1, 3; as the image has them the two runs of a half would lie in the same banks).
// Statistics of a row exist as the pair a lane uses (queries i, 16 + i) and, for what is done once per row, "by rows": of query lane % 32.

__device__ __forceinline__ int lane_key(int lane) { return 16 * (lane >> 5) + 4 * ((lane >> 4) & 1); }      // = tile_key(4 (lane / 16)): 16 (i / 8) + 4 ((i / 4) % 2) + i % 4
__device__ __forceinline__ int k_fill_lane(int lane) { return (lane & ~24) | ((lane & 8) << 1) | ((lane & 16) >> 1); }
// where this lane reads V^T fragment n (channels 16 n .. + 15, the tile's 32 keys), from the V^T section's start: 2048 (n / 2) + 256 (n % 2) behind this;
// K fragment (32 channels c, key half m), from the K part's start: 2048 c + 256 m behind
__device__ __forceinline__ int frag_offset(int lane) { return 512 * (lane >> 4) + 16 * (lane & 15); }
// this lane's number, found again: a kernel that has no register to keep it in forms it where it is used
__device__ __forceinline__ int lane_again() {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}
// exchanges lanes 16 .. 31 of a with 0 .. 15 of b and 48 .. 63 with 32 .. 47 (written out for the reason given at both_halves)
__device__ __forceinline__ void swap_rows16(float& a, float& b) { asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b)); }
__device__ __forceinline__ float row_max(float a, float b) {      // of the two queries' partial values, by rows
    swap_rows16(a, b);
    float lo, hi;
    both_halves(fmaxf(a, b), lo, hi);
    return fmaxf(lo, hi);
}
__device__ __forceinline__ float row_sum(float a, float b) {
    swap_rows16(a, b);
    float lo, hi;
    both_halves(a + b, lo, hi);
    return lo + hi;
}
__device__ __forceinline__ void of_lane(float x, float* two) {    // by rows -> the two queries of this lane
    two[0] = two[1] = x;
    swap_rows16(two[0], two[1]);
}
// Scores of one tile as a lane sees them, two queries x 8 keys -- the accumulator registers of the score MFMAs: element e = 8 n + 4 m + r
// masked keys (>= kv_len, or above the diagonal when causal) get -inf; key0: the tile's first key, row: of this lane's query of half 0
__device__ __forceinline__ void mask_scores16(f32x4* x, int key0, int lane, int kv_len, bool causal, int row) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int key = key0 + lane_key(lane) + 8 * ((e >> 2) & 1) + (e & 3);
        const bool ok = key < kv_len && (!causal || key <= row + 16 * (e >> 3));
        x[e >> 2][e & 3] = ok ? x[e >> 2][e & 3] : -INFINITY;
    }
}
__device__ __forceinline__ float lane_max16(const f32x4* x, int n) {    // of query half n
    float mx = x[2 * n][0];
#pragma unroll
    for (int e = 1; e < 8; ++e) mx = fmaxf(mx, x[2 * n + (e >> 2)][e & 3]);
    return mx;
}

template <typename T, int MODE>
struct ScoreWave16 {
    typedef AttnCfg<128, 128, MODE> C;
    typedef typename VecOf<T>::v8 V8;
    static constexpr bool JVP = C::JVP, FULL = C::FULL;
    static constexpr int PD = COSMOS_ATTN_PREFETCH_SCORE;    // LDS operand fetches run this many fragments ahead of use
    static constexpr int N = 2, NQ = 4, NF = 8;              // query halves; chunks of 32 channels; K fragments of a tile, (chunk f / 2, key half f % 2)

    struct Scores { f32x4 s[4], ds[4]; };

    V8 qf[N * NQ], tqf[N * NQ];             // [query half][chunk]
    float m_run;                            // running row max, by rows
    float m_lane[2], l_run[2], r_run[2];    // of this lane's two queries: the max, the partial sums over its keys
    float scale_log2, sm_scale;
    int lane;

    __device__ __forceinline__ V8 k_frag(const char* base, int f) const {
        return *reinterpret_cast<const V8*>(base + frag_offset(lane) + 256 * (f & 1) + 2048 * (f >> 1));
    }
    __device__ __forceinline__ void start() {
        m_run = m_lane[0] = m_lane[1] = -INFINITY;
        l_run[0] = l_run[1] = r_run[0] = r_run[1] = 0.f;
    }
    __device__ __forceinline__ float l_total() const { return row_sum(l_run[0], l_run[1]); }     // by rows
    __device__ __forceinline__ float r_total() const { return row_sum(r_run[0], r_run[1]); }
    __device__ __forceinline__ void mask(Scores& x, int key0, int kv_len) const { mask_scores16(x.s, key0, lane, kv_len, false, 0); }

    // Fold a tile's scores into the running max.  Returns the factor, by rows, by which everything accumulated
    // so far must be rescaled before this tile is added (exactly 1 when no row's max moved).
    __device__ __forceinline__ float fold_max(const Scores& x) {
        const float m_new = fmaxf(m_run, row_max(lane_max16(x.s, 0), lane_max16(x.s, 1)) * scale_log2);
        float alpha = 1.0f;
        if (__any(m_new > m_run + max_slack_of<T>(JVP))) {
            alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            float by[2];
            of_lane(alpha, by);
            of_lane(m_new, m_lane);
#pragma unroll
            for (int n = 0; n < 2; ++n) { l_run[n] *= by[n]; r_run[n] *= by[n]; }
        }
        return alpha;
    }

    // ScoreWave::softmax_elem
    __device__ __forceinline__ void softmax_elem(const Scores& x, V8* pf, V8* hf, int e) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(x.s[e >> 2][e & 3], scale_log2, -m_lane[e >> 3]));
        l_run[e >> 3] += p;
        pf[e >> 3][e & 7] = (T)p;
        if (JVP) {
            const float hv = p * (x.ds[e >> 2][e & 3] * sm_scale);
            r_run[e >> 3] += hv;
            hf[e >> 3][e & 7] = (T)hv;
        }
    }
    // one K fragment times the two query halves
    __device__ __forceinline__ static void pair(f32x4* x, V8 a, const V8* b, int f) {
        x[f & 1] = mfma16(a, b[f >> 1], x[f & 1]);
        x[2 + (f & 1)] = mfma16(a, b[NQ + (f >> 1)], x[2 + (f & 1)]);
    }

    // ScoreWave::step; `after_chunk(c)` runs right after the MFMAs of channel chunk c, the last use of the qf / tqf of that chunk in the step
    struct NoHook { __device__ __forceinline__ void operator()(int) const {} };
    template <class F = NoHook>
    __device__ __forceinline__ void step(const Scores& x, Scores& xn, const char* kpart, unsigned ph_out, unsigned alpha_out, float alpha, F after_chunk = F()) {
        V8 pf[2], hf[2], fa[NF], fb[NF];
        asm volatile("ds_write_b32 %0, %1" ::"v"(alpha_out + 4 * lane), "v"(alpha) : "memory");
#pragma unroll
        for (int i = 0; i < PD; ++i) { fa[i] = k_frag(kpart, i); if (FULL) fb[i] = k_frag(kpart + C::DK_OFF, i); }
#pragma unroll
        for (int e = 0; e < 16; ++e) { xn.s[e >> 2][e & 3] = 0.f; xn.ds[e >> 2][e & 3] = 0.f; }
#pragma unroll
        for (int f = 0; f < NF; ++f) {   // two softmax elements per fragment, behind the first and the second product
            SCHED_FENCE();
            if (f + PD < NF) { fa[f + PD] = k_frag(kpart, f + PD); if (FULL) fb[f + PD] = k_frag(kpart + C::DK_OFF, f + PD); }
            SCHED_FENCE();
            if (JVP) pair(xn.ds, fa[f], tqf, f);       // (this order: the two products into ds are not next to each other)
            else pair(xn.s, fa[f], qf, f);
            softmax_elem(x, pf, hf, 2 * f);
            if (!JVP) softmax_elem(x, pf, hf, 2 * f + 1);
            SCHED_FENCE();
            if (JVP) {
                pair(xn.s, fa[f], qf, f);
                softmax_elem(x, pf, hf, 2 * f + 1);
                SCHED_FENCE();
            }
            if (FULL) {
                pair(xn.ds, fb[f], qf, f);
                SCHED_FENCE();
            }
            if (f & 1) after_chunk(f >> 1);
        }
        const unsigned pa = ph_out + 16 * lane;        // (asm stores: see ScoreWave::step)
        asm volatile("ds_write_b128 %0, %1" ::"v"(pa), "v"(pf[0]) : "memory");
        asm volatile("ds_write_b128 %0, %1 offset:1024" ::"v"(pa), "v"(pf[1]) : "memory");
        if (JVP) {
            asm volatile("ds_write_b128 %0, %1 offset:2048" ::"v"(pa), "v"(hf[0]) : "memory");
            asm volatile("ds_write_b128 %0, %1 offset:3072" ::"v"(pa), "v"(hf[1]) : "memory");
        }
    }
    __device__ __forceinline__ void scores_plain(Scores& x, const char* kpart) const {
#pragma unroll
        for (int e = 0; e < 16; ++e) { x.s[e >> 2][e & 3] = 0.f; x.ds[e >> 2][e & 3] = 0.f; }
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            const V8 kf = k_frag(kpart, f);
            if (JVP) pair(x.ds, kf, tqf, f);
            pair(x.s, kf, qf, f);
            if (FULL) pair(x.ds, k_frag(kpart + C::DK_OFF, f), qf, f);
        }
    }
};

template <typename T, int MODE>
struct OutputWave16 {
    typedef AttnCfg<128, 128, MODE> C;
    typedef typename VecOf<T>::v8 V8;
    static constexpr bool JVP = C::JVP, FULL = C::FULL;
    static constexpr int N = 2, NB = 8;      // query halves; groups of 16 channels
    static constexpr int PD = COSMOS_ATTN_PREFETCH_OUTPUT;

    f32x4 acc[NB][N], acct[NB][N];           // channels 16 g + 4 (lane / 16) + r of query 16 n + lane % 16
    int lane;

    __device__ __forceinline__ f32x4 acc4(int g, int n) const { return acc[g][n]; }
    __device__ __forceinline__ f32x4 acct4(int g, int n) const { return acct[g][n]; }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < NB; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) { acc[i][e >> 2][e & 3] = 0.f; acct[i][e >> 2][e & 3] = 0.f; }
        }
    }
    __device__ __forceinline__ void fetch_group(int g, const char* vpart, V8& a, V8& b) const {
        const char* at = vpart + frag_offset(lane) + 2048 * (g >> 1) + 256 * (g & 1);
        a = *reinterpret_cast<const V8*>(at);
        if (FULL) b = *reinterpret_cast<const V8*>(at + C::DVT_OFF);
    }
    __device__ __forceinline__ static void pair(f32x4* x, V8 a, const V8* b) {
        x[0] = mfma16(a, b[0], x[0]);
        x[1] = mfma16(a, b[1], x[1]);
    }
    // OutputWave::step
    __device__ __forceinline__ void step(const char* vpart, const char* ph_in, const char* alpha_in) {
        float alpha[N];
        V8 pf[2], hf[2], fa[NB], fb[NB];
#pragma unroll
        for (int n = 0; n < N; ++n) {
            alpha[n] = *reinterpret_cast<const float*>(alpha_in + 64 * n + 4 * (lane & 15));
            pf[n] = *reinterpret_cast<const V8*>(ph_in + n * kFragBytes + lane * 16);
            if (JVP) hf[n] = *reinterpret_cast<const V8*>(ph_in + (2 + n) * kFragBytes + lane * 16);
        }
#pragma unroll
        for (int i = 0; i < PD; ++i) fetch_group(i, vpart, fa[i], fb[i]);
        if (__any(alpha[0] != 1.0f || alpha[1] != 1.0f)) {   // (v_mul_legacy_f32: see OutputWave::step)
#pragma unroll
            for (int i = 0; i < NB; ++i) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    asm("v_mul_legacy_f32 %0, %1, %2" : "=v"(acc[i][e >> 2][e & 3]) : "v"(alpha[e >> 2]), "v"(acc[i][e >> 2][e & 3]));
                    if (JVP) asm("v_mul_legacy_f32 %0, %1, %2" : "=v"(acct[i][e >> 2][e & 3]) : "v"(alpha[e >> 2]), "v"(acct[i][e >> 2][e & 3]));
                }
            }
        }
#pragma unroll
        for (int g = 0; g < NB; ++g) {
            SCHED_FENCE();
            if (g + PD < NB) fetch_group(g + PD, vpart, fa[g + PD], fb[g + PD]);
            SCHED_FENCE();
            if (JVP) pair(acct[g], fa[g], hf);         // (this order: the two products into acct are not next to each other)
            pair(acc[g], fa[g], pf);
            if (FULL) pair(acct[g], fb[g], pf);
        }
        SCHED_FENCE();
    }
};

// (registers: 164 of the 168 that three wavefronts per SIMD leave; a lane's number is formed again where it is used)
template <typename T>
struct SymWave16 {
    typedef typename VecOf<T>::v8 V8;
    typedef T V2 __attribute__((ext_vector_type(2)));
    static constexpr int N = 2, NQ = 4, NF = 8;          // query halves; chunks of 32 channels; K fragments of a tile, (chunk f / 2, key half f % 2)
    static constexpr int NB = 8;                         // P.V MFMA groups of a tile: 16 channels each
    static constexpr int PD = COSMOS_ATTN_PREFETCH_GROUPS;

    struct Scores { f32x4 s[4]; };
    V8 qf[N * NQ];                          // [query half][chunk]
    f32x4 acc[NB][2];                       // [16 channels][query half]: channels 16 g + 4 (lane / 16) + r
    float m_lane[2], l_run[2], scale_log2;  // of this lane's two queries: running max, row sums (this lane's keys)
    float l_tile[2];                        // the current tile's share of the row sums
    float p_even;
    uint32_t pw[8];                         // P^T of the current tile, two values each (B operand of query half n: words 4 n .. + 3)
    int frag_lane;                          // frag_offset
    __device__ __forceinline__ void start(int lane) {
        frag_lane = frag_offset(lane);
        m_lane[0] = m_lane[1] = -INFINITY;
        l_run[0] = l_run[1] = l_tile[0] = l_tile[1] = 0.f;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[i][e >> 2][e & 3] = 0.f;
        }
    }
    __device__ __forceinline__ f32x4 acc4(int g, int n) const { return acc[g][n]; }
    __device__ __forceinline__ float l_total() const { return row_sum(l_run[0], l_run[1]); }                    // by rows
    __device__ __forceinline__ float m_total() const { return lane_again() & 16 ? m_lane[1] : m_lane[0]; }
    __device__ __forceinline__ static void of_rows(float x, float* two) { of_lane(x, two); }
    __device__ __forceinline__ static void mask(Scores& x, int key0, int kv_len, bool causal, int row0) {
        const int l = lane_again();
        mask_scores16(x.s, key0, l, kv_len, causal, row0 + (l & 15));
    }
    __device__ __forceinline__ V8 k_frag(const char* base, int f) const {
        return *reinterpret_cast<const V8*>(base + frag_lane + 256 * (f & 1) + 2048 * (f >> 1));
    }
    __device__ __forceinline__ V8 vt_frag(const char* base, int g) const {
        return *reinterpret_cast<const V8*>(base + frag_lane + 2048 * (g >> 1) + 256 * (g & 1));
    }
    __device__ __forceinline__ void score_pair(Scores& x, V8 a, int f) const {
        x.s[f & 1] = mfma16(a, qf[f >> 1], x.s[f & 1]);
        x.s[2 + (f & 1)] = mfma16(a, qf[NQ + (f >> 1)], x.s[2 + (f & 1)]);
    }
    __device__ __forceinline__ void out_pair(int g, V8 a, const V8* pf) {
        acc[g][0] = mfma16(a, pf[0], acc[g][0]);
        acc[g][1] = mfma16(a, pf[1], acc[g][1]);
    }
    // Move the running max up to a tile's scores; alpha: the rescale factors of everything accumulated so far.
    __device__ __forceinline__ void raise_max(const Scores& x, float* alpha) {
        float m_new[2];
        of_lane(row_max(lane_max16(x.s, 0) * scale_log2, lane_max16(x.s, 1) * scale_log2), m_new);
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            m_new[n] = fmaxf(m_lane[n], m_new[n]);
            alpha[n] = __builtin_amdgcn_exp2f(m_lane[n] - m_new[n]);
            m_lane[n] = m_new[n];
        }
    }
    __device__ __forceinline__ void scores_plain(Scores& x, const char* kpart) const {
#pragma unroll
        for (int e = 0; e < 16; ++e) x.s[e >> 2][e & 3] = 0.f;
#pragma unroll
        for (int f = 0; f < NF; ++f) score_pair(x, k_frag(kpart, f), f);
    }
    __device__ __forceinline__ void first_max(const Scores& x) {
        float alpha[2];
        raise_max(x, alpha);
    }
    // SymWave::softmax_elems
    __device__ __forceinline__ void softmax_elems(const Scores& x, int e0, int n) {
#pragma unroll
        for (int k = 0; k < n; ++k) {
            const int e = e0 + k;
            const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(x.s[e >> 2][e & 3], scale_log2, -m_lane[e >> 3]));
            if (e & 1) {
                float& sum = l_tile[e >> 3];
                sum += p_even;                   // (an instruction between the exponential and its first use)
                asm volatile("" : "+v"(sum));
                const V2 both = {(T)p_even, (T)p};
                pw[e >> 1] = __builtin_bit_cast(uint32_t, both);
                sum += p;
                asm volatile("" : "+v"(pw[e >> 1]), "+v"(sum));
            } else {
                p_even = p;
                asm volatile("" : "+v"(p_even));
            }
        }
    }

    // SymWave::tile_step
    template <class Mask>
    __device__ __forceinline__ void tile_step(const Scores& x, Scores& xn, const char* kpart, const char* vpart, int t_next, Mask mask) {
        V8 fa[NF];
#pragma unroll
        for (int i = 0; i < PD; ++i) fa[i] = k_frag(kpart, i);
#pragma unroll
        for (int e = 0; e < 16; ++e) xn.s[e >> 2][e & 3] = 0.f;
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            SCHED_FENCE();
            if (f + PD < NF) fa[f + PD] = k_frag(kpart, f + PD);
            SCHED_FENCE();
            score_pair(xn, fa[f], f);
            softmax_elems(x, 8 + f, 1);
        }
        SCHED_FENCE();
        V8 pf[2], fv[NB];
#pragma unroll
        for (int i = 0; i < PD; ++i) fv[i] = vt_frag(vpart, i);
        if (__any(!(l_tile[0] + l_tile[1] <= kMaxTileSum))) {
            float alpha[2];
            raise_max(x, alpha);
#pragma unroll
            for (int n = 0; n < 2; ++n) { l_run[n] *= alpha[n]; l_tile[n] = 0.f; }
#pragma unroll
            for (int i = 0; i < NB; ++i) {
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    acc[i][n] *= alpha[n];
                    asm volatile("" : "+v"(acc[i][n]));
                }
            }
            softmax_elems(x, 0, 16);
        }
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            l_run[n] += l_tile[n];
            l_tile[n] = 0.f;
            pf[n] = __builtin_bit_cast(V8, make_uint4(pw[4 * n], pw[4 * n + 1], pw[4 * n + 2], pw[4 * n + 3]));
        }
        mask(xn, t_next);
#pragma unroll
        for (int g = 0; g < NB; ++g) {
            SCHED_FENCE();
            if (g + PD < NB) fv[g + PD] = vt_frag(vpart, g + PD);
            SCHED_FENCE();
            out_pair(g, fv[g], pf);
            softmax_elems(xn, g, 1);
        }
        SCHED_FENCE();
    }
};

