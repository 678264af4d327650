// Pieces shared by the gfx950 attention kernels (forward + JVP, backward): vector types, the MFMA wrapper, the
// 1 KB operand-fragment constant, direct-to-LDS loads.  Included inside each translation unit's anonymous namespace.
#ifndef COSMOS_ATTN_COMMON_GFX950_H
#define COSMOS_ATTN_COMMON_GFX950_H

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

// f(Int<0>{}) ... f(Int<N - 1>{})
template <int I> struct Int { static constexpr int value = I; };
template <typename F, int... I> __device__ __forceinline__ void for_each_of(F&& f, std::integer_sequence<int, I...>) { (f(Int<I>{}), ...); }
template <int N, typename F> __device__ __forceinline__ void for_each(F&& f) { for_each_of(f, std::make_integer_sequence<int, N>{}); }

template <typename T> struct VecOf;
template <> struct VecOf<__bf16> { typedef bf16x8 v8; typedef bf16x4 v4; };
template <> struct VecOf<_Float16> { typedef f16x8 v8; typedef f16x4 v4; };

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(f16x8 a, f16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// A value that exists once per 32-lane half of a wavefront, made visible to both halves: afterwards, in every lane l,
// `lo` is what lane l % 32 held and `hi` what lane 32 + l % 32 held (one v_permlane32_swap, no LDS round trip).  The
// instruction is written out: given one value for both of its operands, the compiler's builtin treats its two results as
// equal and drops one of them.  (s_nop: the instruction may not directly follow the VALU write of its operands.)
__device__ __forceinline__ void both_halves(float x, float& lo, float& hi) {
    unsigned a = __builtin_bit_cast(unsigned, x), b = a;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    lo = __builtin_bit_cast(float, a);
    hi = __builtin_bit_cast(float, b);
}

constexpr int kFragBytes = 1024;   // one MFMA A-operand fragment: 64 lanes x 16 B
// The running row max that the softmax exponentials refer to is allowed to lag the true one.  In the kernels with a score role
// (attn_fwd_jvp_kernel, attn_qstream_kernel) it moves (and everything
// summed so far is rescaled) only when some row of the wavefront has a score more than kMaxSlack above it, in log2
// units, so p = exp2(s c - m) stays below 2^kMaxSlack.  O = sum p v / sum p and LSE = m + log2 sum p hold for any
// reference m, and 16-bit rounding of p is relative, so nothing is lost; what is gained is that the rescaling pass over
// the accumulators, which otherwise runs in nearly every one of a sweep's first dozens of steps (in every step of a short
// sweep), runs about once per sweep.
// (attn_jvp_rows_kernel: kRowsSlack.)
constexpr float kMaxSlack = 6.0f;
// attn_fwd_sym_kernel reads whether the max has to move off the row sums instead: a lane's sum of the exponentials of its 16 keys of a tile is
// at least its largest one, and is formed anyway.  A tile whose lane sums all stay within 2^kMaxSlack is done; otherwise (or if a sum is no
// number) the max moves up to the tile's scores and the tile's softmax is done again from them.  That is the same bound on p; the max moves
// earlier (sixteen scores 2 above it do), never later.  A max over the scores before the exponentials (10 dependent instructions and the wait
// for the last score MFMA in front of them) costs that kernel 4 to 5 %.
constexpr float kMaxTileSum = (float)(1 << (int)kMaxSlack);
// With tangents H = p dS s is rounded to the 16-bit type as well, and fp16 has the range for |dS s| up to 65504 only while
// p <= 1 (the reference's range, flash_attention_jvp_triton.py:114,141); a p of up to 2^6 would overflow from |dS s| ~ 1e3 on.
// So fp16 with tangents keeps the exact running max; bf16 (8 exponent bits) and the forward-only mode of attn_qstream_kernel use the slack.
template <typename T>
__device__ __host__ constexpr float max_slack_of(bool with_tangents) {
    return (with_tangents && __is_same(T, _Float16)) ? 0.0f : kMaxSlack;
}
#ifndef COSMOS_ATTN_PREFETCH_GROUPS
#define COSMOS_ATTN_PREFETCH_GROUPS 2   // LDS operand fetches run this many MFMA groups ahead of use
#endif
// The forward + JVP kernels' two roles have depths of their own.  The output wavefront runs 6 groups ahead (measured at the
// 2B 720p shape, score / output depth: 2/2 137-138 ms, 4/4 134.6-135, 2/6 133.3, 2/8 133.6, 4/8 134.5): it has the
// registers for it, and its MFMAs are what fills the gaps the score wavefront leaves in the pipe.
#ifndef COSMOS_ATTN_PREFETCH_SCORE
#define COSMOS_ATTN_PREFETCH_SCORE 2
#endif
#ifndef COSMOS_ATTN_PREFETCH_OUTPUT
#define COSMOS_ATTN_PREFETCH_OUTPUT 6
#endif
#ifndef COSMOS_ATTN_SWEEP_STAGGER
#define COSMOS_ATTN_SWEEP_STAGGER 3   // tiles between the sweep starts of workgroups that share an L2 (measured at the 2B 720p
                                      // shape: same time for 1 .. 4; traffic past the L2 56 / 48 / 36-38 / 26 / 26 / 82 GB at 0 / 1 / 2 / 3 / 4 / 6)
#endif

#define SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)

// What one wavefront copies per step (one "load group"): its share of the V part of one tile and of the K part
// of another, as VP_LOADS + KP_LOADS wavefront-level direct-to-LDS loads.  buffer_load ... lds (MUBUF) rather than
// global_load_lds: the compiler's wait-count pass treats the latter as a FLAT access that may touch LDS and then
// turns every later LDS wait into lgkmcnt(0).  One wavefront-level load moves one fragment: lane l's 16 bytes
// (voffset = 16 l) land at dst + 16 l.  The share is a contiguous run of fragments (parts with fewer fragments
// than wavefronts are copied redundantly), so one LDS base (M0) and one scalar offset serve the whole run and the
// fragment index travels in the instruction's immediate offset, which is added to both addresses.
struct LoadJob {
    __amdgpu_buffer_rsrc_t rsrc;
    int lane_off, k_lane_off;   // 16 * lane; for K parts 16 * the lane whose unit this one copies
    int k_src, v_src;        // byte offsets of this wavefront's runs in the packed buffer
    char *k_dst, *v_dst;     // LDS destinations of the runs
};
template <int IMM, int AUX = 0>   // AUX: cache policy bits of the instruction (2 = non-temporal)
__device__ __forceinline__ void lds_load(__amdgpu_buffer_rsrc_t rsrc, char* dst, int lane_off, int src) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)dst, 16, lane_off, src, IMM, AUX);
}
template <int LOADS>
__device__ __forceinline__ void issue_part(__amdgpu_buffer_rsrc_t rsrc, char* dst, int lane_off, int src) {
    lds_load<0>(rsrc, dst, lane_off, src);
    if (LOADS > 1) lds_load<kFragBytes>(rsrc, dst, lane_off, src);
    if (LOADS > 2) lds_load<2 * kFragBytes>(rsrc, dst, lane_off, src);
    if (LOADS > 3) lds_load<3 * kFragBytes>(rsrc, dst, lane_off, src);
}

// ---- K and V read where they are (head dim 128): no re-tiling pass in front of a short call.
// Parts of 32 keys in LDS, every load a run of whole 128-byte lines (a load whose lanes take 32 bytes of each of 32 rows, which would make the fragment order of the
// re-tiled image, runs at half of the rate and costs a step 8 %):
//   K: two halves of 32 rows x 128 bytes, 16-byte chunk c of row r at c XOR (r / 2) % 8: a K-type fragment is one ds_read_b128 per lane, from one of four lane addresses;
//   V: 32 rows x 256 bytes, chunk c of row r at c XOR 4 (r % 4): a V^T fragment is two ds_read_b64_tr_b16 (within 16 lanes, lane i passes the address of 8 bytes, row
//   i of a 16 x 4 matrix M, and receives M[i/4 + 4k][i%4], k = 0..3).
// Neither has bank conflicts.
typedef unsigned raw_u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned raw_u32x4 __attribute__((ext_vector_type(4)));
constexpr int kRawRow = 256;                     // bytes of a row
struct RawFill {
    __amdgpu_buffer_rsrc_t rsrc;                 // one (batch, head)'s rows: bytes behind the last row read as zeros
    int row_bytes;                               // between rows
    __device__ __forceinline__ RawFill(const void* head, int64_t row_stride, int rows)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(head), 0, (int)((rows - 1) * row_stride * 2) + kRawRow, 0x00020000)), row_bytes((int)row_stride * 2) {}
    // K: the 1 KB blocks q .. q + N - 1 (half q / 4, rows 8 (q % 4) .. + 7) of the 32 keys from row `key` on
    template <int N> __device__ __forceinline__ void k(char* dst, int key, int q, int lane) const {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int half = (q + i) >> 2, r8 = (q + i) & 3;
            const int off = (key + 8 * r8 + (lane >> 3)) * row_bytes + half * 128 + (((lane & 7) ^ (4 * (r8 & 1) + (lane >> 4))) << 4);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(dst + i * kFragBytes), 16, off, 0, 0, 0);
        }
    }
    // V: 4 N rows from row `key` on
    template <int N> __device__ __forceinline__ void v(char* dst, int key, int lane) const {
        const int off = (key + (lane >> 4)) * row_bytes + (((lane & 15) ^ (4 * ((lane >> 4) & 3))) << 4);
#pragma unroll
        for (int i = 0; i < N; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(dst + i * kFragBytes), 16, off + 4 * i * row_bytes, 0, 0, 0);
    }
};
// where this lane reads K-type fragment c % 4 of a K part's first half; that of the second half (c >= 4) lies 4096 behind
__device__ __forceinline__ int raw_k_offset(int c, int lane) {
    const int row = lane & 31;
    return row * 128 + (((2 * c + (lane >> 5)) ^ ((row >> 1) & 7)) << 4);
}
// where this lane reads V^T fragment (db, 0) of a V part, from the part's start; fragment (db, c) lies 4096 c behind, its second half of keys 2048
__device__ __forceinline__ unsigned raw_vt_offset(int db, int lane) {
    const int i = lane & 15, key = 4 * (lane >> 5) + (i >> 2), chunk = 4 * db + 2 * ((lane >> 4) & 1) + ((i & 3) >> 1);
    return (unsigned)(key * kRawRow + ((chunk ^ (4 * (i >> 2))) << 4) + 8 * (i & 1));
}
// a fragment on its way: valid behind a wait, made so by landed()
struct RawVt {
    raw_u32x2 lo, hi;
    template <int OFF> __device__ __forceinline__ void read(unsigned a) {
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(a), "n"(OFF));
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(a), "n"(OFF + 8 * kRawRow));
    }
    __device__ __forceinline__ void landed() { asm volatile("" : "+v"(lo), "+v"(hi)); }
    template <typename V8> __device__ __forceinline__ V8 get() const { return __builtin_bit_cast(V8, raw_u32x4{lo.x, lo.y, hi.x, hi.y}); }
};
template <int N> __device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory"); }

// Four units of a V^T-type section (channels 4 quad .. + 3, key chunk c, lane half hh of the 32-key tile at row key0): eight 8-byte
// loads, one per key, of which 32 neighbouring threads cover whole rows of 128 channels, transposed in registers into four 16-byte
// stores side by side.  Channels past `width` and rows past `rows` become zeros.
__device__ __forceinline__ void transpose_units(const uint16_t* head, int64_t row_stride, int key0, int rows, int width, int quad, int c, int hh, uint4* section) {
    const int d = 4 * quad;
    uint2 r[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const int key = key0 + 16 * c + 8 * (s >> 2) + 4 * hh + (s & 3);
        r[s] = key < rows && d < width ? *reinterpret_cast<const uint2*>(head + (int64_t)key * row_stride + d) : make_uint2(0u, 0u);
    }
    uint4* dst = section + (2 * (d >> 5) + c) * (kFragBytes / 16) + 32 * hh + (d & 31);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t a = j < 2 ? r[2 * i].x : r[2 * i].y, b = j < 2 ? r[2 * i + 1].x : r[2 * i + 1].y;
            w[i] = j & 1 ? (a >> 16) | (b & 0xFFFF0000u) : (a & 0xFFFFu) | (b << 16);
        }
        dst[j] = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// hipFuncSetAttribute(MaxDynamicSharedMemorySize) once per (device, kernel).  A kernel's LDS size is a compile-time
// constant of its instantiation, so the call never needs repeating; keeping it out of the steady state also keeps
// the entry points usable while a stream is being captured into a graph.  (Needs <mutex>, <set>, <utility>.)
inline bool allow_lds(const void* fn, size_t bytes) {
    static std::mutex mu;
    static std::set<std::pair<int, const void*>> done;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) { (void)hipGetLastError(); return false; }
    std::lock_guard<std::mutex> lock(mu);
    if (done.count(std::make_pair(dev, fn))) return true;
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    done.insert(std::make_pair(dev, fn));
    return true;
}

// One workgroup of the attention kernels fits on a compute unit, so a launch of n_pairs equal workgroups runs in rounds
// of kNumCUs and a partly filled last round costs a whole one.  The `rem` workgroups of that round may instead be cut
// into S ranges of their stream (keys or queries) each: rem * S shorter workgroups, plus a merge kernel.  Returns the S
// (1 = leave it) of the least cost in microseconds, where
//   * a round of workgroups takes `steps` barrier steps of step_us each and range_us to start and end;
//   * the step of a round that fills only a part of the chip is faster, as the part then clocks higher under its power limit:
//     `alone` (0.7 at head dim 128) of the full chip's time for a few workgroups, growing with the square of the filled part
//     (forward only, 384-row steps: 1.74 us for a few workgroups, 2.42 in full rounds);
//     smaller head dims draw less power: 0.9;
//   * every range leaves slot_bytes of partial results, written once and read once by the merge kernel: 3.8 MB of them cost a
//     microsecond, the merge kernel's launch three.
// The constants are fits to B*H = 16 .. 80, 255 .. 17600 positions and S = 1 .. 16, every S measured (the forward's at head dims 16 .. 128
// each, beside kSymShapes and plan_split; the backward's step at 128, taken down with the head dim: at 16 .. 64, B*H = 16 and 40, 700 .. 9000 positions, its
// choice takes 1.014 times the best S on average, 1.11 at most).  What the rule that
// counted rounds alone chose, and this one (us, forward + tangents unless said, head dim 128, with the re-tiling):
//   1 x 16 x 1560: S = 11 243, S = 1 77;   1 x 40 x 512: S = 3 64, S = 1 40;   1 x 16 x 7040: S = 16 1093, S = 2 1012;
//   backward 1 x 16 x 1560: S = 11 267, S = 1 113.
// The cost of a split has to come out at least a twentieth lower: the fits are no better than that.
constexpr int kNumCUs = 256;          // MI355X
constexpr int kMaxSplits = 16;
constexpr int kMinStepsPerSplit = 4;
struct StepCost { double step_us, range_us, alone = 0.7; };   // a barrier step in full rounds, and what a workgroup costs besides its steps
// `pairs` workgroups of n_steps / S steps each, in rounds
inline double rounds_cost(int64_t pairs, double n_steps, StepCost c) {
    if (pairs <= 0) return 0.0;
    const int64_t rounds = (pairs + kNumCUs - 1) / kNumCUs;
    const double filled = (double)pairs / (double)(rounds * kNumCUs);
    return (double)rounds * (n_steps * c.step_us * (c.alone + (1.0 - c.alone) * filled * filled) + c.range_us);
}
// Causal calls: workgroups of unequal length.  They go out by id, to the 8 dies in turn and inside of a die to its 4 shader engines in turn, and one whose engine has none of its 8 units free holds
// up the die's others.  So with 32 .. 36 blocks a head an engine gets the long ones of every head, and both sizes of workgroups take a quarter longer there than their work says.  The time of the
// later of two dies, one of which has workgroup `first`, the longest.  (Up to kCausalPairs workgroups.)
constexpr int kNumDies = 8, kCausalPairs = 16 * kNumCUs;
template <typename F> inline double causal_cost(int64_t first, int64_t pairs, F us_of) {
    constexpr int kEngines = 4, kUnits = kNumCUs / kNumDies / kEngines;
    double end = 0.0;
    for (int64_t die = first; die <= first + 2; die += 2) {
        double free_at[kEngines][kUnits] = {}, now = 0.0;          // heaps: the unit that is free first is [0]
        int engine = 0;
        for (int64_t i = die % kNumDies; i < pairs; i += kNumDies, engine = (engine + 1) % kEngines) {
            double* const unit = free_at[engine];
            now = unit[0] > now ? unit[0] : now;
            const double t = now + us_of(i);
            end = t > end ? t : end;
            int at = 0;
            for (int next = 1; next < kUnits; next = 2 * at + 1) {
                if (next + 1 < kUnits && unit[next + 1] < unit[next]) ++next;
                if (unit[next] >= t) break;
                unit[at] = unit[next];
                at = next;
            }
            unit[at] = t;
        }
    }
    return end;
}
// a value measured at head dims 16, 32, 64 and 128, and on the line between two of them for calls of unequal head dims
inline double by_head_dim(const double (&at)[4], double d) {
    const int i = d > 64.0 ? 2 : d > 32.0 ? 1 : 0;
    const double lo = (double)(16 << i);
    return at[i] + (at[i + 1] - at[i]) * (d - lo) / lo;
}
inline double split_cost(int rem, int n_steps, int S, StepCost c, double slot_bytes) {
    return rounds_cost((int64_t)rem * S, (double)n_steps / S, c) + (S > 1 ? 3.0 + (double)rem * S * slot_bytes / 3.8e6 : 0.0);
}
inline int choose_splits(int rem, int n_steps, StepCost c, double slot_bytes, int most = kMaxSplits) {
    if (rem <= 0) return 1;
    int best = 1;
    double best_cost = 0.95 * split_cost(rem, n_steps, 1, c, slot_bytes);
    for (int S = 2; S <= most && S * kMinStepsPerSplit <= n_steps; ++S) {
        const double cost = split_cost(rem, n_steps, S, c, slot_bytes);
        if (cost < best_cost) { best_cost = cost; best = S; }
    }
    return best;
}

// The workgroup-to-XCD maps and the rounds-of-kNumCUs arithmetic of the attention kernels assume a whole MI355X (256 compute
// units).  A partitioned device (CPX / DPX modes) reports fewer and would silently get wrong piece maps: looked up once per
// device ordinal, refused with a status code.  (Needs <mutex>.)
inline bool device_is_whole_mi355x() {
    static std::mutex mu;
    static signed char state[64] = {};   // 0 = not looked up, 1 = yes, -1 = no
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) { (void)hipGetLastError(); return false; }
    std::lock_guard<std::mutex> lock(mu);
    if (state[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) { (void)hipGetLastError(); return false; }
        state[dev] = n == kNumCUs ? 1 : -1;
    }
    return state[dev] == 1;
}

inline bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }
inline bool strides_ok(const int64_t* s) { return s[0] % 8 == 0 && s[1] % 8 == 0 && s[2] % 8 == 0; }
inline bool head_dim_ok(int d) { return d == 16 || d == 32 || d == 64 || d == 128; }

#endif
