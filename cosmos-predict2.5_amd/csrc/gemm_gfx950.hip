// Matrix products of the linear layers for gfx950: out[rows, cols] = A B on 16-bit operands with fp32 accumulation, in the three
// orders that a layer and its backward pass need (y = x w^T, dx = dy w, dw = dy^T x), up to three products of one shape in a launch
// (the q, k and v projections) or summed into one output (their gradient of x).  C ABI in include/cosmos_attn_hip.h.
//
// What bounds it and what was chosen.  A product of this size is bound by the matrix units under the part's power limit (a large one of
// the vendor library runs at 1.55 PFLOP/s with random operands), a small one by how its tiles divide over 256 compute units.
//   * v_mfma_f32_16x16x32: 1.75 PFLOP/s sustained where the 32x32x16 shape is throttled to 1.33.
//   * Four wavefronts per workgroup, one per SIMD, each with a quarter of the tile: at 256 x 256 its 128 x 128 outputs are all 256
//     accumulation registers, and a 1 KB operand fragment read from LDS feeds eight MFMAs.  (Eight wavefronts of half that: the same time,
//     1.5 times the LDS traffic.)
//   * A wavefront that has its SIMD to itself pays for every instruction that it has to wait for, so the loop is written in slots: an
//     MFMA, at most one LDS read and one direct-to-LDS load each, one half step of operands ahead (LDS reads) and 1.3 to 2 steps ahead (loads).
//     The MFMAs, reads and loads are asm so that neither order nor waits are the compiler's.  Spreading the loads evenly over a step is worth 6 %
//     (in bursts the load path, 64 bytes a clock, is full and the next MFMA waits behind it in program order), taking the address arithmetic
//     out from between the MFMAs another 4 %.
//   * LDS rings of 64-deep steps: at 256 x 256 two stages of A and three of B are exactly the 160 KB.
//   * Both kinds of operand go through the same loop: rows that run along the contraction are read with ds_read_b128, rows that run along the
//     output with the transposing ds_read_b64_tr_b16, so that dx and dw cost what y costs (the library's orders: 1.57 / 1.39 / 1.19 PFLOP/s
//     at 8192^3, these 1.53 / 1.55 / 1.53).  The 16-byte chunks of a row are stored XOR-swizzled (the load's lanes pick their source): no bank conflicts.
//   * Persistent workgroups: the loads run over tile boundaries, so that only a workgroup's first tile waits for memory.  An XCD serves a
//     contiguous run of tiles, 8 rows of tiles high, so that its L2 holds the panels that its compute units share.
// Measured, us, library -> this, bf16 (rows x cols x depth): 37440 x 2048 x 2048 y 287 -> 225, dx 290 -> 230;
// 37440 x 8192 x 2048 931 -> 874, 1127 -> 912, 1042 -> 827; 10920 x 2048 x 2048 78 -> 76, 87 -> 78, 121 -> 84; 3520 x 2048 x 2048 34 -> 30, 36 -> 31.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <set>
#include <utility>

#include "cosmos_attn_hip.h"

namespace {
#include "attn_common_gfx950.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

constexpr int kStep = 64;            // contraction indexes per step
constexpr int kTileGroup = 8;        // rows of tiles that are served together
constexpr int kMostProducts = 3;

struct GemmParams {
    const uint16_t *a[kMostProducts], *b[kMostProducts];
    uint16_t* c[kMostProducts];
    int64_t lda, ldb, ldc;           // elements
    int rows, cols, depth;
    int segments;                    // products that are summed into one output; 1: every product has its own
    int tiles_r, tiles_c;            // of one product
    int tiles, items;                // tiles of one product; of all that have an output of their own
    int steps;                       // of one product
    int group;                       // tiles of a full group
    unsigned m_group, m_last;        // ceil(2^32 / d) of the divisions in place()
};

template <int OFF> __device__ __forceinline__ u32x4 ds_b128(unsigned a) {
    u32x4 r;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(a), "n"(OFF));
    return r;
}
// within 16 lanes, lane j passes the address of 8 bytes, row j of a 16 x 4 matrix M of 16-bit values, and lane i receives M[i/4 + 4k][i%4], k = 0 .. 3
template <int OFF> __device__ __forceinline__ u32x2 ds_transposed(unsigned a) {
    u32x2 r;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(a), "n"(OFF));
    return r;
}
// One MFMA operand: lane l holds output index l % 16, contraction indexes 8 (l / 16) .. + 7 of a half step.  Its registers may be touched only after
// landed(), behind a wait.  read<H, N, TILE>: half H of the step, 16 output indexes number N of this wavefront's.
template <bool COL> struct Frag;
template <> struct Frag<false> {                 // in LDS [index][64 contraction indexes]
    u32x4 v;
    template <int H, int N, int TILE, int NA> __device__ __forceinline__ void read(const unsigned (&a)[NA]) { v = ds_b128<N * 2048>(a[H]); }
    __device__ __forceinline__ void landed() { asm volatile("" : "+v"(v)); }
    __device__ __forceinline__ u32x4 get() const { return v; }
};
template <> struct Frag<true> {                  // in LDS [64 contraction indexes][TILE]
    u32x2 lo, hi;
    template <int H, int N, int TILE, int NA> __device__ __forceinline__ void read(const unsigned (&a)[NA]) {
        lo = ds_transposed<H * 64 * TILE>(a[N]);
        hi = ds_transposed<H * 64 * TILE + 8 * TILE>(a[N]);
    }
    __device__ __forceinline__ void landed() { asm volatile("" : "+v"(lo), "+v"(hi)); }
    __device__ __forceinline__ u32x4 get() const { return u32x4{lo.x, lo.y, hi.x, hi.y}; }
};

// c += b a^T on 16 x 16 outputs: lane l ends up with columns 4 (l / 16) .. + 3 (b's indexes) of row l % 16 (a's)
#define GEMM_MFMA(OP)                                                                                                                             \
    static __device__ __forceinline__ void mfma(f32x4& c, u32x4 b, u32x4 a) { asm volatile(OP " %0, %1, %2, %0" : "+a"(c) : "v"(b), "v"(a)); }    \
    static __device__ __forceinline__ void mfma_zero(f32x4& c, u32x4 b, u32x4 a) { asm volatile(OP " %0, %1, %2, 0" : "=a"(c) : "v"(b), "v"(a)); } \
    template <int I>                                                                                                                              \
    static __device__ __forceinline__ void mfma_load(f32x4& c, u32x4 b, u32x4 a, unsigned dst, int off, u32x4 rs) {                               \
        if constexpr (I % 4 == 0)                                                                                                                 \
            asm volatile("s_add_i32 m0, %3, %6\n\t" OP " %0, %1, %2, %0\n\tbuffer_load_dwordx4 %4, %5, 0 offen lds"                              \
                         : "+a"(c) : "v"(b), "v"(a), "s"(dst), "v"(off), "s"(rs), "n"(I * 1024) : "memory", "scc");                               \
        else                                                                                                                                      \
            asm volatile(OP " %0, %1, %2, %0\n\tbuffer_load_dwordx4 %3, %4, 0 offen offset:%5 lds"                                               \
                         : "+a"(c) : "v"(b), "v"(a), "v"(off), "s"(rs), "n"(I % 4 * 1024) : "memory");                                            \
    }
template <typename T> struct Mfma16;
template <> struct Mfma16<__bf16> { GEMM_MFMA("v_mfma_f32_16x16x32_bf16") };
template <> struct Mfma16<_Float16> { GEMM_MFMA("v_mfma_f32_16x16x32_f16") };
#undef GEMM_MFMA
// Load I of a step: 1 KB at dst + 1024 I.  M0 holds the LDS address of four loads, whose number in the four travels in the instruction's offset (it is
// added to both addresses, so `off` lies that much lower); nothing else in the kernel touches M0.
template <int I> __device__ __forceinline__ void load_to_lds(unsigned dst, int off, u32x4 rs) {
    if constexpr (I % 4 == 0)
        asm volatile("s_add_i32 m0, %0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(dst), "v"(off), "s"(rs), "n"(I * 1024) : "memory", "scc");
    else
        asm volatile("buffer_load_dwordx4 %0, %1, 0 offen offset:%2 lds" ::"v"(off), "s"(rs), "n"(I % 4 * 1024) : "memory");
}
template <int N> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

constexpr int kWaves = 4, kWavesR = 2, kWavesC = 2;
template <int TILE> struct Side {
    static constexpr int BYTES = TILE * kStep * 2;
    static constexpr int LOADS = TILE / 8 / kWaves;        // 1 KB loads per wavefront and step
    static constexpr int FRAGS = TILE / kWavesR / 16;      // of a wavefront
};

// ACOL, BCOL: the operand's rows run along the output (A [depth, rows], B [depth, cols]) instead of along the contraction (A [rows, depth], B [cols, depth]).
// NSA: steps in A's LDS ring (B's holds three).  WPE: wavefronts per SIMD.
template <typename T, int TR, int TC, int NSA, int WPE, bool ACOL, bool BCOL>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void gemm_kernel(const GemmParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    using SA = Side<TR>;
    using SB = Side<TC>;
    constexpr int FR = SA::FRAGS, FC = SB::FRAGS, NA = SA::LOADS, NB = SB::LOADS, NSB = 3;
    constexpr int A_OFF = 0, B_OFF = NSA * SA::BYTES;
    extern __shared__ __align__(1024) char smem[];
    const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = wave % kWavesR, wc = wave / kWavesR;

    // workgroups with ids = x mod 8 run on XCD x: each XCD has a contiguous eighth of the items
    const int xcd = blockIdx.x & 7, wg_per_xcd = gridDim.x >> 3;
    const int x0 = (int)((int64_t)p.items * xcd >> 3), x1 = (int)((int64_t)p.items * (xcd + 1) >> 3);
    int item = x0 + (blockIdx.x >> 3);
    if (item >= x1) return;

    auto place = [&](int t, int& z, int& tr, int& tc) __attribute__((always_inline)) {
        z = t < p.tiles ? 0 : t < 2 * p.tiles ? 1 : 2;
        t -= z * p.tiles;
        const int grp = (int)__umulhi((unsigned)t, p.m_group), r0 = grp * kTileGroup, nr = min(kTileGroup, p.tiles_r - r0);
        t -= grp * p.group;
        tc = nr == kTileGroup ? t / kTileGroup : nr == 1 ? t : (int)__umulhi((unsigned)t, p.m_last);    // (2^32 / 1 has no 32 bits)
        tr = r0 + t - tc * nr;
    };

    // ---- where a lane's 16 bytes of each load come from.  A load is 1 KB of a stage: chunk c of a row lies at c XOR (something of the row).
    auto fill_off = [&](bool col, int tile, int64_t ld, int i) __attribute__((always_inline)) -> int {
        if (!col) {
            const int row = 8 * (wave * (tile / 8 / kWaves) + i) + (lane >> 3);
            return (int)(row * ld * 2) + (((lane & 7) ^ ((row >> 1) & 7)) << 4) - i % 4 * 1024;
        }
        const int per_row = tile / 8, k = 64 / per_row * (wave * (tile / 8 / kWaves) + i) + lane / per_row;
        return (int)(k * ld * 2) + (((lane % per_row) ^ (2 * ((k & 3) + 4 * ((k >> 3) & 1)))) << 4) - i % 4 * 1024;
    };
    int a_off[NA], b_off[NB];
#pragma unroll
    for (int i = 0; i < NA; ++i) a_off[i] = fill_off(ACOL, TR, p.lda, i);
#pragma unroll
    for (int i = 0; i < NB; ++i) b_off[i] = fill_off(BCOL, TC, p.ldb, i);

    // ---- where a lane reads its fragments: per half step, or per 16 output indexes
    constexpr int NAA = ACOL ? FR : 2, NBA = BCOL ? FC : 2;
    unsigned ra[NAA], rb[NBA];
    const int l16 = lane & 15, g = lane >> 4;
    auto row_addr = [&](int base, int h) __attribute__((always_inline)) { return (unsigned)((base + l16) * 128 + (((4 * h + g) ^ (l16 >> 1)) << 4)); };
    auto col_addr = [&](int base, int f, int tile) __attribute__((always_inline)) {
        const int k = 8 * g + l16 / 4, m = base + 16 * f + 4 * (l16 & 3);
        return (unsigned)(k * tile * 2 + (((m / 8) ^ (2 * (l16 / 4 + 4 * (g & 1)))) << 4) + 8 * (l16 & 1));
    };
#pragma unroll
    for (int i = 0; i < NAA; ++i) ra[i] = lds + A_OFF + (ACOL ? col_addr(wr * (TR / kWavesR), i, TR) : row_addr(wr * (TR / kWavesR), i));
#pragma unroll
    for (int i = 0; i < NBA; ++i) rb[i] = lds + B_OFF + (BCOL ? col_addr(wc * (TC / kWavesC), i, TC) : row_addr(wc * (TC / kWavesC), i));

    // ---- one cursor per operand: the step that is loaded next
    struct Cursor {
        int item, segment, left;
        unsigned dst;          // LDS address of this wavefront's first load
        uint64_t ptr;          // memory, and bytes left from there to the operand's end: what lies beyond reads as zeros
        unsigned n, step;
        __device__ __forceinline__ u32x4 rs() const { return u32x4{(unsigned)ptr, (unsigned)(ptr >> 32), n, 0x00020000u}; }
    };
    auto setup = [&](Cursor& f, auto side) __attribute__((always_inline)) {
        constexpr bool IS_A = decltype(side)::value == 0, COL = IS_A ? ACOL : BCOL;
        // (nothing more: the loads are issued all the same, and counted, of a buffer of no bytes)
        unsigned n = 0, step = 0;
        int left = 1 << 30;
        uint64_t ptr = f.ptr;
        if (f.item < x1) {
            int z, tr, tc;
            place(f.item, z, tr, tc);
            z += f.segment;
            const uint16_t *base0 = IS_A ? p.a[0] : p.b[0], *base1 = IS_A ? p.a[1] : p.b[1], *base2 = IS_A ? p.a[2] : p.b[2];
            const uint16_t* base = z == 0 ? base0 : z == 1 ? base1 : base2;
            const int idx0 = IS_A ? tr * TR : tc * TC, n_idx = IS_A ? p.rows : p.cols;
            const int64_t ld = IS_A ? p.lda : p.ldb;
            const int64_t skip = COL ? idx0 : (int64_t)idx0 * ld;
            const int64_t all = COL ? (p.depth - 1) * ld + n_idx : (n_idx - 1) * ld + p.depth;
            ptr = (uint64_t)(base + skip) & 0xFFFFFFFFFFFFull;
            n = (unsigned)((all - skip) * 2);
            step = f.step;
            left = p.steps;
        }
        f.ptr = ptr;
        f.n = n;
        f.step = step;
        f.left = left;
    };
    Cursor ca, cb;
    ca.item = cb.item = item;
    ca.segment = cb.segment = 0;
    ca.dst = lds + A_OFF + wave * NA * 1024;
    cb.dst = lds + B_OFF + wave * NB * 1024;
    const unsigned a_end = ca.dst + NSA * SA::BYTES, b_end = cb.dst + NSB * SB::BYTES;
    ca.step = ACOL ? 2u * kStep * (unsigned)p.lda : 2u * kStep;
    cb.step = BCOL ? 2u * kStep * (unsigned)p.ldb : 2u * kStep;
    ca.ptr = cb.ptr = 0;
    setup(ca, Int<0>{});
    setup(cb, Int<1>{});
    auto step_on = [&](Cursor& f, unsigned end, int bytes, int stages) __attribute__((always_inline)) {
        f.dst += bytes;
        if (f.dst == end) f.dst -= stages * bytes;
        f.ptr += f.step;
        f.n -= f.step;
        if (--f.left) return false;
        if (++f.segment == p.segments) { f.segment = 0; f.item += wg_per_xcd; }
        return true;
    };
    auto move_a = [&]() __attribute__((always_inline)) { if (__builtin_expect(step_on(ca, a_end, SA::BYTES, NSA), 0)) setup(ca, Int<0>{}); };
    auto move_b = [&]() __attribute__((always_inline)) { if (__builtin_expect(step_on(cb, b_end, SB::BYTES, NSB), 0)) setup(cb, Int<1>{}); };

    // ---- fragments: of half step 0 and of half step 1
    Frag<ACOL> fa[2][FR];
    Frag<BCOL> fb[2][FC];
    f32x4 acc[FC][FR];
    constexpr int NRD = FR + FC;
    auto read_frag = [&](auto half, auto n) __attribute__((always_inline)) {
        constexpr int H = decltype(half)::value, N = decltype(n)::value;
        if constexpr (N < FR) fa[H][N].template read<H, N, TR>(ra);
        else fb[H][N - FR].template read<H, N - FR, TC>(rb);
    };
    auto wait_half = [&](auto half) __attribute__((always_inline)) {
        constexpr int H = decltype(half)::value;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        for_each<FR>([&](auto i) { fa[H][decltype(i)::value].landed(); });
        for_each<FC>([&](auto i) { fb[H][decltype(i)::value].landed(); });
    };
    // from a step's stage to the next one's, in A's ring (of two: there and back) and in B's
    int a_to[3] = {SA::BYTES, SA::BYTES, -2 * SA::BYTES}, b_to[3] = {SB::BYTES, SB::BYTES, -2 * SB::BYTES};
    auto advance = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NAA; ++i) ra[i] += a_to[0];
#pragma unroll
        for (int i = 0; i < NBA; ++i) rb[i] += b_to[0];
    };
    auto next_stage = [&]() __attribute__((always_inline)) {
        if constexpr (NSA == 2) a_to[0] = -a_to[0];
        else { const int t = a_to[0]; a_to[0] = a_to[1]; a_to[1] = a_to[2]; a_to[2] = t; }
        const int t = b_to[0];
        b_to[0] = b_to[1];
        b_to[1] = b_to[2];
        b_to[2] = t;
    };

    // ---- slots: a step's MFMAs are numbered 0 .. 2 NM - 1.
    //   A's ring of three: at slot Y = NM everybody has read the step, and the next step's operands are here; the loads of the step three ahead follow,
    //     spread over the 2 NM slots from Y to the next Y.
    //   A's ring of two: at slot X everybody has read the step; A's loads of the step two ahead are spread over NM slots from there, B's of the step
    //     three ahead over the other NM; at slot Y, later, the next step's operands are here.
    // Half 1's fragments are read from slot 0 on, the next step's half 0 from slot Y on.
    constexpr int NM = FR * FC;
    constexpr bool A3 = NSA == 3;
    constexpr int XQ = A3 ? NM : NM * 5 / 8, YQ = A3 ? NM : NM + NM / 8;
    constexpr int RS = NM / 2 / NRD > 0 ? NM / 2 / NRD : 1;          // a read every RS slots
    static_assert((NRD - 1) * RS < XQ && YQ + (NRD - 1) * RS < 2 * NM, "reads end before they are waited for");
    // of n loads that are spread over slots q0 .. q0 + len - 1, how many are issued before slot q
    constexpr auto before = [](int n, int q0, int len, int q) { return q <= q0 ? 0 : q >= q0 + len ? n : n * (q - q0) / len; };
    // the load of slot q: A's number, NA + B's number, or -1
    constexpr auto load_of = [before](int q) {
        if (A3) {
            const int at = q >= NM ? q - NM : q + NM;
            const int lo = before(NA + NB, 0, 2 * NM, at), hi = before(NA + NB, 0, 2 * NM, at + 1);
            return hi > lo ? lo : -1;
        }
        const int alo = before(NA, XQ, NM, q), ahi = before(NA, XQ, NM, q + 1);
        if (ahi > alo) return alo;
        const int at = q >= XQ + NM ? q - (XQ + NM) : q < XQ ? q + (NM - XQ) : -1;
        if (at < 0) return -1;
        const int lo = before(NB, 0, NM, at), hi = before(NB, 0, NM, at + 1);
        return hi > lo ? NA + lo : -1;
    };
    static_assert(NA + NB <= 2 * NM && NA <= NM && NB <= NM, "never two loads in a slot");
    constexpr int NEWER = A3 ? NA + NB : NB + before(NA, XQ, NM, YQ);       // loads issued by slot Y behind the last one that it waits for
    constexpr int STORES = FR * FC / 2;                                     // of a tile; in the order of the loads, behind those

    auto some_a = [&](auto n) __attribute__((always_inline)) { for_each<decltype(n)::value>([&](auto k) { constexpr int I = decltype(k)::value; load_to_lds<I>(ca.dst, a_off[I], ca.rs()); }); };
    auto some_b = [&](auto n) __attribute__((always_inline)) { for_each<decltype(n)::value>([&](auto k) { constexpr int I = decltype(k)::value; load_to_lds<I>(cb.dst, b_off[I], cb.rs()); }); };
    for_each<2>([&](auto) {
        some_a(Int<NA>{});
        some_b(Int<NB>{});
        move_a();
        move_b();
    });
    // what the slots before the first Y (or X) do not issue (slot 0 moves on where the load before it was a part's last)
    constexpr int PRE = A3 ? before(NA + NB, 0, 2 * NM, NM) : before(NB, 0, NM, NM - XQ);
    static_assert(PRE < NA + NB && (A3 || PRE < NB), "the prologue stops inside a step");
    if constexpr (A3) {
        some_a(Int<(PRE < NA ? PRE : NA)>{});
        if constexpr (PRE > NA) {
            move_a();
            some_b(Int<PRE - NA>{});
        }
    } else {
        some_b(Int<PRE>{});
    }
    wait_vm<PRE>();            // the first two steps are here: a tile's first step waits as if stores of the tile before were under way
    __builtin_amdgcn_s_barrier();
    for_each<NRD>([&](auto n) { read_frag(Int<0>{}, n); });
    wait_half(Int<0>{});

    auto slot = [&](auto qi, auto first) __attribute__((always_inline)) {
        constexpr int Q = decltype(qi)::value, H = Q / NM, M = Q % NM, CI = M / FR, J = M % FR;
        constexpr bool FIRST = decltype(first)::value, ZERO = FIRST && H == 0;
        if constexpr (Q == XQ) wait_half(Int<1>{});
        if constexpr (Q == XQ && !A3) __builtin_amdgcn_s_barrier();
        if constexpr (Q == YQ) {
            wait_vm<(FIRST ? (NEWER + STORES > 63 ? 63 : NEWER + STORES) : NEWER)>();
            __builtin_amdgcn_s_barrier();
            advance();
        }
        if constexpr (Q == YQ + 2) next_stage();
        __builtin_amdgcn_sched_barrier(0);
        constexpr int L = load_of(Q), BEFORE = load_of((Q + 2 * NM - 1) % (2 * NM));
        if constexpr (BEFORE == NA - 1) move_a();
        if constexpr (BEFORE == NA + NB - 1) move_b();
        if constexpr (L >= 0 && !ZERO) {
            constexpr int I = L < NA ? L : L - NA;
            if constexpr (L < NA) Mfma16<T>::template mfma_load<I>(acc[CI][J], fb[H][CI].get(), fa[H][J].get(), ca.dst, a_off[I], ca.rs());
            else Mfma16<T>::template mfma_load<I>(acc[CI][J], fb[H][CI].get(), fa[H][J].get(), cb.dst, b_off[I], cb.rs());
        } else {
            if constexpr (ZERO) Mfma16<T>::mfma_zero(acc[CI][J], fb[H][CI].get(), fa[H][J].get());
            else Mfma16<T>::mfma(acc[CI][J], fb[H][CI].get(), fa[H][J].get());
            if constexpr (L >= 0) {
                constexpr int I = L < NA ? L : L - NA;
                if constexpr (L < NA) load_to_lds<I>(ca.dst, a_off[I], ca.rs());
                else load_to_lds<I>(cb.dst, b_off[I], cb.rs());
            }
        }
        constexpr int RQ = Q < NM ? Q : Q - YQ;
        if constexpr (RQ >= 0 && RQ % RS == 0 && RQ / RS < NRD) read_frag(Int<(Q < NM ? 1 : 0)>{}, Int<RQ / RS>{});
        __builtin_amdgcn_sched_barrier(0);
    };

    const int all_steps = p.steps * p.segments;
#pragma clang loop unroll(disable)
    for (; item < x1; item += wg_per_xcd) {
        for_each<2 * NM>([&](auto q) { slot(q, Int<1>{}); });
        wait_half(Int<0>{});
#pragma clang loop unroll(disable)
        for (int s = 1; s < all_steps; ++s) {
            for_each<2 * NM>([&](auto q) { slot(q, Int<0>{}); });
            wait_half(Int<0>{});
        }
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");      // the last products (written as asm: no hazard checks) are in their registers
        int el = lane;
        asm volatile("" : "+v"(el));                            // (the addresses below are not kept over the loop)
        int z, tr, tc;
        place(item, z, tr, tc);
        uint16_t* out = z == 0 ? p.c[0] : z == 1 ? p.c[1] : p.c[2];
        const int m0 = wr * (TR / kWavesR) + (el & 15), n0 = wc * (TC / kWavesC), eg = el >> 4;
        const int rows = min(TR, p.rows - tr * TR), cols = min(TC, p.cols - tc * TC);
        const auto rsc = __builtin_amdgcn_make_buffer_rsrc((void*)(out + (int64_t)tr * TR * p.ldc + tc * TC), 0, (unsigned)(((rows - 1) * p.ldc + cols) * 2), 0x00020000);
#pragma unroll
        for (int j = 0; j < FR; ++j) {
            const int m = m0 + 16 * j;
#pragma unroll
            for (int i = 0; i < FC; i += 2) {
                asm volatile("" : "+a"(acc[i][j]), "+a"(acc[i + 1][j]));     // (out of the accumulation registers only now)
                __builtin_amdgcn_sched_barrier(0);
                typedef T pair_t __attribute__((ext_vector_type(2)));
                unsigned w[2][2];
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int h = 0; h < 2; ++h) w[q][h] = __builtin_bit_cast(unsigned, pair_t{(T)acc[i + q][j][2 * h], (T)acc[i + q][j][2 * h + 1]});
                // a lane has 4 columns of tile i and 4 of tile i + 1; afterwards even groups of 16 lanes have 8 of tile i, odd ones 8 of tile i + 1
                const auto s0 = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
                const auto s1 = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
                const int n = n0 + 16 * (i + (eg & 1)) + 8 * (eg >> 1);
                // (lanes outside the matrix store past the buffer's end: dropped, but the instruction is issued and counted)
                const unsigned at = m < rows && n < cols ? (unsigned)((m * p.ldc + n) * 2) : 0x80000000u;
                __builtin_amdgcn_raw_buffer_store_b128(u32x4{s0[0], s1[0], s0[1], s1[1]}, rsc, at, 0, 0);
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0): drain the (unused) trailing loads before the LDS is released
#endif
}

// The tile shapes, and what they are chosen by: the time of a 64-deep step of a workgroup in full rounds, the part of it that is left when few workgroups
// run (the part clocks higher under its power limit), and what a tile costs besides its steps.  Fits to 2048 and 5120 wide layers (and 4 times that) with
// 256 .. 70400 rows, all orders, every shape measured: the choice is within 1 % of the best on average.
struct Shape { int tr, tc, nsa, per_cu; double step_us, alone, tile_us; };
constexpr Shape kShapes[] = {
    {256, 256, 2, 1, 1.38, 0.71, 4.0},
    {256, 128, 3, 1, 0.81, 0.67, 1.9},
    {128, 256, 3, 1, 0.83, 0.70, 1.8},
    {128, 128, 2, 2, 0.98, 0.70, 0.5},
};
constexpr int kNumShapes = 4;
constexpr double kLaunchUs = 4.4;

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
double cost_of(const Shape& s, int64_t rows, int64_t cols, int64_t steps, int64_t products) {
    const int64_t items = ceil_div(rows, s.tr) * ceil_div(cols, s.tc) * products;
    const int64_t per_xcd = ceil_div(items, 8), slots = kNumCUs / 8 * s.per_cu, full = per_xcd / slots, rest = per_xcd % slots;
    double us = kLaunchUs + (double)full * (steps * s.step_us + s.tile_us);
    if (rest > 0) {
        // two workgroups share a compute unit only where there are more than compute units: one by itself takes a little more than half of their time
        const bool shared = s.per_cu == 2 && rest > slots / 2;
        const double filled = (double)rest / (double)(s.per_cu == 2 && !shared ? slots / 2 : slots);
        us += steps * s.step_us * (s.per_cu == 2 && !shared ? 0.54 : 1.0) * (s.alone + (1.0 - s.alone) * filled * filled) + s.tile_us;
    }
    return us;
}
int choose_shape(const cosmos_attn_gemm_desc* d, double* cost) {
    const bool sum = (d->flags & COSMOS_GEMM_SUM) != 0;
    const int64_t steps = ceil_div(d->depth, kStep) * (sum ? d->count : 1), products = sum ? 1 : d->count;
    int best = 0;
    for (int i = 0; i < kNumShapes; ++i) {
        const double c = cost_of(kShapes[i], d->rows, d->cols, steps, products);
        if (i == 0 || c < *cost) { best = i; *cost = c; }
    }
    return best;
}

template <typename T, int SHAPE, bool ACOL, bool BCOL>
int launch(GemmParams& p, int products, hipStream_t stream) {
    constexpr Shape s = kShapes[SHAPE];
    p.tiles_r = (int)ceil_div(p.rows, s.tr);
    p.tiles_c = (int)ceil_div(p.cols, s.tc);
    const int64_t tiles = (int64_t)p.tiles_r * p.tiles_c, group = (int64_t)kTileGroup * p.tiles_c;
    // (an item number times a divisor stays below 2^32: then the division by its rounded-up reciprocal is exact)
    if (tiles * group >= (int64_t)1 << 32 || tiles * kMostProducts > 0x7FFFFFFF) return COSMOS_ATTN_UNSUPPORTED;
    p.tiles = (int)tiles;
    p.items = (int)(tiles * products);
    p.steps = (int)ceil_div(p.depth, kStep);
    p.group = (int)group;
    auto reciprocal = [](uint64_t d) { return d < 2 ? 0u : (unsigned)((0x100000000ull + d - 1) / d); };
    p.m_group = reciprocal(p.group);
    p.m_last = reciprocal(p.tiles_r % kTileGroup);
    const size_t lds = (size_t)s.nsa * Side<s.tr>::BYTES + 3u * Side<s.tc>::BYTES;
    auto kernel = gemm_kernel<T, s.tr, s.tc, s.nsa, s.per_cu, ACOL, BCOL>;
    if (!allow_lds((const void*)kernel, lds)) return COSMOS_ATTN_LAUNCH_FAILED;
    kernel<<<dim3(kNumCUs * s.per_cu), dim3(64 * kWaves), lds, stream>>>(p);
    return hipGetLastError() == hipSuccess ? COSMOS_ATTN_OK : COSMOS_ATTN_LAUNCH_FAILED;
}
template <typename T, bool ACOL, bool BCOL>
int launch_shape(int shape, GemmParams& p, int products, hipStream_t stream) {
    switch (shape) {
        case 0: return launch<T, 0, ACOL, BCOL>(p, products, stream);
        case 1: return launch<T, 1, ACOL, BCOL>(p, products, stream);
        case 2: return launch<T, 2, ACOL, BCOL>(p, products, stream);
        default: return launch<T, 3, ACOL, BCOL>(p, products, stream);
    }
}
template <typename T>
int launch_order(int order, int shape, GemmParams& p, int products, hipStream_t stream) {
    switch (order) {
        case COSMOS_GEMM_XWT: return launch_shape<T, false, false>(shape, p, products, stream);
        case COSMOS_GEMM_XW: return launch_shape<T, false, true>(shape, p, products, stream);
        default: return launch_shape<T, true, true>(shape, p, products, stream);
    }
}

int check(const cosmos_attn_gemm_desc* d) {
    if (!d || d->abi_version != COSMOS_ATTN_ABI_VERSION) return COSMOS_ATTN_BAD_ARG;
    if (d->dtype != COSMOS_ATTN_BF16 && d->dtype != COSMOS_ATTN_FP16) return COSMOS_ATTN_BAD_ARG;
    if (d->order < COSMOS_GEMM_XWT || d->order > COSMOS_GEMM_XTX || d->count < 1 || d->count > kMostProducts) return COSMOS_ATTN_BAD_ARG;
    if (d->flags & ~COSMOS_GEMM_SUM || d->shape < 0 || d->shape > kNumShapes) return COSMOS_ATTN_BAD_ARG;
    if (d->rows < 1 || d->cols < 1 || d->depth < 1 || d->cols % 8) return COSMOS_ATTN_BAD_SHAPE;
    const bool acol = d->order == COSMOS_GEMM_XTX, bcol = d->order != COSMOS_GEMM_XWT;
    // rows along the contraction are read 64 deep without looking at their end; rows along the output in 16-byte chunks
    if ((!acol || !bcol) && d->depth % kStep) return COSMOS_ATTN_BAD_SHAPE;
    if (acol && d->rows % 8) return COSMOS_ATTN_BAD_SHAPE;
    const int64_t a_width = acol ? d->rows : d->depth, b_width = bcol ? d->cols : d->depth;
    const int64_t a_lines = acol ? d->depth : d->rows, b_lines = bcol ? d->depth : d->cols;
    if (d->lda < a_width || d->ldb < b_width || d->ldc < d->cols) return COSMOS_ATTN_BAD_STRIDE;
    if (d->lda % 8 || d->ldb % 8 || d->ldc % 8) return COSMOS_ATTN_BAD_STRIDE;
    // (four loads share an LDS address: a lane's offset less 3 KB is not negative from here on)
    if ((acol && d->lda < 256) || (bcol && d->ldb < 256)) return COSMOS_ATTN_UNSUPPORTED;
    // 32-bit byte offsets: inside a tile, and from a tile to the operand's end
    const int64_t most = (int64_t)1 << 21;
    if (d->lda > most || d->ldb > most || d->ldc > most) return COSMOS_ATTN_UNSUPPORTED;
    if (((a_lines - 1) * d->lda + a_width) * 2 >= (int64_t)1 << 32 || ((b_lines - 1) * d->ldb + b_width) * 2 >= (int64_t)1 << 32) return COSMOS_ATTN_UNSUPPORTED;
    const bool sum = (d->flags & COSMOS_GEMM_SUM) != 0;
    for (int i = 0; i < d->count; ++i) {
        if (!d->a[i] || !d->b[i] || !aligned16(d->a[i]) || !aligned16(d->b[i])) return COSMOS_ATTN_BAD_ARG;
        if ((i == 0 || !sum) && (!d->c[i] || !aligned16(d->c[i]))) return COSMOS_ATTN_BAD_ARG;
    }
    return COSMOS_ATTN_OK;
}
// Where these kernels are the faster ones and where the library's.  Both sides measured on two cards at 256 .. 90 000 rows (ragged ones and whole frames), layers 512 to 5120 wide
// and MLPs of four times that, 1700 sizes for one product, 1000 for several; below: this one's share of the library's time, mean (worst).  The kernels' own time follows cost_of within
// 10 %.  The library's does not follow from the sizes: its choice of tiles is 7 % faster than this one where they fill the chip and up to twice as slow just past a whole round (9360 x 2048 x 8192
// 506 us, 10920 279), and changes from one number of rows to the next.  What is common to the widths is how many rounds its largest tiles take:
//   y, one product.  A half filled to just full round, the second half of a second one and a fourth one are the library's (1.08 (1.29), 1.02 (1.14), 1.00 (1.10)); third and fifth ones this
//     one's (0.88 (1.15), 0.94 (1.12)), and for short contractions also the first half of a first round and of a second (0.76 (1.03), 0.92 (1.11); deep ones 1.01 (1.56), 1.00 (1.26)).  From
//     five rounds on 0.97 (1.09) up to 5120 deep, 1.01 (1.12) deeper.  In all 0.90 (1.15) where it is chosen; "every 8192 rows and more, small layers from 1024 on" was 0.95 (1.56).
//   dx, one product: from an estimated 1.02 PFLOP/s on, and small ones, where the library is furthest from it; but for the second half of a first round (1.00 (1.17)) and deep
//     contractions just past one (0.95 (1.20)).  0.87 (1.08) where it is chosen.
//   dw: this one, whatever the number of rounds, where a product has three quarters of one (0.74 (0.87)).  Fewer tiles leave the chip to few workgroups, each with the whole contraction, which
//     the library splits if it is long: from a quarter round on up to 8192 deep (0.84 (0.97); 1.01 (1.16) above), an eighth to a quarter (2048 x 2048) up to 27 000 (0.64 (0.91); 1.08 (1.36)
//     above), below that up to 4096 (0.68 (1.06); 0.99 (1.14) up to 16 000, 1.8 from 60 000 on).  Two in a launch are filled twice as well (limits 16 384, none, 32 768: 0.66 (0.99)), three
//     always well enough (0.57 (0.85)).
//   Several products of y, or dx summed, are compared with as many of the library's and their additions, at a rate and a launch that these take at best: 0.81 (1.10), 0.67 (0.96).
//     (Of y, 12 us a launch: the 52 measured sizes that 8 us would leave to the library are 0.86 (1.08), the 38 that 12 leaves 0.93 (1.18).)
// On a third card, at other rows and at widths of 1536, 2560 (MLP) and 4096 that no line was drawn by: y 0.92 (1.10) where chosen and 1.03 where not, dx 0.87 (1.06), dw 0.71 (0.98).
bool preferred(const cosmos_attn_gemm_desc* d) {
    double us = 0.0;
    choose_shape(d, &us);
    const double one = 2.0 * d->rows * d->cols * d->depth, rate = one * d->count / us;     // operations, per microsecond
    const double rounds = (double)(ceil_div(d->rows, 256) * ceil_div(d->cols, 256)) / kNumCUs;      // of one product
    const int64_t depth = d->depth;
    if (d->order == COSMOS_GEMM_XTX) {
        if (depth < 256) return false;
        const bool two = d->count == 2;
        if (d->count == 3 || rounds > 0.75) return true;
        if (rounds > 0.25) return depth <= (two ? 16384 : 8192);
        if (rounds > 0.125) return two || depth <= 27000;
        return depth <= (two ? 32768 : 4096);
    }
    if (d->rows < 1024) return false;
    if (d->order == COSMOS_GEMM_XW) {
        if (d->count > 1) return us <= d->count * (one / 1.25e9 + 10.0);
        if ((rounds > 0.5 && rounds <= 0.75) || (rounds > 1.0 && rounds <= 1.2 && depth > 2048)) return false;
        return rate >= 1.02e9 || (one <= 6e10 && rate >= 0.55e9);
    }
    if (d->count > 1) return us <= d->count * (one / 1.35e9 + 12.0);
    if (rounds <= 0.5 || (rounds > 1.0 && rounds <= 1.5)) return depth <= 2048;
    if (rounds <= 2.0 || (rounds > 3.0 && rounds <= 4.0)) return false;
    return rounds <= 5.0 || depth <= 5120;
}
}  // namespace

extern "C" {

COSMOS_ATTN_API int cosmos_attn_gemm_preferred(const cosmos_attn_gemm_desc* d) {
    return check(d) == COSMOS_ATTN_OK && preferred(d) ? 1 : 0;
}

COSMOS_ATTN_API int cosmos_attn_gemm(const cosmos_attn_gemm_desc* d, void* stream_handle) {
    const int bad = check(d);
    if (bad != COSMOS_ATTN_OK) return bad;
    if (!device_is_whole_mi355x()) return COSMOS_ATTN_WRONG_DEVICE;
    hipStream_t stream = static_cast<hipStream_t>(stream_handle);
    GemmParams p = {};
    for (int i = 0; i < d->count; ++i) {
        p.a[i] = static_cast<const uint16_t*>(d->a[i]);
        p.b[i] = static_cast<const uint16_t*>(d->b[i]);
        p.c[i] = static_cast<uint16_t*>(d->c[i]);
    }
    p.lda = d->lda;
    p.ldb = d->ldb;
    p.ldc = d->ldc;
    p.rows = d->rows;
    p.cols = d->cols;
    p.depth = d->depth;
    const bool sum = (d->flags & COSMOS_GEMM_SUM) != 0;
    p.segments = sum ? d->count : 1;
    double cost = 0.0;
    int shape = choose_shape(d, &cost);
    if (d->shape > 0) shape = d->shape - 1;
    const int products = sum ? 1 : d->count;
    if (d->dtype == COSMOS_ATTN_BF16) return launch_order<__bf16>(d->order, shape, p, products, stream);
    return launch_order<_Float16>(d->order, shape, p, products, stream);
}
}
