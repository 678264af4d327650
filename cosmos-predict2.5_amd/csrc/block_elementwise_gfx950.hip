// Elementwise pieces of the DiT block with their forward-mode tangents, for gfx950: kernels and C ABI.
//
// The DiT block (cosmos_predict2/_src/predict2/networks/minimal_v4_dit.py:1119-1242) wraps each of its three
// sub-layers as
//     n = LayerNorm(x) * (1 + scale) + shift            (:1166-1167; LayerNorm without affine parameters, eps 1e-6, :1031)
//     x = x + gate * sublayer(n)                         (:1199, :1231, :1241)
// with per-(batch, frame) modulation vectors shift / scale / gate (:1131-1162), and its MLP uses the exact GELU
// (:222-249).  When a tangent is carried through the block these steps become, in plain tensor-library ops, some thirty
// passes over tensors of hundreds of megabytes; here each is one pass:
//     ln_modulate_kernel      y = n (1 + scale) + shift,  ty = tn (1 + scale) + n tscale + tshift
//                             n = (x - mean) r,  tn = r (tc - n mean(n tc)),  tc = tx - mean(tx),  r = rsqrt(var + eps)
//     gated_residual_kernel   out = x + gate res,  tout = tx + tgate res + gate tres
//                             (between two sub-layers: inside ln_modulate_kernel, which then reads x, tx from registers)
//     gelu_kernel             a = h Phi(h),  ta = th (Phi(h) + h phi(h))
// and their reverse mode, for training:
//     ln_modulate_bwd_kernel     dx = dskip + r (dn - mean(dn) - n mean(dn n)),  dn = dy (1 + scale);  column sums dy n, dy
//     gated_residual_bwd_kernel  dres = dy gate;  column sums dy res
//     column_sum_kernel          adds the column sums of a group's rows up
// and the three small MLPs that make the modulation vectors (modulation_hidden_kernel, modulation_out_kernel).
// The passes over activations are HBM-bound; 16-bit tensors, fp32 arithmetic, 16-byte accesses.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

#include "cosmos_attn_hip.h"

namespace {

constexpr int kThreads = 256;

template <bool BF16>
__device__ __forceinline__ void unpack8(const uint4& v, float* f) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (BF16) {
            f[2 * i] = __builtin_bit_cast(float, w[i] << 16);
            f[2 * i + 1] = __builtin_bit_cast(float, w[i] & 0xFFFF0000u);
        } else {
            typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
            const half2_t h = __builtin_bit_cast(half2_t, w[i]);
            f[2 * i] = (float)h[0];
            f[2 * i + 1] = (float)h[1];
        }
    }
}
template <bool BF16>
__device__ __forceinline__ uint4 pack8(const float* f) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (BF16) {
            typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
            bf2_t r; r[0] = (__bf16)f[2 * i]; r[1] = (__bf16)f[2 * i + 1];
            w[i] = __builtin_bit_cast(uint32_t, r);
        } else {
            typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
            half2_t r; r[0] = (_Float16)f[2 * i]; r[1] = (_Float16)f[2 * i + 1];
            w[i] = __builtin_bit_cast(uint32_t, r);
        }
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// sum over the 64 lanes of the wavefront, result in every lane
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) v += __shfl_xor(v, m);
    return v;
}

// ------------------------------------------------------------------------------------------------ LayerNorm + modulation
struct LnModParams {
    const uint16_t *x, *tx;                      // [rows, D]; tx may be null
    const uint16_t *shift, *scale;               // [groups, D]
    const uint16_t *tshift, *tscale;             // [groups, D] or null (the modulation does not move)
    uint16_t *y, *ty;                            // [rows, D]
    int64_t rows;
    int D, rows_per_group;
    float eps;
    const uint16_t *res, *tres;                  // GATED: [rows, D]
    const uint16_t *gate, *tgate;                // [groups, D]; tgate may be null
    uint16_t *out, *tout;                        // [rows, D]
};

// v = x + gate res, t = tx + gate tres [+ tgate res], eight elements, rounded to the 16-bit type as they are stored
template <bool TANGENT, bool BF16>
__device__ __forceinline__ void gated_sum(uint4 x, uint4 tx, uint4 res, uint4 tres, uint4 gate, const uint16_t* tgate, uint4& v, uint4& t) {
    float fx[8], fr[8], fg[8], s[8];
    unpack8<BF16>(x, fx);
    unpack8<BF16>(res, fr);
    unpack8<BF16>(gate, fg);
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] = fx[i] + fg[i] * fr[i];
    v = pack8<BF16>(s);
    if (TANGENT) {
        float ft[8], ftr[8], ts[8];
        unpack8<BF16>(tx, ft);
        unpack8<BF16>(tres, ftr);
#pragma unroll
        for (int i = 0; i < 8; ++i) ts[i] = ft[i] + fg[i] * ftr[i];
        if (tgate) {
            float ftg[8];
            unpack8<BF16>(*reinterpret_cast<const uint4*>(tgate), ftg);
#pragma unroll
            for (int i = 0; i < 8; ++i) ts[i] += ftg[i] * fr[i];
        }
        t = pack8<BF16>(ts);
    }
}

// One wavefront per row; lane l holds the 8-element chunks l, l + 64, ... (NCH of them, D <= 512 NCH), so that the
// row stays in registers between the statistics and the output pass.
// GATED: the row is the gated residual of the sub-layer before, formed, rounded and stored here, so that it is not read back from memory
// (memory-bound, 4 tensors of traffic instead of 3 + 2, and 1 launch instead of 2; the same bits).  28 blocks on 3520 x 2048 rows, two such
// pairs each: 18406 -> 18089 us, a block on 37440 rows 13558 -> 13467.  One pair, us, two kernels -> this one: 17600 x 2048 rows 67 -> 52, with tangents
// 148 -> 121; 17600 x 5120 180 -> 168, 399 -> 338; 3520 x 5120 37 -> 33
// (inputs not in cache 40 -> 42), 80 -> 72; slower without tangents around 10000 x 5120, 96 -> 101.  Of a block with tangents the matrix products
// are so much that it shows only where the two ways are timed in turn: 17600 rows 10110 -> 10081, 3520 1143 -> 1133, 1560 638 -> 627.
template <int NCH, bool TANGENT, bool BF16, bool GATED>
__global__ void __launch_bounds__(kThreads) ln_modulate_kernel(const LnModParams p) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
    if (row >= p.rows) return;     // whole wavefronts leave together: the shuffles below stay complete
    const int D = p.D;
    const int64_t grp = row / p.rows_per_group;
    const uint16_t* xr = p.x + row * D;
    const uint16_t* txr = TANGENT ? p.tx + row * D : nullptr;
    float x[NCH][8], t[NCH][8];
    float sx = 0.f, st = 0.f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int off = 8 * (lane + 64 * c);
        const bool in = off < D;
        const uint4 z = make_uint4(0u, 0u, 0u, 0u);
        uint4 v = in ? *reinterpret_cast<const uint4*>(xr + off) : z;
        uint4 tv = TANGENT && in ? *reinterpret_cast<const uint4*>(txr + off) : z;
        if (GATED && in) {
            const int64_t o = row * D + off, g = grp * D + off;
            gated_sum<TANGENT, BF16>(v, tv, *reinterpret_cast<const uint4*>(p.res + o), TANGENT ? *reinterpret_cast<const uint4*>(p.tres + o) : z,
                                     *reinterpret_cast<const uint4*>(p.gate + g), TANGENT && p.tgate ? p.tgate + g : nullptr, v, tv);
            *reinterpret_cast<uint4*>(p.out + o) = v;
            if (TANGENT) *reinterpret_cast<uint4*>(p.tout + o) = tv;
        }
        unpack8<BF16>(v, x[c]);
        if (TANGENT) unpack8<BF16>(tv, t[c]);
#pragma unroll
        for (int i = 0; i < 8; ++i) { sx += x[c][i]; if (TANGENT) st += t[c][i]; }
    }
    const float inv_d = 1.0f / D;
    const float mean = wave_sum(sx) * inv_d;
    const float tmean = TANGENT ? wave_sum(st) * inv_d : 0.f;
    float sv = 0.f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const bool in = 8 * (lane + 64 * c) < D;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            x[c][i] = in ? x[c][i] - mean : 0.f;
            if (TANGENT) t[c][i] = in ? t[c][i] - tmean : 0.f;
            sv += x[c][i] * x[c][i];
        }
    }
    const float r = rsqrtf(wave_sum(sv) * inv_d + p.eps);
    float sd = 0.f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
#pragma unroll
        for (int i = 0; i < 8; ++i) { x[c][i] *= r; if (TANGENT) sd += x[c][i] * t[c][i]; }
    }
    const float s = TANGENT ? wave_sum(sd) * inv_d : 0.f;

    const uint16_t* sh = p.shift + grp * D;
    const uint16_t* sc = p.scale + grp * D;
    const uint16_t* tsh = (TANGENT && p.tshift) ? p.tshift + grp * D : nullptr;
    const uint16_t* tsc = (TANGENT && p.tscale) ? p.tscale + grp * D : nullptr;
    uint16_t* yr = p.y + row * D;
    uint16_t* tyr = TANGENT ? p.ty + row * D : nullptr;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int off = 8 * (lane + 64 * c);
        if (off >= D) continue;
        float a[8], b[8], y[8];
        unpack8<BF16>(*reinterpret_cast<const uint4*>(sc + off), a);
        unpack8<BF16>(*reinterpret_cast<const uint4*>(sh + off), b);
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = x[c][i] * (1.0f + a[i]) + b[i];
        *reinterpret_cast<uint4*>(yr + off) = pack8<BF16>(y);
        if (TANGENT) {
            float ty[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) ty[i] = r * (t[c][i] - x[c][i] * s) * (1.0f + a[i]);
            if (tsc) {
                float ta[8];
                unpack8<BF16>(*reinterpret_cast<const uint4*>(tsc + off), ta);
#pragma unroll
                for (int i = 0; i < 8; ++i) ty[i] += x[c][i] * ta[i];
            }
            if (tsh) {
                float tb[8];
                unpack8<BF16>(*reinterpret_cast<const uint4*>(tsh + off), tb);
#pragma unroll
                for (int i = 0; i < 8; ++i) ty[i] += tb[i];
            }
            *reinterpret_cast<uint4*>(tyr + off) = pack8<BF16>(ty);
        }
    }
}

typedef void (*ln_kernel_t)(const LnModParams);
template <bool TANGENT, bool BF16, bool GATED>
ln_kernel_t pick_ln(int d) {
    const int nch = (d + 511) / 512;
    if (nch <= 1) return ln_modulate_kernel<1, TANGENT, BF16, GATED>;
    if (nch <= 2) return ln_modulate_kernel<2, TANGENT, BF16, GATED>;
    if (nch <= 4) return ln_modulate_kernel<4, TANGENT, BF16, GATED>;
    if (nch <= 8) return ln_modulate_kernel<8, TANGENT, BF16, GATED>;
    if (nch <= 10) return ln_modulate_kernel<10, TANGENT, BF16, GATED>;
    if constexpr (!GATED) if (nch <= 16) return ln_modulate_kernel<16, TANGENT, BF16, false>;
    return nullptr;
}
// Wider rows go through the two kernels.  16 chunks of a row take some 200 registers (340 with tangents), and one pass with its four streams is then
// slower than two, but for calls so small that the launch counts (us, two kernels / one pass: 7040 rows of 5632 79 / 93, 37440 432 / 515, of 8192
// 603 / 678, 1560 of 5632 24 / 20; with tangents either way within a tenth: 3520 of 5632 122 / 133, 10000 of 8192 470 / 445).
constexpr int kMaxGatedLnD = 5120;

// ------------------------------------------------------------------------------------------------ gated residual
struct GatedResidualParams {
    const uint16_t *x, *tx, *res, *tres;         // [rows, D]; tx, tres null together
    const uint16_t *gate, *tgate;                // [groups, D]; tgate may be null
    uint16_t *out, *tout;                        // [rows, D]; may alias x, tx
    int64_t chunks;                              // rows * D / 8
    int D, rows_per_group;
};

template <bool TANGENT, bool BF16>
__global__ void __launch_bounds__(kThreads) gated_residual_kernel(const GatedResidualParams p) {
    const int64_t c = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (c >= p.chunks) return;
    const int cpr = p.D / 8;                      // chunks per row
    const int64_t row = c / cpr;
    const int col = (int)(c - row * cpr) * 8;
    const int64_t g = (row / p.rows_per_group) * p.D + col;
    const int64_t o = c * 8;
    const uint4 z = make_uint4(0u, 0u, 0u, 0u);
    uint4 v, tv;
    gated_sum<TANGENT, BF16>(*reinterpret_cast<const uint4*>(p.x + o), TANGENT ? *reinterpret_cast<const uint4*>(p.tx + o) : z,
                             *reinterpret_cast<const uint4*>(p.res + o), TANGENT ? *reinterpret_cast<const uint4*>(p.tres + o) : z,
                             *reinterpret_cast<const uint4*>(p.gate + g), TANGENT && p.tgate ? p.tgate + g : nullptr, v, tv);
    if (TANGENT) *reinterpret_cast<uint4*>(p.tout + o) = tv;
    *reinterpret_cast<uint4*>(p.out + o) = v;
}

// ------------------------------------------------------------------------------------------------ GELU
struct GeluParams {
    const uint16_t *h, *th;                      // th may be null
    uint16_t *a, *ta;
    int64_t chunks;                              // elements / 8
};

template <bool TANGENT, bool BF16>
__global__ void __launch_bounds__(kThreads) gelu_kernel(const GeluParams p) {
    const int64_t c = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (c >= p.chunks) return;
    const int64_t o = c * 8;
    float h[8], a[8], th[8], ta[8];
    unpack8<BF16>(*reinterpret_cast<const uint4*>(p.h + o), h);
    if (TANGENT) unpack8<BF16>(*reinterpret_cast<const uint4*>(p.th + o), th);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float cdf = 0.5f * (1.0f + erff(h[i] * 0.70710678118654752f));
        a[i] = h[i] * cdf;
        if (TANGENT) {
            const float pdf = 0.3989422804014327f * __expf(-0.5f * h[i] * h[i]);
            ta[i] = th[i] * (cdf + h[i] * pdf);
        }
    }
    *reinterpret_cast<uint4*>(p.a + o) = pack8<BF16>(a);
    if (TANGENT) *reinterpret_cast<uint4*>(p.ta + o) = pack8<BF16>(ta);
}

// ------------------------------------------------------------------------------------------------ reverse mode
// Both kernels read every tensor once and leave the sums over a group's rows (the gradients of its modulation vectors) as
// one fp32 line per workgroup; column_sum_kernel adds the lines up in a fixed order.  A workgroup of 256 threads keeps its
// columns (8 (t + 256 c)) over a run of `chunk` rows, so that the column sums stay in registers; the row sums of LayerNorm
// go through LDS, two exchanges for the R rows that are in flight together.  HBM-bound.  In tensor-library ops this was 13
// passes in fp32 per LayerNorm and 7 per gated residual.
// Measured at 10920 x 2048 bf16, one LayerNorm and one gated residual together: 515 -> 94 us (58 and 25, and 5 twice for the
// column sums); of these the LayerNorm runs at 3.1 TB/s, held back by the exchanges between its loads, the other at 5.3.
struct ColumnSums {
    float* part;              // [blocks][vectors][D] (chunks_per_group > 1)
    uint16_t* out[2];         // [groups, D] (written by the kernel itself when a group is one chunk)
    int chunk, chunks_per_group;
};
// rows of one workgroup: runs long enough that the lines of column sums are a small part of the traffic, short enough for
// four workgroups per compute unit; a group of up to 16 rows is never cut
void plan_column_sums(ColumnSums& s, int64_t rows, int rows_per_group) {
    int64_t c = (rows + 1023) / 1024;
    c = (c + 3) / 4 * 4;
    if (c < 8) c = 8;
    if (c > rows_per_group || rows_per_group <= 16) c = rows_per_group;
    s.chunk = (int)c;
    s.chunks_per_group = (int)((rows_per_group + c - 1) / c);
}
size_t column_sum_bytes(int64_t rows, int rows_per_group, int D, int vectors) {
    ColumnSums s;
    plan_column_sums(s, rows, rows_per_group);
    return s.chunks_per_group == 1 ? 0 : (size_t)(rows / rows_per_group) * s.chunks_per_group * vectors * D * sizeof(float);
}
// this workgroup's line of column sums: vector v of `vectors`, columns off .. off + 7
template <bool BF16>
__device__ __forceinline__ void store_column_sums(const ColumnSums& s, int v, int vectors, int D, int off, const float* sum) {
    if (s.chunks_per_group == 1) {
        if (s.out[v]) *reinterpret_cast<uint4*>(s.out[v] + (int64_t)blockIdx.x * D + off) = pack8<BF16>(sum);
    } else {
        float* to = s.part + ((int64_t)blockIdx.x * vectors + v) * D + off;
        *reinterpret_cast<float4*>(to) = make_float4(sum[0], sum[1], sum[2], sum[3]);
        *reinterpret_cast<float4*>(to + 4) = make_float4(sum[4], sum[5], sum[6], sum[7]);
    }
}

// grid (groups, columns / 64, vectors); thread (i, j): lines i, i + 16, ... of the group, columns 4 j .. 4 j + 3
template <bool BF16>
__global__ void __launch_bounds__(kThreads) column_sum_kernel(const ColumnSums s, int vectors, int D) {
    __shared__ float4 red[16][16];
    const int i = threadIdx.x >> 4, j = threadIdx.x & 15;
    const int col = blockIdx.y * 64 + 4 * j, v = blockIdx.z;
    const int64_t line0 = (int64_t)blockIdx.x * s.chunks_per_group;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    if (col < D) {
        for (int l = i; l < s.chunks_per_group; l += 16) {
            const float4 x = *reinterpret_cast<const float4*>(s.part + ((line0 + l) * vectors + v) * D + col);
            a.x += x.x; a.y += x.y; a.z += x.z; a.w += x.w;
        }
    }
    red[i][j] = a;
    __syncthreads();
    if (i == 0 && col < D && s.out[v]) {
        for (int l = 1; l < 16; ++l) { const float4 x = red[l][j]; a.x += x.x; a.y += x.y; a.z += x.z; a.w += x.w; }
        const float f[8] = {a.x, a.y, a.z, a.w, 0.f, 0.f, 0.f, 0.f};
        const uint4 w = pack8<BF16>(f);
        *reinterpret_cast<uint2*>(s.out[v] + (int64_t)blockIdx.x * D + col) = make_uint2(w.x, w.y);
    }
}

struct LnModBwdParams {
    const uint16_t *x, *dy, *dskip;              // [rows, D]; dskip (gradient that reaches x past the LayerNorm) may be null
    const uint16_t* scale;                       // [groups, D]
    uint16_t* dx;                                // [rows, D]
    ColumnSums sums;                             // dshift, dscale
    int D, rows_per_group;
    float eps;
};

// Sums of four values over a wavefront, 7 exchanges instead of 24: the first two halve the number of values a lane carries.
// Returns the sum of value (lane & 3).
__device__ __forceinline__ float wave_sum4(float v0, float v1, float v2, float v3) {
    const bool b0 = threadIdx.x & 1, b1 = threadIdx.x & 2;
    const float k01 = (b0 ? v1 : v0) + __shfl_xor(b0 ? v0 : v1, 1);
    const float k23 = (b0 ? v3 : v2) + __shfl_xor(b0 ? v2 : v3, 1);
    float k = (b1 ? k23 : k01) + __shfl_xor(b1 ? k01 : k23, 2);
#pragma unroll
    for (int m = 4; m < 64; m <<= 1) k += __shfl_xor(k, m);
    return k;
}
// sums of N values over the workgroup; every thread gets them
template <int N>
__device__ __forceinline__ void block_sums(float* v, float (*red)[16]) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < N; i += 4) {
        const float s = wave_sum4(v[i], i + 1 < N ? v[i + 1 < N ? i + 1 : 0] : 0.f, i + 2 < N ? v[i + 2 < N ? i + 2 : 0] : 0.f,
                                  i + 3 < N ? v[i + 3 < N ? i + 3 : 0] : 0.f);
        if (lane < 4) red[wave][i + lane] = s;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = red[0][i] + red[1][i] + red[2][i] + red[3][i];
}

template <int NCH, int R, bool BF16>
__global__ void __launch_bounds__(kThreads) ln_modulate_bwd_kernel(const LnModBwdParams p) {
    static_assert(3 * R <= 16, "row sums per exchange");
    __shared__ float red1[4][16], red2[4][16];   // written again only after the other one's barrier
    const int D = p.D;
    const int64_t grp = blockIdx.x / p.sums.chunks_per_group;
    const int64_t lo = grp * p.rows_per_group + (int64_t)(blockIdx.x % p.sums.chunks_per_group) * p.sums.chunk;
    const int64_t end = (grp + 1) * p.rows_per_group;
    const int64_t hi = lo + p.sums.chunk < end ? lo + p.sums.chunk : end;
    const float inv_d = 1.0f / D;
    float sc[NCH][8], asc[NCH][8], ash[NCH][8];
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int off = 8 * ((int)threadIdx.x + kThreads * c);
        unpack8<BF16>(off < D ? *reinterpret_cast<const uint4*>(p.scale + grp * D + off) : make_uint4(0u, 0u, 0u, 0u), sc[c]);
#pragma unroll
        for (int i = 0; i < 8; ++i) { sc[c][i] += 1.0f; asc[c][i] = ash[c][i] = 0.f; }
    }
    for (int64_t row0 = lo; row0 < hi; row0 += R) {      // the same for all threads: the barriers below are met by all
        float x[R][NCH][8], dy[R][NCH][8], s[3 * R], m[R];
        uint4 skip[R][NCH];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            m[r] = 0.f;
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                const int off = 8 * ((int)threadIdx.x + kThreads * c);
                const bool in = off < D && row0 + r < hi;
                const int64_t at = (row0 + r) * D + off;
                const uint4 z = make_uint4(0u, 0u, 0u, 0u);
                unpack8<BF16>(in ? *reinterpret_cast<const uint4*>(p.x + at) : z, x[r][c]);
                unpack8<BF16>(in ? *reinterpret_cast<const uint4*>(p.dy + at) : z, dy[r][c]);
                skip[r][c] = in && p.dskip ? *reinterpret_cast<const uint4*>(p.dskip + at) : z;
#pragma unroll
                for (int i = 0; i < 8; ++i) m[r] += x[r][c][i];
            }
        }
        block_sums<R>(m, red1);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            s[3 * r] = s[3 * r + 1] = s[3 * r + 2] = 0.f;
            m[r] *= inv_d;
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                const bool in = 8 * ((int)threadIdx.x + kThreads * c) < D;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float xc = in ? x[r][c][i] - m[r] : 0.f, dn = dy[r][c][i] * sc[c][i];
                    x[r][c][i] = xc;
                    s[3 * r] += xc * xc; s[3 * r + 1] += dn; s[3 * r + 2] += dn * xc;
                }
            }
        }
        block_sums<3 * R>(s, red2);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            // a row past the end has no variance: with eps = 0 its rsqrt is inf, and 0 inf would reach the column sums
            const float rs = row0 + r < hi ? rsqrtf(s[3 * r] * inv_d + p.eps) : 0.f;
            const float m1 = s[3 * r + 1] * inv_d, m2 = s[3 * r + 2] * inv_d * rs;
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                const int off = 8 * ((int)threadIdx.x + kThreads * c);
                float dx[8];
                unpack8<BF16>(skip[r][c], dx);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float n = x[r][c][i] * rs;
                    dx[i] += rs * (dy[r][c][i] * sc[c][i] - m1 - n * m2);
                    asc[c][i] += dy[r][c][i] * n;
                    ash[c][i] += dy[r][c][i];
                }
                if (off < D && row0 + r < hi) *reinterpret_cast<uint4*>(p.dx + (row0 + r) * D + off) = pack8<BF16>(dx);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int off = 8 * ((int)threadIdx.x + kThreads * c);
        if (off >= D) continue;
        store_column_sums<BF16>(p.sums, 0, 2, D, off, ash[c]);
        store_column_sums<BF16>(p.sums, 1, 2, D, off, asc[c]);
    }
}

typedef void (*ln_bwd_kernel_t)(const LnModBwdParams);
template <bool BF16>
ln_bwd_kernel_t pick_ln_bwd(int d) {
    switch ((d + 8 * kThreads - 1) / (8 * kThreads)) {
        case 1: return ln_modulate_bwd_kernel<1, 4, BF16>;
        case 2: return ln_modulate_bwd_kernel<2, 2, BF16>;
        case 3: return ln_modulate_bwd_kernel<3, 1, BF16>;
        case 4: return ln_modulate_bwd_kernel<4, 1, BF16>;
        default: return nullptr;
    }
}

struct GatedBwdParams {
    const uint16_t *dy, *res, *gate;             // [rows, D], [rows, D], [groups, D]
    uint16_t* dres;                              // [rows, D]
    ColumnSums sums;                             // dgate
    int D, rows_per_group;
};

// grid (chunks, columns / 2048)
template <bool BF16>
__global__ void __launch_bounds__(kThreads) gated_residual_bwd_kernel(const GatedBwdParams p) {
    const int D = p.D, off = 8 * ((int)threadIdx.x + kThreads * (int)blockIdx.y);
    if (off >= D) return;
    const int64_t grp = blockIdx.x / p.sums.chunks_per_group;
    const int64_t lo = grp * p.rows_per_group + (int64_t)(blockIdx.x % p.sums.chunks_per_group) * p.sums.chunk;
    const int64_t end = (grp + 1) * p.rows_per_group;
    const int64_t hi = lo + p.sums.chunk < end ? lo + p.sums.chunk : end;
    float gate[8], sum[8];
    unpack8<BF16>(*reinterpret_cast<const uint4*>(p.gate + grp * D + off), gate);
#pragma unroll
    for (int i = 0; i < 8; ++i) sum[i] = 0.f;
    for (int64_t row0 = lo; row0 < hi; row0 += 4) {
        uint4 wy[4], wr[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t row = row0 + r < hi ? row0 + r : hi - 1;
            wy[r] = *reinterpret_cast<const uint4*>(p.dy + row * D + off);
            wr[r] = *reinterpret_cast<const uint4*>(p.res + row * D + off);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (row0 + r >= hi) break;
            float dy[8], res[8], d[8];
            unpack8<BF16>(wy[r], dy);
            unpack8<BF16>(wr[r], res);
#pragma unroll
            for (int i = 0; i < 8; ++i) { d[i] = dy[i] * gate[i]; sum[i] += dy[i] * res[i]; }
            *reinterpret_cast<uint4*>(p.dres + (row0 + r) * D + off) = pack8<BF16>(d);
        }
    }
    store_column_sums<BF16>(p.sums, 0, 1, D, off, sum);
}

// ------------------------------------------------------------------------------------------------ modulation vectors
// The block's three modulation MLPs  m = W2 W1 silu(emb) + lora  (networks/minimal_v4_dit.py:1131-1162) for a handful of rows
// (one per batch row and frame), and their tangents  W2 W1 (silu'(emb) temb) + tlora  as rows of the same products.  What bounds
// them is reading the weights once (12 MB at 2B: 2 us) and the launches: one launch per layer for all three MLPs, instead of five
// to eight library launches for each.  A wavefront forms a 16 x 16 tile (outputs x rows) on v_mfma_f32_16x16x32, its operands read
// straight from memory, 16 bytes a lane (both operands with the same k order, so that order is free).  The first layer has few
// outputs and a long k: sixteen wavefronts share a tile's k and add their parts in LDS, else 48 wavefronts would read all weights.  All loads of a
// wavefront are in flight before the first product, with no branch that differs between lanes among them: with eight wavefronts and one load after the other (a branch
// around a missing row's) the layers took 14.4 and 6.8 us inside a network on one image, now 8.5 and 6.0, of which silu, formed by each workgroup for itself, is some 3.
// Measured per block (2048 channels, in a replayed graph): one row 46 -> 16 us, 24 rows 72 -> 15, 5 rows with tangents 219 -> 14;
// outside a graph the launches count too: a 28-block network on one image 24.0 -> 20.4 ms.
struct ModulationParams {
    const uint16_t *emb, *temb;                  // [rows, K]; temb may be null (it does not move)
    const uint16_t *lora, *tlora;                // [rows, 3 D]; tlora may be null
    const uint16_t *w1[3], *w2[3];               // [hidden, K], [3 D, hidden]
    uint16_t* h;                                 // [3, rows_all, hidden]: the first layer's outputs
    uint16_t *out, *tout;                        // [3 MLPs, 3 vectors, rows, D]
    int rows, rows_all, K, hidden, D;            // rows_all = rows, or twice that with tangents (second half)
};

template <bool BF16> struct Half8;
template <> struct Half8<true> {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    typedef float v4f __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ v4f mfma(uint4 a, uint4 b, v4f c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
    }
};
template <> struct Half8<false> {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    typedef float v4f __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ v4f mfma(uint4 a, uint4 b, v4f c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
    }
};

constexpr int kModSplit = 16;      // wavefronts that share a first-layer tile
constexpr int kModLoads = 4;       // k steps of a wavefront whose loads are in flight together, first layer (twice as many: second)
// grid (3 hidden / 16, ceil(rows_all / 16)), 64 kModSplit threads
template <bool BF16>
__global__ void __launch_bounds__(64 * kModSplit) modulation_hidden_kernel(const ModulationParams p) {
    typedef typename Half8<BF16>::v4f v4f;
    __shared__ float4 part[kModSplit][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tiles = p.hidden / 16, mod = blockIdx.x / tiles, n0 = (blockIdx.x % tiles) * 16;
    const int row = blockIdx.y * 16 + (lane & 15);
    const bool live = row < p.rows_all, tangent = row >= p.rows, moves = p.rows_all > p.rows && p.temb;
    const uint16_t* w = (mod == 0 ? p.w1[0] : mod == 1 ? p.w1[1] : p.w1[2]) + (int64_t)(n0 + (lane & 15)) * p.K;
    // (a row that is not there reads row 0 and forms a column that nobody reads)
    const int64_t at = live ? (int64_t)(tangent ? row - p.rows : row) * p.K : 0;
    const uint16_t *e = p.emb + at, *te = moves ? p.temb + at : nullptr;
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 32 * wave; k0 < p.K; k0 += 32 * kModSplit * kModLoads) {
        uint4 a[kModLoads], x[kModLoads], tx[kModLoads];
#pragma unroll
        for (int i = 0; i < kModLoads; ++i) {
            a[i] = x[i] = tx[i] = make_uint4(0u, 0u, 0u, 0u);
            if (k0 + 32 * kModSplit * i < p.K) {       // (K is a multiple of 32: the same in all lanes)
                const int k = k0 + 32 * kModSplit * i + 8 * (lane >> 4);
                a[i] = *reinterpret_cast<const uint4*>(w + k);
                x[i] = *reinterpret_cast<const uint4*>(e + k);
                if (moves) tx[i] = *reinterpret_cast<const uint4*>(te + k);
            }
        }
#pragma unroll
        for (int i = 0; i < kModLoads; ++i) {
            float f[8], sig[8];
            unpack8<BF16>(x[i], f);
#pragma unroll
            for (int j = 0; j < 8; ++j) sig[j] = 1.0f / (1.0f + __expf(-f[j]));
            if (moves) {
                float t[8];
                unpack8<BF16>(tx[i], t);
#pragma unroll
                for (int j = 0; j < 8; ++j) f[j] = tangent ? t[j] * (sig[j] * (1.0f + f[j] * (1.0f - sig[j]))) : f[j] * sig[j];
            } else {         // (emb does not move: its tangent's activations are zeros, whatever its values)
#pragma unroll
                for (int j = 0; j < 8; ++j) f[j] = tangent ? 0.f : f[j] * sig[j];
            }
            acc = Half8<BF16>::mfma(a[i], pack8<BF16>(f), acc);
        }
    }
    part[wave][lane] = make_float4(acc[0], acc[1], acc[2], acc[3]);
    __syncthreads();
    if (wave == 0 && live) {
        float f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kModSplit; ++i) { const float4 x = part[i][lane]; f[0] += x.x; f[1] += x.y; f[2] += x.z; f[3] += x.w; }
        const uint4 o = pack8<BF16>(f);
        *reinterpret_cast<uint2*>(p.h + ((int64_t)mod * p.rows_all + row) * p.hidden + n0 + 4 * (lane >> 4)) = make_uint2(o.x, o.y);
    }
}

// grid (ceil(9 D / 64), ceil(rows_all / 16)), 256 threads: four tiles
template <bool BF16>
__global__ void __launch_bounds__(kThreads) modulation_out_kernel(const ModulationParams p) {
    typedef typename Half8<BF16>::v4f v4f;
    const int lane = threadIdx.x & 63;
    const int tile = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6), tiles = 3 * p.D / 16, mod = tile / tiles;
    if (mod >= 3) return;
    const int n0 = (tile % tiles) * 16, row = blockIdx.y * 16 + (lane & 15);
    const bool live = row < p.rows_all, tangent = row >= p.rows;
    const uint16_t* w = (mod == 0 ? p.w2[0] : mod == 1 ? p.w2[1] : p.w2[2]) + (int64_t)(n0 + (lane & 15)) * p.hidden;
    const uint16_t* h = p.h + ((int64_t)mod * p.rows_all + (live ? row : 0)) * p.hidden;
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < p.hidden; k0 += 64 * kModLoads) {
        uint4 a[2 * kModLoads], b[2 * kModLoads];
#pragma unroll
        for (int i = 0; i < 2 * kModLoads; ++i) {
            a[i] = b[i] = make_uint4(0u, 0u, 0u, 0u);
            if (k0 + 32 * i < p.hidden) {
                const int k = k0 + 32 * i + 8 * (lane >> 4);
                a[i] = *reinterpret_cast<const uint4*>(w + k);
                b[i] = *reinterpret_cast<const uint4*>(h + k);
            }
        }
#pragma unroll
        for (int i = 0; i < 2 * kModLoads; ++i) acc = Half8<BF16>::mfma(a[i], b[i], acc);
    }
    if (!live) return;
    const int n = n0 + 4 * (lane >> 4), r = tangent ? row - p.rows : row;      // D is a multiple of 16: a tile is in one vector
    const uint16_t* add = tangent ? p.tlora : p.lora;
    float f[8] = {acc[0], acc[1], acc[2], acc[3], 0.f, 0.f, 0.f, 0.f};
    if (add) {
        const uint2 x = *reinterpret_cast<const uint2*>(add + (int64_t)r * 3 * p.D + n);
        float l[8];
        unpack8<BF16>(make_uint4(x.x, x.y, 0u, 0u), l);
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] += l[i];
    }
    const uint4 o = pack8<BF16>(f);
    const int vec = n / p.D;
    uint16_t* to = (tangent ? p.tout : p.out) + ((int64_t)(3 * mod + vec) * p.rows + r) * p.D + (n - vec * p.D);
    *reinterpret_cast<uint2*>(to) = make_uint2(o.x, o.y);
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }
bool dtype_ok(int dtype) { return dtype == COSMOS_ATTN_BF16 || dtype == COSMOS_ATTN_FP16; }
int launched() { return hipGetLastError() == hipSuccess ? COSMOS_ATTN_OK : COSMOS_ATTN_LAUNCH_FAILED; }

template <typename Desc>
bool rows_ok(const Desc* d) {
    return d && d->rows > 0 && d->D > 0 && d->rows_per_group > 0 && d->D % 8 == 0 && d->rows % d->rows_per_group == 0;
}
template <typename Desc>
void fill_ln(LnModParams& p, const Desc* d) {
    p.x = (const uint16_t*)d->x; p.tx = (const uint16_t*)d->tx;
    p.shift = (const uint16_t*)d->shift; p.scale = (const uint16_t*)d->scale;
    p.tshift = (const uint16_t*)d->tshift; p.tscale = (const uint16_t*)d->tscale;
    p.y = (uint16_t*)d->y; p.ty = (uint16_t*)d->ty;
    p.rows = d->rows; p.D = d->D; p.rows_per_group = d->rows_per_group; p.eps = d->eps;
}
template <bool GATED>
int launch_ln(const LnModParams& p, int dtype, void* stream) {
    const bool bf16 = dtype == COSMOS_ATTN_BF16;
    ln_kernel_t fn = p.tx ? (bf16 ? pick_ln<true, true, GATED>(p.D) : pick_ln<true, false, GATED>(p.D))
                          : (bf16 ? pick_ln<false, true, GATED>(p.D) : pick_ln<false, false, GATED>(p.D));
    const int64_t blocks = (p.rows + kThreads / 64 - 1) / (kThreads / 64);
    if (!fn || blocks > 0x7FFFFFFF) return COSMOS_ATTN_BAD_SHAPE;
    hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(kThreads), 0, (hipStream_t)stream, p);
    return launched();
}
template <typename Desc>
int launch_gated(const Desc* d, void* stream) {
    GatedResidualParams p;
    p.x = (const uint16_t*)d->x; p.tx = (const uint16_t*)d->tx; p.res = (const uint16_t*)d->res; p.tres = (const uint16_t*)d->tres;
    p.gate = (const uint16_t*)d->gate; p.tgate = (const uint16_t*)d->tgate;
    p.out = (uint16_t*)d->out; p.tout = (uint16_t*)d->tout;
    p.chunks = d->rows * (d->D / 8); p.D = d->D; p.rows_per_group = d->rows_per_group;
    const int64_t blocks = (p.chunks + kThreads - 1) / kThreads;
    if (blocks > 0x7FFFFFFF) return COSMOS_ATTN_BAD_SHAPE;
    const bool bf16 = d->dtype == COSMOS_ATTN_BF16;
    auto fn = d->tx ? (bf16 ? gated_residual_kernel<true, true> : gated_residual_kernel<true, false>)
                    : (bf16 ? gated_residual_kernel<false, true> : gated_residual_kernel<false, false>);
    hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(kThreads), 0, (hipStream_t)stream, p);
    return launched();
}
int start_column_sums(ColumnSums& s, int64_t rows, int rows_per_group, int D, int vectors, void* out0, void* out1, void* workspace, size_t bytes) {
    plan_column_sums(s, rows, rows_per_group);
    s.out[0] = (uint16_t*)out0; s.out[1] = (uint16_t*)out1;
    s.part = (float*)workspace;
    const size_t need = column_sum_bytes(rows, rows_per_group, D, vectors);
    if (need && (!workspace || bytes < need || !aligned16(workspace))) return COSMOS_ATTN_WORKSPACE_TOO_SMALL;
    return COSMOS_ATTN_OK;
}
int finish_column_sums(const ColumnSums& s, int64_t groups, int D, int vectors, bool bf16, void* stream) {
    if (s.chunks_per_group > 1) {
        const dim3 grid((unsigned)groups, (unsigned)((D + 63) / 64), (unsigned)vectors);
        hipLaunchKernelGGL(bf16 ? column_sum_kernel<true> : column_sum_kernel<false>, grid, dim3(kThreads), 0, (hipStream_t)stream, s, vectors, D);
    }
    return launched();
}

}  // namespace

extern "C" {

COSMOS_ATTN_API int cosmos_ln_modulate(const cosmos_ln_modulate_desc* d, void* stream) {
    if (!d || d->abi_version != COSMOS_ATTN_ABI_VERSION) return COSMOS_ATTN_BAD_ARG;
    if (d->rows <= 0 || d->D <= 0 || d->rows_per_group <= 0 || !(d->eps >= 0.f)) return COSMOS_ATTN_BAD_ARG;
    if (!d->x || !d->y || !d->shift || !d->scale) return COSMOS_ATTN_BAD_ARG;
    if ((d->tx != nullptr) != (d->ty != nullptr)) return COSMOS_ATTN_BAD_ARG;
    if (!d->tx && (d->tshift || d->tscale)) return COSMOS_ATTN_BAD_ARG;
    if (!dtype_ok(d->dtype)) return COSMOS_ATTN_UNSUPPORTED;
    if (d->D % 8 != 0 || d->rows % d->rows_per_group != 0) return COSMOS_ATTN_BAD_SHAPE;
    if (d->D > 8192) return COSMOS_ATTN_UNSUPPORTED;
    const void* ptrs[] = {d->x, d->tx, d->shift, d->scale, d->tshift, d->tscale, d->y, d->ty};
    for (const void* q : ptrs) if (q && !aligned16(q)) return COSMOS_ATTN_BAD_STRIDE;
    LnModParams p = {};
    fill_ln(p, d);
    return launch_ln<false>(p, d->dtype, stream);
}

COSMOS_ATTN_API int cosmos_gated_residual_ln_modulate(const cosmos_gated_residual_ln_modulate_desc* d, void* stream) {
    if (!d || d->abi_version != COSMOS_ATTN_ABI_VERSION) return COSMOS_ATTN_BAD_ARG;
    if (d->rows <= 0 || d->D <= 0 || d->rows_per_group <= 0 || !(d->eps >= 0.f)) return COSMOS_ATTN_BAD_ARG;
    if (!d->x || !d->res || !d->gate || !d->out || !d->y || !d->shift || !d->scale) return COSMOS_ATTN_BAD_ARG;
    const bool tangent = d->tx != nullptr;
    if ((d->tres != nullptr) != tangent || (d->tout != nullptr) != tangent || (d->ty != nullptr) != tangent) return COSMOS_ATTN_BAD_ARG;
    if (!tangent && (d->tgate || d->tshift || d->tscale)) return COSMOS_ATTN_BAD_ARG;
    if (!dtype_ok(d->dtype)) return COSMOS_ATTN_UNSUPPORTED;
    if (d->D % 8 != 0 || d->rows % d->rows_per_group != 0) return COSMOS_ATTN_BAD_SHAPE;
    if (d->D > 8192) return COSMOS_ATTN_UNSUPPORTED;
    const void* ptrs[] = {d->x, d->tx, d->res, d->tres, d->gate, d->tgate, d->shift, d->scale, d->tshift, d->tscale, d->out, d->tout, d->y, d->ty};
    for (const void* q : ptrs) if (q && !aligned16(q)) return COSMOS_ATTN_BAD_STRIDE;
    LnModParams p = {};
    fill_ln(p, d);
    if (d->D > kMaxGatedLnD) {
        const int st = launch_gated(d, stream);
        p.x = (const uint16_t*)d->out; p.tx = (const uint16_t*)d->tout;
        return st == COSMOS_ATTN_OK ? launch_ln<false>(p, d->dtype, stream) : st;
    }
    p.res = (const uint16_t*)d->res; p.tres = (const uint16_t*)d->tres;
    p.gate = (const uint16_t*)d->gate; p.tgate = (const uint16_t*)d->tgate;
    p.out = (uint16_t*)d->out; p.tout = (uint16_t*)d->tout;
    return launch_ln<true>(p, d->dtype, stream);
}

COSMOS_ATTN_API int cosmos_gated_residual(const cosmos_gated_residual_desc* d, void* stream) {
    if (!d || d->abi_version != COSMOS_ATTN_ABI_VERSION) return COSMOS_ATTN_BAD_ARG;
    if (d->rows <= 0 || d->D <= 0 || d->rows_per_group <= 0) return COSMOS_ATTN_BAD_ARG;
    if (!d->x || !d->res || !d->gate || !d->out) return COSMOS_ATTN_BAD_ARG;
    const bool tangent = d->tx != nullptr;
    if ((d->tres != nullptr) != tangent || (d->tout != nullptr) != tangent || (!tangent && d->tgate)) return COSMOS_ATTN_BAD_ARG;
    if (!dtype_ok(d->dtype)) return COSMOS_ATTN_UNSUPPORTED;
    if (d->D % 8 != 0 || d->rows % d->rows_per_group != 0) return COSMOS_ATTN_BAD_SHAPE;
    const void* ptrs[] = {d->x, d->tx, d->res, d->tres, d->gate, d->tgate, d->out, d->tout};
    for (const void* q : ptrs) if (q && !aligned16(q)) return COSMOS_ATTN_BAD_STRIDE;
    return launch_gated(d, stream);
}

COSMOS_ATTN_API int cosmos_gelu(const cosmos_gelu_desc* d, void* stream) {
    if (!d || d->abi_version != COSMOS_ATTN_ABI_VERSION) return COSMOS_ATTN_BAD_ARG;
    if (d->n <= 0 || !d->h || !d->a || (d->th != nullptr) != (d->ta != nullptr)) return COSMOS_ATTN_BAD_ARG;
    if (!dtype_ok(d->dtype)) return COSMOS_ATTN_UNSUPPORTED;
    if (d->n % 8 != 0) return COSMOS_ATTN_BAD_SHAPE;
    const void* ptrs[] = {d->h, d->th, d->a, d->ta};
    for (const void* q : ptrs) if (q && !aligned16(q)) return COSMOS_ATTN_BAD_STRIDE;
    GeluParams p;
    p.h = (const uint16_t*)d->h; p.th = (const uint16_t*)d->th; p.a = (uint16_t*)d->a; p.ta = (uint16_t*)d->ta;
    p.chunks = d->n / 8;
    const int64_t blocks = (p.chunks + kThreads - 1) / kThreads;
    if (blocks > 0x7FFFFFFF) return COSMOS_ATTN_BAD_SHAPE;
    const bool bf16 = d->dtype == COSMOS_ATTN_BF16;
    auto fn = d->th ? (bf16 ? gelu_kernel<true, true> : gelu_kernel<true, false>)
                    : (bf16 ? gelu_kernel<false, true> : gelu_kernel<false, false>);
    hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(kThreads), 0, (hipStream_t)stream, p);
    return launched();
}

COSMOS_ATTN_API size_t cosmos_ln_modulate_bwd_workspace_bytes(const cosmos_ln_modulate_bwd_desc* d) {
    return rows_ok(d) ? column_sum_bytes(d->rows, d->rows_per_group, d->D, 2) : 0;
}

COSMOS_ATTN_API int cosmos_ln_modulate_bwd(const cosmos_ln_modulate_bwd_desc* d, void* workspace, size_t workspace_bytes, void* stream) {
    if (!d || d->abi_version != COSMOS_ATTN_ABI_VERSION) return COSMOS_ATTN_BAD_ARG;
    if (d->rows <= 0 || d->D <= 0 || d->rows_per_group <= 0 || !(d->eps >= 0.f)) return COSMOS_ATTN_BAD_ARG;
    if (!d->x || !d->scale || !d->dy || !d->dx || !d->dshift || !d->dscale) return COSMOS_ATTN_BAD_ARG;
    if (!dtype_ok(d->dtype)) return COSMOS_ATTN_UNSUPPORTED;
    if (!rows_ok(d)) return COSMOS_ATTN_BAD_SHAPE;
    if (d->D > 8192) return COSMOS_ATTN_UNSUPPORTED;
    const void* ptrs[] = {d->x, d->scale, d->dy, d->dskip, d->dx, d->dshift, d->dscale};
    for (const void* q : ptrs) if (q && !aligned16(q)) return COSMOS_ATTN_BAD_STRIDE;
    LnModBwdParams p;
    p.x = (const uint16_t*)d->x; p.dy = (const uint16_t*)d->dy; p.dskip = (const uint16_t*)d->dskip; p.scale = (const uint16_t*)d->scale;
    p.dx = (uint16_t*)d->dx; p.D = d->D; p.rows_per_group = d->rows_per_group; p.eps = d->eps;
    const bool bf16 = d->dtype == COSMOS_ATTN_BF16;
    const ln_bwd_kernel_t fn = bf16 ? pick_ln_bwd<true>(d->D) : pick_ln_bwd<false>(d->D);
    const int64_t groups = d->rows / d->rows_per_group;
    const int st = start_column_sums(p.sums, d->rows, d->rows_per_group, d->D, 2, d->dshift, d->dscale, workspace, workspace_bytes);
    if (st != COSMOS_ATTN_OK) return st;
    if (!fn || groups * p.sums.chunks_per_group > 0x7FFFFFFF) return COSMOS_ATTN_BAD_SHAPE;
    hipLaunchKernelGGL(fn, dim3((unsigned)(groups * p.sums.chunks_per_group)), dim3(kThreads), 0, (hipStream_t)stream, p);
    return finish_column_sums(p.sums, groups, d->D, 2, bf16, stream);
}

COSMOS_ATTN_API size_t cosmos_gated_residual_bwd_workspace_bytes(const cosmos_gated_residual_bwd_desc* d) {
    return rows_ok(d) ? column_sum_bytes(d->rows, d->rows_per_group, d->D, 1) : 0;
}

COSMOS_ATTN_API int cosmos_gated_residual_bwd(const cosmos_gated_residual_bwd_desc* d, void* workspace, size_t workspace_bytes, void* stream) {
    if (!d || d->abi_version != COSMOS_ATTN_ABI_VERSION) return COSMOS_ATTN_BAD_ARG;
    if (d->rows <= 0 || d->D <= 0 || d->rows_per_group <= 0) return COSMOS_ATTN_BAD_ARG;
    if (!d->dy || !d->res || !d->gate || !d->dres || !d->dgate) return COSMOS_ATTN_BAD_ARG;
    if (!dtype_ok(d->dtype)) return COSMOS_ATTN_UNSUPPORTED;
    if (!rows_ok(d)) return COSMOS_ATTN_BAD_SHAPE;
    const void* ptrs[] = {d->dy, d->res, d->gate, d->dres, d->dgate};
    for (const void* q : ptrs) if (!aligned16(q)) return COSMOS_ATTN_BAD_STRIDE;
    GatedBwdParams p;
    p.dy = (const uint16_t*)d->dy; p.res = (const uint16_t*)d->res; p.gate = (const uint16_t*)d->gate; p.dres = (uint16_t*)d->dres;
    p.D = d->D; p.rows_per_group = d->rows_per_group;
    const bool bf16 = d->dtype == COSMOS_ATTN_BF16;
    const int64_t groups = d->rows / d->rows_per_group, cols = ((int64_t)d->D + 8 * kThreads - 1) / (8 * kThreads);
    const int st = start_column_sums(p.sums, d->rows, d->rows_per_group, d->D, 1, d->dgate, nullptr, workspace, workspace_bytes);
    if (st != COSMOS_ATTN_OK) return st;
    if (groups * p.sums.chunks_per_group > 0x7FFFFFFF || d->D > 64 * 65535) return COSMOS_ATTN_BAD_SHAPE;
    const dim3 grid((unsigned)(groups * p.sums.chunks_per_group), (unsigned)cols);
    hipLaunchKernelGGL(bf16 ? gated_residual_bwd_kernel<true> : gated_residual_bwd_kernel<false>, grid, dim3(kThreads), 0, (hipStream_t)stream, p);
    return finish_column_sums(p.sums, groups, d->D, 1, bf16, stream);
}

COSMOS_ATTN_API size_t cosmos_ln_modulation_workspace_bytes(const cosmos_ln_modulation_desc* d) {
    if (!d || d->rows <= 0 || d->hidden <= 0) return 0;
    return (size_t)3 * d->rows * (d->tout ? 2 : 1) * d->hidden * sizeof(uint16_t);
}

COSMOS_ATTN_API int cosmos_ln_modulation(const cosmos_ln_modulation_desc* d, void* workspace, size_t workspace_bytes, void* stream) {
    if (!d || d->abi_version != COSMOS_ATTN_ABI_VERSION) return COSMOS_ATTN_BAD_ARG;
    if (d->rows <= 0 || d->K <= 0 || d->hidden <= 0 || d->D <= 0 || !d->emb || !d->lora || !d->out) return COSMOS_ATTN_BAD_ARG;
    if (!d->tout && (d->temb || d->tlora)) return COSMOS_ATTN_BAD_ARG;
    if (!dtype_ok(d->dtype)) return COSMOS_ATTN_UNSUPPORTED;
    if (d->K % 32 != 0 || d->hidden % 32 != 0 || d->D % 16 != 0) return COSMOS_ATTN_BAD_SHAPE;
    if (d->rows > 65536 || d->K > (1 << 20) || d->hidden > (1 << 20) || d->D > (1 << 20)) return COSMOS_ATTN_BAD_SHAPE;
    const void* ptrs[] = {d->emb, d->temb, d->lora, d->tlora, d->out, d->tout, d->w1[0], d->w1[1], d->w1[2], d->w2[0], d->w2[1], d->w2[2]};
    for (const void* q : ptrs) if (q && !aligned16(q)) return COSMOS_ATTN_BAD_STRIDE;
    ModulationParams p;
    for (int i = 0; i < 3; ++i) {
        if (!d->w1[i] || !d->w2[i]) return COSMOS_ATTN_BAD_ARG;
        p.w1[i] = (const uint16_t*)d->w1[i]; p.w2[i] = (const uint16_t*)d->w2[i];
    }
    if (!workspace || workspace_bytes < cosmos_ln_modulation_workspace_bytes(d) || !aligned16(workspace)) return COSMOS_ATTN_WORKSPACE_TOO_SMALL;
    p.emb = (const uint16_t*)d->emb; p.temb = (const uint16_t*)d->temb; p.lora = (const uint16_t*)d->lora; p.tlora = (const uint16_t*)d->tlora;
    p.h = (uint16_t*)workspace; p.out = (uint16_t*)d->out; p.tout = (uint16_t*)d->tout;
    p.rows = d->rows; p.rows_all = d->tout ? 2 * d->rows : d->rows; p.K = d->K; p.hidden = d->hidden; p.D = d->D;
    const bool bf16 = d->dtype == COSMOS_ATTN_BF16;
    const unsigned row_tiles = (unsigned)((p.rows_all + 15) / 16);
    hipLaunchKernelGGL(bf16 ? modulation_hidden_kernel<true> : modulation_hidden_kernel<false>, dim3((unsigned)(3 * (p.hidden / 16)), row_tiles),
                       dim3(64 * kModSplit), 0, (hipStream_t)stream, p);
    hipLaunchKernelGGL(bf16 ? modulation_out_kernel<true> : modulation_out_kernel<false>, dim3((unsigned)((9 * (p.D / 16) + 3) / 4), row_tiles),
                       dim3(kThreads), 0, (hipStream_t)stream, p);
    return launched();
}

}  // extern "C"
