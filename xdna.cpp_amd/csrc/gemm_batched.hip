// Batched GEMV on the matrix cores for gfx950: y[m] = W x[m] for many
// activation rows m (a prompt's micro-batch), every weight type.
//
// With M rows the path is a contraction of 2 M N K operations over N row_bytes
// of weights, so past a few rows the products bound it, not HBM: one
// v_dot8/v_dot4 row kernel per 1 or 8 activations ran at 10-35 TFLOP/s.  Here
// each lane decodes 8 weights at a time straight into an MFMA operand and
// every decoded operand meets 32 or 64 activation rows.
//
// Arithmetic.  Codes times integer sub-block scales are exact in f16 (11
// bits) for Q3_K, Q4_K, Q5_K, IQ3_S, and for IQ3_XXS / IQ2_S with grids up to
// 66; Q6_K and IQ4_XS need 12 bits and take a second operand with the exact
// remainder, which meets the activations' high plane only (its product with the
// low one is at most 2^-22 of the term); Q4_0 keeps its bare codes and applies
// the block scale to each block's sum.  Activations are split into two f16
// planes, hi = f16(x s) and lo = f16(x s - hi) with s a power of two per row that
// puts its largest |x| in [2^14, 2^15): x s = hi + lo to 2^-23 of x, or 2^-25
// absolute, i.e. 2^-39 of the row's largest value.  Products are exact in f32 and
// sums are f32 over 256 values (32 for Q4_0), scaled by the superblock's d and
// added in f32 over superblocks (FINE kernels: in f64).  This is more accurate
// than the 20- or 16-bit fixed point of the single-row kernels, except that those
// scale every 32 values by themselves: a row with a block of 32 whose largest
// value is more than 2^18 below the row's is wide, and a wavefront sums wide rows
// in f32 after its tiles, four to a pass over its weights, from the activations
// as they are.  (us with none, one and all of the rows wide: Q4_0 17408x5120 M =
// 37 48, 84, 403; IQ3_S 8192x8192 M = 64 45, 72, 459.  Every row's activations go
// through the vector memory path for 64 weight rows at a time.)
//
// Work split.  A workgroup of 4 wavefronts computes 256 output columns (weight
// rows) x 32 or 64 activation rows; a wavefront 64 columns as two 32-wide
// MFMA tiles, so that each activation operand read from LDS feeds two
// products.  K is walked in half superblocks of 8 operand steps: the
// activation planes of the next half travel to LDS directly (global_load_lds)
// and its weights to registers while this half is multiplied, and each step's
// operands are decoded dword by dword between the products of the step before
// (a sched_barrier after every product keeps that order: left alone, the
// compiler decodes a whole half first).  Where the tiles leave CUs idle the
// superblocks are split over gridDim.y segments whose f32 partials a second
// kernel adds in segment order.
//
// What bounds it (rocprof counters, cycles per SIMD or wavefront).  The matrix and
// the vector work of a SIMD's two wavefronts hardly overlap: at M = 512 Q6_K
// 4096x14336 has 172 k cycles of MFMA (32 each; two products, for Q6_K and IQ4_XS
// three, make one useful one) and 144 k of decode in the 328 k that a wavefront
// runs, Q4_0 17408x5120 174 k and 165 k in 318 k.  Q4_0 there has 544 workgroups for
// 512 places, and the last 32 take a round of their own: 292 us against 212.  At M
// = 37 (Q4_K 14336x4096) a workgroup has two superblocks, 15 k and 17 k cycles of
// the 45 k that it runs; the staging and the adding launch take 11 of 38 us.  us
// per call on MI355X (sequential or 8-row passes before): Q4_0 17408x5120 M = 512
// 293 (2710), Q6_K 4096x14336 M = 512 222 (6310), Q4_K 14336x4096 M = 37 35 (252).
#include "internal.h"
#include "kq_device.h"
#include "q4_0_layout.h"

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <type_traits>

namespace mi355x {
namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kGmWaves = 4;
constexpr int kGmThreads = 64 * kGmWaves;
constexpr int kGmNT = 2;                            // 32-wide column tiles per wavefront
constexpr int kGmCols = 32 * kGmNT * kGmWaves;      // weight rows per workgroup
constexpr int kGmHalfBytes = 512;                   // planes of one activation row's half superblock
constexpr int kGmMaxRows = 512;                     // activation rows per pass

struct GemmArgs {
    const uint8_t *W;
    int64_t N;
    int64_t row_bytes;
    int B;        // superblocks per row (Q4_0: of 8 blocks, the last may be partial)
    int blocks;   // Q4_0 blocks per row
    int M;
    int Mp;       // rows of the staged planes (M rounded up to the tile)
    int ntiles, mtiles;
    int per_seg;  // superblocks per segment
    int nseg;
    const uint8_t *planes;  // [superblock][half][Mp][512]
    const _Float16 *sums;   // [superblock][Mp][16]
    const float *unit;      // [Mp]: 1 / s of each row, negative for wide rows
    const float *x;         // the activations themselves, for wide rows
    int64_t x_stride;
    float *out;             // y, or the partials of segment 0
    int64_t out_stride;
    int64_t seg_stride;
    const uint32_t *grid;   // IQ3_XXS, IQ2_S
};

__device__ __forceinline__ f16x2 h2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ uint32_t u2(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ f16x2 h2s(float v) {
    return f16x2{static_cast<_Float16>(v), static_cast<_Float16>(v)};
}
__device__ __forceinline__ f16x2 pk_fma(f16x2 a, f16x2 b, f16x2 c) { return __builtin_elementwise_fma(a, b, c); }

// f16 pattern of 1024 (+ n for n < 1024 in the low bits), in both halves
constexpr uint32_t kH1024 = 0x64006400u;

// A staged 8-value run holds its values in the order 0, 2, 1, 3, 4, 6, 5, 7:
// the f16 pairs that come out of a dword of byte codes by masking are bytes
// (0, 2) and (1, 3).
__device__ __forceinline__ f16x8 frag8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    const u32x4 v{a, b, c, d};
    return __builtin_bit_cast(f16x8, v);
}

// ---- activation planes --------------------------------------------------------
// 16-byte slot of run r (0..15 of a half superblock) of plane p in the 512
// bytes of activation row m: the runs of a row are XORed by m so that the 32
// rows of an MFMA operand read 16 distinct slots.
__device__ __forceinline__ int gm_slot(int p, int r, int m) { return 16 * p + (r ^ (m & 15)); }
// position of sub-block sum j among the 8 of a superblock (the run order above)
__device__ __forceinline__ int gm_sum_pos(int j) { return (j & 4) | ((j & 1) << 1) | ((j >> 1) & 1); }

__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, dpp_mov<0xB1>(v));
    v = fmaxf(v, dpp_mov<0x4E>(v));
    v = fmaxf(v, dpp_mov<0x141>(v));
    v = fmaxf(v, dpp_mov<0x140>(v));
    v = fmaxf(v, dpp_mov<0x142, 0xA>(v));
    v = fmaxf(v, dpp_mov<0x143, 0xC>(v));
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// Four values of a row (`left` of the superblock's 256 exist).
__device__ __forceinline__ float4 load_x4(const float *x, int i0, int left, bool al16) {
    if (al16 && i0 + 3 < left) return *reinterpret_cast<const float4 *>(x + i0);
    float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i0 < left) f.x = x[i0];
    if (i0 + 1 < left) f.y = x[i0 + 1];
    if (i0 + 2 < left) f.z = x[i0 + 2];
    if (i0 + 3 < left) f.w = x[i0 + 3];
    return f;
}
__device__ __forceinline__ float abs_max4(const float4 &f) {
    return fmaxf(fmaxf(fabsf(f.x), fabsf(f.y)), fmaxf(fabsf(f.z), fabsf(f.w)));
}

// Scale of a row whose largest |x| is mx: s = 2^(14 - E) for mx in
// [2^E, 2^(E+1)), E >= -110 (smaller and all-zero rows take 2^124), and 1 / s.
__device__ __forceinline__ float row_scale(float mx, float &unit) {
    const int e = min(max(static_cast<int>(__builtin_bit_cast(uint32_t, mx) >> 23), 17), 254);  // biased E
    unit = __builtin_bit_cast(float, static_cast<uint32_t>(e - 14) << 23);
    return __builtin_bit_cast(float, static_cast<uint32_t>(268 - e) << 23);
}

struct XPlanes {
    uint2 hi, lo;         // this lane's 4 values of each plane, in run order
    _Float16 s_hi, s_lo;  // lanes 8j: sum of sub-block j (times s / 32)
};

// One superblock of one activation row by a whole wavefront: lane l converts
// values 4l .. 4l + 3.
__device__ __forceinline__ XPlanes convert_superblock(const float4 &f, float s) {
    const float w[4] = {f.x * s, f.y * s, f.z * s, f.w * s};
    _Float16 h[4], l[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        h[t] = static_cast<_Float16>(w[t]);
        l[t] = static_cast<_Float16>(w[t] - static_cast<float>(h[t]));
    }
    XPlanes r;
    r.hi = make_uint2(u2(f16x2{h[0], h[2]}), u2(f16x2{h[1], h[3]}));
    r.lo = make_uint2(u2(f16x2{l[0], l[2]}), u2(f16x2{l[1], l[3]}));
    float sum = (w[0] + w[1]) + (w[2] + w[3]);
    sum += dpp_mov<0xB1>(sum);
    sum += dpp_mov<0x4E>(sum);
    sum += dpp_mov<0x141>(sum);  // the 8 lanes of a 32-value sub-block
    sum *= 0.03125f;
    r.s_hi = static_cast<_Float16>(sum);
    r.s_lo = static_cast<_Float16>(sum - static_cast<float>(r.s_hi));
    return r;
}

// Stores a converted superblock: `half0` / `half1` the 512-byte rows of the
// two halves, `sums` the 16 f16 of the row.
template <class P, class S>
__device__ __forceinline__ void store_superblock(const XPlanes &c, int m, int lane, P half0, P half1, S sums) {
    const int r = lane >> 1;
    P row = lane < 32 ? half0 : half1;
    *reinterpret_cast<uint2 *>(row + 16 * gm_slot(0, r & 15, m) + 8 * (lane & 1)) = c.hi;
    *reinterpret_cast<uint2 *>(row + 16 * gm_slot(1, r & 15, m) + 8 * (lane & 1)) = c.lo;
    if ((lane & 7) == 0) {
        const int j = gm_sum_pos(lane >> 3);
        sums[j] = c.s_hi;
        sums[8 + j] = c.s_lo;
    }
}

// Planes, sums and units of the activation rows: one workgroup per row, its
// wavefronts taking the superblocks in turn; the first kPlKeep of each stay in
// registers between the row's maximum and the conversion.  A row is wide if a
// block of 32 has a largest scaled value below kWideBelow but not 0: the planes
// hold a value to 2^-25 at worst, which is then at most 2^-21 of the block's
// largest (the fixed point of the one-row kernels: 2^-18.9 for Q4_0, 2^-16 for the
// other types), or 2^-25 of it where f32 is the measure.
constexpr float kWideBelow = 0.0625f, kWideBelowF32 = 1.0f;
constexpr int kWideRows = 4;
constexpr int kPlThreads = 1024, kPlWavesG = kPlThreads / 64, kPlKeep = 4;
__global__ __launch_bounds__(kPlThreads) void gemm_planes_kernel(const float *x, int64_t x_stride, int64_t K,
                                                                 int x_al16, float wide_below, int Mp, int B,
                                                                 uint8_t *planes, _Float16 *sums, float *unit) {
    __shared__ float smax[kPlWavesG];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, m = blockIdx.x;
    const float *xr = x + m * x_stride;
    auto load = [&](int b) {
        const int64_t left = K - 256 * static_cast<int64_t>(b);
        return load_x4(xr + 256 * static_cast<int64_t>(b), 4 * lane, static_cast<int>(left < 256 ? left : 256), x_al16 != 0);
    };
    float4 keep[kPlKeep];
    float mx = 0.f;
#pragma unroll
    for (int k = 0; k < kPlKeep; ++k) {
        const int b = wave + kPlWavesG * k;
        keep[k] = b < B ? load(b) : make_float4(0.f, 0.f, 0.f, 0.f);
        mx = fmaxf(mx, abs_max4(keep[k]));
    }
    for (int b = wave + kPlWavesG * kPlKeep; b < B; b += kPlWavesG) mx = fmaxf(mx, abs_max4(load(b)));
    mx = wave_max(mx);
    if (lane == 0) smax[wave] = mx;
    __syncthreads();
    mx = wave_max(smax[lane & (kPlWavesG - 1)]);
    float u;
    const float s = row_scale(mx, u);
    int wide = 0;
    auto put = [&](int b, const float4 &f) {
        float bm = abs_max4(f) * s;  // of the block, in its 8 lanes
        bm = fmaxf(bm, dpp_mov<0xB1>(bm));
        bm = fmaxf(bm, dpp_mov<0x4E>(bm));
        bm = fmaxf(bm, dpp_mov<0x141>(bm));
        wide |= bm > 0.f && bm < wide_below;
        uint8_t *h0 = planes + (static_cast<int64_t>(2 * b) * Mp + m) * kGmHalfBytes;
        store_superblock(convert_superblock(f, s), m, lane, h0, h0 + static_cast<int64_t>(Mp) * kGmHalfBytes,
                         sums + (static_cast<int64_t>(b) * Mp + m) * 16);
    };
#pragma unroll
    for (int k = 0; k < kPlKeep; ++k) {
        const int b = wave + kPlWavesG * k;
        if (b < B) put(b, keep[k]);
    }
    for (int b = wave + kPlWavesG * kPlKeep; b < B; b += kPlWavesG) put(b, load(b));
    wide = __syncthreads_or(wide);
    if (threadIdx.x == 0) unit[m] = wide ? -u : u;
}

// ---- weight decode --------------------------------------------------------------
// Gw<TYPE>: the weights of one lane (one weight row) for slice s of a
// superblock as four f16 operands, operand p the run at position p of the
// slice (run_of).  dword(p, j) gives dword j of operand p: the run's values
// (0, 2), (1, 3), (4, 6), (5, 7); kWide types leave the exact remainder of
// code times scale in lo.  half, q, p and j are compile-time constants at
// every call (s = 4 half + 2 q + h, h = lane / 32); what the dwords share
// (scales) is written into each and kept by the compiler.  Codebook types
// read their kLooks table entries of operand p ahead of time (look).  d(regs)
// is the superblock's scale.
template <int TYPE>
struct Gw;

// (scale, min) bytes of sub-blocks 2c and 2c + 1 (scale_min_pair_k4)
__device__ __forceinline__ uint32_t scale_pair_k4(int c, const u32x4 &hd) {
    const uint32_t sh = 16u * static_cast<uint32_t>(c & 1);
    const uint32_t a2 = hd[1] >> sh, c2 = hd[3] >> sh;
    return c < 2 ? (a2 & 0x3F3Fu) : ((c2 & 0x0F0Fu) | ((a2 >> 2) & 0x3030u));
}
// byte B of w less BIAS as f16 in both halves
template <int B, int BIAS = 0>
__device__ __forceinline__ f16x2 byte_h2(uint32_t w) {
    return h2(__builtin_amdgcn_perm(w, w, 0x0C000C00u | (static_cast<uint32_t>(B) << 16) | B) | kH1024) -
           h2s(1024.f + BIAS);
}

// Q4_K, Q5_K: operands 0, 1 the low nibbles of code bytes 0-7, 8-15, operands
// 2, 3 the high nibbles.  The high codes stay in place (16 times the code) and
// the fma that removes the 1024 also applies the scale: sc <= 63, so every
// product and sum is exact.
template <bool Q5, class Regs>
__device__ __forceinline__ uint32_t k45_dword(const Regs &g, int half, int q, int p, int j) {
    const int c = 2 * half + q, i = 2 * (p & 1) + (j >> 1);
    const uint32_t sp = scale_pair_k4(c, g.hd);
    const f16x2 sc = p < 2 ? byte_h2<0>(sp) : byte_h2<1>(sp) * h2s(0.0625f);
    const uint32_t w = (j & 1) ? g.q[i] >> 8 : g.q[i];
    uint32_t a = (w & (p < 2 ? 0x000F000Fu : 0x00F000F0u)) | kH1024;
    if constexpr (Q5) {
        // high bit 2c of each qh byte to bit 4 of the low codes, bit 2c + 1
        // to bit 8 of the in-place high codes
        const uint32_t qh = g.qh[i];
        if (p < 2) {
            const uint32_t t = 2 * c <= 4 ? qh << (4 - 2 * c) : qh >> (2 * c - 4);
            a |= ((j & 1) ? t >> 8 : t) & 0x00100010u;
        } else {
            a |= ((j & 1) ? qh >> (2 * c + 1) : qh << (7 - 2 * c)) & 0x01000100u;
        }
    }
    return u2(pk_fma(h2(a), sc, sc * h2s(-1024.f)));
}
// the 8 sub-block mins of a superblock in run order
__device__ __forceinline__ f16x8 k4_mins(const u32x4 &hd) {
    const uint32_t m0 = hd[2] & 0x3F3F3F3Fu;
    const uint32_t m1 = ((hd[3] >> 4) & 0x0F0F0F0Fu) | ((hd[2] >> 2) & 0x30303030u);
    const f16x2 k = h2s(1024.f);
    return frag8(u2(h2((m0 & 0x00FF00FFu) | kH1024) - k), u2(h2(((m0 >> 8) & 0x00FF00FFu) | kH1024) - k),
                 u2(h2((m1 & 0x00FF00FFu) | kH1024) - k), u2(h2(((m1 >> 8) & 0x00FF00FFu) | kH1024) - k));
}

// the mins of sub-blocks 2c (low byte) and 2c + 1
__device__ __forceinline__ uint32_t min_pair_k4(int c, const u32x4 &hd) {
    const uint32_t sh = 16u * static_cast<uint32_t>(c & 1);
    const uint32_t b2 = hd[2] >> sh, c2 = hd[3] >> sh;
    return c < 2 ? (b2 & 0x3F3Fu) : (((c2 >> 4) & 0x0F0Fu) | ((b2 >> 2) & 0x3030u));
}

template <>
struct Gw<MI355X_TYPE_Q4_K> {
    static constexpr bool kWide = false, kMins = true;
    static constexpr int kLooks = 0;
    using Regs = Kq<MI355X_TYPE_Q4_K>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_Q4_K>::load(r, b, s); }
    __device__ static float d(const Regs &g) { return half_f(g.hd[0] & 0xFFFF); }
    __device__ static void dword(const Regs &g, int half, int q, int p, int j, const uint2 *, uint32_t &hi, uint32_t &) {
        hi = k45_dword<false>(g, half, q, p, j);
    }
};
template <>
struct Gw<MI355X_TYPE_Q5_K> {
    static constexpr bool kWide = false, kMins = true;
    static constexpr int kLooks = 0;
    using Regs = Kq<MI355X_TYPE_Q5_K>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_Q5_K>::load(r, b, s); }
    __device__ static float d(const Regs &g) { return half_f(g.hd[0] & 0xFFFF); }
    __device__ static void dword(const Regs &g, int half, int q, int p, int j, const uint2 *, uint32_t &hi, uint32_t &) {
        hi = k45_dword<true>(g, half, q, p, j);
    }
};

// v * sc split into its f16 rounding and the exact remainder
__device__ __forceinline__ void wide_mul(f16x2 v, f16x2 sc, uint32_t &hi, uint32_t &lo) {
    const f16x2 p = v * sc;
    hi = u2(p);
    lo = u2(pk_fma(v, sc, -p));
}
// w << sh for sh >= 0, else w >> -sh
__device__ __forceinline__ uint32_t shift(uint32_t w, int sh) { return sh >= 0 ? w << sh : w >> -sh; }

template <>
struct Gw<MI355X_TYPE_Q6_K> {
    static constexpr bool kWide = true, kMins = false;
    static constexpr int kLooks = 0;
    using Regs = Kq<MI355X_TYPE_Q6_K>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_Q6_K>::load(r, b, s); }
    __device__ static float d(const Regs &g) { return half_f(g.d); }
    __device__ static void dword(const Regs &g, int, int, int p, int j, const uint2 *, uint32_t &hi, uint32_t &lo) {
        const uint32_t sw = g.sw4 ^ 0x80808080u;  // int8 scales + 128
        const f16x2 sc = p == 0   ? byte_h2<0, 128>(sw)
                         : p == 1 ? byte_h2<1, 128>(sw)
                         : p == 2 ? byte_h2<2, 128>(sw)
                                  : byte_h2<3, 128>(sw);
        // nibble p / 2 of the first (p even) or second ql run, bits 2p of qh above it
        const int w = j >> 1, o = 8 * (j & 1);
        const uint32_t A = (p & 1) ? g.qb[w] : g.qa[w];
        const uint32_t c = ((A >> (4 * (p >> 1) + o)) & 0x000F000Fu) | (shift(g.qh[w], 4 - 2 * p - o) & 0x00300030u);
        wide_mul(h2(c | kH1024) - h2s(1024.f + 32.f), sc, hi, lo);
    }
};

template <>
struct Gw<MI355X_TYPE_Q3_K> {
    static constexpr bool kWide = false, kMins = false;
    static constexpr int kLooks = 0;
    // as Kq<Q3_K>::Regs with both halves of the slice's 8 hmask bytes
    struct Regs {
        u32x2 q, hm, sw01;
        uint32_t sw2, d;
    };
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) {
        const GPos p = gpos(r, 110, b, s);
        const uint32_t k = static_cast<uint32_t>(s & 3);
        const u32x2 q = ld64(r, p.base + 12 * p.m);
        const uint32_t h0 = ld32(r, p.base + 12 * (k * p.g + p.bl) + 8);
        const uint32_t h1 = ld32(r, p.base + 12 * ((4 + k) * p.g + p.bl) + 8);
        const u32x3 sc = ld96(r, p.base + 96 * p.g + 12 * p.bl);
        return {q, u32x2{h0, h1}, u32x2{sc[0], sc[1]}, sc[2], ld16(r, p.d)};
    }
    __device__ static float d(const Regs &g) { return half_f(g.d); }
    __device__ static void dword(const Regs &g, int half, int q, int p, int j, const uint2 *, uint32_t &hi, uint32_t &) {
        // the four 6-bit scales in one word, bytes in run order 0, 2, 1, 3
        // (KqDg<Q3_K>); kk = q, hh = half
        const uint32_t Lw = q ? g.sw01[1] : g.sw01[0];
        const uint32_t Hw = g.sw2 >> (8 * q + 4 * half);
        const uint32_t SC = ((Lw >> (4 * half)) & 0x0F0F0F0Fu) | ((Hw & 0x00030003u) << 4) | ((Hw & 0x000C000Cu) << 10);
        const f16x2 sc = p == 0   ? byte_h2<0, 32>(SC)
                         : p == 1 ? byte_h2<2, 32>(SC)
                         : p == 2 ? byte_h2<1, 32>(SC)
                                  : byte_h2<3, 32>(SC);
        // code bits in place (4^p times the code), the hmask bit above them:
        // bit 4 half + p of the byte to bit 2p + 2
        const int w = j >> 1, o = 8 * (j & 1);
        const uint32_t m2 = 0x00030003u << (2 * p), mh = 0x00040004u << (2 * p);
        const float f = static_cast<float>(1 << (2 * p));
        const uint32_t a = ((g.q[w] >> o) & m2) | (shift(g.hm[w], p + 2 - 4 * half - o) & mh) | kH1024;
        hi = u2((h2(a) - h2s(1024.f + 4.f * f)) * (sc * h2s(1.f / f)));
    }
};

template <>
struct Gw<MI355X_TYPE_IQ4_XS> {
    static constexpr bool kWide = true, kMins = false;
    static constexpr int kLooks = 0;
    using Regs = Kq<MI355X_TYPE_IQ4_XS>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_IQ4_XS>::load(r, b, s); }
    __device__ static float d(const Regs &g) { return half_f(g.hd[0] & 0xFFFF); }
    __device__ static void dword(const Regs &g, int half, int q, int p, int j, const uint2 *, uint32_t &hi, uint32_t &lo) {
        const uint32_t s = static_cast<uint32_t>(4 * half + 2 * q) + (__lane_id() >> 5);
        const uint32_t sh = g.hd[0] >> 16;
        const uint32_t ls = ((g.hd[1] >> (4 * s)) & 15u) | (((sh >> (2 * s)) & 3u) << 4);
        const uint32_t w = g.q[2 * (p & 1) + (j >> 1)];
        const uint32_t a = Kq<MI355X_TYPE_IQ4_XS>::lookup((p < 2 ? w : w >> 4) & 0x0F0F0F0Fu);
        // the codebook bytes are kvalues + 128
        wide_mul(h2((((j & 1) ? a >> 8 : a) & 0x00FF00FFu) | kH1024) - h2s(1024.f + 128.f), byte_h2<0, 32>(ls), hi, lo);
    }
};

// Dword j of 8 grid magnitudes with the signs of byte `signs`, times sc: m the
// f16 pair of values (0, 2), (1, 3), (4, 6) or (5, 7); bit i of the byte and
// its copy at 14 + i meet in the sign bits of one pair.
__device__ __forceinline__ uint32_t signed_dword(uint32_t m, uint32_t signs, int j, f16x2 sc) {
    const uint32_t t = signs | (signs << 14);
    return u2(h2(m ^ ((t << (j < 2 ? 15 - j : 13 - j)) & 0x80008000u)) * sc);
}

template <>
struct Gw<MI355X_TYPE_IQ3_S> {
    static constexpr bool kWide = false, kMins = false;
    static constexpr int kLooks = 2;
    using Regs = Kq<MI355X_TYPE_IQ3_S>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_IQ3_S>::load(r, b, s); }
    __device__ static float d(const Regs &g) { return half_f(g.d); }
    __device__ static uint2 look(const Regs &g, int p, int k, const uint2 *tab) {
        return tab[byte_u(g.qs[p >> 1], 2 * (p & 1) + k) | (((g.qh >> (2 * p + k)) & 1u) << 8)];
    }
    __device__ static void dword(const Regs &g, int, int, int p, int j, const uint2 *e, uint32_t &hi, uint32_t &) {
        const uint32_t n = (g.scb >> ((__lane_id() >> 5) * 4)) & 15u;
        hi = signed_dword((j & 1) ? e[j >> 1].y : e[j >> 1].x, byte_u(g.sg, p), j, byte_h2<0>(2 * n + 1));
    }
};

template <>
struct Gw<MI355X_TYPE_IQ3_XXS> {
    static constexpr bool kWide = false, kMins = false;
    static constexpr int kLooks = 2;
    using Regs = Kq<MI355X_TYPE_IQ3_XXS>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_IQ3_XXS>::load(r, b, s); }
    // (0.5 + n) / 2 = (2 n + 1) / 4
    __device__ static float d(const Regs &g) { return 0.25f * half_f(g.d); }
    __device__ static uint2 look(const Regs &g, int p, int k, const uint2 *tab) {
        return tab[byte_u(g.qs[p >> 1], 2 * (p & 1) + k)];
    }
    __device__ static void dword(const Regs &g, int, int, int p, int j, const uint2 *e, uint32_t &hi, uint32_t &) {
        hi = signed_dword((j & 1) ? e[j >> 1].y : e[j >> 1].x, ksigns((g.aux >> (7 * p)) & 127u), j,
                          byte_h2<0>(2 * (g.aux >> 28) + 1));
    }
};

template <>
struct Gw<MI355X_TYPE_IQ2_S> {
    static constexpr bool kWide = false, kMins = false;
    static constexpr int kLooks = 1;  // 8 magnitudes as bytes (f16 entries would take 16 KB and a workgroup of the CU)
    using Regs = Kq<MI355X_TYPE_IQ2_S>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_IQ2_S>::load(r, b, s); }
    // (0.5 + n) / 4 = (2 n + 1) / 8
    __device__ static float d(const Regs &g) { return 0.125f * half_f(g.d); }
    __device__ static uint2 look(const Regs &g, int p, int, const uint2 *tab) {
        return tab[byte_u(g.qs, p) | (((g.qh >> (2 * p)) & 3u) << 8)];
    }
    __device__ static void dword(const Regs &g, int, int, int p, int j, const uint2 *e, uint32_t &hi, uint32_t &) {
        const uint32_t b = j < 2 ? e[0].x : e[0].y;
        const uint32_t m = u2(h2((((j & 1) ? b >> 8 : b) & 0x00FF00FFu) | kH1024) - h2s(1024.f));
        hi = signed_dword(m, byte_u(g.sg, p), j, byte_h2<0>(2 * (p < 2 ? g.scb & 15u : g.scb >> 4) + 1));
    }
};

// Q4_0: "slice" s of a superblock is its block s; lanes h = 0, 1 load blocks
// 2q, 2q + 1 and exchange halves, so that both lanes of a row hold 8 bytes of
// each: operand (e, j) of the pair has values 16 j + 8 h + (0..7) of block
// 2q + e.
struct Q40Regs {
    u32x4 q;
    uint32_t d[2];  // fp16 of blocks 2q, 2q + 1
};
// dword j of operand i (0: low nibbles, 1: high) of block e
__device__ __forceinline__ uint32_t q40_dword(const Q40Regs &g, int e, int i, int j) {
    const auto sw = j < 2 ? __builtin_amdgcn_permlane32_swap(g.q[0], g.q[2], false, false)
                          : __builtin_amdgcn_permlane32_swap(g.q[1], g.q[3], false, false);
    const uint32_t v = static_cast<uint32_t>(sw[e]);
    const uint32_t a = (j & 1) ? v >> 8 : v;
    // resident nibbles are q - 8 in two's complement: flip the sign bit
    return i == 0 ? u2(h2((a & 0x000F000Fu) ^ 0x64086408u) + h2s(-1032.f))
                  : u2(pk_fma(h2((a & 0x00F000F0u) ^ 0x64806480u), h2s(0.0625f), h2s(-72.f)));
}

// entries of the LDS codebook table
constexpr int gm_table_entries(int type) {
    return type == MI355X_TYPE_IQ3_S     ? kIq3sGridSize
           : type == MI355X_TYPE_IQ3_XXS ? 256
           : type == MI355X_TYPE_IQ2_S   ? 1024
                                         : 1;
}
template <int TYPE>
__device__ __forceinline__ void stage_table(const GemmArgs &a, uint2 *tab) {
    if constexpr (TYPE == MI355X_TYPE_IQ3_S || TYPE == MI355X_TYPE_IQ3_XXS) {
        for (int i = threadIdx.x; i < gm_table_entries(TYPE); i += kGmThreads) {
            const uint32_t w = TYPE == MI355X_TYPE_IQ3_S ? kIq3sGrid[i] : a.grid[i];
            tab[i] = make_uint2(u2(h2((w & 0x00FF00FFu) | kH1024) - h2s(1024.f)),
                                u2(h2(((w >> 8) & 0x00FF00FFu) | kH1024) - h2s(1024.f)));
        }
    } else if constexpr (TYPE == MI355X_TYPE_IQ2_S) {
        for (int i = threadIdx.x; i < 1024; i += kGmThreads) tab[i] = make_uint2(a.grid[2 * i], a.grid[2 * i + 1]);
    }
}

// ---- kernel ----------------------------------------------------------------------
template <int TYPE>
struct RegsOf {
    using T = typename Gw<TYPE>::Regs;
};
template <>
struct RegsOf<MI355X_TYPE_Q4_0> {
    using T = Q40Regs;
};

__device__ __forceinline__ f32x16 mfma(const f16x8 &a, const f16x8 &b, const f32x16 &c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Copies one half superblock's planes of the workgroup's rows (BM x 512
// contiguous bytes) to LDS without passing through registers.
template <int BM>
__device__ __forceinline__ void copy_planes(const uint8_t *src, uint4 *dst, int wave, int lane) {
    constexpr int n = BM * kGmHalfBytes / 1024 / kGmWaves;
#pragma unroll
    for (int i = 0; i < n; ++i) {
        const int c = wave * n + i;
        __builtin_amdgcn_global_load_lds(
            reinterpret_cast<const __attribute__((address_space(1))) uint32_t *>(
                reinterpret_cast<uintptr_t>(src + 1024 * c + 16 * lane)),
            (__attribute__((address_space(3))) uint32_t *)(dst + 64 * c), 16, 0, 0);
    }
}

// All outstanding vector-memory operations of this wavefront done (the LDS
// copies above count there), then the workgroup barrier.
__device__ __forceinline__ void gm_barrier() {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();
}

// FINE: for calls whose one-row kernels sum f32 activations in f32 (IQ types).
// The low planes' products have sums of their own, so that they do not add
// roundings at the size of the high ones', and the sums of each half superblock
// (IQ2_S: quarter) are added in f64.  Error against 64 bits over K = 256 to 16384
// and N = 64 to 12000, f32 rows in brackets: IQ3_S and IQ3_XXS 1.0e-7 (1.2 to
// 1.4e-7), IQ2_S 0.8 to 0.9e-7 (0.9 to 1.2e-7), IQ4_XS 1.05e-7 (2.5e-7); without
// them 1.6 to 1.9e-7.  us, without -> with: IQ3_S 1024x4096 M = 9 18.9 -> 20.1,
// M = 512 61 -> 75; IQ2_S 17408x11008 M = 128 164 -> 331 (one GEMV each: 37, 1993
// and 4134).
template <int TYPE, int MT, bool FINE>
__global__ __launch_bounds__(kGmThreads, 2) void gemm_kernel(GemmArgs a) {
    constexpr int BM = 32 * MT, NT = kGmNT;
    constexpr bool Q40 = TYPE == MI355X_TYPE_Q4_0;
    constexpr bool MINS = TYPE == MI355X_TYPE_Q4_K || TYPE == MI355X_TYPE_Q5_K;
    using Regs = typename RegsOf<TYPE>::T;
    __shared__ uint4 xh0[BM * kGmHalfBytes / 16], xh1[BM * kGmHalfBytes / 16];
    __shared__ uint4 ssum[2][BM * 2];
    __shared__ uint2 tab[gm_table_entries(TYPE)];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int col = lane & 31, h = lane >> 5;
    // workgroups of one column tile run on one XCD (workgroup i runs on XCD
    // i % 8), so the tile's weights stay in that XCD's L2 for every row tile
    const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
    const int mt = seq % a.mtiles, ntile = (seq / a.mtiles) * 8 + xcd;
    if (ntile >= a.ntiles) return;
    const int m0 = mt * BM;
    const int64_t n0 = static_cast<int64_t>(ntile) * kGmCols + wave * (32 * NT);

    // the wavefront's rows of the matrix as one buffer (empty past N)
    const int64_t rows = a.N - n0 < 32 * NT ? (a.N - n0 > 0 ? a.N - n0 : 0) : 32 * NT;
    auto view = [&](int c, LaneRow (&v)[NT]) {  // of the lanes of column c of the tiles
        const uint8_t *base = a.W + (rows > 0 ? n0 : 0) * a.row_bytes;
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t *>(base), 0, static_cast<uint32_t>(rows * a.row_bytes), kBufferWord3);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const uint32_t rl = 32 * t + c;
            v[t].rsrc = rsrc;
            v[t].base = rl * static_cast<uint32_t>(a.row_bytes);
            if constexpr (!Q40) {
                constexpr KqLayout L = kq_layout(TYPE);
                const bool flipped = kq_row_flipped(reinterpret_cast<uintptr_t>(base) + v[t].base);
                if constexpr (L.grouped) {
                    v[t].P[0] = static_cast<uint32_t>(a.B);
                    v[t].P[1] = flipped ? 1u : 0u;
                } else {
#pragma unroll
                    for (int i = 0; i < 5; ++i)
                        v[t].P[i] = i < L.nfields ? static_cast<uint32_t>(kq_plane_start(L, i, a.B, flipped)) : 0u;
                }
            }
        }
    };
    LaneRow lr[NT];
    view(col, lr);
    // raw weights of slice (or blocks) 4 half + 2q + h of superblock b
    auto load_rows = [&](const LaneRow (&lr)[NT], int h, Regs (&r)[NT], int b, int half, int q) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if constexpr (Q40) {
                // rows have an even number of blocks, so a pair exists or not;
                // past the row (a partial last superblock) the scales are 0
                // and the codes whatever follows in the buffer
                const int b0 = 8 * b + 4 * half + 2 * q;
                const bool in = b0 < a.blocks;
                const int bc = in ? b0 : 0;
                r[t].q = ld128(lr[t], static_cast<uint32_t>(128 * b + 16 * h) + 16u * static_cast<uint32_t>(4 * half + 2 * q));
                const uint32_t F = static_cast<uint32_t>(a.blocks) >> 6;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const uint32_t be = static_cast<uint32_t>(bc + e);
                    const uint32_t slot = be < 64 * F ? (be & 63) * F + (be >> 6) : be;  // q4_0_d_slot
                    r[t].d[e] = ld16(lr[t], 16u * static_cast<uint32_t>(a.blocks) + 2 * slot) & (in ? 0xFFFFu : 0u);
                }
            } else {
                r[t] = Gw<TYPE>::load(lr[t], static_cast<uint32_t>(b), 4 * half + 2 * q + h);
            }
        }
    };

    auto load_raw = [&](Regs (&r)[NT], int b, int half, int q) { load_rows(lr, h, r, b, half, q); };

    f32x16 acc[NT][MT];
    double accd[FINE ? NT : 1][FINE ? MT : 1][16];
    auto clear = [&] {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                acc[t][i] = f32x16{};
                if constexpr (FINE) {
#pragma unroll
                    for (int k = 0; k < 16; ++k) accd[t][i][k] = 0.0;
                }
            }
    };
    const int mx = col & 15;  // the rows' slot swizzle (m0 is a multiple of 32)
    auto operand = [&](const uint4 *xb, int plane, int run, int tile) {
        const uint4 v = xb[(32 * tile + col) * 32 + 16 * plane + (run ^ mx)];
        return __builtin_bit_cast(f16x8, v);
    };
    // acc += d * v, in place: sunk to its next use, every block's v would be
    // live at once
    auto add_block = [&](f32x16 &c, const f32x16 &v, float d) {
#pragma unroll
        for (int k = 0; k < 16; ++k) c[k] = fmaf(d, v[k], c[k]);
        asm volatile("" : "+v"(c));
    };

    // Operands ahead of their products, of even / odd steps (Q4_0: blocks)
    u32x4 fw[Q40 ? 1 : NT][2], fl[Q40 ? 1 : NT][2];  // K types: operand and remainder
    uint2 fe[NT][2][2];                              // codebook entries
    u32x4 bw[Q40 ? NT : 1][2][2];                    // Q4_0: the block's two operands
    float bd[NT][2];
    f32x16 tsum[Q40 ? 1 : NT][Q40 ? 1 : MT];
    f32x16 tlow[FINE ? NT : 1][FINE ? MT : 1];
    f32x16 vlast;
    float dlast = 0.f;
    auto op = [](const u32x4 &v) { return __builtin_bit_cast(f16x8, v); };

    // K types: table entry k, and dword j, of operand step n (q = n / 4, p = n % 4)
    auto look = [&](const Regs (&r)[2][NT], int n, int t, int k) {
        if constexpr (!Q40) {
            if constexpr (Gw<TYPE>::kLooks > 0) fe[t][n & 1][k] = Gw<TYPE>::look(r[n >> 2][t], n & 3, k, tab);
        }
    };
    auto decode = [&](const Regs (&r)[2][NT], int half, int n, int t, int j) {
        if constexpr (!Q40) {
            uint32_t hi, lo = 0;
            Gw<TYPE>::dword(r[n >> 2][t], half, n >> 2, n & 3, j, fe[t][n & 1], hi, lo);
            fw[t][n & 1][j] = hi;
            if constexpr (Gw<TYPE>::kWide) fl[t][n & 1][j] = lo;
        }
    };
    // Q4_0: dword j (0..7) of block n
    auto decode_block = [&](const Regs (&r)[2][NT], int n, int t, int j) {
        if constexpr (Q40) {
            bw[t][n & 1][j >> 2][j & 3] = q40_dword(r[n >> 1][t], n & 1, j >> 2, j & 3);
            if (j == 0) bd[t][n & 1] = half_f(r[n >> 1][t].d[n & 1]);
        }
    };
    // first operands of a superblock from its raw weights
    auto decode_first = [&](const Regs (&r)[2][NT]) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int j = 0; j < 8; ++j) decode_block(r, 0, t, j);
            if constexpr (!Q40) {
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int k = 0; k < Gw<TYPE>::kLooks; ++k) look(r, n, t, k);
#pragma unroll
                for (int j = 0; j < 4; ++j) decode(r, 0, 0, t, j);
            }
        }
    };

    // FINE: the sums of a half superblock (IQ2_S: of each quarter, as its f32 rows
    // are the most accurate)
    constexpr bool QUARTERS = FINE && TYPE == MI355X_TYPE_IQ2_S;
    auto finish_fine = [&](const Regs (&r)[NT]) {
        if constexpr (FINE) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const double d = static_cast<double>(Gw<TYPE>::d(r[t]));
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int k = 0; k < 16; ++k)
                        accd[t][i][k] = fma(d, static_cast<double>(tsum[t][i][k] + tlow[t][i][k]), accd[t][i][k]);
            }
        }
    };
    // One half superblock from its raw weights r, its first operands already
    // decoded; `refill` loads r[0] of the next half once this one's are
    // decoded, and the last step decodes that half's first operands.
    auto half_step = [&](Regs (&r)[2][NT], const uint4 *xb, auto HALF, auto refill) {
        constexpr int half = decltype(HALF)::value;
        if constexpr (Q40) {
            f16x8 x[2][4];  // the operands of one (block, row tile), and the next
            auto read = [&](int u, int k) {
                const int e = u / MT, i = u % MT;
                return operand(xb, k & 1, 4 * e + 2 * (k >> 1) + h, i);
            };
#pragma unroll
            for (int k = 0; k < 4; ++k) x[0][k] = read(0, k);
#pragma unroll
            for (int u = 0; u < 4 * MT; ++u) {
                const int e = u / MT, i = u % MT;
                if (u == 2 * MT) refill();  // r[0] is decoded; after the wait for r[1]'s loads at block 1
                f32x16 v;
#pragma unroll
                for (int m = 0; m < 4 * NT; ++m) {
                    const int t = m >> 2, k = m & 3;
                    v = mfma(x[u & 1][k], op(bw[t][e & 1][k >> 1]), k == 0 ? f32x16{} : v);
                    if (u + 1 < 4 * MT && m < 4) x[(u + 1) & 1][m] = read(u + 1, m);
                    // a quarter of the block sum before this one
                    f32x16 &c = t ? acc[t - 1][i] : acc[NT - 1][(i + MT - 1) % MT];
#pragma unroll
                    for (int z = 4 * k; z < 4 * k + 4; ++z) c[z] = fmaf(dlast, vlast[z], c[z]);
                    // the next block's operands, 8 NT dwords over its 4 NT MT products
#pragma unroll
                    for (int z = 0; z < 8 * NT; ++z)
                        if (z * MT / 2 == i * 4 * NT + m) decode_block(r, (e + 1) & 3, z >> 3, z & 7);
                    __builtin_amdgcn_sched_barrier(0);
                    if (k == 3) {
                        vlast = v;
                        dlast = bd[t][e & 1];
                    }
                }
            }
        } else {
            constexpr int SH = slice_shape(TYPE), TM = NT * MT, NM = TM * (Gw<TYPE>::kWide ? 3 : 2);
            constexpr int LOOKS = Gw<TYPE>::kLooks;
            f16x8 x[2][2 * MT];
            auto read = [&](int s, int k) { return operand(xb, k & 1, run_of<SH>(2 * (s >> 2) + h, s & 3), k >> 1); };
#pragma unroll
            for (int k = 0; k < 2 * MT; ++k) x[0][k] = read(0, k);
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                if (QUARTERS && s == 4) finish_fine(r[0]);
                if (s == 4) refill();  // r[0] is decoded; after the wait for r[1]'s loads in step 3
                const int n = (s + 1) & 7, nh = s < 7 ? half : 1 - half;
#pragma unroll
                for (int m = 0; m < NM; ++m) {
                    const int plane = m / TM, i = m / NT % MT, t = m % NT;
                    const bool low = FINE && plane > 0;
                    const bool first = (half == 0 || FINE) && (s == 0 || (QUARTERS && s == 4)) && (low ? plane == 1 : plane == 0);
                    f32x16 &c = low ? tlow[FINE ? t : 0][FINE ? i : 0] : tsum[t][i];
                    c = mfma(x[s & 1][2 * i + (plane == 1)], op(plane == 2 ? fl[t][s & 1] : fw[t][s & 1]),
                             first ? f32x16{} : c);
                    if (s < 7 && m < 2 * MT) x[(s + 1) & 1][m] = read(s + 1, m);
                    // the next step's operands, 4 NT dwords over NM products,
                    // and the table entries of the one after
#pragma unroll
                    for (int z = 0; z < 4 * NT; ++z)
                        if (z * NM / (4 * NT) == m) decode(r, nh, n, z >> 2, z & 3);
#pragma unroll
                    for (int z = 0; z < LOOKS * NT; ++z)
                        if (NM - LOOKS * NT + z == m || (NM < LOOKS * NT && m == NM - 1)) look(r, (s + 2) & 7, z % NT, z / NT);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    };
    // K types, end of a superblock: acc += d * tsum - dmin * mins . sums
    auto finish = [&](const Regs (&r)[NT], int par) {
        if constexpr (!Q40 && !FINE) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const float d = Gw<TYPE>::d(r[t]);
                if constexpr (Gw<TYPE>::kMins) {
                    const f16x8 mins = k4_mins(r[t].hd);
                    const float dm = -32.0f * half_f(r[t].hd[0] >> 16);
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        // operand halves h = 0, 1: the sums' hi and lo planes
                        const f16x8 s = __builtin_bit_cast(f16x8, ssum[par][(32 * i + col) * 2 + h]);
                        const f32x16 mm = mfma(s, mins, f32x16{});
#pragma unroll
                        for (int k = 0; k < 16; ++k) acc[t][i][k] += fmaf(dm, mm[k], d * tsum[t][i][k]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < MT; ++i) add_block(acc[t][i], tsum[t][i], d);
                }
            }
        }
    };
    // Q4_0: the last block sum
    auto flush = [&] {
        if constexpr (Q40) {
            add_block(acc[NT - 1][MT - 1], vlast, dlast);
            vlast = f32x16{};
            dlast = 0.f;
        }
    };
    auto store = [&](int seg) {
        float *out = a.out + seg * a.seg_stride;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            float us[16];  // requested together, negative for wide rows
#pragma unroll
            for (int k = 0; k < 16; ++k) us[k] = a.unit[min(m0 + 32 * i + 8 * (k >> 2) + 4 * h + (k & 3), a.M - 1)];
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int m = m0 + 32 * i + 8 * (k >> 2) + 4 * h + (k & 3);
                const float u = us[k];
                if (m >= a.M || u < 0.f) continue;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int64_t n = n0 + 32 * t + col;
                    if (n >= a.N) continue;
                    if constexpr (FINE) out[m * a.out_stride + n] = static_cast<float>(static_cast<double>(u) * accd[t][i][k]);
                    else out[m * a.out_stride + n] = u * acc[t][i][k];
                }
            }
        }
    };

    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;

    // Wide activation rows m[0..] in f32, over superblocks [b0, b1), up to
    // kWideRows in one pass over the weights: a lane sums its own slices of its
    // weight rows from the operands that the products take.  (Everything of the
    // lane is formed again here, from its number: nothing stays in registers for
    // this over the products.)
    auto wide_rows = [&](int lane, const int (&m)[kWideRows], int b0, int b1, float *out) {
        const int col = lane & 31, h = lane >> 5;
        LaneRow lr[NT];
        view(col, lr);
        const float *x[kWideRows];
#pragma unroll
        for (int r = 0; r < kWideRows; ++r) x[r] = a.x + m[r] * a.x_stride;
        double wacc[kWideRows][NT] = {};
        // an operand's dwords as its 8 values in order
        auto widen = [](const uint32_t (&w)[4], float (&f)[8]) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f[4 * (j >> 1) + (j & 1)] = static_cast<float>(h2(w[j])[0]);
                f[4 * (j >> 1) + (j & 1) + 2] = static_cast<float>(h2(w[j])[1]);
            }
        };
        auto dot8 = [](const float (&w)[8], const float (&v)[8]) {
            return (fmaf(w[0], v[0], w[1] * v[1]) + fmaf(w[2], v[2], w[3] * v[3])) +
                   (fmaf(w[4], v[4], w[5] * v[5]) + fmaf(w[6], v[6], w[7] * v[7]));
        };
        auto load8 = [&](int r, int64_t i, float (&v)[8]) {
            __builtin_memcpy(&v[0], x[r] + i, 16);
            __builtin_memcpy(&v[4], x[r] + i + 4, 16);
        };
        for (int b = b0; b < b1; ++b) {
            float sup[kWideRows][NT] = {}, low[kWideRows][NT] = {}, d[NT], dm[NT];
            auto quarter = [&](auto HALF, auto Q) {
                constexpr int half = decltype(HALF)::value, q = decltype(Q)::value;
                Regs g[NT];
                load_rows(lr, h, g, b, half, q);
                float v[8];
                if constexpr (Q40) {
                    const int blk = 8 * b + 4 * half + 2 * q;
                    if (blk >= a.blocks) return;
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        float s[kWideRows][NT] = {};
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
                            float f[NT][8];
#pragma unroll
                            for (int t = 0; t < NT; ++t) {
                                uint32_t w[4];
#pragma unroll
                                for (int j = 0; j < 4; ++j) w[j] = q40_dword(g[t], e, i, j);
                                widen(w, f[t]);
                            }
#pragma unroll
                            for (int r = 0; r < kWideRows; ++r) {
                                load8(r, 32 * static_cast<int64_t>(blk + e) + 16 * i + 8 * h, v);
#pragma unroll
                                for (int t = 0; t < NT; ++t) s[r][t] += dot8(f[t], v);
                            }
                        }
#pragma unroll
                        for (int r = 0; r < kWideRows; ++r)
#pragma unroll
                            for (int t = 0; t < NT; ++t) sup[r][t] = fmaf(half_f(g[t].d[e]), s[r][t], sup[r][t]);
                    }
                } else {
                    constexpr int SH = slice_shape(TYPE);
                    float sx[MINS ? kWideRows : 1][2] = {};  // of positions 0, 1 and 2, 3
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        float f[NT][8], rest[NT][8];
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            uint2 e[2] = {};
#pragma unroll
                            for (int k = 0; k < Gw<TYPE>::kLooks; ++k) {
                                if constexpr (Gw<TYPE>::kLooks > 0) e[k] = Gw<TYPE>::look(g[t], p, k, tab);
                            }
                            uint32_t w[4], l[4] = {};
#pragma unroll
                            for (int j = 0; j < 4; ++j) Gw<TYPE>::dword(g[t], half, q, p, j, e, w[j], l[j]);
                            widen(w, f[t]);
                            if constexpr (Gw<TYPE>::kWide) {
                                widen(l, rest[t]);
#pragma unroll
                                for (int i = 0; i < 8; ++i) f[t][i] += rest[t][i];  // exact: 12 bits
                            }
                        }
#pragma unroll
                        for (int r = 0; r < kWideRows; ++r) {
                            load8(r, 256 * static_cast<int64_t>(b) + 128 * half + 8 * run_of<SH>(2 * q + h, p), v);
                            if constexpr (MINS)
                                sx[r][p >> 1] += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
#pragma unroll
                            for (int t = 0; t < NT; ++t) sup[r][t] += dot8(f[t], v);
                        }
                    }
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        d[t] = Gw<TYPE>::d(g[t]);
                        if constexpr (MINS) {
                            const uint32_t mn = min_pair_k4(2 * half + q, g[t].hd);
                            const float m0 = static_cast<float>(mn & 0xFFu), m1 = static_cast<float>(mn >> 8);
#pragma unroll
                            for (int r = 0; r < kWideRows; ++r) low[r][t] += fmaf(m0, sx[r][0], m1 * sx[r][1]);
                            dm[t] = half_f(g[t].hd[0] >> 16);
                        }
                    }
                }
            };
            quarter(H0{}, H0{});
            __builtin_amdgcn_sched_barrier(0);
            quarter(H0{}, H1{});
            __builtin_amdgcn_sched_barrier(0);
            quarter(H1{}, H0{});
            __builtin_amdgcn_sched_barrier(0);
            quarter(H1{}, H1{});
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < kWideRows; ++r)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    float v = sup[r][t];
                    if constexpr (!Q40) v *= d[t];
                    if constexpr (MINS) v = fmaf(-dm[t], low[r][t], v);
                    wacc[r][t] += static_cast<double>(v);
                }
        }
        static_assert(NT == 2, "lane half h stores column tile h");
        const int64_t n = n0 + 32 * h + col;
#pragma unroll
        for (int r = 0; r < kWideRows; ++r) {
            const double y0 = wacc[r][0] + __shfl_xor(wacc[r][0], 32), y1 = wacc[r][1] + __shfl_xor(wacc[r][1], 32);
            if (n < a.N) out[m[r] * a.out_stride + n] = static_cast<float>(h ? y1 : y0);
        }
    };
    stage_table<TYPE>(a, tab);
    vlast = f32x16{};

    const int seg = blockIdx.y;
    const int b0 = seg * a.per_seg, b1 = min(b0 + a.per_seg, a.B);
    auto half_src = [&](int b, int half) {
        return a.planes + (static_cast<int64_t>(2 * b + half) * a.Mp + m0) * kGmHalfBytes;
    };
    // sums of superblock b (types with mins): threads 0 .. 2 BM - 1
    auto load_sums = [&](int b, uint4 &s) {
        if (MINS && threadIdx.x < 2 * BM)
            s = reinterpret_cast<const uint4 *>(a.sums)[(static_cast<int64_t>(b) * a.Mp + m0) * 2 + threadIdx.x];
    };
    auto put_sums = [&](int par, const uint4 &s) {
        if (MINS && threadIdx.x < 2 * BM) ssum[par][threadIdx.x] = s;
    };
    clear();
    uint4 s = make_uint4(0, 0, 0, 0);
    Regs r[2][NT];
    copy_planes<BM>(half_src(b0, 0), xh0, wave, lane);
    load_sums(b0, s);
    load_raw(r[0], b0, 0, 0);
    put_sums(b0 & 1, s);
    gm_barrier();
    decode_first(r);
    for (int b = b0; b < b1; ++b) {
        const int bn = b + 1 < b1 ? b + 1 : b;  // the last superblock's look-ahead reads itself again
        copy_planes<BM>(half_src(b, 1), xh1, wave, lane);
        load_raw(r[1], b, 0, 1);
        __builtin_amdgcn_sched_barrier(0);  // the loads go out before this half's work
        half_step(r, xh0, H0{}, [&] { load_raw(r[0], b, 1, 0); });
        finish_fine(r[1]);
        gm_barrier();
        copy_planes<BM>(half_src(bn, 0), xh0, wave, lane);
        load_sums(bn, s);
        load_raw(r[1], b, 1, 1);
        __builtin_amdgcn_sched_barrier(0);
        half_step(r, xh1, H1{}, [&] { load_raw(r[0], bn, 0, 0); });
        finish_fine(r[1]);
        finish(r[1], b & 1);
        put_sums((b + 1) & 1, s);
        gm_barrier();
    }
    flush();
    store(seg);
    uint32_t ones = ~0u;
    asm volatile("" : "+s"(ones));
    const int lid = static_cast<int>(__builtin_amdgcn_mbcnt_hi(ones, __builtin_amdgcn_mbcnt_lo(ones, 0u)));
    const int ml = m0 + (lid & (BM - 1));
    uint64_t wide = __ballot(lid < BM && ml < a.M && a.unit[ml] < 0.f);
    while (wide) {
        int m[kWideRows];  // the last one repeats
#pragma unroll
        for (int r = 0; r < kWideRows; ++r) {
            m[r] = wide ? m0 + __builtin_ctzll(wide) : m[r > 0 ? r - 1 : 0];
            wide &= wide - 1;
        }
        wide_rows(lid, m, b0, b1, a.out + seg * a.seg_stride);
    }
}

// y = partial 0 + partial 1 + ..., in segment order, in Sum (f64, which costs 1.8
// us more at 4 x 512 x 4096, for the FINE kernels' partials and for more than 64,
// whose f32 chain loses: 5e-7 of an output's deviation with 512)
template <class Sum>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const float *part, int64_t seg_stride, int nseg, int M,
                                                          int64_t N, float *y, int64_t y_stride) {
    const int64_t n = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (n >= N) return;
    for (int m = blockIdx.y; m < M; m += gridDim.y) {
        const float *p = part + m * N + n;
        Sum v = p[0];
        for (int s = 1; s < nseg; ++s) v += static_cast<Sum>(p[s * seg_stride]);
        y[m * y_stride + n] = static_cast<float>(v);
    }
}

typedef void (*gemm_fn)(GemmArgs);

template <int TYPE>
gemm_fn pick_gemm_type(int mt) {
    return mt == 1 ? gemm_kernel<TYPE, 1, false> : gemm_kernel<TYPE, 2, false>;
}
// FINE tiles are of 32 activations: the second sums of 64 do not fit the registers
template <int TYPE>
gemm_fn pick_gemm_iq(int mt, bool fine) {
    return fine ? gemm_kernel<TYPE, 1, true> : pick_gemm_type<TYPE>(mt);
}

gemm_fn pick_gemm(int type, int mt, bool fine) {
    switch (type) {
    case MI355X_TYPE_Q4_0: return pick_gemm_type<MI355X_TYPE_Q4_0>(mt);
    case MI355X_TYPE_Q3_K: return pick_gemm_type<MI355X_TYPE_Q3_K>(mt);
    case MI355X_TYPE_Q4_K: return pick_gemm_type<MI355X_TYPE_Q4_K>(mt);
    case MI355X_TYPE_Q5_K: return pick_gemm_type<MI355X_TYPE_Q5_K>(mt);
    case MI355X_TYPE_Q6_K: return pick_gemm_type<MI355X_TYPE_Q6_K>(mt);
    case MI355X_TYPE_IQ4_XS: return pick_gemm_iq<MI355X_TYPE_IQ4_XS>(mt, fine);
    case MI355X_TYPE_IQ3_S: return pick_gemm_iq<MI355X_TYPE_IQ3_S>(mt, fine);
    case MI355X_TYPE_IQ3_XXS: return pick_gemm_iq<MI355X_TYPE_IQ3_XXS>(mt, fine);
    case MI355X_TYPE_IQ2_S: return pick_gemm_iq<MI355X_TYPE_IQ2_S>(mt, fine);
    default: return nullptr;
    }
}

size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

// Rows of activation tiles for M activations, and what their planes, sums and
// units take of the workspace.
int tile_rows(int M, bool fine) { return M <= 32 || fine ? (M + 31) / 32 * 32 : (M + 63) / 64 * 64; }
size_t planes_bytes(int64_t B, int Mp) { return static_cast<size_t>(B) * 2 * Mp * kGmHalfBytes; }
size_t sums_bytes(int64_t B, int Mp) { return align256(static_cast<size_t>(B) * Mp * 32); }
size_t staged_bytes(int64_t B, int Mp) {
    return planes_bytes(B, Mp) + sums_bytes(B, Mp) + align256(static_cast<size_t>(Mp) * 4);
}

}  // namespace

// From how many activations the matrix cores take a call.  For the K/IQ types,
// whose alternative is one GEMV each (us, that first: 34 / 23 at Q4_K 64x16384 M
// = 4, 35 / 25 at 3001x2816), from 4, but from 5 for codebook matrices of few
// rows (IQ3_S 1024x4096: 16 / 19 at M = 4, 20 / 19 at 5).  For Q4_0 past two
// passes of the 8-row kernels; with 2^25 weights of long rows also most of two
// passes (30 / 24 at 4096x8192 M = 12, 39 / 36 at 8192x8192 M = 16; but 16 / 20
// at 256x4096, 97 / 122 at 151936x2048).  Only where the caller leaves arithmetic
// and form to the library: MI355X_VARIANT_DIGITS promises fixed point, and the
// kernels here know no form options and no cap on the workgroups.
bool gemm_batched_supports(const mi355x_ctx *ctx, const GemvArgs &a, int64_t M) {
    if (ctx->kernel_variant != MI355X_VARIANT_AUTO || !form_is_auto(ctx, a.type) || ctx->grid_override != 0) return false;
    if (a.x_bf16 || a.N <= 0 || a.K <= 0 || !ctx->gemm_buf) return false;
    // Q4_0 rows past 16384 values have f32 one-row kernels (error against 64 bits
    // 2.7e-7; here 1.7e-7 at 17408x16640 and 2.3e-7 at 17408x32768, growing with
    // the f32 chain of a row's blocks)
    if (a.type == MI355X_TYPE_Q4_0 && a.K > 32768) return false;
    // 32-bit offsets into the 64 rows of a wavefront
    const int64_t row_bytes = a.type == MI355X_TYPE_Q4_0 ? a.K / 32 * 18 : a.K / 256 * kq_layout(a.type).block_bytes;
    if (row_bytes <= 0 || row_bytes >= (int64_t(1) << 31) / 64 || a.N >= (int64_t(1) << 31)) return false;
    if (staged_bytes((a.K + 255) / 256, 32) > kGemmWorkspace) return false;
    if (a.type == MI355X_TYPE_Q4_0) {
        // dword-aligned loads of code groups
        if (reinterpret_cast<uintptr_t>(a.W) % 4 != 0 || row_bytes % 4 != 0) return false;
        return M >= 17 || (M >= 12 && a.K >= 4096 && a.N * a.K >= (int64_t(1) << 25));
    }
    // codes times scales exact in f16
    if ((a.type == MI355X_TYPE_IQ3_XXS || a.type == MI355X_TYPE_IQ2_S) &&
        (a.type == MI355X_TYPE_IQ3_XXS ? ctx->iq3xxs_max : ctx->iq2s_max) > 66)
        return false;
    return M >= (a.N < 4096 && !kq_digit_rows(ctx, a.type, a.N, a.K) ? 5 : 4);
}

// Whether the launches of a call now run in order on the context's stream, and
// on no other: false while the stream records a graph.
int gemm_batched_in_order(const mi355x_ctx *ctx, bool *in_order) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    MI355X_HIP(hipStreamIsCapturing(ctx->stream, &st));
    *in_order = st == hipStreamCaptureStatusNone;
    return MI355X_OK;
}

// The workspace belongs to the context from its creation to its end and never
// moves, so no call allocates; the context's lock keeps the launches that share
// it together on its stream.  Activations that it cannot hold at once go in
// several passes.  A graph may be replayed on any stream, at the same time as
// the context's own calls, so a call under capture takes a form without the
// workspace instead (gemm_batched_in_order).
int launch_gemm_batched(mi355x_ctx *ctx, const GemvArgs &a, int64_t x_stride, int64_t y_stride, int64_t M_total) {
    const bool q40 = a.type == MI355X_TYPE_Q4_0;
    // calls that replace f32 rows
    const bool f32_rows = q40 ? a.K > 16384 : !kq_digit_rows(ctx, a.type, a.N, a.K);
    const bool fine = f32_rows && !q40;
    GemmArgs g{};
    g.W = a.W;
    g.N = a.N;
    g.row_bytes = q40 ? a.K / 32 * 18 : a.K / 256 * kq_layout(a.type).block_bytes;
    g.B = static_cast<int>((a.K + 255) / 256);
    g.blocks = static_cast<int>(a.K / 32);
    const int x_al16 = reinterpret_cast<uintptr_t>(a.x) % 16 == 0 && x_stride % 4 == 0 ? 1 : 0;
    if (a.type == MI355X_TYPE_IQ3_XXS) g.grid = static_cast<const uint32_t *>(ctx->iq3xxs_grid);
    if (a.type == MI355X_TYPE_IQ2_S) g.grid = static_cast<const uint32_t *>(ctx->iq2s_grid);
    if ((a.type == MI355X_TYPE_IQ3_XXS || a.type == MI355X_TYPE_IQ2_S) && !g.grid)
        return set_error(MI355X_EUNSUPPORTED, "grid table not installed for this IQ type");
    g.ntiles = static_cast<int>((a.N + kGmCols - 1) / kGmCols);
    std::lock_guard<std::mutex> lk(ctx->mu);
    for (int64_t mb = 0; mb < M_total; mb += g.M) {
        int M = static_cast<int>(std::min<int64_t>(kGmMaxRows, M_total - mb));
        while (M > 32 && staged_bytes(g.B, tile_rows(M, fine)) > kGemmWorkspace) M = std::max(32, (M / 2 + 31) / 32 * 32);
        const int mt = M <= 32 || fine ? 1 : 2;
        g.M = M;
        g.Mp = tile_rows(M, fine);
        g.mtiles = g.Mp / (32 * mt);
        float *y = a.y + mb * y_stride;
        const int64_t tiles = static_cast<int64_t>(g.ntiles) * g.mtiles;
        const size_t staged = staged_bytes(g.B, g.Mp);
        // segments of K: enough workgroups for two per CU, at least two
        // superblocks each, partials within the rest of the workspace
        int64_t seg = std::max<int64_t>(1, 2 * ctx->num_cus / tiles);
        seg = std::min<int64_t>(seg, std::max(1, g.B / 2));
        seg = std::min<int64_t>(seg, std::max<int64_t>(1, static_cast<int64_t>(kGemmWorkspace - staged) / (4 * M * a.N)));
        g.per_seg = static_cast<int>((g.B + seg - 1) / seg);
        g.nseg = (g.B + g.per_seg - 1) / g.per_seg;
        const unsigned grid_x = static_cast<unsigned>((g.ntiles + 7) / 8 * 8 * g.mtiles);
        uint8_t *p = static_cast<uint8_t *>(ctx->gemm_buf);
        g.planes = p;
        g.sums = reinterpret_cast<const _Float16 *>(p + planes_bytes(g.B, g.Mp));
        g.x = static_cast<const float *>(a.x) + mb * x_stride;
        g.x_stride = x_stride;
        g.unit = reinterpret_cast<const float *>(p + planes_bytes(g.B, g.Mp) + sums_bytes(g.B, g.Mp));
        float *partial = reinterpret_cast<float *>(p + staged);
        g.out = g.nseg > 1 ? partial : y;
        g.out_stride = g.nseg > 1 ? a.N : y_stride;
        g.seg_stride = static_cast<int64_t>(M) * a.N;
        hipLaunchKernelGGL(gemm_planes_kernel, dim3(static_cast<unsigned>(M)), dim3(kPlThreads), 0, ctx->stream,
                           g.x, x_stride, a.K, x_al16, f32_rows ? kWideBelowF32 : kWideBelow, g.Mp, g.B, p,
                           const_cast<_Float16 *>(g.sums), const_cast<float *>(g.unit));
        MI355X_HIP(hipGetLastError());
        hipLaunchKernelGGL(pick_gemm(a.type, mt, fine), dim3(grid_x, static_cast<unsigned>(g.nseg)), dim3(kGmThreads), 0,
                           ctx->stream, g);
        MI355X_HIP(hipGetLastError());
        if (g.nseg > 1) {
            hipLaunchKernelGGL(fine || g.nseg > 64 ? gemm_reduce_kernel<double> : gemm_reduce_kernel<float>,
                               dim3(static_cast<unsigned>((a.N + 255) / 256), std::min(M, 64)),
                               dim3(256), 0, ctx->stream, partial, g.seg_stride, g.nseg, M, a.N, y, y_stride);
            MI355X_HIP(hipGetLastError());
        }
    }
    return MI355X_OK;
}

}  // namespace mi355x
