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
// remainder; Q4_0 keeps its bare codes and applies the block scale to each
// block's sum.  Activations are split into two f16 planes, hi = f16(x s) and
// lo = f16(x s - hi) with s a power of two per (row, 256 values) that puts the
// largest |x| in [2^14, 2^15): x s = hi + lo to 2^-22 of x, or 2^-25 absolute,
// i.e. 2^-39 of the superblock's largest value.  Products are exact in f32 and
// sums are f32 over 256 values (32 for Q4_0), then scaled by the superblock's
// d and s and added in f32 over superblocks.  This is more accurate than the
// 20- or 16-bit fixed point of the single-row kernels.
//
// Work split.  A workgroup of 4 wavefronts computes 256 output columns (weight
// rows) x 32 or 64 activation rows; a wavefront 64 columns as two 32-wide
// MFMA tiles, so that each activation operand read from LDS feeds two
// products.  K is walked in half superblocks: the activation planes of the
// next half travel to LDS directly (buffer_load ... lds) and the next half's
// weights to registers while this half is multiplied.  Where the tiles leave
// CUs idle the superblocks are split over gridDim.y segments whose f32
// partials a second kernel adds in segment order.
//
// Measured on MI355X, us per call (sequential or 8-row passes before): Q4_0
// 17408x5120 M = 512 395 (2700), Q6_K 4096x14336 M = 512 232 (6330), Q4_K
// 14336x4096 M = 37 40 (256); 231-259 TFLOP/s of useful products, each two
// MFMAs (three for Q6_K).
#include "internal.h"
#include "kq_device.h"
#include "q4_0_layout.h"

#include <algorithm>
#include <cstdint>
#include <mutex>

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
    const float *unit;      // [superblock][Mp]
    const float *x;         // CONV: the activations themselves
    int64_t x_stride;
    int x_al16;
    int64_t K;
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

struct XPlanes {
    uint2 hi, lo;  // this lane's 4 values of each plane, in run order
    float unit;    // 1 / s
    _Float16 s_hi, s_lo;  // lanes 8j: sum of sub-block j (times s / 32)
};

// One superblock of one activation row by a whole wavefront: lane l converts
// values 4l .. 4l + 3 (`left` of the 256 exist, the rest are zero).
__device__ __forceinline__ XPlanes convert_superblock(const float *x, int left, bool al16, int lane) {
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    const int i0 = 4 * lane;
    if (al16 && i0 + 3 < left) {
        const float4 f = *reinterpret_cast<const float4 *>(x + i0);
        v[0] = f.x;
        v[1] = f.y;
        v[2] = f.z;
        v[3] = f.w;
    } else {
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (i0 + t < left) v[t] = x[i0 + t];
    }
    const float mx = wave_max(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
    // s = 2^(14 - E) for max in [2^E, 2^(E+1)), E >= -110 (an all-zero or
    // smaller superblock takes 2^124)
    const int e = max(static_cast<int>(__builtin_bit_cast(uint32_t, mx) >> 23), 17);  // biased E
    const float s = __builtin_bit_cast(float, static_cast<uint32_t>(268 - min(e, 254)) << 23);
    XPlanes r;
    r.unit = __builtin_bit_cast(float, static_cast<uint32_t>(min(e, 254) - 14) << 23);
    float w[4];
    _Float16 h[4], l[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        w[t] = v[t] * s;
        h[t] = static_cast<_Float16>(w[t]);
        l[t] = static_cast<_Float16>(w[t] - static_cast<float>(h[t]));
    }
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

// Planes, sums and units of M activation rows: one wavefront per (row,
// superblock).
__global__ __launch_bounds__(256) void gemm_planes_kernel(const float *x, int64_t x_stride, int64_t K, int x_al16,
                                                          int M, int Mp, int B, uint8_t *planes, _Float16 *sums,
                                                          float *unit) {
    const int lane = threadIdx.x & 63;
    const int64_t task = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (task >= static_cast<int64_t>(M) * B) return;
    const int m = static_cast<int>(task / B), b = static_cast<int>(task % B);
    const int64_t left = K - 256 * static_cast<int64_t>(b);
    const XPlanes c = convert_superblock(x + m * x_stride + 256 * static_cast<int64_t>(b),
                                         static_cast<int>(left < 256 ? left : 256), x_al16 != 0, lane);
    uint8_t *h0 = planes + (static_cast<int64_t>(2 * b) * Mp + m) * kGmHalfBytes;
    store_superblock(c, m, lane, h0, h0 + static_cast<int64_t>(Mp) * kGmHalfBytes,
                     sums + (static_cast<int64_t>(b) * Mp + m) * 16);
    if (lane == 0) unit[static_cast<int64_t>(b) * Mp + m] = c.unit;
}

// ---- weight decode --------------------------------------------------------------
// Gw<TYPE>: the weights of one lane (one weight row) for slice s of a
// superblock as four f16 operands, operand p the run at position p of the
// slice (run_of).  decode's `half` and `q` are compile-time constants at every
// call (s = 4 half + 2 q + h, h = lane / 32).  kWide types leave the exact
// remainder of codes times scales in lo; d(regs) is the superblock's scale.
template <int TYPE>
struct Gw;

// (scale, min) bytes of sub-blocks 2c and 2c + 1 (scale_min_pair_k4)
__device__ __forceinline__ uint32_t scale_pair_k4(int c, const u32x4 &hd) {
    const uint32_t sh = 16u * static_cast<uint32_t>(c & 1);
    const uint32_t a2 = hd[1] >> sh, c2 = hd[3] >> sh;
    return c < 2 ? (a2 & 0x3F3Fu) : ((c2 & 0x0F0Fu) | ((a2 >> 2) & 0x3030u));
}
// byte B of w as an f16 integer in both halves
template <int B>
__device__ __forceinline__ f16x2 byte_h2(uint32_t w) {
    return h2(__builtin_amdgcn_perm(w, w, 0x0C000C00u | (static_cast<uint32_t>(B) << 16) | B) | kH1024) - h2s(1024.f);
}
// the same less BIAS
template <int B, int BIAS>
__device__ __forceinline__ f16x2 byte_h2_biased(uint32_t w) {
    return h2(__builtin_amdgcn_perm(w, w, 0x0C000C00u | (static_cast<uint32_t>(B) << 16) | B) | kH1024) -
           h2s(1024.f + BIAS);
}

template <bool Q5, class Regs>
__device__ __forceinline__ void k45_decode(const Regs &g, int half, int q, f16x8 (&hi)[4]) {
    const int c = 2 * half + q;
    const uint32_t sp = scale_pair_k4(c, g.hd);
    const f16x2 sc0 = byte_h2<0>(sp), sc1 = byte_h2<1>(sp) * h2s(0.0625f);
    const f16x2 o0 = sc0 * h2s(-1024.f), o1 = sc1 * h2s(-1024.f);  // exact: sc <= 63
    uint32_t lo[8], up[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t w = g.q[i], w8 = w >> 8;
        uint32_t a = (w & 0x000F000Fu) | kH1024, b = (w8 & 0x000F000Fu) | kH1024;
        uint32_t e = (w & 0x00F000F0u) | kH1024, f = (w8 & 0x00F000F0u) | kH1024;
        if constexpr (Q5) {
            // high bit 2c of each qh byte to bit 4 of the low codes, bit
            // 2c + 1 to bit 8 of the in-place high codes
            const uint32_t qh = g.qh[i];
            const uint32_t t = 2 * c <= 4 ? qh << (4 - 2 * c) : qh >> (2 * c - 4);
            a |= t & 0x00100010u;
            b |= (t >> 8) & 0x00100010u;
            e |= (7 - 2 * c >= 0 ? qh << (7 - 2 * c) : qh) & 0x01000100u;
            f |= (qh >> (2 * c + 1)) & 0x01000100u;
        }
        lo[2 * i] = u2(pk_fma(h2(a), sc0, o0));
        lo[2 * i + 1] = u2(pk_fma(h2(b), sc0, o0));
        up[2 * i] = u2(pk_fma(h2(e), sc1, o1));
        up[2 * i + 1] = u2(pk_fma(h2(f), sc1, o1));
    }
    hi[0] = frag8(lo[0], lo[1], lo[2], lo[3]);
    hi[1] = frag8(lo[4], lo[5], lo[6], lo[7]);
    hi[2] = frag8(up[0], up[1], up[2], up[3]);
    hi[3] = frag8(up[4], up[5], up[6], up[7]);
}
// the 8 sub-block mins of a superblock in run order
__device__ __forceinline__ f16x8 k4_mins(const u32x4 &hd) {
    const uint32_t m0 = hd[2] & 0x3F3F3F3Fu;
    const uint32_t m1 = ((hd[3] >> 4) & 0x0F0F0F0Fu) | ((hd[2] >> 2) & 0x30303030u);
    const f16x2 k = h2s(1024.f);
    return frag8(u2(h2((m0 & 0x00FF00FFu) | kH1024) - k), u2(h2(((m0 >> 8) & 0x00FF00FFu) | kH1024) - k),
                 u2(h2((m1 & 0x00FF00FFu) | kH1024) - k), u2(h2(((m1 >> 8) & 0x00FF00FFu) | kH1024) - k));
}

template <>
struct Gw<MI355X_TYPE_Q4_K> {
    static constexpr bool kWide = false, kMins = true;
    using Regs = Kq<MI355X_TYPE_Q4_K>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_Q4_K>::load(r, b, s); }
    __device__ static float d(const Regs &g) { return half_f(g.hd[0] & 0xFFFF); }
    __device__ static void decode(const Regs &g, int half, int q, const uint2 *, f16x8 (&hi)[4], f16x8 (&)[4]) {
        k45_decode<false>(g, half, q, hi);
    }
};
template <>
struct Gw<MI355X_TYPE_Q5_K> {
    static constexpr bool kWide = false, kMins = true;
    using Regs = Kq<MI355X_TYPE_Q5_K>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_Q5_K>::load(r, b, s); }
    __device__ static float d(const Regs &g) { return half_f(g.hd[0] & 0xFFFF); }
    __device__ static void decode(const Regs &g, int half, int q, const uint2 *, f16x8 (&hi)[4], f16x8 (&)[4]) {
        k45_decode<true>(g, half, q, hi);
    }
};

// v * sc split into its f16 rounding and the exact remainder
__device__ __forceinline__ void wide_mul(f16x2 v, f16x2 sc, uint32_t &hi, uint32_t &lo) {
    const f16x2 p = v * sc;
    hi = u2(p);
    lo = u2(pk_fma(v, sc, -p));
}

template <>
struct Gw<MI355X_TYPE_Q6_K> {
    static constexpr bool kWide = true, kMins = false;
    using Regs = Kq<MI355X_TYPE_Q6_K>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_Q6_K>::load(r, b, s); }
    __device__ static float d(const Regs &g) { return half_f(g.d); }
    __device__ static void decode(const Regs &g, int, int, const uint2 *, f16x8 (&hi)[4], f16x8 (&lo)[4]) {
        uint32_t H[4][4], L[4][4];
        const uint32_t sw = g.sw4 ^ 0x80808080u;  // int8 scales + 128
        const f16x2 sc[4] = {byte_h2_biased<0, 128>(sw), byte_h2_biased<1, 128>(sw), byte_h2_biased<2, 128>(sw),
                             byte_h2_biased<3, 128>(sw)};
        const f16x2 off = h2s(1024.f + 32.f);
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const uint32_t A = g.qa[w], Bq = g.qb[w], Q = g.qh[w];
            const uint32_t code[4][2] = {
                {(A & 0x000F000Fu) | ((Q << 4) & 0x00300030u), ((A >> 8) & 0x000F000Fu) | ((Q >> 4) & 0x00300030u)},
                {(Bq & 0x000F000Fu) | ((Q << 2) & 0x00300030u), ((Bq >> 8) & 0x000F000Fu) | ((Q >> 6) & 0x00300030u)},
                {((A >> 4) & 0x000F000Fu) | (Q & 0x00300030u), ((A >> 12) & 0x000F000Fu) | ((Q >> 8) & 0x00300030u)},
                {((Bq >> 4) & 0x000F000Fu) | ((Q >> 2) & 0x00300030u),
                 ((Bq >> 12) & 0x000F000Fu) | ((Q >> 10) & 0x00300030u)}};
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    wide_mul(h2(code[j][t] | kH1024) - off, sc[j], H[j][2 * w + t], L[j][2 * w + t]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            hi[j] = frag8(H[j][0], H[j][1], H[j][2], H[j][3]);
            lo[j] = frag8(L[j][0], L[j][1], L[j][2], L[j][3]);
        }
    }
};

template <>
struct Gw<MI355X_TYPE_Q3_K> {
    static constexpr bool kWide = false, kMins = false;
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
    __device__ static void decode(const Regs &g, int half, int q, const uint2 *, f16x8 (&hi)[4], f16x8 (&)[4]) {
        // the four 6-bit scales in one word, bytes in run order 0, 2, 1, 3
        // (KqDg<Q3_K>); kk = q, hh = half
        const uint32_t Lw = q ? g.sw01[1] : g.sw01[0];
        const uint32_t Hw = g.sw2 >> (8 * q + 4 * half);
        const uint32_t SC = ((Lw >> (4 * half)) & 0x0F0F0F0Fu) | ((Hw & 0x00030003u) << 4) | ((Hw & 0x000C000Cu) << 10);
        const f16x2 sc[4] = {byte_h2_biased<0, 32>(SC), byte_h2_biased<2, 32>(SC), byte_h2_biased<1, 32>(SC),
                             byte_h2_biased<3, 32>(SC)};
        uint32_t H[4][4];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                // code bits in place (4^j times the code), the hmask bit above
                const uint32_t m2 = 0x00030003u << (2 * j), mh = 0x00040004u << (2 * j);
                const int sh = j + 2 - 4 * half;  // hmask bit 4 half + j to bit 2j + 2
                const uint32_t h0 = sh >= 0 ? g.hm[w] << sh : g.hm[w] >> -sh;
                const uint32_t h1 = 8 - sh >= 0 ? g.hm[w] >> (8 - sh) : g.hm[w];
                const uint32_t a = (g.q[w] & m2) | (h0 & mh) | kH1024;
                const uint32_t b = ((g.q[w] >> 8) & m2) | (h1 & mh) | kH1024;
                const float f = static_cast<float>(1 << (2 * j));
                const f16x2 o = h2s(1024.f + 4.f * f), sj = sc[j] * h2s(1.f / f);
                H[j][2 * w] = u2((h2(a) - o) * sj);
                H[j][2 * w + 1] = u2((h2(b) - o) * sj);
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) hi[j] = frag8(H[j][0], H[j][1], H[j][2], H[j][3]);
    }
};

template <>
struct Gw<MI355X_TYPE_IQ4_XS> {
    static constexpr bool kWide = true, kMins = false;
    using Regs = Kq<MI355X_TYPE_IQ4_XS>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_IQ4_XS>::load(r, b, s); }
    __device__ static float d(const Regs &g) { return half_f(g.hd[0] & 0xFFFF); }
    __device__ static void decode(const Regs &g, int half, int q, const uint2 *, f16x8 (&hi)[4], f16x8 (&lo)[4]) {
        const uint32_t s = static_cast<uint32_t>(4 * half + 2 * q) + (__lane_id() >> 5);
        const uint32_t sh = g.hd[0] >> 16;
        const uint32_t ls = ((g.hd[1] >> (4 * s)) & 15u) | (((sh >> (2 * s)) & 3u) << 4);
        const f16x2 sc = byte_h2_biased<0, 32>(ls);
        const f16x2 off = h2s(1024.f + 128.f);  // the codebook bytes are kvalues + 128
        uint32_t H[16], L[16];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t a = Kq<MI355X_TYPE_IQ4_XS>::lookup(g.q[i] & 0x0F0F0F0Fu);
            const uint32_t b = Kq<MI355X_TYPE_IQ4_XS>::lookup((g.q[i] >> 4) & 0x0F0F0F0Fu);
            wide_mul(h2((a & 0x00FF00FFu) | kH1024) - off, sc, H[2 * i], L[2 * i]);
            wide_mul(h2(((a >> 8) & 0x00FF00FFu) | kH1024) - off, sc, H[2 * i + 1], L[2 * i + 1]);
            wide_mul(h2((b & 0x00FF00FFu) | kH1024) - off, sc, H[8 + 2 * i], L[8 + 2 * i]);
            wide_mul(h2(((b >> 8) & 0x00FF00FFu) | kH1024) - off, sc, H[9 + 2 * i], L[9 + 2 * i]);
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            hi[p] = frag8(H[4 * p], H[4 * p + 1], H[4 * p + 2], H[4 * p + 3]);
            lo[p] = frag8(L[4 * p], L[4 * p + 1], L[4 * p + 2], L[4 * p + 3]);
        }
    }
};

// Sign masks of the f16 pairs of 8 values from their sign byte: pairs (0, 2),
// (1, 3), (4, 6), (5, 7) of the byte's bits.
struct SignMasks {
    uint32_t m[4];
};
__device__ __forceinline__ SignMasks sign_masks(uint32_t b) {
    const uint32_t t = b | (b << 14);  // bit i also at 14 + i: bits 2i and 16 + .. meet in a halfword pair
    return {{(t << 15) & 0x80008000u, (t << 14) & 0x80008000u, (t << 11) & 0x80008000u, (t << 10) & 0x80008000u}};
}
// 8 grid magnitudes (two f16 table entries of 4) with signs, times sc
__device__ __forceinline__ f16x8 signed_run(uint2 e0, uint2 e1, uint32_t signs, f16x2 sc) {
    const SignMasks s = sign_masks(signs);
    return frag8(u2(h2(e0.x ^ s.m[0]) * sc), u2(h2(e0.y ^ s.m[1]) * sc), u2(h2(e1.x ^ s.m[2]) * sc),
                 u2(h2(e1.y ^ s.m[3]) * sc));
}

template <>
struct Gw<MI355X_TYPE_IQ3_S> {
    static constexpr bool kWide = false, kMins = false;
    using Regs = Kq<MI355X_TYPE_IQ3_S>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_IQ3_S>::load(r, b, s); }
    __device__ static float d(const Regs &g) { return half_f(g.d); }
    __device__ static void decode(const Regs &g, int, int, const uint2 *tab, f16x8 (&hi)[4], f16x8 (&)[4]) {
        const uint32_t n = (g.scb >> ((__lane_id() >> 5) * 4)) & 15u;
        const f16x2 sc = byte_h2<0>(2 * n + 1);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const uint32_t w = g.qs[p >> 1];
            const uint32_t i0 = byte_u(w, 2 * (p & 1)) | (((g.qh >> (2 * p)) & 1u) << 8);
            const uint32_t i1 = byte_u(w, 2 * (p & 1) + 1) | (((g.qh >> (2 * p + 1)) & 1u) << 8);
            hi[p] = signed_run(tab[i0], tab[i1], byte_u(g.sg, p), sc);
        }
    }
};

template <>
struct Gw<MI355X_TYPE_IQ3_XXS> {
    static constexpr bool kWide = false, kMins = false;
    using Regs = Kq<MI355X_TYPE_IQ3_XXS>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_IQ3_XXS>::load(r, b, s); }
    // (0.5 + n) / 2 = (2 n + 1) / 4
    __device__ static float d(const Regs &g) { return 0.25f * half_f(g.d); }
    __device__ static void decode(const Regs &g, int, int, const uint2 *tab, f16x8 (&hi)[4], f16x8 (&)[4]) {
        const f16x2 sc = byte_h2<0>(2 * (g.aux >> 28) + 1);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const uint32_t w = g.qs[p >> 1];
            hi[p] = signed_run(tab[byte_u(w, 2 * (p & 1))], tab[byte_u(w, 2 * (p & 1) + 1)],
                               ksigns((g.aux >> (7 * p)) & 127u), sc);
        }
    }
};

template <>
struct Gw<MI355X_TYPE_IQ2_S> {
    static constexpr bool kWide = false, kMins = false;
    using Regs = Kq<MI355X_TYPE_IQ2_S>::Regs;
    __device__ static Regs load(const LaneRow &r, uint32_t b, int s) { return Kq<MI355X_TYPE_IQ2_S>::load(r, b, s); }
    // (0.5 + n) / 4 = (2 n + 1) / 8
    __device__ static float d(const Regs &g) { return 0.125f * half_f(g.d); }
    __device__ static void decode(const Regs &g, int, int, const uint2 *tab, f16x8 (&hi)[4], f16x8 (&)[4]) {
        // the table keeps the grid's bytes: an f16 table would take 16 KB and
        // the second workgroup of a CU
        const f16x2 sc[2] = {byte_h2<0>(2 * (g.scb & 15u) + 1), byte_h2<0>(2 * (g.scb >> 4) + 1)};
        const f16x2 k = h2s(1024.f);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const uint2 e = tab[byte_u(g.qs, p) | (((g.qh >> (2 * p)) & 3u) << 8)];
            const uint2 e0 = make_uint2(u2(h2((e.x & 0x00FF00FFu) | kH1024) - k),
                                        u2(h2(((e.x >> 8) & 0x00FF00FFu) | kH1024) - k));
            const uint2 e1 = make_uint2(u2(h2((e.y & 0x00FF00FFu) | kH1024) - k),
                                        u2(h2(((e.y >> 8) & 0x00FF00FFu) | kH1024) - k));
            hi[p] = signed_run(e0, e1, byte_u(g.sg, p), sc[p >> 1]);
        }
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
__device__ __forceinline__ void q40_decode(const Q40Regs &g, f16x8 (&w)[2][2]) {
    const auto s0 = __builtin_amdgcn_permlane32_swap(g.q[0], g.q[2], false, false);
    const auto s1 = __builtin_amdgcn_permlane32_swap(g.q[1], g.q[3], false, false);
    const uint32_t v[2][2] = {{static_cast<uint32_t>(s0[0]), static_cast<uint32_t>(s1[0])},
                              {static_cast<uint32_t>(s0[1]), static_cast<uint32_t>(s1[1])}};
    const f16x2 o0 = h2s(-1032.f), o1 = h2s(-72.f), c = h2s(0.0625f);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        uint32_t L[4], U[4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            // resident nibbles are q - 8 in two's complement: flip the sign bit
            const uint32_t a = v[e][i], b = a >> 8;
            L[2 * i] = u2(h2((a & 0x000F000Fu) ^ 0x64086408u) + o0);
            L[2 * i + 1] = u2(h2((b & 0x000F000Fu) ^ 0x64086408u) + o0);
            U[2 * i] = u2(pk_fma(h2((a & 0x00F000F0u) ^ 0x64806480u), c, o1));
            U[2 * i + 1] = u2(pk_fma(h2((b & 0x00F000F0u) ^ 0x64806480u), c, o1));
        }
        w[e][0] = frag8(L[0], L[1], L[2], L[3]);
        w[e][1] = frag8(U[0], U[1], U[2], U[3]);
    }
}

// LDS words of the codebook table
constexpr int gm_table_entries(int type) {
    return type == MI355X_TYPE_IQ3_S ? kIq3sGridSize : type == MI355X_TYPE_IQ3_XXS ? 256 : type == MI355X_TYPE_IQ2_S ? 1024 : 1;
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

template <int TYPE, int MT, bool CONV>
__global__ __launch_bounds__(kGmThreads, 2) void gemm_kernel(GemmArgs a) {
    constexpr int BM = 32 * MT, NT = kGmNT;
    constexpr bool Q40 = TYPE == MI355X_TYPE_Q4_0;
    using Regs = typename RegsOf<TYPE>::T;
    __shared__ uint4 xh0[BM * kGmHalfBytes / 16], xh1[BM * kGmHalfBytes / 16];
    __shared__ uint4 ssum[2][BM * 2];
    __shared__ float sunit[2][BM];
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
    LaneRow lr[NT];
    {
        const uint8_t *base = a.W + (rows > 0 ? n0 : 0) * a.row_bytes;
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t *>(base), 0, static_cast<uint32_t>(rows * a.row_bytes), kBufferWord3);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const uint32_t rl = 32 * t + col;
            lr[t].rsrc = rsrc;
            lr[t].base = rl * static_cast<uint32_t>(a.row_bytes);
            if constexpr (!Q40) {
                constexpr KqLayout L = kq_layout(TYPE);
                const bool flipped = kq_row_flipped(reinterpret_cast<uintptr_t>(base) + lr[t].base);
                if constexpr (L.grouped) {
                    lr[t].P[0] = static_cast<uint32_t>(a.B);
                    lr[t].P[1] = flipped ? 1u : 0u;
                } else {
#pragma unroll
                    for (int i = 0; i < 5; ++i)
                        lr[t].P[i] = i < L.nfields ? static_cast<uint32_t>(kq_plane_start(L, i, a.B, flipped)) : 0u;
                }
            }
        }
    }
    // raw weights of slices (or blocks) 4 half + 2q + h, q = 0, 1
    auto load_raw = [&](Regs (&r)[NT][2], int b, int half) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                if constexpr (Q40) {
                    // rows have an even number of blocks: a pair exists or
                    // not; past the row the scales are 0
                    const int b0 = 8 * b + 4 * half + 2 * q;
                    const bool in = b0 < a.blocks;
                    const int bc = in ? b0 : 0;
                    r[t][q].q = ld128(lr[t], 16u * static_cast<uint32_t>(bc + h));
                    const uint32_t F = static_cast<uint32_t>(a.blocks) >> 6;
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const uint32_t be = static_cast<uint32_t>(bc + e);
                        const uint32_t slot = be < 64 * F ? (be & 63) * F + (be >> 6) : be;  // q4_0_d_slot
                        r[t][q].d[e] = ld16(lr[t], 16u * static_cast<uint32_t>(a.blocks) + 2 * slot) & (in ? 0xFFFFu : 0u);
                    }
                } else {
                    r[t][q] = Gw<TYPE>::load(lr[t], static_cast<uint32_t>(b), 4 * half + 2 * q + h);
                }
            }
        }
    };

    f32x16 acc[NT][MT], tsum[NT][MT];
    const int mx = col & 15;  // the rows' slot swizzle (m0 is a multiple of 32)

    auto operand = [&](const uint4 *xb, int plane, int run, int tile) {
        const uint4 v = xb[(32 * tile + col) * 32 + 16 * plane + (run ^ mx)];
        return __builtin_bit_cast(f16x8, v);
    };

    // tsum (+)= this half superblock
    auto compute = [&](const Regs (&r)[NT][2], const uint4 *xb, int half) {
        if constexpr (Q40) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                f16x8 w[NT][2][2];
#pragma unroll
                for (int t = 0; t < NT; ++t) q40_decode(r[t][q], w[t]);
#pragma unroll
                for (int e = 0; e < 2; ++e) {
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        const int run = 4 * (2 * q + e);
                        const f16x8 h0 = operand(xb, 0, run + h, i), l0 = operand(xb, 1, run + h, i);
                        const f16x8 h1 = operand(xb, 0, run + 2 + h, i), l1 = operand(xb, 1, run + 2 + h, i);
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            f32x16 v = {};
                            v = mfma(h0, w[t][e][0], v);
                            v = mfma(l0, w[t][e][0], v);
                            v = mfma(h1, w[t][e][1], v);
                            v = mfma(l1, w[t][e][1], v);
                            const float d = half_f(r[t][q].d[e]);
#pragma unroll
                            for (int k = 0; k < 16; ++k)
                                tsum[t][i][k] = half == 0 && q == 0 && e == 0 ? d * v[k] : fmaf(d, v[k], tsum[t][i][k]);
                            // stays here: sunk to its next use, every block's
                            // v would be live at once
                            asm volatile("" : "+v"(tsum[t][i]));
                        }
                    }
                }
            }
        } else {
            constexpr int SH = slice_shape(TYPE);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                f16x8 wh[NT][4], wl[NT][4];
#pragma unroll
                for (int t = 0; t < NT; ++t) Gw<TYPE>::decode(r[t][q], half, q, tab, wh[t], wl[t]);
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const int run = run_of<SH>(2 * q + h, p);
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        const f16x8 xh = operand(xb, 0, run, i), xl = operand(xb, 1, run, i);
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            f32x16 v = half == 0 && q == 0 && p == 0 ? f32x16{} : tsum[t][i];
                            v = mfma(xh, wh[t][p], v);
                            v = mfma(xl, wh[t][p], v);
                            if constexpr (Gw<TYPE>::kWide) v = mfma(xh, wl[t][p], v);
                            tsum[t][i] = v;
                        }
                    }
                }
            }
        }
    };
    // acc += unit_m * (d * tsum - dmin * mins . sums)
    auto finish = [&](const Regs (&r)[NT][2], int par) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            float un[16];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float4 u = *reinterpret_cast<const float4 *>(&sunit[par][32 * i + 8 * g + 4 * h]);
                un[4 * g] = u.x;
                un[4 * g + 1] = u.y;
                un[4 * g + 2] = u.z;
                un[4 * g + 3] = u.w;
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if constexpr (Q40) {
#pragma unroll
                    for (int k = 0; k < 16; ++k) acc[t][i][k] = fmaf(un[k], tsum[t][i][k], acc[t][i][k]);
                } else {
                    const float d = Gw<TYPE>::d(r[t][0]);
                    if constexpr (Gw<TYPE>::kMins) {
                        // operand halves h = 0, 1: the sums' hi and lo planes
                        const f16x8 s = __builtin_bit_cast(f16x8, ssum[par][(32 * i + col) * 2 + h]);
                        const f32x16 mm = mfma(s, k4_mins(r[t][0].hd), f32x16{});
                        const float dm = -32.0f * half_f(r[t][0].hd[0] >> 16);
#pragma unroll
                        for (int k = 0; k < 16; ++k)
                            acc[t][i][k] = fmaf(un[k], fmaf(dm, mm[k], d * tsum[t][i][k]), acc[t][i][k]);
                        __builtin_amdgcn_sched_barrier(0);
                    } else {
#pragma unroll
                        for (int k = 0; k < 16; ++k) acc[t][i][k] = fmaf(un[k], d * tsum[t][i][k], acc[t][i][k]);
                    }
                }
            }
        }
    };
    // segment `seg` to out (CONV: added to the segments before it)
    auto store = [&](int seg) {
        float *out = a.out + (CONV ? 0 : seg * a.seg_stride);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int64_t n = n0 + 32 * t + col;
            if (n >= a.N) continue;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
#pragma unroll
                for (int k = 0; k < 16; ++k) {
                    const int m = m0 + 32 * i + 8 * (k >> 2) + 4 * h + (k & 3);
                    if (m < a.M) {
                        float *p = out + m * a.out_stride + n;
                        if constexpr (CONV) *p = seg == 0 ? acc[t][i][k] : *p + acc[t][i][k];
                        else *p = acc[t][i][k];
                    }
                }
            }
        }
    };

    stage_table<TYPE>(a, tab);

    if constexpr (CONV) {
        for (int seg = 0; seg < a.nseg; ++seg) {
            const int b0 = seg * a.per_seg, b1 = min(b0 + a.per_seg, a.B);
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int i = 0; i < MT; ++i) acc[t][i] = f32x16{};
            for (int b = b0; b < b1; ++b) {
                Regs r0[NT][2], r1[NT][2];
                load_raw(r0, b, 0);
                load_raw(r1, b, 1);
                __syncthreads();  // the previous superblock's operands are read
                const int64_t left = a.K - 256 * static_cast<int64_t>(b);
                for (int r = wave; r < BM && m0 + r < a.M; r += kGmWaves) {
                    const XPlanes c = convert_superblock(a.x + (m0 + r) * a.x_stride + 256 * static_cast<int64_t>(b),
                                                         static_cast<int>(left < 256 ? left : 256), a.x_al16 != 0, lane);
                    store_superblock(c, r, lane, reinterpret_cast<uint8_t *>(xh0) + kGmHalfBytes * r,
                                     reinterpret_cast<uint8_t *>(xh1) + kGmHalfBytes * r,
                                     reinterpret_cast<_Float16 *>(ssum[0]) + 16 * r);
                    if (lane == 0) sunit[0][r] = c.unit;
                }
                __syncthreads();
                compute(r0, xh0, 0);
                compute(r1, xh1, 1);
                finish(r1, 0);
            }
            store(seg);
        }
    } else {
        const int seg = blockIdx.y;
        const int b0 = seg * a.per_seg, b1 = min(b0 + a.per_seg, a.B);
        auto half_src = [&](int b, int half) {
            return a.planes + (static_cast<int64_t>(2 * b + half) * a.Mp + m0) * kGmHalfBytes;
        };
        // sums and units of superblock b: threads 0 .. 2 BM - 1 and 0 .. BM - 1
        auto load_tail = [&](int b, uint4 &s, float &u) {
            if (threadIdx.x < 2 * BM)
                s = reinterpret_cast<const uint4 *>(a.sums)[(static_cast<int64_t>(b) * a.Mp + m0) * 2 + threadIdx.x];
            if (threadIdx.x < BM) u = a.unit[static_cast<int64_t>(b) * a.Mp + m0 + threadIdx.x];
        };
        auto put_tail = [&](int par, const uint4 &s, float u) {
            if (threadIdx.x < 2 * BM) ssum[par][threadIdx.x] = s;
            if (threadIdx.x < BM) sunit[par][threadIdx.x] = u;
        };
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[t][i] = f32x16{};
        uint4 s = make_uint4(0, 0, 0, 0);
        float u = 0.f;
        Regs r[NT][2], rn[NT][2];
        copy_planes<BM>(half_src(b0, 0), xh0, wave, lane);
        load_tail(b0, s, u);
        load_raw(r, b0, 0);
        put_tail(b0 & 1, s, u);
        gm_barrier();
        for (int b = b0; b < b1; ++b) {
            const bool more = b + 1 < b1;
            copy_planes<BM>(half_src(b, 1), xh1, wave, lane);
            load_raw(rn, b, 1);
            __builtin_amdgcn_sched_barrier(0);  // the next half's loads go out before this half's work
            compute(r, xh0, 0);
            gm_barrier();
            if (more) {
                copy_planes<BM>(half_src(b + 1, 0), xh0, wave, lane);
                load_tail(b + 1, s, u);
                load_raw(r, b + 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            compute(rn, xh1, 1);
            finish(rn, b & 1);
            if (more) put_tail((b + 1) & 1, s, u);
            gm_barrier();
        }
        store(seg);
    }
}

// y = partial 0 + partial 1 + ..., in segment order
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const float *part, int64_t seg_stride, int nseg, int M,
                                                          int64_t N, float *y, int64_t y_stride) {
    const int64_t n = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (n >= N) return;
    for (int m = blockIdx.y; m < M; m += gridDim.y) {
        const float *p = part + m * N + n;
        float v = p[0];
        for (int s = 1; s < nseg; ++s) v += p[s * seg_stride];
        y[m * y_stride + n] = v;
    }
}

typedef void (*gemm_fn)(GemmArgs);

template <int TYPE>
gemm_fn pick_gemm_type(int mt, bool conv) {
    if (conv) return mt == 1 ? gemm_kernel<TYPE, 1, true> : gemm_kernel<TYPE, 2, true>;
    return mt == 1 ? gemm_kernel<TYPE, 1, false> : gemm_kernel<TYPE, 2, false>;
}

gemm_fn pick_gemm(int type, int mt, bool conv) {
    switch (type) {
    case MI355X_TYPE_Q4_0: return pick_gemm_type<MI355X_TYPE_Q4_0>(mt, conv);
    case MI355X_TYPE_Q3_K: return pick_gemm_type<MI355X_TYPE_Q3_K>(mt, conv);
    case MI355X_TYPE_Q4_K: return pick_gemm_type<MI355X_TYPE_Q4_K>(mt, conv);
    case MI355X_TYPE_Q5_K: return pick_gemm_type<MI355X_TYPE_Q5_K>(mt, conv);
    case MI355X_TYPE_Q6_K: return pick_gemm_type<MI355X_TYPE_Q6_K>(mt, conv);
    case MI355X_TYPE_IQ4_XS: return pick_gemm_type<MI355X_TYPE_IQ4_XS>(mt, conv);
    case MI355X_TYPE_IQ3_S: return pick_gemm_type<MI355X_TYPE_IQ3_S>(mt, conv);
    case MI355X_TYPE_IQ3_XXS: return pick_gemm_type<MI355X_TYPE_IQ3_XXS>(mt, conv);
    case MI355X_TYPE_IQ2_S: return pick_gemm_type<MI355X_TYPE_IQ2_S>(mt, conv);
    default: return nullptr;
    }
}

constexpr size_t kGmPartialMax = size_t(64) << 20;

size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

}  // namespace

// From how many activations the matrix cores take a call: for the K/IQ types,
// whose alternative is one GEMV each (7-12 us at the FFN shapes against 40 us
// for up to 64 here), from 4; for Q4_0 from 16, past two passes of the 8-row
// kernels.
bool gemm_batched_supports(const mi355x_ctx *ctx, const GemvArgs &a, int64_t M) {
    if (ctx->kernel_variant != MI355X_VARIANT_AUTO && ctx->kernel_variant != MI355X_VARIANT_DIGITS) return false;
    if (a.x_bf16 || a.N <= 0 || a.K <= 0) return false;
    // 32-bit offsets into the 64 rows of a wavefront
    const int64_t row_bytes = a.type == MI355X_TYPE_Q4_0 ? a.K / 32 * 18 : a.K / 256 * kq_layout(a.type).block_bytes;
    if (row_bytes <= 0 || row_bytes >= (int64_t(1) << 31) / 64 || a.N >= (int64_t(1) << 31)) return false;
    if (a.type == MI355X_TYPE_Q4_0) {
        // dword-aligned loads of code groups
        if (reinterpret_cast<uintptr_t>(a.W) % 4 != 0 || row_bytes % 4 != 0) return false;
        return M >= 16;
    }
    // codes times scales exact in f16
    if ((a.type == MI355X_TYPE_IQ3_XXS || a.type == MI355X_TYPE_IQ2_S) &&
        (a.type == MI355X_TYPE_IQ3_XXS ? ctx->iq3xxs_max : ctx->iq2s_max) > 66)
        return false;
    return M >= 4;
}

int launch_gemm_batched(mi355x_ctx *ctx, const GemvArgs &a, int64_t x_stride, int64_t y_stride, int64_t M_total,
                        bool noalloc) {
    const bool q40 = a.type == MI355X_TYPE_Q4_0;
    const int64_t row_bytes = q40 ? a.K / 32 * 18 : a.K / 256 * kq_layout(a.type).block_bytes;
    GemmArgs g{};
    g.W = a.W;
    g.N = a.N;
    g.K = a.K;
    g.row_bytes = row_bytes;
    g.B = static_cast<int>((a.K + 255) / 256);
    g.blocks = static_cast<int>(a.K / 32);
    g.x_stride = x_stride;
    g.x_al16 = reinterpret_cast<uintptr_t>(a.x) % 16 == 0 && x_stride % 4 == 0 ? 1 : 0;
    if (a.type == MI355X_TYPE_IQ3_XXS) g.grid = static_cast<const uint32_t *>(ctx->iq3xxs_grid);
    if (a.type == MI355X_TYPE_IQ2_S) g.grid = static_cast<const uint32_t *>(ctx->iq2s_grid);
    if ((a.type == MI355X_TYPE_IQ3_XXS || a.type == MI355X_TYPE_IQ2_S) && !g.grid)
        return set_error(MI355X_EUNSUPPORTED, "grid table not installed for this IQ type");
    g.ntiles = static_cast<int>((a.N + kGmCols - 1) / kGmCols);
    std::unique_lock<std::mutex> lk(ctx->mu, std::defer_lock);
    if (!noalloc) lk.lock();
    for (int64_t mb = 0; mb < M_total; mb += kGmMaxRows) {
        const int M = static_cast<int>(std::min<int64_t>(kGmMaxRows, M_total - mb));
        const int mt = M <= 32 ? 1 : 2;
        g.M = M;
        g.mtiles = (M + 32 * mt - 1) / (32 * mt);
        g.Mp = g.mtiles * 32 * mt;
        g.x = static_cast<const float *>(a.x) + mb * x_stride;
        float *y = a.y + mb * y_stride;
        const int64_t tiles = static_cast<int64_t>(g.ntiles) * g.mtiles;
        // segments of K: enough workgroups for two per CU, at least two
        // superblocks each, partials within kGmPartialMax
        int64_t seg = std::max<int64_t>(1, 2 * ctx->num_cus / tiles);
        seg = std::min<int64_t>(seg, std::max(1, g.B / 2));
        seg = std::min<int64_t>(seg, std::max<int64_t>(1, static_cast<int64_t>(kGmPartialMax / (4 * M * a.N))));
        g.per_seg = static_cast<int>((g.B + seg - 1) / seg);
        g.nseg = (g.B + g.per_seg - 1) / g.per_seg;
        const unsigned grid_x = static_cast<unsigned>((g.ntiles + 7) / 8 * 8 * g.mtiles);
        const gemm_fn k = pick_gemm(a.type, mt, noalloc);
        if (noalloc) {
            // planes converted by each workgroup, segments one after another:
            // the same sums in the same order, no buffer
            g.out = y;
            g.out_stride = y_stride;
            hipLaunchKernelGGL(k, dim3(grid_x), dim3(kGmThreads), 0, ctx->stream, g);
            MI355X_HIP(hipGetLastError());
            continue;
        }
        const size_t planes = static_cast<size_t>(g.B) * 2 * g.Mp * kGmHalfBytes;
        const size_t sums = static_cast<size_t>(g.B) * g.Mp * 32;
        const size_t units = align256(static_cast<size_t>(g.B) * g.Mp * 4);
        const size_t part = g.nseg > 1 ? static_cast<size_t>(g.nseg) * M * a.N * 4 : 0;
        const size_t need = planes + align256(sums) + units + part;
        if (ctx->gemm_bytes < need) {
            const int rc = free_device(ctx, ctx->gemm_buf);
            if (rc) return rc;
            ctx->gemm_buf = nullptr;
            ctx->gemm_bytes = 0;
            MI355X_HIP(hipMalloc(&ctx->gemm_buf, need));
            ctx->gemm_bytes = need;
        }
        uint8_t *p = static_cast<uint8_t *>(ctx->gemm_buf);
        g.planes = p;
        g.sums = reinterpret_cast<const _Float16 *>(p + planes);
        g.unit = reinterpret_cast<const float *>(p + planes + align256(sums));
        float *partial = reinterpret_cast<float *>(p + planes + align256(sums) + units);
        g.out = g.nseg > 1 ? partial : y;
        g.out_stride = g.nseg > 1 ? a.N : y_stride;
        g.seg_stride = static_cast<int64_t>(M) * a.N;
        const int64_t tasks = static_cast<int64_t>(M) * g.B;
        hipLaunchKernelGGL(gemm_planes_kernel, dim3(static_cast<unsigned>((tasks + 3) / 4)), dim3(256), 0, ctx->stream,
                           g.x, x_stride, a.K, g.x_al16, M, g.Mp, g.B, p, const_cast<_Float16 *>(g.sums),
                           const_cast<float *>(g.unit));
        MI355X_HIP(hipGetLastError());
        hipLaunchKernelGGL(k, dim3(grid_x, static_cast<unsigned>(g.nseg)), dim3(kGmThreads), 0, ctx->stream, g);
        MI355X_HIP(hipGetLastError());
        if (g.nseg > 1) {
            hipLaunchKernelGGL(gemm_reduce_kernel, dim3(static_cast<unsigned>((a.N + 255) / 256), std::min(M, 64)),
                               dim3(256), 0, ctx->stream, partial, g.seg_stride, g.nseg, M, a.N, y, y_stride);
            MI355X_HIP(hipGetLastError());
        }
    }
    return MI355X_OK;
}

}  // namespace mi355x
