// K/IQ GEMV for a few activation rows (2 to 8) on the integer matrix cores of
// gfx950, one launch: the digit arithmetic of the one-row kernels (16-bit
// activation digits in two signed-byte planes, exact integer sums per scale
// group) with the products on v_mfma_i32_16x16x64_i8.
//
// Why.  The one-row kernels spend 2.3-3.9 VALU instructions per weight and
// activation; run once per activation they cost M times 7-12 us.  Here the
// codes are decoded once (0.4-1.3 instructions per weight) and stay in
// registers while every activation's digits meet them.  One MFMA multiplies 16
// weight rows x 64 codes, and its 16 result rows keep the scale groups and
// planes apart: lane (n, g) of the weight operand holds 16 codes of weight row
// n that share one scale; the activation operand is zero except in rows
// 4g .. 4g + 3 of lane group g, so lane (n, g) of the result receives exactly
// the sums of its own codes -- rows 4g + 2r + p the sum over digit plane p of
// the operands given row pair r -- and scales them with its own row's scales.
// (For one activation the one-row kernels stay faster: 6.9 against 8.7 us at
// Q4_K 14336x4096, 9 against 17 at IQ3_S 8192x8192; a wavefront's chain of
// operand reads, products and sums is longer than theirs.)
//
// Work split.  A workgroup of 8 wavefronts owns tiles of 16 rows and splits K:
// wavefront v takes units v, v + 8, ... of every tile.  Plane types (Q4_K,
// Q5_K, IQ4_XS): a unit is a superblock, lane group g reads slices g, g + 4 --
// 64 contiguous bytes per row and load.  Group types: a unit is a pair of
// slices (2 sp, 2 sp + 1) of a group's 8 superblocks, lane group g reads
// superblocks g, g + 4, whose records are contiguous.  A unit's registers are
// reloaded with the next tile's right after its decode, so NU units per
// wavefront stay in flight; row sums meet in LDS.
#include "internal.h"
#include "kq_device.h"

#include <algorithm>
#include <cstdint>

namespace mi355x {
namespace {

constexpr int kMxWaves = 8;
constexpr int kMxThreads = 64 * kMxWaves;
constexpr int kMxRows = 16;
constexpr int kMxRowSlots = 32;   // (tiles x activations) whose sums wait in LDS
constexpr int kMxMaxAct = 8;      // activations per launch
constexpr int kMxMaxBlocks = 64;  // superblocks per row

typedef int i32x4 __attribute__((ext_vector_type(4)));

struct MxArgs {
    const uint8_t *W;
    int64_t N;
    int64_t row_bytes;
    int B;       // superblocks per row
    int tiles;
    int M;
    const float *x;
    int64_t x_stride;
    int x_al16;
    float *y;
    int64_t y_stride;
    const uint32_t *grid;
};

constexpr bool mx_grouped(int type) { return kq_layout(type).grouped; }
// units of a row of B superblocks
constexpr int mx_units(int type, int B) { return mx_grouped(type) ? 4 * ((B + 7) / 8) : B; }

__device__ __forceinline__ u32x4 splat_and(const u32x4 &v, uint32_t m) { return v & u32x4{m, m, m, m}; }

// ---- activations ----------------------------------------------------------------
// LDS, per activation: digit planes [2][256 B] in natural order, the units of
// the 32-value blocks [8 B], and (K4 types) u * sum Z of every 16 values, in
// the order 4c + 2h + f of value 64c + 32f + 16h; then 16 zero bytes.
constexpr size_t mx_act_bytes(int type, int B) {
    return static_cast<size_t>(B) * (512 + 32 + (slice_shape(type) == kK4 ? 64 : 0));
}
struct MxLds {
    uint8_t *z;    // of activation 0
    uint32_t act;  // bytes per activation
    int B;
    __device__ const uint8_t *planes(int m) const { return z + m * act; }
    __device__ float *u(int m) const { return reinterpret_cast<float *>(z + m * act + 512 * B); }
    __device__ float *s16(int m) const { return u(m) + 8 * B; }
};

template <int TYPE>
__device__ __forceinline__ void mx_stage(const MxArgs &a, const MxLds &l, int tid) {
    const int runs = 32 * a.B;
    for (int m = 0; m < a.M; ++m) {
        const float *x = a.x + m * a.x_stride;
        uint8_t *z = l.z + m * l.act;
        // runs is a multiple of 32: a quad is inside or outside
        for (int r = tid; r < runs; r += kMxThreads) {
            float4 lo, hi;
            load_x8(x, a.x_al16 ? kXF32 : kXF32Any, 8 * r, lo, hi);
            const float q[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            // digits as stage_run_dg
            float mx = fmaxf(fmaxf(fmaxf(fabsf(q[0]), fabsf(q[1])), fmaxf(fabsf(q[2]), fabsf(q[3]))),
                             fmaxf(fmaxf(fabsf(q[4]), fabsf(q[5])), fmaxf(fabsf(q[6]), fabsf(q[7]))));
            mx = fmaxf(mx, quad_x1_f(mx));
            mx = fmaxf(mx, quad_x2_f(mx));
            float c, u;
            dg_scale(mx, c, u);
            uint32_t F[8], G1[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                F[t] = __builtin_bit_cast(uint32_t, fmaf(q[t], c, 12582912.0f));
                G1[t] = F[t] + 128u;
            }
            *reinterpret_cast<uint2 *>(z + 8 * r) =
                make_uint2(gather_byte<0>(F[0], F[1], F[2], F[3]), gather_byte<0>(F[4], F[5], F[6], F[7]));
            *reinterpret_cast<uint2 *>(z + 256 * a.B + 8 * r) =
                make_uint2(gather_byte<1>(G1[0], G1[1], G1[2], G1[3]), gather_byte<1>(G1[4], G1[5], G1[6], G1[7]));
            if ((r & 3) == 0) l.u(m)[r >> 2] = u;
            if constexpr (slice_shape(TYPE) == kK4) {
                const uint32_t fs = (F[0] + F[1] + F[2]) + (F[3] + F[4] + F[5]) + (F[6] + F[7]);
                const float zs = static_cast<float>(static_cast<int>(fs - 8u * 0x4B400000u));
                const float z2 = zs + quad_x1_f(zs);
                const int g = r >> 1;  // 16-value group 4c + 2f + h -> 4c + 2h + f
                if ((r & 1) == 0) l.s16(m)[(g & ~3) | ((g & 1) << 1) | ((g >> 1) & 1)] = u * z2;
            }
        }
    }
    if (tid < 4) reinterpret_cast<uint32_t *>(l.z + a.M * l.act)[tid] = 0u;
}

// ---- products -------------------------------------------------------------------
struct MxLane {
    int g;            // lane group
    uint32_t on[2];   // row pair r: all ones where this lane holds a digit row
    uint32_t at[2];   // its plane's offset, or the zero bytes'
};
// activation m's operand of row pair r for the 16 values at `off`
__device__ __forceinline__ i32x4 mx_x(const MxLane &q, const MxLds &l, int m, uint32_t off, int r) {
    return *reinterpret_cast<const i32x4 *>(l.z + q.at[r] + ((off + m * l.act) & q.on[r]));
}
__device__ __forceinline__ i32x4 mx_mfma(const i32x4 &x, const u32x4 &w, const i32x4 &c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(x, __builtin_bit_cast(i32x4, w), c, 0, 0, 0);
}
// the sum of row pair r, rounded once
__device__ __forceinline__ float mx_sum(const i32x4 &d, int r) {
    return static_cast<float>(d[2 * r] + d[2 * r + 1] * 256);
}

template <int TYPE>
struct Mx;

// byte `k` of w as a float
__device__ __forceinline__ float mx_byte(uint32_t w, int k) { return static_cast<float>((w >> (8 * k)) & 0xFFu); }

template <bool Q5>
struct MxK4 {
    struct Regs {
        u32x4 q[2], hd, qh;
    };
    __device__ static Regs load(const LaneRow &r, int b, int g) {
        Regs v;
        const uint32_t o = r.P[0] + 128u * b + 16u * g;
        v.q[0] = ld128(r, o);
        v.q[1] = ld128(r, o + 64);
        if constexpr (Q5) v.qh = ld128(r, r.P[1] + 32u * b + 16u * (g & 1));
        v.hd = ld128(r, (Q5 ? r.P[2] : r.P[1]) + 16u * b);
        return v;
    }
    template <int MB>
    __device__ static void compute(const Regs &v, int b, const MxLane &q, const MxLds &l, int M, const uint32_t *,
                                   float (&acc)[MB]) {
        const int c0 = q.g >> 1, h = q.g & 1;
        const uint32_t sh = 16u * c0;
        u32x4 qh{};
        if constexpr (Q5) qh = v.qh >> (2u * c0);
        const float d = half_f(v.hd[0] & 0xFFFF), dmin = half_f(v.hd[0] >> 16);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            u32x4 lo = splat_and(v.q[i], 0x0F0F0F0Fu), hi = splat_and(v.q[i] >> 4u, 0x0F0F0F0Fu);
            if constexpr (Q5) {
                lo |= splat_and(i ? qh : qh << 4u, 0x10101010u);
                hi |= splat_and(i ? qh >> 1u : qh << 3u, 0x10101010u);
            }
            // (scale, min) bytes of sub-blocks 2c, 2c + 1, c = c0 + 2 i
            // (scale_min_pair_k4; c < 2 exactly for i = 0)
            const uint32_t a2 = v.hd[1] >> sh, b2 = v.hd[2] >> sh, c2 = v.hd[3] >> sh;
            const uint32_t sc = i == 0 ? (a2 & 0x3F3Fu) : ((c2 & 0x0F0Fu) | ((a2 >> 2) & 0x3030u));
            const uint32_t mn = i == 0 ? (b2 & 0x3F3Fu) : (((c2 >> 4) & 0x0F0Fu) | ((b2 >> 2) & 0x3030u));
            const float d0 = d * mx_byte(sc, 0), d1 = d * mx_byte(sc, 1);
            const float m0 = dmin * mx_byte(mn, 0), m1 = dmin * mx_byte(mn, 1);
            const int c = c0 + 2 * i;
            const uint32_t off = 256u * b + 64u * c + 16u * h;
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                if (m >= M) break;
                i32x4 p = mx_mfma(mx_x(q, l, m, off, 0), lo, i32x4{0, 0, 0, 0});
                p = mx_mfma(mx_x(q, l, m, off + 32, 1), hi, p);
                const float2 u = *reinterpret_cast<const float2 *>(l.u(m) + 8 * b + 2 * c);
                const float2 z = *reinterpret_cast<const float2 *>(l.s16(m) + 16 * b + 4 * c + 2 * h);
                acc[m] += fmaf(d0, mx_sum(p, 0) * u.x, d1 * (mx_sum(p, 1) * u.y)) - fmaf(m0, z.x, m1 * z.y);
            }
        }
    }
};
template <>
struct Mx<MI355X_TYPE_Q4_K> : MxK4<false> {};
template <>
struct Mx<MI355X_TYPE_Q5_K> : MxK4<true> {};

template <>
struct Mx<MI355X_TYPE_IQ4_XS> {
    struct Regs {
        u32x4 q[2];
        u32x2 hd;
    };
    __device__ static Regs load(const LaneRow &r, int b, int g) {
        const uint32_t o = r.P[0] + 128u * b + 16u * g;
        return {{ld128(r, o), ld128(r, o + 64)}, ld64(r, r.P[1] + 8u * b)};
    }
    template <int MB>
    __device__ static void compute(const Regs &v, int b, const MxLane &q, const MxLds &l, int M, const uint32_t *,
                                   float (&acc)[MB]) {
        using D = KqDg<MI355X_TYPE_IQ4_XS>;
        u32x4 lo[2], hi[2];
        float f[2];
        const float d = half_f(v.hd[0] & 0xFFFF);
        const uint32_t sh = v.hd[0] >> 16;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                lo[i][k] = D::lookup(v.q[i][k] & 0x0F0F0F0Fu);
                hi[i][k] = D::lookup((v.q[i][k] >> 4) & 0x0F0F0F0Fu);
            }
            const int s = q.g + 4 * i;
            const uint32_t ls = ((v.hd[1] >> (4 * s)) & 15u) | (((sh >> (2 * s)) & 3u) << 4);
            f[i] = d * static_cast<float>(static_cast<int>(ls) - 32);
        }
        const uint32_t off = 256u * b + 32u * q.g;
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            if (m >= M) break;
            i32x4 p{0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                p = mx_mfma(mx_x(q, l, m, off + 128 * i, i), lo[i], p);
                p = mx_mfma(mx_x(q, l, m, off + 128 * i + 16, i), hi[i], p);
            }
            const float *u = l.u(m) + 8 * b + q.g;
            acc[m] += fmaf(f[0], mx_sum(p, 0) * u[0], f[1] * (mx_sum(p, 1) * u[4]));
        }
    }
};

// Group types: superblock 8 t + 4 i + g of unit (t, sp); past the last group's
// end the last superblock again, with d = 0.
struct MxPos {
    GPos p;
    uint32_t b;
    bool in;
};
__device__ __forceinline__ MxPos mx_pos(const LaneRow &r, int bb, int unit, int i, int g) {
    const uint32_t want = 8u * (unit >> 2) + 4u * i + g, B = r.P[0];
    const bool in = want < B;
    const uint32_t b = in ? want : B - 1;
    return {gpos(r, bb, b, 2 * (unit & 3)), b, in};
}
// value offset of superblock 4 i + g of the unit's group (clamped alike)
__device__ __forceinline__ uint32_t mx_block(int unit, int i, int g, int B) {
    const int want = 8 * (unit >> 2) + 4 * i + g;
    return static_cast<uint32_t>(want < B ? want : B - 1);
}

template <>
struct Mx<MI355X_TYPE_Q6_K> {
    struct One {
        u32x4 a[2];  // ql, ql runs of the two slices
        u32x2 h[2];  // their qh runs
        uint32_t sw, d;
    };
    struct Regs {
        One v[2];
    };
    __device__ static Regs load(const LaneRow &r, int unit, int g) {
        Regs o;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const MxPos q = mx_pos(r, 210, unit, i, g);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const uint32_t at = q.p.base + 24 * (q.p.m + s * q.p.g);
                o.v[i].a[s] = ld128(r, at);
                o.v[i].h[s] = ld64(r, at + 16);
            }
            o.v[i].sw = ld32(r, q.p.base + 192 * q.p.g + 16 * q.p.bl + 4 * (unit & 3));
            o.v[i].d = q.in ? ld16(r, q.p.d) : 0u;
        }
        return o;
    }
    template <int MB>
    __device__ static void compute(const Regs &o, int unit, const MxLane &q, const MxLds &l, int M, const uint32_t *,
                                   float (&acc)[MB]) {
        const int hh = (unit >> 1) & 1, kk = unit & 1;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const One &v = o.v[i];
            const uint32_t b = mx_block(unit, i, q.g, l.B);
            const float d = 0.25f * half_f(v.d);
            u32x4 w[4];
            float f[4];
            // 4 (code - 32) as signed bytes: the 6-bit code at the top of the
            // byte, its top bit flipped
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        const uint32_t A = v.a[s][2 * (j & 1) + k], H = v.h[s][k];
                        w[j][2 * s + k] = (((j >= 2 ? A >> 2 : A << 2) & 0x3C3C3C3Cu) |
                                           ((j < 3 ? H << (6 - 2 * j) : H) & 0xC0C0C0C0u)) ^ 0x80808080u;
                    }
                f[j] = d * static_cast<float>(static_cast<int32_t>(v.sw << (24 - 8 * j)) >> 24);
            }
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                if (m >= M) break;
                const float4 u = *reinterpret_cast<const float4 *>(l.u(m) + 8 * b + 4 * hh);
                const float uu[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                for (int jp = 0; jp < 2; ++jp) {
                    i32x4 p{0, 0, 0, 0};
#pragma unroll
                    for (int r = 0; r < 2; ++r)
                        p = mx_mfma(mx_x(q, l, m, 256 * b + 128 * hh + 32 * (2 * jp + r) + 16 * kk, r), w[2 * jp + r], p);
                    acc[m] += fmaf(f[2 * jp], mx_sum(p, 0) * uu[2 * jp], f[2 * jp + 1] * (mx_sum(p, 1) * uu[2 * jp + 1]));
                }
            }
        }
    }
};

template <>
struct Mx<MI355X_TYPE_Q3_K> {
    struct One {
        u32x2 q[2];     // code bytes of the two slices
        uint32_t h[2];  // hmask bytes 8k + 0..3
        uint32_t h4[2]; // and 8k + 4..7
        u32x3 sc;
        uint32_t d;
    };
    struct Regs {
        One v[2];
    };
    __device__ static Regs load(const LaneRow &r, int unit, int g) {
        Regs o;
        const uint32_t hh = (unit >> 1) & 1;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const MxPos q = mx_pos(r, 110, unit, i, g);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const uint32_t at = q.p.base + 12 * (q.p.m + s * q.p.g);
                const u32x3 rec = ld96(r, at);
                // the other half's slice (s ^ 4) holds the other four hmask bytes
                const uint32_t other = ld32(r, (hh ? at - 48 * q.p.g : at + 48 * q.p.g) + 8);
                o.v[i].q[s] = u32x2{rec[0], rec[1]};
                o.v[i].h[s] = hh ? other : rec[2];
                o.v[i].h4[s] = hh ? rec[2] : other;
            }
            o.v[i].sc = ld96(r, q.p.base + 96 * q.p.g + 12 * q.p.bl);
            o.v[i].d = q.in ? ld16(r, q.p.d) : 0u;
        }
        return o;
    }
    template <int MB>
    __device__ static void compute(const Regs &o, int unit, const MxLane &q, const MxLds &l, int M, const uint32_t *,
                                   float (&acc)[MB]) {
        const int hh = (unit >> 1) & 1, kk = unit & 1;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const One &v = o.v[i];
            const uint32_t b = mx_block(unit, i, q.g, l.B);
            const float d = 0.03125f * half_f(v.d);
            u32x4 w[4];
            float f[4];
            // the unit's four 6-bit scales, bytes in run order 0, 2, 1, 3, top
            // bit flipped (KqDg<Q3_K>)
            const uint32_t L = kk ? v.sc[1] : v.sc[0];
            const uint32_t H = v.sc[2] >> (8 * kk + 4 * hh);
            const int SX = static_cast<int>((((L >> (4 * hh)) & 0x0F0F0F0Fu) | ((H & 0x00030003u) << 4) |
                                             ((H & 0x000C000Cu) << 10)) ^ 0x20202020u);
            f[0] = d * static_cast<float>((SX << 26) >> 26);
            f[1] = d * static_cast<float>((SX << 10) >> 26);
            f[2] = d * static_cast<float>((SX << 18) >> 26);
            f[3] = d * static_cast<float>((SX << 2) >> 26);
            // 32 (code - 4) as signed bytes: code bits to 5-6, the hmask bit
            // (4 hh + j) flipped to 7
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        const uint32_t c = v.q[s][k], hm = (k ? v.h4[s] : v.h[s]) << (hh ? 0 : 4);
                        w[j][2 * s + k] = (((j < 3 ? c << (5 - 2 * j) : c >> 1) & 0x60606060u) |
                                           ((hm << (3 - j)) & 0x80808080u)) ^ 0x80808080u;
                    }
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                if (m >= M) break;
                const float4 u = *reinterpret_cast<const float4 *>(l.u(m) + 8 * b + 4 * hh);
                const float uu[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                for (int jp = 0; jp < 2; ++jp) {
                    i32x4 p{0, 0, 0, 0};
#pragma unroll
                    for (int r = 0; r < 2; ++r)
                        p = mx_mfma(mx_x(q, l, m, 256 * b + 128 * hh + 32 * (2 * jp + r) + 16 * kk, r), w[2 * jp + r], p);
                    acc[m] += fmaf(f[2 * jp], mx_sum(p, 0) * uu[2 * jp], f[2 * jp + 1] * (mx_sum(p, 1) * uu[2 * jp + 1]));
                }
            }
        }
    }
};

// codebook types: tables as the digit row kernels' (GridRegs::put_dg)
template <>
struct Mx<MI355X_TYPE_IQ3_S> {
    struct One {
        u32x3 rec[2];
        uint32_t qh[2], scb, d;
    };
    struct Regs {
        One v[2];
    };
    __device__ static Regs load(const LaneRow &r, int unit, int g) {
        Regs o;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const MxPos q = mx_pos(r, 110, unit, i, g);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                o.v[i].rec[s] = ld96(r, q.p.base + 12 * (q.p.m + s * q.p.g));
                o.v[i].qh[s] = ld8(r, q.p.base + 96 * q.p.g + q.p.m + s * q.p.g);
            }
            o.v[i].scb = ld8(r, q.p.base + 104 * q.p.g + 4 * q.p.bl + (unit & 3));
            o.v[i].d = q.in ? ld16(r, q.p.d) : 0u;
        }
        return o;
    }
    template <int MB>
    __device__ static void compute(const Regs &o, int unit, const MxLane &q, const MxLds &l, int M,
                                   const uint32_t *grid, float (&acc)[MB]) {
        const uint2 *gt = reinterpret_cast<const uint2 *>(grid);
        const uint2 *st = gt + kIq3sGridSize;
        const int s0 = 2 * (unit & 3);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const One &v = o.v[i];
            const uint32_t b = mx_block(unit, i, q.g, l.B);
            u32x4 w[2][2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
#pragma unroll
                for (int k = 0; k < 8; k += 2) {
                    const uint32_t i0 = byte_u(v.rec[s][k >> 2], k & 3) | (((v.qh[s] >> k) & 1u) << 8);
                    const uint32_t i1 = byte_u(v.rec[s][k >> 2], (k & 3) + 1) | (((v.qh[s] >> (k + 1)) & 1u) << 8);
                    const uint2 e0 = gt[i0], e1 = gt[i1], sl = st[byte_u(v.rec[s][2], k >> 1)];
                    w[s][k >> 2][k & 3] = __builtin_amdgcn_perm(e0.y, e0.x, sl.x);
                    w[s][k >> 2][(k & 3) + 1] = __builtin_amdgcn_perm(e1.y, e1.x, sl.y);
                }
            }
            const float d = half_f(v.d);
            const float f0 = d * static_cast<float>(2 * (v.scb & 15u) + 1), f1 = d * static_cast<float>(2 * (v.scb >> 4) + 1);
            const uint32_t off = 256 * b + 32 * s0;
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                if (m >= M) break;
                i32x4 p{0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    p = mx_mfma(mx_x(q, l, m, off + 32 * s, s), w[s][0], p);
                    p = mx_mfma(mx_x(q, l, m, off + 32 * s + 16, s), w[s][1], p);
                }
                const float2 u = *reinterpret_cast<const float2 *>(l.u(m) + 8 * b + s0);
                acc[m] += fmaf(f0, mx_sum(p, 0) * u.x, f1 * (mx_sum(p, 1) * u.y));
            }
        }
    }
};

template <>
struct Mx<MI355X_TYPE_IQ3_XXS> {
    struct One {
        u32x3 rec[2];
        uint32_t d;
    };
    struct Regs {
        One v[2];
    };
    __device__ static Regs load(const LaneRow &r, int unit, int g) {
        Regs o;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const MxPos q = mx_pos(r, 98, unit, i, g);
#pragma unroll
            for (int s = 0; s < 2; ++s) o.v[i].rec[s] = ld96(r, q.p.base + 12 * (q.p.m + s * q.p.g));
            o.v[i].d = q.in ? ld16(r, q.p.d) : 0u;
        }
        return o;
    }
    template <int MB>
    __device__ static void compute(const Regs &o, int unit, const MxLane &q, const MxLds &l, int M,
                                   const uint32_t *grid, float (&acc)[MB]) {
        const uint2 *gt = reinterpret_cast<const uint2 *>(grid);
        const uint2 *st = gt + 256;
        const int s0 = 2 * (unit & 3);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const One &v = o.v[i];
            const uint32_t b = mx_block(unit, i, q.g, l.B);
            u32x4 w[2][2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t c = v.rec[s][k >> 1];
                    const uint2 e0 = gt[byte_u(c, 2 * (k & 1))], e1 = gt[byte_u(c, 2 * (k & 1) + 1)];
                    const uint2 sl = st[(v.rec[s][2] >> (7 * k)) & 127u];
                    w[s][k >> 1][2 * (k & 1)] = __builtin_amdgcn_perm(e0.y, e0.x, sl.x);
                    w[s][k >> 1][2 * (k & 1) + 1] = __builtin_amdgcn_perm(e1.y, e1.x, sl.y);
                }
            }
            // (0.5 + n) / 2 = (2 n + 1) / 4
            const float d = 0.25f * half_f(v.d);
            const float f0 = d * static_cast<float>(2 * (v.rec[0][2] >> 28) + 1);
            const float f1 = d * static_cast<float>(2 * (v.rec[1][2] >> 28) + 1);
            const uint32_t off = 256 * b + 32 * s0;
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                if (m >= M) break;
                i32x4 p{0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    p = mx_mfma(mx_x(q, l, m, off + 32 * s, s), w[s][0], p);
                    p = mx_mfma(mx_x(q, l, m, off + 32 * s + 16, s), w[s][1], p);
                }
                const float2 u = *reinterpret_cast<const float2 *>(l.u(m) + 8 * b + s0);
                acc[m] += fmaf(f0, mx_sum(p, 0) * u.x, f1 * (mx_sum(p, 1) * u.y));
            }
        }
    }
};

template <>
struct Mx<MI355X_TYPE_IQ2_S> {
    struct One {
        u32x2 rec[2];
        uint32_t p[2], d;
    };
    struct Regs {
        One v[2];
    };
    __device__ static Regs load(const LaneRow &r, int unit, int g) {
        Regs o;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const MxPos q = mx_pos(r, 82, unit, i, g);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                o.v[i].rec[s] = ld64(r, q.p.base + 8 * (q.p.m + s * q.p.g));
                o.v[i].p[s] = ld16(r, q.p.base + 64 * q.p.g + 2 * (q.p.m + s * q.p.g));
            }
            o.v[i].d = q.in ? ld16(r, q.p.d) : 0u;
        }
        return o;
    }
    template <int MB>
    __device__ static void compute(const Regs &o, int unit, const MxLane &q, const MxLds &l, int M,
                                   const uint32_t *grid, float (&acc)[MB]) {
        const uint2 *gt = reinterpret_cast<const uint2 *>(grid);
        const uint2 *st = gt + 1024;
        const int s0 = 2 * (unit & 3);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const One &v = o.v[i];
            const uint32_t b = mx_block(unit, i, q.g, l.B);
            const float d = 0.125f * half_f(v.d);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const uint32_t qh = v.p[s] & 0xFFu, scb = v.p[s] >> 8;
                u32x4 w[2];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint2 e = gt[byte_u(v.rec[s][0], k) | (((qh >> (2 * k)) & 3u) << 8)];
                    const uint2 sl = st[byte_u(v.rec[s][1], k)];
                    w[k >> 1][2 * (k & 1)] = __builtin_amdgcn_perm(0x01010100u - e.x, e.x, sl.x);
                    w[k >> 1][2 * (k & 1) + 1] = __builtin_amdgcn_perm(0x01010100u - e.y, e.y, sl.y);
                }
                // (0.5 + n) / 4 = (2 n + 1) / 8, one nibble per 16 values
                const float f0 = d * static_cast<float>(2 * (scb & 15u) + 1), f1 = d * static_cast<float>(2 * (scb >> 4) + 1);
                const uint32_t off = 256 * b + 32 * (s0 + s);
#pragma unroll
                for (int m = 0; m < MB; ++m) {
                    if (m >= M) break;
                    i32x4 p = mx_mfma(mx_x(q, l, m, off, 0), w[0], i32x4{0, 0, 0, 0});
                    p = mx_mfma(mx_x(q, l, m, off + 16, 1), w[1], p);
                    acc[m] = fmaf(l.u(m)[8 * b + s0 + s], fmaf(f0, mx_sum(p, 0), f1 * mx_sum(p, 1)), acc[m]);
                }
            }
        }
    }
};

// ---- kernel ------------------------------------------------------------------------
template <int TYPE, int NU, int MB>
__global__ __launch_bounds__(kMxThreads, 2) void gemv_kq_mx_kernel(MxArgs a) {
    using X = Mx<TYPE>;
    constexpr int SLOTS = kMxRowSlots / MB;
    extern __shared__ uint4 mx_lds[];
    __shared__ float part[SLOTS][MB][kMxWaves][kMxRows];
    __shared__ uint32_t tab[dg_table_words(TYPE) > 0 ? dg_table_words(TYPE) : 1];
    const MxLds l{reinterpret_cast<uint8_t *>(mx_lds), static_cast<uint32_t>(mx_act_bytes(TYPE, a.B)), a.B};

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    const int U = mx_units(TYPE, a.B);
    MxLane q;
    q.g = g;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const bool on = (n >> 2) == g && ((n >> 1) & 1) == r;
        q.on[r] = on ? ~0u : 0u;
        q.at[r] = on ? (n & 1) * 256u * a.B : a.M * l.act;
    }

    // this lane's row of tile t (an empty buffer past the last tile)
    auto view = [&](int t) {
        const int64_t n0 = static_cast<int64_t>(t) * kMxRows;
        const int64_t rows = t < a.tiles ? (a.N - n0 < kMxRows ? a.N - n0 : kMxRows) : 0;
        const uint8_t *base = a.W + (rows > 0 ? n0 : 0) * a.row_bytes;
        LaneRow r;
        r.rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base), 0,
                                                   static_cast<uint32_t>(rows * a.row_bytes), kBufferWord3);
        r.base = static_cast<uint32_t>(n) * static_cast<uint32_t>(a.row_bytes);
        constexpr KqLayout L = kq_layout(TYPE);
        const bool flipped = kq_row_flipped(reinterpret_cast<uintptr_t>(base) + r.base);
        if constexpr (L.grouped) {
            r.P[0] = static_cast<uint32_t>(a.B);
            r.P[1] = flipped ? 1u : 0u;
        } else {
#pragma unroll
            for (int i = 0; i < 5; ++i)
                r.P[i] = i < L.nfields ? static_cast<uint32_t>(kq_plane_start(L, i, a.B, flipped)) : 0u;
        }
        return r;
    };

    // the first tile's weights in flight while the activations are staged
    KqArgs ga{};
    ga.grid = a.grid;
    GridRegs<TYPE, kMxThreads> gr;
    gr.fetch(ga, tid, kMxThreads);
    typename X::Regs regs[NU];
    {
        const LaneRow r = view(blockIdx.x);
#pragma unroll
        for (int k = 0; k < NU; ++k)
            if (wave + kMxWaves * k < U) regs[k] = X::load(r, wave + kMxWaves * k, g);
    }
    mx_stage<TYPE>(a, l, tid);
    gr.put_dg(tab, tid, kMxThreads);
    __syncthreads();

    for (int t0 = blockIdx.x; t0 < a.tiles; t0 += gridDim.x * SLOTS) {
        int slot = 0;
        for (int t = t0; slot < SLOTS && t < a.tiles; ++slot, t += gridDim.x) {
            const LaneRow next = view(t + static_cast<int>(gridDim.x) < a.tiles ? t + static_cast<int>(gridDim.x) : a.tiles);
            float acc[MB];
#pragma unroll
            for (int m = 0; m < MB; ++m) acc[m] = 0.f;
#pragma unroll
            for (int k = 0; k < NU; ++k) {
                const int unit = wave + kMxWaves * k;
                if (unit < U) {
                    // operand addresses are formed here again, not held in
                    // registers for all (unit, activation) over the tiles
                    MxLds lu = l;
                    MxLane qu = q;
                    asm volatile("" : "+s"(lu.act), "+v"(qu.at[0]), "+v"(qu.at[1]));
                    X::compute(regs[k], unit, qu, lu, a.M, tab, acc);
                    __builtin_amdgcn_sched_barrier(0);
                    regs[k] = X::load(next, unit, g);
                }
            }
            // lanes n, n + 16, n + 32, n + 48 hold one row
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                if (m >= a.M) break;
                float v = acc[m];
                v += __shfl_xor(v, 16);
                v += __shfl_xor(v, 32);
                if (g == 0) part[slot][m][wave][n] = v;
            }
        }
        __syncthreads();
        for (int i = tid; i < slot * MB * kMxRows; i += kMxThreads) {
            const int r = i % kMxRows, m = i / kMxRows % MB, sl = i / (kMxRows * MB);
            const int64_t row = (static_cast<int64_t>(t0) + static_cast<int64_t>(sl) * gridDim.x) * kMxRows + r;
            if (m < a.M && row < a.N) {
                float s = part[sl][m][0][r];
#pragma unroll
                for (int w = 1; w < kMxWaves; ++w) s += part[sl][m][w][r];
                a.y[m * a.y_stride + row] = s;
            }
        }
        __syncthreads();
    }
}

typedef void (*mx_fn)(MxArgs);

template <int TYPE, int MB>
mx_fn pick_mx_nu(int nu) {
    if (nu == 1) return gemv_kq_mx_kernel<TYPE, 1, MB>;
    if (nu == 2) return gemv_kq_mx_kernel<TYPE, 2, MB>;
    if constexpr (mx_grouped(TYPE)) return gemv_kq_mx_kernel<TYPE, 4, MB>;
    else return nu <= 4 ? gemv_kq_mx_kernel<TYPE, 4, MB> : gemv_kq_mx_kernel<TYPE, 8, MB>;
}
template <int TYPE>
mx_fn pick_mx_type(int nu, int mb) {
    return mb <= 2 ? pick_mx_nu<TYPE, 2>(nu) : mb <= 4 ? pick_mx_nu<TYPE, 4>(nu) : pick_mx_nu<TYPE, 8>(nu);
}

mx_fn pick_mx(int type, int nu, int mb) {
    switch (type) {
    case MI355X_TYPE_Q3_K: return pick_mx_type<MI355X_TYPE_Q3_K>(nu, mb);
    case MI355X_TYPE_Q4_K: return pick_mx_type<MI355X_TYPE_Q4_K>(nu, mb);
    case MI355X_TYPE_Q5_K: return pick_mx_type<MI355X_TYPE_Q5_K>(nu, mb);
    case MI355X_TYPE_Q6_K: return pick_mx_type<MI355X_TYPE_Q6_K>(nu, mb);
    case MI355X_TYPE_IQ4_XS: return pick_mx_type<MI355X_TYPE_IQ4_XS>(nu, mb);
    case MI355X_TYPE_IQ3_S: return pick_mx_type<MI355X_TYPE_IQ3_S>(nu, mb);
    case MI355X_TYPE_IQ3_XXS: return pick_mx_type<MI355X_TYPE_IQ3_XXS>(nu, mb);
    case MI355X_TYPE_IQ2_S: return pick_mx_type<MI355X_TYPE_IQ2_S>(nu, mb);
    default: return nullptr;
    }
}

}  // namespace

// What it takes: digit arithmetic (so never where the one-row form of the type
// and size sums in f32), and activations that fit the LDS in one launch (3 to 8;
// a second launch reads and decodes the weights again: Q4_K 4096x8192 M = 8 28
// us in two, 23 in the f16 form of many activations).  us against the better of
// M one-row launches and that form:
//   M = 2  Q4_K 2048x2048 5.1 (8.3), 14336x4096 12.3 (14.8); Q6_K 4096x14336
//          18.6 (24.4), but 1024x16384 24 (22): few tiles of long rows, whose
//          loads of 128 bytes leave most of the chip waiting; IQ2_S 16384x2048
//          10 (12), but 8192x8192 18.1 (16.2): its codebook reads
//   M = 4  Q4_K 14336x4096 15.4 (25.1), Q6_K 4096x14336 23.7 (42.9), IQ3_S
//          8192x8192 22.8 (33.7)
//   M = 8  Q4_K 2048x2048 8.5 (15.7), Q5_K 14336x4096 28.0 (30.2), IQ3_S 8192x8192
//          32.0 (34.0), but Q4_K 14336x4096 26.3 (24.4; 18.9 at M = 6): with
//          more than 6 activations of 4096 values one workgroup fits a CU
bool kq_mx_takes(const mi355x_ctx *ctx, const GemvArgs &a, int64_t M) {
    if (a.type == MI355X_TYPE_Q4_0 || a.x_bf16 || M < 2 || M > kMxMaxAct || a.N <= 0 || a.N >= (int64_t(1) << 31)) return false;
    if (!form_is_auto(ctx, a.type)) return false;
    const int64_t B = a.K / 256;
    if (B < 1 || B > kMxMaxBlocks || !kq_digit_rows(ctx, a.type, a.N, a.K)) return false;
    const size_t fixed = kMxRowSlots * kMxWaves * kMxRows * sizeof(float) + dg_table_words(a.type) * 4u + 256;
    if (fixed + M * mx_act_bytes(a.type, static_cast<int>(B)) > ctx->max_lds_per_block) return false;
    if (M == 2 && ((mx_grouped(a.type) && B > 32 && a.N < 4096) || (a.type == MI355X_TYPE_IQ2_S && B > 16))) return false;
    return a.type != MI355X_TYPE_Q4_K || M <= 6 || B < 16 || a.N * a.K < (int64_t(1) << 25);
}

int launch_gemv_kq_mx(mi355x_ctx *ctx, const GemvArgs &a, int64_t x_stride, int64_t y_stride, int M) {
    MxArgs g{};
    g.W = a.W;
    g.N = a.N;
    g.B = static_cast<int>(a.K / 256);
    g.row_bytes = static_cast<int64_t>(g.B) * kq_layout(a.type).block_bytes;
    g.tiles = static_cast<int>((a.N + kMxRows - 1) / kMxRows);
    g.M = M;
    g.x = static_cast<const float *>(a.x);
    g.x_stride = x_stride;
    g.x_al16 = (reinterpret_cast<uintptr_t>(a.x) & 15) == 0 && x_stride % 4 == 0;
    g.y = a.y;
    g.y_stride = y_stride;
    if (a.type == MI355X_TYPE_IQ3_XXS) g.grid = static_cast<const uint32_t *>(ctx->iq3xxs_grid);
    if (a.type == MI355X_TYPE_IQ2_S) g.grid = static_cast<const uint32_t *>(ctx->iq2s_grid);
    if ((a.type == MI355X_TYPE_IQ3_XXS || a.type == MI355X_TYPE_IQ2_S) && !g.grid)
        return set_error(MI355X_EUNSUPPORTED, "grid table not installed for this IQ type");
    const int nu = (mx_units(a.type, g.B) + kMxWaves - 1) / kMxWaves;
    const mx_fn k = pick_mx(a.type, nu, M);
    const size_t lds = M * mx_act_bytes(a.type, g.B) + 16;
    const int occ = occupancy(reinterpret_cast<const void *>(k), kMxThreads, lds);
    int64_t wgs = std::min<int64_t>(g.tiles, static_cast<int64_t>(ctx->num_cus) * std::max(1, std::min(occ, 2)));
    if (ctx->grid_override > 0) wgs = std::min<int64_t>(wgs, ctx->grid_override);
    hipLaunchKernelGGL(k, dim3(static_cast<unsigned>(std::max<int64_t>(wgs, 1))), dim3(kMxThreads), lds, ctx->stream, g);
    MI355X_HIP(hipGetLastError());
    return MI355X_OK;
}

}  // namespace mi355x
