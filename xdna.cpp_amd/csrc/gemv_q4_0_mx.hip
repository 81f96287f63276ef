// Q4_0 GEMV for 2 to 8 activation rows on the matrix cores of gfx950, one
// launch without a workspace.
//
// Why.  The dot-unit forms spend about one VALU instruction per weight and
// activation (13.5 us of VALU per CU at 8192x8192, M = 8) and, past 2048
// values per row, a staging launch.  Here every weight is decoded once (about
// 2 VALU instructions per weight of a lane, whatever M) and one
// v_mfma_f32_16x16x32_f16 per block and 16 weight rows does all products.
//
// Arithmetic.  The 16 activation rows of an MFMA are 8 activations in two f16
// planes, hi = f16(x s) and lo = f16(x s - hi), s the power of two that puts
// the largest |x| of the wavefront's part of the row in [2^14, 2^15): x to
// 2^-22 of itself, or 2^-39 of that largest value.  Codes are exact, products
// exact in f32; a block's f32 sums are scaled by its d and added in f32.  An
// activation with a block whose largest value is more than 2^18 below that of the
// wavefront's part is wide (the fixed point of the dot-unit forms, with a scale
// per block, held such a block to 2^-18.9): after its tiles the workgroup sums wide
// activations in f32 from their values as they are.  The lanes compare the least
// that they saw of each activation while they stage it; only where that is small
// does the workgroup read the activations again to tell.  (us at 8192x8192 M = 8
// with none, one and all wide 19.8, 47, 97, without the comparison 19.3.)
//
// Work split.  A workgroup of 8 wavefronts owns tiles of 16 weight rows and
// splits K: wavefront v takes QN quads of 4 blocks.  Lane (n, g) = (lane & 15,
// lane >> 4) loads the 16 code bytes of block g of a quad and its d, of weight
// row n; a 4 x 4 exchange between the lane groups (permlane swaps) gives every
// lane dword g of all four blocks, the 8 codes of its MFMA operand.  The
// wavefront's activations stay in registers (4 per block), read from the
// caller once per workgroup: the lanes of the two planes of a row each load half
// of every block and exchange the plane that the other one needs.  A quad's
// registers are reloaded with the next tile's right after its decode, so QN
// quads per wavefront stay in flight; tile sums meet in LDS.  Rows of more than
// 8192 values go in two launches, the second adding to y.
//
// What bounds it: waiting.  At 8192x8192 M = 8 a wavefront runs 45 k cycles, of
// which its SIMD issues vector instructions for 16 k (about 85 per quad and tile
// and 85 per quad to stage the activations) and matrix ones for 2 k (rocprof).
// Every workgroup reads and converts all activations, 256 KB through each CU's L1
// there, before its two tiles, with two wavefronts per SIMD to hide it.
// us per call on MI355X, dot-unit forms -> here: M = 8 8192x8192 25.9 -> 19.8,
// 4096x4096 11.9 -> 8.3, 17408x5120 42.9 -> 20.0, 151936x2048 73.7 -> 50.
#include "internal.h"
#include "kq_device.h"
#include "q4_0_layout.h"

#include <algorithm>
#include <cstdint>

namespace mi355x {
namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kQxWaves = 8;
constexpr int kQxThreads = 64 * kQxWaves;
constexpr int kQxRows = 16;     // weight rows per tile
constexpr int kQxAct = 8;       // activations per launch
constexpr int kQxMaxQuads = 8;  // quads of blocks per wavefront and launch
constexpr float kQxBelow = 0.0625f;  // largest scaled value from which on a block's planes hold it to 2^-21

struct QxArgs {
    const uint8_t *W;
    int N;
    int row_bytes;
    int B;       // blocks per row
    int q0, q1;  // quads of this launch
    int tiles;
    int M;
    const float *x;
    int64_t x_stride;
    float *y;
    int64_t y_stride;
    int add;  // add to y
};

__device__ __forceinline__ f16x2 qx_h2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ uint32_t qx_u2(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ f16x2 qx_splat(float v) {
    return f16x2{static_cast<_Float16>(v), static_cast<_Float16>(v)};
}

// The four code bytes w of a block as the operand of values (0, 2), (1, 3) of
// their low nibbles and of their high ones; resident nibbles are q - 8 in two's
// complement, so flipping the sign bit over 1024 in f16 gives 1024 + q.
__device__ __forceinline__ f16x8 qx_operand(uint32_t w) {
    const uint32_t v = w >> 8;
    const f16x2 c0 = qx_splat(-1032.f), c1 = qx_splat(0.0625f), c2 = qx_splat(-72.f);
    const u32x4 r{qx_u2(qx_h2((w & 0x000F000Fu) ^ 0x64086408u) + c0),
                  qx_u2(qx_h2((v & 0x000F000Fu) ^ 0x64086408u) + c0),
                  qx_u2(__builtin_elementwise_fma(qx_h2((w & 0x00F000F0u) ^ 0x64806480u), c1, c2)),
                  qx_u2(__builtin_elementwise_fma(qx_h2((v & 0x00F000F0u) ^ 0x64806480u), c1, c2))};
    return __builtin_bit_cast(f16x8, r);
}

// r[e] of lane group g: v[g] of lane group e
__device__ __forceinline__ void qx_exchange(const u32x4 &v, uint32_t (&r)[4]) {
    const auto a = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    r[0] = c[0], r[1] = c[1], r[2] = d[0], r[3] = d[1];
}
// r[e] of every lane: v of lane group e
__device__ __forceinline__ void qx_spread(uint32_t v, uint32_t (&r)[4]) {
    const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], a[0], false, false);
    const auto d = __builtin_amdgcn_permlane16_swap(a[1], a[1], false, false);
    r[0] = c[0], r[1] = c[1], r[2] = d[0], r[3] = d[1];
}

// four values at any float address
__device__ __forceinline__ float4 qx_load4(const float *p) {
    float4 f;
    __builtin_memcpy(&f, p, sizeof f);
    return f;
}
// w rounded to f16, and what that leaves
__device__ __forceinline__ f16x2 qx_hi(float w0, float w1) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    return __builtin_convertvector((f32x2{w0, w1}), f16x2);
}
__device__ __forceinline__ f16x2 qx_lo(float w0, float w1, f16x2 h) {
    return f16x2{static_cast<_Float16>(w0 - static_cast<float>(h[0])),
                 static_cast<_Float16>(w1 - static_cast<float>(h[1]))};
}
// `own` in the lanes of one plane (banks of 4 lanes of a 16-lane row), the
// other plane's lanes of `other` in the rest: row_ror:8
template <int BANKS>
__device__ __forceinline__ uint32_t qx_from(f16x2 own, f16x2 other) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(__builtin_bit_cast(int, own),
                                                             __builtin_bit_cast(int, other), 0x128, 0xF, BANKS, false));
}
__device__ __forceinline__ float qx_max4(const float4 &f) {
    return fmaxf(fmaxf(fmaxf(fabsf(f.x), fabsf(f.y)), fabsf(f.z)), fabsf(f.w));
}
// over the 8 lanes of an activation: the two planes' (row_ror:8) and the lane groups
__device__ __forceinline__ float qx_row_max(float v) {
    v = fmaxf(v, dpp_mov<0x128>(v));
    v = fmaxf(v, __shfl_xor(v, 16));
    return fmaxf(v, __shfl_xor(v, 32));
}
__device__ __forceinline__ uint32_t qx_row_or(uint32_t v) {
    v |= static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x128, 0xF, 0xF, false));
    v |= __shfl_xor(v, 16);
    return v | __shfl_xor(v, 32);
}
// s = 2^(14 - E) for mx in [2^E, 2^(E+1)), E >= -110, and unit = 1 / s
constexpr float kQxUnitMin = 0x1p-124f;
__device__ __forceinline__ float qx_scale(float mx, float &unit) {
    const int ex = min(max(static_cast<int>(__builtin_bit_cast(uint32_t, mx) >> 23), 17), 254);
    unit = __builtin_bit_cast(float, static_cast<uint32_t>(ex - 14) << 23);
    return __builtin_bit_cast(float, static_cast<uint32_t>(268 - ex) << 23);
}

// A weight row of a tile: block b of it in lane group b & 3 (the lane's 16 code
// bytes and d).  The tile's rows are one buffer, empty past the last tile and
// where `in` is false (readfirstlane: left alone, the compiler computes the
// descriptor in vector registers and loops over its values).
__device__ __forceinline__ void qx_load(const QxArgs &a, int tile, bool in, uint32_t b, int col, u32x4 &q, uint32_t &d) {
    const int rows = __builtin_amdgcn_readfirstlane(tile < a.tiles && in ? min(a.N - tile * kQxRows, kQxRows) : 0);
    const int at = __builtin_amdgcn_readfirstlane(rows > 0 ? tile : 0);
    const uint8_t *base = a.W + static_cast<int64_t>(at) * (kQxRows * a.row_bytes);
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(base), 0, static_cast<uint32_t>(rows * a.row_bytes), kBufferWord3);
    const uint32_t F = static_cast<uint32_t>(a.B) >> 6;
    const uint32_t slot = b < 64 * F ? (b & 63) * F + (b >> 6) : b;  // q4_0_d_slot
    const uint32_t row = static_cast<uint32_t>(col) * static_cast<uint32_t>(a.row_bytes);
    q = __builtin_amdgcn_raw_buffer_load_b128(rsrc, static_cast<int>(row + 16 * b), 0, kNonTemporal);
    d = __builtin_amdgcn_raw_buffer_load_b16(rsrc, static_cast<int>(row + 16 * static_cast<uint32_t>(a.B) + 2 * slot), 0, 0);
}

// The activations (bits) of which quads [qw, qw + n), n <= 8, hold a block that
// the planes lose, `unit` the lane's activation's: read again, as this is seldom
// asked (parts with such blocks, or with zeros).
__device__ __forceinline__ uint32_t qx_lost(const QxArgs &a, int qw, int n, int lane, float unit) {
    const int m = lane & 7, g = lane >> 4, plane = (lane >> 3) & 1;
    const float *x = a.x + min(m, a.M - 1) * a.x_stride + 4 * g + 16 * plane;
    // the smallest scale takes what it has
    const float below = unit > kQxUnitMin ? kQxBelow * unit : 0.f;
    // bits of the lane's quarters that are large enough, and that are not 0
    uint32_t near = 0, some = 0;
#pragma unroll 16
    for (int k = 0; k < 4 * n; ++k) {
        const float q = qx_max4(qx_load4(x + 32 * static_cast<int64_t>(min(4 * qw + k, 4 * a.q1 - 1))));
        near |= static_cast<uint32_t>(q >= below) << k;
        some |= static_cast<uint32_t>(q > 0.f) << k;
    }
    return static_cast<uint32_t>(__ballot((qx_row_or(some) & ~qx_row_or(near)) != 0)) & 0xFF;
}

// The activations of `wide` over the whole row so far, quads [0, q1), in f32:
// each lane its block of its weight row.  red: 8 wavefronts x 8 activations x 16
// rows.  Called by the whole workgroup with the same `wide`; replaces what the
// tiles stored (and what the launch before did).
__device__ __forceinline__ void qx_wide(const QxArgs &a, uint32_t wide, int wave, int lane, float (*red)[kQxAct][kQxRows]) {
    const int col = lane & 15, g = lane >> 4;
    for (int tile = blockIdx.x; tile < a.tiles; tile += static_cast<int>(gridDim.x)) {
        float acc[kQxAct] = {};
#pragma clang loop unroll(disable)
        for (int qd = wave; qd < a.q1; qd += kQxWaves) {
            const uint32_t b = 4u * static_cast<uint32_t>(qd) + g;
            u32x4 q;
            uint32_t dh;
            qx_load(a, tile, true, b, col, q, dh);
            float w[32];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const f16x8 o = qx_operand(q[k]);  // values 0, 2, 1, 3 of the low nibbles, then of the high ones
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    w[16 * t + 4 * k] = static_cast<float>(o[4 * t]);
                    w[16 * t + 4 * k + 2] = static_cast<float>(o[4 * t + 1]);
                    w[16 * t + 4 * k + 1] = static_cast<float>(o[4 * t + 2]);
                    w[16 * t + 4 * k + 3] = static_cast<float>(o[4 * t + 3]);
                }
            }
            const float d = half_f(dh);
#pragma unroll
            for (int m = 0; m < kQxAct; ++m) {
                if (!(wide >> m & 1)) continue;
                const float *x = a.x + m * a.x_stride + 32 * static_cast<int64_t>(b);
                float s = 0.f;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const float4 v = qx_load4(x + 4 * k);
                    s += fmaf(w[4 * k], v.x, w[4 * k + 1] * v.y) + fmaf(w[4 * k + 2], v.z, w[4 * k + 3] * v.w);
                }
                acc[m] = fmaf(d, s, acc[m]);
            }
        }
        __syncthreads();  // the last readers of red
#pragma unroll
        for (int m = 0; m < kQxAct; ++m) {
            float v = acc[m];
            v += __shfl_xor(v, 16);
            v += __shfl_xor(v, 32);
            if (g == 0) red[wave][m][col] = v;
        }
        __syncthreads();
        const int m = 2 * (wave & 3) + (lane >> 5), r = lane & 31;
        if (wave < 4 && r < kQxRows && (wide >> m & 1) && tile * kQxRows + r < a.N) {
            float v = 0.f;
#pragma unroll
            for (int k = 0; k < kQxWaves; ++k) v += red[k][m][r];
            a.y[m * a.y_stride + tile * kQxRows + r] = v;
        }
    }
}

template <int QN>
__global__ __launch_bounds__(kQxThreads) void gemv_q4_0_mx_kernel(QxArgs a) {
    __shared__ f32x4 part[2][kQxWaves][64];
    __shared__ f32x4 unit[kQxWaves][kQxAct / 4];
    __shared__ uint32_t flags[kQxWaves];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int col = lane & 15, g = lane >> 4;
    const int m = col & 7, plane = col >> 3;
    const int qw = a.q0 + wave * QN;  // first quad of the wavefront

    // 1. its activations: of every block, values 16 plane + 4 g + (0..3), so that
    // the lanes of a row read whole cache lines
    // (rows past M and quads past the launch's repeat the last: their products
    // are not stored, or are with zero weights)
    float4 f[QN][4];
    const float *xr = a.x + min(m, a.M - 1) * a.x_stride + 4 * g + 16 * plane;
#pragma unroll
    for (int i = 0; i < QN; ++i) {
        const float *p = xr + 128 * static_cast<int64_t>(min(qw + i, a.q1 - 1));
#pragma unroll
        for (int e = 0; e < 4; ++e) f[i][e] = qx_load4(p + 32 * e);
    }

    // 2. the first tile's weights
    u32x4 wq[QN];
    uint32_t wd[QN];
    auto load = [&](int i, int tile) {
        qx_load(a, tile, qw + i < a.q1, 4u * static_cast<uint32_t>(qw + i) + g, col, wq[i], wd[i]);
    };
    int tile = blockIdx.x;
#pragma unroll
    for (int i = 0; i < QN; ++i) load(i, tile);
    __builtin_amdgcn_sched_barrier(0);

    // 3. the activations' operands
    // the largest value, and the smallest of the lane's quarters of blocks that is
    // not 0 (its bits less 1, so that 0 is none)
    float mxe[2] = {0.f, 0.f};
    uint32_t mn = ~0u;
#pragma unroll
    for (int i = 0; i < QN; ++i)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float q0 = qx_max4(f[i][2 * e]), q1 = qx_max4(f[i][2 * e + 1]);
            mxe[e] = fmaxf(fmaxf(mxe[e], q0), q1);
            mn = min(min(mn, __builtin_bit_cast(uint32_t, q0) - 1u), __builtin_bit_cast(uint32_t, q1) - 1u);
        }
    const float mx = qx_row_max(fmaxf(mxe[0], mxe[1]));
    float un;
    const float s = qx_scale(mx, un);
    if (lane < kQxAct) reinterpret_cast<float *>(unit[wave])[lane] = un;
    // where each quarter is 0 or large enough, each block is
    const bool suspect = !__all(mn + 1u >= __builtin_bit_cast(uint32_t, kQxBelow * un) || mn == ~0u);
    if (lane == 0) flags[wave] = suspect;
    f16x8 x[QN][4];
#pragma unroll
    for (int i = 0; i < QN; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float4 &v = f[i][e];
            const float w[4] = {v.x * s, v.y * s, v.z * s, v.w * s};
            const f16x2 h0 = qx_hi(w[0], w[2]), h1 = qx_hi(w[1], w[3]);
            const f16x2 l0 = qx_lo(w[0], w[2], h0), l1 = qx_lo(w[1], w[3], h1);
            // values 4 g + (0..3) from the lane of plane 0, 16 + 4 g + (0..3) from plane 1's
            const u32x4 o{qx_from<0xC>(h0, l0), qx_from<0xC>(h1, l1), qx_from<0x3>(l0, h0), qx_from<0x3>(l1, h1)};
            x[i][e] = __builtin_bit_cast(f16x8, o);
        }
    }
    // result row 4 g + k of this wavefront is activation (4 g + k) & 7
    const f32x4 u = unit[wave][g & 1];

    // 4. tiles
    for (int par = 0; tile < a.tiles; par ^= 1) {
        const int next = tile + static_cast<int>(gridDim.x);
        f32x4 acc{};
#pragma unroll
        for (int i = 0; i < QN; ++i) {
            uint32_t q[4], d[4];
            qx_exchange(wq[i], q);
            qx_spread(__builtin_bit_cast(uint32_t, half_f(wd[i])), d);
            load(i, next);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const f32x4 v = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[i][e], qx_operand(q[e]), f32x4{}, 0, 0, 0);
                const float de = __builtin_bit_cast(float, d[e]);
#pragma unroll
                for (int k = 0; k < 4; ++k) acc[k] = fmaf(de, v[k], acc[k]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        part[par][wave][lane] = f32x4{acc[0] * u[0], acc[1] * u[1], acc[2] * u[2], acc[3] * u[3]};
        __syncthreads();  // also keeps this half of part from its next writers until it is read
        // output o = (activation, row) by the four lanes of a quad, two wavefronts' sums each
        const int o = threadIdx.x >> 2, w = 2 * (threadIdx.x & 3);
        const int om = o >> 4, on = o & 15;
        float sum = 0.f;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const float *p = reinterpret_cast<const float *>(&part[par][w + k][16 * (om >> 2) + on]) + (om & 3);
            sum += p[0] + p[4 * 32];  // hi and lo planes
        }
        sum += quad_x1_f(sum);
        sum += quad_x2_f(sum);
        const int n = tile * kQxRows + on;
        if (w == 0 && om < a.M && n < a.N) {
            float *y = a.y + om * a.y_stride + n;
            *y = a.add ? *y + sum : sum;
        }
        tile = next;
    }
    // 5. wide activations (a workgroup has a tile, so a barrier has passed)
    int l = threadIdx.x & 63;
    asm volatile("" : "+v"(l));  // nothing stays in registers for this over the tiles
    if (__builtin_expect(__any(flags[l & (kQxWaves - 1)] != 0), 0)) {
        __syncthreads();  // every wavefront has read its flags
        const uint32_t lost = qx_lost(a, qw, QN, l, reinterpret_cast<const float *>(unit[wave])[l & 7]);
        if (l == 0) flags[wave] = lost;
        __syncthreads();
        uint32_t wide = 0;
#pragma unroll
        for (int k = 0; k < kQxWaves; ++k) wide |= flags[k];
        wide = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(wide))) & ((1u << a.M) - 1);
        if (wide) qx_wide(a, wide, wave, l, reinterpret_cast<float(*)[kQxAct][kQxRows]>(part));
    }
}

typedef void (*qx_fn)(QxArgs);
qx_fn pick_qx(int qn) {
    switch (qn) {
    case 1: return gemv_q4_0_mx_kernel<1>;
    case 2: return gemv_q4_0_mx_kernel<2>;
    case 3: return gemv_q4_0_mx_kernel<3>;
    case 4: return gemv_q4_0_mx_kernel<4>;
    case 5: return gemv_q4_0_mx_kernel<5>;
    case 6: return gemv_q4_0_mx_kernel<6>;
    case 7: return gemv_q4_0_mx_kernel<7>;
    default: return gemv_q4_0_mx_kernel<8>;
    }
}

}  // namespace

// Where this form is faster than the dot-unit ones (us, those first).  From 5
// activations, which cost those as much as 8: rows of up to 4096 values (M = 8
// 256x512 8.0 / 4.6, 1024x4096 9.3 / 8.2), longer ones where enough tiles share
// the staging (M = 8 4096x8192 17.3 / 15.1, 17408x14336 82 / 66; but 1024x8192
// 9.7 / 15.6, 4096x14336 25.5 / 29.9).  Up to 4: where those need a staging
// launch (the pipelined batched form does not: M = 2 4096x4096 5.2 / 7.1) and
// rows are short (M = 4 1024x2560 7.4 / 5.7, M = 2 4096x5120 10.3 / 7.7, M = 4
// 4096x6144 13.3 / 9.8; but M = 2 4096x7168 9.8 / 11.2, M = 4 1024x5120 7.3 /
// 8.8).  Only in the AUTO variant: MI355X_VARIANT_DIGITS promises the fixed-point
// arithmetic of the dot-unit forms.
bool q4_0_mx_takes(const mi355x_ctx *ctx, const GemvArgs &a, int64_t M) {
    if (ctx->kernel_variant != MI355X_VARIANT_AUTO || !form_is_auto(ctx, a.type)) return false;
    if (M >= 5) return a.K <= 4096 || a.N >= (a.K <= 8192 ? 4096 : 16384);
    const bool pipelined = a.K % 2048 == 0 && (a.K <= 4096 || M == 2);
    return !pipelined && (a.K <= 4096 || (a.N >= 4096 && a.K <= (M == 2 ? 5120 : 6144)));
}

// Rows of whole quads, 16-byte aligned (q4_0_mb_capacity() takes no others).
int launch_gemv_q4_0_mx(mi355x_ctx *ctx, const GemvArgs &a, int64_t x_stride, int64_t y_stride, int M) {
    QxArgs q{};
    q.W = a.W;
    q.N = static_cast<int>(a.N);
    q.B = static_cast<int>(a.K / 32);
    q.row_bytes = q.B * 18;
    q.tiles = static_cast<int>((a.N + kQxRows - 1) / kQxRows);
    q.M = M;
    q.x = static_cast<const float *>(a.x);
    q.x_stride = x_stride;
    q.y = a.y;
    q.y_stride = y_stride;
    const int quads = q.B / 4;
    const int launches = (quads + kQxWaves * kQxMaxQuads - 1) / (kQxWaves * kQxMaxQuads);
    const int per = (quads + launches - 1) / launches;
    for (q.q0 = 0; q.q0 < quads; q.q0 += per, q.add = 1) {
        q.q1 = std::min(q.q0 + per, quads);
        const int qn = (q.q1 - q.q0 + kQxWaves - 1) / kQxWaves;
        const qx_fn k = pick_qx(qn);
        // one workgroup per CU where staging is long (14336x4096 M = 2: 12.5
        // us, with two 14.5), two where the loads of one are too few
        const int occ = occupancy(reinterpret_cast<const void *>(k), kQxThreads, 0);
        int64_t wgs = std::min<int64_t>(q.tiles, static_cast<int64_t>(ctx->num_cus) * std::max(1, std::min(occ, qn < 3 ? 2 : 1)));
        if (ctx->grid_override > 0) wgs = std::min<int64_t>(wgs, ctx->grid_override);
        hipLaunchKernelGGL(k, dim3(static_cast<unsigned>(wgs)), dim3(kQxThreads), 0, ctx->stream, q);
        MI355X_HIP(hipGetLastError());
    }
    return MI355X_OK;
}

}  // namespace mi355x
