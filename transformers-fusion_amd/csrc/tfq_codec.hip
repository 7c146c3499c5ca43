// Block codec on the device: bit-exact decode of every supported wire format
// (per-weight arithmetic in tfq_decode.hpp), the closed-form encoders, the wire ->
// Tiled16 layout conversion and the decode from that layout, the iterative encoders.  Decode: a wavefront takes
// four blocks, a lane four weights of each.  The closed-form encoders of the benchmark formats are laid out the same
// way, the others have a workgroup per block; the iterative ones give a scale group (or a run of weights with one
// scale) to a lane or a small team of lanes.  Decode and the closed forms are bound by the fp32 side (4 B per
// weight), the iterative encoders by vector instructions.

#include "tfq_decode.hpp"
#include "tfq_encode_short.hpp"

#include <cmath>

namespace tfq {

namespace {

template <int FMT>
__global__ __launch_bounds__(256) void decode_kernel(const uint8_t* __restrict__ src,
                                                     float* __restrict__ out) {
    constexpr Spec sp = spec_of(FMT);
    const int64_t blk = blockIdx.x;
    out[blk * 256 + threadIdx.x] = decode_weight<FMT>(src + blk * (int64_t)sp.block_bytes, threadIdx.x);
}

// A wavefront per block, four weights per lane from aligned dword reads, kDecodeBlocks consecutive blocks per
// wavefront so that the loads of several are in flight together; the output is not read back by this launch, so its
// stores carry the non-temporal hint.  Bound by the 4 bytes written per weight.
// 58.7 M weights: Q_G_4 200 -> 39.6 us, SB256A3 233 -> 39.8 us, Q_G_8 204 -> 49.4 us, B32S4 164 -> 39.3 us (6.8 TB/s read
// and written) against a lane per weight with byte loads; Q_4 95 -> 42 us against one block per wavefront.
// The short last block of a tensor rides in one more workgroup of the same launch.
constexpr int kDecodeBlocks = 4;
template <int FMT>
__global__ __launch_bounds__(256) void decode_quad_kernel(const uint8_t* __restrict__ src, float* __restrict__ out,
                                                          int64_t nblocks, BlockLayout tail) {
    constexpr Spec sp = spec_of(FMT);
    if (tail.n > 0 && blockIdx.x == gridDim.x - 1) {  // the short last block, a lane per weight
        if ((int)threadIdx.x < tail.n) out[nblocks * 256 + threadIdx.x] = decode_weight_short(tail, src + nblocks * (int64_t)sp.block_bytes, threadIdx.x);
        return;
    }
    typedef float f32x4_t __attribute__((ext_vector_type(4)));
    const int64_t first = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * kDecodeBlocks;
    const uint32_t lane = threadIdx.x & 63;
    const uint8_t* limit = src + nblocks * (int64_t)sp.block_bytes;
#pragma unroll
    for (int u = 0; u < kDecodeBlocks; ++u) {
        const int64_t blk = first + u;
        if (blk >= nblocks) return;
        float v[4];
        decode_quad<FMT>(src + blk * (int64_t)sp.block_bytes, lane, v, limit);
        __builtin_nontemporal_store(f32x4_t{v[0], v[1], v[2], v[3]}, reinterpret_cast<f32x4_t*>(out + blk * 256 + 4 * lane));
    }
}

__global__ __launch_bounds__(256) void decode_short_kernel(BlockLayout L, const uint8_t* __restrict__ src,
                                                           float* __restrict__ out) {
    if ((int)threadIdx.x < L.n) out[threadIdx.x] = decode_weight_short(L, src, threadIdx.x);
}

// Literal symmetric block-32 formats, closed form per 32 weights:
//   d = binary16(absmax / qmax), q = clamp(round_half_away(w / d), lo, qmax),
//   qmax = 7, lo = -8 (4-bit) or qmax = 127, lo = -127 (8-bit); d == 0 or not
//   finite gives q = 0.  (The reference holds this quantizer only as comparator
//   code: src/adapters/tools/bench_ollama_comparison.cpp:61-75, 121-134.)
// Four weights per lane, a wavefront per block, kEncodeBlocks blocks in a row; a group of 32 is eight lanes.  Bound by
// the reads (4 bytes per weight).  The tensor's short last block (tail_n weights, whole groups) is one more block with
// fewer lanes.  58.7 M weights of B32S4: 168 us with a lane per weight and byte stores, 67 us.
constexpr int kEncodeBlocks = 2;
template <int FMT>
__global__ __launch_bounds__(256) void encode_sym32_kernel(const float* __restrict__ w, uint8_t* __restrict__ dst, int64_t nblocks, int tail_n) {
    constexpr Spec sp = spec_of(FMT);
    constexpr float qmax = sp.bits == 4 ? 7.0f : 127.0f;
    constexpr int lo = sp.bits == 4 ? -8 : -127, hi = sp.bits == 4 ? 7 : 127;
    const uint32_t lane = threadIdx.x & 63;
    const int64_t first = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * kEncodeBlocks;
    float4 v[kEncodeBlocks];
#pragma unroll
    for (int k = 0; k < kEncodeBlocks; ++k) {
        const int64_t blk = first + k;
        v[k] = float4{0.0f, 0.0f, 0.0f, 0.0f};
        if (blk < nblocks || (blk == nblocks && 4 * (int)lane < tail_n)) __builtin_memcpy(&v[k], w + blk * 256 + 4 * lane, 16);  // (aligned to a float only)
    }
#pragma unroll
    for (int k = 0; k < kEncodeBlocks; ++k) {
        const int64_t blk = first + k;
        const float x[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
        float amax = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
#pragma unroll
        for (int m = 4; m >= 1; m >>= 1) amax = fmaxf(amax, __shfl_xor(amax, m, 64));
        const uint32_t h = float_to_half_bits(amax / qmax);
        const float d = half_bits_to_float(h);
        uint32_t packed = sp.bits == 4 ? 0x8888u : 0u;
        if (d > 0.0f && (h & 0x7C00u) != 0x7C00u) {
            packed = 0;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float r = roundf(x[t] / d);
                const int q = r <= (float)lo ? lo : r >= (float)hi ? hi : (int)r;
                packed |= sp.bits == 4 ? (uint32_t)(q + 8) << (4 * t) : (uint32_t)(uint8_t)(int8_t)q << (8 * t);
            }
        }
        const int n = blk < nblocks ? 256 : blk == nblocks ? tail_n : 0;
        if (4 * (int)lane < n) {
            uint8_t* p = dst + blk * (int64_t)sp.block_bytes;
            __builtin_memcpy(p + lane * (sp.bits / 2), &packed, sp.bits / 2);
            if ((lane & 7u) == 0) __builtin_memcpy(p + n * sp.bits / 8 + 2 * (lane >> 3), &h, 2);
        }
    }
}

template <int FMT>
static void launch_encode_sym32(const float* w, int64_t nblocks, uint8_t* dst, int tail_n, hipStream_t s) {
    const int64_t grid = (nblocks + (tail_n > 0) + 4 * kEncodeBlocks - 1) / (4 * kEncodeBlocks);
    hipLaunchKernelGGL(encode_sym32_kernel<FMT>, dim3((unsigned)grid), dim3(256), 0, s, w, dst, nblocks, tail_n);
}

__global__ __launch_bounds__(256) void encode_raw32_kernel(const float* __restrict__ w,
                                                           uint8_t* __restrict__ dst) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    reinterpret_cast<float*>(dst)[e] = w[e];
}

// Closed-form encoders of the 16- and 24-bit formats (quant_q16_enhanced / quant_q24,
// src/codec/block_codec.cpp:1690-1757, :1809-1820) and of the residual means the grouped ids append
// (:2450-2493): per 32 weights the binary16 of mean(w - decoded), summed in double in index order.
// One workgroup per block: lane i owns weight i, then output byte pairs, then (8 lanes) a group.
template <int FMT>
__global__ __launch_bounds__(256) void encode_wide_kernel(const float* __restrict__ w, uint8_t* __restrict__ dst) {
    constexpr Spec sp = spec_of(FMT);
    constexpr int plain = 256 * sp.bits / 8;
    __shared__ uint32_t code[256];
    __shared__ float dec[256];
    __shared__ float red[8];
    const int64_t blk = blockIdx.x;
    const uint32_t i = threadIdx.x;
    uint8_t* p = dst + blk * (int64_t)sp.block_bytes;
    const float x = w[blk * 256 + i];
    if constexpr (sp.bits == 24) {
        const uint32_t u = __float_as_uint(x);
        p[3 * i] = (uint8_t)(u >> 8);
        p[3 * i + 1] = (uint8_t)(u >> 16);
        p[3 * i + 2] = (uint8_t)(u >> 24);
        dec[i] = __uint_as_float(u & 0xFFFFFF00u);
    } else {
        // min and max are order independent; the encoder starts them at +-1e30
        float lo = fminf(1e30f, x), hi = fmaxf(-1e30f, x);
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) { lo = fminf(lo, __shfl_xor(lo, m, 64)); hi = fmaxf(hi, __shfl_xor(hi, m, 64)); }
        if ((i & 63u) == 0) { red[i >> 6] = lo; red[4 + (i >> 6)] = hi; }
        __syncthreads();
        lo = fminf(fminf(red[0], red[1]), fminf(red[2], red[3]));
        hi = fmaxf(fmaxf(red[4], red[5]), fmaxf(red[6], red[7]));
        if (lo > hi) { lo = 0.0f; hi = 0.0f; }
        const float range = hi - lo;
        const bool narrow = (i & 3u) == 3u;
        const float top = narrow ? 32767.0f : 65535.0f;
        const float scale = range > 0 ? top / range : 0.0f;
        long q = lroundf((x - lo) * scale);
        q = q < 0 ? 0 : q > (long)top ? (long)top : q;
        code[i] = (uint32_t)q;
        const float dscale = range > 0 ? range / top : 0.0f;
        dec[i] = __builtin_fmaf((float)(uint32_t)q, dscale, lo);
        __syncthreads();
        // output bytes 2 i and 2 i + 1: bits 16 i .. 16 i + 15 of [min][max][64 groups of 63 bits]
        uint32_t out16 = 0;
#pragma unroll
        for (uint32_t b = 0; b < 16; ++b) {
            const uint32_t pos = 16 * i + b;
            uint32_t bit;
            if (pos < 32) bit = (__float_as_uint(lo) >> pos) & 1u;
            else if (pos < 64) bit = (__float_as_uint(hi) >> (pos - 32)) & 1u;
            else {
                const uint32_t g = (pos - 64) / 63, r = (pos - 64) - 63 * g;
                const uint32_t k = r < 48 ? r >> 4 : 3;
                bit = g < 64 ? (code[4 * g + k] >> (r - 16 * k)) & 1u : 0u;
            }
            out16 |= bit << b;
        }
        p[2 * i] = (uint8_t)(out16 & 0xFF);
        p[2 * i + 1] = (uint8_t)(out16 >> 8);
    }
    if constexpr (sp.block_bytes > plain) {
        __syncthreads();
        if (i < 8) {
            uint32_t h = 0;
            if constexpr (sp.scb == 1) {
                double mean = 0.0;
                for (int j = 0; j < 32; ++j) mean += (double)w[blk * 256 + 32 * i + j] - (double)dec[32 * i + j];
                mean /= 32.0;
                h = float_to_half_bits((float)mean);
            }
            p[plain + 2 * i] = (uint8_t)(h & 0xFF);  // ids without residuals pad with zeros
            p[plain + 2 * i + 1] = (uint8_t)(h >> 8);
        }
    }
}

// Sign formats (src/codec/block_codec.cpp:2434-2449, :2523-2549): binary16 scale, then the sign bits of
// the weights that are not slots.  tier < 0: Q_1, scale = sqrt(mean w^2) (rms_scale, :213-218); otherwise
// the mean |w| of the kept weights snapped to binary16 and the best of the 2 * radius neighbouring
// binary16 values by squared error (q1_fit_scale_fp16, :270-299), radius 4, 10 or 24.  Every sum runs
// in double in index order; lane c evaluates candidate c, lane 0 picks the first strict minimum in the
// reference's order (centre, then -radius .. +radius).
__global__ __launch_bounds__(256) void encode_q1_kernel(const float* __restrict__ w, uint8_t* __restrict__ dst, int tier) {
    __shared__ float x[256];
    __shared__ double err[64];
    __shared__ uint32_t scale_bits;
    const int64_t blk = blockIdx.x;
    const uint32_t i = threadIdx.x;
    x[i] = w[blk * 256 + i];
    __syncthreads();
    if (tier < 0) {
        if (i == 0) {
            double sum = 0.0;
            for (int j = 0; j < 256; ++j) sum += (double)x[j] * (double)x[j];
            scale_bits = float_to_half_bits((float)sqrt(sum / 256.0));
        }
    } else {
        const int rad = tier == 0 ? 4 : tier == 1 ? 10 : 24;
        __shared__ uint32_t h0s;
        if (i == 0) {
            double sum_abs = 0.0;
            for (int j = 0; j < 256; ++j)
                if ((j & 15) != 15) sum_abs += fabs((double)x[j]);
            h0s = float_to_half_bits((float)(sum_abs / 240.0));
        }
        __syncthreads();
        const int h0 = (int)h0s;
        // candidate c: 0 = h0, 1 .. rad = h0 - rad .. h0 - 1, rad + 1 .. 2 rad = h0 + 1 .. h0 + rad
        if ((int)i <= 2 * rad) {
            const int delta = i == 0 ? 0 : (int)i <= rad ? (int)i - rad - 1 : (int)i - rad;
            const int hc = h0 + delta;
            double e = -1.0;  // out of range: skipped
            if (hc >= 0 && hc <= 0xFFFF) {
                const float sc = half_bits_to_float((uint32_t)hc);
                e = 0.0;
                for (int j = 0; j < 256; ++j) {
                    if ((j & 15) == 15) continue;
                    const double v = x[j] >= 0 ? (double)sc : -(double)sc;
                    const double d = (double)x[j] - v;
                    e = __builtin_fma(d, d, e);  // fused in the reference's Release build
                }
            }
            err[i] = e;
        }
        __syncthreads();
        if (i == 0) {
            int best = h0;
            double best_e = err[0];
            for (int c = 1; c <= 2 * rad; ++c) {
                const int delta = c <= rad ? c - rad - 1 : c - rad;
                if (err[c] >= 0.0 && err[c] < best_e) { best_e = err[c]; best = h0 + delta; }
            }
            scale_bits = (uint32_t)best;  // a binary16 pattern converts back to itself
        }
    }
    __syncthreads();
    uint8_t* p = dst + blk * 32;
    if (i < 32) {
        uint32_t byte = 0;
#pragma unroll
        for (uint32_t b = 0; b < 8; ++b) {
            const uint32_t pos = 8 * i + b;
            uint32_t bit;
            if (pos < 16) bit = (scale_bits >> pos) & 1u;
            else {
                const uint32_t j = pos - 16;        // kept index -> weight index (15 kept weights per 16)
                bit = x[j + j / 15] >= 0.0f ? 1u : 0u;
            }
            byte |= bit << b;
        }
        p[i] = (uint8_t)byte;
    }
}

// Affine family encoder: quant_affine with grp16_fit_affine (src/codec/block_codec.cpp:1337-1521) for
// Q_G_4 / Q_G_3 / Q_G_2, the superblock formats and Q_1_5.  A lane owns a group and keeps its 32 or 16 weights in
// registers, so a wavefront encodes eight or four blocks: the per-group Lloyd fit (4 x assign + least-squares refit,
// +-15 % scale polish, closing refit) and the per-group part of the 5 joint refinements run in the lane, in the
// reference's order, with double sums; the sums over the groups of a block are read from LDS by all of its lanes.
// Multiply-adds are fused exactly where the reference's Release build (GCC, -ffp-contract=fast) fuses them and
// nowhere else.
// Bound by vector instructions: 17 passes over the weights.  What a pass needs of a weight is its level, lround(clamp((x - m)
// / s) * top) in fp32 (the correctly rounded division alone is ten instructions), and from ten passes the sums over level,
// level squared and weight times level, in double, that s and m are solved from.  Neither is formed as the reference forms
// it: levels come from one multiply-add by top / s with a bound on their distance from the reference's value (group_levels),
// s and m from integer dot products of levels and weights, four to an instruction, with a bound on what the reference's
// roundings can make of them (quick_solve).  A pass takes 3.3 instructions for a weight's level and 1.5 for the sums, where the
// double sums took six.  Where a bound reaches a rounding boundary (a level, a code, a binary16 d or dm) the step is taken
// again: with the reference's own division for the weights in question, or with s and m from its own double sums over the
// last levels, which are kept for that.  So every payload is the reference's.  58.7 M weights of Q_G_4: a third of the
// wavefronts meet the latter in the fit, three quarters once in their five refinements; a build that never does takes 25 us
// less.  The polish compares six errors that are formed in fp32 first.
// 58.7 M weights of Q_G_4: 7.46 ms with one block per wavefront and the division, 268 to 290 us with all sums in double,
// 236 now; Q_G_3 269 -> 233, Q_G_2 344 -> 305, SB256A3 351 -> 301, SB256A2 351 -> 307; smaller calls by
// encode_affine_summed_kernel.  Four wavefronts a SIMD: three have 17 % less of its issue.
__device__ __forceinline__ uint32_t unit_nearest_dev(float value, int bits) {
    const float v = fmaxf(0.0f, fminf(1.0f, value));
    const float top = bits == 1 ? 1.0f : bits == 4 ? 15.0f : bits == 3 ? 7.0f : bits == 6 ? 63.0f : bits == 8 ? 255.0f : 3.0f;
    return (uint32_t)lroundf(v * top);
}
__device__ __forceinline__ double fms2(double a, double b, double c, double d) {  // a b - c d, first product fused
    return __builtin_fma(a, b, -(c * d));
}

// Levels of a lane's group for offset m and scale s, a byte each.  False where some weight may have another level than the
// reference gives it: it lies closer to a rounding boundary than the bound, or the group is `odd` (a NaN, an infinity or a
// magnitude the bound does not cover).  `off_by` is how far s and m together may be from the reference's.
// With u = 2^-24 and T = top (x - m) / s, which matters up to `top`: the reference's three roundings put its value within
// 3 u T, here the reciprocal (1 ulp), m / s and the multiply-adds within 3 u T + u top |m / s|.  T is formed in units of 2^-16
// on top of 2^23 + 2^15 + a, so that the third byte of the float is the level and its lower half how far T is above the
// boundary below; a unit number a above the bound shifts that to where one comparison finds both sides of a boundary.
constexpr float kRound = 12582912.0f;           // 1.5 * 2^23
constexpr float kUlp = 5.9604644775390625e-8f;  // 2^-24
template <int BITS>
struct NearLevel {
    static constexpr float top = (float)((1 << BITS) - 1);
    float r, mr, magic;
    uint32_t least;  // (the lower half of a weight whose level is certain is no less)
    bool usable;
    __device__ __forceinline__ NearLevel(float m, float s, float off_by) : r(__builtin_amdgcn_rcpf(s)), mr(m * r) {
        const float bound = 65536.0f * (kUlp * (6.0f * (top + 1.0f) + 4.0f + 1.01f * top * fabsf(mr)) + 1.02f * top * off_by * fabsf(r));
        const float a = floorf(bound + 1.51f);  // (half a unit for the rounding to units)
        usable = a <= 16384.0f && fabsf(r) >= 1e-36f;  // (a NaN, as from s = 0, is not; a denormal reciprocal lost bits)
        magic = 8421376.0f + a;
        least = 2 * (uint32_t)a;
    }
    __device__ __forceinline__ uint32_t operator()(float v) const {
        const float t = __builtin_amdgcn_fmed3f(__builtin_fmaf(v, r, -mr), 0.0f, 1.0f);
        return __float_as_uint(__builtin_fmaf(t, top * 65536.0f, magic));
    }
};
__device__ __forceinline__ uint32_t third_bytes(const uint32_t (&w)[4]) {
    return __builtin_amdgcn_perm(__builtin_amdgcn_perm(w[3], w[2], 0x0C0C0602u), __builtin_amdgcn_perm(w[1], w[0], 0x0C0C0602u), 0x05040100u);
}
template <int BITS, int GSZ>
__device__ __forceinline__ bool group_levels(const float (&x)[GSZ], float m, float s, float off_by, bool odd, uint32_t (&p)[GSZ / 4]) {
    const NearLevel<BITS> near(m, s, off_by);
    uint32_t low = 0xFFFFu;
#pragma unroll
    for (int i = 0; i < GSZ; i += 4) {
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = near(x[i + j]);
        asm("v_min3_u16 %0, %0, %1, %2" : "+v"(low) : "v"(w[0]), "v"(w[1]));  // (of the lower halves; the compiler packs pairs first)
        asm("v_min3_u16 %0, %0, %1, %2" : "+v"(low) : "v"(w[2]), "v"(w[3]));
        p[i / 4] = third_bytes(w);
    }
    return !odd && (low & 0xFFFFu) >= near.least && near.usable;
}
// The reference's own levels: the division is left to the weights in question, four at a time, which are read again from
// `from` (a rare path of little code: unrolled over the group it filled a third of the instruction cache).
template <int BITS, int GSZ>
__device__ __forceinline__ void group_levels_divided(const float (&x)[GSZ], const float* from, float m, float s, bool odd, uint32_t (&p)[GSZ / 4]) {
    asm volatile("" : "+v"(m), "+v"(s));  // (or what the usual path has of the weights would be kept in registers for this one)
    const NearLevel<BITS> near(m, s, 0.0f);
    const uint32_t least = odd || !near.usable ? 0x10000u : near.least;
    uint32_t open = 0;  // the fours with a weight in question
#pragma unroll
    for (int i = 0; i < GSZ; i += 4) {
        uint32_t w[4], low = 0xFFFFu;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = near(x[i + j]);
        asm("v_min3_u16 %0, %0, %1, %2" : "+v"(low) : "v"(w[0]), "v"(w[1]));
        asm("v_min3_u16 %0, %0, %1, %2" : "+v"(low) : "v"(w[2]), "v"(w[3]));
        p[i / 4] = third_bytes(w);
        open |= (low & 0xFFFFu) < least ? 1u << (i / 4) : 0u;
    }
#pragma unroll 1
    while (open) {
        const int at = __builtin_ctz(open);
        open &= open - 1;
        float v[4];
        __builtin_memcpy(v, from + 4 * at, 16);
        uint32_t four = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t w = near(v[j]);
            four |= ((w & 0xFFFFu) < least ? unit_nearest_dev((v[j] - m) / s, BITS) : w >> 16 & 0x7Fu) << (8 * j);
        }
#pragma unroll
        for (int i = 0; i < GSZ / 4; ++i) p[i] = at == i ? four : p[i];
    }
}
// The roundings of a level n * unit and of its square, relative and in units of 2^-24: the former lie within `level` of
// each other, `ideal` being the unit in their middle, the latter within `square` of the exact square.
struct LevelRounding {
    double level, square, ideal;
};
constexpr LevelRounding level_rounding(int bits) {
    const float unit = bits == 1 ? 1.0f : 1.0f / (float)((1 << bits) - 1);
    double lo = 0, hi = 0, sq = 0;
    for (int n = 1; n < 1 << bits; ++n) {
        const float l = (float)n * unit, l2 = l * l;
        const double e = ((double)l / ((double)n * (double)unit) - 1.0) * 16777216.0, f = ((double)l2 / ((double)l * (double)l) - 1.0) * 16777216.0;
        if (e < lo) lo = e;
        if (e > hi) hi = e;
        if (f > sq) sq = f;
        if (-f > sq) sq = -f;
    }
    return {(hi - lo) / 2, sq, (double)unit * (1.0 + (hi + lo) / 2 / 16777216.0)};
}
__device__ __forceinline__ int byte_dot(uint32_t levels, uint32_t plane, int sum, bool is_signed) {
    return is_signed ? __builtin_amdgcn_sdot4((int)levels, (int)plane, sum, false) : (int)__builtin_amdgcn_udot4(levels, plane, (uint32_t)sum, false);
}
template <int CTRL>
__device__ __forceinline__ float dpp_from(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true)); }

template <int FMT>
__global__ __launch_bounds__(64, 4) void encode_affine_kernel(const float* __restrict__ wg, uint8_t* __restrict__ dst, int64_t nblocks, ShortJob job) {
    constexpr Spec sp = spec_of(FMT);
    constexpr int bits = sp.bits, gsz = sp.gsz, ng = 256 / gsz, quads = gsz / 4;
    constexpr int scq = (1 << sp.scb) - 1, mq = (1 << sp.mb) - 1, bias = (mq + 1) / 2;
    constexpr float eps = 1e-15f, top = (float)((1 << bits) - 1);
    constexpr float unit = bits == 1 ? 1.0f : 1.0f / (float)((1 << bits) - 1);  // unit_level(bits, n) = n * unit
    struct Blocks {
        uint4 planes[gsz == 32 ? 4 : 0][quads / 4][64];  // the weights as integers X
        union {
            float errors[6][64];  // of the fit
            struct {              // of what follows
                float2 sums[2][64];  // (value, its integer code) of every group: scales, and offsets with their sign turned
                double2 joint_level[1 << bits];  // a level, and its square as the refinements have it, a float product
            };
        };
        uint8_t hcode[128];
        double2 level[1 << bits];  // a level n * unit, and its exact square
    };
    // (one or the other: together they would leave room for fewer wavefronts per SIMD)
    __shared__ union { Team team; Blocks blocks; } lds;
    const int with_short = job.L.n > 0;
    if (with_short && blockIdx.x == 0) { encode_short_block<FMT>(job, lds.team); return; }
    auto& planes = lds.blocks.planes;
    auto& sums = lds.blocks.sums;
    auto& errors = lds.blocks.errors;
    auto& hcode = lds.blocks.hcode;
    auto& level = lds.blocks.level;
    auto& joint_level = lds.blocks.joint_level;
    const int t = threadIdx.x, g = t & (ng - 1), first = t & ~(ng - 1);
    const float own_level = (float)t * unit;
    if (t < 1 << bits) level[t] = double2{(double)own_level, (double)own_level * (double)own_level};
    __syncthreads();
    const int64_t mine = (int64_t)(blockIdx.x - with_short) * (64 / ng) + t / ng;
    const int64_t blk = mine < nblocks ? mine : nblocks - 1;  // past the end: the last block again, stored by nobody
    const float* const group = wg + blk * 256 + g * gsz;
    float x[gsz];
#pragma unroll
    for (int i = 0; i < gsz; i += 4) {
        float4 v;  // (the caller's pointer is aligned to a float only)
        __builtin_memcpy(&v, group + i, 16);
        x[i] = v.x; x[i + 1] = v.y; x[i + 2] = v.z; x[i + 3] = v.w;
    }
    float maxw = -1e30f, minw = 1e30f;
    uint32_t top_bits = 0;
    double sx = 0;  // the same in every refit
#pragma unroll
    for (int i = 0; i < gsz; ++i) {
        maxw = fmaxf(maxw, x[i]);
        minw = fminf(minw, x[i]);
        top_bits = max(top_bits, __float_as_uint(x[i]) & 0x7FFFFFFFu);
        sx += (double)x[i];
    }
    const bool odd = top_bits > 0x71000000u;  // above 2^99, infinite or NaN
    constexpr double sw = (double)gsz;

    // ---- the weights as integers X of 31 bits, x = q X within q, a plane of bytes each (the uppermost one signed)
    const float range = maxw - minw;
    const uint32_t up = (283u - (top_bits >> 23)) << 23;  // 2^k: |x| 2^k below 2^30
    const float pw = __uint_as_float(up), q = __uint_as_float(0x7F000000u - up);
    const bool plain = !odd && top_bits >= 0x11000000u && range >= 1e-28f;  // |x| from 2^-93 on
    int sX[4] = {};
    uint32_t X[4][4];  // (of a group of 16; one of 32 has them in LDS, whose registers a fourth wavefront needs)
#pragma unroll
    for (int i = 0; i < gsz; i += 16) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = (uint32_t)(int)(x[i + 4 * c + j] * pw);
            const uint32_t a = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u), b = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u);
            const uint32_t e = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u), f = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
            X[0][c] = __builtin_amdgcn_perm(b, a, 0x05040100u);
            X[1][c] = __builtin_amdgcn_perm(b, a, 0x07060302u);
            X[2][c] = __builtin_amdgcn_perm(f, e, 0x05040100u);
            X[3][c] = __builtin_amdgcn_perm(f, e, 0x07060302u);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
#pragma unroll
            for (int c = 0; c < 4; ++c) sX[k] = byte_dot(0x01010101u, X[k][c], sX[k], k == 3);
            if constexpr (gsz == 32) planes[k][i / 16][t] = uint4{X[k][0], X[k][1], X[k][2], X[k][3]};  // (read by this lane only)
        }
    }
    auto joined = [](const int (&v)[4]) __attribute__((always_inline)) {  // (256 v[3] + v[2] and 256 v[1] + v[0] fit in 31 bits)
        return __builtin_fma((double)(v[2] + 256 * v[3]), 65536.0, (double)(v[0] + 256 * v[1]));
    };
    const double sumX = joined(sX), mean = sumX * ((double)q / sw);

    // ---- scale s and offset m of a group by least squares over (level, weight)
    float s = range, m = minw;
    float off_s = 0.0f, off_m = 0.0f;  // how far s and m may be from the reference's: 0, or they are a quick_solve of `was`
    uint32_t p[quads], was[quads];
    // The reference's double sums over the levels `was`, and its solution.  The fit's squares of levels are fused, and so exact, a
    // refinement's are float products.  JOINT: of is `level` or `joint_level`, a lane's own choice.
    auto solve = [&](const double2* of, auto joint) __attribute__((always_inline)) {
        double sl = 0, sl2 = 0, sxl = 0;
#pragma unroll
        for (int i = 0; i < gsz; ++i) {
            const double2* const at = of + (was[i / 4] >> (8 * (i % 4)) & 0xFFu);
            const double l = at->x;
            sl += l;
            if constexpr (decltype(joint)::value) sl2 += at->y;
            else sl2 = __builtin_fma(l, l, sl2);
            float xi = x[i];
            asm volatile("" : "+v"(xi));  // (or the 32 conversions would be kept in registers for this rarer path)
            sxl = __builtin_fma((double)xi, l, sxl);
            if (i % 8 == 7) __builtin_amdgcn_sched_barrier(0);  // (all factors first would take 128 registers)
        }
        asm volatile("" : "+v"(sxl));  // (or this sum moves behind the branch, and its factors wait in registers)
        const double D = fms2(sw, sl2, sl, sl);
        if (D > 1e-20) {
            s = (float)(fms2(sw, sxl, sx, sl) / D);
            m = (float)(fms2(sl2, sx, sl, sxl) / D);
        }
        off_s = off_m = 0.0f;
    };
    // The same from integer dot products, and a bound on how far the result is from the reference's: what the roundings of
    // the levels n * unit (and, JOINT, of their squares) do to the slope, a unit of X in every weight, and the rounding of
    // either result.  With S = sum (l - mean)^2 = D / (top^2 gsz), k^2 = sum l^2 / S, z^2 = gsz / S and sum (x - mean)^2 at most
    // gsz (range / 2)^2 the levels' part of the slope is u k (z range / 2 + 2 |s|) by Cauchy-Schwarz, the weights' z q.
    // False without a spread.
    constexpr LevelRounding rounding = level_rounding(bits);
    auto quick_solve = [&](const uint32_t (&lv)[quads], auto joint) __attribute__((always_inline)) {
        uint32_t s1 = 0, s2 = 0;
        int dX[4] = {};
#pragma unroll
        for (int i = 0; i < quads; ++i) {
            s1 = __builtin_amdgcn_udot4(lv[i], 0x01010101u, s1, false);
            s2 = __builtin_amdgcn_udot4(lv[i], lv[i], s2, false);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
#pragma unroll
            for (int i = 0; i < quads; i += 4) {
                uint4 v{X[k][0], X[k][1], X[k][2], X[k][3]};
                if constexpr (gsz == 32) v = planes[k][i / 4][t];
                dX[k] = byte_dot(lv[i], v.x, dX[k], k == 3);
                dX[k] = byte_dot(lv[i + 1], v.y, dX[k], k == 3);
                dX[k] = byte_dot(lv[i + 2], v.z, dX[k], k == 3);
                dX[k] = byte_dot(lv[i + 3], v.w, dX[k], k == 3);
            }
        }
        const uint32_t D = (uint32_t)gsz * s2 - s1 * s1;
        if (!plain || D == 0) return false;
        const double n1 = (double)s1, nX = joined(dX), dD = (double)D;
        double rD = __builtin_amdgcn_rcp(dD);
        rD = __builtin_fma(__builtin_fma(-dD, rD, 1.0), rD, rD);
        const double per_level = __builtin_fma(sw, nX, -(sumX * n1)) * rD * (double)q;
        s = (float)(per_level * (1.0 / rounding.ideal));
        m = (float)__builtin_fma(-per_level, n1 * (1.0 / sw), mean);
        const float rq = __builtin_amdgcn_rsqf((float)D), k = __builtin_amdgcn_sqrtf((float)((uint32_t)gsz * s2)) * rq, z = (float)gsz * top * rq;
        const float as = fabsf(s), am = fabsf(m);
        const float slope = __builtin_fmaf(1.02f * (float)rounding.level * kUlp * k, __builtin_fmaf(z, 0.5f * range, 2.0f * as), 1.02f * q * z);
        off_s = __builtin_fmaf(2.05f * kUlp, as, slope);
        off_m = __builtin_fmaf(2.05f * kUlp, am + as, __builtin_fmaf(1.02f, q, slope));
        if constexpr (decltype(joint)::value) {
            const float square = 1.02f * (float)rounding.square * kUlp * k * k;
            off_s = __builtin_fmaf(square, as, off_s);
            off_m = __builtin_fmaf(square, am + fabsf(minw) + range, off_m);
        }
        return true;
    };
    using Group = std::false_type;
    using Joint = std::true_type;
    auto keep_levels = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < quads; ++i) was[i] = p[i];
    };
#pragma unroll
    for (int i = 0; i < quads; ++i) was[i] = p[i] = 0;

    // ---- per-group fit
    if (!(fabsf(s) > 1e-30f)) { s = 0.0f; m = 0.0f; }
    else {
        // assign levels, then refit (s, m): four times, then once more behind the polish.  Where the reference's own s and m are
        // needed, `exact` sends the step back to the head of the loop, the only place where they are solved for (code that is
        // there six times does not fit the instruction cache).
        bool exact = false, polished = false, settled = false, divide = false;
#pragma unroll 1
        for (int iter = 0;;) {
            if (exact) solve(level, Group{});
            exact = false;
            if (iter == 5) break;
            if (iter == 4 && !polished) {
                exact = off_s > 0.0f;
                if (__any(exact)) continue;
                polished = true;
                // Six scales, the one with the least squared error, formed in fp32.  Of a distance y = x - m, cs * unit, the level
                // and the multiply-add are rounded here, the product and the difference there, and a weight between two levels
                // may take the other one: together within `slip` = u (3 max |x| + 6 |m| + 13 |s|), so that a sum of squares e is
                // off by less than 2 sqrt(gsz e) slip + gsz slip^2 + 40 u e <= e (2^-14 + 40 u) + 33 2^14 slip^2.
                // Scales that are as near to the least as that (both sides of an optimum with the same levels are: a third of
                // the groups of 16 at two bits) are compared by the reference's sums.
                float best_s = s, low = 1e38f, high = 0.0f;
                const float slip = kUlp * (3.0f * __uint_as_float(top_bits) + 6.0f * fabsf(m) + 13.0f * fabsf(s));
                auto scale_of = [&](int j) __attribute__((always_inline)) { return s * __builtin_fmaf(0.05f, (float)(j < 3 ? j - 3 : j - 2), 1.0f); };
                const float slip2 = 33.0f * 16384.0f * slip * slip;
#pragma unroll 1
                for (int j = 0; j < 6; ++j) {
                    const float cs = scale_of(j), r = __builtin_amdgcn_rcpf(cs), mr = m * r, cu = cs * unit;
                    float e = 0.0f;
#pragma unroll
                    for (int i = 0; i < gsz; ++i) {
                        const float v = __builtin_amdgcn_fmed3f(__builtin_fmaf(x[i], r, -mr), 0.0f, 1.0f);
                        const float n = __builtin_fmaf(v, top, kRound) - kRound;
                        const float d = __builtin_fmaf(n, cu, m - x[i]);
                        e = __builtin_fmaf(d, d, e);
                    }
                    errors[j][t] = e;  // (read by this lane only)
                    high = fmaxf(high, e);
                    if (e < low) { low = e; best_s = cs; }
                }
                // (an e of NaN does not reach `high`; it takes an odd weight, an infinite scale or offset, or a scale of 0)
                const bool even = !odd && low >= 1e-30f && high <= 1e37f && fabsf(s) <= 1e18f && fabsf(s) >= 1e-18f && fabsf(m) <= 1e18f;
                const float limit = low * 1.0000635f + slip2;
                uint32_t close = 0;
#pragma unroll
                for (int j = 0; j < 6; ++j) close |= (!even || errors[j][t] * 0.9999365f - slip2 <= limit) ? 1u << j : 0u;
                if (close & (close - 1)) {
                    double best = 1e300;
#pragma unroll 1
                    for (int j = 0; j < 6; ++j) {
                        if (!(close >> j & 1)) continue;
                        const float cs = scale_of(j);
                        if (!group_levels<bits>(x, m, cs, 0.0f, odd, p)) group_levels_divided<bits>(x, group, m, cs, odd, p);
                        double e = 0.0;
#pragma unroll
                        for (int i = 0; i < gsz; ++i) {
                            const float d = __builtin_fmaf(cs, (float)(p[i / 4] >> (8 * (i % 4)) & 0xFFu) * unit, m) - x[i];
                            e = __builtin_fma((double)d, (double)d, e);
                            if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                        }
                        if (e < best) { best = e; best_s = cs; }
                    }
                    if (best == 1e300) best_s = s;
                }
                s = best_s;
            }
            if (!settled) {
                divide = !group_levels<bits>(x, m, s, off_s + off_m, odd, p);
                exact = divide && off_s > 0.0f;
                settled = true;
                if (__any(exact)) continue;  // (all lanes: the ones that go ahead alone would have the wavefront go twice)
            }
            if (divide) group_levels_divided<bits>(x, group, m, s, odd, p);
            settled = divide = false;
            if (!quick_solve(p, Group{})) {
                exact = true;
                if (off_s > 0.0f) continue;  // (a solution that fails leaves s and m as they were)
            }
            keep_levels();
            ++iter;
        }
    }

    // ---- global d / dm and the joint refinement
    constexpr int kMirror = ng == 8 ? 0x141 : 0x140;  // row_half_mirror, row_mirror: a block's lanes the other way round
    auto block_max = [&](float v) __attribute__((always_inline)) {
        v = fmaxf(v, dpp_from<kMirror>(v));
        if constexpr (ng == 16) v = fmaxf(v, dpp_from<0x141>(v));  // row_half_mirror
        v = fmaxf(v, dpp_from<0xB1>(v));                           // quad_perm [1,0,3,2]
        return fmaxf(v, dpp_from<0x4E>(v));                        // quad_perm [2,3,0,1]
    };
    // binary16 of (sum of value x code) / (sum of code^2) over the groups in order, 0 where there is no support: of the
    // scales in even lanes, of the offsets in odd ones
    auto joint_scales = [&](float& d, float& dm, float s, int sc, float m, int mc) __attribute__((always_inline)) {
        __syncthreads();
        sums[0][t] = float2{s, (float)sc};
        sums[1][t] = float2{-m, (float)mc};
        __syncthreads();
        const float2* const mine = sums[t & 1] + first;
        double num = 0, den = 0;
#pragma unroll 4
        for (int k = 0; k < ng; ++k) {
            const float2 v = mine[k];
            num = __builtin_fma((double)v.x, (double)v.y, num);
            den = __builtin_fma((double)v.y, (double)v.y, den);
        }
        float q = (den > 1e-20) ? half_bits_to_float(float_to_half_bits((float)(num / den))) : 0.0f;
        q = fabsf(q) <= eps ? 0.0f : q;
        const float other = __shfl_xor(q, 1, 64);
        d = t & 1 ? other : q;
        dm = t & 1 ? q : other;
    };
    auto snap_scale = [&](float s, float d) __attribute__((always_inline)) {
        return (s == 0.0f) ? 0 : max(0, min(scq, (int)lroundf(s / d)));
    };
    auto snap_min = [&](float m, float dm) __attribute__((always_inline)) {
        return max(-bias, min(mq - bias, (int)lroundf(-m / dm)));
    };
    // Codes and binary16 values from s and m that may be off by off_s and off_m; `sure` falls where a difference of that size
    // could change one: a quotient near the middle of two integers, or bounds with different binary16 values.  (Quotients here
    // within 4 u, the reference's own rounding among them.)
    bool sure;
    auto quick_code = [&](float v, float off, float unit_of, int lo, int hi) __attribute__((always_inline)) {
        const float r = __builtin_amdgcn_rcpf(unit_of), c = v * r, n = rintf(c);
        sure = sure && fabsf(c - n) <= 0.5f - __builtin_fmaf(off, fabsf(r), 5.0f * kUlp * fabsf(c)) - 1e-6f;
        return (int)fminf(fmaxf(n, (float)lo), (float)hi);
    };
    auto quick_half = [&](float v, float off) __attribute__((always_inline)) {
        const _Float16 lo = (_Float16)(v - off), hi = (_Float16)(v + off);
        sure = sure && lo == hi && fabsf(v) >= 1.25e-7f && fabsf(v) < 65000.0f;  // (smaller ones the reference does not round)
        return (float)lo;
    };
    __syncthreads();  // (the errors' room)
    if (t < 1 << bits) joint_level[t] = double2{(double)own_level, (double)(own_level * own_level)};
    __syncthreads();
    float d, dm;
    int sc, mc;
    bool dead = false;     // all scales vanish: d = 0, codes 0, dm stays 1
    bool refined = false;  // `was` are a refinement's levels, not the fit's
#pragma unroll 1
    for (;;) {
        const float max_s = block_max(fabsf(s)), max_m = block_max(fabsf(m));
        sure = true;
        d = quick_half(max_s * (1.0f / (float)scq), __builtin_fmaf(block_max(off_s), 1.01f / (float)scq, 5.0f * kUlp / (float)scq * max_s));
        dm = quick_half(max_m * (1.0f / (float)bias), __builtin_fmaf(block_max(off_m), 1.01f / (float)bias, 5.0f * kUlp / (float)bias * max_m));
        sc = quick_code(s, off_s, d, 0, scq);
        mc = quick_code(-m, off_m, dm, -bias, mq - bias);
        if (__all(sure)) break;
        if (__any(off_s > 0.0f)) {
            if (off_s > 0.0f) solve(level, Group{});
            continue;
        }
        dead = max_s <= eps;
        d = 0.0f, dm = 1.0f, sc = mc = 0;
        if (!dead) {
            d = half_bits_to_float(float_to_half_bits(max_s / (float)scq));
            if (max_m > eps) dm = half_bits_to_float(float_to_half_bits(max_m / (float)bias));
            sc = snap_scale(s, d);
            if (max_m > eps) mc = snap_min(m, dm);
        }
        break;
    }
    // A refinement's codes and joint_scales with fp32 sums over a block's lanes, which are within 6 u of their terms.
    auto quick_codes = [&](int& nsc, int& nmc, float& nd, float& ndm) __attribute__((always_inline)) {
        sure = true;
        nsc = quick_code(s, off_s, d, 0, scq);
        nmc = fabsf(dm) > eps ? quick_code(-m, off_m, dm, -bias, mq - bias) : 0;
        const float fs = (float)nsc, fm = (float)nmc, as = s * fs, am = -m * fm;
        // the upper half of a block's lanes takes the offsets, the lower one the scales
        const bool upper = t & (ng / 2);
        auto total = [&](float of_s, float of_m) __attribute__((always_inline)) {
            float v = (upper ? of_m : of_s) + dpp_from<kMirror>(upper ? of_s : of_m);
            if constexpr (ng == 16) v += dpp_from<0x141>(v);
            v += dpp_from<0xB1>(v);
            v += dpp_from<0x4E>(v);
            return v;
        };
        const float num = total(as, am), den = total(fs * fs, fm * fm);
        const float err = total(__builtin_fmaf(6.0f * kUlp, fabsf(as), off_s * fs), __builtin_fmaf(6.0f * kUlp, fabsf(am), off_m * fabsf(fm)));
        const float r = __builtin_amdgcn_rcpf(den), v = num * r, off = 1.02f * __builtin_fmaf(err, r, 5.0f * kUlp * fabsf(v));
        const bool none = den == 0.0f, before = sure;
        float mine = quick_half(v, off);
        if (none) { sure = before; mine = 0.0f; }
        const float other = dpp_from<kMirror>(mine);
        nd = upper ? other : mine;
        ndm = upper ? mine : other;
    };
#pragma unroll 1
    for (int iter = 0;; ++iter) {  // (dead blocks come along for the barriers and keep their values)
        const float eff_s = d * (float)sc;
        const float eff_m = -dm * (float)mc;
        bool failed = false;
        if (eff_s != 0.0f) {
            if (!group_levels<bits>(x, eff_m, eff_s, 0.0f, odd, p)) group_levels_divided<bits>(x, group, eff_m, eff_s, odd, p);
        } else if (iter == 5) {
#pragma unroll
            for (int i = 0; i < quads; ++i) p[i] = 0;
        }
        if (iter == 5) break;  // (the payload's levels)
        if (eff_s != 0.0f) {
            if (quick_solve(p, Joint{})) {
                keep_levels();
                refined = true;
            } else if (plain) {
                // One level for all weights, as where a group's offset is far from dm times its code: the reference's D is the
                // rounding of that level's square, and s and m stay unless it is positive.  (With its sums taken there instead
                // 58.7 M weights of Q_G_2, groups of a spread of 0.004 about offsets of 0.05, 384 us, 305 so.)
                failed = joint_level[p[0] & 0xFFu].y > level[p[0] & 0xFFu].y;
            } else failed = true;
        }
        int nsc, nmc;
        float nd, ndm;
#pragma unroll 1
        for (;;) {
            quick_codes(nsc, nmc, nd, ndm);
            if (__all(dead || (sure && !failed))) break;
            if (__any(failed || off_s > 0.0f)) {
                // Once more with the reference's own s and m, which are the fit's where no refinement has replaced them.
#pragma unroll 1
                for (int again = 0; again < 2; ++again) {
                    if (again && failed) {
                        keep_levels();
                        refined = true;
                    }
                    if (again ? failed : off_s > 0.0f) solve(refined ? joint_level : level, Joint{});
                }
                failed = false;
                continue;
            }
            nsc = dead ? 0 : snap_scale(s, d);
            nmc = (!dead && fabsf(dm) > eps) ? snap_min(m, dm) : 0;
            joint_scales(nd, ndm, s, nsc, m, nmc);
            break;
        }
        if (!dead) { sc = nsc; mc = nmc; d = nd; dm = ndm; }
    }
    // ---- payload: levels | scale codes | biased min codes | binary16 d | binary16 dm, one LSB-first stream.  A lane's
    // levels are whole bytes; the header is put together from the lanes' codes in LDS.
    constexpr int lane_bytes = gsz * bits / 8, lane_dwords = (lane_bytes + 3) / 4;
    uint32_t packed[lane_dwords] = {};
#pragma unroll
    for (int i = 0; i < gsz; ++i) {
        const uint32_t c = p[i / 4] >> (8 * (i % 4)) & 0xFFu;
        packed[i * bits / 32] |= c << (i * bits % 32);
        if (i * bits % 32 + bits > 32) packed[i * bits / 32 + 1] |= c >> (32 - i * bits % 32);
    }
    __syncthreads();
    hcode[t] = (uint8_t)sc;
    hcode[64 + t] = (uint8_t)(mc + bias);
    __syncthreads();
    if (mine >= nblocks) return;
    uint8_t* pay = dst + blk * (int64_t)sp.block_bytes;
#pragma unroll
    for (int i = 0; i < lane_bytes / 4; ++i) __builtin_memcpy(pay + g * lane_bytes + 4 * i, &packed[i], 4);
    if constexpr (lane_bytes % 4 == 2) __builtin_memcpy(pay + g * lane_bytes + lane_bytes - 2, &packed[lane_dwords - 1], 2);
    constexpr int head = 32 * bits, sc_end = ng * sp.scb, mn_end = sc_end + ng * sp.mb;
    const uint32_t dh = float_to_half_bits(d) | (float_to_half_bits(dm) << 16);
    static_assert(sp.scb == sp.mb && (sp.scb == 4 || sp.scb == 6) && sc_end % 8 == 0, "a byte of the header has bits of two codes");
    for (int byte = g; byte < sp.block_bytes - head; byte += ng) {
        const bool offsets = 8 * byte >= sc_end;
        const int pos = 8 * byte - (offsets ? sc_end : 0), k = pos / sp.scb;
        const uint8_t* const codes = hcode + (offsets ? 64 : 0) + first;
        uint32_t v;
        if (8 * byte < mn_end) v = ((uint32_t)codes[k] | (uint32_t)codes[k + 1] << sp.scb) >> (pos - k * sp.scb);
        else v = dh >> (8 * byte - mn_end);
        pay[head + byte] = (uint8_t)v;
    }
}

// The same with the reference's double sums in every pass (17 passes, some 12 instructions per weight and pass; level_pass
// repeats a pass in which a weight lies too close to a rounding boundary).  More instructions and none of the repeated steps of
// encode_affine_kernel: the faster one where the time is that of the slowest wavefront, see launch_encode_affine.
// use(i, n) for every weight of the group, n (float) = its level index for offset m and scale s; `reset` forgets what
// `use` gathered.  odd: the group holds a NaN, an infinity or a magnitude the bound does not cover.
// With u = 2^-24 and T = top (x - m) / s, which matters up to `top`: the reference's three roundings put its value within
// 3 u T, here the reciprocal (1 ulp), m / s and the multiply-add within 3 u T + u top |m / s|; adding 1.5 2^23 rounds to an
// integer without an error of its own.
template <int BITS, int GSZ, class Reset, class Use>
__device__ __forceinline__ void level_pass(const float (&x)[GSZ], float m, float s, bool odd, Reset&& reset, Use&& use) {
    constexpr float top = (float)((1 << BITS) - 1);
    float r = __builtin_amdgcn_rcpf(s);
    const float mr = m * r;
    auto near_level = [&](float v, float& off) __attribute__((always_inline)) {
        const float t = __builtin_amdgcn_fmed3f(__builtin_fmaf(v, r, -mr), 0.0f, 1.0f);
        const float n = __builtin_fmaf(t, top, kRound) - kRound;
        off = __builtin_fmaf(t, top, -n);
        return n;
    };
    float far = 0.0f;
    reset();
#pragma unroll
    for (int i = 0; i < GSZ; i += 2) {
        float o0, o1;
        const float n0 = near_level(x[i], o0), n1 = near_level(x[i + 1], o1);
        far = fmaxf(fmaxf(fabsf(o0), fabsf(o1)), far);
        use(i, n0);
        use(i + 1, n1);
    }
    const float reach = 0.5f - 5.9604644775390625e-8f * (6.0f * (top + 1.0f) + 4.0f + 1.01f * top * fabsf(mr));
    // (written so that a NaN bound, as from s = 0, takes the branch; so does a scale whose reciprocal lost bits)
    if (odd || !(far <= reach) || !(fabsf(r) >= 1e-36f)) {
        const bool all = odd || !(reach > 0.0f) || !(fabsf(r) >= 1e-36f);
        reset();
        asm volatile("" : "+v"(r));  // (or the levels above would be kept in registers for this rare path)
#pragma unroll
        for (int i = 0; i < GSZ; ++i) {
            float o, n = near_level(x[i], o);
            if (all || !(fabsf(o) <= reach)) n = (float)unit_nearest_dev((x[i] - m) / s, BITS);
            use(i, n);
            __builtin_amdgcn_sched_barrier(0);  // one division at a time: interleaved, they would take the registers of the fast path
        }
    }
}

template <int FMT>
__global__ __launch_bounds__(64, spec_of(FMT).gsz == 32 ? 3 : 4) void encode_affine_summed_kernel(const float* __restrict__ wg, uint8_t* __restrict__ dst, int64_t nblocks, ShortJob job) {
    constexpr Spec sp = spec_of(FMT);
    constexpr int bits = sp.bits, gsz = sp.gsz, ng = 256 / gsz;
    constexpr int scq = (1 << sp.scb) - 1, mq = (1 << sp.mb) - 1, bias = (mq + 1) / 2;
    constexpr float eps = 1e-15f;
    constexpr float unit = bits == 1 ? 1.0f : 1.0f / (float)((1 << bits) - 1);  // unit_level(bits, n) = n * unit
    struct Blocks {
        double2 sums[2][64];  // (value, its integer code) of every group: scales, and offsets with their sign turned
        float errors[6][64];
        uint8_t hcode[128];
    };
    // (one or the other: together they would leave room for three wavefronts per SIMD)
    __shared__ union { Team team; Blocks blocks; } lds;
    const int with_short = job.L.n > 0;
    if (with_short && blockIdx.x == 0) { encode_short_block<FMT>(job, lds.team); return; }
    auto& sums = lds.blocks.sums;
    auto& errors = lds.blocks.errors;
    auto& hcode = lds.blocks.hcode;
    const int t = threadIdx.x, g = t & (ng - 1), first = t & ~(ng - 1);
    const int64_t mine = (int64_t)(blockIdx.x - with_short) * (64 / ng) + t / ng;
    const int64_t blk = mine < nblocks ? mine : nblocks - 1;  // past the end: the last block again, stored by nobody
    float x[gsz];
#pragma unroll
    for (int i = 0; i < gsz; i += 4) {
        float4 v;  // (the caller's pointer is aligned to a float only)
        __builtin_memcpy(&v, wg + blk * 256 + g * gsz + i, 16);
        x[i] = v.x; x[i + 1] = v.y; x[i + 2] = v.z; x[i + 3] = v.w;
    }
    float maxw = -1e30f, minw = 1e30f;
    uint32_t top_bits = 0;
    double sx = 0;  // the same in every refit
#pragma unroll
    for (int i = 0; i < gsz; ++i) {
        maxw = fmaxf(maxw, x[i]);
        minw = fminf(minw, x[i]);
        top_bits = max(top_bits, __float_as_uint(x[i]) & 0x7FFFFFFFu);
        sx += (double)x[i];
    }
    const bool odd = top_bits > 0x71000000u;  // above 2^99, infinite or NaN
    constexpr double sw = (double)gsz;

    double sl, sl2, sxl;
    auto solve = [&](float& s, float& m) __attribute__((always_inline)) {
        const double D = fms2(sw, sl2, sl, sl);
        if (D > 1e-20) {
            s = (float)(fms2(sw, sxl, sx, sl) / D);
            m = (float)(fms2(sl2, sx, sl, sxl) / D);
        }
    };
    auto clear = [&]() __attribute__((always_inline)) { sl = 0; sl2 = 0; sxl = 0; };

    // ---- per-group fit
    float s = maxw - minw, m = minw;
    if (!(fabsf(s) > 1e-30f)) { s = 0.0f; m = 0.0f; }
    else {
        // assign levels, then refit (s, m) by least squares over (level, weight): four times, then once more behind the polish
#pragma unroll 1
        for (int iter = 0; iter < 5; ++iter) {
            if (iter == 4) {
                // Six scales, the one with the least squared error, formed in fp32.  Of a distance y = x - m, cs * unit, the level
                // and the multiply-add are rounded here, the product and the difference there, and a weight between two levels
                // may take the other one: together within `slip` = u (3 max |x| + 6 |m| + 13 |s|), so that a sum of squares e is
                // off by less than 2 sqrt(gsz e) slip + gsz slip^2 + 40 u e <= e (2^-14 + 40 u) + 33 2^14 slip^2.
                // Scales that are as near to the least as that (both sides of an optimum with the same levels are: a third of
                // the groups of 16 at two bits) are compared by the reference's sums.
                float best_s = s, low = 1e38f, high = 0.0f;
                const float slip = 5.9604644775390625e-8f * (3.0f * __uint_as_float(top_bits) + 6.0f * fabsf(m) + 13.0f * fabsf(s));
                auto scale_of = [&](int j) __attribute__((always_inline)) { return s * __builtin_fmaf(0.05f, (float)(j < 3 ? j - 3 : j - 2), 1.0f); };
                const float slip2 = 33.0f * 16384.0f * slip * slip;
#pragma unroll 1
                for (int j = 0; j < 6; ++j) {
                    const float cs = scale_of(j), r = __builtin_amdgcn_rcpf(cs), mr = m * r, cu = cs * unit;
                    float e = 0.0f;
#pragma unroll
                    for (int i = 0; i < gsz; ++i) {
                        const float v = __builtin_amdgcn_fmed3f(__builtin_fmaf(x[i], r, -mr), 0.0f, 1.0f);
                        const float n = __builtin_fmaf(v, (float)((1 << bits) - 1), kRound) - kRound;
                        const float d = __builtin_fmaf(n, cu, m - x[i]);
                        e = __builtin_fmaf(d, d, e);
                    }
                    errors[j][t] = e;  // (read by this lane only)
                    high = fmaxf(high, e);
                    if (e < low) { low = e; best_s = cs; }
                }
                // (an e of NaN does not reach `high`; it takes an odd weight, an infinite scale or offset, or a scale of 0)
                const bool plain = !odd && low >= 1e-30f && high <= 1e37f && fabsf(s) <= 1e18f && fabsf(s) >= 1e-18f && fabsf(m) <= 1e18f;
                const float limit = low * 1.0000635f + slip2;
                uint32_t close = 0;
#pragma unroll
                for (int j = 0; j < 6; ++j) close |= (!plain || errors[j][t] * 0.9999365f - slip2 <= limit) ? 1u << j : 0u;
                if (close & (close - 1)) {
                    double best = 1e300;
#pragma unroll 1
                    for (int j = 0; j < 6; ++j) {
                        if (!(close >> j & 1)) continue;
                        const float cs = scale_of(j);
                        double e;
                        level_pass<bits, gsz>(x, m, cs, odd, [&]() __attribute__((always_inline)) { e = 0.0; },
                                              [&](int i, float n) __attribute__((always_inline)) {
                                                  const float d = __builtin_fmaf(cs, n * unit, m) - x[i];
                                                  e = __builtin_fma((double)d, (double)d, e);
                                              });
                        if (e < best) { best = e; best_s = cs; }
                    }
                    if (best == 1e300) best_s = s;
                }
                s = best_s;
            }
            level_pass<bits, gsz>(x, m, s, odd, clear, [&](int i, float n) __attribute__((always_inline)) {
                const double l = (double)(n * unit);
                sl += l;
                sl2 = __builtin_fma(l, l, sl2);
                sxl = __builtin_fma((double)x[i], l, sxl);
            });
            solve(s, m);
        }
    }

    // ---- global d / dm and the joint refinement
    auto block_max = [&](float v) __attribute__((always_inline)) {
#pragma unroll
        for (int k = ng / 2; k >= 1; k >>= 1) v = fmaxf(v, __shfl_xor(v, k, 64));
        return v;
    };
    // binary16 of (sum of value x code) / (sum of code^2) over the groups in order, 0 where there is no support: of the
    // scales in even lanes, of the offsets in odd ones
    auto joint_scales = [&](float& d, float& dm, float s, int sc, float m, int mc) __attribute__((always_inline)) {
        __syncthreads();
        sums[0][t] = double2{(double)s, (double)sc};
        sums[1][t] = double2{(double)-m, (double)mc};
        __syncthreads();
        const double2* const mine = sums[t & 1] + first;
        double num = 0, den = 0;
#pragma unroll
        for (int k = 0; k < ng; ++k) {
            const double2 v = mine[k];
            num = __builtin_fma(v.x, v.y, num);
            den = __builtin_fma(v.y, v.y, den);
        }
        float q = (den > 1e-20) ? half_bits_to_float(float_to_half_bits((float)(num / den))) : 0.0f;
        q = fabsf(q) <= eps ? 0.0f : q;
        const float other = __shfl_xor(q, 1, 64);
        d = t & 1 ? other : q;
        dm = t & 1 ? q : other;
    };
    const float max_s = block_max(fabsf(s)), max_m = block_max(fabsf(m));
    const bool dead = max_s <= eps;  // all scales vanish: d = 0, codes 0, dm stays 1
    float d = 0.0f, dm = 1.0f;
    int sc = 0, mc = 0;
    auto snap_scale = [&](float s, float d) __attribute__((always_inline)) {
        return (s == 0.0f) ? 0 : max(0, min(scq, (int)lroundf(s / d)));
    };
    auto snap_min = [&](float m, float dm) __attribute__((always_inline)) {
        return max(-bias, min(mq - bias, (int)lroundf(-m / dm)));
    };
    if (!dead) {
        d = half_bits_to_float(float_to_half_bits(max_s / (float)scq));
        if (max_m > eps) dm = half_bits_to_float(float_to_half_bits(max_m / (float)bias));
        sc = snap_scale(s, d);
        if (max_m > eps) mc = snap_min(m, dm);
    }
#pragma unroll 1
    for (int iter = 0; iter < 5; ++iter) {  // (dead blocks come along for the barriers and keep their values)
        const float eff_s = d * (float)sc;
        const float eff_m = -dm * (float)mc;
        if (eff_s != 0.0f) {
            level_pass<bits, gsz>(x, eff_m, eff_s, odd, clear, [&](int i, float n) __attribute__((always_inline)) {
                const float l = n * unit;
                sl += (double)l;
                sl2 += (double)(l * l);  // the square is a float product here, not fused
                sxl = __builtin_fma((double)x[i], (double)l, sxl);
            });
            solve(s, m);
        }
        if (!dead) sc = snap_scale(s, d);
        if (!dead) mc = (fabsf(dm) > eps) ? snap_min(m, dm) : 0;
        float nd, ndm;
        joint_scales(nd, ndm, s, sc, m, mc);
        if (!dead) { d = nd; dm = ndm; }
    }
    // ---- payload: levels | scale codes | biased min codes | binary16 d | binary16 dm, one LSB-first stream.  A lane's
    // levels are whole bytes; the header is put together from the lanes' codes in LDS.
    constexpr int lane_bytes = gsz * bits / 8, lane_dwords = (lane_bytes + 3) / 4;
    uint32_t packed[lane_dwords];
    auto clear_packed = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < lane_dwords; ++i) packed[i] = 0;
    };
    const float eff_s = d * (float)sc;
    const float eff_m = -dm * (float)mc;
    clear_packed();
    if (eff_s != 0.0f) {
        level_pass<bits, gsz>(x, eff_m, eff_s, odd, clear_packed, [&](int i, float n) __attribute__((always_inline)) {
            const uint32_t c = (uint32_t)n;
            packed[i * bits / 32] |= c << (i * bits % 32);
            if (i * bits % 32 + bits > 32) packed[i * bits / 32 + 1] |= c >> (32 - i * bits % 32);
        });
    }
    __syncthreads();
    hcode[t] = (uint8_t)sc;
    hcode[64 + t] = (uint8_t)(mc + bias);
    __syncthreads();
    if (mine >= nblocks) return;
    uint8_t* p = dst + blk * (int64_t)sp.block_bytes;
#pragma unroll
    for (int i = 0; i < lane_bytes / 4; ++i) __builtin_memcpy(p + g * lane_bytes + 4 * i, &packed[i], 4);
    if constexpr (lane_bytes % 4 == 2) __builtin_memcpy(p + g * lane_bytes + lane_bytes - 2, &packed[lane_dwords - 1], 2);
    constexpr int head = 32 * bits, sc_end = ng * sp.scb, mn_end = sc_end + ng * sp.mb;
    const uint32_t dh = float_to_half_bits(d) | (float_to_half_bits(dm) << 16);
    for (int byte = g; byte < sp.block_bytes - head; byte += ng) {
        uint32_t v = 0;
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const int pos = 8 * byte + b;
            uint32_t bit;
            if (pos < sc_end) bit = ((uint32_t)hcode[first + pos / sp.scb] >> (pos % sp.scb)) & 1u;
            else if (pos < mn_end) bit = ((uint32_t)hcode[64 + first + (pos - sc_end) / sp.mb] >> ((pos - sc_end) % sp.mb)) & 1u;
            else bit = (dh >> (pos - mn_end)) & 1u;
            v |= bit << b;
        }
        p[head + byte] = (uint8_t)v;
    }
}

// (all launchers of this kind: `job` rides along as the first workgroup)
template <int FMT>
static void launch_encode_affine(const float* w, int64_t nblocks, uint8_t* dst, const ShortJob& job, hipStream_t s) {
    constexpr int per_wave = 64 / (256 / spec_of(FMT).gsz);
    const dim3 grid((unsigned)((nblocks + per_wave - 1) / per_wave + (job.L.n > 0)));
    // Up to some wavefronts a SIMD a call takes as long as its slowest wavefronts, and of a few thousand some meet several of the
    // steps that are taken again, at two and three bits above all; beyond, the number of instructions counts.  us, double sums in
    // every pass and integer sums: Q_G_4 786432 weights 23.5 and 25.0, 5 M 38.7 and 40.9, 8 M 54.5 and 49.6; Q_G_3 1 M 23.7 and 28.8, 5 M 37.7
    // and 38.2, 8 M 53.8 and 49.3; Q_G_2 786432 17.5 and 20.2, 5 M 39.6 and 39.9, 8 M 58.5 and 54.7; SB256A2 524288 18.0 and 20.0, 8 M
    // 59.7 and 55.5; SB256A3 2 M 23.2 and 24.7, 8 M 59.5 and 55.7.  (Between, a few per cent either way with the weights.)  Q_1_5
    // at every size timed: 262144 19.7 and 26.5, 8 M 48.0 and 52.7, 16 M 83.5 and 87.3.  All of normal weights; ones that reach a bound in
    // nearly every refinement are slower at any size (16 M of Q_G_4: of 1e-6 93 and 115, u^8 90 and 104, two values 89 and 94).
    if constexpr (FMT != TFQ_Q_1_5) {
        if (nblocks > 24576) {
            hipLaunchKernelGGL(encode_affine_kernel<FMT>, grid, dim3(64), 0, s, w, dst, nblocks, job);
            return;
        }
    }
    hipLaunchKernelGGL(encode_affine_summed_kernel<FMT>, grid, dim3(64), 0, s, w, dst, nblocks, job);
}

// ---- encoders with one scale per run of weights (a group of 32 or a block of 256)
// (Comp8Team and ordered_sums, which the short blocks use too, are in tfq_encode_short.hpp)
// `width` (<= 48) bits of v at bit `pos` of an LDS image that starts out as zeros
__device__ __forceinline__ void image_bits(uint32_t* img, uint32_t pos, uint64_t v, int width) {
    const uint32_t sh = pos & 31u;
    atomicOr(&img[pos >> 5], (uint32_t)(v << sh));
    if (sh + (uint32_t)width > 32u) atomicOr(&img[(pos >> 5) + 1], (uint32_t)((v << sh) >> 32));
    if (sh + (uint32_t)width > 64u) atomicOr(&img[(pos >> 5) + 2], (uint32_t)(v >> (64u - sh)));
}
// the codes of PER consecutive weights from weight `i0` (a multiple of 4) into a lattice block's image:
// [binary16 scale][16 codes, the last a bit short] x 16
template <int BITS, int PER>
__device__ __forceinline__ void image_lattice(uint32_t* img, int i0, const uint32_t (&code)[PER]) {
#pragma unroll
    for (int k = 0; k < PER; k += 4) {
        const int i = i0 + k;
        const bool slot = (i & 15) == 12;  // weight i + 3 gives up its low bit
        uint64_t v = (uint64_t)code[k] | ((uint64_t)code[k + 1] << BITS) | ((uint64_t)code[k + 2] << (2 * BITS));
        v |= (uint64_t)(slot ? code[k + 3] >> 1 : code[k + 3]) << (3 * BITS);
        image_bits(img, (uint32_t)(16 + BITS * i - (i >> 4)), v, 4 * BITS - (slot ? 1 : 0));
    }
}

// Companded 8-bit encoders: Q_G_8 (quant_grp8_compound, src/codec/block_codec.cpp:365-388, a scale per 32
// weights) and Q_8 (quant_lattice with bits = 8, :458-470, one scale per block, 7-bit slots), both on
// comp8_fit_scale_fp16 (:306-358): three least-squares seeds, 14 golden-section steps on the true squared
// error over [0.75 s, 1.25 s], then the +-4 neighbouring binary16 values, about 29 evaluations of every weight.
// Bound by vector instructions.  The grid is a cubic to within a hundred-thousandth of a step, so a value's place in it, and
// with that the nearest level, takes five instructions (Comp8Team::levels); the comparison of the two distances is left for
// values on a border, and for the codes.  58.7 M weights of Q_G_8: 11.4 ms with a wavefront per group, a bisection and lane 0
// adding, 798 us with both levels around a value and both distances, 571 us; Q_8: 9.84 ms, 1.19 ms, 795 us.  Four wavefronts
// a SIMD, for some spilled registers (two without: 716 us).  Lanes per run: as few as leave a wavefront per SIMD.
template <int FMT, int T>
__global__ __launch_bounds__(64, T == 8 ? 3 : T == 4 ? 2 : 4) void encode_comp8_kernel(const float* __restrict__ wg, uint8_t* __restrict__ dst, float smult, int64_t nunits, ShortJob job) {
    constexpr bool GROUPED = spec_of(FMT).codec == Codec::Grp8;
    constexpr int CNT = GROUPED ? 32 : 256, PER = CNT / T, TEAMS = 64 / T;
    __shared__ float lv[256];
    __shared__ uint32_t img[GROUPED ? 1 : TEAMS * 64];
    __shared__ Team short_team;
    const int with_short = job.L.n > 0;
    if (with_short && blockIdx.x == 0) { encode_short_block<FMT>(job, short_team); return; }
    const int lane = threadIdx.x, tl = lane % T;
    const int64_t mine = (int64_t)(blockIdx.x - with_short) * TEAMS + lane / T;  // group or block
    const int64_t unit = mine < nunits ? mine : nunits - 1;       // past the end: the last one again, stored by nobody
    for (int i = lane; i < 256; i += 64) lv[i] = __uint_as_float(kComp8Bits[i]);
    if constexpr (!GROUPED)
        for (int i = lane; i < TEAMS * 64; i += 64) img[i] = 0;
    Comp8Team<CNT, T> team;
    team.lv = lv;
    team.first = lane - tl;
    float m = 0.0f;
#pragma unroll
    for (int k = 0; k < PER; k += 4) {
        float4 v;  // (the caller's pointer is aligned to a float only)
        __builtin_memcpy(&v, wg + unit * CNT + tl * PER + k, 16);
        team.w[k] = v.x; team.w[k + 1] = v.y; team.w[k + 2] = v.z; team.w[k + 3] = v.w;
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) m = fmaxf(m, fabsf(team.w[k]));
#pragma unroll
    for (int sft = T / 2; sft >= 1; sft >>= 1) m = fmaxf(m, __shfl_xor(m, sft, 64));
    __syncthreads();
    const float s = team.fit((double)m) * smult;  // the _K tiers try scaled copies of the fitted scale
    uint32_t code[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) code[k] = (s > 0.0f) ? team.nearest(team.w[k] / s) : 0u;
    const uint32_t h = float_to_half_bits(s);
    if constexpr (GROUPED) {
        if (mine >= nunits) return;
        uint8_t* p = dst + (unit >> 3) * 272;
        const int g = (int)(unit & 7);
#pragma unroll
        for (int k = 0; k < PER; k += 4) {
            const uint32_t v = code[k] | (code[k + 1] << 8) | (code[k + 2] << 16) | (code[k + 3] << 24);
            __builtin_memcpy(p + 32 * g + tl * PER + k, &v, 4);
        }
        if (tl == 0) { p[256 + 2 * g] = (uint8_t)(h & 0xFF); p[257 + 2 * g] = (uint8_t)(h >> 8); }
    } else {
        uint32_t* mimg = img + (lane / T) * 64;
        image_lattice<8, PER>(mimg, tl * PER, code);
        if (tl == 0) atomicOr(&mimg[0], h);
        __syncthreads();
        const int64_t b0 = (int64_t)(blockIdx.x - with_short) * TEAMS;
        const int words = (int)min((int64_t)TEAMS, nunits - b0) * 64;
        for (int i = lane; i < words; i += 64) __builtin_memcpy(dst + b0 * 256 + 4 * i, &img[i], 4);
    }
}

// Lanes per run: 32 weights per lane keep the index-order sums short in total; where that leaves SIMDs of the chip
// without a wavefront, runs are spread over more lanes.
template <int FMT>
static void launch_encode_comp8(const float* w, int64_t nblocks, uint8_t* dst, float smult, const ShortJob& job, hipStream_t s) {
    constexpr bool GROUPED = spec_of(FMT).codec == Codec::Grp8;
    constexpr int T = GROUPED ? 1 : 8, SPREAD = GROUPED ? 4 : 16;
    const int64_t units = GROUPED ? nblocks * 8 : nblocks;
    const bool wide = (units * T + 63) / 64 < 1024;
    const unsigned grid = (unsigned)((units * (wide ? SPREAD : T) + 63) / 64 + (job.L.n > 0));
    if (grid == 0) return;
    if (wide) hipLaunchKernelGGL((encode_comp8_kernel<FMT, SPREAD>), dim3(grid), dim3(64), 0, s, w, dst, smult, units, job);
    else hipLaunchKernelGGL((encode_comp8_kernel<FMT, T>), dim3(grid), dim3(64), 0, s, w, dst, smult, units, job);
}

// Plain lattice encoders Q_4 / Q_2 (quant_lattice, src/codec/block_codec.cpp:443-497) and the fixed-codebook
// encoders Q_3 / Q_6 / Q_12 (quant_fixed_codebook, :624-663), which differ in the level table only:
// s = absmax / top level * smult, `iters` least-squares refits over the nearest levels, binary16; codes are the
// nearest level of w / s, slots (every 16th weight) keep the even index below.  The base ids run 2 (lattice) or
// 3 (fixed) refits with smult 1; the _K tiers try more.  Teams of sixteen lanes
// (of eight: 190 us, half the wavefronts for their registers).
// The tables of up to sixteen levels are looked up by bucket: a bucket is narrower than the distance of two
// midpoints, so it names the only two levels that can be nearest; the comparison of their distances is the
// reference's, and so is the scan over all levels that far-off values take.  58.7 M weights of Q_4: 1.30 ms with a block
// per wavefront, the scan for every weight and lane 0 adding, 229 us with the lanes of a team adding one after
// the other, 135 us.
template <int FMT>
__global__ __launch_bounds__(64) void encode_lattice_kernel(const float* __restrict__ wg, uint8_t* __restrict__ dst,
                                                            int iters, float smult, int64_t nblocks, ShortJob job) {
    constexpr Spec sp = spec_of(FMT);
    constexpr int T = 16;  // lanes of a team
    constexpr int bits = sp.bits, BB = sp.block_bytes, NL = 1 << bits, PER = 256 / T, TEAMS = 64 / T;
    constexpr bool FIXED = sp.codec == Codec::Fixed;
    constexpr bool SEARCH = FIXED && bits > 3;  // ascending quantile table: binary search on |v| (:596-622)
    __shared__ float tab[NL];
    __shared__ float4 bucket[SEARCH ? 1 : 64];  // (level lo, level lo + 1, lo)
    __shared__ uint32_t img[TEAMS * BB / 4];
    __shared__ Team short_team;
    const int with_short = job.L.n > 0;
    if (with_short && blockIdx.x == 0) { encode_short_block<FMT>(job, short_team); return; }
    const int lane = threadIdx.x, tl = lane % T, first = lane - tl;
    const int64_t mine = (int64_t)(blockIdx.x - with_short) * TEAMS + lane / T;
    const int64_t blk = mine < nblocks ? mine : nblocks - 1;  // past the end: the last block again, stored by nobody
    for (int i = lane; i < NL; i += 64) tab[i] = FIXED ? fixed_value(bits, (uint32_t)i) : grid_value(bits, (uint32_t)i);
    for (int i = lane; i < TEAMS * BB / 4; i += 64) img[i] = 0;
    __syncthreads();
    const float reach = tab[NL - 1] + 0.1f, per_unit = 32.0f / reach;  // buckets over [-reach, reach]
    if constexpr (!SEARCH) {
        const float edge = (float)lane * (reach / 32.0f) - reach - 0.001f;
        int lo = 0;
        for (int i = 1; i < NL - 1; ++i) lo += 0.5f * (tab[i - 1] + tab[i]) < edge;
        bucket[lane] = float4{tab[lo], tab[lo + 1], __int_as_float(lo), 0.0f};
        __syncthreads();
    }
    float w[PER];
    float m = 0.0f;
#pragma unroll
    for (int k = 0; k < PER; k += 4) {
        float4 v;  // (the caller's pointer is aligned to a float only)
        __builtin_memcpy(&v, wg + blk * 256 + tl * PER + k, 16);
        w[k] = v.x; w[k + 1] = v.y; w[k + 2] = v.z; w[k + 3] = v.w;
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) m = fmaxf(m, fabsf(w[k]));
#pragma unroll
    for (int sft = T / 2; sft >= 1; sft >>= 1) m = fmaxf(m, __shfl_xor(m, sft, 64));
    auto nearest = [&](float v, float* level) __attribute__((always_inline)) {
        if constexpr (SEARCH) {
            constexpr int half = NL / 2;
            const float a = fabsf(v);
            int lo = half;  // the first level of the upper half that is not below a, the last one at most
#pragma unroll
            for (int len = half / 2; len >= 1; len /= 2) lo += tab[lo + len - 1] < a ? len : 0;
            if (lo > half) {
                const float d0 = a - tab[lo - 1];
                const float d1 = tab[lo] - a;
                if (d1 >= d0) --lo;
            }
            const uint32_t best = (v >= 0.0f) ? (uint32_t)lo : (uint32_t)(half - 1 - (lo - half));
            *level = tab[best];
            return best;
        } else {
            const float4 e = bucket[(int)fminf(fmaxf((v + reach) * per_unit, 0.0f), 63.0f)];
            const bool up = fabsf(v - e.y) < fabsf(v - e.x);
            uint32_t best = (uint32_t)__float_as_int(e.z) + (up ? 1u : 0u);
            float l = up ? e.y : e.x;
            if (!(fabsf(v) <= 64.0f)) {  // distances may round to the same number, and a NaN is level 0: the scan decides
                best = 0;
                float bd = fabsf(v - tab[0]);
                for (int i = 1; i < NL; ++i) {
                    const float d = fabsf(v - tab[i]);
                    if (d < bd) { bd = d; best = (uint32_t)i; }
                }
                l = tab[best];
            }
            *level = l;
            return best;
        }
    };
    float s = (m > 1e-30f) ? m / tab[NL - 1] * smult : 0.0f;
    if (s > 0.0f) {
#pragma unroll 1
        for (int it = 0; it < iters; ++it) {
            float l[PER];
#pragma unroll
            for (int k = 0; k < PER; ++k) nearest(w[k] / s, &l[k]);
            auto step = [&](double& a, double& b) __attribute__((always_inline)) {
#pragma unroll
                for (int k = 0; k < PER; ++k) {
                    a = __builtin_fma((double)w[k], (double)l[k], a);
                    b = __builtin_fma((double)l[k], (double)l[k], b);
                }
            };
            // Every lane its own part, then the lanes': all terms are positive (a level has its weight's sign), so the order moves
            // either sum by less than 2^-44 of it.  Where that could turn the rounding of their quotient to fp32, or a sum is
            // no number, the team adds in the reference's order, which runs every addition once per lane.
            double num = 0.0, den = 0.0;
            step(num, den);
            num = team_sum<T>(num);
            den = team_sum<T>(den);
            const double q = num / den;
            if (!(den > 1e-10) || (float)(q * (1.0 + 0x1p-42)) != (float)(q * (1.0 - 0x1p-42))) ordered_sums<T>(first, num, den, step);
            if (den > 1e-20) s = (float)(num / den);
        }
    }
    if (!(s > 0.0f)) s = 0.0f;
    uint32_t code[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        float l;
        code[k] = nearest((s == 0.0f) ? 0.0f : w[k] / s, &l);
    }
    uint32_t* mimg = img + (lane / T) * (BB / 4);
    image_lattice<bits, PER>(mimg, tl * PER, code);
    if (tl == 0) atomicOr(&mimg[0], float_to_half_bits(s));
    __syncthreads();
    const int64_t b0 = (int64_t)(blockIdx.x - with_short) * TEAMS;
    const int words = (int)min((int64_t)TEAMS, nblocks - b0) * (BB / 4);
    for (int i = lane; i < words; i += 64) __builtin_memcpy(dst + b0 * BB + 4 * i, &img[i], 4);
}

// 12-bit compound encoder (quant_grp12_compound, src/codec/block_codec.cpp:969-1004): every group of 32 weights
// gets its own least-squares scale against the 4096-level table (same fit as above on 32 weights), then 256
// 12-bit codes and the eight binary16 scales.  A wavefront per block: eight lanes per group hold four weights
// each, the first lane of a group sums it in index order.
__global__ __launch_bounds__(64) void encode_grp12_kernel(const float* __restrict__ wg, uint8_t* __restrict__ dst,
                                                          int iters, float smult) {
    __shared__ float tab[4096];
    __shared__ float w[256];
    __shared__ float lev[256];
    __shared__ float sg[8];
    __shared__ uint16_t code[256];
    const int lane = threadIdx.x, g = lane >> 3;
    const int64_t blk = blockIdx.x;
    for (int i = lane; i < 4096; i += 64) tab[i] = fixed_value(12, (uint32_t)i);
    for (int i = lane; i < 256; i += 64) w[i] = wg[blk * 256 + i];
    __syncthreads();
    auto nearest = [&](float v) __attribute__((always_inline)) {
        const float a = fabsf(v);
        int lo = 2048, hi = 4095;
        while (lo < hi) {
            const int mid = (lo + hi) / 2;
            if (tab[mid] < a) lo = mid + 1; else hi = mid;
        }
        if (lo > 2048) {
            const float d0 = a - tab[lo - 1];
            const float d1 = tab[lo] - a;
            if (d1 >= d0) --lo;
        }
        return (v >= 0.0f) ? (uint32_t)lo : (uint32_t)(2047 - (lo - 2048));
    };
    // weights 4 (lane & 7) .. + 3 of group g: lanes of one group are consecutive, so an 8-lane max suffices
    float m = 0.0f;
    for (int t = 0; t < 4; ++t) m = fmaxf(m, fabsf(w[4 * lane + t]));
#pragma unroll
    for (int sft = 4; sft >= 1; sft >>= 1) m = fmaxf(m, __shfl_xor(m, sft, 64));
    float s = (m > 1e-30f) ? m / tab[4095] * smult : 0.0f;
    const bool live = s > 0.0f;  // per group; the refits run to the end once started, like the reference's
    for (int it = 0; it < iters; ++it) {
        if (live)
            for (int t = 0; t < 4; ++t) lev[4 * lane + t] = tab[nearest(w[4 * lane + t] / s)];
        __syncthreads();
        if (live && (lane & 7) == 0) {
            double num = 0.0, den = 0.0;
            for (int i = 32 * g; i < 32 * g + 32; ++i) {
                num = __builtin_fma((double)w[i], (double)lev[i], num);
                den = __builtin_fma((double)lev[i], (double)lev[i], den);
            }
            sg[g] = (den > 1e-20) ? (float)(num / den) : s;
        }
        __syncthreads();
        if (live) s = sg[g];
        __syncthreads();
    }
    if (!(s > 0.0f)) s = 0.0f;
    for (int t = 0; t < 4; ++t) code[4 * lane + t] = (uint16_t)((s > 0.0f) ? nearest(w[4 * lane + t] / s) : 0u);
    if ((lane & 7) == 0) sg[g] = s;
    __syncthreads();
    uint8_t* p = dst + blk * 400;
    for (int byte = lane; byte < 384; byte += 64) {
        // two codes in three bytes
        const int pair = byte / 3, part = byte - 3 * pair;
        const uint32_t two = (uint32_t)code[2 * pair] | ((uint32_t)code[2 * pair + 1] << 12);
        p[byte] = (uint8_t)(two >> (8 * part));
    }
    if (lane < 8) {
        const uint32_t h = float_to_half_bits(sg[lane]);
        p[384 + 2 * lane] = (uint8_t)(h & 0xFF);
        p[385 + 2 * lane] = (uint8_t)(h >> 8);
    }
}

// Grouped-lattice fallback encoder (quant_grp16 with grp16_fit_scale, src/codec/block_codec.cpp:739-914) for
// the ids that use that layout for full blocks: a wavefront per block, lane g owns group g (32 groups of 8), lane 0
// the sums over groups; fused operations where GCC's Release build fuses.
template <int FMT>
__global__ __launch_bounds__(64) void encode_grp16_kernel(const float* __restrict__ wg, uint8_t* __restrict__ dst) {
    constexpr Spec sp = spec_of(FMT);
    constexpr int bits = sp.bits, ng = 32;
    constexpr float eps = 1e-15f;
    constexpr float top_level = bits == 2 ? 1.5104f : bits == 4 ? 2.7178f : 8.0f;
    __shared__ float w[256];
    __shared__ float s_[32];
    __shared__ int sc_[32];
    __shared__ float dsh;
    __shared__ uint8_t code[256];
    const int64_t blk = blockIdx.x;
    const int t = threadIdx.x;
    for (int i = t; i < 256; i += 64) w[i] = wg[blk * 256 + i];
    __syncthreads();
    const float* x = w + (t & 31) * 8;
    auto nearest = [&](float v) __attribute__((always_inline)) -> uint32_t {
        if constexpr (bits == 2 || bits == 4) {
            uint32_t best = 0;
            float bd = fabsf(v - grid_value(bits, 0));
            for (int i = 1; i < (1 << bits); ++i) {
                const float d = fabsf(v - grid_value(bits, (uint32_t)i));
                if (d < bd) { bd = d; best = (uint32_t)i; }
            }
            return best;
        } else {
            constexpr float top = (float)((1u << bits) - 1u);
            const float c = fmaxf(-8.0f, fminf(8.0f, v));
            return (uint32_t)lroundf((c + 8.0f) * top / 16.0f);
        }
    };
    if (t < ng) {
        float maxa = 0.0f;
        for (int i = 0; i < 8; ++i) maxa = fmaxf(maxa, fabsf(x[i]));
        float s = (maxa > 1e-30f) ? maxa / top_level : 0.0f;
        if (!(fabsf(s) > 1e-30f)) s = 0.0f;
        else {
            auto assign_refit = [&](float as) __attribute__((always_inline)) {
                double num = 0.0, den = 0.0;
                for (int i = 0; i < 8; ++i) {
                    const float l = grid_value(bits, nearest(x[i] / as));
                    num = __builtin_fma((double)x[i], (double)l, num);
                    den = __builtin_fma((double)l, (double)l, den);
                }
                if (den > 1e-20) s = (float)(num / den);
            };
            for (int iter = 0; iter < 4; ++iter) assign_refit(s);
            float best_s = s;
            double best = 1e300;
            for (int k = -3; k <= 3; ++k) {
                if (k == 0) continue;
                const float cs = s * __builtin_fmaf(0.05f, (float)k, 1.0f);
                double e = 0.0;
                for (int i = 0; i < 8; ++i) {
                    const float l = grid_value(bits, nearest(x[i] / cs));
                    const float d = __builtin_fmaf(cs, l, -x[i]);
                    e = __builtin_fma((double)d, (double)d, e);
                }
                if (e < best) { best = e; best_s = cs; }
            }
            s = best_s;
            assign_refit(s);
        }
        s_[t] = s;
        sc_[t] = 0;
    }
    __syncthreads();
    if (t == 0) {
        float max_abs = 0.0f;
        for (int g = 0; g < ng; ++g) max_abs = fmaxf(max_abs, fabsf(s_[g]));
        dsh = (max_abs <= eps) ? 0.0f : half_bits_to_float(float_to_half_bits(max_abs / 7.0f));
    }
    __syncthreads();
    // once d has collapsed to zero the reference's (int)lround(s / 0) comes out as 0 after its clamp
    auto snap = [&](float s, float d) __attribute__((always_inline)) {
        return (s == 0.0f || d == 0.0f) ? 0 : max(0, min(7, (int)lroundf(s / d)));
    };
    if (dsh != 0.0f) {  // an all-zero block keeps d = 0 and every code 0
        if (t < ng) sc_[t] = snap(s_[t], dsh);
        __syncthreads();
        for (int iter = 0; iter < 5; ++iter) {
            const float d = dsh;
            if (t < ng) {
                const float eff = d * (float)sc_[t];
                if (eff != 0.0f) {
                    double num = 0.0, den = 0.0;
                    for (int i = 0; i < 8; ++i) {
                        const float l = grid_value(bits, nearest(x[i] / eff));
                        num = __builtin_fma((double)x[i], (double)l, num);
                        den = __builtin_fma((double)l, (double)l, den);
                    }
                    s_[t] = (den > 1e-20) ? (float)(num / den) : 0.0f;
                }
                sc_[t] = snap(s_[t], d);
            }
            __syncthreads();
            if (t == 0) {
                double num = 0.0, den = 0.0;
                for (int g = 0; g < ng; ++g) {
                    num = __builtin_fma((double)s_[g], (double)sc_[g], num);
                    den = __builtin_fma((double)sc_[g], (double)sc_[g], den);
                }
                float nd = (den > 1e-20) ? (float)(num / den) : 0.0f;
                nd = half_bits_to_float(float_to_half_bits(nd));
                if (fabsf(nd) <= eps) nd = 0.0f;
                dsh = nd;
            }
            __syncthreads();
        }
    }
    const float d = dsh;
    if (t < ng) {
        const float eff = d * (float)sc_[t];
        for (int i = 0; i < 8; ++i) code[t * 8 + i] = (eff == 0.0f) ? 0 : (uint8_t)nearest(x[i] / eff);
    }
    __syncthreads();
    constexpr int lev_bits = 256 * bits, sc_end = lev_bits + 96;
    const uint32_t dh = float_to_half_bits(d);
    uint8_t* p = dst + blk * (int64_t)sp.block_bytes;
    for (int byte = t; byte < sp.block_bytes; byte += 64) {
        uint32_t v = 0;
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const int pos = 8 * byte + b;
            uint32_t bit;
            if (pos < lev_bits) bit = ((uint32_t)code[pos / bits] >> (pos % bits)) & 1u;
            else if (pos < sc_end) bit = ((uint32_t)sc_[(pos - lev_bits) / 3] >> ((pos - lev_bits) % 3)) & 1u;
            else bit = (dh >> (pos - sc_end)) & 1u;
            v |= bit << b;
        }
        p[byte] = (uint8_t)v;
    }
}

__device__ __forceinline__ int q6k_round_dev(float v) {  // round to nearest even through the 1.5 * 2^23 bias
    return (int)(__float_as_uint(v + 12582912.f) & 0x007fffffu) - 0x00400000;
}
__device__ __forceinline__ int q6k_level_dev(float ratio) {
    ratio = fmaxf(-4000.0f, fminf(4000.0f, ratio));
    return max(-32, min(31, q6k_round_dev(ratio)));
}

// giters / polish / joint: the search effort (4, 3, 3 for Q_G_6 and _K_L).  A lane owns a group of 16, a wavefront four
// blocks, as in encode_affine_kernel, and levels are taken from a product by 1 / scale in the same way: its distance to
// the correctly rounded quotient is below 2^-22 |x / scale| and the quotient matters up to 32, so 0.5 - 2^-16 decides.
// 58.7 M weights: 1.96 ms with one block per wavefront, 280 us.
__global__ __launch_bounds__(64, 4) void encode_q6k_kernel(const float* __restrict__ wg, uint8_t* __restrict__ dst,
                                                           int giters, int polish, int joint, int64_t nblocks, ShortJob job) {
    constexpr int ng = 16;
    constexpr float eps = 1e-15f;
    __shared__ double2 sums[64];
    __shared__ uint32_t img[210];  // four blocks
    __shared__ Team short_team;
    const int with_short = job.L.n > 0;
    if (with_short && blockIdx.x == 0) { encode_short_block<TFQ_Q_G_6>(job, short_team); return; }
    const int t = threadIdx.x, g = t & (ng - 1), first = t & ~(ng - 1);
    const int64_t mine = (int64_t)(blockIdx.x - with_short) * 4 + t / ng;
    const int64_t blk = mine < nblocks ? mine : nblocks - 1;  // past the end: the last block again, stored by nobody
    float x[16];
    float maxa = 0.0f;
    uint32_t top_bits = 0;
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
        float4 v;  // (the caller's pointer is aligned to a float only)
        __builtin_memcpy(&v, wg + blk * 256 + g * 16 + i, 16);
        x[i] = v.x; x[i + 1] = v.y; x[i + 2] = v.z; x[i + 3] = v.w;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        maxa = fmaxf(maxa, fabsf(x[i]));
        top_bits = max(top_bits, __float_as_uint(x[i]) & 0x7FFFFFFFu);
    }
    const bool odd = top_bits > 0x71000000u;  // above 2^99, infinite or NaN
    // use(i, l) for every weight, l (float) = its level for `scale`; `reset` forgets what `use` gathered
    auto pass = [&](float scale, auto&& reset, auto&& use) __attribute__((always_inline)) {
        const float r = 1.0f / scale;
        float far = 0.0f;
        reset();
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float q = __builtin_amdgcn_fmed3f(x[i] * r, -32.0f, 31.0f);
            const float n = __builtin_rintf(q);
            far = fmaxf(far, fabsf(q - n));
            use(i, n);
        }
        if (odd || !(far <= 0.5f - 1.52587890625e-5f) || !(fabsf(r) < 1e37f)) {
            reset();
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                use(i, (float)q6k_level_dev(x[i] / scale));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    auto refit16 = [&](float scale, float* out) __attribute__((always_inline)) {
        double num, den;
        pass(scale, [&]() __attribute__((always_inline)) { num = 0.0; den = 0.0; },
             [&](int i, float n) __attribute__((always_inline)) {
                 const double l = (double)n;
                 num = __builtin_fma((double)x[i], l, num);
                 den = __builtin_fma(l, l, den);
             });
        if (den > 1e-20) *out = (float)(num / den);
    };
    float sg = (maxa > eps) ? maxa / 32.0f : 0.0f;
    if (fabsf(sg) <= eps) sg = 0.0f;
    else {
#pragma unroll 1
        for (int iter = 0; iter <= giters; ++iter) {  // the last one behind the polish
            if (iter == giters) {
                float best_s = sg;
                double best = 1e300;
#pragma unroll 1
                for (int k = -polish; k <= polish; ++k) {
                    if (k == 0) continue;
                    const float cs = sg * __builtin_fmaf(0.05f, (float)k, 1.0f);
                    double e;
                    pass(cs, [&]() __attribute__((always_inline)) { e = 0.0; },
                         [&](int i, float n) __attribute__((always_inline)) {
                             const float d = __builtin_fmaf(cs, n, -x[i]);
                             e = __builtin_fma((double)d, (double)d, e);
                         });
                    if (e < best) { best = e; best_s = cs; }
                }
                sg = best_s;
            }
            refit16(sg, &sg);
        }
    }
    float max_abs = fabsf(sg);
#pragma unroll
    for (int k = ng / 2; k >= 1; k >>= 1) max_abs = fmaxf(max_abs, __shfl_xor(max_abs, k, 64));
    const bool dead = max_abs <= eps;
    float d = 0.0f;
    int sc = 0;
    if (!dead) {
        const float iscale = -128.0f / max_abs;
        d = 1.0f / iscale;
        // the product feeds the rounding add directly: one fused operation in the reference's build
        sc = max(-127, min(127, (int)(__float_as_uint(__builtin_fmaf(iscale, sg, 12582912.f)) & 0x007fffffu) - 0x00400000));
    }
#pragma unroll 1
    for (int iter = 0; iter < joint; ++iter) {  // (dead blocks come along for the barriers)
        const float eff = d * (float)sc;
        if (eff != 0.0f) {
            float fitted = 0.0f;
            refit16(eff, &fitted);
            sg = fitted;
        }
        if (!dead) sc = (d == 0.0f) ? 0 : max(-127, min(127, q6k_round_dev(sg / d)));
        __syncthreads();
        sums[t] = double2{(double)sg, (double)sc};
        __syncthreads();
        double num = 0.0, den = 0.0;
#pragma unroll
        for (int k = 0; k < ng; ++k) {
            const double2 v = sums[first + k];
            num = __builtin_fma(v.x, v.y, num);
            den = __builtin_fma(v.y, v.y, den);
        }
        float nd = (den > 1e-20) ? (float)(num / den) : 0.0f;
        if (fabsf(nd) <= eps) nd = 0.0f;
        if (!dead) d = nd;
    }
    uint32_t packed[3] = {0, 0, 0};
    auto level_bits = [&](int i, uint32_t c) __attribute__((always_inline)) {
        packed[i * 6 / 32] |= c << (i * 6 % 32);
        if (i * 6 % 32 + 6 > 32) packed[i * 6 / 32 + 1] |= c >> (32 - i * 6 % 32);
    };
    const float eff = d * (float)sc;
    if (eff != 0.0f) {
        pass(eff, [&]() __attribute__((always_inline)) { packed[0] = packed[1] = packed[2] = 0; },
             [&](int i, float n) __attribute__((always_inline)) { level_bits(i, (uint32_t)((int)n + 32)); });
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) level_bits(i, 32u);
    }
    // a block is 210 bytes: its parts in the image are aligned to two bytes
    uint8_t* bytes = reinterpret_cast<uint8_t*>(img) + (t / ng) * 210;
#pragma unroll
    for (int i = 0; i < 6; ++i) *reinterpret_cast<uint16_t*>(bytes + 12 * g + 2 * i) = (uint16_t)(packed[i >> 1] >> (16 * (i & 1)));
    bytes[192 + g] = (uint8_t)(int8_t)sc;
    if (g == 0) *reinterpret_cast<uint16_t*>(bytes + 208) = (uint16_t)float_to_half_bits(d);
    __syncthreads();
    const int64_t b0 = (int64_t)(blockIdx.x - with_short) * 4;
    const int halves = (int)min((int64_t)4, nblocks - b0) * 105;
    uint8_t* p = dst + b0 * 210;
    for (int i = t; i < halves / 2; i += 64) __builtin_memcpy(p + 4 * i, &img[i], 4);
    if ((halves & 1) && t == 0) __builtin_memcpy(p + 2 * halves - 2, reinterpret_cast<const uint8_t*>(img) + 2 * halves - 2, 2);
}

// _K_M / _K_H tiers (src/codec/block_codec.cpp:2378-2400, :2551-2665, :2733-2824): a candidate payload replaces
// the current one when its decoded mean squared error (double, index order, fused like the reference's k_mse)
// is strictly smaller.  One wavefront per block: lanes decode both payloads, lane 0 compares, all lanes copy.
template <int FMT>
__global__ __launch_bounds__(64) void keep_better_kernel(const float* __restrict__ wg, uint8_t* __restrict__ cur,
                                                         const uint8_t* __restrict__ cand) {
    constexpr int BB = spec_of(FMT).block_bytes;
    __shared__ float dc[256], dn[256];
    __shared__ int take;
    const int64_t blk = blockIdx.x;
    const int t = threadIdx.x;
    uint8_t* pc = cur + blk * BB;
    const uint8_t* pn = cand + blk * BB;
    for (int i = t; i < 256; i += 64) {
        dc[i] = decode_weight<FMT>(pc, i);
        dn[i] = decode_weight<FMT>(pn, i);
    }
    __syncthreads();
    if (t == 0) {
        double ec = 0.0, en = 0.0;
        for (int i = 0; i < 256; ++i) {
            const double w = (double)wg[blk * 256 + i];
            const double a = w - (double)dc[i], b = w - (double)dn[i];
            ec = __builtin_fma(a, a, ec);
            en = __builtin_fma(b, b, en);
        }
        take = (en / 256.0) < (ec / 256.0);
    }
    __syncthreads();
    if (take)
        for (int i = t; i < BB; i += 64) pc[i] = pn[i];
}

// ---- four-tier mixes (Q_MX_*, Q_G_MX_*): a wavefront per block of L.n <= 256 weights
__global__ __launch_bounds__(64) void decode_mix_kernel(MixLayout L, const uint8_t* __restrict__ src, float* __restrict__ out) {
    const uint32_t lane = threadIdx.x;
    const int64_t blk = blockIdx.x;
    float v[4];
    mix_decode_wave(L, src + blk * L.bytes, lane, v);
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (4 * (int)lane + k < L.n) out[blk * L.n + 4 * lane + k] = v[k];
}

__device__ __forceinline__ float mix_level(int bits, uint32_t code) {
    return (bits == 3 || bits == 6 || bits == 12) ? fixed_value(bits, code) : grid_value(bits, code);
}
// nearest_level / nearest_fixed_level for the widths the mixes use (src/codec/block_codec.cpp:190-203, :596-606)
__device__ __forceinline__ uint32_t mix_nearest(int bits, float v) {
    if (bits == 8) {
        const float c = fmaxf(-8.0f, fminf(8.0f, v));
        return (uint32_t)lroundf((c + 8.0f) * 255.0f / 16.0f);
    }
    if (bits == 6 || bits == 12) {  // ascending quantile tables: search |v| in the upper half (:596-622)
        const int half = 1 << (bits - 1);
        const float a = fabsf(v);
        int lo = half, hi = 2 * half - 1;
        while (lo < hi) {
            const int mid = (lo + hi) / 2;
            if (fixed_value(bits, (uint32_t)mid) < a) lo = mid + 1; else hi = mid;
        }
        if (lo > half && fixed_value(bits, (uint32_t)lo) - a >= a - fixed_value(bits, (uint32_t)lo - 1u)) --lo;
        return v >= 0.0f ? (uint32_t)lo : (uint32_t)(half - 1 - (lo - half));
    }
    uint32_t best = 0;
    float bd = fabsf(v - mix_level(bits, 0));
    for (int i = 1; i < (1 << bits); ++i) {
        const float d = fabsf(v - mix_level(bits, (uint32_t)i));
        if (d < bd) { bd = d; best = (uint32_t)i; }
    }
    return best;
}

// Encoder of a block of L.n <= 256 weights (quant_quad_mix, src/codec/block_codec.cpp:2102-2205): weights ranked by
// magnitude, the c[3] largest into tier 3 and so on down; per tier (per 32 values of the most populated
// tier of a grouped id) s = max / top level and two least-squares refits on the first 32 values the scale
// covers; then tiers, values and scales as laid out in MixLayout.  Equal magnitudes rank by index here;
// the reference leaves their order to an unstable sort, so a block with a tie across a tier boundary may
// get the two weights' tiers the other way round.
__global__ __launch_bounds__(64) void encode_mix_kernel(MixLayout L, const float* __restrict__ wg, uint8_t* __restrict__ dst) {
    __shared__ float w[256], tv[256], lev[256];
    __shared__ uint32_t mag[256];  // |w| as its bit pattern: the same order as the values, and total (NaN sorts above inf)
    __shared__ float sc[4][8];
    __shared__ int live[8];
    __shared__ uint32_t words[200];  // the largest block is 784 bytes
    const uint32_t lane = threadIdx.x;
    const int64_t blk = blockIdx.x;
    const int n = L.n, valid = max(0, min(4, n - 4 * (int)lane));  // lane l holds weights 4 l .. 4 l + 3
    for (int i = lane; i < 256; i += 64) { const float x = i < n ? wg[blk * n + i] : 0.0f; w[i] = x; mag[i] = __float_as_uint(x) & 0x7FFFFFFFu; }
    for (int i = lane; i < 200; i += 64) words[i] = 0;
    if (lane < 32) sc[lane >> 3][lane & 7] = 0.0f;
    __syncthreads();
    const int n3 = L.c[3], n2 = n3 + L.c[2], n1 = n2 + L.c[1];
    uint32_t tiers = 0;
    for (int k = 0; k < valid; ++k) {
        const int i = 4 * lane + k;
        const uint32_t m = mag[i];
        int rank = 0;
        for (int j = 0; j < n; ++j) {
            const uint32_t mj = mag[j];
            rank += (mj > m || (mj == m && j < i)) ? 1 : 0;
        }
        const uint32_t t = rank < n3 ? 3u : rank < n2 ? 2u : rank < n1 ? 1u : 0u;
        tiers |= t << (2 * k);
    }
    uint32_t before[4], total[4];
    mix_scan(tiers, valid, lane, before, total);
    const int first[4] = {0, L.c[0], L.c[0] + L.c[1], L.c[0] + L.c[1] + L.c[2]};  // tier runs inside tv
    uint32_t rk[4] = {0, 0, 0, 0};
    for (int k = 0; k < valid; ++k) {
        const uint32_t t = (tiers >> (2 * k)) & 3u;
        rk[k] = before[t]++;
        tv[first[t] + rk[k]] = w[4 * lane + k];
    }
    __syncthreads();
    for (int t = 0; t < 4; ++t) {
        const int nsc = L.nsc[t];
        if (nsc == 0) continue;
        const int bits = L.bits[t], cnt = min(L.c[t], nsc * 32);
        const float top = bits == 2 ? 1.5104f : bits == 3 ? 3.0776f : bits == 4 ? 2.7178f : bits == 8 ? 8.0f
                                                                  : (bits == 6 || bits == 12) ? fixed_value(bits, (1u << bits) - 1u) : 1.0f;
        const float* x = tv + first[t];
        if ((int)lane < nsc) {
            float maxa = 0.0f;
            for (int j = 32 * lane; j < min(cnt, 32 * (int)lane + 32); ++j) maxa = fmaxf(maxa, fabsf(x[j]));
            const float s = (maxa > 1e-30f) ? maxa / top : 0.0f;
            sc[t][lane] = s;
            live[lane] = s > 0.0f;
        }
        __syncthreads();
        for (int it = 0; it < 2; ++it) {
            for (int j = lane; j < cnt; j += 64) {
                if (!live[j >> 5]) continue;
                lev[j] = bits == 1 ? (x[j] >= 0.0f ? 1.0f : -1.0f) : mix_level(bits, mix_nearest(bits, x[j] / sc[t][j >> 5]));
            }
            __syncthreads();
            if ((int)lane < nsc && live[lane]) {
                double num = 0.0, den = 0.0;
                for (int j = 32 * lane; j < min(cnt, 32 * (int)lane + 32); ++j) {
                    num = __builtin_fma((double)x[j], (double)lev[j], num);
                    den = __builtin_fma((double)lev[j], (double)lev[j], den);
                }
                if (den > 1e-20) sc[t][lane] = (float)(num / den);
            }
            __syncthreads();
        }
        if ((int)lane < nsc && !(sc[t][lane] > 0.0f)) sc[t][lane] = 0.0f;
        __syncthreads();
    }
    // the stream: byte l holds the tiers of lane l's weights, values at (start of the tier's run) + rank * width
    atomicOr(&words[lane >> 2], tiers << (8 * (lane & 3u)));
    uint32_t start[4];
    uint32_t at = 2u * (uint32_t)n;
    for (int t = 0; t < 4; ++t) { start[t] = at; at += (uint32_t)(L.c[t] * L.bits[t]); }
    for (int k = 0; k < valid; ++k) {
        const uint32_t t = (tiers >> (2 * k)) & 3u;
        const int bits = L.bits[t];
        const float v = w[4 * lane + k];
        const float s = L.nsc[t] > 0 ? sc[t][min((int)(rk[k] >> 5), L.nsc[t] - 1)] : 1.0f;
        uint32_t code;
        switch (bits) {
            case 1: code = v >= 0.0f ? 1u : 0u; break;
            case 16: code = float_to_half_bits(v); break;
            case 24: code = __float_as_uint(v) >> 8; break;
            case 32: code = __float_as_uint(v); break;
            default: code = mix_nearest(bits, (s == 0.0f) ? 0.0f : v / s); break;
        }
        const uint32_t pos = start[t] + rk[k] * (uint32_t)bits, sh = pos & 31u;
        atomicOr(&words[pos >> 5], code << sh);
        if (sh + (uint32_t)bits > 32u) atomicOr(&words[(pos >> 5) + 1], code >> (32u - sh));
    }
    __syncthreads();
    uint8_t* p = dst + blk * L.bytes;
    for (int byte = lane; byte < L.payload_bytes; byte += 64) p[byte] = (uint8_t)(words[byte >> 2] >> (8 * (byte & 3)));
    if (lane < 32) {
        const int t = lane >> 3, g = lane & 7;
        if (g < L.nsc[t]) {
            const uint32_t h = float_to_half_bits(sc[t][g]);
            p[L.sc_at[t] + 2 * g] = (uint8_t)(h & 0xFF);
            p[L.sc_at[t] + 2 * g + 1] = (uint8_t)(h >> 8);
        }
    }
}

// Wire -> Tiled16: one lane per 16-byte piece of the tiled buffer.  Piece p of a unit: p < 64 code
// slot of k-step 0, p < 128 of k-step 1, else a 16-byte part of a row header.  Codes narrower
// than 4 bits are widened to nibbles.
template <int FMT>
__global__ __launch_bounds__(256) void tile16_kernel(const uint8_t* __restrict__ wire, uint4* __restrict__ tiled,
                                                     int64_t N, int nblocks, int64_t npieces) {
    constexpr Spec sp = spec_of(FMT);
    constexpr int HB = tiled_header_bytes(FMT), HP = HB / 16, NP = tiled_planes(FMT), CW = tiled_code_width(FMT);
    constexpr int CP = tiled_code_bytes(FMT) / 16, PIECES = CP + 16 * HP;  // code pieces, all pieces of a unit
    constexpr uint32_t BB = sp.block_bytes, code_bytes = 256u * sp.bits / 8;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= npieces) return;
    const int64_t unit = i / PIECES;
    const int p = (int)(i - unit * PIECES);
    const int64_t tile = unit / nblocks;
    const int blk = (int)(unit - tile * nblocks);
    uint32_t o[4] = {0, 0, 0, 0};
    if (CW < 4 && p < CP) {
        // true-width code area: piece p = the 2-bit fields of lane p
        const int l = p, n = l & 15, c = l >> 4;
        const int64_t row = tile * 16 + n;
        if (row < N) {
            const uint8_t* src = wire + (row * nblocks + blk) * (int64_t)BB;
            for (int h = 0; h < 2; ++h)
                for (int e = 0; e < 32; ++e) {  // element e of the lane's 32-slot of k-step h
                    const uint32_t code = stream_bits(src, code_bytes, (uint32_t)(128 * h + 32 * c + e) * sp.bits, sp.bits);
                    const int j = e >> 3, t = e & 3, upper = (e >> 2) & 1;  // MFMA j, pair t, low / high half-word
                    o[2 * h + (j >> 1)] |= code << (16 * upper + 2 * (t + 4 * (j & 1)));
                }
        }
    } else if (p < CP) {
        const int plane = p >> 7, l = p & 63, n = l & 15, g32 = (l >> 4) + 4 * ((p >> 6) & 1);
        const int64_t row = tile * 16 + n;
        if (row < N) {
            const uint8_t* src = wire + (row * nblocks + blk) * (int64_t)BB;
#pragma unroll
            for (int j = 0; j < 32; ++j) {
                uint32_t code;
                if constexpr (NP == 2) {  // 8-bit code as an unsigned byte, split into nibbles
                    uint32_t u;
                    if constexpr (sp.codec == Codec::Sym32) {
                        u = (uint32_t)src[32 * g32 + j] ^ 0x80u;  // int8 code + 128
                    } else if constexpr (sp.codec == Codec::Grp8) {
                        u = src[32 * g32 + j];
                    } else {  // plain Q_8: every 16th weight is a 7-bit slot that decodes as an even index
                        const uint32_t e = (uint32_t)(32 * g32 + j);
                        const bool slot = (e & 15u) == 15u;
                        u = stream_bits(src, BB, 16u + 8u * e - (e >> 4), slot ? 7 : 8);
                        if (slot) u <<= 1;
                    }
                    code = plane ? u >> 4 : u & 15u;
                } else {
                    code = stream_bits(src, code_bytes, (uint32_t)(32 * g32 + j) * sp.bits, sp.bits);
                }
                o[j >> 3] |= code << (4 * (j & 7));
            }
        }
    } else {
        // header pieces: one per row, or part-major planes of sixteen rows (tiled_header_offset)
        const int n = HP == 1 ? p - CP : (p - CP) % 16, part = HP == 1 ? 0 : (p - CP) / 16;
        const int64_t row = tile * 16 + n;
        if (row < N) {
            const uint8_t* src = wire + (row * nblocks + blk) * (int64_t)BB;
            if constexpr (sp.codec == Codec::Lattice) {  // the block's one binary16 scale, for each of the 8 groups
                const uint32_t s2 = (uint32_t)src[0] | ((uint32_t)src[1] << 8);
                o[0] = o[1] = o[2] = o[3] = s2 | (s2 << 16);
            } else if constexpr (tiled_header_in_bytes(FMT)) {
                // part 0: the 16 scale codes, one per byte; part 1: the 16 offset codes (still biased); part 2: d, dm
                constexpr uint32_t ng = 256 / sp.gsz, sc_bits = ((ng * sp.scb + 7) / 8) * 8, mn_bits = ((ng * sp.mb + 7) / 8) * 8;
                const uint8_t* hsrc = src + code_bytes;
                const uint32_t hbytes = BB - code_bytes;
                if (part < 2) {
#pragma unroll
                    for (int g = 0; g < 16; ++g) {
                        const uint32_t code = part == 0 ? stream_bits(hsrc, hbytes, (uint32_t)g * sp.scb, sp.scb)
                                                        : stream_bits(hsrc, hbytes, sc_bits + (uint32_t)g * sp.mb, sp.mb);
                        o[g >> 2] |= code << (8 * (g & 3));
                    }
                } else {
                    o[0] = stream_bits(hsrc, hbytes, sc_bits + mn_bits, 16) | (stream_bits(hsrc, hbytes, sc_bits + mn_bits + 16, 16) << 16);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const uint32_t off = code_bytes + 16 * part + j;
                    if (off < BB) o[j >> 2] |= (uint32_t)src[off] << (8 * (j & 3));
                }
            }
        }
    }
    tiled[i] = uint4{o[0], o[1], o[2], o[3]};
}

// Decode straight from the Tiled16 layout: one workgroup per (row, block), one lane per weight,
// the arithmetic of decode_weight on the same header bytes.
template <int FMT>
__global__ __launch_bounds__(256) void decode_tiled_kernel(const uint8_t* __restrict__ tiled, float* __restrict__ out,
                                                           int nblocks) {
    constexpr Spec sp = spec_of(FMT);
    constexpr int HB = tiled_header_bytes(FMT), UB = tiled_unit_bytes(FMT);
    const int64_t rb = blockIdx.x;  // row * nblocks + blk
    const int64_t row = rb / nblocks;
    const int blk = (int)(rb - row * nblocks);
    const uint32_t i = threadIdx.x;
    const uint8_t* unit = tiled + ((row >> 4) * nblocks + blk) * (int64_t)UB;
    const int n = (int)(row & 15);
    const uint32_t g32 = i >> 5, j = i & 31;
    const uint8_t* codes = unit + (g32 >> 2) * 1024 + (n + 16 * (g32 & 3)) * 16;
    uint32_t idx;
    if constexpr (tiled_code_width(FMT) < 4) {
        const uint32_t ks = g32 >> 2, lane = (uint32_t)n + 16 * (g32 & 3), mj = j >> 3, t = j & 3, upper = (j >> 2) & 1;
        const uint32_t* lo = reinterpret_cast<const uint32_t*>(unit + 16 * lane);
        idx = (lo[2 * ks + (mj >> 1)] >> (16 * upper + 2 * (t + 4 * (mj & 1)))) & 3u;
    } else {
        idx = (codes[j >> 1] >> ((j & 1u) * 4)) & 15u;
    }
    const uint8_t* h = unit + tiled_code_bytes(FMT) + n * HB;
    float v;
    if constexpr (sp.codec == Codec::Grp8 || sp.codec == Codec::Lattice) {
        const float d = half_bits_to_float((uint32_t)h[2 * g32] | ((uint32_t)h[2 * g32 + 1] << 8));
        const uint32_t u = idx | (((codes[2048 + (j >> 1)] >> ((j & 1u) * 4)) & 15u) << 4);
        v = d * __uint_as_float(kComp8Bits[u]);
    } else if constexpr (sp.codec == Codec::Sym32) {
        const float d = half_bits_to_float((uint32_t)h[2 * g32] | ((uint32_t)h[2 * g32 + 1] << 8));
        int q = (int)idx - 8;
        if constexpr (tiled_planes(FMT) == 2) q = (int)(idx | (((codes[2048 + (j >> 1)] >> ((j & 1u) * 4)) & 15u) << 4)) - 128;
        v = (float)q * d;
    } else {
        constexpr uint32_t ng = 256 / sp.gsz;
        constexpr uint32_t sc_bits = ((ng * sp.scb + 7) / 8) * 8;
        constexpr uint32_t mn_bits = ((ng * sp.mb + 7) / 8) * 8;
        constexpr int bias = (1 << sp.mb) / 2;
        const uint32_t g = i / sp.gsz;
        float sc, mc, d, dm;
        if constexpr (tiled_header_in_bytes(FMT)) {
            const uint8_t* h0 = unit + tiled_header_offset(FMT, n, 0);
            const uint8_t* h1 = unit + tiled_header_offset(FMT, n, 1);
            const uint8_t* h2 = unit + tiled_header_offset(FMT, n, 2);
            sc = (float)h0[g];
            mc = (float)h1[g] - (float)bias;
            d = half_bits_to_float((uint32_t)h2[0] | ((uint32_t)h2[1] << 8));
            dm = half_bits_to_float((uint32_t)h2[2] | ((uint32_t)h2[3] << 8));
        } else {
            sc = (float)stream_bits(h, HB, g * sp.scb, sp.scb);
            mc = (float)stream_bits(h, HB, sc_bits + g * sp.mb, sp.mb) - (float)bias;
            d = half_bits_to_float(stream_bits(h, HB, sc_bits + mn_bits, 16));
            dm = half_bits_to_float(stream_bits(h, HB, sc_bits + mn_bits + 16, 16));
        }
        const float es = d * sc;
        const float neg = -(dm * mc);
        v = __builtin_fmaf(es, unit_level(sp.bits, idx), neg);
    }
    out[rb * 256 + i] = v;
}

template <int FMT>
int run_decode(const uint8_t* src, int64_t nblocks, float* out, const BlockLayout& tail, hipStream_t s) {
    if constexpr (kHasQuad<FMT>) {
        // dword reads need a 4-byte aligned payload and a 16-byte aligned destination; anything else
        // takes the byte-wise kernel
        if ((reinterpret_cast<uintptr_t>(src) & 3u) == 0 && (reinterpret_cast<uintptr_t>(out) & 15u) == 0) {
            const int64_t grid = (nblocks + 4 * kDecodeBlocks - 1) / (4 * kDecodeBlocks) + (tail.n > 0);
            hipLaunchKernelGGL(decode_quad_kernel<FMT>, dim3((unsigned)grid), dim3(256), 0, s, src, out, nblocks, tail);
            return hip_fail(hipGetLastError(), "decode launch");
        }
    }
    if (nblocks > 0) hipLaunchKernelGGL(decode_kernel<FMT>, dim3((unsigned)nblocks), dim3(256), 0, s, src, out);
    if (tail.n > 0) return launch_decode_short(tail, src + nblocks * (int64_t)spec_of(FMT).block_bytes, out + nblocks * 256, s);
    return hip_fail(hipGetLastError(), "decode launch");
}

}  // namespace

// Sizes as the reference's encoders choose them (src/codec/block_codec.cpp): lattice :443-455,
// affine :1394-1411, grouped-lattice fallback :788-815, Q_G_6 :1070-1082, Q_G_8 :2501-2510.
static bool affine_or_fallback(int bits, int gsz, int scb, int mb, double claimed, int n, BlockLayout* L) {
    const int levels = (n * bits + 7) / 8;
    const int budget = (int)std::ceil(claimed * (double)n / 8.0);
    const int ng = n >= gsz ? n / gsz : 0;
    const int total = levels + (ng * scb + 7) / 8 + (ng * mb + 7) / 8 + 4;
    if (ng > 0 && total <= budget) {
        *L = {BK_AFFINE, bits, n, total, gsz, ng, scb, mb, 0};
        return true;
    }
    const int ng8 = n >= 8 ? n / 8 : 0;
    const int sc_bytes = (ng8 * 3 + 7) / 8;
    const bool scales = n == 256 || (n >= 8 && levels + sc_bytes + 2 <= budget);
    const bool d_only = n >= 8 && levels + 2 <= budget;
    *L = {BK_GRP16, bits, n, levels + (scales ? sc_bytes : 0) + ((scales || d_only) ? 2 : 0), 8, ng8, 3, 0,
          scales ? 2 : d_only ? 1 : 0};
    return true;
}

bool block_layout(int fmt, int n, BlockLayout* L) {
    const Spec sp = spec_of(fmt);
    if (n <= 0 || n > 256) return false;
    switch (sp.codec) {
        case Codec::Mix: *L = {BK_MIX, 0, n, mix_layout(fmt, n).bytes, 0, 0, 0, 0, fmt}; return true;
        case Codec::Raw32: *L = {BK_RAW32, 32, n, n * 4, 0, 0, 0, 0, 0}; return true;
        case Codec::Lattice:
            *L = {n < 16 ? BK_LEVELS : BK_LATTICE, sp.bits, n, ((int)std::ceil(sp.bpw * (double)n) + 7) / 8, 0, 0, 0, 0, 0};
            return true;
        case Codec::Affine: case Codec::Grp16:
            return affine_or_fallback(sp.bits, sp.gsz, sp.scb, sp.mb, (double)sp.bpw, n, L);
        case Codec::Grp8:
            if (n >= 32 && n % 32 == 0) { *L = {BK_GRP8, 8, n, n + (n / 32) * 2, 32, n / 32, 0, 0, 0}; return true; }
            return affine_or_fallback(8, 32, 6, 6, (double)sp.bpw, n, L);  // 8.5, or 8.0 for the _K tiers
        case Codec::Fixed:
            *L = {n < 16 ? BK_LEVELS : BK_LATTICE, sp.bits, n, (sp.bits * n + 7) / 8, 0, 0, 0, 0, 1};
            return true;
        case Codec::Grp12:
            if (n >= 32 && n % 32 == 0) { *L = {BK_GRP12, 12, n, n * 3 / 2 + (n / 32) * 2, 32, n / 32, 0, 0, 0}; return true; }
            if (sp.scb) { *L = {n < 16 ? BK_LEVELS : BK_LATTICE, 12, n, (12 * n + 7) / 8, 0, 0, 0, 0, 1}; return true; }
            return affine_or_fallback(12, 512, 0, 0, 12.5, n, L);  // no affine layout: the grouped-lattice fallback
        case Codec::Q6K: {
            const int levels = (n * 6 + 7) / 8, sc_count = n >= 32 ? n / 16 : 0;
            const int budget = (int)std::ceil(6.5625 * (double)n / 8.0);
            const bool scales = n == 256 || (n >= 32 && levels + sc_count + 2 <= budget);
            *L = {BK_Q6K, 6, n, levels + (scales ? sc_count : 0) + (n >= 8 ? 2 : 0), 16, sc_count, 8, 0,
                  (n >= 8 ? 1 : 0) | ((scales ? sc_count : 0) << 8)};
            return true;
        }
        case Codec::Q1: *L = {BK_Q1, 1, n, (n + 7) / 8, 0, 0, 0, 0, 0}; return true;
        case Codec::Q16: case Codec::Q24: {
            // plain part, padded to the claim; the grouped ids fill the padding with residual means
            // when the block is a whole number of 32-groups (src/codec/block_codec.cpp:2450-2493, :2836-2847)
            const int plain = n * sp.bits / 8, claimed = (int)std::ceil((double)sp.bpw * (double)n / 8.0);
            const bool residual = sp.scb == 1 && claimed > plain && n % 32 == 0;
            *L = {BK_WIDE, sp.bits, n, claimed > plain ? claimed : plain, 0, 0, 0, 0,
                  (residual ? 1 : 0) | (sp.bits == 16 && n == 256 ? 2 : 0)};
            return true;
        }
        case Codec::Sym32:
            if (n < 32 || n % 32) return false;
            *L = {BK_SYM32, sp.bits, n, n * sp.bits / 8 + (n / 32) * 2, 32, n / 32, 0, 0, 0};
            return true;
        default: return false;
    }
}

int launch_decode_short(const BlockLayout& L, const uint8_t* src, float* out, hipStream_t s) {
    if (L.n <= 0 || L.n > 256 || L.bytes <= 0) return fail(TFQ_ERR_SHAPE, "decode: bad short-block layout");
    if (L.kind == BK_MIX) {
        hipLaunchKernelGGL(decode_mix_kernel, dim3(1), dim3(64), 0, s, mix_layout(L.aux, L.n), src, out);
        return hip_fail(hipGetLastError(), "decode launch");
    }
    hipLaunchKernelGGL(decode_short_kernel, dim3(1), dim3(256), 0, s, L, src, out);
    return hip_fail(hipGetLastError(), "decode launch");
}

int launch_decode(int fmt, const uint8_t* src, int64_t nblocks, float* out, hipStream_t s, const BlockLayout* short_block) {
    const BlockLayout tail = short_block ? *short_block : BlockLayout{};
    if (nblocks <= 0 && tail.n <= 0) return TFQ_OK;
    if (nblocks > 0x7FFFFFFF) return fail(TFQ_ERR_SHAPE, "decode: more than 2^31-1 blocks in one call");
    if (is_mix(fmt)) {
        const MixLayout L = mix_layout(fmt, 256);
        if (nblocks > 0) hipLaunchKernelGGL(decode_mix_kernel, dim3((unsigned)nblocks), dim3(64), 0, s, L, src, out);
        if (tail.n > 0) return launch_decode_short(tail, src + nblocks * L.bytes, out + nblocks * 256, s);
        return hip_fail(hipGetLastError(), "decode launch");
    }
    switch (canonical(fmt)) {
        case TFQ_Q_1: return run_decode<TFQ_Q_1>(src, nblocks, out, tail, s);
        case TFQ_Q_1_5: return run_decode<TFQ_Q_1_5>(src, nblocks, out, tail, s);
        case TFQ_Q_16: return run_decode<TFQ_Q_16>(src, nblocks, out, tail, s);
        case TFQ_Q_16_5: return run_decode<TFQ_Q_16_5>(src, nblocks, out, tail, s);
        case TFQ_Q_G_16: return run_decode<TFQ_Q_G_16>(src, nblocks, out, tail, s);
        case TFQ_Q_24: return run_decode<TFQ_Q_24>(src, nblocks, out, tail, s);
        case TFQ_Q_24_5: return run_decode<TFQ_Q_24_5>(src, nblocks, out, tail, s);
        case TFQ_Q_G_24: return run_decode<TFQ_Q_G_24>(src, nblocks, out, tail, s);
        case TFQ_Q_2: return run_decode<TFQ_Q_2>(src, nblocks, out, tail, s);
        case TFQ_Q_3: return run_decode<TFQ_Q_3>(src, nblocks, out, tail, s);
        case TFQ_Q_6: return run_decode<TFQ_Q_6>(src, nblocks, out, tail, s);
        case TFQ_Q_12: return run_decode<TFQ_Q_12>(src, nblocks, out, tail, s);
        case TFQ_Q_G_12: return run_decode<TFQ_Q_G_12>(src, nblocks, out, tail, s);
        case TFQ_Q_G_6: return run_decode<TFQ_Q_G_6>(src, nblocks, out, tail, s);
        case TFQ_Q_G_2_K_L: return run_decode<TFQ_Q_G_2_K_L>(src, nblocks, out, tail, s);
        case TFQ_Q_G_3_K_L: return run_decode<TFQ_Q_G_3_K_L>(src, nblocks, out, tail, s);
        case TFQ_Q_G_4_K_L: return run_decode<TFQ_Q_G_4_K_L>(src, nblocks, out, tail, s);
        case TFQ_Q_6_5: return run_decode<TFQ_Q_6_5>(src, nblocks, out, tail, s);
        case TFQ_Q_32: return run_decode<TFQ_Q_32>(src, nblocks, out, tail, s);
        case TFQ_Q_4: return run_decode<TFQ_Q_4>(src, nblocks, out, tail, s);
        case TFQ_Q_8: return run_decode<TFQ_Q_8>(src, nblocks, out, tail, s);
        case TFQ_Q_G_4: return run_decode<TFQ_Q_G_4>(src, nblocks, out, tail, s);
        case TFQ_Q_G_3: return run_decode<TFQ_Q_G_3>(src, nblocks, out, tail, s);
        case TFQ_Q_G_2: return run_decode<TFQ_Q_G_2>(src, nblocks, out, tail, s);
        case TFQ_Q_G_8: return run_decode<TFQ_Q_G_8>(src, nblocks, out, tail, s);
        case TFQ_SB256A3: return run_decode<TFQ_SB256A3>(src, nblocks, out, tail, s);
        case TFQ_SB256A2: return run_decode<TFQ_SB256A2>(src, nblocks, out, tail, s);
        case TFQ_B32S4: return run_decode<TFQ_B32S4>(src, nblocks, out, tail, s);
        case TFQ_B32S8: return run_decode<TFQ_B32S8>(src, nblocks, out, tail, s);
        default: return fail(TFQ_ERR_FORMAT, "decode: wire id " + std::to_string(fmt) + " is not handled");
    }
}

template <int FMT>
static int run_tile16(const uint8_t* wire, uint8_t* tiled, int64_t N, int64_t K, hipStream_t s) {
    const int nblocks = (int)(K / 256);
    const int64_t tiles = (N + 15) / 16;
    const int64_t npieces = tiles * nblocks * (tiled_unit_bytes(FMT) / 16);
    const int64_t grid = (npieces + 255) / 256;
    if (grid > 0x7FFFFFFF) return fail(TFQ_ERR_SHAPE, "matrix too large for one layout pass");
    hipLaunchKernelGGL(tile16_kernel<FMT>, dim3((unsigned)grid), dim3(256), 0, s, wire, reinterpret_cast<uint4*>(tiled), N,
                       nblocks, npieces);
    return hip_fail(hipGetLastError(), "layout launch");
}

int launch_tile16(int fmt, const uint8_t* wire, uint8_t* tiled, int64_t N, int64_t K, hipStream_t s) {
    switch (canonical(fmt)) {
        case TFQ_Q_G_4: return run_tile16<TFQ_Q_G_4>(wire, tiled, N, K, s);
        case TFQ_B32S4: return run_tile16<TFQ_B32S4>(wire, tiled, N, K, s);
        case TFQ_B32S8: return run_tile16<TFQ_B32S8>(wire, tiled, N, K, s);
        case TFQ_Q_G_8: return run_tile16<TFQ_Q_G_8>(wire, tiled, N, K, s);
        case TFQ_Q_8: return run_tile16<TFQ_Q_8>(wire, tiled, N, K, s);
        case TFQ_Q_G_3: return run_tile16<TFQ_Q_G_3>(wire, tiled, N, K, s);
        case TFQ_Q_G_2: return run_tile16<TFQ_Q_G_2>(wire, tiled, N, K, s);
        case TFQ_SB256A3: return run_tile16<TFQ_SB256A3>(wire, tiled, N, K, s);
        case TFQ_SB256A2: return run_tile16<TFQ_SB256A2>(wire, tiled, N, K, s);
        default: return fail(TFQ_ERR_FORMAT, "layout: wire id " + std::to_string(fmt) + " has no tiled layout");
    }
}

template <int FMT>
static int run_decode_tiled(const uint8_t* tiled, int64_t N, int64_t K, float* out, hipStream_t s) {
    const int nblocks = (int)(K / 256);
    const int64_t grid = N * nblocks;
    if (grid > 0x7FFFFFFF) return fail(TFQ_ERR_SHAPE, "decode: more than 2^31-1 blocks in one call");
    hipLaunchKernelGGL(decode_tiled_kernel<FMT>, dim3((unsigned)grid), dim3(256), 0, s, tiled, out, nblocks);
    return hip_fail(hipGetLastError(), "decode launch");
}

int launch_decode_tiled(int fmt, const uint8_t* tiled, int64_t N, int64_t K, float* out, hipStream_t s) {
    switch (canonical(fmt)) {
        case TFQ_Q_G_4: return run_decode_tiled<TFQ_Q_G_4>(tiled, N, K, out, s);
        case TFQ_B32S4: return run_decode_tiled<TFQ_B32S4>(tiled, N, K, out, s);
        case TFQ_B32S8: return run_decode_tiled<TFQ_B32S8>(tiled, N, K, out, s);
        case TFQ_Q_G_8: return run_decode_tiled<TFQ_Q_G_8>(tiled, N, K, out, s);
        case TFQ_Q_8: return run_decode_tiled<TFQ_Q_8>(tiled, N, K, out, s);
        case TFQ_Q_G_3: return run_decode_tiled<TFQ_Q_G_3>(tiled, N, K, out, s);
        case TFQ_Q_G_2: return run_decode_tiled<TFQ_Q_G_2>(tiled, N, K, out, s);
        case TFQ_SB256A3: return run_decode_tiled<TFQ_SB256A3>(tiled, N, K, out, s);
        case TFQ_SB256A2: return run_decode_tiled<TFQ_SB256A2>(tiled, N, K, out, s);
        default: return fail(TFQ_ERR_FORMAT, "decode: wire id " + std::to_string(fmt) + " has no tiled layout");
    }
}

// One more search per candidate (iters, smult), each kept only where it decodes strictly better than what
// `dst` holds.  `launch(out, iters, smult)` enqueues the encoder of the family.
struct TierTry { int iters; float smult; };

template <int FMT, class Launch>
static int encode_tiers(const TierTry* tries, int count, const float* w, int64_t nblocks, uint8_t* dst, hipStream_t s,
                        Launch&& launch) {
    if (count <= 0 || nblocks <= 0) return TFQ_OK;
    constexpr size_t BB = spec_of(FMT).block_bytes;
    uint8_t* cand = nullptr;
    TFQ_HIP(hipMalloc(&cand, (size_t)nblocks * BB));
    for (int c = 0; c < count; ++c) {
        launch(cand, tries[c].iters, tries[c].smult);
        hipLaunchKernelGGL(keep_better_kernel<FMT>, dim3((unsigned)nblocks), dim3(64), 0, s, w, dst, (const uint8_t*)cand);
    }
    const hipError_t e1 = hipStreamSynchronize(s);
    (void)hipFree(cand);
    if (e1 != hipSuccess) return hip_fail(e1, "hipStreamSynchronize");
    return TFQ_OK;
}

// Lattice and fixed-codebook ids with their tiers: base (iters0, 1.0), _K_M one longer search, _K_H six
// (src/codec/block_codec.cpp:2551-2665).
template <int FMT>
static int encode_lattice_family(int fmt, const float* w, int64_t nblocks, uint8_t* dst, const ShortJob& job, hipStream_t s) {
    constexpr bool FIXED = spec_of(FMT).codec == Codec::Fixed;
    auto launch = [&](uint8_t* out, int iters, float smult, const ShortJob& job) {
        const unsigned grid = (unsigned)((nblocks + 3) / 4 + (job.L.n > 0));
        hipLaunchKernelGGL((encode_lattice_kernel<FMT>), dim3(grid), dim3(64), 0, s, w, out, iters, smult, nblocks, job);
    };
    launch(dst, FIXED ? 3 : 2, 1.0f, job);
    const int a = FIXED ? 10 : 6, b = FIXED ? 24 : 14;
    const TierTry tries[6] = {{a, 1.0f}, {b, 1.0f}, {b, 0.9f}, {b, 1.1f}, {b, 0.7f}, {b, 1.3f}};
    const int tier = tier_of(fmt);
    return encode_tiers<FMT>(tries, tier >= 2 ? 6 : tier, w, nblocks, dst, s,
                             [&](uint8_t* out, int iters, float smult) { launch(out, iters, smult, ShortJob{}); });
}

// The job of a tensor's short last block (behind nblocks full ones); job->L.n = 0 where there is none.
static int short_job(int fmt, const BlockLayout* L, const float* w, int64_t nblocks, uint8_t* dst, ShortJob* job) {
    *job = ShortJob{};
    if (!L || L->n <= 0) return TFQ_OK;
    if (L->n >= 256 || L->bytes <= 0 || L->bytes > kMaxShortBytes) return fail(TFQ_ERR_SHAPE, "encode: bad short-block layout");
    job->L = *L;
    job->w = w + nblocks * 256;
    job->dst = dst + nblocks * (int64_t)spec_of(fmt).block_bytes;
    job->tier = tier_of(fmt);
    if (L->kind == BK_Q1)
        job->tier = fmt == TFQ_Q_1 ? -1 : (fmt == TFQ_Q_1_K_M || fmt == TFQ_Q_G_1_K_M) ? 1 : (fmt == TFQ_Q_1_K_H || fmt == TFQ_Q_G_1_K_H) ? 2 : 0;
    if (L->kind == BK_Q6K) job->tier = fmt == TFQ_Q_G_6_K_M ? 1 : fmt == TFQ_Q_G_6_K_H ? 2 : 0;
    // A short Q_G_8_K_M / _K_H block that still holds an affine header would take the searched affine encoder
    // of :2775-2785; with their claim of 8.0 bits the header never fits, so this does not occur.
    if (spec_of(fmt).codec == Codec::Grp8 && L->kind == BK_AFFINE && tier_of(fmt) > 0)
        return fail(TFQ_ERR_FORMAT, "encode: a short block of this id in the affine layout has no device encoder");
    return TFQ_OK;
}

// formats whose full-block encoder takes the short block along as a workgroup
static bool short_rides_along(int fmt) {
    switch (spec_of(fmt).codec) {
        case Codec::Affine: case Codec::Lattice: case Codec::Fixed: case Codec::Grp8: case Codec::Q6K: case Codec::Sym32: return true;
        default: return false;
    }
}

static int launch_encode_short(int fmt, const ShortJob& job, hipStream_t s) {
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(1), dim3(64), 0, s, job); };
    switch (canonical(fmt)) {
        case TFQ_Q_32: launch(encode_short_kernel<TFQ_Q_32>); break;
        case TFQ_Q_G_12: launch(encode_short_kernel<TFQ_Q_G_12>); break;
        case TFQ_Q_G_2_K_L: launch(encode_short_kernel<TFQ_Q_G_2_K_L>); break;
        case TFQ_Q_G_3_K_L: launch(encode_short_kernel<TFQ_Q_G_3_K_L>); break;
        case TFQ_Q_G_4_K_L: launch(encode_short_kernel<TFQ_Q_G_4_K_L>); break;
        case TFQ_Q_6_5: launch(encode_short_kernel<TFQ_Q_6_5>); break;
        case TFQ_Q_24: launch(encode_short_kernel<TFQ_Q_24>); break;
        case TFQ_Q_24_5: launch(encode_short_kernel<TFQ_Q_24_5>); break;
        case TFQ_Q_G_24: launch(encode_short_kernel<TFQ_Q_G_24>); break;
        case TFQ_Q_16: launch(encode_short_kernel<TFQ_Q_16>); break;
        case TFQ_Q_16_5: launch(encode_short_kernel<TFQ_Q_16_5>); break;
        case TFQ_Q_G_16: launch(encode_short_kernel<TFQ_Q_G_16>); break;
        case TFQ_Q_1: launch(encode_short_kernel<TFQ_Q_1>); break;
        default: return fail(TFQ_ERR_FORMAT, "encode: wire id " + std::to_string(fmt) + " has no device encoder in this build");
    }
    return hip_fail(hipGetLastError(), "encode launch");
}

int launch_encode(int fmt, const float* w, int64_t nblocks, uint8_t* dst, hipStream_t s, const BlockLayout* short_block) {
    if (nblocks > 0x7FFFFFFF) return fail(TFQ_ERR_SHAPE, "encode: more than 2^31-1 blocks in one call");
    ShortJob job;
    if (int r = short_job(fmt, short_block, w, nblocks, dst, &job)) return r;
    if (nblocks <= 0 && job.L.n <= 0) return TFQ_OK;
    const dim3 grid((unsigned)nblocks), grid4((unsigned)((nblocks + 3) / 4)), block(256);
    if (is_mix(fmt)) {
        if (nblocks > 0) hipLaunchKernelGGL(encode_mix_kernel, grid, dim3(64), 0, s, mix_layout(fmt, 256), w, dst);
        if (job.L.n > 0) hipLaunchKernelGGL(encode_mix_kernel, dim3(1), dim3(64), 0, s, mix_layout(fmt, job.L.n), job.w, job.dst);
        return hip_fail(hipGetLastError(), "encode launch");
    }
    if (job.L.n > 0 && !short_rides_along(fmt)) {
        if (nblocks > 0)
            if (int r = launch_encode(fmt, w, nblocks, dst, s)) return r;
        return launch_encode_short(fmt, job, s);
    }
    switch (canonical(fmt)) {
        case TFQ_Q_32: hipLaunchKernelGGL(encode_raw32_kernel, grid, block, 0, s, w, dst); break;
        case TFQ_B32S4: launch_encode_sym32<TFQ_B32S4>(w, nblocks, dst, job.L.n, s); break;
        case TFQ_B32S8: launch_encode_sym32<TFQ_B32S8>(w, nblocks, dst, job.L.n, s); break;
        case TFQ_Q_G_4: launch_encode_affine<TFQ_Q_G_4>(w, nblocks, dst, job, s); break;
        case TFQ_Q_G_3: launch_encode_affine<TFQ_Q_G_3>(w, nblocks, dst, job, s); break;
        case TFQ_Q_G_2: launch_encode_affine<TFQ_Q_G_2>(w, nblocks, dst, job, s); break;
        case TFQ_SB256A3: launch_encode_affine<TFQ_SB256A3>(w, nblocks, dst, job, s); break;
        case TFQ_SB256A2: launch_encode_affine<TFQ_SB256A2>(w, nblocks, dst, job, s); break;
        case TFQ_Q_1_5: launch_encode_affine<TFQ_Q_1_5>(w, nblocks, dst, job, s); break;
        case TFQ_Q_G_8:
            if (nblocks * 8 > 0x7FFFFFFF) return fail(TFQ_ERR_SHAPE, "encode: too many groups in one call");
            launch_encode_comp8<TFQ_Q_G_8>(w, nblocks, dst, 1.0f, job, s);
            if (const int tier = tier_of(fmt)) {
                // :2756-2772: scaled copies of every group's fitted scale, the last two for _K_M, all six for _K_H
                const TierTry tries[6] = {{0, 0.7f}, {0, 0.9f}, {0, 0.95f}, {0, 1.05f}, {0, 1.1f}, {0, 1.3f}};
                const int count = tier >= 2 ? 6 : 2;
                const int rc = encode_tiers<TFQ_Q_G_8>(tries + 6 - count, count, w, nblocks, dst, s, [&](uint8_t* out, int, float smult) {
                    launch_encode_comp8<TFQ_Q_G_8>(w, nblocks, out, smult, ShortJob{}, s);
                });
                if (rc != TFQ_OK) return rc;
            }
            break;
        case TFQ_Q_8:
            launch_encode_comp8<TFQ_Q_8>(w, nblocks, dst, 1.0f, job, s);
            if (tier_of(fmt) >= 2) {
                // :2627-2645: the tries with smult 1 repeat the base payload (the 8-bit fit takes no iteration
                // count), so _K_M equals _K_L and _K_H has four scaled tries
                const TierTry tries[4] = {{0, 0.9f}, {0, 1.1f}, {0, 0.7f}, {0, 1.3f}};
                const int rc = encode_tiers<TFQ_Q_8>(tries, 4, w, nblocks, dst, s, [&](uint8_t* out, int, float smult) {
                    launch_encode_comp8<TFQ_Q_8>(w, nblocks, out, smult, ShortJob{}, s);
                });
                if (rc != TFQ_OK) return rc;
            }
            break;
        case TFQ_Q_4: { const int rc = encode_lattice_family<TFQ_Q_4>(fmt, w, nblocks, dst, job, s); if (rc != TFQ_OK) return rc; break; }
        case TFQ_Q_2: { const int rc = encode_lattice_family<TFQ_Q_2>(fmt, w, nblocks, dst, job, s); if (rc != TFQ_OK) return rc; break; }
        case TFQ_Q_3: { const int rc = encode_lattice_family<TFQ_Q_3>(fmt, w, nblocks, dst, job, s); if (rc != TFQ_OK) return rc; break; }
        case TFQ_Q_6: { const int rc = encode_lattice_family<TFQ_Q_6>(fmt, w, nblocks, dst, job, s); if (rc != TFQ_OK) return rc; break; }
        case TFQ_Q_12: { const int rc = encode_lattice_family<TFQ_Q_12>(fmt, w, nblocks, dst, job, s); if (rc != TFQ_OK) return rc; break; }
        case TFQ_Q_G_12: {
            auto launch = [&](uint8_t* out, int iters, float smult) {
                hipLaunchKernelGGL(encode_grp12_kernel, grid, dim3(64), 0, s, w, out, iters, smult);
            };
            launch(dst, 3, 1.0f);
            // :2788-2810; the second try repeats the first
            const TierTry tries[5] = {{8, 1.0f}, {20, 0.93f}, {20, 1.07f}, {20, 0.7f}, {20, 1.3f}};
            const int tier = tier_of(fmt);
            const int rc = encode_tiers<TFQ_Q_G_12>(tries, tier >= 2 ? 5 : tier, w, nblocks, dst, s, launch);
            if (rc != TFQ_OK) return rc;
            break;
        }
        case TFQ_Q_G_2_K_L: hipLaunchKernelGGL(encode_grp16_kernel<TFQ_Q_G_2_K_L>, grid, dim3(64), 0, s, w, dst); break;
        case TFQ_Q_G_3_K_L: hipLaunchKernelGGL(encode_grp16_kernel<TFQ_Q_G_3_K_L>, grid, dim3(64), 0, s, w, dst); break;
        case TFQ_Q_G_4_K_L: hipLaunchKernelGGL(encode_grp16_kernel<TFQ_Q_G_4_K_L>, grid, dim3(64), 0, s, w, dst); break;
        case TFQ_Q_6_5: hipLaunchKernelGGL(encode_grp16_kernel<TFQ_Q_6_5>, grid, dim3(64), 0, s, w, dst); break;
        case TFQ_Q_G_6:
            // the _K_M / _K_H tiers re-run the search with more effort and keep the better candidate by decoded
            // error (src/codec/block_codec.cpp:2733-2755); that selection is not on the device
            hipLaunchKernelGGL(encode_q6k_kernel, dim3(grid4.x + (job.L.n > 0)), dim3(64), 0, s, w, dst, 4, 3, 3, nblocks, job);
            if (nblocks > 0 && (fmt == TFQ_Q_G_6_K_M || fmt == TFQ_Q_G_6_K_H)) {
                // longer searches, each kept only where it decodes strictly better (src/codec/block_codec.cpp:2733-2755)
                uint8_t* cand = nullptr;
                TFQ_HIP(hipMalloc(&cand, (size_t)nblocks * 210));
                const int effort[2][3] = {{8, 5, 6}, {14, 8, 10}};
                for (int c = 0; c < (fmt == TFQ_Q_G_6_K_H ? 2 : 1); ++c) {
                    hipLaunchKernelGGL(encode_q6k_kernel, grid4, dim3(64), 0, s, w, cand, effort[c][0], effort[c][1], effort[c][2], nblocks, ShortJob{});
                    hipLaunchKernelGGL(keep_better_kernel<TFQ_Q_G_6>, grid, dim3(64), 0, s, w, dst, (const uint8_t*)cand);
                }
                const hipError_t e1 = hipStreamSynchronize(s);
                (void)hipFree(cand);
                if (e1 != hipSuccess) return hip_fail(e1, "hipStreamSynchronize");
            }
            break;
        case TFQ_Q_24: hipLaunchKernelGGL(encode_wide_kernel<TFQ_Q_24>, grid, block, 0, s, w, dst); break;
        case TFQ_Q_24_5: hipLaunchKernelGGL(encode_wide_kernel<TFQ_Q_24_5>, grid, block, 0, s, w, dst); break;
        case TFQ_Q_G_24: hipLaunchKernelGGL(encode_wide_kernel<TFQ_Q_G_24>, grid, block, 0, s, w, dst); break;
        case TFQ_Q_16: hipLaunchKernelGGL(encode_wide_kernel<TFQ_Q_16>, grid, block, 0, s, w, dst); break;
        case TFQ_Q_16_5: hipLaunchKernelGGL(encode_wide_kernel<TFQ_Q_16_5>, grid, block, 0, s, w, dst); break;
        case TFQ_Q_G_16: hipLaunchKernelGGL(encode_wide_kernel<TFQ_Q_G_16>, grid, block, 0, s, w, dst); break;
        case TFQ_Q_1: {
            const int tier = fmt == TFQ_Q_1 ? -1 : (fmt == TFQ_Q_1_K_M || fmt == TFQ_Q_G_1_K_M) ? 1
                             : (fmt == TFQ_Q_1_K_H || fmt == TFQ_Q_G_1_K_H) ? 2 : 0;
            hipLaunchKernelGGL(encode_q1_kernel, grid, block, 0, s, w, dst, tier);
            break;
        }
        default:
            return fail(TFQ_ERR_FORMAT, "encode: wire id " + std::to_string(fmt) +
                                            " has no device encoder in this build");
    }
    return hip_fail(hipGetLastError(), "encode launch");
}

}  // namespace tfq
