// Prefill products whose weights may not be rounded: Y[m][n] = sum_k X[m][k] * W[n][k] for tall X (M > 16) on the
// matrix cores with integer operands.  Serves fp32 activations on the Tiled16 formats, the 16-weight-group formats
// (Q_G_2, SB256A3, SB256A2) and the two formats kept in wire layout that a prompt meets (Q_4, Q_G_6).
// Replaces Qwen35Engine::gemm for those (src/adapters/tools/qwen35_engine.cpp:54-101), which decodes a block to fp32
// and accumulates in fp32.
//
// Every weight of a block is  scale * I + offset  with an integer I that one or two bf16 numbers hold exactly, so a
// bf16 MFMA with fp32 accumulation multiplies the integers without any rounding of the weight; scales are applied to
// the sums in fp32:
//   Q_G_4, Q_G_3          I = code,            scale d sc / top per 32 weights, offset -dm mc per 32
//   B32S4, B32S8          I = code - 8 / 128,  scale per 32
//   Q_G_8, Q_8            I = 2 code - 255,    scale per 32 (the line that stands for the companded grid)
//   Q_G_2, SB256A2        I = sc code <= 189,  scale d / 3 per 256,             offset -dm mc per 16
//   SB256A3               I = sc (code - 4),   scale d / 7 per 256,             offset 4 sc d / 7 - dm mc per 16
//   Q_4                   I = 10^4 level (14 bits and sign, two bf16), scale per 256
//   Q_G_6                 I = sc (code - 32)   (13 bits, two bf16),    scale d per 256
// (of the last two the operands are I 2^-23 and I 2^-20, so that no sum of 256 leaves the range before its scale; of
// the three formats above them, and of their offsets, the integers times 2^-6: as plain integers the sums of 256 left
// the range one power of two before those of the decode kernels, which scale sums of 16; now 3 to 7 powers after them)
// bf16 activations are exact operands.  fp32 activations go in as a bf16 high part and the bf16 of the rest (two
// operands, the 16 bits that the decode kernels keep too), for the wire formats, whose other kernel multiplies in
// fp32, as three (24 bits).  The offsets times the activations' group sums are a product of their own, one MFMA per
// block: its 32 K-slots hold the group sums as three bf16 parts (24 bits) against the integers mc (and sc).
//
// A workgroup of four wavefronts owns 128 tokens x 128 weight rows and walks K in steps of 32, both operands staged
// in LDS (two buffers, one barrier per step); a wavefront multiplies 64 x 64.  What bounds it is vector issue next
// to the MFMAs (splitting activations, decoding codes, the scale's multiply-adds; counted on 333 fp32 rows of Q_G_4
// 4096 x 14336: 245 vector instructions, 38 of them MFMAs, per wavefront and step, vector issue busy for 52 % of the
// cycles, the matrix cores for 33 %, LDS for 34 %; SB256A3 with bf16 rows 123 / 26, 39, 33 and 38 %), so two workgroups
// share a compute unit (LDS <= 80 KB, <= 256 registers): one's staging runs under the other's MFMAs.  256-row tiles with one workgroup per unit would stage less per product,
// but a ragged prompt (333 rows) then pads to 512 rows instead of 384.  Activations are fetched two steps ahead, codes
// three.  Few rows take 64-row tiles, three workgroups per unit.
// Measured, before (slices of 4 to 16 rows through the decode kernels) and now: Q_G_4 fp32 333 rows 4096 x 14336
// 657 -> 146 us, B32S8 the same 700 -> 133 us; 512 bf16 rows of 14336 x 4096: Q_4 7580 -> 189 us, Q_G_6 5360 -> 184 us,
// SB256A3 789 -> 141 us.  Up to 16 rows tfq_gemv's kernels serve every format, above that the faster of the two
// by a model (exact_cheaper).  For the wire formats the step at 17 rows is where the entry points part,
// not where the kernels cross: 14336 x 4096 bf16 Q_4 takes 93 us at 16 rows (four passes) and 40 us at 17 to 24 rows here,
// Q_G_6 90 and 45 us; at 1024 x 4096 the two meet (16 us).  The Tiled16 formats cross between 16 and 20 rows.

#include <algorithm>
#include <atomic>
#include <cmath>

#include "tfq_decode.hpp"
#include "tfq_gemm_decode.hpp"

namespace tfq {

namespace {

constexpr float kSumScale = 64.0f;  // the 16-weight-group formats' operands are divided by it (see above), their scales multiplied
constexpr int TN = 128, THREADS = 256;  // tokens of a tile: a template parameter, 128 or 64

template <int FMT>
struct Form {
    static constexpr bool WIRE = FMT == TFQ_Q_4 || FMT == TFQ_Q_G_6;
    static constexpr bool BYTES = tiled_header_in_bytes(FMT);  // sixteen groups of 16, header one code per byte
    static constexpr bool BLOCK_SCALE = WIRE || BYTES;         // the sums of a block of 256 stay unscaled until its end
    static constexpr int WP = WIRE ? 2 : 1;                    // bf16 operands per weight
    static constexpr int OG = BYTES ? 16 : (FMT == TFQ_Q_G_4 || FMT == TFQ_Q_G_3) ? 8 : 0;  // offset groups per block
    static constexpr bool SC_OFFSET = FMT == TFQ_SB256A3;      // the centred codes bring a second offset product
    static constexpr int RAW = WIRE ? 3 : FMT == TFQ_Q_G_2 || FMT == TFQ_SB256A2 ? 1 : 2 * tiled_planes(FMT);  // code dwords per thread and step
};

struct ExactArgs {
    const uint8_t* W;
    const void* X;
    void* Y;
    float* partial;  // [ksplit][M][N] when ksplit > 1
    int M, N, K;
    int y_bf16;
    int tiles_m, tiles_n, ksplit;
};

__device__ __forceinline__ uint32_t pk(float lo, float hi) { return pack_bf16(lo, hi); }
__device__ __forceinline__ float bf_lo(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float bf_hi(uint32_t v) { return __uint_as_float(v & 0xFFFF0000u); }

// ---- Q_4: level = +-L / 10^4, L = 1260 ... 27178; two bf16 numbers hold L exactly
struct Q4Table {
    uint32_t hi_b[2], hi_t[2], lo_b[2], lo_t[2];  // low / high bytes of the two parts, entry m in byte m % 4 of word m / 4
};
constexpr uint32_t bf16_of_int(int v) {  // v 2^-23, exact: at most eight significant bits
    if (v == 0) return 0;
    const uint32_t sign = v < 0 ? 0x8000u : 0u;
    uint32_t m = v < 0 ? (uint32_t)-v : (uint32_t)v;
    int e = 0;
    while ((m >> e) > 1) ++e;
    const uint32_t frac = e >= 7 ? (m >> (e - 7)) : (m << (7 - e));
    return sign | ((uint32_t)(127 - 23 + e) << 7) | (frac & 0x7Fu);
}
constexpr Q4Table make_q4_table() {
    constexpr int L[8] = {1260, 3976, 6508, 9275, 12392, 15995, 20522, 27178};
    Q4Table t{};
    for (int m = 0; m < 8; ++m) {
        int e = 0;
        while ((L[m] >> e) > 1) ++e;
        const int hi = ((L[m] + (1 << (e - 8))) >> (e - 7)) << (e - 7), lo = L[m] - hi;  // |lo| <= 2^(e - 8) <= 2^6
        const uint32_t h = bf16_of_int(hi), l = bf16_of_int(lo);
        t.hi_b[m / 4] |= (h & 255u) << (8 * (m % 4));
        t.hi_t[m / 4] |= (h >> 8) << (8 * (m % 4));
        t.lo_b[m / 4] |= (l & 255u) << (8 * (m % 4));
        t.lo_t[m / 4] |= (l >> 8) << (8 * (m % 4));
    }
    return t;
}

// four codes, one per byte -> the two bf16 parts as dwords (codes 0, 1) and (2, 3): the magnitudes are byte look-ups
// by v_perm_b32 (level 15 - i is minus level i), the sign goes onto the high bytes
__device__ __forceinline__ void q4_levels(uint32_t q, uint32_t (&hi)[2], uint32_t (&lo)[2]) {
    constexpr Q4Table T = make_q4_table();
    const uint32_t neg = (q & 0x08080808u) ^ 0x08080808u;          // 8 where the level is negative
    const uint32_t sel = (q & 0x07070707u) ^ (neg - (neg >> 3));   // 7 - (q & 7) there
    const uint32_t sgn = neg << 4;
    const uint32_t hb = __builtin_amdgcn_perm(T.hi_b[1], T.hi_b[0], sel), ht = __builtin_amdgcn_perm(T.hi_t[1], T.hi_t[0], sel) ^ sgn;
    const uint32_t lb = __builtin_amdgcn_perm(T.lo_b[1], T.lo_b[0], sel), lt = __builtin_amdgcn_perm(T.lo_t[1], T.lo_t[0], sel) ^ sgn;
    hi[0] = __builtin_amdgcn_perm(ht, hb, 0x05010400u);
    hi[1] = __builtin_amdgcn_perm(ht, hb, 0x07030602u);
    lo[0] = __builtin_amdgcn_perm(lt, lb, 0x05010400u);
    lo[1] = __builtin_amdgcn_perm(lt, lb, 0x07030602u);
}

// sixteen 2-bit codes of the true-width layout -> I = sc * code / kSumScale as bf16, in order (C: see f16_bias)
__device__ __forceinline__ void decode16x2(uint32_t v, float sc, uint32_t C, uint4& o0, uint4& o1) {
    const float c2 = -16.0f * sc;
    uint32_t o[8];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        float w[8];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const f16x2_t p = __builtin_bit_cast(f16x2_t, ((v >> (2 * (t + 4 * j))) & 0x00030003u) | C);
            w[t] = __builtin_fmaf(sc, (float)p.x, c2);
            w[t + 4] = __builtin_fmaf(sc, (float)p.y, c2);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) o[4 * j + t] = pk(w[2 * t], w[2 * t + 1]);
    }
    o0 = uint4{o[0], o[1], o[2], o[3]};
    o1 = uint4{o[4], o[5], o[6], o[7]};
}

__device__ __forceinline__ bool finite_f32(float v) { return (__float_as_uint(v) & 0x7F800000u) != 0x7F800000u; }

// An infinite activation meets two parts of a weight here, which may differ in sign or be zero, and gives a NaN where
// the fp32 product gives an infinity.  Where outputs of the wire formats (whose other kernel multiplies in fp32) are
// not finite, the wavefront looks the activation row over: a NaN makes the output a NaN; else the infinities alone
// decide, by the signs of their weights (and stop as soon as every output is a NaN); fp32 values that round to an
// infinite bf16 part have their outputs formed again weight by weight.  All 64 lanes call this together.
template <int FMT, int XP>
__device__ __attribute__((noinline)) float repair_non_finite(const uint8_t* W, const void* X, int K, int m, int col, bool valid, float v) {
    const int nblk = K >> 8, lane = threadIdx.x & 63;
    constexpr int BB = spec_of(FMT).block_bytes;
    const bool flag = valid && !finite_f32(v);
    auto value = [&](int row, int k) {
        return XP == 1 ? __uint_as_float((uint32_t)static_cast<const unsigned short*>(X)[(size_t)row * K + k] << 16)
                       : static_cast<const float*>(X)[(size_t)row * K + k];
    };
    auto weight = [&](int k) { return decode_weight<FMT>(W + ((size_t)col * nblk + (k >> 8)) * BB, (uint32_t)(k & 255)); };
    uint64_t todo = __ballot(flag);
    while (todo) {
        const int row = __builtin_amdgcn_readlane(m, __builtin_ctzll(todo));
        const bool mine = flag && m == row;
        todo &= ~__ballot(mine);
        bool nan = false, inf = false, huge = false;
        for (int k = lane; k < K; k += 64) {
            const uint32_t u = __float_as_uint(value(row, k)) & 0x7FFFFFFFu;
            nan |= u > 0x7F800000u;
            inf |= u == 0x7F800000u;
            huge |= u >= 0x7F7F8000u && u < 0x7F800000u;
        }
        if (__ballot(nan)) {
            if (mine) v = __uint_as_float(0x7FC00000u);
        } else if (__ballot(inf)) {
            float r = 0.0f;
            for (int k0 = 0; k0 < K && __ballot(mine && r == r); k0 += 64) {
                const float xv = value(row, k0 + lane);
                uint64_t at = __ballot(!finite_f32(xv));
                while (at) {
                    const int p = __builtin_ctzll(at);
                    at &= at - 1;
                    const float xi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(xv), p));
                    if (mine) r += weight(k0 + p) * xi;
                }
            }
            if (mine) v = r;
        } else if (__ballot(huge)) {
            if (mine) {
                float r = 0.0f;
                for (int k = 0; k < K; ++k) r = __builtin_fmaf(weight(k), value(row, k), r);
                v = r;
            }
        }
    }
    return v;
}

template <int FMT, int XP, int TM>
constexpr int lds_uint4s() {
    using F = Form<FMT>;
    return 2 * XP * TM * 4 + 2 * F::WP * 512 + (F::OG == 16 ? 6 * TM + 512 * (F::SC_OFFSET ? 2 : 1) : F::OG == 8 ? 3 * TM + 256 : 0) + 64 + (F::OG ? 64 : 0);
}

template <int FMT, int XP, int TM>
__global__ __launch_bounds__(THREADS, TM == 128 || XP == 3 ? 2 : 3) void gemm_exact_kernel(ExactArgs args) {
    using F = Form<FMT>;
    constexpr int WP = F::WP, OG = F::OG, UB = F::WIRE ? spec_of(FMT).block_bytes : tiled_unit_bytes(FMT);
    constexpr int MI = TM / 32, NJ = 4, XPL = TM * 4;  // XPL: 16-byte pieces of an activation part in LDS
    extern __shared__ uint4 smem[];
    uint4* const xs = smem;                      // [2][XP][TM rows x 4 pieces]
    uint4* const wsm = xs + 2 * XP * XPL;        // [2][WP][128 rows x 4 pieces]
    uint4* const sums = wsm + 2 * WP * 512;      // group sums of a block, three bf16 parts: [row][3 x 8 groups] or [row][6 x 8]
    uint4* const mcs = sums + (OG == 16 ? 6 * TM : OG == 8 ? 3 * TM : 0);           // [2] offset integers of a block, bf16
    uint4* const scs = mcs + (OG == 16 ? 512 : OG == 8 ? 256 : 0);              // [2] the scale integers where they are an offset too
    float* const wscale = reinterpret_cast<float*>(scs + (F::SC_OFFSET ? 512 : 0));  // [2][128], per step or per block
    float* const woff = wscale + 256;            // [2][128] dm

    const int M = args.M, N = args.N, K = args.K, S = args.ksplit;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // as in the other tile kernel: an XCD gets a contiguous run of the token-tile-major list, so that the workgroups
    // running together on it read the same activations through its L2
    const int items = args.tiles_m * args.tiles_n * S, per_xcd = (items + 7) >> 3;
    const int item = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || item >= items) return;
    const int tms = item / args.tiles_n, strip = item - tms * args.tiles_n;
    const int tm = tms / S, split = __builtin_amdgcn_readfirstlane(tms - tm * S);
    const int m0 = tm * TM, n0 = strip * TN;
    const int nblocks = K >> 8;
    const int blk0 = (int)((long)split * nblocks / S), blk1 = (int)((long)(split + 1) * nblocks / S);

    // staging of the weights: a thread takes 16 of a row's 32 K-slots; eight consecutive threads take eight rows of one
    // half, whose LDS slots are consecutive
    const int row = (tid & 7) | ((tid >> 4) << 3), half = (tid >> 3) & 1;
    const int wslot = ((row >> 3) << 5) + (half << 4) + (row & 7);  // piece 2 half; + 8 for the next piece
    // K order of a step: the Tiled16 formats take 32 consecutive weights; the wire formats 16 of the block's first half and
    // 16 of the second, so that a thread stays in one half of its block's bit stream
    const int wtile = F::WIRE ? min(n0 + row, N - 1) - n0 : min((n0 + row) >> 4, ((N + 15) >> 4) - 1) - (n0 >> 4);
    const uint8_t* const wbase = args.W + (size_t)(F::WIRE ? n0 : n0 >> 4) * nblocks * UB;
    const uint32_t woffs = (uint32_t)wtile * (uint32_t)nblocks * UB;  // below 4 GiB: K is at most 2^22
    const int r16 = (n0 + row) & 15;
    // staging of the activations: 16-byte pieces, adjacent threads take adjacent pieces of a row (64 bytes of
    // a row per thread, every lane on a line of its own: B32S8 fp32 333 x 4096 x 14336 144 us against 133 us).
    // LDS slot of (row, piece of eight values): row * 4 + (piece ^ row / 2 % 4), free of bank conflicts both ways.
    constexpr int XE = XP == 1 ? 2 : 4, TPR = XP == 1 ? 4 : 8, RPP = THREADS / TPR, XC = TM / RPP;
    const int xrow0 = tid / TPR, xpiece = tid % TPR;
    const uint8_t* const xbase = static_cast<const uint8_t*>(args.X) + (size_t)m0 * K * XE;
    uint32_t xoff[XC];
#pragma unroll
    for (int i = 0; i < XC; ++i)
        xoff[i] = (uint32_t)(((uint32_t)(min(m0 + xrow0 + i * RPP, M - 1) - m0) * (uint32_t)K + (F::WIRE ? (xpiece / (TPR / 2)) * 128 + (xpiece % (TPR / 2)) * (16 / XE) : xpiece * (16 / XE))) * XE);
    // (RPP is a multiple of 8: the swizzle is the same for all of a thread's rows)
    const int xslot = XP == 1 ? xrow0 * 4 + (xpiece ^ ((xrow0 >> 1) & 3)) : xrow0 * 4 + ((xpiece >> 1) ^ ((xrow0 >> 1) & 3));

    u32x4_t xr[2][XC];        // the activations of the next step and of the one after it
    uint32_t raw[4][F::RAW];  // ring: set r holds the code dwords of a step with index % 4 == r
    uint4 hdr = {0, 0, 0, 0}, hnext = {0, 0, 0, 0}, hmc = {0, 0, 0, 0};
    uint32_t hdd = 0;

    auto load_x = [&]<int U>(int blk) __attribute__((always_inline)) {
        const uint8_t* p = xbase + ((size_t)blk * 256 + (F::WIRE ? 16 : 32) * U) * XE;
#pragma unroll
        for (int i = 0; i < XC; ++i) xr[U & 1][i] = *reinterpret_cast<const u32x4_t*>(p + xoff[i]);
    };
    auto load_w = [&]<int U>(int blk) __attribute__((always_inline)) {
        const uint8_t* p = wbase + (size_t)blk * UB + woffs;
        uint32_t(&r)[F::RAW] = raw[U & 3];
        if constexpr (FMT == TFQ_Q_4) {
            // 63 bits from bit 16 + 63 (U + 8 half): inside three dwords; the block's last 63 bits end with its dword 31
            constexpr int d0 = (16 + 63 * U) >> 5, d1 = (520 + 63 * U) >> 5;
            const uint32_t* q = reinterpret_cast<const uint32_t*>(p) + (half ? (d1 < 29 ? d1 : 29) : d0);
#pragma unroll
            for (int i = 0; i < 3; ++i) r[i] = q[i];
        } else if constexpr (FMT == TFQ_Q_G_6) {
            // 96 bits; a block starts at an even address
            const unsigned short* q = reinterpret_cast<const unsigned short*>(p + 96 * half + 12 * U);
            __builtin_memcpy(r, __builtin_assume_aligned(q, 2), 12);
        } else if constexpr (tiled_code_width(FMT) == 2) {
            r[0] = *reinterpret_cast<const uint32_t*>(p + (r16 + 16 * (U & 3)) * 16 + (2 * (U >> 2) + half) * 4);
        } else {
            const uint8_t* q = p + (U >> 2) * 1024 + (U & 3) * 256 + 16 * r16 + 8 * half;
            const uint2 a = *reinterpret_cast<const uint2*>(q);
            r[0] = a.x; r[1] = a.y;
            if constexpr (F::RAW == 4) {
                const uint2 b = *reinterpret_cast<const uint2*>(q + 2048);
                r[2] = b.x; r[3] = b.y;
            }
        }
    };
    auto load_hdr = [&](int blk) __attribute__((always_inline)) {
        const uint8_t* p = wbase + (size_t)blk * UB + woffs;
        if constexpr (FMT == TFQ_Q_4) {
            hdd = *reinterpret_cast<const uint16_t*>(p);
        } else if constexpr (FMT == TFQ_Q_G_6) {
            __builtin_memcpy(&hnext, __builtin_assume_aligned(p + 192 + 8 * half, 2), 8);
            hdd = *reinterpret_cast<const uint16_t*>(p + 208);
        } else if constexpr (F::BYTES) {
            hnext = *reinterpret_cast<const uint4*>(p + tiled_header_offset(FMT, r16, 0));
            hmc = *reinterpret_cast<const uint4*>(p + tiled_header_offset(FMT, r16, 1));
            hdd = *reinterpret_cast<const uint32_t*>(p + tiled_header_offset(FMT, r16, 2));
        } else {
            hnext = *reinterpret_cast<const uint4*>(p + tiled_header_offset(FMT, r16, 0));
        }
    };
    // f16_bias: OR-ed under a code n it makes the binary16 number 1024 + n, of the 16-weight-group formats 16 + n / 64,
    // which divides their operands without an operation (a multiplication of sc: SB256A3 142 -> 144 us, 512 x 14336 x 4096)
    static_assert(kSumScale == 64.0f);
    uint32_t nib_mask = 0x000F000Fu, f16_bias = F::BYTES ? 0x4C004C00u : 0x64006400u;
    float one = 1.0f;
    asm volatile("" : "+v"(nib_mask), "+v"(f16_bias), "+v"(one));  // kept in registers (see decode8); a literal 1 would split its mixed multiply-add

    // stage step U (its loads have been issued) into buffer U & 1; par: parity of its block, for what a block has once
    auto stage = [&]<int U>(int par) __attribute__((always_inline)) {
        uint4* const wd = wsm + (U & 1) * WP * 512 + wslot;
#pragma unroll
        for (int i = 0; i < XC; ++i) {
            const u32x4_t v = xr[U & 1][i];
            uint4* const xd = xs + (U & 1) * XP * XPL + xslot + i * RPP * 4;
            if constexpr (XP == 1) {
                if constexpr (FMT == TFQ_Q_4) {  // order 0 2 4 6 1 3 5 7, as q4_levels leaves the weights
                    uint4 o;
                    o.x = __builtin_amdgcn_perm(v[1], v[0], 0x05040100u);
                    o.y = __builtin_amdgcn_perm(v[3], v[2], 0x05040100u);
                    o.z = __builtin_amdgcn_perm(v[1], v[0], 0x07060302u);
                    o.w = __builtin_amdgcn_perm(v[3], v[2], 0x07060302u);
                    *xd = o;
                } else {
                    *xd = uint4{v[0], v[1], v[2], v[3]};
                }
            } else {
                float f[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) f[t] = __uint_as_float(v[t]);
#pragma unroll
                for (int p = 0; p < XP; ++p) {
                    uint32_t o[2];
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const int a = FMT == TFQ_Q_4 ? t : 2 * t, b = FMT == TFQ_Q_4 ? a + 2 : a + 1;
                        o[t] = pk(f[a], f[b]);
                        if (p + 1 < XP) {
                            f[a] -= bf_lo(o[t]);
                            f[b] -= bf_hi(o[t]);
                        }
                    }
                    uint32_t* const d = reinterpret_cast<uint32_t*>(xd + p * XPL);
                    if constexpr (FMT == TFQ_Q_4) {  // values 0..3 of the eight: dwords (0, 2) and (1, 3); 4..7: one dword on
                        d[xpiece & 1] = o[0];
                        d[2 + (xpiece & 1)] = o[1];
                    } else {
                        *reinterpret_cast<uint2*>(d + 2 * (xpiece & 1)) = uint2{o[0], o[1]};
                    }
                }
            }
        }
        // ---- weights
        const uint32_t(&r)[F::RAW] = raw[U & 3];
        if constexpr (U == 0) hdr = hnext;
        if constexpr (FMT == TFQ_Q_4) {
            constexpr int d0 = (16 + 63 * U) >> 5, s0 = (16 + 63 * U) & 31, d1 = (520 + 63 * U) >> 5, s1 = (520 + 63 * U) & 31;
            uint32_t a = r[0], b = r[1], c = r[2];
            if constexpr (d1 > 29) {
                if (half) { a = b; b = c; c = 0; }
            }
            (void)d0;
            const uint32_t sh = half ? s1 : s0;
            const uint32_t v0 = __builtin_amdgcn_alignbit(b, a, sh);
            uint32_t v1 = __builtin_amdgcn_alignbit(c, b, sh);
            v1 = (v1 & 0x0FFFFFFFu) | ((v1 << 1) & 0xE0000000u);  // the sixteenth code has three bits, an even level
            const uint32_t q[4] = {v0 & 0x0F0F0F0Fu, (v0 >> 4) & 0x0F0F0F0Fu, v1 & 0x0F0F0F0Fu, (v1 >> 4) & 0x0F0F0F0Fu};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint32_t eh[2], el[2], oh[2], ol[2];
                q4_levels(q[2 * h], eh, el);
                q4_levels(q[2 * h + 1], oh, ol);
                wd[8 * h] = uint4{eh[0], eh[1], oh[0], oh[1]};
                wd[512 + 8 * h] = uint4{el[0], el[1], ol[0], ol[1]};
            }
            // the scale takes 10^-4 in one rounding
            if constexpr (U == 0) wscale[par * 128 + row] = (float)((double)half_bits_to_float(hdd) * (8388608.0 * 1e-4));
        } else if constexpr (FMT == TFQ_Q_G_6) {
            const uint32_t scw = U < 4 ? hdr.x : hdr.y;
            const float sc = (float)((int32_t)(scw << (24 - 8 * (U & 3))) >> 24) * (1.0f / 1048576.0f), c = -32.0f * sc;
            uint32_t hi[8], lo[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                float w[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int pos = 6 * (2 * t + e), i = pos >> 5, s = pos & 31;
                    uint32_t code = r[i] >> s;
                    if (s > 26) code = __builtin_amdgcn_alignbit(r[i + 1 < 3 ? i + 1 : 2], r[i], s);
                    w[e] = __builtin_fmaf(sc, (float)(code & 63u), c);  // exact
                }
                hi[t] = pk(w[0], w[1]);
                lo[t] = pk(w[0] - bf_lo(hi[t]), w[1] - bf_hi(hi[t]));  // exact
            }
            wd[0] = uint4{hi[0], hi[1], hi[2], hi[3]};
            wd[8] = uint4{hi[4], hi[5], hi[6], hi[7]};
            wd[512] = uint4{lo[0], lo[1], lo[2], lo[3]};
            wd[520] = uint4{lo[4], lo[5], lo[6], lo[7]};
            if constexpr (U == 0) wscale[par * 128 + row] = half_bits_to_float(hdd) * 1048576.0f;
        } else if constexpr (F::BYTES) {
            const uint32_t scw = (U >> 1) == 0 ? hdr.x : (U >> 1) == 1 ? hdr.y : (U >> 1) == 2 ? hdr.z : hdr.w;
            const float sc = (float)((scw >> (16 * (U & 1) + 8 * half)) & 255u);
            if constexpr (tiled_code_width(FMT) == 2) {
                uint4 o0, o1;
                decode16x2(r[0], sc, f16_bias, o0, o1);
                wd[0] = o0;
                wd[8] = o1;
            } else {
                // decode8 takes 1024 sc off its addend: -(16 + 4 / 64) sc is left, exactly
                wd[0] = decode8(r[0], sc, (1024.0f - 16.0f - 4.0f / kSumScale) * sc, nib_mask, f16_bias);
                wd[8] = decode8(r[1], sc, (1024.0f - 16.0f - 4.0f / kSumScale) * sc, nib_mask, f16_bias);
            }
            if constexpr (U == 0) {
                constexpr Spec sp = spec_of(FMT);
                constexpr float bias = (float)((1 << sp.mb) / 2);
                auto ints = [&](uint32_t w0, uint32_t w1, float b, float s) {  // eight codes -> s * code + b as bf16
                    uint4 o;
                    o.x = pk(__builtin_fmaf(s, (float)(w0 & 255u), b), __builtin_fmaf(s, (float)((w0 >> 8) & 255u), b));
                    o.y = pk(__builtin_fmaf(s, (float)((w0 >> 16) & 255u), b), __builtin_fmaf(s, (float)(w0 >> 24), b));
                    o.z = pk(__builtin_fmaf(s, (float)(w1 & 255u), b), __builtin_fmaf(s, (float)((w1 >> 8) & 255u), b));
                    o.w = pk(__builtin_fmaf(s, (float)((w1 >> 16) & 255u), b), __builtin_fmaf(s, (float)(w1 >> 24), b));
                    return o;
                };
                mcs[par * 256 + half * 128 + row] = ints(half ? hmc.z : hmc.x, half ? hmc.w : hmc.y, bias / kSumScale, -1.0f / kSumScale);
                if constexpr (F::SC_OFFSET) scs[par * 256 + half * 128 + row] = ints(half ? hdr.z : hdr.x, half ? hdr.w : hdr.y, 0.0f, 4.0f / kSumScale);
                wscale[par * 128 + row] = half_fast(hdd & 0xFFFFu) * (sp.bits == 3 ? 1.0f / 7.0f : 1.0f / 3.0f) * kSumScale;
                woff[par * 128 + row] = half_fast(hdd >> 16) * kSumScale;
            }
        } else {
            float a, c;
            group_coeffs<FMT>(hdr, U, a, c);
            if constexpr (tiled_planes(FMT) == 1) {
                constexpr float c0 = FMT == TFQ_B32S4 ? -8.0f : 0.0f;
                wd[0] = decode8(r[0], one, c0, nib_mask, f16_bias);
                wd[8] = decode8(r[1], one, c0, nib_mask, f16_bias);
            } else {
                constexpr float s = FMT == TFQ_B32S8 ? 1.0f : 2.0f, c0 = FMT == TFQ_B32S8 ? -128.0f : -255.0f;
                wd[0] = decode8x2(r[0], r[2], s, c0);
                wd[8] = decode8x2(r[1], r[3], s, c0);
                if constexpr (FMT != TFQ_B32S8) a *= 0.5f;
            }
            // (the halves hold the same value; without the offsets' longer step one write of it is the faster form:
            // B32S8 133 against 137 us, Q_G_4 172 against 171 us, fp32 333 x 4096 x 14336)
            if (OG > 0 || half == 0) wscale[(U & 1) * 128 + row] = a;
            if constexpr (U == 0 && OG == 8) {
                // the 6-bit offset codes of the eight groups, 32 - code
                const uint64_t mw = (uint64_t)(hdr.y >> 16) | ((uint64_t)hdr.z << 16);
                uint32_t o[4];
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    o[t] = pk(32.0f - (float)(uint32_t)((mw >> (12 * t)) & 63u), 32.0f - (float)(uint32_t)((mw >> (12 * t + 6)) & 63u));
                mcs[par * 128 + row] = uint4{o[0], o[1], o[2], o[3]};
                woff[par * 128 + row] = half_fast(hdr.w >> 16);
            }
        }
    };

    const int wm = wave >> 1, wn_ = wave & 1, fr = lane & 15, fk = lane >> 4;
    const f32x4_t zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4_t acc[MI][NJ], blk_acc[F::BLOCK_SCALE ? MI : 1][F::BLOCK_SCALE ? NJ : 1];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = zero4;
    auto mm = [](uint4 a, uint4 b, f32x4_t c) __attribute__((always_inline)) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    };
    const int afrag = (wm * (TM / 2) + fr) * 4 + (fk ^ ((fr >> 1) & 3)), bfrag = ((wn_ * 64 + fr) >> 3) * 32 + (fk << 3) + (fr & 7);

    constexpr uint32_t kOnes = 0x3F803F80u;
    const uint4 ones = OG == 16 && (fk < 2) != ((fr & 1) == 0) ? uint4{0, 0, 0, 0} : uint4{kOnes, kOnes, kOnes, kOnes};
    auto step = [&]<int U>(int blk) __attribute__((always_inline)) {
        const int par = (blk - blk0) & 1;
        const int nblk = min(blk + 1, blk1 - 1);  // past the end: the last block again
        load_x.template operator()<(U + 2) & 7>(U + 2 > 7 ? nblk : blk);
        load_w.template operator()<(U + 3) & 7>(U + 3 > 7 ? nblk : blk);
        if constexpr (U == 4) load_hdr(nblk);
        const uint4* const xb = xs + (U & 1) * XP * XPL + afrag;
        const uint4* const wb = wsm + (U & 1) * WP * 512 + bfrag;
        uint4 bf[WP][NJ];
        float sc[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
#pragma unroll
            for (int p = 0; p < WP; ++p) bf[p][j] = wb[p * 512 + j * 64];
            if constexpr (!F::BLOCK_SCALE) sc[j] = wscale[(U & 1) * 128 + wn_ * 64 + j * 16 + fr];
        }
        constexpr int TS = F::WIRE ? 1 : 2;  // (the wire formats' registers are full)
        f32x4_t t[TS][NJ];
        auto apply = [&](int i) __attribute__((always_inline)) {  // the step's scale
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[i][j][e] = __builtin_fmaf(sc[j], t[i % TS][j][e], acc[i][j][e]);
                // (the optimizer would otherwise keep a block's eight sums and add them at its end, out of registers)
                f32x4_t& done = acc[i][j];
                asm volatile("" : "+v"(done));
            }
        };
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            uint4 af[XP];
#pragma unroll
            for (int p = 0; p < XP; ++p) af[p] = xb[p * XPL + i * 64];
            // The small parts first.  The wire formats add a step's products to the block's sum in fp32: kept in the matrix
            // cores over its 16 products its error was up to 1.45 times the fp32 kernel's.
#pragma unroll
            for (int p = XP - 1; p >= 0; --p)
#pragma unroll
                for (int q = WP - 1; q >= 0; --q)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        const bool first = p == XP - 1 && q == WP - 1;
                        if constexpr (F::BYTES) blk_acc[i][j] = mm(af[p], bf[q][j], first && U == 0 ? zero4 : blk_acc[i][j]);
                        else t[i % TS][j] = mm(af[p], bf[q][j], first ? zero4 : t[i % TS][j]);
                    }
            if constexpr (F::WIRE) {
#pragma unroll
                for (int j = 0; j < NJ; ++j) blk_acc[i][j] = U == 0 ? t[i % TS][j] : blk_acc[i][j] + t[i % TS][j];
            }
            // one row of tiles behind the matrix instructions, which then have no result to wait for
            if constexpr (!F::BLOCK_SCALE) {
                if (i > 0) apply(i - 1);
            }
        }
        if constexpr (!F::BLOCK_SCALE) apply(MI - 1);
        if constexpr (OG > 0) {
            // The step's group sums, by MFMAs against ones (16-weight groups: even columns take the first group, odd ones
            // the second), each wavefront of a pair half of their rows: as sums of the parts that the codes meet, what the
            // parts leave out of x counts with the weight itself and not with code and offset apart (twice the error).
#pragma unroll
            for (int h = 0; h < MI / 2; ++h) {
                const int i = wn_ * (MI / 2) + h;
                f32x4_t v4 = zero4;
#pragma unroll
                for (int p = XP - 1; p >= 0; --p) v4 = mm(xb[p * XPL + i * 64], ones, v4);
                // (lanes beyond the four rows write what those write: no branch in the middle of the step)
                const int e = (OG == 16 ? fr >> 1 : fr) & 3;
                const float v01 = e & 1 ? v4[1] : v4[0], v23 = e & 1 ? v4[3] : v4[2], v = e & 2 ? v23 : v01;
                const uint32_t p0 = pk(v, 0.0f), p1 = pk(v - bf_lo(p0), 0.0f), p2 = pk(v - bf_lo(p0) - bf_lo(p1), 0.0f);
                const int r = wm * (TM / 2) + i * 16 + 4 * fk + e;
                unsigned short* const sd = reinterpret_cast<unsigned short*>(sums) + (OG == 16 ? r * 48 + 2 * U + (fr & 1) : r * 24 + U);
                sd[0] = (unsigned short)p0;
                sd[OG] = (unsigned short)p1;
                sd[2 * OG] = (unsigned short)p2;
            }
        }
        if constexpr (U == 7) {
            if constexpr (OG > 0) __syncthreads();  // the block's group sums are complete
            if constexpr (F::BLOCK_SCALE) {
                float bs[NJ];
#pragma unroll
                for (int j = 0; j < NJ; ++j) bs[j] = wscale[par * 128 + wn_ * 64 + j * 16 + fr];
                if constexpr (F::SC_OFFSET) {  // 4 sc times the group sums, at the block's scale
#pragma unroll
                    for (int i = 0; i < MI; ++i) {
                        const uint4* sp = sums + (wm * (TM / 2) + i * 16 + fr) * 6;
                        const uint4 a1 = sp[fk], a2 = fk < 2 ? sp[4 + fk] : uint4{0, 0, 0, 0};
#pragma unroll
                        for (int j = 0; j < NJ; ++j) {
                            const uint4 b = scs[par * 256 + (fk & 1) * 128 + wn_ * 64 + j * 16 + fr];
                            blk_acc[i][j] = mm(a1, b, mm(a2, fk < 2 ? b : uint4{0, 0, 0, 0}, blk_acc[i][j]));
                        }
                    }
                }
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][j][e] = __builtin_fmaf(bs[j], blk_acc[i][j][e], acc[i][j][e]);
                        f32x4_t& done = acc[i][j];
                        asm volatile("" : "+v"(done));
                    }
            }
            if constexpr (OG > 0) {
                float dm[NJ];
#pragma unroll
                for (int j = 0; j < NJ; ++j) dm[j] = woff[par * 128 + wn_ * 64 + j * 16 + fr];
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    const uint4 none = {0, 0, 0, 0};
                    const uint4* sp = sums + (wm * (TM / 2) + i * 16 + fr) * (OG == 16 ? 6 : 3);
                    f32x4_t u[NJ];
                    if constexpr (OG == 16) {
                        const uint4 a1 = sp[fk], a2 = fk < 2 ? sp[4 + fk] : none;
#pragma unroll
                        for (int j = 0; j < NJ; ++j) {
                            const uint4 b = mcs[par * 256 + (fk & 1) * 128 + wn_ * 64 + j * 16 + fr];
                            u[j] = mm(a1, b, mm(a2, fk < 2 ? b : none, zero4));
                        }
                    } else {
                        const uint4 a1 = fk < 3 ? sp[fk < 3 ? fk : 0] : none;
#pragma unroll
                        for (int j = 0; j < NJ; ++j) u[j] = mm(a1, fk < 3 ? mcs[par * 128 + wn_ * 64 + j * 16 + fr] : none, zero4);
                    }
#pragma unroll
                    for (int j = 0; j < NJ; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][j][e] = __builtin_fmaf(dm[j], u[j][e], acc[i][j][e]);
                }
            }
        }
        stage.template operator()<(U + 1) & 7>(U == 7 ? par ^ 1 : par);
        __syncthreads();
    };

    load_hdr(blk0);
    load_x.template operator()<0>(blk0);
    load_x.template operator()<1>(blk0);
    load_w.template operator()<0>(blk0);
    load_w.template operator()<1>(blk0);
    load_w.template operator()<2>(blk0);
    stage.template operator()<0>(0);
    __syncthreads();
    for (int blk = blk0; blk < blk1; ++blk) {
        step.template operator()<0>(blk);
        step.template operator()<1>(blk);
        step.template operator()<2>(blk);
        step.template operator()<3>(blk);
        step.template operator()<4>(blk);
        step.template operator()<5>(blk);
        step.template operator()<6>(blk);
        step.template operator()<7>(blk);
    }

    // ---- store: lane holds column fr, rows 4 fk + e of each 16 x 16 tile
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int col = n0 + wn_ * 64 + j * 16 + fr;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = m0 + wm * (TM / 2) + i * 16 + 4 * fk + e;
                const bool valid = m < M && col < N;
                const size_t o = (size_t)m * N + col;
                float v = acc[i][j][e];
                if constexpr (F::WIRE) {
                    if (S == 1 && __ballot(valid && !finite_f32(v))) v = repair_non_finite<FMT, XP>(args.W, args.X, K, m, col, valid, v);
                }
                if (valid) {
                    if (S > 1) args.partial[(size_t)split * M * N + o] = v;
                    else if (args.y_bf16) reinterpret_cast<unsigned short*>(args.Y)[o] = (unsigned short)bf16_rne(v);
                    else reinterpret_cast<float*>(args.Y)[o] = v;
                }
            }
        }
}

// y = sum over the K splits of their partial tiles, in split order
template <int FMT, int XP>
__global__ __launch_bounds__(256) void reduce_exact_kernel(ExactArgs args) {
    const size_t n = (size_t)args.M * args.N, i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const bool valid = i < n;
    float v = 0.0f;
    for (int sp = 0; sp < args.ksplit; ++sp) v += valid ? args.partial[(size_t)sp * n + i] : 0.0f;
    if constexpr (Form<FMT>::WIRE) {
        if (__ballot(valid && !finite_f32(v)))
            v = repair_non_finite<FMT, XP>(args.W, args.X, args.K, (int)(i / args.N), (int)(i % args.N), valid, v);
    }
    if (!valid) return;
    if (args.y_bf16) reinterpret_cast<unsigned short*>(args.Y)[i] = (unsigned short)bf16_rne(v);
    else reinterpret_cast<float*>(args.Y)[i] = v;
}

// Tile height, K split and time (us) of M rows by a model of measurements (14336 x 4096): two workgroups of 128 rows
// or three of 64 run on a compute unit at once; a step takes t[n - 1] us with n workgroups on every unit.  Rows are the
// operand products per weight: one (bf16 activations, 16-weight groups), two (fp32 activations, or bf16 ones on the
// wire formats) or six (fp32 on the wire formats, whose 128-row tile fits a unit only once and lost: 1.7 us against
// 1.44 us for two of 64).  The partials' traffic at 5 TB/s.
struct ExactPlan {
    int tm, ksplit;
    double us;
};
ExactPlan plan_exact(int64_t N, int64_t K, int M, int planes, size_t scratch_bytes) {
    static constexpr double kStep64[3][3] = {{0.50, 0.78, 1.05}, {0.56, 0.93, 1.30}, {0.84, 1.44, 0.0}}, kStep128[2][2] = {{0.75, 1.00}, {0.85, 1.30}};
    const int nblocks = (int)(K >> 8), kind = planes == 1 ? 0 : planes == 2 ? 1 : 2;
    ExactPlan best{64, 1, 1e30};
    for (int tm = 64; tm <= (kind == 2 ? 64 : 128); tm *= 2) {
        const long tiles = (long)((M + tm - 1) / tm) * (long)((N + TN - 1) / TN);
        const int per_cu = tm == 128 || kind == 2 ? 2 : 3;
        const double* t = tm == 64 ? kStep64[kind] : kStep128[kind];
        const long slots = 256L * per_cu;
        for (int S = 1; S <= 16 && S <= nblocks; ++S) {
            const double part_bytes = (double)S * (double)M * (double)N * 4.0;
            if (S > 1 && (tiles * S > 2 * slots || part_bytes > (double)scratch_bytes)) continue;
            const long wgs = tiles * S, rest = wgs % slots;
            const double steps = 8.0 * (double)((nblocks + S - 1) / S);
            double us = 4.0 + steps * ((double)(wgs / slots) * t[per_cu - 1] + (rest ? t[(rest + 255) / 256 - 1] : 0.0));
            if (S > 1) us += 3.0 + part_bytes * (1.0 + 1.0 / S) / 5e6;
            if (us < best.us) best = {tm, S, us};
        }
    }
    return best;
}

template <int FMT, int XP, int TM>
int run_exact_tm(ExactArgs a, hipStream_t s) {
    constexpr size_t lds = (size_t)lds_uint4s<FMT, XP, TM>() * 16;
    if constexpr (lds > 64 * 1024) {  // (two fp32 parts of 128 rows beside the byte headers' offsets: 70 or 78 KB)
        static std::atomic<bool> lds_limit_raised = false;  // once per kernel, as for the other tile kernel
        if (!lds_limit_raised) {
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_exact_kernel<FMT, XP, TM>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute");
            lds_limit_raised = true;
        }
    }
    a.tiles_m = (a.M + TM - 1) / TM;
    const long items = (long)a.tiles_m * a.tiles_n * a.ksplit;
    hipLaunchKernelGGL((gemm_exact_kernel<FMT, XP, TM>), dim3((unsigned)(8 * ((items + 7) / 8))), dim3(THREADS), lds, s, a);
    if (a.ksplit > 1) {
        const size_t n = (size_t)a.M * a.N;
        hipLaunchKernelGGL((reduce_exact_kernel<FMT, XP>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
    }
    return hip_fail(hipGetLastError(), "gemm launch");
}

template <int FMT, int XP>
int run_exact(const ExactArgs& a, int tm, hipStream_t s) {
    if constexpr (XP == 3) return run_exact_tm<FMT, XP, 64>(a, s);
    else return tm == 64 ? run_exact_tm<FMT, XP, 64>(a, s) : run_exact_tm<FMT, XP, 128>(a, s);
}

int run_exact_fmt(int fmt, const ExactArgs& a, bool f32, int tm, hipStream_t s) {
    switch (canonical(fmt)) {
        case TFQ_Q_G_4: return run_exact<TFQ_Q_G_4, 2>(a, tm, s);
        case TFQ_Q_G_3: return run_exact<TFQ_Q_G_3, 2>(a, tm, s);
        case TFQ_B32S4: return run_exact<TFQ_B32S4, 2>(a, tm, s);
        case TFQ_B32S8: return run_exact<TFQ_B32S8, 2>(a, tm, s);
        case TFQ_Q_G_8: return run_exact<TFQ_Q_G_8, 2>(a, tm, s);
        case TFQ_Q_8: return run_exact<TFQ_Q_8, 2>(a, tm, s);
        case TFQ_Q_G_2: return f32 ? run_exact<TFQ_Q_G_2, 2>(a, tm, s) : run_exact<TFQ_Q_G_2, 1>(a, tm, s);
        case TFQ_SB256A3: return f32 ? run_exact<TFQ_SB256A3, 2>(a, tm, s) : run_exact<TFQ_SB256A3, 1>(a, tm, s);
        case TFQ_SB256A2: return f32 ? run_exact<TFQ_SB256A2, 2>(a, tm, s) : run_exact<TFQ_SB256A2, 1>(a, tm, s);
        case TFQ_Q_4: return f32 ? run_exact<TFQ_Q_4, 3>(a, tm, s) : run_exact<TFQ_Q_4, 1>(a, tm, s);
        case TFQ_Q_G_6: return f32 ? run_exact<TFQ_Q_G_6, 3>(a, tm, s) : run_exact<TFQ_Q_G_6, 1>(a, tm, s);
        default: return fail(TFQ_ERR_FORMAT, "gemm: no tile kernel for this format");
    }
}

int planes_of(const tfq_weight* w, int x_dtype) {
    const bool wire = w->layout == TFQ_LAYOUT_WIRE;
    return (x_dtype == TFQ_BF16 ? 1 : wire ? 3 : 2) * (wire ? 2 : 1);
}

}  // namespace

bool gemm_exact_serves(const tfq_weight* w, int x_dtype, int M) {
    if (M <= 16 || w->N > 0x7FFFFF00 || w->K > (1 << 22)) return false;
    if ((double)((M + 63) / 64) * (double)((w->N + TN - 1) / TN) * 16.0 > 2e9) return false;
    const int f = canonical(w->fmt);
    if (w->layout == TFQ_LAYOUT_WIRE) return f == TFQ_Q_4 || f == TFQ_Q_G_6;
    return w->layout == TFQ_LAYOUT_TILED16 && (x_dtype == TFQ_F32 || tiled_header_bytes(w->fmt) == 48);
}

size_t gemm_exact_scratch_bytes(const tfq_weight* w, int x_dtype, int M) {
    const ExactPlan p = plan_exact(w->N, w->K, M, planes_of(w, x_dtype), ~(size_t)0);
    return p.ksplit > 1 ? (size_t)p.ksplit * (size_t)M * (size_t)w->N * 4 : 0;
}

// What a call with this much scratch takes (us): the plan's model, which prices every format of a kind alike, times
// about the median of measured over modelled (17 to 200 rows, 256 x 1024 to 128256 x 4096; nine tenths within 25 % of it).
double gemm_exact_us(const tfq_weight* w, int x_dtype, int M, size_t scratch_bytes) {
    const bool f32 = x_dtype == TFQ_F32;
    double fit = 1.0;
    switch (canonical(w->fmt)) {
        case TFQ_B32S4: fit = 0.86; break;
        case TFQ_B32S8: case TFQ_Q_G_8: case TFQ_Q_8: fit = 0.9; break;
        case TFQ_Q_G_4: case TFQ_Q_G_3: fit = 1.05; break;
        case TFQ_SB256A3: fit = f32 ? 1.1 : 0.95; break;
        case TFQ_Q_G_2: case TFQ_SB256A2: fit = f32 ? 1.0 : 0.89; break;
        default: fit = f32 ? 1.1 : 1.25; break;
    }
    return fit * plan_exact(w->N, w->K, M, planes_of(w, x_dtype), scratch_bytes).us;
}

// keep_split: the K split is the one that a scratch of any size would give; where its partial tiles need more than there
// is, the rows go through in runs of whole tiles (a split has at most two rounds of workgroups, so 32 MiB hold the parts
// of 42 rows or more; a row's sums do not depend on the tile it is in).
int launch_gemm_exact(const tfq_weight* w, const void* x, int x_dtype, int M, void* y, int y_dtype, hipStream_t s, void* scratch,
                      size_t scratch_bytes, bool keep_split) {
    const size_t have = scratch ? scratch_bytes : 0;
    const ExactPlan p = plan_exact(w->N, w->K, M, planes_of(w, x_dtype), keep_split ? ~(size_t)0 : have);
    int rows = M;
    if (keep_split && p.ksplit > 1) {
        const size_t fit = have / ((size_t)p.ksplit * (size_t)w->N * 4);
        if (fit < (size_t)M) rows = (int)(fit < (size_t)p.tm ? fit : fit / p.tm * p.tm);
        if (rows < 1) return fail(TFQ_ERR_SHAPE, "gemm: no scratch for the K split");
    }
    const size_t xe = x_dtype == TFQ_F32 ? 4 : 2, ye = y_dtype == TFQ_F32 ? 4 : 2;
    for (int m0 = 0; m0 < M; m0 += rows) {
        ExactArgs a{};
        a.W = w->dev;
        a.X = static_cast<const uint8_t*>(x) + (size_t)m0 * (size_t)w->K * xe;
        a.Y = static_cast<uint8_t*>(y) + (size_t)m0 * (size_t)w->N * ye;
        a.M = std::min(rows, M - m0);
        a.N = (int)w->N;
        a.K = (int)w->K;
        a.y_bf16 = y_dtype == TFQ_BF16;
        a.tiles_n = (int)((w->N + TN - 1) / TN);
        a.ksplit = p.ksplit;
        a.partial = reinterpret_cast<float*>(scratch);
        if (int rc = run_exact_fmt(w->fmt, a, x_dtype == TFQ_F32, p.tm, s)) return rc;
    }
    return TFQ_OK;
}

}  // namespace tfq
