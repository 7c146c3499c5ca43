// Encoder of ONE block of fewer than 256 weights: the last block of a tensor whose size is not a
// multiple of 256 (FormatRegistry::quantize cuts a tensor into 256-blocks and hands the encoder the
// remainder as a short block, src/codec/format_registry.cpp:168-207).  The reference's block encoders
// (src/codec/block_codec.cpp:2402-2867) choose a short block's layout from (format, n): headers shrink or
// vanish, group counts follow n, and the sixteen shortened codes sit where floor(16 i / n) steps.
// block_layout() restates those rules on the host; this file encodes into whatever layout it names.
//
// One wavefront works on the block:
//   * a lane per weight, four weights each, for everything that is independent per weight (nearest level, residual, code),
//   * a lane per scale group for the sums of a group's fit, in index order in double, as the results must not
//     depend on how the work is split,
//   * lane 0 for the sums that run over the whole block or over the groups,
//   * every field of the payload (a code, a scale code, a binary16) is OR-ed into a zeroed image of the
//     block at its bit position by the lane that owns it: the parts of a short block are one LSB-first
//     stream with no alignment between them, so there is no byte a single lane could own.
// It is a chain of dependent steps whatever the tensor's size (a Q_G_4 block took 150 us with the fit of a group in
// one lane, five times the time of 65536 weights), so the code is compiled for the format (level tables are
// constants of the unrolled scans), and the encoders of tfq_codec.hip run it in a workgroup of the launch that
// encodes the full blocks.
// The _K_M / _K_H ids encode further candidates (more refits, scaled start values) into a second image
// and keep one where the decoded error is strictly smaller, as their full blocks do.
// Multiply-adds are fused where the reference's Release build (GCC, -ffp-contract=fast) fuses them.

#pragma once

#include "tfq_decode.hpp"

namespace tfq {

namespace {

constexpr int kMaxShortBytes = 1024;  // 255 weights of the widest format are 1020 bytes
constexpr float kTiny = 1e-15f;

struct ShortJob {  // L.n = 0: there is no short block
    BlockLayout L;
    int tier;  // search effort of the _K ids: 0, 1, 2; BK_Q1: -1 = the RMS scale of plain Q_1
    const float* w;
    uint8_t* dst;
};

// What the wavefront shares.
struct Team {
    float w[256];        // the block
    float table[256];    // the companded 8-bit levels
    float lev[256];      // per weight: the level it is assigned, or a residual
    double dres[256];    // per weight: a residual in double
    float gs[32];        // per group: scale
    float gm[32];        // per group: offset
    float gtry[32];      // per group: a scale that is being tried
    int gc[32];          // per group: scale code
    int gk[32];          // per group: offset code
    uint32_t img[2][kMaxShortBytes / 4];  // payload images: [0] the block, [1] a candidate
    double d0, d1;       // results lane 0 publishes
    float f0, f1;
    int i0;
};

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = fmaxf(v, __shfl_xor(v, m, 64));
    return v;
}

// is_slot (:176-180): sixteen positions of a block give up the low bit of their code
__device__ __forceinline__ int slots_before(int i, int n) { return (i * 16) / n; }
__device__ __forceinline__ bool slot_at(int i, int n) { return ((i + 1) * 16) / n != (i * 16) / n; }

// `width` bits of `value` at bit `pos` of an image of `cap` bits; what would fall behind the end is dropped
__device__ __forceinline__ void put_bits(uint32_t* img, uint32_t cap, uint32_t pos, uint32_t value, int width) {
    if (pos >= cap || width <= 0) return;
    if (pos + (uint32_t)width > cap) width = (int)(cap - pos);
    if (width < 32) value &= (1u << width) - 1u;
    const uint32_t sh = pos & 31u;
    atomicOr(&img[pos >> 5], value << sh);
    if (sh + (uint32_t)width > 32u) atomicOr(&img[(pos >> 5) + 1], value >> (32u - sh));
}

// f(i) for every weight of the run [0, cnt), four per lane at once (a lane without a fourth weight repeats the last one)
template <class F>
__device__ __forceinline__ void each(int lane, int cnt, F&& f) {
    if (cnt <= 0) return;
#pragma unroll
    for (int k = 0; k < 4; ++k) f(min(lane + 64 * k, cnt - 1));
}

// ---- level tables and nearest-level searches
// FIXED: the fixed N(0,1) codebooks (3, 6, 12 bits) instead of the lattice grids
template <int BITS, bool FIXED>
struct Grid {
    static __device__ __forceinline__ float level(uint32_t idx) { return FIXED ? fixed_value(BITS, idx) : grid_value(BITS, idx); }
    static __device__ __forceinline__ float top() { return level((1u << BITS) - 1u); }
    static __device__ __forceinline__ uint32_t pick(float v) {
        if constexpr (FIXED && BITS > 3) {  // ascending quantile table, symmetric: search |v| in the upper half (:596-622)
            constexpr int half = 1 << (BITS - 1);
            const float a = fabsf(v);
            int lo = half;  // the first level of the upper half that is not below a, the last one at most
#pragma unroll
            for (int len = half / 2; len >= 1; len /= 2) lo += fixed_value(BITS, (uint32_t)(lo + len - 1)) < a ? len : 0;
            if (lo > half && fixed_value(BITS, (uint32_t)lo) - a >= a - fixed_value(BITS, (uint32_t)lo - 1u)) --lo;
            return v >= 0.0f ? (uint32_t)lo : (uint32_t)(half - 1 - (lo - half));
        } else if constexpr (FIXED || BITS == 2 || BITS == 4) {  // short tables: the first level at the smallest distance
            uint32_t best = 0;
            float bd = fabsf(v - level(0));
#pragma unroll
            for (uint32_t i = 1; i < (1u << BITS); ++i) {
                const float d = fabsf(v - level(i));
                if (d < bd) { bd = d; best = i; }
            }
            return best;
        } else {
            constexpr float span = (float)(BITS >= 24 ? 16777215u : (1u << (BITS & 31)) - 1u);  // uniform grid on [-8, 8]
            return (uint32_t)lroundf((fmaxf(-8.0f, fminf(8.0f, v)) + 8.0f) * span / 16.0f);
        }
    }
};

__device__ __forceinline__ uint32_t unit_pick(float value, int bits) {  // nearest code of the [0, 1] grid
    const float top = (float)((1 << bits) - 1);
    return (uint32_t)lroundf(fmaxf(0.0f, fminf(1.0f, value)) * top);
}

__device__ __forceinline__ int six_round(float v) {  // to nearest, ties to even, through the 1.5 * 2^23 bias
    return (int)(__float_as_uint(v + 12582912.f) & 0x007fffffu) - 0x00400000;
}
__device__ __forceinline__ int six_level(float ratio) {
    return max(-32, min(31, six_round(fmaxf(-4000.0f, fminf(4000.0f, ratio)))));
}

// sums over [0, cnt) of a[i] * b[i] and of b[i] * b[i], in index order, in double
__device__ __forceinline__ void dots_in_order(const float* a, const float* b, int cnt, double* ab, double* bb) {
    double x = 0.0, y = 0.0;
#pragma unroll 8
    for (int i = 0; i < cnt; ++i) {
        const double l = (double)b[i];
        x = __builtin_fma((double)a[i], l, x);
        y = __builtin_fma(l, l, y);
    }
    *ab = x;
    *bb = y;
}

// ------------------------------------------------------------------------------------------------
// One scale for a run of weights against a level table: s = absmax / top * smult, then `iters`
// least-squares refits over the nearest levels.  The whole wavefront works on the run [0, n).
template <class G>
__device__ float fit_run(Team& T, int lane, int n, int iters, float smult) {
    float m = 0.0f;
    each(lane, n, [&](int i) { m = fmaxf(m, fabsf(T.w[i])); });
    m = wave_max(m);
    float s = (m > 1e-30f) ? m / G::top() * smult : 0.0f;
    if (s > 0.0f) {
        for (int it = 0; it < iters; ++it) {
            each(lane, n, [&](int i) { T.lev[i] = G::level(G::pick(T.w[i] / s)); });
            __syncthreads();
            if (lane == 0) {
                double num, den;
                dots_in_order(T.w, T.lev, n, &num, &den);
                T.f0 = (den > 1e-20) ? (float)(num / den) : s;
            }
            __syncthreads();
            s = T.f0;
            __syncthreads();
        }
    }
    return s > 0.0f ? s : 0.0f;
}

// The same for whole groups of 32 weights at once: lane g fits group g (its sums), the lanes assign levels.
// T.gs[g] receives the scales.
template <class G>
__device__ void fit_groups32(Team& T, int lane, int ng, int iters, float smult) {
    if (lane < ng) {
        float m = 0.0f;
        for (int i = 32 * lane; i < 32 * lane + 32; ++i) m = fmaxf(m, fabsf(T.w[i]));
        T.gs[lane] = (m > 1e-30f) ? m / G::top() * smult : 0.0f;
        T.gc[lane] = T.gs[lane] > 0.0f;  // a group whose start value is zero is never refit
    }
    __syncthreads();
    for (int it = 0; it < iters; ++it) {
        each(lane, 32 * ng, [&](int i) {
            if (T.gc[i >> 5]) T.lev[i] = G::level(G::pick(T.w[i] / T.gs[i >> 5]));
        });
        __syncthreads();
        if (lane < ng && T.gc[lane]) {
            double num, den;
            dots_in_order(T.w + 32 * lane, T.lev + 32 * lane, 32, &num, &den);
            if (den > 1e-20) T.gs[lane] = (float)(num / den);
        }
        __syncthreads();
    }
    if (lane < ng && !(T.gs[lane] > 0.0f)) T.gs[lane] = 0.0f;
    __syncthreads();
}

// Golden-section search of the companded grid's scale from the seed s, then the +-4 neighbouring binary16 values
// (comp8_fit_scale_fp16, src/codec/block_codec.cpp:306-358).  The evaluations are steps of one loop, so that their code
// is there once: 0, 1 the first two section points; 2..15 the golden-section steps; 16 the middle; 17 its binary16;
// 18..25 the neighbours of that.
template <class SqErr>
__device__ __forceinline__ float comp8_search(double s, double hi, SqErr&& sq_err) {
    const double phi = 0.6180339887498949;
    double a = s * 0.75, b = s * 1.25, c = 0.0, d = 0.0, fc = 0.0, fd = 0.0, raw = 0.0, best_e = 0.0;
    uint32_t hf = 0;
    float best = 0.0f;
#pragma unroll 1
    for (int step = 0; step < 26; ++step) {
        bool left = false;
        double at;
        if (step == 0) at = c = __builtin_fma(-phi, b - a, b);
        else if (step == 1) at = d = __builtin_fma(phi, b - a, a);
        else if (step < 16) {
            if (!((b - a) > 1e-11 * (a + b))) { step = 15; continue; }
            left = fc < fd;
            if (left) { b = d; d = c; fd = fc; at = c = __builtin_fma(-phi, b - a, b); }
            else { a = c; c = d; fc = fd; at = d = __builtin_fma(phi, b - a, a); }
        } else if (step == 16) at = raw = 0.5 * (a + b);
        else if (step == 17) {
            hf = float_to_half_bits((float)raw);
            at = (double)half_bits_to_float(hf);
        } else {
            const int hc = (int)hf + (step < 22 ? step - 22 : step - 21);
            if (hc < 0 || hc > 0xFFFF) continue;
            const float cand = half_bits_to_float((uint32_t)hc);
            if (!(cand > 0.0f) || !((double)cand <= hi * 1.02)) continue;
            at = (double)cand;
        }
        const double e = sq_err(at);
        if (step == 0) fc = e;
        else if (step == 1) fd = e;
        else if (step < 16) (left ? fc : fd) = e;
        else if (step == 16) {
            if (e > fc && fc <= fd) raw = c;
            else if (e > fd) raw = d;
        } else if (step == 17) { best_e = e; best = (float)at; }
        else if (e < best_e) { best_e = e; best = (float)at; }
    }
    return best;
}

// A team of T lanes owns a run, PER = CNT / T consecutive weights in each lane's registers; a wavefront holds 64 / T
// teams.  What is independent per weight (division, nearest level, residual) runs in all lanes; the sums must be added
// in index order (double, as the reference adds them), so they go round the team: the lanes all run their PER steps
// from the sum they were given and the sum of lane st is what lane st + 1 starts from.
__device__ __forceinline__ double from_lane_below(double v) {  // within a row of sixteen lanes
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x111, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x111, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
// step(a, b) adds the lane's part to both sums; every lane of the team gets the totals
template <int T, class Step>
__device__ __forceinline__ void ordered_sums(int first, double& a, double& b, Step&& step) {
    static_assert(T <= 16, "a team lies in one row of lanes");
    a = 0.0;
    b = 0.0;
    step(a, b);
    if constexpr (T > 1) {
        const int tl = (int)(threadIdx.x & 63) - first;
#pragma unroll 1
        for (int st = 1; st < T; ++st) {
            double na = from_lane_below(a), nb = from_lane_below(b);
            if (tl == 0) { na = 0.0; nb = 0.0; }
            step(na, nb);
            a = na;
            b = nb;
        }
        a = __shfl(a, first + T - 1, 64);
        b = __shfl(b, first + T - 1, 64);
    }
}

// Scale fit of a run of CNT weights on the companded grid by a team (see encode_comp8_kernel)
template <int CNT, int T>
struct Comp8Team {
    static constexpr int PER = CNT / T;
    const float* lv;  // 256 levels, LDS
    float w[PER];
    int first;  // the team's first lane
    static __device__ __forceinline__ int below(float v) {
        return (int)fminf(fmaxf(__builtin_fmaf(v, 127.5f / 1.0000742443371564f, 127.5f), 0.0f), 254.0f);
    }
    __device__ __forceinline__ uint32_t nearest(float v) const {
        const int lo = below(v);
        return (v - lv[lo] <= lv[lo + 1] - v) ? (uint32_t)lo : (uint32_t)lo + 1u;
    }
    __device__ __forceinline__ float level(float v) const {
        const int lo = below(v);
        const float a = lv[lo], b = lv[lo + 1];
        return (v - a <= b - v) ? a : b;
    }
    __device__ __forceinline__ double sq_err(double s) const {
        const double inv = 1.0 / s;
        double r[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k) r[k] = __builtin_fma((double)level((float)((double)w[k] * inv)), s, -(double)w[k]);
        double e, unused;
        ordered_sums<T>(first, e, unused, [&](double& a, double&) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < PER; ++k) a = __builtin_fma(r[k], r[k], a);
        });
        return e;
    }
    // false when the refit has no support (den <= 1e-20)
    __device__ __forceinline__ bool seed(double s, double* out) const {
        float l[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k) l[k] = level((float)((double)w[k] / s));
        double num, den;
        ordered_sums<T>(first, num, den, [&](double& a, double& b) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                a = __builtin_fma((double)w[k], (double)l[k], a);
                b = __builtin_fma((double)l[k], (double)l[k], b);
            }
        });
        if (!(den > 1e-20)) return false;
        *out = num / den;
        return true;
    }
    __device__ __forceinline__ float fit(double maxa) const {
        if (!(maxa > 0.0)) return 0.0f;
        const double hi = maxa * 1.0000001;
        double s = maxa;
#pragma unroll 1
        for (int it = 0; it < 3; ++it) {
            double ls;
            if (!seed(s, &ls)) break;
            s = ls < hi ? ls : hi;
        }
        return comp8_search(s, hi, [&](double at) __attribute__((always_inline)) { return sq_err(at); });
    }
};

// ------------------------------------------------------------------------------------------------
// Scale of the 8-bit companded grid for the run [first, first + cnt) (comp8_fit_scale_fp16, :306-358): three
// least-squares seeds, a golden-section search on the true squared error over [0.75 s, 1.25 s], then the +-4
// neighbouring binary16 values.  The lanes evaluate the weights, lane 0 adds in index order; the search itself
// runs in every lane on the values lane 0 publishes.
struct Comp8Run {
    Team& T;
    int lane, first, cnt;
    // the two levels around a value from the line through the grid (see encode_comp8_kernel), then the nearer one
    __device__ __forceinline__ uint32_t pick(float v) const {
        const int lo = (int)fminf(fmaxf(__builtin_fmaf(v, 127.5f / 1.0000742443371564f, 127.5f), 0.0f), 254.0f);
        return (v - T.table[lo] <= T.table[lo + 1] - v) ? (uint32_t)lo : (uint32_t)lo + 1u;
    }
    __device__ double sq_err(double s) const {
        const double inv = 1.0 / s;
        each(lane, cnt, [&](int i) {
            const float x = T.w[first + i];
            T.dres[i] = __builtin_fma((double)T.table[pick((float)((double)x * inv))], s, -(double)x);
        });
        __syncthreads();
        if (lane == 0) {
            double e = 0.0;
#pragma unroll 8
            for (int i = 0; i < cnt; ++i) e = __builtin_fma(T.dres[i], T.dres[i], e);
            T.d0 = e;
        }
        __syncthreads();
        const double e = T.d0;
        __syncthreads();
        return e;
    }
    __device__ bool seed(double s, double* refit) const {
        each(lane, cnt, [&](int i) { T.dres[i] = (double)T.table[pick((float)((double)T.w[first + i] / s))]; });
        __syncthreads();
        if (lane == 0) {
            double num = 0.0, den = 0.0;
#pragma unroll 8
            for (int i = 0; i < cnt; ++i) {
                num = __builtin_fma((double)T.w[first + i], T.dres[i], num);
                den = __builtin_fma(T.dres[i], T.dres[i], den);
            }
            T.d0 = num;
            T.d1 = den;
        }
        __syncthreads();
        const double num = T.d0, den = T.d1;
        __syncthreads();
        if (!(den > 1e-20)) return false;
        *refit = num / den;
        return true;
    }
    __device__ float fit() const {
        float m = 0.0f;
        each(lane, cnt, [&](int i) { m = fmaxf(m, fabsf(T.w[first + i])); });
        const double maxa = (double)wave_max(m);
        if (!(maxa > 0.0)) return 0.0f;
        const double hi = maxa * 1.0000001;
        double s = maxa;
        for (int it = 0; it < 3; ++it) {
            double ls;
            if (!seed(s, &ls)) break;
            s = ls < hi ? ls : hi;
        }
        return comp8_search(s, hi, [&](double at) { return sq_err(at); });
    }
};

// ------------------------------------------------------------------------------------------------
// Plain lattice and fixed-codebook blocks: [binary16 scale][n codes, sixteen of them a bit short]; fewer
// than sixteen weights are bare codes against a scale of one (quant_lattice :443-497, quant_fixed_codebook
// :624-663).
template <int BITS, bool FIXED>
__device__ void encode_lattice(Team& T, int lane, const BlockLayout& L, uint32_t* img, int iters, float smult) {
    using G = Grid<BITS, FIXED>;
    const int n = L.n;
    const uint32_t cap = (uint32_t)L.bytes * 8u;
    constexpr bool comp8 = !FIXED && BITS == 8;
    if (L.kind == BK_LEVELS) {
        each(lane, n, [&](int i) { put_bits(img, cap, (uint32_t)(i * BITS), G::pick(T.w[i]), BITS); });
        return;
    }
    const Comp8Run run{T, lane, 0, n};
    float s;
    if constexpr (comp8) s = run.fit() * smult;
    else s = fit_run<G>(T, lane, n, iters, smult);
    if (lane == 0) put_bits(img, cap, 0, float_to_half_bits(s), 16);
    each(lane, n, [&](int i) {
        uint32_t idx;
        if constexpr (comp8) idx = (s > 0.0f) ? run.pick(T.w[i] / s) : 0u;
        else idx = G::pick((s == 0.0f) ? 0.0f : T.w[i] / s);
        const bool sl = slot_at(i, n);
        put_bits(img, cap, (uint32_t)(16 + BITS * i - slots_before(i, n)), sl ? idx >> 1 : idx, BITS - (sl ? 1 : 0));
    });
}

// 12-bit codes with a binary16 scale per 32 weights (quant_grp12_compound, :969-1004) and the 8-bit
// companded counterpart (quant_grp8_compound, :365-388); n is a multiple of 32 here.
__device__ inline void encode_grp12(Team& T, int lane, const BlockLayout& L, uint32_t* img, int iters, float smult) {
    using G = Grid<12, true>;
    const int n = L.n, ng = n / 32;
    const uint32_t cap = (uint32_t)L.bytes * 8u;
    fit_groups32<G>(T, lane, ng, iters, smult);
    each(lane, n, [&](int i) {
        const float s = T.gs[i >> 5];
        put_bits(img, cap, (uint32_t)(12 * i), s > 0.0f ? G::pick(T.w[i] / s) : 0u, 12);
    });
    if (lane < ng) put_bits(img, cap, (uint32_t)(12 * n + 16 * lane), float_to_half_bits(T.gs[lane]), 16);
}

__device__ inline void encode_grp8(Team& T, int lane, const BlockLayout& L, uint32_t* img, float smult) {
    const int n = L.n, ng = n / 32, g = lane >> 3, tl = lane & 7;  // eight lanes per group, all groups at once
    const uint32_t cap = (uint32_t)L.bytes * 8u;
    Comp8Team<32, 8> team;
    team.lv = T.table;
    team.first = lane & ~7;
    float m = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        team.w[k] = T.w[32 * min(g, ng - 1) + 4 * tl + k];  // (lanes past the last group repeat it and store nothing)
        m = fmaxf(m, fabsf(team.w[k]));
    }
#pragma unroll
    for (int sft = 4; sft >= 1; sft >>= 1) m = fmaxf(m, __shfl_xor(m, sft, 64));
    const float s = team.fit((double)m) * smult;
    if (g >= ng) return;
#pragma unroll
    for (int k = 0; k < 4; ++k) put_bits(img, cap, (uint32_t)(8 * (32 * g + 4 * tl + k)), (s > 0.0f) ? team.nearest(team.w[k] / s) : 0u, 8);
    if (tl == 0) put_bits(img, cap, (uint32_t)(8 * n + 16 * g), float_to_half_bits(s), 16);
}

// ------------------------------------------------------------------------------------------------
// Affine groups (quant_affine with grp16_fit_affine, :1337-1521): ng whole groups of gsz weights, each with a
// scale code and an offset code under two binary16 super-values.  Lane g owns group g; lane 0 the sums over
// groups.  Only the whole groups are written: the levels of ng * gsz weights, then the header at once.
template <int BITS, int GSZ>
__device__ void encode_affine(Team& T, int lane, const BlockLayout& L, uint32_t* img) {
    constexpr int bits = BITS, gsz = GSZ;
    const int ng = L.ng;
    const int scq = (1 << L.scb) - 1, mq = (1 << L.mb) - 1, bias = (mq + 1) / 2;
    const uint32_t cap = (uint32_t)L.bytes * 8u;
    const bool own = lane < ng;
    const float* x = T.w + (own ? lane : 0) * gsz;
    const float* lev = T.lev + (own ? lane : 0) * gsz;
    double sx = 0;  // the same in every refit
#pragma unroll
    for (int i = 0; i < gsz; ++i) sx += (double)x[i];
    // T.lev = the levels that every group's offset and scale (the lanes' own values) assign to its weights
    auto assign = [&](float m, float s) {
        if (own) { T.gm[lane] = m; T.gtry[lane] = s; }
        __syncthreads();
        each(lane, ng * gsz, [&](int i) { T.lev[i] = unit_level(bits, unit_pick((T.w[i] - T.gm[i / gsz]) / T.gtry[i / gsz], bits)); });
        __syncthreads();
    };
    // least squares of the group's weights over the assigned levels
    auto lsq = [&](bool square_in_float, float* s_out, float* m_out) {
        constexpr double sw = (double)gsz;
        double sl = 0, sl2 = 0, sxl = 0;
#pragma unroll
        for (int i = 0; i < gsz; ++i) {
            const float lf = lev[i];
            const double l = (double)lf;
            sl += l;
            if (square_in_float) sl2 += lf * lf; else sl2 = __builtin_fma(l, l, sl2);
            sxl = __builtin_fma((double)x[i], l, sxl);
        }
        const double D = __builtin_fma(sw, sl2, -(sl * sl));
        if (D > 1e-20) {
            *s_out = (float)(__builtin_fma(sw, sxl, -(sx * sl)) / D);
            *m_out = (float)(__builtin_fma(sl2, sx, -(sl * sxl)) / D);
        }
    };
    float hi = -1e30f, lo = 1e30f;
#pragma unroll
    for (int i = 0; i < gsz; ++i) { hi = fmaxf(hi, x[i]); lo = fminf(lo, x[i]); }
    float s = hi - lo, m = lo;
    const bool flat = !(fabsf(s) > 1e-30f);  // stays at scale and offset zero
    for (int it = 0; it < 5; ++it) {
        if (it == 4) {
            // the scale 5, 10, 15 % up and down: the first with the smallest squared error stays
            float keep = s;
            double least = 1e300;
            for (int k = -3; k <= 3; ++k) {
                if (k == 0) continue;
                const float cs = s * __builtin_fmaf(0.05f, (float)k, 1.0f);
                assign(m, cs);
                double e = 0.0;
#pragma unroll
                for (int i = 0; i < gsz; ++i) {
                    const float r = __builtin_fmaf(cs, lev[i], m) - x[i];
                    e = __builtin_fma((double)r, (double)r, e);
                }
                if (e < least) { least = e; keep = cs; }
            }
            s = keep;
        }
        assign(m, s);
        lsq(false, &s, &m);
    }
    if (own) {
        T.gs[lane] = flat ? 0.0f : s;
        T.gm[lane] = flat ? 0.0f : m;
        T.gc[lane] = 0;
        T.gk[lane] = 0;
    }
    __syncthreads();
    if (lane == 0) {
        float top_s = 0.0f, top_m = 0.0f;
        for (int g = 0; g < ng; ++g) { top_s = fmaxf(top_s, fabsf(T.gs[g])); top_m = fmaxf(top_m, fabsf(T.gm[g])); }
        const bool dead = top_s <= kTiny, offsets = top_m > kTiny;
        T.f0 = dead ? 0.0f : half_bits_to_float(float_to_half_bits(top_s / (float)scq));
        T.f1 = (!dead && offsets) ? half_bits_to_float(float_to_half_bits(top_m / (float)bias)) : 1.0f;
        T.i0 = (dead ? 1 : 0) | (offsets ? 2 : 0);
    }
    __syncthreads();
    const bool dead = (T.i0 & 1) != 0, offsets = (T.i0 & 2) != 0;
    __syncthreads();
    auto scale_code = [&](float s, float d) __attribute__((always_inline)) { return (s == 0.0f) ? 0 : max(0, min(scq, (int)lroundf(s / d))); };
    auto offset_code = [&](float m, float dm) __attribute__((always_inline)) { return max(-bias, min(mq - bias, (int)lroundf(-m / dm))); };
    if (!dead) {
        if (lane < ng) {
            T.gc[lane] = scale_code(T.gs[lane], T.f0);
            if (offsets) T.gk[lane] = offset_code(T.gm[lane], T.f1);
        }
        __syncthreads();
        for (int it = 0; it < 5; ++it) {
            const float d = T.f0, dm = T.f1;
            const float es = own ? d * (float)T.gc[lane] : 0.0f, em = own ? -dm * (float)T.gk[lane] : 0.0f;
            const float gm = own ? T.gm[lane] : 0.0f;  // (assign() takes the place for em)
            assign(em, es);
            if (own) {
                T.gm[lane] = gm;
                if (es != 0.0f) lsq(true, &T.gs[lane], &T.gm[lane]);
                T.gc[lane] = scale_code(T.gs[lane], d);
            }
            __syncthreads();
            if (lane == 0) {
                double num = 0, den = 0;
                for (int g = 0; g < ng; ++g) {
                    num = __builtin_fma((double)T.gs[g], (double)T.gc[g], num);
                    den = __builtin_fma((double)T.gc[g], (double)T.gc[g], den);
                }
                float nd = (den > 1e-20) ? half_bits_to_float(float_to_half_bits((float)(num / den))) : 0.0f;
                T.f0 = fabsf(nd) <= kTiny ? 0.0f : nd;
            }
            if (lane < ng) T.gk[lane] = (fabsf(dm) > kTiny) ? offset_code(T.gm[lane], dm) : 0;
            __syncthreads();
            if (lane == 0) {
                double num = 0, den = 0;
                for (int g = 0; g < ng; ++g) {
                    num = __builtin_fma(-(double)T.gm[g], (double)T.gk[g], num);
                    den = __builtin_fma((double)T.gk[g], (double)T.gk[g], den);
                }
                float nd = (den > 1e-20) ? half_bits_to_float(float_to_half_bits((float)(num / den))) : 0.0f;
                T.f1 = fabsf(nd) <= kTiny ? 0.0f : nd;
            }
            __syncthreads();
        }
    }
    const float d = T.f0, dm = T.f1;
    const int covered = ng * gsz;
    each(lane, covered, [&](int i) {
        const int g = i / gsz;
        const float es = d * (float)T.gc[g], em = -dm * (float)T.gk[g];
        put_bits(img, cap, (uint32_t)(i * bits), (es == 0.0f) ? 0u : unit_pick((T.w[i] - em) / es, bits), bits);
    });
    const uint32_t head = (uint32_t)(covered * bits);
    if (lane < ng) {
        put_bits(img, cap, head + (uint32_t)(lane * L.scb), (uint32_t)T.gc[lane], L.scb);
        put_bits(img, cap, head + (uint32_t)(ng * L.scb + lane * L.mb), (uint32_t)(T.gk[lane] + bias), L.mb);
    }
    if (lane == 0) {
        const uint32_t tail = head + (uint32_t)(ng * (L.scb + L.mb));
        put_bits(img, cap, tail, float_to_half_bits(d), 16);
        put_bits(img, cap, tail + 16, float_to_half_bits(dm), 16);
    }
}

// ------------------------------------------------------------------------------------------------
// Grouped-lattice fallback (quant_grp16 with grp16_fit_scale, :739-914) in its three short forms: bare codes,
// one binary16 scale for the block, or a 3-bit scale code per 8 weights under a binary16 super-scale.
//
// One scale for a run: four (assign, refit) rounds, the scale 5, 10, 15 % up and down by squared error, a
// closing refit.
template <class G>
__device__ float fallback_fit_block(Team& T, int lane, int n) {
    float m = 0.0f;
    each(lane, n, [&](int i) { m = fmaxf(m, fabsf(T.w[i])); });
    m = wave_max(m);
    float s = (m > 1e-30f) ? m / G::top() : 0.0f;
    if (!(fabsf(s) > 1e-30f)) return 0.0f;
    for (int it = 0; it < 5; ++it) {
        if (it == 4) {
            float keep = s;
            double least = 1e300;
            for (int k = -3; k <= 3; ++k) {
                if (k == 0) continue;
                const float cs = s * __builtin_fmaf(0.05f, (float)k, 1.0f);
                each(lane, n, [&](int i) { T.lev[i] = __builtin_fmaf(cs, G::level(G::pick(T.w[i] / cs)), -T.w[i]); });
                __syncthreads();
                if (lane == 0) {
                    double unused;
                    dots_in_order(T.lev, T.lev, n, &T.d0, &unused);
                }
                __syncthreads();
                const double e = T.d0;
                __syncthreads();
                if (e < least) { least = e; keep = cs; }
            }
            s = keep;
        }
        each(lane, n, [&](int i) { T.lev[i] = G::level(G::pick(T.w[i] / s)); });
        __syncthreads();
        if (lane == 0) {
            double num, den;
            dots_in_order(T.w, T.lev, n, &num, &den);
            T.f0 = (den > 1e-20) ? (float)(num / den) : s;
        }
        __syncthreads();
        s = T.f0;
        __syncthreads();
    }
    return s;
}

template <int BITS>
__device__ void encode_fallback(Team& T, int lane, const BlockLayout& L, uint32_t* img) {
    using G = Grid<BITS, false>;
    constexpr int bits = BITS;
    const int n = L.n;
    const uint32_t cap = (uint32_t)L.bytes * 8u;
    if (L.aux == 0) {
        each(lane, n, [&](int i) { put_bits(img, cap, (uint32_t)(i * bits), G::pick(T.w[i]), bits); });
        return;
    }
    if (L.aux == 1) {
        float d = fallback_fit_block<G>(T, lane, n);
        if (!(fabsf(d) > kTiny)) d = 0.0f;
        each(lane, n, [&](int i) { put_bits(img, cap, (uint32_t)(i * bits), (d == 0.0f) ? 0u : G::pick(T.w[i] / d), bits); });
        if (lane == 0) put_bits(img, cap, (uint32_t)(((n * bits + 7) / 8) * 8), float_to_half_bits(d), 16);
        return;
    }
    const int ng = L.ng;  // whole groups of eight
    const bool own = lane < ng;
    const float* x = T.w + (own ? lane : 0) * 8;
    const float* lev = T.lev + (own ? lane : 0) * 8;
    // T.lev = the levels of the groups' weights under the scales the lanes hold
    auto assign = [&](float s) {
        if (own) T.gtry[lane] = s;
        __syncthreads();
        each(lane, 8 * ng, [&](int i) { T.lev[i] = G::level(G::pick(T.w[i] / T.gtry[i >> 3])); });
        __syncthreads();
    };
    auto refit = [&](float* s) {  // false where the levels give no support
        double num = 0.0, den = 0.0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float l = lev[i];
            num = __builtin_fma((double)x[i], (double)l, num);
            den = __builtin_fma((double)l, (double)l, den);
        }
        if (den > 1e-20) *s = (float)(num / den);
        return den > 1e-20;
    };
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) m = fmaxf(m, fabsf(x[i]));
    float s = (m > 1e-30f) ? m / G::top() : 0.0f;
    const bool flat = !(fabsf(s) > 1e-30f);
    for (int it = 0; it < 5; ++it) {
        if (it == 4) {
            float keep = s;
            double least = 1e300;
            for (int k = -3; k <= 3; ++k) {
                if (k == 0) continue;
                const float cs = s * __builtin_fmaf(0.05f, (float)k, 1.0f);
                assign(cs);
                double e = 0.0;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float r = __builtin_fmaf(cs, lev[i], -x[i]);
                    e = __builtin_fma((double)r, (double)r, e);
                }
                if (e < least) { least = e; keep = cs; }
            }
            s = keep;
        }
        assign(s);
        refit(&s);
    }
    if (own) {
        T.gs[lane] = flat ? 0.0f : s;
        T.gc[lane] = 0;
    }
    __syncthreads();
    if (lane == 0) {
        float top_s = 0.0f;
        for (int k = 0; k < ng; ++k) top_s = fmaxf(top_s, fabsf(T.gs[k]));
        T.f0 = (top_s <= kTiny) ? 0.0f : half_bits_to_float(float_to_half_bits(top_s / 7.0f));
    }
    __syncthreads();
    // (once d has collapsed to zero the reference's lround(s / 0) comes out as 0 after its clamp)
    auto scale_code = [&](float s, float d) __attribute__((always_inline)) { return (s == 0.0f || d == 0.0f) ? 0 : max(0, min(7, (int)lroundf(s / d))); };
    if (T.f0 != 0.0f) {
        if (lane < ng) T.gc[lane] = scale_code(T.gs[lane], T.f0);
        __syncthreads();
        for (int it = 0; it < 5; ++it) {
            const float d = T.f0;
            const float eff = own ? d * (float)T.gc[lane] : 0.0f;
            assign(eff);
            if (own) {
                if (eff != 0.0f && !refit(&T.gs[lane])) T.gs[lane] = 0.0f;
                T.gc[lane] = scale_code(T.gs[lane], d);
            }
            __syncthreads();
            if (lane == 0) {
                double num = 0.0, den = 0.0;
                for (int k = 0; k < ng; ++k) {
                    num = __builtin_fma((double)T.gs[k], (double)T.gc[k], num);
                    den = __builtin_fma((double)T.gc[k], (double)T.gc[k], den);
                }
                float nd = half_bits_to_float(float_to_half_bits((den > 1e-20) ? (float)(num / den) : 0.0f));
                T.f0 = fabsf(nd) <= kTiny ? 0.0f : nd;
            }
            __syncthreads();
        }
    }
    const float d = T.f0;
    each(lane, n, [&](int i) {  // the weights behind the last whole group go with its scale
        const float eff = d * (float)T.gc[min(i >> 3, ng - 1)];
        put_bits(img, cap, (uint32_t)(i * bits), (eff == 0.0f) ? 0u : G::pick(T.w[i] / eff), bits);
    });
    if (lane < ng) put_bits(img, cap, (uint32_t)(n * bits + 3 * lane), (uint32_t)T.gc[lane], 3);
    if (lane == 0) put_bits(img, cap, (uint32_t)(n * bits + 3 * ng), float_to_half_bits(d), 16);
}

// ------------------------------------------------------------------------------------------------
// Q_G_6 (quant_6k, :1070-1238): signed 6-bit levels; bare below eight weights, one binary16 d up to the
// size that has room for scales, else an int8 scale per 16 weights under d.
__device__ inline void encode_six(Team& T, int lane, const BlockLayout& L, uint32_t* img, int passes, int giters, int polish, int joint) {
    const int n = L.n;
    const uint32_t cap = (uint32_t)L.bytes * 8u;
    const int level_bytes = (n * 6 + 7) / 8, ng = L.aux >> 8;
    if (!(L.aux & 1)) {
        each(lane, n, [&](int i) { put_bits(img, cap, (uint32_t)(6 * i), (uint32_t)(six_level(T.w[i]) + 32), 6); });
        return;
    }
    if (ng == 0) {
        // one d by least squares weighted with (mean |w| + |w|) (:1095-1125)
        float m = 0.0f;
        each(lane, n, [&](int i) { m = fmaxf(m, fabsf(T.w[i])); T.lev[i] = fabsf(T.w[i]); });
        m = wave_max(m);
        __syncthreads();
        if (lane == 0) {
            float av = 0.0f;
#pragma unroll 8
            for (int i = 0; i < n; ++i) av += T.lev[i];
            T.f1 = av / (float)n;
        }
        __syncthreads();
        const float av = T.f1;
        float d = m / 32.0f;
        for (int pass = 0; pass < passes; ++pass) {
            each(lane, n, [&](int i) { T.lev[i] = (float)six_level(T.w[i] / d); });
            __syncthreads();
            if (lane == 0) {
                double num = 0.0, den = 0.0;
#pragma unroll 8
                for (int i = 0; i < n; ++i) {
                    const double wgt = (double)(av + fabsf(T.w[i])), l = (double)T.lev[i];
                    num += wgt * (double)T.w[i] * l;
                    den += wgt * l * l;
                }
                T.f0 = (den > 1e-20) ? (float)(num / den) : d;
            }
            __syncthreads();
            d = T.f0;
            __syncthreads();
        }
        if (!(fabsf(d) > kTiny)) d = 0.0f;
        each(lane, n, [&](int i) { put_bits(img, cap, (uint32_t)(6 * i), (uint32_t)(((d == 0.0f) ? 0 : six_level(T.w[i] / d)) + 32), 6); });
        if (lane == 0) put_bits(img, cap, (uint32_t)(8 * level_bytes), float_to_half_bits(d), 16);
        return;
    }
    const bool own = lane < ng;
    const float* x = T.w + (own ? lane : 0) * 16;
    const float* lev = T.lev + (own ? lane : 0) * 16;
    // T.lev = the levels of the groups' weights under the scales the lanes hold
    auto assign = [&](float s) {
        if (own) T.gtry[lane] = s;
        __syncthreads();
        each(lane, 16 * ng, [&](int i) { T.lev[i] = (float)six_level(T.w[i] / T.gtry[i >> 4]); });
        __syncthreads();
    };
    auto refit16 = [&](float* out) {
        double num = 0.0, den = 0.0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const double l = (double)lev[i];
            num = __builtin_fma((double)x[i], l, num);
            den = __builtin_fma(l, l, den);
        }
        if (den > 1e-20) *out = (float)(num / den);
    };
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) m = fmaxf(m, fabsf(x[i]));
    float sg = (m > kTiny) ? m / 32.0f : 0.0f;
    const bool flat = fabsf(sg) <= kTiny;
    for (int it = 0; it <= giters; ++it) {
        if (it == giters) {
            float keep = sg;
            double least = 1e300;
            for (int k = -polish; k <= polish; ++k) {
                if (k == 0) continue;
                const float cs = sg * __builtin_fmaf(0.05f, (float)k, 1.0f);
                assign(cs);
                double e = 0.0;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float r = __builtin_fmaf(cs, lev[i], -x[i]);
                    e = __builtin_fma((double)r, (double)r, e);
                }
                if (e < least) { least = e; keep = cs; }
            }
            sg = keep;
        }
        assign(sg);
        refit16(&sg);
    }
    if (own) {
        T.gs[lane] = flat ? 0.0f : sg;
        T.gc[lane] = 0;
    }
    __syncthreads();
    float top_s = 0.0f;
    for (int g = 0; g < ng; ++g) top_s = fmaxf(top_s, fabsf(T.gs[g]));
    if (top_s <= kTiny) {
        if (lane == 0) T.f0 = 0.0f;
        __syncthreads();
    } else {
        const float iscale = -128.0f / top_s;
        if (lane == 0) T.f0 = 1.0f / iscale;
        // the product feeds the rounding add directly: one fused operation in the reference's build
        if (lane < ng) T.gc[lane] = max(-127, min(127, (int)(__float_as_uint(__builtin_fmaf(iscale, T.gs[lane], 12582912.f)) & 0x007fffffu) - 0x00400000));
        __syncthreads();
        for (int it = 0; it < joint; ++it) {
            const float d = T.f0;
            const float eff = own ? d * (float)T.gc[lane] : 0.0f;
            assign(eff);
            if (own) {
                if (eff != 0.0f) {
                    float fitted = 0.0f;
                    refit16(&fitted);
                    T.gs[lane] = fitted;
                }
                T.gc[lane] = (d == 0.0f) ? 0 : max(-127, min(127, six_round(T.gs[lane] / d)));
            }
            __syncthreads();
            if (lane == 0) {
                double num = 0.0, den = 0.0;
                for (int g = 0; g < ng; ++g) {
                    num = __builtin_fma((double)T.gs[g], (double)T.gc[g], num);
                    den = __builtin_fma((double)T.gc[g], (double)T.gc[g], den);
                }
                const float nd = (den > 1e-20) ? (float)(num / den) : 0.0f;
                T.f0 = fabsf(nd) <= kTiny ? 0.0f : nd;
            }
            __syncthreads();
        }
    }
    const float d = T.f0;
    each(lane, n, [&](int i) {
        const float eff = d * (float)T.gc[min(i >> 4, ng - 1)];
        put_bits(img, cap, (uint32_t)(6 * i), (uint32_t)(((eff == 0.0f) ? 0 : six_level(T.w[i] / eff)) + 32), 6);
    });
    if (lane < ng) put_bits(img, cap, (uint32_t)(8 * (level_bytes + lane)), (uint32_t)(uint8_t)(int8_t)T.gc[lane], 8);
    if (lane == 0) put_bits(img, cap, (uint32_t)(8 * (level_bytes + ng)), float_to_half_bits(d), 16);
}

// ------------------------------------------------------------------------------------------------
// Sign formats (:2434-2449, :2523-2549): fewer than 32 weights are bare signs; otherwise a binary16 scale and
// the signs of the weights that are not slots.  Lane c evaluates candidate scale c.
__device__ inline void encode_signs(Team& T, int lane, const BlockLayout& L, uint32_t* img, int tier) {
    const int n = L.n;
    const uint32_t cap = (uint32_t)L.bytes * 8u;
    if (n < 32) {
        for (int i = lane; i < n; i += 64) put_bits(img, cap, (uint32_t)i, T.w[i] >= 0.0f ? 1u : 0u, 1);
        return;
    }
    if (tier < 0) {  // Q_1: sqrt(mean w^2)
        if (lane == 0) {
            double sum, same;
            dots_in_order(T.w, T.w, n, &sum, &same);
            T.i0 = (int)float_to_half_bits((float)sqrt(sum / (double)n));
        }
    } else {
        if (lane == 0) {
            double sum_abs = 0.0;
            int kept = 0;
            for (int i = 0; i < n; ++i)
                if (!slot_at(i, n)) { sum_abs += fabs((double)T.w[i]); ++kept; }
            T.i0 = kept ? (int)float_to_half_bits((float)(sum_abs / kept)) : -1;
        }
        __syncthreads();
        const int h0 = T.i0;
        __syncthreads();
        if (h0 >= 0) {
            // candidate c: 0 = h0, 1 .. rad = h0 - rad .. h0 - 1, rad + 1 .. 2 rad = h0 + 1 .. h0 + rad
            const int rad = tier == 0 ? 4 : tier == 1 ? 10 : 24;
            auto delta_of = [&](int c) __attribute__((always_inline)) { return c == 0 ? 0 : c <= rad ? c - rad - 1 : c - rad; };
            if (lane <= 2 * rad) {
                const int hc = h0 + delta_of(lane);
                double e = -1.0;  // outside binary16: skipped
                if (hc >= 0 && hc <= 0xFFFF) {
                    const float sc = half_bits_to_float((uint32_t)hc);
                    e = 0.0;
                    for (int i = 0; i < n; ++i) {
                        if (slot_at(i, n)) continue;
                        const double r = (double)T.w[i] - (T.w[i] >= 0 ? (double)sc : -(double)sc);
                        e = __builtin_fma(r, r, e);
                    }
                }
                T.dres[lane] = e;
            }
            __syncthreads();
            if (lane == 0) {
                int best = h0;
                double least = T.dres[0];
                for (int c = 1; c <= 2 * rad; ++c)
                    if (T.dres[c] >= 0.0 && T.dres[c] < least) { least = T.dres[c]; best = h0 + delta_of(c); }
                T.i0 = best;
            }
        } else if (lane == 0) {
            T.i0 = 0;  // no weight is kept: scale 0
        }
    }
    __syncthreads();
    if (lane == 0) put_bits(img, cap, 0, (uint32_t)T.i0, 16);
    for (int i = lane; i < n; i += 64)
        if (!slot_at(i, n)) put_bits(img, cap, (uint32_t)(16 + i - slots_before(i, n)), T.w[i] >= 0.0f ? 1u : 0u, 1);
}

// 16- and 24-bit formats: fewer than 256 weights are raw binary16 / the top three bytes of the binary32; the
// grouped ids append a binary16 mean of (w - decoded) per 32 weights (:1690-1873, :2450-2493)
__device__ inline void encode_wide(Team& T, int lane, const BlockLayout& L, uint32_t* img) {
    const int n = L.n, width = L.bits;
    const uint32_t cap = (uint32_t)L.bytes * 8u;
    for (int i = lane; i < n; i += 64) {
        const uint32_t u = __float_as_uint(T.w[i]);
        if (width == 16) {
            const uint32_t h = float_to_half_bits(T.w[i]);
            put_bits(img, cap, (uint32_t)(16 * i), h, 16);
            T.lev[i] = half_bits_to_float(h);
        } else {
            put_bits(img, cap, (uint32_t)(24 * i), u >> 8, 24);
            T.lev[i] = __uint_as_float(u & 0xFFFFFF00u);
        }
    }
    __syncthreads();
    if ((L.aux & 1) && lane < n / 32) {
        double mean = 0.0;
        for (int i = 32 * lane; i < 32 * lane + 32; ++i) mean += (double)T.w[i] - (double)T.lev[i];
        put_bits(img, cap, (uint32_t)(width * n + 16 * lane), float_to_half_bits((float)(mean / 32.0)), 16);
    }
}

// ------------------------------------------------------------------------------------------------
// true when the candidate image decodes with a strictly smaller mean squared error than the block's
__device__ inline bool candidate_wins(Team& T, int lane, const BlockLayout& L) {
    const uint8_t* cur = reinterpret_cast<const uint8_t*>(T.img[0]);
    const uint8_t* cand = reinterpret_cast<const uint8_t*>(T.img[1]);
    for (int i = lane; i < L.n; i += 64) {
        T.lev[i] = decode_weight_short(L, cur, (uint32_t)i);
        T.dres[i] = (double)decode_weight_short(L, cand, (uint32_t)i);
    }
    __syncthreads();
    if (lane == 0) {
        double ec = 0.0, en = 0.0;
        for (int i = 0; i < L.n; ++i) {
            const double x = (double)T.w[i], a = x - (double)T.lev[i], b = x - T.dres[i];
            ec = __builtin_fma(a, a, ec);
            en = __builtin_fma(b, b, en);
        }
        T.i0 = (en / (double)L.n) < (ec / (double)L.n);
    }
    __syncthreads();
    const bool take = T.i0 != 0;
    __syncthreads();
    return take;
}

// One workgroup of 64 lanes encodes the job's block.
template <int FMT>
__device__ __forceinline__ void encode_short_block(const ShortJob& job, Team& T) {
    constexpr Spec sp = spec_of(FMT);
    const BlockLayout& L = job.L;
    const int lane = threadIdx.x, n = L.n, words = (L.bytes + 3) / 4;
    for (int i = lane; i < n; i += 64) T.w[i] = job.w[i];
    for (int i = lane; i < kMaxShortBytes / 4; i += 64) { T.img[0][i] = 0; T.img[1][i] = 0; }
    if constexpr (sp.bits == 8)
        for (int i = lane; i < 256; i += 64) T.table[i] = __uint_as_float(kComp8Bits[i]);
    __syncthreads();
    // the further tries of the _K_M (one) and _K_H (all) ids, each kept only where it decodes strictly better
    // (:2551-2665, :2733-2824); `encode_try(c)` writes try c into the candidate image
    auto search = [&](int count, auto&& encode_try) {
        for (int c = 0; c < count; ++c) {
            for (int i = lane; i < words; i += 64) T.img[1][i] = 0;
            __syncthreads();
            encode_try(c);
            __syncthreads();
            if (candidate_wins(T, lane, L))
                for (int i = lane; i < words; i += 64) T.img[0][i] = T.img[1][i];
            __syncthreads();
        }
    };
    const int tries = job.tier >= 2 ? 6 : 1;
    if constexpr (sp.codec == Codec::Raw32) {
        for (int i = lane; i < n; i += 64) T.img[0][i] = __float_as_uint(T.w[i]);
    } else if constexpr (sp.codec == Codec::Q1) {
        encode_signs(T, lane, L, T.img[0], job.tier);
    } else if constexpr (sp.codec == Codec::Q16 || sp.codec == Codec::Q24) {
        encode_wide(T, lane, L, T.img[0]);
    } else if constexpr (sp.codec == Codec::Q6K) {
        const int effort[3][4] = {{2, 4, 3, 3}, {5, 8, 5, 6}, {10, 14, 8, 10}};
        for (int c = -1; c < (job.tier >= 2 ? 2 : job.tier); ++c) {
            auto one = [&](uint32_t* img) { encode_six(T, lane, L, img, effort[c + 1][0], effort[c + 1][1], effort[c + 1][2], effort[c + 1][3]); };
            if (c < 0) { one(T.img[0]); __syncthreads(); }
            else search(1, [&](int) { one(T.img[1]); });
        }
    } else {
        constexpr bool fixed = sp.codec == Codec::Fixed || sp.codec == Codec::Grp12;
        if (L.kind == BK_LEVELS || L.kind == BK_LATTICE) {
            if constexpr (sp.codec == Codec::Lattice || sp.codec == Codec::Fixed || sp.codec == Codec::Grp12) {
                const float start[6] = {1.0f, 1.0f, 0.9f, 1.1f, 0.7f, 1.3f};
                encode_lattice<sp.bits, fixed>(T, lane, L, T.img[0], fixed ? 3 : 2, 1.0f);
                __syncthreads();
                if (job.tier > 0)
                    search(tries, [&](int c) { encode_lattice<sp.bits, fixed>(T, lane, L, T.img[1], c == 0 ? (fixed ? 10 : 6) : (fixed ? 24 : 14), start[c]); });
            }
        } else if (L.kind == BK_GRP12) {
            if constexpr (sp.codec == Codec::Grp12) {
                const int its[6] = {8, 8, 20, 20, 20, 20};
                const float start[6] = {1.0f, 1.0f, 0.93f, 1.07f, 0.7f, 1.3f};
                encode_grp12(T, lane, L, T.img[0], 3, 1.0f);
                __syncthreads();
                if (job.tier > 0) search(tries, [&](int c) { encode_grp12(T, lane, L, T.img[1], its[c], start[c]); });
            }
        } else if (L.kind == BK_GRP8) {
            if constexpr (sp.codec == Codec::Grp8) {
                const float start[6] = {0.7f, 0.9f, 0.95f, 1.05f, 1.1f, 1.3f};
                const int count = job.tier >= 2 ? 6 : 2;
                encode_grp8(T, lane, L, T.img[0], 1.0f);
                __syncthreads();
                if (job.tier > 0) search(count, [&](int c) { encode_grp8(T, lane, L, T.img[1], start[6 - count + c]); });
            }
        } else if (L.kind == BK_AFFINE) {
            if constexpr (sp.codec == Codec::Affine || sp.codec == Codec::Grp16) encode_affine<sp.bits, sp.gsz>(T, lane, L, T.img[0]);
            else if constexpr (sp.codec == Codec::Grp8) encode_affine<8, 32>(T, lane, L, T.img[0]);
        } else if (L.kind == BK_GRP16) {
            if constexpr (sp.codec == Codec::Affine || sp.codec == Codec::Grp16 || sp.codec == Codec::Grp8 || sp.codec == Codec::Grp12)
                encode_fallback<sp.bits>(T, lane, L, T.img[0]);
        }
    }
    __syncthreads();
    const uint8_t* image = reinterpret_cast<const uint8_t*>(T.img[0]);
    for (int i = lane; i < L.bytes; i += 64) job.dst[i] = image[i];
}

// The block in a launch of its own, for the formats whose encoder does not take it along.
template <int FMT>
__global__ __launch_bounds__(64) void encode_short_kernel(ShortJob job) {
    __shared__ Team T;
    encode_short_block<FMT>(job, T);
}

}  // namespace

}  // namespace tfq
