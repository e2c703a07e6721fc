// Shared by the split matrix-core form of the L2 Similarity modes (similarity_split.hip) and the direct kernels that
// pack its parameters and recompute the tiles it flags (similarity_direct.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "fast_div.h"
#include "internal.h"
#include "sim_step.h"

namespace simnets {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kSplitPixels = 128;   // output pixels of a workgroup, consecutive over the whole batch
constexpr int kSplitRows = 32;      // templates of one matrix tile
constexpr float kSplitLogScale = 512.0f;   // of the logarithm terms, at most 120 in size
constexpr int kSplitMaxC = 4096;    // channels whose centres and scales the packing kernel keeps in LDS

// Geometry of one call on the split form.
struct SplitPlan {
    bool on;
    int cg;       // channels of a staged chunk: 16 (a matrix step is one tap) or 8 (a step is two taps)
    int chunks;   // ceil(C / cg)
    int steps;    // matrix steps per chunk: taps, or ceil(taps / 2)
    int pieces;   // 16-bit pieces of the packed parameters per step: 4, with missing values 8 (input gradient: 6)
    int n_mtiles; // ceil(O / 32)
    int n_ptiles; // ceil(B oh ow / 128)
    int Wp, Hv;   // columns of a staged row; rows of one image's staged stack
    size_t packed, chan, rows, flags, exact, logs, total;   // workspace, from its own start
};

SplitPlan sim_split_plan(const SimPlan &p);

// Per template four floats: what the sums of a row lack (bias, in two floats; with missing values the guard: outputs below
// it times the sum of the present w (t'^2 + m / s^2) are recomputed), the power of two that takes back what the packed
// parameters were multiplied by, and the line below which outputs are recomputed.  Behind those of the n_mtiles * 32
// templates the constants of the normalized modes, and pairs by which the line rises with the staged values.
enum SplitRow { SPLIT_BIAS, SPLIT_BIAS_LESSER, SPLIT_UNSCALE, SPLIT_THR, SPLIT_GUARD = SPLIT_BIAS };
// Per channel, [level][field][chunks * cg], zeros behind the last channel: the scale s, -c s, and m.
enum SplitChannel { SPLIT_S, SPLIT_NCS, SPLIT_M, SPLIT_CHANNEL_FIELDS };

struct SplitPack {
    const float *templates, *weights;
    unsigned short *packed;
    float *chan, *rows;
    float2 *exact;   // [O][K] template and negative weight as the term-by-term kernels take them ...
    float *logs;     // ... and the normalized modes' logarithm terms
    int O, C, taps, K, cg, chunks, steps, pieces, n_mtiles, mode;
    float fudge, norm_const;
    float line;   // outputs below `line` times sum w t'^2 are recomputed term by term
    float *ctr;   // input gradient: centres of the rows
    int pack_blocks;   // ... workgroups of its packing launch, chunks * n_mtiles * ceil(steps / 4)
    FastDiv d_taps, d_steps;
    int blocks;   // of the packing launch: each template of the n_mtiles * 32, one at a time
};

int sim_split_launch(const SimPlan &p, const SplitPlan &sp, const float *input, float *output, char *ws, hipStream_t s);
SplitPack sim_split_pack_args(const SimPlan &p, const SplitPlan &sp, const float *templates, const float *weights,
                              char *ws);

// Parameter gradients (similarity_split_params.hip).
struct SplitParamsPlan {
    bool on;
    int n_mtiles, m_groups, k_groups, TH, TW, rows, cols, pitch, chan, tiles_r, tiles_c, units, S, Opad, Kpad;
    size_t partial, centres, ctr, ctr64, spread, packed, total;
};

SplitParamsPlan sim_split_params_plan(const SimPlan &p);
int sim_split_params_launch(const SimPlan &p, const SplitParamsPlan &sp, const float *input, const float *templates,
                            const float *output_grad, char *ws, hipStream_t s);

// v = p0 + p1 + p2, each the nearest 16-bit value to what is left: 24 bits of mantissa, exact for every v whose pieces
// are normal numbers.
__device__ __forceinline__ void split3(float v, __bf16 &p0, __bf16 &p1, __bf16 &p2)
{
    p0 = (__bf16)v;
    const float r = v - (float)p0;
    p1 = (__bf16)r;
    p2 = (__bf16)(r - (float)p1);
}

// The same for values that may be infinite or NaN, which stay in one piece.
__device__ __forceinline__ void split3_any(float v, __bf16 &p0, __bf16 &p1, __bf16 &p2)
{
    split3(v, p0, p1, p2);
    const bool finite = __builtin_fabsf(v) < INFINITY;
    p1 = finite ? p1 : (__bf16)0.0f;
    p2 = finite ? p2 : (__bf16)0.0f;
}

// A sum of products of such pieces, hi the leading one's and lo the lesser ones'.  An infinite factor meets the other's
// lesser pieces, zeros and either sign among them, so lo says nothing there; hi holds the infinity with the sign it has.
__device__ __forceinline__ float split_sum(float hi, float lo)
{
    return __builtin_isfinite(hi) ? hi + lo : hi;
}

// v = hi + lo / 2048, each the nearest half-precision value to what is left: 24 bits for |v| from 2^-14 to 65504, and to
// 2^-36 absolutely below that.  A v beyond 65504 gives an infinity and a NaN.
constexpr float kSplitLow = 2048.0f;
// The forward's scales: levels of 2^-3 of the packed ones (a parameter times 2^-24 is still a half-precision value; with missing
// values the lesser pieces meet twice as much).
constexpr int kSplitLevels = 9, kSplitMaskedLevels = 5, kSplitLevelBits = 3;
constexpr float kSplitParamShare = 0.07f;   // 2^-25.8 / 2^-22
constexpr float kSplitSeen = 2.0f;     // staged values up to this need no attention
constexpr float kSplitMost = 181.0f;   // the largest staged value, its square below 2^15

__device__ __forceinline__ void split2(float v, _Float16 &hi, _Float16 &lo)
{
    hi = (_Float16)v;
    lo = (_Float16)__builtin_fmaf((float)hi, -kSplitLow, v * kSplitLow);
}

// The same for parameters, which are scaled to at most 2^14: v = hi + lo.
__device__ __forceinline__ void split2_param(float v, _Float16 &hi, _Float16 &lo)
{
    hi = (_Float16)v;
    lo = (_Float16)(v - (float)hi);
}

// Sum over a channel's sampled template elements: up to 32, spread over the channel; sixteen lanes share a channel and
// all of them get the result, the same wherever it is computed.
struct SplitSample {
    float t[2], w[2];
    bool there[2];
};

__device__ __forceinline__ SplitSample split_sample(const SplitPack &a, int c)
{
    const int n = a.O * a.taps, ns = min(32, n), apart = n / ns;
    SplitSample s;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int q = (threadIdx.x & 15) + 16 * i, e = q * apart, m = (int)fast_div((unsigned)e, a.d_taps);
        s.there[i] = q < ns && c < a.C;
        const size_t at = s.there[i] ? ((size_t)m * a.C + c) * a.taps + (e - m * a.taps) : 0;
        s.t[i] = a.templates[at];
        s.w[i] = a.weights[at];
    }
    return s;
}

__device__ __forceinline__ float split_sample_sum(float v)
{
    for (int d = 8; d > 0; d >>= 1)
        v += __shfl_xor(v, d, 16);
    return v;
}

// What is subtracted from every value of a channel: the mean of the sampled elements.  Any value is correct; one near the
// data keeps the three sums of w (x - t)^2 from cancelling.
__device__ __forceinline__ float split_centre(const SplitPack &a, const SplitSample &s)
{
    const float c = split_sample_sum((s.there[0] ? s.t[0] : 0.0f) + (s.there[1] ? s.t[1] : 0.0f)) / (float)min(32, a.O * a.taps);
    return __builtin_fabsf(c) < 1e18f ? c : 0.0f;
}

constexpr int kSplitRowLds = 1536;      // elements of a template that its packing workgroup keeps in LDS
constexpr int kNoExponent = -100000;   // of zero and of what is not finite

__device__ __forceinline__ int split_exponent(float v)   // floor(log2 |v|)
{
    return v != 0.0f && __builtin_fabsf(v) < INFINITY ? __builtin_amdgcn_frexp_expf(v) - 1 : kNoExponent;
}

__device__ __forceinline__ int split_wave_max(int v)
{
    for (int d = 32; d > 0; d >>= 1)
        v = max(v, __shfl_xor(v, d, 64));
    return v;
}

// Templates pack in their packing launch's first a.blocks workgroups (256 threads); `lds` holds 3 ceil(C / 16) 16 floats,
// then 32 doubles, 16 ints and min(K, kSplitRowLds) pairs of floats.
//
// Scales, all powers of two.  A channel's s: w s^-2 of about one size for all channels, so that the terms of a sum are
// as its values x'^2 s^2 are, and the largest of 256 sampled w (t - t2)^2 / 2 at 2^-3.  So a value is 24 bits while its
// term is above 2^-14, is off by 2^-36 absolutely below, and its square overflows 250 to 700 times further from the
// centre than the templates are from one another; workgroups that meet many such inputs take smaller scales (levels).  m:
// the sampled mean of t'^2 s^2, see similarity_split.hip.
// A template's row: its largest parameter at 2^13.
__device__ inline void split_pack_block(const SplitPack &a, int index, float *lds)
{
    // Consecutive workgroups go to the eight XCDs in turn; eight templates' 16-byte pieces share a line, which their XCD's
    // L2 should write once: neighbouring templates to one XCD (a.blocks is a multiple of 32).
    const int block = index % 8 * (a.blocks / 8) + index / 8;
    const int tid = threadIdx.x, wave = tid >> 6;
    const bool masked = a.mode == SIM_MODE_L2_NORM_IGNORE_NAN;
    const int Cp = (a.C + 15) / 16 * 16;
    float *lc = lds, *lm = lds + 2 * Cp;
    int *le = reinterpret_cast<int *>(lds + Cp);                 // exponent of s
    double *sums = reinterpret_cast<double *>(lds + 3 * Cp);     // [4 waves][8]
    int *ints = reinterpret_cast<int *>(sums + 32);              // [4 waves][4]
    float2 *row_tw = reinterpret_cast<float2 *>(ints + 16);      // the first kSplitRowLds of a template's elements

    // this workgroup's first template and the first channels' samples are requested before anything is waited for
    constexpr int kAhead = 4;
    float t_ahead[kAhead], w_ahead[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
        const size_t at = (size_t)min(block, a.O - 1) * a.K + min(tid + 256 * i, a.K - 1);
        t_ahead[i] = a.templates[at];
        w_ahead[i] = a.weights[at];
    }
    SplitSample s[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        s[i] = split_sample(a, 16 * i + (tid >> 4));
    int global;   // exponent of s^2 w
    {
        const long long total = (long long)a.O * a.K, e = total * tid / 256;
        const int m1 = (int)(e / a.K), k = (int)(e - (long long)m1 * a.K), m2 = (m1 + (a.O + 1) / 2) % a.O;
        const float t1 = a.templates[e], t2 = a.templates[(size_t)m2 * a.K + k];
        const int ew = split_exponent(a.weights[e]);
        int v[3] = {ew + 2 * split_exponent(t1 - t2) - 1, ew + 2 * split_exponent(t1), ew};
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            v[i] = split_wave_max(v[i]);
            if ((tid & 63) == 0)
                ints[4 * wave + i] = v[i];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 3; ++i)
            v[i] = max(max(ints[i], ints[4 + i]), max(ints[8 + i], ints[12 + i]));
        // templates all equal: their own size, or that of the weights alone
        const int size = v[0] > kNoExponent / 2 ? v[0] : v[1] > kNoExponent / 2 ? v[1] : v[2] > kNoExponent / 2 ? v[2] : 0;
        global = (-3 - size) >> 1;
        __syncthreads();
        if (tid == 0)
            ints[0] = v[2] > kNoExponent / 2 ? v[2] : 0;
    }
    __syncthreads();
    const int typical_w = ints[0];
    for (int c0 = 0; c0 < a.C; c0 += 64) {   // the loads of four channels in flight
        if (c0 > 0)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                s[i] = split_sample(a, c0 + 16 * i + (tid >> 4));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = c0 + 16 * i + (tid >> 4);
            const float centre = split_centre(a, s[i]);
            int ew = kNoExponent;
            float var = 0.0f;
#pragma unroll
            for (int j = 0; j < 2; ++j)
                if (s[i].there[j]) {
                    ew = max(ew, split_exponent(s[i].w[j]));
                    var += (s[i].t[j] - centre) * (s[i].t[j] - centre);
                }
            for (int d = 8; d > 0; d >>= 1)
                ew = max(ew, __shfl_xor(ew, d, 16));
            const int es = min(100, max(-100, global + ((ew > kNoExponent ? ew : typical_w) >> 1)));
            float mean = ldexpf(split_sample_sum(var) / (float)min(32, a.O * a.taps), 2 * es);
            mean = mean < 1e4f ? mean : 0.0f;
            if ((tid & 15) == 0 && c < Cp) {
                lc[c] = centre;
                le[c] = es;
                lm[c] = mean;
            }
        }
    }
    __syncthreads();
    if (block == 0)
        for (int c = tid; c < a.chunks * a.cg; c += 256) {
            const bool there = c < a.C;
            float *dst = a.chan + c;
            for (int level = 0; level < kSplitLevels; ++level, dst += SPLIT_CHANNEL_FIELDS * a.chunks * a.cg) {
                const float s = there ? ldexpf(1.0f, le[c] - kSplitLevelBits * level) : 0.0f;
                dst[SPLIT_S * a.chunks * a.cg] = s;
                dst[SPLIT_NCS * a.chunks * a.cg] = there ? -(lc[c] * s) : 0.0f;
                dst[SPLIT_M * a.chunks * a.cg] = there ? ldexpf(lm[c], -2 * kSplitLevelBits * level) : 0.0f;
            }
        }
    for (int m = block; m < a.n_mtiles * kSplitRows; m += a.blocks) {
        // The loops below run once or twice in a workgroup: unrolled, their code takes longer to fetch than to run.
        const float *mt = a.templates + (size_t)min(m, a.O - 1) * a.K, *mw = a.weights + (size_t)min(m, a.O - 1) * a.K;
        const int in_lds = min(a.K, kSplitRowLds);
        if (m == block)
#pragma unroll
            for (int i = 0; i < kAhead; ++i)
                if (tid + 256 * i < in_lds)
                    row_tw[tid + 256 * i] = make_float2(t_ahead[i], w_ahead[i]);
#pragma unroll 1
        for (int k = tid + (m == block ? 256 * kAhead : 0); k < in_lds; k += 256)
            row_tw[k] = make_float2(mt[k], mw[k]);
        double sum[3] = {};   // w t'^2, w m / s^2, logarithms
        float size[2] = {};   // w / s^2 or 2 w |t'| / s, w t^2
        bool bad = false, weighted = false;
        int top = kNoExponent, bottom = kNoExponent;   // the largest of the parameters' exponents, and of -(those of w / s^2)
#pragma unroll 1
        for (int k = tid; k < (m < a.O ? a.K : 0); k += 256) {   // (a thread's own elements of the row)
            const float2 own = k < in_lds ? row_tw[k] : make_float2(mt[k], mw[k]);
            const int c = (int)fast_div((unsigned)k, a.d_taps), es = le[c];
            const float t = own.x, w = own.y, tc = t - lc[c], spread = ldexpf(lm[c], -2 * es);
            float2 tw;
            float l;
            sim_pack_element(a.mode, true, t, w, a.fudge, tw.x, tw.y, l);
            a.exact[(size_t)m * a.K + k] = tw;
            weighted |= w != 0.0f;
            sum[0] += (double)w * tc * tc;
            sum[1] += (double)w * spread;
            size[0] += fmaxf(ldexpf(w, -2 * es), ldexpf(2.0f * w * __builtin_fabsf(tc), -es));
            size[1] += w * t * t;
            const int ew = split_exponent(w);
            top = max(top, max(ew - 2 * es, ew + split_exponent(tc) + 2 - es));
            bottom = ew > kNoExponent ? max(bottom, 2 * es - ew) : bottom;
            // weights and templates outside this range: the pieces of their products may leave the range of
            // normal numbers, so such a template is left to the term-by-term kernel
            bad |= !(w == 0.0f || (w >= 0x1p-60f && w <= 0x1p20f)) || !(__builtin_fabsf(t) <= 0x1p60f);
            if (a.mode != SIM_MODE_L2) {
                a.logs[(size_t)m * a.K + k] = l;
                sum[2] += l;
                bad |= !(__builtin_fabsf(l) <= 120.0f);
            }
            if (masked)
                top = max(top, ew + split_exponent(__builtin_fmaf(tc, tc, spread)) + 1);
        }
        for (int d = 32; d > 0; d >>= 1) {
#pragma unroll
            for (int i = 0; i < 3; ++i)
                sum[i] += __shfl_xor(sum[i], d, 64);
#pragma unroll
            for (int i = 0; i < 2; ++i)
                size[i] += __shfl_xor(size[i], d, 64);
            top = max(top, __shfl_xor(top, d, 64));
            bottom = max(bottom, __shfl_xor(bottom, d, 64));
        }
        if ((tid & 63) == 0) {
#pragma unroll
            for (int i = 0; i < 3; ++i)
                sums[8 * wave + i] = sum[i];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                sums[8 * wave + 3 + i] = size[i];
            ints[4 * wave] = top;
            ints[4 * wave + 1] = bottom;
        }
        bad = __syncthreads_or(bad);
        weighted = __syncthreads_or(weighted);
        top = max(max(ints[0], ints[4]), max(ints[8], ints[12]));
        bottom = max(max(ints[1], ints[5]), max(ints[9], ints[13]));
        const int shift = top > kNoExponent / 2 ? min(120, max(-120, 13 - top)) : 0;
        if (tid == 0) {
            double all[5];
#pragma unroll
            for (int i = 0; i < 5; ++i)
                all[i] = (sums[i] + sums[8 + i]) + (sums[16 + i] + sums[24 + i]);
            sum[2] = all[2];
            const double both = all[0] + all[1], line = a.line * fmax(all[0], 0.5 * both);
            double thr = weighted ? 0x1p-60 : 0.0;   // without weights zero is the exact sum
            // The values' absolute error, 2^-36 each, stays below 2^-23 of such a sum; 2^6 times as much with each level.
            const double root = (double)sqrtf((float)a.K), values = all[3] * 0x1p-13 / root;
            // The parameters' is 2^-25 of the scaled ones, 2^-25.8 in the mean of its square: of a sum with d_k scaled values
            // and weights a_k, 2^-25.8 sqrt(sum d_k^4), which is at most D^2 sqrt(K) and D sqrt(sum / min a_k), D the largest
            // value.  It stays below 2^-22 of the sum.
            const double params = fmin(kSplitParamShare * root, ldexp(1.0, min(100, bottom - shift - 6))) * ldexp(1.0, -shift);
            thr = fmax(thr, fmax(values, params * (kSplitSeen * kSplitSeen)));
            if (masked)   // (the third operand's parameters meet ones)
                thr = fmax(thr, ldexp(kSplitParamShare * root, -shift));
            if (!masked)
                thr = fmax(thr, fmax(line, all[4] / 1024.0));
            const double first = masked ? (both > 0.0 ? line / both : 0.0) : -both;
            float4 row;
            row.x = (float)first;
            row.y = __builtin_fabs(first) < 1e37 ? (float)(first - (double)row.x) : 0.0f;
            row.z = ldexpf(1.0f, -shift);
            row.w = bad || !(thr < 1e37) ? INFINITY : (float)thr;
            reinterpret_cast<float4 *>(a.rows)[m] = row;
            reinterpret_cast<float2 *>(a.rows + (size_t)5 * a.n_mtiles * kSplitRows)[m] = make_float2((float)values, (float)params);
            a.rows[(size_t)4 * a.n_mtiles * kSplitRows + m] = masked || a.mode == SIM_MODE_L2 ? 0.0f : (float)(sum[2] + (double)a.norm_const);
        }
        // the row's packed parameters: 16 bytes are eight channels at one tap
        const int mtile = m / kSplitRows, row = m % kSplitRows;
#pragma unroll 1
        for (int i = tid; i < a.chunks * a.steps * 2; i += 256) {
            const int half = i & 1, at = i >> 1, chunk = (int)fast_div((unsigned)at, a.d_steps), step = at - chunk * a.steps;
            const int tap = a.cg == 16 ? step : 2 * step + half;
            f16x8 v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int c = chunk * a.cg + (a.cg == 16 ? 8 * half : 0) + j;
                const bool there = m < a.O && c < a.C && tap < a.taps;
                const int k = there ? c * a.taps + tap : 0;
                float2 tw = row_tw[min(k, in_lds - 1)];
                if (a.K > kSplitRowLds && k >= in_lds)
                    tw = make_float2(mt[k], mw[k]);
                const float t = tw.x, w = tw.y;
                const int cl = there ? c : 0, es = le[cl];
                const float tc = t - lc[cl];
                _Float16 hi, lo;
                auto put = [&](int at, float value) {
                    split2_param(there ? value : 0.0f, hi, lo);
                    v[at][j] = hi;
                    v[at + 1][j] = lo;
                };
                put(0, -ldexpf(w, shift - 2 * es));
                put(2, ldexpf(2.0f * w * tc, shift - es));
                if (masked) {
                    const float l = a.logs[(size_t)min(m, a.O - 1) * a.K + k];   // (written in front of the barriers above)
                    put(4, -ldexpf(w * __builtin_fmaf(tc, tc, ldexpf(lm[cl], -2 * es)), shift));
                    put(6, l * kSplitLogScale);
                }
            }
            f16x8 *dst = reinterpret_cast<f16x8 *>(a.packed) + ((size_t)mtile * a.chunks * a.steps + at) * a.pieces * 64 +
                         32 * half + row;
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (q < a.pieces)
                    dst[q * 64] = v[q];
        }
        __syncthreads();
    }
}

inline size_t split_pack_lds_bytes(int C, int K)
{
    return (C + 15) / 16 * 16 * 3 * sizeof(float) + 32 * sizeof(double) + 16 * sizeof(int) +
           std::min(K, kSplitRowLds) * sizeof(float2);
}

}  // namespace simnets
