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
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

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
    FastDiv d_taps, d_steps, d_K;
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
    float t[2];
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
    }
    return s;
}

__device__ __forceinline__ float split_sample_sum(float v)
{
    for (int d = 8; d > 0; d >>= 1)
        v += __shfl_xor(v, d, 16);
    return v;
}

constexpr int kSplitRowLds = 1536;      // elements of a template that its packing workgroup keeps in LDS
constexpr int kNoExponent = -100000;   // of zero and of what is not finite

__device__ __forceinline__ int split_exponent(float v)   // floor(log2 |v|)
{
    return v != 0.0f && __builtin_fabsf(v) < INFINITY ? __builtin_amdgcn_frexp_expf(v) - 1 : kNoExponent;
}

// A value of another lane of the same row of sixteen: the one SHIFT lanes on, in a circle.
template <int SHIFT>
__device__ __forceinline__ int split_row_turn(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, 0x120 + SHIFT, 0xf, 0xf, true);
}

// ... and of the same four: the lane whose number differs in the bits of X, 1 or 2.
template <int X>
__device__ __forceinline__ int split_quad_swap(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, X == 1 ? 0xB1 : 0x4E, 0xf, 0xf, true);
}

__device__ __forceinline__ float split_quad_sum(float v)
{
    v += __int_as_float(split_quad_swap<2>(__float_as_int(v)));
    return v + __int_as_float(split_quad_swap<1>(__float_as_int(v)));
}

template <int N>
__device__ __forceinline__ void split_row_max(int (&v)[N])   // every lane of the row has the result
{
    auto step = [&](auto turn) {
#pragma unroll
        for (int i = 0; i < N; ++i)
            v[i] = max(v[i], turn(v[i]));
    };
    step([](int x) { return split_row_turn<8>(x); });
    step([](int x) { return split_row_turn<4>(x); });
    step([](int x) { return split_row_turn<2>(x); });
    step([](int x) { return split_row_turn<1>(x); });
}

template <int N>
__device__ __forceinline__ void split_row_sum(double (&v)[N])
{
    auto step = [&](auto turn) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const unsigned long long bits = __builtin_bit_cast(unsigned long long, v[i]);
            const unsigned lo = (unsigned)turn((int)(unsigned)bits), hi = (unsigned)turn((int)(unsigned)(bits >> 32));
            v[i] += __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
        }
    };
    step([](int x) { return split_row_turn<8>(x); });
    step([](int x) { return split_row_turn<4>(x); });
    step([](int x) { return split_row_turn<2>(x); });
    step([](int x) { return split_row_turn<1>(x); });
}

// What the packing workgroups exchange, of each of their sixteen rows of lanes.
struct SplitPackRows {
    double sums[16][5];
    int most[16][4];
};

// Templates pack in their packing launch's first a.blocks workgroups (256 threads); `lds` holds SplitPackRows, 3 ceil(C / 16) 16
// floats and min(K, kSplitRowLds) pairs of floats.
//
// Scales, all powers of two.  A channel's s: w s^-2 of about one size for all channels, so that the terms of a sum are
// as its values x'^2 s^2 are, and the largest of 256 sampled w (t - t2)^2 / 2 at 2^-3.  So a value is 24 bits while its
// term is above 2^-14, is off by 2^-36 absolutely below, and its square overflows 250 to 700 times further from the
// centre than the templates are from one another; workgroups that meet many such inputs take smaller scales (levels).  m:
// the sampled mean of t'^2 s^2, see similarity_split.hip.
// A template's row: its largest parameter at 2^13.
//
// Every instruction runs once or twice in a workgroup and is fetched from beyond the caches, some eight cycles each: what
// counts is their number (7.6 KB; 19 with unrolled channels and reductions through LDS moves), and loads requested in front of
// what they are not needed for.  The launch, us: 64 channels, 3 x 3, 128 templates 15.3 -> 9.8; 45, 75 10.9 -> 6.6; 128, 128
// 17.7 -> 11.7.
__device__ inline void split_pack_block(const SplitPack &a, int index, float *lds)
{
    // Consecutive workgroups go to the eight XCDs in turn; eight templates' 16-byte pieces share a line, which their XCD's
    // L2 should write once: neighbouring templates to one XCD (a.blocks is a multiple of 32).
    const int block = index % 8 * (a.blocks / 8) + index / 8;
    const int tid = threadIdx.x, row16 = tid >> 4, col16 = tid & 15;
    const bool masked = a.mode == SIM_MODE_L2_NORM_IGNORE_NAN;
    const int Cp = (a.C + 15) / 16 * 16;
    SplitPackRows &rows = *reinterpret_cast<SplitPackRows *>(lds);
    float *lc = lds + sizeof(SplitPackRows) / sizeof(float), *lm = lc + 2 * Cp;
    int *le = reinterpret_cast<int *>(lc + Cp);                  // exponent of s
    float2 *row_tw = reinterpret_cast<float2 *>(lc + 3 * Cp);    // the first kSplitRowLds of a template's elements

    // this workgroup's first template, 256 elements of all and the first channels' samples are requested before anything is
    // waited for
    constexpr int kAhead = 4;
    float t_ahead[kAhead], w_ahead[kAhead];
    {
        const size_t first = (size_t)min(block, a.O - 1) * a.K;
        const float *mt = a.templates + first, *mw = a.weights + first;
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const unsigned k = min(tid + 256 * i, a.K - 1);
            t_ahead[i] = mt[k];
            w_ahead[i] = mw[k];
        }
    }
    float some_t, some_t2, some_w;
    {
        const long long total = (long long)a.O * a.K, e = (total >> 8) * tid + ((total & 255) * tid >> 8);   // total tid / 256
        const int m1 = total < (1ll << 31) ? (int)fast_div((unsigned)e, a.d_K) : (int)(e / a.K);
        const int m2 = m1 + (a.O + 1) / 2, apart = (m2 < a.O ? m2 : m2 - a.O) - m1;
        const float *t = a.templates + e;
        some_t = t[0];
        some_t2 = t[(long long)apart * a.K];
        some_w = a.weights[e];
    }
    // A channel's samples are up to 32 template elements, spread over the channel: eight a lane, four lanes a channel.
    struct Samples {
        float t[8], w[8];
    } next, s;
    const int n_samples = min(32, a.O * a.taps), samples_apart = a.O * a.taps / n_samples;
    const float per_sample = 1.0f / (float)n_samples;
    int typical_w = 0, global = 0;   // exponents, the second that of s^2 w
    for (int c0 = -64; c0 < a.C; c0 += 64) {
        if (c0 + 64 < a.C) {
            const int c = min(c0 + 64 + (tid >> 2), a.C - 1);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int q = (tid & 3) + 4 * i, e = min(q, n_samples - 1) * samples_apart, m = (int)fast_div((unsigned)e, a.d_taps);
                const size_t at = (size_t)m * ((a.C - 1) * a.taps) + (c * a.taps + e);
                next.t[i] = a.templates[at];
                next.w[i] = a.weights[at];
            }
        }
        if (c0 < 0) {
            const int ew = split_exponent(some_w);
            int v[3] = {ew + 2 * split_exponent(some_t - some_t2) - 1, ew + 2 * split_exponent(some_t), ew};
#pragma unroll 1
            for (int half = 0; half < 2; ++half) {   // of the row's lanes, of the rows
                split_row_max(v);
                if (half == 0) {
                    if (col16 == 0)
#pragma unroll
                        for (int i = 0; i < 3; ++i)
                            rows.most[row16][i] = v[i];
                    __syncthreads();
#pragma unroll
                    for (int i = 0; i < 3; ++i)
                        v[i] = rows.most[col16][i];
                }
            }
            // templates all equal: their own size, or that of the weights alone
            const int size = v[0] > kNoExponent / 2 ? v[0] : v[1] > kNoExponent / 2 ? v[1] : v[2] > kNoExponent / 2 ? v[2] : 0;
            global = (-3 - size) >> 1;
            typical_w = v[2] > kNoExponent / 2 ? v[2] : 0;
        } else {
            auto there = [&](int i) { return (tid & 3) + 4 * i < n_samples; };
            float part[4], var[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                part[i] = (there(i) ? s.t[i] : 0.0f) + (there(i + 4) ? s.t[i + 4] : 0.0f);
            float centre = split_quad_sum((part[0] + part[2]) + (part[1] + part[3])) * per_sample;
            centre = __builtin_fabsf(centre) < 1e18f ? centre : 0.0f;
            int ew = kNoExponent;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float d = there(i) ? s.t[i] - centre : 0.0f, d2 = there(i + 4) ? s.t[i + 4] - centre : 0.0f;
                var[i] = __builtin_fmaf(d2, d2, d * d);
                ew = max(ew, max(there(i) ? split_exponent(s.w[i]) : kNoExponent, there(i + 4) ? split_exponent(s.w[i + 4]) : kNoExponent));
            }
            ew = max(ew, split_quad_swap<2>(ew));
            ew = max(ew, split_quad_swap<1>(ew));
            const int es = min(100, max(-100, global + ((ew > kNoExponent ? ew : typical_w) >> 1)));
            float mean = ldexpf(split_quad_sum((var[0] + var[2]) + (var[1] + var[3])) * per_sample, 2 * es);
            mean = mean < 1e4f ? mean : 0.0f;
            const int c = c0 + (tid >> 2);
            if ((tid & 3) == 0 && c < Cp) {
                lc[c] = centre;
                le[c] = es;
                lm[c] = mean;
            }
        }
        s = next;
    }
    // (the loops below run once or twice in a workgroup)
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
        if (tid + 256 * i < min(a.K, kSplitRowLds))
            row_tw[tid + 256 * i] = make_float2(t_ahead[i], w_ahead[i]);
    __syncthreads();
    if (block < kSplitLevels)   // (there are 32 of them at least)
#pragma unroll 1
        for (int c = tid; c < a.chunks * a.cg; c += 256) {
            const bool there = c < a.C;
            float *dst = a.chan + block * SPLIT_CHANNEL_FIELDS * a.chunks * a.cg + c;
            const float s = there ? ldexpf(1.0f, le[c] - kSplitLevelBits * block) : 0.0f;
            dst[SPLIT_S * a.chunks * a.cg] = s;
            dst[SPLIT_NCS * a.chunks * a.cg] = there ? -(lc[c] * s) : 0.0f;
            dst[SPLIT_M * a.chunks * a.cg] = there ? ldexpf(lm[c], -2 * kSplitLevelBits * block) : 0.0f;
        }
    for (int m = block; m < a.n_mtiles * kSplitRows; m += a.blocks) {
        const float *mt = a.templates + (size_t)min(m, a.O - 1) * a.K, *mw = a.weights + (size_t)min(m, a.O - 1) * a.K;
        const int in_lds = min(a.K, kSplitRowLds);
#pragma unroll 1
        for (int k = tid + (m == block ? 256 * kAhead : 0); k < in_lds; k += 256)
            row_tw[k] = make_float2(mt[k], mw[k]);
        double sum[5] = {};   // w t'^2, w m / s^2, logarithms, w / s^2 or 2 w |t'| / s, w t^2
        bool bad = false, weighted = false;
        int most[4] = {kNoExponent, kNoExponent};   // of the parameters' exponents, of -(those of w / s^2), and the two flags
        {
            float size[2] = {};
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
                most[0] = max(most[0], max(ew - 2 * es, ew + split_exponent(tc) + 2 - es));
                most[1] = ew > kNoExponent ? max(most[1], 2 * es - ew) : most[1];
                // weights and templates outside this range: the pieces of their products may leave the range of
                // normal numbers, so such a template is left to the term-by-term kernel
                bad |= !(w == 0.0f || (w >= 0x1p-60f && w <= 0x1p20f)) || !(__builtin_fabsf(t) <= 0x1p60f);
                if (a.mode != SIM_MODE_L2) {
                    a.logs[(size_t)m * a.K + k] = l;
                    sum[2] += l;
                    bad |= !(__builtin_fabsf(l) <= 120.0f);
                }
                if (masked)
                    most[0] = max(most[0], ew + split_exponent(__builtin_fmaf(tc, tc, spread)) + 1);
            }
            sum[3] = size[0];
            sum[4] = size[1];
        }
        most[2] = bad;
        most[3] = weighted;
#pragma unroll 1
        for (int half = 0; half < 2; ++half) {   // of the row's lanes, of the rows
            split_row_sum(sum);
            split_row_max(most);
            if (half == 0) {
                __syncthreads();   // (rows.most has been read)
                if (col16 == 0) {
#pragma unroll
                    for (int i = 0; i < 5; ++i)
                        rows.sums[row16][i] = sum[i];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        rows.most[row16][i] = most[i];
                }
                __syncthreads();
#pragma unroll
                for (int i = 0; i < 5; ++i)
                    sum[i] = rows.sums[col16][i];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    most[i] = rows.most[col16][i];
            }
        }
        const int top = most[0], bottom = most[1];
        const int shift = top > kNoExponent / 2 ? min(120, max(-120, 13 - top)) : 0;
        // the row's packed parameters: 16 bytes are eight channels at one tap, a lane takes two of them
        const int mtile = m / kSplitRows, row = m % kSplitRows;
#pragma unroll 1
        for (int i = tid; i < a.chunks * a.steps * 8; i += 256) {
            const int pair = i & 3, half = i >> 2 & 1, at = i >> 3;
            const int chunk = (int)fast_div((unsigned)at, a.d_steps), step = at - chunk * a.steps;
            const int tap = a.cg == 16 ? step : 2 * step + half;
            f16x2 v[8];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int c = chunk * a.cg + (a.cg == 16 ? 8 * half : 0) + 2 * pair + j;
                const bool there = m < a.O && c < a.C && tap < a.taps;
                const int k = there ? c * a.taps + tap : 0;
                float2 tw = row_tw[min(k, in_lds - 1)];
                if (k >= in_lds)
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
            f16x2 *dst = reinterpret_cast<f16x2 *>(a.packed) +
                         (((size_t)mtile * a.chunks * a.steps + at) * a.pieces * 64 + 32 * half + row) * 4 + pair;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                dst[q * 256] = v[q];
            if (masked)
#pragma unroll
                for (int q = 4; q < 8; ++q)
                    dst[q * 256] = v[q];
        }
        if (tid == 192) {   // (the wave with the fewest of the elements above)
            const double both = sum[0] + sum[1], line = a.line * fmax(sum[0], 0.5 * both);
            double thr = most[3] ? 0x1p-60 : 0.0;   // without weights zero is the exact sum
            // The values' absolute error, 2^-36 each, stays below 2^-23 of such a sum; 2^6 times as much with each level.
            const double root = (double)sqrtf((float)a.K), values = sum[3] * 0x1p-13 / root;
            // The parameters' is 2^-25 of the scaled ones, 2^-25.8 in the mean of its square: of a sum with d_k scaled values
            // and weights a_k, 2^-25.8 sqrt(sum d_k^4), which is at most D^2 sqrt(K) and D sqrt(sum / min a_k), D the largest
            // value.  It stays below 2^-22 of the sum.
            const double params = fmin(kSplitParamShare * root, ldexp(1.0, min(100, bottom - shift - 6))) * ldexp(1.0, -shift);
            thr = fmax(thr, fmax(values, params * (kSplitSeen * kSplitSeen)));
            if (masked)   // (the third operand's parameters meet ones)
                thr = fmax(thr, ldexp(kSplitParamShare * root, -shift));
            if (!masked)
                thr = fmax(thr, fmax(line, sum[4] / 1024.0));
            const double first = masked ? (both > 0.0 ? line / both : 0.0) : -both;
            float4 row;
            row.x = (float)first;
            row.y = __builtin_fabs(first) < 1e37 ? (float)(first - (double)row.x) : 0.0f;
            row.z = ldexpf(1.0f, -shift);
            row.w = most[2] || !(thr < 1e37) ? INFINITY : (float)thr;
            reinterpret_cast<float4 *>(a.rows)[m] = row;
            reinterpret_cast<float2 *>(a.rows + (size_t)5 * a.n_mtiles * kSplitRows)[m] = make_float2((float)values, (float)params);
            a.rows[(size_t)4 * a.n_mtiles * kSplitRows + m] = masked || a.mode == SIM_MODE_L2 ? 0.0f : (float)(sum[2] + (double)a.norm_const);
        }
        __syncthreads();
    }
}

inline size_t split_pack_lds_bytes(int C, int K)
{
    return sizeof(SplitPackRows) + (C + 15) / 16 * 16 * 3 * sizeof(float) + std::min(K, kSplitRowLds) * sizeof(float2);
}

}  // namespace simnets
