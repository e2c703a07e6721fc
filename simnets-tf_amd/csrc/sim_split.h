// Shared by the split matrix-core form of the L2 Similarity modes (similarity_split.hip) and the direct kernels that
// pack its parameters and recompute the tiles it flags (similarity_direct.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "internal.h"
#include "sim_step.h"

namespace simnets {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kSplitPixels = 128;   // output pixels of a workgroup, consecutive over the whole batch
constexpr int kSplitRows = 32;      // templates of one matrix tile
constexpr float kSplitLead = 0.125f;   // of sum w t'^2, added to an output's sum in advance and taken off at its end
constexpr int kSplitMaxC = 4096;    // channels whose centres the packing kernel keeps in LDS

// Geometry of one call on the split form.
struct SplitPlan {
    bool on;
    int cg;       // channels of a staged chunk: 16 (a matrix step is one tap) or 8 (a step is two taps)
    int chunks;   // ceil(C / cg)
    int steps;    // matrix steps per chunk: taps, or ceil(taps / 2)
    int pieces;   // 16-bit pieces of the packed parameters per step: 6, with missing values 12
    int n_mtiles; // ceil(O / 32)
    int n_ptiles; // ceil(B oh ow / 128)
    int Wp, Hv;   // columns of a staged row; rows of one image's staged stack
    size_t packed, ctr, bias, lg, thr, flags, exact, logs, total;   // workspace, from its own start
};

SplitPlan sim_split_plan(const SimPlan &p);

struct SplitPack {
    const float *templates, *weights;
    unsigned short *packed;
    float *ctr, *bias, *lg, *thr;
    float2 *exact;   // [O][K] template and negative weight as the term-by-term kernels take them ...
    float *logs;     // ... and the normalized modes' logarithm terms
    int O, C, taps, K, cg, chunks, steps, pieces, n_mtiles, mode;
    float fudge, norm_const;
    float line;   // outputs below `line` times sum w t'^2 are recomputed term by term
    int pack_blocks, thr_blocks;   // pack_blocks = chunks * n_mtiles * ceil(steps / 4)
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

// What is subtracted from every value of a channel: the mean of up to 32 template elements spread over the channel.  Any
// value is correct; one near the data keeps the three sums of w (x - t)^2 from cancelling.  Sixteen lanes share a
// channel; all of them get the result, the same wherever it is computed.
__device__ __forceinline__ float split_centre_part(const SplitPack &a, int c)
{
    const int n = a.O * a.taps, ns = min(32, n), apart = n / ns;
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int q = (threadIdx.x & 15) + 16 * i, e = q * apart, m = e / a.taps;
        if (q < ns && c < a.C)
            s += a.templates[((size_t)m * a.C + c) * a.taps + (e - m * a.taps)];
    }
    return s;
}

__device__ __forceinline__ float split_centre(const SplitPack &a, float part)
{
    for (int d = 8; d > 0; d >>= 1)
        part += __shfl_xor(part, d, 16);
    part /= (float)min(32, a.O * a.taps);
    return __builtin_fabsf(part) < 1e18f ? part : 0.0f;
}

// The parameter-only part, run by the first pack_blocks + thr_blocks workgroups (256 threads) of the packing launch;
// `lds` holds max(C, 16) floats and then 12 doubles.
__device__ inline void split_pack_block(const SplitPack &a, int block, float *lds)
{
    const int tid = threadIdx.x;
    const bool masked = a.mode == SIM_MODE_L2_NORM_IGNORE_NAN;
    if (block < a.pack_blocks) {
        const int parts = (a.steps + 3) / 4;   // of a chunk's steps, four to a workgroup
        const int mtile = block / (a.chunks * parts), rest = block - mtile * a.chunks * parts;
        const int chunk = rest / parts, part = rest - chunk * parts;
        if (tid < a.cg * 16) {
            const int cl = tid >> 4;
            const float centre = split_centre(a, split_centre_part(a, chunk * a.cg + cl));
            if ((tid & 15) == 0) {
                lds[cl] = centre;
                if (mtile == 0 && part == 0)
                    a.ctr[chunk * a.cg + cl] = centre;
            }
        }
        __syncthreads();
        const int step = 4 * part + (tid >> 6);
        if (step < a.steps) {
            const int lane = tid & 63, half = lane >> 5, m = mtile * kSplitRows + (lane & 31);
            const int tap = a.cg == 16 ? step : 2 * step + half;
            bf16x8 v[12];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int cl = a.cg == 16 ? 8 * half + j : j, c = chunk * a.cg + cl;
                float t = 0.0f, w = 0.0f, l = 0.0f;
                if (m < a.O && c < a.C && tap < a.taps) {
                    const size_t at = ((size_t)m * a.C + c) * a.taps + tap;
                    w = a.weights[at];
                    t = a.templates[at] - lds[cl];
                    float unused0, unused1;
                    if (masked)
                        sim_pack_element(a.mode, true, t, w, a.fudge, unused0, unused1, l);
                }
                __bf16 p0, p1, p2;
                auto put = [&](int at, float value) {
                    split3(value, p0, p1, p2);
                    v[at][j] = p0;
                    v[at + 1][j] = p1;
                    v[at + 2][j] = p2;
                };
                put(0, -w);
                put(3, 2.0f * w * t);
                if (masked) {
                    put(6, -(w * t) * t);
                    put(9, l);
                }
            }
            bf16x8 *dst = reinterpret_cast<bf16x8 *>(a.packed) +
                          (((size_t)mtile * a.chunks + chunk) * a.steps + step) * a.pieces * 64 + lane;
#pragma unroll
            for (int q = 0; q < 12; ++q)
                if (q < a.pieces)
                    dst[q * 64] = v[q];
        }
        return;
    }
    // biases and thresholds, one template per workgroup (at a time)
    for (int c0 = 0; c0 < a.C; c0 += 64) {   // the loads of four channels in flight
        float part[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            part[i] = split_centre_part(a, c0 + 16 * i + (tid >> 4));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = c0 + 16 * i + (tid >> 4);
            const float centre = split_centre(a, part[i]);
            if ((tid & 15) == 0 && c < a.C)
                lds[c] = centre;
        }
    }
    __syncthreads();
    double *sums = reinterpret_cast<double *>(lds + ((a.C + 15) / 16 * 16));   // [4 waves][3]
    for (int m = block - a.pack_blocks; m < a.n_mtiles * kSplitRows; m += a.thr_blocks) {
        double tc2 = 0.0, traw = 0.0, lsum = 0.0;
        bool bad = false, weighted = false;
        if (m < a.O)
#pragma unroll 4
            for (int k = tid; k < a.K; k += 256) {
                const float t = a.templates[(size_t)m * a.K + k], w = a.weights[(size_t)m * a.K + k];
                const float tc = t - lds[k / a.taps];
                float2 tw;
                float l;
                sim_pack_element(a.mode, true, t, w, a.fudge, tw.x, tw.y, l);
                a.exact[(size_t)m * a.K + k] = tw;
                weighted |= w != 0.0f;
                tc2 += (double)w * tc * tc;
                traw += (double)w * t * t;
                // weights and templates outside this range: the pieces of their products may leave the range of
                // normal numbers, so such a template is left to the term-by-term kernel
                bad |= !(w == 0.0f || (w >= 0x1p-60f && w <= 0x1p20f)) || !(__builtin_fabsf(t) <= 0x1p60f);
                if (a.mode != SIM_MODE_L2) {
                    a.logs[(size_t)m * a.K + k] = l;
                    lsum += l;
                    bad |= !(__builtin_fabsf(l) <= 1e6f);
                }
            }
        for (int d = 32; d > 0; d >>= 1) {
            tc2 += __shfl_xor(tc2, d, 64);
            traw += __shfl_xor(traw, d, 64);
            lsum += __shfl_xor(lsum, d, 64);
        }
        if ((tid & 63) == 0) {
            double *mine = sums + 3 * (tid >> 6);
            mine[0] = tc2; mine[1] = traw; mine[2] = lsum;
        }
        bad = __syncthreads_or(bad);
        weighted = __syncthreads_or(weighted);
        if (tid == 0) {
            tc2 = (sums[0] + sums[3]) + (sums[6] + sums[9]);
            traw = (sums[1] + sums[4]) + (sums[7] + sums[10]);
            lsum = (sums[2] + sums[5]) + (sums[8] + sums[11]);
            a.bias[m] = masked ? 0.0f : (float)(-(1.0 + kSplitLead) * tc2);
            a.lg[m] = masked || a.mode == SIM_MODE_L2 ? 0.0f : (float)(lsum + (double)a.norm_const);
            double thr = weighted ? 0x1p-60 : 0.0;   // without weights zero is the exact sum
            if (!masked)
                thr = fmax(thr, fmax((double)a.line * tc2, traw / 1024.0));
            a.thr[m] = bad || !(thr < 1e37) ? INFINITY : (float)thr;
        }
        __syncthreads();
    }
}

}  // namespace simnets
