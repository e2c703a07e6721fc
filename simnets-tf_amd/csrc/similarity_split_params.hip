// Parameter gradients of the L2 Similarity modes on the bf16 matrix cores, at the precision of fp32 (gfx950): the moments
//   S1[o, k] = sum_px g[px, o] x'[px, k],   S2[o, k] = sum_px g[px, o] x'[px, k]^2,   x' = x - c, c one value per channel
// or, where templates share a pattern, per patch element (and G[o] = sum_px g) that the finish kernel of similarity_grad.hip combines, every factor as three 16-bit pieces and
// the six products of pieces that matter, as in similarity_split.hip; the leading one has accumulators of its own.
//
// The contraction runs over images and output pixels.  A lane's eight values of a matrix operand are eight images at one
// pixel, so a tap moves a lane's operand by whole 16-byte slots - with eight pixels per operand every odd tap would be
// misaligned - and the patches need no copy of their own: the input tile of a few output pixels is staged once in LDS as
// [piece of x'^2, x'][channel, pixel][8 images] and read by every tap.  Rows are templates: g is packed once per call
// into the order the lanes read (1.5 times its size, read again for every 64 patch elements), its sums G on the way.
// A workgroup takes 64 patch elements x up to 128 templates over a share of the pixels; its partial sums go to the
// workspace and are added in order by the finish kernel.
//
// Measured (32 x 128 x 28 x 28, 128 templates, 3 x 3): 207 us on the fp32 matrix instructions -> 86 us + 10 us of packing,
// 1.04 PFLOP/s of matrix products; the finish kernel 20 -> 9 us with 28 shares of the pixels for 170.  Error against 64
// bits 2.5e-7 -> 2.0e-7 (templates) and 1.9e-7 (weights) of the gradient's 2-norm; with one set of accumulators 2.9e-7.
//
// LDS pitches are chosen so that slot = patch element modulo 8: the eight lanes that read together hit different banks.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fast_div.h"
#include "internal.h"
#include "sim_split.h"

namespace simnets {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kThreads = 256;
constexpr int kSlots = 816;          // 16-byte slots of one piece; the last holds zeros
constexpr int kColumns = 64;         // patch elements of a workgroup
constexpr int kImages = 8;           // images of a matrix operand
constexpr int kPackRows = 8, kPackGroups = kSplitRows / kPackRows;   // templates of a workgroup that packs g

struct ParamsArgs {
    const float *g, *x, *templates;
    bf16x8 *packed;      // g: [mtile][unit][pixel pair][piece][64 lanes]
    float *partial, *centres;   // [2 S1, S2; 2: G][S][Opad][Kpad]; [Opad][Kpad] what was subtracted, for the finish kernel
    float *ctr, *ctr64;         // centres: [C], and [64 templates][Kpad]
    float2 *spread;             // [Kpad] sum of the squares of t about the channel's centre and about the 64 templates' own
    int B, C, H, W, O, K, oh, ow, bh, bw, sh, sw, ph, pw, taps;
    int Opad, Kpad, S, n_mtiles;
    int TH, TW, pairs;   // output tile; TH * TW / 2 pixel pairs
    int rows, cols, pitch, chan;      // staged input rows and columns, slots of a row and of a channel
    int tiles_r, tiles_c, units;      // output tiles of an image, and of all groups of eight images
    float oob;
    FastDiv d_pairs, d_tw2, d_tiles, d_tc, d_chan, d_pitch, d_taps;
};

struct Unit {
    int img, r0, c0;     // first image, first output row and column
};

__device__ __forceinline__ Unit unit_of(const ParamsArgs &a, int u)
{
    Unit q;
    const int group = (int)fast_div((unsigned)u, a.d_tiles), t = u - group * a.tiles_r * a.tiles_c;
    const int tr = (int)fast_div((unsigned)t, a.d_tc);
    q.img = group * kImages;
    q.r0 = tr * a.TH;
    q.c0 = (t - tr * a.tiles_c) * a.TW;
    return q;
}

__device__ __forceinline__ int first_unit(const ParamsArgs &a, int s) { return (int)((long long)s * a.units / a.S); }

// One channel's centre, the mean of its template elements (any value is correct); its patch elements' centres, the mean
// over each 64 templates, and how far the templates lie from the two.
__device__ __forceinline__ void params_channel_block(const ParamsArgs &a, int c)
{
    __shared__ float wave_sum[kThreads / 64];
    const int tid = threadIdx.x, n = a.O * a.taps, l8 = tid & 7;
    float sum = 0.0f;
#pragma unroll 4
    for (int i = tid; i < n; i += kThreads) {
        const int o = (int)fast_div((unsigned)i, a.d_taps);
        sum += a.templates[((size_t)o * a.C + c) * a.taps + (i - o * a.taps)];
    }
    for (int d = 32; d > 0; d >>= 1)
        sum += __shfl_xor(sum, d, 64);
    if ((tid & 63) == 0)
        wave_sum[tid >> 6] = sum;
    __syncthreads();
    sum = ((wave_sum[0] + wave_sum[1]) + (wave_sum[2] + wave_sum[3])) / (float)n;
    const float centre = __builtin_fabsf(sum) < 1e18f ? sum : 0.0f;
    if (tid == 0)
        a.ctr[c] = centre;
    for (int tap = tid >> 3; tap < a.taps; tap += kThreads / 8) {   // eight lanes to a patch element
        const int k = c * a.taps + tap;
        float2 spread = make_float2(0.0f, 0.0f);
        for (int o0 = 0; o0 < a.O; o0 += 64) {
            float t[8], s1 = 0.0f, s2 = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                t[i] = a.templates[((size_t)min(o0 + 8 * i + l8, a.O - 1) * a.C + c) * a.taps + tap] - centre;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                t[i] = o0 + 8 * i + l8 < a.O ? t[i] : 0.0f;
                s1 += t[i];
                s2 += t[i] * t[i];
            }
            for (int d = 4; d > 0; d >>= 1) {
                s1 += __shfl_xor(s1, d, 8);
                s2 += __shfl_xor(s2, d, 8);
            }
            const float mean = s1 / (float)min(64, a.O - o0);
            if (l8 == 0)
                a.ctr64[(size_t)(o0 / 64) * a.Kpad + k] = __builtin_fabsf(centre + mean) < 1e18f ? centre + mean : 0.0f;
            spread.x += s2;
            spread.y += s2 - s1 * mean;
        }
        if (l8 == 0)
            a.spread[k] = spread;
    }
}

// The first C blocks: params_channel_block.  The 4 S n_mtiles behind: g of one share of the pixels and eight templates, a
// thread one template's pairs of pixels (eight neighbouring lanes read 64 contiguous bytes, a wave writes whole lines of
// 128), and the share's sums G.  32 x 128 x 28 x 28, 128 templates, 3 x 3 (32 MB to move): with 32 templates to a workgroup, 112
// of them, 17.7 us, so 10.5.
__global__ __launch_bounds__(kThreads) void sim_split_params_pack_kernel(const ParamsArgs a)
{
    if ((int)blockIdx.x < a.C) {
        params_channel_block(a, blockIdx.x);
        return;
    }
    __shared__ float wave_sum[kThreads / 64][kPackRows];
    const int tid = threadIdx.x, lane = tid & 63, block = (blockIdx.x - a.C) / kPackGroups;
    const int mtile = block / a.S, s = block - mtile * a.S;
    const int row = (blockIdx.x - a.C) % kPackGroups * kPackRows + (lane >> 3), o = mtile * kSplitRows + row;
    const int q0 = first_unit(a, s) * a.pairs, q1 = first_unit(a, s + 1) * a.pairs;
    const size_t npix = (size_t)a.oh * a.ow;
    float sum = 0.0f;
    for (int q = q0 + (tid >> 6) * 8 + (lane & 7); q < q1; q += kThreads / 8) {
        const int u = (int)fast_div((unsigned)q, a.d_pairs), pp = q - u * a.pairs;
        const Unit un = unit_of(a, u);
        const int py = (int)fast_div((unsigned)pp, a.d_tw2);
        const int r = un.r0 + py, c = un.c0 + 2 * (pp - py * (a.TW / 2));
        const float *src = a.g + ((size_t)un.img * a.O + o) * npix + (size_t)r * a.ow + c;
        float v[2][kImages];
#pragma unroll
        for (int j = 0; j < kImages; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                v[h][j] = o < a.O && r < a.oh && c + h < a.ow && un.img + j < a.B ? src[(size_t)j * a.O * npix + h] : 0.0f;
        bf16x8 *dst = a.packed + (((size_t)mtile * a.units * a.pairs + q) * 3) * 64 + row;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            bf16x8 p[3];
#pragma unroll
            for (int j = 0; j < kImages; ++j) {
                __bf16 p0, p1, p2;
                split3_any(v[h][j], p0, p1, p2);
                p[0][j] = p0; p[1][j] = p1; p[2][j] = p2;
            }
#pragma unroll
            for (int i = 0; i < 3; ++i)
                dst[i * 64 + h * 32] = p[i];
        }
        // sixteen values to one addition: with each added in turn the error of G was 2.2e-7 of it (32 x 128 x 28 x 28, 128
        // templates; now 1.1e-7, the fp32 matrix form 1.6e-7), and more than the moments' in a gradient
        float pair[kImages];
#pragma unroll
        for (int j = 0; j < kImages; ++j)
            pair[j] = v[0][j] + v[1][j];
        sum += ((pair[0] + pair[1]) + (pair[2] + pair[3])) + ((pair[4] + pair[5]) + (pair[6] + pair[7]));
    }
    for (int d = 4; d > 0; d >>= 1)
        sum += __shfl_xor(sum, d, 8);
    if ((lane & 7) == 0)
        wave_sum[tid >> 6][lane >> 3] = sum;
    __syncthreads();
    if (tid < 64 && (lane & 7) == 0 && o < a.O)
        a.partial[((size_t)2 * a.S + s) * a.Opad * a.Kpad + (size_t)o * a.Kpad] =
            (wave_sum[0][lane >> 3] + wave_sum[1][lane >> 3]) + (wave_sum[2][lane >> 3] + wave_sum[3][lane >> 3]);
}

// This share's sums of one patch element k and a lane's sixteen templates; with the first share what was subtracted.
__device__ __forceinline__ void params_store(const ParamsArgs &a, int mtile, int k, int s, int half, float centre,
                                             const f32x16 &hi2, const f32x16 &lo2, const f32x16 &hi1, const f32x16 &lo1)
{
    const size_t slab = (size_t)a.Opad * a.Kpad;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int o = mtile * kSplitRows + 8 * (r / 4) + 4 * half + r % 4;
        if (o >= a.O)
            continue;
        const size_t at = (size_t)o * a.Kpad + k;
        float *dst = a.partial + (size_t)s * slab + at;
        dst[0] = split_sum(hi1[r], lo1[r]);
        dst[(size_t)a.S * slab] = split_sum(hi2[r], lo2[r]);
        if (s == 0)
            a.centres[at] = centre;
    }
}

// G template tiles from mtile0 x 64 patch elements; a wave holds one template tile x NI column tiles.
template <int G>
__device__ __forceinline__ void params_body(const ParamsArgs &a, char *lds, int mtile0)
{
    constexpr int NI = G == 4 ? 2 : 1;   // two column tiles among 4 / G waves (G = 1: two waves only stage)
    constexpr int kPlane = kSlots * 16;
    constexpr int kItems = (kSlots + kThreads - 1) / kThreads;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, col = lane & 31;
    const int mtile = mtile0 + wave % G;
    const bool active = mtile < a.n_mtiles && (wave / G) * NI < kColumns / 32;
    const int k0 = blockIdx.y * kColumns;
    const int ch0 = (int)fast_div((unsigned)k0, a.d_taps);
    const int nch = (int)fast_div((unsigned)(min(k0 + kColumns, a.K) - 1), a.d_taps) - ch0 + 1;
    const int s = blockIdx.x;
    const int u0 = first_unit(a, s), u1 = first_unit(a, s + 1);

    // slot of this lane's patch elements relative to their pixel's
    int at[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int k = min(k0 + ((wave / G) * NI + i) * 32 + col, a.K - 1);
        const int c = (int)fast_div((unsigned)k, a.d_taps), tap = k - c * a.taps;
        const int dh = tap / a.bw;
        at[i] = (c - ch0) * a.chan + dh * a.pitch + (tap - dh * a.bw);
    }
    // this thread's staged slots: channel, row and column of the tile
    int src[kItems], rc[kItems];
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        const int e = tid + i * kThreads;
        const int c = (int)fast_div((unsigned)e, a.d_chan), rem = e - c * a.chan;
        const int r = (int)fast_div((unsigned)rem, a.d_pitch), cc = rem - r * a.pitch;
        rc[i] = c < nch && r < a.rows && cc < a.cols ? r << 16 | cc : -1;
        src[i] = (ch0 + c) * a.H * a.W;
    }
    if (tid < 6)
        *reinterpret_cast<float4 *>(lds + tid * kPlane + (kSlots - 1) * 16) = make_float4(0, 0, 0, 0);

    // [S2, S1], the leading product's and the lesser ones'
    f32x16 hi[2][NI], lo[2][NI];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            hi[f][i] = 0.0f;
            lo[f][i] = 0.0f;
        }
    const bf16x8 *pp = a.packed + ((size_t)(active ? mtile : 0) * a.units + u0) * a.pairs * 192 + lane;
    const bf16x8 *last = a.packed + (((size_t)(active ? mtile : 0) * a.units + u1) * a.pairs - 1) * 192 + lane;
    bf16x8 next[3];
#pragma unroll
    for (int q = 0; q < 3; ++q)
        next[q] = pp[q * 64];

    const size_t image = (size_t)a.C * a.H * a.W;
    const int vh = (a.oh - 1) * a.sh + a.bh, vw = (a.ow - 1) * a.sw + a.bw;   // what any output reads, padding included
    for (int u = u0; u < u1; ++u) {
        const Unit un = unit_of(a, u);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            if (rc[i] < 0)
                continue;
            const int e = tid + i * kThreads;
            const int vr = un.r0 * a.sh + (rc[i] >> 16), vc = un.c0 * a.sw + (rc[i] & 0xffff);
            const int r = vr - a.ph, c = vc - a.pw;
            const bool in = r >= 0 && r < a.H && c >= 0 && c < a.W, used = vr < vh && vc < vw;
            const float *p = a.x + (size_t)un.img * image + src[i] + (size_t)r * a.W + c;
            const float centre = a.ctr[ch0 + (int)fast_div((unsigned)e, a.d_chan)];
            float x[kImages];
#pragma unroll
            for (int j = 0; j < kImages; ++j)
                x[j] = in && un.img + j < a.B ? p[j * image] : a.oob;
            bf16x8 v[6];
#pragma unroll
            for (int j = 0; j < kImages; ++j) {
                const float d = used && un.img + j < a.B ? x[j] - centre : 0.0f;
                __bf16 p0, p1, p2;
                split3_any(d * d, p0, p1, p2);
                v[0][j] = p0; v[1][j] = p1; v[2][j] = p2;
                split3_any(d, p0, p1, p2);
                v[3][j] = p0; v[4][j] = p1; v[5][j] = p2;
            }
#pragma unroll
            for (int b = 0; b < 6; ++b)
                *reinterpret_cast<bf16x8 *>(lds + b * kPlane + e * 16) = v[b];
        }
        __syncthreads();
        int py = 0, pc = 0;
        for (int q = 0; q < a.pairs; ++q) {
            bf16x8 A[3];
#pragma unroll
            for (int i = 0; i < 3; ++i)
                A[i] = next[i];
            pp = pp < last ? pp + 192 : pp;
#pragma unroll
            for (int i = 0; i < 3; ++i)
                next[i] = pp[i * 64];
            const int px = 2 * pc + half;
            const int pix = py * a.sh * a.pitch + px * a.sw;
            const bool there = un.r0 + py < a.oh && un.c0 + px < a.ow;
            if (++pc == a.TW / 2) {
                pc = 0;
                ++py;
            }
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                // a pixel past the edge: zeros (its g is zero, but the input it would read may be infinite)
                const char *src_at = lds + (there ? at[i] + pix : kSlots - 1) * 16;
                bf16x8 B[6];
#pragma unroll
                for (int b = 0; b < 6; ++b)
                    B[b] = *reinterpret_cast<const bf16x8 *>(src_at + b * kPlane);
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    auto mul = [&](f32x16 &acc, int x, int y) {
                        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[x], B[3 * f + y], acc, 0, 0, 0);
                    };
                    mul(lo[f][i], 2, 0);
                    mul(lo[f][i], 0, 2);
                    mul(hi[f][i], 0, 0);
                    mul(lo[f][i], 1, 1);
                    mul(lo[f][i], 1, 0);
                    mul(lo[f][i], 0, 1);
                }
            }
        }
    }
    if (!active)
        return;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int k = k0 + ((wave / G) * NI + i) * 32 + col;
        if (k >= a.K)
            continue;
        params_store(a, mtile, k, s, half, a.ctr[(int)fast_div((unsigned)k, a.d_taps)], hi[0][i], lo[0][i], hi[1][i], lo[1][i]);
    }
}

// The same for 64 patch elements whose templates lie far from their channel's centre and near one another (whole-image
// patches, templates that began as one prototype): there S2 - 2 t' S1 + t'^2 G, t' = t - c, cancels, by 3e-4 of the
// gradient where what the templates share is 30 times what they differ by.  Centred element by element, over the 64
// templates of two tiles, t' is that difference.  A pixel that several taps read then needs a value for each, so a slot
// of LDS holds one patch element at one pixel: ten pixels at a time, staged for every 64 templates.  The gradients of
// 64 x 16 x 32 x 32, 64 templates, 4 x 4 at stride 4 take 21 us (one centre to a channel: 22, the fp32 form: 33) and have
// 1.0e-7 of error whatever is shared (fp32 form: 1.4e-7); 32 x 128 x 28 x 28, 128 templates, 3 x 3: 188 us (111, 212).
constexpr int kElemPairs = 5, kElemPitch = 2 * kElemPairs + 1;   // odd: see the note on pitches

__device__ __forceinline__ void params_elements_body(const ParamsArgs &a, char *lds, int mtile0)
{
    constexpr int kPlane = kSlots * 16;
    constexpr int kUsed = kColumns * kElemPitch, kItems = (kUsed + kThreads - 1) / kThreads;
    static_assert(kUsed <= kSlots, "a slot for every element and pixel");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, col = lane & 31;
    const int mtile = mtile0 + (wave & 1), kcol = (wave >> 1) * 32 + col;
    const bool active = mtile < a.n_mtiles;
    const int k0 = blockIdx.y * kColumns, s = blockIdx.x;
    const int u0 = first_unit(a, s), u1 = first_unit(a, s + 1);
    const float *centres = a.ctr64 + (size_t)(mtile0 / 2) * a.Kpad;

    // this thread's slots: patch element (tap and channel) and pixel of the ten (-1: none)
    int src[kItems], tap[kItems], pos[kItems];
    float ctr[kItems];
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        const int e = tid + i * kThreads, kl = e / kElemPitch, k = min(k0 + kl, a.K - 1);
        const int c = (int)fast_div((unsigned)k, a.d_taps), t = k - c * a.taps, dh = t / a.bw;
        pos[i] = e < kUsed && e - kl * kElemPitch < 2 * kElemPairs ? e - kl * kElemPitch : -1;
        tap[i] = dh << 16 | (t - dh * a.bw);
        src[i] = c * a.H * a.W;
        ctr[i] = centres[k];
    }
    f32x16 hi[2], lo[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        hi[f] = 0.0f;
        lo[f] = 0.0f;
    }
    const bf16x8 *pp = a.packed + ((size_t)(active ? mtile : 0) * a.units + u0) * a.pairs * 192 + lane;
    const size_t image = (size_t)a.C * a.H * a.W;
    for (int u = u0; u < u1; ++u) {
        const Unit un = unit_of(a, u);
        for (int q0 = 0; q0 < a.pairs; q0 += kElemPairs) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kItems; ++i) {
                if (pos[i] < 0)
                    continue;
                const int q = q0 + (pos[i] >> 1), py = (int)fast_div((unsigned)q, a.d_tw2);
                const int ro = un.r0 + py, co = un.c0 + 2 * (q - py * (a.TW / 2)) + (pos[i] & 1);
                const int r = ro * a.sh - a.ph + (tap[i] >> 16), c = co * a.sw - a.pw + (tap[i] & 0xffff);
                const bool in = r >= 0 && r < a.H && c >= 0 && c < a.W, there = q < a.pairs && ro < a.oh && co < a.ow;
                const float *p = a.x + (size_t)un.img * image + src[i] + (ptrdiff_t)r * a.W + c;
                float x[kImages];
#pragma unroll
                for (int j = 0; j < kImages; ++j)
                    x[j] = in && there && un.img + j < a.B ? p[j * image] : a.oob;
                bf16x8 v[6];
#pragma unroll
                for (int j = 0; j < kImages; ++j) {
                    const float d = there && un.img + j < a.B ? x[j] - ctr[i] : 0.0f;
                    __bf16 p0, p1, p2;
                    split3_any(d * d, p0, p1, p2);
                    v[0][j] = p0; v[1][j] = p1; v[2][j] = p2;
                    split3_any(d, p0, p1, p2);
                    v[3][j] = p0; v[4][j] = p1; v[5][j] = p2;
                }
#pragma unroll
                for (int b = 0; b < 6; ++b)
                    *reinterpret_cast<bf16x8 *>(lds + b * kPlane + (tid + i * kThreads) * 16) = v[b];
            }
            __syncthreads();
            const int n = min(kElemPairs, a.pairs - q0);
            for (int j = 0; j < n; ++j, pp += 192) {
                bf16x8 A[3], B[6];
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    A[i] = pp[i * 64];
#pragma unroll
                for (int b = 0; b < 6; ++b)
                    B[b] = *reinterpret_cast<const bf16x8 *>(lds + b * kPlane + (kcol * kElemPitch + 2 * j + half) * 16);
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    auto mul = [&](f32x16 &acc, int x, int y) {
                        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[x], B[3 * f + y], acc, 0, 0, 0);
                    };
                    mul(lo[f], 2, 0);
                    mul(lo[f], 0, 2);
                    mul(hi[f], 0, 0);
                    mul(lo[f], 1, 1);
                    mul(lo[f], 1, 0);
                    mul(lo[f], 0, 1);
                }
            }
        }
    }
    if (active && k0 + kcol < a.K)
        params_store(a, mtile, k0 + kcol, s, half, centres[k0 + kcol], hi[0], lo[0], hi[1], lo[1]);
}

// Whether these 64 patch elements' templates lie further from their channels' centres than the fp32 form, which centres
// each 64 templates element by element, would leave them: by a tenth of the sum of squares.  There the two forms' errors
// are equal (64 x 16 x 32 x 32, 64 templates, 4 x 4 at stride 4: 1.3e-7 and 1.4e-7; at twice the sum 4.1e-7 and 1.4e-7);
// templates without a common part stay below (1 + 1/24 on average with 24 of them, fewer do not come here).
__device__ __forceinline__ bool params_elements(const ParamsArgs &a)
{
    const int k = blockIdx.y * kColumns + (threadIdx.x & 63);
    float2 v = k < a.K ? a.spread[k] : make_float2(0.0f, 0.0f);
    for (int d = 32; d > 0; d >>= 1) {
        v.x += __shfl_xor(v.x, d, 64);
        v.y += __shfl_xor(v.y, d, 64);
    }
    return __builtin_amdgcn_readfirstlane(!(v.x <= 1.1f * v.y));
}

// blockIdx: (share of the pixels, 64 patch elements, template tiles dealt out as groups of 4, the rest as one of 4, 2 or 1)
__global__ __launch_bounds__(kThreads, 2) void sim_split_params_kernel(const ParamsArgs a)
{
    __shared__ __align__(16) char lds[kSlots * 16 * 6];
    const int mtile0 = blockIdx.z * 4, rest = a.n_mtiles - mtile0;
    if (params_elements(a)) {
        for (int two = 0; two < min(rest, 4); two += 2)
            params_elements_body(a, lds, mtile0 + two);
        return;
    }
    const int g = rest >= 3 ? 4 : rest;
    if (g == 4)
        params_body<4>(a, lds, mtile0);
    else if (g == 2)
        params_body<2>(a, lds, mtile0);
    else
        params_body<1>(a, lds, mtile0);
}

int round_to(int v, int residue)   // the smallest number from v on that is `residue` modulo 8
{
    return v + ((residue - v) % 8 + 8) % 8;
}

}  // namespace

SplitParamsPlan sim_split_params_plan(const SimPlan &p)
{
    SplitParamsPlan s = {};
    if (!p.split || (p.mode != SIM_MODE_L2 && p.mode != SIM_MODE_L2_NORM) || p.B == 0 || p.bh > 64 || p.bw > 64)
        return s;
    const int taps = p.bh * p.bw;
    const long long npix = 1LL * p.oh * p.ow, image = 1LL * p.C * p.H * p.W;
    if (p.K < 64 || p.O < 24 || image >= (1LL << 30) || 1LL * p.O * p.K >= (1LL << 30))
        return s;
    const int groups = (p.B + kImages - 1) / kImages;
    int most = 0;   // channels that 64 consecutive patch elements touch
    for (int k0 = 0; k0 < p.K && k0 < kColumns * taps; k0 += kColumns)
        most = std::max(most, (std::min(k0 + kColumns, p.K) - 1) / taps - k0 / taps + 1);
    s.n_mtiles = (p.O + kSplitRows - 1) / kSplitRows;
    const int g = s.n_mtiles >= 3 ? 4 : s.n_mtiles;
    // The output tile: per tile, cycles to stage (about 500 per round of 256 slots, and two barriers) and to multiply
    // (384 per pixel pair and column tile of a wave), over the image's tiles
    double best = 0;
    for (int th = 1; th <= std::min(p.oh, 16); ++th)
        for (int tw = 2; tw <= std::min((p.ow + 1) / 2 * 2, 64); tw += 2) {
            const int rows = (th - 1) * p.sh + p.bh, cols = (tw - 1) * p.sw + p.bw;
            const int pitch = round_to(cols, p.bw % 8), chan = round_to(rows * pitch, taps % 8);
            if (1LL * most * chan > kSlots - 1)
                break;
            const double tiles = 1.0 * ((p.oh + th - 1) / th) * ((p.ow + tw - 1) / tw);
            const double cost = tiles * (500.0 * ((most * chan + kThreads - 1) / kThreads) + 1000 + 384.0 * ((g + 1) / 2) * th * tw / 2);
            if (best == 0 || cost < best) {
                best = cost;
                s.TH = th; s.TW = tw; s.rows = rows; s.cols = cols; s.pitch = pitch; s.chan = chan;
            }
        }
    if (best == 0)
        return s;
    s.tiles_r = (p.oh + s.TH - 1) / s.TH;
    s.tiles_c = (p.ow + s.TW - 1) / s.TW;
    const long long units = 1LL * groups * s.tiles_r * s.tiles_c, pairs = s.TH * s.TW / 2;
    s.k_groups = (p.K + kColumns - 1) / kColumns;
    s.m_groups = (s.n_mtiles + 3) / 4;
    // worth it: enough of the products useful, enough of them, and the packed g of ordinary size
    const double useful = 1.0 * p.B * npix * p.O * p.K;
    const double padded = 2.0 * kImages * units * pairs * s.n_mtiles * kSplitRows * s.k_groups * kColumns;
    const long long packed = units * pairs * s.n_mtiles * 3 * 1024;
    if (useful < 0.3 * padded || useful < 3e7 || units * pairs >= (1LL << 30) || packed > (1LL << 30))
        return s;
    // shares of the pixels: two workgroups for every compute unit, of whole tiles
    const long long want = std::max<long long>(1, 512 / (s.k_groups * s.m_groups));
    const long long per = std::max<long long>(1, (units + want - 1) / want);
    s.S = (int)((units + per - 1) / per);
    s.units = (int)units;
    s.Opad = s.n_mtiles * kSplitRows;
    s.Kpad = s.k_groups * kColumns;
    const size_t slab = (size_t)s.Opad * s.Kpad * sizeof(float);
    s.partial = 0;
    s.centres = 3 * (size_t)s.S * slab;    // where the finish kernel reads them
    s.ctr = s.centres + slab;
    s.ctr64 = s.ctr + align_up((size_t)p.C * sizeof(float), 256);
    s.spread = s.ctr64 + (size_t)(s.n_mtiles + 1) / 2 * s.Kpad * sizeof(float);
    s.packed = s.spread + (size_t)s.Kpad * sizeof(float2);
    s.total = s.packed + (size_t)packed;
    s.on = true;
    return s;
}

int sim_split_params_launch(const SimPlan &p, const SplitParamsPlan &sp, const float *input, const float *templates,
                            const float *output_grad, char *ws, hipStream_t s)
{
    ParamsArgs a;
    a.g = output_grad; a.x = input; a.templates = templates;
    a.packed = reinterpret_cast<bf16x8 *>(ws + sp.packed);
    a.partial = reinterpret_cast<float *>(ws + sp.partial);
    a.centres = reinterpret_cast<float *>(ws + sp.centres);
    a.ctr = reinterpret_cast<float *>(ws + sp.ctr);
    a.ctr64 = reinterpret_cast<float *>(ws + sp.ctr64);
    a.spread = reinterpret_cast<float2 *>(ws + sp.spread);
    a.B = p.B; a.C = p.C; a.H = p.H; a.W = p.W; a.O = p.O; a.K = p.K; a.oh = p.oh; a.ow = p.ow;
    a.bh = p.bh; a.bw = p.bw; a.sh = p.sh; a.sw = p.sw; a.ph = p.ph; a.pw = p.pw; a.taps = p.bh * p.bw;
    a.Opad = sp.Opad; a.Kpad = sp.Kpad; a.S = sp.S; a.n_mtiles = sp.n_mtiles;
    a.TH = sp.TH; a.TW = sp.TW; a.pairs = sp.TH * sp.TW / 2;
    a.rows = sp.rows; a.cols = sp.cols; a.pitch = sp.pitch; a.chan = sp.chan;
    a.tiles_r = sp.tiles_r; a.tiles_c = sp.tiles_c; a.units = sp.units;
    a.oob = p.oob;
    a.d_pairs = make_fast_div((unsigned)a.pairs);
    a.d_tw2 = make_fast_div((unsigned)(sp.TW / 2));
    a.d_tiles = make_fast_div((unsigned)(sp.tiles_r * sp.tiles_c));
    a.d_tc = make_fast_div((unsigned)sp.tiles_c);
    a.d_chan = make_fast_div((unsigned)sp.chan);
    a.d_pitch = make_fast_div((unsigned)sp.pitch);
    a.d_taps = make_fast_div((unsigned)a.taps);
    hipLaunchKernelGGL(sim_split_params_pack_kernel, dim3(p.C + sp.S * sp.n_mtiles * kPackGroups), dim3(kThreads), 0, s, a);
    hipLaunchKernelGGL(sim_split_params_kernel, dim3(sp.S, sp.k_groups, sp.m_groups), dim3(kThreads), 0, s, a);
    return hipGetLastError() == hipSuccess ? SIMNETS_OK : SIMNETS_ERR_HIP;
}

}  // namespace simnets
