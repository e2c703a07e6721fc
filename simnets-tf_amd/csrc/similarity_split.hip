// The L2 Similarity modes as a matrix product on the 16-bit matrix cores, at the precision of fp32 (gfx950).
//
//   sum_k w (x - t)^2 = sum_k w x'^2 - 2 w t' x' + w t'^2,   x' = x - c, t' = t - c, c one value per channel
// is a contraction of (w, -2 w t') with (x'^2, x').  Forward: every factor is the sum of two half-precision pieces of 11
// bits, hi + lo (split2), and three products of pieces are formed on v_mfma_f32_32x32x16_f16; the one left out, lo lo, is
// below 2^-22 of the whole with either sign.  Half precision has a narrow exponent: the packing kernel scales channels and
// templates by powers of two (split_pack_block), the lesser piece of a value is kept times 2048 and meets a copy of hi
// divided by as much, workgroups whose inputs are on another scale than the templates take smaller ones (split_body), and a
// value that overflows all the same makes its outputs NaN, which the guard below hands on.  Input gradient: three bf16
// pieces and six products (see the end of the file).
//
// Precision.  The matrix unit cuts what lies below 2^-26 of a sum off each of its products, and these have 22 bits: of
// terms of one sign that is a bias (4.4e-7 at 576 elements).  So the squares are those about their channel's sampled mean,
// x'^2 - m, whose sums stay small and have no bias, and a chunk's products (144 elements of 3 x 3) have a sum of their own
// that is added in fp32.  Error against 64 bits (2-norm, relative; weights 0.1 to 2): 64 channels, 3 x 3, inputs unrelated to
// the templates 0.45e-7 (three bf16 pieces 0.8e-7, term by term 3.6e-7), all zero 0.65e-7 (0.6e-7, 4.1e-7), without their
// negative values 0.4e-7, ten to 10^7 times the templates 0.7e-7 (1.7e-7, 3.5e-7); 256 channels, 1 x 1, 0.4e-7 to 0.6e-7 (2.3e-7).
// Inputs near a template lose to cancellation, as T / out, T = sum w t'^2.  A patch at out / T = 2, 1 and 0.5 from its
// template, 576 elements: 0.9e-7, 1.4e-7 and 2.4e-7 (root mean square; term by term 3.6e-7), 2304: 0.6e-7, 0.9e-7, 2.1e-7
// (7.2e-7), 64: 0.8e-7, 1.1e-7, 1.2e-7 (1.2e-7).  The guard's line lies at 0.43 T (half for the shortest patches,
// split_line).  It also lies where the pieces' own limits would show: parameters far below their template's largest,
// values far below what the tile holds (split_pack_block).
// An output below the line (or below 1/1024 of the uncentred sum w t^2, the guard of the sqrt-weight form; or not finite) is
// computed again term by term by its workgroup (split_recompute), and the others keep their value.  A tile with more of
// them than that is worth, or with a template whose parameters are negative, huge or tiny, is flagged and left whole to
// the direct kernel's launch behind this one, which otherwise returns at once.
// Templates fitted to the inputs (k-means of 1/f images with three factors over the channels): 256 x 64 x 32 x 32 -> 128, 3 x 3,
// 0.3 % of the outputs below the line: 319 us (unrelated templates 228, sqrt-weight form 764, direct kernel 1017); 64 x
// 16 x 32 x 32 -> 64, 0.3 %: 36 (28, 49, 49); 64 x 8 x 32 x 32 -> 32, 72 elements, 1.5 % and 2.1 %: 28 and 30 (22, 25, 26).  Where many
// tiles are left: 64 x 32 x 32 x 32 -> 64 of two factors, 1.2 %: 136 (35, 85, 86); 256 x 8 x 32 x 32 -> 32, 3 %: 109 (42, 49, 50); 256 x 576 x
// 14 x 14 -> 128, 1 x 1, 7 %: 585 (132, 864, 455).
//
// Missing values (NaN inputs ignored): both operands 0 and a third, the 0/1 mask of present values, which contracts with
// -w (t'^2 + m) and with the logarithm term, two pieces each; T is that of the present values.
//
// Layout.  A workgroup of four waves computes 128 consecutive output pixels (over the batch: images are a stack of
// padded rows, so a tile may span images and no lane idles at an image's end) x up to 128 templates.  16 channels (or
// 8) of the rows it touches are staged in LDS as [piece][channel group of 8][pixel][8 channels], converted once and read
// by every tap and template; a lane's matrix operand - 8 channels of its pixel - is one ds_read_b128, consecutive
// lanes' in consecutive 16 bytes.  The parameters are packed in the order the lanes read them and come from L2 straight
// into registers, one step ahead; the next chunk's input is requested during a chunk's last step, by buffer loads (an
// offset per pixel, one per channel, zeros outside of the image: no 64-bit address per value).  256 registers: two
// workgroups per compute unit, so that one stages while the other multiplies.
// Where tiles are few for that, or the input gradient's rows many, a workgroup of eight waves to a compute unit, with two buffers:
// split_forward_wide, split_grad_wide.
//
// Measured (whole call, vector form, three bf16 pieces, this form): 256 x 64 x 32 x 32 -> 128, 3 x 3: 0.80, 0.372, 0.229 ms.
// The kernel's 211 us are 1.1 PFLOP/s of matrix products at 1.55 GHz, matrix units busy 56 %: the clock sinks with them
// (products of random numbers alone run at 1.57 PFLOP/s and 1.65 GHz, of zeros at 2.35), 155 us would be that rate.  37 x 45 x
// 29 x 35 -> 75: 172, 66, 50 us, where half of the products are padding (96 templates, 48 channels, 37632 pixels).  64 images of
// the first with a quarter missing: 427, 160, 110 us.
// Tried: 2 x 2 tiles a wave (half of the LDS reads, twice the parameter loads): 250 us for 228.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "fast_div.h"
#include "internal.h"
#include "sim_split.h"
#include "split_channel.h"

namespace simnets {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(1))) float global_float;
typedef __attribute__((address_space(1))) float2_t global_float2;

constexpr int kThreads = 256;
enum SplitKind { SPLIT_FWD, SPLIT_MASKED /* forward, NaN inputs ignored */, SPLIT_GRAD /* input gradient */ };

// staged pixels of a chunk of 16 channels (twice as many of 8): two workgroups' tiles fit the 160 KB of a compute unit
constexpr int split_lds_pixels(int kind) { return kind == SPLIT_MASKED ? 360 : kind == SPLIT_FWD ? 408 : 816; }
constexpr int split_operands(int kind) { return kind == SPLIT_MASKED ? 5 : kind == SPLIT_FWD ? 4 : 3; }
constexpr int split_lds_bytes(int kind) { return split_lds_pixels(kind) * 32 * split_operands(kind); }
// pixels of one staged plane [channel group][pixel]
constexpr int split_plane_pixels(int kind, int cg) { return split_lds_pixels(kind) * (cg == 16 ? 1 : 2); }
constexpr int split_pieces(int kind) { return kind == SPLIT_MASKED ? 8 : kind == SPLIT_FWD ? 4 : 6; }

struct SplitArgs {
    const float *in;
    float *out;
    const void *packed;
    const float *chan, *rows;   // see SplitPack
    const float *ctr;           // input gradient: centres of the rows
    const float2 *exact;   // see SplitPack
    const float *logs;
    int *flags;      // [pixel tile][mtile]
    int C, H, W, O, ow, npix, total;   // npix = oh ow, total = B npix
    int bw, sh, sw, ph, pw, taps, chunks, steps, n_mtiles, Wp, Hv;
    int gmax;        // matrix tiles of templates per workgroup: 4, 2 or 1
    int per_sum;     // chunks whose products share accumulators
    float oob;
    const float *x;  // input gradient: the forward's input, of the output's shape; templates and weights [C][O][taps]
    const float *templates, *weights;
    float scale;
    float norm_const;
    int K;
    FastDiv d_npix, d_ow, d_wp, d_hv, d_taps, d_bw;
};

// Cold paths read the kernel's arguments again from its argument segment (they end where the implicit arguments begin; the
// kernel's other argument is an int), instead of keeping them in registers past the main loop.
#if defined(__HIP_DEVICE_COMPILE__)
static_assert(sizeof(SplitArgs) % 8 == 0, "the explicit arguments end 8 bytes behind the block");
__device__ __forceinline__ const SplitArgs &split_kernel_args()
{
    return *reinterpret_cast<const SplitArgs *>(reinterpret_cast<const char *>(__builtin_amdgcn_implicitarg_ptr()) -
                                                (sizeof(SplitArgs) + 8));
}

// Input gradient of one element (input channel ch, pixel rem of its image) term by term: where the sums A and (x - c) B are
// infinite with one sign, only the terms tell which way their difference goes.  Not inlined: the main loop's registers and
// schedule stay as they are.
__device__ __noinline__ float split_grad_terms(int img, int ch, int rem, float x)
{
    const SplitArgs &a = split_kernel_args();
    const int y = rem / a.ow, xo = rem - y * a.ow;
    float sum = 0.0f;
    for (int o = 0; o < a.C; ++o)
        for (int tap = 0; tap < a.taps; ++tap) {
            const int dh = tap / a.bw, r = y + dh - a.ph, c = xo + tap - dh * a.bw - a.pw;
            if (r < 0 || r >= a.H || c < 0 || c >= a.W)
                continue;
            const size_t at = ((size_t)o * a.O + ch) * a.taps + (a.taps - 1 - tap);
            sum += a.in[(((size_t)img * a.C + o) * a.H + r) * a.W + c] * (a.scale * a.weights[at]) * (a.templates[at] - x);
        }
    return sum;
}

// Outputs of a tile (of 4096) that a workgroup recomputes by itself.  One at a time 2.5 % of them (256 x 576 x 14 x 14 -> 128, 1 x
// 1: 17.9 ms for all, the direct kernel 0.45) to 3.3 % (64 x 144 x 32 x 32 -> 64: 2.3 ms, 0.08) take as long as the tile does
// on the direct kernel.
constexpr int kSplitListed = 192;   // (fitted templates have a few tiles with five times the mean)

// LDS of a workgroup whose products are done and that has outputs to recompute.
template <int KIND, int CG>
struct NearOutputs {
    static constexpr int kPlane = split_plane_pixels(KIND, CG);
    int count[4], total;                            // of each template tile, and of the list
    float sum[4 * kSplitListed];
    float x[CG * kPlane];                           // a chunk's channels of the rows that the pixels read
    unsigned short list[4 * kSplitListed];          // pixel << 7 | template
    unsigned short element[CG * kPlane];            // where a patch element of the chunk lies in x
};

// Outputs below the guard's line, term by term with the direct kernels' arithmetic, eight lanes to an output and twelve
// terms of a lane in flight; their patches from memory where they are few, else from the rows, staged again in fp32, chunk
// by chunk.  near[i]: this lane's, bit r.  A tile with more of them than kSplitListed, or with a template whose
// parameters are out of range, is flagged for the direct kernel instead.  G: the workgroup's template tiles, 4, 2 or 1.
// LOGS: the mode has logarithm terms.  Inlined once, at the kernel's end: a call, or a copy in each split_body, spills SGPRs of
// the bodies (37 x 45 x 29 x 35 -> 75 62 -> 65 to 72 us).
template <int KIND, int CG, bool LOGS, int WAVES>
__device__ __forceinline__ void split_recompute(lds_char *lds, int ptile, int mtile0, int G, u32x4 near)
{
    constexpr int kThreads = 64 * WAVES, kLanes = 8, kTerms = 12, kOutputs = kThreads / kLanes;
    typedef NearOutputs<KIND, CG> Near;
    static_assert(sizeof(Near) <= split_lds_bytes(KIND), "in the memory of the staged pieces");
    const SplitArgs a = split_kernel_args();
    __attribute__((address_space(3))) Near &q = *(__attribute__((address_space(3))) Near *)lds;
    const int tid = threadIdx.x, wave = tid >> 6, n0 = ptile * kSplitPixels;
    if (tid < 4)
        q.count[tid] = 0;
    if (tid == 4)
        q.total = 0;
    __syncthreads();
    int bits = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        bits += __builtin_popcount(near[i]);
    if (bits)
        atomicAdd((int *)&q.count[wave % G], bits);
    if (tid < G * kSplitRows && mtile0 + tid / kSplitRows < a.n_mtiles && a.rows[4 * (mtile0 * kSplitRows + tid) + SPLIT_THR] == INFINITY)
        atomicAdd((int *)&q.count[tid / kSplitRows], kSplitPixels * kSplitRows);
    __syncthreads();
    for (int g = 0; g < G && mtile0 + g < a.n_mtiles; ++g) {
        const int outputs = min(kSplitPixels, a.total - n0) * min(kSplitRows, a.O - (mtile0 + g) * kSplitRows);
        const bool leave = q.count[g] > min(kSplitListed, outputs / 2);
        if (tid == 0)
            a.flags[(size_t)ptile * a.n_mtiles + mtile0 + g] = leave;
        if (wave % G != g || leave || !bits)
            continue;
        int slot = atomicAdd((int *)&q.total, bits);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            for (unsigned rest = near[i]; rest; rest &= rest - 1, ++slot) {
                const int r = __builtin_ctz(rest), ml = g * kSplitRows + 8 * (r / 4) + 4 * (tid >> 5 & 1) + r % 4;
                q.list[slot] = (unsigned short)((((wave / G) * (4 * G / WAVES) + i) * 32 + (tid & 31)) << 7 | ml);
            }
    }
    __syncthreads();
    const int listed = q.total, lane = tid % kLanes;
    const global_float *in = (const global_float *)a.in, *logs = (const global_float *)a.logs;
    const global_float2 *exact = (const global_float2 *)a.exact;
    auto pixel = [&](int e, int &img, int &rem, int &r, int &c) {   // its image, place in it, output row and column
        const int n = n0 + (q.list[e] >> 7);
        img = (int)fast_div((unsigned)n, a.d_npix);
        rem = n - img * a.npix;
        r = (int)fast_div((unsigned)rem, a.d_ow);
        c = rem - r * a.ow;
    };
    auto store = [&](int e, float sum) {
        int img, rem, r, c;
        pixel(e, img, rem, r, c);
        const int m = mtile0 * kSplitRows + (q.list[e] & 127);
        ((global_float *)a.out)[((size_t)img * a.O + m) * a.npix + rem] = LOGS ? sum + a.norm_const : sum;
    };
    // n terms of list entry e, from patch element k on, summed over its lanes; value(j): the input under the j-th
    auto terms = [&](int e, int k, int n, auto value) {
        const size_t at = (size_t)(mtile0 * kSplitRows + (q.list[e] & 127)) * a.K + k;
        float sum = 0.0f;
        for (int j0 = lane; j0 < n; j0 += kLanes * kTerms) {
            float x[kTerms], l[kTerms];
            float2_t tw[kTerms];
#pragma unroll
            for (int i = 0; i < kTerms; ++i) {   // behind the last: the last
                const int j = min(j0 + kLanes * i, n - 1);
                tw[i] = exact[at + j];
                l[i] = LOGS ? logs[at + j] : 0.0f;
                x[i] = value(j);
            }
#pragma unroll
            for (int i = 0; i < kTerms; ++i) {
                const float d = tw[i].x - x[i], term = __builtin_fmaf(tw[i].y * d, d, l[i]);
                sum += j0 + kLanes * i >= n || (KIND == SPLIT_MASKED && x[i] != x[i]) ? 0.0f : term;
            }
        }
        for (int d = kLanes / 2; d > 0; d >>= 1)
            sum += __shfl_xor(sum, d, kLanes);
        return sum;
    };
    if (listed <= kOutputs) {
        const int e = tid / kLanes;
        if (e >= listed)
            return;
        int img, rem, r, c;
        pixel(e, img, rem, r, c);
        const int r0 = r * a.sh - a.ph, c0 = c * a.sw - a.pw, first = (img * a.C * a.H + r0) * a.W + c0;
        const float sum = terms(e, 0, a.K, [&](int k) {
            const int ch = (int)fast_div((unsigned)k, a.d_taps), tap = k - ch * a.taps;
            const int dh = (int)fast_div((unsigned)tap, a.d_bw), dw = tap - dh * a.bw, h = r0 + dh, w = c0 + dw;
            const bool inside = (h >= 0) & (h < a.H) & (w >= 0) & (w < a.W);
            const float x = in[inside ? first + (ch * a.H + dh) * a.W + dw : 0];
            return inside ? x : a.oob;
        });
        if (lane == 0)
            store(e, sum);
        return;
    }
    auto virtual_row = [&](int n) {   // of the stack of padded images, as in split_body
        const int img = (int)fast_div((unsigned)n, a.d_npix);
        return img * a.Hv + (int)fast_div((unsigned)(n - img * a.npix), a.d_ow) * a.sh;
    };
    const int v0 = virtual_row(n0);
    const int rows = virtual_row(min(n0 + kSplitPixels, a.total) - 1) - v0 + a.taps / a.bw;
    const int staged = min(rows * a.Wp, Near::kPlane);
    for (int k = tid; k < CG * a.taps; k += kThreads) {
        const int ch = (int)fast_div((unsigned)k, a.d_taps), tap = k - ch * a.taps;
        const int dh = (int)fast_div((unsigned)tap, a.d_bw);
        q.element[k] = (unsigned short)(ch * Near::kPlane + dh * a.Wp + tap - dh * a.bw);
    }
    const size_t plane = (size_t)a.H * a.W;
    for (int chunk = 0; chunk < a.chunks; ++chunk) {
        const int channels = min(CG, a.C - chunk * CG);
        for (int p = tid; p < staged; p += kThreads) {
            const int vr = (int)fast_div((unsigned)p, a.d_wp), c = p - vr * a.Wp - a.pw;
            const int img = (int)fast_div((unsigned)(v0 + vr), a.d_hv), r = v0 + vr - img * a.Hv - a.ph;
            const bool inside = (r >= 0) & (r < a.H) & (c >= 0) & (c < a.W);
            const size_t at = inside ? ((size_t)(img * a.C + chunk * CG) * a.H + r) * a.W + c : 0;
            float x[CG];
#pragma unroll
            for (int j = 0; j < CG; ++j)
                x[j] = in[inside ? at + min(j, channels - 1) * plane : 0];
#pragma unroll
            for (int j = 0; j < CG; ++j)
                q.x[j * Near::kPlane + p] = inside ? x[j] : a.oob;
        }
        __syncthreads();
        for (int e = tid / kLanes; e < listed; e += kOutputs) {
            int img, rem, r, c;
            pixel(e, img, rem, r, c);
            const int base = (img * a.Hv + r * a.sh - v0) * a.Wp + c * a.sw;
            float sum = terms(e, chunk * CG * a.taps, channels * a.taps, [&](int j) { return q.x[base + q.element[j]]; });
            if (lane == 0) {
                sum += chunk == 0 ? 0.0f : q.sum[e];
                if (chunk + 1 < a.chunks)
                    q.sum[e] = sum;
                else
                    store(e, sum);
            }
        }
        __syncthreads();
    }
}
#endif

// How a workgroup's pixels, 128 from n0 on, lie in the stack of padded images: the virtual row of the first, and what is
// staged for them.
__device__ __forceinline__ int split_virtual_row(const SplitArgs &a, int n, int &img, int &c)
{
    img = (int)fast_div((unsigned)n, a.d_npix);
    const int rem = n - img * a.npix, r = (int)fast_div((unsigned)rem, a.d_ow);
    c = rem - r * a.ow;
    return img * a.Hv + r * a.sh;
}

// Input gradient.  One workgroup of WAVES waves: G template tiles of 32 (from mtile0) x 128 pixels; a wave holds one template
// tile x NI pixel tiles.  Four waves, two workgroups to a compute unit: each stages a chunk between two barriers while the other
// multiplies.  Eight waves (G = 4 or 2), one to a compute unit: twice the rows from what is staged; the next chunk's values are
// requested two steps ahead and converted into a second buffer, so that a wave does so while another one multiplies.
template <int CG, int G, int WAVES>
__device__ __forceinline__ void split_grad_body(const SplitArgs &a, char *lds, int ptile, int mtile0, int flag)
{
    constexpr int KIND = SPLIT_GRAD;
    constexpr bool WIDE = WAVES == 8;
    constexpr int NI = 4 * G / WAVES, NB = split_operands(KIND), NA = split_pieces(KIND);
    constexpr int P = split_plane_pixels(KIND, CG);
    constexpr int kPlane = split_lds_pixels(KIND) * 32;
    constexpr int kHalves = CG / 8;                               // groups of eight channels
    constexpr int kItems = (kHalves * ((P + 63) / 64) + WAVES - 1) / WAVES;   // of 64 pixels and eight channels
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, col = lane & 31;
    const int mtile = mtile0 + wave % G;
    const int ntile0 = (wave / G) * NI;

    const int n0 = ptile * kSplitPixels;
    int img0, img1, c0, c1;
    const int v0 = split_virtual_row(a, n0, img0, c0);
    const int rows = split_virtual_row(a, min(n0 + kSplitPixels, a.total) - 1, img1, c1) - v0 + a.taps / a.bw;
    const int staged = min(rows * a.Wp, P), per_half = (staged + 63) / 64;

    // where this lane's staged elements come from (the same for every chunk): bytes from the tile's first image for the loads
    // of eight waves, which give zero outside of it; elements of the whole tensor, which may be larger, for those of four
    constexpr unsigned kOutside = WIDE ? 0x80000000u : 0xffffffffu;
    const unsigned plane = (unsigned)a.H * a.W;
    const int first = WIDE ? img0 : 0;
    const float *base = a.in + (size_t)first * a.C * plane;
    const size_t behind = (size_t)(a.total / a.npix - first) * a.C * plane * 4u;
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)(behind < 0x7ffffffcu ? behind : 0x7ffffffcu), 0x00020000);
    unsigned src[kItems];
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        const int item = wave + WAVES * i, g = CG == 16 && item >= per_half, q = (item - (g ? per_half : 0)) * 64 + lane;
        const int vr = (int)fast_div((unsigned)q, a.d_wp), c = q - vr * a.Wp - a.pw;
        const int v = v0 + vr, img = (int)fast_div((unsigned)v, a.d_hv), r = v - img * a.Hv - a.ph;
        const bool in = q < staged && r >= 0 && r < a.H && c >= 0 && c < a.W;
        src[i] = in ? (unsigned)((((img - first) * a.C + split_group_start(a.C, g)) * a.H + r) * a.W + c) * (WIDE ? 4u : 1u) : kOutside;
    }
    // and this lane's operands: the LDS byte address of its pixel's first tap
    int at[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        int img, c;
        const int v = split_virtual_row(a, min(n0 + (ntile0 + i) * 32 + col, a.total - 1), img, c);
        at[i] = ((CG == 16 ? half * P : 0) + (v - v0) * a.Wp + c * a.sw) * 16;
    }

    // hi[0] + lo[0] = A, hi[1] + lo[1] = B
    f32x16 hi[2][NI], lo[2][NI];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            hi[f][i] = 0.0f;
            lo[f][i] = 0.0f;
        }
    const bool active = mtile < a.n_mtiles;
    const bf16x8 *pp = (const bf16x8 *)a.packed + (size_t)(active ? mtile : 0) * a.chunks * a.steps * NA * 64;
    bf16x8 next[NA];
#pragma unroll
    for (int q = 0; q < NA; ++q)
        next[q] = pp[q * 64 + lane];

    constexpr int kAhead = WIDE ? 2 : 0;   // items requested ahead: up to 512 pixels' of sixteen channels
    float x[kItems][8];
    auto request_item = [&](int i, int chunk) {   // channels behind the last as the last
        const int item = wave + WAVES * i;
        if (item >= kHalves * per_half)
            return;
        const int g = CG == 16 && item >= per_half, start = split_group_start(a.C, g);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const unsigned channel = split_channel_offset(a.C, start, chunk * CG, j);
            if (WIDE)
                x[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, src[i], channel * plane * 4u, 0));
            else
                x[i][j] = src[i] != kOutside ? base[(size_t)src[i] + (size_t)channel * plane] : 0.0f;
        }
    };
    auto stage_item = [&](int i, int chunk, char *to) {
        const int item = wave + WAVES * i;
        if (item >= kHalves * per_half)
            return;
        const int g = CG == 16 && item >= per_half, q = (item - (g ? per_half : 0)) * 64 + lane;
        const int c0 = chunk * CG + 8 * g;
        if (c0 + 8 > a.C)   // channels behind the last have zero parameters: any finite value will do
#pragma unroll
            for (int j = 0; j < 8; ++j)
                x[i][j] = c0 + j < a.C ? x[i][j] : 0.0f;
        bf16x8 v[3];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            __bf16 p0, p1, p2;
            split3_any(x[i][j], p0, p1, p2);
            v[0][j] = p0; v[1][j] = p1; v[2][j] = p2;
        }
        if (q < staged) {
            char *dst = to + (g * P + q) * 16;
#pragma unroll
            for (int b = 0; b < NB; ++b)
                *reinterpret_cast<bf16x8 *>(dst + b * kPlane) = v[b];
        }
    };
    auto request = [&](int chunk) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
            request_item(i, chunk);
    };
    auto stage = [&](int chunk, char *to) {
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            if (i >= kAhead)
                request_item(i, chunk);
            stage_item(i, chunk, to);
        }
    };
    if (WIDE) {
        request(0);
        stage(0, lds);
    }
    for (int chunk = 0; chunk < a.chunks; ++chunk) {
        const char *from = lds + (WIDE && (chunk & 1) ? split_lds_bytes(KIND) : 0);
        const bool more = chunk + 1 < a.chunks;
        __syncthreads();
        if (!WIDE) {
            stage(chunk, lds);
            __syncthreads();
        }
        int dh = 0, dw = 0;
        const int taps_h = a.taps / a.bw;
        auto next_tap = [&]() {   // LDS offset of the next tap (behind the last: of the first, with zero parameters)
            const int off = dh < taps_h ? (dh * a.Wp + dw) * 16 : 0;
            if (++dw == a.bw) {
                dw = 0;
                ++dh;
            }
            return off;
        };
        auto next_offset = [&]() {   // of a step's operands
            const int off = next_tap();
            if (CG == 16)
                return off;
            const int off2 = next_tap();
            return half ? off2 : off;
        };
        constexpr int kNext = WIDE && NI > 1 ? 1 : 0;   // (of a pixel tile and of the one behind it; no registers left for it with four waves)
        bf16x8 B[1 + kNext][NB];
        auto fetch = [&](bf16x8 (&to)[NB], int off) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
                to[b] = *reinterpret_cast<const bf16x8 *>(from + off + b * kPlane);
        };
        int off = next_offset();
        if (kNext)
            fetch(B[0], at[0] + off);
        auto multiply = [&](int step, bool ask) {   // ask: for the next chunk's values, behind the next step's parameters
            bf16x8 A[NA];
#pragma unroll
            for (int q = 0; q < NA; ++q)
                A[q] = next[q];
            if (more || step + 1 < a.steps)
                pp += NA * 64;
#pragma unroll
            for (int q = 0; q < NA; ++q)
                next[q] = pp[q * 64 + lane];
            if (ask)
                request(chunk + 1);
            const int off_next = next_offset();
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                if (kNext) {
                    fetch(B[(i + 1) & kNext], i + 1 < NI ? at[(i + 1) % NI] + off : at[0] + off_next);
                    __builtin_amdgcn_sched_barrier(0);
                } else
                    fetch(B[0], at[i] + off);
                // an accumulator's products follow one another at 48 cycles, two accumulators' in turn at 32
                auto products = [&](f32x16 (&to)[2][NI], int p, int v) {
#pragma unroll
                    for (int f = 0; f < 2; ++f)
                        to[f][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[3 * f + p], B[i & kNext][v], to[f][i], 0, 0, 0);
                };
                products(lo, 2, 0);
                products(lo, 0, 2);
                products(hi, 0, 0);
                products(lo, 1, 1);
                products(lo, 1, 0);
                products(lo, 0, 1);
                if (kNext)
                    __builtin_amdgcn_sched_barrier(0);
            }
            static_assert(!kNext || NI % 2 == 0, "the last of a step fetches the next one's first into place 0");
            off = off_next;
        };
        for (int step = 0; step < a.steps; ++step)
            multiply(step, WIDE && more && step == max(0, a.steps - 2));
        if (WIDE && more)
            stage(chunk + 1, lds + (chunk & 1 ? 0 : split_lds_bytes(KIND)));
    }

    // lane: pixel col of each tile, templates (input gradient: channels) 8 (r / 4) + 4 half + r % 4
    if (!active)
        return;
    float ctr[16];
#pragma unroll
    for (int r = 0; r < 16; ++r)
        ctr[r] = a.ctr[mtile * kSplitRows + 8 * (r / 4) + 4 * half + r % 4];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int n = n0 + (ntile0 + i) * 32 + col;
        if (n >= a.total)
            continue;
        const int img = (int)fast_div((unsigned)n, a.d_npix);
        const size_t base = ((size_t)img * a.O + mtile * kSplitRows) * a.npix + (n - img * a.npix);
        float x[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int ml = min(8 * (r / 4) + 4 * half + r % 4, a.O - 1 - mtile * kSplitRows);
            x[r] = a.x[base + (size_t)ml * a.npix];
        }
        float v[16], any = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            v[r] = __builtin_fmaf(-(x[r] - ctr[r]), hi[1][i][r] + lo[1][i][r], hi[0][i][r] + lo[0][i][r]);
            any = __builtin_fmaf(v[r], 0.0f, any);   // NaN once a value is not finite
        }
        if (any != any) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float A = split_sum(hi[0][i][r], lo[0][i][r]);
                v[r] = __builtin_fmaf(-(x[r] - ctr[r]), split_sum(hi[1][i][r], lo[1][i][r]), A);
#if defined(__HIP_DEVICE_COMPILE__)
                if (v[r] != v[r] && __builtin_isinf(A))
                    v[r] = split_grad_terms(img, min(mtile * kSplitRows + 8 * (r / 4) + 4 * half + r % 4, a.O - 1),
                                            n - img * a.npix, x[r]);
#endif
                if (flag && x[r] != x[r])
                    v[r] = 0.0f;
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int ml = 8 * (r / 4) + 4 * half + r % 4;
            if (mtile * kSplitRows + ml < a.O)
                a.out[base + (size_t)ml * a.npix] = v[r];
        }
    }
}

#if defined(__HIP_DEVICE_COMPILE__)
typedef const __attribute__((address_space(4))) float uniform_float;

// What a workgroup knows of the sizes it has staged.
struct SplitFar {
    int most[2];                       // the largest |x'| s so far: a float's bits, as which they are compared; chunks of even and odd numbers
    int lanes[3][kSplitLevels - 1];    // of three chunks in turn: with a value that the next level keeps, see split_body
};

// Raises far.most to a lane's value, rounded up to a quarter of an octave: so a workgroup does it a few times.  (One instruction
// and not the compiler's loop over the lanes.)
__device__ __forceinline__ void split_far_most(__attribute__((address_space(3))) int &most, float value)
{
    asm volatile("ds_max_i32 %0, %1\n\ts_waitcnt lgkmcnt(0)"
                 :
                 : "v"((unsigned)(uintptr_t)&most), "v"(__float_as_int(value) | 0x1fffff)
                 : "memory");
}

// Forward.  One workgroup: G template tiles of 32 (from mtile0) x 128 pixels; a wave holds one template tile x NI pixel
// tiles.  Where the inputs are much larger than what the templates differ by, so that the square of one is beyond half
// precision, the workgroup goes on at a smaller scale of the channels (a level, 2^-3 each, packed by the packing kernel): its
// sums are scaled, the chunk is staged again, and the cross terms' parameters are multiplied on the way.  Ordinary values
// keep their bits at the first level (what it may lose, 2^-7 / sqrt(K) of the weights' sum, is below the guard's line);
// for the higher ones an eighth of the lanes need values that count there, and where only a few pixels are that large
// their outputs become NaN and are recomputed.  256 x 64 x 32 x 32 -> 128, 3 x 3, templates of size 0.05, inputs 0..255 or 0..10^7:
// 220 us, where all tiles left to the direct kernel took 1190; inputs 0.05 and a border of 100: 222 and 1222; one pixel in a
// hundred 10^3 times the others: 225 and 1440, 10^4 times: 1490 and 1470.  What it costs ordinary inputs: 1 to 2 us there,
// 1 of 50 on 37 x 45 x 29 x 35 -> 75, 2 of 54 on 64 x 256 x 32 x 32 -> 64, 1 x 1.
//
// WAVES: four, two workgroups to a compute unit, each of which stages a chunk between two barriers while the other multiplies;
// or eight, one to a unit, all rows from what is staged once: the next chunk's values are requested two steps ahead and
// converted into a second buffer.  A barrier a chunk then: a wave may be a chunk ahead of another that has yet to read far, so
// that consecutive chunks have places of their own there.
template <int KIND, int CG, int G, int WAVES>
__device__ __forceinline__ void split_body(const SplitArgs &a, char *lds, __attribute__((address_space(3))) SplitFar &far,
                                           u32x4 &near, int ptile, int mtile0, int norm)
{
    constexpr bool MASKED = KIND == SPLIT_MASKED;
    constexpr bool WIDE = WAVES == 8;
    constexpr int NI = 4 * G / WAVES, NB = split_operands(KIND), NA = split_pieces(KIND), kWaves = WAVES;
    constexpr int P = split_plane_pixels(KIND, CG);
    constexpr int kPlane = split_lds_pixels(KIND) * 32;
    constexpr int kHalves = CG / 8;                               // groups of eight channels
    constexpr int kItems = (kHalves * ((P + 63) / 64) + kWaves - 1) / kWaves;   // of 64 pixels and eight channels
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, col = lane & 31;
    const int mtile = mtile0 + wave % G;
    const int ntile0 = wave / G * NI;
    constexpr int kLastLevel = MASKED ? kSplitMaskedLevels - 1 : kSplitLevels - 1;

    const int n0 = ptile * kSplitPixels;
    int img0, img1, c0, c1;
    const int v0 = split_virtual_row(a, n0, img0, c0);
    const int rows = split_virtual_row(a, min(n0 + kSplitPixels, a.total) - 1, img1, c1) - v0 + a.taps / a.bw;
    const int staged = min(rows * a.Wp, P), per_half = (staged + 63) / 64;

    // The images from this tile's first on, for loads that give zero outside of them (and wherever voffset is kOutside).
    const unsigned plane = (unsigned)a.H * a.W * 4u;
    constexpr unsigned kOutside = 0x80000000u;
    const float *base = a.in + (size_t)img0 * a.C * a.H * a.W;
    const size_t behind = (size_t)(a.total / a.npix - img0) * a.C * plane;
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)(behind < 0x7ffffffcu ? behind : 0x7ffffffcu), 0x00020000);
    // where this lane's staged elements come from (the same for every chunk)
    unsigned src[kItems];
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        const int item = wave + kWaves * i, g = CG == 16 && item >= per_half, q = (item - (g ? per_half : 0)) * 64 + lane;
        const int vr = (int)fast_div((unsigned)q, a.d_wp), c = q - vr * a.Wp - a.pw;
        const int v = v0 + vr, img = (int)fast_div((unsigned)v, a.d_hv), r = v - img * a.Hv - a.ph;
        const bool in = q < staged && r >= 0 && r < a.H && c >= 0 && c < a.W;
        src[i] = in ? (unsigned)((((img - img0) * a.C + 8 * g) * a.H + r) * a.W + c) * 4u : kOutside;
    }
    // and this lane's operands: the LDS byte address of its pixel's first tap
    int at[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        int img, c;
        const int v = split_virtual_row(a, min(n0 + (ntile0 + i) * 32 + col, a.total - 1), img, c);
        at[i] = ((CG == 16 ? half * P : 0) + (v - v0) * a.Wp + c * a.sw) * 16;
    }

    // sum: of the chunks before this one, whose own is acc; with missing values tm, the present -w (t'^2 + m / s^2), and lg
    constexpr bool TWO = !MASKED && NI <= 2;   // the two products' chunk sums apart: room for them
    f32x16 sum[NI], acc[NI], ac2[TWO ? NI : 1], tm[MASKED ? NI : 1], lg[MASKED ? NI : 1];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        sum[i] = 0.0f;
        acc[i] = 0.0f;
        if (TWO)
            ac2[i] = 0.0f;
        if (MASKED) {
            tm[i] = 0.0f;
            lg[i] = 0.0f;
        }
    }
    const bool active = mtile < a.n_mtiles;
    const int taps_h = a.taps / a.bw;
    const f16x8 *pp = (const f16x8 *)a.packed + (size_t)(active ? mtile : 0) * a.chunks * a.steps * NA * 64;
    f16x8 next[NA];   // the packed parameters of the next step
#pragma unroll
    for (int q = 0; q < NA; ++q)
        next[q] = pp[q * 64 + lane];

    float x[kItems][8];
    // a chunk's values of this lane's pixels (patches of 64 elements at least: eight channels or fewer come in chunks of eight, so
    // that a group's start has a channel)
    auto request = [&](int chunk) {
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            const int item = wave + kWaves * i;
            if (item >= kHalves * per_half)
                continue;
            const int g = CG == 16 && item >= per_half, there = a.C - 1 - (chunk * CG + 8 * g);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                x[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                    rsrc, src[i], (chunk * CG + max(-8 * g, min(j, there))) * plane, 0));
        }
    };
    int level = 0;
    // (sizes as a float's bits) the largest |x'| s so far, what is larger than it, and than the level keeps, among staged values
    int seen = __float_as_int(kSplitSeen), ask = seen, limit = __float_as_int(kSplitMost);
    const float *channels = a.chan;
    auto buffer = [&](int chunk) { return lds + (WIDE && (chunk & 1) ? split_lds_bytes(KIND) : 0); };
    auto stage = [&](int chunk) {   // converts the requested values; returns the largest staged |x'| of this lane's
        float most = 0.0f;
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            const int item = wave + kWaves * i;
            if (item >= kHalves * per_half)
                continue;
            const int g = CG == 16 && item >= per_half, q = (item - (g ? per_half : 0)) * 64 + lane;
            const int c0 = chunk * CG + 8 * g;
            uniform_float *chan = (uniform_float *)(channels + c0);
            if (a.oob != 0.0f)   // (a NaN too)
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    x[i][j] = src[i] == kOutside ? a.oob : x[i][j];
            if (c0 + 8 > a.C)    // channels behind the last have zero parameters: any finite value will do
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    x[i][j] = c0 + j < a.C ? x[i][j] : 0.0f;
            f16x8 v[5];
            float item_most = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float s = chan[SPLIT_S * a.chunks * CG + j], ncs = chan[SPLIT_NCS * a.chunks * CG + j];
                float d = __builtin_fmaf(x[i][j], s, ncs);
                float d2 = __builtin_fmaf(d, d, -chan[SPLIT_M * a.chunks * CG + j]);
                if (MASKED) {
                    const bool ok = x[i][j] == x[i][j];
                    d = ok ? d : 0.0f;
                    d2 = ok ? d2 : 0.0f;
                    v[4][j] = ok ? (_Float16)1.0f : (_Float16)0.0f;
                }
                item_most = fmaxf(item_most, __builtin_fabsf(d));
                _Float16 hi, lo;
                split2(d2, hi, lo);
                v[0][j] = hi; v[1][j] = lo;
                split2(d, hi, lo);
                v[2][j] = hi; v[3][j] = lo;
            }
            if (q < staged) {
                most = fmaxf(most, item_most);
                char *dst = buffer(chunk) + (g * P + q) * 16;
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    *reinterpret_cast<f16x8 *>(dst + b * kPlane) = v[b];
            }
        }
        return __float_as_int(most);
    };
    auto stage_and_tell = [&](int chunk) {
        // Both blocks out of the ordinary: code that is not in the instruction cache takes a microsecond or two to get.
        const int most = stage(chunk);
        if (most > ask)
            split_far_most(far.most[chunk & 1], most < __float_as_int(INFINITY) ? ldexpf(__int_as_float(most), kSplitLevelBits * level) : 0.0f);
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(most > limit) != 0, 0))
            for (int i = level; i < kLastLevel; ++i) {
                const float keeps = ldexpf(kSplitMost / 32, kSplitLevelBits * (i - level));
                const int lanes = __popcll(__builtin_amdgcn_ballot_w64(__int_as_float(most) > keeps));
                if (lane == 0)
                    __hip_atomic_fetch_add(&far.lanes[chunk % 3][i], lanes, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
    };
    request(0);
    if (WIDE)
        stage_and_tell(0);
    for (int chunk = 0; chunk < a.chunks; ++chunk) {
        __syncthreads();
        if (!WIDE) {
            stage_and_tell(chunk);
            __syncthreads();
        }
        seen = max(seen, __builtin_amdgcn_readfirstlane(far.most[chunk & 1]));
        ask = seen;
        if (__builtin_expect(seen > __float_as_int(kSplitMost), 0)) {
            int next_level = level;
            while (next_level < kLastLevel && __int_as_float(seen) > ldexpf(kSplitMost, kSplitLevelBits * next_level) &&
                   (next_level == 0 || __builtin_amdgcn_readfirstlane(far.lanes[chunk % 3][next_level]) > 64 * WAVES / 8))
                ++next_level;
            if (next_level > level) {
                const float ratio = ldexpf(1.0f, 2 * kSplitLevelBits * (level - next_level));
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    sum[i] *= ratio;
                    acc[i] *= ratio;
                    if (TWO)
                        ac2[i] *= ratio;
                }
                level = next_level;
                limit = __float_as_int(level < kLastLevel ? kSplitMost : INFINITY);
                channels = a.chan + level * SPLIT_CHANNEL_FIELDS * a.chunks * CG;
                stage(chunk);
                __syncthreads();
            }
            ask = __float_as_int(ldexpf(__int_as_float(seen), -kSplitLevelBits * level));
            if (tid < kSplitLevels - 1)
                far.lanes[(chunk + 2) % 3][tid] = 0;
        }
        // Products go in front of the conversions of the unit's other waves, which wait for memory more than for their turn: 62.7 ->
        // 60.6 us with eight waves, 32 x 128 x 28 x 28 -> 128, 3 x 3; missing values, 64 x 64 x 32 x 32 -> 128, 105.3 -> 103.3, 64 x 128 x 28 x
        // 28 -> 128, 1 x 1, 59.7 -> 57.7.  (The other forms: no difference.)
        if (WIDE || MASKED)
            __builtin_amdgcn_s_setprio(1);
        int dh = 0, dw = 0;
        auto next_tap = [&]() {   // LDS offset of the next tap (behind the last: of the first, with zero parameters)
            const int off = dh < taps_h ? (dh * a.Wp + dw) * 16 : 0;
            if (++dw == a.bw) {
                dw = 0;
                ++dh;
            }
            return off;
        };
        auto next_offset = [&]() {   // of a step's operands
            const int off = next_tap();
            if (CG == 16)
                return off;
            const int off2 = next_tap();
            return half ? off2 : off;
        };
        const char *staged_here = buffer(chunk);
        auto fetch = [&](f16x8 &to, int from, int b) { to = *reinterpret_cast<const f16x8 *>(staged_here + from + b * kPlane); };
        auto mul = [](f32x16 &to, const f16x8 &p, const f16x8 &v) {
            to = __builtin_amdgcn_mfma_f32_32x32x16_f16(p, v, to, 0, 0, 0);
        };
        const f16x8 low = (_Float16)(1.0f / kSplitLow);
        f16x8 A[NA];
        auto advance = [&](int step) {   // this step's parameters from those ahead, and the request of the next ones
#pragma unroll
            for (int q = 0; q < NA; ++q)
                A[q] = next[q];
            if (__builtin_expect(level > 0, 0)) {
                const f16x8 shrink = (_Float16)ldexpf(1.0f, -kSplitLevelBits * level);
                A[2] *= shrink;
                A[3] *= shrink;
                if (MASKED)   // (the lesser piece of what tm sums is added to the squares)
                    A[NA - 3] *= shrink * shrink;
            }
            if (chunk + 1 < a.chunks || step + 1 < a.steps)
                pp += NA * 64;
#pragma unroll
            for (int q = 0; q < NA; ++q)
                next[q] = pp[q * 64 + lane];
            if (step == (WIDE ? max(0, a.steps - 2) : a.steps - 1) && chunk + 1 < a.chunks)
                request(chunk + 1);
        };
        int off = next_offset();
        if (!active) {
            if (chunk + 1 < a.chunks)
                request(chunk + 1);
        } else if constexpr (NI == 4) {
            // An accumulator's products follow one another at 48 cycles, two accumulators' in turn at 32: two pixel tiles at
            // a time, their squares while their cross terms' operands are requested, then the other way round.
            f16x8 Bq[2][2], Be[2][2];
            auto fetch_pair = [&](f16x8 (&to)[2][2], int pair, int from, int b) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    fetch(to[i][1], at[2 * pair + i] + from, b + 1);
                    fetch(to[i][0], at[2 * pair + i] + from, b);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            auto products = [&](int pair, const f16x8 &hi, const f16x8 &lo, const f16x8 (&b)[2][2]) {
                const f16x8 lower = hi * low;
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    mul(acc[2 * pair + i], lower, b[i][1]);
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    mul(acc[2 * pair + i], lo, b[i][0]);
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    mul(acc[2 * pair + i], hi, b[i][0]);
                __builtin_amdgcn_sched_barrier(0);
            };
            fetch_pair(Bq, 0, off, 0);
            for (int step = 0; step < a.steps; ++step) {
                advance(step);
                const int off_next = next_offset();
#pragma unroll
                for (int pair = 0; pair < 2; ++pair) {
                    fetch_pair(Be, pair, off, 2);
                    products(pair, A[0], A[1], Bq);
                    fetch_pair(Bq, 1 - pair, pair == 0 ? off : off_next, 0);
                    products(pair, A[2], A[3], Be);
                }
                off = off_next;
            }
        } else {
            constexpr int kAhead = MASKED ? 0 : 1;   // (missing values: no registers left for it)
            f16x8 B[1 + kAhead][NB];
            auto fetch_all = [&](f16x8 (&to)[NB], int from) {
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    fetch(to[b], from, b);
            };
            if (kAhead)
                fetch_all(B[0], at[0] + off);
            for (int step = 0; step < a.steps; ++step) {
                advance(step);
                const int off_next = next_offset();
                const f16x8 A0 = A[0] * low, A2 = A[2] * low;
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    if (kAhead) {
                        fetch_all(B[(i + 1) & kAhead], i + 1 < NI ? at[(i + 1) % NI] + off : at[0] + off_next);
                        __builtin_amdgcn_sched_barrier(0);
                    } else
                        fetch_all(B[0], at[i] + off);
                    const f16x8 (&b)[NB] = B[i & kAhead];
                    f32x16 &cross = TWO ? ac2[TWO ? i : 0] : acc[i];
                    mul(acc[i], A0, b[1]);
                    if (MASKED)
                        mul(lg[MASKED ? i : 0], A[NA - 1], b[NB - 1]);
                    mul(cross, A2, b[3]);
                    if (MASKED)
                        mul(tm[MASKED ? i : 0], A[NA - 4], b[NB - 1]);
                    mul(acc[i], A[1], b[0]);
                    if (MASKED)
                        mul(lg[MASKED ? i : 0], A[NA - 2], b[NB - 1]);
                    mul(cross, A[3], b[2]);
                    if (MASKED)   // (the lesser piece of what tm sums, where small sums are kept)
                        mul(acc[i], A[NA - 3], b[NB - 1]);
                    mul(acc[i], A[0], b[0]);
                    mul(cross, A[2], b[2]);
                    if (kAhead)
                        __builtin_amdgcn_sched_barrier(0);
                }
                if (kAhead && (NI & 1))
#pragma unroll
                    for (int b = 0; b < NB; ++b)
                        B[0][b] = B[kAhead][b];
                off = off_next;
            }
        }
        if (WIDE || MASKED)
            __builtin_amdgcn_s_setprio(0);
        // a sum of its own for every so many products: see the head of the file
        if ((chunk + 1) % a.per_sum == 0 || chunk + 1 == a.chunks)
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                sum[i] += TWO ? acc[i] + ac2[TWO ? i : 0] : acc[i];
                acc[i] = 0.0f;
                if (TWO)
                    ac2[i] = 0.0f;
            }
        if (WIDE && chunk + 1 < a.chunks)
            stage_and_tell(chunk + 1);
    }

    // lane: pixel col of each tile, templates 8 (r / 4) + 4 half + r % 4
    if (!active)
        return;
    const f32x4 *rows4 = reinterpret_cast<const f32x4 *>(a.rows) + mtile * kSplitRows + 4 * half;
    const float *lgs = a.rows + (size_t)4 * a.n_mtiles * kSplitRows + mtile * kSplitRows + 4 * half;
    f32x4 row[16];
    float lgm[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        row[r] = rows4[8 * (r / 4) + r % 4];
        lgm[r] = !MASKED && norm ? lgs[8 * (r / 4) + r % 4] : 0.0f;
    }
    const float grow = ldexpf(1.0f, 2 * kSplitLevelBits * level);
    if (__builtin_expect(seen > __float_as_int(kSplitSeen), 0)) {   // the guard's line rises with the staged values: see split_pack_block
        const float2 *more = reinterpret_cast<const float2 *>(a.rows + (size_t)5 * a.n_mtiles * kSplitRows) + mtile * kSplitRows + 4 * half;
        // (what is beyond 2^8 of the level's leaves its outputs NaN)
        const float largest = fminf(__int_as_float(seen), ldexpf(256.0f, kSplitLevelBits * level)), square = largest * largest;
        const float scaled = MASKED && level > 0 ? kSplitParamShare * sqrtf((float)a.K) * grow : 0.0f;   // (the scaled lesser pieces)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float2 by = more[8 * (r / 4) + r % 4];
            row[r][SPLIT_THR] = fmaxf(fmaxf(row[r][SPLIT_THR], by.x * grow), fmaxf(by.y * square, row[r][SPLIT_UNSCALE] * scaled));
            if (!MASKED)
                row[r][SPLIT_UNSCALE] *= grow;
        }
    }
    // stores by a pixel's offset and a row's; rows behind the last template go outside of the buffer
    const int left = a.O - mtile * kSplitRows;
    const unsigned image = (unsigned)a.npix * 4u;
    float *tile = a.out + ((size_t)img0 * a.O + mtile * kSplitRows) * a.npix;
    const size_t room = ((size_t)(a.total / a.npix - img0) * a.O - mtile * kSplitRows) * image;
    const __amdgpu_buffer_rsrc_t to =
        __builtin_amdgcn_make_buffer_rsrc((void *)tile, 0, (int)(room < 0x7ffffffcu ? room : 0x7ffffffcu), 0x00020000);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int n = n0 + (ntile0 + i) * 32 + col;
        const int img = (int)fast_div((unsigned)n, a.d_npix);
        const unsigned pixel = n < a.total ? ((unsigned)((img - img0) * a.O + 4 * half) * a.npix + (n - img * a.npix)) * 4u : kOutside;
        unsigned flagged = 0;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int ml = 8 * (r / 4) + r % 4;
            float v;
            bool fine;
            if (MASKED) {
                v = __builtin_fmaf(sum[i][r], grow, tm[i][r]) * row[r][SPLIT_UNSCALE];
                const float mag = __builtin_fabsf(v);
                fine = mag < 1e37f && mag >= row[r][SPLIT_GUARD] * -(tm[i][r] * row[r][SPLIT_UNSCALE]) &&
                       (mag >= row[r][SPLIT_THR] || (v == 0.0f && tm[i][r] == 0.0f && row[r][SPLIT_THR] < 1e37f));
                v = __builtin_fmaf(0.5f, v, lg[i][r] * (1.0f / kSplitLogScale));
            } else {
                v = __builtin_fmaf(sum[i][r], row[r][SPLIT_UNSCALE], row[r][SPLIT_BIAS]) + row[r][SPLIT_BIAS_LESSER];
                const float mag = __builtin_fabsf(v);
                fine = mag >= row[r][SPLIT_THR] && mag < 1e37f;
                if (norm)
                    v = __builtin_fmaf(0.5f, v, lgm[r]);
            }
            flagged |= fine ? 0u : 1u << r;
            unsigned at = pixel;
            if (left < kSplitRows)
                at = ml + 4 * half < left ? at : kOutside;
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), to, at, ml * image, 0);
        }
        if (left < kSplitRows)   // of the rows that are templates
#pragma unroll
            for (int r = 0; r < 16; ++r)
                flagged &= 8 * (r / 4) + r % 4 + 4 * half < left ? ~0u : ~(1u << r);
        near[i] = n < a.total ? flagged : 0u;
    }
}

// What a forward workgroup does around its body: body(far, near).
template <int KIND, int CG, int WAVES, class Body>
__device__ __forceinline__ void split_forward(const SplitArgs &a, char *lds, int ptile, int mtile0, int g, int norm, Body &&body)
{
    __shared__ int any_near;   // of the workgroup's outputs, one below the guard's line
    __shared__ SplitFar far;
    if (threadIdx.x == 0)
        any_near = 0;
    if (threadIdx.x < 2)
        far.most[threadIdx.x] = __float_as_int(kSplitSeen);
    if (threadIdx.x < kSplitLevels - 1)
        far.lanes[0][threadIdx.x] = far.lanes[1][threadIdx.x] = far.lanes[2][threadIdx.x] = 0;
    if (WAVES == 8)   // (its first chunk is staged, and told of, in front of the first barrier)
        __syncthreads();
    u32x4 near = 0;   // [i] bit r: output r of this lane's pixel tile i is
    body(*(__attribute__((address_space(3))) SplitFar *)&far, near);
    if (near[0] | near[1] | near[2] | near[3])
        any_near = 1;
    __syncthreads();
    // (unlikely: the code behind everything else; between the bodies it costs 37 x 45 x 29 x 35 -> 75 4 us of 62)
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(any_near), 0)) {
        if (KIND == SPLIT_MASKED || norm)
            split_recompute<KIND, CG, true, WAVES>((lds_char *)lds, ptile, mtile0, g, near);
        else
            split_recompute<KIND, CG, KIND == SPLIT_MASKED, WAVES>((lds_char *)lds, ptile, mtile0, g, near);
    } else if ((int)threadIdx.x < g && mtile0 + (int)threadIdx.x < a.n_mtiles)
        a.flags[(size_t)ptile * a.n_mtiles + mtile0 + threadIdx.x] = 0;
}
#endif

// Consecutive workgroups go to the eight XCDs in turn: a run of neighbouring pixel tiles, which share rows, to each.
__device__ __forceinline__ int split_ptile()
{
    const int run = gridDim.x / 8, x = blockIdx.x;
    return x < run * 8 ? x % 8 * run + x / 8 : x;
}

// The template tiles of a pixel tile are dealt out as groups of gmax and, of the rest, 2 and 1 (forward, of four: the rest
// as one).  flag: forward, the normalized mode; input gradient, NaN inputs ignored.
template <int KIND, int CG>
__global__ __launch_bounds__(kThreads, 2) void sim_split_kernel(const SplitArgs a, int flag)
{
#if defined(__HIP_DEVICE_COMPILE__)
    __shared__ __align__(16) char split_lds[split_lds_bytes(KIND)];
    const int full = a.n_mtiles / a.gmax, y = blockIdx.y;
    int mtile0 = y * a.gmax, g = a.gmax;
    if (y >= full) {
        const int rest = a.n_mtiles - full * a.gmax;   // 1..3
        mtile0 = full * a.gmax;
        g = rest == 3 && KIND == SPLIT_FWD ? 4 : rest >= 2 ? 2 : 1;
        if (y > full) {   // the last one of three
            mtile0 += 2;
            g = 1;
        }
    }
    const int ptile = split_ptile();
    if constexpr (KIND == SPLIT_GRAD) {
        if (g == 2)
            split_grad_body<CG, 2, 4>(a, split_lds, ptile, mtile0, flag);
        else
            split_grad_body<CG, 1, 4>(a, split_lds, ptile, mtile0, flag);
    } else
        split_forward<KIND, CG, 4>(a, split_lds, ptile, mtile0, g, flag, [&](auto &far, u32x4 &near) __attribute__((always_inline)) {
            if (KIND == SPLIT_FWD && g == 4)
                split_body<KIND, CG, KIND == SPLIT_FWD ? 4 : 2, 4>(a, split_lds, far, near, ptile, mtile0, flag);
            else if (g == 2)
                split_body<KIND, CG, 2, 4>(a, split_lds, far, near, ptile, mtile0, flag);
            else
                split_body<KIND, CG, 1, 4>(a, split_lds, far, near, ptile, mtile0, flag);
        });
#endif
}

// Forward without missing values, G template tiles, four or two, to a workgroup of eight waves.
template <int CG, int G>
__global__ __launch_bounds__(2 * kThreads, 2) void sim_split_forward_wide_kernel(const SplitArgs a, int flag)
{
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int KIND = SPLIT_FWD;
    __shared__ __align__(16) char split_lds[2 * split_lds_bytes(KIND)];
    const int ptile = split_ptile(), mtile0 = blockIdx.y * G;
    split_forward<KIND, CG, 8>(a, split_lds, ptile, mtile0, G, flag, [&](auto &far, u32x4 &near) __attribute__((always_inline)) {
        split_body<KIND, CG, G, 8>(a, split_lds, far, near, ptile, mtile0, flag);
    });
#endif
}

// Input gradient, G template tiles, four or two, to a workgroup of eight waves.
template <int CG, int G>
__global__ __launch_bounds__(2 * kThreads, 2) void sim_split_grad_wide_kernel(const SplitArgs a, int flag)
{
#if defined(__HIP_DEVICE_COMPILE__)
    __shared__ __align__(16) char split_lds[2 * split_lds_bytes(SPLIT_GRAD)];
    split_grad_body<CG, G, 8>(a, split_lds, split_ptile(), blockIdx.y * G, flag);
#endif
}

// The sum of a channel's sampled template elements, and their mean.
__device__ __forceinline__ float split_grad_centre_part(const SplitPack &a, int c)
{
    const SplitSample s = split_sample(a, c);
    return (s.there[0] ? s.t[0] : 0.0f) + (s.there[1] ? s.t[1] : 0.0f);
}

__device__ __forceinline__ float split_grad_centre(const SplitPack &a, float part)
{
    part = split_sample_sum(part) / (float)min(32, a.O * a.taps);
    return __builtin_fabsf(part) < 1e18f ? part : 0.0f;
}

// Packs the input gradient's coefficients, rows = input channels, contraction = (template, flipped tap): three pieces
// each of s w (t - c) and s w.  Same blocks as split_pack_block.
__global__ __launch_bounds__(kThreads) void sim_split_grad_pack_kernel(const SplitPack a, float scale)
{
    __shared__ float centre[kSplitRows];
    const int tid = threadIdx.x, parts = (a.steps + 3) / 4;
    const int mtile = blockIdx.x / (a.chunks * parts), rest = blockIdx.x - mtile * a.chunks * parts;
    const int chunk = rest / parts, part = rest - chunk * parts;
    // this lane's elements first: they arrive while the centres are formed (7.6 -> 4.9 us, 128 channels, 128 templates, 3 x 3)
    const int step = 4 * part + (tid >> 6);
    const int lane = tid & 63, half = lane >> 5, row = lane & 31, c = mtile * kSplitRows + row;
    const int tap = a.cg == 16 ? step : 2 * step + half;
    float t[8], w[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {   // (any value outside)
        const int o = chunk * a.cg + (a.cg == 16 ? 8 * half : 0) + j;
        const size_t at = ((size_t)min(o, a.O - 1) * a.C + min(c, a.C - 1)) * a.taps + (a.taps - 1 - min(tap, a.taps - 1));
        t[j] = a.templates[at];
        w[j] = a.weights[at];
    }
    float sum[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
        sum[i] = split_grad_centre_part(a, mtile * kSplitRows + 16 * i + (tid >> 4));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float centred = split_grad_centre(a, sum[i]);
        if ((tid & 15) == 0) {
            centre[16 * i + (tid >> 4)] = centred;
            if (chunk == 0 && part == 0)
                a.ctr[mtile * kSplitRows + 16 * i + (tid >> 4)] = centred;
        }
    }
    __syncthreads();
    if (step >= a.steps)
        return;
    const float middle = centre[row];
    bf16x8 v[6];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int o = chunk * a.cg + (a.cg == 16 ? 8 * half : 0) + j;
        const bool there = c < a.C && o < a.O && tap < a.taps;
        const float ws = there ? scale * w[j] : 0.0f, td = there ? t[j] - middle : 0.0f;
        __bf16 p0, p1, p2;
        split3_any(ws * td, p0, p1, p2);
        v[0][j] = p0; v[1][j] = p1; v[2][j] = p2;
        split3_any(ws, p0, p1, p2);
        v[3][j] = p0; v[4][j] = p1; v[5][j] = p2;
    }
    bf16x8 *dst = reinterpret_cast<bf16x8 *>(a.packed) +
                  (((size_t)mtile * a.chunks + chunk) * a.steps + step) * a.pieces * 64 + lane;
#pragma unroll
    for (int q = 0; q < 6; ++q)
        dst[q * 64] = v[q];
}

}  // namespace

// The guard's line as a share of sum w t'^2: where this form's error (see the head of the file) is that of the sum it
// stands for, term by term or with square roots of the weights.  Its last roundings weigh more in a short sum.
static float split_line(int K) { return K < 128 ? 0.5f : 0.43f; }

// Chunks, tiles and workspace of the contraction that `p` describes, with `kind`'s operands; .on if it fits and is worth
// while.
static SplitPlan split_geometry(const SimPlan &p, int kind)
{
    SplitPlan s = {};
    const int taps = p.bh * p.bw;
    const long long total = 1LL * p.B * p.oh * p.ow;
    if (p.C > kSplitMaxC || 1LL * p.B * p.C * p.H * p.W >= (1LL << 31) || total >= (1LL << 30) ||
        1LL * p.B * ((p.oh - 1) * p.sh + p.bh) >= (1LL << 30))
        return s;
    // a workgroup addresses the images it touches by 31 bits
    const long long touched = (kSplitPixels - 1) / (1LL * p.oh * p.ow) + 2;
    if (kind != SPLIT_GRAD && 4 * touched * std::max(1LL * p.C * p.H * p.W, 1LL * p.O * p.oh * p.ow) >= (1LL << 31))
        return s;
    s.Wp = (p.ow - 1) * p.sw + p.bw;
    s.Hv = (p.oh - 1) * p.sh + p.bh;
    // the most rows of the stack that 128 consecutive pixels touch
    int g = p.ow, h = kSplitPixels;
    while (h) {
        const int r = g % h;
        g = h;
        h = r;
    }
    const int out_rows = (p.ow - g + kSplitPixels - 1) / p.ow + 1;
    const int crossings = 1LL * p.oh * p.ow % kSplitPixels == 0 ? 0 : (out_rows - 1 + p.oh - 1) / p.oh;
    const long long staged = 1LL * ((out_rows - 1) * p.sh + p.bh + crossings * std::max(0, p.bh - p.sh)) * s.Wp;
    const int room = split_lds_pixels(kind);
    const int c16 = (p.C + 15) / 16 * taps, c8 = (p.C + 7) / 8 * ((taps + 1) / 2);   // matrix steps
    if (staged > 2 * room)
        return s;
    s.cg = staged > room || (c8 < c16 && 8 * c8 < 7 * c16) ? 8 : 16;
    s.chunks = (p.C + s.cg - 1) / s.cg;
    s.steps = s.cg == 16 ? taps : (taps + 1) / 2;
    s.pieces = split_pieces(kind);
    s.n_mtiles = (p.O + kSplitRows - 1) / kSplitRows;
    s.n_ptiles = (int)((total + kSplitPixels - 1) / kSplitPixels);
    const double useful = 1.0 * total * p.O * p.K;
    const double padded = 1.0 * s.n_ptiles * kSplitPixels * s.n_mtiles * kSplitRows * s.chunks * s.steps * 16;
    // few of the products useful (64 x 17 x 28 x 28 -> 33, 0.33 of them: still 48 -> 35 us; 32 x 3 x 64 x 64 -> 64, 5 x 5, 0.36
    // in a single chunk: 50 -> 53), or a handful of workgroups: no gain over the vector forms
    if (useful < (s.chunks > 1 ? 0.3 : 0.4) * padded || 1LL * s.n_ptiles * s.n_mtiles < 32)
        return s;
    const int mpad = s.n_mtiles * kSplitRows;
    s.packed = 0;
    s.chan = s.packed + (size_t)s.n_mtiles * s.chunks * s.steps * s.pieces * 1024;
    s.rows = s.chan + align_up((size_t)std::max(kSplitLevels * SPLIT_CHANNEL_FIELDS * s.chunks * s.cg, mpad) * sizeof(float), 256);
    s.flags = s.rows + align_up((size_t)7 * mpad * sizeof(float), 256);
    s.exact = s.flags + align_up((size_t)s.n_ptiles * s.n_mtiles * sizeof(int), 256);
    s.logs = s.exact + (kind == SPLIT_GRAD ? 0 : align_up((size_t)p.O * p.K * sizeof(float2), 256));
    s.total = s.logs + (kind == SPLIT_GRAD || p.mode == SIM_MODE_L2 ? 0 : align_up((size_t)p.O * p.K * sizeof(float), 256));
    s.on = true;
    return s;
}

SplitPlan sim_split_plan(const SimPlan &p)
{
    // few elements per patch: outputs below the guard's line are ordinary there
    if (!p.split || p.mode == SIM_MODE_L1 || (p.mode == SIM_MODE_L2_NORM && p.norm_const_every_iteration) ||
        p.B == 0 || p.K < 64)
        return SplitPlan();
    return split_geometry(p, p.mode == SIM_MODE_L2_NORM_IGNORE_NAN ? SPLIT_MASKED : SPLIT_FWD);
}

static float split_norm_const(int K) { return (float)((double)(-0.5f * (float)K) * std::log(2.0 * M_PI)); }

SplitPack sim_split_pack_args(const SimPlan &p, const SplitPlan &sp, const float *templates, const float *weights,
                              char *ws)
{
    SplitPack a;
    a.templates = templates; a.weights = weights;
    a.packed = reinterpret_cast<unsigned short *>(ws + sp.packed);
    a.chan = a.ctr = reinterpret_cast<float *>(ws + sp.chan);
    a.rows = reinterpret_cast<float *>(ws + sp.rows);
    a.exact = reinterpret_cast<float2 *>(ws + sp.exact);
    a.logs = reinterpret_cast<float *>(ws + sp.logs);
    a.O = p.O; a.C = p.C; a.taps = p.bh * p.bw; a.K = p.K; a.cg = sp.cg; a.chunks = sp.chunks; a.steps = sp.steps;
    a.pieces = sp.pieces; a.n_mtiles = sp.n_mtiles; a.mode = p.mode; a.fudge = p.fudge;
    a.line = split_line(p.K);
    a.d_taps = make_fast_div((unsigned)a.taps);
    a.d_K = make_fast_div((unsigned)a.K);
    a.d_steps = make_fast_div((unsigned)std::max(1, sp.steps));
    a.norm_const = p.mode == SIM_MODE_L2_NORM ? split_norm_const(p.K) : 0.0f;
    a.pack_blocks = sp.on ? sp.chunks * sp.n_mtiles * ((sp.steps + 3) / 4) : 0;
    a.blocks = sp.on ? std::min(sp.n_mtiles * kSplitRows, 512) : 0;
    return a;
}

// Workgroups that are more than half and at most one to a compute unit: eight waves take four template tiles then, or two where
// four leave fewer, instead of half as many tiles to four waves, two workgroups to a unit, which stage the same pixels twice.
static bool split_wide_round(long long groups) { return groups > 128 && groups <= 256; }

// Workgroups of eight waves and four template tiles, one to a compute unit, instead of four waves and two, two to a unit: 0.93 of
// the time of a chip that either kind fills.  A compute unit that gets a single one of the lesser takes 0.55.  All template
// tiles in fours (96 channels, the last of three tiles' two waves idle: 32 x 96 x 28 x 28 -> 128 76 -> 81 us), and 31 bits for
// the images of a tile.  Measured, 128 channels, 28 x 28 -> 128, 3 x 3, by the number of tiles (us, before and after):
// 135 97 -> 83, 172 97 -> 84, 196 93 -> 82, 252 100 -> 92, 392 176 -> 162, 503 189 -> 178; 258 148 -> 159, 343 149 -> 162, left to the others.
// 1 x 1, 196: 29 -> 22; 5 x 5, 196: 216 -> 204.
// Two tiles of rows, instead of one to four waves: 64 channels, 32 images -> 50, 32.3 -> 29.1; 128 channels, 20 images, 59 -> 55, 12 55 ->
// 51; 48 x 14 x 14, 192 templates, 72 -> 70; not in chunks of eight channels (5 x 5, 64 -> 64: 62.6 -> 63.6).
static int split_grad_wide(const SimPlan &p, const SplitPlan &s)
{
    const long long touched = (kSplitPixels - 1) / (1LL * p.oh * p.ow) + 2;
    if (4 * touched * p.C * p.H * p.W >= (1LL << 31))
        return 0;
    const long long groups = 1LL * s.n_ptiles * (s.n_mtiles / 4), full = groups / 256, rest = groups % 256;
    if (s.n_mtiles % 4 == 0 && 0.93 * (full + (rest != 0)) < full + (rest == 0 ? 0.0 : rest <= 128 ? 0.55 : 1.0))
        return 4;
    return s.cg == 16 && s.n_mtiles % 2 == 0 && split_wide_round(1LL * s.n_ptiles * (s.n_mtiles / 2)) ? 2 : 0;
}

// The forward's: where the workgroups of four waves and two template tiles are more than one and at most two to a compute
// unit.  Fewer leave compute units to share; more run as four tiles to four waves, two workgroups to a unit, which is the faster
// form of a full chip (256 x 64 x 32 x 32 -> 128, 3 x 3: 219 us, this form 267).  Measured, 128 channels, 28 x 28 -> 128, 3 x 3, by the
// number of tiles (us, before and after): 135 64 -> 58, 196 68 -> 62, 252 72 -> 67; 1 x 1, 196: 28 -> 23; 5 x 5, 196: 143 -> 143;
// two tiles to a workgroup, 64 templates 51.6 -> 46.0, 1 x 1 24 -> 21, 128 templates, 20 images, 52 -> 46, 12 images 48 -> 43;
// three tiles of 75 templates, 30 x 45 x 29 x 35, 238: 32 -> 28.  With missing values no gain (22 x 128 x 28 x 28: 95 -> 95; 64 x 64 x 32 x
// 32: 103 -> 107).
static int split_forward_wide(const SplitPlan &s)
{
    if ((s.n_mtiles % 4 == 0 || s.n_mtiles % 4 == 3) && split_wide_round(1LL * s.n_ptiles * ((s.n_mtiles + 3) / 4)))
        return 4;
    return s.n_mtiles % 2 == 0 && split_wide_round(1LL * s.n_ptiles * (s.n_mtiles / 2)) ? 2 : 0;
}

template <int KIND>
static int split_launch(const SimPlan &p, const SplitPlan &sp, const float *input, float *output, char *ws, int flag,
                        hipStream_t s, SplitArgs a = {})
{
    a.in = input; a.out = output;
    a.packed = ws + sp.packed;
    a.chan = a.ctr = reinterpret_cast<const float *>(ws + sp.chan);
    a.rows = reinterpret_cast<const float *>(ws + sp.rows);
    a.flags = reinterpret_cast<int *>(ws + sp.flags);
    a.exact = reinterpret_cast<const float2 *>(ws + sp.exact);
    a.logs = reinterpret_cast<const float *>(ws + sp.logs);
    a.norm_const = p.mode == SIM_MODE_L2_NORM ? split_norm_const(p.K) : 0.0f;
    a.K = p.K;
    a.C = p.C; a.H = p.H; a.W = p.W; a.O = p.O; a.ow = p.ow; a.npix = p.oh * p.ow; a.total = p.B * a.npix;
    a.bw = p.bw; a.sh = p.sh; a.sw = p.sw; a.ph = p.ph; a.pw = p.pw; a.taps = p.bh * p.bw;
    a.chunks = sp.chunks; a.steps = sp.steps; a.n_mtiles = sp.n_mtiles; a.Wp = sp.Wp; a.Hv = sp.Hv;
    a.oob = p.oob;
    a.per_sum = std::max(1, 2 / sp.steps);
    a.d_npix = make_fast_div((unsigned)a.npix);
    a.d_ow = make_fast_div((unsigned)p.ow);
    a.d_wp = make_fast_div((unsigned)sp.Wp);
    a.d_hv = make_fast_div((unsigned)sp.Hv);
    a.d_taps = make_fast_div((unsigned)a.taps);
    a.d_bw = make_fast_div((unsigned)p.bw);
    const int wide = KIND == SPLIT_FWD ? split_forward_wide(sp) : KIND == SPLIT_GRAD ? split_grad_wide(p, sp) : 0;
    if (wide) {
        const dim3 grid((unsigned)sp.n_ptiles, (unsigned)((sp.n_mtiles + wide - 1) / wide));
        void (*const kernels[2][2][2])(SplitArgs, int) = {
            {{sim_split_forward_wide_kernel<8, 2>, sim_split_forward_wide_kernel<8, 4>},
             {sim_split_forward_wide_kernel<16, 2>, sim_split_forward_wide_kernel<16, 4>}},
            {{nullptr /* see split_grad_wide */, sim_split_grad_wide_kernel<8, 4>},
             {sim_split_grad_wide_kernel<16, 2>, sim_split_grad_wide_kernel<16, 4>}}};
        hipLaunchKernelGGL(kernels[KIND == SPLIT_GRAD][sp.cg == 16][wide == 4], grid, dim3(2 * kThreads), 0, s, a, flag);
        return hipGetLastError() == hipSuccess ? SIMNETS_OK : SIMNETS_ERR_HIP;
    }
    // as many template tiles per staged pixel tile as leave a workgroup for every compute unit
    a.gmax = KIND == SPLIT_FWD ? 4 : 2;
    while (a.gmax > 1 && (a.gmax / 2 >= sp.n_mtiles || (long long)sp.n_ptiles * ((sp.n_mtiles + a.gmax - 1) / a.gmax) < 256))
        a.gmax /= 2;
    const int rest = sp.n_mtiles % a.gmax;
    const dim3 grid((unsigned)sp.n_ptiles, (unsigned)(sp.n_mtiles / a.gmax + (rest == 0 ? 0 : rest == 3 && KIND != SPLIT_FWD ? 2 : 1)));
    if (sp.cg == 16)
        hipLaunchKernelGGL((sim_split_kernel<KIND, 16>), grid, dim3(kThreads), 0, s, a, flag);
    else
        hipLaunchKernelGGL((sim_split_kernel<KIND, 8>), grid, dim3(kThreads), 0, s, a, flag);
    return hipGetLastError() == hipSuccess ? SIMNETS_OK : SIMNETS_ERR_HIP;
}

int sim_split_launch(const SimPlan &p, const SplitPlan &sp, const float *input, float *output, char *ws, hipStream_t s)
{
    if (p.mode == SIM_MODE_L2_NORM_IGNORE_NAN)
        return split_launch<SPLIT_MASKED>(p, sp, input, output, ws, 0, s);
    return split_launch<SPLIT_FWD>(p, sp, input, output, ws, p.mode == SIM_MODE_L2_NORM, s);
}

// ------------------------------------------------------------------------------------------------
// Input gradient of the L2 modes at stride 1:  dX = A - (X - c) B,  A = sum g s w (t - c),  B = sum g s w  over (template,
// tap) - the forward's contraction with g as the image (its channels are the templates, the taps flipped) and the input
// channels as rows, g in three pieces against the three of each coefficient: eight bits each, but with the exponents of fp32,
// which g and the weights use (gradients of one template, or of one pixel, may be many orders below others').  32 x 128 x 28 x 28, 128 templates, 3 x 3: 196 us
// on the fp32 matrix instructions -> 93 us, 82 with workgroups of eight waves (split_grad_wide), error against 64 bits 6.0e-7 -> 2.0e-7 of the gradient's 2-norm.  Small grids
// keep that kernel (sim_mfma_kernel), which splits the contraction over workgroups.
// ------------------------------------------------------------------------------------------------
static SimPlan grad_as_forward(const SimPlan &p)
{
    SimPlan q = p;
    q.C = p.O; q.O = p.C; q.H = p.oh; q.W = p.ow; q.oh = p.H; q.ow = p.W;
    q.ph = p.bh - 1 - p.ph; q.pw = p.bw - 1 - p.pw;
    q.K = q.C * p.bh * p.bw;
    q.oob = 0.0f;
    return q;
}

static SplitPlan split_grad_plan(const SimPlan &p)
{
    if (!p.split || p.mode == SIM_MODE_L1 || p.B == 0 || p.sh != 1 || p.sw != 1 || p.ph > p.bh - 1 || p.pw > p.bw - 1)
        return SplitPlan();
    const SimPlan q = grad_as_forward(p);
    const SplitPlan s = split_geometry(q, SPLIT_GRAD);
    // Fewer tiles than fill the chip twice: a workgroup walks the whole contraction, 1.6 us to stage a chunk and 0.49 a step,
    // where the fp32 form splits it over workgroups and takes some 45 us + 1 per tap + 38 per 10^9 terms.  Short
    // contractions are the faster ones here (8 x 128 x 16 x 16, 128 templates, 3 x 3, 64 tiles: 53 us, fp32 form 62; 64 templates 30
    // and 58; 8 x 64 x 28 x 28, 64, 5 x 5, 59 and 98), long ones there (1 x 32 x 64 x 64, 256 templates, 32 tiles: 98 and 57; 4 x 256 x
    // 14 x 14, 256: 106 and 76; 6 x 64 x 28 x 28, 1024, 1 x 1: 138 and 55); 6 x 128 x 32 x 32, 256, 192 tiles: 100 and 95.
    const double here = 6 + s.chunks * (1.6 + 0.49 * s.steps), there = 45 + p.bh * p.bw + 38e-9 * p.B * p.H * p.W * p.C * q.K;
    return s.on && 1LL * s.n_ptiles * s.n_mtiles < 512 && here > there ? SplitPlan() : s;
}

size_t sim_split_grad_input_workspace_bytes(const SimPlan &p)
{
    const SplitPlan s = split_grad_plan(p);
    return s.on ? s.total : 0;
}

int sim_split_grad_input_launch(const SimPlan &p, const float *input, const float *templates, const float *weights,
                                const float *output_grad, float *input_grad, void *workspace, size_t workspace_bytes,
                                void *stream)
{
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const SimPlan q = grad_as_forward(p);
    const SplitPlan sp = split_grad_plan(p);
    if (workspace_bytes < sp.total)
        return SIMNETS_ERR_WORKSPACE;
    char *ws = reinterpret_cast<char *>(workspace);
    SplitPack a = sim_split_pack_args(q, sp, templates, weights, ws);
    a.O = p.O; a.C = p.C;   // of the templates' layout
    SplitArgs g = {};
    g.x = input; g.templates = templates; g.weights = weights;
    g.scale = p.mode != SIM_MODE_L2 ? 1.0f : 2.0f;   // the normalized functor halves the plain one
    hipLaunchKernelGGL(sim_split_grad_pack_kernel, dim3(a.pack_blocks), dim3(kThreads), 0, s, a, g.scale);
    if (hipGetLastError() != hipSuccess)
        return SIMNETS_ERR_HIP;
    return split_launch<SPLIT_GRAD>(q, sp, output_grad, input_grad, ws, p.mode == SIM_MODE_L2_NORM_IGNORE_NAN, s, g);
}

}  // namespace simnets
