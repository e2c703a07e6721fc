// MEX backward (gfx950): gradients w.r.t. the input and w.r.t. the offsets.
//
// Replaces MEXGradInputKernelGPU / MEXGradOffsetsKernelGPU (src/kernels/mex_grad_kernel_gpu.cu), i.e.
// per image im2col_3d_gpu + split_patches + ggemm_readc_gpu with mex_backward_bottom_finite /
// _infinite (include/utils/mex_utils.hpp:31-46) + reverse split_patches + col2im_3d_gpu (input) or
// the accumulation over images (offsets), by one launch over the whole batch each.
//
// Both gradients are sums of the same term
//   e(px, m, k) = g[px,m] * exp(eps * (patch(px)[k] + off[r(px),m,k] - out[px,m]) + ey)        finite eps
//               = g[px,m] * (patch(px)[k] + off[r(px),m,k] == out[px,m])                        eps = +-inf
//   d patch(px)[k]  = sum_m e(px, m, k)          (then stored to the input element the patch element is; patches
//                                                 that overlap are added per element by mex_col2im_kernel)
//   d off[r, m, k]  = sum_{px in region r} e(px, m, k)
// Output pixels are enumerated region-major exactly like the forward kernel does, a lane owns
// pixel slots, so the offsets a wave needs are the same for all its lanes (scalar loads).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "fast_div.h"
#include "internal.h"
#include "mex_common.h"
#include "valu_tile.h"

namespace simnets {

namespace {

struct MexGradArgs {
    MexKernelArgs k;       // geometry; k.in = input, k.out unused
    const float *off;      // [R][M][K] offsets as the forward op used them
    const float *out;      // forward output
    const float *g;        // output gradient
    int gpool;             // g is the gradient of the 2 x 2 sum-pooled output, [B][M][H/2][W/2]: the gradient of output
                           // pixel (h, w) is its window's, g[h / 2][w / 2]
    float *dx;             // input gradient
    float *partial;        // offsets gradient partial sums [chunk][R][M][K]
    int overlap;           // patches overlap: the per-patch gradients go to `col`, mex_col2im_kernel adds them up
    float *col;            // [B][K][Co*Ho*Wo] gradient of every patch element (overlapping patches only): lanes hold
                           // consecutive output pixels both where it is written and where it is added up
    int cpr;               // pixel chunks per region
    int msplit;            // input gradient: the instances are split over gridDim.z workgroups (1: no split) ...
    int mg_per_split;      // ... of this many packed groups (GM_TM instances) each, which write their partial
    float *dx_splits;      // gradients to [split][input] for mex_sum_splits_kernel
    // Factor buffers (finite epsilon, optional): the pixel factors W [R][slots_pad][Mp] and the patch exponentials
    // EX [R][slots_pad][Kp] of mex_grad_factors_kernel, which the matrix kernels then load instead of forming them
    // (again and again: once per tile of the other dimension).  nullptr: the kernels form them themselves.
    float *wbuf, *exbuf;
    int slots_pad, Mp, Kp;
    int pxl;               // pixel slots per lane (offsets gradient)
};

// Output gradient given as the gradient of the 2 x 2 sum-pooled output (ga.gpool; one output channel per instance,
// even height and width): plane size and the offset of output pixel `out_off`'s window.
__device__ __forceinline__ size_t pooled_g_plane(const MexGradArgs &ga, size_t plane)
{
    return ga.gpool ? plane >> 2 : plane;
}

__device__ __forceinline__ int pooled_g_offset(const MexGradArgs &ga, int out_off)
{
    if (!ga.gpool)
        return out_off;
    const int h = out_off / ga.k.Wo, w = out_off - h * ga.k.Wo;
    return (h >> 1) * (ga.k.Wo >> 1) + (w >> 1);
}

// patch element k of the pixel -> value (im2col_3d rule) and, if inside the image, its offset from the
// image start; -1 otherwise
__device__ __forceinline__ float patch_element(const MexKernelArgs &a, const PixelRef &px, int k, ptrdiff_t *img_off)
{
    const int bhw = a.bh * a.bw;
    const int dc = k / bhw;
    const int rem = k - dc * bhw;
    const int dh = rem / a.bw;
    const int dw = rem - dh * a.bw;
    const int ci = px.ci0 + dc, hi = px.hi0 + dh, wi = px.wi0 + dw;
    const bool ok = mex_inside(a, ci, hi, wi);
    const ptrdiff_t o = ((ptrdiff_t)ci * a.H + hi) * a.W + wi;
    *img_off = ok ? o : -1;
    // (the load on an address that is always valid, the choice afterwards: loads inside conditions are waited for one
    // by one)
    const float v = a.in[(size_t)px.b * a.C * a.H * a.W + (ok ? o : 0)];
    return ok ? v : a.oob;
}

__device__ __forceinline__ float mex_term(float x_plus_off, float out, float g, float c1, float c0, bool finite)
{
    if (finite)
        return g * __builtin_amdgcn_exp2f(__builtin_fmaf(x_plus_off - out, c1, c0));
    return x_plus_off == out ? g : 0.0f;
}

constexpr int GX_KT = 8;   // patch elements per lane (input gradient)

// One wave: the 64 pixel slots of (region r, chunk) x GX_KT patch elements from k0, term by term.
__device__ __forceinline__ void mex_grad_input_wave(const MexGradArgs &ga, int r, int chunk, int k0, int lane,
                                                    int m_begin, int m_end, float *dx)
{
    const MexKernelArgs &a = ga.k;
    const PixelRef px = locate(a, r, chunk * 64 + lane);
    const bool valid = px.out_off >= 0;

    float xk[GX_KT], acc[GX_KT];
    ptrdiff_t io[GX_KT];
#pragma unroll
    for (int j = 0; j < GX_KT; ++j) {
        acc[j] = 0.0f;
        io[j] = -1;
        xk[j] = 0.0f;
        if (k0 + j < a.K)
            xk[j] = patch_element(a, px, k0 + j, &io[j]);
    }
    const size_t plane = (size_t)a.Co * a.Ho * a.Wo;
    const size_t gplane = pooled_g_plane(ga, plane);
    const float *gp = ga.g + (size_t)px.b * a.M * gplane + (valid ? pooled_g_offset(ga, px.out_off) : 0);
    const float *op = ga.out + (size_t)px.b * a.M * plane + (valid ? px.out_off : 0);
    const float SIMNETS_CONST_AS *off = (const float SIMNETS_CONST_AS *)(ga.off) + (size_t)r * a.M * a.K + k0;
    const bool finite = a.finite_eps != 0;
    // four instances at a time: their gradient and output values requested together (the additions keep their order)
    for (int m4 = m_begin; m4 < m_end; m4 += 4) {
        float gv[4], ov[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int mc = min(m4 + u, m_end - 1);
            gv[u] = gp[(size_t)mc * gplane];
            ov[u] = op[(size_t)mc * plane];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int m = m4 + u;
            if (m < m_end) {
                const float g = valid ? gv[u] : 0.0f;
#pragma unroll
                for (int j = 0; j < GX_KT; ++j) {
                    const float of = (k0 + j < a.K) ? off[(size_t)m * a.K + j] : 0.0f;
                    acc[j] += mex_term(xk[j] + of, ov[u], g, a.c1, a.c0, finite);
                }
            }
        }
    }
    if (!valid)
        return;
    float *dimg = dx + (size_t)px.b * a.C * a.H * a.W;
    float *dcol = ga.col + ((size_t)px.b * a.K + k0) * plane + px.out_off;
#pragma unroll
    for (int j = 0; j < GX_KT; ++j) {
        if (io[j] < 0)
            continue;
        if (ga.overlap)
            dcol[j * plane] = acc[j];
        else
            dimg[io[j]] = acc[j];
    }
}

// grid.x: (region, pixel chunk of 64 slots); grid.y: tile of 4*GX_KT patch elements (one GX_KT per wave)
__global__ __launch_bounds__(256) void mex_grad_input_kernel(const MexGradArgs ga)
{
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = blockIdx.x / ga.cpr;
    const int chunk = blockIdx.x - r * ga.cpr;
    const int k0 = (blockIdx.y * 4 + wave) * GX_KT;
    if (k0 < ga.k.K)
        mex_grad_input_wave(ga, r, chunk, k0, lane, 0, ga.k.M, ga.dx);
}

// Finite epsilon, product form on the fp32 matrix cores.  In the scaled domain (xs = c1 x, os = c1 off, outs = c1 out,
// c1 = eps log2 e) a term is g 2^(xs_k + os_mk - outs_m + c0), and outs_m - c0 = log2 sum_k 2^(xs_k + os_mk) bounds every
// xs_k + os_mk from above.  With lo_m = min_k os_mk and a = min_m (outs_m - c0 - lo_m) >= every xs_k of the pixel:
//   term = 2^(xs_k - a) * 2^(os_mk - mo_m) * [ g_m 2^(a + mo_m - outs_m + c0) ],
// all three factors at most 2^(range of the instance's offsets), and for the terms that matter (near 1) at least
// 2^-range: d patch_k = 2^(xs_k - a) * sum_m W_m EO_mk is a GEMM over the instances (v_mfma_f32_16x16x4_f32 tiles:
// 16 patch elements x 16 pixels x 4 instances) of the pixel factors W (computed from g and out, which the kernel
// reads anyway: no pass over the patches is needed for the bound) with the packed offset exponentials EO of the
// forward pass.  Used when every instance of the region has an offsets range of at most kGradProductRange; otherwise the
// workgroup falls back to the term-by-term waves.
// grid.x: (region, pixel chunk of 64 slots); grid.y: tile of GM_KT patch elements (16 per wave)
constexpr int GM_TM = kGradPackTm;   // (32) instances per packed group = contraction chunk
// Widest offsets range (an exponent of two) the gradients' product form takes on the loose bound a (below).  Its factors
// 2^(xs - a), 2^(os - mo) and W then carry exponents of up to the range, each rounded once: an error of ulp(range) in an
// exponent is a relative error of about 4e-8 * range in the factor - two to four times the error of the reference's own
// fp32 arithmetic on the same data.  Measured against the fp64 oracle the gradients stay within the 1e-4 bar up to
// ranges of about 50 (at most 8e-5 at 48, 1.15e-4 at 64, 1.2e-4 at 77 on the tests' data; the reference's fp32 arithmetic:
// 1.5 ... 3e-5); the forward pass's 90 is a bound against overflow, not this one.  Beyond it the gathering kernels take
// a region term by term (about 12 times slower); the row-wise kernels switch to a tight bound (kGradRowsRange).
constexpr float kGradProductRange = 48.0f;
// Row-wise kernels: widest patch range of a pixel (exponents of two) for which a region with large offsets ranges
// keeps the product form on the pixel's own maximum as the bound (the factors' exponents stay within this range)
constexpr float kGradPixelRange = 64.0f;
// ... and the widest offsets range such a region may have.  With the tight bound the factors' errors follow the size of
// the offsets themselves, as the reference's own do, at 1.5 to 4 times its error; what an element of the gradient sees
// of it depends on how far its terms cancel: 4e-5 ... 7e-5 at 77 and 1.5e-4 at 88 on the tests' seeded layers, but
// 1.1e-4 at a range of 55 on another (a sum of 4.8 in absolute terms that cancels to 0.08; error 2e-6 of the terms).  The
// same limit as the gathering kernels' keeps such elements rare; beyond it a region goes term by term.
constexpr float kGradRowsRange = 48.0f;
constexpr float kLooseBoundRange = 24.0f;  // offsets ranges (exponents of two) up to which a few instances give the bound
constexpr int GM_KT = 64;
typedef float floatx4 __attribute__((ext_vector_type(4)));

// Pixel factors and patch exponentials of the product form, once per pixel: for the 64 pixel slots of
// (region, chunk) the bound a, W_m = g_m 2^(a + mo_m - outs_m + c0) for every instance and 2^(xs_k - a) for every
// patch element, written as rows [slot][Mp] and [slot][Kp] (through LDS, so that the stores run along the rows);
// a workgroup forms one block of 32 instances or 32 patch elements (grid.y), each from the same bound.
// Regions with an offsets range beyond kGradProductRange are left alone: the matrix kernels fall back to the
// term-by-term waves there and never look at the buffers.
__global__ __launch_bounds__(256) void mex_grad_factors_kernel(const MexGradArgs ga)
{
    const MexKernelArgs &a = ga.k;
    __shared__ float tile[32 * 65];   // [instance or patch element][pixel], padded rows
    __shared__ float pmn[4 * 64];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = blockIdx.x / ga.cpr;
    const int chunk = blockIdx.x - r * ga.cpr;
    const int n_mg = a.n_mgroups;
    const float *omax_r = a.omax + (size_t)r * n_mg * GM_TM, *orng_r = a.orng + (size_t)r * n_mg * GM_TM;
    int wide = 0, big = 0;
    for (int m = tid; m < a.M; m += 256) {
        wide |= !(orng_r[m] <= kGradProductRange);
        big |= !(orng_r[m] <= kLooseBoundRange);
    }
    const int roomy = __syncthreads_or(big);
    if (__syncthreads_or(wide))
        return;
    const PixelRef px = locate(a, r, chunk * 64 + lane);
    const bool valid = px.out_off >= 0;
    const size_t plane = (size_t)a.Co * a.Ho * a.Wo, gplane = pooled_g_plane(ga, plane);
    const float *gp = ga.g + (size_t)px.b * a.M * gplane + (valid ? pooled_g_offset(ga, px.out_off) : 0);
    const float *op = ga.out + (size_t)px.b * a.M * plane + (valid ? px.out_off : 0);
    const int m_scan = roomy ? a.M : min(a.M, 4);   // see mex_grad_input_mfma_kernel
    float amin = INFINITY;
#pragma unroll 4
    for (int m = wave; m < m_scan; m += 4)   // (unrolled: four loads in flight instead of one)
        amin = fminf(amin, __builtin_fmaf(op[(size_t)m * plane], a.c1, -(a.c0 + (omax_r[m] - orng_r[m]))));
    pmn[wave * 64 + lane] = amin;
    __syncthreads();
    const float a_p = valid ? fminf(fminf(pmn[lane], pmn[64 + lane]), fminf(pmn[128 + lane], pmn[192 + lane])) : 0.0f;
    // (below, all loads of a block go out first, those past the last instance or patch element on a clamped
    // address: a load inside the condition would be waited for before the next one is issued)
    // rows of this chunk; thread (column c, pixels pr, pr + 8, ...) writes the tile out
    const size_t row0 = (size_t)r * ga.slots_pad + (size_t)chunk * 64;
    const int c = tid & 31, pr = tid >> 5;
    // grid.y: one block of 32 columns per workgroup - the instance groups first, then the patch-element blocks
    if ((int)blockIdx.y < n_mg) {
        const int mg = blockIdx.y;
        float ovv[GM_TM / 4], gvv[GM_TM / 4], omv[GM_TM / 4];
#pragma unroll
        for (int i = 0; i < GM_TM / 4; ++i) {
            const int mc = min(mg * GM_TM + wave + 4 * i, a.M - 1);
            ovv[i] = op[(size_t)mc * plane];
            gvv[i] = gp[(size_t)mc * gplane];
            omv[i] = omax_r[mc];
        }
#pragma unroll
        for (int i = 0; i < GM_TM / 4; ++i) {
            const int mm = wave + 4 * i, m = mg * GM_TM + mm;
            float w = 0.0f;
            if (valid && m < a.M) {
                const float e = __builtin_fmaf(-ovv[i], a.c1, a_p) + (omv[i] + a.c0);
                w = gvv[i] * __builtin_amdgcn_exp2f(e);
            }
            tile[mm * 65 + lane] = w;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; ++j)
            ga.wbuf[(row0 + pr + 8 * j) * ga.Mp + mg * GM_TM + c] = tile[c * 65 + pr + 8 * j];
    } else {
        const int kb = ((int)blockIdx.y - n_mg) * 32;
        int4 ke[8];  // wave-uniform: {offset inside an image, dc, dh, dw}
#pragma unroll
        for (int i = 0; i < 8; ++i)
            ke[i] = a.ktab[min(kb + wave + 4 * i, a.K - 1)];
        float xg[8];
        unsigned inside = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int ci = px.ci0 + ke[i].y, hi = px.hi0 + ke[i].z, wi = px.wi0 + ke[i].w;
            const bool ok = mex_inside(a, ci, hi, wi);
            inside |= ok ? 1u << i : 0u;
            const float *src = ok ? px.base + ke[i].x : a.in;
            xg[i] = *src;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int kk = wave + 4 * i, k = kb + kk;
            float e = 0.0f;
            if (valid && k < a.K) {
                const float x = (inside >> i) & 1u ? xg[i] : a.oob;
                e = __builtin_amdgcn_exp2f(__builtin_fmaf(x, a.c1, -a_p));
            }
            tile[kk * 65 + lane] = e;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; ++j)
            ga.exbuf[(row0 + pr + 8 * j) * ga.Kp + kb + c] = tile[c * 65 + pr + 8 * j];
    }
}

__global__ __launch_bounds__(256) void mex_grad_input_mfma_kernel(const MexGradArgs ga)
{
    const MexKernelArgs &a = ga.k;
    __shared__ float eo[GM_KT * (GM_TM + 1)];   // [k][instance], padded rows
    __shared__ float wt[GM_TM * 65];            // [instance][pixel], padded rows
    __shared__ float pmn[4 * 64], ap[64];
    __shared__ int pb[64], pc0[64], ph0[64], pw0[64];   // pixel table: image (-1: empty slot), patch origin
    __shared__ int pout[64];                            // ... and the pixel's offset within the image's output
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = blockIdx.x / ga.cpr;
    const int chunk = blockIdx.x - r * ga.cpr;
    const int k0 = blockIdx.y * GM_KT;
    const int n_mg = a.n_mgroups;
    // this workgroup's share of the instances (all of them unless the launch splits them over gridDim.z) and where
    // its gradients go
    const int mg_begin = blockIdx.z * ga.mg_per_split, mg_end = min(n_mg, mg_begin + ga.mg_per_split);
    float *dxo = ga.msplit > 1 ? ga.dx_splits + (size_t)blockIdx.z * a.B * a.C * a.H * a.W : ga.dx;
    const float *omax_r = a.omax + (size_t)r * n_mg * GM_TM, *orng_r = a.orng + (size_t)r * n_mg * GM_TM;
    // (everything the product form reads first is requested before the barriers that decide on it: the pixel, its
    // table entries, the first output value of the bound, the patch element records of this lane's gradients)
    const int lr = lane & 15, lq = lane >> 4;
    int4 kel[4];
#pragma unroll
    for (int v = 0; v < 4; ++v)
        kel[v] = a.ktab[min(k0 + wave * 16 + 4 * lq + v, a.K - 1)];
    const PixelRef px = locate(a, r, chunk * 64 + lane);
    const bool valid = px.out_off >= 0;
    if (wave == 0) {
        pb[lane] = valid ? px.b : -1;
        pc0[lane] = px.ci0; ph0[lane] = px.hi0; pw0[lane] = px.wi0;
        pout[lane] = px.out_off;
    }
    const size_t plane = (size_t)a.Co * a.Ho * a.Wo, gplane = pooled_g_plane(ga, plane);
    const float *gp = ga.g + (size_t)px.b * a.M * gplane + (valid ? pooled_g_offset(ga, px.out_off) : 0);
    const float *op = ga.out + (size_t)px.b * a.M * plane + (valid ? px.out_off : 0);
    const float o_first = op[(size_t)min(wave, a.M - 1) * plane];
    const float lo_first = omax_r[min(wave, a.M - 1)] - orng_r[min(wave, a.M - 1)];
    int roomy;  // some instance's offsets range is large enough for the choice of the bound to matter (below)
    {
        int wide = 0, big = 0;
        for (int m = tid; m < a.M; m += 256) {
            wide |= !(orng_r[m] <= kGradProductRange);
            big |= !(orng_r[m] <= kLooseBoundRange);
        }
        roomy = __syncthreads_or(big);
        if (__syncthreads_or(wide)) {
#pragma unroll
            for (int h = 0; h < GM_KT / (4 * GX_KT); ++h) {
                const int kk0 = k0 + (wave * (GM_KT / (4 * GX_KT)) + h) * GX_KT;
                if (kk0 < a.K)
                    mex_grad_input_wave(ga, r, chunk, kk0, lane, min(a.M, mg_begin * GM_TM), min(a.M, mg_end * GM_TM),
                                        dxo);
            }
            return;
        }
    }
    const bool buffered = ga.wbuf != nullptr;   // W and 2^(xs - a) come from mex_grad_factors_kernel
    const size_t row0 = (size_t)r * ga.slots_pad + (size_t)chunk * 64;
    // the pixel's bound a = min_m (outs_m - c0 - lo_m).  Every single term of the minimum is a valid bound
    // (>= every xs_k); with the minimum over all instances the exponent of W_m stays below the instance's own
    // offsets range, with the minimum over a few it stays below that range + the range of those few + log2 K.
    // While no range exceeds kLooseBoundRange that is far from overflow, and the first four instances (one
    // strided load per thread instead of M / 4) do.
    const int m_scan = buffered ? 0 : (roomy ? a.M : min(a.M, 4));
    float amin = INFINITY;
    for (int m = wave; m < m_scan; m += 4)
        amin = fminf(amin, m == wave ? __builtin_fmaf(o_first, a.c1, -(a.c0 + lo_first))
                                     : __builtin_fmaf(op[(size_t)m * plane], a.c1, -(a.c0 + (omax_r[m] - orng_r[m]))));
    pmn[wave * 64 + lane] = amin;
    __syncthreads();
    if (wave == 0)
        ap[lane] = valid ? fminf(fminf(pmn[lane], pmn[64 + lane]), fminf(pmn[128 + lane], pmn[192 + lane])) : 0.0f;
    __syncthreads();
    const float a_p = ap[lane];

    // where this lane's 16 gradients go (the pixel tables are in place behind the barriers above) and the input
    // values their factors 2^(xs_k - a) are made of: requested here, used after the matrix loop (a load in front of
    // each store made the lane wait for 16 memory round trips in turn, 45 % of the kernel on a 64 x 32 x 16 x 16 -> 64
    // layer)
    const size_t chw = (size_t)a.C * a.H * a.W;
    size_t at[4][4];
    float xin[4][4];
    bool ok[4][4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int k = k0 + wave * 16 + 4 * lq + v;
        const int dc = kel[v].y, dh = kel[v].z, dw = kel[v].w;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int p = t * 16 + lr;
            const int b = pb[p];
            const int ci = pc0[p] + dc, hi = ph0[p] + dh, wi = pw0[p] + dw;
            ok[v][t] = (k < a.K) & (b >= 0) & mex_inside(a, ci, hi, wi);
            at[v][t] = ok[v][t] ? (size_t)b * chw + ((size_t)ci * a.H + hi) * a.W + wi : 0;
            if (buffered)
                xin[v][t] = ga.exbuf[ok[v][t] ? (row0 + p) * ga.Kp + k : 0];
            else
                xin[v][t] = a.in[at[v][t]];
        }
    }

    floatx4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
        acc[t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    // operands of an instance group: the offsets tile (two float4 per thread) and, unless the pixel factors come from
    // the buffers, this thread's eight output and gradient values - requested a group ahead
    constexpr int EO4 = GM_KT * (GM_TM / 4) / 256;
    float4 eo_n[EO4];
    float ov_n[GM_TM / 4], gv_n[GM_TM / 4], om_n[GM_TM / 4];
    auto request = [&](int mg) {
        const float4 *src = reinterpret_cast<const float4 *>(a.offe + (((size_t)r * n_mg + mg) * a.K + k0) * GM_TM);
#pragma unroll
        for (int j = 0; j < EO4; ++j) {
            const int i = tid + j * 256;
            eo_n[j] = k0 + i / (GM_TM / 4) < a.K ? src[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        if (!buffered) {
#pragma unroll
            for (int i = 0; i < GM_TM / 4; ++i) {
                const int m = min(mg * GM_TM + wave + 4 * i, a.M - 1);
                ov_n[i] = op[(size_t)m * plane];
                gv_n[i] = gp[(size_t)m * gplane];
                om_n[i] = omax_r[m];
            }
        }
    };
    if (mg_begin < mg_end)
        request(mg_begin);
    for (int mg = mg_begin; mg < mg_end; ++mg) {
        __syncthreads();  // the previous chunk's matrix instructions are done with eo / wt
#pragma unroll
        for (int j = 0; j < EO4; ++j) {
            const int i = tid + j * 256;
            const int row = i / (GM_TM / 4), c4 = i % (GM_TM / 4);
            const float4 v = eo_n[j];
            float *d = eo + row * (GM_TM + 1) + 4 * c4;
            d[0] = v.x; d[1] = v.y; d[2] = v.z; d[3] = v.w;
        }
        if (buffered) {
            // rows of 32 instances: thread (instance c, pixels pr, pr + 8, ...)
            const int c = tid & 31, pr = tid >> 5;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                wt[c * 65 + pr + 8 * j] = ga.wbuf[(row0 + pr + 8 * j) * ga.Mp + mg * GM_TM + c];
        } else {
#pragma unroll
            for (int i = 0; i < GM_TM / 4; ++i) {
                const int mm = wave + 4 * i, m = mg * GM_TM + mm;
                float w = 0.0f;
                if (valid && m < a.M) {
                    // (a - outs) first: a small, once-rounded difference; the instance constant is added to that
                    const float e = __builtin_fmaf(-ov_n[i], a.c1, a_p) + (om_n[i] + a.c0);
                    w = gv_n[i] * __builtin_amdgcn_exp2f(e);
                }
                wt[mm * 65 + lane] = w;
            }
        }
        if (mg + 1 < mg_end)
            request(mg + 1);   // in flight during the matrix steps
        __syncthreads();
#pragma unroll
        for (int ms = 0; ms < GM_TM; ms += 4) {
            const float av = eo[(wave * 16 + lr) * (GM_TM + 1) + ms + lq];
#pragma unroll
            for (int t = 0; t < 4; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, wt[(ms + lq) * 65 + t * 16 + lr], acc[t], 0, 0, 0);
        }
    }
    // ---- d patch_k = 2^(xs_k - a) * acc, scattered to the input element the patch element is ----
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int k = k0 + wave * 16 + 4 * lq + v;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (!ok[v][t])
                continue;
            const int p = t * 16 + lr;
            const float val = acc[t][v] * (buffered ? xin[v][t]
                                                    : __builtin_amdgcn_exp2f(__builtin_fmaf(xin[v][t], a.c1, -ap[p])));
            if (ga.overlap)
                ga.col[((size_t)pb[p] * a.K + k) * plane + pout[p]] = val;
            else
                dxo[at[v][t]] = val;
        }
    }
}

// Instances split over several workgroups: input gradient = sum of their partial gradients, in split order.
__global__ __launch_bounds__(256) void mex_sum_splits_kernel(const float *__restrict__ parts, long long n, int splits,
                                                            float *__restrict__ dx)
{
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        float s = parts[i];
        for (int z = 1; z < splits; ++z)
            s += parts[(size_t)z * n + i];
        dx[i] = s;
    }
}

// ... four elements per thread with all the splits' loads (at most 8) in flight together: n a multiple of 4, 16-byte
// aligned pointers.  The same additions in the same order.
__device__ __forceinline__ void sum_splits4(const float4 *__restrict__ parts, long long n4, int splits, float4 *__restrict__ dx,
                                            long long i)
{
    if (i >= n4)
        return;
    float4 v[8];
#pragma unroll
    for (int z = 0; z < 8; ++z)
        v[z] = parts[(size_t)min(z, splits - 1) * n4 + i];
    float4 s = v[0];
#pragma unroll
    for (int z = 1; z < 8; ++z)
        if (z < splits) {
            s.x += v[z].x; s.y += v[z].y; s.z += v[z].z; s.w += v[z].w;
        }
    dx[i] = s;
}

__global__ __launch_bounds__(256) void mex_sum_splits4_kernel(const float4 *__restrict__ parts, long long n4, int splits,
                                                             float4 *__restrict__ dx)
{
    sum_splits4(parts, n4, splits, dx, (long long)blockIdx.x * 256 + threadIdx.x);
}

void launch_sum_splits(const float *parts, long long n, int splits, float *dx, hipStream_t s)
{
    if (splits <= 8 && n % 4 == 0 && reinterpret_cast<uintptr_t>(parts) % 16 == 0 &&
        reinterpret_cast<uintptr_t>(dx) % 16 == 0 && (n / 4 + 255) / 256 <= 0x7fffffffLL)
        hipLaunchKernelGGL(mex_sum_splits4_kernel, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, s,
                           reinterpret_cast<const float4 *>(parts), n / 4, splits, reinterpret_cast<float4 *>(dx));
    else
        hipLaunchKernelGGL(mex_sum_splits_kernel, dim3((unsigned)std::min<long long>((n + 255) / 256, 65535)), dim3(256),
                           0, s, parts, n, splits, dx);
}

// Overlapping patches: input gradient = sum, over the patches that cover the element, of the patch-element
// gradients in `col` (the reference's col2im_3d, src/utils/im2col.cpp:297-328), patches in ascending (c, h, w)
// order.  One thread per input element; elements no patch covers get 0.
__global__ __launch_bounds__(256) void mex_col2im_kernel(const MexKernelArgs a, const float *__restrict__ col,
                                                         float *__restrict__ dx, long long n)
{
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= n)
        return;
    const int w = (int)(idx % a.W);
    long long q = idx / a.W;
    const int h = (int)(q % a.H); q /= a.H;
    const int c = (int)(q % a.C);
    const long long b = q / a.C;
    // patches o along an axis that cover coordinate x: 0 <= x + pad - o * stride < block
    auto first = [](int x, int pad, int block, int stride) {
        const int lo = x + pad - block + 1;
        return lo <= 0 ? 0 : (lo + stride - 1) / stride;
    };
    const int co_lo = first(c, a.pc, a.bc, a.sc), co_hi = min(a.Co - 1, (c + a.pc) / a.sc);
    const int ho_lo = first(h, a.ph, a.bh, a.sh), ho_hi = min(a.Ho - 1, (h + a.ph) / a.sh);
    const int wo_lo = first(w, a.pw, a.bw, a.sw), wo_hi = min(a.Wo - 1, (w + a.pw) / a.sw);
    const size_t plane = (size_t)a.Co * a.Ho * a.Wo;
    const float *cb = col + (size_t)b * plane * a.K;
    float acc = 0.0f;
    for (int co = co_lo; co <= co_hi; ++co) {
        const int dc = c + a.pc - co * a.sc;
        for (int ho = ho_lo; ho <= ho_hi; ++ho) {
            const int dh = h + a.ph - ho * a.sh;
            for (int wo = wo_lo; wo <= wo_hi; ++wo) {
                const int dw = w + a.pw - wo * a.sw;
                acc += cb[((dc * a.bh + dh) * a.bw + dw) * plane + ((size_t)co * a.Ho + ho) * a.Wo + wo];
            }
        }
    }
    dx[idx] = acc;
}

constexpr int GO_MT = 4, GO_KT = 8;  // instances x patch elements per lane (offsets gradient)

// One wave: GO_MT instances from m0 x GO_KT patch elements from k0 over the 64*pxl pixel slots of (region r,
// chunk), term by term; writes its partial sums.
__device__ __forceinline__ void mex_grad_offsets_wave(const MexGradArgs &ga, int r, int chunk, int m0, int k0, int lane)
{
    const MexKernelArgs &a = ga.k;

    float acc[GO_MT][GO_KT];
#pragma unroll
    for (int i = 0; i < GO_MT; ++i)
#pragma unroll
        for (int j = 0; j < GO_KT; ++j)
            acc[i][j] = 0.0f;
    // the offsets of this wave's tile are the same for every pixel
    float of[GO_MT][GO_KT];
    const float SIMNETS_CONST_AS *off = (const float SIMNETS_CONST_AS *)(ga.off) + (size_t)r * a.M * a.K;
#pragma unroll
    for (int i = 0; i < GO_MT; ++i)
#pragma unroll
        for (int j = 0; j < GO_KT; ++j)
            of[i][j] = (m0 + i < a.M && k0 + j < a.K) ? to_vgpr(off[(size_t)(m0 + i) * a.K + k0 + j]) : 0.0f;

    const size_t plane = (size_t)a.Co * a.Ho * a.Wo;
    const bool finite = a.finite_eps != 0;
    for (int s = 0; s < ga.pxl; ++s) {
        const PixelRef px = locate(a, r, (chunk * ga.pxl + s) * 64 + lane);
        const bool valid = px.out_off >= 0;
        float xk[GO_KT];
#pragma unroll
        for (int j = 0; j < GO_KT; ++j) {
            ptrdiff_t unused;
            xk[j] = (k0 + j < a.K) ? patch_element(a, px, k0 + j, &unused) : 0.0f;
        }
        const size_t gplane = pooled_g_plane(ga, plane);
        const float *gp = ga.g + (size_t)px.b * a.M * gplane + (valid ? pooled_g_offset(ga, px.out_off) : 0);
        const float *op = ga.out + (size_t)px.b * a.M * plane + (valid ? px.out_off : 0);
        float gv[GO_MT], ov[GO_MT];
#pragma unroll
        for (int i = 0; i < GO_MT; ++i) {   // (all requests first, on clamped rows)
            const int mc = min(m0 + i, a.M - 1);
            gv[i] = gp[(size_t)mc * gplane];
            ov[i] = op[(size_t)mc * plane];
        }
#pragma unroll
        for (int i = 0; i < GO_MT; ++i) {
            const bool mok = valid && m0 + i < a.M;
            const float g = mok ? gv[i] : 0.0f;
            const float o = mok ? ov[i] : 0.0f;
#pragma unroll
            for (int j = 0; j < GO_KT; ++j) {
                const float e = mex_term(xk[j] + of[i][j], o, g, a.c1, a.c0, finite);
                acc[i][j] += mok ? e : 0.0f;
            }
        }
    }
    // sum over the 64 lanes; lane 0 holds the result
#pragma unroll
    for (int i = 0; i < GO_MT; ++i)
#pragma unroll
        for (int j = 0; j < GO_KT; ++j) {
            float v = acc[i][j];
            for (int d = 32; d > 0; d >>= 1)
                v += __shfl_xor(v, d, 64);
            acc[i][j] = v;
        }
    if (lane == 0) {
        float *dst = ga.partial + ((size_t)chunk * a.R + r) * a.M * a.K;
#pragma unroll
        for (int i = 0; i < GO_MT; ++i)
#pragma unroll
            for (int j = 0; j < GO_KT; ++j)
                if (m0 + i < a.M && k0 + j < a.K)
                    dst[(size_t)(m0 + i) * a.K + k0 + j] = acc[i][j];
    }
}

// grid.x: (region, pixel chunk of 64*pxl slots); grid.y: tile of 4*GO_MT instances (one GO_MT per wave);
// grid.z: tile of GO_KT patch elements
__global__ __launch_bounds__(256) void mex_grad_offsets_kernel(const MexGradArgs ga)
{
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = blockIdx.x / ga.cpr;
    const int chunk = blockIdx.x - r * ga.cpr;
    const int m0 = (blockIdx.y * 4 + wave) * GO_MT;
    if (m0 < ga.k.M)
        mex_grad_offsets_wave(ga, r, chunk, m0, blockIdx.z * GO_KT, lane);
}

// Finite epsilon, product form (see mex_grad_input_mfma_kernel): d off_mk = 2^(os_mk - mo_m) * sum_px W_px,m 2^(xs_px,k - a_px)
// is a GEMM over the pixels.  The bound a of a pixel only has to hold for the instances of the workgroup's tile, so
// it is the minimum over those.  A workgroup owns 64 instances x 64 patch elements (wave: 16 x 64, four 16 x 16
// tiles) and walks its pxl groups of 64 pixel slots: pixel factors W [pixel][instance] and patch exponentials
// [pixel][k] go to LDS, 16 matrix steps of 4 pixels each.
// grid.x: (region, pixel chunk of 64*pxl slots); grid.y: tile of 64 instances; grid.z: tile of 64 patch elements
constexpr int GOM_MT = 64, GOM_KT = 64;

//
// PIPE: the next group's values are requested in front of the current group's arithmetic (two sets of 48 registers:
// one workgroup per compute unit's share of registers less); a launch of one group per workgroup has no next one and
// fits three workgroups to a compute unit (32 x 16 x 20 x 20, 3 x 3 blocks, 32 instances: 28.8 us with one resident
// workgroup and a branch per gathered element, 13.8 now).
template <bool PIPE>
__global__ __launch_bounds__(256, PIPE ? 2 : 3) void mex_grad_offsets_mfma_kernel(const MexGradArgs ga)
{
    const MexKernelArgs &a = ga.k;
    __shared__ float wt[64 * 65];   // [pixel][instance], padded rows
    __shared__ float ex[64 * 65];   // [pixel][k], padded rows
    __shared__ float pmn[4 * 64];
    __shared__ __attribute__((aligned(16))) float cst[2 * GOM_MT];   // per instance: bound term, exponent term
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = blockIdx.x / ga.cpr;
    const int chunk = blockIdx.x - r * ga.cpr;
    const int m0 = blockIdx.y * GOM_MT, k0 = blockIdx.z * GOM_KT;
    const int n_mg = a.n_mgroups;
    const float *omax_r = a.omax + (size_t)r * n_mg * GM_TM, *orng_r = a.orng + (size_t)r * n_mg * GM_TM;
    // this thread's instances when staging (16 of the tile, the same for the whole wave)
    const int ms0 = m0 + wave * 16;
    const bool wave_active = ms0 < a.M;
    // the records of the wave's 16 patch elements: one vector load (lane i holds element i), read back lane by lane
    // where they are used - as 16 wave-uniform loads in front of the 16 gathers each was waited for on its own
    const int4 kl = a.ktab[min(k0 + wave * 16 + (lane & 15), a.K - 1)];
    if (tid < GOM_MT) {
        const int m = min(m0 + tid, a.M - 1);
        cst[tid] = a.c0 + (omax_r[m] - orng_r[m]);
        cst[GOM_MT + tid] = omax_r[m] + a.c0;
    }
    {
        int wide = 0;
        for (int m = tid; m < a.M; m += 256)
            wide |= !(orng_r[m] <= kGradProductRange);
        if (__syncthreads_or(wide)) {
            // term by term: this workgroup's tile as GO_MT x GO_KT wave tiles
            for (int i = wave; i < (GOM_MT / GO_MT) * (GOM_KT / GO_KT); i += 4) {
                const int mm0 = m0 + (i / (GOM_KT / GO_KT)) * GO_MT, kk0 = k0 + (i % (GOM_KT / GO_KT)) * GO_KT;
                if (mm0 < a.M && kk0 < a.K)
                    mex_grad_offsets_wave(ga, r, chunk, mm0, kk0, lane);
            }
            return;
        }
    }
    const size_t plane = (size_t)a.Co * a.Ho * a.Wo, gplane = pooled_g_plane(ga, plane);
    const int lr = lane & 15, lq = lane >> 4;
    floatx4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
        acc[t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    const bool buffered = ga.wbuf != nullptr;   // W and 2^(xs - a) come from mex_grad_factors_kernel
    // global loads of a group of 64 pixel slots: this thread's pixel, its 16 instances' output and gradient values
    // and 16 of the tile's patch elements; the loads of group s + 1 are issued before group s is processed
    struct Group {
        bool valid;
        float ov[16], gv[16], xr[16];
    };
    auto load_group = [&](int s, Group &q) {
        const PixelRef px = locate(a, r, (chunk * ga.pxl + s) * 64 + lane);
        q.valid = px.out_off >= 0;
        const float *gp = ga.g + (size_t)px.b * a.M * gplane + (q.valid ? pooled_g_offset(ga, px.out_off) : 0);
        const float *op = ga.out + (size_t)px.b * a.M * plane + (q.valid ? px.out_off : 0);
        // Every load on a valid address and no branches: inside a condition each would be waited for in front of the
        // next.  Instances and patch elements past the last one repeat it; their rows and columns are not stored.
        if (wave_active) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int m = min(ms0 + i, a.M - 1);
                q.ov[i] = op[(size_t)m * plane];
                q.gv[i] = gp[(size_t)m * gplane];
            }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            // {offset inside an image, dc, dh, dw} of element i
            const int kx = __builtin_amdgcn_readlane(kl.x, i), ky = __builtin_amdgcn_readlane(kl.y, i);
            const int kz = __builtin_amdgcn_readlane(kl.z, i), kw = __builtin_amdgcn_readlane(kl.w, i);
            const bool ok = mex_inside(a, px.ci0 + ky, px.hi0 + kz, px.wi0 + kw);
            const float raw = *(ok ? px.base + kx : a.in);
            q.xr[i] = ok ? raw : a.oob;
        }
    };
    Group cur;
    for (int s = 0; s < ga.pxl; ++s) {
        if (buffered) {
            // rows of the group's 64 pixel slots: thread (column cc of the tile, pixels pq, pq + 4, ...)
            const int grp = chunk * ga.pxl + s;
            if (grp * 64 >= ga.slots_pad)
                break;  // no slots left in the region (uniform)
            const size_t row0 = (size_t)r * ga.slots_pad + (size_t)grp * 64;
            const int cc = tid & 63, pq = tid >> 6;
            __syncthreads();  // the previous group's matrix instructions are done with wt / ex
            // (sixteen loads at a time, columns past the buffers' rows on a clamped address: inside the condition
            // each would be waited for in front of its LDS write)
            const int mcol_c = min(m0 + cc, ga.Mp - 1), kcol_c = min(k0 + cc, ga.Kp - 1);
#pragma unroll
            for (int j0 = 0; j0 < 16; j0 += 8) {
                float wv[8], ev[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int pp = pq + 4 * (j0 + j);
                    wv[j] = ga.wbuf[(row0 + pp) * ga.Mp + mcol_c];
                    ev[j] = ga.exbuf[(row0 + pp) * ga.Kp + kcol_c];
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int pp = pq + 4 * (j0 + j);
                    wt[pp * 65 + cc] = m0 + cc < ga.Mp ? wv[j] : 0.0f;
                    ex[pp * 65 + cc] = k0 + cc < ga.Kp ? ev[j] : 0.0f;
                }
            }
            __syncthreads();
#pragma unroll 4
            for (int ps = 0; ps < 64; ps += 4) {
                const float av = wt[(ps + lq) * 65 + wave * 16 + lr];
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, ex[(ps + lq) * 65 + t * 16 + lr], acc[t], 0, 0, 0);
            }
            continue;
        }
        if (s == 0 || !PIPE)
            load_group(s, cur);
        Group nxt;
        if (PIPE && s + 1 < ga.pxl)
            load_group(s + 1, nxt);   // in flight while this group is processed
        float amin = INFINITY;
        if (wave_active)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                amin = fminf(amin, __builtin_fmaf(cur.ov[i], a.c1, -cst[wave * 16 + i]));
        __syncthreads();  // the previous group's matrix instructions are done with wt / ex / pmn
        pmn[wave * 64 + lane] = amin;
        __syncthreads();
        const float a_p = cur.valid ? fminf(fminf(pmn[lane], pmn[64 + lane]), fminf(pmn[128 + lane], pmn[192 + lane])) : 0.0f;
        if (wave_active) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                // (an empty slot holds the values of another region's pixel: its exponent can be anything, and zero times
                // an overflowed factor would put NaN into the sums)
                const float w = cur.gv[i] * __builtin_amdgcn_exp2f(__builtin_fmaf(-cur.ov[i], a.c1, a_p) + cst[GOM_MT + wave * 16 + i]);
                wt[lane * 65 + wave * 16 + i] = cur.valid ? w : 0.0f;
            }
        }
        // patch exponentials: this thread's pixel, 16 of the tile's patch elements
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(cur.xr[i], a.c1, -a_p));
            ex[lane * 65 + wave * 16 + i] = cur.valid ? e : 0.0f;
        }
        __syncthreads();
        if (wave_active) {
#pragma unroll 4
            for (int ps = 0; ps < 64; ps += 4) {
                const float av = wt[(ps + lq) * 65 + wave * 16 + lr];
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, ex[(ps + lq) * 65 + t * 16 + lr], acc[t], 0, 0, 0);
            }
        }
        if (PIPE && s + 1 < ga.pxl)
            cur = nxt;
    }
    if (!wave_active)
        return;
    // ---- partial sums of this pixel chunk: acc * 2^(os_mk - mo_m) ----
    float *dst = ga.partial + ((size_t)chunk * a.R + r) * a.M * a.K;
    // (the 16 offset exponentials first, on clamped indices, then the products and stores)
    float eov[4][4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int m = min(m0 + wave * 16 + 4 * lq + v, a.M - 1);
        const float *eo = a.offe + (((size_t)r * n_mg + m / GM_TM) * a.K) * GM_TM + m % GM_TM;
#pragma unroll
        for (int t = 0; t < 4; ++t)
            eov[v][t] = eo[(size_t)min(k0 + t * 16 + lr, a.K - 1) * GM_TM];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int m = m0 + wave * 16 + 4 * lq + v;
        if (m >= a.M)
            continue;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int k = k0 + t * 16 + lr;
            if (k < a.K)
                dst[(size_t)m * a.K + k] = acc[t][v] * eov[v][t];
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// Row-wise forms of the two matrix kernels for the layers of the reference's networks: 2 x 2 unshared offsets over
// whole-channel patches (blocks [C, 1, 1], stride 1, no padding) on maps whose height and width are powers of two.
// There the pixel slots of a region are every other pixel of every other row.  A wave that walks one region's slots
// touches 16 to 64 separate 32-byte sectors per load and uses half of each or less, the four regions write the
// input gradient into each other's sectors at different times, and the address units, not the arithmetic, set the
// time of the kernels above.  Here a workgroup takes the 64 slots of a chunk for ALL four regions - 256 pixels that
// are whole rows of one image or whole small images - so that every plane (an instance of `out` / `g`, a channel
// of the input or of its gradient) is read and written as one run of 1 KB, or runs of whole images, with 16-byte
// accesses.  The values pass through LDS tiles [plane][column] with column = region * 64 + slot, and wave r does
// the matrix steps of region r on its 64 columns.
// Everything the kernel reads outside of its term-by-term path, in one block: fetched at once, and not piece by piece where
// it is first needed (a round trip to memory each).
struct RowsArgs {
    const float *in, *out, *g;
    const float *offe, *omax, *orng;   // the packed offsets
    float *dx, *partial;               // (of split 0; null: not wanted)
    long long dx_split;                // floats from one split's input gradient to the next's
    float c0, c1;
    int B, M, K, n_mg, mg_per_split;
    int lgW, Ws, RS;   // log2(width), windows per row, windows per image
    int lgHW, HW;      // pixels of an image
    int chunks, pxl;   // of 256 pixels: in all, per workgroup
    int nx, ty, tz;    // workgroup numbering (rows_block): pixel groups, tiles along the two other grid dimensions,
    int per_die;       // ... an eighth of them all
    FastDiv d_tiles, d_ty;   // ty * tz; ty
};

// Workgroups that read the same rows - the tiles (y, z) of one pixel group x - get turns on ONE accelerator die (linear
// workgroup id mod 8), so that the rows come from memory once and from that die's L2 for the other tiles: each die takes an
// eighth of all tiles, in order.  (Whole groups to a die, x mod 8, leave dies idle where there are few: the 2 x 2
// maps of 32 images, one group, 35.5 -> 16.0 us.)  The launch is one-dimensional with 8 g.per_die workgroups; false:
// nothing is left for this one.
__device__ __forceinline__ bool rows_block(const RowsArgs &g, int *x, int *y, int *z)
{
    const int l = blockIdx.x, tiles = g.ty * g.tz, i = (l & 7) * g.per_die + (l >> 3);
    if (i >= g.nx * tiles)
        return false;
    *x = (int)fast_div((unsigned)i, g.d_tiles);
    const int tile = i - *x * tiles;
    *z = (int)fast_div((unsigned)tile, g.d_ty);
    *y = tile - *z * g.ty;
    return true;
}

// A thread's four neighbouring pixels (16 bytes) of the chunk's 256: image, first pixel, tile columns.  They share a row, and
// pixels 0 and 2 belong to region rbase, 1 and 3 to rbase + 1; on maps of two columns (W2) they are a window and belong to
// the four regions in turn.  A chunk starts on an even row (or a whole image), so columns and regions depend on the quad
// alone, not on the chunk.
template <bool W2>
struct RowsQuad {
    int img, pix0, rbase, col0;
    __device__ __forceinline__ RowsQuad(const RowsArgs &g, int chunk, int quad)
    {
        const int gpix = chunk * 256 + 4 * quad;
        img = gpix >> g.lgHW;
        pix0 = gpix & (g.HW - 1);
        const int h = pix0 >> g.lgW, w0 = pix0 & ((1 << g.lgW) - 1);
        rbase = W2 ? 0 : (h & 1) * 2;
        col0 = (rbase << 6) + img * g.RS + (h >> 1) * g.Ws + (w0 >> 1) - chunk * 64;
    }
    __device__ __forceinline__ int region(int e) const { return W2 ? e : rbase + (e & 1); }
    __device__ __forceinline__ int col(int e) const { return W2 ? col0 + (e << 6) : col0 + ((e & 1) << 6) + (e >> 1); }
    // of the pooled map: the quad's first window
    __device__ __forceinline__ int window(const RowsArgs &g) const
    {
        const int h = pix0 >> g.lgW, w0 = pix0 & ((1 << g.lgW) - 1);
        return (h >> 1) * g.Ws + (w0 >> 1);
    }
};

// The output gradients of a thread's pixel quad as they come from memory: 16 bytes of g, or - POOLED, g is that of the
// windows' sums - the gradients of the windows the quad lies in (x, y; each belongs to two pixels; W2: one, x).
// rows_quad_g expands them where they are used: expanding here would wait for the load where it is issued.
template <bool W2, bool POOLED>
struct RowsGrad {
    typedef std::conditional_t<!POOLED, float4, std::conditional_t<W2, float, float2>> type;
};

__device__ __forceinline__ void rows_quad_g(const float4 &v, float (&gg)[4])
{
    gg[0] = v.x; gg[1] = v.y; gg[2] = v.z; gg[3] = v.w;
}

__device__ __forceinline__ void rows_quad_g(const float2 &v, float (&gg)[4])
{
    gg[0] = gg[1] = v.x;
    gg[2] = gg[3] = v.y;
}

__device__ __forceinline__ void rows_quad_g(float v, float (&gg)[4])
{
    gg[0] = gg[1] = gg[2] = gg[3] = v;
}

// A uniform address and a lane's offset in elements (less than 2^31 bytes: rows_geometry)
template <typename T>
__device__ __forceinline__ T rows_load(const float *base, unsigned at)
{
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + 4 * at);
}

// What a region does term by term: bits of the flags below.
enum { kRowsInput = 1, kRowsOffsets = 2 };

// per region: is some instance's offsets range beyond kGradRowsRange or not finite (flags[r]: both gradients term by term);
// flags[4]: does some range exceed kLooseBoundRange.  All threads of the workgroup call flag(); the flags (five, zero before a
// barrier) are in place behind the next one.  The constructor requests the first 256 instances' ranges.
struct RowsRanges {
    float v[4];
    __device__ __forceinline__ RowsRanges(const RowsArgs &g, int tid)
    {
        load(g, min(tid, g.M - 1));
    }
    __device__ __forceinline__ void load(const RowsArgs &g, int m)
    {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            v[r] = g.orng[r * g.n_mg * GM_TM + m];
    }
    __device__ __forceinline__ void flag(const RowsArgs &g, int tid, int *flags)
    {
        for (int m = tid;;) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (m < g.M && !(v[r] <= kLooseBoundRange)) {
                    flags[4] = 1;      // (every writer writes the same value)
                    if (!(v[r] <= kGradRowsRange))
                        flags[r] = kRowsInput | kRowsOffsets;
                }
            m += 256;
            if (m >= g.M)
                break;
            load(g, m);
        }
    }
};

constexpr int kLateOffsets = 1 << 16;

// A product and a sum with a rounding each, whatever else is fused: two kernels add up the same partial sums, bit for bit.
__device__ __forceinline__ float rows_product(float a, float b)
{
#pragma clang fp contract(off)
    return a * b;
}

__device__ __forceinline__ float rows_sum(float a, float b)
{
#pragma clang fp contract(off)
    return a + b;
}

#if defined(__HIP_DEVICE_COMPILE__)
// The term-by-term path of the kernel below reads its arguments from the kernel's argument segment (they are the last, in front
// of the implicit ones) and is a call: inlined, what it keeps in scalar registers is fetched, and spilled, at the kernel's start.
static_assert(sizeof(MexGradArgs) % 8 == 0, "the explicit arguments end with the block");
__device__ __forceinline__ const MexGradArgs &rows_term_args()
{
    return *reinterpret_cast<const MexGradArgs *>(reinterpret_cast<const char *>(__builtin_amdgcn_implicitarg_ptr()) -
                                                  sizeof(MexGradArgs));
}

// The regions with a wide offsets range, or with a chunk's wide pixels: late holds a bit per chunk (sixteen at most) for the input
// gradient of each, and kLateOffsets.  GX_KT patch elements of a region per wave and turn for the input gradient; for the offsets
// the tile of KT patch elements as GO_MT x GO_KT wave tiles over all chunks.
// (Arguments of a call are in vector registers: all are uniform.)
template <int KT>
__device__ __noinline__ void rows_terms(int bx_v, int n_chunks_v, int k0_v, int mg_begin_v, int mg_end_v, float *dx_v, int offsets_v,
                                        int4 late_v)
{
    const MexGradArgs &ga = rows_term_args();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    const int bx = uniform(bx_v), n_chunks = uniform(n_chunks_v), k0 = uniform(k0_v), mg_begin = uniform(mg_begin_v),
              mg_end = uniform(mg_end_v), offsets = uniform(offsets_v);
    const int late[4] = {uniform(late_v.x), uniform(late_v.y), uniform(late_v.z), uniform(late_v.w)};
    const unsigned long long dx_bits = (unsigned long long)(uintptr_t)dx_v;
    float *dx = reinterpret_cast<float *>((unsigned long long)(unsigned)uniform((int)(dx_bits >> 32)) << 32 | (unsigned)uniform((int)dx_bits));
    const int M = ga.k.M, K = ga.k.K, m_begin = min(M, mg_begin * GM_TM), m_end = min(M, mg_end * GM_TM);
    constexpr int NX = KT / GX_KT, NO = KT / GO_KT, NM = 32 / GO_MT;
    if (dx != nullptr)
        for (int s = 0; s < n_chunks; ++s)
            for (int u = wave; u < 4 * NX; u += 4) {
                const int r = u / NX, kk0 = k0 + u % NX * GX_KT;
                if ((late[r] >> s & 1) && kk0 < K)
                    mex_grad_input_wave(ga, r, bx * ga.pxl + s, kk0, lane, m_begin, m_end, dx);
            }
    if (offsets)
        for (int m0 = m_begin; m0 < m_end; m0 += 32)
            for (int u = wave; u < 4 * NM * NO; u += 4) {
                const int r = u / (NM * NO), i = u % (NM * NO), mm0 = m0 + i / NO * GO_MT, kk0 = k0 + i % NO * GO_KT;
                if ((late[r] & kLateOffsets) && mm0 < M && kk0 < K)
                    mex_grad_offsets_wave(ga, r, bx, mm0, kk0, lane);
            }
}
#endif

// Both gradients, or either.  Workgroup (rows_block) x: group of ga.pxl chunks of 256 pixels; y: tile of 16 * KSUB patch
// elements; z: split of the instance groups.  A thread's pixels are one quad of the chunk, its planes pl0, pl0 + 4, ... of
// every block of 32: a wave's load is four planes of sixteen quads, whole runs of memory on maps of any size (2 x 2 ones
// included: neighbouring planes of an image are neighbours in memory), and what concerns one pixel - its bound a - needs
// no LDS.  Per instance group the pixel factors W [32][256] are formed once, from rows of `out` and `g`, and serve both
// products: wave r multiplies region r's W with the offset exponentials (input gradient, added up over the groups) and
// with the tile's patch exponentials 2^(xs - a) of its 64 columns, which it holds as matrix operands in registers
// (offsets gradient, to the partial sums at once; with several chunks the workgroup adds to what it has stored).  The input gradient
// leaves through a tile [patch element][column], times 2^(xs - a), as rows.  A region with a wide offsets range is done
// term by term (the other three are not held up by it).
//
// Bound by the latency of a workgroup's phases, two workgroups to a compute unit, of which the matrix steps are a third.
// The two gradients were a kernel each: both read `out` and `g` and formed W, the one for the offsets once more for every 32 patch
// elements.  512 images, whole call, 32 channels of 16 x 16 -> 64
// instances, 64 of 8 x 8 -> 128, 128 of 4 x 4 -> 256, 256 of 2 x 2 -> 512: both gradients 57, 54, 59, 72 -> 44, 39, 41, 52 us, the
// input's alone 27, 27, 33, 47 -> 24.5, 21, 27, 34, the offsets' alone 34, 30, 32, 45 -> 31.5 (mex_grad_offsets_rows_kernel), 30, 29, 37.
// 32 images, both, the kernels of four such layers and their sums: 118 -> 75.  The bound is taken over the first group's
// instances: errors against 64 bits as before, and a third to a half of it for offsets that span 24 to 48 exponents on 2 x 2 maps.
// W2: the map has two columns, a quad is a window and its pixels belong to the four regions.
// WANT: the only gradient wanted, or 0.  Compiled for one alone the kernel needs 20 to 30 registers less, none of them in memory: 28.5, 25,
// 28.5, 37.5 and 37.5, 33.5, 32.5, 40.5 us where both are decided at run time.  (Compiled for both: 44 -> 46.5, 39 -> 41 on the
// first and third.)
//
// The tile's pitch, 20 modulo 64: sixteen lanes' 16-byte operands of a column of rows, or of a row, lie in different banks.
template <int KSUB, bool W2, bool POOLED, int WANT>
__global__ __launch_bounds__(256, KSUB == 1 ? 3 : 2) void mex_grads_rows_kernel(const RowsArgs g, const MexGradArgs ga)
{
    constexpr int KT = 16 * KSUB, NJ = KT / 4;
    constexpr int TP = 276, EP = 36;
    // The pixel's own maximum as the bound where the tile holds all of K: at hand for the offsets, one pass more over those rows for
    // the input alone.  Both 44 -> 42.6 us (512 x 32 x 16 x 16 -> 64), input 22.8 -> 24.5, errors of offsets that span 20 exponents 3.8e-7
    // -> 2.7e-7.  (KSUB 1: no registers left for it, 512 x 64 x 8 x 8 -> 128 37.8 -> 38.7.)
    constexpr bool kTight = KSUB == 2;
    __shared__ __attribute__((aligned(16))) float wt[32 * TP];        // W, and before and behind it the patch elements' tile
    __shared__ __attribute__((aligned(16))) float eo[4 * KT * EP];    // [region][patch element][instance]
    __shared__ float tab[2][128];      // per (region, instance of the group): omax + c0, for this group and the next
    __shared__ float lo_tab[128];      // ... and c0 + the offsets' minimum, of the first group
    __shared__ int wide_sh[5];         // see RowsRanges
    __shared__ int late[4];            // per region: the chunks (bits) that are left to the term-by-term waves
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lq = lane >> 4;
    int bx, by, bz;
    if (!rows_block(g, &bx, &by, &bz))
        return;
    const bool want_input = WANT == kRowsInput || (WANT == 0 && g.dx != nullptr);
    const bool want_offsets = WANT == kRowsOffsets || (WANT == 0 && g.partial != nullptr);
    const int k0 = by * KT;
    const int n_mg = g.n_mg, per = n_mg * GM_TM;
    const int mg_begin = bz * g.mg_per_split, mg_end = min(n_mg, mg_begin + g.mg_per_split);
    float *dxo = g.dx + bz * g.dx_split;
    int pl0 = lane >> 4;
    const RowsQuad<W2> q0(g, 0, wave * 16 + (lane & 15));   // (its columns and regions are the same in every chunk)
    // where pixel e of the quad lies in row pl0 + 4 j
    const int tile0 = pl0 * TP + q0.col(0);
    auto tile_index = [&](int j, int e) { return tile0 + 4 * j * TP + (W2 ? e * 64 : (e & 1) * 64 + (e >> 1)); };
    // Matrix operands, 16 bytes to a read: the terms of a product are added in any order both operands agree on, so lane (lr,
    // lq) takes four columns 16 lq + 4 i ... of row lr (four steps of a contraction over columns); and a product's columns
    // may stand for any pixels: column lr of product t is pixel 4 lr + t (the four products' operands of one row).
    auto read4 = [&](const float *at, float (&v)[4]) {
        const float4 f = *reinterpret_cast<const float4 *>(at);
        v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
    };
    const float *const by_row = wt + lr * TP + wave * 64 + 16 * lq;
    float *const by_col = wt + wave * 64 + 4 * lr;

    // operands of an instance group: this thread's eight pieces of rows of `out` and `g`, its share of the four regions'
    // offset exponentials, the next group's instance constants - requested a group ahead, while the matrix steps run
    typedef typename RowsGrad<W2, POOLED>::type Grad;
    float4 ov[8], en[2 * KSUB];
    Grad gv[8];
    float tn = 0.0f;
    // a chunk's first image, and this lane's pixels from there on
    const int gplane = POOLED ? g.HW >> 2 : g.HW;
    const float *out_c, *g_c, *x_c;
    unsigned out_at, g_at, x_at;
    size_t first;
    bool img_ok;
    auto locate_chunk = [&](int chunk) {
        const RowsQuad<W2> q(g, chunk, wave * 16 + (lane & 15));
        const int img0 = chunk * 256 >> g.lgHW;
        img_ok = q.img < g.B;
        const unsigned img = img_ok ? q.img - img0 : 0;
        first = (size_t)img0 * g.K * g.HW;
        out_c = g.out + (size_t)img0 * g.M * g.HW;
        g_c = g.g + (size_t)img0 * g.M * gplane;
        x_c = g.in + first;
        out_at = img * g.M * g.HW + q.pix0;
        g_at = img * g.M * gplane + (POOLED ? q.window(g) : q.pix0);
        x_at = img * g.K * g.HW + q.pix0;
    };
    auto request = [&](int mg) {
        // (those past the last instance, image or patch element on a clamped address)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const unsigned m = min(mg * GM_TM + pl0 + 4 * j, g.M - 1);
            ov[j] = rows_load<float4>(out_c, out_at + m * g.HW);
            gv[j] = rows_load<Grad>(g_c, g_at + m * gplane);
        }
#pragma unroll
        for (int j = 0; j < 2 * KSUB; ++j) {
            const int i = tid + 256 * j;
            const int r = i / (KT * 8), row = (i % (KT * 8)) >> 3, c4 = i & 7;
            en[j] = rows_load<float4>(g.offe, ((r * n_mg + mg) * g.K + min(k0 + row, g.K - 1)) * GM_TM + 4 * c4);
        }
        tn = g.omax[(tid >> 5 & 3) * per + min(mg + 1, n_mg - 1) * GM_TM + (tid & 31)];
    };
    float4 xv[NJ];                     // rows of the input's tile, for 2^(xs - a)
    auto request_input = [&]() {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            xv[j] = rows_load<float4>(x_c, x_at + (unsigned)min(k0 + pl0 + 4 * j, g.K - 1) * g.HW);
    };

    const int n_chunks = min(g.pxl, g.chunks - bx * g.pxl);
    // (loads return in order: the small ones, which the flags wait for, in front of the rows)
    RowsRanges ranges(g, tid);
    const int own = (tid >> 5 & 3) * per + mg_begin * GM_TM + (tid & 31);   // (the packed arrays are padded to whole groups)
    const float om = g.omax[own], rng = g.orng[own];
    if (tid < 5)
        wide_sh[tid] = 0;
    if (tid < 4)
        late[tid] = 0;
    locate_chunk(bx * g.pxl);
    request(mg_begin);
    if (want_offsets)
        request_input();
    __syncthreads();
    if (tid < 128) {
        tab[mg_begin & 1][tid] = om + g.c0;
        lo_tab[tid] = g.c0 + (om - rng);
    }
    ranges.flag(g, tid, wide_sh);
    __syncthreads();
    const bool roomy = wide_sh[4] != 0;
    const int unbounded = __builtin_amdgcn_readfirstlane(wide_sh[wave]);   // this wave's region: term by term whatever its pixels

    const bool nothing = (wide_sh[0] & wide_sh[1] & wide_sh[2] & wide_sh[3]) != 0;   // all four regions
    if (nothing && tid < 4)
        late[tid] = (1 << n_chunks) - 1 | kLateOffsets;
    for (int s = nothing ? n_chunks : 0; s < n_chunks; ++s) {
        asm volatile("" : "+v"(pl0));   // (what follows from it is cheap to form again, and too much to keep across the chunks)
        if (s > 0) {
            locate_chunk(bx * g.pxl + s);
            request(mg_begin);
            if (want_offsets)
                request_input();
            if (tid < 128)
                tab[mg_begin & 1][tid] = g.omax[(tid >> 5) * per + mg_begin * GM_TM + (tid & 31)] + g.c0;
        }
        // ---- the bound of every pixel: a >= every xs_k of its patch ----
        // The minimum over a group of instances of outs_m - c0 - lo_m, see mex_grad_input_mfma_kernel.  Where some offsets
        // range is large that is loose by up to the range, which costs the factors their precision (and, beyond
        // kGradProductRange, the product form): there it is the pixel's own maximum over all of K, from one sweep over
        // the rows of the input.  The exponents then stay within the pixel's patch range, and a region keeps the
        // product form while those ranges are at most kGradPixelRange and its offsets span at most kGradRowsRange.
        // (Where the tile holds all of K the maximum is at hand, whatever the ranges.)
        float bound[4], alo[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            bound[e] = -INFINITY;
            alo[e] = INFINITY;
        }
        if (roomy || (kTight && g.K <= KT && !want_offsets)) {
            for (int k = pl0; k < g.K; k += 32) {
                float4 xr[8];
#pragma unroll
                for (int j = 0; j < 8; ++j)   // (behind the last: the last)
                    xr[j] = rows_load<float4>(x_c, x_at + (unsigned)min(k + 4 * j, g.K - 1) * g.HW);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float v[4] = {xr[j].x, xr[j].y, xr[j].z, xr[j].w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {   // (fmax / fmin skip NaN)
                        bound[e] = fmaxf(bound[e], v[e] * g.c1);
                        alo[e] = fminf(alo[e], v[e] * g.c1);
                    }
                }
            }
        } else if (kTight && g.K <= KT) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const float v[4] = {xv[j].x, xv[j].y, xv[j].z, xv[j].w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    bound[e] = fmaxf(bound[e], v[e] * g.c1);
            }
        }
        if (roomy) {
            // each chunk decides for itself: behind the readers of the ranges' flags above, or of the chunk's before
            if (s > 0 && lane == 0)
                wide_sh[wave] = unbounded;
            __syncthreads();
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                for (int d = 16; d < 64; d <<= 1) {
                    bound[e] = fmaxf(bound[e], __shfl_xor(bound[e], d, 64));
                    alo[e] = fminf(alo[e], __shfl_xor(alo[e], d, 64));
                }
                // A pixel with an infinite value or nothing finite sends its region term by term, one with a patch range
                // beyond the bound the region's input gradient.  (To the offsets' gradient a patch element far below the pixel's
                // largest adds next to nothing: W is 2^kGradRowsRange of g at most.  512 x 32 x 16 x 16 -> 64, such a
                // pixel in each image: 45 us where the offsets' gradient took 192 term by term, both 105 and 255.)
                const bool finite = fabsf(bound[e]) < INFINITY;
                if (img_ok && !(finite && bound[e] - alo[e] <= kGradPixelRange))
                    atomicOr(&wide_sh[q0.region(e)], finite ? kRowsInput : kRowsInput | kRowsOffsets);
            }
        } else if (kTight && g.K <= KT) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                for (int d = 16; d < 64; d <<= 1)
                    bound[e] = fmaxf(bound[e], __shfl_xor(bound[e], d, 64));
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                bound[e] = INFINITY;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float o[4] = {ov[j].x, ov[j].y, ov[j].z, ov[j].w};
                const bool there = mg_begin * GM_TM + pl0 + 4 * j < g.M;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float b = __builtin_fmaf(o[e], g.c1, -lo_tab[q0.region(e) * 32 + pl0 + 4 * j]);
                    bound[e] = fminf(bound[e], there ? b : INFINITY);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                for (int d = 16; d < 64; d <<= 1)
                    bound[e] = fminf(bound[e], __shfl_xor(bound[e], d, 64));
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            bound[e] = img_ok ? bound[e] : 0.0f;

        // ---- the patch exponentials as matrix operands: patch element 16 kt + lr, columns 16 lq + 4 i + ... of this wave's ----
        float exr[KSUB][4][4];
        if (want_offsets) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const float x[4] = {xv[j].x, xv[j].y, xv[j].z, xv[j].w};
                const bool use = img_ok && k0 + pl0 + 4 * j < g.K;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float v = __builtin_amdgcn_exp2f(__builtin_fmaf(x[e], g.c1, -bound[e]));
                    wt[tile_index(j, e)] = use ? v : 0.0f;
                }
            }
            __syncthreads();
#pragma unroll
            for (int kt = 0; kt < KSUB; ++kt)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    read4(by_row + kt * 16 * TP + 4 * i, exr[kt][i]);
        }

        floatx4 acc[KSUB][4];
#pragma unroll
        for (int ks = 0; ks < KSUB; ++ks)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                acc[ks][t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int mg = mg_begin; mg < mg_end; ++mg) {
            __syncthreads();           // everyone is done with the tile, the offset exponentials and the flags
            const float *tb = tab[mg & 1];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int pl = pl0 + 4 * j;
                const bool use = img_ok && mg * GM_TM + pl < g.M;
                const float o[4] = {ov[j].x, ov[j].y, ov[j].z, ov[j].w};
                float gg[4];
                rows_quad_g(gv[j], gg);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    // (a - outs) first: a small, once-rounded difference; the instance constant is added to that (forming
                    // a + mo first, about the size of outs, was tried for the tight bound: worse on half of the data)
                    const float ex = __builtin_fmaf(-o[e], g.c1, bound[e]) + tb[q0.region(e) * 32 + pl];
                    const float w = gg[e] * __builtin_amdgcn_exp2f(ex);
                    wt[tile_index(j, e)] = use ? w : 0.0f;
                }
            }
#pragma unroll
            for (int j = 0; j < 2 * KSUB; ++j) {
                const int i = tid + 256 * j;
                const int r = i / (KT * 8), row = (i % (KT * 8)) >> 3, c4 = i & 7;
                const bool use = k0 + row < g.K;
                *reinterpret_cast<float4 *>(eo + (r * KT + row) * EP + 4 * c4) = use ? en[j] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
            if (tid < 128)
                tab[(mg + 1) & 1][tid] = tn + g.c0;
            if (mg + 1 < mg_end)
                request(mg + 1);
            else if (want_input)
                request_input();
            __syncthreads();
            if (want_input) {
                // (lane lq: instances 8 lq + i)
                float av[KSUB][2][4];
#pragma unroll
                for (int ks = 0; ks < KSUB; ++ks)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        read4(eo + (wave * KT + ks * 16 + lr) * EP + 8 * lq + 4 * h, av[ks][h]);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    float bv[4];
                    read4(by_col + (8 * lq + i) * TP, bv);
#pragma unroll
                    for (int ks = 0; ks < KSUB; ++ks)
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                            acc[ks][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[ks][i / 4][i % 4], bv[t], acc[ks][t], 0, 0, 0);
                }
            }
            if (want_offsets) {
                floatx4 sum[2][KSUB];
#pragma unroll
                for (int mt = 0; mt < 2; ++mt)
#pragma unroll
                    for (int kt = 0; kt < KSUB; ++kt)
                        sum[mt][kt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float wa[2][4];
#pragma unroll
                    for (int mt = 0; mt < 2; ++mt)
                        read4(by_row + mt * 16 * TP + 4 * i, wa[mt]);
#pragma unroll
                    for (int c = 0; c < 4; ++c)
#pragma unroll
                        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
                            for (int kt = 0; kt < KSUB; ++kt)
                                sum[mt][kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(exr[kt][i][c], wa[mt][c], sum[mt][kt], 0, 0, 0);
                }
                // partial sums, times 2^(os_mk - mo_m): a lane's are four neighbouring patch elements of an instance
                float *dst = g.partial + ((size_t)bx * 4 + wave) * g.M * g.K;
#pragma unroll
                for (int mt = 0; mt < 2; ++mt)
#pragma unroll
                    for (int kt = 0; kt < KSUB; ++kt) {
                        const int m = mg * GM_TM + mt * 16 + lr, k = k0 + kt * 16 + 4 * lq;
                        const float *e = eo + (wave * KT + kt * 16 + 4 * lq) * EP + mt * 16 + lr;
                        float add[4];
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            add[v] = rows_product(sum[mt][kt][v], e[v * EP]);
                        if (m >= g.M || k >= g.K)
                            continue;
                        float *at = reinterpret_cast<float *>(reinterpret_cast<char *>(dst) + 4 * ((unsigned)m * g.K + k));
                        if ((g.K & 3) == 0) {
                            float4 old = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                            if (s > 0)
                                old = *reinterpret_cast<const float4 *>(at);
                            *reinterpret_cast<float4 *>(at) = make_float4(rows_sum(old.x, add[0]), rows_sum(old.y, add[1]),
                                                                          rows_sum(old.z, add[2]), rows_sum(old.w, add[3]));
                        } else {
#pragma unroll
                            for (int v = 0; v < 4; ++v)
                                if (k + v < g.K)
                                    at[v] = s > 0 ? rows_sum(at[v], add[v]) : add[v];
                        }
                    }
            }
        }
        const int my_wide = __builtin_amdgcn_readfirstlane(wide_sh[wave]);   // (its products are left unused)
        if (my_wide && lane == 0)
            late[wave] |= ((my_wide & kRowsInput) != 0 ? 1 << s : 0) | ((my_wide & kRowsOffsets) != 0 ? kLateOffsets : 0);

        // ---- d patch_k = 2^(xs_k - a) * acc: through the tile [patch element][column] to rows of the gradient ----
        __syncthreads();               // the last matrix steps are done with the tile and the tables
        if (want_input) {
#pragma unroll
            for (int ks = 0; ks < KSUB; ++ks)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    *reinterpret_cast<float4 *>(by_col + (ks * 16 + 4 * lq + v) * TP) =
                        make_float4(acc[ks][0][v], acc[ks][1][v], acc[ks][2][v], acc[ks][3][v]);
            __syncthreads();
            const bool any_wide = ((wide_sh[0] | wide_sh[1] | wide_sh[2] | wide_sh[3]) & kRowsInput) != 0;
            float *dst = dxo + first;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int k = k0 + pl0 + 4 * j;
                if (!img_ok || k >= g.K)
                    continue;
                const float x[4] = {xv[j].x, xv[j].y, xv[j].z, xv[j].w};
                float d[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    d[e] = wt[tile_index(j, e)] * __builtin_amdgcn_exp2f(__builtin_fmaf(x[e], g.c1, -bound[e]));
                float *to = reinterpret_cast<float *>(reinterpret_cast<char *>(dst) + 4 * (x_at + (unsigned)k * g.HW));
                if (!any_wide) {
                    *reinterpret_cast<float4 *>(to) = make_float4(d[0], d[1], d[2], d[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (!(wide_sh[q0.region(e)] & kRowsInput))
                            to[e] = d[e];
                }
            }
            __syncthreads();           // everyone is done with the tile and the flags
        }
    }
    __syncthreads();
#if defined(__HIP_DEVICE_COMPILE__)
    if ((late[0] | late[1] | late[2] | late[3]) != 0)
        rows_terms<KT>(bx, n_chunks, k0, mg_begin, mg_end, want_input ? dxo : nullptr, want_offsets,
                       make_int4(late[0], late[1], late[2], late[3]));
#endif
}

// The offsets gradient by itself, on maps of four columns and more: of layers whose two gradients are a kernel each
// (MexGradTiling::rows_apart), and wanted alone where the tile holds all of K, bit for bit as mex_grads_rows_kernel gives it.
// Workgroup (rows_block) x: group of ga.pxl chunks; y: tile of 32 patch elements; z: group of instances.  Per chunk the group's
// pixel factors W and the tile's patch exponentials are formed side by side, and wave r takes region r's 32 x 32 products over
// its 64 columns: the sums stay in registers over the chunks, and the next chunk's rows are requested in front of the matrix
// steps.  (In the other kernel a workgroup's sums, of all instance groups, are too many for that: each chunk's are added to
// what is stored.)  The bound is the pixel's maximum where the tile holds all of K or some offsets range is large, as there, and
// over the group's own instances otherwise.
// Bound by the exponentials and their way through LDS, two workgroups to a compute unit.  Offsets alone, this kernel and the
// other: 512 x 32 x 16 x 16 -> 64 31.5, 32.8 us, 2048 x 32 x 16 x 16 -> 64 82, 103; 512 x 96 x 16 x 16 -> 192 134, 177.
template <bool POOLED>
__global__ __launch_bounds__(256, 2) void mex_grad_offsets_rows_kernel(const RowsArgs g, const MexGradArgs ga)
{
    constexpr int TP = 276;            // (see mex_grads_rows_kernel)
    __shared__ __attribute__((aligned(16))) float wt[32 * TP];   // [instance][column]
    __shared__ __attribute__((aligned(16))) float et[32 * TP];   // [patch element][column]
    __shared__ int wide_sh[5];         // see RowsRanges
    __shared__ int odd_sh[4];          // per region: met a pixel that only the term-by-term path can take
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lq = lane >> 4;
    int bx, by, mg;
    if (!rows_block(g, &bx, &by, &mg))
        return;
    const int k0 = by * 32, per = g.n_mg * GM_TM;
    const RowsQuad<false> q0(g, 0, wave * 16 + (lane & 15));
    const int tile0 = lq * TP + q0.col(0);   // of row lq + 4 j
    auto tile_index = [&](int j, int e) { return tile0 + 4 * j * TP + (e & 1) * 64 + (e >> 1); };

    typedef typename RowsGrad<false, POOLED>::type Grad;
    float4 ov[8], xv[8];
    Grad gv[8];
    const int gplane = POOLED ? g.HW >> 2 : g.HW;
    const float *x_c;
    unsigned x_at;
    bool img_ok;
    auto request = [&](int chunk) {    // (those past the last instance, image or patch element on a clamped address)
        const RowsQuad<false> q(g, chunk, wave * 16 + (lane & 15));
        const int img0 = chunk * 256 >> g.lgHW;
        img_ok = q.img < g.B;
        const unsigned img = img_ok ? q.img - img0 : 0;
        const float *out_c = g.out + (size_t)img0 * g.M * g.HW, *g_c = g.g + (size_t)img0 * g.M * gplane;
        const unsigned out_at = img * g.M * g.HW + q.pix0, g_at = img * g.M * gplane + (POOLED ? q.window(g) : q.pix0);
        x_c = g.in + (size_t)img0 * g.K * g.HW;
        x_at = img * g.K * g.HW + q.pix0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const unsigned m = min(mg * GM_TM + lq + 4 * j, g.M - 1);
            ov[j] = rows_load<float4>(out_c, out_at + m * g.HW);
            gv[j] = rows_load<Grad>(g_c, g_at + m * gplane);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j)
            xv[j] = rows_load<float4>(x_c, x_at + (unsigned)min(k0 + lq + 4 * j, g.K - 1) * g.HW);
    };
    const int n_chunks = min(g.pxl, g.chunks - bx * g.pxl);
    RowsRanges ranges(g, tid);
    // this thread's instances in its two regions: c0 + the offsets' largest, and smallest
    float hi[8][2], lo[8][2];
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int at = q0.region(e) * per + mg * GM_TM + lq + 4 * j;   // (the packed arrays are padded to whole groups)
            hi[j][e] = g.omax[at];
            lo[j][e] = g.orng[at];
        }
    if (tid < 5)
        wide_sh[tid] = 0;
    if (tid < 4)
        odd_sh[tid] = 0;
    request(bx * g.pxl);
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            lo[j][e] = g.c0 + (hi[j][e] - lo[j][e]);
            hi[j][e] += g.c0;
        }
    __syncthreads();
    ranges.flag(g, tid, wide_sh);
    __syncthreads();
    const bool roomy = wide_sh[4] != 0;
    const bool nothing = (wide_sh[0] & wide_sh[1] & wide_sh[2] & wide_sh[3]) != 0;   // all four regions term by term

    floatx4 total[2][2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
            total[mt][kt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    float eov[2][2][4];                // the offset exponentials of the sums
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                eov[mt][kt][v] = g.offe[(((size_t)wave * g.n_mg + mg) * g.K + min(k0 + kt * 16 + 4 * lq + v, g.K - 1)) * GM_TM +
                                        mt * 16 + lr];
    for (int s = nothing ? n_chunks : 0; s < n_chunks; ++s) {
        // the bound of every pixel, see mex_grads_rows_kernel
        float bound[4];
        if (g.K <= 32 || roomy) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                bound[e] = -INFINITY;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float v[4] = {xv[j].x, xv[j].y, xv[j].z, xv[j].w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    bound[e] = fmaxf(bound[e], v[e] * g.c1);
            }
            for (int k = lq; k < g.K && g.K > 32; k += 32) {
                float4 xr[8];
#pragma unroll
                for (int j = 0; j < 8; ++j)   // (behind the last: the last)
                    xr[j] = rows_load<float4>(x_c, x_at + (unsigned)min(k + 4 * j, g.K - 1) * g.HW);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float v[4] = {xr[j].x, xr[j].y, xr[j].z, xr[j].w};
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        bound[e] = fmaxf(bound[e], v[e] * g.c1);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                for (int d = 16; d < 64; d <<= 1)
                    bound[e] = fmaxf(bound[e], __shfl_xor(bound[e], d, 64));
                if (roomy && img_ok && !(fabsf(bound[e]) < INFINITY))
                    odd_sh[q0.region(e)] = 1;   // (every writer writes the same value)
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                bound[e] = INFINITY;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float o[4] = {ov[j].x, ov[j].y, ov[j].z, ov[j].w};
                const bool there = mg * GM_TM + lq + 4 * j < g.M;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    bound[e] = fminf(bound[e], there ? __builtin_fmaf(o[e], g.c1, -lo[j][e & 1]) : INFINITY);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                for (int d = 16; d < 64; d <<= 1)
                    bound[e] = fminf(bound[e], __shfl_xor(bound[e], d, 64));
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            bound[e] = img_ok ? bound[e] : 0.0f;
        __syncthreads();               // everyone is done with the tiles
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const bool use_m = img_ok && mg * GM_TM + lq + 4 * j < g.M, use_k = img_ok && k0 + lq + 4 * j < g.K;
            const float o[4] = {ov[j].x, ov[j].y, ov[j].z, ov[j].w}, x[4] = {xv[j].x, xv[j].y, xv[j].z, xv[j].w};
            float gg[4];
            rows_quad_g(gv[j], gg);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float w = gg[e] * __builtin_amdgcn_exp2f(__builtin_fmaf(-o[e], g.c1, bound[e]) + hi[j][e & 1]);
                const float v = __builtin_amdgcn_exp2f(__builtin_fmaf(x[e], g.c1, -bound[e]));
                wt[tile_index(j, e)] = use_m ? w : 0.0f;
                et[tile_index(j, e)] = use_k ? v : 0.0f;
            }
        }
        if (s + 1 < n_chunks)
            request(bx * g.pxl + s + 1);
        __syncthreads();
        floatx4 sum[2][2];
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
                sum[mt][kt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float wa[2][4], xa[2][4];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int at = (h * 16 + lr) * TP + wave * 64 + 16 * lq + 4 * i;
                const float4 w = *reinterpret_cast<const float4 *>(wt + at), x = *reinterpret_cast<const float4 *>(et + at);
                wa[h][0] = w.x; wa[h][1] = w.y; wa[h][2] = w.z; wa[h][3] = w.w;
                xa[h][0] = x.x; xa[h][1] = x.y; xa[h][2] = x.z; xa[h][3] = x.w;
            }
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int mt = 0; mt < 2; ++mt)
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt)
                        sum[mt][kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[kt][c], wa[mt][c], sum[mt][kt], 0, 0, 0);
        }
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int v = 0; v < 4; ++v)   // times 2^(os_mk - mo_m), as mex_grads_rows_kernel adds them
                    total[mt][kt][v] = rows_sum(total[mt][kt][v], rows_product(sum[mt][kt][v], eov[mt][kt][v]));
    }
    __syncthreads();                   // (odd_sh is in place)
    int late[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        late[r] = __builtin_amdgcn_readfirstlane(wide_sh[r] | odd_sh[r]) != 0 ? kLateOffsets : 0;
    if (!__builtin_amdgcn_readfirstlane(wide_sh[wave] | odd_sh[wave])) {
        // partial sums: a lane's are four neighbouring patch elements of an instance
        float *dst = g.partial + ((size_t)bx * 4 + wave) * g.M * g.K;
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                const int m = mg * GM_TM + mt * 16 + lr, k = k0 + kt * 16 + 4 * lq;
                if (m >= g.M || k >= g.K)
                    continue;
                const floatx4 &t = total[mt][kt];
                float *at = reinterpret_cast<float *>(reinterpret_cast<char *>(dst) + 4 * ((unsigned)m * g.K + k));
                if ((g.K & 3) == 0) {
                    *reinterpret_cast<float4 *>(at) = make_float4(t[0], t[1], t[2], t[3]);
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (k + v < g.K)
                            at[v] = t[v];
                }
            }
    }
#if defined(__HIP_DEVICE_COMPILE__)
    if ((late[0] | late[1] | late[2] | late[3]) != 0)
        rows_terms<32>(bx, n_chunks, k0, mg, mg + 1, nullptr, 1, make_int4(late[0], late[1], late[2], late[3]));
#endif
}

// dOff[r,m,k] = sum over pixel chunks, in a fixed order (reproducible): a workgroup takes 32 consecutive elements,
// its 8 groups of 32 threads each sum every 8th chunk in chunk order, and the 8 sums are added in group order.
__global__ __launch_bounds__(256) void mex_grad_offsets_finish_kernel(const float *__restrict__ partial, long long n,
                                                                     int chunks, float *__restrict__ doff)
{
    __shared__ float sm[8][32];
    const int e = threadIdx.x & 31, sub = threadIdx.x >> 5;
    for (long long i0 = (long long)blockIdx.x * 32; i0 < n; i0 += (long long)gridDim.x * 32) {
        const long long i = i0 + e;
        float s = 0.0f;
        if (i < n)
            for (int c = sub; c < chunks; c += 8)
                s += partial[(size_t)c * n + i];
        sm[sub][e] = s;
        __syncthreads();
        if (sub == 0 && i < n) {
            float t = sm[0][e];
#pragma unroll
            for (int j = 1; j < 8; ++j)
                t += sm[j][e];
            doff[i] = t;
        }
        __syncthreads();
    }
}

// One wave per (region, instance) row: n = o - logsumexp(o)  (python/simnets/keras.py:155-160).
__global__ __launch_bounds__(256) void mex_normalize_rows_kernel(const float *__restrict__ src, long long rows, int K,
                                                                float *__restrict__ dst)
{
    const int lane = threadIdx.x & 63;
    const long long row = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows)
        return;
    const float *s = src + (size_t)row * K;
    float mxv = -INFINITY;
    for (int k = lane; k < K; k += 64)
        mxv = fmaxf(mxv, s[k]);
    for (int d = 32; d > 0; d >>= 1)
        mxv = fmaxf(mxv, __shfl_xor(mxv, d, 64));
    if (!(fabsf(mxv) < INFINITY))
        mxv = 0.0f;
    float sum = 0.0f;
    for (int k = lane; k < K; k += 64)
        sum += mex_exp_term(s[k] - mxv);   // (the pack kernel's arithmetic: both write the same normalised rows)
    for (int d = 32; d > 0; d >>= 1)
        sum += __shfl_xor(sum, d, 64);
    const float lse = mex_lse_of(sum, mxv);
    for (int k = lane; k < K; k += 64)
        dst[(size_t)row * K + k] = s[k] - lse;
}

// Chain rule through the normalisation n = o - logsumexp(o): d/do_j = G_j - exp(n_j) * sum_k G_k, in place.
__global__ __launch_bounds__(256) void mex_normalize_rows_backward_kernel(const float *__restrict__ normalized,
                                                                         long long rows, int K, float *__restrict__ grad)
{
    const int lane = threadIdx.x & 63;
    const long long row = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows)
        return;
    float *gr = grad + (size_t)row * K;
    const float *n = normalized + (size_t)row * K;
    float sum = 0.0f;
    for (int k = lane; k < K; k += 64)
        sum += gr[k];
    for (int d = 32; d > 0; d >>= 1)
        sum += __shfl_xor(sum, d, 64);
    for (int k = lane; k < K; k += 64)
        gr[k] -= expf(n[k]) * sum;
}

// Elements lane, lane + 64, ... of one row of the offsets gradient from its partial sums (eight interleaved sums in
// chunk order, added in order), E elements at a time; returns the lane's share of the row sum (in element order).
// (NB: rounds of eight chunks requested together; the additions keep the order of one round at a time)
template <int E, int STRIDE = 64, int NB = 1>
__device__ __forceinline__ float finish_long_row(const float *__restrict__ pr, float *__restrict__ gr, long long n,
                                                 int chunks, int K, int lane)
{
    float sum = 0.0f;
    for (int k0 = lane; k0 < K; k0 += STRIDE * E) {
        float s8[E][8];
#pragma unroll
        for (int e = 0; e < E; ++e)
#pragma unroll
            for (int j = 0; j < 8; ++j)
                s8[e][j] = 0.0f;
        for (int c0 = 0; c0 < chunks; c0 += 8 * NB) {
            // all requests first, those past the last chunk or the row's end on a valid address (a load inside the
            // condition would be waited for before the next one is issued)
            float v[NB][E][8];
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int e = 0; e < E; ++e)
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        v[b][e][j] = pr[(size_t)min(c0 + 8 * b + j, chunks - 1) * n + min(k0 + STRIDE * e, K - 1)];
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int e = 0; e < E; ++e)
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        s8[e][j] = c0 + 8 * b + j < chunks ? s8[e][j] + v[b][e][j] : s8[e][j];
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            float t = s8[e][0];
#pragma unroll
            for (int j = 1; j < 8; ++j)
                t += s8[e][j];
            if (k0 + STRIDE * e < K) {
                gr[k0 + STRIDE * e] = t;
                sum += t;
            }
        }
    }
    return sum;
}

// Both of the above for short rows, one wave per (region, instance) row: element k of the row is the sum of its
// partial sums in the order of mex_grad_offsets_finish_kernel (eight interleaved sums in chunk order, added in
// order), then, if `normalized` is given, the chain rule of mex_normalize_rows_backward_kernel with the same
// reduction over the row: the same values as the two launches, in one.
constexpr int kFinishRowsMaxK = 1024;
__global__ __launch_bounds__(256) void mex_grad_offsets_finish_rows_kernel(const float *__restrict__ partial, long long n,
                                                                          int chunks, long long rows, int K,
                                                                          const float *__restrict__ normalized,
                                                                          float *__restrict__ doff)
{
    const int lane = threadIdx.x & 63;
    const long long row = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows)
        return;
    float *gr = doff + (size_t)row * K;
    const float *pr = partial + (size_t)row * K;
    float sum = 0.0f;
    if (K <= 32 && (K & 3) == 0) {
        // short rows of whole 16-byte pieces: lane (q, j) = (lane & 7, lane >> 3) takes piece q (elements 4 q ... 4 q + 3)
        // of the chunks j, j + 8, ... - the interleaved sum j -, eight of them requested at a time; lane (q, 0) then
        // adds the eight sums in order.  The values are those of the loops below.
        const int Kq = K >> 2, q = lane & 7, j = lane >> 3, qc = min(q, Kq - 1);
        const long long n4 = n >> 2;
        const float4 *pr4 = reinterpret_cast<const float4 *>(pr) + qc;
        float4 sj = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        for (int c0 = j; c0 < chunks; c0 += 64) {
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                v[u] = pr4[(size_t)min(c0 + 8 * u, chunks - 1) * n4];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (c0 + 8 * u < chunks) {
                    sj.x += v[u].x; sj.y += v[u].y; sj.z += v[u].z; sj.w += v[u].w;
                }
        }
        float4 t4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
            const float4 val = make_float4(__shfl(sj.x, q + 8 * jj, 64), __shfl(sj.y, q + 8 * jj, 64),
                                           __shfl(sj.z, q + 8 * jj, 64), __shfl(sj.w, q + 8 * jj, 64));
            if (jj == 0)
                t4 = val;
            else {
                t4.x += val.x; t4.y += val.y; t4.z += val.z; t4.w += val.w;
            }
        }
        if (normalized == nullptr) {
            if (j == 0 && q < Kq) {
                if ((reinterpret_cast<uintptr_t>(gr) & 15) == 0)
                    reinterpret_cast<float4 *>(gr)[q] = t4;
                else {
                    gr[4 * q] = t4.x; gr[4 * q + 1] = t4.y; gr[4 * q + 2] = t4.z; gr[4 * q + 3] = t4.w;
                }
            }
            return;
        }
        // element k to lane k (it lives in lane k / 4), then the row sum and the chain rule as below
        const int k = lane & 31;
        const float a0 = __shfl(t4.x, k >> 2, 64), a1 = __shfl(t4.y, k >> 2, 64), a2 = __shfl(t4.z, k >> 2, 64),
                    a3 = __shfl(t4.w, k >> 2, 64);
        const float t = (k & 3) == 0 ? a0 : (k & 3) == 1 ? a1 : (k & 3) == 2 ? a2 : a3;
        const bool owner = lane < K;
        sum = owner ? t : 0.0f;
        for (int d = 32; d > 0; d >>= 1)
            sum += __shfl_xor(sum, d, 64);
        if (owner)
            gr[k] = t - expf(normalized[(size_t)row * K + k]) * sum;
        return;
    }
    if (K <= 32) {
        // rows shorter than a wave: the lanes form 64 / Kp groups (Kp = 8, 16 or 32 >= K) that each take 8 / groups
        // of the eight interleaved sums, four rounds of chunks requested at a time; every lane then adds the eight
        // sums in order (read from the lanes that hold them), so the values are those of the loop below
        const int lg = K <= 8 ? 3 : K <= 16 ? 4 : 5, Kp = 1 << lg;
        const int per = 8 >> (6 - lg);               // sums per group: 1, 2 or 4
        const int gi = lane >> lg, k = lane & (Kp - 1), kc = min(k, K - 1);
        float sj[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int c0 = 0; c0 < chunks; c0 += 32) {
            float v[4][4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (i < per)
                        v[u][i] = pr[(size_t)min(c0 + 8 * u + gi * per + i, chunks - 1) * n + kc];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (i < per && c0 + 8 * u + gi * per + i < chunks)
                        sj[i] += v[u][i];
        }
        float t = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int i = j & (per - 1), src = ((j >> (lg - 3)) << lg) + k;   // sum j lives in group j / per, slot j % per
            const float mine = i == 0 ? sj[0] : i == 1 ? sj[1] : i == 2 ? sj[2] : sj[3];
            const float val = __shfl(mine, src, 64);
            t = j == 0 ? val : t + val;
        }
        const bool owner = gi == 0 && k < K;
        if (owner)
            gr[k] = t;
        if (normalized == nullptr)
            return;
        sum = owner ? t : 0.0f;
        for (int d = 32; d > 0; d >>= 1)
            sum += __shfl_xor(sum, d, 64);
        if (owner)
            gr[k] = t - expf(normalized[(size_t)row * K + k]) * sum;
        return;
    }
    // up to four elements of the row per lane at a time (64 apart): 8 requests each in flight
    if (K <= 64)
        sum = finish_long_row<1>(pr, gr, n, chunks, K, lane);
    else if (K <= 128)
        sum = finish_long_row<2>(pr, gr, n, chunks, K, lane);
    else
        sum = finish_long_row<4>(pr, gr, n, chunks, K, lane);
    if (normalized == nullptr)
        return;
    for (int d = 32; d > 0; d >>= 1)
        sum += __shfl_xor(sum, d, 64);
    const float *nr = normalized + (size_t)row * K;
    for (int k = lane; k < K; k += 64)
        gr[k] -= expf(nr[k]) * sum;   // reads back what this lane stored above
}

// The same for few rows of many chunks: one workgroup of 1024 per row, 128 threads on each of the eight interleaved sums,
// eight chunks of two elements requested at a time.  With a wave per row the chunks are one chain of round trips to
// memory (32 rows of 144 elements, 200 chunks: eight workgroups, 25 round trips, 21.7 us; here four, 6.2 us); with
// many rows the waves of others hide it, and with few chunks there is no chain.  Same values: the additions, the row
// sum's included, keep their order.
__global__ __launch_bounds__(1024) void mex_grad_offsets_finish_tall_rows_kernel(const float *__restrict__ partial,
                                                                                long long n, int chunks, int K,
                                                                                const float *__restrict__ normalized,
                                                                                float *__restrict__ doff)
{
    __shared__ float sm[8 * kFinishRowsMaxK];
    const long long row = blockIdx.x;
    const float *pr = partial + (size_t)row * K;
    float *gr = doff + (size_t)row * K;
    const int tid = threadIdx.x, j = tid >> 7;
    for (int k0 = tid & 127; k0 < K; k0 += 256) {
        float s2[2] = {0.0f, 0.0f};
        for (int c0 = j; c0 < chunks; c0 += 64) {
            float v[8][2];
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    v[u][e] = pr[(size_t)min(c0 + 8 * u, chunks - 1) * n + min(k0 + 128 * e, K - 1)];
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    s2[e] = c0 + 8 * u < chunks ? s2[e] + v[u][e] : s2[e];
        }
#pragma unroll
        for (int e = 0; e < 2; ++e)
            if (k0 + 128 * e < K)
                sm[j * K + k0 + 128 * e] = s2[e];
    }
    __syncthreads();
    float t = 0.0f;
    if (tid < K) {   // K <= kFinishRowsMaxK = the workgroup's threads
        t = sm[tid];
#pragma unroll
        for (int i = 1; i < 8; ++i)
            t += sm[i * K + tid];
        sm[tid] = t;
        if (normalized == nullptr)
            gr[tid] = t;
    }
    if (normalized == nullptr)
        return;
    __syncthreads();
    float sum = 0.0f;
    for (int k = tid & 63; k < K; k += 64)
        sum += sm[k];
    for (int d = 32; d > 0; d >>= 1)
        sum += __shfl_xor(sum, d, 64);
    if (tid < K)
        gr[tid] = t - expf(normalized[(size_t)row * K + tid]) * sum;
}

// The same for few long rows: one workgroup per row, the four waves split its
// elements (thread t takes t, t + 256, ...), the row sum of the chain rule goes through LDS.
__global__ __launch_bounds__(256) void mex_grad_offsets_finish_wide_rows_kernel(const float *__restrict__ partial,
                                                                               long long n, int chunks, int K,
                                                                               const float *__restrict__ normalized,
                                                                               float *__restrict__ doff)
{
    __shared__ float ws[4];
    const long long row = blockIdx.x;
    float *gr = doff + (size_t)row * K;
    const float *pr = partial + (size_t)row * K;
    const int tid = threadIdx.x;
    float sum = K <= 256 ? finish_long_row<1, 256, 4>(pr, gr, n, chunks, K, tid)
                         : (K <= 512 ? finish_long_row<2, 256, 2>(pr, gr, n, chunks, K, tid)
                                     : finish_long_row<4, 256, 1>(pr, gr, n, chunks, K, tid));
    if (normalized == nullptr)
        return;
    for (int d = 32; d > 0; d >>= 1)
        sum += __shfl_xor(sum, d, 64);
    if ((tid & 63) == 0)
        ws[tid >> 6] = sum;
    __syncthreads();
    sum = (ws[0] + ws[1]) + (ws[2] + ws[3]);
    const float *nr = normalized + (size_t)row * K;
    for (int k = tid; k < K; k += 256)
        gr[k] -= expf(nr[k]) * sum;   // reads back what this thread stored above
}

// What is left after mex_grads_rows_kernel, in one launch: the first `rows` workgroups take a row of the offsets gradient each
// (K a multiple of 4, at most kFinishRowsMaxK), the others the sums of the input gradient's splits (mex_sum_splits4_kernel).
// K / 4 threads hold four elements of the row each, 1024 / K groups of them every so many chunks; the groups' sums are
// added in order, then the chain rule through the normalisation, if `normalized` is given.  Eight chunks are requested at
// a time.  512 images, 64 channels of 8 x 8, 128 instances, two splits: 10.4 us in two launches, 8.2 in one; 32 channels of 16 x
// 16, 512 partial sums of 256 rows: 9.4 us with a wave to a row, 5.6.
__global__ __launch_bounds__(256) void mex_grads_finish_kernel(const float *__restrict__ partial, long long n, int chunks,
                                                              int rows, int K, const float *__restrict__ normalized,
                                                              float *__restrict__ doff, const float4 *__restrict__ parts,
                                                              long long n4, int splits, float4 *__restrict__ dx)
{
    __shared__ __attribute__((aligned(16))) float4 sm[256];
    __shared__ float wave_sum[4];
    const int tid = threadIdx.x;
    if ((int)blockIdx.x >= rows) {
        sum_splits4(parts, n4, splits, dx, (long long)(blockIdx.x - rows) * 256 + tid);
        return;
    }
    const int row = blockIdx.x, Kq = K >> 2, G = 256 / Kq;
    const int grp = tid / Kq, q = tid - grp * Kq;
    const bool first = grp == 0;
    float nv[4];
    if (normalized != nullptr)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            nv[e] = normalized[(size_t)row * K + 4 * q + e];
    float4 t = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (grp < G) {
        const float4 *src = reinterpret_cast<const float4 *>(partial + (size_t)row * K) + q;
        for (int c0 = grp; c0 < chunks; c0 += 8 * G) {
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)   // (behind the last: this group's first)
                v[u] = src[(size_t)(c0 + u * G < chunks ? c0 + u * G : grp) * (n >> 2)];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (c0 + u * G < chunks) {
                    t.x += v[u].x; t.y += v[u].y; t.z += v[u].z; t.w += v[u].w;
                }
        }
    }
    sm[tid] = t;
    __syncthreads();
    float sum = 0.0f;
    if (first) {
        for (int j = 1; j < min(G, chunks); ++j) {
            const float4 v = sm[j * Kq + q];
            t.x += v.x; t.y += v.y; t.z += v.z; t.w += v.w;
        }
        sum = (t.x + t.y) + (t.z + t.w);
    }
    float v[4] = {t.x, t.y, t.z, t.w};
    if (normalized != nullptr) {
        for (int d = 32; d > 0; d >>= 1)
            sum += __shfl_xor(sum, d, 64);
        if ((tid & 63) == 0)
            wave_sum[tid >> 6] = sum;
        __syncthreads();
        sum = (wave_sum[0] + wave_sum[1]) + (wave_sum[2] + wave_sum[3]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            v[e] -= expf(nv[e]) * sum;
    }
    if (!first)
        return;
    float *dst = doff + (size_t)row * K + 4 * q;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        dst[e] = v[e];
}

// Few instances over long patches on few pixels (a network's classifier head: 10 instances x 512 channels on one
// pixel per image): the tiled kernels above would run a handful of workgroups in long serial chains, in three
// launches.  Here a thread owns one patch element k (a workgroup spans K) and keeps the region's offsets for that
// element in registers; the workgroup walks its share of the pixels, four at a time (their loads in flight
// together), and forms every term as the reference does (mex_term: either epsilon, any offsets range): summed over
// the instances it is the input gradient of (pixel, k), summed over the pixels - in registers - the offsets gradient
// of (instance, k).  No LDS, no barriers; one partial sum [M][K] per workgroup for the finish kernel.
// A chain of round trips: 512 pixels of 512 elements, 10 instances, in 64 workgroups of two rounds 13.7 us + 6.5 to finish, in 128 of one 9.8 +
// 7.1 (with four times the requests in flight).
constexpr int kHeadMaxM = 16, kHeadPixels = 4;
template <int MH, bool FINITE>
__global__ __launch_bounds__(1024) void mex_grad_head_kernel(const MexGradArgs ga, int wgs_per_region, int want_input,
                                                             int want_offsets)
{
    static_assert(MH <= 16, "one lane per instance in the load of the gradients and outputs");
    const MexKernelArgs &a = ga.k;
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x / wgs_per_region, wg = blockIdx.x - r * wgs_per_region;
    const int k = threadIdx.x;
    const bool kv = k < a.K;
    const int kk = kv ? k : 0;
    const int bhw = a.bh * a.bw;
    const int dc = kk / bhw, rem = kk - dc * bhw, dh = rem / a.bw, dw = rem - dh * a.bw;
    float of[MH], acc[MH];
#pragma unroll
    for (int m = 0; m < MH; ++m) {
        of[m] = ga.off[((size_t)r * a.M + min(m, a.M - 1)) * a.K + kk];
        acc[m] = 0.0f;
    }
    const size_t plane = (size_t)a.Co * a.Ho * a.Wo, gplane = pooled_g_plane(ga, plane);
    const int ml = min(lane & 15, a.M - 1);
    for (int s0 = wg * kHeadPixels; s0 < a.slots; s0 += wgs_per_region * kHeadPixels) {
        float x[kHeadPixels], go[kHeadPixels];
        int io[kHeadPixels];
        bool valid[kHeadPixels];
        size_t img[kHeadPixels], col[kHeadPixels];
#pragma unroll
        for (int p = 0; p < kHeadPixels; ++p) {
            const int slot = s0 + p;
            const PixelRef px = locate(a, r, min(slot, a.slots - 1));   // (the same pixel for the whole workgroup)
            valid[p] = slot < a.slots && px.out_off >= 0;
            const int ci = px.ci0 + dc, hi = px.hi0 + dh, wi = px.wi0 + dw;
            const bool ok = kv && mex_inside(a, ci, hi, wi);
            io[p] = ok ? (ci * a.H + hi) * a.W + wi : -1;
            img[p] = (size_t)px.b * a.C * a.H * a.W;
            // (loads on addresses that are always valid, the choice made afterwards: a load inside a condition is
            // waited for before the next one is issued)
            const float xv = a.in[img[p] + (ok ? io[p] : 0)];
            x[p] = ok ? xv : a.oob;
            const int oo = valid[p] ? px.out_off : 0;
            // every instance's gradient (lanes 0 ... 15) and output value (lanes 16 ... 31) through one load, read back
            // lane by lane below
            const float *src = (lane & 16) ? ga.out + ((size_t)px.b * a.M + ml) * plane + oo
                                           : ga.g + ((size_t)px.b * a.M + ml) * gplane + pooled_g_offset(ga, oo);
            go[p] = *src;
            col[p] = (size_t)px.b * a.K * plane + oo;
        }
        // Straight-line arithmetic: instances past the last one repeat it with a zero gradient (their sums are never
        // stored), threads past the last patch element compute on the out-of-bounds value (nothing of theirs is
        // stored either); only an empty pixel slot is skipped.
#pragma unroll
        for (int p = 0; p < kHeadPixels; ++p) {
            if (!valid[p])
                continue;
            float dxa = 0.0f;
#pragma unroll
            for (int m = 0; m < MH; ++m) {
                float gm = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, go[p]), m));
                const float om = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, go[p]), 16 + m));
                gm = m < a.M ? gm : 0.0f;
                const float e = mex_term(x[p] + of[m], om, gm, a.c1, a.c0, FINITE);
                dxa += e;
                acc[m] += e;
            }
            if (want_input && io[p] >= 0) {
                if (ga.overlap)
                    ga.col[col[p] + k * plane] = dxa;
                else
                    ga.dx[img[p] + io[p]] = dxa;
            }
        }
    }
    if (!want_offsets || !kv)
        return;
    float *part = ga.partial + ((size_t)wg * a.R + r) * a.M * a.K + k;
#pragma unroll
    for (int m = 0; m < MH; ++m)
        if (m < a.M)
            part[(size_t)m * a.K] = acc[m];
}

__global__ void mex_fill_zero_kernel(float *__restrict__ p, long long n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        p[i] = 0.0f;
}

struct MexGradTiling {
    int pxl, cpr_offsets;
    bool head;           // few instances over long patches on few pixels: mex_grad_head_kernel, both gradients
    int head_wgs;        // ... with this many workgroups per region (= partial sums per region)
    bool mfma;           // finite epsilon: the matrix-core kernels, fed by the forward pass's packed offsets
    size_t norm_bytes, partial_bytes, packed_bytes;
    bool overlap;        // input gradient: patches overlap
    size_t col_bytes;    // ... and their per-patch gradients pass through a [B][K][Co*Ho*Wo] buffer
    bool tiles_input;    // patches tile the input exactly: every element is written by exactly one patch
    int msplit, mg_per_split;  // input gradient, matrix form: instance groups split over gridDim.z workgroups
    size_t split_bytes;  // ... whose partial gradients [split][input] are added by mex_sum_splits_kernel
    // factor buffers of mex_grad_factors_kernel: used when a matrix kernel would otherwise form the same factors
    // in several workgroups (more than one tile along the dimension it does not contract)
    bool factors_input, factors_offsets;
    int slots_pad, Mp, Kp;
    size_t factor_bytes;
    // the row-wise kernel (mex_grads_rows_kernel): the layer qualifies (the pointers are checked at the launch), and its
    // tiling
    bool rows;
    int rows_ksub;                        // 16 * ksub patch elements per workgroup
    int rows_msplit, rows_mg_per_split;   // ... and the split of its instance groups
    int rows_pxl, rows_cpr;               // chunks per workgroup, workgroups along the pixels
    bool rows_apart;                      // the offsets gradient in a kernel of its own: mex_grad_offsets_rows_kernel
    int offsets_pxl, offsets_cpr;         // chunks per workgroup and workgroups along the pixels of either's partial sums
};

inline int log2_exact(int v)   // log2 of a power of two, -1 otherwise
{
    int l = 0;
    while ((1 << l) < v)
        ++l;
    return v > 0 && (1 << l) == v ? l : -1;
}

// 2 x 2 unshared offsets over whole-channel patches on a map with power-of-two sides: see the row-wise kernels.
// A chunk of 256 pixels must be whole images or an even number of whole rows (width <= 128), so that it holds
// exactly the 64 slots [64 chunk, 64 chunk + 64) of each of the four regions; a 16-byte piece lies in one row
// (width 4 and more) or is a window (width 2).
bool rows_geometry(const MexPlan &p)
{
    const simnets_mex_dims &d = p.d;
    return std::isfinite(p.epsilon) && p.use_unshared && d.offsets_c == 1 && d.offsets_h == 2 && d.offsets_w == 2 &&
           d.channels_out == 1 && d.block_c == p.C && d.block_h == 1 && d.block_w == 1 && d.stride_h == 1 &&
           d.stride_w == 1 && d.pad_c == 0 && d.pad_h == 0 && d.pad_w == 0 && d.height_out == p.H &&
           d.width_out == p.W && log2_exact(p.H) >= 1 && log2_exact(p.W) >= 1 && p.W <= 128 &&
           d.region_size == (p.H / 2) * (p.W / 2) && (long long)p.B * p.H * p.W <= 0x3fffffffLL &&
           // (32-bit offsets in bytes: of an image or a chunk's images, and of the packed offsets)
           std::max<long long>(256, 1LL * p.H * p.W) * std::max<long long>(d.M, d.K) < (1LL << 29) &&
           4LL * (d.M + GM_TM - 1) / GM_TM * GM_TM * d.K < (1LL << 29);
}

MexGradTiling mex_grad_tiling(const MexPlan &p)
{
    const simnets_mex_dims &d = p.d;
    MexGradTiling t;
    const long long slots = (long long)p.B * d.region_size;
    t.mfma = std::isfinite(p.epsilon);
    const long long mk = t.mfma ? 4LL * ((d.M + GOM_MT - 1) / GOM_MT) * ((d.K + GOM_KT - 1) / GOM_KT)
                                : (long long)((d.M + GO_MT - 1) / GO_MT) * ((d.K + GO_KT - 1) / GO_KT);
    auto waves = [&](int pxl) { return d.num_regions * ((slots + 64LL * pxl - 1) / (64LL * pxl)) * mk; };
    t.pxl = 16;
    while (t.pxl > 1 && waves(t.pxl) < (t.mfma ? 2048 : 4096))
        t.pxl >>= 1;
    t.cpr_offsets = (int)((slots + 64LL * t.pxl - 1) / (64LL * t.pxl));
    const size_t rmk = (size_t)d.num_regions * d.M * d.K * sizeof(float);
    t.norm_bytes = p.normalize_offsets ? align_up(rmk, 256) : 0;
    t.partial_bytes = align_up(rmk * t.cpr_offsets, 256);
    t.packed_bytes = t.mfma ? mex_packed_bytes(p, GM_TM, (d.M + GM_TM - 1) / GM_TM) : 0;
    t.overlap = (d.block_c > d.stride_c && d.channels_out > 1) || (d.block_h > d.stride_h && d.height_out > 1) ||
                (d.block_w > d.stride_w && d.width_out > 1);
    t.col_bytes = t.overlap ? align_up((size_t)p.B * d.channels_out * d.height_out * d.width_out * d.K * sizeof(float),
                                       256) : 0;
    t.tiles_input = d.pad_c == 0 && d.pad_h == 0 && d.pad_w == 0 && d.stride_c == d.block_c &&
                    d.stride_h == d.block_h && d.stride_w == d.block_w && d.channels_out * d.block_c == p.C &&
                    d.height_out * d.block_h == p.H && d.width_out * d.block_w == p.W;
    // Few pixels and many instances (deep layers on small maps): a workgroup would walk all instance groups alone
    // while most of the chip idles.  Then the groups are split over up to 8 workgroups (two groups each at least)
    // until the launch has about two workgroups per compute unit.
    t.msplit = 1;
    const int n_mg = (d.M + GM_TM - 1) / GM_TM;
    const long long wgs = (long long)d.num_regions * ((slots + 63) / 64) * ((d.K + GM_KT - 1) / GM_KT);
    if (t.mfma && t.tiles_input && wgs <= 256 && n_mg >= 4)
        t.msplit = (int)std::max<long long>(1, std::min<long long>(std::min(8, n_mg / 2), 512 / std::max<long long>(wgs, 1)));
    t.mg_per_split = (n_mg + t.msplit - 1) / t.msplit;
    t.msplit = (n_mg + t.mg_per_split - 1) / t.mg_per_split;
    t.split_bytes = t.msplit > 1 ? align_up((size_t)t.msplit * p.B * p.C * p.H * p.W * sizeof(float), 256) : 0;
    t.slots_pad = (int)((slots + 63) / 64 * 64);
    t.Mp = n_mg * GM_TM;
    t.Kp = (d.K + 31) / 32 * 32;
    const int k_tiles = (d.K + GM_KT - 1) / GM_KT, m_tiles = (d.M + GOM_MT - 1) / GOM_MT;
    // (the extra launch and the round trip through memory cost about 10 us: measured to pay from 4 tiles of patch
    // elements and 128 instances on for the input gradient and from 16 tiles on for the offsets gradient)
    t.factors_input = t.mfma && k_tiles >= 4 && d.M >= 128;
    t.factors_offsets = t.mfma && m_tiles * ((d.K + GOM_KT - 1) / GOM_KT) >= 16;
    t.factor_bytes = align_up((size_t)d.num_regions * t.slots_pad * ((size_t)t.Mp + t.Kp) * sizeof(float), 256);
    // The head kernel: terms few enough for one exponential each (a classifier head has 512 x 10 x 512 of them)
    t.head = d.M <= kHeadMaxM && d.K >= 64 && d.K <= 1024 && slots >= 1 &&
             (long long)d.num_regions * slots * d.M * d.K <= (16LL << 20) && (long long)p.C * p.H * p.W <= 0x7fffffffLL;
    // (a round of pixels per workgroup, at most 128 partial sums per region for the finish kernel)
    t.head_wgs = (int)std::max<long long>(1, std::min<long long>((slots + kHeadPixels - 1) / kHeadPixels, std::max(1, 128 / d.num_regions)));
    if (t.head)
        t.partial_bytes = std::max(t.partial_bytes, align_up(rmk * t.head_wgs, 256));
    t.rows = rows_geometry(p);
    t.rows_ksub = 1; t.rows_msplit = 1; t.rows_mg_per_split = n_mg; t.rows_pxl = 1; t.rows_cpr = 0;
    t.rows_apart = false; t.offsets_pxl = 1; t.offsets_cpr = 0;
    if (t.rows) {
        const long long chunks = t.slots_pad / 64;
        // Row-wise kernels, about two workgroups per compute unit at least: tiles of patch elements (each reads all of `out` and `g`), the
        // split of the instance groups (of the input gradient's sums), and as many chunks to a workgroup as that allows (each
        // writes a partial sum of its tile).
        // 32 patch elements to a workgroup, or 16 if 32 leave the chip short of two workgroups to a compute unit and 16 leave
        // it less so, whatever the split of the instance groups, or if 32 need a split where 16 do not (512 images, 64 channels of 8 x 8, 128
        // instances: 27.4 + 8.2 us with two splits and their sums, 28.0 + 5.1 without)
        auto split_of = [&](long long wgs) {
            return wgs >= 512 || n_mg < 4 ? 1LL : std::max<long long>(1, std::min<long long>(std::min(8, n_mg / 2), 512 / std::max<long long>(wgs, 1)));
        };
        const long long wide = chunks * ((d.K + 31) / 32), narrow = chunks * ((d.K + 15) / 16);
        const long long wide_wgs = wide * split_of(wide);
        t.rows_ksub = d.K <= 16 || (wide_wgs < 512 && narrow * split_of(narrow) > wide_wgs) || (wide < 512 && narrow >= 512) ? 1 : 2;
        const long long tiles = (d.K + 16 * t.rows_ksub - 1) / (16 * t.rows_ksub);
        t.rows_msplit = (int)split_of(chunks * tiles);
        t.rows_mg_per_split = (n_mg + t.rows_msplit - 1) / t.rows_msplit;
        t.rows_msplit = (n_mg + t.rows_mg_per_split - 1) / t.rows_mg_per_split;
        if (t.rows_msplit > 1)
            t.split_bytes = std::max(t.split_bytes, align_up((size_t)t.rows_msplit * p.B * p.C * p.H * p.W * sizeof(float), 256));
        t.rows_pxl = 16;
        while (t.rows_pxl > 1 && (chunks + t.rows_pxl - 1) / t.rows_pxl * tiles < 512)
            t.rows_pxl >>= 1;
        t.rows_cpr = (int)((chunks + t.rows_pxl - 1) / t.rows_pxl);
        t.offsets_pxl = t.rows_pxl;
        // The two gradients in a kernel each: W is formed twice, but the offsets' sums stay in registers and partial sums are fewer.
        // Several tiles of patch elements, so that `out` and `g` are read several times either way, and either several chunks to a
        // workgroup or many terms.  Both gradients, in one kernel and in two, and the offsets' alone (us): 512 x 96 x 16 x 16 -> 192 262,
        // 242; 177, 134.  256 x 128 x 16 x 16 -> 256 190, 162; 123, 87.  1024 x 64 x 16 x 16 -> 64 130, 110; 76, 53.  2048 x 128 x 4 x 4 -> 512 181, 162;
        // 135, 90.  Left in one: 512 x 48 x 16 x 16 -> 96 79, 83 (half of the second tile empty), 256 x 128 x 8 x 8 -> 512 106, 109.  A single tile
        // and many groups, whose partial sums are many: 2048 x 32 x 8 x 8 -> 256 118, 117; 94, 65; with fewer groups
        // 512 x 32 x 32 x 32 -> 128 243, 300.  16 elements fill half a tile: left in one.
        t.rows_apart = p.W > 2 && (d.K > 48 ? t.rows_pxl > 1 || 256.0 * chunks * d.M * d.K >= 0x1p31 : d.K > 16 && d.K <= 32 && n_mg >= 8);
        if (t.rows_apart) {
            t.offsets_pxl = 16;
            while (t.offsets_pxl > 1 && (chunks + t.offsets_pxl - 1) / t.offsets_pxl * ((d.K + 31) / 32) * n_mg < 512)
                t.offsets_pxl >>= 1;
        }
        t.offsets_cpr = (int)((chunks + t.offsets_pxl - 1) / t.offsets_pxl);
        t.partial_bytes = std::max(t.partial_bytes, align_up(rmk * t.offsets_cpr, 256));
    }
    return t;
}

// offsets as the forward op used them: the caller's, or their normalised copy in the workspace
int prepare_offsets(const MexPlan &p, const float *offsets, void *workspace, hipStream_t s, const float **used)
{
    *used = offsets;
    if (!p.normalize_offsets)
        return SIMNETS_OK;
    float *norm = reinterpret_cast<float *>(workspace);
    const long long rows = (long long)p.d.num_regions * p.d.M;
    hipLaunchKernelGGL(mex_normalize_rows_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, offsets, rows,
                       p.d.K, norm);
    *used = norm;
    return hipGetLastError() == hipSuccess ? SIMNETS_OK : SIMNETS_ERR_HIP;
}

// Launches mex_grad_factors_kernel into `buffers` and points ga at them (ga.k must hold the packed offsets).
int launch_factors(const MexPlan &p, const MexGradTiling &t, MexGradArgs &ga, void *buffers, hipStream_t s)
{
    ga.slots_pad = t.slots_pad; ga.Mp = t.Mp; ga.Kp = t.Kp;
    ga.wbuf = reinterpret_cast<float *>(buffers);
    ga.exbuf = ga.wbuf + (size_t)p.d.num_regions * t.slots_pad * t.Mp;
    MexGradArgs fa = ga;
    fa.cpr = t.slots_pad / 64;
    const long long gx = (long long)p.d.num_regions * fa.cpr;
    if (gx > 0x7fffffffLL)
        return SIMNETS_ERR_TOO_LARGE;
    const int gy = t.Mp / GM_TM + t.Kp / 32;
    if (gy > 65535)
        return SIMNETS_ERR_TOO_LARGE;
    if (gx > 0)
        hipLaunchKernelGGL(mex_grad_factors_kernel, dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, s, fa);
    return hipGetLastError() == hipSuccess ? SIMNETS_OK : SIMNETS_ERR_HIP;
}

}  // namespace

namespace {

// Scratch of a gradient call, in this order: normalised offsets | packed offsets | offsets-gradient partial sums |
// patch gradients of overlapping patches | partial input gradients of the instance split | factor buffers.
struct MexGradScratch {
    size_t norm, packed, partial, col, split, factors, total;
    bool use_factors;
};

MexGradScratch mex_grad_scratch(const MexGradTiling &t, bool want_input, bool want_offsets)
{
    MexGradScratch w;
    // both gradients in one call: the factors are formed once for the kernels that want them
    w.use_factors = (want_input && t.factors_input) || (want_offsets && t.factors_offsets);
    size_t at = 0;
    w.norm = at;    at += t.norm_bytes;
    w.packed = at;  at += t.packed_bytes;
    w.partial = at; at += want_offsets ? t.partial_bytes : 0;
    w.col = at;     at += want_input ? t.col_bytes : 0;
    w.split = at;   at += want_input ? t.split_bytes : 0;
    w.factors = at; at += w.use_factors ? t.factor_bytes : 0;
    w.total = at;
    return w;
}

}  // namespace

size_t mex_grads_workspace_bytes(const MexPlan &p, bool want_input, bool want_offsets)
{
    return mex_grad_scratch(mex_grad_tiling(p), want_input, want_offsets).total;
}

size_t mex_grad_input_workspace_bytes(const MexPlan &p) { return mex_grads_workspace_bytes(p, true, false); }

size_t mex_grad_offsets_workspace_bytes(const MexPlan &p) { return mex_grads_workspace_bytes(p, false, true); }

// Either gradient or both (a null pointer skips one).  The offsets as the forward op used them, their packed form
// and, where used, the factor buffers are prepared once and shared.
bool mex_grads_take_pooled(const MexPlan &p, const float *input, const float *output, const float *pooled_grad,
                           const float *input_grad)
{
    (void)input; (void)output; (void)pooled_grad; (void)input_grad;   // (any alignment: only the row-wise kernels care)
    // every kernel maps an output pixel to its window (pooled_g_offset): one output channel per instance and no
    // trailing row or column that the pooling dropped
    return p.d.channels_out == 1 && p.d.height_out % 2 == 0 && p.d.width_out % 2 == 0;
}

bool mex_grads_read_packed(const MexPlan &p)
{
    const MexGradTiling t = mex_grad_tiling(p);
    return t.mfma && !t.head;
}

int mex_grad_pack_launch(const MexPlan &p, const float *offsets, void *buffer, void *stream)
{
    MexPlan q = p;
    q.grad_pack = nullptr;
    MexPackTwin tw;
    float *norm;
    mex_grad_pack_layout(q, buffer, &tw, &norm);
    if (tw.offp == nullptr) {   // only the normalised copy is kept
        const float *used;
        return prepare_offsets(q, offsets, norm, reinterpret_cast<hipStream_t>(stream), &used);
    }
    MexKernelArgs a = mex_kernel_args(q);
    return mex_pack_offsets(q, offsets, GM_TM, tw.n_mgroups, buffer, &a, stream, nullptr, true, norm, true);
}

int mex_grads(const MexPlan &p, const float *input, const float *offsets, const float *output,
              const float *output_grad, float *input_grad, float *offsets_grad, void *workspace,
              size_t workspace_bytes, void *stream, bool grad_is_pooled, const void *saved)
{
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const bool want_input = input_grad != nullptr, want_offsets = offsets_grad != nullptr;
    const MexGradTiling t = mex_grad_tiling(p);
    const MexGradScratch w = mex_grad_scratch(t, want_input, want_offsets);
    if (workspace_bytes < w.total)
        return SIMNETS_ERR_WORKSPACE;
    const simnets_mex_dims &d = p.d;
    const long long n_in = (long long)p.B * p.C * p.H * p.W;
    const long long n_off = (long long)d.num_regions * d.M * d.K;
    if (p.B == 0) {  // an empty batch has an empty input gradient and a zero offsets gradient
        if (want_offsets) {
            hipLaunchKernelGGL(mex_fill_zero_kernel, dim3((unsigned)std::min<long long>((n_off + 255) / 256, 65535)),
                               dim3(256), 0, s, offsets_grad, n_off);
            return hipGetLastError() == hipSuccess ? SIMNETS_OK : SIMNETS_ERR_HIP;
        }
        return SIMNETS_OK;
    }
    if ((n_in + 255) / 256 > 0x7fffffffLL)
        return SIMNETS_ERR_TOO_LARGE;
    char *ws = reinterpret_cast<char *>(workspace);

    MexGradArgs ga;
    ga.k = mex_kernel_args(p);
    ga.k.in = input;
    // the offsets as the forward op used them: with the matrix kernels the pack launch below writes the normalised
    // copy as well, otherwise a launch of its own does
    const bool pack_normalizes = t.mfma && p.normalize_offsets;
    // ... or the forward call left them (and their packed form) in `saved`
    const bool packed_already = saved != nullptr && t.mfma;
    char *packed_at = ws + w.packed;
    float *norm_at = reinterpret_cast<float *>(ws + w.norm);
    if (packed_already) {
        MexPackTwin tw;
        packed_at = reinterpret_cast<char *>(const_cast<void *>(saved));
        mex_grad_pack_layout(p, packed_at, &tw, &norm_at);
    }
    int rc = SIMNETS_OK;
    if (pack_normalizes)
        ga.off = norm_at;
    else
        rc = prepare_offsets(p, offsets, ws + w.norm, s, &ga.off);
    if (rc)
        return rc;
    ga.out = output; ga.g = output_grad;
    ga.gpool = grad_is_pooled ? 1 : 0;
    ga.dx = input_grad;
    ga.partial = reinterpret_cast<float *>(ws + w.partial);
    ga.overlap = 0;
    ga.col = reinterpret_cast<float *>(ws + w.col);
    if (grad_is_pooled && !mex_grads_take_pooled(p, input, output, output_grad, input_grad))
        return SIMNETS_ERR_ALGO;   // (the callers ask first)
    if (t.head) {
        // one launch for both gradients, on the offsets as they are (or their normalised copy): nothing is packed
        if (pack_normalizes && !packed_already) {
            rc = prepare_offsets(p, offsets, ws + w.norm, s, &ga.off);
            if (rc)
                return rc;
        }
        ga.overlap = t.overlap ? 1 : 0;
        if (want_input && !t.overlap && !t.tiles_input) {
            hipLaunchKernelGGL(mex_fill_zero_kernel, dim3((unsigned)std::min<long long>((n_in + 255) / 256, 65535)),
                               dim3(256), 0, s, input_grad, n_in);
            if (hipGetLastError() != hipSuccess)
                return SIMNETS_ERR_HIP;
        }
        const dim3 grid((unsigned)(d.num_regions * t.head_wgs)), block((unsigned)((d.K + 63) / 64 * 64));
        const int wi = want_input ? 1 : 0, wo = want_offsets ? 1 : 0;
#define SIMNETS_HEAD_LAUNCH(MH)                                                                                      \
    if (t.mfma)                                                                                                      \
        hipLaunchKernelGGL((mex_grad_head_kernel<MH, true>), grid, block, 0, s, ga, t.head_wgs, wi, wo);              \
    else                                                                                                             \
        hipLaunchKernelGGL((mex_grad_head_kernel<MH, false>), grid, block, 0, s, ga, t.head_wgs, wi, wo)
        if (d.M <= 4) {
            SIMNETS_HEAD_LAUNCH(4);
        } else if (d.M <= 8) {
            SIMNETS_HEAD_LAUNCH(8);
        } else if (d.M <= 12) {
            SIMNETS_HEAD_LAUNCH(12);
        } else {
            SIMNETS_HEAD_LAUNCH(kHeadMaxM);
        }
#undef SIMNETS_HEAD_LAUNCH
        if (hipGetLastError() != hipSuccess)
            return SIMNETS_ERR_HIP;
        if (want_input && t.overlap) {
            hipLaunchKernelGGL(mex_col2im_kernel, dim3((unsigned)((n_in + 255) / 256)), dim3(256), 0, s, ga.k, ga.col,
                               input_grad, n_in);
            if (hipGetLastError() != hipSuccess)
                return SIMNETS_ERR_HIP;
        }
        if (want_offsets) {
            const long long rows = (long long)d.num_regions * d.M;
            // (1024 threads to a row pay from some 48 partial sums on: 512 elements, 10 instances, the offsets' gradient alone, 8 of them
            // 14.9 us with 256 threads and 16.4 with 1024, 32 16.0 and 16.6, 60 17.9 and 16.7, 128 21.9 and 19.3; 256 regions of 64
            // elements, one 49.0 and 52.3)
            if (t.head_wgs >= 48)
                hipLaunchKernelGGL(mex_grad_offsets_finish_tall_rows_kernel, dim3((unsigned)rows), dim3(1024), 0, s, ga.partial,
                                   n_off, t.head_wgs, d.K, p.normalize_offsets ? ga.off : nullptr, offsets_grad);
            else
                hipLaunchKernelGGL(mex_grad_offsets_finish_wide_rows_kernel, dim3((unsigned)rows), dim3(256), 0, s, ga.partial,
                                   n_off, t.head_wgs, d.K, p.normalize_offsets ? ga.off : nullptr, offsets_grad);
            if (hipGetLastError() != hipSuccess)
                return SIMNETS_ERR_HIP;
        }
        return SIMNETS_OK;
    }
    ga.msplit = 1; ga.mg_per_split = (d.M + GM_TM - 1) / GM_TM;
    ga.dx_splits = reinterpret_cast<float *>(ws + w.split);
    ga.wbuf = nullptr; ga.exbuf = nullptr; ga.slots_pad = 0; ga.Mp = 0; ga.Kp = 0;
    ga.pxl = 1;
    ga.cpr = (ga.k.slots + 63) / 64;
    // the row-wise kernels read and write 16 bytes at a time
    auto aligned16 = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    // (of a pooled gradient they read a window row's two values: 8 bytes)
    const bool g_aligned = grad_is_pooled ? (reinterpret_cast<uintptr_t>(output_grad) & 7) == 0 : aligned16(output_grad);
    const bool use_rows = t.mfma && t.rows && aligned16(input) && aligned16(output) && g_aligned &&
                          (!want_input || aligned16(input_grad));
    if (t.mfma) {
        rc = mex_pack_offsets(p, offsets, GM_TM, (d.M + GM_TM - 1) / GM_TM, packed_at, &ga.k, stream, nullptr,
                              !packed_already, pack_normalizes ? norm_at : nullptr, true);
        if (rc)
            return rc;
        if (w.use_factors && !use_rows) {
            rc = launch_factors(p, t, ga, ws + w.factors, s);
            if (rc)
                return rc;
        }
    }
    if (use_rows) {
        RowsArgs rg;
        rg.in = input; rg.out = output; rg.g = output_grad;
        rg.offe = ga.k.offe; rg.omax = ga.k.omax; rg.orng = ga.k.orng;
        rg.dx_split = n_in;
        rg.c0 = ga.k.c0; rg.c1 = ga.k.c1;
        rg.B = p.B; rg.M = d.M; rg.K = d.K; rg.n_mg = (d.M + GM_TM - 1) / GM_TM; rg.mg_per_split = t.rows_mg_per_split;
        rg.lgW = log2_exact(p.W); rg.Ws = p.W / 2; rg.RS = d.region_size; rg.HW = p.H * p.W; rg.lgHW = log2_exact(rg.HW);
        rg.chunks = t.slots_pad / 64;
        MexGradArgs gr = ga;   // for the term-by-term path
        gr.wbuf = gr.exbuf = nullptr;
        gr.slots_pad = t.slots_pad;
        typedef void (*RowsKernel)(RowsArgs, MexGradArgs);
        auto launch = [&](RowsKernel kernel, bool input, bool offsets, int ksub, int tz, int pxl, int cpr) {
            rg.dx = !input ? nullptr : t.rows_msplit > 1 ? ga.dx_splits : input_grad;
            rg.partial = offsets ? ga.partial : nullptr;
            rg.pxl = gr.pxl = pxl;
            rg.nx = gr.cpr = cpr; rg.ty = (d.K + 16 * ksub - 1) / (16 * ksub); rg.tz = tz;
            rg.d_tiles = make_fast_div((unsigned)(rg.ty * rg.tz)); rg.d_ty = make_fast_div((unsigned)rg.ty);
            const long long per_die = (1LL * rg.nx * rg.ty * rg.tz + 7) / 8, wgs = 8 * per_die;
            if (wgs > 0x7fffffffLL)
                return SIMNETS_ERR_TOO_LARGE;
            rg.per_die = (int)per_die;
            hipLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(256), 0, s, rg, gr);
            return hipGetLastError() == hipSuccess ? SIMNETS_OK : SIMNETS_ERR_HIP;
        };
        auto kernel_of = [&](auto ksub, auto w2) -> RowsKernel {
            constexpr int k = decltype(ksub)::value;
            constexpr bool w = decltype(w2)::value;
            if (!want_offsets || t.rows_apart)
                return grad_is_pooled ? mex_grads_rows_kernel<k, w, true, kRowsInput> : mex_grads_rows_kernel<k, w, false, kRowsInput>;
            if (!want_input)
                return grad_is_pooled ? mex_grads_rows_kernel<k, w, true, kRowsOffsets> : mex_grads_rows_kernel<k, w, false, kRowsOffsets>;
            return grad_is_pooled ? mex_grads_rows_kernel<k, w, true, 0> : mex_grads_rows_kernel<k, w, false, 0>;
        };
        // (alone, in a tile that holds all of K: 16 elements would fill half of it, 1024 x 16 x 16 x 16 -> 64 44 us, 41 in the other kernel)
        const bool offsets_apart = want_offsets && (t.rows_apart || (!want_input && p.W > 2 && d.K > 16 && d.K <= 16 * t.rows_ksub));
        const std::integral_constant<int, 1> one;
        const std::integral_constant<int, 2> two;
        if (want_input || !offsets_apart) {
            rc = launch(t.rows_ksub == 2 ? p.W > 2 ? kernel_of(two, std::false_type()) : kernel_of(two, std::true_type())
                        : p.W > 2        ? kernel_of(one, std::false_type())
                                         : kernel_of(one, std::true_type()),
                        want_input, want_offsets && !offsets_apart, t.rows_ksub, t.rows_msplit, t.rows_pxl, t.rows_cpr);
            if (rc)
                return rc;
        }
        if (offsets_apart) {
            rc = launch(grad_is_pooled ? mex_grad_offsets_rows_kernel<true> : mex_grad_offsets_rows_kernel<false>, false, true, 2, rg.n_mg,
                        t.offsets_pxl, t.offsets_cpr);
            if (rc)
                return rc;
        }
        // sums of the splits and of the chunks, in one launch if both are there to do (n_in is a multiple of 4: whole planes
        // of at least four pixels)
        const long long rows = (long long)d.num_regions * d.M, n4 = want_input && t.rows_msplit > 1 ? n_in / 4 : 0;
        const long long wgs_sum = (n4 + 255) / 256;
        if (want_offsets && d.K % 4 == 0 && d.K <= kFinishRowsMaxK && rows + wgs_sum <= 0x7fffffffLL) {
            hipLaunchKernelGGL(mex_grads_finish_kernel, dim3((unsigned)(rows + wgs_sum)), dim3(256), 0, s, ga.partial, n_off,
                               t.offsets_cpr, (int)rows, d.K, p.normalize_offsets ? ga.off : nullptr, offsets_grad,
                               reinterpret_cast<const float4 *>(ga.dx_splits), n4, t.rows_msplit,
                               reinterpret_cast<float4 *>(input_grad));
            return hipGetLastError() == hipSuccess ? SIMNETS_OK : SIMNETS_ERR_HIP;
        }
        if (n4 > 0) {
            launch_sum_splits(ga.dx_splits, n_in, t.rows_msplit, input_grad, s);
            if (hipGetLastError() != hipSuccess)
                return SIMNETS_ERR_HIP;
        }
    }

    if (want_input && !use_rows) {
        MexGradArgs gi = ga;
        gi.overlap = t.overlap ? 1 : 0;
        gi.msplit = t.msplit; gi.mg_per_split = t.mg_per_split;
        gi.pxl = 1;
        gi.cpr = (ga.k.slots + 63) / 64;
        if (!t.factors_input)
            gi.wbuf = gi.exbuf = nullptr;  // (each gradient forms its factors as it does in a call of its own)
        if (!t.overlap && !t.tiles_input) {
            // every element belongs to at most one patch, which stores its gradient; the others keep 0 (patches
            // that tile the input exactly write every element; overlapping ones go through mex_col2im_kernel)
            hipLaunchKernelGGL(mex_fill_zero_kernel, dim3((unsigned)std::min<long long>((n_in + 255) / 256, 65535)),
                               dim3(256), 0, s, input_grad, n_in);
            if (hipGetLastError() != hipSuccess)
                return SIMNETS_ERR_HIP;
        }
        const long long gx = (long long)d.num_regions * gi.cpr;
        if (t.mfma) {
            const int gy = (d.K + GM_KT - 1) / GM_KT;
            if (gx > 0x7fffffffLL || gy > 65535)
                return SIMNETS_ERR_TOO_LARGE;
            if (gx > 0)
                hipLaunchKernelGGL(mex_grad_input_mfma_kernel, dim3((unsigned)gx, (unsigned)gy, (unsigned)t.msplit),
                                   dim3(256), 0, s, gi);
            if (gx > 0 && t.msplit > 1) {
                if (hipGetLastError() != hipSuccess)
                    return SIMNETS_ERR_HIP;
                launch_sum_splits(gi.dx_splits, n_in, t.msplit, input_grad, s);
            }
        } else {
            const int gy = (d.K + 4 * GX_KT - 1) / (4 * GX_KT);
            if (gx > 0x7fffffffLL || gy > 65535)
                return SIMNETS_ERR_TOO_LARGE;
            if (gx > 0)
                hipLaunchKernelGGL(mex_grad_input_kernel, dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, s, gi);
        }
        if (hipGetLastError() != hipSuccess)
            return SIMNETS_ERR_HIP;
        if (t.overlap) {
            hipLaunchKernelGGL(mex_col2im_kernel, dim3((unsigned)((n_in + 255) / 256)), dim3(256), 0, s, gi.k, gi.col,
                               input_grad, n_in);
            if (hipGetLastError() != hipSuccess)
                return SIMNETS_ERR_HIP;
        }
    }

    if (want_offsets) {
        MexGradArgs go = ga;
        go.dx = nullptr; go.col = nullptr; go.dx_splits = nullptr;
        go.overlap = 0; go.msplit = 1;
        go.pxl = t.pxl;
        go.cpr = t.cpr_offsets;
        if (!t.factors_offsets)
            go.wbuf = go.exbuf = nullptr;
        const long long gx = (long long)d.num_regions * go.cpr;
        if (use_rows) {
            go.cpr = t.offsets_cpr;   // (launched above)
        } else if (t.mfma) {
            const int gy = (d.M + GOM_MT - 1) / GOM_MT, gz = (d.K + GOM_KT - 1) / GOM_KT;
            if (gx > 0x7fffffffLL || gy > 65535 || gz > 65535)
                return SIMNETS_ERR_TOO_LARGE;
            const dim3 grid((unsigned)gx, (unsigned)gy, (unsigned)gz);
            if (go.pxl > 1)
                hipLaunchKernelGGL(mex_grad_offsets_mfma_kernel<true>, grid, dim3(256), 0, s, go);
            else
                hipLaunchKernelGGL(mex_grad_offsets_mfma_kernel<false>, grid, dim3(256), 0, s, go);
        } else {
            const int gy = (d.M + 4 * GO_MT - 1) / (4 * GO_MT);
            const int gz = (d.K + GO_KT - 1) / GO_KT;
            if (gx > 0x7fffffffLL || gy > 65535 || gz > 65535)
                return SIMNETS_ERR_TOO_LARGE;
            hipLaunchKernelGGL(mex_grad_offsets_kernel, dim3((unsigned)gx, (unsigned)gy, (unsigned)gz), dim3(256), 0, s,
                               go);
        }
        if (hipGetLastError() != hipSuccess)
            return SIMNETS_ERR_HIP;
        const long long rows = (long long)d.num_regions * d.M;
        if (rows <= 64 && d.K >= 256 && d.K <= kFinishRowsMaxK) {
            // few long rows: a workgroup per row
            hipLaunchKernelGGL(mex_grad_offsets_finish_wide_rows_kernel, dim3((unsigned)rows), dim3(256), 0, s, go.partial,
                               n_off, go.cpr, d.K, p.normalize_offsets ? go.off : nullptr, offsets_grad);
            return hipGetLastError() == hipSuccess ? SIMNETS_OK : SIMNETS_ERR_HIP;
        }
        // (33 elements and more: shorter rows have several lanes to an element in the kernel below)
        if (d.K > 32 && d.K <= kFinishRowsMaxK && rows <= 512 && go.cpr >= 64) {
            hipLaunchKernelGGL(mex_grad_offsets_finish_tall_rows_kernel, dim3((unsigned)rows), dim3(1024), 0, s, go.partial,
                               n_off, go.cpr, d.K, p.normalize_offsets ? go.off : nullptr, offsets_grad);
            return hipGetLastError() == hipSuccess ? SIMNETS_OK : SIMNETS_ERR_HIP;
        }
        if (d.K <= kFinishRowsMaxK && (rows + 3) / 4 <= 0x7fffffffLL) {
            // short rows: the sum over the pixel chunks and the chain rule through the normalisation in one launch
            hipLaunchKernelGGL(mex_grad_offsets_finish_rows_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s,
                               go.partial, n_off, go.cpr, rows, d.K, p.normalize_offsets ? go.off : nullptr,
                               offsets_grad);
            return hipGetLastError() == hipSuccess ? SIMNETS_OK : SIMNETS_ERR_HIP;
        }
        hipLaunchKernelGGL(mex_grad_offsets_finish_kernel,
                           dim3((unsigned)std::min<long long>((n_off + 31) / 32, 65535)), dim3(256), 0, s, go.partial,
                           n_off, go.cpr, offsets_grad);
        if (hipGetLastError() != hipSuccess)
            return SIMNETS_ERR_HIP;
        if (p.normalize_offsets) {
            hipLaunchKernelGGL(mex_normalize_rows_backward_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s,
                               go.off, rows, d.K, offsets_grad);
            if (hipGetLastError() != hipSuccess)
                return SIMNETS_ERR_HIP;
        }
    }
    return SIMNETS_OK;
}

int mex_grad_input(const MexPlan &p, const float *input, const float *offsets, const float *output,
                   const float *output_grad, float *input_grad, void *workspace, size_t workspace_bytes, void *stream)
{
    return mex_grads(p, input, offsets, output, output_grad, input_grad, nullptr, workspace, workspace_bytes, stream);
}

int mex_grad_offsets(const MexPlan &p, const float *input, const float *offsets, const float *output,
                     const float *output_grad, float *offsets_grad, void *workspace, size_t workspace_bytes,
                     void *stream)
{
    return mex_grads(p, input, offsets, output, output_grad, nullptr, offsets_grad, workspace, workspace_bytes, stream);
}

}  // namespace simnets
