// fp_adjoint.hip -- matched adjoint of the ray-driven FP (gfx950): cell-driven where
// every sample lies in the image's texel cells [-1, n-1], else gathered per pixel.
//
// The FP (fp.hip; reference FP/transform.cu:103-146) forms
//     p[v][c] = 0.125 dx * sum_k  sum_taps  w_tap(u_k, w_k) * img[clamp(tap)]
// with u_k = fma(k, du, u0), w_k = fma(k, dw, w0) in FP32.  Its transpose is
//     img[j][i] = 0.125 dx * sum_v sum_c p[v][c] * W_c(i, j),
//     W_c(i, j) = sum_k  T_i(u_k) * T_j(w_k),
// where T_i(u) = max(0, 1 - |clamp(u, 0, nX-1) - i|) is the total bilinear weight the
// clamped taps of a sample give pixel i (the clamp folds the taps -1 and nX, and any
// sample beyond the image edge, into the border pixels).
//
// Both forms write every pixel exactly once, without atomics.  The cell-driven kernels
// (section "cell-driven variant" below) sum each ray's samples per texel cell in closed
// form.  The per-pixel gather: each thread owns one output pixel and accumulates over
// all views.  Per view, the candidate rays are
// the columns whose lines pass within the support of the pixel (radius rho around its
// centre, rho = sqrt(2) inside the image), found from the pixel's fan angle; per
// candidate ray the sample range whose positions fall in the support is computed in
// closed form and the samples are evaluated at exactly the FP32 positions the forward
// kernel interpolates at.  A group of S <= 16 slices that share the geometry is
// processed together: the per-(pixel, view, ray) weight W_c is computed once and applied
// to S sinograms.  Sums over blocks of 8 views accumulate in FP32, across blocks in FP64.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "dtype.hpp"
#include "fbct_internal.hpp"

namespace fbct {
namespace {

constexpr int kAdjThreads = 256;
constexpr int kAdjTx = 16, kAdjTy = kAdjThreads / kAdjTx;  // tile of the regular launches
constexpr float kBig = 1e30f;

struct FpaArgs {
    const void *sino;  // TI[n][nViews][nCols]
    void *img;         // TO[n][nY][nX]
    const float4 *ray_geo;
    const int32_t *ray_n;
    const float2 *ray_inv;  // (1/du, 1/dw), 1e30 for a zero step
    const float2 *cs;       // (cos beta, sin beta)
    long long img_stride, sino_stride;
    int nX, nY, nViews, nCols, nSlices;
    float scale;            // 0.125 dx
    float r;                // rFOV/dx: FP texel coordinate of the image centre is r - 1/2
    float dx, R;
    float c_scale, c_off;   // column coordinate c_f = atan(t/U) * c_scale + c_off (ray c at c_f = c)
    float c_abs;            // |1/dCol|: radians -> columns
    float far_x, far_y;     // how far samples reach beyond the last pixel centre (texels)
};

// Sample window of one pixel.  kBorder: the pixel's tile touches the image edge, so the
// clamp window and the unbounded outer support of border pixels apply; interior tiles
// skip them.
struct PixelWin {
    float xlo_c, xhi_c, ylo_c, yhi_c;  // clamp window of the sample coordinate (border plateaus)
    float xlo_b, xhi_b, ylo_b, yhi_b;  // support of T_i in (u - i), unbounded outside border pixels
    float rho;                          // support radius (texels)
};

template <bool kBorder>
__device__ __forceinline__ PixelWin pixel_window(const FpaArgs &A, int i, int j)
{
    PixelWin w{-kBig, kBig, -kBig, kBig, -1.0f, 1.0f, -1.0f, 1.0f, 1.41421356f};
    if (kBorder) {
        if (i == 0) w.xlo_c = 0.0f, w.xlo_b = -kBig;
        if (i == A.nX - 1) w.xhi_c = 0.0f, w.xhi_b = kBig;
        if (j == 0) w.ylo_c = 0.0f, w.ylo_b = -kBig;
        if (j == A.nY - 1) w.yhi_c = 0.0f, w.yhi_b = kBig;
        const float ex = (i == A.nX - 1) ? fmaxf(1.0f, A.far_x) : 1.0f;
        const float ey = (j == A.nY - 1) ? fmaxf(1.0f, A.far_y) : 1.0f;
        w.rho = sqrtf(ex * ex + ey * ey);
    }
    return w;
}

// atan(q) for |q| <= 1/2 by the odd polynomial q P(q^2) of degree 7 (coefficients a
// weighted least-squares fit to atan on [0, 1/2]); its error, FP32 evaluation included,
// is below 5.5e-7 rad on [-1/2, 1/2] (checked on 2e5 points against FP64 atan), and
// kCandAtanErr bounds it.
constexpr float kCandAtanErr = 2.0e-6f;
__device__ __forceinline__ float cand_atan(float q)
{
    if (fabsf(q) > 0.5f) return atanf(q);
    const float s = q * q;
    return q * fmaf(fmaf(fmaf(-9.581676484e-02f, s, 1.920663981e-01f), s, -3.328139539e-01f), s,
                    9.999906794e-01f);
}

// Candidate rays of a pixel in one view: columns [clo, chi] whose lines pass within rho
// (texels) of the pixel centre (x, y) (mm).  Such rays subtend at most asin(rho dx / L)
// from the pixel's fan angle; L >= U and asin(z) <= z (1 + z^2) for z <= 0.9.  The fan
// angle comes from cand_atan and the range is widened by its error bound, so it holds
// every column the exact angle admits (an extra candidate adds zero samples).
__device__ __forceinline__ void candidate_rays(const FpaArgs &A, float2 cs, float x, float y, float rho, int &clo,
                                               int &chi)
{
    const float U = fmaf(-y, cs.y, fmaf(-x, cs.x, A.R));
    const float t = fmaf(x, cs.y, -y * cs.x);
    const float rU = __builtin_amdgcn_rcpf(U);
    const float cf = fmaf(cand_atan(t * rU), A.c_scale, A.c_off);
    const float z = rho * A.dx * rU;
    const float hw = z < 0.9f ? fmaf(z * fmaf(z, z, 1.0f), A.c_abs, fmaf(kCandAtanErr, A.c_abs, 1e-3f)) : 1e9f;
    clo = (int)fmaxf(ceilf(cf - hw), 0.0f);
    chi = (int)fminf(floorf(cf + hw), (float)(A.nCols - 1));
}

// Candidate rays of the cells of one square block in one view, from a linear model of the
// column coordinate about the block centre (xc, yc) (mm): cf(p) = c_scale atan(t/U) +
// c_off is c_scale times the polar angle of p about the source, whose Hessian has norm
// 1/r^2 (r the distance to the source).  Over the block's cell centres, within h of the
// centre along each axis (3.5 dx for a tile of 8 x 8 cells), the linear model is therefore off by at most
// |c_scale| h^2 / Rmin^2, Rmin the least r over the block.  A ray at fan-angle offset g
// from a cell centre passes r sin|g| from it, so the rays that meet the cell lie within
// asin(rs dx / Rmin) <= z (1 + z^2), z = rs dx / Rmin, of its fan angle (rs the cell's
// support radius, below); the half-width adds the model's error and the atan bound to
// that, so every cell's range holds every column whose ray meets the cell.  One lane
// evaluates a view's model for all of the tile's cells.
struct BlockCand {
    float cf, gx, gy, hw;  // centre column, d cf / dx, d cf / dy (per mm), half-width
    float dx, dy, spread;  // ray direction at the centre; a bound on how far any candidate's differs
};

__device__ __forceinline__ BlockCand block_candidates(const FpaArgs &A, float2 cs, float xc, float yc, float rho,
                                                      float h)
{
    const float U = fmaf(-yc, cs.y, fmaf(-xc, cs.x, A.R));
    const float t = fmaf(xc, cs.y, -yc * cs.x);
    const float rU = __builtin_amdgcn_rcpf(U);
    BlockCand b;
    b.cf = fmaf(cand_atan(t * rU), A.c_scale, A.c_off);
    // d atan(t/U) = (U dt - t dU) / (U^2 + t^2) with dt = (sin b, -cos b) . dp and
    // dU = -(cos b, sin b) . dp
    const float k = A.c_scale * __builtin_amdgcn_rcpf(fmaf(U, U, t * t));
    b.gx = k * fmaf(U, cs.y, t * cs.x);
    b.gy = k * fmaf(t, cs.y, -U * cs.x);
    const float Umin = U - (fabsf(cs.x) + fabsf(cs.y)) * h;
    // every point of the block is at least Rmin from the source: its U is at least Umin,
    // and it lies within 1.415 h of the block centre, at sqrt(U^2 + t^2) from the source
    const float q = fmaf(U, U, t * t);
    const float rL = rsqrtf(q);
    const float rRm = __builtin_amdgcn_rcpf(fmaxf(Umin, fmaf(q, rL, -1.415f * h)));
    auto half_width = [&](float rs) {  // for a support of radius rs (texels) about each cell centre
        const float z = rs * A.dx * rRm;
        return (Umin > 0.0f && z < 0.9f)
                   ? fmaf(z * fmaf(z, z, 1.0f), A.c_abs,
                          fmaf(kCandAtanErr, A.c_abs, fmaf(A.c_abs * h * h, rRm * rRm, 1e-3f)))
                   : 1e9f;
    };
    // A line of unit direction d meets a square cell iff it passes within (|d_x| + |d_y|)/2
    // texels of its centre, which is below rho = 1/sqrt(2) except along the diagonals.  The
    // direction from the source to the block centre is (t sin b - U cos b, -U sin b - t cos b)
    // / sqrt(U^2 + t^2); a candidate ray's direction differs from it by at most 1.415 h / Rmin
    // (its cell's place in the block) plus hw / |c_scale| (its column, within the disk's
    // half-width hw), and (|d_x| + |d_y|)/2 changes by at most 0.7072 per radian; 0.004 texel
    // covers the FP32 sample positions (within 3e-4 texel of the line).  Only rays without
    // samples in the cell are dropped.
    const float hw_disk = half_width(rho);
    const float ax = fmaf(t, cs.y, -U * cs.x), ay = -fmaf(U, cs.y, t * cs.x);
    const float spread = fmaf(1.415f * h, rRm, hw_disk * __builtin_amdgcn_rcpf(A.c_abs));
    const float rs = fminf(rho, fmaf(0.5f * (fabsf(ax) + fabsf(ay)), rL, fmaf(0.7072f, spread, 0.004f)));
    b.hw = half_width(rs);
    b.dx = ax * rL, b.dy = ay * rL, b.spread = spread;
    return b;
}

// W_c(i, j): total bilinear weight pixel (fi, fj) receives from the N samples of ray
// (u0, w0, du, dw) = g, evaluated at the FP32 sample positions; inv = (1/du, 1/dw).
template <bool kBorder>
__device__ __forceinline__ float ray_weight(float4 g, float2 inv, int N, float fi, float fj, const PixelWin &w)
{
    const float X0 = g.x - fi, Y0 = g.y - fj;
    const float a1 = (w.xlo_b - X0) * inv.x, a2 = (w.xhi_b - X0) * inv.x;
    const float b1 = (w.ylo_b - Y0) * inv.y, b2 = (w.yhi_b - Y0) * inv.y;
    const float lo = fmaxf(fmaxf(fminf(a1, a2), fminf(b1, b2)), 0.0f);
    const float hi = fminf(fminf(fmaxf(a1, a2), fmaxf(b1, b2)), (float)(N - 1));
    float wsum = 0.0f;
    const float kend = floorf(hi);
    auto sample = [&](float kf) {
        const float X = fmaf(kf, g.z, X0);
        const float Y = fmaf(kf, g.w, Y0);
        if (kBorder) {
            const float wx = 1.0f - fabsf(fminf(fmaxf(X, w.xlo_c), w.xhi_c));
            const float wy = 1.0f - fabsf(fminf(fmaxf(Y, w.ylo_c), w.yhi_c));
            wsum = fmaf(fmaxf(wx, 0.0f), fmaxf(wy, 0.0f), wsum);
        } else {
            // inside the support |X|, |Y| < 1 up to rounding at its two ends
            wsum = fmaf(1.0f - fabsf(X), 1.0f - fabsf(Y), wsum);
        }
    };
    float kf = ceilf(lo);
    for (; kf + 1.0f <= kend; kf += 2.0f) {  // two samples per iteration
        sample(kf);
        sample(kf + 1.0f);
    }
    if (kf <= kend) sample(kf);
    return wsum;
}

// FP32 sums over blocks of kViewBlock views, FP64 across blocks.
constexpr int kViewBlock = 8;

// Per-pixel accumulation over all views, every ray's tables and S sinogram values read
// from global memory.
template <int S, bool kBorder, typename TI, typename TO>
__device__ __forceinline__ void adjoint_pixel(const FpaArgs &A, int i, int j, int s0)
{
    const float fi = (float)i, fj = (float)j;
    // pixel centre in mm, in the FP's frame (dx on both axes, centre at texel r - 1/2)
    const float x = (fi + 0.5f - A.r) * A.dx;
    const float y = (fj + 0.5f - A.r) * A.dx;
    const PixelWin pw = pixel_window<kBorder>(A, i, j);

    const TI *sino[S];
#pragma unroll
    for (int s = 0; s < S; ++s)
        sino[s] = static_cast<const TI *>(A.sino) + (size_t)min(s0 + s, A.nSlices - 1) * A.sino_stride;

    double acc[S];
    float vsum[S];
#pragma unroll
    for (int s = 0; s < S; ++s) acc[s] = 0.0, vsum[s] = 0.0f;

    for (int v = 0; v < A.nViews; ++v) {
        int clo, chi;
        candidate_rays(A, A.cs[v], x, y, pw.rho, clo, chi);
        const size_t rbase = (size_t)v * A.nCols;
        for (int c = clo; c <= chi; ++c) {
            // The S sinogram values are loaded first, unconditionally, so their latency
            // overlaps the weight computation (a ray that misses the support, or has no
            // samples, ends with wsum = 0; sinograms are expected to be finite).
            const int N = A.ray_n[rbase + c];
            const float4 g = A.ray_geo[rbase + c];
            const float2 inv = A.ray_inv[rbase + c];
            // one 32-bit byte offset serves all S sinograms (a slice's sinogram is < 4 GiB)
            const unsigned boff = (unsigned)(rbase + c) * (unsigned)sizeof(TI);
            float sv[S];
#pragma unroll
            for (int s = 0; s < S; ++s) sv[s] = load_f_at(sino[s], boff);
            const float wsum = ray_weight<kBorder>(g, inv, N, fi, fj, pw);
#pragma unroll
            for (int s = 0; s < S; ++s) vsum[s] = fmaf(wsum, sv[s], vsum[s]);
        }
        if (v % kViewBlock == kViewBlock - 1 || v == A.nViews - 1) {
#pragma unroll
            for (int s = 0; s < S; ++s) acc[s] += (double)vsum[s], vsum[s] = 0.0f;
        }
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s0 + s < A.nSlices)
            store_f(static_cast<TO *>(A.img), (size_t)(s0 + s) * A.img_stride + (size_t)j * A.nX + i,
                    (float)(acc[s] * (double)A.scale));
}

// ---------------------------------------------------------------- staged variant
// For S >= 4 slices the per-ray loads dominate: S sinogram values and the ray's tables,
// gathered per pixel.  The staged variant copies, per batch of kStageVB views, the 64
// sinogram columns around the tile's candidate rays into LDS once (coalesced, slices
// interleaved per column, converted to FP32) together with the columns' ray tables; a
// pixel then reads a ray's S values with S/4 16-byte LDS reads.  The window of a view
// is derived from the four corner pixels of the tile (t/U, and so the fan angle, is
// extremal at a corner), lane 4m + c evaluating corner c of view m; a candidate column
// outside the window is read from global memory.
constexpr int kStageCols = 64;  // staged columns per view: one per lane
constexpr int kStageVB = 4;     // views per staging batch

template <int S>
struct AdjStage {
    static constexpr int kPitch = S + 4;  // floats per staged column: 16-byte multiple, off the bank period
    float val[kStageVB][kStageCols][kPitch];
    float4 geo[kStageVB][kStageCols];
    float2 inv[kStageVB][kStageCols];
    int n[kStageVB][kStageCols];
};

template <int S, bool kBorder, typename TI, typename TO>
__device__ __forceinline__ void adjoint_staged_tile(const FpaArgs &A, AdjStage<S> &st, int tx, int ty, int s0)
{
    static_assert(S % 4 == 0, "a staged column is read four slices at a time");
    constexpr int VB = kStageVB;
    constexpr int SQ = S / 4;  // slices staged per wave
    const int i = tx * kAdjTx + (int)threadIdx.x % kAdjTx;
    const int j = ty * kAdjTy + (int)threadIdx.x / kAdjTx;
    const bool valid = i < A.nX && j < A.nY;  // no early exit: every thread stages and waits
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const float fi = (float)i, fj = (float)j;
    const float x = (fi + 0.5f - A.r) * A.dx;
    const float y = (fj + 0.5f - A.r) * A.dx;
    const PixelWin pw = pixel_window<kBorder>(A, i, j);
    // corner of this lane for the window: lane 4m + c evaluates corner c
    const int ci = min(tx * kAdjTx + ((lane & 1) ? kAdjTx - 1 : 0), A.nX - 1);
    const int cj = min(ty * kAdjTy + ((lane & 2) ? kAdjTy - 1 : 0), A.nY - 1);
    const float cx = ((float)ci + 0.5f - A.r) * A.dx;
    const float cy = ((float)cj + 0.5f - A.r) * A.dx;
    // this wave stages slices [s0 + wave SQ, s0 + (wave + 1) SQ)
    const TI *sino_w[SQ];
#pragma unroll
    for (int q = 0; q < SQ; ++q)
        sino_w[q] = static_cast<const TI *>(A.sino) + (size_t)min(s0 + wave * SQ + q, A.nSlices - 1) * A.sino_stride;
    const TI *sino[S];
#pragma unroll
    for (int s = 0; s < S; ++s)
        sino[s] = static_cast<const TI *>(A.sino) + (size_t)min(s0 + s, A.nSlices - 1) * A.sino_stride;

    double acc[S];
    float vsum[S];
#pragma unroll
    for (int s = 0; s < S; ++s) acc[s] = 0.0, vsum[s] = 0.0f;

    for (int v0 = 0; v0 < A.nViews; v0 += VB) {
        int c_lo[VB];
        {
            int wlo, whi;
            candidate_rays(A, A.cs[min(v0 + (lane >> 2) % VB, A.nViews - 1)], cx, cy, 1.41421356f, wlo, whi);
#pragma unroll
            for (int sh = 1; sh <= 2; sh <<= 1) wlo = min(wlo, __shfl_xor(wlo, sh));
#pragma unroll
            for (int m = 0; m < VB; ++m)
                c_lo[m] = min(max(__builtin_amdgcn_readlane(wlo, 4 * m) - 1, 0), max(A.nCols - kStageCols, 0));
        }
        __syncthreads();  // the previous batch's reads are done
#pragma unroll
        for (int m = 0; m < VB; ++m) {
            const int c = c_lo[m] + lane;
            if (v0 + m >= A.nViews || c >= A.nCols) continue;
            const size_t rb = (size_t)(v0 + m) * A.nCols + c;
            const unsigned boff = (unsigned)rb * (unsigned)sizeof(TI);
            float q4[SQ];
#pragma unroll
            for (int q = 0; q < SQ; ++q) q4[q] = load_f_at(sino_w[q], boff);
            float *dst = &st.val[m][lane][wave * SQ];  // this wave's SQ slots of the column
            if constexpr (SQ % 4 == 0) {
#pragma unroll
                for (int q = 0; q < SQ; q += 4)
                    *reinterpret_cast<float4 *>(dst + q) = make_float4(q4[q], q4[q + 1], q4[q + 2], q4[q + 3]);
            } else if constexpr (SQ == 2) {
                *reinterpret_cast<float2 *>(dst) = make_float2(q4[0], q4[1]);
            } else {
#pragma unroll
                for (int q = 0; q < SQ; ++q) dst[q] = q4[q];
            }
            if (wave == 0) st.geo[m][lane] = A.ray_geo[rb];
            else if (wave == 1) st.inv[m][lane] = A.ray_inv[rb];
            else if (wave == 2) st.n[m][lane] = A.ray_n[rb];
        }
        __syncthreads();
        if (!valid) continue;
#pragma unroll 1
        for (int m = 0; m < VB; ++m) {
            const int v = v0 + m;
            if (v >= A.nViews) break;
            int clo, chi;
            candidate_rays(A, A.cs[v], x, y, pw.rho, clo, chi);
            for (int c = clo; c <= chi; ++c) {
                const int lc = c - c_lo[m];
                int N;
                float4 g;
                float2 inv;
                float sv[S];
                if ((unsigned)lc < (unsigned)kStageCols) {
                    N = st.n[m][lc];
                    g = st.geo[m][lc];
                    inv = st.inv[m][lc];
#pragma unroll
                    for (int s = 0; s < S; s += 4) {
                        const float4 t4 = *reinterpret_cast<const float4 *>(&st.val[m][lc][s]);
                        sv[s] = t4.x, sv[s + 1] = t4.y, sv[s + 2] = t4.z, sv[s + 3] = t4.w;
                    }
                } else {
                    const size_t rb = (size_t)v * A.nCols + c;
                    N = A.ray_n[rb];
                    g = A.ray_geo[rb];
                    inv = A.ray_inv[rb];
                    const unsigned boff = (unsigned)rb * (unsigned)sizeof(TI);
#pragma unroll
                    for (int s = 0; s < S; ++s) sv[s] = load_f_at(sino[s], boff);
                }
                const float wsum = ray_weight<kBorder>(g, inv, N, fi, fj, pw);
#pragma unroll
                for (int s = 0; s < S; ++s) vsum[s] = fmaf(wsum, sv[s], vsum[s]);
            }
            if (v % kViewBlock == kViewBlock - 1 || v == A.nViews - 1) {
#pragma unroll
                for (int s = 0; s < S; ++s) acc[s] += (double)vsum[s], vsum[s] = 0.0f;
            }
        }
    }
    if (!valid) return;
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s0 + s < A.nSlices)
            store_f(static_cast<TO *>(A.img), (size_t)(s0 + s) * A.img_stride + (size_t)j * A.nX + i,
                    (float)(acc[s] * (double)A.scale));
}

template <int S, typename TI, typename TO>
__global__ __launch_bounds__(kAdjThreads) void fp_adjoint_staged_kernel(FpaArgs A)
{
    __shared__ AdjStage<S> st;
    const int tx = blockIdx.x, ty = blockIdx.y;
    const bool border_tile = tx == 0 || ty == 0 || (tx + 1) * kAdjTx >= A.nX || (ty + 1) * kAdjTy >= A.nY;
    if (border_tile)
        adjoint_staged_tile<S, true, TI, TO>(A, st, tx, ty, blockIdx.z * S);
    else
        adjoint_staged_tile<S, false, TI, TO>(A, st, tx, ty, blockIdx.z * S);
}

// Pixel tile (tx, ty) of TX x (256/TX) pixels for slices [s0, s0+S).
template <int S, int TX, typename TI, typename TO>
__device__ __forceinline__ void adjoint_tile(const FpaArgs &A, int tx, int ty, int s0)
{
    constexpr int TY = kAdjThreads / TX;
    const int i = tx * TX + threadIdx.x % TX;
    const int j = ty * TY + threadIdx.x / TX;
    if (i >= A.nX || j >= A.nY) return;
    const bool border_tile = tx == 0 || ty == 0 || (tx + 1) * TX >= A.nX || (ty + 1) * TY >= A.nY;
    if (border_tile)
        adjoint_pixel<S, true, TI, TO>(A, i, j, s0);
    else
        adjoint_pixel<S, false, TI, TO>(A, i, j, s0);
}

template <int S, typename TI, typename TO>
__global__ __launch_bounds__(kAdjThreads) void fp_adjoint_kernel(FpaArgs A)
{
    adjoint_tile<S, kAdjTx, TI, TO>(A, blockIdx.x, blockIdx.y, blockIdx.z * S);
}

// ---------------------------------------------------------------- cell-driven variant
// The per-pixel gather evaluates each sample once for every pixel of its 2x2 support.
// Here a thread owns a texel cell (ci, cj), the square between the pixel centres
// ci..ci+1 and cj..cj+1 (samples inside it interpolate between those four pixels).  Per
// view and candidate ray (lines within half a cell diagonal of the cell centre) it finds
// the ray's samples inside the cell: along each axis the samples before boundary b number
// ceil((b - u0) / du) in either direction, evaluated by the same expression in both cells
// that share b, so the cells partition every ray's samples exactly.  The sums
// over those n samples of 1, the u- and w-fractions and their products (fractions
// ta + j du, tm + j dw) are closed-form, as in the forward kernel's cell walk, and
// accumulate (FP32) times the ray's value per slice; at the end they give the four corner
// weights, which are combined per pixel through LDS, clamp-to-edge folding the outer
// corners of cells -1 and n-1 into the border pixels.  Valid while every sample lies in the cells [-1, n-1] of both axes
// (2 rFOV/dx - n + 1/2 < 1, square images); otherwise the gather kernels run.  Every
// variant below evaluates a slice with the same arithmetic in the same order, so results
// do not depend on how many slices share a launch.
constexpr int kCellTile = kAdjCellTile;  // cells per tile side; a tile yields 7 x 7 pixels
constexpr int kCellOut = kCellTile - 1;
constexpr int kCells = kCellTile * kCellTile;  // one per lane
constexpr int kCombineS = 4;                   // slices combined per LDS pass
constexpr float kCellRho = 0.70710678f;        // half a cell diagonal (texels)

// A ray as the cell kernels read it: u0, w0, du, dw; 1/du, 1/dw, -u0/du, -w0/dw; samples N,
// du dw / 12.
struct RayRec {
    float4 p, q;
    float2 n;
};

// Closed-form sums over the samples of a ray that lie in cell (fci, fcj): their number n, and
// the sums n ta of the u-fractions, n tm of the w-fractions and n g of their products.  The
// bilinear weights the cell's corners (0,0) (1,0) (0,1) (1,1) receive are n (1 - ta - tm + g),
// n (ta - g), n (tm - g) and n g (formed once per cell from the accumulated sums in
// cell_combine).
//
// (ulo, uhi) and (wlo, whi) are the cell's boundaries in the order the ray meets them: (fci, fci +
// 1) for du > 0, the other way round for du < 0; kMixed: in either order, sorted here.
struct CellSums {
    float n, ta, tm, g;  // samples, their mean fractions, the mean of the fractions' products
};
template <bool kMixed>
__device__ __forceinline__ CellSums cell_sums(const RayRec &ray, float fci, float fcj, float ulo, float uhi, float wlo,
                                              float whi)
{
    // sample range inside the cell, per axis, then intersected with [0, N): the samples
    // that precede boundary b along the ray number ceil((b - u0) / du) in either
    // direction (a sample exactly on b goes to the cell it leaves, where its bilinear
    // weights are the same), so the range is [ceil(min q), ceil(max q)); both cells that share
    // a boundary evaluate the same expression for it
    float qul = fmaf(ulo, ray.q.x, ray.q.z), quh = fmaf(uhi, ray.q.x, ray.q.z);
    float qwl = fmaf(wlo, ray.q.y, ray.q.w), qwh = fmaf(whi, ray.q.y, ray.q.w);
    if constexpr (kMixed) {
        const float a = fminf(qul, quh), b = fminf(qwl, qwh);
        quh = fmaxf(qul, quh), qwh = fmaxf(qwl, qwh);
        qul = a, qwl = b;
    }
    const float klo = ceilf(fmaxf(fmaxf(qul, qwl), 0.0f));
    const float khi = ceilf(fminf(fminf(quh, qwh), ray.n.x));
    CellSums c;
    c.n = fmaxf(khi - klo, 0.0f);
    // the fractions are linear in the sample index, so their means are those of the middle
    // (half-integer) index, and the mean of their products is the product of the means plus
    // du dw times the variance (n^2 - 1) / 12 of the indices.  The cell index is subtracted
    // before the step is added, so the FP32 rounding is that of the distance, not of the texel
    // coordinate.
    const float kc = fmaf(c.n, 0.5f, klo - 0.5f);
    c.ta = fmaf(kc, ray.p.z, ray.p.x - fci), c.tm = fmaf(kc, ray.p.w, ray.p.y - fcj);
    c.g = fmaf(ray.n.y, fmaf(c.n, c.n, -1.0f), c.ta * c.tm);
    return c;
}

// True when cell (ci, cj) can hold samples: every sample lies in the FOV disk of radius
// r about texel coordinate (r - 1/2, r - 1/2) (its chord endpoints are on the circle), so
// a cell whose nearest point is farther away (plus 0.01 texel for FP32 positions)
// receives none and its views can be skipped.
__device__ __forceinline__ bool cell_in_fov(const FpaArgs &A, float fci, float fcj)
{
    const float c0 = A.r - 0.5f;
    const float ex = fmaxf(fmaxf(fci - c0, c0 - (fci + 1.0f)), 0.0f);
    const float ey = fmaxf(fmaxf(fcj - c0, c0 - (fcj + 1.0f)), 0.0f);
    const float rr = A.r + 0.01f;
    return fmaf(ex, ex, ey * ey) <= rr * rr;
}

// A workgroup owns a tile of 8 x 8 cells, one per lane, and its four waves a quarter of the views
// each (their sums meet in LDS at the end, see cell_combine), so that small images fill the chip too.  A wave runs
// without workgroup barriers: the columns around its candidate rays are staged by the wave, for
// itself, in 64 LDS slots (the windows of 4, 3, 2 or 1 views, 16, 21, 32 or 64 columns wide, as
// the tile's geometry in the current group of views needs), each slot holding a ray's record and
// its S values.  LDS operations of a wave complete in order, so rewriting the slots needs no
// wait.
//
// The candidate columns of a cell come from one linear model per (tile, view) -- evaluated for
// 16 views at a time, one per lane, and read back as wave-uniform scalars: a cell's first
// candidate is two FMAs and a ceil, and the number of candidates is uniform (the widest range
// that fits the half-width), so the candidate loop has no divergence.  Columns beyond the
// detector are staged as rays without samples, so it has no clamps either.
//
// Bound: VALU issue (0.7 of it, a third of the instructions issued in pairs): per wave and view
// about 2.15 candidates (1.55 rays meet a cell at 512 x 512 / 888 columns) of 25 instructions and
// 4 S multiply-adds, and 30 for the model, the staging and the loop.  Measured on 512 x 512 pixels, 984
// views, 888 columns: 1 slice 940 -> 630 us, 4 slices 1.30 ms -> 829 us (with the rays read by every
// cell from global memory, and staged per workgroup between barriers); 16 slices 2.0 -> 1.75 ms;
// 256 x 256, 360 views, 512 columns: 1 slice 162 -> 117 us, 4 slices 614 -> 151 us; 104 x 104, 147
// views: 81 -> 19 us.  Tiles of 16 x 16 cells (four waves side by side) have less overlap (1.14
// against 1.31 cells per pixel) and measured the same within 5% at 512 x 512 (596 us for 1 slice) and
// slower on smaller images (156 us at 256 x 256).
constexpr int kWvGroup = 16;      // views whose models are evaluated together
constexpr int kWvSlots = 64;      // staged columns per wave
constexpr int kWvSplit = 4;       // waves per workgroup, each a quarter of the views
constexpr float kWvHalf = 3.5f;   // cell centres lie within this many texels of the tile's centre

// Slot stride in dwords: record (10), S values (from dword 10, or 12 for S >= 4), and padding
// so that 16 adjacent slots start in different bank groups (an odd multiple of 4 dwords).
template <int S>
struct alignas(16) WvStage {
    static constexpr int kDw = S == 16 ? 28 : S >= 4 ? 20 : 12;
    float slot[kWvSlots * kDw];
};

template <int S>
union CellShared {
    static constexpr int kC = S < kCombineS ? S : kCombineS;
    WvStage<S> stage[kWvSplit];
    struct {
        float part[kWvSplit][4][kC][kCells];  // the waves' sums
        float corner[kC][4][kCells];
    } sum;
};

// Cell (lx, ly) of this lane in the tile: each 16 lanes a 4 x 4 block, whose candidate columns
// lie close together (few LDS bank conflicts).
__device__ __forceinline__ void tile_cell(int &lx, int &ly)
{
    const int lane = (int)threadIdx.x & 63;
    lx = 4 * ((lane >> 4) & 1) + (lane & 3);
    ly = 4 * (lane >> 5) + ((lane >> 2) & 3);
}

// LDS accesses of a wave complete in order; this keeps the compiler from moving them across each
// other where lanes read what other lanes of their wave wrote.
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
}

// Adds the waves' cell sums acc[4][S] (n, Su, Sw, Suw, each times the ray values; FP32, in pairs) and
// combines them, as corner partials, into the tile's 7 x 7 pixels of slices [s0, s0 + S), kCombineS
// slices per pass, a wave each (one wave for all of them took 340 of the 890 us of 64 slices of 512 x
// 512 over 90 views).  Pixel (px, py) collects corner dx of cell px - dx (dx = 0, 1), and, on the
// borders, the clamped outer corner of cell -1 (pixel 0) or of cell n-1 (pixel n-1).  sh is free when
// called; every thread of the workgroup calls it.
template <int S, typename TO>
__device__ __forceinline__ void cell_combine(const FpaArgs &A, CellShared<S> &sh, const float (&acc)[4][S], int tx,
                                             int ty, int s0)
{
    constexpr int kC = CellShared<S>::kC;
    int lane = (int)threadIdx.x;
    asm volatile("" : "+v"(lane));  // nothing of this is kept in registers while the views are summed
    const int wave = __builtin_amdgcn_readfirstlane(lane >> 6);
    lane &= 63;
    const int lx = 4 * ((lane >> 4) & 1) + (lane & 3), ly = 4 * (lane >> 5) + ((lane >> 2) & 3);
    const int cid = ly * kCellTile + lx;
    const int px = tx * kCellOut + lx, py = ty * kCellOut + ly;
    const bool out = lx < kCellOut && ly < kCellOut && px < A.nX && py < A.nY;
#pragma unroll
    for (int sb = 0; sb < S; sb += kCombineS) {
        if (sb > 0) __syncthreads();  // the previous pass's reads
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int k = 0; k < kC; ++k) sh.sum.part[wave][q][k][lane] = acc[q][sb + k];
        __syncthreads();
        if (wave >= kC || s0 + sb + wave >= A.nSlices) continue;
        float r[4];  // corner weights from the sums (n, Su, Sw, Suw)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            r[q] = (sh.sum.part[0][q][wave][lane] + sh.sum.part[1][q][wave][lane]) +
                   (sh.sum.part[2][q][wave][lane] + sh.sum.part[3][q][wave][lane]);
        float(&corner)[4][kCells] = sh.sum.corner[wave];
        const float c01 = r[2] - r[3];
        wave_lds_order();  // the previous pass's corners are read
        corner[0][cid] = (r[0] - r[1]) - c01;
        corner[1][cid] = r[1] - r[3];
        corner[2][cid] = c01;
        corner[3][cid] = r[3];
        wave_lds_order();
        if (out) {
            double sum = 0.0;
            auto row = [&](int cy, int dy) {
                const float *c0 = &corner[2 * dy][cy * kCellTile + lx], *c1 = c0 + kCells;
                sum += (double)c0[1];
                sum += (double)c1[0];
                if (px == 0) sum += (double)c0[0];
                if (px == A.nX - 1) sum += (double)c1[1];
            };
            row(ly + 1, 0);
            row(ly, 1);
            if (py == 0) row(ly, 0);
            if (py == A.nY - 1) row(ly + 1, 1);
            store_f(static_cast<TO *>(A.img), (size_t)(s0 + sb + wave) * A.img_stride + (size_t)py * A.nX + px,
                    (float)(sum * (double)A.scale));
        }
    }
}

// First view of quarter r of the views: a multiple of 4 (whole staging batches).
__device__ __forceinline__ int view_quarter(int nViews, int r)
{
    return r == 4 ? nViews : min(4 * (int)(((long long)nViews * r + 8) / 16), nViews);
}

// Cell tile (tx, ty): cells tx*7-1 .. tx*7+6 (and likewise in y), output pixels tx*7 .. tx*7+6,
// slices [s0, s0 + S) (a ragged last group repeats its last slice).  Every thread of the
// workgroup calls it.
template <int S, typename TI, typename TO>
__device__ __forceinline__ void cell_tile(const FpaArgs &A, CellShared<S> &sh, int tx, int ty, int s0)
{
    static_assert(kCells == 64 && kWvSplit * kCells == kAdjThreads, "a tile's cells on the lanes of a wave");
    constexpr int kDw = WvStage<S>::kDw;
    // 16 slices: the next batch's rays are loaded into registers while the current ones are
    // evaluated (three waves per SIMD: 1.78 against 2.16 ms for 16 slices); with fewer slices the
    // other waves hide the loads, and the registers are worth more (1 slice 656 against 702 us)
    constexpr bool kAhead = S == 16;
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int lx, ly;
    tile_cell(lx, ly);
    const int ci = tx * kCellOut - 1 + lx, cj = ty * kCellOut - 1 + ly;  // >= -1
    const float fci = (float)ci, fcj = (float)cj;
    float *slots = sh.stage[wave].slot;
    const TI *sino[S];
#pragma unroll
    for (int s = 0; s < S; ++s)
        sino[s] = static_cast<const TI *>(A.sino) + (size_t)min(s0 + s, A.nSlices - 1) * A.sino_stride;
    // the tile's centre and this cell's offset from it (mm); cell c's centre is texel
    // coordinate c + 1/2, at (c + 1 - r) dx
    const float bx = ((float)(ci - lx) + 4.5f - A.r) * A.dx, by = ((float)(cj - ly) + 4.5f - A.r) * A.dx;
    const float dxl = ((float)lx - kWvHalf) * A.dx, dyl = ((float)ly - kWvHalf) * A.dx;

    // Of view vb + (lane & 15): a cell's first candidate is slot ceil(gx dxl + gy dyl + e) of the
    // view's window, which starts at column wlo; nit candidates follow one another.
    struct Model {
        float gx, gy, e;
        int nit, wlo;
    };
    // Models of the views [vb, min(vb + 16, vend)); returns the widest window among them.
    auto models = [&](int vb, int vend, Model &M, int &dirs) {
        const int v = min(vb + (lane & (kWvGroup - 1)), vend - 1);
        const BlockCand b = block_candidates(A, A.cs[v], bx, by, kCellRho, kWvHalf * A.dx);
        // candidates of a cell: ceil(cf - hw) and the following nit - 1 columns (no interval of
        // length 2 hw holds more integers; 0.001 and 0.01 cover the FP32 column coordinates)
        const float ext = kWvHalf * A.dx * (fabsf(b.gx) + fabsf(b.gy));
        const float nit = floorf(fmaf(2.0f, b.hw, 0.001f)) + 1.0f;
        const float lo = ceilf(b.cf - ext - b.hw - 0.01f);
        M.gx = b.gx, M.gy = b.gy, M.e = (b.cf - lo) - b.hw;
        M.wlo = (int)fminf(fmaxf(lo, -1.0e9f), 1.0e9f);
        // the signs of du (1: positive, 2: negative) and dw (4, 8) that every ray in reach of the
        // tile shares, in all the group's views (0: mixed): any slot read lies within hw + 2
        // columns of the cell's own, and samples run towards the source, against (dx, dy)
        const float sp = b.spread + (b.hw + 2.0f) * __builtin_amdgcn_rcpf(A.c_abs);
        dirs = (__all(b.dx < -sp) ? 1 : 0) | (__all(b.dx > sp) ? 2 : 0) | (__all(b.dy < -sp) ? 4 : 0) |
               (__all(b.dy > sp) ? 8 : 0);
        M.nit = (int)fminf(nit, 1.0e9f);
        float need = ceilf(M.e + ext + 0.01f) + nit;
        need = need < 1.0e9f ? need : 1.0e9f;  // also for a block at the source (not a number)
#pragma unroll
        for (int sh2 = 1; sh2 < kWvGroup; sh2 <<= 1) need = fmaxf(need, __shfl_xor(need, sh2));
        return __builtin_amdgcn_readfirstlane((int)need);
    };
    auto lane_f = [](float x, int k) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), k)); };

    float acc[4][S];
    float4 pg;  // the slot's next ray: u0, w0, du, dw,
    float2 pi;  // 1/du, 1/dw,
    int pn;     // samples,
    TI pv[S];   // and its values (storage bits: widened when they are written to LDS)
    auto load_ray = [&](bool ok, int v, int c) {
        pg = make_float4(0.0f, 0.0f, 0.0f, 0.0f), pi = make_float2(0.0f, 0.0f), pn = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) pv[s] = 0;
        if (ok) {
            const unsigned rb = (unsigned)v * (unsigned)A.nCols + (unsigned)c;
            pg = A.ray_geo[rb];
            pi = A.ray_inv[rb];
            pn = A.ray_n[rb];
#pragma unroll
            for (int s = 0; s < S; ++s) pv[s] = sino[s][rb];
        }
    };
    auto store_ray = [&]() {
        float *d = slots + lane * kDw;
        const float n = (float)pn, dd = pg.z * pg.w * (1.0f / 12.0f);
        wave_lds_order();  // the previous rays' reads
        *reinterpret_cast<float4 *>(d) = pg;
        *reinterpret_cast<float4 *>(d + 4) = make_float4(pi.x, pi.y, -pg.x * pi.x, -pg.y * pi.y);
        if constexpr (S >= 4) {
            *reinterpret_cast<float2 *>(d + 8) = make_float2(n, dd);
#pragma unroll
            for (int s = 0; s < S; s += 4)
                *reinterpret_cast<float4 *>(d + 12 + s) =
                    make_float4(widen(pv[s]), widen(pv[s + 1]), widen(pv[s + 2]), widen(pv[s + 3]));
        } else {
            *reinterpret_cast<float4 *>(d + 8) = make_float4(n, dd, widen(pv[0]), widen(pv[S - 1]));
        }
        wave_lds_order();
    };
    struct Ray {
        RayRec rec;
        float v[S];
    };
    auto read_ray = [&](const float *d, Ray &r) {
        r.rec.p = *reinterpret_cast<const float4 *>(d);
        r.rec.q = *reinterpret_cast<const float4 *>(d + 4);
        if constexpr (S >= 4) {
            r.rec.n = *reinterpret_cast<const float2 *>(d + 8);
#pragma unroll
            for (int s = 0; s < S; s += 4) {
                const float4 t4 = *reinterpret_cast<const float4 *>(d + 12 + s);
                r.v[s] = t4.x, r.v[s + 1] = t4.y, r.v[s + 2] = t4.z, r.v[s + 3] = t4.w;
            }
        } else {
            const float4 t4 = *reinterpret_cast<const float4 *>(d + 8);
            r.rec.n = make_float2(t4.x, t4.y);
            r.v[0] = t4.z;
            if constexpr (S == 2) r.v[1] = t4.w;
        }
    };
    float ulo = fci, uhi = fci + 1.0f, wlo = fcj, whi = fcj + 1.0f;  // boundaries in the order of the group's rays
    auto add_ray = [&](auto mixed, const Ray &ray, auto skip_empty) {
        constexpr bool kMixed = decltype(mixed)::value;
        const CellSums c = cell_sums<kMixed>(ray.rec, fci, fcj, kMixed ? fci : ulo, kMixed ? fci + 1.0f : uhi,
                                             kMixed ? fcj : wlo, kMixed ? fcj + 1.0f : whi);
        if (decltype(skip_empty)::value && c.n == 0.0f) return;
        const float r[4] = {c.n, c.n * c.ta, c.n * c.tm, c.n * c.g};
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int s = 0; s < S; ++s) acc[q][s] = fmaf(r[q], ray.v[s], acc[q][s]);
    };
    // nit >= 1 adjacent slots from d
    auto add_rays = [&](auto mixed, const float *d, int nit) {
        if constexpr (S <= 2) {  // two rays in flight
            for (; nit > 1; nit -= 2, d += 2 * kDw) {
                Ray r0, r1;
                read_ray(d, r0);
                read_ray(d + kDw, r1);
                add_ray(mixed, r0, std::false_type{});
                add_ray(mixed, r1, std::false_type{});
            }
            if (nit > 0) {
                Ray r;
                read_ray(d, r);
                add_ray(mixed, r, std::false_type{});
            }
        } else {
            do {
                Ray r;
                read_ray(d, r);
                add_ray(mixed, r, std::false_type{});
                d += kDw;
            } while (--nit > 0);
        }
    };

    // A view by itself: 64 columns at a time, each cell's range per lane, without the rays that have no
    // samples in the cell.  Where windows are wider than the slots.
    auto wide_view = [&](int v) {
        const BlockCand b = block_candidates(A, A.cs[v], bx, by, kCellRho, kWvHalf * A.dx);
        const float cf = fmaf(b.gx, dxl, fmaf(b.gy, dyl, b.cf));
        const int clo = (int)fmaxf(ceilf(cf - b.hw), 0.0f);
        const int chi = (int)fminf(floorf(cf + b.hw), (float)(A.nCols - 1));
        const float ext = kWvHalf * A.dx * (fabsf(b.gx) + fabsf(b.gy)) + b.hw + 0.01f;
        const int first = __builtin_amdgcn_readfirstlane((int)fmaxf(ceilf(b.cf - ext), 0.0f));
        const int last = __builtin_amdgcn_readfirstlane((int)fminf(floorf(b.cf + ext), (float)(A.nCols - 1)));
        for (int w = first; w <= last; w += kWvSlots) {
            load_ray(w + lane < A.nCols, v, w + lane);
            store_ray();
            for (int c = max(clo, w); c <= min(chi, w + kWvSlots - 1); ++c) {
                Ray r;
                read_ray(slots + (c - w) * kDw, r);
                add_ray(std::true_type{}, r, std::true_type{});
            }
        }
    };

    // Cells add rays that have no samples in them with weights 0, which would spread an infinity or NaN:
    // where there is one, the rest of its group of views (16 slices: all of the wave's views, found from
    // the sums) is taken view by view without such rays; the other sums come out the same.  (Looking at
    // the staged values costs 16 slices 1.5%, looking at the sums 8 slices 5%, in registers.)
    auto nonfinite = [&](auto &&value) {
        float most = fabsf(value(0));
#pragma unroll
        for (int s = 1; s < S; ++s) most = __builtin_elementwise_maximum(most, fabsf(value(s)));  // keeps NaN
        return __any(!(most < __builtin_inff())) != 0;
    };
    auto clear = [&]() {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int s = 0; s < S; ++s) acc[q][s] = 0.0f;
    };

    // Sums of the views [v_begin, v_end) into acc.
    auto run = [&](int v_begin, int v_end) {
        Model M;
        int dirs;
        int need = models(v_begin, v_end, M, dirs);
        int wd, nv, lm, lc;  // window width, views per batch, this lane's view and column in them
        auto set_window = [&]() {
            nv = __builtin_amdgcn_readfirstlane(need <= 16 ? 4 : need <= 21 ? 3 : need <= 32 ? 2 : 1);
            wd = __builtin_amdgcn_readfirstlane(need <= 16 ? 16 : need <= 21 ? 21 : need <= 32 ? 32 : 64);
            lm = (int)(lane >= wd) + (int)(lane >= 2 * wd) + (int)(lane >= 3 * wd);
            lc = lane - lm * wd;
        };
        auto load_batch = [&](int vb, int v0, int gend) {
            const int v = v0 + lm;
            const int c = __shfl(M.wlo, min(v - vb, kWvGroup - 1)) + lc;
            load_ray(lm < nv && v < gend && (unsigned)c < (unsigned)A.nCols, v, c);
        };
        set_window();
        if (kAhead && need <= kWvSlots) load_batch(v_begin, v_begin, min(v_begin + kWvGroup, v_end));
        bool one_by_one = false;
        for (int vb = v_begin; vb < v_end; vb += kWvGroup) {
            const int gend = min(vb + kWvGroup, v_end), vn = gend;
            const Model C = M;
            int left = vb;  // first view that is taken by itself
            if (need <= kWvSlots && !one_by_one) {
                left = gend;
                const int cwd = wd, cnv = nv, cdirs = dirs;
                ulo = cdirs & 2 ? fci + 1.0f : fci, uhi = cdirs & 2 ? fci : fci + 1.0f;
                wlo = cdirs & 8 ? fcj + 1.0f : fcj, whi = cdirs & 8 ? fcj : fcj + 1.0f;
                auto group = [&](auto mixed) {
                    for (int v0 = vb; v0 < gend; v0 += cnv) {
                        if (!kAhead) load_batch(vb, v0, gend);
                        store_ray();
                        if (!kAhead && nonfinite([&](int s) { return widen(pv[s]); })) {
                            left = v0;
                            break;
                        }
                        if constexpr (kAhead) {
                            if (v0 + cnv < gend) {
                                load_batch(vb, v0 + cnv, gend);
                            } else if (vn < v_end) {  // the next group's models and first batch
                                need = models(vn, v_end, M, dirs);
                                set_window();
                                if (need <= kWvSlots) load_batch(vn, vn, min(vn + kWvGroup, v_end));
                            }
                        }
                        const int nb = min(cnv, gend - v0);
                        for (int m = 0; m < nb; ++m) {
                            const int k = v0 + m - vb;
                            const float f = fmaf(lane_f(C.gx, k), dxl, fmaf(lane_f(C.gy, k), dyl, lane_f(C.e, k)));
                            add_rays(mixed, slots + ((int)ceilf(f) + m * cwd) * kDw, __builtin_amdgcn_readlane(C.nit, k));
                        }
                    }
                };
                // (one copy of the loop for 16 slices: the other costs a wave per SIMD)
                if (S < 16 && (cdirs & 3) && (cdirs & 12)) group(std::false_type{});
                else group(std::true_type{});
            }
            if (left < gend) {
                for (int v = left; v < gend; ++v) wide_view(v);
                if (kAhead && vn < v_end) {
                    need = models(vn, v_end, M, dirs);
                    set_window();
                    if (need <= kWvSlots) load_batch(vn, vn, min(vn + kWvGroup, v_end));
                }
            }
            if (!kAhead && vn < v_end) {
                need = models(vn, v_end, M, dirs);
                set_window();
            }
            if (kAhead && vn == v_end && !one_by_one && nonfinite([&](int s) { return acc[0][s]; })) {
                one_by_one = true;
                clear();
                vb = v_begin - kWvGroup;
            }
        }
    };

    clear();
    // cells outside the FOV disk hold no samples; a tile without any other cell skips the views
    if (__any(ci <= A.nX - 1 && cj <= A.nY - 1 && cell_in_fov(A, fci, fcj))) {
        const int v0 = view_quarter(A.nViews, wave), v1 = view_quarter(A.nViews, wave + 1);
        if (v0 < v1) run(v0, v1);
    }
    __syncthreads();  // the staging space turns into partial sums
    cell_combine<S, TO>(A, sh, acc, tx, ty, s0);
}

// Waves per SIMD that the registers are held to: one slice 667, 662, 668 us at 5, 6, 8; four 878,
// 835, 1234 (spills) at 5, 6, 8.
template <int S, typename TI, typename TO>
__global__ __launch_bounds__(kAdjThreads, S == 16 ? 2 : S == 8 ? 4 : 6) void fp_adjoint_cell_kernel(FpaArgs A, int slice0)
{
    __shared__ CellShared<S> sh;
    unsigned tx, ty, g;  // blocked, XCD-aware order (neighbouring tiles share staged columns in L2)
    xcd_blocked_tile(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gridDim.x, gridDim.y, gridDim.z,
                     tx, ty, g);
    cell_tile<S, TI, TO>(A, sh, (int)tx, (int)ty, slice0 + (int)g * S);
}

// Uneven batch: slice s has its own geometry (desc[s]); work item = (slice, tile), items
// of slice s are [prefix[s], prefix[s+1]).  A slice whose samples stay in the cells
// [-1, n-1] takes 7 x 7-pixel cell tiles, as a single-slice call does; any other slice
// TX x (256/TX) gather tiles.  A fixed grid strides over all items, the XCDs taking
// them in chunks of 64, and a slice's tiles run in blocked order, so the tiles resident
// on one XCD cover a compact part of one image and share their rays through its L2.
template <int TX, typename TI, typename TO>
__global__ __launch_bounds__(kAdjThreads, 6) void fp_adjoint_batch_kernel(const FpaSliceDesc *__restrict__ desc,
                                                                       const int *__restrict__ prefix, int n,
                                                                       int total, const TI *sino, TO *img)
{
    __shared__ CellShared<1> sh;
    const unsigned first = xcd_chunk(blockIdx.x, gridDim.x);
    for (unsigned at = first; at < (unsigned)total; at += gridDim.x) {  // (total < 2^31, the grid below 2^24)
        const int item = (int)at;
        int lo = 0, hi = n - 1;  // last slice with prefix[s] <= item
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (prefix[mid] <= item) lo = mid;
            else hi = mid - 1;
        }
        const FpaSliceDesc &d = desc[lo];
        FpaArgs A;
        A.sino = sino + d.sino_off;
        A.img = img + d.img_off;
        // the slice's tables, as workgroup-uniform global-memory pointers (read from the
        // descriptor they would be generic, per-lane addresses: flat loads)
        A.ray_geo = uniform_global(d.ray_geo);
        A.ray_n = uniform_global(d.ray_n);
        A.ray_inv = uniform_global(d.ray_inv);
        A.cs = uniform_global(d.cs);
        A.img_stride = 0;
        A.sino_stride = 0;
        A.nX = d.nX;
        A.nY = d.nY;
        A.nViews = d.nViews;
        A.nCols = d.nCols;
        A.nSlices = 1;
        A.scale = d.scale;
        A.r = d.r;
        A.dx = d.dx;
        A.R = d.R;
        A.c_scale = d.c_scale;
        A.c_off = d.c_off;
        A.c_abs = d.c_abs;
        A.far_x = d.far_x;
        A.far_y = d.far_y;
        const unsigned local = (unsigned)(item - prefix[lo]);
        unsigned tx, ty;
        if (adj_cells_fit(A.far_x, A.far_y)) {  // same test as the single-slice launch
            blocked_tile(local, adj_cell_tiles(A.nX), adj_cell_tiles(A.nY), tx, ty);
            cell_tile<1, TI, TO>(A, sh, (int)tx, (int)ty, 0);
            __syncthreads();  // sh is free again
        } else {
            blocked_tile(local, (A.nX + TX - 1) / TX, (A.nY + 256 / TX - 1) / (256 / TX), tx, ty);
            adjoint_tile<1, TX, TI, TO>(A, (int)tx, (int)ty, 0);
        }
    }
}

}  // namespace

template <int S, typename TI, typename TO>
static void launch_fpa_k(int groups, hipStream_t stream, const FpaArgs &A, int slice0)
{
    if (adj_cells_fit(A.far_x, A.far_y)) {
        const dim3 grid(adj_cell_tiles(A.nX), adj_cell_tiles(A.nY), groups);
        hipLaunchKernelGGL((fp_adjoint_cell_kernel<S, TI, TO>), grid, dim3(kAdjThreads), 0, stream, A, slice0);
        return;
    }
    const dim3 grid((A.nX + kAdjTx - 1) / kAdjTx, (A.nY + kAdjTy - 1) / kAdjTy, groups);
    if constexpr (S >= 4)
        hipLaunchKernelGGL((fp_adjoint_staged_kernel<S, TI, TO>), grid, dim3(kAdjThreads), 0, stream, A);
    else
        hipLaunchKernelGGL((fp_adjoint_kernel<S, TI, TO>), grid, dim3(kAdjThreads), 0, stream, A);
}

template <int S>
static fbct_status launch_fpa_t(fbct_dtype ti, fbct_dtype to, int groups, hipStream_t stream, const FpaArgs &A,
                                int slice0)
{
    if (ti == FBCT_F32 && to == FBCT_F32) launch_fpa_k<S, float, float>(groups, stream, A, slice0);
    else if (ti == FBCT_BF16 && to == FBCT_F32) launch_fpa_k<S, bf16_t, float>(groups, stream, A, slice0);
    else if (ti == FBCT_F32 && to == FBCT_BF16) launch_fpa_k<S, float, bf16_t>(groups, stream, A, slice0);
    else if (ti == FBCT_BF16 && to == FBCT_BF16) launch_fpa_k<S, bf16_t, bf16_t>(groups, stream, A, slice0);
    else return fail(FBCT_ERR_INVALID_ARGUMENT, "fbct_fp_adjoint: unknown storage type");
    return FBCT_OK;
}

fbct_status launch_fp_adjoint(const fbct_plan &p, const DeviceTables &t, const void *sino, fbct_dtype ti,
                              void *img, fbct_dtype to, int n, hipStream_t stream)
{
    FpaArgs A;
    A.sino = sino;
    A.img = img;
    A.ray_geo = t.ray_geo;
    A.ray_n = t.ray_n;
    A.ray_inv = t.ray_inv;
    A.cs = t.view_cs;
    A.img_stride = (long long)p.g.nX * p.g.nY;
    A.sino_stride = (long long)p.g.nViews * p.g.nCols;
    A.nX = p.g.nX;
    A.nY = p.g.nY;
    A.nViews = p.g.nViews;
    A.nCols = p.g.nCols;
    A.nSlices = n;
    A.scale = p.d.fp_scale;
    A.r = p.d.fpa_r;
    A.dx = p.g.dx;
    A.R = p.g.R;
    A.c_scale = p.d.fpa_c_scale;
    A.c_off = p.d.fpa_c_off;
    A.c_abs = fabsf(p.d.fpa_c_scale);
    A.far_x = p.d.fpa_far_x;
    A.far_y = p.d.fpa_far_y;
    const long long gx = (p.g.nX + kAdjTx - 1) / kAdjTx, gy = (p.g.nY + kAdjTy - 1) / kAdjTy;
    fbct_status st = FBCT_OK;
    if (adj_cells_fit(A.far_x, A.far_y)) {
        // Groups of 16 slices, the rest in groups of the next size up, padded with the last slice
        // (512 x 512: 1, 2, 4, 8, 16 slices take 630, 671, 829, 1139, 1747 us, and 603, 656, 835, 1117,
        // 1780 when the costs below were taken, so that 11 to 15 go as 16, but 9 and 10 as 8 and the rest); or all slices in one launch of one group size,
        // where the costs say so: a launch costs about its group's time on the tiles times (its
        // workgroups + 800), 800 standing for the time a launch takes that does not fill the chip
        // (64 x 64 over 90 views, 9 slices: 8 and 1 44 us, pairs 21; 73 x 73 over 102, 41 slices:
        // 16, 8 and 1 76 us, eights 34; 174 x 174 over 328, 21 slices: 207, eights 174; 256 x 256
        // over 360, 17 slices: 16 and 1 399, eights 464).
        static constexpr struct { int s; double time; } kGroups[] = {{1, 603}, {2, 656}, {4, 835}, {8, 1117}, {16, 1780}};
        const long long tiles = (long long)adj_cell_tiles(A.nX) * adj_cell_tiles(A.nY);
        auto cost = [&](int S, int groups) {
            for (const auto &k : kGroups)
                if (k.s == S) return k.time * ((double)(tiles * groups) + 800.0);
            return 0.0;
        };
        auto rule = [](int left) { return left >= 11 ? 16 : left >= 5 ? 8 : left >= 3 ? 4 : left; };
        double least = 0.0;
        for (int left = n; left > 0; left -= rule(left) * std::max(left / rule(left), 1))
            least += cost(rule(left), std::max(left / rule(left), 1));
        int all = 0;
        for (const auto &k : kGroups)
            if (const double c = cost(k.s, (n + k.s - 1) / k.s); c < least) least = c, all = k.s;
        for (int done = 0; done < n && st == FBCT_OK;) {
            const int left = n - done;
            const int S = all ? all : rule(left);
            const int groups = all ? (left + S - 1) / S : std::max(left / S, 1);
            if (S == 16) st = launch_fpa_t<16>(ti, to, groups, stream, A, done);
            else if (S == 8) st = launch_fpa_t<8>(ti, to, groups, stream, A, done);
            else if (S == 4) st = launch_fpa_t<4>(ti, to, groups, stream, A, done);
            else if (S == 2) st = launch_fpa_t<2>(ti, to, groups, stream, A, done);
            else st = launch_fpa_t<1>(ti, to, groups, stream, A, done);
            done += groups * S;
        }
    } else {
        // Slices that share the geometry are processed together when there are enough
        // workgroups left to fill the device.
        const long long tiles = gx * gy;
        if (n >= 16 && tiles * ((n + 15) / 16) >= 1024) st = launch_fpa_t<16>(ti, to, (n + 15) / 16, stream, A, 0);
        else if (n >= 8 && tiles * ((n + 7) / 8) >= 1024) st = launch_fpa_t<8>(ti, to, (n + 7) / 8, stream, A, 0);
        else if (n >= 4 && tiles * ((n + 3) / 4) >= 1024) st = launch_fpa_t<4>(ti, to, (n + 3) / 4, stream, A, 0);
        else if (n >= 2 && tiles * ((n + 1) / 2) >= 1024) st = launch_fpa_t<2>(ti, to, (n + 1) / 2, stream, A, 0);
        else st = launch_fpa_t<1>(ti, to, n, stream, A, 0);
    }
    if (st != FBCT_OK) return st;
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(FBCT_ERR_DEVICE, "fp_adjoint_kernel launch: %s", hipGetErrorString(e));
    return FBCT_OK;
}

template <int TX, typename TI, typename TO>
static void launch_fpa_batch_t(dim3 grid, hipStream_t stream, const BatchDevice &bd, const int *prefix, int n,
                               int total, const void *sino, void *img)
{
    hipLaunchKernelGGL((fp_adjoint_batch_kernel<TX, TI, TO>), grid, dim3(kAdjThreads), 0, stream, bd.fpa_desc, prefix, n,
                       total, static_cast<const TI *>(sino), static_cast<TO *>(img));
}

template <int TX>
static void launch_fpa_batch_x(fbct_dtype ti, fbct_dtype to, dim3 grid, hipStream_t stream, const BatchDevice &bd,
                               const int *prefix, int n, int total, const void *sino, void *img)
{
    if (ti == FBCT_F32 && to == FBCT_F32) launch_fpa_batch_t<TX, float, float>(grid, stream, bd, prefix, n, total, sino, img);
    else if (ti == FBCT_BF16 && to == FBCT_F32) launch_fpa_batch_t<TX, bf16_t, float>(grid, stream, bd, prefix, n, total, sino, img);
    else if (ti == FBCT_F32 && to == FBCT_BF16) launch_fpa_batch_t<TX, float, bf16_t>(grid, stream, bd, prefix, n, total, sino, img);
    else launch_fpa_batch_t<TX, bf16_t, bf16_t>(grid, stream, bd, prefix, n, total, sino, img);
}

fbct_status launch_fp_adjoint_batch(const fbct_batch &b, const BatchDevice &bd, const void *sino, fbct_dtype ti,
                                    void *img, fbct_dtype to, hipStream_t stream)
{
    const int n = (int)b.plans.size();
    int k = 0;
    while (k < kAdjNumTiles && kAdjTileX[k] != b.shape.adj_tile_x) ++k;
    if (k == kAdjNumTiles) return fail(FBCT_ERR_INVALID_ARGUMENT, "fbct_batch_fp_adjoint: tile width %d", b.shape.adj_tile_x);
    const int total = b.fpa_prefix[k][n];
    if (total == 0) return FBCT_OK;
    // (a grid holds fewer than 2^32 threads; beyond, its workgroups stride over the items)
    const long long most = b.shape.adj_wgs_per_cu == 0 ? 0xffffffffLL / kAdjThreads
                                                       : (long long)b.shape.adj_wgs_per_cu * bd.num_cu;
    const long long wgs = std::min<long long>(total, most);
    const dim3 grid((unsigned)wgs);
    const int *prefix = bd.fpa_prefix[k];
    switch (b.shape.adj_tile_x) {
    case 8: launch_fpa_batch_x<8>(ti, to, grid, stream, bd, prefix, n, total, sino, img); break;
    case 32: launch_fpa_batch_x<32>(ti, to, grid, stream, bd, prefix, n, total, sino, img); break;
    case 64: launch_fpa_batch_x<64>(ti, to, grid, stream, bd, prefix, n, total, sino, img); break;
    default: launch_fpa_batch_x<16>(ti, to, grid, stream, bd, prefix, n, total, sino, img); break;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(FBCT_ERR_DEVICE, "fp_adjoint_batch_kernel launch: %s", hipGetErrorString(e));
    return FBCT_OK;
}

}  // namespace fbct
