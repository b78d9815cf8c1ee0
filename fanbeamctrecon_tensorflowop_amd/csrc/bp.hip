// bp.hip -- pixel-driven fan-beam backprojection (plain and 1/L^2-weighted) and its
// transpose (gfx950).
//
// Reference: BackProjOneView_fan_curve_kernel, BP/transform.cu:67-95 (unweighted) and
// FBP/transform.cu:61-89 (times 1/(U^2+t^2)), launched once per view with a memcpy
// and a device sync per view (BP/transform.cu:110-118).
//
// Here one launch covers every view and a group of slices: a thread owns a pixel of S
// slices, loops over its views with the per-view (cos, sin) read as uniform scalars, computes the
// column coordinate, in-range decision, taps and weight once per (pixel, view) and
// applies them to the S slices, accumulates in registers and stores once.  Both taps of an
// update come in one load from global memory (few slices) or from columns staged in LDS; the
// 1-D texture's clamp-to-edge linear filter is reproduced with exact FP32 weights.
//
// atan(t/U) is evaluated as z + z^3 R(z^2) with a correction polynomial R fitted per
// plan over the range FOV pixels reach, |t/U| <= rFOV/sqrt(R^2 - rFOV^2) (relative error
// below 1e-8 before FP32 evaluation, about one ulp after); plans whose range needs more
// than 9 terms use atanf.
//
// The reference's hard cut-off 0 < xi < nCols is a discontinuity: where a pixel sits
// within 0.01 column of a fan edge the decision is retaken in FP64 (tangent test on
// U, t from FP64 pixel coordinates and FP64 cos/sin), so FP32 rounding of xi cannot
// flip it.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <type_traits>

#include "dtype.hpp"
#include "fbct_internal.hpp"

namespace fbct {
namespace {

struct BpArgs {
    const float *sino;
    float *img;
    const float2 *cs;
    const double2 *csd;
    const int2 *fov_row;  // per row the FOV pixel range (FP64 membership of the centres)
    long long img_stride, sino_stride;
    int nX, nY, nViews, nCols;
    float R, xmin, ymin, dx, dy;
    float xi_scale;
    // dShift - dLeft/dCol - 1/2 = ct_col + ct_offset, |ct_offset| <= 1/2: the column coordinate between the
    // column centres is formed relative to column ct_col (mid-detector as a rule), where its
    // FP32 rounding is that of the distance from it
    float ct_offset;
    int ct_col;
    int edge_exact;
    double tan_min, tan_max;
    float atan_c[kBpAtanMax];  // correction polynomial R(s), s = z^2, lowest order first
};

constexpr int kBpTx = 16, kBpTy = 16;
constexpr float kEdgeBand = 0.01f;  // columns

struct PixelGeo {
    float x, y;     // FP32 pixel centre (mm), as the reference computes it
    double xd, yd;  // FP64 pixel centre for edge decisions
};

__device__ __forceinline__ PixelGeo pixel_geo(const BpArgs &A, int i, int j)
{
    PixelGeo p;
    p.x = fmaf(A.dx, (float)i + 0.5f, A.xmin);
    p.y = fmaf(A.dy, (float)j + 0.5f, A.ymin);
    p.xd = (double)A.xmin + (double)A.dx * ((double)i + 0.5);
    p.yd = (double)A.ymin + (double)A.dy * ((double)j + 0.5);
    return p;
}

// atan(z) for |z| within the fitted range: z + z*s*R(s), s = z^2 (kNc terms of R);
// kNc = 0 calls atanf.
template <int kNc>
__device__ __forceinline__ float fan_atan(const BpArgs &A, float z)
{
    if constexpr (kNc == 0) {
        return atanf(z);
    } else {
        const float s = z * z;
        float r = A.atan_c[kNc - 1];
#pragma unroll
        for (int k = kNc - 2; k >= 0; --k) r = fmaf(r, s, A.atan_c[k]);
        return fmaf(z * s, r, z);
    }
}

// Column coordinate of the pixel in view v relative to the centre of column ct_col (xi_raw of
// BP/transform.cu:85 less 1/2 and ct_col), and the FP32 U, t.
template <int kNc>
__device__ __forceinline__ float column_of(const BpArgs &A, const PixelGeo &p, int v, float &U, float &t)
{
    const float2 cs = A.cs[v];
    U = fmaf(-p.y, cs.y, fmaf(-p.x, cs.x, A.R));  // projection onto the iso-ray
    t = fmaf(p.x, cs.y, -p.y * cs.x);             // distance to the centre ray
    return fmaf(fan_atan<kNc>(A, t * __builtin_amdgcn_rcpf(U)), A.xi_scale, A.ct_offset);
}

// The in-range decision 0 < xi < nCols.
__device__ __forceinline__ bool in_range(const BpArgs &A, const PixelGeo &p, int v, float ct)
{
    const float lo = -0.5f - (float)A.ct_col, hi = lo + (float)A.nCols;
    bool in = ct > lo && ct < hi;
    if (A.edge_exact && (fabsf(ct - lo) < kEdgeBand || fabsf(ct - hi) < kEdgeBand)) {
        const double2 c = A.csd[v];
        const double Ud = (double)A.R - p.xd * c.x - p.yd * c.y;
        const double td = p.xd * c.y - p.yd * c.x;
        in = (td - Ud * A.tan_min > 0.0) && (td - Ud * A.tan_max < 0.0);
    }
    return in;
}

// Linear interpolation position: ct clamped to the column centres; returns the left tap c0
// in [0, nCols-2] and the weight of c0+1.
__device__ __forceinline__ int interp_pos(const BpArgs &A, float ct, float &al)
{
    const float first = (float)-A.ct_col;
    const float cc = fminf(fmaxf(ct, first), first + (float)(A.nCols - 1));
    const float fc = fminf(floorf(cc), first + (float)max(A.nCols - 2, 0));
    al = cc - fc;
    return (int)fc + A.ct_col;
}

// Weights of the taps c0 and c0 + 1 of one view: (1 - al, al), times the fan-beam
// distance weight 1 / (U^2 + t^2) for the weighted (FBP) form, so that a slice's update
// is two FMAs.
template <bool kWeighted>
__device__ __forceinline__ void bp_tap_weights(float al, float U, float t, float &w0, float &w1)
{
    if constexpr (kWeighted) {
        const float w = __builtin_amdgcn_rcpf(fmaf(U, U, t * t));
        w1 = al * w;
        w0 = w - w1;
    } else {
        w1 = al;
        w0 = 1.0f - al;
    }
}

// Few slices (S = 1..4): a wave owns an 8 x 8 pixel block and reads its taps from global
// memory, both columns of an update (of all S slices, where they lie interleaved) in one
// load.  The W waves of a workgroup share the block and split the views (chunks of kBpChunk
// views dealt round-robin), so a small image still fills the chip; their FP32 partial sums
// meet in LDS and are added in FP64 in wave order.  A chunk's coordinates are computed together
// (independent chains, the loads of kBpChunk views in flight); when every active pixel of the
// wave lies between the centres of the first and the last column in all of them, which one
// comparison per view decides, the taps need no clamp and the update no in-range test.  Any
// other chunk takes the general path, view by view.
//
// Bound: VALU issue for one slice (about 36 instruction slots per update, a quarter of them two
// reciprocals; 512 x 512 pixels, 984 views: 177 us, and 284 us for the one-thread-per-pixel loop
// over all views that this replaces; 256 x 256, 360 views: 147 -> 24 us), for more slices the
// vector L1, which takes about 20 cycles per gathered load whatever its width: 224 / 327 / 431 us
// for 2 / 3 / 4 planes, 201 / 256 / 236 us interleaved (one, two and two loads per update).
constexpr int kBpBlk = 8;    // pixel block side: one pixel per lane
constexpr int kBpChunk = 4;  // views evaluated together

// taps c0 and c0 + 1 of S interleaved slices, as they lie in memory
template <int S>
struct __attribute__((packed, aligned(4))) TapPair {
    float v[2 * S];
};

template <bool kWeighted, bool kIl, int S, int kNc, int W>
__global__ __launch_bounds__(64 * W) void bp_direct_kernel(BpArgs A, int slice0)
{
    unsigned tbx, tby, g;
    xcd_blocked_tile(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gridDim.x, gridDim.y, gridDim.z,
                     tbx, tby, g);
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int i = (int)tbx * kBpBlk + (lane & 7), j = (int)tby * kBpBlk + (lane >> 3);
    const size_t sl = (size_t)slice0 + (size_t)S * g;
    const PixelGeo pg = pixel_geo(A, min(i, A.nX - 1), min(j, A.nY - 1));
    const int2 fr = A.fov_row[min(j, A.nY - 1)];
    const bool valid = i < A.nX && j < A.nY;
    constexpr int kSl = kIl ? S : 1;       // slices a tap holds
    constexpr int kPl = kIl ? 1 : S;       // planes read per update
    const float *sino[kPl];
#pragma unroll
    for (int s = 0; s < kPl; ++s) sino[s] = A.sino + (sl + s) * A.sino_stride;
    float acc[S];
#pragma unroll
    for (int s = 0; s < S; ++s) acc[s] = 0.0f;
    const float mid = 0.5f * (float)(A.nCols - 1), midr = mid - (float)A.ct_col;

    if (valid && i >= fr.x && i <= fr.y) {
        // one update by the general path
        auto update = [&](int v) {
            float U, t, al;
            const float ct = column_of<kNc>(A, pg, v, U, t);
            if (!in_range(A, pg, v, ct)) return;
            const int c0 = interp_pos(A, ct, al);
            const int c1 = min(c0 + 1, A.nCols - 1);
            float w0, w1;
            bp_tap_weights<kWeighted>(al, U, t, w0, w1);
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const float *P = sino[s / kSl] + (size_t)v * A.nCols * kSl + s % kSl;
                acc[s] = fmaf(w1, P[c1 * kSl], fmaf(w0, P[c0 * kSl], acc[s]));
            }
        };
        int v0 = wave * kBpChunk;
        for (; v0 + kBpChunk <= A.nViews; v0 += W * kBpChunk) {
            float ct[kBpChunk], U[kBpChunk], t[kBpChunk];
            bool ok = true;
#pragma unroll
            for (int m = 0; m < kBpChunk; ++m) {
                ct[m] = column_of<kNc>(A, pg, v0 + m, U[m], t[m]);
                ok = ok && fabsf(ct[m] - midr) < mid - kEdgeBand;
            }
            if (__all(ok)) {
                const size_t row = (size_t)v0 * A.nCols * kSl;
                TapPair<kSl> p[kBpChunk][kPl];
                float w0[kBpChunk], w1[kBpChunk];
#pragma unroll
                for (int m = 0; m < kBpChunk; ++m) {
                    const float fc = floorf(ct[m]);
                    const unsigned off = (unsigned)((int)fc + A.ct_col) * (4u * kSl);
#pragma unroll
                    for (int s = 0; s < kPl; ++s)
                        p[m][s] = load_at(
                            reinterpret_cast<const TapPair<kSl> *>(sino[s] + row + (size_t)m * A.nCols * kSl), off);
                    bp_tap_weights<kWeighted>(ct[m] - fc, U[m], t[m], w0[m], w1[m]);
                }
#pragma unroll
                for (int m = 0; m < kBpChunk; ++m)
#pragma unroll
                    for (int s = 0; s < S; ++s)
                        acc[s] = fmaf(w1[m], p[m][s / kSl].v[kSl + s % kSl], fmaf(w0[m], p[m][s / kSl].v[s % kSl], acc[s]));
            } else {
                for (int m = 0; m < kBpChunk; ++m) update(v0 + m);
            }
        }
        for (int v = v0; v < min(v0 + kBpChunk, A.nViews); ++v) update(v);
    }

    __shared__ float part[W][S][64];
#pragma unroll
    for (int s = 0; s < S; ++s) part[wave][s][lane] = acc[s];
    __syncthreads();
    // slice s of the block is summed by wave s mod W
    for (int s = wave; s < S; s += W) {
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < W; ++w) sum += (double)part[w][s][lane];
        if (valid) A.img[(sl + s) * A.img_stride + (size_t)j * A.nX + i] = (float)sum;
    }
}

// Staged variant for S = 8, 16 slices: per batch of kBpStageVB views the workgroup
// copies the 64 detector columns around its tile into LDS once (coalesced, the S slices
// of a column contiguous, so a tap of all S slices is S/4 16-byte LDS reads instead of
// S gathers).  The window of a view starts at the smallest column coordinate of the
// tile's four corner pixels (t/U, and so xi, is extremal at a corner; lane 4m + c
// evaluates corner c of view m); a pixel whose taps leave the window reads them from
// global memory.  A batch whose taps all lie in the window and between the detector's end
// columns runs without clamps and in-range tests, its views' coordinates computed together,
// as in bp_direct_kernel.  VG view groups of 256 threads each stage and sum every VG-th
// batch of the same tile (partial sums added in FP64 at the end), so that few tiles still
// fill the chip.
//
// Bound: VALU issue and the LDS reads, about even.  64 slices of 512 x 512 pixels, 984 views:
// 3.29 -> 2.33 ms by giving each wave an 8 x 8 block (its 16-byte reads stop conflicting: a
// 16 x 4 strip spans more columns than the 16 that fall in distinct bank groups) and by the
// batch path (4 independent chains instead of one).
constexpr int kBpStageCols = 64;
constexpr int kBpStageVB = 4;

template <int S>
struct BpStage {
    static constexpr int kPitch = S + 4;  // floats per staged column: 16-byte multiple, off the bank period
    float val[kBpStageVB][kBpStageCols][kPitch];
};

template <bool kWeighted, bool kIl, int S, int kNc, int VG>
__global__ __launch_bounds__(kBpTx *kBpTy *VG) void bp_staged_kernel(BpArgs A, int slice0)
{
    static_assert(S % 4 == 0, "a staged column is read four slices at a time");
    constexpr int VB = kBpStageVB, SQ = S / 4;
    __shared__ BpStage<S> stages[VG];
    unsigned tbx, tby, g;  // blocked, XCD-aware order (neighbouring tiles share staged columns in L2)
    xcd_blocked_tile(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gridDim.x, gridDim.y, gridDim.z,
                     tbx, tby, g);
    const int tx0 = (int)tbx * kBpTx, ty0 = (int)tby * kBpTy;
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6) & 3);
    const int vg = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 8));
    BpStage<S> &st = stages[vg];
    // each wave an 8x8 quarter of the tile, each 16 lanes of it a 4x4 block: the wave's taps
    // lie within 14 adjacent staged columns or so (8 pixels along the diagonal at 1.2 columns
    // a pixel), and 16 adjacent columns (pitch S + 4) start in different bank groups
    static_assert(kBpTx == 16 && kBpTy == 16, "lane layout assumes 16x16 tiles");
    const int i = tx0 + 8 * (wave & 1) + 4 * ((lane >> 4) & 1) + (lane & 3);
    const int j = ty0 + 8 * (wave >> 1) + 4 * (lane >> 5) + ((lane >> 2) & 3);
    const size_t sl = (size_t)slice0 + (size_t)S * g;
    // every thread of a tile with FOV pixels stages and waits
    const bool valid = i < A.nX && j < A.nY;
    const PixelGeo pg = pixel_geo(A, min(i, A.nX - 1), min(j, A.nY - 1));
    const int2 fr = A.fov_row[min(j, A.nY - 1)];
    const bool inside = valid && i >= fr.x && i <= fr.y;
    float *out = A.img + (size_t)j * A.nX + i;
    if (!__syncthreads_or(inside)) {
        if (valid && vg == 0)
            for (int s = 0; s < S; ++s) out[(sl + s) * A.img_stride] = 0.0f;
        return;
    }
    const PixelGeo pc = pixel_geo(A, min(tx0 + ((lane & 1) ? kBpTx - 1 : 0), A.nX - 1),
                                  min(ty0 + ((lane & 2) ? kBpTy - 1 : 0), A.nY - 1));
    const float *sino = A.sino + sl * A.sino_stride;  // slice group base
    // this wave stages slices wave*SQ..: planes of them, or (interleaved by four) a quarter
    // of a quad of slices (SQ < 4) or a quad (SQ = 4)
    constexpr int kSl = kIl ? 4 : 1;
    const float *sino_w = sino + (size_t)(wave * SQ / kSl * kSl) * A.sino_stride + wave * SQ % kSl;
    const unsigned sbytes = (unsigned)A.sino_stride * 4u;
    float acc[S];
#pragma unroll
    for (int s = 0; s < S; ++s) acc[s] = 0.0f;
    const float mid = 0.5f * (float)(A.nCols - 1), midr = mid - (float)A.ct_col;

    // Staging is software-pipelined: while a batch is read from LDS, the next batch's
    // columns are loaded into registers, and written to LDS between the two barriers that
    // follow.
    auto window = [&](int v0, int (&c_lo)[VB]) {
        float U, tt;
        const float ct = column_of<kNc>(A, pc, min(v0 + (lane >> 2) % VB, A.nViews - 1), U, tt);
        int wlo = (int)floorf(fminf(fmaxf(ct, -1.0e6f), 1.0e6f)) + A.ct_col;
#pragma unroll
        for (int sh = 1; sh <= 2; sh <<= 1) wlo = min(wlo, __shfl_xor(wlo, sh));
#pragma unroll
        for (int m = 0; m < VB; ++m)
            c_lo[m] = min(max(__builtin_amdgcn_readlane(wlo, 4 * m) - 1, 0), max(A.nCols - kBpStageCols, 0));
    };
    struct __attribute__((packed, aligned(4))) Cols {
        float v[SQ];
    };
    Cols q[VB];  // next batch: this wave's slices of lane's column, per view
    auto load_batch = [&](int v0, const int (&c_lo)[VB]) {
#pragma unroll
        for (int m = 0; m < VB; ++m) {
            // 32-bit byte offsets from the wave's first slice (the launch stages slice
            // groups only when four sinograms span less than 4 GiB)
            const unsigned off =
                ((unsigned)min(v0 + m, A.nViews - 1) * (unsigned)A.nCols + (unsigned)min(c_lo[m] + lane, A.nCols - 1)) *
                (4u * kSl);
            if constexpr (kIl) {
                q[m] = load_at(reinterpret_cast<const Cols *>(sino_w), off);
            } else {
#pragma unroll
                for (int k = 0; k < SQ; ++k) q[m].v[k] = load_at(sino_w, off + (unsigned)k * sbytes);
            }
        }
    };
    auto store_batch = [&](int v0, const int (&c_lo)[VB]) {
#pragma unroll
        for (int m = 0; m < VB; ++m) {
            if (v0 + m >= A.nViews || c_lo[m] + lane >= A.nCols) continue;
            float *dst = &st.val[m][lane][wave * SQ];
            if constexpr (SQ % 4 == 0) {
                *reinterpret_cast<float4 *>(dst) = make_float4(q[m].v[0], q[m].v[1], q[m].v[2], q[m].v[3]);
            } else if constexpr (SQ == 2) {
                *reinterpret_cast<float2 *>(dst) = make_float2(q[m].v[0], q[m].v[1]);
            } else {
                dst[0] = q[m].v[0];
            }
        }
    };
    // one update of view v0 + m by the general path
    auto update = [&](int v, int wlo, int m) {
        float U, tt, al;
        const float ct = column_of<kNc>(A, pg, v, U, tt);
        if (!in_range(A, pg, v, ct)) return;
        const int c0 = interp_pos(A, ct, al);
        float w0, w1;
        bp_tap_weights<kWeighted>(al, U, tt, w0, w1);
        const int lc = c0 - wlo;
        if ((unsigned)lc < (unsigned)(kBpStageCols - 1) && c0 + 1 < A.nCols) {
#pragma unroll
            for (int s = 0; s < S; ++s)
                acc[s] = fmaf(w1, st.val[m][lc + 1][s], fmaf(w0, st.val[m][lc][s], acc[s]));
        } else {
            const int c1 = min(c0 + 1, A.nCols - 1);
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const float *P = sino + (size_t)(s / kSl * kSl) * A.sino_stride + (size_t)v * A.nCols * kSl + s % kSl;
                acc[s] = fmaf(w1, P[c1 * kSl], fmaf(w0, P[c0 * kSl], acc[s]));
            }
        }
    };
    int c_lo[VB], c_nx[VB];
    window(vg * VB, c_nx);
    load_batch(vg * VB, c_nx);
    for (int vb = 0; vb < A.nViews; vb += VG * VB) {
        const int v0 = vb + vg * VB;
#pragma unroll
        for (int m = 0; m < VB; ++m) c_lo[m] = c_nx[m];
        __syncthreads();  // the previous batch's reads are done
        store_batch(v0, c_lo);
        __syncthreads();
        if (vb + VG * VB < A.nViews) {
            window(v0 + VG * VB, c_nx);
            load_batch(v0 + VG * VB, c_nx);
        }
        if (!inside) continue;
        if (v0 + VB <= A.nViews) {
            float ct[VB], U[VB], tt[VB];
            bool ok = true;
#pragma unroll
            for (int m = 0; m < VB; ++m) {
                ct[m] = column_of<kNc>(A, pg, v0 + m, U[m], tt[m]);
                ok = ok && fabsf(ct[m] - midr) < mid - kEdgeBand;
                ok = ok && (unsigned)((int)floorf(ct[m]) + (A.ct_col - c_lo[m])) < (unsigned)(kBpStageCols - 1);
            }
            if (__all(ok)) {
#pragma unroll
                for (int m = 0; m < VB; ++m) {
                    const float fc = floorf(ct[m]);
                    const int lc = (int)fc + (A.ct_col - c_lo[m]);
                    float w0, w1;
                    bp_tap_weights<kWeighted>(ct[m] - fc, U[m], tt[m], w0, w1);
                    const float *p = &st.val[m][lc][0];
#pragma unroll
                    for (int s = 0; s < S; s += 4) {
                        const float4 a = *reinterpret_cast<const float4 *>(p + s);
                        const float4 b = *reinterpret_cast<const float4 *>(p + BpStage<S>::kPitch + s);
                        acc[s] = fmaf(w1, b.x, fmaf(w0, a.x, acc[s]));
                        acc[s + 1] = fmaf(w1, b.y, fmaf(w0, a.y, acc[s + 1]));
                        acc[s + 2] = fmaf(w1, b.z, fmaf(w0, a.z, acc[s + 2]));
                        acc[s + 3] = fmaf(w1, b.w, fmaf(w0, a.w, acc[s + 3]));
                    }
                }
                continue;
            }
        }
#pragma unroll 1
        for (int m = 0; m < VB && v0 + m < A.nViews; ++m) {
            int wlo = c_lo[0];
#pragma unroll
            for (int k = 1; k < VB; ++k) wlo = m == k ? c_lo[k] : wlo;
            update(v0 + m, wlo, m);
        }
    }
    if constexpr (VG == 1) {
        if (!valid) return;
#pragma unroll
        for (int s = 0; s < S; ++s) out[(sl + s) * A.img_stride] = acc[s];
    } else {
        // the groups' partial sums meet in LDS; group g adds and stores slices g, g + VG, ...
        static_assert(sizeof(BpStage<S>) >= sizeof(float) * S * kBpTx * kBpTy, "partial sums fit the staging space");
        const int t = (int)threadIdx.x & 255;
        __syncthreads();
        float *part = &st.val[0][0][0];
#pragma unroll
        for (int s = 0; s < S; ++s) part[s * 256 + t] = acc[s];
        __syncthreads();
        for (int s = vg; s < S; s += VG) {
            double sum = 0.0;
#pragma unroll
            for (int w = 0; w < VG; ++w) sum += (double)(&stages[w].val[0][0][0])[s * 256 + t];
            if (valid) out[(sl + s) * A.img_stride] = (float)sum;
        }
    }
}

// ------------------------------------------------------------------ transpose
// BP^T: sino[v][c] = sum over FOV pixels p of img[p] w_p hat_c(xi_p), the transpose of
// the two-tap interpolation above (clamped taps folded into the edge columns, the
// 0 < xi < nCols cut kept; w_p = 1 or 1/(U^2+t^2)), gathered per (view, column), so every
// sum has a fixed order and no atomics are needed.
//
// Column c's taps come from the pixels whose column coordinate lies within one column of
// its node xi = c + 1/2, i.e. between the node rays of columns c - 1 and c + 1.  A node
// ray (theta = beta + gamma_c) is marched along image lines: rows or columns of pixels.
// On line k the ray crosses the other axis at pixel coordinate m*(k) = a k + b (one FP64
// FMA), and the candidates are the pixels within hw(k) = L*(k) tan|dCol| /
// ((|pd| - |pl| tan|dCol|) h) of m*(k), cut to the line's FOV range.  Each candidate's
// position relative to the node ray comes from its small offset Delta = (m - m*(k)) h
// along the line: perpendicular distance d = Delta pd, distance from the source
// L = L*(k) + Delta pl, and (xi - 1/2) - c = atan(d/L) / dCol = z (1 - z^2/3) / dCol,
// z = d/L (|z| is at most about tan|dCol|, so the next term is below 1e-9 column).  Every
// quantity is small, so the column offset is accurate to a few 1e-7 column, where an FP32
// column coordinate carries half an ulp of nCols (3e-5 column at 888 columns); that
// error, amplified about 70-fold by the ramp filter that follows in FBP^T, is what a
// scatter with the forward kernels' coordinate would leave.  Sums are FP32 over the lines
// of a chunk and FP64 across chunks, for the same reason.
//
// Work: a workgroup takes 64 adjacent columns (one per lane) of 4 adjacent views (a wave each;
// kSplit: of one view, whose lines the four waves share) and S slices.  Its rays march a
// common axis (the one its middle ray runs closest to) in chunks of 8 lines; per chunk the
// workgroup stages the pixels its candidates span -- the union of every ray's candidate
// range over the chunk's lines, each bound linear in k and so extreme at a chunk end --
// for its S slices in LDS, pixels outside the FOV disk as zeros, and each candidate is one LDS
// read of S slices.  The crossing m*(k) is followed in FP32 from the chunk's first line (exact
// products, so the fraction keeps an ulp of 1), and the number of candidates is the same for
// the wave: lanes with fewer, and lines outside a ray's range, read a zero pixel.  A ray more
// than 60 degrees off the axis (wide fans with few columns) is gathered on its own axis
// from global memory.
//
// Bound: VALU issue (0.6) and the latency of a chunk (two barriers, the staging loads, the
// candidates' chains).  With the distance weight, 512 x 512 pixels, 984 views, 888 columns, against
// two views per thread with a candidate loop per lane: 1 slice 805 -> 598 us, 4 slices 887 -> 682 us, 16
// slices 1.94 -> 1.62 ms; 256 x 256, 360 views, 512 columns, 1 slice 172 -> 104 us.  With 8 slices (1.12
// ms -> 884 us) float4 planes apart gave 3% (a 32-byte pixel made 16-byte reads conflict two-fold), the
// window sized by the plan instead of 160 pixels (four workgroups per CU instead of three) 15%.
// Against 64 bits the results are 5 to 18% closer than with a candidate's place from an FP64 crossing
// rounded to FP32 (RMS of 1 slice as above 5.9e-8 against 6.8e-8); the crossing in single FP32 steps was 4%
// faster and up to 13% further off than that.
struct BpaArgs {
    const float *img;
    float *sino;
    const double2 *csd;     // [nViews] cos, sin beta
    const double2 *col_csd; // [nCols] cos, sin gamma_c
    const int2 *fov_row, *fov_col;
    long long img_stride, sino_stride;
    int nX, nY, nViews, nCols, nSlices, win;
    unsigned cblocks, vgroups;  // workgroups along the columns and the views
    double R, xmin, ymin, dx, dy;
    double icol;       // 1/dCol
    float rFOV, tanc;  // rFOV, tan|dCol|
};

constexpr int kBpaChunk = 8;                 // lines per staged chunk
constexpr float kBpaTan = 0.0125f;           // 1.2 tan^4 < 2^-25
constexpr int kBpaFar = 1 << 24;             // beyond any window
constexpr int kBpaWin = 160;                 // most staged pixels per line

// A staged pixel of S slices lies in S / 4 planes of float4 (16 lanes that read adjacent pixels
// then cover all banks once), or in one plane of S floats.
template <int S> struct BpaPlane { using T = float4; };
template <> struct BpaPlane<1> { using T = float; };
template <> struct BpaPlane<2> { using T = float2; };

template <int S>
struct BpaTap {
    static constexpr int kP = S > 4 ? S / 4 : 1;
    typename BpaPlane<S>::T p[kP];
    __device__ __forceinline__ float operator[](int s) const { return reinterpret_cast<const float *>(p)[s]; }
};

// Node ray of one (view, column) on a marching axis.
struct BpaRay {
    double a, b;               // m*(k) = a k + b
    float L0, Ls, pd, pl, hwc;
    int klo, khi;              // lines holding candidates (klo > khi: none)
};

// The same for the staged chunks: a = a32 + da with a32 a multiple of 2^-23; pd, pl times the pixel
// pitch along the line; 1/dCol for these.
struct BpaStep {
    float a32, da, hpd, hpl, icol;
};

__device__ __forceinline__ void bpa_ray(const BpaArgs &A, double cth, double sth, double Rs, double Rc, bool along_y,
                                        BpaRay &r)
{
    double p0, ext;
    float h;
    if (along_y) {  // lines are image rows j; candidates along x
        const double cot = cth / sth, y0 = A.ymin + 0.5 * A.dy, xs0 = cot * y0 + Rs / sth;
        r.a = cot * A.dy / A.dx;
        r.b = (xs0 - A.xmin) / A.dx - 0.5;
        r.L0 = (float)(Rc - cth * xs0 - sth * y0);
        r.Ls = (float)(-A.dy / sth);
        r.pd = (float)sth, r.pl = (float)(-cth), h = (float)A.dx;
        p0 = -Rs * cth, ext = fabs(sth);
    } else {  // lines are image columns i; candidates along y
        const double tn = sth / cth, x0 = A.xmin + 0.5 * A.dx, ys0 = tn * x0 - Rs / cth;
        r.a = tn * A.dx / A.dy;
        r.b = (ys0 - A.ymin) / A.dy - 0.5;
        r.L0 = (float)(Rc - cth * x0 - sth * ys0);
        r.Ls = (float)(-A.dx / cth);
        r.pd = (float)(-cth), r.pl = (float)(-sth), h = (float)A.dy;
        p0 = Rs * sth, ext = fabs(cth);
    }
    const float apd = fabsf(r.pd) - fabsf(r.pl) * A.tanc;
    r.hwc = apd > 0.05f ? A.tanc / (apd * h) * 1.0001f : 1e9f;
    // lines holding candidates: points within delta of the node ray (delta bounds every
    // candidate's |d|) and inside the FOV disk have |s| <= H along the ray from its foot
    // Rs (sin th, -cos th); their coordinate on the marching axis is p0 + s dir +- delta
    const double delta = ((double)A.R + A.rFOV) * A.tanc * 1.01 + 2.0 * fmax(A.dx, A.dy);
    const double dn = fmax(fabs(Rs) - delta, 0.0);
    const double H2 = (double)A.rFOV * A.rFOV - dn * dn;
    if (!(H2 > 0.0)) {
        r.klo = 1, r.khi = 0;
        return;
    }
    const double span = sqrt(H2) * ext + delta * (along_y ? fabs(cth) : fabs(sth));
    const double org = along_y ? A.ymin : A.xmin, step = along_y ? A.dy : A.dx;
    const int n_major = along_y ? A.nY : A.nX;
    r.klo = max((int)floor((p0 - span - org) / step - 0.5) - 1, 0);
    r.khi = min((int)ceil((p0 + span - org) / step - 0.5) + 1, n_major - 1);
}

// Hat of column c in rel = (xi - 1/2) - c: 1 - |rel| on (-1, 1); the edge columns take
// the clamped taps (weight 1 for xi - 1/2 beyond their node) up to the cut 0 < xi < nCols.
struct BpaHat {
    float clo, chi, cut_lo, cut_hi, icol, c3;
};

// Calls fn(m, w) for the candidates m of line k (FOV range fr) of ray r, w the hat weight
// (times 1/L^2 for the weighted form); n_minor bounds the candidate range.
template <bool kWeighted, typename Fn>
__device__ __forceinline__ void bpa_line(const BpaRay &r, const BpaHat &hh, float h, int k, int2 fr, int n_minor, Fn &&fn)
{
    const double ms = fma(r.a, (double)k, r.b);
    const double mfl = floor(ms);
    const int mi = (int)mfl;
    const float mf = (float)(ms - mfl);
    const float Lk = fmaf((float)k, r.Ls, r.L0);
    const float hw = fminf(fmaf(Lk, r.hwc, 1.0e-3f), (float)(2 * n_minor + 2));
    const int lo = max(fr.x, mi + (int)ceilf(mf - hw));
    const int hi = min(fr.y, mi + (int)floorf(mf + hw));
    for (int m = lo; m <= hi; ++m) {
        const float dl = ((float)(m - mi) - mf) * h;
        const float d = dl * r.pd;
        const float L = fmaf(dl, r.pl, Lk);
        const float z = d * __builtin_amdgcn_rcpf(L);
        const float rel = z * fmaf(z * z, hh.c3, hh.icol);
        float w = 1.0f - fabsf(fminf(fmaxf(rel, hh.clo), hh.chi));
        w = (rel > hh.cut_lo && rel < hh.cut_hi) ? w : 0.0f;
        if constexpr (kWeighted) w *= __builtin_amdgcn_rcpf(fmaf(L, L, d * d));
        fn(m, w);
    }
}

// Reductions over the wave's 64 lanes by DPP (rows of 16 lanes by shifts, then across rows): the
// result is in lane 63, read back as a wave-uniform value.
template <typename Op>
__device__ __forceinline__ int wave_reduce(int x, Op &&op)
{
    x = op(x, __builtin_amdgcn_update_dpp(x, x, 0x111, 0xf, 0xf, false));  // row_shr:1
    x = op(x, __builtin_amdgcn_update_dpp(x, x, 0x112, 0xf, 0xf, false));  // row_shr:2
    x = op(x, __builtin_amdgcn_update_dpp(x, x, 0x114, 0xf, 0xf, false));  // row_shr:4
    x = op(x, __builtin_amdgcn_update_dpp(x, x, 0x118, 0xf, 0xf, false));  // row_shr:8
    x = op(x, __builtin_amdgcn_update_dpp(x, x, 0x142, 0xa, 0xf, false));  // row_bcast:15
    x = op(x, __builtin_amdgcn_update_dpp(x, x, 0x143, 0xc, 0xf, false));  // row_bcast:31
    return __builtin_amdgcn_readlane(x, 63);
}

__device__ __forceinline__ int wave_min(int x)
{
    return wave_reduce(x, [](int a, int b) { return min(a, b); });
}

__device__ __forceinline__ int wave_max(int x)
{
    return wave_reduce(x, [](int a, int b) { return max(a, b); });
}

// Slices [slice0 + S*g, +S) of the batch, g = the workgroup's slice group.  The waves per SIMD are what
// the LDS window leaves room for (one fewer, from 3 registers more: 4 slices 5%).
template <bool kWeighted, int S, bool kSplit>
__global__ __launch_bounds__(256, S == 8 ? 4 : S == 4 ? 6 : S == 2 ? 7 : 8) void bp_adjoint_staged_kernel(BpaArgs A, int slice0)
{
    constexpr int kLines = kBpaChunk / 4;  // kSplit: lines of a chunk per wave
    constexpr int kBpaViewsWg = kSplit ? 1 : 4;  // views per workgroup
    using TapT = BpaTap<S>;
    constexpr int kP = TapT::kP;
    // A.win staged pixels per line, and one more for the chunk, always zero: what a lane reads past
    // its own candidates
    extern __shared__ float4 bpa_lds[];
    auto *tile = reinterpret_cast<typename BpaPlane<S>::T *>(bpa_lds);
    const int zero_at = kBpaChunk * A.win, plane = zero_at + 1;
    auto put = [&](int at, const TapT &t) {
#pragma unroll
        for (int q = 0; q < kP; ++q) tile[q * plane + at] = t.p[q];
    };
    auto get = [&](int at) {
        TapT t;
#pragma unroll
        for (int q = 0; q < kP; ++q) t.p[q] = tile[q * plane + at];
        return t;
    };
    if (threadIdx.x == 0) put(zero_at, TapT{});
    __shared__ int2 fovc[kBpaChunk];  // FOV ranges of the chunk's lines
    __shared__ int red[2][4];
    // blocked, XCD-aware order over (column block, view group, slice group); the first two share the grid's
    // x, since either may exceed what its y holds
    unsigned cb, vg, g;
    xcd_blocked_tile(blockIdx.x + gridDim.x * blockIdx.z, A.cblocks, A.vgroups, gridDim.z, cb, vg, g);
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int c = (int)cb * 64 + lane;
    const bool cvalid = c < A.nCols;
    // the workgroup holds the first or the last column (uniform)
    const bool edge_wg = cb == 0 || (int)cb * 64 + 63 >= A.nCols - 1;
    const int cc = min(c, A.nCols - 1);
    const size_t sl = (size_t)slice0 + (size_t)S * g;
    const float *img = A.img + sl * A.img_stride;

    // the workgroup's marching axis: the one its middle ray runs closest to
    bool along_y;
    {
        const double2 vm = A.csd[min((int)vg * kBpaViewsWg + kBpaViewsWg / 2, A.nViews - 1)];
        const double2 cm = A.col_csd[min((int)cb * 64 + 32, A.nCols - 1)];
        along_y = fabs(vm.y * cm.x + vm.x * cm.y) >= fabs(vm.x * cm.x - vm.y * cm.y);
    }
    const double2 cg = A.col_csd[cc];
    const double Rs = A.R * cg.y, Rc = A.R * cg.x;
    BpaHat hh;
    hh.clo = c == 0 ? 0.0f : -3.0e38f;
    hh.chi = c == A.nCols - 1 ? 0.0f : 3.0e38f;
    hh.cut_lo = c == 0 ? -0.5f : -1.0f;
    hh.cut_hi = c == A.nCols - 1 ? 0.5f : 1.0f;
    hh.icol = (float)A.icol;
    hh.c3 = -hh.icol * (1.0f / 3.0f);

    BpaRay r;
    int kmin = INT_MAX, kmax = INT_MIN;
    const int v = kSplit ? (int)vg : (int)vg * kBpaViewsWg + wave;
    const double2 vb = A.csd[min(v, A.nViews - 1)];
    const double cth = vb.x * cg.x - vb.y * cg.y, sth = vb.y * cg.x + vb.x * cg.y;
    const bool own = (along_y ? fabs(sth) : fabs(cth)) < 0.5;  // marched on its own axis (far from the workgroup's)
    bpa_ray(A, cth, sth, Rs, Rc, own ? fabs(sth) >= fabs(cth) : along_y, r);
    if (!cvalid || v >= A.nViews) r.klo = 1, r.khi = 0;
    if (!own && r.klo <= r.khi) kmin = min(kmin, r.klo), kmax = max(kmax, r.khi);
    kmin = wave_min(kmin);
    kmax = wave_max(kmax);
    if (lane == 0) red[0][wave] = kmin, red[1][wave] = kmax;
    __syncthreads();
    const int Klo = min(min(red[0][0], red[0][1]), min(red[0][2], red[0][3]));
    const int Khi = max(max(red[1][0], red[1][1]), max(red[1][2], red[1][3]));
    __syncthreads();  // red is rewritten per chunk

    const int s_major = along_y ? A.nX : 1, s_minor = along_y ? 1 : A.nX;
    const int n_minor = along_y ? A.nX : A.nY, n_major = along_y ? A.nY : A.nX;
    const int2 *fov = along_y ? A.fov_row : A.fov_col;
    const float h = along_y ? (float)A.dx : (float)A.dy;
    // pixel off of the group's S slices: 32-bit byte offsets from the group's first image
    // (the launch keeps S images under 4 GiB)
    // (a padded group repeats its last slice)
    const unsigned sbytes = (unsigned)A.img_stride * (unsigned)sizeof(float);
    const int last = A.nSlices - 1 - (int)sl;
    auto load_taps = [&](unsigned off) {
        TapT t;
        float *tp = reinterpret_cast<float *>(t.p);
        const unsigned b = off * (unsigned)sizeof(float);
#pragma unroll
        for (int s = 0; s < S; ++s) tp[s] = load_f_at(img, b + (unsigned)min(s, last) * sbytes);
        return t;
    };
    // the rare global-memory paths (wide windows, rays on their own axis): one slice at a
    // time, so that they hold few registers (the scheduling barrier keeps the loads from
    // being hoisted together); the same FMAs in the same order as the staged path
    auto add_taps = [&](unsigned off, float w, float (&lacc)[S]) {
        const unsigned b = off * (unsigned)sizeof(float);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            lacc[s] = fmaf(w, load_f_at(img, b + (unsigned)min(s, last) * sbytes), lacc[s]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    double accd[S];
#pragma unroll
    for (int s = 0; s < S; ++s) accd[s] = 0.0;

    BpaStep st;
    st.a32 = (float)(rint(r.a * 0x1p23) * 0x1p-23);
    st.da = (float)(r.a - (double)st.a32);
    // (what rounds hpd would be an error of all of the ray's weights: icol takes it back)
    const double hpd = along_y ? A.dx * sth : -A.dy * cth;
    st.hpd = (float)hpd, st.hpl = (float)(along_y ? -A.dx * cth : -A.dy * sth);
    st.icol = (float)(A.icol * hpd / (double)st.hpd);

    // chunks at multiples of kBpaChunk lines: a ray's sums do not depend on its workgroup
    for (int k0 = Klo & ~(kBpaChunk - 1); k0 <= Khi; k0 += kBpaChunk) {
        const int k1 = min(k0 + kBpaChunk - 1, n_major - 1);
        // this thread's ray at the chunk's first line, the candidates per line, the same for the
        // wave (no interval of length 2 hw holds more), and the pixels these reach (bounds linear
        // in k: the ends suffice)
        int wlo = INT_MAX, whi = INT_MIN;
        const double m0 = fma(r.a, (double)k0, r.b);
        const double fl = floor(m0);
        // the crossing's fraction as a multiple of 2^-23 and the rest
        const float fr0 = (float)(floor((m0 - fl) * 0x1p23) * 0x1p-23);
        const float fr1 = (float)((m0 - fl) - (double)fr0);
        const int mi0 = (int)fl;
        const int ka = max(k0, r.klo), kb = min(k1, r.khi);
        const bool on = !own && ka <= kb;
        const float hwa = fmaf(fmaf((float)ka, r.Ls, r.L0), r.hwc, 1.0e-3f);
        const float hwb = fmaf(fmaf((float)kb, r.Ls, r.L0), r.hwc, 1.0e-3f);
        const float hw2 = on ? 2.0f * fmaxf(hwa, hwb) + 1.0e-3f : 0.0f;
        int nit = 1;
        while (nit < A.win && __any(hw2 >= (float)nit)) ++nit;
        if (on && !(hw2 < (float)A.win)) {
            wlo = -kBpaFar, whi = kBpaFar;
        } else if (on) {
            const float xa = fmaf((float)(ka - k0), st.a32, fr0) - hwa;
            const float xb = fmaf((float)(kb - k0), st.a32, fr0) - hwb;
            wlo = min(wlo, mi0 + (int)floorf(fminf(xa, xb)));
            whi = max(whi, mi0 + (int)ceilf(fmaxf(xa, xb)) + nit);
        }
        wlo = wave_min(wlo);
        whi = wave_max(whi);
        if (lane == 0) red[0][wave] = wlo, red[1][wave] = whi;
        __syncthreads();  // also: the previous chunk's reads of the tile are done
        const int mlo = min(min(red[0][0], red[0][1]), min(red[0][2], red[0][3])) - 1;
        const int mhi = max(max(red[1][0], red[1][1]), max(red[1][2], red[1][3])) + 1;
        if (mlo > mhi) {  // no candidates in this chunk (uniform)
            __syncthreads();
            continue;
        }
        // a window wider than the tile (wide fans): this chunk reads global memory
        const bool wide = (long long)mhi - mlo + 1 > A.win;
        const int nl = k1 - k0 + 1;
        if (wide) {
            if (threadIdx.x < (unsigned)nl) fovc[threadIdx.x] = fov[k0 + threadIdx.x];
        } else {
            const int nw = mhi - mlo + 1;
            // pixels outside the FOV disk (and outside the image) are staged as zeros.
            // rows (lines along x): a wave per line, lanes along it; columns: 8 lanes along
            // the chunk's lines, which are consecutive pixels of an image row
            static_assert(kBpaChunk == 8, "column staging puts the chunk's lines on 8 lanes");
            const TapT zero{};
            if (along_y) {
                for (int li = wave; li < nl; li += 4) {
                    const int2 f = fov[k0 + li];
                    for (int mm = lane; mm < nw; mm += 64) {
                        const int m = mlo + mm;
                        put(li * A.win + mm, m >= f.x && m <= f.y ? load_taps((unsigned)((k0 + li) * A.nX + m)) : zero);
                    }
                }
            } else {
                const int li = lane & 7;
                if (li < nl) {
                    const int2 f = fov[k0 + li];
                    for (int mm = (int)threadIdx.x >> 3; mm < nw; mm += 32) {
                        const int m = mlo + mm;
                        put(li * A.win + mm, m >= f.x && m <= f.y ? load_taps((unsigned)(m * A.nX + k0 + li)) : zero);
                    }
                }
            }
        }
        __syncthreads();  // tile ready
        if (!wide) {
            // general: the hat of any column and the weight at any column pitch; else max(1 - |rel|, 0)
            // and the series of narrow columns
            auto staged = [&](auto general) {
                constexpr bool kGen = decltype(general)::value;
                if (own || r.klo > r.khi) return;
                float lacc[S];
#pragma unroll
                for (int s = 0; s < S; ++s) lacc[s] = 0.0f;
                int row = mi0 - mlo + (kSplit ? wave * kLines * A.win : 0);
                const unsigned span = (unsigned)(r.khi - r.klo);
                const int kka = kSplit ? wave * kLines : 0, kkb = kSplit ? min(kka + kLines, nl) : nl;
                for (int kk = kka; kk < kkb; ++kk, row += A.win) {
                    const int k = k0 + kk;
                    // m* = mi0 + mint + mh + ml: mh is exact (kk a32 - mint and fr0 are multiples of
                    // 2^-23 below 2), and so are a candidate's dl = j0 + it - mh; ml, below 2^-22,
                    // enters d alone, which is rounded once, at its own size
                    const float kf = (float)kk;
                    const float mint = floorf(fmaf(kf, st.a32, fr0));
                    const float mh = fmaf(kf, st.a32, -mint) + fr0, mld = fmaf(kf, st.da, fr1) * st.hpd;
                    const float Lk = fmaf((float)k, r.Ls, r.L0);
                    const float hw = fmaf(Lk, r.hwc, 1.0e-3f);
                    const float j0 = ceilf(mh - hw);
                    const int at0 = row + (int)(mint + j0);
                    // candidates beyond hw, and all of a line outside the ray's range, read zeros
                    const float last_dl = (unsigned)(k - r.klo) <= span ? hw : -3.0e38f;
                    // (a candidate that reads zeros may lie at the source: its weight stays finite)
                    auto weight = [&](float dl, bool own_cand) {
                        const float L = fmaf(dl, st.hpl, Lk), d = fmaf(dl, st.hpd, -mld);
                        // z = d / L is the tangent of the angle off the column's ray, and rel =
                        // icol (z - z^3 / 3).  With the distance weight iq = 1 / (L^2 + d^2) the one
                        // reciprocal serves both: s = d L iq = z / (1 + z^2), rel = icol (s + 2/3 s^3)
                        // up to 1.2 s^4 of itself, |z| <= tan|dCol| < kBpaTan
                        constexpr bool kOne = kWeighted && !kGen;
                        const float iq = own_cand ? __builtin_amdgcn_rcpf(kOne ? fmaf(L, L, d * d) : L) : 0.0f;
                        const float z = kOne ? d * (L * iq) : d * iq;
                        const float rel = z * fmaf(z * z, kOne ? -2.0f * hh.c3 : hh.c3, st.icol);
                        float w;
                        if constexpr (kGen) {
                            w = 1.0f - fabsf(fminf(fmaxf(rel, hh.clo), hh.chi));
                            w = rel > hh.cut_lo && rel < hh.cut_hi ? w : 0.0f;
                        } else {
                            w = fmaxf(1.0f - fabsf(rel), 0.0f);
                        }
                        if constexpr (kWeighted && kGen) w = own_cand ? w * __builtin_amdgcn_rcpf(fmaf(L, L, d * d)) : 0.0f;
                        if constexpr (kOne) w *= iq;
                        return w;
                    };
                    const float dl0 = j0 - mh;
                    int it = 0;
                    for (; it + 2 <= nit; it += 2) {  // two independent chains
                        const float da = dl0 + (float)it, db = da + 1.0f;
                        const bool ia = da <= last_dl, ib = db <= last_dl;
                        const TapT ta = get(ia ? at0 + it : zero_at), tb = get(ib ? at0 + it + 1 : zero_at);
                        const float wa = weight(da, ia), wb = weight(db, ib);
#pragma unroll
                        for (int s = 0; s < S; ++s) lacc[s] = fmaf(wb, tb[s], fmaf(wa, ta[s], lacc[s]));
                    }
                    if (it < nit) {
                        const float da = dl0 + (float)it;
                        const bool ia = da <= last_dl;
                        const TapT ta = get(ia ? at0 + it : zero_at);
                        const float wa = weight(da, ia);
#pragma unroll
                        for (int s = 0; s < S; ++s) lacc[s] = fmaf(wa, ta[s], lacc[s]);
                    }
                }
#pragma unroll
                for (int s = 0; s < S; ++s) accd[s] += (double)lacc[s];
            };
            if (edge_wg || A.tanc >= kBpaTan) staged(std::true_type{});
            else staged(std::false_type{});
        } else {
            if (own) continue;
            float lacc[S];
#pragma unroll
            for (int s = 0; s < S; ++s) lacc[s] = 0.0f;
            for (int k = max(kSplit ? k0 + wave * kLines : k0, r.klo);
                 k <= min(kSplit ? min(k1, k0 + wave * kLines + kLines - 1) : k1, r.khi); ++k)
                bpa_line<kWeighted>(r, hh, h, k, fovc[k - k0], n_minor, [&](int m, float w) {
                    add_taps((unsigned)(k * s_major + m * s_minor), w, lacc);
                });
#pragma unroll
            for (int s = 0; s < S; ++s) accd[s] += (double)lacc[s];
        }
    }

    // rays far from the workgroup's axis: their own axis, taps from global memory, FP32
    // sums over 8 lines and FP64 across them (kSplit: the chunks dealt to the waves)
    if (own && r.klo <= r.khi) {
        const bool ay = fabs(sth) >= fabs(cth);
        const int sj = ay ? A.nX : 1, si = ay ? 1 : A.nX;
        const int nm = ay ? A.nX : A.nY;
        const int2 *fv = ay ? A.fov_row : A.fov_col;
        const float ho = ay ? (float)A.dx : (float)A.dy;
        for (int k0 = r.klo + (kSplit ? wave * kBpaChunk : 0); k0 <= r.khi; k0 += (kSplit ? 4 : 1) * kBpaChunk) {
            float lacc[S];
#pragma unroll
            for (int s = 0; s < S; ++s) lacc[s] = 0.0f;
            for (int k = k0; k <= min(k0 + kBpaChunk - 1, r.khi); ++k)
                bpa_line<kWeighted>(r, hh, ho, k, fv[k], nm, [&](int m, float w) {
                    add_taps((unsigned)(k * sj + m * si), w, lacc);
                });
#pragma unroll
            for (int s = 0; s < S; ++s) accd[s] += (double)lacc[s];
        }
    }

    if constexpr (kSplit) {  // the waves' lines, added in wave order
        double *part = reinterpret_cast<double *>(bpa_lds);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            __syncthreads();
            part[threadIdx.x] = accd[s];
            __syncthreads();
            accd[s] = (part[lane] + part[64 + lane]) + (part[128 + lane] + part[192 + lane]);
        }
        if (wave != 0) return;
    }
    if (!cvalid || v >= A.nViews) return;
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s <= last) A.sino[(sl + s) * A.sino_stride + (size_t)v * A.nCols + c] = (float)accd[s];
}

BpArgs make_args(const fbct_plan &p, const DeviceTables &t, const float *sino, float *img)
{
    BpArgs A;
    A.sino = sino;
    A.img = img;
    A.cs = t.view_cs;
    A.csd = t.view_csd;
    A.img_stride = (long long)p.g.nX * p.g.nY;
    A.sino_stride = (long long)p.g.nViews * p.g.nCols;
    A.nX = p.g.nX;
    A.nY = p.g.nY;
    A.nViews = p.g.nViews;
    A.nCols = p.g.nCols;
    A.R = p.g.R;
    A.xmin = p.g.xmin;
    A.ymin = p.g.ymin;
    A.dx = p.g.dx;
    A.dy = p.g.dy;
    A.fov_row = t.fov_row;
    A.xi_scale = p.d.bp_xi_scale;
    A.ct_offset = p.d.bp_ct_offset;
    A.ct_col = p.d.bp_ct_col;
    A.edge_exact = p.d.bp_edge_exact;
    A.tan_min = p.d.bp_tan_min;
    A.tan_max = p.d.bp_tan_max;
    for (int k = 0; k < kBpAtanMax; ++k) A.atan_c[k] = p.d.bp_atan_c[k];
    return A;
}

// Waves per block: the views are split until the launch has 8192 waves (8 per SIMD), at
// least 4 ways (256 x 256 pixels, one slice: 51, 31, 27, 24, 29 us with 1, 2, 4, 8, 16; 512 x
// 512: 216, 210, 180, 177, 231 us).
template <bool kWeighted, bool kIl, int S, int kNc>
void launch_bp_direct(const BpArgs &A, int groups, int slice0, hipStream_t stream)
{
    const dim3 grid((A.nX + kBpBlk - 1) / kBpBlk, (A.nY + kBpBlk - 1) / kBpBlk, groups);
    const long long blocks = (long long)grid.x * grid.y * groups;
    if (blocks * 4 >= 8192)
        hipLaunchKernelGGL((bp_direct_kernel<kWeighted, kIl, S, kNc, 4>), grid, dim3(64 * 4), 0, stream, A, slice0);
    else if (blocks * 8 >= 8192)
        hipLaunchKernelGGL((bp_direct_kernel<kWeighted, kIl, S, kNc, 8>), grid, dim3(64 * 8), 0, stream, A, slice0);
    else
        hipLaunchKernelGGL((bp_direct_kernel<kWeighted, kIl, S, kNc, 16>), grid, dim3(64 * 16), 0, stream, A, slice0);
}

// View groups per workgroup: 1 from four workgroups per CU on, 2 from two, else 4 (256 x 256
// pixels, 256 workgroups of 16 slices: 158, 100, 79 us with 1, 2, 4; 512 workgroups: 177, 131,
// 153; 512 x 512, 1024 workgroups: 591, 637, 759).
template <bool kWeighted, bool kIl, int S, int kNc>
void launch_bp_staged(const BpArgs &A, dim3 tiles, int groups, int slice0, hipStream_t stream)
{
    const dim3 grid(tiles.x, tiles.y, groups);
    const long long wgs = (long long)tiles.x * tiles.y * groups;
    constexpr int nt = kBpTx * kBpTy;
    if (wgs >= 1024)
        hipLaunchKernelGGL((bp_staged_kernel<kWeighted, kIl, S, kNc, 1>), grid, dim3(nt), 0, stream, A, slice0);
    else if (wgs >= 512)
        hipLaunchKernelGGL((bp_staged_kernel<kWeighted, kIl, S, kNc, 2>), grid, dim3(2 * nt), 0, stream, A, slice0);
    else
        hipLaunchKernelGGL((bp_staged_kernel<kWeighted, kIl, S, kNc, 4>), grid, dim3(4 * nt), 0, stream, A, slice0);
}

// Slice groups.  Interleaved (the filtered sinograms of FBP): 16 slices staged where the
// tiles fill the chip evenly -- four workgroups per CU or more, or a count close below a
// multiple of the CUs, since a CU left with one workgroup more than the others sets the time --
// else groups of four and the rest read directly (16 slices of 512 x 512: 558 us staged, 737
// direct; of 256 x 256, 256 tiles: 74 and 87; of 373 x 373, 576 tiles on 256 CUs: 242 and 211;
// of 96 x 96, 36 tiles: 26 and 13).  As planes [slice][view][column]: 16, then 8 slices staged
// from half a workgroup per CU on (8 slices of 512 x 512: 433 us staged, 859 direct; of 256 x
// 256: 57 and 91; of 96 x 96: 23 and 14), since the direct kernel gathers each slice.
template <bool kWeighted, bool kIl, int kNc>
void launch_bp_groups(const BpArgs &A, dim3 tiles, int n, hipStream_t stream)
{
    const long long nt = (long long)tiles.x * tiles.y;
    // the staged kernels address a wave's (up to 4) sinograms by 32-bit byte offsets
    const bool stage_ok = (unsigned long long)A.sino_stride * 16ull < (1ull << 32);
    const long long cus = 256;
    int done = 0;
    const int g16 = n / 16;
    const long long w16 = nt * g16;
    const bool fills = w16 >= 4 * cus || 100 * w16 >= 85 * cus * ((w16 + cus - 1) / cus);
    if (stage_ok && g16 > 0 && (kIl ? fills : w16 >= cus / 2)) {
        launch_bp_staged<kWeighted, kIl, 16, kNc>(A, tiles, g16, done, stream);
        done += 16 * g16;
    }
    if constexpr (!kIl) {
        const int g8 = (n - done) / 8;
        if (stage_ok && g8 > 0 && nt * g8 >= cus / 2) {
            launch_bp_staged<kWeighted, kIl, 8, kNc>(A, tiles, g8, done, stream);
            done += 8 * g8;
        }
    }
    for (int S : {4, 3, 2, 1}) {
        const int groups = (n - done) / S;
        if (groups == 0) continue;
        if (S == 4) launch_bp_direct<kWeighted, kIl, 4, kNc>(A, groups, done, stream);
        else if (S == 3) launch_bp_direct<kWeighted, kIl, 3, kNc>(A, groups, done, stream);
        else if (S == 2) launch_bp_direct<kWeighted, kIl, 2, kNc>(A, groups, done, stream);
        else launch_bp_direct<kWeighted, kIl, 1, kNc>(A, groups, done, stream);
        done += groups * S;
    }
}

template <bool kWeighted, bool kIl>
void launch_bp_nc(const BpArgs &A, int nc, int n, hipStream_t stream)
{
    const dim3 tiles((A.nX + kBpTx - 1) / kBpTx, (A.nY + kBpTy - 1) / kBpTy);
    if (nc == 9) launch_bp_groups<kWeighted, kIl, 9>(A, tiles, n, stream);
    else if (nc == 5) launch_bp_groups<kWeighted, kIl, 5>(A, tiles, n, stream);
    else launch_bp_groups<kWeighted, kIl, 0>(A, tiles, n, stream);
}

}  // namespace

fbct_status launch_bp(const fbct_plan &p, const DeviceTables &t, const float *sino, float *img, int n,
                      bool weighted, bool interleaved, hipStream_t stream)
{
    const BpArgs A = make_args(p, t, sino, img);
    const int nc = p.d.bp_atan_nc;
    if (interleaved) launch_bp_nc<true, true>(A, nc, n, stream);
    else if (weighted) launch_bp_nc<true, false>(A, nc, n, stream);
    else launch_bp_nc<false, false>(A, nc, n, stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(FBCT_ERR_DEVICE, "backprojection launch: %s", hipGetErrorString(e));
    return FBCT_OK;
}

fbct_status launch_bp_adjoint(const fbct_plan &p, const DeviceTables &t, const float *img, float *sino, int n,
                              bool weighted, hipStream_t stream)
{
    BpaArgs A;
    A.img = img;
    A.sino = sino;
    A.csd = t.view_csd;
    A.col_csd = t.col_csd;
    A.fov_row = t.fov_row;
    A.fov_col = t.fov_col;
    A.img_stride = (long long)p.g.nX * p.g.nY;
    A.sino_stride = (long long)p.g.nViews * p.g.nCols;
    A.nX = p.g.nX;
    A.nY = p.g.nY;
    A.nViews = p.g.nViews;
    A.nCols = p.g.nCols;
    A.R = p.g.R;
    A.xmin = p.g.xmin;
    A.ymin = p.g.ymin;
    A.dx = p.g.dx;
    A.dy = p.g.dy;
    A.rFOV = p.g.rFOV;
    A.tanc = p.d.bpa_tan;
    A.icol = 1.0 / (double)p.g.dCol;
    A.nSlices = n;
    // a group's images are addressed by 32-bit byte offsets: its S images stay below 4 GiB
    const unsigned long long img_bytes = (unsigned long long)p.g.nX * p.g.nY * sizeof(float);
    if (img_bytes >= (1ULL << 32))
        return fail(FBCT_ERR_UNSUPPORTED, "fbct_bp_adjoint: an image of %llu bytes exceeds 4 GiB", img_bytes);
    // Four views a workgroup, a wave each, or (split) one view whose lines the waves share.  Split
    // where few workgroups leave the chip idle -- 96 x 96 pixels, 130 views, 140 columns, 99
    // workgroups: 82 -> 26 us for one slice; 128 x 128, 200 workgroups: 63 -> 43 us; but 200 x 200,
    // 375 workgroups: 99 -> 76 us for one slice and 122 -> 127 us for eight, 256 x 256, 720
    // workgroups: 107 -> 132 us -- and where the rays of four views spread so far that some march
    // their own axis from global memory (96 x 96, 16 slices: 199 -> 42 us).  The rule looks at the
    // plan only, so that a slice's result does not depend on the slices with it.
    const double dcol = fabs((double)p.g.dCol), pitch = std::min(p.g.dx, p.g.dy);
    const double dview = p.g.nViews > 1 ? fabs((double)p.angles[p.g.nViews - 1] - p.angles[0]) / (p.g.nViews - 1) : 0.0;
    const int cblocks = (p.g.nCols + 63) / 64;
    const bool split = (long long)cblocks * ((p.g.nViews + 3) / 4) < 300 || 64.0 * dcol + 4.0 * dview > 0.52;
    A.cblocks = cblocks;
    A.vgroups = split ? p.g.nViews : (p.g.nViews + 3) / 4;
    // Staged pixels per line: what 64 columns reach at the far end of the FOV disk on a ray 45
    // degrees off the axis, the views' spread, a chunk's slant and margins; at most the image and
    // kBpaWin (wider windows read global memory)
    const double reach = 64.0 * dcol * ((double)p.g.R + p.g.rFOV) / (0.7 * pitch) + 16.0 +
                         (split ? 0.0 : 4.0 * dview * p.g.rFOV / (0.7 * pitch));
    A.win = (int)std::min(std::min(reach, 24.0 + std::max(p.g.nX, p.g.nY)), (double)kBpaWin);
    for (int done = 0; done < n;) {
        const int left = n - done;
        int S = left >= 5 ? 8 : left >= 3 ? 4 : left;  // padded with the last slice
        while ((unsigned long long)S * img_bytes >= (1ULL << 32)) S /= 2;
        const int groups = std::max(left / S, 1);
        const dim3 grid(A.cblocks * A.vgroups, 1, groups);
        const size_t lds = std::max(sizeof(float) * S * (kBpaChunk * (size_t)A.win + 1), sizeof(double) * 256);
#define FBCT_BPA(SS)                                                                                            \
    if (split && weighted) hipLaunchKernelGGL((bp_adjoint_staged_kernel<true, SS, true>), grid, dim3(256), lds, stream, A, done); \
    else if (split) hipLaunchKernelGGL((bp_adjoint_staged_kernel<false, SS, true>), grid, dim3(256), lds, stream, A, done); \
    else if (weighted) hipLaunchKernelGGL((bp_adjoint_staged_kernel<true, SS, false>), grid, dim3(256), lds, stream, A, done); \
    else hipLaunchKernelGGL((bp_adjoint_staged_kernel<false, SS, false>), grid, dim3(256), lds, stream, A, done)
        switch (S) {
        case 8: FBCT_BPA(8); break;
        case 4: FBCT_BPA(4); break;
        case 2: FBCT_BPA(2); break;
        default: FBCT_BPA(1); break;
        }
#undef FBCT_BPA
        done += groups * S;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(FBCT_ERR_DEVICE, "bp_adjoint_staged_kernel launch: %s", hipGetErrorString(e));
    return FBCT_OK;
}

}  // namespace fbct
