// cone_bp.hip -- voxel-driven cone-beam backprojection (gfx950).
//
// Reference: BackProjOneView_CB_EA_kernel (FDK/GPURecon_GPU.cu:15-50): a thread per
// (x, y) column computes U, t, the column index and 1/(U^2+t^2) once per view and
// loops over z with the row index ((z - zs) D / U - detBottom) / dRow, reading a 2-D
// clamp/linear texture; the host launches it once per view (:245-250).
//
// Here one launch covers all views and volumes.  A thread owns an (x, y) column of KZ
// voxels of one volume, accumulates its views in registers and stores once.  Per
// (column, view) the column coordinate, its taps and weight and the in-range decision
// are computed once; per voxel only the row coordinate (one fma), the taps and a
// bilinear blend.  Texture semantics are reproduced with exact FP32 weights; coordinates are
// relative to the detector's centre, where FP32 keeps their fraction.  Near the two fan edges the
// in-range decision is retaken in FP64 on t/U.
//
// Three kernels (choose() below says which):
//   * tile: a 16 x 16 pixel workgroup stages each view's footprint (a 16 x 16 x 16 voxel tile's
//     taps span about 30 x 25 detector samples, read by 4096 voxels) in LDS.  Large volumes.
//   * wave: a wave owns 8 x 8 pixels of 8 voxels and some of the views and stages its own
//     footprint, so nothing waits at a barrier and small volumes still fill the chip.
//   * direct: as wave, taps from global memory.  Thin volumes and steep row steps, where most
//     staged rows would not be read.

#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>

#include "dtype.hpp"
#include "fbct_internal.hpp"

namespace fbct {
namespace {

constexpr int kTx = 16, kTy = 16;
constexpr float kEdgeBand = 0.01f;  // columns

struct ConeArgs {
    const float *q;        // [n][nViews][nRows][nCols] filtered projections
    void *vol;             // TO[n][nZ][nY][nX]
    const float2 *cs;
    const double2 *csd;
    int nX, nY, nZ, nViews, nCols, nRows, nzc;
    long long gz0;  // first (z-chunk of a volume) of the launch
    float R, xmin, ymin, zmin, dx, dy, dz, r2;
    float xi_scale, ct_offset, zr_scale, rt_offset;  // coordinates relative to column ct_col, row rt_row
    int ct_col, rt_row;
    float ct_lo, ct_hi;  // the detector's edges on the relative column axis
    double tan_min, tan_max;
    float z_fit;  // the polynomial of atan holds for |t/U| <= z_fit, which covers the FOV disk
    float atan_c[kBpAtanMax];
};

template <int kNc>
__host__ __device__ __forceinline__ float fan_atan(const ConeArgs &A, float z)
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

// floor(v) as an integer in one instruction (v_cvt_flr_i32_f32); v is a finite row
// coordinate well inside the int range.
__device__ __forceinline__ int cvt_floor(float v)
{
    int r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

__host__ __device__ __forceinline__ int floor_to_int(float v)
{
    return (int)floorf(fminf(fmaxf(v, -1.0e6f), 1.0e6f));
}

__host__ __device__ __forceinline__ float reciprocal(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcpf(x);
#else
    return 1.0f / x;
#endif
}

// cos and sin of a uniform view's angle, by a scalar load: a vector load would wait behind the rows in
// flight (vector loads return in order).
__device__ __forceinline__ float2 view_cs(const ConeArgs &A, int v)
{
    typedef float f2 __attribute__((ext_vector_type(2)));
    const f2 c = ((const __attribute__((address_space(4))) f2 *)A.cs)[v];
    return make_float2(c.x, c.y);
}

// A voxel column's place in one view.
struct ColumnView {
    float ct;  // column coordinate relative to ct_col (texel centres at integers)
    float w;   // distance weight
    float a;   // row coordinate per unit z
    float U;   // distance from the source along the central ray
};

// kAnywhere: (x, y) may lie outside the FOV disk, where the polynomial of atan turns away from it; t/U
// is cut to the range it was fitted on.
template <bool kFlat, int kNc, bool kAnywhere = false>
__host__ __device__ __forceinline__ ColumnView column_view(const ConeArgs &A, float2 cs, float x, float y)
{
    const float U = fmaf(-y, cs.y, fmaf(-x, cs.x, A.R));
    const float t = fmaf(x, cs.y, -y * cs.x);
    const float rU = reciprocal(U);
    float z = t * rU;
    if constexpr (kAnywhere && !kFlat && kNc > 0) z = fminf(fmaxf(z, -A.z_fit), A.z_fit);
    ColumnView c;
    c.ct = fmaf(kFlat ? z : fan_atan<kNc>(A, z), A.xi_scale, A.ct_offset);
    c.w = kFlat ? rU * rU : reciprocal(fmaf(U, U, t * t));
    c.a = rU * A.zr_scale;
    c.U = U;
    return c;
}

// The reference's column test, retaken in FP64 near the two fan edges.
__device__ __forceinline__ bool in_view(const ConeArgs &A, int v, float ct, double xd, double yd)
{
    bool in = ct > A.ct_lo && ct < A.ct_hi;
    if (fabsf(ct - A.ct_lo) < kEdgeBand || fabsf(ct - A.ct_hi) < kEdgeBand) {
        const double2 d = A.csd[v];
        const double Ud = (double)A.R - xd * d.x - yd * d.y;
        const double td = xd * d.y - yd * d.x;
        in = (td - Ud * A.tan_min > 0.0) && (td - Ud * A.tan_max < 0.0);
    }
    return in;
}

// Elements o and o + 1 of a view in one 8-byte load: taps c0 and c0 + 1 <= nCols - 1 of a row.  Views
// of one column (!kPair) have one element a row.
struct __attribute__((packed, aligned(4))) TapPair {
    float l, r;
};
template <bool kPair>
__device__ __forceinline__ TapPair row_taps(const float *qv, unsigned o)
{
    if constexpr (!kPair) return TapPair{qv[o], qv[o]};
    else return *reinterpret_cast<const TapPair *>(reinterpret_cast<const char *>(qv) + 4u * o);
}

// KZ voxels of a column from global memory, any coordinates (clamp to edge).
template <int KZ, bool kPair = true>
__device__ __forceinline__ void column_global(const ConeArgs &A, const float *qv, float ct, float w, float rt0, float step,
                                              float (&acc)[KZ])
{
    const float cmin = -(float)A.ct_col, rmin = -(float)A.rt_row;
    const float cmax = cmin + (float)(A.nCols - 1), rmax = rmin + (float)(A.nRows - 1);
    const float cfl = cmin + (kPair ? (float)(A.nCols - 2) : 0.0f), rfl = rmin + (float)max(A.nRows - 2, 0);
    ct = fminf(fmaxf(ct, cmin), cmax);
    const float fc = fminf(floorf(ct), cfl);
    const float al = ct - fc;
    // row r of the relative axis starts at r nCols + org (modulo 2^32: a view is smaller)
    const unsigned nC = (unsigned)A.nCols, org = (unsigned)(A.ct_col + (int)fc) + (unsigned)A.rt_row * nC;
    const unsigned dr = A.nRows > 1 ? nC : 0u;
#pragma unroll
    for (int k = 0; k < KZ; ++k) {
        if (k % 4 == 0) asm volatile("" : "+v"(rt0)::"memory");  // four voxels' loads in flight
        const float rt = fminf(fmaxf(fmaf(step, (float)k, rt0), rmin), rmax);
        const float fr = fminf(floorf(rt), rfl);
        const float be = rt - fr;
        const unsigned o = (unsigned)(int)fr * nC + org;
        const TapPair p = row_taps<kPair>(qv, o), q = row_taps<kPair>(qv, o + dr);
        const float top = fmaf(al, p.r - p.l, p.l);
        const float bot = fmaf(al, q.r - q.l, q.l);
        acc[k] = fmaf(w, fmaf(be, bot - top, top), acc[k]);
    }
}

// Taps of KZ voxels from a staged window whose row and column 0 would be at byte `base` of LDS (row
// stride P floats), the whole column inside it.  Coordinates are not clamped: the staged rows and
// columns repeat the edges.  Rows are blended first, then the columns with weights w (1 - al), w al.
template <int KZ, int P>
__device__ __forceinline__ void column_staged(const ColumnView &c, float rt0, float step, unsigned base, float (&acc)[KZ])
{
    using LdsF = __attribute__((address_space(3))) const float;
    const float al = __builtin_amdgcn_fractf(c.ct);
    const float wr = c.w * al, wl = c.w - wr;
#pragma unroll
    for (int k = 0; k < KZ; ++k) {
        const float rt = fmaf(step, (float)k, rt0);
        const float be = __builtin_amdgcn_fractf(rt);
        LdsF *p = reinterpret_cast<LdsF *>((size_t)((unsigned)__mul24(cvt_floor(rt), 4 * P) + base));
        const float left = fmaf(be, p[P] - p[0], p[0]);
        const float right = fmaf(be, p[P + 1] - p[1], p[1]);
        acc[k] = fmaf(wl, left, fmaf(wr, right, acc[k]));
    }
}

// What one corner column of a tile says about a view's window: its column coordinate (least and
// greatest, apart where the window is not to be used) and its row coordinates at the ends of the
// z-chunk.  A corner outside the FOV disk is cut to the range of t/U that the disk's voxels keep to,
// and t/U and 1/U are extremal at a corner, so the corners bound every voxel of the disk in the tile.
// A corner at or behind the source, or rows beyond +-1e6 (where the window's ends would be cut), put
// the window off the detector.
struct Corner {
    float cn, cm, rn, rx;
};
template <bool kFlat, int kNc>
__host__ __device__ __forceinline__ Corner corner_of(const ConeArgs &A, float2 cs, int i, int j, float z0, float z1)
{
    const ColumnView c = column_view<kFlat, kNc, true>(A, cs, fmaf(A.dx, (float)i + 0.5f, A.xmin),
                                                       fmaf(A.dy, (float)j + 0.5f, A.ymin));
    const float ra = fmaf(z0, c.a, A.rt_offset), rb = fmaf(z1, c.a, A.rt_offset);
    const Corner k{c.ct, c.ct, fminf(ra, rb), fmaxf(ra, rb)};
    const bool usable = c.U > 1.0e-3f * A.R && k.rn > -1.0e6f && k.rx < 1.0e6f;
    return usable ? k : Corner{-1.0e6f, c.ct, k.rn, k.rx};
}

// The first and last column and row (relative to ct_col and rt_row) of a tile's taps in a view, from
// the extremes over its corners, with a margin of one sample, which absorbs the rounding between
// corner and voxel.
struct Range {
    int c0, c1, r0, r1;
};
__host__ __device__ __forceinline__ Range range_of(const Corner &k)
{
    return {floor_to_int(k.cn) - 1, floor_to_int(k.cm) + 2, floor_to_int(k.rn) - 1, floor_to_int(k.rx) + 2};
}
// Whether a tile is staged in a view: its window inside the detector's columns and at most `cols` x
// `rows`.
__host__ __device__ __forceinline__ bool is_staged(const ConeArgs &A, const Range &r, int cols, int rows)
{
    return r.c0 + A.ct_col >= 0 && r.c1 + A.ct_col < A.nCols && r.c1 - r.c0 < cols && r.r1 - r.r0 < rows;
}

// Windows of sixteen views, view vg + m's in lane 4m, corner c's evaluated by lane 4m + c.
struct Window {
    Range w;
    template <bool kFlat, int kNc>
    __device__ __forceinline__ void eval(const ConeArgs &A, int vg, int i0, int i1, int j0, int j1, float z0, float z1)
    {
        const int lane = (int)threadIdx.x & 63;
        const int v = min(vg + (lane >> 2), A.nViews - 1);
        Corner k = corner_of<kFlat, kNc>(A, A.cs[v], (lane & 1) ? i1 : i0, (lane & 2) ? j1 : j0, z0, z1);
#pragma unroll
        for (int sh = 1; sh <= 2; sh <<= 1) {
            k.cn = fminf(k.cn, __shfl_xor(k.cn, sh));
            k.cm = fmaxf(k.cm, __shfl_xor(k.cm, sh));
            k.rn = fminf(k.rn, __shfl_xor(k.rn, sh));
            k.rx = fmaxf(k.rx, __shfl_xor(k.rx, sh));
        }
        w = range_of(k);
    }
    // View vg + m's window (its first column and row and its rows), and whether the tile is staged.
    __device__ __forceinline__ bool view(const ConeArgs &A, int m, int cols, int rows, int &vc0, int &vr0, int &nrow) const
    {
        const Range r{__builtin_amdgcn_readlane(w.c0, 4 * m), __builtin_amdgcn_readlane(w.c1, 4 * m),
                      __builtin_amdgcn_readlane(w.r0, 4 * m), __builtin_amdgcn_readlane(w.r1, 4 * m)};
        vc0 = r.c0, vr0 = r.r0, nrow = r.r1 - r.r0 + 1;
        return is_staged(A, r, cols, rows);
    }
};

// The staged loops' columns: lanes outside the FOV disk evaluate the first column of the wave inside it
// (their own may lie outside the windows) and are not stored.
__device__ __forceinline__ float inside_column(float xy, bool active, unsigned long long in)
{
    const float first = __shfl(xy, in != 0 ? __builtin_ctzll(in) : 0);
    return active ? xy : first;
}

// The views of [vbeg, vend) in which a tile is not staged, from global memory.  (A pass of its own:
// the staged views' loop then updates its sums in one place, and reads taps well ahead of their use.)
template <bool kFlat, int kNc, int KZ>
__device__ __forceinline__ void unstaged_views(const ConeArgs &A, int vbeg, int vend, int i0, int i1, int j0, int j1, int i,
                                               int j, bool active, float z0, float z1, int cols, int rows, size_t vi,
                                               float (&acc)[KZ])
{
    const float x = fmaf(A.dx, (float)i + 0.5f, A.xmin);
    const float y = fmaf(A.dy, (float)j + 0.5f, A.ymin);
    const double xd = (double)A.xmin + (double)A.dx * ((double)i + 0.5);
    const double yd = (double)A.ymin + (double)A.dy * ((double)j + 0.5);
    const size_t view_elems = (size_t)A.nRows * A.nCols;
    Window win;
    for (int v = vbeg, m = 0; v < vend; ++v, m = (m + 1) % 16) {
        if (m == 0) win.eval<kFlat, kNc>(A, v, i0, i1, j0, j1, z0, z1);
        int c0, r0, nrow;
        if (win.view(A, m, cols, rows, c0, r0, nrow)) continue;
        const ColumnView c = column_view<kFlat, kNc>(A, view_cs(A, v), x, y);
        if (!active || !in_view(A, v, c.ct, xd, yd)) continue;
        column_global<KZ>(A, A.q + (vi * (size_t)A.nViews + (size_t)v) * view_elems, c.ct, c.w, fmaf(z0, c.a, A.rt_offset),
                          c.a * A.dz, acc);
    }
}

// Orders a wave's LDS accesses where its lanes read what others wrote, or write over what others read: the
// hardware completes them in program order, so nothing waits, but the compiler sees one lane's addresses
// and must not move them across.
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
}

// The wave kernels: a workgroup owns an 8 x 8 pixel tile of KZ voxels; its waves split the
// views and add their sums at the end (in wave order).  LDS: per wave `wave_floats` floats.
extern __shared__ float cone_lds[];

template <int KZ, typename TO>
__device__ __forceinline__ void store_columns(const ConeArgs &A, const float (&acc)[KZ], int i0, int j0, int k0, size_t vi,
                                              int wave_floats)
{
    const int lane = (int)threadIdx.x & 63;
    const int wave = (int)threadIdx.x >> 6, waves = (int)blockDim.x >> 6;
    TO *out = static_cast<TO *>(A.vol) + vi * (size_t)A.nZ * A.nY * A.nX;
    auto put = [&](int k, float v) {
        const int i = i0 + (lane & 7), j = j0 + (lane >> 3);
        if (i < A.nX && j < A.nY && k0 + k < A.nZ) store_f(out, ((size_t)(k0 + k) * A.nY + j) * A.nX + i, v);
    };
    float *mine = cone_lds + wave * wave_floats + lane;
    wave_lds_order();  // the last window's reads
#pragma unroll
    for (int k = 0; k < KZ; ++k) mine[64 * k] = acc[k];  // its own staging area: no wait for others
    __syncthreads();
    for (int k = wave; k < KZ; k += waves) {
        float v = 0.0f;
        for (int w = 0; w < waves; ++w) v += cone_lds[w * wave_floats + 64 * k + lane];
        put(k, v);
    }
}

// Bound by the L1's gather rate: about 20 cycles a wave load whatever its width, two loads (of both
// columns) a voxel.  64 x 64 x 4 voxels over 90 views 65 -> 12 us, 200 x 200 x 10 over 300 334 -> 131
// us (one wave a tile before, four loads a voxel).  Chunks of 4: 200 x 200 x 32 over 300 364 us, 397
// with chunks of 2, 411 with 8.
template <bool kFlat, int kNc, int KZ, bool kPair, typename TO>
__global__ __launch_bounds__(1024) void cone_bp_direct_kernel(ConeArgs A)
{
    unsigned t, gz;  // XCD-aware (tile, z-chunk of a volume): an XCD keeps whole z-chunks
    xcd_tile(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gridDim.x * gridDim.y, gridDim.z, t, gz);
    const int i0 = (int)(t % gridDim.x) * 8, j0 = (int)(t / gridDim.x) * 8;
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), waves = (int)blockDim.x >> 6;
    const int i = i0 + (lane & 7), j = j0 + (lane >> 3);
    const unsigned zg = (unsigned)A.gz0 + gz;
    const int k0 = (int)(zg % A.nzc) * KZ;
    const size_t vi = zg / A.nzc;
    const float x = fmaf(A.dx, (float)i + 0.5f, A.xmin);
    const float y = fmaf(A.dy, (float)j + 0.5f, A.ymin);
    const double xd = (double)A.xmin + (double)A.dx * ((double)i + 0.5);
    const double yd = (double)A.ymin + (double)A.dy * ((double)j + 0.5);
    const float z0 = fmaf(A.dz, (float)k0 + 0.5f, A.zmin);
    float acc[KZ];
#pragma unroll
    for (int k = 0; k < KZ; ++k) acc[k] = 0.0f;
    if (i < A.nX && j < A.nY && x * x + y * y <= A.r2) {
        const int v1 = A.nViews * (wave + 1) / waves;
        const size_t view_elems = (size_t)A.nRows * A.nCols;
        int v = A.nViews * wave / waves;
        const float *qv = A.q + (vi * (size_t)A.nViews + (size_t)v) * view_elems;
        for (; v < v1; ++v, qv += view_elems) {
            const ColumnView c = column_view<kFlat, kNc>(A, view_cs(A, v), x, y);
            if (!in_view(A, v, c.ct, xd, yd)) continue;
            column_global<KZ, kPair>(A, qv, c.ct, c.w, fmaf(z0, c.a, A.rt_offset), c.a * A.dz, acc);
        }
    }
    store_columns<KZ, TO>(A, acc, i0, j0, k0, vi, KZ * 64);
}

constexpr int kWaveKz = 8;
constexpr int kWaveRows = 32, kWaveCols = 32;  // staged window: two rows per load of a wave
constexpr int kWavePitch = 37;
constexpr int kWaveFloats = kWaveRows * kWavePitch;  // LDS per wave
static_assert(kWaveRows % 16 == 0, "staged sixteen rows at a time");
static_assert(kWaveFloats >= kWaveKz * 64, "a wave's sums fit its window");

// Bound by VALU issue and the L1 loads of its staging.  128 x 128 x 64 voxels over 180 views 686 ->
// 135 us (a launch of 128 workgroups of the tile kernel before), 128 x 128 x 32 over 200 397 -> 62 us,
// 400 x 400 x 64 over 500 at 2.5 rows a voxel 7.4 -> 2.8 ms.  Chunks of 16 with windows of 64 rows
// 133 us, of 32 185 us on the first, and 1.6 and 3.0 ms to 1.24 at 300 x 300 x 48 over 360; pitch 33:
// +17%, 45: +11%.  Eight waves per SIMD (SGPRs spill a little): 81 -> 63 us on the second.
template <bool kFlat, int kNc, typename TO>
__global__ __launch_bounds__(1024, 8) void cone_bp_wave_kernel(ConeArgs A)
{
    constexpr int P = kWavePitch, KZ = kWaveKz;
    unsigned t, gz;
    xcd_tile(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gridDim.x * gridDim.y, gridDim.z, t, gz);
    const int i0 = (int)(t % gridDim.x) * 8, j0 = (int)(t / gridDim.x) * 8;
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), waves = (int)blockDim.x >> 6;
    const int ie = min(i0 + 7, A.nX - 1), je = min(j0 + 7, A.nY - 1);
    // lanes past the image take its last pixels' coordinates and are not stored
    const int i = min(i0 + (lane & 7), ie), j = min(j0 + (lane >> 3), je);
    const unsigned zg = (unsigned)A.gz0 + gz;
    const int k0 = (int)(zg % A.nzc) * KZ;
    const size_t vi = zg / A.nzc;
    const float xp = fmaf(A.dx, (float)i + 0.5f, A.xmin);
    const float yp = fmaf(A.dy, (float)j + 0.5f, A.ymin);
    const bool active = xp * xp + yp * yp <= A.r2;
    const unsigned long long in = __ballot(active);
    const float x = inside_column(xp, active, in), y = inside_column(yp, active, in);
    const float z0 = fmaf(A.dz, (float)k0 + 0.5f, A.zmin);
    const float z1 = fmaf(A.dz, (float)(k0 + KZ - 1) + 0.5f, A.zmin);
    const int nC = A.nCols, nR = A.nRows;
    const size_t view_elems = (size_t)nR * nC;
    const unsigned row_bytes = 4u * (unsigned)nC;
    const float *qvol = A.q + vi * (size_t)A.nViews * view_elems;
    float *stage = cone_lds + wave * kWaveFloats;
    const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) float *)stage);
    float acc[KZ];
#pragma unroll
    for (int k = 0; k < KZ; ++k) acc[k] = 0.0f;

    const int vbeg = A.nViews * wave / waves;
    const int vend = in != 0 ? A.nViews * (wave + 1) / waves : vbeg;
    Window win;
    // staging of a window, two rows per load and sixteen rows at a time (a wave's LDS accesses
    // complete in order, so it waits for nothing but its own loads)
    const int lcol = lane & 31, lrow = lane >> 5;
    float *dst = stage + lrow * P + lcol;
    bool unstaged = false;
    for (int v = vbeg, m = 0; v < vend; ++v, m = (m + 1) % 16) {
        if (m == 0) win.eval<kFlat, kNc>(A, v, i0, ie, j0, je, z0, z1);
        int c0, r0, nrow;
        if (!win.view(A, m, kWaveCols, kWaveRows, c0, r0, nrow)) {
            unstaged = true;
            continue;
        }
        const float *qv = qvol + (size_t)v * view_elems;
        const ColumnView c = column_view<kFlat, kNc>(A, view_cs(A, v), x, y);
        const float rt0 = fmaf(z0, c.a, A.rt_offset), step = c.a * A.dz;
        const int gc = c0 + A.ct_col, gr = r0 + A.rt_row;  // the window's corner in the view
        const unsigned c4 = 4u * (unsigned)min(gc + lcol, nC - 1);
        for (int k = 0; k < nrow; k += 16) {
            float p[8];
            if (gr >= 0 && gr + k + 16 <= nR) {
                const float *qr = uniform_global(qv + (size_t)(gr + k) * nC);
                const unsigned o = c4 + (unsigned)lrow * row_bytes;
#pragma unroll
                for (int u = 0; u < 8; ++u) p[u] = load_at(qr + (size_t)(2 * u) * nC, o);
            } else {
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    p[u] = load_at(qv, (unsigned)min(max(gr + k + lrow + 2 * u, 0), nR - 1) * row_bytes + c4);
            }
            if (k == 0) wave_lds_order();  // the previous window's reads
#pragma unroll
            for (int u = 0; u < 8; ++u) dst[(k + 2 * u) * P] = p[u];
        }
        wave_lds_order();
        column_staged<KZ, P>(c, rt0, step, lds0 + 4u * (unsigned)(cvt_floor(c.ct) - c0 - r0 * P), acc);
    }
    if (unstaged)
        unstaged_views<kFlat, kNc, KZ>(A, vbeg, vend, i0, ie, j0, je, i, j, active, z0, z1, kWaveCols, kWaveRows, vi, acc);
#pragma unroll
    for (int k = 0; k < KZ; ++k) acc[k] = active ? acc[k] : 0.0f;
    store_columns<KZ, TO>(A, acc, i0, j0, k0, vi, kWaveFloats);
}

// Workgroup-tile kernel.  The workgroup's detector footprint per view is derived from the four
// corner columns of its 16 x 16 tile (t/U, and so the column coordinate, is extremal at a corner; the
// row coordinate at a corner and an end of the z-chunk), kTileGroup views at a time: lane 4m + c
// evaluates corner c of view m.  Per view the workgroup stages the footprint's rows once (one
// detector row per wave instruction, lane = column, indices clamped to the detector, which reproduces
// clamp-to-edge), and every voxel reads its four taps from LDS.  The next view's rows are loaded
// straight into the other half of the stage while the current one is evaluated: no registers, no
// stores, one barrier a view.  Tiles whose footprint is taller than kTileRows, wider than kTileCols
// or over a fan edge in a view take that view's taps from global memory.
//
// Bound by VALU issue (10 instructions a voxel) and the LDS reads (two ds_read2_b32).  512 x 512 x 256
// over 720 views 15.6 -> 14.9 ms, 300 x 300 x 256 over 360 3.09 -> 2.75 (rows through registers before,
// chunks of 32 voxels at four waves per SIMD); a window of 46 rows holds 16 voxels up to 1.7 rows
// apart anywhere and most at 2.2 (320 x 320 x 160 over 400 at 1.5 rows 3.15 -> 2.31 ms).  The row
// stride sets the bank conflicts (512 x 512 x 256: 65: 20.6 ms, 67: 19.6, 69: 17.5, 71: 15.9, 73 to 77:
// 14.9, 81: 15.3).  Staging (row, row difference) pairs would save two instructions a voxel, but their
// 16-byte reads at 8-byte alignment take twice the time (34.8 ms).
constexpr int kTileGroup = 16;     // views per footprint evaluation (64 lanes / 4 corners)
constexpr int kTileCols = 64;      // staged columns per row: one per lane
constexpr int kTileStride = 73;    // floats between staged rows
constexpr int kTileRows = 46, kTileKz = 16;

template <bool kFlat, int kNc, typename TO>
__global__ __launch_bounds__(kTx *kTy, 6) void cone_bp_tile_kernel(ConeArgs A)
{
    constexpr int kRows = kTileRows, RS = kTileStride, KZ = kTileKz;
    __shared__ float stage[2 * kRows * RS];
    unsigned t, gz;
    xcd_tile(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gridDim.x * gridDim.y, gridDim.z, t, gz);
    // tiles in blocked order: the footprints of those that run together overlap in an XCD's L2 (512 x
    // 512 x 256, 720 views: 15.3 -> 14.85 ms)
    unsigned tbx, tby;
    blocked_tile(t, gridDim.x, gridDim.y, tbx, tby);
    const int tx0 = (int)tbx * kTx, ty0 = (int)tby * kTy;
    // each wave takes an 8x8 pixel quarter of the tile: its taps spread over fewer staged
    // rows and columns than a 16x4 strip's (fewer LDS bank conflicts)
    static_assert(kTx == 16 && kTy == 16, "lane layout assumes 16x16 tiles");
    const int ie = min(tx0 + kTx - 1, A.nX - 1), je = min(ty0 + kTy - 1, A.nY - 1);
    const int iu = tx0 + 8 * (((int)threadIdx.x >> 6) & 1) + ((int)threadIdx.x & 7);
    const int ju = ty0 + 8 * ((int)threadIdx.x >> 7) + (((int)threadIdx.x >> 3) & 7);
    // threads past the image take its last pixels' coordinates and are not stored
    const int i = min(iu, ie), j = min(ju, je);
    const unsigned zg = (unsigned)A.gz0 + gz;
    const int k0 = (int)(zg % A.nzc) * KZ;
    const size_t vi = zg / A.nzc;
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const float xp = fmaf(A.dx, (float)i + 0.5f, A.xmin);
    const float yp = fmaf(A.dy, (float)j + 0.5f, A.ymin);
    const bool active = xp * xp + yp * yp <= A.r2;
    const unsigned long long in = __ballot(active);
    const bool wave_active = in != 0;
    const float x = inside_column(xp, active, in), y = inside_column(yp, active, in);
    // Row coordinate of voxel k: rt_k = rt_0 + k (dz a), rt_0 = z_0 a + rt_offset and
    // a = zr_scale / U -- one fma with k as an immediate.
    const float z0 = fmaf(A.dz, (float)k0 + 0.5f, A.zmin);
    const float z1 = fmaf(A.dz, (float)(k0 + KZ - 1) + 0.5f, A.zmin);
    float acc[KZ];
#pragma unroll
    for (int k = 0; k < KZ; ++k) acc[k] = 0.0f;
    const int nC = A.nCols, nR = A.nRows;
    const size_t view_elems = (size_t)nR * nC;
    const unsigned row_bytes = 4u * (unsigned)nC;
    const float *qvol = A.q + vi * (size_t)A.nViews * view_elems;

    Window win;
    // the next view's window (no rows: not staged)
    int nc0, nr0, nrow;
    bool unstaged = false;
    auto next_window = [&](int m) {
        if (!win.view(A, m, kTileCols, kRows, nc0, nr0, nrow)) {
            nrow = 0;
            unstaged = true;
        }
    };
    // rows of view v's window into half `h` of `stage`, wave w's rows w, w + 4, ...: loads straight to
    // LDS, one detector row each
    auto load_view = [&](int v, int h) {
        const char *qv = reinterpret_cast<const char *>(qvol + (size_t)v * view_elems);
        const unsigned c4 = 4u * (unsigned)min(max(nc0 + A.ct_col + lane, 0), nC - 1);
        const int gr = nr0 + A.rt_row;
        for (int r = wave; r < nrow; r += 4) {
            const char *row = qv + (size_t)((unsigned)min(max(gr + r, 0), nR - 1) * row_bytes);
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void *)(row + c4),
                (__attribute__((address_space(3))) void *)(stage + (h * kRows + r) * RS), 4, 0, 0);
        }
    };
    win.template eval<kFlat, kNc>(A, 0, tx0, ie, ty0, je, z0, z1);
    next_window(0);
    load_view(0, 0);
    for (int v = 0, m = 0; v < A.nViews; ++v) {
        const int c0 = nc0, r0 = nr0;
        const bool staged = nrow > 0;
        // this view's rows have arrived, and the other half's reads are done
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (v + 1 < A.nViews) {
            m = (m + 1) % kTileGroup;
            if (m == 0) win.template eval<kFlat, kNc>(A, v + 1, tx0, ie, ty0, je, z0, z1);
            next_window(m);
            load_view(v + 1, (v + 1) & 1);
        }
        if (!wave_active || !staged) continue;
        const ColumnView c = column_view<kFlat, kNc>(A, view_cs(A, v), x, y);
        const float rt0 = fmaf(z0, c.a, A.rt_offset), step = c.a * A.dz;
        const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) float *)stage);
        column_staged<KZ, RS>(c, rt0, step, lds0 + 4u * (unsigned)(cvt_floor(c.ct) - c0 + ((v & 1) * kRows - r0) * RS), acc);
    }
    if (unstaged && wave_active)
        unstaged_views<kFlat, kNc, KZ>(A, 0, A.nViews, tx0, ie, ty0, je, i, j, active, z0, z1, kTileCols, kRows, vi, acc);
    if (iu >= A.nX || ju >= A.nY) return;
    TO *out = static_cast<TO *>(A.vol) + vi * (size_t)A.nZ * A.nY * A.nX + (size_t)ju * A.nX + iu;
#pragma unroll
    for (int k = 0; k < KZ; ++k)
        if (k0 + k < A.nZ) store_f(out, (size_t)(k0 + k) * A.nY * A.nX, active ? acc[k] : 0.0f);
}

template <bool kFlat, int kNc>
void launch_tile(dim3 grid, hipStream_t st, const ConeArgs &A, fbct_dtype to)
{
    if (to == FBCT_BF16)
        hipLaunchKernelGGL((cone_bp_tile_kernel<kFlat, kNc, bf16_t>), grid, dim3(kTx * kTy), 0, st, A);
    else
        hipLaunchKernelGGL((cone_bp_tile_kernel<kFlat, kNc, float>), grid, dim3(kTx * kTy), 0, st, A);
}

template <bool kFlat, int kNc, int KZ, bool kPair = true>
void launch_direct(dim3 grid, int waves, hipStream_t st, const ConeArgs &A, fbct_dtype to)
{
    const size_t lds = (size_t)waves * KZ * 64 * sizeof(float);
    if (to == FBCT_BF16)
        hipLaunchKernelGGL((cone_bp_direct_kernel<kFlat, kNc, KZ, kPair, bf16_t>), grid, dim3(64 * waves), lds, st, A);
    else
        hipLaunchKernelGGL((cone_bp_direct_kernel<kFlat, kNc, KZ, kPair, float>), grid, dim3(64 * waves), lds, st, A);
}

template <bool kFlat, int kNc>
void launch_wave(dim3 grid, int waves, hipStream_t st, const ConeArgs &A, fbct_dtype to)
{
    const size_t lds = (size_t)waves * kWaveFloats * sizeof(float);
    if (to == FBCT_BF16)
        hipLaunchKernelGGL((cone_bp_wave_kernel<kFlat, kNc, bf16_t>), grid, dim3(64 * waves), lds, st, A);
    else
        hipLaunchKernelGGL((cone_bp_wave_kernel<kFlat, kNc, float>), grid, dim3(64 * waves), lds, st, A);
}

// Which kernel takes a volume, its voxels per thread along z and (direct, wave) its waves per tile.
struct ConeLaunch {
    enum { kDirect, kOneColumn, kWave, kTile } kind;
    int kz, waves;
};

template <bool kFlat, int kNc>
void launch_nc(const ConeLaunch &L, dim3 grid, hipStream_t st, const ConeArgs &A, fbct_dtype to)
{
    if (L.kind == ConeLaunch::kTile) {
        launch_tile<kFlat, kNc>(grid, st, A, to);
    } else if (L.kind == ConeLaunch::kWave) {
        launch_wave<kFlat, kNc>(grid, L.waves, st, A, to);
    } else {
        if (L.kind == ConeLaunch::kOneColumn) launch_direct<kFlat, kNc, 32, false>(grid, L.waves, st, A, to);
        else if (L.kz == 4) launch_direct<kFlat, kNc, 4>(grid, L.waves, st, A, to);
        else if (L.kz == 2) launch_direct<kFlat, kNc, 2>(grid, L.waves, st, A, to);
        else launch_direct<kFlat, kNc, 1>(grid, L.waves, st, A, to);
    }
}

// The rule looks at the plan only, so that a volume's result does not depend on the volumes it
// is called with.  `step` is the detector rows between two voxels of a column at the centre.
//
// The workgroup tile does the least work per voxel but needs four workgroups per CU to hide its
// barriers, and its voxels' rows in its window (step 2.2: rows are magnified up to half as much
// again near the source).  192 x 192 x 128 over 300 views (1152 workgroups): tile 660 us, wave 715;
// 160 x 160 x 160 over 250 (1000): 501, 505; 200 x 200 x 64 over 300 (676): 494, 353; 128 x 128 x 64
// over 180 (256): 381, 135; 400 x 400 x 64 over 500 at step 2.46 (2500): 3.74 ms, 2.8.
//
// Wave or direct: a staged voxel costs 0.3 + 0.17 step of a gathered one (rows are staged whether
// voxels use them or not), over z-chunks of 8 or of 4 and less.  128 x 128 x 32 over 200, step
// 1.23: wave 62 us, direct 107; 256 x 256 x 20 over 400, step 3.9: 481, 509; 200 x 200 x 10 over
// 300, step 4.9: 204, 129; 64 x 64 x 4 over 90: 14, 12.
//
// Waves per tile: sixteen for wave (400 x 400 x 64 over 500: 2.8 ms, eight 3.4, four 3.7) and where
// there are fewer than 512 tiles (direct, 64 x 64 x 16 over 120 views: 15 us, eight 18), else eight.
// With few views each wave's share gets short beside its windows' evaluation and the sum over the
// waves: from 1500 tiles on wave takes eight below a twelfth of the tiles (180 x 180 x 86, 5819 tiles: 90
// views 119 us, sixteen 143; 250: 294, 328; 500: 602, 625; 720: 1037, 952; curved 128 x 128 x 64, 2048
// tiles: 90 views 71, 75; 180: 146, 145) and four below 56 (24 views: 40 us, eight 46, sixteen 68; 64: 85,
// 89, 110), from 700 on eight below 64 (128 x 128 x 32, 40 views: 23 us, sixteen 26; 90: 43, 45; 180: 92,
// 81) and four below 32; direct four below 32 (200 x 200 x 64, 12 views: 30 us, eight 36; 24: 53, 53).
ConeLaunch choose(const fbct_cone_geom &g, double zr_scale)
{
    auto chunks = [&](int kz) { return (long long)((g.nZ + kz - 1) / kz); };
    const long long tiles = (long long)((g.nX + kTx - 1) / kTx) * ((g.nY + kTy - 1) / kTy);
    const double step = std::fabs((double)g.dz * zr_scale / g.R);
    if (g.nCols < 2) return {ConeLaunch::kOneColumn, 32, 4};
    if (g.nZ >= 16 && step < 2.2 && tiles * chunks(kTileKz) > 1024) return {ConeLaunch::kTile, kTileKz, 4};
    // a chunk's column geometry costs about 0.6 of a voxel
    int kz = 4;
    for (int k : {2, 1})
        if (chunks(k) * (k + 0.6) < chunks(kz) * (kz + 0.6)) kz = k;
    const bool wave = chunks(kWaveKz) * kWaveKz * (0.3 + 0.17 * step) < (double)chunks(kz) * kz;
    if (wave) kz = kWaveKz;
    const long long wgs = (long long)((g.nX + 7) / 8) * ((g.nY + 7) / 8) * chunks(kz);
    const int few = g.nViews < 32 ? 4 : 8;
    int waves = 16;
    if (!wave && wgs >= 512) waves = few;
    else if (wave && wgs >= 1500 && 12LL * g.nViews < wgs) waves = g.nViews < 56 ? 4 : 8;
    else if (wave && wgs >= 700 && g.nViews < 64) waves = few;
    return {wave ? ConeLaunch::kWave : ConeLaunch::kDirect, kz, waves};
}

}  // namespace

// The launch's arguments that the plan fixes; `cs` and `csd`: its angles, on the device or (csd unused) on
// the host.
static ConeArgs cone_args(const fbct_cone_plan &p, const float2 *cs, const double2 *csd)
{
    const fbct_cone_geom &g = p.g;
    ConeArgs A{};
    A.cs = cs;
    A.csd = csd;
    A.nX = g.nX;
    A.nY = g.nY;
    A.nZ = g.nZ;
    A.nViews = g.nViews;
    A.nCols = g.nCols;
    A.nRows = g.nRows;
    A.R = g.R;
    A.xmin = g.xmin;
    A.ymin = g.ymin;
    A.zmin = g.zmin;
    A.dx = g.dx;
    A.dy = g.dy;
    A.dz = g.dz;
    A.r2 = p.d.r2;
    A.xi_scale = p.d.xi_scale;
    A.ct_offset = p.d.ct_offset;
    A.zr_scale = p.d.zr_scale;
    A.rt_offset = p.d.rt_offset;
    A.ct_col = p.d.ct_col;
    A.rt_row = p.d.rt_row;
    A.ct_lo = -0.5f - (float)p.d.ct_col;
    A.ct_hi = (float)(g.nCols - p.d.ct_col) - 0.5f;
    A.tan_min = p.d.tan_min;
    A.tan_max = p.d.tan_max;
    A.z_fit = p.d.atan_zmax;
    for (int k = 0; k < kBpAtanMax; ++k) A.atan_c[k] = p.d.atan_c[k];
    return A;
}

fbct_status launch_cone_bp(const fbct_cone_plan &p, const ConeDeviceTables &t, const float *q,
                           void *vol, fbct_dtype to, int n, hipStream_t stream)
{
    const fbct_cone_geom &g = p.g;
    ConeArgs A = cone_args(p, t.view_cs, t.view_csd);
    A.q = q;
    A.vol = vol;
    const ConeLaunch L = choose(g, p.d.zr_scale);
    // the most z-chunks (of 32, 16, 4 or one slice) that a call may hold, whatever chunks its kernel takes
    const int kz_most = g.nZ >= 32 ? 32 : (g.nZ >= 16 ? 16 : (g.nZ >= 4 ? 4 : 1));
    const long long most = (long long)((g.nZ + kz_most - 1) / kz_most) * n;
    if (most > 65535) return fail(FBCT_ERR_UNSUPPORTED, "cone backprojection: %lld z-chunks, at most 65535 a call", most);
    A.nzc = (g.nZ + L.kz - 1) / L.kz;
    const long long gz = (long long)A.nzc * n;
    if ((unsigned long long)g.nRows * (unsigned long long)g.nCols * 4ull >= (1ull << 32))
        return fail(FBCT_ERR_UNSUPPORTED, "cone backprojection: a view of %d x %d exceeds 4 GiB", g.nRows, g.nCols);
    for (A.gz0 = 0; A.gz0 < gz; A.gz0 += 65535) {  // z-groups of one grid
        const unsigned groups = (unsigned)std::min(gz - A.gz0, 65535LL);
        const int side = L.kind == ConeLaunch::kTile ? kTx : 8;
        const dim3 grid((g.nX + side - 1) / side, (g.nY + side - 1) / side, groups);
        if (g.detector == FBCT_DETECTOR_FLAT) launch_nc<true, 0>(L, grid, stream, A, to);
        else if (p.d.atan_nc == 9) launch_nc<false, 9>(L, grid, stream, A, to);
        else if (p.d.atan_nc == 5) launch_nc<false, 5>(L, grid, stream, A, to);
        else launch_nc<false, 0>(L, grid, stream, A, to);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return fail(FBCT_ERR_DEVICE, "cone backprojection launch: %s", hipGetErrorString(e));
    }
    return FBCT_OK;
}

}  // namespace fbct

extern "C" fbct_status fbct_cone_plan_windows(const fbct_cone_plan *plan, int side, int i0, int j0, int k0, int32_t *out)
{
    using namespace fbct;
    if (!plan || !out) return fail(FBCT_ERR_INVALID_ARGUMENT, "fbct_cone_plan_windows: null pointer");
    const fbct_cone_geom &g = plan->g;
    if ((side != 8 && side != 16) || i0 < 0 || i0 >= g.nX || j0 < 0 || j0 >= g.nY || k0 < 0 || k0 >= g.nZ)
        return fail(FBCT_ERR_INVALID_ARGUMENT, "fbct_cone_plan_windows: side 8 or 16 and a voxel of the volume");
    const ConeArgs A = cone_args(*plan, nullptr, nullptr);
    const int kz = side == 8 ? kWaveKz : kTileKz;
    const int cols = side == 8 ? kWaveCols : kTileCols, rows = side == 8 ? kWaveRows : kTileRows;
    const int i1 = std::min(i0 + side - 1, g.nX - 1), j1 = std::min(j0 + side - 1, g.nY - 1);
    const float z0 = fmaf(A.dz, (float)k0 + 0.5f, A.zmin), z1 = fmaf(A.dz, (float)(k0 + kz - 1) + 0.5f, A.zmin);
    const bool flat = g.detector == FBCT_DETECTOR_FLAT;
    for (int v = 0; v < g.nViews; ++v) {
        const float2 cs = make_float2(plan->view_cs[2 * v], plan->view_cs[2 * v + 1]);
        Corner k{};
        for (int c = 0; c < 4; ++c) {
            const int i = (c & 1) ? i1 : i0, j = (c & 2) ? j1 : j0;
            const Corner q = flat                     ? corner_of<true, 0>(A, cs, i, j, z0, z1)
                             : plan->d.atan_nc == 9 ? corner_of<false, 9>(A, cs, i, j, z0, z1)
                             : plan->d.atan_nc == 5 ? corner_of<false, 5>(A, cs, i, j, z0, z1)
                                                    : corner_of<false, 0>(A, cs, i, j, z0, z1);
            k = c == 0 ? q
                       : Corner{fminf(k.cn, q.cn), fmaxf(k.cm, q.cm), fminf(k.rn, q.rn), fmaxf(k.rx, q.rx)};
        }
        const Range r = range_of(k);
        int32_t *o = out + 5 * v;
        o[0] = is_staged(A, r, cols, rows);
        o[1] = r.c0 + A.ct_col, o[2] = r.c1 + A.ct_col, o[3] = r.r0 + A.rt_row, o[4] = r.r1 + A.rt_row;
    }
    return FBCT_OK;
}
