// filter_mfma.hip -- ramp filter as a Toeplitz GEMM on the gfx950 BF16 matrix cores.
//
// The centre-cropped convolution of FBP/transform.cu:163-174 is the product
//     Q[rows][nC] = P[rows][nC] * H[nC][nC],   H[m][c] = h[c - m],
// with H symmetric (h[-n] = h[n]).  BF16 keeps the FP32 exponent range but only 8
// mantissa bits, so both operands are split three ways, x = x_hi + x_lo + x_ll (each
// a BF16 number), and six products are accumulated in FP32 by
// v_mfma_f32_16x16x32_bf16:
//     hi*hi + hi*lo + lo*hi + lo*lo + hi*ll + ll*hi,
// which carries the same information as an FP32 product (the dropped terms are below
// 2^-24 relative).  The taps' three planes are precomputed per plan; P is split in
// registers as it is loaded (optionally multiplied by a per-sample weight first, the
// cone-beam pre-weight; a BF16 input needs no split).
//
// Tiling: a workgroup of 4 waves computes a tile of rows x columns; per K step it
// stages the BF16 planes of its P rows (split once per element) and the window of split
// taps its H columns read (H is Toeplitz and symmetric: the B fragment of column c at k is
// h[k - c .. k - c + 7], read from skewed copies of the taps so that every fragment is one
// aligned 16-byte LDS read) in LDS, and each wave multiplies its part in 16 x 16 MFMA tiles.
// Lane layout of v_mfma_f32_16x16x32_bf16: A lane l holds row l%16, k = 8*(l/16)+j;
// B lane l holds column l%16, k = 8*(l/16)+j; D lane l holds rows 4*(l/16)+j, column l%16.

#include <hip/hip_runtime.h>

#include "fbct_internal.hpp"

namespace fbct {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));


struct MfmaArgs {
    const void *in;    // TI[rows][nC]
    float *out;        // [rows][nC]
    const __bf16 *hp;  // [3][kRampSkew][Lg] skewed split taps (fbct_internal.hpp)
    const float *w;    // optional per-sample weights [wrows][nC], row r uses w[r % wrows]
    const float *w2;   // optional second factor [w2rows][nC], row r uses w2[(r / w2div) % w2rows]
    long long rows;
    int nC, Np, Kp, Lg, wrows, w2div, w2rows;
    int il_views;      // > 0: outputs interleaved (RampLayout), views per slice; 0: as the inputs
    long long il_full; // rows in groups of four slices
    int il_rest;       // slices of the last group (0: none)
};

// Interleaved output: slices in groups of four (the last group holds the rest), a group's
// sinograms as [view][column][slice of the group].  The GEMM's rows then run over the views
// with the group's slices innermost: row r of the product is the input row in_row(r), and
// its column c is stored at out_base(r) + c * group size.
struct __attribute__((packed, aligned(4))) Quad {
    float v[4];
};

struct IlRow {
    long long in_row, out_base;
    int step;
};

__device__ __forceinline__ IlRow il_row(const MfmaArgs &A, long long r)
{
    if (A.il_views == 0) return {r, r * A.nC, 1};
    const bool rest = r >= A.il_full;
    const int sl = rest ? max(A.il_rest, 1) : 4;  // (rows past the last one may be asked for)
    const long long block = 4LL * A.il_views;
    const long long b0 = rest ? A.il_full : r / block * block;
    const int local = (int)(r - b0), v = local / sl, s = local - v * sl;
    return {b0 + (long long)s * A.il_views + v, (b0 + (long long)v * sl) * A.nC + s, sl};
}

__device__ __forceinline__ void split3(float x, __bf16 &hi, __bf16 &lo, __bf16 &ll)
{
    hi = (__bf16)x;
    const float r1 = x - (float)hi;
    lo = (__bf16)r1;
    const float r2 = r1 - (float)lo;
    ll = (__bf16)r2;
}

__device__ __forceinline__ float widen(float x) { return x; }
__device__ __forceinline__ float widen(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// 16 consecutive elements of a row, at the alignment of an element: rows of any length and
// base take 16-byte loads (a row length that is no multiple of 16 bytes took scalar loads
// before: 300 columns of BF16, 17280 rows, 55 us, now 33 us).
template <typename TI>
struct __attribute__((packed, aligned(sizeof(TI)))) Run {
    TI v[16];
};

constexpr int kGemmThreads = 256;

// A workgroup (4 waves) computes BM rows x BN columns; per K step of BK it stages the BF16
// planes of its P rows (split once per element, weights applied first; 16 consecutive values
// per thread) and the tap window of its H columns in LDS, then each wave multiplies its part
// (MT x NT tiles of 16 x 16) from LDS.  Rows of the P planes are padded by 8 BF16, so the 16
// rows a fragment read touches start in distinct bank groups.  Staged taps per plane and
// copy and K step: the fragments reach offsets s in [k0 - c0 - BN + 1, k0 - c0 + BK - 1], plus
// 7 for the copies' shift and 7 for the window's 8-alignment: BN + BK + 16 BF16 per row, an
// odd multiple of 8 dwords (so the 16 lanes of a fragment read, 8 copies x 2 windows 16 bytes
// apart, fall in distinct bank groups).
//
// What bounds it: a workgroup's K steps are a serial chain of load, split, barrier, multiply,
// barrier (about 3.5 us a step at two waves per SIMD), hidden only by other workgroups.  Three
// tile shapes, see launch_ramp_gemm.
template <typename TI, bool kW, int BM, int BN, int BK>
__global__ __launch_bounds__(kGemmThreads) void ramp_gemm_kernel(MfmaArgs A)
{
    constexpr int kTW = BN + BK + 16;
    constexpr int kKS = BK + 8;                        // BF16 per staged P row
    constexpr int WR = BM >= 128 ? 2 : 1, WC = 4 / WR;  // waves along rows and columns
    constexpr int MT = BM / WR / 16, NT = BN / WC / 16;  // 16 x 16 tiles per wave
    static_assert(BM * BK == 16 * kGemmThreads, "a thread stages 16 values of one row");
    static_assert((kTW / 2 / 8) % 2 == 1, "tap rows an odd multiple of 8 dwords");
    constexpr bool kExactA = sizeof(TI) == 2 && !kW;
    constexpr int kPA = kExactA ? 1 : 3;  // A planes in use
    __shared__ __bf16 As[kPA][BM][kKS];
    __shared__ __bf16 Ts[3][kRampSkew][kTW];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave / WC, wc = wave % WC;
    // each XCD takes whole row tiles, their column tiles consecutive (P rows stay in its L2)
    const unsigned lblk = xcd_block(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    const long long r0 = (long long)(lblk / gridDim.y) * BM;
    const int c0 = (int)(lblk % gridDim.y) * BN;
    // staging assignment: thread -> (row, 16 k-values at kh)
    const int srow = tid / (BK / 16), kh = tid % (BK / 16) * 16;
    const bool arow_ok = r0 + srow < A.rows;
    const long long arow = arow_ok ? il_row(A, r0 + srow).in_row : 0;
    const TI *prow = static_cast<const TI *>(A.in) + arow * (long long)A.nC;
    const float *wrow = kW && A.w ? A.w + arow % A.wrows * (long long)A.nC : nullptr;
    const float *w2row =
        kW && A.w2 ? A.w2 + (arow / A.w2div) % A.w2rows * (long long)A.nC : nullptr;
    // B from the tap table: per K step the window of kTW taps (each plane, each skewed
    // copy) from which column c of H reads h[k0 + k - c], k < 32; the window starts at
    // u0 + k0, and each lane's B fragment of tile t sits at a fixed offset in it
    const int dlo = ramp_table_dlo(A.Np);
    const int u0 = (-c0 - (BN - 1) - dlo) & ~7;  // >= 8: c0 <= Np - BN
    const int fr = lane & 15, fk = 8 * (lane >> 4);
    int boff[NT];  // Ts element offset of the fragment h[s .. s + 7], s = k0 + fk - c
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int s0 = fk - (c0 + wc * (BN / WC) + 16 * t + fr);  // s at k0 = 0
        const int r = (-s0) & (kRampSkew - 1);               // copy whose row holds it aligned
        boff[t] = r * kTW + (s0 - dlo + r - u0);             // in [0, kTW - 8], a multiple of 8
    }

    f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};

    for (int k0 = 0; k0 < A.Kp; k0 += BK) {
        // ---- stage A: 16 consecutive k of one row, weighted and split
        {
            float x[16];
            const int kb = k0 + kh;
            if (arow_ok && kb + 16 <= A.nC) {
                const Run<TI> u = *reinterpret_cast<const Run<TI> *>(prow + kb);
#pragma unroll
                for (int j = 0; j < 16; ++j) x[j] = widen(u.v[j]);
            } else {
#pragma unroll
                for (int j = 0; j < 16; ++j) x[j] = (arow_ok && kb + j < A.nC) ? widen(prow[kb + j]) : 0.0f;
            }
            // per-sample weights (kW): the product is formed where the split reads it, as
            // one expression
            float wt[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) wt[j] = 1.0f;
            if constexpr (kW) {
                if (arow_ok && kb + 16 <= A.nC) {
                    // 16-byte loads: a wave's scalar weight loads each touch 32 rows' cache
                    // lines, and 16 of them per step bound the kernel by its memory
                    // instruction rate
                    if (wrow) {
                        const Run<float> u = *reinterpret_cast<const Run<float> *>(wrow + kb);
#pragma unroll
                        for (int j = 0; j < 16; ++j) wt[j] *= u.v[j];
                    }
                    if (w2row) {
                        const Run<float> u = *reinterpret_cast<const Run<float> *>(w2row + kb);
#pragma unroll
                        for (int j = 0; j < 16; ++j) wt[j] *= u.v[j];
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < 16; ++j) {
                        const bool ok = arow_ok && kb + j < A.nC;
                        float w1 = ok ? 1.0f : 0.0f;
                        if (wrow) w1 *= ok ? wrow[kb + j] : 0.0f;
                        if (w2row) w1 *= ok ? w2row[kb + j] : 0.0f;
                        wt[j] = w1;
                    }
                }
            }
            bf16x8 h[2], l[2], m[2];
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                if constexpr (kExactA) {
                    h[j >> 3][j & 7] = (__bf16)x[j];
                } else {
                    __bf16 a, b, c;
                    split3(kW ? x[j] * wt[j] : x[j], a, b, c);
                    h[j >> 3][j & 7] = a, l[j >> 3][j & 7] = b, m[j >> 3][j & 7] = c;
                }
            }
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                *reinterpret_cast<bf16x8 *>(&As[0][srow][kh + 8 * q]) = h[q];
                if constexpr (!kExactA) {
                    *reinterpret_cast<bf16x8 *>(&As[1][srow][kh + 8 * q]) = l[q];
                    *reinterpret_cast<bf16x8 *>(&As[2][srow][kh + 8 * q]) = m[q];
                }
            }
        }
        // ---- stage B: the tap window of this K step (3 planes x 8 copies x kTW taps)
        for (int q = tid; q < 3 * kRampSkew * (kTW / 8); q += 256) {
            const int row = q / (kTW / 8), ch = q % (kTW / 8);  // row = plane * 8 + copy
            *reinterpret_cast<bf16x8 *>(&Ts[0][0][0] + row * kTW + 8 * ch) =
                *reinterpret_cast<const bf16x8 *>(A.hp + (size_t)row * A.Lg + (u0 + k0) + 8 * ch);
        }
        __syncthreads();

        // ---- multiply this wave's part, 32 k at a time
#pragma unroll
        for (int kk = 0; kk < BK; kk += 32) {
            bf16x8 ah[MT], al[MT], all[MT];
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const int r = wr * (BM / WR) + 16 * i + fr;
                ah[i] = *reinterpret_cast<const bf16x8 *>(&As[0][r][kk + fk]);
                if constexpr (!kExactA) {
                    al[i] = *reinterpret_cast<const bf16x8 *>(&As[1][r][kk + fk]);
                    all[i] = *reinterpret_cast<const bf16x8 *>(&As[2][r][kk + fk]);
                }
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const bf16x8 bh = *reinterpret_cast<const bf16x8 *>(&Ts[0][0][0] + boff[t] + kk);
                const bf16x8 bl = *reinterpret_cast<const bf16x8 *>(&Ts[1][0][0] + boff[t] + kk);
                const bf16x8 bll = *reinterpret_cast<const bf16x8 *>(&Ts[2][0][0] + boff[t] + kk);
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    if constexpr (!kExactA) {
                        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(all[i], bh, acc[i][t], 0, 0, 0);
                        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bl, acc[i][t], 0, 0, 0);
                        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bh, acc[i][t], 0, 0, 0);
                    }
                    acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bll, acc[i][t], 0, 0, 0);
                    acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bl, acc[i][t], 0, 0, 0);
                    acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bh, acc[i][t], 0, 0, 0);
                }
            }
        }
        __syncthreads();  // the next K step overwrites the planes
    }

    // ---- store: D lane l holds rows 4 (l / 16) + j, column l % 16 of each 16 x 16 tile
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const long long row0 = r0 + wr * (BM / WR) + 16 * i + 4 * (lane >> 4);
        // a lane's four rows are the four slices of one (view, column): one 16-byte store
        const bool quad = A.il_views > 0 && row0 < A.il_full;
        IlRow o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = il_row(A, row0 + j);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int col = c0 + wc * (BN / WC) + 16 * t + (lane & 15);
            if (col >= A.nC) continue;
            if (quad) {
                *reinterpret_cast<Quad *>(A.out + o[0].out_base + 4LL * col) = Quad{{acc[i][t][0], acc[i][t][1], acc[i][t][2], acc[i][t][3]}};
                continue;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (row0 + j < A.rows) A.out[o[j].out_base + (long long)col * o[j].step] = acc[i][t][j];
        }
    }
}

template <typename TI, bool kW>
void launch_gemm_p(int bm, dim3 grid, hipStream_t stream, const MfmaArgs &A)
{
    const dim3 wg(kGemmThreads);
    if (bm == 32) hipLaunchKernelGGL((ramp_gemm_kernel<TI, kW, 32, 64, 128>), grid, wg, 0, stream, A);
    else if (bm == 64) hipLaunchKernelGGL((ramp_gemm_kernel<TI, kW, 64, 128, 64>), grid, wg, 0, stream, A);
    else hipLaunchKernelGGL((ramp_gemm_kernel<TI, kW, 128, 256, 32>), grid, wg, 0, stream, A);
}

}  // namespace

fbct_status launch_ramp_gemm(const RampOperand &H, const void *in, fbct_dtype ti, float *out, int64_t rows,
                             const RowWeights &rw, hipStream_t stream, int il_views)
{
    if (rows <= 0) return FBCT_OK;
    if ((rw.w && rw.wrows <= 0) || (rw.w2 && (rw.w2div <= 0 || rw.w2rows <= 0)))
        return fail(FBCT_ERR_INVALID_ARGUMENT, "ramp filter: weight row counts must be positive");
    const float *w = (rw.w || rw.w2) ? (rw.w ? rw.w : rw.w2) : nullptr;  // non-null: weighted kernel
    MfmaArgs A;
    A.in = in;
    A.out = out;
    A.hp = reinterpret_cast<const __bf16 *>(H.planes);
    A.w = rw.w;
    A.w2 = rw.w2;
    A.rows = rows;
    A.nC = H.nC;
    A.Np = H.Np;
    A.Kp = H.Kp;
    A.Lg = H.Lg;
    A.wrows = rw.w ? rw.wrows : 1;
    A.w2div = rw.w2 ? rw.w2div : 1;
    A.w2rows = rw.w2 ? rw.w2rows : 1;
    A.il_views = il_views;
    A.il_full = 0;
    A.il_rest = 0;
    if (il_views > 0) {
        const int64_t n = rows / il_views;
        if (n * il_views != rows) return fail(FBCT_ERR_INVALID_ARGUMENT, "ramp filter: rows are not whole slices");
        A.il_full = n / 4 * 4 * il_views;
        A.il_rest = (int)(n % 4);
    }
    if (H.Np % kRampTileN != 0 || H.Np < H.nC || H.Kp % 32 != 0 || H.Kp < H.nC || H.Lg != ramp_table_len(H.Np, H.Kp))
        return fail(FBCT_ERR_UNSUPPORTED, "ramp filter: operand planes not padded to the tile");
    // Tile shape (rows x columns x K step).  The widest, 128 x 256 x 32, splits each input
    // element for the fewest workgroups and is the fastest where it pads the columns no further
    // than 128-wide tiles and leaves enough workgroups (1024 columns: 184320 BF16 rows 1.64 ms
    // against 1.73 with 64 x 128; 15744 rows 133 against 147 us; but 512 columns, 23040 rows 75
    // against 63 us).  Else 64 x 128 x 64, half the K steps and twice the workgroups of the
    // 128 x 128 x 32 tile used before (888 columns, 62976 rows: 447 against 464 us).  With fewer
    // than about 320 such tiles the chip is not full and the length of a workgroup's chain is
    // what counts: 32 x 64 x 128 has four times the workgroups and half the K steps (512
    // columns, 360 rows: 10.7 against 21 us, 55 us before; 888 columns, 1968 rows: 32.7
    // against 34.8; 3936 rows, 434 tiles: 52.9 against 45.1).
    const auto cdiv = [](long long a, long long b) { return (a + b - 1) / b; };
    int bm, bn;
    const bool wide = H.nC >= 768 && cdiv(H.nC, 256) * 256 == cdiv(H.nC, 128) * 128 &&
                      cdiv(rows, 128) * cdiv(H.nC, 256) >= 384;
    if (wide || rows > (1LL << 29))  // (the grid holds fewer than 2^32 threads per axis)
        bm = 128, bn = 256;
    else if (cdiv(rows, 64) * cdiv(H.nC, 128) >= 320)
        bm = 64, bn = 128;
    else
        bm = 32, bn = 64;
    const long long gx = (rows + bm - 1) / bm;
    if (gx > 0x7fffffffLL || gx * ((H.nC + bn - 1) / bn) > 0xffffffffLL)
        return fail(FBCT_ERR_UNSUPPORTED, "ramp filter: too many rows");
    const dim3 grid((unsigned)gx, (H.nC + bn - 1) / bn);
    if (ti == FBCT_BF16) {
        if (w) launch_gemm_p<uint16_t, true>(bm, grid, stream, A);
        else launch_gemm_p<uint16_t, false>(bm, grid, stream, A);
    } else {
        if (w) launch_gemm_p<float, true>(bm, grid, stream, A);
        else launch_gemm_p<float, false>(bm, grid, stream, A);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(FBCT_ERR_DEVICE, "ramp_gemm_kernel launch: %s", hipGetErrorString(e));
    return FBCT_OK;
}

fbct_status launch_ramp_filter_mfma(const fbct_plan &p, const DeviceTables &t, const float *in, float *out,
                                    int64_t rows, const RowWeights &rw, bool interleaved, hipStream_t stream)
{
    RampOperand H{t.ramp_planes, p.g.nCols, p.d.ramp_np, p.d.ramp_kp, p.d.ramp_lg};
    return launch_ramp_gemm(H, in, FBCT_F32, out, rows, rw, stream, interleaved ? p.g.nViews : 0);
}

}  // namespace fbct
