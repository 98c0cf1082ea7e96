// Batch sums of the dynamic backward that no kernel can finish by itself: the column sums of the
// virtual matrix [u | dt],
//     u  [rows_u,  C]    -> dw[C]                 (skipped when dw == nullptr)
//     dt [rows_dt, D+3]  -> dbias[D], dalpha[3]
// as a device routine, so that they can run either as blocks of the finalize launch or as a few extra
// workgroups of a large kernel that comes last in the stream anyway.  One block = 64 columns x RG
// row groups; float64 accumulation: dalpha is a sum of B * n^2 terms of mixed sign whose total can be a
// hundred times smaller than the terms, and a float32 running sum loses what the 1e-5 parity tier
// needs.  The terms themselves (a sample's row, or the row of a few samples that one workgroup added up) are
// float32; where a split batch makes the sums in two launches, the parts in between are float64 too
// (rows of the same layout, BatchSumArgs::rows64 / OUT64).
#pragma once
#include "mhc_common.h"

namespace mhc {

// Where dw goes: fp32, or bf16 (rounded once from the float64 sum's float32 value) for a bf16 weight whose
// gradient the caller hands back in the weight's type, which saves a conversion launch.
struct DwOut {
    void *p;
    bool bf16;
    explicit operator bool() const { return p != nullptr; }
};

struct BatchSumArgs {
    const void *u; int rows_u, C; void *dw;
    const void *dt; int rows_dt, D; float *dbias, *dalpha;
    int nblk;  // blocks of 64 columns
    bool dw_bf16;
    bool rows64;  // u and dt are rows of float64 (else float32)
};

inline BatchSumArgs make_batch_sums(const void *u, int rows_u, int C, DwOut dw, const void *dt, int rows_dt,
                                    int D, float *dbias, float *dalpha, bool rows64 = false) {
    const int ncols = (dw ? C : 0) + (dt ? D + 3 : 0);  // dt == nullptr: the u columns only
    return BatchSumArgs{u, rows_u, C, dw.p, dt, rows_dt, D, dbias, dalpha, (ncols + 63) / 64, dw.bf16, rows64};
}

// Sum of src[r * ld] over r = first, first + RG, ... < rows.
template <int RG, typename T> __device__ __forceinline__ double batch_sum_column(const T *src, int ld, int first, int rows) {
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    int r = first;
    // many rows (per-sample rows of a large batch): sixteen loads in flight, the round trips decide
    for (; r + 15 * RG < rows; r += 16 * RG) {
        T t[16];
#pragma unroll
        for (int k = 0; k < 16; k++) t[k] = src[(size_t)(r + k * RG) * ld];
#pragma unroll
        for (int k = 0; k < 16; k += 4) {
            a0 += (double)t[k]; a1 += (double)t[k + 1]; a2 += (double)t[k + 2]; a3 += (double)t[k + 3];
        }
    }
    for (; r + 3 * RG < rows; r += 4 * RG) {
        const T t0 = src[(size_t)r * ld], t1 = src[(size_t)(r + RG) * ld];
        const T t2 = src[(size_t)(r + 2 * RG) * ld], t3 = src[(size_t)(r + 3 * RG) * ld];
        a0 += (double)t0; a1 += (double)t1; a2 += (double)t2; a3 += (double)t3;
    }
    for (; r < rows; r += RG) a0 += (double)src[(size_t)r * ld];
    return (a0 + a1) + (a2 + a3);
}

// red: RG * (CW + 1) doubles of LDS; called by all CW * RG threads of the workgroup (contains a barrier).
// CW = columns per block: 64, or fewer (down to 16, half a 128-byte line per row) where more blocks are
// wanted; a.nblk must count blocks of CW columns.
// IN64: a.rows64 is looked at (otherwise the rows are float32).  OUT64: the results are parts of sums, one row of
// float64 in dw ([C]) and in dbias ([D + 3], dalpha unused).
template <int RG, int CW = 64, bool IN64 = false, bool OUT64 = false>
__device__ __forceinline__ void batch_sum_block(const BatchSumArgs &a, int blk, int tid, double *red) {
    const int cl = tid % CW, rg = tid / CW;
    const int col = blk * CW + cl;
    const int ncol_u = a.dw ? a.C : 0;
    const int ncols = ncol_u + (a.dt ? a.D + 3 : 0);
    double acc = 0.0;
    if (col < ncols) {
        const bool is_u = col < ncol_u;
        const void *base = is_u ? a.u : a.dt;
        const int at = is_u ? col : col - ncol_u, ld = is_u ? a.C : a.D + 3, rows = is_u ? a.rows_u : a.rows_dt;
        if (IN64 && a.rows64) acc = batch_sum_column<RG>(static_cast<const double *>(base) + at, ld, rg, rows);
        else acc = batch_sum_column<RG>(static_cast<const float *>(base) + at, ld, rg, rows);
    }
    red[rg * (CW + 1) + cl] = acc;
    __syncthreads();
    if (rg == 0 && col < ncols) {
        double v = 0.0;
#pragma unroll
        for (int i = 0; i < RG; i++) v += red[i * (CW + 1) + cl];
        if constexpr (OUT64) {
            if (col < ncol_u) static_cast<double *>(a.dw)[col] = v;
            else reinterpret_cast<double *>(a.dbias)[col - ncol_u] = v;
        } else if (col < ncol_u) {
            if (a.dw_bf16) static_cast<unsigned short *>(a.dw)[col] = f32_to_bf16((float)v);
            else static_cast<float *>(a.dw)[col] = (float)v;
        }
        else if (col - ncol_u < a.D) a.dbias[col - ncol_u] = (float)v;
        else a.dalpha[col - ncol_u - a.D] = (float)v;
    }
}

}  // namespace mhc
