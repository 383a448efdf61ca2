// Products of the GEMM backward on row-major operands as they are (gemm.hip):
// the MFMA tile kernels with transposed LDS fragment reads, bf16, contiguous.
#pragma once

#include "q3_common.h"

namespace q3 {

// Whether gemm_nn (xt false) / gemm_tn (xt true) take these operands: rows of
// a multiple of 8 elements, 16-byte aligned bases, 32-bit byte offsets.
bool gemm_t_ok(const void* x, const void* w, int64_t M, int64_t N, int64_t K, bool xt);
// GEMM workspace (as q3_matmul's) with which a few-tile, long-K product runs split over K.
int64_t gemm_t_workspace_bytes(int64_t M, int64_t N, int64_t K);
// y (M, N) = x (M, K) . w (K, N)
int gemm_nn(const void* x, const void* w, void* y, int64_t M, int64_t N, int64_t K, void* ws, int64_t ws_bytes,
            hipStream_t st);
// y (M, N) = x (K, M)^T . w (K, N)
int gemm_tn(const void* x, const void* w, void* y, int64_t M, int64_t N, int64_t K, void* ws, int64_t ws_bytes,
            hipStream_t st);
// y[z] (M, N) = x[k_off[z] .. k_off[z + 1])^T . w[the same rows] for z < nz, x (rows, M), w (rows, N); k_off (nz + 1)
// on the device, ascending, at most `rows`. An empty range gives zeros. M, N multiples of 8.
int gemm_tn_ranges(const void* x, const void* w, void* y, int64_t M, int64_t N, int64_t rows, const int* k_off,
                   int64_t nz, hipStream_t st);

// fp32: y (M, N) = x . w (K, N) with x (M, K), or with xt x (K, M) transposed. The
// plain x needs 16-byte rows of whole pieces; w and a transposed x any layout.
bool gemm_f32_t_ok(const void* x, int64_t M, int64_t K, bool xt);
int gemm_f32_t(const void* x, const void* w, void* y, int64_t M, int64_t N, int64_t K, bool xt, hipStream_t st);

// out[c] = the sum of the nparts rows of `part` (cols fp32 each), in a fixed order, rounded once (train.hip).
int colsum_reduce_rows(const float* part, void* out, int64_t nparts, int64_t cols, int dtype, hipStream_t st);

}  // namespace q3
