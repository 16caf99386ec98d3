// Products of the double base type (gemm_f64.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace mch {

// C(i,j) = alpha sum_k A(i,k) B(k,j) + beta C(i,j): A(i,k) at A + i ars + k acs, B(k,j) at B + k brs + j bcs, C(i,j) at C + i crs +
// j ccs; matrix z of the batch at z sA, z sB and (z / zdiv) sC + (z % zdiv) sC2.  bias (may be null): one value per column.
struct GemmD { int m, n, k; double alpha, beta; const double *A, *B; double* C; long long ars, acs, brs, bcs, crs, ccs, sA, sB, sC, sC2; int zdiv; const double* bias; };
// Instead of to C: row r = (b, t) of rows of T positions, column c = (which, h, d) of parts of H heads of hs to element (b, h, t, d) of
// dst[which]; with fcos / fsin (tables [seq][hs / 2]) the pairs (2 i, 2 i + 1) of the first two parts are rotated.
struct HeadsD { double* dst[3]; int T, H, hs; const double *fcos, *fsin; int seq; };

hipError_t d_gemm(hipStream_t s, int batch, int m, int n, int k, double alpha, const double* A, long long ars, long long acs, const double* B, long long brs,
                  long long bcs, double beta, double* C, long long crs, long long ccs, long long sA, long long sB, long long sC, int zdiv = 1, long long sC2 = 0,
                  const double* bias = nullptr);

// where one launch of small tiles is what the sizes call for (*done): X W^T + bias through the heads; the gradients of an inner product
hipError_t d_gemm_heads(hipStream_t s, int m, int n, int k, const double* X, const double* W, const double* bias, const HeadsD& he, bool* done);
hipError_t d_linear_bwd_small(hipStream_t s, int m, int n, int k, const double* X, const double* W, const double* dY, double* dW, double* db, double* dX,
                              double beta, bool* done);

}  // namespace mch
