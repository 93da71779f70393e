// tqsv_grad.h - kernels behind the differentiable one-gate functions
// (tqsv_grad.hip).
#ifndef TQSV_GRAD_H
#define TQSV_GRAD_H

#include "tqsv_internal.h"

namespace tqsv {

// out = U psi (out of place)
hipError_t k_apply_1q_to(const float2* psi, float2* out, int n, int bit, const Mat2f& u, hipStream_t st);
hipError_t k_apply_2q_to(const float2* psi, float2* out, int n, int bh, int bl, const Mat4f& u,
                         hipStream_t st);
// out[i] = 2 *ge (-1)^{bit of i} psi[i], ge in device memory
hipError_t k_z_grad(const float2* psi, float2* out, int n, int bit, const double* ge, hipStream_t st);
// Block partials of G[a][c] = sum over the other bits of g[a] conj(psi[c]), 2 *
// 4^k doubles per block (re, im), rows and columns numbered with bits[0] most
// significant; k <= 4.
uint32_t matrix_grad_grid(int n, int k);
hipError_t k_matrix_grad(const float2* psi, const float2* g, int n, int k, const int* bits,
                         double* partials, hipStream_t st);

}  // namespace tqsv

#endif
