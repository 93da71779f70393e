// tqsv_kraus.h - kernels of stochastic Kraus channels and of <Z> on every
// qubit (tqsv_kraus.hip).
#ifndef TQSV_KRAUS_H
#define TQSV_KRAUS_H

#include "tqsv_internal.h"

namespace tqsv {

// one channel of a chain, in device memory: its random number and the range
// of its operators (8 doubles each, row-major re/im)
struct KrausItem {
  double status;
  uint32_t first, count;
};
// partial sums of a sweep: kraus_grid(n) blocks of 4 doubles
uint32_t kraus_grid(int n);
// partials of (rho00, rho11, Re rho01, Im rho01) of the qubit at `bit`
hipError_t k_kraus_rho(const float2* psi, int n, int bit, double* partials, hipStream_t st);
// Chooses the item's operator from the sums in `in` (all blocks the same
// way), applies it to `bit`, scaled by a power of two to a norm in [1, 2), and
// writes the partials of the result: of the qubit at `next`, or with next < 0 of
// the same qubit.
hipError_t k_kraus_apply(float2* psi, int n, int bit, int next, const KrausItem* item,
                         const double* ops, const double* in, double* out, hipStream_t st);
// psi /= sqrt(sum of rho00 + rho11 in `in`) unless that is 0
hipError_t k_kraus_normalise(float2* psi, int n, const double* in, hipStream_t st);

// <Z_b> for every index bit b at (*result)[b], in `partials` (zall_doubles(n)
// doubles) when one block sums the state, else in out
size_t zall_doubles(int n);
hipError_t k_zall(const float2* psi, int n, double* partials, double* out, const double** result,
                  hipStream_t st);

}  // namespace tqsv

#endif
