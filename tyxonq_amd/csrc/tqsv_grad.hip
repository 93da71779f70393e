// tqsv_grad.hip - kernels behind the differentiable one-gate functions:
// out-of-place gates, the gradient of <Z>, and gate-matrix gradients.
#include <hip/hip_runtime.h>

#include "tqsv_device.h"
#include "tqsv_grad.h"

namespace tqsv {

namespace {

constexpr int BLK = 256;
constexpr int NWAVE = BLK / 64;

__device__ __forceinline__ uint64_t ins0(uint64_t x, uint32_t b) {
  return ((x >> b) << (b + 1)) | (x & ((1ull << b) - 1ull));
}

uint32_t grid_of(uint64_t work) {
  const uint64_t g = (work + BLK - 1) / BLK;
  return (uint32_t)(g > 65536u ? 65536u : (g ? g : 1u));
}

// One thread per amplitude pair (quad).  Bound: one read and one write of the
// state (4.3 us at 20 qubits); a copy and an in-place kernel were two launches
// and two of each.
__global__ void apply_1q_to_kernel(const float2* __restrict__ psi, float2* __restrict__ out,
                                   uint64_t npairs, uint32_t bit, Mat2f u) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < npairs; t += stride) {
    const uint64_t i0 = ins0(t, bit), i1 = i0 | (1ull << bit);
    const float2 x0 = psi[i0], x1 = psi[i1];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const float* m = u.v + 4 * r;
      out[r ? i1 : i0] = make_float2(m[0] * x0.x - m[1] * x0.y + m[2] * x1.x - m[3] * x1.y,
                                     m[0] * x0.y + m[1] * x0.x + m[2] * x1.y + m[3] * x1.x);
    }
  }
}

__global__ void apply_2q_to_kernel(const float2* __restrict__ psi, float2* __restrict__ out,
                                   uint64_t nquads, uint32_t bh, uint32_t bl, Mat4f u) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint32_t blo = bh < bl ? bh : bl, bhi = bh < bl ? bl : bh;
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < nquads; t += stride) {
    const uint64_t i00 = ins0(ins0(t, blo), bhi);
    const uint64_t idx[4] = {i00, i00 | (1ull << bl), i00 | (1ull << bh),
                             i00 | (1ull << bh) | (1ull << bl)};
    float2 x[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) x[c] = psi[idx[c]];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float yr = 0.f, yi = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float mr = u.v[8 * r + 2 * c], mi = u.v[8 * r + 2 * c + 1];
        yr += mr * x[c].x - mi * x[c].y;
        yi += mr * x[c].y + mi * x[c].x;
      }
      out[idx[r]] = make_float2(yr, yi);
    }
  }
}

__global__ void z_grad_kernel(const float2* __restrict__ psi, float2* __restrict__ out, uint64_t dim,
                              uint32_t bit, const double* __restrict__ ge) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const float f = (float)(2.0 * ge[0]);
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < dim; i += stride) {
    const float2 v = psi[i];
    const float s = ((i >> bit) & 1ull) ? -f : f;
    out[i] = make_float2(v.x * s, v.y * s);
  }
}

struct GradBits {
  uint32_t sorted[4];  // target bits, ascending
  uint64_t off[16];    // target bits of each row / column number
};

// G[a][c] = sum_rest g[rest | off a] conj(psi[rest | off c]): one sweep over
// both states for all entries, 6.2 us at 20 qubits (sums by flip and sign
// masks took 4 or 16 sweeps, each with its own launches and host round trip).
// With 10 such gates, 5 of k = 2 and 20 <Z>, forward and backward at 20 qubits:
// 661 -> 216 launches, 7.9 -> 3.06 ms, host-bound (767 us of kernels).
// FP64 products and sums.  ROWS of the 2^K rows per thread: all for K <= 2 (32
// accumulators); one, with blockIdx.y the row, for K = 3, 4.
template <int K, int ROWS>
__global__ __launch_bounds__(BLK) void matrix_grad_kernel(const float2* __restrict__ psi,
                                                          const float2* __restrict__ g,
                                                          uint64_t nrest, GradBits gb,
                                                          double* __restrict__ partials) {
  constexpr int D = 1 << K;
  const int row0 = ROWS == D ? 0 : (int)blockIdx.y;
  double acc[ROWS][D][2] = {};
  const uint64_t stride = (uint64_t)gridDim.x * BLK;
  for (uint64_t t = (uint64_t)blockIdx.x * BLK + threadIdx.x; t < nrest; t += stride) {
    uint64_t base = t;
#pragma unroll
    for (int j = 0; j < K; ++j) base = ins0(base, gb.sorted[j]);
    float2 x[D], y[ROWS];
#pragma unroll
    for (int c = 0; c < D; ++c) x[c] = psi[base | gb.off[c]];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) y[r] = g[base | gb.off[row0 + r]];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int c = 0; c < D; ++c) {
        const double gx = y[r].x, gy = y[r].y, px = x[c].x, py = x[c].y;
        acc[r][c][0] += gx * px + gy * py;
        acc[r][c][1] += gy * px - gx * py;
      }
  }
  __shared__ double red[NWAVE][ROWS * D * 2];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int c = 0; c < D; ++c)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const double s = wave_sum_last_d(acc[r][c][p]);
        if (lane == 63) red[wave][(r * D + c) * 2 + p] = s;
      }
  __syncthreads();
  for (uint32_t v = threadIdx.x; v < (uint32_t)(ROWS * D * 2); v += BLK) {
    double s = 0.0;
    for (int w = 0; w < NWAVE; ++w) s += red[w][v];
    partials[(size_t)blockIdx.x * (2 * D * D) + (size_t)row0 * D * 2 + v] = s;
  }
}

}  // namespace

hipError_t k_apply_1q_to(const float2* psi, float2* out, int n, int bit, const Mat2f& u,
                         hipStream_t st) {
  const uint64_t np = 1ull << (n - 1);
  hipLaunchKernelGGL(apply_1q_to_kernel, dim3(grid_of(np)), dim3(BLK), 0, st, psi, out, np,
                     (uint32_t)bit, u);
  return hipGetLastError();
}

hipError_t k_apply_2q_to(const float2* psi, float2* out, int n, int bh, int bl, const Mat4f& u,
                         hipStream_t st) {
  const uint64_t nq = 1ull << (n - 2);
  hipLaunchKernelGGL(apply_2q_to_kernel, dim3(grid_of(nq)), dim3(BLK), 0, st, psi, out, nq,
                     (uint32_t)bh, (uint32_t)bl, u);
  return hipGetLastError();
}

hipError_t k_z_grad(const float2* psi, float2* out, int n, int bit, const double* ge, hipStream_t st) {
  const uint64_t dim = 1ull << n;
  hipLaunchKernelGGL(z_grad_kernel, dim3(grid_of(dim)), dim3(BLK), 0, st, psi, out, dim,
                     (uint32_t)bit, ge);
  return hipGetLastError();
}

uint32_t matrix_grad_grid(int n, int k) {
  // 4 items per thread, at most 512 blocks of partials for the final sums
  const uint64_t g = ((1ull << (n - k)) + BLK * 4 - 1) / (BLK * 4);
  return (uint32_t)(g > 512 ? 512 : g);
}

hipError_t k_matrix_grad(const float2* psi, const float2* g, int n, int k, const int* bits,
                         double* partials, hipStream_t st) {
  GradBits b{};
  for (int j = 0; j < k; ++j) b.sorted[j] = (uint32_t)bits[j];
  for (int j = 1; j < k; ++j)  // ascending
    for (int i = j; i > 0 && b.sorted[i] < b.sorted[i - 1]; --i) {
      const uint32_t t = b.sorted[i];
      b.sorted[i] = b.sorted[i - 1];
      b.sorted[i - 1] = t;
    }
  for (int v = 0; v < (1 << k); ++v)
    for (int j = 0; j < k; ++j)
      if ((v >> (k - 1 - j)) & 1) b.off[v] |= 1ull << bits[j];
  const uint64_t nrest = 1ull << (n - k);
  const uint32_t gx = matrix_grad_grid(n, k);
  switch (k) {
    case 1:
      hipLaunchKernelGGL((matrix_grad_kernel<1, 2>), dim3(gx), dim3(BLK), 0, st, psi, g, nrest, b, partials);
      break;
    case 2:
      hipLaunchKernelGGL((matrix_grad_kernel<2, 4>), dim3(gx), dim3(BLK), 0, st, psi, g, nrest, b, partials);
      break;
    case 3:
      hipLaunchKernelGGL((matrix_grad_kernel<3, 1>), dim3(gx, 8), dim3(BLK), 0, st, psi, g, nrest, b, partials);
      break;
    case 4:
      hipLaunchKernelGGL((matrix_grad_kernel<4, 1>), dim3(gx, 16), dim3(BLK), 0, st, psi, g, nrest, b, partials);
      break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace tqsv
