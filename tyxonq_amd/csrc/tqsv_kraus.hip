// tqsv_kraus.hip - stochastic Kraus channels without host round trips, and
// <Z> of every qubit in one sweep.
//
// A channel {K_i} on one qubit keeps K_i with probability |K_i psi|^2 =
// Tr(K_i^dagger K_i rho), rho the qubit's 2x2 density matrix.  A chain of
// channels is one sweep per channel: every block sums the partials that the
// previous sweep left (all in the same order, so all choose alike), applies
// the chosen operator (times a power of two) to its amplitudes and accumulates
// the density matrix of the next channel's qubit from the result.  Bound: one read and one write of
// the state per channel, and launch latency below about 22 qubits.  FP64 sums.
// 20 qubits, a trajectory of 3 layers with 20 two-operator channels each and
// <Z> of every qubit: 9.3 ms when every operator was applied to a copy, reduced
// and brought to the host (970 launches), 1.14 ms here (82; 7.5 us per channel).
#include <hip/hip_runtime.h>

#include "tqsv_device.h"
#include "tqsv_kraus.h"

namespace tqsv {

namespace {

constexpr int BLK = 256;
constexpr int NWAVE = BLK / 64;

__device__ __forceinline__ uint64_t ins0(uint64_t x, uint32_t b) {
  return ((x >> b) << (b + 1)) | (x & ((1ull << b) - 1ull));
}

// block sums of 4 values, in every thread (red: NWAVE * 4 doubles)
__device__ __forceinline__ void block_sum4(double (&v)[4], double* red) {
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const double s = wave_sum_last_d(v[j]);
    if (lane == 63) red[wave * 4 + j] = s;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v[j] = 0.0;
    for (int w = 0; w < NWAVE; ++w) v[j] += red[w * 4 + j];
  }
  __syncthreads();
}

__device__ __forceinline__ void sum_partials(const double* in, uint32_t nblk, double (&v)[4],
                                             double* red) {
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = 0.0;
  for (uint32_t g = threadIdx.x; g < nblk; g += BLK)
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] += in[4 * (size_t)g + j];
  block_sum4(v, red);
}

// acc += density matrix entries of the pair (a: bit clear, b: bit set)
__device__ __forceinline__ void add_rho(double (&acc)[4], float2 a, float2 b) {
  const double ax = a.x, ay = a.y, bx = b.x, by = b.y;
  acc[0] += ax * ax + ay * ay;
  acc[1] += bx * bx + by * by;
  acc[2] += ax * bx + ay * by;  // rho01 = a conj(b)
  acc[3] += ay * bx - ax * by;
}

__device__ __forceinline__ void put_partials(double (&acc)[4], double* out, double* red) {
  block_sum4(acc, red);
  if (threadIdx.x < 4) out[4 * (size_t)blockIdx.x + threadIdx.x] = acc[threadIdx.x];
}

__global__ __launch_bounds__(BLK) void kraus_rho_kernel(const float2* __restrict__ psi,
                                                        uint64_t npairs, uint32_t bit,
                                                        double* __restrict__ out) {
  __shared__ double red[NWAVE * 4];
  double acc[4] = {};
  const uint64_t stride = (uint64_t)gridDim.x * BLK;
  for (uint64_t t = (uint64_t)blockIdx.x * BLK + threadIdx.x; t < npairs; t += stride) {
    const uint64_t i0 = ins0(t, bit);
    add_rho(acc, psi[i0], psi[i0 | (1ull << bit)]);
  }
  put_partials(acc, out, red);
}

// QUAD: amplitudes in fours over (bit, next), the result's density matrix of
// `next`; else pairs over bit and the result's density matrix of bit
template <bool QUAD>
__global__ __launch_bounds__(BLK) void kraus_apply_kernel(float2* __restrict__ psi, uint64_t nitems,
                                                          uint32_t bit, uint32_t next,
                                                          const KrausItem* __restrict__ item,
                                                          const double* __restrict__ ops,
                                                          const double* __restrict__ in,
                                                          double* __restrict__ out) {
  __shared__ double red[NWAVE * 4];
  __shared__ float mat[8];
  {
    double r[4];
    sum_partials(in, gridDim.x, r, red);
    if (threadIdx.x == 0) {
      // weights |K psi|^2 = A rho00 + B rho11 + 2 Re(C rho01), C = sum_row
      // K[row][0] conj(K[row][1])
      auto weight = [&](const double* k) {
        const double A = k[0] * k[0] + k[1] * k[1] + k[4] * k[4] + k[5] * k[5];
        const double B = k[2] * k[2] + k[3] * k[3] + k[6] * k[6] + k[7] * k[7];
        const double cr = k[0] * k[2] + k[1] * k[3] + k[4] * k[6] + k[5] * k[7];
        const double ci = k[1] * k[2] - k[0] * k[3] + k[5] * k[6] - k[4] * k[7];
        const double w = A * r[0] + B * r[1] + 2.0 * (cr * r[2] - ci * r[3]);
        return w < 0.0 ? 0.0 : w;  // (a rounded zero)
      };
      const double* k0 = ops + 8 * (size_t)item->first;
      double tot = 0.0;
      for (uint32_t i = 0; i < item->count; ++i) tot += weight(k0 + 8 * i);
      // the first operator whose cumulative probability reaches the random
      // number; none (rounding, a zero state): the first operator
      uint32_t sel = 0;
      double cum = 0.0;
      for (uint32_t i = 0; i < item->count; ++i) {
        cum += weight(k0 + 8 * i) / tot;
        if (item->status <= cum) {
          sel = i;
          break;
        }
      }
      const double* k = k0 + 8 * (size_t)sel;
      const double w = weight(k);
      // a power of two, which brings the norm sqrt(w) into [1, 2): exact, so that
      // the operator's entries are rounded as they are given, whatever w is; the
      // chain's last sweep normalises
      int x = 0;
      (void)frexp(w, &x);
      const int e2 = w > 0.0 ? -((x - 1) >> 1) : 0;
      for (int j = 0; j < 8; ++j) mat[j] = ldexpf((float)k[j], e2);
    }
    __syncthreads();
  }
  float m[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) m[j] = mat[j];
  auto row = [&](int r, float2 a, float2 b) {
    return make_float2(m[4 * r] * a.x - m[4 * r + 1] * a.y + m[4 * r + 2] * b.x - m[4 * r + 3] * b.y,
                       m[4 * r] * a.y + m[4 * r + 1] * a.x + m[4 * r + 2] * b.y + m[4 * r + 3] * b.x);
  };
  double acc[4] = {};
  const uint64_t stride = (uint64_t)gridDim.x * BLK;
  const uint32_t lo = bit < next ? bit : next, hi = bit < next ? next : bit;
  const uint64_t mb = 1ull << bit, mn = 1ull << next;
  for (uint64_t t = (uint64_t)blockIdx.x * BLK + threadIdx.x; t < nitems; t += stride) {
    if constexpr (QUAD) {
      const uint64_t i = ins0(ins0(t, lo), hi);
      const float2 x00 = psi[i], x10 = psi[i | mb], x01 = psi[i | mn], x11 = psi[i | mb | mn];
      const float2 y00 = row(0, x00, x10), y10 = row(1, x00, x10);
      const float2 y01 = row(0, x01, x11), y11 = row(1, x01, x11);
      psi[i] = y00;
      psi[i | mb] = y10;
      psi[i | mn] = y01;
      psi[i | mb | mn] = y11;
      add_rho(acc, y00, y01);
      add_rho(acc, y10, y11);
    } else {
      const uint64_t i = ins0(t, bit);
      const float2 x0 = psi[i], x1 = psi[i | mb];
      const float2 y0 = row(0, x0, x1), y1 = row(1, x0, x1);
      psi[i] = y0;
      psi[i | mb] = y1;
      add_rho(acc, y0, y1);
    }
  }
  put_partials(acc, out, red);
}

__global__ __launch_bounds__(BLK) void kraus_normalise_kernel(float2* __restrict__ psi, uint64_t dim,
                                                              const double* __restrict__ in) {
  __shared__ double red[NWAVE * 4];
  double r[4];
  sum_partials(in, gridDim.x, r, red);
  const double nrm = r[0] + r[1];
  if (!(nrm > 0.0)) return;
  const float f = (float)(1.0 / sqrt(nrm));
  const uint64_t stride = (uint64_t)gridDim.x * BLK;
  for (uint64_t i = (uint64_t)blockIdx.x * BLK + threadIdx.x; i < dim; i += stride) {
    const float2 v = psi[i];
    psi[i] = make_float2(v.x * f, v.y * f);
  }
}

// ---- <Z> of every bit -------------------------------------------------------
// A chunk is 2^ZB consecutive amplitudes: index bits 0-5 are lane bits, 6-7
// wave bits, 8 to ZB-1 the thread's 2^(ZB-8) loads; higher bits are the
// block's, and beyond 2^ZGRID blocks a block takes the 2^r chunks that differ in
// the top r index bits.  Per block: the signed sum of each low and top bit and
// the total.  One read of the state for all bits instead of one per bit (20
// qubits: 20 reductions with a host round trip each).
constexpr int ZB = 12;
constexpr int ZGRID = 12;
constexpr int ZTOP = 34 - ZB - ZGRID;      // top bits at most
constexpr int ZVALS = ZB + 1 + ZTOP;       // low bits, total, top bits

template <bool TOP>
__global__ __launch_bounds__(BLK) void zall_kernel(const float2* __restrict__ psi, uint64_t dim,
                                                   uint32_t nchunk, double* __restrict__ partials) {
  constexpr int NV = TOP ? ZVALS : ZB + 1;
  __shared__ double red[NWAVE][ZVALS];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  double tot = 0.0, hi[ZB - 8] = {}, top[ZTOP] = {};
  for (uint32_t j = 0; j < nchunk; ++j) {
    const uint64_t base = ((uint64_t)(j * gridDim.x + blockIdx.x) << ZB) + threadIdx.x;
    double tj = 0.0;
#pragma unroll
    for (int k = 0; k < (1 << (ZB - 8)); ++k) {
      const uint64_t i = base + ((uint64_t)k << 8);
      double p = 0.0;
      if (i < dim) {
        const float2 v = psi[i];
        p = (double)v.x * v.x + (double)v.y * v.y;
      }
      tj += p;
#pragma unroll
      for (int b = 0; b < ZB - 8; ++b) hi[b] += (k >> b) & 1 ? -p : p;
    }
    tot += tj;
    if constexpr (TOP)
#pragma unroll
      for (int b = 0; b < ZTOP; ++b) top[b] += (j >> b) & 1u ? -tj : tj;
  }
  auto put = [&](int slot, double v) {
    const double s = wave_sum_last_d(v);
    if (lane == 63) red[wave][slot] = s;
  };
#pragma unroll
  for (int b = 0; b < 6; ++b) put(b, (lane >> b) & 1u ? -tot : tot);
#pragma unroll
  for (int b = 6; b < 8; ++b) put(b, (wave >> (b - 6)) & 1u ? -tot : tot);
#pragma unroll
  for (int b = 8; b < ZB; ++b) put(b, hi[b - 8]);
  put(ZB, tot);
  if constexpr (TOP)
#pragma unroll
    for (int b = 0; b < ZTOP; ++b) put(ZB + 1 + b, top[b]);
  __syncthreads();
  if (threadIdx.x < (uint32_t)NV) {
    double s = 0.0;
    for (int w = 0; w < NWAVE; ++w) s += red[w][threadIdx.x];
    partials[(size_t)blockIdx.x * ZVALS + threadIdx.x] = s;
  }
}

// one block per bit
__global__ __launch_bounds__(BLK) void zall_final_kernel(const double* __restrict__ partials,
                                                         uint32_t nblk, double* __restrict__ out) {
  __shared__ double red[NWAVE * 4];
  const uint32_t b = blockIdx.x;
  double v[4] = {};
  for (uint32_t g = threadIdx.x; g < nblk; g += BLK) {
    const double* p = partials + (size_t)g * ZVALS;
    if (b < (uint32_t)ZB)
      v[0] += p[b];
    else if (b < (uint32_t)(ZB + ZGRID))
      v[0] += (g >> (b - ZB)) & 1u ? -p[ZB] : p[ZB];
    else
      v[0] += p[ZB + 1 + b - (ZB + ZGRID)];
  }
  block_sum4(v, red);
  if (threadIdx.x == 0) out[b] = v[0];
}

}  // namespace

// at least 4 quads per thread, at most 1024 blocks (every block sums all
// partials)
uint32_t kraus_grid(int n) {
  const uint64_t g = ((1ull << n) + BLK * 16 - 1) / (BLK * 16);
  return (uint32_t)(g > 1024 ? 1024 : g);
}

hipError_t k_kraus_rho(const float2* psi, int n, int bit, double* partials, hipStream_t st) {
  hipLaunchKernelGGL(kraus_rho_kernel, dim3(kraus_grid(n)), dim3(BLK), 0, st, psi, 1ull << (n - 1),
                     (uint32_t)bit, partials);
  return hipGetLastError();
}

hipError_t k_kraus_apply(float2* psi, int n, int bit, int next, const KrausItem* item,
                         const double* ops, const double* in, double* out, hipStream_t st) {
  if (next >= 0 && next != bit)
    hipLaunchKernelGGL(kraus_apply_kernel<true>, dim3(kraus_grid(n)), dim3(BLK), 0, st, psi,
                       1ull << (n - 2), (uint32_t)bit, (uint32_t)next, item, ops, in, out);
  else
    hipLaunchKernelGGL(kraus_apply_kernel<false>, dim3(kraus_grid(n)), dim3(BLK), 0, st, psi,
                       1ull << (n - 1), (uint32_t)bit, (uint32_t)bit, item, ops, in, out);
  return hipGetLastError();
}

hipError_t k_kraus_normalise(float2* psi, int n, const double* in, hipStream_t st) {
  hipLaunchKernelGGL(kraus_normalise_kernel, dim3(kraus_grid(n)), dim3(BLK), 0, st, psi, 1ull << n, in);
  return hipGetLastError();
}

static uint32_t zall_blocks(int n) {
  return n > ZB + ZGRID ? 1u << ZGRID : (n > ZB ? 1u << (n - ZB) : 1u);
}
size_t zall_doubles(int n) { return (size_t)zall_blocks(n) * ZVALS; }

hipError_t k_zall(const float2* psi, int n, double* partials, double* out, const double** result,
                  hipStream_t st) {
  const dim3 G(zall_blocks(n)), B(BLK);
  if (n > ZB + ZGRID)
    hipLaunchKernelGGL(zall_kernel<true>, G, B, 0, st, psi, 1ull << n, 1u << (n - ZB - ZGRID), partials);
  else
    hipLaunchKernelGGL(zall_kernel<false>, G, B, 0, st, psi, 1ull << n, 1u, partials);
  if (n <= ZB) {  // one block, and every bit is a low one: its sums are the result
    *result = partials;
    return hipGetLastError();
  }
  *result = out;
  hipLaunchKernelGGL(zall_final_kernel, dim3((uint32_t)n), B, 0, st, partials, zall_blocks(n), out);
  return hipGetLastError();
}

}  // namespace tqsv
