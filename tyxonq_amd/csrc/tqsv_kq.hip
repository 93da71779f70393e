// tqsv_kq.hip - dense k-qubit unitaries: on the matrix cores, and k = 3 in vector
// arithmetic (below).
//
// A k-qubit matrix on a state is a complex product U (2^k x 2^k) * X (2^k x
// 2^(n-k)), X's rows the target-bit patterns and its columns the other index
// bits.  In real numbers a row pair (re, im) of U is [[Ur, -Ui], [Ui, Ur]], so
// one v_mfma_f32_32x32x2 multiplies 16 complex rows by 32 columns; operands,
// products and sums stay FP32.
//
// Bound: 16 * 2^n bytes at HBM rate for k <= 5, the FP32 matrix rate for k >=
// 6 (8 * 2^(n+k) flops; 64 cycles per 32x32x2).  Tile: a work-group of 4 waves
// takes 4096 amplitudes (32 KB of LDS), the product of 2^LK target patterns
// (LK = min(k, 6)) and the lowest 12 - LK other bits, so that its global
// accesses are runs of at least 64 amplitudes whatever the targets are.  A
// wave owns 16 complex rows and 64 columns (two accumulators); its part of U
// stays in registers over all tiles of the work-group for k <= 6 and is read
// per chunk of 64 columns of U for k >= 7, where each work-group computes 64
// of the 2^k output rows.
// Measured per call (one thread per amplitude -> here; random targets): 24
// qubits, k = 4: 379 -> 58 us, 5: 704 -> 72, 6: 1124 -> 107 (80 TFLOP/s with the
// call, of the 150 a large FP32 matrix product reaches); 27 qubits, k = 5: 4.41
// -> 0.45 ms (4.8 TB/s); 24 qubits, k = 8: 8.9 -> 0.35 ms.
// Error against 64 bits at k = 6: 1.5e-7 -> 1.1e-7.
#include <hip/hip_runtime.h>

#include "tqsv_internal.h"

namespace tqsv {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint64_t dep12(const KqGeo& g, uint32_t p) {
  uint64_t v = 0;
#pragma unroll
  for (int b = 0; b < KQ_TILE_BITS; ++b) v |= (uint64_t)((p >> b) & 1u) << g.pos[b];
  return v;
}

__device__ __forceinline__ uint32_t lds12(const KqGeo& g, uint32_t p) {
  uint32_t v = 0;
#pragma unroll
  for (int b = 0; b < KQ_TILE_BITS; ++b) v ^= ((p >> b) & 1u) ? g.lmap[b] : 0u;
  return v;
}

__device__ __forceinline__ uint64_t tile_base_of(const KqGeo& g, uint64_t tile) {
  uint64_t v = tile;
  for (uint32_t j = 0; j < g.nskip; ++j) {
    const uint32_t b = g.skip[j];
    v = ((v >> b) << (b + 1)) | (v & ((1ull << b) - 1ull));
  }
  return v;
}

__device__ __forceinline__ uint64_t chunk_bits(const KqGeo& g, uint32_t c) {
  uint64_t v = 0;
#pragma unroll
  for (int b = 0; b < 4; ++b) v |= (uint64_t)((c >> b) & 1u) << g.hpos[b];
  return v;
}

// row r of the LDS tile starts at r << CB; columns are XORed with the reversed
// low row bits, so that the store of a run that walks target bits and column
// bits in any order touches distinct banks, as does the read of one row
__host__ __device__ constexpr uint32_t rev5(uint32_t r) {
  return ((r & 1u) << 4) | ((r & 2u) << 2) | (r & 4u) | ((r & 8u) >> 2) | ((r & 16u) >> 4);
}

template <int LK, bool MULTI>
__global__ __launch_bounds__(256, 2) void kq_mfma_kernel(const float2* __restrict__ psi,
                                                      float2* __restrict__ out, KqGeo g,
                                                      const float2* __restrict__ A,
                                                      uint32_t nwork) {
  constexpr int CB = KQ_TILE_BITS - LK;    // column bits of a tile
  constexpr int MT = 1 << (LK - 4);        // 16-row blocks per work-group
  constexpr int NF = 1 << (LK - 1);        // complex entries of U per lane and chunk
  // products per accumulator chain (4 * RUN real ones), then added to the sum:
  // one chain over all 2^(k+1) products had 1.35 times the rounding error of a
  // chain over complex products
  constexpr int RUN = NF / 4;
  __shared__ __align__(16) float2 tile[1 << KQ_TILE_BITS];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t mt = wave % MT, ng = wave / MT;
  const uint32_t h = lane >> 5, lc = lane & 31u;
  const uint32_t nchunk = MULTI ? g.nchunk : 1u;

  // thread's loads: positions 2*tid + 512*i (16-byte pairs, ascending bits)
  const uint64_t gt = dep12(g, 2u * tid);
  const uint32_t lt = lds12(g, 2u * tid), l1 = g.lmap[0];
  float4 st[8];
  float2 af[NF];

  auto load_tile = [&](uint64_t base) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      st[i] = *reinterpret_cast<const float4*>(psi + (base | gt | dep12(g, 512u * i)));
  };
  // work item w: tile and (MULTI) block of 64 output rows; the row blocks of a
  // tile are 8 work-groups apart, on one XCD, whose L2 then holds the tile
  auto split = [&](uint32_t w, uint32_t& mb) -> uint64_t {
    if constexpr (MULTI) {
      if ((g.ntiles & 7u) == 0) {
        const uint32_t i = w >> 3;
        mb = i % nchunk;
        return (uint64_t)(w & 7u) + 8u * (i / nchunk);
      }
      mb = w % nchunk;
      return w / nchunk;
    } else {
      mb = 0;
      return w;
    }
  };
  auto load_u = [&](uint32_t mb, uint32_t kc) {
    const float2* a = A + ((size_t)((mb * MT + mt) * nchunk + kc) * NF) * 32u + h * 16u + (lc >> 1);
#pragma unroll
    for (int t = 0; t < NF; ++t) {
      const float2 u = a[32 * t];
      af[t] = (lc & 1u) ? make_float2(u.y, u.x) : make_float2(u.x, -u.y);
    }
  };

  uint32_t w = blockIdx.x;
  if (w >= nwork) return;
  uint32_t mb;
  uint64_t base = tile_base_of(g, split(w, mb));
  if constexpr (!MULTI) load_u(0, 0);
  load_tile(base);
  for (;;) {
    f16v sum0 = {}, sum1 = {}, acc0 = {}, acc1 = {};
    const uint32_t wn = w + gridDim.x;
    uint32_t mbn = 0;
    uint64_t basen = 0;
    if (wn < nwork) basen = tile_base_of(g, split(wn, mbn));
    for (uint32_t kc = 0; kc < nchunk; ++kc) {
      if constexpr (MULTI) load_u(mb, kc);
      __syncthreads();  // the previous chunk (or the stores of the previous tile) has been read
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t l = lt ^ lds12(g, 512u * i);
        tile[l] = make_float2(st[i].x, st[i].y);
        tile[l ^ l1] = make_float2(st[i].z, st[i].w);
      }
      __syncthreads();
      // the next chunk or tile travels while this one is multiplied
      if (kc + 1 < nchunk)
        load_tile(base | chunk_bits(g, kc + 1));
      else if (wn < nwork)
        load_tile(basen);
      const float2* row = tile + (h << CB) + ng * 64u;
      const uint32_t lx = lc ^ (h << 4);
#pragma unroll
      for (int t = 0; t < NF; ++t) {
        const uint32_t c = lx ^ rev5((2 * t) & 31);
        const float2 b0 = row[((2 * t) << CB) + c], b1 = row[((2 * t) << CB) + 32 + c];
        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(af[t].x, b0.x, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(af[t].x, b1.x, acc1, 0, 0, 0);
        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(af[t].y, b0.y, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(af[t].y, b1.y, acc1, 0, 0, 0);
        if (t % RUN == RUN - 1) {
          sum0 += acc0;
          sum1 += acc1;
          acc0 = f16v{};
          acc1 = f16v{};
        }
      }
    }
    __syncthreads();
    // entry v of a lane's sum: real row 8 (v/4) + 4 h + v%4, column lc
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint32_t r = mt * 16u + 4u * q + 2u * h + e;
        const uint32_t l = (r << CB) + ng * 64u + (lc ^ rev5(r & 31u));
        tile[l] = make_float2(sum0[4 * q + 2 * e], sum0[4 * q + 2 * e + 1]);
        tile[l + 32] = make_float2(sum1[4 * q + 2 * e], sum1[4 * q + 2 * e + 1]);
      }
    __syncthreads();
    const uint64_t ob = base | (MULTI ? chunk_bits(g, mb) : 0ull);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t l = lt ^ lds12(g, 512u * i);
      const float2 x = tile[l], y = tile[l ^ l1];
      *reinterpret_cast<float4*>(out + (ob | gt | dep12(g, 512u * i))) =
          make_float4(x.x, x.y, y.x, y.y);
    }
    if (wn >= nwork) break;
    w = wn;
    mb = mbn;
    base = basen;
  }
}

// ---- k = 3 --------------------------------------------------------------------
// A thread takes two groups of 8 amplitudes that differ in index bit 0, or with
// bit 0 a target (LOW) the 8 amplitudes of one, in 16-byte accesses; U in scalar
// registers.  Bound: 16 * 2^n bytes at HBM rate (64 flops per amplitude).  As a
// 4-qubit matrix U x I on the matrix cores it multiplied every amplitude by
// zeros of another group too, which an infinity turned into NaN there.
// 24 qubits, a call among others: 52-62 us -> 44-49; 27 qubits: 414-530 -> 367-453
// (4.7-5.8 TB/s); error against 64 bits 6.28e-8 -> 6.18e-8.
struct Kq3 {
  uint32_t sorted[3];  // target bits, ascending
  uint64_t off[8];     // target bits of each row / column number
};
__device__ __forceinline__ uint64_t ins0(uint64_t x, uint32_t b) {
  return ((x >> b) << (b + 1)) | (x & ((1ull << b) - 1ull));
}
// (pairs of products, then their sums: one sum of all eight had 1.1 times the
// rounding error)
__device__ __forceinline__ void kq3_row(const Mat8f& u, int r, const float2 (&x)[8], float2& y) {
  float re[4], im[4];
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    re[h] = im[h] = 0.f;
#pragma unroll
    for (int c = 2 * h; c < 2 * h + 2; ++c) {
      const float ur = u.v[16 * r + 2 * c], ui = u.v[16 * r + 2 * c + 1];
      re[h] += ur * x[c].x - ui * x[c].y;
      im[h] += ur * x[c].y + ui * x[c].x;
    }
  }
  y = make_float2((re[0] + re[1]) + (re[2] + re[3]), (im[0] + im[1]) + (im[2] + im[3]));
}

template <bool LOW>
__global__ __launch_bounds__(256) void kq3_kernel(const float2* __restrict__ psi,
                                                  float2* __restrict__ out, uint64_t nitems, Kq3 g,
                                                  Mat8f u) {
  const uint64_t stride = (uint64_t)gridDim.x * 256u;
  for (uint64_t t = (uint64_t)blockIdx.x * 256u + threadIdx.x; t < nitems; t += stride) {
    if constexpr (LOW) {
      const uint64_t base = ins0(ins0(t << 1, g.sorted[1]), g.sorted[2]);
      float2 x[8], y[2];
#pragma unroll
      for (int c = 0; c < 8; c += 2) {
        const float4 v = *reinterpret_cast<const float4*>(psi + (base | g.off[c]));
        x[c] = make_float2(v.x, v.y);
        x[c + 1] = make_float2(v.z, v.w);
      }
#pragma unroll
      for (int r = 0; r < 8; r += 2) {
        kq3_row(u, r, x, y[0]);
        kq3_row(u, r + 1, x, y[1]);
        *reinterpret_cast<float4*>(out + (base | g.off[r])) =
            make_float4(y[0].x, y[0].y, y[1].x, y[1].y);
      }
    } else {
      const uint64_t base = ins0(ins0(ins0(t << 1, g.sorted[0]), g.sorted[1]), g.sorted[2]);
      float2 x[8], z[8], y[2];
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const float4 v = *reinterpret_cast<const float4*>(psi + (base | g.off[c]));
        x[c] = make_float2(v.x, v.y);
        z[c] = make_float2(v.z, v.w);
      }
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        kq3_row(u, r, x, y[0]);
        kq3_row(u, r, z, y[1]);
        *reinterpret_cast<float4*>(out + (base | g.off[r])) =
            make_float4(y[0].x, y[0].y, y[1].x, y[1].y);
      }
    }
  }
}

// The same through LDS: tiles as in kq_mfma_kernel (8 rows, 512 columns), whose
// global accesses are runs of 64 amplitudes or more.  A thread multiplies columns
// tid and tid + 256.
__global__ __launch_bounds__(256) void kq3_tile_kernel(const float2* __restrict__ psi,
                                                       float2* __restrict__ out, KqGeo g, Mat8f u) {
  constexpr int CB = KQ_TILE_BITS - 3;
  __shared__ __align__(16) float2 tile[1 << KQ_TILE_BITS];
  const uint32_t tid = threadIdx.x;
  const uint64_t gt = dep12(g, 2u * tid);
  const uint32_t lt = lds12(g, 2u * tid), l1 = g.lmap[0];
  float4 st[8];
  auto load_tile = [&](uint64_t base) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      st[i] = *reinterpret_cast<const float4*>(psi + (base | gt | dep12(g, 512u * i)));
  };
  uint32_t w = blockIdx.x;
  if (w >= g.ntiles) return;
  uint64_t base = tile_base_of(g, w);
  load_tile(base);
  for (;;) {
    const uint32_t wn = w + gridDim.x;
    const uint64_t basen = wn < g.ntiles ? tile_base_of(g, wn) : 0ull;
    __syncthreads();  // the stores of the previous tile have been read
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t l = lt ^ lds12(g, 512u * i);
      tile[l] = make_float2(st[i].x, st[i].y);
      tile[l ^ l1] = make_float2(st[i].z, st[i].w);
    }
    __syncthreads();
    if (wn < g.ntiles) load_tile(basen);
#pragma unroll
    for (int k = 0; k < 2; ++k) {  // (a column is one thread's: no barrier in between)
      const uint32_t c = tid + 256u * k;
      float2 x[8], y;
#pragma unroll
      for (int r = 0; r < 8; ++r) x[r] = tile[((uint32_t)r << CB) + (c ^ rev5(r))];
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        kq3_row(u, r, x, y);
        tile[((uint32_t)r << CB) + (c ^ rev5(r))] = y;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t l = lt ^ lds12(g, 512u * i);
      const float2 x = tile[l], y = tile[l ^ l1];
      *reinterpret_cast<float4*>(out + (base | gt | dep12(g, 512u * i))) =
          make_float4(x.x, x.y, y.x, y.y);
    }
    if (wn >= g.ntiles) break;
    w = wn;
    base = basen;
  }
}

}  // namespace

static bool kq_geo(int n, int k, const uint32_t* bits, KqGeo* geo);

hipError_t k_apply_3q_to(const float2* psi, float2* out, int n, const int* bits, const Mat8f& u,
                         hipStream_t st) {
  // targets in ascending order, and U's rows and columns numbered by them
  int at[3] = {0, 1, 2};
  for (int i = 0; i < 3; ++i)
    for (int j = i + 1; j < 3; ++j)
      if (bits[at[j]] < bits[at[i]]) {
        const int s = at[i];
        at[i] = at[j];
        at[j] = s;
      }
  Kq3 g{};
  int num[8];
  for (int i = 0; i < 3; ++i) g.sorted[i] = (uint32_t)bits[at[i]];
  for (int v = 0; v < 8; ++v) {
    num[v] = 0;
    for (int i = 0; i < 3; ++i)
      if ((v >> i) & 1) {
        g.off[v] |= 1ull << bits[at[i]];
        num[v] |= 1 << (2 - at[i]);
      }
  }
  Mat8f m;
  for (int r = 0; r < 8; ++r)
    for (int c = 0; c < 8; ++c)
      for (int p = 0; p < 2; ++p) m.v[16 * r + 2 * c + p] = u.v[16 * num[r] + 2 * num[c] + p];
  const dim3 B(256);
  // Two targets below bit 5 leave a thread's accesses as pieces of cache lines that
  // other loads take the rest of (27 qubits, bits 1-3: 784 us, through LDS 407;
  // 2, 4 and 26: 398, 397); with wider gaps they are runs of at least 32
  // amplitudes, and LDS only costs (bits 0, 5 and 9: 367, through LDS 409).
  KqGeo geo;
  if (g.sorted[1] < 5 && kq_geo(n, 3, g.sorted, &geo)) {
    const dim3 G(geo.ntiles < 16384u ? geo.ntiles : 16384u);
    hipLaunchKernelGGL(kq3_tile_kernel, G, B, 0, st, psi, out, geo, m);
    return hipGetLastError();
  }
  const bool low = g.sorted[0] == 0;
  const uint64_t items = 1ull << (low ? n - 3 : n - 4);
  const uint64_t want = (items + 255) / 256;
  const dim3 G((uint32_t)(want < (1u << 20) ? want : (1u << 20)));
  if (low)
    hipLaunchKernelGGL(kq3_kernel<true>, G, B, 0, st, psi, out, items, g, m);
  else
    hipLaunchKernelGGL(kq3_kernel<false>, G, B, 0, st, psi, out, items, g, m);
  return hipGetLastError();
}

bool kq_mfma_geo(int n, int k, const uint32_t* bits, KqGeo* geo) {
  return k >= 4 && k <= 10 && kq_geo(n, k, bits, geo);
}

static bool kq_geo(int n, int k, const uint32_t* bits, KqGeo* geo) {
  const int lk = k < 6 ? k : 6, cb = KQ_TILE_BITS - lk;
  if (n - k < cb) return false;
  KqGeo g{};
  uint64_t tm = 0;
  for (int b = 0; b < k; ++b) tm |= 1ull << bits[b];
  // the tile: the lk lowest targets and the cb lowest other bits
  int nt = 0, nc = 0, np = 0, ns = 0, nh = 0;
  for (int b = 0; b < n; ++b) {
    if ((tm >> b) & 1u) {
      if (nt < lk) {
        g.pos[np] = (uint32_t)b;
        g.lmap[np++] = (1u << (cb + nt)) ^ (nt < 5 ? 1u << (4 - nt) : 0u);
        ++nt;
      } else {
        g.hpos[nh++] = (uint32_t)b;
      }
      g.skip[ns++] = (uint32_t)b;
    } else if (nc < cb) {
      g.pos[np] = (uint32_t)b;
      g.lmap[np++] = 1u << nc;
      ++nc;
      g.skip[ns++] = (uint32_t)b;
    }
  }
  g.nskip = (uint32_t)ns;
  g.nchunk = 1u << (k - lk);
  g.ntiles = 1u << (n - k - cb);
  *geo = g;
  return true;
}

hipError_t k_apply_kq_mfma(const float2* psi, float2* out, int k, const KqGeo& g, const float2* A,
                           hipStream_t st) {
  const uint64_t nwork = (uint64_t)g.ntiles * g.nchunk;
  if (nwork > 0xffffffffull - 4096u) return hipErrorInvalidValue;
  // 2 work-groups per CU fit by registers; 4 to 8 tiles each balance the load
  // (24 qubits, k = 5: 512 or 1024 work-groups 71 us, 768 82; 27 qubits, k = 5:
  // 1024 516 us, 4096 449)
  const uint64_t want = nwork / 8 < 1024u ? 1024u : (nwork / 8 > 4096u ? 4096u : nwork / 8);
  const uint32_t grid = (uint32_t)(nwork < want ? nwork : want);
  const dim3 G(grid), B(256);
  const uint32_t nw = (uint32_t)nwork;
  if (k == 4)
    hipLaunchKernelGGL((kq_mfma_kernel<4, false>), G, B, 0, st, psi, out, g, A, nw);
  else if (k == 5)
    hipLaunchKernelGGL((kq_mfma_kernel<5, false>), G, B, 0, st, psi, out, g, A, nw);
  else if (k == 6)
    hipLaunchKernelGGL((kq_mfma_kernel<6, false>), G, B, 0, st, psi, out, g, A, nw);
  else
    hipLaunchKernelGGL((kq_mfma_kernel<6, true>), G, B, 0, st, psi, out, g, A, nw);
  return hipGetLastError();
}

}  // namespace tqsv
