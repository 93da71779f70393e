// tqsv_pass_impl.h - the precompiled expectation-pass kernel, which interprets
// the reduction steps of a pass program at run time (psi is read only;
// templates; each tqsv_pass_*.hip translation unit instantiates one variant).
// The step functions are in tqsv_device.h; the program format is in
// tqsv_prog.h.
#ifndef TQSV_PASS_IMPL_H
#define TQSV_PASS_IMPL_H

#include <hip/hip_runtime.h>

#include "tqsv_device.h"
#include "tqsv_internal.h"

namespace tqsv {

template <int TB, typename IDX>
__global__ __launch_bounds__(1 << TB) void k_pass(const float2* __restrict__ psi,
                                                  const uint32_t* __restrict__ prog_g,
                                                  double* __restrict__ partials, uint32_t ntiles) {
  constexpr int NT = 1 << TB;
  constexpr int T = TB + RB;
  constexpr uint32_t TSIZE = 1u << T;
  constexpr int NCHUNK = (TSIZE / 2) / NT;  // float4 chunks per thread
  extern __shared__ __align__(16) unsigned char smem[];
  float2* tA = reinterpret_cast<float2*>(smem);
  double* acc = reinterpret_cast<double*>(smem + TSIZE * sizeof(float2));

  const cw_t prog = (cw_t)prog_g;
  const uint32_t tid = threadIdx.x;
  const uint32_t L = prog[PH_L], m = prog[PH_M];
  const uint32_t nred = prog[PH_NRED];
  const cw_t H = prog + PH_H;
  constexpr uint32_t NWAVE = NT / 64 > 0 ? NT / 64 : 1;

  for (uint32_t i = tid; i < NWAVE * nred; i += NT) acc[i] = 0.0;

  // global index bits of the thread's first load chunk (tile position 2*tid)
  const IDX gthr = pos_map<IDX>(2u * tid, L, m, H);
  const uint32_t lthr = swz(2u * tid);

  for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const IDX base = tile_base<IDX>(tile, L, m, H);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NCHUNK; ++k) {
      const uint32_t pk = (uint32_t)k << (TB + 1);
      const IDX g = base | gthr | pos_map<IDX>(pk, L, m, H);
      const uint32_t l = lthr ^ swz(pk);
      *reinterpret_cast<float4*>(tA + l) = reinterpret_cast<const float4*>(psi)[g >> 1];
    }
    __syncthreads();

    // per phase, every thread gathers its 32 slots and runs the phase's steps
    const uint32_t nphase = prog[PH_NPHASE];
    cw_t ph = prog + PH_SIZE;
    for (uint32_t iph = 0; iph < nphase; ++iph) {
      const uint32_t nsteps = ph[PS_NSTEPS];
      PhaseGeo<IDX> G;
      uint32_t tpos = tid;
      G.rmask = 0;
#pragma unroll
      for (int j = 0; j < RB; ++j) {
        const uint32_t r = ph[PS_R + j];
        tpos = ((tpos >> r) << (r + 1)) | (tpos & ((1u << r) - 1u));
        G.sph[j] = swz(1u << r);
        G.gR[j] = pos_map<IDX>(1u << r, L, m, H);
        G.rmask |= G.gR[j];
      }
      G.bt = swz(tpos);
      G.gb = base | pos_map<IDX>(tpos, L, m, H);

      float2 a[NSLOT];
#pragma unroll
      for (int s = 0; s < NSLOT; ++s) a[s] = tA[G.bt ^ ls_of(G, s)];

      cw_t w = ph + PS_SIZE;
      for (uint32_t is = 0; is < nsteps; ++is) {
        const uint32_t op = w[0] & 0xffffu;
        const uint32_t nw = w[0] >> 16;
        // the slot registers do not change in a read-only pass; marking
        // them as rewritten here keeps the compiler from hoisting the pair
        // products of all 32 reduction arms out of the step loop
#pragma unroll
        for (int s = 0; s < NSLOT; ++s) __asm__ volatile("" : "+v"(a[s].x), "+v"(a[s].y));
        if (op == OP_RED) red_switch<IDX>(w[1], a, w, G, acc, nred);
        w += nw;
      }
      __syncthreads();
      ph = w;
    }
  }

  if (nred) {
    __syncthreads();
    for (uint32_t r = tid; r < nred; r += NT) {
      double sum = 0.0;
      for (uint32_t wv = 0; wv < NWAVE; ++wv) sum += acc[wv * nred + r];
      partials[(size_t)blockIdx.x * nred + r] = sum;
    }
  }
}

template <int TB, typename IDX>
hipError_t launch_one(const PassLaunch& pl, hipStream_t st) {
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_pass<TB, IDX>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  hipLaunchKernelGGL((k_pass<TB, IDX>), dim3(pl.grid), dim3(1 << TB), pl.lds_bytes, st, pl.psi,
                     pl.prog, pl.partials, pl.ntiles);
  return hipGetLastError();
}

}  // namespace tqsv

#endif
