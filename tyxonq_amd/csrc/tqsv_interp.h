// tqsv_interp.h - the interpreting tile-pass kernel (gate and dual passes):
// reads the step sequence of a pass program (tqsv_prog.h) at run time.
//
// A phase's 32 slots (5 register positions) are shared by 4 neighbouring
// lanes: slot bits 0 and 1 are lane bits 0 and 1, slot bits 2-4 are 8 registers
// per state.  Gates on the lane bits exchange by DPP inside the quad.  With all
// 32 slots in one thread's registers (128 for psi and lambda) the compiler kept
// them in accumulation registers and moved them in and out around every step
// arm (20 of 85 thousand instructions of the dual kernel were such reads), and
// a 2^13-amplitude tile filled one wave per SIMD, so that the latency of each
// step's scalar loads and of its wave reduction showed in full.  Here a tile
// is 4 waves per SIMD.  Bound: instruction issue (vector and scalar about
// equal) on the CUs that have a tile.  Measured per pass, 2^13-amplitude tiles,
// 18 qubits (32 tiles), about 50 gates: gate 75 -> 34 us, dual 287 -> 108 us;
// 14 qubits (2 tiles), UCCSD rotation groups: gate 211 -> 127, dual 454 -> 329 us.
// With 2^12 tiles, and the register positions' index bits and LDS offsets from
// the phase header (one load) instead of formed per phase: 18 qubits gate 19.8
// -> 18.6, dual 45.3 -> 35.4 us; 14 qubits gate 34.4 -> 30.0, dual 76 -> 64 us.
#ifndef TQSV_INTERP_H
#define TQSV_INTERP_H

#include <hip/hip_runtime.h>

#include "tqsv_device.h"
#include "tqsv_internal.h"

namespace tqsv {

constexpr int NR = NSLOT / 4;  // slots per lane

// first words of a step; the next step's are fetched while one runs (programs
// on the device are followed by STEP_SLACK words)
typedef uint32_t step_t __attribute__((ext_vector_type(16), aligned(4)));
typedef const __attribute__((address_space(4))) step_t* cstep_t;

template <typename IDX>
__device__ __forceinline__ IDX widx(uint32_t lo, uint32_t hi) {
  if constexpr (sizeof(IDX) == 8) return (IDX)lo | ((IDX)hi << 32);
  return (IDX)lo;
}

// The tile's bit map, read once per pass (unused entries are zero, and tile
// positions have no bits there)
struct TileBits {
  uint32_t L, H[MAXH];
};
__device__ __forceinline__ TileBits tile_bits(cw_t prog) {
  TileBits t;
  t.L = prog[PH_L];
#pragma unroll
  for (int k = 0; k < MAXH; ++k) t.H[k] = prog[PH_H + k];
  return t;
}
// tile position -> global index bits (no tile base)
template <typename IDX>
__device__ __forceinline__ IDX tile_pos(const TileBits& t, uint32_t p) {
  IDX v = (IDX)(p & ((1u << t.L) - 1u));
  const uint32_t hi = p >> t.L;
#pragma unroll
  for (int k = 0; k < MAXH; ++k) v |= (IDX)((hi >> k) & 1u) << t.H[k];
  return v;
}

template <typename IDX>
struct QuadGeo {
  IDX gb;        // global index of the quad's slot 0 (register positions zero)
  IDX gq;        // this lane's two register positions
  IDX gr[3];     // the register positions of slot bits 2-4 (uniform)
  IDX rmask;     // all five register positions
  uint32_t q;    // lane in the quad: slot bits 0 and 1
};
template <typename IDX>
__device__ __forceinline__ IDX gs_reg(const QuadGeo<IDX>& G, int s) {
  IDX v = 0;
#pragma unroll
  for (int j = 0; j < 3; ++j)
    if (s & (1 << j)) v ^= G.gr[j];
  return v;
}

// the value of the lane whose slot bits 0 and 1 differ by X
template <int X>
__device__ __forceinline__ float qx(float v) {
  if constexpr (X == 0) return v;
  constexpr int CTRL = X == 1 ? 0xB1 : (X == 2 ? 0x4E : 0x1B);
  return __uint_as_float(
      (uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), CTRL, 0xf, 0xf, true));
}
template <int X>
__device__ __forceinline__ float2 qx2(float2 v) {
  return make_float2(qx<X>(v.x), qx<X>(v.y));
}
__device__ __forceinline__ float flip(float v, uint32_t sign) {
  return __uint_as_float(__float_as_uint(v) ^ sign);
}
__device__ __forceinline__ void touch8(float2 (&a)[NR]) {
#pragma unroll
  for (int s = 0; s < NR; ++s) __asm__ volatile("" : "+v"(a[s].x), "+v"(a[s].y));
}

// ---- rotations -------------------------------------------------------------
template <int K, int MD>
__device__ __forceinline__ void qrot(float2 (&a)[NR], float t, uint32_t q) {
  if constexpr (K >= 2) {
#pragma unroll
    for (int s = 0; s < NR; ++s) {
      if (s & (1 << (K - 2))) continue;
      const int s1 = s | (1 << (K - 2));
      const float2 x0 = a[s], x1 = a[s1];
      if constexpr (MD == 0) {
        a[s] = make_float2(fmaf(-t, x1.x, x0.x), fmaf(-t, x1.y, x0.y));
        a[s1] = make_float2(fmaf(t, x0.x, x1.x), fmaf(t, x0.y, x1.y));
      } else if constexpr (MD == 1) {
        a[s] = make_float2(fmaf(t, x0.x, -x1.x), fmaf(t, x0.y, -x1.y));
        a[s1] = make_float2(fmaf(t, x1.x, x0.x), fmaf(t, x1.y, x0.y));
      } else if constexpr (MD == 2) {
        a[s] = make_float2(fmaf(t, x1.y, x0.x), fmaf(-t, x1.x, x0.y));
        a[s1] = make_float2(fmaf(t, x0.y, x1.x), fmaf(-t, x0.x, x1.y));
      } else {
        a[s] = make_float2(fmaf(t, x0.x, x1.y), fmaf(t, x0.y, -x1.x));
        a[s1] = make_float2(fmaf(t, x1.x, x0.y), fmaf(t, x1.y, -x0.x));
      }
    }
  } else {
    // lane bit K: lo = 1 in the lane of x0
    const uint32_t lo = (~(q >> K) & 1u) << 31;
    const float ts = flip(t, lo);
#pragma unroll
    for (int s = 0; s < NR; ++s) {
      const float2 p = qx2<1 << K>(a[s]);
      if constexpr (MD == 0)
        a[s] = make_float2(fmaf(ts, p.x, a[s].x), fmaf(ts, p.y, a[s].y));
      else if constexpr (MD == 1)
        a[s] = make_float2(fmaf(t, a[s].x, flip(p.x, lo)), fmaf(t, a[s].y, flip(p.y, lo)));
      else if constexpr (MD == 2)
        a[s] = make_float2(fmaf(t, p.y, a[s].x), fmaf(-t, p.x, a[s].y));
      else
        a[s] = make_float2(fmaf(t, a[s].x, p.y), fmaf(t, a[s].y, -p.x));
    }
  }
}

// ---- one-sided phase ---------------------------------------------------------
template <int K>
__device__ __forceinline__ void qph(float2 (&a)[NR], float2 u, uint32_t q) {
  if constexpr (K >= 2) {
#pragma unroll
    for (int s = 0; s < NR; ++s)
      if (s & (1 << (K - 2))) a[s] = cmul(a[s], u);
  } else {
    if ((q >> K) & 1u) {
#pragma unroll
      for (int s = 0; s < NR; ++s) a[s] = cmul(a[s], u);
    }
  }
}

// ---- controlled swap ----------------------------------------------------------
template <int K>
__device__ __forceinline__ void qcxp(float2 (&a)[NR], bool ton, uint32_t smask, uint32_t q) {
  if constexpr (K >= 2) {
    const uint32_t m = ton ? smask >> q : 0u;
#pragma unroll
    for (int s = 0; s < NR; ++s) {
      if (s & (1 << (K - 2))) continue;
      const int s1 = s | (1 << (K - 2));
      const bool on = ((m >> (4 * s)) & 1u) != 0;
      const float2 x0 = a[s], x1 = a[s1];
      a[s] = sel2(on, x1, x0);
      a[s1] = sel2(on, x0, x1);
    }
  } else {
    const uint32_t m = ton ? smask >> (q & ~(1u << K)) : 0u;
#pragma unroll
    for (int s = 0; s < NR; ++s) {
      const bool on = ((m >> (4 * s)) & 1u) != 0;
      a[s] = sel2(on, qx2<1 << K>(a[s]), a[s]);
    }
  }
}

// ---- 2x2 with controls ---------------------------------------------------------
template <typename IDX>
__device__ __forceinline__ bool q_on(const QuadGeo<IDX>& G, int s, IDX cm, IDX cv, bool ton) {
  return ton && ((gs_reg(G, s) ^ G.gq) & cm & G.rmask) == (cv & G.rmask);
}
// (products with the zeros of a TYPE are left out: an infinity times 0 is NaN)
template <int K, uint32_t TYPE, typename IDX>
__device__ __forceinline__ void qu1(float2 (&a)[NR], const M2f& u, const QuadGeo<IDX>& G, IDX cm,
                                    IDX cv, bool ton) {
  if constexpr (K >= 2) {
#pragma unroll
    for (int s = 0; s < NR; ++s) {
      if (s & (1 << (K - 2))) continue;
      const int s1 = s | (1 << (K - 2));
      const bool on = q_on(G, s, cm, cv, ton);
      float2 y0, y1;
      mul2<TYPE>(u, a[s], a[s1], y0, y1);
      a[s] = sel2(on, y0, a[s]);
      a[s1] = sel2(on, y1, a[s1]);
    }
  } else {
    const bool hi = ((G.q >> K) & 1u) != 0;
    const float dr = hi ? u.r11 : u.r00, di = hi ? u.i11 : u.i00;
    const float er = hi ? u.r10 : u.r01, ei = hi ? u.i10 : u.i01;
#pragma unroll
    for (int s = 0; s < NR; ++s) {
      const bool on = q_on(G, s, cm, cv, ton);
      const float2 x = a[s], p = qx2<1 << K>(a[s]);
      float2 y;
      if constexpr (TYPE == U1_REAL)
        y = make_float2(dr * x.x + er * p.x, dr * x.y + er * p.y);
      else if constexpr (TYPE == U1_RXLIKE)
        y = make_float2(dr * x.x - ei * p.y, dr * x.y + ei * p.x);
      else
        y = make_float2(dr * x.x - di * x.y + er * p.x - ei * p.y,
                        dr * x.y + di * x.x + er * p.y + ei * p.x);
      a[s] = sel2(on, y, x);
    }
  }
}

// ---- 4x4 with controls (KH > KL slot bits, KH the basis' most significant) ------
__device__ __forceinline__ float2 cmac(float2 y, float2 m, float2 x) {
  y.x += m.x * x.x - m.y * x.y;
  y.y += m.x * x.y + m.y * x.x;
  return y;
}
template <int KH, int KL, typename IDX>
__device__ __forceinline__ void qu2(float2 (&a)[NR], cw_t m, const QuadGeo<IDX>& G, IDX cm, IDX cv,
                                    bool ton) {
  auto el = [&](uint32_t r, uint32_t c) {
    return make_float2(fl(m + 8 * r + 2 * c), fl(m + 8 * r + 2 * c + 1));
  };
  if constexpr (KL >= 2) {
    constexpr int bl = 1 << (KL - 2), bh = 1 << (KH - 2);
#pragma unroll
    for (int s = 0; s < NR; ++s) {
      if (s & (bl | bh)) continue;
      const int idx[4] = {s, s | bl, s | bh, s | bh | bl};
      const bool on = q_on(G, s, cm, cv, ton);
      float2 x[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) x[c] = a[idx[c]];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float2 y = make_float2(0.f, 0.f);
#pragma unroll
        for (int c = 0; c < 4; ++c) y = cmac(y, el(r, c), x[c]);
        a[idx[r]] = sel2(on, y, x[r]);
      }
    }
  } else if constexpr (KH >= 2) {
    // KL a lane bit: rows and columns of this lane's bit and of its partner's
    constexpr int bh = 1 << (KH - 2);
    const uint32_t l = (G.q >> KL) & 1u;
    float2 e[2][2][2];  // [row KH][column KH][own, partner]
#pragma unroll
    for (uint32_t r = 0; r < 2; ++r)
#pragma unroll
      for (uint32_t c = 0; c < 2; ++c) {
        e[r][c][0] = el(2 * r + l, 2 * c + l);
        e[r][c][1] = el(2 * r + l, 2 * c + (l ^ 1u));
      }
#pragma unroll
    for (int s = 0; s < NR; ++s) {
      if (s & bh) continue;
      const int s1 = s | bh;
      const bool on = q_on(G, s, cm, cv, ton);
      const float2 x0 = a[s], x1 = a[s1], p0 = qx2<1 << KL>(x0), p1 = qx2<1 << KL>(x1);
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        float2 y = make_float2(0.f, 0.f);
        y = cmac(y, e[r][0][0], x0);
        y = cmac(y, e[r][0][1], p0);
        y = cmac(y, e[r][1][0], x1);
        y = cmac(y, e[r][1][1], p1);
        a[r ? s1 : s] = sel2(on, y, r ? x1 : x0);
      }
    }
  } else {
    // both lane bits: row q
    float2 e[4];
#pragma unroll
    for (uint32_t x = 0; x < 4; ++x) e[x] = el(G.q, G.q ^ x);
#pragma unroll
    for (int s = 0; s < NR; ++s) {
      const bool on = q_on(G, s, cm, cv, ton);
      const float2 v = a[s];
      float2 y = make_float2(0.f, 0.f);
      y = cmac(y, e[0], v);
      y = cmac(y, e[1], qx2<1>(v));
      y = cmac(y, e[2], qx2<2>(v));
      y = cmac(y, e[3], qx2<3>(v));
      a[s] = sel2(on, y, v);
    }
  }
}

// ---- partner of every slot under a flip mask ------------------------------------
template <int X>
__device__ __forceinline__ void partner_x(const float2 (&a)[NR], float2 (&p)[NR]) {
#pragma unroll
  for (int s = 0; s < NR; ++s) p[s] = qx2<X & 3>(a[s ^ (X >> 2)]);
}
__device__ __forceinline__ void partner(uint32_t x, const float2 (&a)[NR], float2 (&p)[NR]) {
#define TQSV_PX(X)            \
  case X:                     \
    partner_x<X>(a, p);       \
    touch8(p);                \
    TQSV_ARM_END("px", X);    \
    break;
#define TQSV_PX8(X) TQSV_PX(X) TQSV_PX(X + 1) TQSV_PX(X + 2) TQSV_PX(X + 3) \
  TQSV_PX(X + 4) TQSV_PX(X + 5) TQSV_PX(X + 6) TQSV_PX(X + 7)
  switch (x & 31u) { TQSV_PX8(0) TQSV_PX8(8) TQSV_PX8(16) TQSV_PX8(24) }
#undef TQSV_PX8
#undef TQSV_PX
}

// Slots (bit = slot) of the pairs of class c of flip mask x: Mi those with x's
// lowest bit clear, Mj their partners
__device__ __forceinline__ void class_slots(uint32_t x, uint32_t c, uint32_t& Mi, uint32_t& Mj) {
  const uint32_t B[5] = {0xAAAAAAAAu, 0xCCCCCCCCu, 0xF0F0F0F0u, 0xFF00FF00u, 0xFFFF0000u};
  Mi = Mj = ~0u;
  uint32_t v = c << 1;  // bit 0: the lowest bit of x, clear in Mi
#pragma unroll
  for (int b = 0; b < 5; ++b)
    if ((x >> b) & 1u) {
      const uint32_t on = (v & 1u) ? B[b] : ~B[b];
      Mi &= on;
      Mj &= ~on;
      v >>= 1;
    }
}

// exp(-i theta/2 P): new[s] = c a[s] + sg(s ^ x) sn i^k a[s ^ x], -i i^|x&z| = i^k
__device__ __forceinline__ void qprot(float2 (&a)[NR], const float2 (&p)[NR], bool diag, float c,
                                      float sn, uint32_t odd, uint32_t tsign, uint32_t sm) {
#pragma unroll
  for (int s = 0; s < NR; ++s) {
    const float f = flip(sn, tsign ^ (((sm >> s) & 1u) << 31));
    const float2 v = a[s], w = p[s];
    if (diag)
      a[s] = make_float2(c * v.x + f * v.y, c * v.y - f * v.x);
    else if (odd)
      a[s] = make_float2(c * v.x - f * w.y, c * v.y + f * w.x);
    else
      a[s] = make_float2(c * v.x + f * w.x, c * v.y + f * w.y);
  }
}

__device__ __forceinline__ void qpgrp(float2 (&a)[NR], const float2 (&p)[NR], uint32_t Mi,
                                      uint32_t Mj, uint32_t q, cw_t e, uint32_t tsign, uint32_t sm) {
  const float cm1 = fl(e), uir = fl(e + 1), uii = fl(e + 2), ujr = fl(e + 3), uji = fl(e + 4);
  const uint32_t mi = Mi >> q, mj = Mj >> q;
#pragma unroll
  for (int s = 0; s < NR; ++s) {
    if ((((Mi | Mj) >> (4 * s)) & 15u) == 0) continue;  // uniform: no lane's slot is active
    const bool i = ((mi >> (4 * s)) & 1u) != 0, j = ((mj >> (4 * s)) & 1u) != 0;
    const uint32_t sg = tsign ^ (((sm >> (4 * s)) & 1u) << 31);
    const float ur = flip(i ? ujr : uir, sg), ui = flip(i ? uji : uii, sg);
    const float2 x = a[s], w = p[s];
    const float tr = fmaf(-ui, w.y, fmaf(cm1, x.x, ur * w.x));
    const float ti = fmaf(ui, w.x, fmaf(cm1, x.y, ur * w.y));
    a[s] = sel2(i || j, make_float2(x.x + tr, x.y + ti), x);
  }
}

// adds the wave's sum of v to its FP64 accumulator of the slot
__device__ __forceinline__ void put_red(float v, double* acc, uint32_t nred, uint32_t slot) {
  const double d = wave_sum_last_d((double)v);
  if ((threadIdx.x & 63u) == 63u) acc[(threadIdx.x >> 6) * nred + slot] += d;
}

// Runs the step h at w.  (Nothing here may depend on the next step's words: they
// would be waited for before this step's work.)
template <int MODE, typename IDX>
__device__ __forceinline__ void run_step(const step_t& h, cw_t w, float2 (&a)[NR], float2 (&b)[NR],
                                         QuadGeo<IDX> G, double* acc, uint32_t nred) {
  constexpr bool DUAL = MODE == MODE_DUAL;
  // opaque copies: what the arms derive from the geometry is formed in the arm
  // and not kept in registers through the step loop
  __asm__ volatile("" : "+v"(G.q), "+v"(G.gb), "+v"(G.gq));
  __asm__ volatile("" : "+s"(G.gr[0]), "+s"(G.gr[1]), "+s"(G.gr[2]), "+s"(G.rmask));
  const uint32_t q = G.q;
  auto F = [&](int j) { return __uint_as_float(h[j]); };
  switch (h[0] & 0xffffu) {
    case OP_ROT: {
      float t = F(3);
      const IDX zs = widx<IDX>(h[4], h[5]);
      if (zs != 0) t = parity((IDX)(G.gb & zs)) ? -t : t;
#define TQSV_QR(K, MD)                      \
  case 4 * K + MD:                          \
    qrot<K, MD>(a, t, q);                   \
    if constexpr (DUAL) qrot<K, MD>(b, t, q); \
    TQSV_ARM_END("rot", 4 * K + MD);        \
    break;
#define TQSV_QRK(K) TQSV_QR(K, 0) TQSV_QR(K, 1) TQSV_QR(K, 2) TQSV_QR(K, 3)
      switch (4u * h[1] + h[2]) {
        TQSV_QRK(0) TQSV_QRK(1) TQSV_QRK(2) TQSV_QRK(3) TQSV_QRK(4)
        default: break;
      }
#undef TQSV_QRK
#undef TQSV_QR
      break;
    }
    case OP_PH: {
      float2 u = make_float2(F(4), F(5));
      const uint32_t nent = h[2];
      cw_t e = w + OPH_HDR;
#pragma unroll 4
      for (uint32_t i = 0; i < nent; ++i, e += OPH_ENT) {
        const float2 v = cmul(u, make_float2(fl(e + 1), fl(e + 2)));
        u = sel2(((G.gb >> e[0]) & 1u) != 0, v, u);
      }
#define TQSV_QP(K)                       \
  case K:                                \
    qph<K>(a, u, q);                     \
    if constexpr (DUAL) qph<K>(b, u, q); \
    touch8(a);                           \
    if constexpr (DUAL) touch8(b);       \
    TQSV_ARM_END("ph", K);               \
    break;
      switch (h[1]) {
        TQSV_QP(0) TQSV_QP(1) TQSV_QP(2) TQSV_QP(3) TQSV_QP(4)
        default: break;
      }
#undef TQSV_QP
      break;
    }
    case OP_SGN: {
      const uint32_t m = h[1] >> q;
#pragma unroll
      for (int s = 0; s < NR; ++s) {
        const uint32_t sg = (m << (31 - 4 * s)) & 0x80000000u;
        a[s] = make_float2(flip(a[s].x, sg), flip(a[s].y, sg));
        if constexpr (DUAL) b[s] = make_float2(flip(b[s].x, sg), flip(b[s].y, sg));
      }
      break;
    }
    case OP_TAB: {
      cw_t t = w + TAB_OFF + 2 * q;
#pragma unroll
      for (int s = 0; s < NR; ++s) {
        const float2 f = make_float2(fl(t + 8 * s), fl(t + 8 * s + 1));
        a[s] = cmul(a[s], f);
        if constexpr (DUAL) b[s] = cmul(b[s], f);
      }
      break;
    }
    case OP_THR: {
      const uint32_t nent = h[1];
      float2 f = make_float2(F(2), F(3));
      cw_t e = w + THR_HDR;
#pragma unroll 4
      for (uint32_t i = 0; i < nent; ++i, e += THR_ENT) {
        const float2 v = cmul(f, make_float2(fl(e + 2), fl(e + 3)));
        f = sel2((((G.gb >> e[0]) & (G.gb >> e[1])) & 1u) != 0, v, f);
      }
#pragma unroll
      for (int s = 0; s < NR; ++s) {
        a[s] = cmul(a[s], f);
        if constexpr (DUAL) b[s] = cmul(b[s], f);
      }
      break;
    }
    case OP_SCL: {
      const float f = F(1);
#pragma unroll
      for (int s = 0; s < NR; ++s) {
        a[s] = make_float2(a[s].x * f, a[s].y * f);
        if constexpr (DUAL) b[s] = make_float2(b[s].x * f, b[s].y * f);
      }
      break;
    }
    case OP_CXP: {
      const bool ton = h[2] == CX_THREAD
                           ? (G.gb & widx<IDX>(h[4], h[5])) == widx<IDX>(h[6], h[7])
                           : true;
#define TQSV_QC(K)                                  \
  case K:                                           \
    qcxp<K>(a, ton, h[8], q);                       \
    if constexpr (DUAL) qcxp<K>(b, ton, h[8], q);   \
    touch8(a);                                      \
    if constexpr (DUAL) touch8(b);                  \
    TQSV_ARM_END("cxp", K);                         \
    break;
      switch (h[1]) {
        TQSV_QC(0) TQSV_QC(1) TQSV_QC(2) TQSV_QC(3) TQSV_QC(4)
        default: break;
      }
#undef TQSV_QC
      break;
    }
    case OP_U1: {
      const IDX cm = widx<IDX>(h[4], h[5]), cv = widx<IDX>(h[6], h[7]);
      const bool ton = (G.gb & cm) == (cv & ~G.rmask);
      const M2f u{F(8), F(9), F(10), F(11), F(12), F(13), F(14), F(15)};
#define TQSV_QU(K, TY)                                              \
  case 4 * K + TY:                                                  \
    qu1<K, TY, IDX>(a, u, G, cm, cv, ton);                          \
    if constexpr (DUAL) qu1<K, TY, IDX>(b, u, G, cm, cv, ton);      \
    TQSV_ARM_END("u1", 4 * K + TY);                                 \
    break;
#define TQSV_QUK(K) TQSV_QU(K, 1) TQSV_QU(K, 2)
      const uint32_t arm = 4u * h[1] + h[2];
      // (the other types' arms are placed after the kernel's: in line they took 1 us
      // of 50 from 66 general matrices at 11 qubits)
      if (__builtin_expect(h[2] == U1_GENERAL, 1)) {
        switch (arm) {
          TQSV_QU(0, 0) TQSV_QU(1, 0) TQSV_QU(2, 0) TQSV_QU(3, 0) TQSV_QU(4, 0)
          default: break;
        }
      } else {
        switch (arm) {
          TQSV_QUK(0) TQSV_QUK(1) TQSV_QUK(2) TQSV_QUK(3) TQSV_QUK(4)
          default: break;
        }
      }
#undef TQSV_QUK
#undef TQSV_QU
      break;
    }
    case OP_U2: {
      const IDX cm = widx<IDX>(h[4], h[5]), cv = widx<IDX>(h[6], h[7]);
      const bool ton = (G.gb & cm) == (cv & ~G.rmask);
#define TQSV_Q2(KH, KL)                                                \
  case 8 * KH + KL:                                                    \
    qu2<KH, KL, IDX>(a, w + 8, G, cm, cv, ton);                        \
    if constexpr (DUAL) qu2<KH, KL, IDX>(b, w + 8, G, cm, cv, ton);    \
    TQSV_ARM_END("u2", 8 * KH + KL);                                   \
    break;
      switch (8u * h[1] + h[2]) {
        TQSV_Q2(1, 0) TQSV_Q2(2, 0) TQSV_Q2(2, 1) TQSV_Q2(3, 0) TQSV_Q2(3, 1)
        TQSV_Q2(3, 2) TQSV_Q2(4, 0) TQSV_Q2(4, 1) TQSV_Q2(4, 2) TQSV_Q2(4, 3)
        default: break;
      }
#undef TQSV_Q2
      break;
    }
    case OP_D2: {
      const float2 d0 = make_float2(F(4), F(5)), d1 = make_float2(F(6), F(7));
      const float2 d2 = make_float2(F(8), F(9)), d3 = make_float2(F(10), F(11));
#pragma unroll
      for (int s = 0; s < NR; ++s) {
        const IDX g = G.gb ^ G.gq ^ gs_reg(G, s);
        const uint32_t sel = 2u * (uint32_t)((g >> h[1]) & 1u) + (uint32_t)((g >> h[2]) & 1u);
        const float2 d = sel2((sel & 2u) != 0, sel2((sel & 1u) != 0, d3, d2),
                              sel2((sel & 1u) != 0, d1, d0));
        a[s] = cmul(a[s], d);
        if constexpr (DUAL) b[s] = cmul(b[s], d);
      }
      break;
    }
    case OP_PROT: {
      float2 p[NR];
      const IDX z = widx<IDX>(h[2], h[3]);
      const uint32_t xr = h[1], k = (h[6] + 3u) & 3u;  // -i i^|x&z| = i^k
      // the partner's sign; i^(k + 2) = -i^k
      uint32_t ts = (uint32_t)(parity((IDX)((G.gb ^ G.gq) & z)) ^ (h[6] & 1u)) << 31;
      if (xr != 0) ts ^= (k & 2u) << 30;
      uint32_t sm = 0;
#pragma unroll
      for (int s = 0; s < NR; ++s) sm |= (uint32_t)parity((IDX)(gs_reg(G, s) & z)) << s;
      partner(xr, a, p);
      qprot(a, p, xr == 0, F(4), F(5), k & 1u, ts, sm);
      if constexpr (DUAL) {
        partner(xr, b, p);
        qprot(b, p, xr == 0, F(4), F(5), k & 1u, ts, sm);
      }
      break;
    }
    case OP_PGRP: {
      float2 p[NR];
      const uint32_t xr = h[1], sm = h[6];
      const uint32_t ts =
          (uint32_t)(parity((IDX)(G.gb & widx<IDX>(h[2], h[3]))) ^ ((sm >> q) & 1u) ^ (h[4] & 1u)) << 31;
      uint32_t Mi = 0, Mj = 0;
      partner(xr, a, p);
      for (uint32_t act = h[5]; act; act &= act - 1u) {
        const uint32_t c = (uint32_t)__builtin_ctz(act);
        class_slots(xr, c, Mi, Mj);
        qpgrp(a, p, Mi, Mj, q, w + PG_HDR + PG_ENT * c, ts, sm);
      }
      if constexpr (DUAL) {
        partner(xr, b, p);
        const bool one = (h[5] & (h[5] - 1u)) == 0;  // the masks are still its
        for (uint32_t act = h[5]; act; act &= act - 1u) {
          const uint32_t c = (uint32_t)__builtin_ctz(act);
          if (!one) class_slots(xr, c, Mi, Mj);
          qpgrp(b, p, Mi, Mj, q, w + PG_HDR + PG_ENT * c, ts, sm);
        }
      }
      break;
    }
    case OP_RED: {
      if constexpr (DUAL) {
        const uint32_t xr = h[1], slot = h[4], sm = h[7];
        // slot signs are a parity of the slot bits: the lane's part once
        const uint32_t tp = parity((IDX)(G.gb & widx<IDX>(h[5], h[6]))) ^ ((sm >> q) & 1u);
        float2 p[NR];
        partner(xr, a, p);
        if (h[2] == RED_CROSS) {
          float v0 = 0.f, v1 = 0.f;
          if (h[8]) {
#pragma unroll
            for (int s = 0; s < NR; ++s) {
              float& v = s & 1 ? v1 : v0;
              v = fmaf(sgn1(sm, 4 * s), b[s].x * p[s].y - b[s].y * p[s].x, v);
            }
          } else {
#pragma unroll
            for (int s = 0; s < NR; ++s) {
              float& v = s & 1 ? v1 : v0;
              v = fmaf(sgn1(sm, 4 * s), b[s].x * p[s].x + b[s].y * p[s].y, v);
            }
          }
          put_red(flip(v0 + v1, tp << 31), acc, nred, slot);
        } else {
          const uint32_t ts = (tp ^ (h[9] & 1u)) << 31;
          float v = 0.f;
          for (uint32_t act = h[10]; act; act &= act - 1u) {
            const uint32_t c = (uint32_t)__builtin_ctz(act);
            uint32_t Mi, Mj;
            class_slots(xr, c, Mi, Mj);
            cw_t e = w + RED_HDR + RED_ENT + 2 + RGRP_ENT * c;
            const float vir = fl(e), vii = fl(e + 1), vjr = fl(e + 2), vji = fl(e + 3);
            const uint32_t mi = Mi >> q, mj = Mj >> q;
#pragma unroll
            for (int s = 0; s < NR; ++s) {
              if ((((Mi | Mj) >> (4 * s)) & 15u) == 0) continue;
              const bool i = ((mi >> (4 * s)) & 1u) != 0, j = ((mj >> (4 * s)) & 1u) != 0;
              const uint32_t sg = ts ^ (((sm >> (4 * s)) & 1u) << 31);
              const float wr = flip(i ? vjr : vir, sg), wi = flip(i ? vji : vii, sg);
              // Im(conj(l) w a) = l.x (w.r a.y + w.i a.x) - l.y (w.r a.x - w.i a.y)
              const float t = fmaf(b[s].x, wr * p[s].y + wi * p[s].x, v);
              v = i || j ? fmaf(-b[s].y, wr * p[s].x - wi * p[s].y, t) : v;
            }
          }
          put_red(v, acc, nred, slot);
        }
      }
      break;
    }
    default: break;
  }
}

// The phases of one pass over the tile(s) in LDS.  NT threads, NT / 4 quads; a
// tile of more quads is worked off in turns.  `base` is the global index of
// the tile's position 0.  LIM: amplitudes from index `lim` up are zero and stay
// zero, so waves that hold nothing else skip the phase.
template <int T, int NT, int MODE, typename IDX, bool LIM = false>
__device__ __forceinline__ void run_phases(cw_t prog, float2* tA, float2* tB, double* acc,
                                           uint32_t nred, IDX base, const TileBits& tb,
                                           IDX lim = 0) {
  constexpr bool DUAL = MODE == MODE_DUAL;
  constexpr int TURNS = (1 << (T - RB)) / (NT / 4);
  const uint32_t q = threadIdx.x & 3u;
  const uint32_t nphase = prog[PH_NPHASE];
  cw_t ph = prog + PH_SIZE;
  for (uint32_t iph = 0; iph < nphase; ++iph) {
    const step_t hd = *(cstep_t)ph;  // (PS_SIZE words)
    const uint32_t nsteps = hd[PS_NSTEPS];
    cw_t w = ph + PS_SIZE;
#pragma unroll 1
    for (int turn = 0; turn < TURNS; ++turn) {
      QuadGeo<IDX> G;
      uint32_t tpos = (threadIdx.x >> 2) + turn * (NT / 4);
      uint32_t sp[RB];
      IDX gR[RB];
      G.rmask = 0;
#pragma unroll
      for (int j = 0; j < RB; ++j) {
        const uint32_t r = hd[PS_R + j];
        tpos = ((tpos >> r) << (r + 1)) | (tpos & ((1u << r) - 1u));
        sp[j] = hd[PS_S + j];
        gR[j] = (IDX)1 << hd[PS_G + j];
        G.rmask |= gR[j];
      }
      G.q = q;
      G.gb = base | tile_pos<IDX>(tb, tpos);
      if constexpr (LIM)
        if (__ballot(G.gb < lim) == 0) {
          w = ph + PS_SIZE;
          for (uint32_t is = 0; is < nsteps; ++is) w += w[0] >> 16;
          continue;
        }
      G.gq = (q & 1u ? gR[0] : 0) ^ (q & 2u ? gR[1] : 0);
      G.gr[0] = gR[2];
      G.gr[1] = gR[3];
      G.gr[2] = gR[4];
      uint32_t bt = swq(tpos) ^ (q & 1u ? sp[0] : 0u) ^ (q & 2u ? sp[1] : 0u);
      auto ls = [&](int s) {
        return (s & 1 ? sp[2] : 0u) ^ (s & 2 ? sp[3] : 0u) ^ (s & 4 ? sp[4] : 0u);
      };
      float2 a[NR], b[NR];
#pragma unroll
      for (int s = 0; s < NR; ++s) {
        const uint32_t l = bt ^ ls(s);
        a[s] = tA[l];
        if constexpr (DUAL) b[s] = tB[l];
      }
      w = ph + PS_SIZE;
      step_t h = *(cstep_t)w;
#pragma unroll 1
      for (uint32_t is = 0; is < nsteps; ++is) {
        cw_t wn = w + (h[0] >> 16);
        const step_t hn = *(cstep_t)wn;
        run_step<MODE, IDX>(h, w, a, b, G, acc, nred);
        w = wn;
        h = hn;
      }
      // the slot addresses are formed again instead of being kept through the phase
      __asm__ volatile("" : "+v"(bt));
#pragma unroll
      for (int s = 0; s < NR; ++s) {
        const uint32_t l = bt ^ ls(s);
        tA[l] = a[s];
        if constexpr (DUAL) tB[l] = b[s];
      }
    }
    __syncthreads();
    ph = w;
  }
}

constexpr int interp_threads(int T) { return T >= 13 ? 1024 : 1 << (T - 3); }

template <int T, int MODE, typename IDX>
__global__ __launch_bounds__(interp_threads(T)) void k_interp(float2* __restrict__ psi,
                                                              float2* __restrict__ lam,
                                                              const uint32_t* __restrict__ prog_g,
                                                              double* __restrict__ partials,
                                                              uint32_t ntiles) {
  constexpr bool DUAL = MODE == MODE_DUAL;
  constexpr int NT = interp_threads(T);
  constexpr uint32_t TSIZE = 1u << T;
  constexpr int NCHUNK = (TSIZE / 2) / NT;  // float4 chunks per thread
  extern __shared__ __align__(16) unsigned char smem[];
  float2* tA = reinterpret_cast<float2*>(smem);
  float2* tB = tA + TSIZE;  // only used in dual passes
  double* acc = reinterpret_cast<double*>(smem + (DUAL ? 2 : 1) * TSIZE * sizeof(float2));

  const cw_t prog = (cw_t)prog_g;
  const uint32_t tid = threadIdx.x;
  const TileBits tb = tile_bits(prog);
  const uint32_t m = prog[PH_M];
  const uint32_t nred = DUAL ? prog[PH_NRED] : 0u;
  constexpr uint32_t NWAVE = NT / 64;

  if constexpr (DUAL)
    for (uint32_t i = tid; i < NWAVE * nred; i += NT) acc[i] = 0.0;

  const IDX gthr = tile_pos<IDX>(tb, 2u * tid);
  const uint32_t lthr = swq(2u * tid);
  for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const IDX base = tile_base<IDX>(tile, tb.L, m, prog + PH_H);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NCHUNK; ++k) {
      const uint32_t pk = 2u * (uint32_t)k * NT;
      const IDX g = base | gthr | tile_pos<IDX>(tb, pk);
      const uint32_t l = lthr ^ swq(pk);
      *reinterpret_cast<float4*>(tA + l) = reinterpret_cast<const float4*>(psi)[g >> 1];
      if constexpr (DUAL)
        *reinterpret_cast<float4*>(tB + l) = reinterpret_cast<const float4*>(lam)[g >> 1];
    }
    __syncthreads();
    run_phases<T, NT, MODE, IDX>(prog, tA, tB, acc, nred, base, tb);
#pragma unroll
    for (int k = 0; k < NCHUNK; ++k) {
      const uint32_t pk = 2u * (uint32_t)k * NT;
      const IDX g = base | gthr | tile_pos<IDX>(tb, pk);
      const uint32_t l = lthr ^ swq(pk);
      reinterpret_cast<float4*>(psi)[g >> 1] = *reinterpret_cast<const float4*>(tA + l);
      if constexpr (DUAL)
        reinterpret_cast<float4*>(lam)[g >> 1] = *reinterpret_cast<const float4*>(tB + l);
    }
  }
  if constexpr (DUAL) {
    if (nred) {
      __syncthreads();
      for (uint32_t r = tid; r < nred; r += NT) {
        double sum = 0.0;
        for (uint32_t wv = 0; wv < NWAVE; ++wv) sum += acc[wv * nred + r];
        partials[(size_t)blockIdx.x * nred + r] = sum;
      }
    }
  }
}

template <int T, int MODE, typename IDX>
hipError_t launch_interp(const PassLaunch& pl, hipStream_t st) {
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_interp<T, MODE, IDX>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  hipLaunchKernelGGL((k_interp<T, MODE, IDX>), dim3(pl.grid), dim3(interp_threads(T)), pl.lds_bytes,
                     st, pl.psi, pl.lam, pl.prog, pl.partials, pl.ntiles);
  return hipGetLastError();
}

}  // namespace tqsv

#endif
