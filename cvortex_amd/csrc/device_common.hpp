// device_common.hpp -- shared device-side definitions for the gfx950 kernels.
//
// Pair kernels are written in the reduced form
//     vel    = -(1/4pi)       * sum_s  Kv(r2) (d x a_s)
//     dvort  = sign(sigma)/4pi * [ a_t x sum_s Kv a_s  +  sum_s Kh (a_t . (d x a_s)) d ]
//     visc   = (2 nu / sigma^2) * [ V_t sum_s eta a_s  -  a_t sum_s eta V_s ]
// with d = x_t - x_s, Kv = g(rho)/r^3 and Kh = (3 g(rho)/r^3 - zeta(rho)/sigma^3)/r^2.
// This is algebraically the reference's pair arithmetic (reference
// src/P3D.cpp:51-144) after using d.(a_t x a_s) = -a_t.(d x a_s) and
// sum_s (a_t x a_s) Kv = a_t x sum_s Kv a_s; the rearrangement lets vel,
// dvort and visc share one evaluation of d, r2 and the regularisation per
// pair and moves two cross products out of the pair loop.
//
// Each regularisation computes (Kv, Kh, eta) up to per-call constant factors
// that the epilogue applies in FP64 (Scales below).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cvtx {

enum Reg : int { REG_SINGULAR = 0, REG_WINCKELMANS = 1, REG_PLANETARY = 2, REG_GAUSSIAN = 3 };
enum OutMask : int { OUT_VEL = 1, OUT_DVORT = 2, OUT_VISC = 4 };
// ACC_PLAIN: one FP32 running sum per accumulator.  ACC_COMP: FP32 tile
// sums folded by TwoSum, and the P3D stretching (and PSE) sums and the P2D
// viscous exchange per pair in FP64.  ACC_TILES: FP32 tile sums folded by
// TwoSum for every accumulator, no per-pair FP64 (F3D and the vorticity
// field have no per-pair FP64, so there it is ACC_COMP).
enum AccMode : int { ACC_PLAIN = 0, ACC_COMP = 1, ACC_TILES = 2 };
inline bool valid_acc(int a) { return a == ACC_PLAIN || a == ACC_COMP || a == ACC_TILES; }

// Gaussian near-field table: cubic pieces of the reduced kernels
//   G(rho) = g(rho)/rho^3,  H(rho) = (3 G(rho) - zeta(rho)) / rho^2
// on rho in [0, GTAB_RHO_MAX) with GTAB_PER_UNIT pieces per unit of rho.
// Piece i covers rho = (i + t)/GTAB_PER_UNIT, t in [0,1):
//   G = ((g3 t + g2) t + g1) t + g0, same for H; stored as two float4.
constexpr int GTAB_PER_UNIT = 16;
constexpr int GTAB_RHO_MAX = 6;
constexpr int GTAB_N = GTAB_PER_UNIT * GTAB_RHO_MAX;  // 96 pieces

// Per-call constants for the regularisations (all FP32, set by the host).
struct RegConsts {
  float s2;        // sigma^2
  float inv_s2;    // 1/sigma^2
  float c1;        // gaussian: -log2(e)/2 (3D: /t^2) | winckelmans: 2D eta 4 log2(e), 3D 1.5 sigma^2
  float c2;        // gaussian: sqrt(2/pi)
  float q_far = 208.f;  // gaussian: rho^2 from which the far form is taken (p3d_consts)
  float q_exp = 46.f;   // 3D gaussian: rho^2 from which 1 - rho zeta and G - zeta/3 round to 1 and G
  float q_tab = (float)(GTAB_RHO_MAX * GTAB_RHO_MAX);  // gaussian: table range in rho^2
  float xs = 1.f;  // 3D winckelmans, gaussian: power of two that positions are multiplied by
};

// The 3D kernels' constants.  (A struct of their own: the other kernels' schedules
// suffer from a larger argument; the 2D planetary velocity with four targets per
// lane takes 12.5 ms instead of 11.3 for 262144 particles.)
struct P3DConsts : RegConsts {
  // 3D gaussian, with t from GaussianKernel: -1/t, -1/(3 t^3), GTAB_PER_UNIT/t, and
  // log(2) times what c1 lacks of its value in FP64 (used by the near ranges only)
  float nt1 = -1.f, nt3 = -1.f / 3.f, tp = GTAB_PER_UNIT, c1_rest = 0.f;
  double g3 = 1, h5 = 1;  // 1/t^3, 1/t^5: factors of the table's G and H/3
  double tp_error = 0;    // relative rounding of tp
};

// A uniform value that a pair loop reads on every pair, held in a VGPR.  On
// gfx950 a VALU instruction with an SGPR operand issues at about half the
// rate of one whose operands are VGPRs, inline constants or a literal
// (measured: 1.8 issue slots against 1), and the compiler keeps uniform
// values in SGPRs.  The empty asm makes the value opaque, so it stays in a
// VGPR for the loop.
__device__ __forceinline__ float in_vgpr(float x) {
  asm volatile("" : "+v"(x));
  return x;
}

__device__ __forceinline__ int in_vgpr(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// The constants of `k` as VGPR values (see in_vgpr), for use inside pair loops.
__device__ __forceinline__ RegConsts loop_consts(const RegConsts& k) {
  RegConsts v;
  v.s2 = in_vgpr(k.s2);
  v.inv_s2 = in_vgpr(k.inv_s2);
  v.c1 = in_vgpr(k.c1);
  v.c2 = in_vgpr(k.c2);
  v.q_far = in_vgpr(k.q_far);
  v.q_exp = in_vgpr(k.q_exp);
  v.q_tab = in_vgpr(k.q_tab);
  return v;
}
__device__ __forceinline__ P3DConsts loop_consts(const P3DConsts& k) {
  P3DConsts v = k;
  static_cast<RegConsts&>(v) = loop_consts(static_cast<const RegConsts&>(k));
  return v;
}

// ---- separately rounded FP32 operations --------------------------------
// For code that must reproduce another program's FP32 operation sequence:
// each product and sum is rounded on its own.  (HIP's __fmul_rn family is
// plain arithmetic, which floating-point contraction may fuse into a
// multiply-add with a single rounding.)
__device__ __forceinline__ float rn_mul(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}
__device__ __forceinline__ float rn_add(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}
__device__ __forceinline__ float rn_sub(float a, float b) {
#pragma clang fp contract(off)
  return a - b;
}

// ---- compensated (TwoSum) accumulation ----------------------------------
// Knuth's TwoSum: hi + lo carries the running sum exactly up to the final
// rounding of lo.  Six FP32 operations per update; applied once per source
// tile per accumulator, so its cost is amortised over the tile.
__device__ __forceinline__ void two_sum_add(float& hi, float& lo, float x) {
  float s = hi + x;
  float bp = s - hi;
  float err = (hi - (s - bp)) + (x - bp);
  hi = s;
  lo += err;
}

// ---- regularisation kernels (reduced form) -------------------------------
// eval<SELF>(r2, K, lds_table, Kv, Kh, eta) (Winckelmans: see there)
//   Kv: velocity / stretching kernel, zero when r2 == 0 (self and
//       coincident pairs are excluded, reference src/P3D.cpp:58,94,127)
//   Kh: gradient kernel; Kh * 0 must be 0 when r2 == 0
//   eta: PSE kernel, zero when r2 == 0
// SELF = false (velocity only) drops the r2 == 0 test where Kv is finite
// there: the velocity term Kv (d x a_s) is then exactly 0 for d = 0, and the
// test is a compare and a select per pair, which are not dual-issued.
template <int REG>
struct RegKernel;

template <>
struct RegKernel<REG_SINGULAR> {
  // Kv = r^-3, Kh = r^-5 (x3 in the epilogue); infinite at r2 = 0: SELF = false
  // only where the caller finds such pairs itself (SELF_WATCH)
  template <bool SELF = true>
  static __device__ __forceinline__ void eval(float r2, const RegConsts&, const float4*,
                                              float& Kv, float& Kh, float& eta) {
    float y = __builtin_amdgcn_rsqf(r2);
    float y2 = y * y;
    float kv = y * y2;
    float kh = kv * y2;
    bool z = SELF && (r2 == 0.f);
    Kv = z ? 0.f : kv;
    Kh = z ? 0.f : kh;
    eta = 0.f;
  }
};

template <>
struct RegKernel<REG_WINCKELMANS> {
  // Positions come multiplied by a power of two (RegConsts::xs, exact) that
  // puts sigma in [1, 2), so that S = r^2 + sigma^2 can be formed in three
  // multiply-adds started from sigma^2 (rather than r^2 and then r^2/sigma^2
  // + 1) and its powers stay in range; with the exchange (winckelmans_reduced)
  // S = r^2/sigma^2 + 1 and sigma is 1 here.  With y = S^-1/2, in those units:
  //   Kv  = (r^2 + 2.5 sigma^2) y^5 = y^3 (1 + 1.5 sigma^2 y^2)
  //   Kh  = (r^2 + 3.5 sigma^2) y^7 = (Kv + sigma^2 y^5) y^2
  //   eta = y^9
  // (x 3 and x 52.5 in the epilogue).  None is zero at r = 0: the caller drops
  // coincident pairs where that matters.  k: s2 = sigma^2, c1 = 1.5 sigma^2, but
  // for the rounding (p3d_consts).
  static __device__ __forceinline__ void eval(float S, const RegConsts& k, float& Kv, float& Kh,
                                              float& eta) {
    const float y = __builtin_amdgcn_rsqf(S);
    const float y2 = y * y;
    const float y3 = y2 * y;
    Kv = y3 * __builtin_fmaf(k.c1, y2, 1.f);
    const float y5 = y3 * y2;
    Kh = __builtin_fmaf(k.s2, y5, Kv) * y2;
    eta = (y5 * y2) * y2;
  }
};

template <>
struct RegKernel<REG_PLANETARY> {
  // Reduced units, q = rho^2.  Inside the core (q < 1): g = rho^3, zeta = 3,
  // so G = 1 and H = 0; outside: g = 1, zeta = 0, so G = q^-3/2 and
  // H / 3 = q^-5/2.  The epilogue applies |sigma|^-3 and 3 |sigma|^-5.
  template <bool SELF = true>
  static __device__ __forceinline__ void eval(float r2, const RegConsts& k, const float4*,
                                              float& Kv, float& Kh, float& eta) {
    float q = r2 * k.inv_s2;
    float y = __builtin_amdgcn_rsqf(q);
    float y2 = y * y;
    float kv = y * y2;
    float kh = kv * y2;
    bool in = q < 1.f;
    bool z = SELF && (r2 == 0.f);
    Kv = z ? 0.f : (in ? 1.f : kv);
    Kh = in ? 0.f : kh;
    eta = 0.f;
  }
};

// DIRECT: see below; the other regularisations have one form.
template <bool DIRECT>
struct GaussianKernel {
  // Positions come multiplied by a power of two (RegConsts::xs, exact) that puts
  // sigma in [1, 2).  In those units, with t = sigma (DIRECT), Kv = G(rho)/t^3, Kh
  // = H(rho)/(3 t^5), eta = zeta = sqrt(2/pi) exp(-rho^2/2): beyond the core Kv =
  // r^-3 and Kh = r^-5, so the usual pair does without rho^2 = r^2/sigma^2, one
  // issue slot of about 33 for velocity and stretching, and one rounding.  The
  // near ranges, which need rho, pay two multiplications and a rounding instead.
  // So !DIRECT (r^2 taken in units of sigma^2, t = 1) where most rounds (a wave
  // and a source) have a near pair: targets that are not ordered, that is clouds
  // and small problems (q = 4).  Reduced -> DIRECT: ring of 2^20 661.8 -> 635 ms,
  // velocity of a ring of 100000 4005 -> 3953 us, the error of velocity and
  // stretching of a ring of 65536 against 64 bits 1.2e-7 -> 5.4e-8; but 48 clouds
  // 16.3 -> 17.0 ms.
  // Three ranges of rho^2 (limits in r^2), nested so that a wave runs only the ranges its
  // lanes need (for spatially ordered targets, order.hip, a wave's lanes
  // are close together and most sources fall in the first range for all):
  //   rho^2 >= 208: exp(-rho^2/2) < 2^-149 is zero in FP32, so
  //                 G = rho^-3, H/3 = rho^-5, zeta = 0: Kv = r^-3, Kh = r^-5;
  //   rho^2 >= 36:  erf(rho/sqrt2) = 1 to below 2e-9, so
  //                 G = rho^-3 (1 - rho zeta), H/3 = (G - zeta/3) rho^-2;
  //   rho^2 < 36:   cubic pieces of G and H/3 from the LDS table, built on the host from
  //                 exact FP64 values (series below rho = 0.5), so the
  //                 small-rho behaviour has no cancellation.
  // A self or coincident pair falls in the last range, where same() is asked and
  // G and zeta are zeroed; H stays finite and only ever multiplies d = 0.  1e-30
  // added to r2 (by the caller if DIRECT) keeps 1/r finite.
  //
  // eval_ranges also reports the split between the ranges: near(G, eta) is
  // called inside the rho^2 < 208 branch (only there is eta nonzero), and
  // Kfar is Kv for the pairs beyond it and 0 for the others.  A caller can so
  // accumulate the near pairs in a wider type at the cost of the branch only.
  // The evaluation in two steps, for callers that interleave pairs:
  // far() is the rho^2 >= 208 form every pair starts from, near() replaces
  // g and h and sets zeta for a pair with rho^2 < 208 (the caller tests
  // r2 < k.q_far).  eval_ranges is the two combined.
  struct Far {
    float pinv, pinv2, g, h;
  };
  static __device__ __forceinline__ Far far(float& r2, const P3DConsts& k) {
    if constexpr (!DIRECT) r2 = __builtin_fmaf(r2, k.inv_s2, 1e-30f);
    Far f;
    f.pinv = __builtin_amdgcn_rsqf(r2);  // 1/r
    f.pinv2 = f.pinv * f.pinv;
    f.g = f.pinv2 * f.pinv;
    f.h = f.g * f.pinv2;
    return f;
  }
  // The table's G and H/3 come multiplied by 1/t^3 and 1/t^5, in FP64 and each
  // coefficient rounded by itself (table_entry): a factor rounded to FP32 would be off
  // the same way for every near pair (velocity where all pairs are near, sigma 0.61:
  // 4.8e-8 against 64 bits with such factors, 3.3e-8 so).
  // ZETA: zeta itself is used: the rounding of c1, times rho^2/2, is common to all
  // pairs too and made up for (exchange, sigma 0.013: 1.0e-7 -> 3.2e-8).  G and H,
  // against which zeta is small, take it as it is, the same with and without ZETA.
  template <bool ZETA, class Same>
  static __device__ __forceinline__ void near(const Far& f, float r2, const P3DConsts& k,
                                              const float4* tab, Same&& same, float& g, float& h,
                                              float& z) {
    z = k.c2 * __builtin_amdgcn_exp2f(r2 * k.c1);
    if constexpr (DIRECT) {
      g = f.pinv2 * __builtin_fmaf(z, k.nt1, f.pinv);
      h = __builtin_fmaf(z, k.nt3, g) * f.pinv2;
    } else {
      g = f.pinv2 * (f.pinv - z);
      h = __builtin_fmaf(z, -1.f / 3.f, g) * f.pinv2;
    }
    if constexpr (ZETA) z = __builtin_fmaf(z, r2 * k.c1_rest, z);
    if (r2 < k.q_tab) {
      float t = r2 * f.pinv * (DIRECT ? k.tp : (float)GTAB_PER_UNIT);  // rho * 16
      int i = (int)t;
      i = i < (GTAB_N - 1) ? i : (GTAB_N - 1);
      i = i > 0 ? i : 0;
      float u = t - (float)i;
      float4 cg = tab[2 * i];
      float4 ch = tab[2 * i + 1];
      g = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(cg.w, u, cg.z), u, cg.y), u, cg.x);
      h = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(ch.w, u, ch.z), u, ch.y), u, ch.x);
      const bool zr = same();
      g = zr ? 0.f : g;
      z = zr ? 0.f : z;
    }
  }

  // Entry i of the table in the kernel's units.  DIRECT: from the FP64 copy behind
  // the FP32 one, so that it is rounded once, and as a function of the argument
  // that the kernel forms, 1 + d times the true one for the rounding d of tp:
  // p(u) - d (i + u) p'(u) for the piece i, to first order in d, again a cubic.
  static __device__ __forceinline__ float4 table_entry(const float4* __restrict__ gtab, int i,
                                                       const P3DConsts& k) {
    if constexpr (!DIRECT) return gtab[i];
    const double2* d = reinterpret_cast<const double2*>(gtab + 2 * GTAB_N) + 2 * i;
    const double f = i & 1 ? k.h5 : k.g3, e = k.tp_error, t = (double)(i >> 1);
    const double2 a = d[0], b = d[1];  // p(u) = a.x + a.y u + b.x u^2 + b.y u^3
    return make_float4((float)(f * (a.x - e * (t * a.y))),
                       (float)(f * (a.y - e * (a.y + 2.0 * t * b.x))),
                       (float)(f * (b.x - e * (2.0 * b.x + 3.0 * t * b.y))),
                       (float)(f * (b.y - e * (3.0 * b.y))));
  }

  // PIN: keep the near range a branch.  With no work of its own in
  // near_cb the compiler if-converts it, and every pair then pays the exp (a
  // transcendental, about three issue slots) and the selects.  Where near_cb
  // does FP64 sums it stays a branch by itself, and the pin would only stop
  // the loop around it from unrolling.  Measured on the 2^20 ring: the
  // compensated vel-only kernel 593 -> 515 ms with the pin; the plain FP32
  // vel+dvort kernel (two targets per lane) 680 -> 700 ms, so eval() does
  // not pin.
  template <bool ZETA, bool PIN = false, class Same, class Near>
  static __device__ __forceinline__ void eval_ranges(float r2, const P3DConsts& k,
                                                     const float4* tab, Same&& same, float& Kv,
                                                     float& Kh, float& eta, float& Kfar,
                                                     Near&& near_cb) {
    const Far f = far(r2, k);
    float g = f.g, h = f.h, z = 0.f, kf = f.g;
    if (r2 < k.q_far) {
      if constexpr (PIN) asm volatile("");
      near<ZETA>(f, r2, k, tab, same, g, h, z);
      near_cb(g, z);
      kf = 0.f;
    }
    Kv = g;
    Kh = h;
    eta = z;
    Kfar = kf;
  }

  // The same with the far range's own work in a callback on an else
  // branch, far_cb(G): the caller needs no copy of G that the near branch
  // would zero (a register copy per pair otherwise).  Ring of 2^20, fused
  // vel + dvort: 694.5 -> 679.1 ms (three runs of each in turn).
  // NEST: for callers that use neither zeta nor, below rho^2 = 208, anything
  // but FP64 sums of G: beyond q_exp (there 1 - rho zeta and 1 - zeta/(3 G) round
  // to 1) G and H are the far form's, bit for bit, and the exp is skipped.  Of
  // the ring's rounds (a wave and a source) 9.4 % have a pair below 208 and 3.6 %
  // one below 46: 65536 2685 -> 2652 us, cube of 50000 1681 -> 1636 (targets not
  // ordered, where nearly every such round has both: 6000 59.8 -> 61.1 with it).
  template <bool ZETA, bool NEST, class Same, class Near, class FarCb>
  static __device__ __forceinline__ void eval_split(float r2, const P3DConsts& k,
                                                    const float4* tab, Same&& same, float& Kv,
                                                    float& Kh, float& eta, Near&& near_cb,
                                                    FarCb&& far_cb) {
    const Far f = far(r2, k);
    float g = f.g, h = f.h, z = 0.f;
    if (r2 < k.q_far) {
      if (!NEST || r2 < k.q_exp) near<ZETA>(f, r2, k, tab, same, g, h, z);
      near_cb(g, z);
    } else {
      far_cb(f.g);
    }
    Kv = g;
    Kh = h;
    eta = z;
  }

  template <bool ZETA, class Same>
  static __device__ __forceinline__ void eval(float r2, const P3DConsts& k, const float4* tab,
                                              Same&& same, float& Kv, float& Kh, float& eta) {
    float kf;
    eval_ranges<ZETA>(r2, k, tab, same, Kv, Kh, eta, kf, [](float, float) {});
  }
};

// Waves that share their targets (Q > 1): the part [wave_part, wave_part_end)
// of a tile of cnt sources that a wave takes, a multiple of four long except
// for the last (the loops are unrolled by two and four).  The bounds are scalar,
// and so is the loop (bounds in VGPRs, us: 3D velocity of 10000 particles 51.5
// -> 48.4, 3600 filaments on 20000 targets 161 -> 154, 2D Gaussian with the
// viscous term 12000 100.4 -> 93.4).
template <int Q>
__device__ __forceinline__ int wave_part(int cnt, int tid) {
  if constexpr (Q == 1) return 0;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  return min(cnt, w * (((cnt + 4 * Q - 1) / (4 * Q)) * 4));
}
template <int Q>
__device__ __forceinline__ int wave_part_end(int cnt, int part) {
  if constexpr (Q == 1) return cnt;
  return min(cnt, part + ((cnt + 4 * Q - 1) / (4 * Q)) * 4);
}

// The target whose partials a thread of a 256-thread reduction sums, and their
// sum over the partitions in d; true where this thread holds the total.
// ROWS = 1: 256 targets per workgroup.  ROWS = 4, for few targets, where the
// loads' latency bounds it: 64 targets, wave w adding partitions w, w + 4, ...,
// then the first wave the others' sums.  1 -> 4, us a call: Gaussian vel +
// dvort + visc of 2000 particles 25.2 -> 21.4, Winckelmans vel + dvort of 5000
// 37.7 -> 33.6; but 65536 Gaussian 2629 -> 2639 (reduce_rows).
template <int NA, int ROWS>
__device__ __forceinline__ bool sum_partitions(const double* __restrict__ partial, int n_split,
                                               int n_tgt, int& i, double (&d)[NA]) {
  __shared__ double share[ROWS > 1 ? ROWS - 1 : 1][ROWS > 1 ? NA : 1][64];
  const int lane = threadIdx.x & 63, w = ROWS > 1 ? threadIdx.x >> 6 : 0;
  i = ROWS > 1 ? blockIdx.x * 64 + lane : blockIdx.x * 256 + threadIdx.x;
#pragma unroll
  for (int a = 0; a < NA; ++a) d[a] = 0.0;
  if (i < n_tgt) {
    // the loads of several partitions in flight at once
#pragma unroll 4
    for (int s = w; s < n_split; s += ROWS)
#pragma unroll
      for (int a = 0; a < NA; ++a) d[a] += partial[((size_t)s * NA + a) * n_tgt + i];
  }
  if constexpr (ROWS > 1) {
    if (w > 0) {
#pragma unroll
      for (int a = 0; a < NA; ++a) share[w - 1][a][lane] = d[a];
    }
    __syncthreads();
    if (w > 0) return false;
#pragma unroll
    for (int v = 0; v < ROWS - 1; ++v)
#pragma unroll
      for (int a = 0; a < NA; ++a) d[a] += share[v][a][lane];
  }
  return i < n_tgt;
}
inline int reduce_rows(int n_tgt) { return n_tgt <= 32768 ? 4 : 1; }

}  // namespace cvtx
