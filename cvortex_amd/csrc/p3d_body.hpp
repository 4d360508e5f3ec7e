// p3d_body.hpp -- the P3D pair loop shared by the regular kernel (p3d.hip)
// and the persistent multi-cloud kernel (batched.hip).  See p3d.hip for the
// scheme.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.hpp"

namespace cvtx {

// Canonical layout of the per-target sums (FP64 partials and epilogue).
template <int MASK>
struct P3DLayout {
  static constexpr int VEL = 0;
  static constexpr int A = (MASK & OUT_VEL) ? 3 : 0;       // sum Kv a_s
  static constexpr int H = A + 3;                           // sum Kh (a_t.c) d
  static constexpr int E = A + ((MASK & OUT_DVORT) ? 6 : 0); // sum eta a_s
  static constexpr int EV = E + 3;                          // sum eta V_s
  static constexpr int N = E + ((MASK & OUT_VISC) ? 4 : 0);
  static constexpr bool NEED_TA = (MASK & (OUT_DVORT | OUT_VISC)) != 0;
};

// Register layout of the accumulators.  FP32 accumulators hold the sums
// whose terms carry no coherent large component: vel (sum Kv d x a_s) and
// the gradient term (sum Kh (a_t.c) d).  With ACC_COMP the stretching sum
// sum Kv a_s and the PSE sums sum eta a_s, sum eta V_s are accumulated per
// pair in FP64: their near-field terms are large and nearly parallel to a_t,
// and only their small component normal to a_t (or the small difference
// V_t E - a_t e) survives, so FP32 tile sums would lose several digits
// there.  With ACC_PLAIN and ACC_TILES everything is FP32 (ACC_TILES folds
// the tile sums by TwoSum, which suits fields whose near terms are not
// coherent, e.g. i.i.d. strengths).
// SPLIT (Gaussian with ACC_COMP): only pairs with rho^2 < 208 go to FP64,
// inside the regularisation's near branch; the stretching terms of the
// pairs beyond (Kv < 208^-3/2 in reduced units, and eta = 0 there) are
// summed in FP32 tiles combined by TwoSum, in the F_A slots, on the far
// branch (GaussianKernel::eval_split).
template <int REG, int MASK, int ACC>
struct P3DRegs {
  static constexpr bool DBL = (ACC == ACC_COMP);
  static constexpr bool SPLIT = DBL && REG == REG_GAUSSIAN;
  static constexpr int F_VEL = 0;
  static constexpr int F_A = (MASK & OUT_VEL) ? 3 : 0;  // plain, or the far part with SPLIT
  static constexpr int F_H = F_A + (((!DBL || SPLIT) && (MASK & OUT_DVORT)) ? 3 : 0);
  static constexpr int F_E = F_H + ((MASK & OUT_DVORT) ? 3 : 0);  // plain only
  static constexpr int NF = F_E + ((!DBL && (MASK & OUT_VISC)) ? 4 : 0);
  static constexpr int D_A = 0;
  static constexpr int D_E = (MASK & OUT_DVORT) ? 3 : 0;
  static constexpr int ND = DBL ? (D_E + ((MASK & OUT_VISC) ? 4 : 0)) : 0;
};

struct P3DKParams {
  const float4* __restrict__ src_pv;
  const float4* __restrict__ src_a;
  const float4* __restrict__ tgt_pv;
  const float4* __restrict__ tgt_a;
  const float4* __restrict__ gtab;
  float* __restrict__ out_vel;
  float* __restrict__ out_dvort;
  float* __restrict__ out_visc;
  double* __restrict__ partial;          // indexed by target slot
  const int* __restrict__ tgt_perm;      // slot -> target (nullptr: identity)
  int n_src, n_tgt, split_len, n_split;
  P3DConsts rc;
  Scales sc;
};

// How a Winckelmans pair with equal coordinates, or a singular one with r^2 = 0,
// is dropped (the others test for it in their own kernels).  SELF_NONE: it need
// not be, the velocity term being Kv (d x a_s) with d = 0 and Kv finite.
// SELF_TEST: a compare per pair.  SELF_WATCH: only the tile's smallest r^2 is kept
// (r^2 + sigma^2 for Winckelmans without the exchange), a third as many
// instructions; where it is that of such a pair the caller repeats the tile with
// SELF_TEST (see p3d_block).
enum SelfMode : int { SELF_NONE, SELF_TEST, SELF_WATCH };

// A coordinate in the kernel's units.  Gaussian: one that overflows there (a particle
// parked at FLT_MAX) stays as it is: the square of its distance to any other is
// infinite in either unit, and its pairs give 0, where an infinite difference gives
// NaN.  (Winckelmans, whose pairs at infinite r^2 are NaN in reduced units too, does
// without: in its staging the test costs 128 clouds 41.4 -> 42.7 ms.)
template <int REG>
__device__ __forceinline__ float scaled(float x, float xs) {
  const float y = x * xs;
  return REG == REG_GAUSSIAN && __builtin_isinf(y) ? x : y;
}

template <int REG, int MASK, int ACC, int SELF, bool DIRECT>
__device__ __forceinline__ void p3d_pair(const float4 sp, const float4 sa, const double2* pxy,
                                         const double2* pzv, const float3 xt, const float3 at,
                                         const P3DConsts& rc, const float4* tab, float* acc,
                                         double* dacc, float& smin) {
  using R = P3DRegs<REG, MASK, ACC>;
  const float dx = xt.x - sp.x;
  const float dy = xt.y - sp.y;
  const float dz = xt.z - sp.z;
  constexpr bool REDUCED = REG == REG_WINCKELMANS && winckelmans_reduced(MASK);
  const float z2 = REG == REG_WINCKELMANS && !REDUCED ? __builtin_fmaf(dz, dz, rc.s2)
                   : REG == REG_GAUSSIAN && DIRECT ? __builtin_fmaf(dz, dz, 1e-30f)
                                                   : dz * dz;
  const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, z2));
  auto same_place = [&] {
    if constexpr (REDUCED || (REG == REG_GAUSSIAN && !DIRECT)) return r2 == 0.f;
    // zeros of either sign: -0.0 - (+0.0) is -0.0
    // (the larger of three that propagates NaN: one instruction and a compare)
    const float x = __builtin_elementwise_abs(dx), y = __builtin_elementwise_abs(dy);
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(x, y),
                                         __builtin_elementwise_abs(dz)) == 0.f;
  };
  constexpr bool ZETA = (MASK & OUT_VISC) != 0;
  float Kv, Kh, eta, Kfar = 0.f;
  if constexpr (REG == REG_WINCKELMANS) {
    const float S = REDUCED ? __builtin_fmaf(r2, rc.inv_s2, 1.f) : r2;
    RegKernel<REG_WINCKELMANS>::eval(S, rc, Kv, Kh, eta);
    if constexpr (SELF == SELF_WATCH) smin = fminf(smin, r2);
    if constexpr (SELF == SELF_TEST) {
      const bool same = same_place();
      Kv = same ? 0.f : Kv;
      eta = same ? 0.f : eta;
    }
  } else if constexpr (R::SPLIT && (MASK & OUT_DVORT) != 0) {
    GaussianKernel<DIRECT>::template eval_split<ZETA, DIRECT && !ZETA>(
        r2, rc, tab, same_place, Kv, Kh, eta, [&](float kn, float en) {
      const double2 sxy = *pxy, szv = *pzv;
      const double k = (double)kn;
      dacc[R::D_A + 0] = __builtin_fma(k, sxy.x, dacc[R::D_A + 0]);
      dacc[R::D_A + 1] = __builtin_fma(k, sxy.y, dacc[R::D_A + 1]);
      dacc[R::D_A + 2] = __builtin_fma(k, szv.x, dacc[R::D_A + 2]);
      if constexpr ((MASK & OUT_VISC) != 0) {
        const double e = (double)en;
        dacc[R::D_E + 0] = __builtin_fma(e, sxy.x, dacc[R::D_E + 0]);
        dacc[R::D_E + 1] = __builtin_fma(e, sxy.y, dacc[R::D_E + 1]);
        dacc[R::D_E + 2] = __builtin_fma(e, szv.x, dacc[R::D_E + 2]);
        dacc[R::D_E + 3] = __builtin_fma(e, szv.y, dacc[R::D_E + 3]);
      }
    }, [&](float kf) {
      acc[R::F_A + 0] = __builtin_fmaf(kf, sa.x, acc[R::F_A + 0]);
      acc[R::F_A + 1] = __builtin_fmaf(kf, sa.y, acc[R::F_A + 1]);
      acc[R::F_A + 2] = __builtin_fmaf(kf, sa.z, acc[R::F_A + 2]);
    });
  } else if constexpr (R::SPLIT) {
    constexpr bool PIN = (MASK & (OUT_DVORT | OUT_VISC)) == 0;  // no FP64 near sums
    GaussianKernel<DIRECT>::template eval_ranges<ZETA, PIN>(r2, rc, tab, same_place, Kv, Kh, eta, Kfar,
                                                       [&](float kn, float en) {
      // FP64 source strengths are read from LDS here, on the rare path (a
      // conversion of sa would be speculated out of the branch)
      const double2 sxy = *pxy, szv = *pzv;
      if constexpr ((MASK & OUT_DVORT) != 0) {
        const double k = (double)kn;
        dacc[R::D_A + 0] = __builtin_fma(k, sxy.x, dacc[R::D_A + 0]);
        dacc[R::D_A + 1] = __builtin_fma(k, sxy.y, dacc[R::D_A + 1]);
        dacc[R::D_A + 2] = __builtin_fma(k, szv.x, dacc[R::D_A + 2]);
      }
      if constexpr ((MASK & OUT_VISC) != 0) {
        const double e = (double)en;
        dacc[R::D_E + 0] = __builtin_fma(e, sxy.x, dacc[R::D_E + 0]);
        dacc[R::D_E + 1] = __builtin_fma(e, sxy.y, dacc[R::D_E + 1]);
        dacc[R::D_E + 2] = __builtin_fma(e, szv.x, dacc[R::D_E + 2]);
        dacc[R::D_E + 3] = __builtin_fma(e, szv.y, dacc[R::D_E + 3]);
      }
    });
  } else if constexpr (REG == REG_GAUSSIAN) {
    GaussianKernel<DIRECT>::template eval<ZETA>(r2, rc, tab, same_place, Kv, Kh, eta);
  } else if constexpr (REG == REG_SINGULAR) {
    RegKernel<REG_SINGULAR>::template eval<SELF != SELF_WATCH>(r2, rc, tab, Kv, Kh, eta);
    if constexpr (SELF == SELF_WATCH) smin = fminf(smin, r2);
  } else {
    RegKernel<REG>::template eval<(MASK & (OUT_DVORT | OUT_VISC)) != 0>(r2, rc, tab, Kv, Kh, eta);
  }
  if constexpr ((MASK & (OUT_VEL | OUT_DVORT)) != 0) {
    // c = d x a_s
    const float cx = __builtin_fmaf(dy, sa.z, -dz * sa.y);
    const float cy = __builtin_fmaf(dz, sa.x, -dx * sa.z);
    const float cz = __builtin_fmaf(dx, sa.y, -dy * sa.x);
    if constexpr ((MASK & OUT_VEL) != 0) {
      acc[R::F_VEL + 0] = __builtin_fmaf(Kv, cx, acc[R::F_VEL + 0]);
      acc[R::F_VEL + 1] = __builtin_fmaf(Kv, cy, acc[R::F_VEL + 1]);
      acc[R::F_VEL + 2] = __builtin_fmaf(Kv, cz, acc[R::F_VEL + 2]);
    }
    if constexpr ((MASK & OUT_DVORT) != 0) {
      if constexpr (R::SPLIT) {
        // the far range's stretching sum was added by eval_split's callback
      } else if constexpr (R::DBL) {
        const double2 sxy = *pxy, szv = *pzv;
        const double k = (double)Kv;
        dacc[R::D_A + 0] = __builtin_fma(k, sxy.x, dacc[R::D_A + 0]);
        dacc[R::D_A + 1] = __builtin_fma(k, sxy.y, dacc[R::D_A + 1]);
        dacc[R::D_A + 2] = __builtin_fma(k, szv.x, dacc[R::D_A + 2]);
      } else {
        acc[R::F_A + 0] = __builtin_fmaf(Kv, sa.x, acc[R::F_A + 0]);
        acc[R::F_A + 1] = __builtin_fmaf(Kv, sa.y, acc[R::F_A + 1]);
        acc[R::F_A + 2] = __builtin_fmaf(Kv, sa.z, acc[R::F_A + 2]);
      }
      const float t = Kh * __builtin_fmaf(at.x, cx, __builtin_fmaf(at.y, cy, at.z * cz));
      acc[R::F_H + 0] = __builtin_fmaf(t, dx, acc[R::F_H + 0]);
      acc[R::F_H + 1] = __builtin_fmaf(t, dy, acc[R::F_H + 1]);
      acc[R::F_H + 2] = __builtin_fmaf(t, dz, acc[R::F_H + 2]);
    }
  }
  if constexpr ((MASK & OUT_VISC) != 0 && !R::SPLIT) {
    if constexpr (R::DBL) {
      const double2 sxy = *pxy, szv = *pzv;
      const double e = (double)eta;
      dacc[R::D_E + 0] = __builtin_fma(e, sxy.x, dacc[R::D_E + 0]);
      dacc[R::D_E + 1] = __builtin_fma(e, sxy.y, dacc[R::D_E + 1]);
      dacc[R::D_E + 2] = __builtin_fma(e, szv.x, dacc[R::D_E + 2]);
      dacc[R::D_E + 3] = __builtin_fma(e, szv.y, dacc[R::D_E + 3]);
    } else {
      acc[R::F_E + 0] = __builtin_fmaf(eta, sa.x, acc[R::F_E + 0]);
      acc[R::F_E + 1] = __builtin_fmaf(eta, sa.y, acc[R::F_E + 1]);
      acc[R::F_E + 2] = __builtin_fmaf(eta, sa.z, acc[R::F_E + 2]);
      acc[R::F_E + 3] = __builtin_fmaf(eta, sp.w, acc[R::F_E + 3]);
    }
  }
}

// Final combination of the reduced sums for one target (FP64).
template <int MASK>
__device__ __forceinline__ void p3d_finish(const double* a, float3 at, float vt, const Scales& sc,
                                           float* out_vel, float* out_dvort, float* out_visc,
                                           int i) {
  using L = P3DLayout<MASK>;
  if constexpr ((MASK & OUT_VEL) != 0) {
    out_vel[3 * (size_t)i + 0] = (float)(sc.vel * a[L::VEL + 0]);
    out_vel[3 * (size_t)i + 1] = (float)(sc.vel * a[L::VEL + 1]);
    out_vel[3 * (size_t)i + 2] = (float)(sc.vel * a[L::VEL + 2]);
  }
  if constexpr ((MASK & OUT_DVORT) != 0) {
    const double ax = at.x, ay = at.y, az = at.z;
    const double Ax = a[L::A + 0], Ay = a[L::A + 1], Az = a[L::A + 2];
    const double wx = ay * Az - az * Ay;
    const double wy = az * Ax - ax * Az;
    const double wz = ax * Ay - ay * Ax;
    out_dvort[3 * (size_t)i + 0] = (float)(sc.dG * wx + sc.dH * a[L::H + 0]);
    out_dvort[3 * (size_t)i + 1] = (float)(sc.dG * wy + sc.dH * a[L::H + 1]);
    out_dvort[3 * (size_t)i + 2] = (float)(sc.dG * wz + sc.dH * a[L::H + 2]);
  }
  if constexpr ((MASK & OUT_VISC) != 0) {
    const double v = vt, e = a[L::EV];
    out_visc[3 * (size_t)i + 0] = (float)(sc.visc * (v * a[L::E + 0] - (double)at.x * e));
    out_visc[3 * (size_t)i + 1] = (float)(sc.visc * (v * a[L::E + 1] - (double)at.y * e));
    out_visc[3 * (size_t)i + 2] = (float)(sc.visc * (v * a[L::E + 2] - (double)at.z * e));
  }
}

// Shared-memory staging of one workgroup.  A source is read from LDS on
// every pair: staged as {x, y, z, ax} and {ay, az} (with the viscous term
// {ay, az, volume, -}), it is one 16-byte and one 8-byte read, where
// {x, y, z, volume} and {ax, ay, az, -} took two 12-byte reads.  Measured on
// the 2^20 ring: fused vel + dvort 671.4 -> 659.7 ms, dvort alone
// 595.0 -> 585.6 ms, vel + dvort + visc 695.4 -> 673.0 ms, identical results.
template <int REG, int MASK, int ACC, int WG>
struct P3DSmem {
  static constexpr bool DBL = P3DRegs<REG, MASK, ACC>::ND > 0;  // FP64 source strengths
  static constexpr bool VOL = (MASK & OUT_VISC) != 0;
  using Tail = typename std::conditional<VOL, float4, float2>::type;
  float4 xa[WG];   // x, y, z, ax
  Tail tl[WG];     // ay, az (, volume)
  double2 xy[DBL ? WG : 1];
  double2 zv[DBL ? WG : 1];
  float4 tab[REG == REG_GAUSSIAN ? 2 * GTAB_N : 1];
};

// FP64 sums of the waves that share targets (Q > 1), one set per wave but the
// first.
template <int MASK, int Q>
struct P3DShare {
  double d[Q > 1 ? Q - 1 : 1][Q > 1 ? P3DLayout<MASK>::N : 1][64];
};

// One workgroup: targets base + k*WG + lane (k < T) that are < tgt_end,
// against sources [s0, s1).  Q > 1 (T = 1): targets base + lane of 64, the
// same in all Q waves, each of which takes 1/Q of every tile's sources; their
// sums are added in FP64 at the end (see narrow_cfg).  Writes the outputs
// (n_split == 1) or the FP64 partials of partition `split`.  The caller has loaded sm.tab (Gaussian)
// and issues no barrier-sensitive work on sm around the call.
// DIRECT: which form of the Gaussian pair (GaussianKernel).
template <int REG, int MASK, int ACC, int T, int WG, bool DIRECT, int Q = 1>
__device__ __forceinline__ void p3d_block(const P3DKParams& p, const P3DConsts& rc,
                                          const Scales& sc, int base, int tgt_end, int s0,
                                          int s1, int split, P3DSmem<REG, MASK, ACC, WG>& sm,
                                          P3DShare<MASK, Q>* share = nullptr) {
  static_assert(Q == 1 || (T == 1 && WG == 64 * Q), "a group of shared targets is one wave wide");
  using L = P3DLayout<MASK>;
  using R = P3DRegs<REG, MASK, ACC>;
  constexpr int NF = R::NF;
  constexpr int ND = R::ND > 0 ? R::ND : 1;
  // P3DConsts::xs
  constexpr bool SCALED = (REG == REG_WINCKELMANS && !winckelmans_reduced(MASK)) || REG == REG_GAUSSIAN;
  constexpr bool DBL_ = P3DSmem<REG, MASK, ACC, WG>::DBL;
  const int tid = threadIdx.x;
  const int tl = Q == 1 ? tid : tid & 63;  // target within the group
  float3 xt[T], at[T];
  float vt[T];
#pragma unroll
  for (int k = 0; k < T; ++k) {
    int i = base + k * WG + tl;
    i = i < tgt_end ? i : tgt_end - 1;
    if (p.tgt_perm) i = p.tgt_perm[i];
    const float4 q = p.tgt_pv[i];
    xt[k] = SCALED ? make_float3(scaled<REG>(q.x, rc.xs), scaled<REG>(q.y, rc.xs), scaled<REG>(q.z, rc.xs))
                   : make_float3(q.x, q.y, q.z);
    vt[k] = q.w;
    if constexpr (L::NEED_TA) {
      const float4 w = p.tgt_a[i];
      at[k] = make_float3(w.x, w.y, w.z);
    } else {
      at[k] = make_float3(0.f, 0.f, 0.f);
    }
  }

  float acc[T][NF];
  float lo[T][NF];
  float hi[T][NF];
  double dacc[T][ND];
#pragma unroll
  for (int k = 0; k < T; ++k) {
#pragma unroll
    for (int a = 0; a < NF; ++a) { acc[k][a] = 0.f; lo[k][a] = 0.f; hi[k][a] = 0.f; }
#pragma unroll
    for (int a = 0; a < ND; ++a) dacc[k][a] = 0.0;
  }

  const P3DConsts rv = loop_consts(rc);
  const bool one_array = p.src_pv == p.tgt_pv && p.tgt_perm == nullptr;
  for (int ts = s0; ts < s1; ts += WG) {
    const int cnt = min(WG, s1 - ts);
    const int part = wave_part<Q>(cnt, tid), end = wave_part_end<Q>(cnt, part);
    __syncthreads();
    if (tid < cnt) {
      float4 q = p.src_pv[ts + tid];
      const float4 w = p.src_a[ts + tid];
      if constexpr (SCALED) {
        q.x = scaled<REG>(q.x, rc.xs);
        q.y = scaled<REG>(q.y, rc.xs);
        q.z = scaled<REG>(q.z, rc.xs);
      }
      sm.xa[tid] = make_float4(q.x, q.y, q.z, w.x);
      if constexpr (P3DSmem<REG, MASK, ACC, WG>::VOL)
        sm.tl[tid] = make_float4(w.y, w.z, q.w, 0.f);
      else
        sm.tl[tid] = make_float2(w.y, w.z);
      if constexpr (DBL_) {
        sm.xy[tid] = make_double2((double)w.x, (double)w.y);
        sm.zv[tid] = make_double2((double)w.z, (double)q.w);
      }
    }
    __syncthreads();
    // two sources per iteration, except around the velocity-only Gaussian's
    // pinned near-range branch, which cannot be unrolled, and four for the
    // short velocity-only pair with one target per lane (uniform cube of
    // 8192, Winckelmans: 41.0 -> 39.0 us per evaluation; 79.7 -> 63.0 us
    // with one wave per SIMD; eight sources: 40.9 us)
    constexpr int kUnroll = (R::SPLIT && (MASK & (OUT_DVORT | OUT_VISC)) == 0)
                                ? 1
                                : ((MASK == OUT_VEL && T == 1) ? 4 : 2);
    float smin = __builtin_inff();
    auto tile = [&](auto mode) {
      if constexpr (ACC != ACC_PLAIN) {
#pragma unroll
        for (int k = 0; k < T; ++k)
#pragma unroll
          for (int a = 0; a < NF; ++a) acc[k][a] = 0.f;
      }
      // the LDS index runs in a VGPR too: an SGPR index would cost an
      // SGPR-reading move per source to form the ds_read address
      int jv = in_vgpr(part);
      // The place of this loop in its 32 bytes matters where the issue is full: 128
      // clouds take 41.9 ms with its start at 12 or 16 of them, where this puts it,
      // 42.4 at 20 or 28 and 43.6 at 0, 4 or 8 (measured for this form only).
      if constexpr (REG == REG_WINCKELMANS && MASK == (OUT_VEL | OUT_DVORT) && ACC == ACC_TILES &&
                    T == 1 && decltype(mode)::value == SELF_WATCH)
        asm volatile(".p2align 5");
#pragma unroll kUnroll
      for (int j = part; j < end; ++j, ++jv) {
        const float4 xa = sm.xa[jv];
        const auto tl = sm.tl[jv];
        float vol = 0.f;
        if constexpr (P3DSmem<REG, MASK, ACC, WG>::VOL) vol = tl.z;
        const float4 sp = make_float4(xa.x, xa.y, xa.z, vol);
        const float4 sa = make_float4(xa.w, tl.x, tl.y, 0.f);
#pragma unroll
        for (int k = 0; k < T; ++k)
          p3d_pair<REG, MASK, ACC, decltype(mode)::value, DIRECT>(sp, sa, &sm.xy[DBL_ ? jv : 0],
                                                          &sm.zv[DBL_ ? jv : 0], xt[k], at[k], rv,
                                                          sm.tab, acc[k], dacc[k], smin);
      }
    };
    // Winckelmans with stretching or viscous terms: a target meets itself (or
    // another particle at its place) in one tile of many, so the tile's sums
    // are formed without a test and formed again with it only where some
    // pair's r^2 was 0 or, where S starts from sigma^2, S was (r below 2^-12
    // sigma).  Both give the same value
    // for every other pair.  One FP32 running sum cannot be taken back.
    // With Q > 1 the partitions are of a few tiles, and it tests each pair
    // (4000 particles, vel + dvort, 31.0 -> 26.0 us).
    // With S formed from sigma^2 (RegKernel) 36 issue slots per pair instead
    // of 41, ms: 128 clouds, tile-compensated 51.1 -> 46.6; 64 clouds, FP64
    // stretching 32.1 -> 30.8; velocity of 100000 (S alone) 4.40 -> 4.07.  With the
    // exchange, where S is r^2/sigma^2 + 1, 400000 particles 146.7 -> 143.4 by the
    // test per tile alone.
    // Singular, whose Kv is infinite there, likewise (r^2 = 0) for every output:
    // a compare and one or two selects less.  100000 particles on 300000, velocity
    // 11.95 -> 11.16 ms, with the stretching 20.50 -> 19.23.
    constexpr bool WATCH = Q == 1 && ACC != ACC_PLAIN &&
                           (REG == REG_SINGULAR ||
                            (REG == REG_WINCKELMANS && (MASK & (OUT_DVORT | OUT_VISC)) != 0));
    if constexpr (WATCH) {
      // (a block's own tiles, where sources and targets are one array, are known)
      bool test = one_array && ts < base + T * WG && ts + cnt > base;
      if (!test) {
        double before[T][ND];
#pragma unroll
        for (int k = 0; k < T; ++k)
#pragma unroll
          for (int a = 0; a < ND; ++a) before[k][a] = dacc[k][a];
        tile(std::integral_constant<int, SELF_WATCH>());
        if (__any(smin <= (REG == REG_SINGULAR || winckelmans_reduced(MASK) ? 0.f : rc.s2))) {
          test = true;
#pragma unroll
          for (int k = 0; k < T; ++k)
#pragma unroll
            for (int a = 0; a < ND; ++a) dacc[k][a] = before[k][a];
        }
      }
      if (test) tile(std::integral_constant<int, SELF_TEST>());
    } else {
      tile(std::integral_constant<int, MASK == OUT_VEL ? SELF_NONE : SELF_TEST>());
    }
    if constexpr (ACC != ACC_PLAIN) {
#pragma unroll
      for (int k = 0; k < T; ++k)
#pragma unroll
        for (int a = 0; a < NF; ++a) two_sum_add(hi[k][a], lo[k][a], acc[k][a]);
    }
  }

#pragma unroll
  for (int k = 0; k < T; ++k) {
    const int i = base + k * WG + tl;
    if (Q == 1 && i >= tgt_end) continue;
    // gather the canonical layout
    double d[L::N];
    auto fval = [&](int a) -> double {
      return (ACC != ACC_PLAIN) ? (double)hi[k][a] + (double)lo[k][a] : (double)acc[k][a];
    };
    if constexpr ((MASK & OUT_VEL) != 0) {
#pragma unroll
      for (int c = 0; c < 3; ++c) d[L::VEL + c] = fval(R::F_VEL + c);
    }
    if constexpr ((MASK & OUT_DVORT) != 0) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if constexpr (R::SPLIT)
          d[L::A + c] = dacc[k][R::D_A + c] + fval(R::F_A + c);
        else
          d[L::A + c] = R::DBL ? dacc[k][R::D_A + c] : fval(R::F_A + c);
        d[L::H + c] = fval(R::F_H + c);
      }
    }
    if constexpr ((MASK & OUT_VISC) != 0) {
#pragma unroll
      for (int c = 0; c < 4; ++c) d[L::E + c] = R::DBL ? dacc[k][R::D_E + c] : fval(R::F_E + c);
    }
    if constexpr (Q > 1) {
      const int w = tid >> 6;
      if (w > 0) {
#pragma unroll
        for (int a = 0; a < L::N; ++a) share->d[w - 1][a][tl] = d[a];
      }
      __syncthreads();
      if (w > 0 || i >= tgt_end) return;
#pragma unroll
      for (int v = 0; v < Q - 1; ++v)
#pragma unroll
        for (int a = 0; a < L::N; ++a) d[a] += share->d[v][a][tl];
    }
    if (p.n_split == 1) {
      p3d_finish<MASK>(d, at[k], vt[k], sc, p.out_vel, p.out_dvort, p.out_visc,
                       p.tgt_perm ? p.tgt_perm[i] : i);
    } else {
#pragma unroll
      for (int a = 0; a < L::N; ++a)
        p.partial[((size_t)split * L::N + a) * p.n_tgt + i] = d[a];
    }
  }
}


}  // namespace cvtx
