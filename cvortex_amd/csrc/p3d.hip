// p3d.hip -- 3D vortex particle direct-sum kernels for gfx950.
//
// One kernel evaluates any subset of {vel, dvort, visc} for the targets of a
// workgroup against one partition of the sources:
//   * each lane owns T targets in registers (targets k*WG + lane of the
//     workgroup's block, so target loads are coalesced);
//   * sources stream through LDS in tiles of WG particles, loaded coalesced
//     by the whole workgroup and then read by every lane at the same address
//     (an LDS broadcast), so each source is fetched from memory once per
//     workgroup and shared by WG*T targets;
//   * per pair: d, r2, one regularisation evaluation shared by all outputs,
//     then FMA accumulation into the reduced sums of device_common.hpp;
//   * ACC_COMP: per-tile FP32 sums folded into a TwoSum (hi, lo) pair per
//     accumulator, FP64 stretching and PSE sums per pair; ACC_TILES: the
//     folded tile sums for every accumulator; ACC_PLAIN: one FP32 running sum;
//   * n_split > 1: each grid row handles one source partition and writes FP64
//     partial sums; p3d_reduce adds the partitions in FP64 and applies the
//     epilogue.  Otherwise the epilogue runs in the main kernel.
// Reference semantics: src/P3D.cpp:51-144 (pairs), :230-296 (sums),
// :324-456 (M2M); GPU scaling ocl_P3D.cpp:164,299-304,337,482-487,698-702.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "kernels.hpp"
#include "p3d_body.hpp"

namespace cvtx {

int p3d_nacc(int mask) {
  return ((mask & OUT_VEL) ? 3 : 0) + ((mask & OUT_DVORT) ? 6 : 0) + ((mask & OUT_VISC) ? 4 : 0);
}

template <int REG, int MASK, int ACC, int T, int WG, int Q = 1>
__global__ __launch_bounds__(WG) void p3d_kernel(P3DKParams p) {
  __shared__ P3DSmem<REG, MASK, ACC, WG> sm;
  __shared__ P3DShare<MASK, Q> share;
  if constexpr (REG == REG_GAUSSIAN) {
    for (int i = threadIdx.x; i < 2 * GTAB_N; i += WG)
      sm.tab[i] = GaussianKernel<Q == 1>::table_entry(p.gtab, i, p.rc);
  }
  const int s0 = blockIdx.y * p.split_len;
  const int s1 = min(s0 + p.split_len, p.n_src);
  p3d_block<REG, MASK, ACC, T, WG, Q == 1, Q>(p, p.rc, p.sc, blockIdx.x * (WG * T / Q), p.n_tgt, s0, s1,
                                      blockIdx.y, sm, &share);
}

template <int MASK, int ROWS>
__global__ __launch_bounds__(256) void p3d_reduce(P3DKParams p) {
  using L = P3DLayout<MASK>;
  constexpr int NA = L::N;
  int i;
  double d[NA];
  if (!sum_partitions<NA, ROWS>(p.partial, p.n_split, p.n_tgt, i, d)) return;
  const int t = p.tgt_perm ? p.tgt_perm[i] : i;
  const float4 q = p.tgt_pv[t];
  float3 at = make_float3(0.f, 0.f, 0.f);
  if constexpr (L::NEED_TA) {
    const float4 w = p.tgt_a[t];
    at = make_float3(w.x, w.y, w.z);
  }
  p3d_finish<MASK>(d, at, q.w, p.sc, p.out_vel, p.out_dvort, p.out_visc, t);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

bool p3d_supported(int reg, int mask) {
  if (reg < REG_SINGULAR || reg > REG_GAUSSIAN) return false;
  if (mask <= 0 || mask > 7) return false;
  if ((mask & OUT_VISC) && (reg == REG_SINGULAR || reg == REG_PLANETARY)) return false;
  return true;
}

// The exponent e for which sigma 2^e is in [1, 2) (0 for a radius
// that is zero, infinite or NaN).
static int radius_exponent(float sigma) {
  const double s = std::fabs((double)sigma);
  if (!(s > 0.0) || !std::isfinite(s)) return 0;
  return std::min(126, std::max(-126, -std::ilogb(s)));
}

// Winckelmans in reduced units: the relative rounding a of 1/sigma^2 as the kernel
// has it, S = 1 + a q.
static double reduced_rounding(double s) {
  const float inv = (float)(1.0 / (s * s));
  return std::isfinite(inv) && inv > 0.f ? (double)inv * (s * s) : 1.0;
}

P3DConsts p3d_consts(int reg, float sigma, int mask, int acc, bool direct) {
  P3DConsts k{};
  const double s = std::fabs((double)sigma);
  k.s2 = (float)(s * s);
  k.inv_s2 = (float)(1.0 / (s * s));
  if (reg == REG_GAUSSIAN) {
    k.xs = (float)std::ldexp(1.0, radius_exponent(sigma));
    // (an infinite radius is scaled by 0 below, 0 and NaN give NaN there)
    const double sx = std::isinf(s) || s == 0.0 ? 1.0 : s * (double)k.xs;
    k.inv_s2 = (float)(1.0 / (sx * sx));
    const double t = direct ? sx : 1.0, t2 = t * t;
    // (r^2 comes in the units of t, or multiplied by 1/sigma^2 as rounded)
    const double c1 = -0.5 / (std::log(2.0) * (direct ? t2 : sx * sx * (double)k.inv_s2));
    k.c1 = (float)c1;
    k.c1_rest = (float)((c1 - (double)k.c1) * std::log(2.0));
    k.c2 = (float)std::sqrt(2.0 / M_PI);
    k.g3 = 1.0 / (t2 * t);
    k.h5 = 1.0 / (t2 * t2 * t);
    k.nt1 = (float)(-1.0 / t);
    k.nt3 = (float)(-1.0 / (3.0 * t2 * t));
    k.tp = (float)(GTAB_PER_UNIT / t);
    k.tp_error = (double)k.tp * t / GTAB_PER_UNIT - 1.0;
    // Where no pair's FP64 sum and no zeta depends on it, the far form is taken
    // from where the near one rounds to it: 1 - rho zeta = 1 from rho^2 = 38 on,
    // and G - zeta/3 = G from 44 on.  Bit for bit the same results; velocity, us:
    // ring of 100000 4113 -> 4005, box of 50000 1401 -> 1193.
    if (mask == OUT_VEL) k.q_far = 40.f;
    else if (!(mask & OUT_VISC) && acc != ACC_COMP) k.q_far = k.q_exp;
    // as limits of r^2 (in units of sigma^2 where not direct)
    k.q_far = (float)(k.q_far * t2);
    k.q_exp = (float)(k.q_exp * t2);
    k.q_tab = (float)(k.q_tab * t2);
  }
  if (reg == REG_WINCKELMANS) {
    // sigma^2 or its reciprocal is rounded, one relative error for all pairs, and
    // the constants are chosen so that Kv is exact far away and at r = 0 all the
    // same (and Kh, in reduced units): the radii whose squares round most, error
    // common to all pairs of a core, 1.0e-7 -> 4e-8.
    if (winckelmans_reduced(mask)) {
      const double a = reduced_rounding(s);
      k.c1 = (float)(2.5 * std::pow(a, -1.5) - 1.0);
      k.s2 = (float)(3.5 * std::pow(a, -2.5) - 1.0 - (double)k.c1);
    } else {
      k.xs = (float)std::ldexp(1.0, radius_exponent(sigma));
      const double t = s * (double)k.xs;
      // no field of a radius that is no length: 0 and NaN give NaN, an infinite
      // one is scaled by 0 (p3d_scales)
      const double t2 = std::isinf(s) ? 1.0 : (s == 0.0 ? std::nan("") : t * t);
      k.s2 = (float)t2;
      k.c1 = (float)((double)k.s2 * (2.5 * std::pow((double)k.s2 / t2, 1.5) - 1.0));
    }
  }
  return k;
}

Scales p3d_scales(int reg, float sigma, float nu, int mask, bool direct) {
  Scales sc;
  const double s = std::fabs((double)sigma);
  const double sgn = sigma < 0 ? -1.0 : 1.0;
  const double k4pi = 1.0 / (4.0 * M_PI);
  const double s3 = s * s * s, s5 = s3 * s * s;
  switch (reg) {
    case REG_GAUSSIAN: {
      // as for Winckelmans below
      const double x = std::ldexp(1.0, radius_exponent(sigma)), t = std::isinf(s) ? 1.0 : s * x;
      const double on = std::isinf(s) ? 0.0 : (s > 0.0 ? 1.0 : std::nan(""));
      const double f = direct ? 1.0 : 1.0 / (t * t * t);
      sc.vel = -k4pi * x * x * on * f;
      sc.dG = sgn * k4pi * x * x * x * on * f;
      sc.dH = 3.0 * sc.dG * (direct ? 1.0 : 1.0 / (t * t));
      sc.visc = on * (2.0 * (double)nu / (s * s)) *
                (std::sqrt(2.0 / M_PI) / (double)(float)std::sqrt(2.0 / M_PI));
      break;
    }
    case REG_WINCKELMANS: {
      const double on = std::isinf(s) ? 0.0 : (s > 0.0 ? 1.0 : std::nan(""));
      if (winckelmans_reduced(mask)) {
        // S^-3/2 and S^-5/2 far away; S^-9/2 on average over a uniform
        // neighbourhood, where q / (1 + q) has the mean 1/3 under the weight
        // (1 + q)^-4.5 q^1/2 dq
        const double a = reduced_rounding(s);
        sc.vel = -k4pi / s3 * on * std::pow(a, 1.5);
        sc.dG = -sgn * sc.vel;
        sc.dH = 3.0 * sgn * k4pi / s5 * on * std::pow(a, 2.5);
        sc.visc = 2.0 * (double)nu / (s * s) * on * 52.5 * std::pow(a, 1.5);
      } else {
        // in positions multiplied by x: Kv is x^-3 of the dimensional one, each
        // position factor x
        const double x = std::ldexp(1.0, radius_exponent(sigma));
        sc.vel = -k4pi * x * x * on;
        sc.dG = sgn * k4pi * x * x * x * on;
        sc.dH = 3.0 * sc.dG;
      }
      break;
    }
    case REG_PLANETARY:
      sc.vel = -k4pi / s3;
      sc.dG = sgn * k4pi / s3;
      sc.dH = 3.0 * sgn * k4pi / s5;
      break;
    default:  // singular: Kv = r^-3, Kh = r^-5 are dimensional
      sc.vel = -k4pi;
      sc.dG = sgn * k4pi;
      sc.dH = 3.0 * sgn * k4pi;
      break;
  }
  return sc;
}

size_t p3d_workspace_bytes(const P3DJob& j, const LaunchCfg& c) {
  if (c.n_split <= 1) return 0;
  return (size_t)c.n_split * p3d_nacc(j.mask) * (size_t)j.n_tgt * sizeof(double);
}

namespace {

using KernelFn = void (*)(P3DKParams);

template <int REG, int MASK, int ACC>
KernelFn pick_T(int T, int q) {
  if (q == 4) return T == 1 ? p3d_kernel<REG, MASK, ACC, 1, 256, 4> : nullptr;
  switch (T) {
    case 1: return p3d_kernel<REG, MASK, ACC, 1, 256>;
    case 4: return p3d_kernel<REG, MASK, ACC, 4, 256>;
    default: return p3d_kernel<REG, MASK, ACC, 2, 256>;
  }
}

template <int REG, int MASK>
KernelFn pick_acc(int acc, int T, int q) {
  if (acc == ACC_PLAIN) return pick_T<REG, MASK, ACC_PLAIN>(T, q);
  if (acc == ACC_TILES) return pick_T<REG, MASK, ACC_TILES>(T, q);
  return pick_T<REG, MASK, ACC_COMP>(T, q);
}

template <int REG>
KernelFn pick_mask_inviscid(int mask, int acc, int T, int q) {
  switch (mask) {
    case OUT_VEL: return pick_acc<REG, OUT_VEL>(acc, T, q);
    case OUT_DVORT: return pick_acc<REG, OUT_DVORT>(acc, T, q);
    case OUT_VEL | OUT_DVORT: return pick_acc<REG, OUT_VEL | OUT_DVORT>(acc, T, q);
    default: return nullptr;
  }
}

template <int REG>
KernelFn pick_mask_viscous(int mask, int acc, int T, int q) {
  switch (mask) {
    case OUT_VEL: return pick_acc<REG, OUT_VEL>(acc, T, q);
    case OUT_DVORT: return pick_acc<REG, OUT_DVORT>(acc, T, q);
    case OUT_VISC: return pick_acc<REG, OUT_VISC>(acc, T, q);
    case OUT_VEL | OUT_DVORT: return pick_acc<REG, OUT_VEL | OUT_DVORT>(acc, T, q);
    case OUT_DVORT | OUT_VISC: return pick_acc<REG, OUT_DVORT | OUT_VISC>(acc, T, q);
    case OUT_VEL | OUT_DVORT | OUT_VISC: return pick_acc<REG, OUT_VEL | OUT_DVORT | OUT_VISC>(acc, T, q);
    default: return nullptr;
  }
}

KernelFn pick_kernel(int reg, int mask, int acc, int T, int q) {
  switch (reg) {
    case REG_SINGULAR: return pick_mask_inviscid<REG_SINGULAR>(mask, acc, T, q);
    case REG_PLANETARY: return pick_mask_inviscid<REG_PLANETARY>(mask, acc, T, q);
    case REG_WINCKELMANS: return pick_mask_viscous<REG_WINCKELMANS>(mask, acc, T, q);
    case REG_GAUSSIAN: return pick_mask_viscous<REG_GAUSSIAN>(mask, acc, T, q);
    default: return nullptr;
  }
}

template <int ROWS>
KernelFn pick_reduce(int mask) {
  switch (mask) {
    case OUT_VEL: return p3d_reduce<OUT_VEL, ROWS>;
    case OUT_DVORT: return p3d_reduce<OUT_DVORT, ROWS>;
    case OUT_VISC: return p3d_reduce<OUT_VISC, ROWS>;
    case OUT_VEL | OUT_DVORT: return p3d_reduce<OUT_VEL | OUT_DVORT, ROWS>;
    case OUT_DVORT | OUT_VISC: return p3d_reduce<OUT_DVORT | OUT_VISC, ROWS>;
    case OUT_VEL | OUT_DVORT | OUT_VISC: return p3d_reduce<OUT_VEL | OUT_DVORT | OUT_VISC, ROWS>;
    default: return nullptr;
  }
}

}  // namespace

hipError_t launch_p3d(const P3DJob& j, const LaunchCfg& c, hipStream_t s) {
  if (j.n_tgt <= 0) return hipSuccess;
  if (!p3d_supported(j.reg, j.mask)) return hipErrorInvalidValue;
  if (j.n_src < 0 || c.wg != 256) return hipErrorInvalidValue;
  if ((j.mask & (OUT_DVORT | OUT_VISC)) && j.tgt_a == nullptr) return hipErrorInvalidValue;
  if (j.reg == REG_GAUSSIAN && j.gtab == nullptr) return hipErrorInvalidValue;
  // every output the mask selects must exist, and the inputs it reads
  if (((j.mask & OUT_VEL) && !j.out_vel) || ((j.mask & OUT_DVORT) && !j.out_dvort) ||
      ((j.mask & OUT_VISC) && !j.out_visc) || !j.tgt_pv || (j.n_src > 0 && (!j.src_pv || !j.src_a)))
    return hipErrorInvalidValue;
  KernelFn k = pick_kernel(j.reg, j.mask, j.acc, c.T, c.q);
  if (!k) return hipErrorInvalidValue;

  P3DKParams p{};
  p.src_pv = j.src_pv;
  p.src_a = j.src_a;
  p.tgt_pv = j.tgt_pv;
  p.tgt_a = j.tgt_a;
  p.gtab = j.gtab;
  p.out_vel = j.out_vel;
  p.out_dvort = j.out_dvort;
  p.out_visc = j.out_visc;
  p.partial = j.partial;
  p.tgt_perm = j.tgt_perm;
  p.n_src = j.n_src;
  p.n_tgt = j.n_tgt;
  p.rc = p3d_consts(j.reg, j.sigma, j.mask, j.acc, c.q == 1);
  p.sc = p3d_scales(j.reg, j.sigma, j.nu, j.mask, c.q == 1);

  int n_split = c.n_split;
  int split_len = c.split_len;
  if (n_split <= 1 || j.n_src == 0) {
    n_split = 1;
    split_len = j.n_src > 0 ? j.n_src : 1;
  } else {
    if (split_len <= 0 || split_len % (c.wg / c.q) != 0) return hipErrorInvalidValue;
    if ((long long)split_len * n_split < j.n_src) return hipErrorInvalidValue;
    if (j.partial == nullptr) return hipErrorInvalidValue;
  }
  p.n_split = n_split;
  p.split_len = split_len;

  const int tgt_per_block = c.wg * c.T / c.q;
  dim3 grid((j.n_tgt + tgt_per_block - 1) / tgt_per_block, n_split);
  hipLaunchKernelGGL(k, grid, dim3(c.wg), 0, s, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || n_split == 1) return e;
  const int rows = reduce_rows(j.n_tgt), sums = 256 / rows;
  hipLaunchKernelGGL(rows == 4 ? pick_reduce<4>(j.mask) : pick_reduce<1>(j.mask),
                     dim3((j.n_tgt + sums - 1) / sums), dim3(256), 0, s, p);
  return hipGetLastError();
}

}  // namespace cvtx
