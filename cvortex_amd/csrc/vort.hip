// vort.hip -- vorticity field of 3D vortex particles (cvtx_P3D_M2M_vort) and
// the Pedrizzetti relaxation update, for gfx950.
//
// Semantics are those of the reference CPU path (src/P3D.cpp:298-322,
// 458-498, 669-707):
//   omega(x) = sum over sources s with |dx|, |dy|, |dz| < 5 sigma of
//              zeta(|x_s - x| / sigma) alpha_s,   then / (4 pi sigma^3)
// with d = x_s - x, the cut-off box tested component-wise in FP32 exactly as
// the reference tests it, and the self-pair included (zeta(0) is finite).
// (The reference's OpenCL kernel has neither the cut-off nor the self-pair;
// the CPU path is the one followed here.)
//
// Structure: as the pair kernels -- 256-source LDS tiles shared by the
// workgroup, T targets per lane, FP32 tile sums combined by TwoSum, optional
// source partitions with an FP64 reduction.  Because the cut-off makes the
// interaction short-ranged, large problems run on Morton-sorted sources and
// targets (vort_sorted_kernel): every 64-source chunk carries its bounding
// box, and each wave visits only the chunks whose box is not separated from
// the box of its own targets by the cut-off or more along any axis.  FP32
// subtraction is monotonic, so every pair of a skipped chunk would fail the
// reference's own box test, and every pair of a chunk whose farthest corner
// is inside would pass it: neither changes a result.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "kernels.hpp"

namespace cvtx {

namespace {

// zeta(rho) up to the per-call constant the epilogue applies (vort_scale).
template <int REG>
struct Zeta;

// eval(dx, dy, dz, rsigma, sigma, divide, consts): rsigma = 1/sigma and
// sigma feed only the planetary core test (rho = |d| rsigma, or |d| / sigma
// when `divide`, as the reference's two vorticity forms compute it).
template <>
struct Zeta<REG_SINGULAR> {  // zeta = 0
  static __device__ __forceinline__ float eval(float, float, float, float, float, bool,
                                               const RegConsts&) {
    return 0.f;
  }
};

template <>
struct Zeta<REG_WINCKELMANS> {  // 7.5 (rho^2 + 1)^-3.5 -> y^7, y = (q + 1)^-1/2
  static __device__ __forceinline__ float eval(float dx, float dy, float dz, float, float, bool,
                                               const RegConsts& k) {
    const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
    const float y = __builtin_amdgcn_rsqf(__builtin_fmaf(r2, k.inv_s2, 1.f));
    const float y2 = y * y;
    const float y3 = y2 * y;
    return (y3 * y3) * y;
  }
};

template <>
struct Zeta<REG_PLANETARY> {  // 3 inside the core, 0 outside -> 1 / 0
  // The core test is a discontinuity, so rho is formed with the reference's
  // FP32 operations: |d| = sqrt(dx dx + dy dy + dz dz) rounded at every
  // step, then rho = |d| * (1/sigma) (src/P3D.cpp:314-315) or |d| / sigma
  // (src/P3D.cpp:154-155).
  static __device__ __forceinline__ float eval(float dx, float dy, float dz, float rsigma,
                                               float sigma, bool divide, const RegConsts&) {
    const float r2 = rn_add(rn_add(rn_mul(dx, dx), rn_mul(dy, dy)), rn_mul(dz, dz));
    const float r = __fsqrt_rn(r2);
    const float rho = divide ? __fdiv_rn(r, sigma) : rn_mul(r, rsigma);
    return rho < 1.f ? 1.f : 0.f;
  }
};

template <>
struct Zeta<REG_GAUSSIAN> {  // sqrt(2/pi) exp(-rho^2 / 2) -> 2^(r^2 c1)
  static __device__ __forceinline__ float eval(float dx, float dy, float dz, float, float, bool,
                                               const RegConsts& k) {
    const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
    return __builtin_amdgcn_exp2f(r2 * k.c1);  // c1 = -log2(e) / (2 sigma^2)
  }
};

struct VortKParams {
  const float4* __restrict__ src_pv;
  const float4* __restrict__ src_a;
  const float4* __restrict__ tgt;
  const int* __restrict__ tgt_perm;   // slot -> target (nullptr: identity)
  const float4* __restrict__ src_xa;  // sorted sources {x, y, z, alpha x}, 64 per chunk
  const float2* __restrict__ src_bc;  // {alpha y, alpha z}
  const float4* __restrict__ box_lo;  // bounding box of each chunk's finite sources
  const float4* __restrict__ box_hi;
  float* __restrict__ out;
  double* __restrict__ partial;
  int n_src, n_tgt, split_len, n_split;
  float cutoff;  // 5 sigma in FP32, as the reference forms it (+inf: no cut-off)
  float rsigma;  // 1 / sigma in FP32
  float sigma;
  int divide;    // planetary rho = |d| / sigma instead of |d| * rsigma
  RegConsts rc;
  double scale;  // zeta constant / (4 pi sigma^3)
};

__device__ __forceinline__ float wave_min(float v) {
  for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}

template <int REG, int ACC, int T, int WG>
__global__ __launch_bounds__(WG) void vort_kernel(VortKParams p) {
  __shared__ float4 s_pv[WG];
  __shared__ float4 s_a[WG];
  const int tid = threadIdx.x;
  const int base = blockIdx.x * (WG * T);
  float3 xt[T];
#pragma unroll
  for (int k = 0; k < T; ++k) {
    int i = base + k * WG + tid;
    i = i < p.n_tgt ? i : p.n_tgt - 1;
    if (p.tgt_perm) i = p.tgt_perm[i];
    const float4 q = p.tgt[i];
    xt[k] = make_float3(q.x, q.y, q.z);
  }
  float acc[T][3], sh[T][3], sl[T][3];
#pragma unroll
  for (int k = 0; k < T; ++k)
#pragma unroll
    for (int a = 0; a < 3; ++a) { acc[k][a] = 0.f; sh[k][a] = 0.f; sl[k][a] = 0.f; }

  const float c = p.cutoff;
  // per-pair uniform values in VGPRs (an SGPR operand blocks dual issue)
  const float cv = in_vgpr(c);
  const RegConsts rv = loop_consts(p.rc);
  const int s0 = blockIdx.y * p.split_len;
  const int s1 = min(s0 + p.split_len, p.n_src);
  for (int ts = s0; ts < s1; ts += WG) {
    const int cnt = min(WG, s1 - ts);
    __syncthreads();
    if (tid < cnt) {
      s_pv[tid] = p.src_pv[ts + tid];
      s_a[tid] = p.src_a[ts + tid];
    }
    __syncthreads();
    if constexpr (ACC == ACC_COMP) {
#pragma unroll
      for (int k = 0; k < T; ++k)
#pragma unroll
        for (int a = 0; a < 3; ++a) acc[k][a] = 0.f;
    }
    int jv = in_vgpr(0);  // LDS index in a VGPR
#pragma unroll 2
    for (int j = 0; j < cnt; ++j, ++jv) {
      const float4 sp = s_pv[jv];
      const float4 sa = s_a[jv];
#pragma unroll
      for (int k = 0; k < T; ++k) {
        const float dx = sp.x - xt[k].x;
        const float dy = sp.y - xt[k].y;
        const float dz = sp.z - xt[k].z;
        const bool in = (__builtin_fabsf(dx) < cv) && (__builtin_fabsf(dy) < cv) &&
                        (__builtin_fabsf(dz) < cv);
        float z = Zeta<REG>::eval(dx, dy, dz, p.rsigma, p.sigma, p.divide != 0, rv);
        z = in ? z : 0.f;
        acc[k][0] = __builtin_fmaf(z, sa.x, acc[k][0]);
        acc[k][1] = __builtin_fmaf(z, sa.y, acc[k][1]);
        acc[k][2] = __builtin_fmaf(z, sa.z, acc[k][2]);
      }
    }
    if constexpr (ACC == ACC_COMP) {
#pragma unroll
      for (int k = 0; k < T; ++k)
#pragma unroll
        for (int a = 0; a < 3; ++a) two_sum_add(sh[k][a], sl[k][a], acc[k][a]);
    }
  }

#pragma unroll
  for (int k = 0; k < T; ++k) {
    const int i = base + k * WG + tid;
    if (i >= p.n_tgt) continue;
    double d[3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
      d[a] = (ACC == ACC_COMP) ? (double)sh[k][a] + (double)sl[k][a] : (double)acc[k][a];
    if (p.n_split == 1) {
      const int o = p.tgt_perm ? p.tgt_perm[i] : i;
#pragma unroll
      for (int a = 0; a < 3; ++a) p.out[3 * (size_t)o + a] = (float)(p.scale * d[a]);
    } else {
#pragma unroll
      for (int a = 0; a < 3; ++a) p.partial[((size_t)blockIdx.y * 3 + a) * p.n_tgt + i] = d[a];
    }
  }
}

// The sorted form.  A wave owns 64 T targets and walks the source chunks of
// its partition on its own: 64 lanes test 64 chunk boxes at once and a ballot
// gives the chunks to visit; in a visited chunk each lane tests one source
// against the box of the wave's targets and appends it to one of two queues
// in the wave's part of LDS (or drops it): sources within the cut-off of all
// the targets along every axis, whose pairs need no test, and sources that
// are apart for some of them.  A full queue block of 64 is then summed.
// Nothing in the loop is shared between waves, so there is no barrier and no
// wave waits for another's chunks.  A source with a coordinate that is not
// finite is dropped and a target with one gets zero: the reference's box test
// fails for all its pairs.
//
// Bound by the LDS: with one target per lane a source's 24 bytes take its port
// 12 cycles per wave, 48 for the four SIMDs of a CU, as long as 24 issue slots,
// where an untested pair needs about 13 and a tested one 18.  On the 2^20 ring
// the port is busy in 76 % of the cycles and the vector units issue 0.34
// instructions per SIMD and cycle (68 % of the most they can), in 10.9 ms.
// There (sigma 0.02) 2.3 % of all pairs are within the box; chunk boxes alone
// leave 4.2 % to visit (20 % of them untested), the per-source test 3.2 % (43 %
// untested).  A relaxation step, ms: 22.9 with one box test per workgroup and
// tile, shared tiles and every pair tested; 15.8 with a wave's own chunks; 11.85
// with the queues and partitions of interleaved chunks.  2^18: 2.29 -> 1.13,
// 2^16: 0.37 -> 0.225, 2^14: 0.106 -> 0.077.
template <int REG, int ACC, int T>
__global__ __launch_bounds__(256) void vort_sorted_kernel(VortKParams p) {
  // queue entries {x, y, z, alpha x}, {alpha y, alpha z}: a ring of two
  // blocks of 64 each for the tested (0) and the untested (1) sources
  __shared__ float4 s_xa[4][2][128];
  __shared__ float2 s_bc[4][2][128];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int base = (blockIdx.x * 4 + w) * (64 * T);
  if (base >= p.n_tgt) return;  // whole waves; no barrier below
  float3 xt[T];
  bool finite[T];
  const float inf = __builtin_inff();
  float3 lo = make_float3(inf, inf, inf), hi = make_float3(-inf, -inf, -inf);
#pragma unroll
  for (int k = 0; k < T; ++k) {
    int i = min(base + k * 64 + lane, p.n_tgt - 1);
    if (p.tgt_perm) i = p.tgt_perm[i];
    const float4 q = p.tgt[i];
    xt[k] = make_float3(q.x, q.y, q.z);
    finite[k] = __builtin_isfinite(q.x) && __builtin_isfinite(q.y) && __builtin_isfinite(q.z);
    if (finite[k]) {
      lo.x = fminf(lo.x, q.x); lo.y = fminf(lo.y, q.y); lo.z = fminf(lo.z, q.z);
      hi.x = fmaxf(hi.x, q.x); hi.y = fmaxf(hi.y, q.y); hi.z = fmaxf(hi.z, q.z);
    }
  }
  lo.x = wave_min(lo.x); lo.y = wave_min(lo.y); lo.z = wave_min(lo.z);
  hi.x = wave_max(hi.x); hi.y = wave_max(hi.y); hi.z = wave_max(hi.z);

  float acc[T][3], sh[T][3], sl[T][3];
#pragma unroll
  for (int k = 0; k < T; ++k)
#pragma unroll
    for (int a = 0; a < 3; ++a) { acc[k][a] = 0.f; sh[k][a] = 0.f; sl[k][a] = 0.f; }

  const float c = p.cutoff;
  const float cv = in_vgpr(c);
  const RegConsts rv = loop_consts(p.rc);
  auto pair = [&](auto untested, const float4 xa, const float2 bc) {
#pragma unroll
    for (int k = 0; k < T; ++k) {
      const float dx = xa.x - xt[k].x;
      const float dy = xa.y - xt[k].y;
      const float dz = xa.z - xt[k].z;
      float z = Zeta<REG>::eval(dx, dy, dz, p.rsigma, p.sigma, p.divide != 0, rv);
      if constexpr (!decltype(untested)::value)
        z = fmaxf(fmaxf(__builtin_fabsf(dx), __builtin_fabsf(dy)), __builtin_fabsf(dz)) < cv ? z : 0.f;
      acc[k][0] = __builtin_fmaf(z, xa.w, acc[k][0]);
      acc[k][1] = __builtin_fmaf(z, bc.x, acc[k][1]);
      acc[k][2] = __builtin_fmaf(z, bc.y, acc[k][2]);
    }
  };
  // sum n (at most 64) entries of a queue from slot `at`
  auto sum = [&](auto untested, int at, int n) {
    constexpr int Q = decltype(untested)::value ? 1 : 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if constexpr (ACC == ACC_COMP) {
#pragma unroll
      for (int k = 0; k < T; ++k)
#pragma unroll
        for (int a = 0; a < 3; ++a) acc[k][a] = 0.f;
    }
    int jv = in_vgpr(at);
    if (n == 64) {
#pragma unroll 4
      for (int j = 0; j < 64; ++j, ++jv) pair(untested, s_xa[w][Q][jv], s_bc[w][Q][jv]);
    } else {
      for (int j = 0; j < n; ++j, ++jv) pair(untested, s_xa[w][Q][jv], s_bc[w][Q][jv]);
    }
    if constexpr (ACC == ACC_COMP) {
#pragma unroll
      for (int k = 0; k < T; ++k)
#pragma unroll
        for (int a = 0; a < 3; ++a) two_sum_add(sh[k][a], sl[k][a], acc[k][a]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  using Tested = std::integral_constant<bool, false>;
  using Untested = std::integral_constant<bool, true>;

  // chunks y, y + n_split, y + 2 n_split, ...: neighbouring chunks go to
  // different partitions, so a wave's work is the same in each
  const int chunks = (p.n_src + 63) / 64;
  const int per = (chunks - (int)blockIdx.y + p.n_split - 1) / p.n_split;
  int at[2] = {0, 0}, count[2] = {0, 0};  // first block and length of the queues
  for (int cb = 0; cb < per; cb += 64) {
    const size_t ci = (size_t)min(cb + lane, per - 1) * p.n_split + blockIdx.y;
    const float4 bl = p.box_lo[ci], bh = p.box_hi[ci];
    const bool apart = (bl.x - hi.x >= c) || (lo.x - bh.x >= c) || (bl.y - hi.y >= c) ||
                       (lo.y - bh.y >= c) || (bl.z - hi.z >= c) || (lo.z - bh.z >= c);
    unsigned long long visit = __ballot(!apart && cb + lane < per);
    if (visit == 0) continue;
    auto source = [&](int b) { return ((size_t)(cb + b) * p.n_split + blockIdx.y) * 64 + lane; };
    size_t i = source(__builtin_ctzll(visit));
    float4 xa = p.src_xa[i];
    float2 bc = p.src_bc[i];
    while (visit != 0) {
      visit &= visit - 1;
      const float4 s = xa;
      const float2 sb = bc;
      if (visit != 0) {  // the next chunk's sources while this one's are handled
        i = source(__builtin_ctzll(visit));
        xa = p.src_xa[i];
        bc = p.src_bc[i];
      }
      // differences from the box's faces: any pair's lies between them
      const float ax = s.x - hi.x, bx = lo.x - s.x;
      const float ay = s.y - hi.y, by = lo.y - s.y;
      const float az = s.z - hi.z, bz = lo.z - s.z;
      const bool fin = __builtin_isfinite(s.x) && __builtin_isfinite(s.y) && __builtin_isfinite(s.z);
      const bool in = fin && fmaxf(fmaxf(fmaxf(ax, bx), fmaxf(ay, by)), fmaxf(az, bz)) < c;
      const bool all = in && fmaxf(fmaxf(fmaxf(-ax, -bx), fmaxf(-ay, -by)), fmaxf(-az, -bz)) < c;
      const unsigned long long m[2] = {__ballot(in && !all), __ballot(all)};
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (q == 0 ? (in && !all) : all) {
          const int slot = (at[q] + count[q] + __popcll(m[q] & ((1ull << lane) - 1))) & 127;
          s_xa[w][q][slot] = s;
          s_bc[w][q][slot] = sb;
        }
        count[q] += __popcll(m[q]);
      }
      if (count[0] >= 64) {
        sum(Tested(), at[0], 64);
        at[0] ^= 64;
        count[0] -= 64;
      }
      if (count[1] >= 64) {
        sum(Untested(), at[1], 64);
        at[1] ^= 64;
        count[1] -= 64;
      }
    }
  }
  sum(Tested(), at[0], count[0]);
  sum(Untested(), at[1], count[1]);

#pragma unroll
  for (int k = 0; k < T; ++k) {
    const int i = base + k * 64 + lane;
    if (i >= p.n_tgt) continue;
    double d[3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
      d[a] = !finite[k] ? 0.0
             : (ACC == ACC_COMP) ? (double)sh[k][a] + (double)sl[k][a] : (double)acc[k][a];
    if (p.n_split == 1) {
      const int o = p.tgt_perm ? p.tgt_perm[i] : i;
#pragma unroll
      for (int a = 0; a < 3; ++a) p.out[3 * (size_t)o + a] = (float)(p.scale * d[a]);
    } else {
#pragma unroll
      for (int a = 0; a < 3; ++a) p.partial[((size_t)blockIdx.y * 3 + a) * p.n_tgt + i] = d[a];
    }
  }
}

// (One thread per target added up to 2048 partitions after one another: 2^20 sources
// on 64 targets 297 -> 180 us, on 1000 582 -> 504, 300000 on 1000 206 -> 176.)
template <int ROWS>
__global__ __launch_bounds__(256) void vort_reduce(VortKParams p) {
  int i;
  double d[3];
  if (!sum_partitions<3, ROWS>(p.partial, p.n_split, p.n_tgt, i, d)) return;
  const int o = p.tgt_perm ? p.tgt_perm[i] : i;
#pragma unroll
  for (int a = 0; a < 3; ++a) p.out[3 * (size_t)o + a] = (float)(p.scale * d[a]);
}

// The sources in sorted order, as the pair loop reads them, and the bounding
// box of each 64-source chunk (one wave each).  Slots past n repeat the last
// source's position with zero strength, so that every chunk is whole.
__global__ __launch_bounds__(256) void sort_sources(const float4* __restrict__ pv,
                                                    const float4* __restrict__ a,
                                                    const int* __restrict__ perm, int n,
                                                    float4* __restrict__ xa,
                                                    float2* __restrict__ bc,
                                                    float4* __restrict__ lo,
                                                    float4* __restrict__ hi) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int j = perm[min(i, n - 1)];
  const float4 q = pv[j], w = a[j];
  xa[i] = make_float4(q.x, q.y, q.z, i < n ? w.x : 0.f);
  bc[i] = i < n ? make_float2(w.y, w.z) : make_float2(0.f, 0.f);
  const bool fin = __builtin_isfinite(q.x) && __builtin_isfinite(q.y) && __builtin_isfinite(q.z);
  const float inf = __builtin_inff();
  const float3 l = make_float3(wave_min(fin ? q.x : inf), wave_min(fin ? q.y : inf), wave_min(fin ? q.z : inf));
  const float3 h = make_float3(wave_max(fin ? q.x : -inf), wave_max(fin ? q.y : -inf), wave_max(fin ? q.z : -inf));
  if ((threadIdx.x & 63) == 0) {
    lo[i >> 6] = make_float4(l.x, l.y, l.z, 0.f);
    hi[i >> 6] = make_float4(h.x, h.y, h.z, 0.f);
  }
}

// Pedrizzetti update (reference src/P3D.cpp:690-702), FP32 in the
// reference's operation order: new = a (1 - fdt) + omega (|a| / |omega|) fdt,
// zero where |omega| == 0.  a is float4 {alpha, 0}; omega float[3 n].
__global__ __launch_bounds__(256) void relax_kernel(float4* __restrict__ a,
                                                    const float* __restrict__ omega, int n,
                                                    float fdt) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float4 ov = a[i];
  const float wx = omega[3 * (size_t)i + 0], wy = omega[3 * (size_t)i + 1], wz = omega[3 * (size_t)i + 2];
  const float aw =
      __fsqrt_rn(rn_add(rn_add(rn_mul(wx, wx), rn_mul(wy, wy)), rn_mul(wz, wz)));
  const float aa = __fsqrt_rn(
      rn_add(rn_add(rn_mul(ov.x, ov.x), rn_mul(ov.y, ov.y)), rn_mul(ov.z, ov.z)));
  const float coeff = __fdiv_rn(aa, aw);
  const float tmp = rn_sub(1.f, fdt);
  const float cf = rn_mul(coeff, fdt);
  float4 nv;
  nv.x = rn_add(rn_mul(ov.x, tmp), rn_mul(wx, cf));
  nv.y = rn_add(rn_mul(ov.y, tmp), rn_mul(wy, cf));
  nv.z = rn_add(rn_mul(ov.z, tmp), rn_mul(wz, cf));
  nv.w = ov.w;
  if (aw == 0.f) nv = make_float4(0.f, 0.f, 0.f, ov.w);
  a[i] = nv;
}

using VFn = void (*)(VortKParams);

template <int REG, int ACC>
VFn vort_T(int T, bool sorted) {
  switch (T) {
    case 1: return sorted ? vort_sorted_kernel<REG, ACC, 1> : vort_kernel<REG, ACC, 1, 256>;
    case 4: return sorted ? vort_sorted_kernel<REG, ACC, 4> : vort_kernel<REG, ACC, 4, 256>;
    default: return sorted ? vort_sorted_kernel<REG, ACC, 2> : vort_kernel<REG, ACC, 2, 256>;
  }
}
template <int REG>
VFn vort_acc(int acc, int T, bool sorted) {
  return acc == ACC_PLAIN ? vort_T<REG, ACC_PLAIN>(T, sorted) : vort_T<REG, ACC_COMP>(T, sorted);
}
VFn vort_pick(int reg, int acc, int T, bool sorted) {
  switch (reg) {
    case REG_SINGULAR: return vort_acc<REG_SINGULAR>(acc, T, sorted);
    case REG_WINCKELMANS: return vort_acc<REG_WINCKELMANS>(acc, T, sorted);
    case REG_PLANETARY: return vort_acc<REG_PLANETARY>(acc, T, sorted);
    case REG_GAUSSIAN: return vort_acc<REG_GAUSSIAN>(acc, T, sorted);
    default: return nullptr;
  }
}

size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

}  // namespace

double vort_scale(int reg, float sigma) {
  // zeta constants: Winckelmans 7.5, planetary 3, Gaussian sqrt(2/pi).  The
  // reference divides by 4 pi sigma^3 with the signed sigma
  // (src/P3D.cpp:320-321); sigma = 0 gives 0 * inf = NaN as there.
  const double s = (double)sigma;
  const double k = reg == REG_WINCKELMANS ? 7.5
                   : reg == REG_PLANETARY ? 3.0
                   : reg == REG_GAUSSIAN  ? std::sqrt(2.0 / M_PI)
                                          : 0.0;
  return k * (1.0 / (4.0 * M_PI * s * s * s));
}

// waves a launch with few targets is split into
constexpr long long VORT_FILL = 24576;

LaunchCfg vort_default_cfg(int n_src, int n_tgt, int n_cu, bool sorted) {
  if (!sorted) return default_cfg(n_src, n_tgt, n_cu);
  // One target per lane: the box of a wave's targets is smaller than with two,
  // so it visits fewer sources (ring 2^20, 16 partitions: 11.9 ms, with two
  // 13.2).  Partitions: the work left is very uneven over the target waves, so
  // 32 of them even for many waves (ring 2^20, ms, 4 / 8 / 16 / 32 / 64:
  // 13.6 / 12.4 / 11.9 / 11.8 / 12.2; 2^16: 0.35 / 0.26 / 0.24 / 0.23 / 0.24),
  // more where the targets are too few to fill the chip (300000 sources on
  // 20000 targets, 32 / 64: 0.48 / 0.44), but eight chunks (two tiles) each (2^14: 32
  // partitions 77 us, 64 84 us).  The FP64 partial sums (24 B per target and
  // partition) are held to 2^26 target-partitions, 1.5 GiB.
  LaunchCfg c;
  c.T = 1;
  const long long tiles = ((long long)n_src + 255) / 256;
  const long long waves = ((long long)n_tgt + 63) / 64;
  long long k = std::max<long long>(32, VORT_FILL / std::max<long long>(waves, 1));
  k = std::min(k, std::max<long long>(1, tiles / 2));
  k = std::min<long long>(k, std::max<long long>(1, (1LL << 26) / std::max(n_tgt, 1)));
  if (k <= 1) return c;
  c.n_split = (int)k;
  c.split_len = (int)((tiles + k - 1) / k * 256);
  return c;
}

size_t vort_workspace_bytes(const VortJob& j, const LaunchCfg& c, bool sorted) {
  size_t b = 0;
  if (c.n_split > 1) b += align256((size_t)c.n_split * 3 * (size_t)j.n_tgt * sizeof(double));
  if (sorted) {
    const size_t tiles = ((size_t)j.n_src + 255) / 256;
    b += (sizeof(float4) + sizeof(float2)) * 256 * tiles + 2 * align256(sizeof(float4) * tiles * 4);
  }
  return b;
}

hipError_t launch_vort(const VortJob& j, const LaunchCfg& c, void* ws, size_t ws_bytes,
                       hipStream_t s) {
  if (j.n_tgt <= 0) return hipSuccess;
  if (j.n_src < 0 || c.wg != 256 || j.reg < REG_SINGULAR || j.reg > REG_GAUSSIAN)
    return hipErrorInvalidValue;
  const bool sorted = j.src_perm != nullptr;
  if (ws_bytes < vort_workspace_bytes(j, c, sorted)) return hipErrorInvalidValue;
  VFn k = vort_pick(j.reg, j.acc, c.T, sorted);
  if (!k) return hipErrorInvalidValue;
  VortKParams p{};
  p.src_pv = j.src_pv;
  p.src_a = j.src_a;
  p.tgt = j.tgt;
  p.tgt_perm = j.tgt_perm;
  p.out = j.out;
  p.n_src = j.n_src;
  p.n_tgt = j.n_tgt;
  // the reference's single-source forms (S2S, S2M) have no cut-off and
  // divide by sigma (src/P3D.cpp:146-161); M2S and M2M cut at 5 sigma
  p.cutoff = j.cutoff ? 5.f * j.sigma : __builtin_inff();
  p.rsigma = 1.f / j.sigma;
  p.sigma = j.sigma;
  p.divide = j.cutoff ? 0 : 1;
  const double sa = (double)j.sigma;
  p.rc.s2 = (float)(sa * sa);
  p.rc.inv_s2 = (float)(1.0 / (sa * sa));
  p.rc.c1 = (float)(-0.5 / (std::log(2.0) * sa * sa));
  p.scale = vort_scale(j.reg, j.sigma);
  char* w = (char*)ws;
  int n_split = c.n_split, split_len = c.split_len;
  if (n_split <= 1 || j.n_src <= 0) {
    n_split = 1;
    split_len = j.n_src > 0 ? j.n_src : 1;
  } else {
    p.partial = (double*)w;
    w += align256((size_t)n_split * 3 * (size_t)j.n_tgt * sizeof(double));
  }
  p.n_split = n_split;
  p.split_len = split_len;
  if (sorted && j.n_src > 0) {
    const int tiles = (j.n_src + 255) / 256;
    float4* xa = (float4*)w;
    w += sizeof(float4) * 256 * (size_t)tiles;
    float2* bc = (float2*)w;
    w += sizeof(float2) * 256 * (size_t)tiles;
    float4* lo = (float4*)w;
    w += align256(sizeof(float4) * (size_t)tiles * 4);
    float4* hi = (float4*)w;
    hipLaunchKernelGGL(sort_sources, dim3(tiles), dim3(256), 0, s, j.src_pv, j.src_a, j.src_perm,
                       j.n_src, xa, bc, lo, hi);
    p.src_xa = xa;
    p.src_bc = bc;
    p.box_lo = lo;
    p.box_hi = hi;
  }
  // (a sorted problem's workgroup is four waves of 64 T targets: as many)
  const int gx = (j.n_tgt + 256 * c.T - 1) / (256 * c.T);
  hipLaunchKernelGGL(k, dim3(gx, n_split), dim3(256), 0, s, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || n_split == 1) return e;
  const int rows = reduce_rows(j.n_tgt), sums = 256 / rows;
  hipLaunchKernelGGL(rows == 4 ? vort_reduce<4> : vort_reduce<1>, dim3((j.n_tgt + sums - 1) / sums),
                     dim3(256), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_relax(float4* a, const float* omega, int n, float fdt, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(relax_kernel, dim3((n + 255) / 256), dim3(256), 0, s, a, omega, n, fdt);
  return hipGetLastError();
}

}  // namespace cvtx
