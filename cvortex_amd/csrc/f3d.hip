// f3d.hip -- straight singular vortex filament kernels for gfx950.
//
// Filaments stream through LDS in tiles; when a tile is staged each
// filament is expanded once per workgroup into
//   { a (start), Gamma/(4pi) },  { b (end), -6 Gamma/(4pi |r0|) },
//   { r0 = b - a, |r0|^2 / 2 },
// so the per-pair work only involves the target-dependent quantities.
//
// Per pair (x the target): r1 = x - a, r2 = x - b, c = r1 x r2 (= r0 x r1),
// P = |r1||r2|, s = |r1| + |r2|, d = r1.r2.  The reference's factors
// (F3D.cpp:34-85)
//   t2 = r0.r1/|r1| - r0.r2/|r2|            and   1/|r1| - 1/|r2|
// cancel in FP32 for targets far from the segment or near its end points,
// so they are evaluated in the algebraically identical forms
//   k = (Gamma/4pi) t2 / |c|^2 = (Gamma/4pi) s / (P (P + d))          (d >= 0)
//                              = (Gamma/4pi) s (P - d) / (P |c|^2)    (d < 0)
//   1/|r1| - 1/|r2| = -r0.(r1 + r2) / (P s)
// (using |c|^2 = P^2 - d^2 and |r2|^2 - |r1|^2 = -r0.(r1 + r2)).  Then
//   vel:   v += k c
//   dvort: B += 3 Gamma/(4pi|r0|) |c| (1/|r1| - 1/|r2|),  S += k r0,
//          dvort = a_t B - S x a_t
// A pair whose terms are not finite (target on a filament's line or an end
// point) contributes zero, as in the reference's GPU kernels
// (nbody.cl:637,718); on the line's extension the velocity term is exactly
// zero there (c = 0) and the stretching term is dropped.
#include <hip/hip_runtime.h>

#include <cmath>

#include "kernels.hpp"
#include "tile_cull.hpp"

namespace cvtx {

int f3d_nacc(int mask) { return ((mask & OUT_VEL) ? 3 : 0) + ((mask & OUT_DVORT) ? 4 : 0); }

struct F3DKParams {
  const float4* __restrict__ fa;
  const float4* __restrict__ fb;
  const float4* __restrict__ tgt_pv;
  const float4* __restrict__ tgt_a;
  float* __restrict__ out_vel;
  float* __restrict__ out_dvort;
  double* __restrict__ partial;
  const int* __restrict__ tgt_perm;  // slot -> target (nullptr: identity)
  int n_fil, n_tgt, split_len, n_split;
};

template <int MASK>
__device__ __forceinline__ void f3d_finish(const double* a, float3 at, const F3DKParams& p, int i) {
  constexpr int D = (MASK & OUT_VEL) ? 3 : 0;
  if constexpr ((MASK & OUT_VEL) != 0) {
    p.out_vel[3 * (size_t)i + 0] = (float)a[0];
    p.out_vel[3 * (size_t)i + 1] = (float)a[1];
    p.out_vel[3 * (size_t)i + 2] = (float)a[2];
  }
  if constexpr ((MASK & OUT_DVORT) != 0) {
    const double B = a[D], Sx = a[D + 1], Sy = a[D + 2], Sz = a[D + 3];
    const double ax = at.x, ay = at.y, az = at.z;
    p.out_dvort[3 * (size_t)i + 0] = (float)(ax * B - (Sy * az - Sz * ay));
    p.out_dvort[3 * (size_t)i + 1] = (float)(ay * B - (Sz * ax - Sx * az));
    p.out_dvort[3 * (size_t)i + 2] = (float)(az * B - (Sx * ay - Sy * ax));
  }
}

// One pair by the general formula (any target position): accumulates into
// acc[0..NA) of one target.  fa = {a, Gamma/(4pi)}, fb = {b, -6 Gamma/(4pi|r0|)},
// f0 = {r0, |r0|^2 / 2}.
template <int MASK>
__device__ __forceinline__ void f3d_pair(const float4 fa, const float4 fb, const float4 f0,
                                         const float3 xt, const float fin, float* acc) {
  constexpr int D = (MASK & OUT_VEL) ? 3 : 0;
  const float r1x = xt.x - fa.x, r1y = xt.y - fa.y, r1z = xt.z - fa.z;
  const float r2x = xt.x - fb.x, r2y = xt.y - fb.y, r2z = xt.z - fb.z;
  // c = r1 x r2 (= r0 x r1); for targets beside the segment its
  // products are smaller than those of r0 x r1, so it loses less to
  // cancellation near the filament
  const float cx = __builtin_fmaf(r1y, r2z, -r1z * r2y);
  const float cy = __builtin_fmaf(r1z, r2x, -r1x * r2z);
  const float cz = __builtin_fmaf(r1x, r2y, -r1y * r2x);
  const float cc = __builtin_fmaf(cx, cx, __builtin_fmaf(cy, cy, cz * cz));
  const float n1s = __builtin_fmaf(r1x, r1x, __builtin_fmaf(r1y, r1y, r1z * r1z));
  const float n2s = __builtin_fmaf(r2x, r2x, __builtin_fmaf(r2y, r2y, r2z * r2z));
  const float n1 = n1s * __builtin_amdgcn_rsqf(n1s);
  const float n2 = n2s * __builtin_amdgcn_rsqf(n2s);
  const float P = n1 * n2;
  const float sum = n1 + n2;
  const float d12 = __builtin_fmaf(r1x, r2x, __builtin_fmaf(r1y, r2y, r1z * r2z));
  const bool same_side = d12 >= 0.f;
  const float den = same_side ? P * (P + d12) : P * cc;
  const float num = same_side ? sum : sum * (P - d12);
  float kk = fa.w * num * __builtin_amdgcn_rcpf(den);
  if constexpr ((MASK & OUT_DVORT) != 0) {
    const float rcc = __builtin_amdgcn_rsqf(cc);
    const float cn = cc * rcc;  // |c|; 0 * inf = NaN when c = 0
    const float p12 = __builtin_fmaf(f0.x, r1x + r2x, __builtin_fmaf(f0.y, r1y + r2y, f0.z * (r1z + r2z)));
    float B = fb.w * cn * (0.5f * p12) * __builtin_amdgcn_rcpf(P * sum);
    // B is NaN whenever c = 0 (target on the filament's line), so the
    // finiteness of B also drops those pairs
    const bool ok = (__builtin_fabsf(kk) < __builtin_inff()) &&
                    (__builtin_fabsf(B) < __builtin_inff());
    B = ok ? B : 0.f;
    const float kd = ok ? kk : 0.f;
    if constexpr ((MASK & OUT_VEL) != 0) {
      kk = (__builtin_fabsf(kk) < __builtin_inff()) ? kk : 0.f;
      acc[0] = __builtin_fmaf(kk, cx, acc[0]);
      acc[1] = __builtin_fmaf(kk, cy, acc[1]);
      acc[2] = __builtin_fmaf(kk, cz, acc[2]);
    }
    acc[D + 0] += B;
    acc[D + 1] = __builtin_fmaf(kd, f0.x, acc[D + 1]);
    acc[D + 2] = __builtin_fmaf(kd, f0.y, acc[D + 2]);
    acc[D + 3] = __builtin_fmaf(kd, f0.z, acc[D + 3]);
  } else {
    kk = (__builtin_fabsf(kk) < fin) ? kk : 0.f;
    acc[0] = __builtin_fmaf(kk, cx, acc[0]);
    acc[1] = __builtin_fmaf(kk, cy, acc[1]);
    acc[2] = __builtin_fmaf(kk, cz, acc[2]);
  }
}

// Far tiles (tile_cull.hpp).  When every target of the block is at least
// half the longest filament of the tile away from the tile's box, every
// pair has r1.r2 = |x - m|^2 - |r0|^2/4 >= 0 (m the filament's midpoint),
// so the same-side form holds for all of them and no pair's terms can be
// infinite.  With y_i = 1/|r_i|, S = |r1| + |r2|, L = |r0| and
// h = |r1||r2| + r1.r2 = (S^2 - L^2) / 2 (which loses at most a bit or two
// at the nearest targets):
//   k = (Gamma/4pi) S / (|r1||r2| h) = (Gamma/4pi) (y1 + y2) / h,
//   1/|r1| - 1/|r2| = -r0.(r1 + r2) y1 y2 / S,  r0.(r1 + r2) / 2 = r0.r1 - L^2/2,
// and c = r0 x r1, the better conditioned product away from the segment.
// The stretching takes 1/h and 1/S from one value, 1/(S h):
//   k = (Gamma/4pi) S^2 z,  B = -(3 Gamma/4pi L) |c| r0.(r1 + r2) h z,
//   z = y1 y2 / (S h);
// the reciprocals of a group's pairs come from one (batch_rcp).  Against the
// form with r1.r2 and one reciprocal each for h and S it saves three
// operations of 30 per pair for the velocity and ten of 58 for both outputs.
// The stretching terms of a pair with c = 0 (a target on the extension of a
// filament's line) are dropped, as the general form does (there |c| = 0 and
// the reference's terms are NaN).
// Bound by vector issue: 2.25 transcendentals per pair along a chain (rsq of
// the new end point, sqrt of |c|^2, half a rcp), 1.5 for the velocity.
// 16384 filaments in chains of 128 x 2^20 targets, ms, old form -> this:
// fused 18.44 -> 14.95, stretching 17.08 -> 14.18, velocity 9.96 -> 9.04.
// Two pairs per group: the velocity with four takes 9.99 ms (more registers:
// 12.35 held to 6 waves per SIMD, with spills), with one 12.2.
template <int MASK, int T>
struct F3DFar {
  static constexpr int U = T >= 2 ? 1 : 2;  // filaments per group
  static constexpr int NP = U * T;          // pairs per group
};

// Waves per SIMD the register allocation must leave room for: the fused
// kernel with one target per lane is held to 5 (96 VGPRs; held to 4 it takes
// 15.25 ms against 14.98), the velocity to 6 (5, 7 and 8: 9.09, 9.10, 9.17
// ms against 9.04); the stretching takes 93 and 5 waves unbounded.
template <int MASK, int T>
constexpr int f3d_min_waves() {
  if constexpr (T != 1) return 1;
  return MASK == (OUT_VEL | OUT_DVORT) ? 5 : (MASK == OUT_VEL ? 6 : 1);
}

// Q > 1 (T = 1): 64 targets per workgroup, the same in all Q waves, each of
// which takes 1/Q of every tile's filaments; their FP64 sums are added at the
// end (see narrow_cfg).
template <int MASK, int ACC, int T, int WG, int Q = 1>
__global__ __launch_bounds__(WG, (f3d_min_waves<MASK, T>())) void f3d_kernel(F3DKParams p) {
  static_assert(Q == 1 || (T == 1 && WG == 64 * Q), "a group of shared targets is one wave wide");
  constexpr int NA = ((MASK & OUT_VEL) ? 3 : 0) + ((MASK & OUT_DVORT) ? 4 : 0);
  constexpr int D = (MASK & OUT_VEL) ? 3 : 0;
  constexpr int WAVES = WG / 64;
  using FF = F3DFar<MASK, T>;
  __shared__ float4 s_a[WG];
  __shared__ float4 s_b[WG];
  __shared__ float4 s_r0[WG];
  __shared__ unsigned long long s_link[WAVES];
  __shared__ BoxPartials<3, WAVES> s_box;
  __shared__ double s_share[Q > 1 ? Q - 1 : 1][Q > 1 ? NA : 1][64];
  const int tid = threadIdx.x;
  const int tl = Q == 1 ? tid : tid & 63;               // target within the group
  const int base = blockIdx.x * (WG * T / Q);
  float3 xt[T], at[T];
#pragma unroll
  for (int k = 0; k < T; ++k) {
    int i = base + k * WG + tl;
    i = i < p.n_tgt ? i : p.n_tgt - 1;
    if (p.tgt_perm) i = p.tgt_perm[i];
    const float4 q = p.tgt_pv[i];
    xt[k] = make_float3(q.x, q.y, q.z);
    if constexpr ((MASK & OUT_DVORT) != 0) {
      const float4 w = p.tgt_a[i];
      at[k] = make_float3(w.x, w.y, w.z);
    } else {
      at[k] = make_float3(0.f, 0.f, 0.f);
    }
  }
  float acc[T][NA], hi[T][NA], lo[T][NA];
#pragma unroll
  for (int k = 0; k < T; ++k)
#pragma unroll
    for (int a = 0; a < NA; ++a) { acc[k][a] = 0.f; hi[k][a] = 0.f; lo[k][a] = 0.f; }

  // box of the block's targets (the clamped duplicates are real targets)
  Box<3> tbox;
  {
    float l3[3] = {xt[0].x, xt[0].y, xt[0].z}, h3[3] = {xt[0].x, xt[0].y, xt[0].z};
    bool fin = true;
#pragma unroll
    for (int k = 0; k < T; ++k) {
      l3[0] = fminf(l3[0], xt[k].x); l3[1] = fminf(l3[1], xt[k].y); l3[2] = fminf(l3[2], xt[k].z);
      h3[0] = fmaxf(h3[0], xt[k].x); h3[1] = fmaxf(h3[1], xt[k].y); h3[2] = fmaxf(h3[2], xt[k].z);
      fin = fin && __builtin_isfinite(xt[k].x) && __builtin_isfinite(xt[k].y) &&
            __builtin_isfinite(xt[k].z);
    }
    tbox = block_box<3, WAVES>(l3, h3, fin, s_box);
  }

  const float k4pi = (float)(1.0 / (4.0 * M_PI));
  const int s0 = blockIdx.y * p.split_len;
  const int s1 = min(s0 + p.split_len, p.n_fil);
  for (int ts = s0; ts < s1; ts += WG) {
    const int cnt = min(WG, s1 - ts);
    __syncthreads();
    {
      float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
      // link: this filament ends where the next one of the tile starts,
      // bit for bit (a polyline), so the two can share that point's
      // distance terms in the far loop
      int link = 0;
      if (tid < cnt) {
        a = p.fa[ts + tid];
        b = p.fb[ts + tid];
        const float rx = b.x - a.x, ry = b.y - a.y, rz = b.z - a.z;
        const float g = a.w * k4pi;
        const float l2 = rx * rx + ry * ry + rz * rz;
        if (tid + 1 < cnt) {
          const float4 an = p.fa[ts + tid + 1];
          link = (int)(__float_as_uint(an.x) == __float_as_uint(b.x)) &
                 (int)(__float_as_uint(an.y) == __float_as_uint(b.y)) &
                 (int)(__float_as_uint(an.z) == __float_as_uint(b.z));
        }
        s_a[tid] = make_float4(a.x, a.y, a.z, g);
        // (a filament of no length contributes nothing: its factor, infinite
        // here, times |c| = 0 would make the far loop's sum NaN)
        s_b[tid] = make_float4(b.x, b.y, b.z, l2 > 0.f ? -6.f * g / __builtin_sqrtf(l2) : 0.f);
        s_r0[tid] = make_float4(rx, ry, rz, 0.5f * l2);
      }
      const unsigned long long links = __ballot(link != 0);
      if ((tid & 63) == 0) s_link[tid >> 6] = links;
      // the tile's box holds both ends of every filament; extra: the
      // longest filament's squared length
      const float l3[3] = {fminf(a.x, b.x), fminf(a.y, b.y), fminf(a.z, b.z)};
      const float h3[3] = {fmaxf(a.x, b.x), fmaxf(a.y, b.y), fmaxf(a.z, b.z)};
      const float rx = b.x - a.x, ry = b.y - a.y, rz = b.z - a.z;
      const bool fin = __builtin_isfinite(a.x) && __builtin_isfinite(a.y) &&
                       __builtin_isfinite(a.z) && __builtin_isfinite(b.x) &&
                       __builtin_isfinite(b.y) && __builtin_isfinite(b.z) &&
                       __builtin_isfinite(a.w);
      box_partial<3, WAVES>(l3, h3, rx * rx + ry * ry + rz * rz, fin, tid < cnt, s_box);
    }
    __syncthreads();
    if constexpr (ACC == ACC_COMP) {
#pragma unroll
      for (int k = 0; k < T; ++k)
#pragma unroll
        for (int a = 0; a < NA; ++a) acc[k][a] = 0.f;
    }
    const int part = wave_part<Q>(cnt, tid), end = wave_part_end<Q>(cnt, part);
    int jv = in_vgpr(part);  // LDS index in a VGPR (no SGPR operand per filament)
    // velocity only: +inf in a VGPR, so |kk| < fin is a VGPR compare (against
    // the literal the compiler emits a class test whose mask operand is an
    // SGPR).  Measured on 16384 filaments x 2^20 targets: vel 16.79 -> 16.54
    // ms; the dvort and fused kernels were slower with it (23.06 -> 23.27,
    // 24.46 -> 24.91) and keep the literal.
    const float fin = [] {
      if constexpr ((MASK & OUT_DVORT) == 0) return in_vgpr(__builtin_inff());
      else return __builtin_inff();
    }();
    const float c126 = in_vgpr(0x1p126f);
    float l2max;
    const Box<3> fbox = box_combine<3, WAVES>(s_box, &l2max);
    // every pair same-side and finite, and the product of the NP values that
    // share a reciprocal normal: h is in [dmin^2, 2 dmax^2], S, by which the
    // stretching multiplies it, in [2 dmin, 2 dmax], so the product of two
    // S h or of four h is within 2^(+-124) in the wide range, that of four
    // S h in the narrow one
    bool far = false;
    if (tbox.finite && fbox.finite) {
      float dmin2, dmax2;
      box_dist2<3>(tbox, fbox, dmin2, dmax2);
      constexpr bool few = FF::NP <= 2 || (MASK & OUT_DVORT) == 0;
      const float lo_ok = few ? 9.3e-10f : 3.1e-5f;   // 2^-30, 2^-15
      const float hi_ok = few ? 5.3e8f : 1.6e4f;      // 2^29, 2^14
      far = dmin2 >= 0.2501f * l2max && dmin2 >= lo_ok && dmax2 <= hi_ok;
    }
    if (far) {
      constexpr int U = FF::U;
      int j = part;
      // the last end point of a group, kept for the next group when the
      // chain runs on into it (its first filament starts there, bit for bit,
      // so the values are those the next group would compute): a third of the
      // end points of a chain's groups of two.  Both paths leave the point,
      // which keeps the register allocator from copying it around the branch.
      float lpx[T], lpy[T], lpz[T], lpn[T], lpy1[T];
      bool carry = false;
      unsigned long long links = 0;
      for (; j + U <= end; j += U, jv += U) {
        if ((j & 63) == 0 || (Q > 1 && j == part)) {
          const unsigned long long m = s_link[j >> 6];
          links = ((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(m >> 32)) << 32) |
                  (unsigned)__builtin_amdgcn_readfirstlane((int)m);
          if (Q > 1) links >>= j & 63;
        }
        float4 fa[U], fb[U], f0[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          fa[u] = s_a[jv + u];
          fb[u] = s_b[jv + u];
          f0[u] = s_r0[jv + u];
        }
        float cx[FF::NP], cy[FF::NP], cz[FF::NP], ys[FF::NP], S2[FF::NP], p12[FF::NP],
            cn[FF::NP], den[FF::NP], X[FF::NP], inv[FF::NP];
        // the terms of pair q (filament u) from r1 = x - a, the norms of r1
        // and r2 and their reciprocals
        auto terms = [&](int q, int u, float r1x, float r1y, float r1z, float n1, float n2,
                         float y1, float y2) {
          cx[q] = __builtin_fmaf(f0[u].y, r1z, -f0[u].z * r1y);
          cy[q] = __builtin_fmaf(f0[u].z, r1x, -f0[u].x * r1z);
          cz[q] = __builtin_fmaf(f0[u].x, r1y, -f0[u].y * r1x);
          const float S = n1 + n2;
          S2[q] = S * S;
          den[q] = __builtin_fmaf(0.5f, S2[q], -f0[u].w);  // |r1||r2| + r1.r2
          if constexpr ((MASK & OUT_DVORT) != 0) {
            ys[q] = y1 * y2;
            X[q] = S * den[q];
            const float cc = __builtin_fmaf(cx[q], cx[q], __builtin_fmaf(cy[q], cy[q], cz[q] * cz[q]));
            cn[q] = __builtin_amdgcn_sqrtf(cc);
            // r0.(r1 + r2) / 2
            p12[q] = __builtin_fmaf(f0[u].x, r1x, __builtin_fmaf(f0[u].y, r1y,
                                                                 __builtin_fmaf(f0[u].z, r1z, -f0[u].w)));
          } else {
            ys[q] = y1 + y2;
            X[q] = den[q];
          }
        };
        // a chained group (each filament ends where the next begins) has
        // U + 1 distinct end points: each point's distance and rsq serve
        // the two filaments that meet there (same formulas as below)
        constexpr unsigned in_group = (1u << (U - 1)) - 1u;
        const bool chained = U > 1 && ((unsigned)links & in_group) == in_group;
        if (chained) {
          if (!carry) {
#pragma unroll
            for (int k = 0; k < T; ++k) {
              lpx[k] = xt[k].x - fa[0].x;
              lpy[k] = xt[k].y - fa[0].y;
              lpz[k] = xt[k].z - fa[0].z;
              const float ns = __builtin_fmaf(lpx[k], lpx[k], __builtin_fmaf(lpy[k], lpy[k], lpz[k] * lpz[k]));
              lpy1[k] = __builtin_amdgcn_rsqf(ns);
              lpn[k] = ns * lpy1[k];
            }
          }
#pragma unroll
          for (int k = 0; k < T; ++k) {
            // walk the points: each filament's terms as soon as its end is known
            float px = lpx[k], py = lpy[k], pz = lpz[k], pn = lpn[k], py1 = lpy1[k];
#pragma unroll
            for (int u = 0; u < U; ++u) {
              const float4 pt = u + 1 < U ? fa[u + 1] : fb[U - 1];
              const float qx = xt[k].x - pt.x, qy = xt[k].y - pt.y, qz = xt[k].z - pt.z;
              const float qns = __builtin_fmaf(qx, qx, __builtin_fmaf(qy, qy, qz * qz));
              const float qy1 = __builtin_amdgcn_rsqf(qns);
              const float qn = qns * qy1;
              terms(u * T + k, u, px, py, pz, pn, qn, py1, qy1);
              px = qx; py = qy; pz = qz; pn = qn; py1 = qy1;
            }
            lpx[k] = px; lpy[k] = py; lpz[k] = pz; lpn[k] = pn; lpy1[k] = py1;
          }
        } else {
#pragma unroll
          for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < T; ++k) {
              const float r1x = xt[k].x - fa[u].x, r1y = xt[k].y - fa[u].y, r1z = xt[k].z - fa[u].z;
              const float r2x = xt[k].x - fb[u].x, r2y = xt[k].y - fb[u].y, r2z = xt[k].z - fb[u].z;
              const float n1s = __builtin_fmaf(r1x, r1x, __builtin_fmaf(r1y, r1y, r1z * r1z));
              const float n2s = __builtin_fmaf(r2x, r2x, __builtin_fmaf(r2y, r2y, r2z * r2z));
              const float y1 = __builtin_amdgcn_rsqf(n1s), y2 = __builtin_amdgcn_rsqf(n2s);
              const float n2 = n2s * y2;
              terms(u * T + k, u, r1x, r1y, r1z, n1s * y1, n2, y1, y2);
              if (u == U - 1) {
                // the group's last end point, as the chained walk leaves it
                lpx[k] = r2x; lpy[k] = r2y; lpz[k] = r2z; lpn[k] = n2; lpy1[k] = y2;
              }
            }
        }
        carry = (links >> (U - 1)) & 1;
        links >>= U;
        batch_rcp<FF::NP>(X, inv);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int k = 0; k < T; ++k) {
            const int q = u * T + k;
            float kk;
            if constexpr ((MASK & OUT_DVORT) != 0) {
              const float z = ys[q] * inv[q];  // y1 y2 / (S (P + r1.r2))
              kk = fa[u].w * S2[q] * z;
              acc[k][D + 0] = __builtin_fmaf(fb[u].w, cn[q] * p12[q] * (den[q] * z), acc[k][D + 0]);
            } else {
              kk = fa[u].w * ys[q] * inv[q];
            }
            if constexpr ((MASK & OUT_VEL) != 0) {
              acc[k][0] = __builtin_fmaf(kk, cx[q], acc[k][0]);
              acc[k][1] = __builtin_fmaf(kk, cy[q], acc[k][1]);
              acc[k][2] = __builtin_fmaf(kk, cz[q], acc[k][2]);
            }
            if constexpr ((MASK & OUT_DVORT) != 0) {
              // kk, or 0 when c = 0: |c| is 0 or at least 2^-75 (the root
              // of a float), so |c| 2^126 clamped to [0, 1] is 0 or 1 (one
              // multiplication with the clamp modifier, where a compare does
              // not dual-issue): lattice fused 19.18 -> 19.03 ms
              // (kk is finite in far tiles, so kk * 0 is 0)
              const float kd = kk * __builtin_amdgcn_fmed3f(cn[q] * c126, 0.f, 1.f);
              acc[k][D + 1] = __builtin_fmaf(kd, f0[u].x, acc[k][D + 1]);
              acc[k][D + 2] = __builtin_fmaf(kd, f0[u].y, acc[k][D + 2]);
              acc[k][D + 3] = __builtin_fmaf(kd, f0[u].z, acc[k][D + 3]);
            }
          }
      }
      for (; j < end; ++j, ++jv) {
        const float4 fa = s_a[jv], fb = s_b[jv], f0 = s_r0[jv];
#pragma unroll
        for (int k = 0; k < T; ++k) f3d_pair<MASK>(fa, fb, f0, xt[k], fin, acc[k]);
      }
    } else {
#pragma unroll 2
      for (int j = part; j < end; ++j, ++jv) {
        const float4 fa = s_a[jv];
        const float4 fb = s_b[jv];
        const float4 f0 = s_r0[jv];
#pragma unroll
        for (int k = 0; k < T; ++k) f3d_pair<MASK>(fa, fb, f0, xt[k], fin, acc[k]);
      }
    }
    if constexpr (ACC == ACC_COMP) {
#pragma unroll
      for (int k = 0; k < T; ++k)
#pragma unroll
        for (int a = 0; a < NA; ++a) two_sum_add(hi[k][a], lo[k][a], acc[k][a]);
    }
  }

#pragma unroll
  for (int k = 0; k < T; ++k) {
    const int i = base + k * WG + tl;
    if (Q == 1 && i >= p.n_tgt) continue;
    double d[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a)
      d[a] = (ACC == ACC_COMP) ? (double)hi[k][a] + (double)lo[k][a] : (double)acc[k][a];
    if constexpr (Q > 1) {
      const int w = tid >> 6;
      if (w > 0) {
#pragma unroll
        for (int a = 0; a < NA; ++a) s_share[w - 1][a][tl] = d[a];
      }
      __syncthreads();
      if (w > 0 || i >= p.n_tgt) return;
#pragma unroll
      for (int v = 0; v < Q - 1; ++v)
#pragma unroll
        for (int a = 0; a < NA; ++a) d[a] += s_share[v][a][tl];
    }
    if (p.n_split == 1) {
      f3d_finish<MASK>(d, at[k], p, p.tgt_perm ? p.tgt_perm[i] : i);
    } else {
#pragma unroll
      for (int a = 0; a < NA; ++a) p.partial[((size_t)blockIdx.y * NA + a) * p.n_tgt + i] = d[a];
    }
  }
}

template <int MASK, int ROWS>
__global__ __launch_bounds__(256) void f3d_reduce(F3DKParams p) {
  constexpr int NA = ((MASK & OUT_VEL) ? 3 : 0) + ((MASK & OUT_DVORT) ? 4 : 0);
  int i;
  double d[NA];
  if (!sum_partitions<NA, ROWS>(p.partial, p.n_split, p.n_tgt, i, d)) return;
  const int t = p.tgt_perm ? p.tgt_perm[i] : i;
  float3 at = make_float3(0.f, 0.f, 0.f);
  if constexpr ((MASK & OUT_DVORT) != 0) {
    const float4 w = p.tgt_a[t];
    at = make_float3(w.x, w.y, w.z);
  }
  f3d_finish<MASK>(d, at, p, t);
}

size_t f3d_workspace_bytes(const F3DJob& j, const LaunchCfg& c) {
  if (c.n_split <= 1) return 0;
  return (size_t)c.n_split * f3d_nacc(j.mask) * (size_t)j.n_tgt * sizeof(double);
}

namespace {
using F3Fn = void (*)(F3DKParams);
template <int MASK, int ACC>
F3Fn f3_T(int T, int q) {
  if (q == 4) return T == 1 ? f3d_kernel<MASK, ACC, 1, 256, 4> : nullptr;
  switch (T) {
    case 1: return f3d_kernel<MASK, ACC, 1, 256>;
    case 4: return f3d_kernel<MASK, ACC, 4, 256>;
    default: return f3d_kernel<MASK, ACC, 2, 256>;
  }
}
template <int MASK>
F3Fn f3_acc(int acc, int T, int q) {
  return acc == ACC_PLAIN ? f3_T<MASK, ACC_PLAIN>(T, q) : f3_T<MASK, ACC_COMP>(T, q);
}
F3Fn f3_pick(int mask, int acc, int T, int q) {
  switch (mask) {
    case OUT_VEL: return f3_acc<OUT_VEL>(acc, T, q);
    case OUT_DVORT: return f3_acc<OUT_DVORT>(acc, T, q);
    case OUT_VEL | OUT_DVORT: return f3_acc<OUT_VEL | OUT_DVORT>(acc, T, q);
    default: return nullptr;
  }
}
template <int ROWS>
F3Fn f3_reduce(int mask) {
  switch (mask) {
    case OUT_VEL: return f3d_reduce<OUT_VEL, ROWS>;
    case OUT_DVORT: return f3d_reduce<OUT_DVORT, ROWS>;
    case OUT_VEL | OUT_DVORT: return f3d_reduce<OUT_VEL | OUT_DVORT, ROWS>;
    default: return nullptr;
  }
}
// Influence matrix (cvtx_F3D_inf_mtrx, reference src/F3D.cpp:204-227):
//   out[i * n_fil + j] = vel(filament j, point i) . dir_i
// with the filament's own strength and, as in f3d_kernel, non-finite terms
// flushed to zero (a strength that is not finite where the columns are loaded, the
// rest by the general form below).  Each lane owns NF adjacent filaments (columns) of its
// workgroup's block and the workgroup walks `rows` consecutive points, staged
// in LDS (a broadcast read puts them in VGPRs; an SGPR operand would halve
// the issue rate of every instruction that reads it).
//
// Two forms of the element.  inf_general is f3d_pair's, right for any point.
// The far form holds where S^2 >= 2 L^2 for S = |r1| + |r2| and the
// filament's length L (then r1.r2 >= 0 and no term is infinite): with
// S^2 - L^2 = 2 (|r1||r2| + r1.r2),
//   k = (Gamma/4pi) (y1 + y2) / (|r1||r2| + r1.r2) = (Gamma/2pi) S y1 y2 / (S^2 - L^2)
// needs neither r1.r2 nor |c|^2 nor the selects, and c = r0 x r1 (r0 = b - a,
// kept in registers) is, away from the segment, the better conditioned
// product.  S^2 - L^2 loses at most one bit there.  A row for which any lane
// of the wave fails the test (or has a NaN) is computed again by the general
// form.  (One test per wave and row against the box around the wave's
// filaments, decided for all rows by one ballot, gave 217 us instead of 222
// on the matrix below, but its wave reductions cost every workgroup more than
// a small matrix's rows: 1786 x 2069 8.4 -> 11.9 us.)  Where the filaments of
// every lane of the wave form a polyline (each starts, bit for bit, where the
// previous one ends, as the spanwise segments of a vortex lattice do), a
// shared end point's distance terms are computed once per row.
//
// What bounds it: the matrix's write and the vector units about equally.  For
// 16384 x 16384 (1 GiB) the kernel takes 222 us, 4.8 TB/s of writes (294 us
// before: every element by the general form, two columns per lane, points in
// SGPRs); with the element arithmetic left out it takes 167 us with 8 rows
// per workgroup and 213 with 32.  16383 x 16384 320 -> 263 us, 4096 x 4096
// 23.4 -> 19.3, 3280 x 1149 10.3 -> 8.6, 923 x 18510 26.6 -> 25.0.
template <int NF>
struct InfCols {
  float3 a[NF], b[NF], r0[NF];
  float g[NF], L2[NF];  // Gamma / (2 pi), |r0|^2
};

__device__ __forceinline__ float3 sub3(float4 x, float3 a) {
  return make_float3(x.x - a.x, x.y - a.y, x.z - a.z);
}
__device__ __forceinline__ float dot3(float3 a, float3 b) {
  return __builtin_fmaf(a.x, b.x, __builtin_fmaf(a.y, b.y, a.z * b.z));
}
__device__ __forceinline__ float3 cross3(float3 a, float3 b) {
  return make_float3(__builtin_fmaf(a.y, b.z, -a.z * b.y), __builtin_fmaf(a.z, b.x, -a.x * b.z),
                     __builtin_fmaf(a.x, b.y, -a.y * b.x));
}

// One element by f3d_pair's formula, projected on e (g = Gamma / (4 pi)).
__device__ __forceinline__ float inf_general(float3 r1, float3 r2, float g, float3 e) {
  const float3 c = cross3(r1, r2);
  const float cc = dot3(c, c);
  const float n1s = dot3(r1, r1), n2s = dot3(r2, r2);
  const float n1 = n1s * __builtin_amdgcn_rsqf(n1s);
  const float n2 = n2s * __builtin_amdgcn_rsqf(n2s);
  const float P = n1 * n2;
  const float sum = n1 + n2;
  const float d12 = dot3(r1, r2);
  const bool same_side = d12 >= 0.f;
  const float den = same_side ? P * (P + d12) : P * cc;
  const float num = same_side ? sum : sum * (P - d12);
  float kk = g * num * __builtin_amdgcn_rcpf(den);
  kk = (__builtin_fabsf(kk) < __builtin_inff()) ? kk : 0.f;
  return kk * dot3(c, e);
}

constexpr long INF_STREAM_ELEMENTS = 64l << 20;  // 256 MiB of floats
constexpr int INF_ROWS = 32;  // rows a workgroup stages at most

// The rows of one workgroup.  WHOLE: the lane's columns are all inside the
// matrix and may be written as one NF * 4-byte store
// (STREAM: past the caches).
template <int NF, bool SHARE, bool WHOLE, bool STREAM>
__device__ __forceinline__ void inf_rows(const InfCols<NF>& c, const float4* s_x, const float4* s_e,
                                         int nr, int j0, int n_fil, float* __restrict__ o) {
  using Vec = float __attribute__((ext_vector_type(NF)));
  using Vec4 = float __attribute__((ext_vector_type(NF), aligned(4)));  // any float's address
  // Added to the squared distances (no instruction more): the reciprocal root of a
  // denormal one is infinite, and the far form would turn that into NaN.
  const float tiny = in_vgpr(0x1p-120f);
  auto norm2 = [&](float3 r) {
    return __builtin_fmaf(r.x, r.x, __builtin_fmaf(r.y, r.y, __builtin_fmaf(r.z, r.z, tiny)));
  };
  int iv = in_vgpr(0);
  float4 xn = s_x[iv], en = s_e[iv];
  for (int i = 0; i < nr; ++i, o += n_fil) {
    const float4 x = xn;
    const float3 e = make_float3(en.x, en.y, en.z);
    ++iv;
    // the next row's point is read while this row's elements are computed
    // (the arrays have a slot past the last row)
    xn = s_x[iv];
    en = s_e[iv];
    Vec v;
    bool far = true;
    float3 r2;
    float y2, n2;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      float3 r1 = r2;
      float y1 = y2, n1 = n2;
      if (f == 0 || !SHARE) {
        r1 = sub3(x, c.a[f]);
        const float ns = norm2(r1);
        y1 = __builtin_amdgcn_rsqf(ns);
        n1 = ns * y1;
      }
      r2 = sub3(x, c.b[f]);
      const float ns = norm2(r2);
      y2 = __builtin_amdgcn_rsqf(ns);
      n2 = ns * y2;
      const float S = n1 + n2;
      const float den = __builtin_fmaf(S, S, -c.L2[f]);
      far = far && den >= c.L2[f];
      const float ce = dot3(cross3(c.r0[f], r1), e);
      v[f] = ((c.g[f] * (S * y1)) * y2) * (ce * __builtin_amdgcn_rcpf(den));
    }
    if (!__all(far)) {
#pragma unroll
      for (int f = 0; f < NF; ++f) v[f] = inf_general(sub3(x, c.a[f]), sub3(x, c.b[f]), 0.5f * c.g[f], e);
    }
    if constexpr (WHOLE) {
      if constexpr (STREAM) __builtin_nontemporal_store(v, reinterpret_cast<Vec*>(o + j0));
      else *reinterpret_cast<Vec4*>(o + j0) = v;
    } else {
#pragma unroll
      for (int f = 0; f < NF; ++f)
        if (j0 + f < n_fil) o[j0 + f] = v[f];
    }
  }
}

template <int NF, bool STREAM>
__global__ __launch_bounds__(256) void f3d_inf_kernel(const float4* __restrict__ fa,
                                                      const float4* __restrict__ fb, int n_fil,
                                                      const float4* __restrict__ mes,
                                                      const float4* __restrict__ dir, int n_mes,
                                                      int rows, float* __restrict__ out) {
  __shared__ float4 s_x[INF_ROWS + 1], s_e[INF_ROWS + 1];
  const int tid = threadIdx.x;
  const int j0 = (blockIdx.x * 256 + tid) * NF;
  const int i0 = blockIdx.y * rows;
  const int nr = min(rows, n_mes - i0);
  if (tid <= nr) {
    const bool in = tid < nr;
    s_x[tid] = in ? mes[i0 + tid] : make_float4(0.f, 0.f, 0.f, 0.f);
    s_e[tid] = in ? dir[i0 + tid] : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  InfCols<NF> c;
  bool linked = true;
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int j = min(j0 + f, n_fil - 1);
    const float4 fa4 = fa[j], fb4 = fb[j];
    c.a[f] = make_float3(fa4.x, fa4.y, fa4.z);
    c.b[f] = make_float3(fb4.x, fb4.y, fb4.z);
    c.r0[f] = make_float3(fb4.x - fa4.x, fb4.y - fa4.y, fb4.z - fa4.z);
    c.L2[f] = dot3(c.r0[f], c.r0[f]);
    // (a strength that is not finite and a filament of no length give elements of 0,
    // in either form: c = 0 times a factor that overflows would be NaN)
    const float g = fa4.w * (float)(1.0 / (4.0 * M_PI));
    const bool none = c.r0[f].x == 0.f && c.r0[f].y == 0.f && c.r0[f].z == 0.f;
    c.g[f] = __builtin_isfinite(g) && !none ? 2.f * g : 0.f;
    if (f > 0)
      linked = linked && __float_as_uint(c.a[f].x) == __float_as_uint(c.b[f - 1].x) &&
               __float_as_uint(c.a[f].y) == __float_as_uint(c.b[f - 1].y) &&
               __float_as_uint(c.a[f].z) == __float_as_uint(c.b[f - 1].z);
  }
  const bool whole = ((int)blockIdx.x + 1) * (256 * NF) <= n_fil;
  __syncthreads();
  // a wave beyond the last column has nothing to do (no barrier below); us, its rows
  // computed -> not: 1 column of 4 10^6 rows 1560 -> 444, 128 x 500000 210 -> 77
  if ((int)(blockIdx.x * 256 + (tid & ~63)) * NF >= n_fil) return;
  float* o = out + (size_t)i0 * (size_t)n_fil;
  // one answer for the whole wave, so the row loop branches uniformly
  const bool share = __all(linked);
  if (whole) {
    if (share) inf_rows<NF, true, true, STREAM>(c, s_x, s_e, nr, j0, n_fil, o);
    else inf_rows<NF, false, true, STREAM>(c, s_x, s_e, nr, j0, n_fil, o);
  } else {
    if (share) inf_rows<NF, true, false, STREAM>(c, s_x, s_e, nr, j0, n_fil, o);
    else inf_rows<NF, false, false, STREAM>(c, s_x, s_e, nr, j0, n_fil, o);
  }
}

}  // namespace

hipError_t launch_f3d_inf(const float4* fa, const float4* fb, int n_fil, const float4* mes,
                          const float4* dir, int n_mes, float* out, hipStream_t s) {
  if (n_fil <= 0 || n_mes <= 0) return hipSuccess;
  if (!fa || !fb || !mes || !dir || !out) return hipErrorInvalidValue;
  // A matrix that outgrows the last-level cache, with rows of whole 128-byte
  // lines, is written past the caches in 16-byte stores: 16384 x 16384 237 us
  // with two columns per lane and cached stores, 217 us so.  Where it fits
  // (3280 x 1149, 15 MB) streaming takes 21 us against 10, and where lines are
  // shared between rows (127 x 130 columns) 345 us against 260.
  const bool stream = n_fil % 32 == 0 && ((uintptr_t)out & 127) == 0 &&
                      (size_t)n_fil * n_mes >= (size_t)INF_STREAM_ELEMENTS;
  const int per = 256 * (stream ? 4 : 2);
  // rows per workgroup: eight workgroups per CU at least (3280 x 1149, us with
  // 2 / 4 / 8 / 16 per CU: 8.5 / 8.3 / 8.6 / 10.7; 923 x 18510: 25.6 / 25.9 /
  // 25.0 / 24.0; 1786 x 2069: 9.9 / 8.8 / 8.4 / 8.4)
  const int gx = (n_fil + per - 1) / per;
  int rows = 1;
  while (rows < INF_ROWS && (long long)gx * ((n_mes + 2 * rows - 1) / (2 * rows)) >= 2048) rows *= 2;
  const auto k = stream ? f3d_inf_kernel<4, true> : f3d_inf_kernel<2, false>;
  hipLaunchKernelGGL(k, dim3(gx, (n_mes + rows - 1) / rows), dim3(256), 0, s, fa, fb, n_fil, mes,
                     dir, n_mes, rows, out);
  return hipGetLastError();
}

hipError_t launch_f3d(const F3DJob& j, const LaunchCfg& c, hipStream_t s) {
  if (j.n_tgt <= 0) return hipSuccess;
  if (j.n_fil < 0 || c.wg != 256) return hipErrorInvalidValue;
  if ((j.mask & OUT_DVORT) && j.tgt_a == nullptr) return hipErrorInvalidValue;
  // every output the mask selects must exist, and the inputs it reads
  if (((j.mask & OUT_VEL) && !j.out_vel) || ((j.mask & OUT_DVORT) && !j.out_dvort) || !j.tgt_pv ||
      (j.n_fil > 0 && (!j.fa || !j.fb)))
    return hipErrorInvalidValue;
  F3Fn k = f3_pick(j.mask, j.acc, c.T, c.q);
  if (!k) return hipErrorInvalidValue;
  F3DKParams p{};
  p.fa = j.fa;
  p.fb = j.fb;
  p.tgt_pv = j.tgt_pv;
  p.tgt_a = j.tgt_a;
  p.out_vel = j.out_vel;
  p.out_dvort = j.out_dvort;
  p.partial = j.partial;
  p.tgt_perm = j.tgt_perm;
  p.n_fil = j.n_fil;
  p.n_tgt = j.n_tgt;
  int n_split = c.n_split, split_len = c.split_len;
  if (n_split <= 1 || j.n_fil == 0) {
    n_split = 1;
    split_len = j.n_fil > 0 ? j.n_fil : 1;
  } else {
    if (split_len <= 0 || split_len % (c.wg / c.q) != 0) return hipErrorInvalidValue;
    if ((long long)split_len * n_split < j.n_fil || j.partial == nullptr) return hipErrorInvalidValue;
  }
  p.n_split = n_split;
  p.split_len = split_len;
  const int per = c.wg * c.T / c.q;
  hipLaunchKernelGGL(k, dim3((j.n_tgt + per - 1) / per, n_split), dim3(c.wg), 0, s, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || n_split == 1) return e;
  const int rows = reduce_rows(j.n_tgt), sums = 256 / rows;
  hipLaunchKernelGGL(rows == 4 ? f3_reduce<4>(j.mask) : f3_reduce<1>(j.mask),
                     dim3((j.n_tgt + sums - 1) / sums), dim3(256), 0, s, p);
  return hipGetLastError();
}

}  // namespace cvtx
