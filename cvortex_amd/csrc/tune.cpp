// tune.cpp -- launch-shape cache and autotuner.
//
// The autotuner times candidate launch shapes (targets per lane T, number of
// source partitions) for a caller's device-resident problem with HIP events
// and records the fastest in a cache keyed by
//   (kind, regularisation, outputs, accumulation, log2 n_src, log2 n_tgt).
// choose_cfg() consults the cache before falling back to default_cfg().
// The cache can be saved to and loaded from a small text file, one entry
// per line: "kind reg mask acc bucket_src bucket_tgt T n_split ms wg" (kind 3:
// a multi-cloud batch, keyed by its pair count and cloud count; n_split is
// then the resident workgroups per CU), and a last column 4 for the variant
// with 64 targets per workgroup (LaunchCfg::q).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include <cvortex_hip.h>

#include "api_common.hpp"
#include "runtime.hpp"
#include "tune.hpp"

namespace cvtx {

namespace {

using Key = std::tuple<int, int, int, int, int, int>;
// n_split is the number of source partitions, or for KIND_BATCH the
// resident workgroups per CU; wg the workgroup size.
struct Entry {
  int T;
  int n_split;
  float ms;
  int wg = 256;
  int q = 1;
};

std::map<Key, Entry>& cache() {
  static std::map<Key, Entry> c;
  return c;
}

}  // namespace

LaunchCfg launch_shape(int T, int n_split, int n_src) {
  LaunchCfg c;
  c.T = T;
  c.wg = 256;
  const long tiles = ((long)n_src + 255) / 256;
  if (n_split <= 1 || tiles <= 1) return c;
  c.split_len = (int)((tiles + n_split - 1) / n_split * 256);
  c.n_split = (int)((n_src + c.split_len - 1) / c.split_len);
  if (c.n_split <= 1) {
    c.n_split = 1;
    c.split_len = 0;
  }
  return c;
}

int size_bucket(int n) {
  int b = 0;
  while (n > 1) {
    n >>= 1;
    ++b;
  }
  return b;
}

// Whether a launch of this kind orders its targets spatially (api.cpp), which
// changes the cost of its launch shapes: part of the cache key, folded into
// the kind field (kind + 16).
int ordered_kind(int kind, int reg, int n_src, int n_tgt) {
  const Runtime& rt = runtime();
  const bool ordered =
      rt.order_targets && ((kind == KIND_P3D && p3d_wants_order(reg, n_src, n_tgt)) ||
                           (kind == KIND_F3D && f3d_wants_order(n_src, n_tgt)));
  return ordered ? kind + 16 : kind;
}

namespace {

// Small problems: 64 targets per workgroup, shared by its four waves, each of
// which takes a quarter of every source tile.  Bound by the waves in flight
// and by the length of the longest one: with 256 targets per workgroup a
// problem of a few tiles leaves most SIMDs idle, and one a little larger ends
// in a wave of workgroups that is nearly empty.  The price is one staging of
// a tile and its barriers per 64 pairs of a lane instead of 256, so the rule
// ends at 24 target-block tiles of 256 x 256 per CU.  256 targets per
// workgroup -> 64, us: Winckelmans vel + dvort of 2000 particles 32.4 -> 13.7,
// 6000 60.6 -> 48.2, 9000 99.7 -> 82.3, 15000 215 -> 191, 18000 289 -> 275;
// velocity of 1000 on the host's arrays 43.7 -> 34.8 a call; 2D Gaussian with
// the viscous term, 3000 51.0 -> 20.5, 9000 103 -> 65, 18000 229 -> 196;
// 3600 filaments on 20000 targets 242 -> 167, 10000 on 30000 467 -> 418 (on
// 100000, 60 tiles per CU, 1054 -> 1190: a block of 64 targets has a smaller
// box than one of 256, but its tiles are staged four times as often).
// 2D velocities by the singular or the planetary kernel end at 16, where two
// targets per lane win (planetary 15000 62.6 -> 56.2, 17000 68.4 -> 71.9).
// Few sources on many targets don't go here either: where blocks of 256 targets
// fill the chip, four times as many workgroups, each with its own staging (and
// table), cost more than they share out.  The line lies at 10 sources per block of
// targets and CU (40 for the lighter 2D and the filament pairs), 32 at least, and 12
// blocks per CU.  256 targets per workgroup -> 64, us: 1 source on 2^20 targets,
// velocity 6.2 -> 12.0, 2D Gaussian 9.5 -> 45, filament 21 -> 71; on 65536 targets 1
// filament 4.9 -> 8.2, 64 3D Gaussian 17.2 -> 10.0; on 131072 64 filaments 16.5 -> 18.8,
// 64 3D Gaussian 18.1 -> 15.2; on 262144 64 2D Gaussian 12.3 -> 18.1, 250 3D Gaussian
// 101 -> 72, 500 velocity 82 -> 60, 500 filaments 377 -> 322; on 600000 500 velocity
// 176 -> 130, 500 filaments 587 -> 477; on 2^20 250 3D singular
// 186 -> 198, 512 3D Gaussian 547 -> 596.
bool narrow(int kind, int reg, int mask, int n_src, int n_tgt, int cus) {
  const long long nb = ((long long)n_tgt + 255) / 256, tiles = ((long long)n_src + 255) / 256;
  if (nb >= 12LL * cus || n_src < 32 || (long long)n_src * cus < (kind == KIND_P3D ? 10 : 40) * nb)
    return false;
  const bool light = kind == KIND_P2D && !(mask & OUT_VISC) &&
                     (reg == REG_PLANETARY || reg == REG_SINGULAR);
  return n_tgt > 0 && tiles > 0 && nb * tiles < (light ? 16LL : 24LL) * cus;
}

// Partitions for 16 workgroups per CU of two tiles or more each, and for 4 per
// CU down to one tile: 8192 particles (velocity, us) 40.9 with two tiles each,
// 44.2 with four; 7000 (vel + dvort) 54.2 with three, 57.0 with two.
// Below 2 workgroups per CU a tile is split too, into quarters, so that each
// wave's run of pairs, a chain it walks alone on its SIMD, is as short as 16:
// Gaussian vel + dvort + visc of 500 particles 20.9 -> 10.4 us, 2000 21.4 ->
// 15.4; Winckelmans vel + dvort of 1000 11.5 -> 8.4; 2D Gaussian with the
// viscous term 1000 17.1 -> 8.9, 3D velocity of 1000 8.8 -> 7.0.  At most 64
// partitions (20000 sources on 50 targets: 15.7 us with 79, 27.5 with 313, whose
// sums are one group's reduction), and where one tile holds all sources, only
// for pairs that cost more than the second launch: 256 particles by the Gaussian
// 18.2 -> 10.4 and Winckelmans vel + dvort 8.5 -> 7.0, but velocity 5.7 -> 6.8
// and 100 particles 5.2 -> 6.8.  Without quarters a few targets' many partitions pay:
// 2^20 sources on 64 targets, us, against 256 targets per workgroup: velocity 161 ->
// 89, with stretching and exchange 541 -> 256, Gaussian 434 -> 203, filaments 593 -> 243.
LaunchCfg narrow_cfg(int kind, int reg, int mask, int n_src, int n_tgt, int cus) {
  const long long groups = ((long long)n_tgt + 63) / 64, tiles = ((long long)n_src + 255) / 256;
  auto fill = [&](long long per_cu) { return std::max(1LL, (per_cu * cus + groups - 1) / groups); };
  const long long k = std::min(std::max(fill(4), std::min(fill(16), tiles / 2)), tiles);
  LaunchCfg c = launch_shape(1, (int)k, n_src);
  c.q = 4;
  const bool heavy = reg == REG_GAUSSIAN || (kind == KIND_P3D && mask != OUT_VEL);
  if (groups * tiles < 2LL * cus && (tiles > 1 || (heavy && n_src > 128))) {
    const long long quarters = ((long long)n_src + 63) / 64;
    const long long kq = std::min({quarters, fill(2), 64LL});
    if (kq > k) {
      c.split_len = (int)((quarters + kq - 1) / kq * 64);
      c.n_split = (n_src + c.split_len - 1) / c.split_len;
    }
  }
  return c;
}

// Each partition's sums are read by one lane after another in the reduction: 2^20
// 2D sources on 64 targets, us, with 256 / 512 / 1024 / 2048 partitions 106 / 92 / 99
// / 120 (planetary).
constexpr long long MOST_PARTITIONS = 512;

// 2D problems that are not narrow.  One target per lane is bound by the LDS: a
// source's 16 bytes take its port 8 cycles per wave, 32 for the four SIMDs of a
// CU, as long as 16 issue slots, where a far pair needs 11.  So two targets per
// lane as soon as there is enough work, in tiles of 256 x 256 per CU, and four
// from 1024 on for the velocity without the Gaussian's ranges (their wider blocks
// have fewer far tiles), with partitions of two tiles or more for 64 workgroups
// per CU, or of one for 32.  One target -> two, us: planetary 21000 particles
// 125 -> 98, 100003 2349 -> 1600 (four: 1588), 200000 9209 -> 6108 with four;
// Gaussian velocity 50000 697 -> 618 (30000: 292 with one, 302 with two),
// exchange 100003 3063 -> 2925; Winckelmans with the exchange 35000 817 -> 733,
// 200000 25185 -> 22259; its velocity at 262144 14976 -> 14846 with four, 15537
// with two.  More partitions alone:
// Gaussian velocity and exchange 21000 particles 307 -> 208, singular 9000 34.3
// -> 29.7.
// Two targets per lane at least where that leaves 4 workgroups per CU, one for up to
// 2048 targets; tiles halved among partitions below 2 workgroups per CU only, whose
// partial sums cost more than an uneven end where targets are many; and at most
// MOST_PARTITIONS.  us, without these lines -> with them: 1 source on 2^20 targets,
// Gaussian with the exchange 14.5 -> 10.4, 250, Winckelmans with it 166 -> 156, 512,
// planetary 136 -> 123; 2^20 sources on 64 targets, planetary 227 -> 92, on 1000 344
// -> 264.
LaunchCfg p2d_cfg(int reg, int mask, int n_src, int n_tgt, int cus) {
  const long long tiles = ((long long)n_src + 255) / 256;
  auto blocks = [&](int T) { return ((long long)n_tgt + 256LL * T - 1) / (256LL * T); };
  const bool visc = (mask & OUT_VISC) != 0;
  const long long work = blocks(1) * tiles / cus;
  int T = 1;
  if (reg == REG_GAUSSIAN) T = work >= 100 ? 2 : 1;
  else if (visc) T = work >= 24 ? 2 : 1;
  else if (reg == REG_PLANETARY || reg == REG_SINGULAR) T = work >= 1024 ? 4 : (work >= 16 ? 2 : 1);
  else T = work >= 1024 ? 4 : 1;
  if (blocks(2) >= 4LL * cus) T = std::max(T, 2);
  if (blocks(1) <= 8) T = 1;
  const long long nb = blocks(T);
  long long k = std::min((64LL * cus + nb - 1) / std::max(1LL, nb), std::max(1LL, tiles / 2));
  if (nb * k < 32LL * cus && nb < 2LL * cus)
    k = std::min((32LL * cus + nb - 1) / std::max(1LL, nb), tiles);
  return launch_shape(T, (int)std::max(1LL, std::min(k, MOST_PARTITIONS)), n_src);
}

}  // namespace

LaunchCfg choose_cfg(int kind, int reg, int mask, int acc, int n_src, int n_tgt, int n_cu) {
  auto it = cache().find(Key{ordered_kind(kind, reg, n_src, n_tgt), reg, mask, acc,
                             size_bucket(n_src), size_bucket(n_tgt)});
  const int cus = n_cu > 0 ? n_cu : 256;
  if (it != cache().end())
    return it->second.q == 4 && n_tgt > 0 ? narrow_cfg(kind, reg, mask, n_src, n_tgt, cus)
                                          : launch_shape(it->second.T, it->second.n_split, n_src);
  // Spatially ordered targets (Gaussian P3D, compensated sums).  One target
  // per lane: a 64-target wave of Morton-ordered targets is more compact
  // than a 128-target one, so fewer of its source rounds take the FP64
  // near-field branch.  Source partitions: the near-field work is
  // concentrated in the workgroups whose targets sit in dense regions, and
  // partitioning spreads each of them over several workgroups instead of
  // leaving them as the launch's tail.  Enough partitions for about 64
  // workgroups per CU, and at least one per 65536 sources, but no more than
  // about 256 workgroups per CU.  Measured on the ring (vel+dvort, ms; one
  // partition -> this rule, on different machines):
  //   2^14: 0.29 -> 0.26 (64 partitions),  2^16: 3.73 -> 2.85 (64),
  //   2^18: 58.0 -> 42.4 (16; 32 and 64 the same),
  //   2^20: 710.6 -> 665.5 (16; 4 partitions: 673.6, 32: 665.3),
  //   2^22: 13742 -> 10564 (4; 1 partition on that machine: 10703).
  // vel alone and vel+dvort+visc at 2^20 also gain 1.2-1.4 % from 4 to 16.
  // The plain FP32 kernel has no FP64 branch and keeps the general shape
  // (two targets per lane: 678 ms against 861 ms with one at 2^20).
  if (kind == KIND_P3D && acc == ACC_COMP && p3d_wants_order(reg, n_src, n_tgt)) {
    // The velocity alone has no FP64 near sums, so the near branch costs
    // little and four targets per lane share each source's LDS reads: four
    // targets per lane and partitions for about 256 workgroups per CU (ring
    // 2^20 vel: 475.7 ms with the rule below, 419.6 ms with this).
    const int T = mask == OUT_VEL ? 4 : 1;
    const long long blocks = ((long long)n_tgt + 256LL * T - 1) / (256LL * T);
    const long long few = (64LL * cus + blocks - 1) / blocks;
    const long long per = ((long long)n_src + 65535) / 65536;
    const long long many = (256LL * cus + blocks - 1) / blocks;
    long long k = T == 4 ? many : std::min(std::max(few, per), many);
    // partitions of one tile spend much of a workgroup on its prologue and
    // epilogue: two tiles each while that still leaves 32 workgroups per CU
    // (ring 32768: 128 partitions 0.85 ms, 64 partitions 0.77 ms)
    const long long tiles = ((long long)n_src + 255) / 256;
    if (k > tiles / 2 && blocks * (tiles / 2) >= 32LL * cus) k = tiles / 2;
    return launch_shape(T, (int)std::min<long long>(k, 1 << 20), n_src);
  }
  if (narrow(kind, reg, mask, n_src, n_tgt, cus)) return narrow_cfg(kind, reg, mask, n_src, n_tgt, cus);
  if (kind == KIND_P2D) return p2d_cfg(reg, mask, n_src, n_tgt, cus);
  // Filaments: a block's tiles near it take several times the far ones' time, so
  // partitions go down to one tile for 64 workgroups per CU, which spread them
  // (a kernel of one or two tiles' worth of filaments gains nothing from it).
  // Partitions of six, three and two tiles -> this, us: 14000 filaments on 40000
  // targets velocity 509 -> 418, both 737 -> 622, 4293 on 156344 558 -> 491, 801 ->
  // 759, 11475 on 312258 2186 -> 2087, 16384 on 2^20 9368 -> 9195; but 459 on 394673
  // 341 -> 351.
  if (kind == KIND_F3D && n_src >= 12 * 256) {
    const long long nb = ((long long)n_tgt + 255) / 256, tiles = ((long long)n_src + 255) / 256;
    return launch_shape(1, (int)std::min(tiles, (64LL * cus + nb - 1) / std::max(1LL, nb)), n_src);
  }
  LaunchCfg c = default_cfg(n_src, n_tgt, n_cu);
  const bool many_blocks = (long long)(n_tgt + 255) / 256 >= 4LL * cus;
  // Filaments: one target per lane.  It fits in fewer VGPRs (more waves per
  // SIMD to pair instructions for dual issue) and, with ordered targets,
  // makes a block's box smaller, so more filament tiles take the far-tile
  // loop.  16384 filaments x 2^20 targets, 4 partitions (ms, two targets
  // per lane -> one): vel 13.7 -> 13.1, dvort 21.1 -> 19.2, fused 21.4 ->
  // 20.4.
  if (kind == KIND_F3D && c.T > 1 && many_blocks) c = partitioned_cfg(1, n_src, n_tgt, n_cu);
  return c;
}

void record_cfg(int kind, int reg, int mask, int acc, int n_src, int n_tgt, int T, int n_split) {
  cache()[Key{ordered_kind(kind, reg, n_src, n_tgt), reg, mask, acc, size_bucket(n_src),
              size_bucket(n_tgt)}] = Entry{T, n_split, 0.f};
}

namespace {
int bucket64(long long n) {
  int b = 0;
  while (n > 1) {
    n >>= 1;
    ++b;
  }
  return b;
}
Key batch_key(const BatchSignature& g) {
  return Key{KIND_BATCH, g.reg, g.mask, g.acc, bucket64(g.pairs), size_bucket(g.n_clouds)};
}
}  // namespace

bool batch_shape_lookup(const BatchSignature& g, BatchShape* out) {
  auto it = cache().find(batch_key(g));
  if (it == cache().end()) return false;
  *out = BatchShape{it->second.T, it->second.wg, it->second.n_split, it->second.ms, it->second.q};
  return true;
}

void batch_shape_record(const BatchSignature& g, const BatchShape& s) {
  cache()[batch_key(g)] = Entry{s.T, s.wpc, s.ms, s.wg, s.q};
}

}  // namespace cvtx

using namespace cvtx;

namespace {

// Time `reps` launches of one shape; returns ms per launch or -1 on error.
template <class Launch>
float time_shape(hipStream_t s, int reps, Launch launch) {
  hipEvent_t a, b;
  if (hipEventCreate(&a) != hipSuccess) return -1.f;
  if (hipEventCreate(&b) != hipSuccess) {
    (void)hipEventDestroy(a);
    return -1.f;
  }
  float ms = -1.f;
  if (launch() == hipSuccess && hipEventRecord(a, s) == hipSuccess) {
    bool ok = true;
    for (int r = 0; r < reps && ok; ++r) ok = launch() == hipSuccess;
    if (ok && hipEventRecord(b, s) == hipSuccess && hipEventSynchronize(b) == hipSuccess) {
      float t = 0.f;
      if (hipEventElapsedTime(&t, a, b) == hipSuccess) ms = t / (float)reps;
    }
  }
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  return ms;
}

std::vector<LaunchCfg> candidates(int n_src, int n_tgt, int n_cu) {
  std::vector<LaunchCfg> out;
  const long tiles = ((long)n_src + 255) / 256;
  for (int T : {1, 2, 4}) {
    const long blocks = ((long)n_tgt + 256L * T - 1) / (256L * T);
    if (T > 1 && blocks < 8) continue;
    for (int k = 1; k <= 256; k *= 2) {
      if (k > 1 && k > tiles) break;
      if (blocks * k > 256L * (n_cu > 0 ? n_cu : 256)) break;
      out.push_back(launch_shape(T, k, n_src));
    }
  }
  return out;
}

}  // namespace

extern "C" {

// Autotune the launch shape of a device-resident P3D problem; the winner is
// recorded in the shape cache for the problem's size bucket.  Returns 0 and
// the fastest shape that two numbers name (the winner, unless that shares its
// targets among the waves of a workgroup), or -1.
int cvtx_hip_autotune_p3d(const cvtx_hip_p3d_problem* p, int reps, int* best_T, int* best_split,
                          float* best_ms) {
  Runtime& rt = runtime();
  std::lock_guard<std::recursive_mutex> lk(rt.mu);
  if (!p || reps < 1) return -1;
  Device* d = active_device(rt);
  if (!d) return -1;
  StreamUse use(*d, d->stream);
  P3DJob j;
  j.src_pv = (const float4*)p->src_pv;
  j.src_a = (const float4*)p->src_a;
  j.n_src = p->n_src;
  j.tgt_pv = (const float4*)p->tgt_pv;
  j.tgt_a = (const float4*)p->tgt_a;
  j.n_tgt = p->n_tgt;
  j.out_vel = p->vel;
  j.out_dvort = p->dvort;
  j.out_visc = p->visc;
  j.reg = p->regularisation;
  j.mask = (p->vel ? OUT_VEL : 0) | (p->dvort ? OUT_DVORT : 0) | (p->visc ? OUT_VISC : 0);
  j.acc = p->accumulate;
  j.sigma = p->sigma;
  j.nu = p->nu;
  j.gtab = d->gtab;
  if (!p3d_supported(j.reg, j.mask) || j.n_tgt <= 0 || j.n_src < 0) return -1;
  // time the shapes on the target order the real calls will use
  if (rt.order_targets && p3d_wants_order(j.reg, j.n_src, j.n_tgt)) {
    j.tgt_perm = order_points(rt, *d, j.tgt_pv, j.n_tgt, SLOT_PERM, d->stream);
    if (!j.tgt_perm) return -1;
  }
  float best = -1.f, named_best = -1.f;
  LaunchCfg win, named;  // the fastest, and the fastest that (T, n_split) names
  std::vector<LaunchCfg> shapes = candidates(j.n_src, j.n_tgt, d->n_cu);
  if (!j.tgt_perm && narrow(KIND_P3D, j.reg, j.mask, j.n_src, j.n_tgt, d->n_cu))
    shapes.push_back(narrow_cfg(KIND_P3D, j.reg, j.mask, j.n_src, j.n_tgt, d->n_cu));
  for (const LaunchCfg& c : shapes) {
    P3DJob jj = j;
    const size_t wb = p3d_workspace_bytes(jj, c);
    if (wb) {
      jj.partial = (double*)device_buffer(rt, *d, SLOT_WORK, wb);
      if (!jj.partial) return -1;
    }
    const float ms = time_shape(d->stream, reps, [&]() { return launch_p3d(jj, c, d->stream); });
    if (ms > 0.f && (best < 0.f || ms < best)) {
      best = ms;
      win = c;
    }
    if (ms > 0.f && c.q == 1 && (named_best < 0.f || ms < named_best)) {
      named_best = ms;
      named = c;
    }
  }
  if (named_best < 0.f) return -1;
  cache()[Key{ordered_kind(KIND_P3D, j.reg, j.n_src, j.n_tgt), j.reg, j.mask, j.acc,
              size_bucket(j.n_src), size_bucket(j.n_tgt)}] = Entry{win.T, win.n_split, best, 256, win.q};
  if (best_T) *best_T = named.T;
  if (best_split) *best_split = named.n_split;
  if (best_ms) *best_ms = named_best;
  return 0;
}

int cvtx_hip_tune_save(const char* path) {
  FILE* f = std::fopen(path, "w");
  if (!f) return -1;
  for (auto& kv : cache()) {
    const Key& k = kv.first;
    std::fprintf(f, "%d %d %d %d %d %d %d %d %.6f %d%s\n", std::get<0>(k), std::get<1>(k),
                 std::get<2>(k), std::get<3>(k), std::get<4>(k), std::get<5>(k), kv.second.T,
                 kv.second.n_split, kv.second.ms, kv.second.wg, kv.second.q == 4 ? " 4" : "");
  }
  std::fclose(f);
  return 0;
}

int cvtx_hip_tune_load(const char* path) {
  FILE* f = std::fopen(path, "r");
  if (!f) return -1;
  int kind, reg, mask, acc, bs, bt, T, ns, wg, q;
  float ms;
  int n = 0;
  char line[256];
  // one entry per line; the last two columns may be absent (256, 1)
  while (std::fgets(line, sizeof(line), f)) {
    wg = 256;
    q = 1;
    const int got = std::sscanf(line, "%d %d %d %d %d %d %d %d %f %d %d", &kind, &reg, &mask, &acc,
                                &bs, &bt, &T, &ns, &ms, &wg, &q);
    if (got >= 9 && (T == 1 || T == 2 || T == 4) && ns >= 1 && (wg == 128 || wg == 256)) {
      if (q != 4 || T != 1 || wg != 256) q = 1;
      cache()[Key{kind, reg, mask, acc, bs, bt}] = Entry{T, ns, ms, wg, q};
      ++n;
    }
  }
  std::fclose(f);
  return n;
}

void cvtx_hip_tune_clear(void) { cache().clear(); }

int cvtx_hip_gaussian_table(float* out, int capacity) {
  if (out == nullptr || capacity < 8 * GTAB_N) return -1;
  double tab[8 * GTAB_N];
  build_gaussian_table(tab);
  for (int i = 0; i < 8 * GTAB_N; ++i) out[i] = (float)tab[i];
  return 8 * GTAB_N;
}

}  // extern "C"
