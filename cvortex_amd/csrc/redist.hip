// redist.hip -- redistribution of vortex particles onto a regular grid
// (remeshing): cvtx_P3D_redistribute_on_grid, cvtx_P2D_redistribute_on_grid.
//
// Semantics of the reference CPU path (src/P3D.cpp:509-665,
// src/P2D.cpp:283-436, src/RedistFunc.cpp:36-96,
// src/redistribution_helper_funcs.cpp:33-80):
//   1. grid origin from the particles' minimum and mean (one cell layout for
//      the whole call), node key = round((x - origin) / h) per axis;
//   2. every particle gives strength alpha * f(U) f(W) (f(V)) to the
//      (2R+1)^dim nodes around its nearest node, R = round(radius), with
//      U = |x - x_node| / h per axis; exactly-zero contributions make no node;
//   3. the nodes' summed strengths become particles of volume h^dim, in the
//      ascending Morton order of the node keys (octant index x + 2y + 4z,
//      quadrant x + 2y), the order the reference's tree emits them in;
//   4. particles weaker than negligible x mean strength are removed and their
//      strength shared equally by the rest;
//   5. with an output array and more particles than it holds, a histogram
//      search picks a strength threshold for about max_output survivors, and
//      of the first max_output particles those above it are kept, again
//      sharing the removed strength.
// The weights use the reference's FP32 operations in its order (no fused
// multiply-adds), so the set of nodes, their positions and the weights of
// every contribution are the reference's; node sums are formed in FP64 in
// particle order (the reference sums in FP32).
//
// GPU structure: particles are sorted by grid cell and the nodes summed block
// by block of the grid (by_blocks); grids whose keys are too long for its
// bitmaps, or particles too scattered, take the general form (by_entries): one
// thread per (particle, neighbour) writes a (Morton key, contribution) entry,
// rocPRIM's stable radix sort groups the entries by node and a wave per node
// sums its run.  Removal and truncation are order-preserving compactions
// (rocPRIM select) with the removed strength reduced in FP64; the threshold
// and the shared strength stay on the device.  Scalar control (grid origin,
// counts, the histogram search's loop) runs on the host between kernels.
#include <hip/hip_runtime.h>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/device/device_select.hpp>
#include <rocprim/iterator/counting_iterator.hpp>

#include <algorithm>
#include <cmath>
#include <vector>

#include "kernels.hpp"
#include "runtime.hpp"

namespace cvtx {

namespace {

constexpr int kPartBlocks = 512;  // fixed grid of the reductions (deterministic)

// Redistribution functions, reference src/RedistFunc.cpp:36-96, in FP32
// with the reference's operation order.
template <int RID>
__device__ __forceinline__ float rd_f(float U) {
  if constexpr (RID == 0) {  // lambda0
    return U < 0.5f ? 1.f : 0.f;
  } else if constexpr (RID == 1) {  // lambda1
    return U <= 1.f ? rn_sub(1.f, U) : 0.f;
  } else if constexpr (RID == 2) {  // lambda2
    return U < 0.5f ? rn_sub(1.f, rn_mul(U, U))
                    : (U < 1.5f ? rn_mul(rn_mul(0.5f, rn_sub(1.f, U)), rn_sub(2.f, U))
                                : 0.f);
  } else if constexpr (RID == 3) {  // lambda3
    return U < 1.f ? rn_mul(rn_mul(0.5f, rn_sub(1.f, rn_mul(U, U))), rn_sub(2.f, U))
                   : (U < 2.f ? rn_mul(rn_mul(rn_mul(1.f / 6.f, rn_sub(1.f, U)),
                                                    rn_sub(2.f, U)),
                                          rn_sub(3.f, U))
                              : 0.f);
  } else {  // m4'
    return U < 1.f ? rn_add(rn_sub(1.f, rn_mul(rn_mul(2.5f, U), U)),
                               rn_mul(rn_mul(rn_mul(1.5f, U), U), U))
                   : (U < 2.f ? rn_mul(rn_mul(rn_mul(0.5f, rn_sub(1.f, U)),
                                                    rn_sub(2.f, U)),
                                          rn_sub(2.f, U))
                              : 0.f);
  }
}

__host__ __device__ __forceinline__ unsigned long long spread3(unsigned v) {
  unsigned long long x = v & 0x1fffffull;
  x = (x | (x << 32)) & 0x1f00000000ffffull;
  x = (x | (x << 16)) & 0x1f0000ff0000ffull;
  x = (x | (x << 8)) & 0x100f00f00f00f00full;
  x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
  x = (x | (x << 2)) & 0x1249249249249249ull;
  return x;
}
__host__ __device__ __forceinline__ unsigned compact3(unsigned long long x) {
  x &= 0x1249249249249249ull;
  x = (x ^ (x >> 2)) & 0x10c30c30c30c30c3ull;
  x = (x ^ (x >> 4)) & 0x100f00f00f00f00full;
  x = (x ^ (x >> 8)) & 0x1f0000ff0000ffull;
  x = (x ^ (x >> 16)) & 0x1f00000000ffffull;
  x = (x ^ (x >> 32)) & 0x1fffffull;
  return (unsigned)x;
}
__host__ __device__ __forceinline__ unsigned long long spread2(unsigned v) {
  unsigned long long x = v;
  x = (x | (x << 16)) & 0x0000ffff0000ffffull;
  x = (x | (x << 8)) & 0x00ff00ff00ff00ffull;
  x = (x | (x << 4)) & 0x0f0f0f0f0f0f0f0full;
  x = (x | (x << 2)) & 0x3333333333333333ull;
  x = (x | (x << 1)) & 0x5555555555555555ull;
  return x;
}
__host__ __device__ __forceinline__ unsigned compact2(unsigned long long x) {
  x &= 0x5555555555555555ull;
  x = (x ^ (x >> 1)) & 0x3333333333333333ull;
  x = (x ^ (x >> 2)) & 0x0f0f0f0f0f0f0f0full;
  x = (x ^ (x >> 4)) & 0x00ff00ff00ff00ffull;
  x = (x ^ (x >> 8)) & 0x0000ffff0000ffffull;
  x = (x ^ (x >> 16)) & 0x00000000ffffffffull;
  return (unsigned)x;
}

struct Grid {
  float mn[3];  // origin
  float h, rh;  // spacing and its reciprocal (FP32 as the reference)
  int R;        // neighbourhood half-width
};

// Per-block min (FP32) and sum (FP64) of each coordinate.
template <int DIM>
__global__ __launch_bounds__(256) void rd_bounds(const float4* __restrict__ pv, int n,
                                                 float* __restrict__ pmin,
                                                 float* __restrict__ pmax,
                                                 double* __restrict__ psum) {
  __shared__ float smin[DIM][256];
  __shared__ float smax[DIM][256];
  __shared__ double ssum[DIM][256];
  float m[DIM], M[DIM];
  double s[DIM];
  for (int c = 0; c < DIM; ++c) { m[c] = __builtin_inff(); M[c] = -__builtin_inff(); s[c] = 0.0; }
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const float4 p = pv[i];
    const float x[3] = {p.x, p.y, p.z};
    for (int c = 0; c < DIM; ++c) {
      m[c] = fminf(m[c], x[c]);
      M[c] = fmaxf(M[c], x[c]);
      s[c] += (double)x[c];
    }
  }
  for (int c = 0; c < DIM; ++c) {
    smin[c][threadIdx.x] = m[c];
    smax[c][threadIdx.x] = M[c];
    ssum[c][threadIdx.x] = s[c];
  }
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w)
      for (int c = 0; c < DIM; ++c) {
        smin[c][threadIdx.x] = fminf(smin[c][threadIdx.x], smin[c][threadIdx.x + w]);
        smax[c][threadIdx.x] = fmaxf(smax[c][threadIdx.x], smax[c][threadIdx.x + w]);
        ssum[c][threadIdx.x] += ssum[c][threadIdx.x + w];
      }
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int c = 0; c < DIM; ++c) {
      pmin[blockIdx.x * DIM + c] = smin[c][0];
      pmax[blockIdx.x * DIM + c] = smax[c][0];
      psum[blockIdx.x * DIM + c] = ssum[c][0];
    }
}

// Entry e = i * W^DIM + j: the contribution of particle i to its j-th
// neighbour node (a window of W = 2R + 1 nodes per axis around the nearest
// node).  3D: pv = {x, y, z, -}, a = {alpha, -}; 2D: pv = {x, y, alpha, -}.
// Returns false for an exactly-zero contribution (the reference makes no
// node for it).
template <int DIM, int RID>
__device__ __forceinline__ bool rd_entry(const float4* __restrict__ pv,
                                         const float4* __restrict__ a, int e, const Grid& g,
                                         unsigned long long& key, float4& v) {
  const int W = 2 * g.R + 1;
  const int WD = DIM == 3 ? W * W * W : W * W;
  const int i = e / WD;
  const int j = e - i * WD;
  const float4 p = pv[i];
  const float x[3] = {p.x, p.y, p.z};
  unsigned q[3];
  int off[3];
  if constexpr (DIM == 3) {
    off[0] = j / (W * W) - g.R;
    off[1] = (j / W) % W - g.R;
    off[2] = j % W - g.R;
  } else {
    off[0] = j / W - g.R;
    off[1] = j % W - g.R;
  }
  float frac = 1.f;
#pragma unroll
  for (int c = 0; c < DIM; ++c) {
    float k;
    if constexpr (DIM == 3) {  // reference UIntKey96.cpp: FP32 offset
      k = roundf(rn_mul(rn_sub(x[c], g.mn[c]), g.rh));
    } else {  // reference UIntKey64.cpp:79-96: the offset is formed in FP64
      k = roundf((float)(((double)x[c] - (double)g.mn[c]) * (double)g.rh));
    }
    q[c] = (unsigned)k + (unsigned)off[c];
    const float node = rn_add(g.mn[c], rn_mul(g.h, (float)q[c]));
    const float U = fabsf(rn_mul(rn_sub(x[c], node), g.rh));
    frac = c == 0 ? rd_f<RID>(U) : rn_mul(frac, rd_f<RID>(U));
  }
  if constexpr (DIM == 3) {
    const float4 al = a[i];
    v = make_float4(rn_mul(al.x, frac), rn_mul(al.y, frac), rn_mul(al.z, frac), 0.f);
    key = spread3(q[0]) | (spread3(q[1]) << 1) | (spread3(q[2]) << 2);
    return !(v.x == 0.f && v.y == 0.f && v.z == 0.f);
  } else {
    v = make_float4(rn_mul(p.z, frac), 0.f, 0.f, 0.f);
    key = spread2(q[0]) | (spread2(q[1]) << 1);
    return v.x != 0.f;
  }
}

// Chunked stable compaction (used for the nonzero entries and for the node
// starts): a first kernel counts the selected items of each chunk of kChunk
// = 16 rounds of 256, an inclusive scan of the counts gives each chunk's end
// offset, and a second kernel writes the chunk's items from its start
// offset in their original order, a wave ballot ranking them within a round.
constexpr int kChunk = 4096;

__device__ __forceinline__ int block_sum(int c, int* s_w) {
  for (int off = 32; off > 0; off >>= 1) c += __shfl_down(c, off, 64);
  if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = c;
  __syncthreads();
  return s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

// Within one round of a chunk: the output slot of this lane's item (if it is
// selected), given the round's first slot; advances `off` past the round.
__device__ __forceinline__ int round_slot(bool sel, int& off, int* s_w) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned long long m = __ballot(sel);
  const int rank = __popcll(m & ((1ull << lane) - 1ull));
  __syncthreads();  // s_w of the previous round has been read
  if (lane == 0) s_w[w] = __popcll(m);
  __syncthreads();
  int wo = 0;
  for (int q = 0; q < w; ++q) wo += s_w[q];
  const int slot = off + wo + rank;
  off += s_w[0] + s_w[1] + s_w[2] + s_w[3];
  return slot;
}

template <int DIM, int RID>
__global__ __launch_bounds__(256) void rd_contrib_count(const float4* __restrict__ pv,
                                                        const float4* __restrict__ a, long ne,
                                                        Grid g, int* __restrict__ counts) {
  __shared__ int s_w[4];
  const long base = (long)blockIdx.x * kChunk;
  int c = 0;
  for (int r = 0; r < kChunk / 256; ++r) {
    const long e = base + r * 256 + threadIdx.x;
    unsigned long long key;
    float4 v;
    if (e < ne && rd_entry<DIM, RID>(pv, a, (int)e, g, key, v)) ++c;
  }
  c = block_sum(c, s_w);
  if (threadIdx.x == 0) counts[blockIdx.x] = c;
}

// The nonzero entries, compacted in entry order (ne < 2^31, checked on the
// host: 32-bit entry indices).
template <int DIM, int RID>
__global__ __launch_bounds__(256) void rd_contrib_write(const float4* __restrict__ pv,
                                                        const float4* __restrict__ a, long ne,
                                                        Grid g, const int* __restrict__ incl,
                                                        unsigned long long* __restrict__ keys,
                                                        float4* __restrict__ vals) {
  __shared__ int s_w[4];
  const long base = (long)blockIdx.x * kChunk;
  int off = blockIdx.x > 0 ? incl[blockIdx.x - 1] : 0;
  for (int r = 0; r < kChunk / 256; ++r) {
    const long e = base + r * 256 + threadIdx.x;
    unsigned long long key = 0;
    float4 v;
    const bool sel = e < ne && rd_entry<DIM, RID>(pv, a, (int)e, g, key, v);
    const int slot = round_slot(sel, off, s_w);
    if (sel) {
      keys[slot] = key;
      vals[slot] = v;
    }
  }
}

// Node starts: the heads of the runs of equal keys among the sorted nonzero
// entries, in increasing order, by the chunked compaction above.  Heads are
// sparse (one per node, a few per hundred entries), so no flag array is
// written.
__device__ __forceinline__ bool run_head(const unsigned long long* __restrict__ keys, long i,
                                         long n) {
  return i < n && (i == 0 || keys[i - 1] != keys[i]);
}

__global__ __launch_bounds__(256) void rd_head_counts(const unsigned long long* __restrict__ keys,
                                                      long n, int* __restrict__ counts) {
  __shared__ int s_w[4];
  const long base = (long)blockIdx.x * kChunk;
  int c = 0;
  for (int r = 0; r < kChunk / 256; ++r) c += run_head(keys, base + r * 256 + threadIdx.x, n);
  c = block_sum(c, s_w);
  if (threadIdx.x == 0) counts[blockIdx.x] = c;
}

__global__ __launch_bounds__(256) void rd_head_write(const unsigned long long* __restrict__ keys,
                                                     long n, const int* __restrict__ incl,
                                                     long* __restrict__ starts) {
  __shared__ int s_w[4];
  const long base = (long)blockIdx.x * kChunk;
  int off = blockIdx.x > 0 ? incl[blockIdx.x - 1] : 0;
  for (int r = 0; r < kChunk / 256; ++r) {
    const long i = base + r * 256 + threadIdx.x;
    const bool h = run_head(keys, i, n);
    const int slot = round_slot(h, off, s_w);
    if (h) starts[slot] = i;
  }
}

// Position, strength and |strength| of a node from its FP64 sum.
template <int DIM>
__device__ __forceinline__ void rd_node(unsigned long long key, double a0, double a1, double a2,
                                        const Grid& g, float4& pos, float4& w, float& str) {
  const float vol = DIM == 3 ? rn_mul(rn_mul(g.h, g.h), g.h) : rn_mul(g.h, g.h);
  if constexpr (DIM == 3) {
    pos = make_float4(rn_add(g.mn[0], rn_mul(g.h, (float)compact3(key))),
                      rn_add(g.mn[1], rn_mul(g.h, (float)compact3(key >> 1))),
                      rn_add(g.mn[2], rn_mul(g.h, (float)compact3(key >> 2))), vol);
  } else {
    pos = make_float4(rn_add(g.mn[0], rn_mul(g.h, (float)compact2(key))),
                      rn_add(g.mn[1], rn_mul(g.h, (float)compact2(key >> 1))), 0.f, vol);
  }
  w = make_float4((float)a0, (float)a1, (float)a2, 0.f);
  str = DIM == 3 ? __fsqrt_rn(rn_add(rn_add(rn_mul(w.x, w.x), rn_mul(w.y, w.y)), rn_mul(w.z, w.z)))
                 : fabsf(w.x);
}

// One wave per node: the wave reads the node's run of entries 64 at a time
// (coalesced) and reduces it in FP64 with a fixed shuffle tree, so the sum
// is the same on every call; the run ends at the first different key.
// pos = {x, y, z, volume} (2D: {x, y, -, area}); w = strength; str = |w|.
template <int DIM>
__global__ __launch_bounds__(256) void rd_nodes(const unsigned long long* __restrict__ keys,
                                                const float4* __restrict__ vals, long n_entries,
                                                const long* __restrict__ starts, int n_nodes,
                                                Grid g, float4* __restrict__ pos,
                                                float4* __restrict__ w, float* __restrict__ str) {
  const int lane = threadIdx.x & 63;
  const int k = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (k >= n_nodes) return;  // whole waves leave together
  const long s = starts[k];
  const unsigned long long key = keys[s];
  double a0 = 0.0, a1 = 0.0, a2 = 0.0;
  for (long base = s;; base += 64) {
    const long i = base + lane;
    const bool in = i < n_entries && keys[i] == key;
    if (in) {
      const float4 v = vals[i];
      a0 += (double)v.x;
      a1 += (double)v.y;
      a2 += (double)v.z;
    }
    // the run is contiguous: it continues only if every lane was inside it
    if (__ballot(in) != ~0ull) break;
  }
  for (int o = 32; o > 0; o >>= 1) {
    a0 += __shfl_xor(a0, o);
    a1 += __shfl_xor(a1, o);
    a2 += __shfl_xor(a2, o);
  }
  if (lane != 0) return;
  rd_node<DIM>(key, a0, a1, a2, g, pos[k], w[k], str[k]);
}

// ---------------------------------------------------------------------------
// Nodes by blocks of the grid (the usual case: keys of at most kBlockKeyBits).
//
// The nodes of a block of 64 (4^3, or 8^2 in 2D: the low six bits of the
// Morton key, one node per lane) receive only from particles whose nearest
// node is within two of the block.  Particles are sorted by cell of 2^DIM
// nodes; a bitmap of the occupied cells with a running count of its bits
// turns a cell into its range of sorted particles, and a second bitmap holds
// the blocks in reach of an occupied cell.  A wave takes a block's region (64
// cells, 36 in 2D), stages 64 particles at a time as the weights of the
// block's nodes along each axis (separable: 12 or 16 evaluations per particle
// and block instead of one per particle, node and axis), and every lane sums
// its node in FP64 in sorted order.  Particles with no weight in the block on
// some axis, a third of a region's for a radius of 2 and three quarters for 1,
// are left out of the staging.  Regions of many particles are split into items
// of kItem, whose partial sums a second kernel adds in order: a wave walks its
// item alone, so the longest item bounds a launch on a coarse grid, where there
// are few blocks.  Items of 2048 without that culling -> 512 with it: 308618
// particles on 0.0177, lambda1 1260 -> 1107 us a call, on 0.03, m4' 1155 ->
// 1010; 10^6 on 0.0177, m4' 2017 -> 1848.
//
// Ring of 2^20 particles, m4', h = 0.01 (131 million candidate contributions):
// by_entries writes, sorts three times and reads 1.6 GB of entries, 4.5 ms of
// kernels; here rd_block_sums took 0.50 ms before the culling (8 blocks of 64
// nodes per particle, 24 % of whose products are nonzero: vector and LDS
// issue), the rest 0.3 ms.  A call on host arrays 6.24 -> 2.29 ms; 800000 particles on
// 0.03 (lambda3) 4.31 -> 1.66; 300000 in 2D 0.96 -> 0.89.
// ---------------------------------------------------------------------------
constexpr int kBlockKeyBits = 30;
constexpr int kItem = 512;

template <int DIM>
struct Blk {
  static constexpr int SIDE = DIM == 3 ? 4 : 8;       // nodes per axis
  static constexpr int CELL_BITS = DIM;               // a cell: 2 nodes per axis
  static constexpr int SPAN = SIDE / 2 + 2;           // cells of a region per axis
  static constexpr int CELLS = DIM == 3 ? 64 : 36;
};

template <int DIM>
__device__ __forceinline__ unsigned key_of(const unsigned* q) {
  if constexpr (DIM == 3)
    return (unsigned)(spread3(q[0]) | (spread3(q[1]) << 1) | (spread3(q[2]) << 2));
  else
    return (unsigned)(spread2(q[0]) | (spread2(q[1]) << 1));
}
template <int DIM>
__device__ __forceinline__ void axes_of(unsigned key, unsigned* q) {
#pragma unroll
  for (int c = 0; c < DIM; ++c) q[c] = DIM == 3 ? compact3(key >> c) : compact2(key >> c);
}

// Index of a particle's nearest node along axis c (as rd_entry).
template <int DIM>
__device__ __forceinline__ unsigned nearest(float x, const Grid& g, int c) {
  if constexpr (DIM == 3) return (unsigned)roundf(rn_mul(rn_sub(x, g.mn[c]), g.rh));
  return (unsigned)roundf((float)(((double)x - (double)g.mn[c]) * (double)g.rh));
}

template <int DIM>
__global__ __launch_bounds__(256) void rd_keys(const float4* __restrict__ pv, int n, Grid g,
                                               unsigned* __restrict__ keys, int* __restrict__ idx) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float4 p = pv[i];
  const float x[3] = {p.x, p.y, p.z};
  unsigned q[3];
#pragma unroll
  for (int c = 0; c < DIM; ++c) q[c] = nearest<DIM>(x[c], g, c);
  keys[i] = key_of<DIM>(q);
  idx[i] = i;
}

// Particles in sorted order, and the bitmap of the occupied cells.
template <int DIM>
__global__ __launch_bounds__(256) void rd_place(const float4* __restrict__ pv,
                                                const float4* __restrict__ a,
                                                const unsigned* __restrict__ keys,
                                                const int* __restrict__ idx, int n,
                                                float4* __restrict__ spv, float4* __restrict__ sa,
                                                unsigned* __restrict__ cells) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int j = idx[i];
  spv[i] = pv[j];
  if constexpr (DIM == 3) sa[i] = a[j];
  const unsigned cell = keys[i] >> Blk<DIM>::CELL_BITS;
  if (i == 0 || keys[i - 1] >> Blk<DIM>::CELL_BITS != cell)
    atomicOr(&cells[cell >> 5], 1u << (cell & 31));
}

// Cells of a block (by their bit in the block's part of the cell bitmap) that
// are in the region of the neighbour at offset d in {-1, 0, 1}^DIM: those on
// its side.
template <int DIM>
constexpr unsigned facing(int dx, int dy, int dz) {
  constexpr int H = Blk<DIM>::SIDE / 2, N = DIM == 3 ? 8 : 16;
  unsigned m = 0;
  for (int k = 0; k < N; ++k) {
    int x = 0, y = 0, z = 0;  // the cell's coordinates from its Morton index
    for (int b = 0; b < (DIM == 3 ? 1 : 2); ++b) {
      x |= ((k >> (DIM * b)) & 1) << b;
      y |= ((k >> (DIM * b + 1)) & 1) << b;
      if (DIM == 3) z |= ((k >> (DIM * b + 2)) & 1) << b;
    }
    const bool in = (dx == 0 || x == (dx < 0 ? 0 : H - 1)) && (dy == 0 || y == (dy < 0 ? 0 : H - 1)) &&
                    (DIM == 2 || dz == 0 || z == (dz < 0 ? 0 : H - 1));
    if (in) m |= 1u << k;
  }
  return m;
}

// The blocks in reach of an occupied cell (one thread per word of cells).
template <int DIM>
__global__ __launch_bounds__(256) void rd_reach(const unsigned* __restrict__ cells, int n_words,
                                                unsigned* __restrict__ blocks,
                                                unsigned n_block_keys) {
  constexpr int PER = DIM == 3 ? 8 : 16;  // cells of a block
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n_words) return;
  const unsigned w = cells[i];
  if (w == 0) return;
  for (int h = 0; h < 32 / PER; ++h) {
    const unsigned own = (w >> (PER * h)) & ((1u << PER) - 1u);
    if (own == 0) continue;
    unsigned b[3];
    axes_of<DIM>((unsigned)i * (32 / PER) + h, b);
#pragma unroll
    for (int m = 0; m < (DIM == 3 ? 27 : 9); ++m) {
      const int dx = m % 3 - 1, dy = (m / 3) % 3 - 1, dz = DIM == 3 ? m / 9 - 1 : 0;
      if (!(own & facing<DIM>(dx, dy, dz))) continue;
      // (node indices start at 5: a neighbour below 0 faces no occupied cell)
      const unsigned o[3] = {b[0] + dx, b[1] + dy, b[2] + dz};
      const unsigned k = key_of<DIM>(o);
      if (k < n_block_keys) atomicOr(&blocks[k >> 5], 1u << (k & 31));
    }
  }
}

__global__ __launch_bounds__(256) void rd_popcounts(const unsigned* __restrict__ words, int n,
                                                    int* __restrict__ counts) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) counts[i] = __popc(words[i]);
}

// Position of bit k among the set bits (incl: running count by word).
__device__ __forceinline__ int bit_rank(const unsigned* __restrict__ words,
                                        const int* __restrict__ incl, unsigned k) {
  const unsigned w = words[k >> 5];
  return incl[k >> 5] - __popc(w >> (k & 31));
}

template <int DIM>
__global__ __launch_bounds__(256) void rd_starts(const unsigned* __restrict__ keys, int n,
                                                 const unsigned* __restrict__ cells,
                                                 const int* __restrict__ incl,
                                                 int* __restrict__ starts) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const unsigned cell = keys[i] >> Blk<DIM>::CELL_BITS;
  const bool head = i == 0 || keys[i - 1] >> Blk<DIM>::CELL_BITS != cell;
  const int r = head || i == n - 1 ? bit_rank(cells, incl, cell) : 0;
  if (head) starts[r] = i;
  if (i == n - 1) starts[r + 1] = n;
}

// The set bits of a bitmap in order.
__global__ __launch_bounds__(256) void rd_bit_list(const unsigned* __restrict__ words, int n,
                                                   const int* __restrict__ incl,
                                                   unsigned* __restrict__ list) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  unsigned w = words[i];
  int at = incl[i] - __popc(w);
  for (; w != 0; w &= w - 1) list[at++] = 32u * i + (unsigned)(__ffs(w) - 1);
}

// This lane's cell of a block's region: its range of sorted particles.
template <int DIM>
__device__ __forceinline__ int2 region_cell(unsigned block, int lane, unsigned n_cells,
                                            const unsigned* __restrict__ cells,
                                            const int* __restrict__ incl,
                                            const int* __restrict__ starts) {
  constexpr int S = Blk<DIM>::SPAN;
  unsigned b[3], o[3];
  axes_of<DIM>(block, b);
  const int s[3] = {lane % S, (lane / S) % S, lane / (S * S)};
  bool in = lane < Blk<DIM>::CELLS;
#pragma unroll
  for (int c = 0; c < DIM; ++c) {
    const int v = (int)b[c] * (Blk<DIM>::SIDE / 2) - 1 + s[c];
    in = in && v >= 0;
    o[c] = v < 0 ? 0u : (unsigned)v;
  }
  const unsigned cell = key_of<DIM>(o);
  in = in && cell < n_cells;
  if (!in || !((cells[cell >> 5] >> (cell & 31)) & 1)) return make_int2(0, 0);
  const int r = bit_rank(cells, incl, cell);
  return make_int2(starts[r], starts[r + 1]);
}

// Items of each block's region (one wave per block).
template <int DIM>
__global__ __launch_bounds__(256) void rd_region_items(const unsigned* __restrict__ list,
                                                       int n_blocks, unsigned n_cells,
                                                       const unsigned* __restrict__ cells,
                                                       const int* __restrict__ incl,
                                                       const int* __restrict__ starts,
                                                       int* __restrict__ items) {
  const int lane = threadIdx.x & 63, k = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (k >= n_blocks) return;
  const int2 r = region_cell<DIM>(list[k], lane, n_cells, cells, incl, starts);
  int c = r.y - r.x;
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
  if (lane == 0) items[k] = (c + kItem - 1) / kItem;
}

// (block, item within it) of every item.
__global__ __launch_bounds__(256) void rd_item_list(const int* __restrict__ items,
                                                    const int* __restrict__ incl, int n_blocks,
                                                    int2* __restrict__ out) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n_blocks) return;
  const int n = items[k], at = incl[k] - n;
  for (int i = 0; i < n; ++i) out[at + i] = make_int2(k, i);
}

// One item: partial sums of a block's 64 nodes over at most kItem particles
// of its region, and whether any contribution was nonzero.  (A strength that
// is not finite makes the mean strength, and with it the removal threshold,
// infinite or NaN, which no node exceeds: the nodes that a zero weight times
// it would add here are removed with all others.)
template <int DIM, int RID>
__global__ __launch_bounds__(256) void rd_block_sums(
    const float4* __restrict__ spv, const float4* __restrict__ sa, Grid g,
    const unsigned* __restrict__ list, unsigned n_cells, const unsigned* __restrict__ cells,
    const int* __restrict__ incl, const int* __restrict__ starts, const int2* __restrict__ items,
    const int* __restrict__ n_items, double* __restrict__ sums, unsigned long long* __restrict__ nonzero) {
  constexpr int SIDE = Blk<DIM>::SIDE, SW = DIM == 3 ? 3 : 1;  // sums per node
  __shared__ float s_w[4][64][DIM * SIDE];
  __shared__ float4 s_a[4][64];
  __shared__ int s_pref[4][64], s_start[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, it = blockIdx.x * 4 + w;
  if (it >= *n_items) return;  // whole waves; no barrier below
  const int2 item = items[it];
  const unsigned block = list[item.x];
  const int2 r = region_cell<DIM>(block, lane, n_cells, cells, incl, starts);
  int pre = r.y - r.x;
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(pre, o, 64);
    if (lane >= o) pre += v;
  }
  const int total = __shfl(pre, 63, 64);
  s_pref[w][lane] = pre - (r.y - r.x);
  s_start[w][lane] = r.x;
  unsigned b[3], q0[3], node[3];
  axes_of<DIM>(block, b);
  axes_of<DIM>((unsigned)lane, node);  // this lane's node within the block
#pragma unroll
  for (int c = 0; c < DIM; ++c) q0[c] = b[c] * SIDE;
  double a0 = 0.0, a1 = 0.0, a2 = 0.0;
  unsigned bits = 0;
  const int i1 = min(total, (item.y + 1) * kItem);
  for (int base = item.y * kItem; base < i1; base += 64) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int e = base + lane;
    float wt[DIM * SIDE];
    float4 al = make_float4(0.f, 0.f, 0.f, 0.f);
    bool live = e < i1;
    if (live) {
      int s = 0;  // the last cell that starts at or before e
#pragma unroll
      for (int h = 32; h > 0; h >>= 1)
        if (s_pref[w][s + h] <= e) s += h;
      const int i = s_start[w][s] + e - s_pref[w][s];
      const float4 p = spv[i];
      const float x[3] = {p.x, p.y, p.z};
      if constexpr (DIM == 3) al = sa[i];
      else al = make_float4(p.z, 0.f, 0.f, 0.f);
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        const unsigned q = nearest<DIM>(x[c], g, c);
        bool reaches = false;
#pragma unroll
        for (int m = 0; m < SIDE; ++m) {
          const unsigned nd = q0[c] + m;
          const bool in = nd - q + (unsigned)g.R <= 2u * (unsigned)g.R;
          const float pos = rn_add(g.mn[c], rn_mul(g.h, (float)nd));
          const float U = fabsf(rn_mul(rn_sub(x[c], pos), g.rh));
          wt[c * SIDE + m] = in ? rd_f<RID>(U) : 0.f;
          reaches = reaches || wt[c * SIDE + m] != 0.f;
        }
        live = live && reaches;
      }
    }
    // only the particles with a weight on every axis are staged, in order
    const unsigned long long lives = __ballot(live);
    if (live) {
      const int at = __popcll(lives & ((1ull << lane) - 1));
#pragma unroll
      for (int m = 0; m < DIM * SIDE; ++m) s_w[w][at][m] = wt[m];
      s_a[w][at] = al;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int cnt = __popcll(lives);
#pragma unroll 4
    for (int j = 0; j < cnt; ++j) {
      float frac = s_w[w][j][node[0]];
      frac = rn_mul(frac, s_w[w][j][SIDE + node[1]]);
      if constexpr (DIM == 3) frac = rn_mul(frac, s_w[w][j][2 * SIDE + node[2]]);
      const float4 al = s_a[w][j];
      float vx = rn_mul(al.x, frac), vy = 0.f, vz = 0.f;
      if constexpr (DIM == 3) {
        vy = rn_mul(al.y, frac);
        vz = rn_mul(al.z, frac);
      }
      a0 += (double)vx;
      bits |= __float_as_uint(vx);
      if constexpr (DIM == 3) {
        a1 += (double)vy;
        a2 += (double)vz;
        bits |= __float_as_uint(vy) | __float_as_uint(vz);
      }
    }
  }
  double* o = sums + (size_t)it * (64 * SW) + lane;
  o[0] = a0;
  if constexpr (DIM == 3) {
    o[64] = a1;
    o[128] = a2;
  }
  const unsigned long long nz = __ballot((bits & 0x7fffffffu) != 0);
  if (lane == 0) nonzero[it] = nz;
}

// Nodes of each block: which there are, and how many.
__global__ __launch_bounds__(256) void rd_block_nodes(const int* __restrict__ items,
                                                      const int* __restrict__ incl, int n_blocks,
                                                      const unsigned long long* __restrict__ nonzero,
                                                      unsigned long long* __restrict__ mask,
                                                      int* __restrict__ counts) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n_blocks) return;
  unsigned long long m = 0;
  for (int i = incl[k] - items[k]; i < incl[k]; ++i) m |= nonzero[i];
  mask[k] = m;
  counts[k] = __popcll(m);
}

// The nodes in Morton order (one wave per block): blocks are listed in key
// order and a block's lanes are its keys in order.
template <int DIM>
__global__ __launch_bounds__(256) void rd_emit(const unsigned* __restrict__ list,
                                               const int* __restrict__ items,
                                               const int* __restrict__ item_incl, int n_blocks,
                                               const unsigned long long* __restrict__ mask,
                                               const int* __restrict__ node_incl,
                                               const double* __restrict__ sums, Grid g,
                                               float4* __restrict__ pos, float4* __restrict__ wo,
                                               float* __restrict__ str) {
  constexpr int SW = DIM == 3 ? 3 : 1;
  const int lane = threadIdx.x & 63, k = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (k >= n_blocks) return;
  const unsigned long long m = mask[k];
  if (!((m >> lane) & 1)) return;
  double a[3] = {0.0, 0.0, 0.0};
  for (int i = item_incl[k] - items[k]; i < item_incl[k]; ++i)
#pragma unroll
    for (int c = 0; c < SW; ++c) a[c] += sums[(size_t)i * (64 * SW) + 64 * c + lane];
  const int at = node_incl[k] - __popcll(m) + __popcll(m & ((1ull << lane) - 1));
  float4 p, w;
  float s;
  rd_node<DIM>((unsigned long long)list[k] * 64 + lane, a[0], a[1], a[2], g, p, w, s);
  pos[at] = p;
  wo[at] = w;
  str[at] = s;
}

// Per-block FP64 sum and FP32 min / max of the strengths.
__global__ __launch_bounds__(256) void rd_str_stats(const float* __restrict__ str, int n,
                                                    double* __restrict__ psum,
                                                    float* __restrict__ pmin,
                                                    float* __restrict__ pmax) {
  __shared__ double ss[256];
  __shared__ float sl[256], sh[256];
  double s = 0.0;
  float lo = __builtin_inff(), hi = -__builtin_inff();
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const float v = str[i];
    s += (double)v;
    lo = fminf(lo, v);
    hi = fmaxf(hi, v);
  }
  ss[threadIdx.x] = s;
  sl[threadIdx.x] = lo;
  sh[threadIdx.x] = hi;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      ss[threadIdx.x] += ss[threadIdx.x + w];
      sl[threadIdx.x] = fminf(sl[threadIdx.x], sl[threadIdx.x + w]);
      sh[threadIdx.x] = fmaxf(sh[threadIdx.x], sh[threadIdx.x + w]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    psum[blockIdx.x] = ss[0];
    pmin[blockIdx.x] = sl[0];
    pmax[blockIdx.x] = sh[0];
  }
}

// The removal threshold, negligible x the mean strength, from the blocks' sums
// (added in block order, in the reference's types: src/P3D.cpp:600-605).
__global__ __launch_bounds__(kPartBlocks) void rd_threshold(const double* __restrict__ psum, int n,
                                                   float negligible, float* __restrict__ thr) {
  __shared__ double s[kPartBlocks];
  s[threadIdx.x] = psum[threadIdx.x];
  __syncthreads();
  if (threadIdx.x != 0) return;
  double a = 0.0;
#pragma unroll 16
  for (int b = 0; b < kPartBlocks; ++b) a += s[b];
  const float mean = __fdiv_rn((float)a, (float)n);
  *thr = rn_mul(mean, negligible);
}

// Each kept particle's share of the removed strength.
__global__ __launch_bounds__(kPartBlocks) void rd_share(const double* __restrict__ pdef,
                                               const int* __restrict__ n_kept,
                                               float4* __restrict__ share) {
  __shared__ double s[kPartBlocks * 3];
#pragma unroll
  for (int k = 0; k < 3; ++k) s[k * kPartBlocks + threadIdx.x] = pdef[k * kPartBlocks + threadIdx.x];
  __syncthreads();
  const int c = threadIdx.x;
  if (c >= 4) return;
  double d = 0.0;
  if (c < 3) {
#pragma unroll 16
    for (int b = 0; b < kPartBlocks; ++b) d += s[b * 3 + c];
  }
  // the reference divides the removed strength by the kept count in FP32
  reinterpret_cast<float*>(share)[c] = c < 3 ? __fdiv_rn((float)d, (float)*n_kept) : 0.f;
}

// keep[i] = str[i] > *thr_p && i < max_keep; per-block FP64 sums of the
// removed strength (3 components).
__global__ __launch_bounds__(256) void rd_flags(const float* __restrict__ str,
                                                const float4* __restrict__ w, int n,
                                                const float* __restrict__ thr_p, int max_keep,
                                                unsigned char* __restrict__ keep,
                                                double* __restrict__ pdef) {
  __shared__ double sd[3][256];
  const float thr = *thr_p;
  double d0 = 0.0, d1 = 0.0, d2 = 0.0;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const bool k = str[i] > thr && i < max_keep;
    keep[i] = k ? 1 : 0;
    if (!k) {
      const float4 v = w[i];
      d0 += (double)v.x;
      d1 += (double)v.y;
      d2 += (double)v.z;
    }
  }
  sd[0][threadIdx.x] = d0;
  sd[1][threadIdx.x] = d1;
  sd[2][threadIdx.x] = d2;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s)
      for (int c = 0; c < 3; ++c) sd[c][threadIdx.x] += sd[c][threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int c = 0; c < 3; ++c) pdef[blockIdx.x * 3 + c] = sd[c][0];
}

// Gather the kept particles, add the shared deficit, refresh |w|.
template <int DIM>
__global__ __launch_bounds__(256) void rd_keep(const int* __restrict__ idx,
                                               const int* __restrict__ n_kept,
                                               const float4* __restrict__ pos_in,
                                               const float4* __restrict__ w_in,
                                               const float4* __restrict__ share,
                                               float4* __restrict__ pos_out,
                                               float4* __restrict__ w_out,
                                               float* __restrict__ str_out) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= *n_kept) return;
  const float4 def = *share;
  const int i = idx[j];
  pos_out[j] = pos_in[i];
  const float4 v = w_in[i];
  const float4 ww = make_float4(rn_add(v.x, def.x), rn_add(v.y, def.y),
                                rn_add(v.z, def.z), 0.f);
  w_out[j] = ww;
  str_out[j] = DIM == 3 ? __fsqrt_rn(rn_add(rn_add(rn_mul(ww.x, ww.x), rn_mul(ww.y, ww.y)),
                                               rn_mul(ww.z, ww.z)))
                        : fabsf(ww.x);
}

// Histogram of the strength-threshold search (reference
// src/redistribution_helper_funcs.cpp:54-60): bin = floor(1023 (s - minv) / range).
__global__ __launch_bounds__(256) void rd_hist(const float* __restrict__ str, int n, double minv,
                                               double range, int* __restrict__ counts) {
  __shared__ int sc[1024];
  for (int b = threadIdx.x; b < 1024; b += 256) sc[b] = 0;
  __syncthreads();
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    int b = (int)floor((double)1023 * ((double)str[i] - minv) / range);
    b = b < 0 ? 0 : (b > 1023 ? 1023 : b);
    atomicAdd(&sc[b], 1);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < 1024; b += 256)
    if (sc[b]) atomicAdd(&counts[b], sc[b]);
}

// AoS output records: 3D {coord[3], vorticity[3], volume} (7 floats),
// 2D {coord[2], vorticity, area} (4 floats).
template <int DIM>
__global__ __launch_bounds__(256) void rd_pack(const float4* __restrict__ pos,
                                               const float4* __restrict__ w, int n,
                                               float* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float4 p = pos[i];
  const float4 v = w[i];
  if constexpr (DIM == 3) {
    float* r = out + 7 * (size_t)i;
    r[0] = p.x; r[1] = p.y; r[2] = p.z; r[3] = v.x; r[4] = v.y; r[5] = v.z; r[6] = p.w;
  } else {
    float* r = out + 4 * (size_t)i;
    r[0] = p.x; r[1] = p.y; r[2] = v.x; r[3] = p.w;
  }
}

size_t al256(size_t b) { return (b + 255) & ~size_t(255); }

// Bump allocator over one runtime workspace slot.
struct Arena {
  char* base = nullptr;
  size_t used = 0, cap = 0;
  template <class T>
  T* take(size_t n) {
    T* p = (T*)(base + used);
    used += al256(sizeof(T) * (n > 0 ? n : 1));
    return used <= cap ? p : nullptr;
  }
};

template <int DIM>
hipError_t launch_contrib_count(int rid, const float4* pv, const float4* a, long ne, const Grid& g,
                                int* counts, hipStream_t s) {
  const dim3 grid((unsigned)((ne + kChunk - 1) / kChunk));
  switch (rid) {
    case 0: hipLaunchKernelGGL((rd_contrib_count<DIM, 0>), grid, dim3(256), 0, s, pv, a, ne, g, counts); break;
    case 1: hipLaunchKernelGGL((rd_contrib_count<DIM, 1>), grid, dim3(256), 0, s, pv, a, ne, g, counts); break;
    case 2: hipLaunchKernelGGL((rd_contrib_count<DIM, 2>), grid, dim3(256), 0, s, pv, a, ne, g, counts); break;
    case 3: hipLaunchKernelGGL((rd_contrib_count<DIM, 3>), grid, dim3(256), 0, s, pv, a, ne, g, counts); break;
    default: hipLaunchKernelGGL((rd_contrib_count<DIM, 4>), grid, dim3(256), 0, s, pv, a, ne, g, counts); break;
  }
  return hipGetLastError();
}

template <int DIM>
hipError_t launch_contrib_write(int rid, const float4* pv, const float4* a, long ne, const Grid& g,
                                const int* incl, unsigned long long* keys, float4* vals,
                                hipStream_t s) {
  const dim3 grid((unsigned)((ne + kChunk - 1) / kChunk));
  switch (rid) {
    case 0: hipLaunchKernelGGL((rd_contrib_write<DIM, 0>), grid, dim3(256), 0, s, pv, a, ne, g, incl, keys, vals); break;
    case 1: hipLaunchKernelGGL((rd_contrib_write<DIM, 1>), grid, dim3(256), 0, s, pv, a, ne, g, incl, keys, vals); break;
    case 2: hipLaunchKernelGGL((rd_contrib_write<DIM, 2>), grid, dim3(256), 0, s, pv, a, ne, g, incl, keys, vals); break;
    case 3: hipLaunchKernelGGL((rd_contrib_write<DIM, 3>), grid, dim3(256), 0, s, pv, a, ne, g, incl, keys, vals); break;
    default: hipLaunchKernelGGL((rd_contrib_write<DIM, 4>), grid, dim3(256), 0, s, pv, a, ne, g, incl, keys, vals); break;
  }
  return hipGetLastError();
}

}  // namespace

float redist_radius(int rid) {
  static const float r[5] = {0.5f, 1.0f, 1.5f, 2.0f, 2.0f};
  return (rid >= 0 && rid < 5) ? r[rid] : -1.f;
}

namespace {

// The nodes of a redistribution and the scratch of what follows, in the
// runtime's node workspace.
struct Nodes {
  float4 *pos0, *w0, *pos1, *w1;
  float *str0, *str1;
  unsigned char* head;
  int *kidx, *nkept, *counts;
  double* pdef;
  float *psmin, *psmax, *thr, *packed;
  float4* share;
  void* sel;
  size_t sel_bytes;
};

int rd_fail(Runtime& rt, const char* what, hipError_t e) {
  if (e != hipSuccess) check_hip(rt, e, what);
  else set_error(rt, what);
  return -1;
}

bool alloc_nodes(Runtime& rt, Device& d, int nn, Nodes* n, hipStream_t s) {
  n->sel_bytes = 0;
  const hipError_t e = rocprim::select(nullptr, n->sel_bytes, rocprim::counting_iterator<int>(0),
                                       (unsigned char*)nullptr, (int*)nullptr, (int*)nullptr,
                                       (size_t)nn, s);
  if (e != hipSuccess) return rd_fail(rt, "select size", e), false;
  const size_t need = al256(n->sel_bytes) + al256(nn) + al256(sizeof(float4) * nn) * 4 +
                      al256(sizeof(float) * nn) * 2 + al256(sizeof(int) * nn) + al256(sizeof(int)) +
                      al256(sizeof(double) * kPartBlocks * 3) + al256(sizeof(float) * kPartBlocks * 2) +
                      al256(sizeof(int) * 1024) + al256(sizeof(float4)) * 2 +
                      al256(sizeof(float) * 7 * (size_t)nn);
  Arena na;
  na.base = (char*)device_buffer(rt, d, SLOT_RD_NODES, need);
  na.cap = need;
  if (!na.base) return false;
  n->sel = na.take<char>(n->sel_bytes);
  n->head = na.take<unsigned char>(nn);
  n->pos0 = na.take<float4>(nn);
  n->w0 = na.take<float4>(nn);
  n->pos1 = na.take<float4>(nn);
  n->w1 = na.take<float4>(nn);
  n->str0 = na.take<float>(nn);
  n->str1 = na.take<float>(nn);
  n->kidx = na.take<int>(nn);
  n->nkept = na.take<int>(1);
  n->pdef = na.take<double>(kPartBlocks * 3);
  n->psmin = na.take<float>(2 * kPartBlocks);
  n->psmax = n->psmin + kPartBlocks;
  n->counts = na.take<int>(1024);
  n->thr = na.take<float>(1);
  n->share = na.take<float4>(1);
  n->packed = na.take<float>(7 * (size_t)nn);
  if (!n->packed) return rd_fail(rt, "redistribution workspace", hipSuccess), false;
  return true;
}

// What comes back to the host, in pinned memory: a copy to pageable memory goes
// through a staging buffer and waits for it on its own.  A call makes four to ten
// such copies; with the three of the bounds in one, and rd_threshold's and
// rd_share's loads in flight at once, us a call: 8000 particles on 0.008
// 548 -> 405, on 0.03 393 -> 300, 308618 on 0.0177 1107 -> 1006, 8000 in 2D
// 350 -> 282.
struct Bounds {
  float mn[kPartBlocks * 3], mx[kPartBlocks * 3];
  double sum[kPartBlocks * 3];
};
struct Landing {
  Bounds bounds;
  float smin[kPartBlocks], smax[kPartBlocks];  // adjacent on the device too
  int bins[1024];
  int total;
  float threshold;
};

// Running counts (in place of `counts`, into `incl`); with `land`, their total
// in land->total.
bool running_counts(Runtime& rt, int* counts, int* incl, size_t n, void* tmp, size_t tmp_bytes,
                    Landing* land, hipStream_t s) {
  hipError_t e = rocprim::inclusive_scan(tmp, tmp_bytes, counts, incl, n, rocprim::plus<int>(), s);
  if (e == hipSuccess && land)
    e = hipMemcpyAsync(&land->total, incl + (n - 1), sizeof(int), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess && land) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return rd_fail(rt, "redistribution scan", e), false;
  return true;
}

// A particle of one block's region is one of at most this many blocks'.
constexpr int kRegionsOfACell = 8;
constexpr int kNotByBlocks = -2;

// Nodes by blocks of the grid (see above): their number, -1 with the error
// recorded, or kNotByBlocks where the grid's keys are too long for the
// bitmaps or particles so scattered that the blocks' regions would make more
// than kMostItems items, whose sums (1.5 KB each in 3D) take 1.5 GiB.
constexpr size_t kMostItems = (size_t)1 << 20;

template <int DIM>
int by_blocks(Runtime& rt, Device& d, const RedistJob& j, const Grid& g, int key_bits, Nodes* out,
              Landing* land, hipStream_t s) {
  using B = Blk<DIM>;
  if (key_bits > kBlockKeyBits || key_bits < 6) return kNotByBlocks;
  const int n = j.n;
  const unsigned n_cells = 1u << (key_bits - B::CELL_BITS), n_block_keys = 1u << (key_bits - 6);
  const int cw = (int)((n_cells + 31) / 32), bw = (int)((n_block_keys + 31) / 32);
  size_t sort_tmp = 0, scan_tmp = 0;
  using Sort = rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config,
                                          rocprim::default_config, 1 << 16>;
  hipError_t e = rocprim::radix_sort_pairs<Sort>(nullptr, sort_tmp, (unsigned*)nullptr, (unsigned*)nullptr,
                                                 (int*)nullptr, (int*)nullptr, (size_t)n, B::CELL_BITS,
                                                 key_bits, s);
  if (e == hipSuccess)
    e = rocprim::inclusive_scan(nullptr, scan_tmp, (int*)nullptr, (int*)nullptr,
                                std::max((size_t)cw, kMostItems), rocprim::plus<int>(), s);
  if (e != hipSuccess) return rd_fail(rt, "redistribution sort size", e);
  // ---- particles by cell, the bitmaps and their running counts ----
  const size_t need = al256(sizeof(unsigned) * n) * 2 + al256(sizeof(int) * n) * 2 +
                      al256(sizeof(float4) * n) * 2 + al256(sizeof(int) * ((size_t)n + 1)) +
                      al256(sizeof(unsigned) * ((size_t)cw + bw)) + al256(sizeof(int) * cw) * 2 +
                      al256(sizeof(int) * bw) + al256(std::max(sort_tmp, scan_tmp));
  Arena ar;
  ar.base = (char*)device_buffer(rt, d, SLOT_RD_CHUNKS, need);
  ar.cap = need;
  if (!ar.base) return -1;
  auto* k_in = ar.take<unsigned>(n);
  auto* keys = ar.take<unsigned>(n);
  auto* i_in = ar.take<int>(n);
  auto* idx = ar.take<int>(n);
  auto* spv = ar.take<float4>(n);
  auto* sa = ar.take<float4>(n);
  auto* starts = ar.take<int>((size_t)n + 1);
  auto* cells = ar.take<unsigned>((size_t)cw + bw);
  unsigned* blocks = cells + cw;
  auto* pop = ar.take<int>(cw);
  auto* cincl = ar.take<int>(cw);
  auto* bincl = ar.take<int>(bw);
  void* tmp = ar.take<char>(std::max(sort_tmp, scan_tmp));
  if (!tmp) return rd_fail(rt, "redistribution workspace", hipSuccess);
  const dim3 pg((n + 255) / 256), blk(256);
  e = hipMemsetAsync(cells, 0, sizeof(unsigned) * ((size_t)cw + bw), s);
  if (e != hipSuccess) return rd_fail(rt, "redistribution cells", e);
  hipLaunchKernelGGL(rd_keys<DIM>, pg, blk, 0, s, j.pv, n, g, k_in, i_in);
  e = rocprim::radix_sort_pairs<Sort>(tmp, sort_tmp, k_in, keys, i_in, idx, (size_t)n, B::CELL_BITS,
                                      key_bits, s);
  if (e != hipSuccess) return rd_fail(rt, "redistribution sort", e);
  hipLaunchKernelGGL(rd_place<DIM>, pg, blk, 0, s, j.pv, j.a, keys, idx, n, spv, sa, cells);
  hipLaunchKernelGGL(rd_reach<DIM>, dim3((cw + 255) / 256), blk, 0, s, cells, cw, blocks, n_block_keys);
  hipLaunchKernelGGL(rd_popcounts, dim3((cw + 255) / 256), blk, 0, s, cells, cw, pop);
  if (!running_counts(rt, pop, cincl, cw, tmp, scan_tmp, nullptr, s)) return -1;
  hipLaunchKernelGGL(rd_starts<DIM>, pg, blk, 0, s, keys, n, cells, cincl, starts);
  hipLaunchKernelGGL(rd_popcounts, dim3((bw + 255) / 256), blk, 0, s, blocks, bw, pop);
  if (!running_counts(rt, pop, bincl, bw, tmp, scan_tmp, land, s)) return -1;
  const int nb = land->total;
  if (nb == 0) return kNotByBlocks;
  // ---- items of each block's region, their sums ----
  const size_t most = (size_t)nb + (size_t)kRegionsOfACell * n / kItem + 1;
  if (most > kMostItems) return kNotByBlocks;
  constexpr int SW = DIM == 3 ? 3 : 1;
  const size_t sneed = al256(sizeof(unsigned) * nb) + al256(sizeof(int) * nb) * 4 +
                       al256(sizeof(int2) * most) + al256(sizeof(double) * 64 * SW * most) +
                       al256(8 * most) + al256(8 * (size_t)nb) + al256(scan_tmp);
  Arena sr;
  sr.base = (char*)device_buffer(rt, d, SLOT_RD, sneed);
  sr.cap = sneed;
  if (!sr.base) return -1;
  auto* list = sr.take<unsigned>(nb);
  auto* items = sr.take<int>(nb);
  auto* iincl = sr.take<int>(nb);
  auto* ncount = sr.take<int>(nb);
  auto* nincl = sr.take<int>(nb);
  auto* ilist = sr.take<int2>(most);
  auto* sums = sr.take<double>(64 * SW * most);
  auto* nonzero = sr.take<unsigned long long>(most);
  auto* mask = sr.take<unsigned long long>(nb);
  void* tmp2 = sr.take<char>(scan_tmp);
  if (!tmp2) return rd_fail(rt, "redistribution workspace", hipSuccess);
  const dim3 bg((nb + 255) / 256), wg((nb + 3) / 4);
  hipLaunchKernelGGL(rd_bit_list, dim3((bw + 255) / 256), blk, 0, s, blocks, bw, bincl, list);
  hipLaunchKernelGGL(rd_region_items<DIM>, wg, blk, 0, s, list, nb, n_cells, cells, cincl, starts,
                     items);
  if (!running_counts(rt, items, iincl, nb, tmp2, scan_tmp, nullptr, s)) return -1;
  hipLaunchKernelGGL(rd_item_list, bg, blk, 0, s, items, iincl, nb, ilist);
  const auto sum = j.rid == 0   ? rd_block_sums<DIM, 0>
                   : j.rid == 1 ? rd_block_sums<DIM, 1>
                   : j.rid == 2 ? rd_block_sums<DIM, 2>
                   : j.rid == 3 ? rd_block_sums<DIM, 3>
                                : rd_block_sums<DIM, 4>;
  hipLaunchKernelGGL(sum, dim3((unsigned)((most + 3) / 4)), blk, 0, s, spv, sa, g, list, n_cells,
                     cells, cincl, starts, ilist, iincl + (nb - 1), sums, nonzero);
  hipLaunchKernelGGL(rd_block_nodes, bg, blk, 0, s, items, iincl, nb, nonzero, mask, ncount);
  if (!running_counts(rt, ncount, nincl, nb, tmp2, scan_tmp, land, s)) return -1;
  const int nn = land->total;
  if (nn == 0) return 0;
  if (!alloc_nodes(rt, d, nn, out, s)) return -1;
  hipLaunchKernelGGL(rd_emit<DIM>, wg, blk, 0, s, list, items, iincl, nb, mask, nincl, sums, g,
                     out->pos0, out->w0, out->str0);
  e = hipGetLastError();
  if (e != hipSuccess) return rd_fail(rt, "redistribution nodes", e);
  return nn;
}

// Nodes by sorting every nonzero (node, contribution) entry: any grid.
template <int DIM>
int by_entries(Runtime& rt, Device& d, const RedistJob& j, const Grid& g, int key_bits, Nodes* out,
               Landing* land, hipStream_t s) {
  auto fail = [&](const char* what, hipError_t e) { return rd_fail(rt, what, e); };
  const int n = j.n;
  const int W = 2 * g.R + 1;
  const long WD = DIM == 3 ? (long)W * W * W : (long)W * W;
  const long ne = (long)n * WD;
  // ---- nonzero entries: count per chunk, scan, compacting write ----
  const long nc = (ne + kChunk - 1) / kChunk;
  size_t scan_tmp = 0;
  hipError_t e = rocprim::inclusive_scan(nullptr, scan_tmp, (int*)nullptr, (int*)nullptr, (size_t)nc,
                              rocprim::plus<int>(), s);
  if (e != hipSuccess) return fail("scan size", e);
  Arena ca;
  const size_t cneed = al256(sizeof(int) * nc) * 2 + al256(scan_tmp);
  ca.base = (char*)device_buffer(rt, d, SLOT_RD_CHUNKS, cneed);
  ca.cap = cneed;
  if (!ca.base) return -1;
  auto* ccount = ca.take<int>(nc);
  auto* cincl = ca.take<int>(nc);
  void* ct = ca.take<char>(scan_tmp);
  // the count of the chunks' items (in cincl's last element) on the host
  auto scan_total = [&](long chunks, int* total) {
    if (!running_counts(rt, ccount, cincl, (size_t)chunks, ct, scan_tmp, land, s)) return false;
    *total = land->total;
    return true;
  };
  e = launch_contrib_count<DIM>(j.rid, j.pv, j.a, ne, g, ccount, s);
  if (e != hipSuccess) return fail("redistribution contributions", e);
  int nz = 0;
  if (!scan_total(nc, &nz)) return -1;
  if (nz == 0) return 0;
  // ---- workspace: the nonzero entries and the sort ----
  size_t sort_tmp = 0;
  e = rocprim::radix_sort_pairs(nullptr, sort_tmp, (unsigned long long*)nullptr,
                                (unsigned long long*)nullptr, (float4*)nullptr, (float4*)nullptr,
                                (size_t)nz, 0, 64, s);
  if (e != hipSuccess) return fail("radix sort size", e);
  const size_t need = al256(sizeof(unsigned long long) * nz) * 2 + al256(sizeof(float4) * nz) * 2 +
                      al256(sort_tmp);
  Arena ar;
  ar.base = (char*)device_buffer(rt, d, SLOT_RD, need);
  ar.cap = need;
  if (!ar.base) return -1;
  auto* k_in = ar.take<unsigned long long>(nz);
  auto* k_out = ar.take<unsigned long long>(nz);
  auto* v_in = ar.take<float4>(nz);
  auto* v_out = ar.take<float4>(nz);
  void* t = ar.take<char>(sort_tmp);
  if (!t) return fail("redistribution workspace", hipSuccess);
  e = launch_contrib_write<DIM>(j.rid, j.pv, j.a, ne, g, cincl, k_in, v_in, s);
  if (e != hipSuccess) return fail("redistribution contributions", e);
  size_t tb = sort_tmp;
  e = rocprim::radix_sort_pairs(t, tb, k_in, k_out, v_in, v_out, (size_t)nz, 0, key_bits, s);
  if (e != hipSuccess) return fail("redistribution sort", e);
  // ---- node starts ----
  const long nh = (nz + kChunk - 1) / kChunk;
  hipLaunchKernelGGL(rd_head_counts, dim3((unsigned)nh), dim3(256), 0, s, k_out, (long)nz, ccount);
  int nn = 0;
  if (!scan_total(nh, &nn)) return -1;
  if (nn == 0) return 0;
  // ---- nodes (their starts take the place of the unsorted keys) ----
  if (!alloc_nodes(rt, d, nn, out, s)) return -1;
  long* starts = (long*)k_in;
  hipLaunchKernelGGL(rd_head_write, dim3((unsigned)nh), dim3(256), 0, s, k_out, (long)nz, cincl,
                     starts);
  hipLaunchKernelGGL((rd_nodes<DIM>), dim3((nn + 3) / 4), dim3(256), 0, s, k_out, v_out, (long)nz,
                     starts, nn, g, out->pos0, out->w0, out->str0);
  e = hipGetLastError();
  if (e != hipSuccess) return fail("redistribution nodes", e);
  return nn;
}

}  // namespace

template <int DIM>
static int redistribute_dim(Runtime& rt, Device& d, const RedistJob& j, float** out_dev,
                            hipStream_t s) {
  auto fail = [&](const char* what, hipError_t e) {
    if (e != hipSuccess) check_hip(rt, e, what);
    else set_error(rt, what);
    return -1;
  };
  const int n = j.n;
  *out_dev = nullptr;
  if (n == 0) return 0;
  // ---- grid origin (reference src/P3D.cpp:538-548) ----
  Bounds* db = (Bounds*)device_buffer(rt, d, SLOT_RD_SMALL, sizeof(Bounds));
  Landing* land = (Landing*)host_buffer(rt, d, SLOT_RD_SMALL, sizeof(Landing));
  if (!db || !land) return -1;
  hipLaunchKernelGGL((rd_bounds<DIM>), dim3(kPartBlocks), dim3(256), 0, s, j.pv, n, db->mn, db->mx,
                     db->sum);
  hipError_t e = hipMemcpyAsync(&land->bounds, db, sizeof(Bounds), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return fail("redistribution bounds", e);
  const float *hmin = land->bounds.mn, *hmax = land->bounds.mx;
  const double* hsum = land->bounds.sum;
  Grid g{};
  g.h = j.h;
  g.rh = 1.f / j.h;
  g.R = (int)roundf(redist_radius(j.rid));
  int axis_bits = 1;  // bits of the largest node index on any axis
  for (int c = 0; c < DIM; ++c) {
    float m = hmin[c], M = hmax[c];
    double sum = 0.0;
    for (int b = 0; b < kPartBlocks; ++b) {
      m = hmin[b * DIM + c] < m ? hmin[b * DIM + c] : m;
      M = hmax[b * DIM + c] > M ? hmax[b * DIM + c] : M;
      sum += hsum[b * DIM + c];
    }
    if (!std::isfinite(m) || !std::isfinite(M)) return fail("non-finite particle coordinates", hipSuccess);
    const float mean = (float)(sum / (double)n);
    float mn = m - 1.f * ((float)g.R * j.h);
    float dc = (mean - mn) / j.h;
    dc = roundf(dc) + 5;
    g.mn[c] = mean - dc * j.h;
    // node indices must fit the Morton key: 21 bits per axis in 3D, 32 in 2D
    const double span = ((double)M - (double)g.mn[c]) / (double)j.h + g.R + 2;
    if (span >= (DIM == 3 ? 2097152.0 : 4294967295.0))
      return fail("grid too fine for the particles' extent", hipSuccess);
    while (axis_bits < 32 && (double)(1ull << axis_bits) <= span) ++axis_bits;
  }
  const int key_bits = DIM * axis_bits < 64 ? DIM * axis_bits : 64;
  const long W = 2 * g.R + 1;  // nodes of a particle's window, per axis
  if ((long)n * (DIM == 3 ? W * W * W : W * W) >= 2147483647L)
    return fail("too many grid contributions for one call", hipSuccess);
  Nodes nd;
  int nn = by_blocks<DIM>(rt, d, j, g, key_bits, &nd, land, s);
  if (nn == kNotByBlocks) nn = by_entries<DIM>(rt, d, j, g, key_bits, &nd, land, s);
  if (nn <= 0) return nn;
  // ---- removal: strength <= threshold (in nd.thr) or index >= max_keep ----
  auto remove = [&](int max_keep) -> int {
    hipLaunchKernelGGL(rd_flags, dim3(kPartBlocks), dim3(256), 0, s, nd.str0, nd.w0, nn, nd.thr,
                       max_keep, nd.head, nd.pdef);
    size_t tb2 = nd.sel_bytes;
    hipError_t ee = rocprim::select(nd.sel, tb2, rocprim::counting_iterator<int>(0), nd.head,
                                    nd.kidx, nd.nkept, (size_t)nn, s);
    if (ee != hipSuccess) return fail("redistribution compaction", ee);
    hipLaunchKernelGGL(rd_share, dim3(1), dim3(kPartBlocks), 0, s, nd.pdef, nd.nkept, nd.share);
    hipLaunchKernelGGL((rd_keep<DIM>), dim3((nn + 255) / 256), dim3(256), 0, s, nd.kidx, nd.nkept,
                       nd.pos0, nd.w0, nd.share, nd.pos1, nd.w1, nd.str1);
    ee = hipMemcpyAsync(&land->total, nd.nkept, sizeof(int), hipMemcpyDeviceToHost, s);
    if (ee == hipSuccess) ee = hipStreamSynchronize(s);
    if (ee != hipSuccess) return fail("redistribution compaction", ee);
    std::swap(nd.pos0, nd.pos1);
    std::swap(nd.w0, nd.w1);
    std::swap(nd.str0, nd.str1);
    nn = land->total;
    return 0;
  };
  hipLaunchKernelGGL(rd_str_stats, dim3(kPartBlocks), dim3(256), 0, s, nd.str0, nn, nd.pdef,
                     nd.psmin, nd.psmax);
  hipLaunchKernelGGL(rd_threshold, dim3(1), dim3(kPartBlocks), 0, s, nd.pdef, nn, j.negligible, nd.thr);
  if (remove(nn) != 0) return -1;
  if (j.max_out >= 0 && nn > j.max_out) {
    // strength threshold, reference src/redistribution_helper_funcs.cpp:33-80
    hipLaunchKernelGGL(rd_str_stats, dim3(kPartBlocks), dim3(256), 0, s, nd.str0, nn, nd.pdef,
                       nd.psmin, nd.psmax);
    static_assert(offsetof(Landing, smax) - offsetof(Landing, smin) == sizeof(float) * kPartBlocks,
                  "adjacent");
    e = hipMemcpyAsync(land->smin, nd.psmin, sizeof(float) * kPartBlocks * 2, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return fail("redistribution strengths", e);
    float smin = __builtin_inff(), smax = -__builtin_inff();
    for (int b = 0; b < kPartBlocks; ++b) {
      smin = land->smin[b] < smin ? land->smin[b] : smin;
      smax = land->smax[b] > smax ? land->smax[b] : smax;
    }
    double minv = smin, maxv = smax, range;
    const int n_guesses = 1024;
    std::vector<float> guesses(n_guesses);
    int* gc = land->bins;
    int k = 0;
    const float tol = 0.01f;
    for (int iter = 0; iter < 4096; ++iter) {
      range = (maxv - minv) * 1.05;
      for (int i = 0; i < n_guesses; ++i)
        guesses[i] = (float)(minv + i * range / (float)(n_guesses - 1));
      e = hipMemsetAsync(nd.counts, 0, sizeof(int) * 1024, s);
      if (e != hipSuccess) return fail("redistribution histogram", e);
      hipLaunchKernelGGL(rd_hist, dim3(kPartBlocks), dim3(256), 0, s, nd.str0, nn, minv, range,
                         nd.counts);
      e = hipMemcpyAsync(gc, nd.counts, sizeof(int) * 1024, hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipStreamSynchronize(s);
      if (e != hipSuccess) return fail("redistribution histogram", e);
      int interp = gc[n_guesses - 1];
      for (int i = n_guesses - 2; i >= 0; --i) {
        maxv = guesses[i + 1];
        minv = guesses[i];
        interp += gc[i];
        gc[i] = interp;
        if (interp > j.max_out) {
          k = i + 1;
          break;
        }
      }
      if (minv == maxv || gc[k] == gc[k - 1] ||
          std::fabs((float)(j.max_out - gc[k]) / ((float)j.max_out)) < tol * 0.6)
        break;
    }
    land->threshold = guesses[k];
    e = hipMemcpyAsync(nd.thr, &land->threshold, sizeof(float), hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return fail("redistribution threshold", e);
    if (remove(j.max_out) != 0) return -1;
  }
  if (j.max_out < 0 || nn == 0) return nn;
  hipLaunchKernelGGL((rd_pack<DIM>), dim3((nn + 255) / 256), dim3(256), 0, s, nd.pos0, nd.w0, nn,
                     nd.packed);
  e = hipGetLastError();
  if (e != hipSuccess) return fail("redistribution output", e);
  *out_dev = nd.packed;
  return nn;
}

int redistribute(Runtime& rt, Device& d, const RedistJob& j, float** out_dev, hipStream_t s) {
  if (j.rid < 0 || j.rid > 4 || !(j.h > 0.f) || j.n < 0 || (j.n > 0 && !j.pv) ||
      (j.dim == 3 && j.n > 0 && !j.a)) {
    set_error(rt, "invalid redistribution job");
    return -1;
  }
  return j.dim == 3 ? redistribute_dim<3>(rt, d, j, out_dev, s)
                    : redistribute_dim<2>(rt, d, j, out_dev, s);
}

}  // namespace cvtx
