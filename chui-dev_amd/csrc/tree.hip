// tree.hip — periodic unwrap, octant-path keys, octree from shared key digits,
// preorder numbering, in-leaf Morton order and FP64 multipoles on gfx950.
//
// The reference builds its octree top-down by recursive stable octant
// partitions of the Morton-presorted particle list against FP64 cube centres
// (tree_gravity.cpp:1081-1206). The same tree is produced here without
// recursion:
//   1. every particle computes its 21-level octant path against the exact FP64
//      centre sequence c +- h/2 (the centres the recursion would visit);
//   2. one stable radix sort by that path gives the preorder leaf sequence;
//   3. the nodes follow from the octant digits that sorted paths share, all
//      levels in one pass (a node is split while count > leaf_size and
//      half > 1e-12);
//   4. inside each leaf the particles are put back into Morton order, because
//      stable partitions preserve the Morton order of a leaf's members.
// All FP64 arithmetic that decides topology or feeds multipoles is written in
// the reference's operation order and compiled with -ffp-contract=off, so keys,
// order, node membership and moments are bit-identical to the CPU path.
#include "tree.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "primitives.hpp"

namespace chui {
namespace {

constexpr uint64_t kEmpty = ~0ull;
constexpr uint32_t kInvalidIndex = 0xFFFFFFFFu;
constexpr int kPathLevels = 21;

struct Axes3 {
  const double* p[3];
};
struct UnwrapArgs {
  double L[3];
  int canonical[3];
  double anchor[3];
};

__device__ __forceinline__ double wrap_coord(double x, double L, int canonical) {
  // tree_pm_coupling.cpp:164-175
  double v = canonical ? x : x - L * floor(x / L);
  if (v >= L) v = 0.0;
  else if (v < 0.0) v += L;
  if (v == 0.0) v = 0.0;
  return v;
}

// ---------------------------------------------------------------------------
// Source statistics: per-axis min/max (order keys), finiteness and mass checks.
struct SourceStats {
  uint64_t lo[3];
  uint64_t hi[3];
  uint32_t bad_coord;
  uint32_t bad_mass;
  uint32_t mass_nonuniform;
  uint32_t pad;
  double mass0;  // m[0] (the uniform mass when every mass equals it)
};

// Each block writes its partial statistics to part[blockIdx.x]; one block then
// folds the partials (same-address atomics from every block would serialise
// at the L2, about 75 us for 1024 blocks whatever n is).
__global__ __launch_bounds__(256) void source_stats_kernel(Axes3 p, const double* __restrict__ m, std::size_t n,
                                                           SourceStats* __restrict__ part) {
  uint64_t lo[3] = {kEmpty, kEmpty, kEmpty}, hi[3] = {0, 0, 0};
  uint32_t bc = 0, bm = 0, nu = 0;
  const double m0 = (m != nullptr && n > 0) ? m[0] : 0.0;
  auto take = [&](const double* v, double mm) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      if (!isfinite(v[a])) {
        bc = 1;
      } else {
        const uint64_t k = order_key(v[a]);
        lo[a] = k < lo[a] ? k : lo[a];
        hi[a] = k > hi[a] ? k : hi[a];
      }
    }
    if (m != nullptr) {
      if (!(isfinite(mm) && mm >= 0.0)) bm = 1;
      if (mm != m0) nu = 1;
    }
  };
  const std::size_t stride = static_cast<std::size_t>(gridDim.x) * blockDim.x;
  std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  constexpr int kU = 4;  // loads of kU elements in flight per thread
  for (; i + (kU - 1) * stride < n; i += kU * stride) {
    double v[kU][3], mm[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
#pragma unroll
      for (int a = 0; a < 3; ++a) v[u][a] = p.p[a][i + u * stride];
      mm[u] = m != nullptr ? m[i + u * stride] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) take(v[u], mm[u]);
  }
  for (; i < n; i += stride) {
    const double v[3] = {p.p[0][i], p.p[1][i], p.p[2][i]};
    take(v, m != nullptr ? m[i] : 0.0);
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    lo[a] = wave_min(lo[a]);
    hi[a] = wave_max(hi[a]);
  }
  bc = wave_max(bc);
  bm = wave_max(bm);
  nu = wave_max(nu);
  // block reduction, then one set of atomics per block (few blocks)
  __shared__ uint64_t slo[4][3], shi[4][3];
  __shared__ uint32_t sflag[4][3];
  const int w = threadIdx.x / kWave;
  if (lane_id() == 0) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      slo[w][a] = lo[a];
      shi[w][a] = hi[a];
    }
    sflag[w][0] = bc;
    sflag[w][1] = bm;
    sflag[w][2] = nu;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int v = 1; v < static_cast<int>(blockDim.x) / kWave; ++v) {
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        lo[a] = slo[v][a] < lo[a] ? slo[v][a] : lo[a];
        hi[a] = shi[v][a] > hi[a] ? shi[v][a] : hi[a];
      }
      bc |= sflag[v][0];
      bm |= sflag[v][1];
      nu |= sflag[v][2];
    }
    SourceStats r;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      r.lo[a] = lo[a];
      r.hi[a] = hi[a];
    }
    r.bad_coord = bc;
    r.bad_mass = bm;
    r.mass_nonuniform = nu;
    r.pad = 0u;
    part[blockIdx.x] = r;
  }
}

__global__ __launch_bounds__(256) void stats_final_kernel(const SourceStats* __restrict__ part, uint32_t nb,
                                                          const double* __restrict__ m, SourceStats* __restrict__ st) {
  uint64_t lo[3] = {kEmpty, kEmpty, kEmpty}, hi[3] = {0, 0, 0};
  uint32_t bc = 0, bm = 0, nu = 0;
  for (uint32_t b = threadIdx.x; b < nb; b += blockDim.x) {
    const SourceStats& q = part[b];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      lo[a] = q.lo[a] < lo[a] ? q.lo[a] : lo[a];
      hi[a] = q.hi[a] > hi[a] ? q.hi[a] : hi[a];
    }
    bc |= q.bad_coord;
    bm |= q.bad_mass;
    nu |= q.mass_nonuniform;
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    lo[a] = wave_min(lo[a]);
    hi[a] = wave_max(hi[a]);
  }
  bc = wave_max(bc);
  bm = wave_max(bm);
  nu = wave_max(nu);
  __shared__ SourceStats sw[256 / kWave];
  const int w = threadIdx.x / kWave;
  if (lane_id() == 0) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      sw[w].lo[a] = lo[a];
      sw[w].hi[a] = hi[a];
    }
    sw[w].bad_coord = bc;
    sw[w].bad_mass = bm;
    sw[w].mass_nonuniform = nu;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    SourceStats r = sw[0];
    for (int v = 1; v < static_cast<int>(blockDim.x) / kWave; ++v) {
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        r.lo[a] = sw[v].lo[a] < r.lo[a] ? sw[v].lo[a] : r.lo[a];
        r.hi[a] = sw[v].hi[a] > r.hi[a] ? sw[v].hi[a] : r.hi[a];
      }
      r.bad_coord |= sw[v].bad_coord;
      r.bad_mass |= sw[v].bad_mass;
      r.mass_nonuniform |= sw[v].mass_nonuniform;
    }
    r.pad = 0u;
    r.mass0 = m ? m[0] : 0.0;
    *st = r;
  }
}

// ---------------------------------------------------------------------------
// Periodic unwrap (tree_pm_coupling.cpp:141-218) without a sort.
// Values are binned into B >= 2n buckets of width w = L/B. The largest
// circular gap is >= L/n = 2w, while two values in one bucket differ by less
// than w (up to rounding), so the largest gap, and every gap tying with it,
// runs from the maximum of an occupied bucket p to the minimum of the next
// occupied bucket i. If e = i - p - 1 empty buckets lie between them, the gap
// is within (e w, (e + 2) w) up to rounding of the bucket computation, so only
// runs with e >= R - 2 (R the longest empty run) can hold the largest gap.
// Steps per axis: an occupancy bitmap (one byte store per value, packed); R from a scan
// of the bitmap; the end buckets of candidate runs and their predecessors are
// marked; exact FP64 min/max (IEEE bits; non-negative doubles order like their
// bits) are gathered only for marked buckets, ranked by a popcount scan; the
// candidate gaps are evaluated with the reference's tie rule (smaller anchor).
struct BucketArgs {
  double L[3];
  double scale[3];  // B / L
  int canonical[3];
  int naxes;
  uint64_t B;       // multiple of 32
  uint64_t W;       // B / 32 bitmap words per axis
};

// The per-build values that a capture-safe build keeps on the device instead
// of reading them back: the canonical flags (from the source statistics), the
// unwrap anchors, the root cube and the in-leaf Morton frame (from the unwrap
// result). Kernels given a Frame take these fields from it.
struct Frame {
  int canonical[3];
  int pad;
  double anchor[3];
  double centre[3];
  double half;
  double mlo[3];
  double mext;
};

__device__ __forceinline__ uint64_t bucket_of(double v, const BucketArgs& a, int ax) {
  uint64_t b = static_cast<uint64_t>(v * a.scale[ax]);
  return b >= a.B ? a.B - 1 : b;
}

// Occupancy as one byte per bucket: every value stores 1 into its bucket's
// byte. The stores are idempotent, so they need no atomics (a device-scope
// atomic per value and axis ran at about 1e10 per second, scattered); a
// coalesced pass then packs 32 bytes into each bitmap word.
__global__ __launch_bounds__(256) void occupancy_bytes_kernel(Axes3 p, std::size_t n, BucketArgs a,
                                                              uint8_t* __restrict__ occb,
                                                              const Frame* __restrict__ fr) {
  if (fr)
    for (int ax = 0; ax < 3; ++ax) a.canonical[ax] = fr->canonical[ax];
  for (std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<std::size_t>(gridDim.x) * blockDim.x) {
    for (int ax = 0; ax < a.naxes; ++ax)
      occb[ax * a.B + bucket_of(wrap_coord(p.p[ax][i], a.L[ax], a.canonical[ax]), a, ax)] = 1u;
  }
}

__global__ __launch_bounds__(256) void occupancy_pack_kernel(const uint8_t* __restrict__ occb, std::size_t words,
                                                             uint32_t* __restrict__ occ) {
  const std::size_t wi = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (wi >= words) return;
  const uint4* src = reinterpret_cast<const uint4*>(occb + 32 * wi);
  const uint4 b0 = src[0], b1 = src[1];
  const uint32_t q[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
  uint32_t bits = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
#pragma unroll
    for (int c = 0; c < 4; ++c) bits |= ((q[k] >> (8 * c)) & 1u) << (4 * k + c);
  }
  occ[wi] = bits;
}

// Exact min/max (IEEE bits, max stored +1 so 0 = empty) of the marked buckets.
__global__ __launch_bounds__(256) void marked_minmax_kernel(Axes3 p, std::size_t n, BucketArgs a,
                                                            const uint32_t* __restrict__ mark,
                                                            const uint32_t* __restrict__ rank_base,
                                                            uint64_t* __restrict__ cmin, uint64_t* __restrict__ cmax,
                                                            const Frame* __restrict__ fr) {
  if (fr)
    for (int ax = 0; ax < 3; ++ax) a.canonical[ax] = fr->canonical[ax];
  for (std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<std::size_t>(gridDim.x) * blockDim.x) {
    for (int ax = 0; ax < a.naxes; ++ax) {
      const double v = wrap_coord(p.p[ax][i], a.L[ax], a.canonical[ax]);
      const uint64_t b = bucket_of(v, a, ax);
      const uint64_t wi = ax * a.W + (b >> 5);
      const uint32_t mw = mark[wi];
      const uint32_t bit = 1u << (b & 31);
      if (mw & bit) {
        const uint32_t r = rank_base[wi] + __popc(mw & (bit - 1u));
        const uint64_t bits = dbits(v);
        atomicMin(reinterpret_cast<unsigned long long*>(&cmin[r]), bits);
        atomicMax(reinterpret_cast<unsigned long long*>(&cmax[r]), bits + 1);
      }
    }
  }
}

__global__ __launch_bounds__(256) void popc_kernel(const uint32_t* __restrict__ w, std::size_t nw,
                                                   uint32_t* __restrict__ out) {
  const std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < nw) out[i] = __popc(w[i]);
}

constexpr int kGapThreads = 256;
constexpr int kGapItems = 2;  // 8 left the walks of small boxes to a block per axis (17 us a pass)
constexpr int kGapTile = kGapThreads * kGapItems;

__device__ __forceinline__ uint64_t block_max_u64(uint64_t v) {
  __shared__ uint64_t wmax[kGapThreads / kWave];
  v = wave_max(v);
  if (lane_id() == 0) wmax[threadIdx.x / kWave] = v;
  __syncthreads();
  uint64_t r = 0;
#pragma unroll
  for (int i = 0; i < kGapThreads / kWave; ++i) r = wmax[i] > r ? wmax[i] : r;
  __syncthreads();
  return r;
}

// Exclusive max-scan over the block (blocked thread order); returns the
// exclusive prefix for this thread and the block total.
__device__ __forceinline__ uint64_t block_excl_max_u64(uint64_t v, uint64_t* total) {
  __shared__ uint64_t wtot[kGapThreads / kWave];
  const int lane = lane_id(), w = threadIdx.x / kWave;
  uint64_t inc = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint64_t o = __shfl_up(inc, off, kWave);
    if (lane >= off) inc = o > inc ? o : inc;
  }
  uint64_t excl = __shfl_up(inc, 1, kWave);
  if (lane == 0) excl = 0;
  if (lane == kWave - 1) wtot[w] = inc;
  __syncthreads();
  uint64_t woff = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < kGapThreads / kWave; ++i) {
    if (i < w) woff = wtot[i] > woff ? wtot[i] : woff;
    tot = wtot[i] > tot ? wtot[i] : tot;
  }
  __syncthreads();
  *total = tot;
  return excl > woff ? excl : woff;
}

// Per block of kGapTile bitmap words: 1 + the last occupied bucket (0 if none).
__global__ __launch_bounds__(kGapThreads) void occ_blockmax_kernel(const uint32_t* __restrict__ occ, uint64_t W,
                                                                   uint64_t* __restrict__ blockmax, uint64_t nblk) {
  const int ax = blockIdx.y;
  const uint64_t base = static_cast<uint64_t>(blockIdx.x) * kGapTile;
  uint64_t mx = 0;
#pragma unroll
  for (int k = 0; k < kGapItems; ++k) {
    const uint64_t wi = base + static_cast<uint64_t>(k) * kGapThreads + threadIdx.x;
    if (wi < W) {
      const uint32_t v = occ[ax * W + wi];
      if (v) {
        const uint64_t last = wi * 32 + 31 - __clz(v);
        mx = last + 1 > mx ? last + 1 : mx;
      }
    }
  }
  mx = block_max_u64(mx);
  if (threadIdx.x == 0) blockmax[ax * nblk + blockIdx.x] = mx;
}

// One block per axis: exclusive max-scan of the block maxima in place.
__global__ __launch_bounds__(kGapThreads) void blockmax_scan_kernel(uint64_t* blockmax, uint64_t nblk,
                                                                    uint64_t* total) {
  const int ax = blockIdx.x;
  uint64_t carry = 0;
  for (uint64_t c = 0; c < nblk; c += kGapThreads) {
    const uint64_t idx = c + threadIdx.x;
    const uint64_t v = idx < nblk ? blockmax[ax * nblk + idx] : 0;
    uint64_t tot;
    uint64_t ex = block_excl_max_u64(v, &tot);
    ex = ex > carry ? ex : carry;
    if (idx < nblk) blockmax[ax * nblk + idx] = ex;
    carry = tot > carry ? tot : carry;
  }
  if (threadIdx.x == 0) total[ax] = carry;
}

struct GapBest {
  double gap;
  double anchor;
  double umax;  // largest unwrapped coordinate if this gap is chosen
  int valid;
  int pad;
};

__device__ __forceinline__ bool better(const GapBest& a, const GapBest& b) {
  if (!a.valid) return false;
  if (!b.valid) return true;
  if (a.gap > b.gap) return true;
  if (a.gap == b.gap && a.anchor < b.anchor) return true;
  return false;
}

__device__ __forceinline__ GapBest shfl_best(const GapBest& v, int src) {
  GapBest r;
  r.gap = __shfl(v.gap, src, kWave);
  r.anchor = __shfl(v.anchor, src, kWave);
  r.umax = __shfl(v.umax, src, kWave);
  r.valid = __shfl(v.valid, src, kWave);
  r.pad = 0;
  return r;
}

__device__ GapBest block_best(GapBest b) {
  __shared__ GapBest wb[kGapThreads / kWave];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const GapBest o = shfl_best(b, lane_id() ^ off);
    if (better(o, b)) b = o;
  }
  if (lane_id() == 0) wb[threadIdx.x / kWave] = b;
  __syncthreads();
  GapBest r = wb[0];
  for (int i = 1; i < kGapThreads / kWave; ++i)
    if (better(wb[i], r)) r = wb[i];
  __syncthreads();
  return r;
}

// Walks the occupied buckets of a block's words in order. For each occupied
// bucket i it knows its predecessor p (the previous occupied bucket, or for the
// first one the last occupied bucket minus B: the wrap) and the empty run
// e = i - p - 1. MODE 0: the longest run per axis (atomicMax). MODE 1: marks
// the end buckets of runs with e >= R - 2 and their predecessors. MODE 2:
// evaluates the marked gaps from the exact min/max and keeps the best per block.
struct RunArgs {
  const uint32_t* occ;
  const uint64_t* block_prefix;  // exclusive max-scan of the block maxima
  const uint64_t* total;         // 1 + last occupied bucket, per axis
  unsigned long long* longest;   // per axis (MODE 0 writes, MODE 1 reads)
  uint32_t* mark;                // MODE 1 writes
  uint32_t* ends;                // MODE 1 writes
  const uint32_t* rank_base;     // MODE 2
  const uint64_t* cmin;          // MODE 2
  const uint64_t* cmax;          // MODE 2
  GapBest* block_out;            // MODE 2
  uint64_t nblk;
};

template <int MODE>
__global__ __launch_bounds__(kGapThreads) void runs_kernel(BucketArgs a, RunArgs r) {
  const int ax = blockIdx.y;
  const uint64_t W = a.W, B = a.B;
  const uint64_t wbase = static_cast<uint64_t>(blockIdx.x) * kGapTile + static_cast<uint64_t>(threadIdx.x) * kGapItems;
  // 1 + last occupied bucket among this thread's words
  uint64_t tmax = 0;
  uint32_t words[kGapItems];
#pragma unroll
  for (int k = 0; k < kGapItems; ++k) {
    const uint64_t wi = wbase + k;
    words[k] = wi < W ? r.occ[ax * W + wi] : 0u;
    if (words[k]) {
      const uint64_t last = wi * 32 + 31 - __clz(words[k]);
      tmax = last + 1 > tmax ? last + 1 : tmax;
    }
  }
  uint64_t tot;
  uint64_t run = block_excl_max_u64(tmax, &tot);
  const uint64_t bp = r.block_prefix[ax * r.nblk + blockIdx.x];
  run = run > bp ? run : bp;
  const uint64_t last_all = r.total[ax] - 1;  // last occupied bucket of the axis
  const unsigned long long R = MODE == 1 ? r.longest[ax] : 0ull;
  const double L = a.L[ax];
  uint64_t longest = 0;
  GapBest best{0.0, 0.0, 0.0, 0, 0};
  const auto rank_of = [&](uint64_t b) -> uint32_t {
    const uint64_t wi = ax * W + (b >> 5);
    const uint32_t bit = 1u << (b & 31);
    return r.rank_base[wi] + __popc(r.mark[wi] & (bit - 1u));
  };
  for (int k = 0; k < kGapItems; ++k) {
    uint32_t v = words[k];
    const uint64_t wi = wbase + k;
    uint32_t endbits = 0;
    while (v) {
      const int bitpos = __ffs(v) - 1;
      v &= v - 1;
      const uint64_t i = wi * 32 + bitpos;
      // run == 0: first occupied bucket; its predecessor is the last one, across the wrap
      const uint64_t e = run == 0 ? (B - 1 - last_all) + i : i - run;  // run = 1 + predecessor
      if (MODE == 0) {
        longest = e > longest ? e : longest;
      } else if (MODE == 1) {
        if (e + 2 >= R) {
          endbits |= 1u << bitpos;
          const uint64_t pb = run == 0 ? last_all : run - 1;
          atomicOr(&r.mark[ax * W + (pb >> 5)], 1u << (pb & 31));
          atomicOr(&r.mark[ax * W + (i >> 5)], 1u << (i & 31));
        }
      } else {
        if ((r.ends[ax * W + wi] >> bitpos) & 1u) {
          const double vmin = bitsd(r.cmin[rank_of(i)]);
          GapBest c;
          c.valid = 1;
          c.pad = 0;
          c.anchor = vmin;
          if (run == 0) {
            const double gmax = bitsd(r.cmax[rank_of(last_all)] - 1);
            c.gap = (vmin + L) - gmax;
            c.umax = gmax;
          } else {
            const double pr = bitsd(r.cmax[rank_of(run - 1)] - 1);
            c.gap = vmin - pr;
            c.umax = pr + L;
          }
          if (better(c, best)) best = c;
        }
      }
      run = i + 1;
    }
    if (MODE == 1 && endbits) r.ends[ax * W + wi] = endbits;
  }
  if (MODE == 0) {
    longest = wave_max(longest);
    if (lane_id() == 0 && longest) atomicMax(&r.longest[ax], static_cast<unsigned long long>(longest));
  } else if (MODE == 2) {
    best = block_best(best);
    if (threadIdx.x == 0) r.block_out[ax * r.nblk + blockIdx.x] = best;
  }
}

__global__ __launch_bounds__(kGapThreads) void gap_final_kernel(const GapBest* __restrict__ block_out, uint64_t nblk,
                                                                UnwrapResult* res) {
  const int ax = blockIdx.x;
  GapBest best{0.0, 0.0, 0.0, 0, 0};
  for (uint64_t i = threadIdx.x; i < nblk; i += kGapThreads) {
    const GapBest c = block_out[ax * nblk + i];
    if (better(c, best)) best = c;
  }
  best = block_best(best);
  if (threadIdx.x == 0) {
    res->anchor[ax] = best.anchor;
    res->umin[ax] = best.anchor;
    res->umax[ax] = best.umax;
  }
}

// ---------------------------------------------------------------------------
// Keys.
__device__ __forceinline__ uint64_t expand21(uint32_t v) {
  uint64_t x = v & 0x1FFFFFu;
  x = (x | (x << 32)) & 0x1F00000000FFFFull;
  x = (x | (x << 16)) & 0x1F0000FF0000FFull;
  x = (x | (x << 8)) & 0x100F00F00F00F00Full;
  x = (x | (x << 4)) & 0x10C30C30C30C30C3ull;
  x = (x | (x << 2)) & 0x1249249249249249ull;
  return x;
}

struct MortonArgs {
  double lo[3];
  double extent;  // max(max extent, 1e-12)  (tree_ordering.cpp:151)
};

// tree_ordering.cpp:159-167: clamp((x-min)/extent,0,1) * (2^21-1), llround.
__device__ __forceinline__ uint64_t morton_key(double x, double y, double z, const MortonArgs& a) {
  const double grid = 2097151.0;
  const double nx = fmin(fmax((x - a.lo[0]) / a.extent, 0.0), 1.0);
  const double ny = fmin(fmax((y - a.lo[1]) / a.extent, 0.0), 1.0);
  const double nz = fmin(fmax((z - a.lo[2]) / a.extent, 0.0), 1.0);
  const uint32_t qx = static_cast<uint32_t>(llround(nx * grid));
  const uint32_t qy = static_cast<uint32_t>(llround(ny * grid));
  const uint32_t qz = static_cast<uint32_t>(llround(nz * grid));
  return (expand21(qx) << 2) | (expand21(qy) << 1) | expand21(qz);
}

__device__ __forceinline__ double unwrap_coord(double x, double L, int canonical, double anchor) {
  const double v = wrap_coord(x, L, canonical);
  return v < anchor ? v + L : v;
}

struct PathArgs {
  UnwrapArgs u;
  double c0[3];
  double h0;
};

// 21-level octant path of every particle against the reference's FP64 centres.
// Also writes the sources in input order as canonical coordinates and mass
// (double4), so that the tree-order gather reads one 32-byte record per source.
__global__ __launch_bounds__(256) void path_key_kernel(Axes3 p, const double* __restrict__ m, std::size_t n,
                                                       PathArgs a, uint64_t* __restrict__ keys,
                                                       uint32_t* __restrict__ vals, double4* __restrict__ packed,
                                                       const Frame* __restrict__ fr) {
  const std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (fr) {
    for (int ax = 0; ax < 3; ++ax) {
      a.u.canonical[ax] = fr->canonical[ax];
      a.u.anchor[ax] = fr->anchor[ax];
      a.c0[ax] = fr->centre[ax];
    }
    a.h0 = fr->half;
  }
  double x = p.p[0][i], y = p.p[1][i], z = p.p[2][i];
  if (fr) {
    // a capture-safe build reports non-finite coordinates through the fault
    // word and carries on; zeros keep every later cell index in range
    x = isfinite(x) ? x : 0.0;
    y = isfinite(y) ? y : 0.0;
    z = isfinite(z) ? z : 0.0;
  }
  packed[i] = make_double4(wrap_coord(x, a.u.L[0], a.u.canonical[0]), wrap_coord(y, a.u.L[1], a.u.canonical[1]),
                           wrap_coord(z, a.u.L[2], a.u.canonical[2]), m[i]);
  const double ux = unwrap_coord(x, a.u.L[0], a.u.canonical[0], a.u.anchor[0]);
  const double uy = unwrap_coord(y, a.u.L[1], a.u.canonical[1], a.u.anchor[1]);
  const double uz = unwrap_coord(z, a.u.L[2], a.u.canonical[2], a.u.anchor[2]);
  double cx = a.c0[0], cy = a.c0[1], cz = a.c0[2], h = a.h0;
  uint64_t key = 0;
  for (int lvl = 0; lvl < kPathLevels; ++lvl) {
    const uint32_t ox = ux >= cx ? 1u : 0u, oy = uy >= cy ? 1u : 0u, oz = uz >= cz ? 1u : 0u;
    key = (key << 3) | (ox << 2) | (oy << 1) | oz;
    const double ch = 0.5 * h;
    cx = cx + (ox ? ch : -ch);
    cy = cy + (oy ? ch : -ch);
    cz = cz + (oz ? ch : -ch);
    h = ch;
  }
  keys[i] = key;
  vals[i] = static_cast<uint32_t>(i);
}

__global__ __launch_bounds__(256) void morton_keys_kernel(Axes3 p, std::size_t n, MortonArgs a,
                                                          uint64_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  keys[i] = morton_key(p.p[0][i], p.p[1][i], p.p[2][i], a);
  vals[i] = static_cast<uint32_t>(i);
}

// unwrap_coord of a canonical coordinate
__device__ __forceinline__ double unwrap_canonical(double v, double anchor, double L) {
  return v < anchor ? v + L : v;
}

// ---------------------------------------------------------------------------
// Octree from the sorted path keys, without a pass per level.
//
// Let cl(i) be the number of octant digits that the keys of particles i - 1
// and i share (-1 for i = 0), and ld(i) the depth of particle i's leaf. A cell
// of depth d holds more than leaf_size particles around i exactly when two
// sorted keys leaf_size apart, at and around i, share d digits, so
//   ld(i) = 1 + max over j in [i - leaf_size, i] of common(j, j + leaf_size),
// capped by the depth whose cells reach the smallest half size
// (tree_gravity.cpp:1133). The nodes that begin at particle i are those of
// depths cl(i) + 1 .. ld(i). Preorder is the order of (begin, depth), so one
// scan of the counts ld - cl numbers the nodes in preorder; a scan per depth
// numbers them breadth first, a node's children being consecutive and its
// first child the next depth's node at the same particle. A node ends at the
// first later key outside its cell, which also gives its subtree size. The
// former discovery took three launches per level to split the nodes and two
// more for subtree sizes and preorder (60 to 75 launches of 4 to 40 us).
// meta = depth | octant << 8 | leaf << 16 | last sibling << 17
constexpr int kMaxLevels = kPathLevels + 1;             // depths 0..21
constexpr int kLvTooDeep = kMaxLevels + 1;              // lv[0, kMaxLevels]: level starts
constexpr int kLvOverflow = kLvTooDeep + 1;             // nodes beyond the node capacity
constexpr int kLvDeepSplit = kLvTooDeep + 2;            // a node below the partial sort's depth splits
constexpr int kLvLeaves = kLvTooDeep + 3;               // nodes without children
constexpr int kLvTotal = kLvTooDeep + 4;                // node count
constexpr int kLvDepth = kLvTooDeep + 5;                // deepest level with nodes
constexpr int kLvSubs = kLvTooDeep + 6;                 // moment subtrees
constexpr int kLvTops = kLvTooDeep + 7;                 // per depth: nodes above the moment subtrees
constexpr int kLvWords = kLvTops + kMaxLevels;

constexpr int kNodeThreads = 512;                       // particles per block of the node passes
constexpr int kNodeRows = kMaxLevels + 1;               // per-block counts: nodes of each depth, all nodes
constexpr uint32_t kMaxLeafSize = 1024;

// What a build reads back: the level words, and with a device frame the source
// statistics and the unwrap result.
struct BuildReport {
  uint32_t lv[kLvWords];
  uint32_t pad;
  SourceStats stats;
  UnwrapResult unwrap;
};

struct NodeArgs {
  uint32_t n, leaf_size;
  int sorted_levels;   // digits the keys are sorted by
  uint32_t nblk;       // blocks of kNodeThreads particles
  double c0[3], h0;    // root cube (unless a frame is given)
  uint32_t capacity;   // node arrays
  uint32_t cut;        // moment subtrees hold at most this many particles
  uint32_t max_top;    // nodes of one depth above them, at most
};

// octant digits two keys share, at most `levels`
__device__ __forceinline__ int common_digits(uint64_t a, uint64_t b, int levels) {
  const uint64_t x = a ^ b;
  const int c = x == 0 ? kPathLevels : (__clzll(static_cast<long long>(x)) - 1) / 3;
  return c < levels ? c : levels;
}

// depth whose cells have half <= 1e-12 (they are leaves whatever they hold), or kMaxLevels
__device__ __forceinline__ int smallest_cell_depth(double half) {
  int d = 0;
  while (d < kMaxLevels && !(half <= 1.0e-12)) {
    half = 0.5 * half;
    ++d;
  }
  return d;
}

// cl + 1 and ld of every particle (cld = cl + 1 | ld << 8), and per block the
// node counts of each depth and in all (cnt[row * nblk + block]).
__global__ __launch_bounds__(kNodeThreads) void node_count_kernel(NodeArgs a, const uint64_t* __restrict__ keys,
                                                                  uint16_t* __restrict__ cld,
                                                                  uint32_t* __restrict__ cnt,
                                                                  uint32_t* __restrict__ flags,
                                                                  const Frame* __restrict__ fr) {
  __shared__ int win[2][kNodeThreads + kMaxLeafSize];
  __shared__ uint32_t hist[kNodeRows];
  __shared__ uint32_t leaves;
  const int t = threadIdx.x;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kNodeThreads;
  const int leaf = static_cast<int>(a.leaf_size), len = kNodeThreads + leaf;
  if (t < kNodeRows) hist[t] = 0;
  if (t == 0) leaves = 0;
  for (int k = t; k < len; k += kNodeThreads) {
    const int64_t j = base - leaf + k;
    win[0][k] = j >= 0 && j + leaf < static_cast<int64_t>(a.n)
                    ? common_digits(keys[j], keys[j + leaf], a.sorted_levels)
                    : -1;
  }
  __syncthreads();
  // maxima over 2, 4, .. entries while they fit the window of leaf + 1
  int cur = 0, span = 1;
  while (2 * span <= leaf + 1) {
    for (int k = t; k < len; k += kNodeThreads) {
      const int v = win[cur][k], o = k + span < len ? win[cur][k + span] : -1;
      win[cur ^ 1][k] = v > o ? v : o;
    }
    cur ^= 1;
    span *= 2;
    __syncthreads();
  }
  const int64_t i = base + t;
  const bool in = i < static_cast<int64_t>(a.n);
  const int s0 = win[cur][t], s1 = win[cur][t + leaf + 1 - span];
  const int split = s0 > s1 ? s0 : s1;  // deepest cell around i with more than leaf_size particles
  const int cap = smallest_cell_depth(fr ? fr->half : a.h0);
  int cl = -1, ld = -1;
  bool deep = false, too = false;
  if (in) {
    cl = i == 0 ? -1 : common_digits(keys[i - 1], keys[i], a.sorted_levels);
    ld = split + 1 < cap ? split + 1 : cap;
    if (split >= a.sorted_levels && cap > a.sorted_levels) {
      deep = a.sorted_levels < kPathLevels;
      too = !deep;
      ld = a.sorted_levels;
    }
    cld[i] = static_cast<uint16_t>((cl + 1) | (ld << 8));
  }
  if (__ballot(deep) && lane_id() == 0) atomicOr(&flags[kLvDeepSplit], 1u);
  if (__ballot(too) && lane_id() == 0) atomicOr(&flags[kLvTooDeep], 1u);
  const int dmax = static_cast<int>(wave_max_u32(static_cast<uint32_t>(ld + 1))) - 1;
  uint32_t all = 0;
  for (int d = 0; d <= dmax; ++d) {
    const uint32_t c = static_cast<uint32_t>(__popcll(__ballot(in && cl < d && d <= ld)));
    all += c;
    if (c && lane_id() == 0) atomicAdd(&hist[d], c);
  }
  const uint32_t lf = static_cast<uint32_t>(__popcll(__ballot(in && cl < ld)));
  if (lane_id() == 0) {
    if (all) atomicAdd(&hist[kMaxLevels], all);
    if (lf) atomicAdd(&leaves, lf);
  }
  __syncthreads();
  if (t < kNodeRows) cnt[static_cast<std::size_t>(t) * a.nblk + blockIdx.x] = hist[t];
  if (t == 0 && leaves) atomicAdd(&flags[kLvLeaves], leaves);
}

// Level starts, node count and deepest level from the row totals; the report
// of the build. A capture-safe build reads nothing back: a tree beyond the
// prepared capacity or sorted depth, or deeper than 21 levels, sets fault bits
// and becomes empty.
__global__ __launch_bounds__(64) void node_levels_kernel(NodeArgs a, const uint32_t* __restrict__ totals,
                                                         BuildReport* __restrict__ rep,
                                                         const SourceStats* __restrict__ stats,
                                                         const UnwrapResult* __restrict__ unwrap,
                                                         unsigned long long* __restrict__ fault) {
  const int t = threadIdx.x;
  uint32_t* lv = rep->lv;
  if (t < kMaxLevels) lv[kLvTops + t] = 0;
  if (t != 0) return;
  uint32_t run = 0, depth = 0;
  for (int d = 0; d < kMaxLevels; ++d) {
    lv[d] = run;
    if (totals[d]) depth = static_cast<uint32_t>(d);
    run += totals[d];
  }
  lv[kMaxLevels] = run;
  lv[kLvTotal] = run;
  lv[kLvDepth] = depth;
  lv[kLvSubs] = 0;
  lv[kLvOverflow] = run > a.capacity ? 1u : 0u;
  if (stats) rep->stats = *stats;
  if (unwrap) rep->unwrap = *unwrap;
  if (fault) {
    unsigned long long f = 0;
    if (lv[kLvOverflow] || lv[kLvDeepSplit]) f |= kFaultPrepared;
    if (lv[kLvTooDeep]) f |= kFaultTooDeep;
    if (f) {
      for (int d = 0; d <= kMaxLevels; ++d) lv[d] = 0;
      lv[kLvTotal] = 0;
      atomicOr(fault, f);
    }
  }
}

struct NodeArrays {
  uint32_t *begin, *count, *first_child, *nchild, *meta, *pre, *subtree;
  double4* geo;
};

// Writes the nodes that begin at each particle (breadth-first slots): begin,
// depth and octant, preorder index, cell, first child. The cell is the root's
// halved along the key's digits, the arithmetic of the path keys.
__global__ __launch_bounds__(kNodeThreads) void node_emit_kernel(NodeArgs a, const uint64_t* __restrict__ keys,
                                                                 const uint16_t* __restrict__ cld,
                                                                 const uint32_t* __restrict__ offs,
                                                                 const uint32_t* __restrict__ lv, NodeArrays o,
                                                                 uint32_t* __restrict__ pbase,
                                                                 const Frame* __restrict__ fr) {
  __shared__ uint32_t wcnt[kNodeThreads / kWave][kNodeRows];
  __shared__ uint32_t start[kNodeRows];
  if (lv[kLvTotal] == 0 || lv[kLvTotal] > a.capacity) return;  // block-uniform
  const int t = threadIdx.x, w = t / kWave, lane = lane_id();
  const uint32_t i = blockIdx.x * kNodeThreads + t;
  const bool in = i < a.n;
  int cl = -1, ld = -2;
  uint64_t key = 0;
  if (in) {
    const uint32_t v = cld[i];
    cl = static_cast<int>(v & 0xFFu) - 1;
    ld = static_cast<int>(v >> 8);
    key = keys[i];
  }
  const int dmax = static_cast<int>(wave_max_u32(static_cast<uint32_t>(ld + 2))) - 2;
  if (t < kNodeRows) {
    start[t] = (t < kMaxLevels ? lv[t] : 0u) + offs[static_cast<std::size_t>(t) * a.nblk + blockIdx.x];
  }
  if (lane < kNodeRows) wcnt[w][lane] = 0;
  __builtin_amdgcn_wave_barrier();
  const uint32_t mine = in && ld > cl ? static_cast<uint32_t>(ld - cl) : 0u;
  for (int d = 0; d <= dmax; ++d) {
    const uint32_t c = static_cast<uint32_t>(__popcll(__ballot(in && cl < d && d <= ld)));
    if (lane == 0) wcnt[w][d] = c;
  }
  uint32_t inc = mine;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint32_t u = __shfl_up(inc, off, kWave);
    if (lane >= off) inc += u;
  }
  if (lane == kWave - 1) wcnt[w][kMaxLevels] = inc;
  __syncthreads();
  uint32_t pb = start[kMaxLevels] + inc - mine;
  for (int k = 0; k < w; ++k) pb += wcnt[k][kMaxLevels];
  if (in) pbase[i] = pb;
  double cx, cy, cz, h;
  if (fr) {
    cx = fr->centre[0];
    cy = fr->centre[1];
    cz = fr->centre[2];
    h = fr->half;
  } else {
    cx = a.c0[0];
    cy = a.c0[1];
    cz = a.c0[2];
    h = a.h0;
  }
  uint32_t prev = kInvalidIndex;  // this particle's node one depth up
  for (int d = 0; d <= dmax; ++d) {
    const bool on = in && cl < d && d <= ld;
    uint32_t oct = 0;
    if (d > 0) {
      oct = static_cast<uint32_t>(key >> (3 * (kPathLevels - d))) & 7u;
      const double ch = 0.5 * h;
      cx = cx + ((oct & 4u) ? ch : -ch);
      cy = cy + ((oct & 2u) ? ch : -ch);
      cz = cz + ((oct & 1u) ? ch : -ch);
      h = ch;
    }
    const unsigned long long m = __ballot(on);
    if (m == 0) continue;
    uint32_t slot = start[d] + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                                         __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u));
    for (int k = 0; k < w; ++k) slot += wcnt[k][d];
    if (on) {
      o.begin[slot] = i;
      o.meta[slot] = static_cast<uint32_t>(d) | (oct << 8) | (d == ld ? 1u << 16 : 0u) | (d == 0 ? 1u << 17 : 0u);
      o.pre[slot] = pb + static_cast<uint32_t>(d - cl - 1);
      o.geo[slot] = make_double4(cx, cy, cz, h);
      if (d == ld) o.first_child[slot] = kInvalidIndex;
      if (prev != kInvalidIndex) o.first_child[prev] = slot;
      prev = slot;
    }
  }
}

// Per node: particle count, subtree size, child count and the last child's
// mark; the moment passes' work lists: subtrees of at most a.cut particles
// whose parent holds more, and the nodes above them by depth.
__global__ __launch_bounds__(256) void node_links_kernel(NodeArgs a, const uint64_t* __restrict__ keys,
                                                         uint32_t* __restrict__ lv, NodeArrays o,
                                                         const uint32_t* __restrict__ pbase,
                                                         uint32_t* __restrict__ subs, uint32_t* __restrict__ tops) {
  const uint32_t total = lv[kLvTotal];
  if (total > a.capacity) return;
  for (uint32_t b = blockIdx.x * blockDim.x + threadIdx.x; b < total; b += gridDim.x * blockDim.x) {
    const uint32_t i = o.begin[b], meta = o.meta[b];
    const int d = static_cast<int>(meta & 0xFFu);
    const bool leaf = (meta >> 16) & 1u;
    uint32_t end = a.n;
    if (d > 0) {
      const int sh = 3 * (kPathLevels - d);
      const uint64_t cell = keys[i] >> sh;
      // keys[lo] is in the cell, keys[hi] is not (or hi = n)
      uint32_t lo = i, step = a.leaf_size < 16u ? a.leaf_size : 16u;
      uint32_t hi = i + step < a.n && i + step > i ? i + step : a.n;
      while (hi < a.n && (keys[hi] >> sh) == cell) {
        lo = hi;
        step *= 2u;
        hi = a.n - hi > step ? hi + step : a.n;
      }
      while (hi - lo > 1u) {
        const uint32_t mid = lo + (hi - lo) / 2u;
        if ((keys[mid] >> sh) == cell) lo = mid;
        else hi = mid;
      }
      end = hi;
    }
    const uint32_t count = end - i;
    o.count[b] = count;
    o.subtree[b] = (end < a.n ? pbase[end] : total) - o.pre[b];
    uint32_t c = 0;
    const uint32_t fc = o.first_child[b];
    if (!leaf) {
      const uint32_t le = lv[d + 2];
      uint32_t first = i;  // begin of child c
      while (c < 8u && fc + c < le && first < end) {
        const uint32_t nxt = fc + c + 1u < le ? o.begin[fc + c + 1u] : a.n;
        const uint32_t ce = nxt < end ? nxt : end;
        if (count > a.cut && ce - first <= a.cut) subs[atomicAdd(&lv[kLvSubs], 1u)] = fc + c;
        first = nxt;
        ++c;
      }
      if (c) atomicOr(&o.meta[fc + c - 1u], 1u << 17);
    }
    o.nchild[b] = c;
    if (d == 0 && count <= a.cut) subs[atomicAdd(&lv[kLvSubs], 1u)] = b;
    if (count > a.cut) tops[static_cast<std::size_t>(d) * a.max_top + atomicAdd(&lv[kLvTops + d], 1u)] = b;
  }
}

// Multipoles, bottom up (tree_gravity.cpp:1208-1380, same operation order). A
// particle or child has a lane: its terms go to LDS, and one lane per sum adds
// them in tree order, so a wave's loads are independent and contiguous. One
// thread per node left a wave to chains of dependent loads. Leaf order, subtrees
// and top, thread per node and now: 128^3 71 + 270 + 84 and 118 + 76 + 39 us,
// 256^3 594 + 983 + 77 and 995 + 417 + 38 us.
struct MomArgs {
  UnwrapArgs u;
  int quad;
  uint32_t done;  // leaves of at most this many particles have their moments from the leaf pass
};

struct MomArrays {
  const double4* pk;
  const uint32_t *begin, *count, *nchild, *first_child;
  const double4* geo;
  double4* mom;
  double* quad;  // 8 per node
  double* box;   // 6 per node: the tight bounding box of its particles (unwrapped), lo[3], hi[3]
};

constexpr int kSumTerms = 7;
constexpr int kSumStride = kWave + 2;  // doubles: the lanes of a group's sums read different banks
using WaveTerms = double[kSumTerms * kSumStride];

// Lane l < N of every group of G lanes adds term l of the group's first
// `steps` lanes to `acc`, in lane order. All lanes active, steps wave-uniform.
template <int G, int N>
__device__ __forceinline__ double ordered_sums(WaveTerms& buf, const double (&v)[N], uint32_t steps, double acc) {
  const int lane = lane_id(), l = lane % G;
#pragma unroll
  for (int k = 0; k < N; ++k) buf[k * kSumStride + lane] = v[k];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const double* src = &buf[(l < N ? l : 0) * kSumStride + lane - l];
  for (uint32_t j = 0; j < steps; ++j) acc += src[j];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  return acc;
}

// Minima and maxima over groups of G consecutive lanes (8, 16 or 64), in every
// lane. All lanes must be active.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const uint64_t b = static_cast<uint64_t>(__double_as_longlong(v));
  const uint32_t lo = CHUI_DPP(static_cast<uint32_t>(b), CTRL, 0xf, 0u);
  const uint32_t hi = CHUI_DPP(static_cast<uint32_t>(b >> 32), CTRL, 0xf, 0u);
  return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}
template <int G, class Op>
__device__ __forceinline__ double group_reduce(double v, Op op) {
  v = op(v, dpp_f64<0xb1>(v));                // quad_perm [1,0,3,2]
  v = op(v, dpp_f64<0x4e>(v));                // quad_perm [2,3,0,1]
  v = op(v, dpp_f64<0x141>(v));               // row_half_mirror: the other quad of 8
  if (G >= 16) v = op(v, dpp_f64<0x140>(v));  // row_mirror: the other 8 of 16
  if (G >= 32) v = op(v, __shfl_xor(v, 16, kWave));
  if (G >= 64) v = op(v, __shfl_xor(v, 32, kWave));
  return v;
}
template <int G>
__device__ __forceinline__ double group_min(double v) {
  return group_reduce<G>(v, [](double x, double y) { return fmin(x, y); });
}
template <int G>
__device__ __forceinline__ double group_max(double v) {
  return group_reduce<G>(v, [](double x, double y) { return fmax(x, y); });
}

// The centre of mass from lane l < 4's sums (mass and first moments), in every
// lane; lane l stores its component.
template <int G>
__device__ __forceinline__ double4 mass_centre(const MomArrays& o, uint32_t node, bool store, const double4& g,
                                               double sum) {
  const int lane = lane_id(), l = lane % G, first = lane - l;
  const double tm = __shfl(sum, first, kWave);
  const bool on = tm > 0.0;
  const double c = l == 1 ? g.x : l == 2 ? g.y : g.z;
  const double v = l == 0 ? tm : on ? sum / tm : c;
  if (store && l < 4) reinterpret_cast<double*>(o.mom + node)[(l + 3) & 3] = v;
  return make_double4(__shfl(v, first + 1, kWave), __shfl(v, first + 2, kWave), __shfl(v, first + 3, kWave), tm);
}

// Lane l < 7 stores its quadrupole value, lane 7 the distance of the centre of
// mass from the cell's centre; the box is stored by lane 0.
template <int G>
__device__ __forceinline__ void store_quad_box(const MomArrays& o, uint32_t node, bool store, const double4& g,
                                               const double4& M, double q, const double (&lo)[3],
                                               const double (&hi)[3]) {
  const int l = lane_id() % G;
  if (store && l < 8) {
    const double ox = g.x - M.x, oy = g.y - M.y, oz = g.z - M.z;
    o.quad[8ull * node + l] = l == 7 ? sqrt(ox * ox + oy * oy + oz * oz) : M.w > 0.0 ? q : 0.0;
  }
  if (store && l == 0) {
    double2* bx = reinterpret_cast<double2*>(o.box + 6ull * node);
    bx[0] = make_double2(lo[0], lo[1]);
    bx[1] = make_double2(lo[2], hi[0]);
    bx[2] = make_double2(hi[1], hi[2]);
  }
}

// Lane l < 6's second moments (xx, xy, xz, yy, yz, zz) to the traceless
// quadrupole, lane 6 the trace.
template <int G>
__device__ __forceinline__ double traceless(double s) {
  const int lane = lane_id(), l = lane % G, first = lane - l;
  const double tr = __shfl(s, first, kWave) + __shfl(s, first + 3, kWave) + __shfl(s, first + 5, kWave);
  return l == 6 ? tr : l == 0 || l == 3 || l == 5 ? 3.0 * s - tr : 3.0 * s;
}

// Moments of leaves whose particles lie one to a lane of a group of G lanes in
// tree order (on: mass and unwrapped position), at most `steps` in a group.
template <int G>
__device__ __forceinline__ void leaf_moments(const MomArgs& a, const MomArrays& o, WaveTerms& buf, uint32_t node,
                                             bool leaf, bool any, bool on, uint32_t steps, double mass, double ux,
                                             double uy, double uz) {
  const double4 g = leaf ? o.geo[node] : make_double4(0.0, 0.0, 0.0, 0.0);
  const double mm = on ? mass : 0.0;
  double lo[3] = {group_min<G>(on ? ux : INFINITY), group_min<G>(on ? uy : INFINITY), group_min<G>(on ? uz : INFINITY)};
  double hi[3] = {group_max<G>(on ? ux : -INFINITY), group_max<G>(on ? uy : -INFINITY),
                  group_max<G>(on ? uz : -INFINITY)};
  if (!any) {
    lo[0] = hi[0] = g.x;
    lo[1] = hi[1] = g.y;
    lo[2] = hi[2] = g.z;
  }
  const double t4[4] = {mm, on ? mm * ux : 0.0, on ? mm * uy : 0.0, on ? mm * uz : 0.0};
  const double4 M = mass_centre<G>(o, node, leaf, g, ordered_sums<G>(buf, t4, steps, 0.0));
  double q = 0.0;
  if (a.quad) {  // wave-uniform
    const double rx = ux - M.x, ry = uy - M.y, rz = uz - M.z;
    const double t6[6] = {on ? mm * rx * rx : 0.0, on ? mm * rx * ry : 0.0, on ? mm * rx * rz : 0.0,
                          on ? mm * ry * ry : 0.0, on ? mm * ry * rz : 0.0, on ? mm * rz * rz : 0.0};
    q = traceless<G>(ordered_sums<G>(buf, t6, steps, 0.0));
  }
  store_quad_box<G>(o, node, leaf, g, M, q, lo, hi);
}

// Moments of a leaf of any size by one whole wave, 64 particles at a time.
__device__ __forceinline__ void leaf_moments_wave(const MomArgs& a, const MomArrays& o, WaveTerms& buf,
                                                  uint32_t node) {
  const uint32_t b = o.begin[node], c = o.count[node];
  const double4 g = o.geo[node];
  double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  double sum = 0.0;
  for (uint32_t k = 0; k < c; k += kWave) {  // wave-uniform
    const uint32_t left = c - k, steps = left < kWave ? left : kWave;
    double t4[4] = {0.0, 0.0, 0.0, 0.0};
    if (lane_id() < steps) {
      const double4 p = o.pk[b + k + lane_id()];
      const double u[3] = {unwrap_canonical(p.x, a.u.anchor[0], a.u.L[0]),
                           unwrap_canonical(p.y, a.u.anchor[1], a.u.L[1]),
                           unwrap_canonical(p.z, a.u.anchor[2], a.u.L[2])};
      t4[0] = p.w;
      for (int ax = 0; ax < 3; ++ax) {
        t4[ax + 1] = p.w * u[ax];
        lo[ax] = fmin(lo[ax], u[ax]);
        hi[ax] = fmax(hi[ax], u[ax]);
      }
    }
    sum = ordered_sums<kWave>(buf, t4, steps, sum);
  }
  for (int ax = 0; ax < 3; ++ax) {
    lo[ax] = group_min<kWave>(lo[ax]);
    hi[ax] = group_max<kWave>(hi[ax]);
  }
  const double4 M = mass_centre<kWave>(o, node, true, g, sum);
  double q = 0.0;
  if (a.quad) {
    for (uint32_t k = 0; k < c; k += kWave) {
      const uint32_t left = c - k, steps = left < kWave ? left : kWave;
      double t6[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      if (lane_id() < steps) {
        const double4 p = o.pk[b + k + lane_id()];
        const double rx = unwrap_canonical(p.x, a.u.anchor[0], a.u.L[0]) - M.x;
        const double ry = unwrap_canonical(p.y, a.u.anchor[1], a.u.L[1]) - M.y;
        const double rz = unwrap_canonical(p.z, a.u.anchor[2], a.u.L[2]) - M.z;
        t6[0] = p.w * rx * rx;
        t6[1] = p.w * rx * ry;
        t6[2] = p.w * rx * rz;
        t6[3] = p.w * ry * ry;
        t6[4] = p.w * ry * rz;
        t6[5] = p.w * rz * rz;
      }
      q = ordered_sums<kWave>(buf, t6, steps, q);
    }
    q = traceless<kWave>(q);
  }
  store_quad_box<kWave>(o, node, true, g, M, q, lo, hi);
}

// Moments of eight nodes per wave, a child to a lane (c: children of the
// group's node, 0 for none).
__device__ __forceinline__ void inner_moments(const MomArgs& a, const MomArrays& o, WaveTerms& buf, uint32_t node,
                                              uint32_t c) {
  const uint32_t j = lane_id() & 7u;
  const bool inner = c > 0u, child = j < c;
  double4 g = make_double4(0.0, 0.0, 0.0, 0.0), cm = g;
  double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  double cq[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (inner) g = o.geo[node];
  if (child) {
    const uint32_t ch = o.first_child[node] + j;
    cm = o.mom[ch];
    const double2* bx = reinterpret_cast<const double2*>(o.box + 6ull * ch);
    const double2 b0 = bx[0], b1 = bx[1], b2 = bx[2];
    lo[0] = b0.x; lo[1] = b0.y; lo[2] = b1.x;
    hi[0] = b1.y; hi[1] = b2.x; hi[2] = b2.y;
    if (a.quad) {
      const double4* qd = reinterpret_cast<const double4*>(o.quad + 8ull * ch);
      const double4 q0 = qd[0], q1 = qd[1];
      cq[0] = q0.x; cq[1] = q0.y; cq[2] = q0.z; cq[3] = q0.w;
      cq[4] = q1.x; cq[5] = q1.y; cq[6] = q1.z;
    }
  }
#pragma unroll
  for (int ax = 0; ax < 3; ++ax) {
    lo[ax] = group_min<8>(lo[ax]);
    hi[ax] = group_max<8>(hi[ax]);
  }
  const double t4[4] = {cm.w, cm.w * cm.x, cm.w * cm.y, cm.w * cm.z};
  const double4 M = mass_centre<8>(o, node, inner, g, ordered_sums<8>(buf, t4, 8u, 0.0));
  double q = 0.0;
  if (a.quad) {  // wave-uniform
    const double dx = child ? cm.x - M.x : 0.0, dy = child ? cm.y - M.y : 0.0, dz = child ? cm.z - M.z : 0.0;
    const double mm = cm.w, d2 = dx * dx + dy * dy + dz * dz;
    const double t7[7] = {cq[0] + mm * (3.0 * dx * dx - d2), cq[1] + mm * (3.0 * dx * dy),
                          cq[2] + mm * (3.0 * dx * dz),      cq[3] + mm * (3.0 * dy * dy - d2),
                          cq[4] + mm * (3.0 * dy * dz),      cq[5] + mm * (3.0 * dz * dz - d2),
                          cq[6] + mm * d2};
    q = ordered_sums<8>(buf, t7, 8u, 0.0);
  }
  store_quad_box<8>(o, node, inner, g, M, q, lo, hi);
}

// Moments of eight nodes (on: the lane's group has one). Leaves beyond the leaf
// pass are summed by the whole wave, one by one.
__device__ __forceinline__ void node_moments(const MomArgs& a, const MomArrays& o, WaveTerms& buf, uint32_t node,
                                             bool on) {
  const uint32_t c = on ? o.nchild[node] : 0u;
  if (__ballot(c > 0u)) inner_moments(a, o, buf, node, c);
  unsigned long long big = __ballot(on && c == 0u && (lane_id() & 7u) == 0u && o.count[node] > a.done);
  while (big) {
    const int l = __ffsll(static_cast<long long>(big)) - 1;
    big &= big - 1ull;
    leaf_moments_wave(a, o, buf, readlane_u32(node, l));
  }
}

// v moved to the lane at byte address `to` / 4; all lanes active, `to` a permutation
__device__ __forceinline__ double permute_f64(int to, double v) {
  const uint64_t b = static_cast<uint64_t>(__double_as_longlong(v));
  const uint32_t lo = __builtin_amdgcn_ds_permute(to, static_cast<int>(static_cast<uint32_t>(b)));
  const uint32_t hi = __builtin_amdgcn_ds_permute(to, static_cast<int>(static_cast<uint32_t>(b >> 32)));
  return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}

// In-leaf Morton order (tree_ordering.cpp:151): the (Morton key, row) ranks of
// a leaf's particles by comparison, G lanes per node; leaves of more than G
// particles are ranked by the whole wave unless they are in order. Reads the sort's order and the
// input-order records, writes the final order and the tree-order copy of the
// sources (canonical coordinates and mass), so the gather, the Morton keys and
// the permutation are one pass (256^3: 0.85 ms in three). The records move to
// their rank's lane first: the stores are contiguous, and the leaf's moments
// are summed in tree order while its particles are in registers.
template <int G>
__global__ __launch_bounds__(256) void leaf_order_kernel(uint32_t total_nodes, const uint32_t* __restrict__ total_dev,
                                                         MomArgs mo, MomArrays o,
                                                         MortonArgs a,
                                                         const double4* __restrict__ packed,
                                                         const uint32_t* __restrict__ order_in,
                                                         uint32_t* __restrict__ order_out, double4* __restrict__ pk,
                                                         const Frame* __restrict__ fr) {
  const uint32_t total = total_dev ? *total_dev : total_nodes;
  __shared__ WaveTerms terms[256 / kWave];
  UnwrapArgs& u = mo.u;
  if (fr) {
    for (int ax = 0; ax < 3; ++ax) {
      u.anchor[ax] = fr->anchor[ax];
      a.lo[ax] = fr->mlo[ax];
    }
    a.extent = fr->mext;
  }
  auto key_of = [&](const double4& q) -> uint64_t {
    return morton_key(unwrap_canonical(q.x, u.anchor[0], u.L[0]), unwrap_canonical(q.y, u.anchor[1], u.L[1]),
                      unwrap_canonical(q.z, u.anchor[2], u.L[2]), a);
  };
  const int lane = lane_id(), sub = lane / G, l = lane % G;
  const uint32_t per = kWave / G;
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave, waves = gridDim.x * blockDim.x / kWave;
  for (uint32_t first = wave * per; first < total; first += waves * per) {  // wave-uniform
    const uint32_t node = first + sub;
    uint32_t b = 0, c = 0;
    const bool leaf = node < total && o.nchild[node] == 0;
    if (leaf) {
      b = o.begin[node];
      c = o.count[node];
    }
    const bool small = c <= static_cast<uint32_t>(G);
    const bool on = small && static_cast<uint32_t>(l) < c;
    uint32_t row = 0;
    double4 q = make_double4(0.0, 0.0, 0.0, 0.0);
    uint64_t mk = 0;
    if (on) {
      row = order_in[b + l];
      q = packed[row];
      mk = key_of(q);
    }
    uint32_t rank = 0;
    const uint32_t steps = wave_max_u32(small ? c : 0u);
    for (uint32_t k = 0; k < steps; ++k) {
      const int src = sub * G + static_cast<int>(k);
      const uint64_t ok = __shfl(mk, src, kWave);
      const uint32_t orow = __shfl(row, src, kWave);
      if (k < c && (ok < mk || (ok == mk && orow < row))) ++rank;
    }
    // lanes beyond the leaf keep their place, so this is a permutation of the group
    const int to = 4 * (sub * G + (on ? static_cast<int>(rank) : l));
    row = static_cast<uint32_t>(__builtin_amdgcn_ds_permute(to, static_cast<int>(row)));
    q.x = permute_f64(to, q.x);
    q.y = permute_f64(to, q.y);
    q.z = permute_f64(to, q.z);
    q.w = permute_f64(to, q.w);
    if (on) {
      order_out[b + l] = row;
      pk[b + l] = q;
    }
    leaf_moments<G>(mo, o, terms[threadIdx.x / kWave], node, leaf && small, c > 0u, on, steps, q.w, unwrap_canonical(q.x, u.anchor[0], u.L[0]),
                    unwrap_canonical(q.y, u.anchor[1], u.L[1]), unwrap_canonical(q.z, u.anchor[2], u.L[2]));
    unsigned long long big = __ballot(!small && l == 0);
    while (big) {
      const int s = __ffsll(static_cast<long long>(big)) - 1;
      big &= big - 1ull;
      const uint32_t bb = readlane_u32(b, s), bc = readlane_u32(c, s);
      // coincident sources come in order from the stable sort, any number of
      // them in one leaf: they are only copied (a solve of 6000: ranked 282 ms,
      // copied 1.1 ms)
      bool sorted = true;
      for (uint32_t e0 = 0; e0 + 1u < bc && sorted; e0 += kWave) {
        bool ok = true;
        if (e0 + lane + 1u < bc) {
          const uint32_t r0 = order_in[bb + e0 + lane], r1 = order_in[bb + e0 + lane + 1u];
          const uint64_t k0 = key_of(packed[r0]), k1 = key_of(packed[r1]);
          ok = k0 < k1 || (k0 == k1 && r0 < r1);
        }
        sorted = __ballot(!ok) == 0ull;
      }
      for (uint32_t e = lane; e < bc; e += kWave) {
        const uint32_t er = order_in[bb + e];
        const double4 eq = packed[er];
        if (sorted) {
          order_out[bb + e] = er;
          pk[bb + e] = eq;
          continue;
        }
        const uint64_t ek = key_of(eq);
        uint32_t r = 0;
        for (uint32_t k = 0; k < bc; ++k) {
          const uint32_t orow = order_in[bb + k];
          const uint64_t ok = key_of(packed[orow]);
          if (ok < ek || (ok == ek && orow < er)) ++r;
        }
        order_out[bb + r] = er;
        pk[bb + r] = eq;
      }
    }
  }
}

// Moments of one subtree per block, all its levels in one launch (bound by the
// loads of each level waiting for the level below; a launch per level took 13
// to 15 launches of 4 to 60 us, hence subtrees of max(512, n / 1024) particles:
// above 5e5 particles a thousand or more blocks and at most a few thousand nodes
// above them; 32^3 has about 64 blocks). A subtree's nodes of each depth are consecutive, from the first child of the first split
// node of the depth above to the last child of the last.
__global__ __launch_bounds__(256) void moment_subtree_kernel(MomArgs a, MomArrays o, const uint32_t* __restrict__ lv,
                                                             const uint32_t* __restrict__ subs,
                                                             const Frame* __restrict__ fr) {
  __shared__ uint32_t lo[kMaxLevels + 1], hi[kMaxLevels + 1];
  __shared__ WaveTerms terms[256 / kWave];
  if (fr)
    for (int ax = 0; ax < 3; ++ax) a.u.anchor[ax] = fr->anchor[ax];
  const uint32_t nsub = lv[kLvTotal] ? lv[kLvSubs] : 0u;
  for (uint32_t s = blockIdx.x; s < nsub; s += gridDim.x) {
    __syncthreads();  // the last subtree's levels are done with lo, hi
    if (threadIdx.x <= kMaxLevels) {
      const uint32_t root = subs[s];
      lo[threadIdx.x] = threadIdx.x == 0 ? root : kInvalidIndex;
      hi[threadIdx.x] = threadIdx.x == 0 ? root + 1u : 0u;
    }
    __syncthreads();
    int levels = 0;
    for (;;) {
      const uint32_t l0 = lo[levels], l1 = hi[levels];
      ++levels;
      if (levels > kMaxLevels) break;
      uint32_t mn = kInvalidIndex, mx = 0;
      for (uint32_t b = l0 + threadIdx.x; b < l1; b += blockDim.x) {
        const uint32_t c = o.nchild[b];
        if (c) {
          const uint32_t f = o.first_child[b];
          mn = f < mn ? f : mn;
          mx = f + c > mx ? f + c : mx;
        }
      }
      if (mx) {
        atomicMin(&lo[levels], mn);
        atomicMax(&hi[levels], mx);
      }
      __syncthreads();
      if (hi[levels] == 0u) break;  // block-uniform
    }
    for (int d = levels - 1; d >= 0; --d) {
      for (uint32_t b = lo[d] + threadIdx.x / kWave * 8u; b < hi[d]; b += blockDim.x / 8u)  // wave-uniform
        node_moments(a, o, terms[threadIdx.x / kWave], b + lane_id() / 8u, b + lane_id() / 8u < hi[d]);
      __syncthreads();
    }
  }
}

// The nodes above the subtrees, deepest level first (one block: about n / cut
// of them per level).
__global__ __launch_bounds__(1024) void moment_top_kernel(MomArgs a, MomArrays o, const uint32_t* __restrict__ lv,
                                                          const uint32_t* __restrict__ tops, uint32_t max_top) {
  __shared__ WaveTerms terms[1024 / kWave];
  if (lv[kLvTotal] == 0) return;
  for (int d = kPathLevels; d >= 0; --d) {
    const uint32_t n = lv[kLvTops + d];
    for (uint32_t k0 = threadIdx.x / kWave * 8u; k0 < n; k0 += blockDim.x / 8u) {  // wave-uniform
      const uint32_t k = k0 + lane_id() / 8u;
      node_moments(a, o, terms[threadIdx.x / kWave], k < n ? tops[static_cast<std::size_t>(d) * max_top + k] : 0u, k < n);
    }
    __syncthreads();
  }
}

__device__ __forceinline__ uint32_t to_fixed(double c, double scale) {
  // scale = 2^32 / L; wraps modulo 2^32 (periodic)
  const double f = floor(c * scale);
  return static_cast<uint32_t>(static_cast<uint64_t>(static_cast<int64_t>(f)));
}

struct RecordArgs {
  uint32_t total;
  int fp64;   // FP64 records and child indices
  int mixed;  // fixed-point/FP32 records and tight boxes
  int cubic;  // separation units of the mixed walk: fixed point (cubic box) or lengths
  double fscale[3];
};

// x rounded up to a float (x >= 0)
__device__ __forceinline__ float float_up(double x) {
  const float f = static_cast<float>(x);
  return static_cast<double>(f) < x ? nextafterf(f, INFINITY) : f;
}

// BFS -> preorder records: links always, FP64 records and/or the mixed walk's
// fixed-point/FP32 records.
__global__ __launch_bounds__(256) void records_kernel(RecordArgs a, const uint32_t* __restrict__ pre,
                                                      const uint32_t* __restrict__ nb, const uint32_t* __restrict__ nc,
                                                      const uint32_t* __restrict__ nchild,
                                                      const uint32_t* __restrict__ first_child,
                                                      const uint32_t* __restrict__ meta,
                                                      const uint32_t* __restrict__ subtree,
                                                      const double4* __restrict__ geo,
                                                      const double4* __restrict__ mom,
                                                      const double* __restrict__ quad, NodeLink* __restrict__ link,
                                                      NodeGeo64* __restrict__ geo64, NodeMom64* __restrict__ mom64,
                                                      NodeQuad64* __restrict__ quad64,
                                                      uint32_t* __restrict__ child_index, NodeGeo32* __restrict__ geo32,
                                                      NodeMom32* __restrict__ mom32,
                                                      NodeQuad32* __restrict__ quad32,
                                                      const double* __restrict__ box,
                                                      NodeBox32* __restrict__ box32, WalkNode* __restrict__ wnode,
                                                      const uint32_t* __restrict__ total_dev) {
  const uint32_t total = total_dev ? *total_dev : a.total;
  for (uint32_t node = blockIdx.x * blockDim.x + threadIdx.x; node < total; node += gridDim.x * blockDim.x) {
  const uint32_t p = pre[node];
  const uint32_t c = nchild[node];
  link[p] = NodeLink{nb[node], nc[node], subtree[node], c};
  const double4 g = geo[node];
  const double4 M = mom[node];
  const double* q = quad + 8ull * node;
  if (a.fp64) {
    geo64[p] = NodeGeo64{g.x, g.y, g.z, g.w};
    mom64[p] = NodeMom64{M.x, M.y, M.z, M.w};
    quad64[p] = NodeQuad64{q[0], q[1], q[2], q[3], q[4], q[5], q[6], q[7]};
    uint32_t ci[8];
#pragma unroll
    for (int o = 0; o < 8; ++o) ci[o] = kInvalidIndex;
    for (uint32_t j = 0; j < c; ++j) {
      const uint32_t ch = first_child[node] + j;
      ci[(meta[ch] >> 8) & 7u] = pre[ch];
    }
#pragma unroll
    for (int o = 0; o < 8; ++o) child_index[8ull * p + o] = ci[o];
  }
  if (a.mixed) {
    geo32[p] = NodeGeo32{to_fixed(g.x, a.fscale[0]), to_fixed(g.y, a.fscale[1]), to_fixed(g.z, a.fscale[2]),
                         static_cast<float>(g.w)};
    mom32[p] = NodeMom32{to_fixed(M.x, a.fscale[0]), to_fixed(M.y, a.fscale[1]), to_fixed(M.z, a.fscale[2]),
                         static_cast<float>(M.w)};
    quad32[p] = NodeQuad32{static_cast<float>(q[0]), static_cast<float>(q[1]), static_cast<float>(q[2]),
                           static_cast<float>(q[3]), static_cast<float>(q[4]), static_cast<float>(q[5]),
                           static_cast<float>(q[6]), static_cast<float>(q[7])};
  }
  if (wnode) {
    // Fixed point floors: the centre and every particle move by less than one
    // unit each, so two units on top of the half-extent keep every particle's
    // fixed-point position inside the box.
    const double* bx = box + 6ull * node;
    NodeBox32 r;
    uint32_t cf[3];
    float hf[3];
    for (int ax = 0; ax < 3; ++ax) {
      const double half = 0.5 * (bx[3 + ax] - bx[ax]);
      cf[ax] = to_fixed(0.5 * (bx[ax] + bx[3 + ax]), a.fscale[ax]);
      hf[ax] = a.cubic ? float_up(half * a.fscale[ax] + 2.0) : float_up(half + 2.0 / a.fscale[ax]);
    }
    r.cx = cf[0];
    r.cy = cf[1];
    r.cz = cf[2];
    r.hx = hf[0];
    r.hy = hf[1];
    r.hz = hf[2];
    r.cell_half = static_cast<float>(g.w);
    r.pad = 0u;
    if (box32) box32[p] = r;
    wnode[node] = WalkNode{r.cx, r.cy, r.cz, r.hx, r.hy, r.hz, r.cell_half,
                           c | ((meta[node] >> 17) & 1u ? kLastSibling : 0u), c == 0 ? nb[node] : first_child[node],
                           nc[node], p, subtree[node]};
  }
  }
}

__global__ void unwrap_apply_kernel(const double* in, std::size_t n, double L, int canonical, double anchor,
                                    double* out) {
  const std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) out[i] = unwrap_coord(in[i], L, canonical, anchor);
}

__global__ void pos_of_row_kernel(const uint32_t* __restrict__ order, std::size_t n, uint32_t* __restrict__ pos) {
  const std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) pos[order[i]] = static_cast<uint32_t>(i);
}

// ---- capture-safe build: per-build values kept on the device ------------------
struct FrameCheck {
  double L[3];
  int expect_uniform;  // mass uniformity of the prepared build
  double expect_mass;  // its uniform mass
};

// Canonical flags from the statistics (tree_pm_coupling.cpp:3185-3195, as the
// ordinary build decides them on the host); invalid inputs and a mass
// uniformity other than the prepared build's set fault bits.
__global__ void frame_stats_kernel(const SourceStats* __restrict__ st, const double* __restrict__ m, FrameCheck c,
                                   Frame* __restrict__ fr, unsigned long long* __restrict__ fault) {
  if (threadIdx.x != 0) return;
  unsigned long long f = 0;
  if (st->bad_coord) f |= kFaultCoordinates;
  if (st->bad_mass) f |= kFaultMasses;
  const int uniform = st->mass_nonuniform == 0 ? 1 : 0;
  if (uniform != c.expect_uniform || (uniform && m[0] != c.expect_mass)) f |= kFaultPrepared;
  for (int a = 0; a < 3; ++a) {
    const double lo = order_key_inv(st->lo[a]), hi = order_key_inv(st->hi[a]);
    fr->canonical[a] = (lo >= 0.0 && hi < c.L[a]) ? 1 : 0;
  }
  fr->pad = 0;
  if (f && fault) atomicOr(fault, f);
}

// Root cube (tree_gravity.cpp:443-452) and the in-leaf Morton frame
// (tree_ordering.cpp:151) from the unwrap result, with the ordinary build's
// host arithmetic (max as (a < b) ? b : a, no contraction).
__global__ void frame_root_kernel(const UnwrapResult* __restrict__ res, Frame* __restrict__ fr) {
  if (threadIdx.x != 0) return;
  double ext = 0.0;
  for (int a = 0; a < 3; ++a) {
    const double e = res->umax[a] - res->umin[a];
    ext = ext < e ? e : ext;
  }
  const double max_extent = ext < 1.0e-10 ? 1.0e-10 : ext;
  for (int a = 0; a < 3; ++a) {
    fr->anchor[a] = res->anchor[a];
    fr->centre[a] = 0.5 * (res->umin[a] + res->umax[a]);
    fr->mlo[a] = res->umin[a];
  }
  fr->half = 0.5 * max_extent * (1.0 + 1.0e-8);
  fr->mext = ext < 1.0e-12 ? 1.0e-12 : ext;
}

// p[0, *count) = v, the count read on the device.
template <class T>
__global__ __launch_bounds__(256) void fill_count_kernel(T* __restrict__ p, T v, const uint32_t* __restrict__ count) {
  const uint32_t n = *count;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = v;
}

// Source statistics -> host.
SourceStats compute_stats(Tree& t, Axes3 p, const double* m, std::size_t n, hipStream_t s) {
  const unsigned nb = n > 0 ? std::min<unsigned>(grid_for(n, 256), 1024u) : 0u;
  t.bounds.reserve((1 + std::max(nb, 1u)) * sizeof(SourceStats));
  SourceStats* st = t.bounds.as<SourceStats>();
  if (n > 0) {
    source_stats_kernel<<<nb, 256, 0, s>>>(p, m, n, st + 1);
    CHUI_LAUNCH_CHECK("source_stats_kernel");
  }
  stats_final_kernel<<<1, 256, 0, s>>>(st + 1, nb, n > 0 ? m : nullptr, st);
  CHUI_LAUNCH_CHECK("stats_final_kernel");
  SourceStats h{};
  t.readback.read(&h, st, sizeof(SourceStats), s);
  return h;
}

double host_order_key_inv(uint64_t k) {
  const uint64_t b = (k & 0x8000000000000000ull) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k;
  double d;
  std::memcpy(&d, &b, 8);
  return d;
}

// Unwraps naxes axes at once; fills res (host).
// With fr (a capture-safe build) the canonical flags come from the frame, the
// marked-bucket buffers are sized by their bound (marked buckets are occupied
// buckets, at most n per axis) and nothing is read back: the result stays in
// the device UnwrapResult (returned).
UnwrapResult* unwrap_axes(Tree& t, Axes3 p, int naxes, std::size_t n, const double* L, const int* canonical,
                          UnwrapResult& res, hipStream_t s, const Frame* fr = nullptr, bool size_bound = false) {
  for (int ax = 0; ax < naxes; ++ax) {
    res.anchor[ax] = 0.0;
    res.umin[ax] = 0.0;
    res.umax[ax] = 0.0;
    res.canonical[ax] = canonical[ax];
  }
  if (n == 0) return nullptr;
  BucketArgs a{};
  const uint64_t B = (std::max<uint64_t>(2ull * n, 64ull) + 31) / 32 * 32;
  a.B = B;
  a.W = B / 32;
  a.naxes = naxes;
  for (int ax = 0; ax < naxes; ++ax) {
    a.L[ax] = L[ax];
    a.scale[ax] = static_cast<double>(B) / L[ax];
    a.canonical[ax] = canonical[ax];
  }
  const uint64_t W = a.W, NW = naxes * W;
  const uint64_t nblk = (W + kGapTile - 1) / kGapTile;
  // bitmaps: occupancy, marks, run ends; ranks; block scan data
  t.bucket_min.reserve(3 * NW * sizeof(uint32_t) + 2 * NW * sizeof(uint32_t));
  uint32_t* occ = t.bucket_min.as<uint32_t>();
  uint32_t* mark = occ + NW;
  uint32_t* ends = mark + NW;
  uint32_t* popc = ends + NW;
  uint32_t* rank_base = popc + NW;
  t.block_max.reserve((naxes * nblk + 8) * sizeof(uint64_t));
  uint64_t* blockmax = t.block_max.as<uint64_t>();
  uint64_t* total = blockmax + naxes * nblk;               // 3 entries
  unsigned long long* longest = reinterpret_cast<unsigned long long*>(total + 3);  // 3 entries
  uint32_t* marked = reinterpret_cast<uint32_t*>(total + 6);  // total marked buckets
  t.block_best.reserve((naxes * nblk + 1) * sizeof(GapBest) + sizeof(UnwrapResult));
  GapBest* best = t.block_best.as<GapBest>();
  UnwrapResult* dres = reinterpret_cast<UnwrapResult*>(best + naxes * nblk + 1);
  fill_u32(occ, 0u, 3 * NW, s);
  fill_u64(total, 0ull, 8, s);
  const unsigned pgrid = std::min<unsigned>(grid_for(n, 256), 8192u);
  // bytes per bucket (B per axis, a multiple of 32), then packed into occ
  t.occ_bytes.reserve(naxes * B);
  uint8_t* occb = t.occ_bytes.as<uint8_t>();
  fill_u32(reinterpret_cast<uint32_t*>(occb), 0u, naxes * B / 4, s);
  occupancy_bytes_kernel<<<pgrid, 256, 0, s>>>(p, n, a, occb, fr);
  CHUI_LAUNCH_CHECK("occupancy_bytes_kernel");
  occupancy_pack_kernel<<<grid_for(NW, 256), 256, 0, s>>>(occb, NW, occ);
  CHUI_LAUNCH_CHECK("occupancy_pack_kernel");
  occ_blockmax_kernel<<<dim3(static_cast<unsigned>(nblk), naxes), kGapThreads, 0, s>>>(occ, W, blockmax, nblk);
  CHUI_LAUNCH_CHECK("occ_blockmax_kernel");
  blockmax_scan_kernel<<<naxes, kGapThreads, 0, s>>>(blockmax, nblk, total);
  CHUI_LAUNCH_CHECK("blockmax_scan_kernel");
  RunArgs ra{};
  ra.occ = occ;
  ra.block_prefix = blockmax;
  ra.total = total;
  ra.longest = longest;
  ra.mark = mark;
  ra.ends = ends;
  ra.rank_base = rank_base;
  ra.block_out = best;
  ra.nblk = nblk;
  const dim3 rgrid(static_cast<unsigned>(nblk), naxes);
  runs_kernel<0><<<rgrid, kGapThreads, 0, s>>>(a, ra);
  CHUI_LAUNCH_CHECK("runs_kernel<0>");
  runs_kernel<1><<<rgrid, kGapThreads, 0, s>>>(a, ra);
  CHUI_LAUNCH_CHECK("runs_kernel<1>");
  popc_kernel<<<grid_for(NW, 256), 256, 0, s>>>(mark, NW, popc);
  CHUI_LAUNCH_CHECK("popc_kernel");
  t.bfs_scan.reserve(scan_scratch_bytes(NW) + 64);
  exclusive_scan_u32(popc, rank_base, NW, marked, t.bfs_scan.ptr, s);
  uint64_t* cmin = nullptr;
  uint64_t* cmax = nullptr;
  if (fr) {
    const uint64_t cap = static_cast<uint64_t>(naxes) * n + 64;
    t.bucket_max.reserve(2 * cap * sizeof(uint64_t));
    cmin = t.bucket_max.as<uint64_t>();
    cmax = cmin + cap;
    fill_count_kernel<uint64_t><<<256, 256, 0, s>>>(cmin, kEmpty, marked);
    CHUI_LAUNCH_CHECK("fill_count_kernel");
    fill_count_kernel<uint64_t><<<256, 256, 0, s>>>(cmax, 0ull, marked);
    CHUI_LAUNCH_CHECK("fill_count_kernel");
  } else {
    uint32_t hm = 0;
    t.readback.read(&hm, marked, sizeof(hm), s);
    if (size_bound) t.bucket_max.reserve(2 * (static_cast<uint64_t>(naxes) * n + 64) * sizeof(uint64_t));
    t.bucket_max.reserve(2 * std::max<uint64_t>(hm, 1) * sizeof(uint64_t));
    cmin = t.bucket_max.as<uint64_t>();
    cmax = cmin + std::max<uint64_t>(hm, 1);
    fill_u64(cmin, kEmpty, hm, s);
    fill_u64(cmax, 0ull, hm, s);
  }
  marked_minmax_kernel<<<pgrid, 256, 0, s>>>(p, n, a, mark, rank_base, cmin, cmax, fr);
  CHUI_LAUNCH_CHECK("marked_minmax_kernel");
  ra.cmin = cmin;
  ra.cmax = cmax;
  runs_kernel<2><<<rgrid, kGapThreads, 0, s>>>(a, ra);
  CHUI_LAUNCH_CHECK("runs_kernel<2>");
  gap_final_kernel<<<naxes, kGapThreads, 0, s>>>(best, nblk, dres);
  CHUI_LAUNCH_CHECK("gap_final_kernel");
  if (fr) return dres;
  UnwrapResult h{};
  t.readback.read(&h, dres, sizeof(UnwrapResult), s);
  for (int ax = 0; ax < naxes; ++ax) {
    res.anchor[ax] = h.anchor[ax];
    res.umin[ax] = h.umin[ax];
    res.umax[ax] = h.umax[ax];
  }
  return dres;
}

void launch_records(Tree& t, bool fp64, bool mixed, hipStream_t s) {
  const std::size_t total = t.node_count;
  const std::size_t nsz = t.sized_for_capture ? std::max(total, t.bfs_capacity) : total;
  if (fp64) {
    t.geo64.reserve(nsz * sizeof(NodeGeo64));
    t.mom64.reserve(nsz * sizeof(NodeMom64));
    t.quad64.reserve(nsz * sizeof(NodeQuad64));
    t.child_index.reserve(nsz * 8 * sizeof(uint32_t));
  }
  // the walk records go with the build's own records, not with a later
  // ensure_records64
  const bool walk_nodes = mixed || !t.wnodes_current;
  RecordArgs ra{};
  ra.total = static_cast<uint32_t>(total);
  ra.fp64 = fp64 ? 1 : 0;
  ra.mixed = mixed ? 1 : 0;
  ra.cubic = t.cubic ? 1 : 0;
  for (int a = 0; a < 3; ++a) ra.fscale[a] = t.fscale[a];
  records_kernel<<<grid_for(total, 256), 256, 0, s>>>(
      ra, t.bfs_pre.as<uint32_t>(), t.bfs_begin.as<uint32_t>(), t.bfs_count.as<uint32_t>(),
      t.bfs_nchild.as<uint32_t>(), t.bfs_first_child.as<uint32_t>(), t.bfs_meta.as<uint32_t>(),
      t.bfs_subtree.as<uint32_t>(), t.bfs_geo.as<double4>(), t.bfs_mom.as<double4>(), t.bfs_quad.as<double>(),
      t.link.as<NodeLink>(), fp64 ? t.geo64.as<NodeGeo64>() : nullptr, fp64 ? t.mom64.as<NodeMom64>() : nullptr,
      fp64 ? t.quad64.as<NodeQuad64>() : nullptr, fp64 ? t.child_index.as<uint32_t>() : nullptr,
      mixed ? t.geo32.as<NodeGeo32>() : nullptr, mixed ? t.mom32.as<NodeMom32>() : nullptr,
      mixed ? t.quad32.as<NodeQuad32>() : nullptr, t.bfs_box.as<double>(),
      mixed ? t.box32.as<NodeBox32>() : nullptr, walk_nodes ? t.wnode.as<WalkNode>() : nullptr,
      device_node_count(t));
  CHUI_LAUNCH_CHECK("records_kernel");
  t.wnodes_current = true;
  if (fp64) t.records64 = true;
}

}  // namespace

void ensure_records64(Tree& t, hipStream_t s) {
  if (t.records64 || t.node_count == 0) return;
  launch_records(t, true, false, s);
}

// ---------------------------------------------------------------------------
void build_tree(Tree& t, const double* x, const double* y, const double* z, const double* m, const TreeParams& P,
                double softening, hipStream_t s) {
  (void)softening;
  const std::size_t n = P.n;
  if (n > 0xFFFFFFFEull) throw std::overflow_error("Tree gravity source count exceeds the 32-bit tree-index contract");
  const bool safe = P.capture_safe;
  if (safe) {
    if (!P.fault) throw std::logic_error("capture-safe tree builds report through a fault word");
    if (n == 0 || n != t.prepared_n || !t.sized_for_capture || t.safe_levels <= 0 || t.bfs_capacity == 0)
      throw std::runtime_error(
          "capture-safe solve on a context not prepared for these sources (run an ordinary solve of the same "
          "source count first)");
  }
  t.n = n;
  t.node_count = 0;
  t.leaf_count = 0;
  t.counts_on_device = false;
  if (!safe) t.max_depth = 0;
  Axes3 p{{x, y, z}};
  Frame* fr = nullptr;
  UnwrapArgs ua{};
  for (int a = 0; a < 3; ++a) ua.L[a] = P.L[a];
  SourceStats* st_dev = nullptr;
  UnwrapResult* unwrap_dev = nullptr;
  // The canonical flags, anchors and root cube stay on the device (Frame) in a
  // capture-safe build and for up to kFrameMax sources: an ordinary build then
  // reads back once, after its nodes are counted, instead of four times (each
  // read-back idles the GPU for about 30 us: 32^3 builds took 0.55 ms so).
  // Above it the waits are below 1% of a solve, and the unwrap's min/max
  // buffers (bounded by n per axis without a read-back) matter more.
  if (n > 0 && (safe || n <= kFrameMax)) {
    t.frame.reserve(sizeof(Frame));
    fr = t.frame.as<Frame>();
    const unsigned nb = std::min<unsigned>(grid_for(n, 256), 1024u);
    t.bounds.reserve((1 + nb) * sizeof(SourceStats));
    st_dev = t.bounds.as<SourceStats>();
    source_stats_kernel<<<nb, 256, 0, s>>>(p, m, n, st_dev + 1);
    CHUI_LAUNCH_CHECK("source_stats_kernel");
    stats_final_kernel<<<1, 256, 0, s>>>(st_dev + 1, nb, m, st_dev);
    CHUI_LAUNCH_CHECK("stats_final_kernel");
    FrameCheck fc{};
    for (int a = 0; a < 3; ++a) fc.L[a] = P.L[a];
    fc.expect_uniform = t.mass_uniform ? 1 : 0;
    fc.expect_mass = t.uniform_mass;
    frame_stats_kernel<<<1, 64, 0, s>>>(st_dev, m, fc, fr, safe ? P.fault : nullptr);
    CHUI_LAUNCH_CHECK("frame_stats_kernel");
    int unused[3] = {0, 0, 0};
    unwrap_dev = unwrap_axes(t, p, 3, n, P.L, unused, t.unwrap, s, fr);
    frame_root_kernel<<<1, 64, 0, s>>>(unwrap_dev, fr);
    CHUI_LAUNCH_CHECK("frame_root_kernel");
  }
  // Source checks, canonical flags and root cube on the host (from a read-back).
  auto take_stats = [&](const SourceStats& st) {
    if (st.bad_coord) throw std::invalid_argument("Periodic TreePM tree geometry requires finite source coordinates");
    if (st.bad_mass)
      throw std::invalid_argument("Tree gravity requires finite coordinates and finite non-negative masses");
    if (n == 0) return;
    t.mass_uniform = st.mass_nonuniform == 0;
    t.uniform_mass = st.mass0;
    for (int a = 0; a < 3; ++a) {
      const double lo = host_order_key_inv(st.lo[a]);
      const double hi = host_order_key_inv(st.hi[a]);
      t.unwrap.canonical[a] = (lo >= 0.0 && hi < P.L[a]) ? 1 : 0;  // tree_pm_coupling.cpp:3185-3195
    }
  };
  auto take_unwrap = [&]() {
    const UnwrapResult& U = t.unwrap;
    // Root cube (tree_gravity.cpp:443-452) from the unwrapped bounds.
    double ext = 0.0;
    for (int a = 0; a < 3; ++a) ext = std::max(ext, U.umax[a] - U.umin[a]);
    const double max_extent = std::max(ext, 1.0e-10);
    for (int a = 0; a < 3; ++a) t.root_centre[a] = 0.5 * (U.umin[a] + U.umax[a]);
    t.root_half = 0.5 * max_extent * (1.0 + 1.0e-8);
    for (int a = 0; a < 3; ++a) {
      ua.canonical[a] = U.canonical[a];
      ua.anchor[a] = U.anchor[a];
    }
  };
  if (!fr) {
    take_stats(compute_stats(t, p, m, n, s));
    if (n == 0) return;
    int canonical[3];
    for (int a = 0; a < 3; ++a) canonical[a] = t.unwrap.canonical[a];
    unwrap_axes(t, p, 3, n, P.L, canonical, t.unwrap, s, nullptr, P.size_for_capture);
    take_unwrap();
    if (P.size_for_capture) t.frame.reserve(sizeof(Frame));
  }

  // Path keys + stable sort.
  t.keys.reserve(n * sizeof(uint64_t));
  t.keys_alt.reserve(n * sizeof(uint64_t));
  t.order.reserve(n * sizeof(uint32_t));
  t.sort_vals.reserve(n * sizeof(uint32_t));
  t.vals_alt.reserve(n * sizeof(uint32_t));
  t.sort_scratch.reserve(radix_sort_scratch_bytes(n));
  PathArgs pa{};
  pa.u = ua;
  for (int a = 0; a < 3; ++a) pa.c0[a] = t.root_centre[a];
  pa.h0 = t.root_half;
  uint64_t* keys = t.keys.as<uint64_t>();
  uint32_t* vals = t.sort_vals.as<uint32_t>();
  t.pk.reserve(n * sizeof(double4));
  t.pk_in.reserve(n * sizeof(double4));
  path_key_kernel<<<grid_for(n, 256), 256, 0, s>>>(p, m, n, pa, keys, vals, t.pk_in.as<double4>(), fr);
  CHUI_LAUNCH_CHECK("path_key_kernel");
  // Sort by the digits of the last build's depth + 2 levels (16 in the first
  // build): the reference's partition order for every node up to that depth,
  // and the order inside a leaf is rebuilt below by (Morton key, row). If a
  // node of the last sorted level still splits, the keys are sorted on by all
  // 21 levels and the nodes counted again. A capture-safe build cannot: it
  // sorts by the prepared depth + 5 levels, and a deeper tree sets a fault bit.
  int levels = safe ? t.safe_levels : (t.level_hint > 0 ? t.level_hint : 16);
  auto sort_keys = [&](int from_level) {
    uint64_t* alt = keys == t.keys.as<uint64_t>() ? t.keys_alt.as<uint64_t>() : t.keys.as<uint64_t>();
    uint32_t* valt = vals == t.sort_vals.as<uint32_t>() ? t.vals_alt.as<uint32_t>() : t.sort_vals.as<uint32_t>();
    if (radix_sort_pairs_swap(keys, vals, alt, valt, n, 3 * (kPathLevels - from_level), 3 * kPathLevels,
                              t.sort_scratch.ptr, s)) {
      std::swap(keys, alt);
      std::swap(vals, valt);
    }
  };
  sort_keys(levels);

  const std::size_t initial_cap = std::max<std::size_t>(1024, n / 4 + 64);
  auto ensure = [&](std::size_t need) {
    if (need <= t.bfs_capacity && t.bfs_begin.ptr) return;
    const std::size_t nc = std::max({need, 2 * t.bfs_capacity, initial_cap});
    for (DeviceBuffer* b : {&t.bfs_begin, &t.bfs_count, &t.bfs_first_child, &t.bfs_nchild, &t.bfs_meta, &t.bfs_subtree,
                            &t.bfs_pre, &t.node_subs})
      b->reserve(nc * sizeof(uint32_t));
    t.bfs_geo.reserve(nc * sizeof(double4));
    t.bfs_capacity = nc;
  };
  if (!safe) ensure(initial_cap);
  NodeArgs na{};
  na.n = static_cast<uint32_t>(n);
  na.leaf_size = P.leaf_size;
  na.nblk = static_cast<uint32_t>((n + kNodeThreads - 1) / kNodeThreads);
  for (int a = 0; a < 3; ++a) na.c0[a] = t.root_centre[a];
  na.h0 = t.root_half;
  na.cut = static_cast<uint32_t>(std::max<std::size_t>(512, n / 1024));
  na.max_top = static_cast<uint32_t>(n / na.cut + 1);
  t.node_cld.reserve(n * sizeof(uint16_t));
  t.node_pbase.reserve(n * sizeof(uint32_t));
  t.node_cnt.reserve((static_cast<std::size_t>(na.nblk) + 1) * kNodeRows * sizeof(uint32_t));
  t.node_tops.reserve(static_cast<std::size_t>(na.max_top) * kMaxLevels * sizeof(uint32_t));
  t.level_dev.reserve(sizeof(BuildReport));
  BuildReport* rep = t.level_dev.as<BuildReport>();
  uint32_t* lv = rep->lv;
  uint32_t* cnt = t.node_cnt.as<uint32_t>();
  uint32_t* totals = cnt + static_cast<std::size_t>(na.nblk) * kNodeRows;
  std::size_t total = 0;  // node count, or the capacity for a capture-safe build
  for (;;) {
    na.sorted_levels = levels;
    na.capacity = static_cast<uint32_t>(std::min<std::size_t>(t.bfs_capacity, 0xFFFFFFFFull));
    fill_u32(lv + kLvTooDeep, 0u, kLvTops - kLvTooDeep, s);
    node_count_kernel<<<na.nblk, kNodeThreads, 0, s>>>(na, keys, t.node_cld.as<uint16_t>(), cnt, lv, fr);
    CHUI_LAUNCH_CHECK("node_count_kernel");
    exclusive_scan_rows(cnt, totals, kNodeRows, na.nblk, s);
    node_levels_kernel<<<1, 64, 0, s>>>(na, totals, rep, fr ? st_dev : nullptr, fr ? unwrap_dev : nullptr,
                                        safe ? P.fault : nullptr);
    CHUI_LAUNCH_CHECK("node_levels_kernel");
    if (safe) {
      total = na.capacity;
      break;
    }
    BuildReport h;
    t.readback.read(&h, rep, sizeof(h), s);
    if (fr) {
      take_stats(h.stats);
      for (int a = 0; a < 3; ++a) {
        t.unwrap.anchor[a] = h.unwrap.anchor[a];
        t.unwrap.umin[a] = h.unwrap.umin[a];
        t.unwrap.umax[a] = h.unwrap.umax[a];
      }
      take_unwrap();
    }
    if (h.lv[kLvDeepSplit]) {
      levels = kPathLevels;
      sort_keys(levels);
      continue;
    }
    if (h.lv[kLvTooDeep])
      throw UnsupportedError(
          "octree deeper than 21 levels (more than max_leaf_size coincident or near-coincident particles) "
          "is not built by the GPU path yet");
    total = h.lv[kLvTotal];
    ensure(total);
    na.capacity = static_cast<uint32_t>(std::min<std::size_t>(t.bfs_capacity, 0xFFFFFFFFull));
    t.max_depth = h.lv[kLvDepth];
    t.leaf_count = h.lv[kLvLeaves];
    t.level_hint = std::min(kPathLevels, static_cast<int>(t.max_depth) + 2);
    t.safe_levels = std::min(kPathLevels, static_cast<int>(t.max_depth) + 5);
    t.prepared_n = n;
    t.sized_for_capture = P.size_for_capture;
    break;
  }
  t.node_count = total;
  t.counts_on_device = safe;
  const uint32_t* total_dev = device_node_count(t);
  // node arrays: the node count, or the capacity when capture-safe builds follow
  const std::size_t nsz = P.size_for_capture ? std::max(total, t.bfs_capacity) : total;
  const NodeArrays nodes{t.bfs_begin.as<uint32_t>(),  t.bfs_count.as<uint32_t>(), t.bfs_first_child.as<uint32_t>(),
                         t.bfs_nchild.as<uint32_t>(), t.bfs_meta.as<uint32_t>(),  t.bfs_pre.as<uint32_t>(),
                         t.bfs_subtree.as<uint32_t>(), t.bfs_geo.as<double4>()};
  node_emit_kernel<<<na.nblk, kNodeThreads, 0, s>>>(na, keys, t.node_cld.as<uint16_t>(), cnt, lv, nodes,
                                                    t.node_pbase.as<uint32_t>(), fr);
  CHUI_LAUNCH_CHECK("node_emit_kernel");
  const unsigned node_grid = std::min<unsigned>(grid_for(total, 256), 65536u);
  node_links_kernel<<<node_grid, 256, 0, s>>>(na, keys, lv, nodes, t.node_pbase.as<uint32_t>(),
                                              t.node_subs.as<uint32_t>(), t.node_tops.as<uint32_t>());
  CHUI_LAUNCH_CHECK("node_links_kernel");
  // In-leaf Morton order (tree_ordering.cpp:151 extent with the 1e-12 floor)
  // and the tree-order copy of the sources.
  MortonArgs ma{};
  if (!fr) {
    const UnwrapResult& U = t.unwrap;
    double mext = 0.0;
    for (int a = 0; a < 3; ++a) {
      ma.lo[a] = U.umin[a];
      mext = std::max(mext, U.umax[a] - U.umin[a]);
    }
    ma.extent = std::max(mext, 1.0e-12);
  }
  double4* pk = t.pk.as<double4>();
  // Multipoles and tight particle boxes, the leaves' with their order, then bottom-up.
  t.bfs_mom.reserve(nsz * sizeof(double4));
  t.bfs_quad.reserve(nsz * 8 * sizeof(double));
  t.bfs_box.reserve(nsz * 6 * sizeof(double));
  MomArgs mo{};
  mo.u = ua;
  mo.quad = P.quadrupole ? 1 : 0;
  mo.done = P.leaf_size <= 16 ? 16u : P.leaf_size <= 32 ? 32u : 64u;  // lanes per leaf below
  const MomArrays mv{pk, nodes.begin, nodes.count, nodes.nchild, nodes.first_child, nodes.geo,
                     t.bfs_mom.as<double4>(), t.bfs_quad.as<double>(), t.bfs_box.as<double>()};
  auto order_leaves = [&](auto kernel, int lanes) {
    const unsigned grid = std::min<unsigned>(grid_for(total * lanes, 256), 65536u);
    kernel<<<grid, 256, 0, s>>>(static_cast<uint32_t>(total), total_dev, mo, mv, ma, t.pk_in.as<double4>(), vals,
                                t.order.as<uint32_t>(), pk, fr);
    CHUI_LAUNCH_CHECK("leaf_order_kernel");
  };
  if (mo.done == 16u) order_leaves(leaf_order_kernel<16>, 16);
  else if (mo.done == 32u) order_leaves(leaf_order_kernel<32>, 32);
  else order_leaves(leaf_order_kernel<64>, 64);
  moment_subtree_kernel<<<2048, 256, 0, s>>>(mo, mv, lv, t.node_subs.as<uint32_t>(), fr);
  CHUI_LAUNCH_CHECK("moment_subtree_kernel");
  moment_top_kernel<<<1, 1024, 0, s>>>(mo, mv, lv, t.node_tops.as<uint32_t>(), na.max_top);
  CHUI_LAUNCH_CHECK("moment_top_kernel");
  // Preorder records: links and, for mixed builds, the fixed-point records;
  // the FP64 records for FP64 builds (or later, on demand).
  t.link.reserve(nsz * sizeof(NodeLink));
  if (P.mixed) {
    t.geo32.reserve(nsz * sizeof(NodeGeo32));
    t.mom32.reserve(nsz * sizeof(NodeMom32));
    t.quad32.reserve(nsz * sizeof(NodeQuad32));
    t.box32.reserve(nsz * sizeof(NodeBox32));
  }
  t.wnode.reserve((nsz + kWalkNodePad) * sizeof(WalkNode));
  t.records64 = false;
  t.wnodes_current = false;
  t.cubic = (P.L[0] == P.L[1] && P.L[0] == P.L[2]);
  for (int a = 0; a < 3; ++a) t.fscale[a] = 4294967296.0 / P.L[a];
  launch_records(t, !P.mixed, P.mixed, s);
}

// ---- mesh-deposit units ---------------------------------------------------------
// The first cell a particle at unwrapped coordinate u writes (CIC: its cell;
// TSC: the cell below the nearest one); the deposit kernels wrap it into the
// mesh, so the tile of a box is [first(lo), first(hi) + span - 1] per axis.
__device__ __forceinline__ long deposit_first_cell(double u, double inv_h, int scheme) {
  const double g = u * inv_h;
  return scheme == 0 ? static_cast<long>(floor(g)) : static_cast<long>(floor(g + 0.5)) - 1;
}

__device__ bool deposit_tile(const double* box, const DepositTiling& d, int32_t lo[3], int32_t dims[3]) {
  const long span = d.scheme == 0 ? 2 : 3;
  long vol = 1;
  bool ok = true;
  for (int a = 0; a < 3; ++a) {
    const long l = deposit_first_cell(box[a], d.inv_h[a], d.scheme);
    const long ext = deposit_first_cell(box[3 + a], d.inv_h[a], d.scheme) + span - l;
    long w = l % d.n[a];
    if (w < 0) w += d.n[a];
    lo[a] = static_cast<int32_t>(w);
    ok = ok && ext <= d.n[a];
    dims[a] = ok ? static_cast<int32_t>(ext) : 0;
    vol *= ok ? ext : 1;
  }
  return ok && vol <= static_cast<long>(d.max_cells);
}

// Units form a cut of the tree: a node is one when it fits (or is a leaf) and
// its parent does not, so every particle lies in exactly one unit. The parent
// decides for its children; flags start at zero.
__global__ __launch_bounds__(256) void deposit_flag_kernel(uint32_t total_nodes, const uint32_t* __restrict__ total_dev,
                                                           const uint32_t* __restrict__ nchild,
                                                           const uint32_t* __restrict__ first_child,
                                                           const double* __restrict__ box, DepositTiling d,
                                                           uint32_t* __restrict__ flag) {
  const uint32_t total = total_dev ? *total_dev : total_nodes;
  for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < total; k += gridDim.x * blockDim.x) {
    int32_t lo[3], dims[3];
    const uint32_t c = nchild[k];
    const bool fits = deposit_tile(box + 6ull * k, d, lo, dims);
    if (k == 0) flag[0] = (fits || c == 0) ? 1u : 0u;
    if (fits || c == 0) continue;
    const uint32_t fc = first_child[k];
    for (uint32_t j = 0; j < c; ++j) {
      const uint32_t ch = fc + j;
      flag[ch] = (nchild[ch] == 0 || deposit_tile(box + 6ull * ch, d, lo, dims)) ? 1u : 0u;
    }
  }
}

__global__ __launch_bounds__(256) void deposit_emit_kernel(uint32_t total_nodes, const uint32_t* __restrict__ total_dev,
                                                           const uint32_t* __restrict__ flag,
                                                           const uint32_t* __restrict__ index,
                                                           const uint32_t* __restrict__ nb,
                                                           const uint32_t* __restrict__ nc,
                                                           const double* __restrict__ box, DepositTiling d,
                                                           DepositUnit* __restrict__ units,
                                                           uint32_t* __restrict__ blocks) {
  const uint32_t total = total_dev ? *total_dev : total_nodes;
  for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < total; k += gridDim.x * blockDim.x) {
    if (!flag[k]) continue;
    DepositUnit u;
    u.begin = nb[k];
    u.count = nc[k];
    if (!deposit_tile(box + 6ull * k, d, u.lo, u.dims)) u.dims[0] = 0;  // leaf spanning too many cells
    const uint32_t i = index[k];
    units[i] = u;
    blocks[i] = (u.count + d.chunk - 1) / d.chunk;
  }
}

DepositUnits build_deposit_units(Tree& t, const DepositTiling& d, hipStream_t s) {
  DepositUnits r;
  const std::size_t total = t.node_count;
  if (total == 0 || t.n == 0) return r;
  const std::size_t nsz = t.sized_for_capture ? std::max(total, t.bfs_capacity) : total;
  t.dep_flag.reserve(nsz * sizeof(uint32_t));
  t.dep_index.reserve(nsz * sizeof(uint32_t));
  t.dep_units.reserve(nsz * sizeof(DepositUnit));
  t.dep_blocks.reserve((nsz + 1) * sizeof(uint32_t));
  t.dep_scan.reserve(scan_scratch_bytes(nsz) + 64);
  t.dep_total.reserve(2 * sizeof(uint32_t));
  uint32_t* flag = t.dep_flag.as<uint32_t>();
  uint32_t* totals = t.dep_total.as<uint32_t>();  // [0] units, [1] blocks
  const uint32_t* total_dev = device_node_count(t);
  // counts left on the device: capture-safe builds, and sources few enough for
  // the two read-backs to matter (kFrameMax)
  const bool on_device = total_dev || t.n <= kFrameMax;
  fill_u32(flag, 0u, total, s);
  deposit_flag_kernel<<<grid_for(total, 256), 256, 0, s>>>(static_cast<uint32_t>(total), total_dev,
                                                           t.bfs_nchild.as<uint32_t>(),
                                                           t.bfs_first_child.as<uint32_t>(), t.bfs_box.as<double>(),
                                                           d, flag);
  CHUI_LAUNCH_CHECK("deposit_flag_kernel");
  exclusive_scan_u32(flag, t.dep_index.as<uint32_t>(), total, totals, t.dep_scan.ptr, s);
  if (on_device) fill_u32(t.dep_blocks.as<uint32_t>(), 0u, total, s);  // blocks past the last unit stay 0
  deposit_emit_kernel<<<grid_for(total, 256), 256, 0, s>>>(
      static_cast<uint32_t>(total), total_dev, flag, t.dep_index.as<uint32_t>(), t.bfs_begin.as<uint32_t>(),
      t.bfs_count.as<uint32_t>(), t.bfs_box.as<double>(), d, t.dep_units.as<DepositUnit>(),
      t.dep_blocks.as<uint32_t>());
  CHUI_LAUNCH_CHECK("deposit_emit_kernel");
  r.units = t.dep_units.as<DepositUnit>();
  r.first_block = t.dep_blocks.as<uint32_t>();
  if (on_device) {
    // scan the blocks of every node slot (zero past the last unit) and leave
    // both counts on the device; the deposit's grid is a fixed size that
    // strides over the real block count
    exclusive_scan_u32(t.dep_blocks.as<uint32_t>(), t.dep_blocks.as<uint32_t>(), total, totals + 1, t.dep_scan.ptr,
                       s);
    r.dev_counts = totals;
    r.count = 0;
    r.blocks = static_cast<uint32_t>(std::min<std::size_t>(total + t.n / d.chunk + 1, kDepositSafeGrid));
    return r;
  }
  uint32_t host[2] = {0, 0};
  t.readback.read(host, totals, sizeof(uint32_t), s);
  exclusive_scan_u32(t.dep_blocks.as<uint32_t>(), t.dep_blocks.as<uint32_t>(), host[0], totals + 1, t.dep_scan.ptr, s);
  t.readback.read(host + 1, totals + 1, sizeof(uint32_t), s);
  r.count = host[0];
  r.blocks = host[1];
  return r;
}

const uint32_t* device_node_count(const Tree& t) {
  return t.counts_on_device ? t.level_dev.as<BuildReport>()->lv + kLvTotal : nullptr;
}

void build_pos_of_row(Tree& t, hipStream_t s) {
  t.pos_of_row.reserve(std::max<std::size_t>(t.n, 1) * sizeof(uint32_t));
  if (t.n == 0) return;
  pos_of_row_kernel<<<grid_for(t.n, 256), 256, 0, s>>>(t.order.as<uint32_t>(), t.n, t.pos_of_row.as<uint32_t>());
  CHUI_LAUNCH_CHECK("pos_of_row_kernel");
}

void morton_order_device(Tree& t, const double* x, const double* y, const double* z, std::size_t n,
                         uint64_t* keys_sorted, uint32_t* order, hipStream_t s) {
  Axes3 p{{x, y, z}};
  const SourceStats st = compute_stats(t, p, nullptr, n, s);
  if (st.bad_coord) throw std::invalid_argument("Tree bounds requires finite particle coordinates");
  if (n == 0) return;
  MortonArgs ma{};
  double ext = 0.0;
  for (int a = 0; a < 3; ++a) {
    ma.lo[a] = host_order_key_inv(st.lo[a]);
    ext = std::max(ext, host_order_key_inv(st.hi[a]) - ma.lo[a]);
  }
  ma.extent = std::max(ext, 1.0e-12);
  t.keys_alt.reserve(n * sizeof(uint64_t));
  t.vals_alt.reserve(n * sizeof(uint32_t));
  t.sort_scratch.reserve(radix_sort_scratch_bytes(n));
  morton_keys_kernel<<<grid_for(n, 256), 256, 0, s>>>(p, n, ma, keys_sorted, order);
  CHUI_LAUNCH_CHECK("morton_keys_kernel");
  radix_sort_pairs(keys_sorted, order, t.keys_alt.as<uint64_t>(), t.vals_alt.as<uint32_t>(), n, 0, 63,
                   t.sort_scratch.ptr, s);
}

double unwrap_axis_device(Tree& t, const double* in, std::size_t n, double L, double* out, hipStream_t s) {
  if (!(std::isfinite(L) && L > 0.0))
    throw std::invalid_argument("Periodic TreePM tree geometry requires finite positive axis lengths");
  Axes3 p{{in, in, in}};
  const SourceStats st = compute_stats(t, p, nullptr, n, s);
  if (st.bad_coord) throw std::invalid_argument("Periodic TreePM tree geometry requires finite source coordinates");
  if (n == 0) return 0.0;
  const double lo = host_order_key_inv(st.lo[0]), hi = host_order_key_inv(st.hi[0]);
  int canonical[3] = {(lo >= 0.0 && hi < L) ? 1 : 0, 0, 0};
  double Ls[3] = {L, L, L};
  UnwrapResult r{};
  unwrap_axes(t, p, 1, n, Ls, canonical, r, s);
  unwrap_apply_kernel<<<grid_for(n, 256), 256, 0, s>>>(in, n, L, canonical[0], r.anchor[0], out);
  CHUI_LAUNCH_CHECK("unwrap_apply_kernel");
  return r.anchor[0];
}

}  // namespace chui
