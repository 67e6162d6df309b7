// spx_gravity.hpp -- TreeGravity on the device (3-D octree; 2-D quadtree).
//
// Tree: the reference's octree (Gravity/TreeGravityInline.hh:37-160, TreeGravity.cc:362-477)
// rebuilt from 60-bit Morton keys.  The level-l cell of a point is the l-level prefix of its
// key (floor(u*2^l) with u = (x - xmin)/boxLength is the prefix of floor(u*2^20), since the
// scaling is by a power of two), and the reference's split rule -- a cell is subdivided when a
// second point arrives, down to level 20 where points are listed -- gives: cells at level l are
// the l-prefix groups of points whose (l-1)-group holds at least two points.  Point p owns the
// cells (p, l) for l from 1 + lcp(p-1, p) to its leaf level min(20, 1 + max lcp with its
// sorted neighbours); numbering them by (p, l) is a pre-order walk, so each cell's subtree is
// the contiguous index range [c, skip[c]) and the force walk needs no stack.
//
// Walk: TreeGravity::applyTreeForces (TreeGravity.cc:818-950) per point from the root's
// daughters: accept a cell's monopole when |xcm - xi|^2 > cellsize^2/opening^2 + rcm2cc2,
// otherwise sum a leaf's points directly (self screened by r^2/soft^2 > 1e-10) or descend.
// Force M/(r^2+soft^2) along the unit vector, potential -M/sqrt(r^2+soft^2) in 3-D; in 2-D
// M/sqrt(r^2+soft^2) and -M log(sqrt(r^2+soft^2)) (TreeGravity.cc:54-90); then DvDt *= G,
// potential *= G, dt vote ftimestep*min sqrt(soft/|a|)/sqrt(G) (TreeGravity.cc:143-328,483-497).
//
// 2-D: the points get z = 0, so the interleaved keys' z bits are all zero and the octree's cells
// are exactly the quadtree's (level-l cell = floor(u*2^l) in x and y, TreeGravityInline.hh:16-33);
// the cell-centre offset rcm2cc2 is summed over x and y only.
#pragma once

#include <rocprim/rocprim.hpp>

#include <algorithm>
#include <vector>

#include "spx_device.hpp"
#include "spx_error.hpp"

namespace spx {

constexpr int kTreeBits = 20;   // deepest level (num1dbits - 1)

struct TreePoints { const double* x[3]; };
struct TreeBox { double lo[3], box; };       // cube of the tree: lower corner, edge

// Points up to which the keys are sorted by the sample sort below, and cells are allocated for the
// worst case (kTreeBits per point): building then takes no wait on the host, and the step is replayed
// from a graph.  The line bounds that worst case, 1.1 KB per point (usual trees have 1.4 to 1.7 of
// its 20 cells), 294 MB at 2^18.  Beyond it, the library's radix sort and a download of the cell count.
// It is no crossover: own / library, Evrard, build 117 / 177 us at 131k, 146 / 232 at 262k, 155 / 259
// at 300k, 286 / 381 at 800k, a step 1.34 / 1.47, 2.22 / 2.40, 2.55 / 2.83 and 6.41 / 6.65 ms.
constexpr int kTreeOwnSort = 1 << 18;
constexpr int kTreeBuckets = 1024;      // of the sort, half as many up to kTreeFewer points: as many
constexpr int kTreeFewer = 1 << 16;     // points are sampled, and one block sorts them
constexpr int kTreeBucketRoom = 16;     // mean bucket sizes up to which a bucket is sorted in LDS
constexpr int kTreeBoxBlocks = 256;
constexpr int kTreeChunk = 512;         // points per block of the cells' kernel
constexpr int kTreeCellsLds = 1280;     // cells of a chunk whose moments are kept in LDS
constexpr int kTreeTopUnits = 48;       // lists of 21 levels per block of k_tree_top

__device__ __forceinline__ int lcp_levels(uint64_t a, uint64_t b) {
  const uint64_t x = a ^ b;
  if (x == 0) return kTreeBits;
  const int lz = __clzll(x) - (64 - 3*kTreeBits);   // leading equal bits within the 60-bit key
  return lz/3;
}

// Every third bit of a key from bit 0 on, packed; and the inverse.
__device__ __forceinline__ uint64_t third_bits(uint64_t v) {
  v &= 0x1249249249249249ull;
  v = (v | v >> 2) & 0x10c30c30c30c30c3ull;
  v = (v | v >> 4) & 0x100f00f00f00f00full;
  v = (v | v >> 8) & 0x001f0000ff0000ffull;
  v = (v | v >> 16) & 0x001f00000000ffffull;
  return (v | v >> 32) & 0x1fffffull;
}
__device__ __forceinline__ uint64_t third_spread(uint64_t v) {
  v = (v | v << 32) & 0x001f00000000ffffull;
  v = (v | v << 16) & 0x001f0000ff0000ffull;
  v = (v | v << 8) & 0x100f00f00f00f00full;
  v = (v | v << 4) & 0x10c30c30c30c30c3ull;
  return (v | v << 2) & 0x1249249249249249ull;
}

// Extent of the points: per block and axis the minimum of x and of -x.
__global__ void __launch_bounds__(kBlock) k_tree_bbox(TreePoints xs, int n, double* part) {
  __shared__ double red[kBlock/64][6];
  double v[6];
#pragma unroll
  for (int q = 0; q < 6; ++q) v[q] = 1.7976931348623157e308;
  for (int i = blockIdx.x*kBlock + threadIdx.x; i < n; i += gridDim.x*kBlock)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const double x = xs.x[a][i];
      v[2*a] = fmin(v[2*a], x);
      v[2*a + 1] = fmin(v[2*a + 1], -x);
    }
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    for (int s = 32; s > 0; s >>= 1) v[q] = fmin(v[q], __shfl_xor(v[q], s));
    if (threadIdx.x % 64 == 0) red[threadIdx.x/64][q] = v[q];
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    double m = red[0][threadIdx.x];
    for (int w = 1; w < kBlock/64; ++w) m = fmin(m, red[w][threadIdx.x]);
    part[(size_t)blockIdx.x*6 + threadIdx.x] = m;
  }
}

__device__ __forceinline__ uint64_t tree_key(const TreePoints& xs, int i, const double* lo, double box) {
  const uint64_t ncell = 1ull << kTreeBits;
  uint64_t key = 0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    uint64_t c = 0;
    if (box > 0.0) {
      const double u = (xs.x[a][i] - lo[a])/box*(double)ncell;   // TreeGravityInline.hh buildCellKey
      c = u <= 0.0 ? 0 : (uint64_t)u;
      c = c < ncell - 1 ? c : ncell - 1;
    }
    key |= third_spread(c) << a;
  }
  return key;
}

// Order of the sort: by key, equal keys by index (as a stable sort leaves them).
__device__ __forceinline__ bool tree_less(uint64_t ka, uint32_t ia, uint64_t kb, uint32_t ib) {
  return ka < kb || (ka == kb && ia < ib);
}

// The block sorts key[0..cnt), id[0..cnt) in place by a bitonic network whose comparators all put
// the smaller first: entries beyond cnt count as larger than any and never move.
__device__ __forceinline__ void tree_bitonic(uint64_t* key, uint32_t* id, int cnt) {
  auto order = [&](int i, int j) {
    if (j >= cnt) return;
    const uint64_t a = key[i], b = key[j];
    const uint32_t p = id[i], q = id[j];
    if (tree_less(b, q, a, p)) {
      key[i] = b; key[j] = a;
      id[i] = q; id[j] = p;
    }
  };
  int lg = 0;
  while ((1 << lg) < cnt) ++lg;
  for (int k = 1; k <= lg; ++k) {
    const int half = 1 << (k - 1);
    for (int c = threadIdx.x; c < 1 << (lg - 1); c += blockDim.x) {
      const int g = (c >> (k - 1)) << k, o = c & (half - 1);
      order(g + o, g + 2*half - 1 - o);
    }
    __syncthreads();
    for (int h = k - 2; h >= 0; --h) {
      for (int c = threadIdx.x; c < 1 << (lg - 1); c += blockDim.x) {
        const int i = ((c >> h) << (h + 1)) | (c & ((1 << h) - 1));
        order(i, i + (1 << h));
      }
      __syncthreads();
    }
  }
}

// One entry per thread, in order over the block's first `size` threads (a power of two; the other
// entries end anywhere behind them): a bitonic network, by lane exchanges within wavefronts and
// through LDS across them.
__device__ __forceinline__ void tree_bitonic_lanes(uint64_t& key, uint32_t& id, int size, uint64_t* skey, uint32_t* sid) {
  const int t = threadIdx.x;
  for (int k = 2; k <= size; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      uint64_t ok;
      uint32_t oi;
      if (j >= 64) {
        skey[t] = key;
        sid[t] = id;
        __syncthreads();
        ok = skey[t ^ j];
        oi = sid[t ^ j];
        __syncthreads();
      } else {
        ok = __shfl_xor((unsigned long long)key, j);
        oi = __shfl_xor(id, j);
      }
      const bool low = ((t & j) == 0) == ((t & k) == 0);      // this thread keeps the smaller
      if (tree_less(ok, oi, key, id) == low) {
        key = ok;
        id = oi;
      }
    }
}

// One block: the cube from the blocks' extents; and, for the sample sort, its splitters
// (key, index), sampled points in order.  Clears the counters of the build.
template <int BUCKETS>
__global__ void __launch_bounds__(BUCKETS) k_tree_split(TreePoints xs, int n, const double* part, int nparts, bool sample,
                                                     TreeBox* out, uint64_t* splitKey, uint32_t* splitId, int* count) {
  __shared__ double ext[6];
  __shared__ uint64_t skey[BUCKETS];
  __shared__ uint32_t sid[BUCKETS];
  const int t = threadIdx.x;
  static_assert(BUCKETS >= 6*64);
  if (t/64 < 6) {
    double v = 1.7976931348623157e308;
    for (int b = t % 64; b < nparts; b += 64) v = fmin(v, part[(size_t)b*6 + t/64]);
    for (int s = 32; s > 0; s >>= 1) v = fmin(v, __shfl_xor(v, s));
    if (t % 64 == 0) ext[t/64] = v;
  }
  count[t] = 0;
  __syncthreads();
  const double lo[3] = {ext[0], ext[2], ext[4]};
  double box = 0.0;
#pragma unroll
  for (int a = 0; a < 3; ++a) box = fmax(box, fabs(-ext[2*a + 1] - lo[a]));
  if (t == 0) *out = TreeBox{{lo[0], lo[1], lo[2]}, box};
  if (!sample) return;
  const int ns = n < BUCKETS ? n : BUCKETS;
  uint64_t key = ~0ull;
  uint32_t id = ~0u;
  if (t < ns) {
    // one out of each of ns equal stretches, at a scrambled place: no period of the particles' order
    const int64_t i0 = (int64_t)t*n/ns, i1 = (int64_t)(t + 1)*n/ns;
    const int i = (int)(i0 + (int64_t)(((uint64_t)((uint32_t)t*2654435769u)*(uint64_t)(i1 - i0)) >> 32));
    key = tree_key(xs, i, lo, box);
    id = (uint32_t)i;
  }
  tree_bitonic_lanes(key, id, BUCKETS, skey, sid);
  splitKey[t] = key;
  splitId[t] = id;
}

// Keys alone, in particle order (for the library's sort).
__global__ void __launch_bounds__(kBlock) k_tree_codes(TreePoints xs, int n, const TreeBox* bx, uint64_t* codes,
                                                       uint32_t* idx) {
  const int i = blockIdx.x*kBlock + threadIdx.x;
  if (i >= n) return;
  codes[i] = tree_key(xs, i, bx->lo, bx->box);
  idx[i] = (uint32_t)i;
}

// Keys, and each point's bucket and place in it (any order: the bucket is sorted afterwards).  The
// block counts its points per bucket in LDS and reserves their places with one atomic each.
template <int BUCKETS>
__global__ void __launch_bounds__(kBlock) k_tree_rank(TreePoints xs, int n, const TreeBox* bx, const uint64_t* splitKey,
                                                      const uint32_t* splitId, int* count, uint64_t* codes, int2* slot) {
  __shared__ uint64_t sk[BUCKETS];
  __shared__ uint32_t si[BUCKETS];
  __shared__ int cnt[BUCKETS];
  for (int b = threadIdx.x; b < BUCKETS; b += kBlock) {
    sk[b] = splitKey[b];
    si[b] = splitId[b];
    cnt[b] = 0;
  }
  __syncthreads();
  const int i = blockIdx.x*kBlock + threadIdx.x;
  int b = 0, r = 0;
  if (i < n) {
    const uint64_t key = tree_key(xs, i, bx->lo, bx->box);
    codes[i] = key;
    for (int step = BUCKETS/2; step > 0; step >>= 1)
      if (!tree_less(key, (uint32_t)i, sk[b + step], si[b + step])) b += step;
    r = atomicAdd(&cnt[b], 1);
  }
  __syncthreads();
  for (int c = threadIdx.x; c < BUCKETS; c += kBlock)
    if (cnt[c] > 0) cnt[c] = atomicAdd(&count[c], cnt[c]);
  __syncthreads();
  if (i < n) slot[i] = make_int2(b, cnt[b] + r);
}

// Points into their buckets' places.
template <int BUCKETS>
__global__ void __launch_bounds__(kBlock) k_tree_scatter(int n, const int* count, const uint64_t* codes, const int2* slot,
                                                         uint64_t* keys, uint32_t* idx) {
  constexpr int per = BUCKETS/kBlock;
  __shared__ int start[BUCKETS];
  __shared__ int wsum[kBlock/64];
  const int t = threadIdx.x;
  int own[per], sum = 0;
#pragma unroll
  for (int k = 0; k < per; ++k) { own[k] = sum; sum += count[t*per + k]; }
  int incl = sum;
  for (int s = 1; s < 64; s <<= 1) { const int o = __shfl_up(incl, s); if (t % 64 >= s) incl += o; }
  if (t % 64 == 63) wsum[t/64] = incl;
  __syncthreads();
  int base = incl - sum;
  for (int w = 0; w < t/64; ++w) base += wsum[w];
#pragma unroll
  for (int k = 0; k < per; ++k) start[t*per + k] = base + own[k];
  __syncthreads();
  const int i = blockIdx.x*kBlock + t;
  if (i >= n) return;
  const int2 s = slot[i];
  const int p = start[s.x] + s.y;
  keys[p] = codes[i];
  idx[p] = (uint32_t)i;
}

// A point into tree order: position, mass, and the walk's record of a listed point, (x, y), (z, m).
struct TreeOrder {
  double* x[3];
  double* m;
  double2* tp;
};
__device__ __forceinline__ void tree_place(const TreePoints& xs, const double* m, uint32_t q, int p, const TreeOrder& o) {
  const double x = xs.x[0][q], y = xs.x[1][q], z = xs.x[2][q], mq = m[q];
  o.x[0][p] = x; o.x[1][p] = y; o.x[2][p] = z;
  o.m[p] = mq;
  o.tp[2*(size_t)p] = make_double2(x, y);
  o.tp[2*(size_t)p + 1] = make_double2(z, mq);
}
__global__ void __launch_bounds__(kBlock) k_tree_gather(TreePoints xs, const double* m, const uint32_t* perm, int n,
                                                        TreeOrder o) {
  const int p = blockIdx.x*kBlock + threadIdx.x;
  if (p < n) tree_place(xs, m, perm[p], p, o);
}

// One block per bucket sorts it: in registers, in LDS or, where far more points than expected fell
// between two splitters, in place in memory; then the points go into tree order.
template <int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_tree_sort(const int* count, int room, uint64_t* keys, uint32_t* idx, TreePoints xs,
                                                     const double* m, uint64_t* codes, uint32_t* perm, TreeOrder o) {
  extern __shared__ char shared[];
  uint64_t* key = reinterpret_cast<uint64_t*>(shared);
  uint32_t* id = reinterpret_cast<uint32_t*>(key + room);
  __shared__ int wsum[BLOCK/64];
  const int t = threadIdx.x, cnt = count[blockIdx.x];
  if (cnt == 0) return;
  int before = 0;
  for (int b = t; b < (int)blockIdx.x; b += BLOCK) before += count[b];
  for (int s = 32; s > 0; s >>= 1) before += __shfl_xor(before, s);
  if (t % 64 == 0) wsum[t/64] = before;
  __syncthreads();
  before = 0;
  for (int w = 0; w < BLOCK/64; ++w) before += wsum[w];
  uint64_t* gk = keys + before;
  uint32_t* gi = idx + before;
  if (cnt <= BLOCK) {
    uint64_t k = ~0ull;
    uint32_t q = ~0u;
    if (t < cnt) { k = gk[t]; q = gi[t]; }
    int size = 1;
    while (size < cnt) size <<= 1;
    tree_bitonic_lanes(k, q, size, key, id);
    if (t < cnt) {
      codes[before + t] = k;
      perm[before + t] = q;
      tree_place(xs, m, q, before + t, o);
    }
    return;
  }
  const bool inLds = cnt <= room;
  if (inLds) {
    for (int j = t; j < cnt; j += BLOCK) { key[j] = gk[j]; id[j] = gi[j]; }
    __syncthreads();
    tree_bitonic(key, id, cnt);
  } else {
    tree_bitonic(gk, gi, cnt);
  }
  for (int j = t; j < cnt; j += BLOCK) {
    const uint32_t q = inLds ? id[j] : gi[j];
    codes[before + j] = inLds ? key[j] : gk[j];
    perm[before + j] = q;
    tree_place(xs, m, q, before + j, o);
  }
}

// The cells that sorted point p heads: levels start .. leaf (none if start > leaf).
struct TreeHead {
  int start, leaf, after;       // after: levels shared with the next point, -1 at the end
  __device__ int count() const { return leaf >= start ? leaf - start + 1 : 0; }
};
__device__ __forceinline__ TreeHead tree_head(const uint64_t* code, int p, int n, uint64_t key) {
  const int lp = p > 0 ? lcp_levels(code[p - 1], key) : -1;
  const int ln = p + 1 < n ? lcp_levels(key, code[p + 1]) : -1;
  TreeHead h;
  h.leaf = min(1 + max(lp, ln), kTreeBits);
  if (n == 1) h.leaf = 0;
  h.start = p == 0 ? 0 : 1 + lp;
  h.after = ln;
  return h;
}

template <int BLOCK>
__device__ __forceinline__ int block_sum(int v, int* wsum) {
  for (int s = 32; s > 0; s >>= 1) v += __shfl_xor(v, s);
  if (threadIdx.x % 64 == 0) wsum[threadIdx.x/64] = v;
  __syncthreads();
  v = 0;
  for (int w = 0; w < BLOCK/64; ++w) v += wsum[w];
  __syncthreads();
  return v;
}

// Cells headed by the points of each chunk.
__global__ void __launch_bounds__(kTreeChunk) k_tree_count(const uint64_t* code, int n, int* total) {
  __shared__ int wsum[kTreeChunk/64];
  const int p = blockIdx.x*kTreeChunk + threadIdx.x;
  const int c = block_sum<kTreeChunk>(p < n ? tree_head(code, p, n, code[p]).count() : 0, wsum);
  if (threadIdx.x == 0) total[blockIdx.x] = c;
}

// A cell as the walk reads it, in one record: the centre of mass, the mass, the opening radius^2
// l^2/theta^2 + |xcm - centre|^2 for the walk's opening angle, the next cell behind its subtree,
// and what a point too close for the monopole does with it: open it (kCellOpen), take its one
// point (kCellPoint) or, at the deepest level, take its list of points (kCellList).
enum : int { kCellOpen = 0, kCellPoint = 1, kCellList = 2 };
struct alignas(16) TreeCell {
  double x, y, z, M;
  double open;
  int skip, kind;
};
static_assert(sizeof(TreeCell) == 48, "TreeCell is read as three 16-byte words");

// What the cells are formed with: the walk's opening angle^2 and self-screen radius^2, dimension.
struct TreeShape {
  const TreeBox* bx;
  double open2, self2;
  int dim, n;
  TreeCell* cells;
  int *first, *last;            // point range of the cells of kind kCellList
};

// Cell coordinates of a key at the deepest level.
struct TreeCoord { uint32_t i[3]; };
__device__ __forceinline__ TreeCoord tree_coord(uint64_t key) {
  return TreeCoord{{(uint32_t)third_bits(key), (uint32_t)third_bits(key >> 1), (uint32_t)third_bits(key >> 2)}};
}

// The record of cell c at level l that holds points p..end-1 (only lists need the exact end).
__device__ __forceinline__ void tree_store(const TreeShape& f, int c, int l, const TreeCoord& at, int p, int end, int skip,
                                           double m, double x, double y, double z) {
  const double cs = ldexp(f.bx->box, -l), xc[3] = {x, y, z};
  double r2 = 0.0;
#pragma unroll
  for (int a = 0; a < 3; ++a)
    if (a < f.dim) {
      const double d = xc[a] - fused(cs, (double)(at.i[a] >> (kTreeBits - l)) + 0.5, f.bx->lo[a]);
      r2 = fused(d, d, r2);
    }
  TreeCell t{x, y, z, m, ldexp(rounded_product(f.bx->box, f.bx->box), -2*l)/f.open2 + r2, skip, kCellOpen};
  // A one-point cell acts through its monopole from its opening radius on and as its point down
  // to the self screen, by the same formula: one radius.  (Below 1e-100 the formulas differ, and
  // such a cell keeps both, the point in a list of one.)
  const bool one = end == p + 1;
  if (one && t.open >= 1.0e-100) {
    t.kind = kCellPoint;
    t.open = fmin(t.open, f.self2);
  } else if (one || l == kTreeBits) {
    t.kind = kCellList;
    f.first[c] = p;
    f.last[c] = end - 1;
  }
  f.cells[c] = t;
}

// A cell whose points reach beyond the chunk of its first one.
struct alignas(16) TreeTop {
  int c, p, end, skip;
  int child[8];                 // per octant: its first point, then its cell; -1: empty
};

// First point in [p, n) whose key is at least v: four ways per step, as a step is one read's latency.
__device__ __forceinline__ int tree_bound(const uint64_t* code, int p, int n, uint64_t v) {
  while (p < n) {
    const int len = n - p, a = p + len/4, b = p + len/2, c = p + (int)(3*(int64_t)len/4);
    const uint64_t ka = code[a], kb = code[b], kc = code[c];
    if (kc < v) p = c + 1;
    else if (kb < v) { p = b + 1; n = c; }
    else if (ka < v) { p = a + 1; n = b; }
    else n = a;
  }
  return p;
}

// The cells headed by a chunk of points, with all that lies within the chunk: numbers by a scan on
// top of the chunks before, ranges by search in the keys in LDS, moments level by level from the
// daughters in LDS (in memory where deep chains give the chunk more than kTreeCellsLds cells),
// summed in the daughters' order.  Cells that reach beyond the chunk (at most one per level) are
// listed with their daughters for k_tree_top.  One launch instead of one per level: see build().
__global__ void __launch_bounds__(kTreeChunk) k_tree_cells(TreeShape f, const uint64_t* code, TreeOrder o,
                                                           const int* total, const int* before, int* cstart, int* ncells,
                                                           TreeTop* top) {
  __shared__ uint64_t key[kTreeChunk];
  __shared__ int at[kTreeChunk + 1], skips[kTreeCellsLds + 1];
  __shared__ double lm[kTreeCellsLds], lx[kTreeCellsLds], ly[kTreeCellsLds], lz[kTreeCellsLds];
  __shared__ int wsum[kTreeChunk/64], topHead[kTreeBits + 1];
  __shared__ unsigned levels;
  const int t = threadIdx.x, n = f.n, s = blockIdx.x*kTreeChunk, nloc = min(kTreeChunk, n - s), p = s + t;
  const uint64_t kk = t < nloc ? code[p] : 0;
  key[t] = kk;
  if (t <= kTreeBits) topHead[t] = -1;
  if (t == 0) levels = 0;
  TreeHead h{1, 0, -1};
  if (t < nloc) h = tree_head(code, p, n, kk);
  const int nh = h.count();
  int base = 0;
  if (before) base = before[blockIdx.x];
  else for (int b = t; b < (int)blockIdx.x; b += kTreeChunk) base += total[b];
  if (!before) base = block_sum<kTreeChunk>(base, wsum);
  int incl = nh;
  for (int d = 1; d < 64; d <<= 1) { const int u = __shfl_up(incl, d); if (t % 64 >= d) incl += u; }
  if (t % 64 == 63) wsum[t/64] = incl;
  __syncthreads();
  int j0 = incl - nh, nc = 0;
  for (int w = 0; w < kTreeChunk/64; ++w) {
    if (w < t/64) j0 += wsum[w];
    nc += wsum[w];
  }
  at[t] = j0;
  if (t == 0) at[kTreeChunk] = nc;
  const int e = s + nloc;                       // the next chunk's first point
  if (t < nloc) cstart[p] = base + j0;
  if (e == n && t == 0) {
    cstart[n] = *ncells = base + nc;
    f.cells[base + nc] = TreeCell{0.0, 0.0, 0.0, 0.0, INFINITY, base + nc, kCellPoint};   // nothing acts
  }
  const int out = nh > 0 && e < n ? lcp_levels(kk, code[e]) : -1;   // levels whose cells reach beyond
  for (int l = h.start; l <= min(out, h.leaf); ++l) topHead[l] = t;
  const bool inLds = nc <= kTreeCellsLds;
  __syncthreads();
  const bool single = h.after < h.leaf;         // the leaf holds this point alone
  // Levels at which this thread's cell has its moments formed from daughters (or a list): those
  // within the chunk.  skips: the next cell behind the subtree, and the cell's level below it.
  const int fine = h.leaf - (single ? 1 : 0), coarse = max(h.start, out + 1);
  const unsigned mine = nh > 0 && fine >= coarse ? (2u << fine) - (1u << coarse) : 0u;
  if (mine) atomicOr(&levels, mine);
  const TreeCoord coord = tree_coord(kk);
  if (inLds) {
    for (int k = 0; k < nh; ++k) skips[j0 + k] = h.start + k;
    if (t == 0) skips[nc] = 0;                  // ends any subtree
  }
  if (nh > 0 && single) {
    const int j = j0 + nh - 1;
    const double m = o.m[p], x = o.x[0][p], y = o.x[1][p], z = o.x[2][p];
    if (inLds) { lm[j] = m; lx[j] = x; ly[j] = y; lz[j] = z; skips[j] |= (j + 1) << 5; }
    tree_store(f, base + j, h.leaf, coord, p, p + 1, base + j + 1, m, x, y, z);
  }
  __syncthreads();
  int lo = t;                                   // the last point found so far, of the finer level
  for (unsigned todo = levels; todo;) {
    const int l = 31 - __clz(todo);
    todo ^= 1u << l;
    __syncthreads();
    if (!(mine >> l & 1)) continue;
    const int j = j0 + l - h.start;
    int je = j + 1;
    if (l == kTreeBits || !inLds) {
      const int sh = 3*(kTreeBits - l);
      int hi = nloc - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (key[mid] >> sh == kk >> sh) lo = mid; else hi = mid - 1;
      }
      je = at[lo + 1];
    }
    double m = 0.0, x = 0.0, y = 0.0, z = 0.0;
    if (l == kTreeBits) {
      for (int q = p; q <= s + lo; ++q) {
        const double mq = o.m[q];
        m += mq;
        x = fused(mq, o.x[0][q], x);
        y = fused(mq, o.x[1][q], y);
        z = fused(mq, o.x[2][q], z);
      }
    } else if (inLds) {
      // the daughters' subtrees end where a cell of level <= l starts
      for (int sk = skips[je]; (sk & 31) > l;) {
        const int to = sk >> 5;
        sk = skips[to];
        const double md = lm[je];
        m += md;
        x = fused(md, lx[je], x);
        y = fused(md, ly[je], y);
        z = fused(md, lz[je], z);
        je = to;
      }
    } else {
      for (int d = base + j + 1; d < base + je;) {
        const TreeCell q = f.cells[d];
        m += q.M;
        x = fused(q.M, q.x, x);
        y = fused(q.M, q.y, y);
        z = fused(q.M, q.z, z);
        d = q.skip;
      }
    }
    x /= m;
    y /= m;
    z /= m;
    if (inLds) { lm[j] = m; lx[j] = x; ly[j] = y; lz[j] = z; skips[j] = je << 5 | l; }
    tree_store(f, base + j, l, coord, p, l == kTreeBits ? s + lo + 1 : p + 2, base + je, m, x, y, z);
  }
  // Rows of 16 lanes: one level's listed cell each, a lane per octant and one for the end.
  const int l = t/16, r = t % 16;
  if (l > kTreeBits) return;
  TreeTop* w = top + (size_t)blockIdx.x*(kTreeBits + 1) + l;
  const int q = topHead[l], sh = 3*(kTreeBits - l);
  if (q < 0) {
    if (r == 9) w->c = -1;
    return;
  }
  const uint64_t pre = key[q] >> sh;
  if (r < 8) {
    int c = -1;
    if (l < kTreeBits) {
      const uint64_t want = pre << 3 | (uint64_t)r;
      c = tree_bound(code, s + q, n, want << (sh - 3));
      if (c >= n || code[c] >> (sh - 3) != want) c = -1;
    }
    w->child[r] = c;
  } else if (r == 8) {
    w->end = tree_bound(code, s + q, n, (pre + 1) << sh);
  } else if (r == 9) {
    w->p = s + q;
    w->c = base + at[q] + l - tree_head(code, s + q, n, key[q]).start;
  }
}

// The listed cells of kTreeTopUnits units (chunks at first), `span` points each, that end within
// them: moments level by level, a thread per cell.  Cells that reach on are listed for the next
// launch, in which these units are one (again at most one cell per level).  first: the daughters
// are still points.
__global__ void __launch_bounds__(1024) k_tree_top(TreeShape f, const uint64_t* code, TreeOrder o, int units, int64_t span,
                                                   bool first, const int* cstart, const int* ncells, const TreeTop* top,
                                                   TreeTop* up) {
  __shared__ unsigned levels;
  // by level, so that a level's cells are in one or two wavefronts
  const int t = threadIdx.x, l = t/kTreeTopUnits, u = blockIdx.x*kTreeTopUnits + t % kTreeTopUnits;
  const bool slot = l <= kTreeBits && u < units;
  TreeTop w{-1};
  if (slot) w = top[(size_t)u*(kTreeBits + 1) + l];
  if (t == 0) levels = 0;
  if (t <= kTreeBits) up[(size_t)blockIdx.x*(kTreeBits + 1) + t].c = -1;
  if (first && w.c >= 0) {
    int child[8];
#pragma unroll
    for (int a = 0; a < 8; ++a) child[a] = cstart[max(w.child[a], 0)];
    w.skip = w.end < f.n ? cstart[w.end] : *ncells;
#pragma unroll
    for (int a = 0; a < 8; ++a)
      if (w.child[a] >= 0) w.child[a] = w.child[a] == w.p ? w.c + 1 : child[a];
  }
  const bool here = w.c >= 0 && (blockIdx.x + 1 == gridDim.x || w.end <= (blockIdx.x + 1)*kTreeTopUnits*span);
  __syncthreads();
  if (w.c >= 0 && !here) up[(size_t)blockIdx.x*(kTreeBits + 1) + l] = w;
  if (here) atomicOr(&levels, 1u << l);
  __syncthreads();
  for (unsigned todo = levels; todo;) {
    const int lvl = 31 - __clz(todo);
    todo ^= 1u << lvl;
    __syncthreads();
    if (!here || l != lvl) continue;
    double m = 0.0, x = 0.0, y = 0.0, z = 0.0;
    if (l == kTreeBits) {
      for (int q = w.p; q < w.end; ++q) {
        const double mq = o.m[q];
        m += mq;
        x = fused(mq, o.x[0][q], x);
        y = fused(mq, o.x[1][q], y);
        z = fused(mq, o.x[2][q], z);
      }
    } else {
      double2 xy[8], zm[8];
#pragma unroll
      for (int a = 0; a < 8; ++a) {
        const double2* d = reinterpret_cast<const double2*>(f.cells + max(w.child[a], 0));
        xy[a] = d[0];
        zm[a] = d[1];
      }
#pragma unroll
      for (int a = 0; a < 8; ++a)
        if (w.child[a] >= 0) {
          m += zm[a].y;
          x = fused(zm[a].y, xy[a].x, x);
          y = fused(zm[a].y, xy[a].y, y);
          z = fused(zm[a].y, zm[a].x, z);
        }
    }
    tree_store(f, w.c, l, tree_coord(code[w.p]), w.p, w.end, w.skip, m, x/m, y/m, z/m);
  }
}

// Neighbouring points that walk the tree together.  In a group of four a wavefront reads 16 records
// per step instead of 64 but visits the cells that any of the four needs (21 to 42 % more steps
// than a point by itself).  With many wavefronts per SIMD the reads count, with few the number of
// dependent steps.  Evrard collapse, per walk with 1 / 2 / 4 together: 16k points 312 / 386 / 428 us,
// 60k 371 / 476 / 550, 120k 665 / 620 / 665, 250k 1293 / 1055 / 928; uniform sphere of 33k with a
// wide opening angle 69 / 102 / 115.  The line is at 1.5 wavefronts per SIMD.  Same bits either way.
constexpr int kTreeGroup = 4;
constexpr int kTreeAlone = 98304;

// Minimum over a point by itself or over each quad of lanes (quad permutes [1,0,3,2], [2,3,0,1]).
template <int GROUP>
__device__ __forceinline__ int group_min(int v) {
  static_assert(GROUP == 1 || GROUP == 4);
  if (GROUP == 4) {
    v = min(v, __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true));
    v = min(v, __builtin_amdgcn_mov_dpp(v, 0x4E, 0xf, 0xf, true));
  }
  return v;
}

// applyTreeForces for the point in tree slot p; results scattered to its hydro slot.
// GROUP neighbouring points walk the pre-order cells together: each lane keeps the next cell its
// own walk would visit, the group visits the smallest of them, and only the lanes waiting on that
// cell act on it.  Every lane therefore takes exactly the decisions, in exactly the order, of an
// independent stackless walk (same bits).  A wavefront walks 64/GROUP groups side by side.
//
// Bound by the vector instructions of a step (58 per visited cell) while wavefronts are plenty and
// by a step's chain -- read a record, compare, choose the next -- where they are not.  So the next
// record is requested before the force of the present one is formed, the record is 48 bytes, and
// the decision is one comparison: the self screen's division became a radius, and a one-point
// cell's two radii one (tree_store).  250k Evrard 1591 -> 928 us per walk, 33k sphere 202 -> 69
// (with the point by itself).  COUNT (a measurement variant, never in a step): counts each point's
// monopole (accepted cell) and point-point interactions into counts[2p], counts[2p+1].
template <int GROUP, bool COUNT = false, int DIM = 3>
__global__ void __launch_bounds__(kBlock) k_tree_walk(
    const double* __restrict__ tx0, const double* __restrict__ tx1, const double* __restrict__ tx2,
    const double2* __restrict__ tp, const TreeCell* __restrict__ cells, const int* __restrict__ first,
    const int* __restrict__ last, const int* __restrict__ pncells, int npts, const uint32_t* __restrict__ perm, double soft2, double self2,
    double soft, double G, double* __restrict__ acc0, double* __restrict__ acc1, double* __restrict__ acc2,
    double* __restrict__ pot, double* __restrict__ blockMin, unsigned long long* __restrict__ counts = nullptr) {
  const int p = blockIdx.x*blockDim.x + threadIdx.x;
  const int ncells = *pncells;
  unsigned long long nCell = 0, nPoint = 0;
  const bool valid = p < npts;
  double dtv = 1.7976931348623157e308;
  double xi = 0.0, yi = 0.0, zi = 0.0;
  if (valid) { xi = tx0[p]; yi = tx1[p]; zi = tx2[p]; }
  double ax = 0.0, ay = 0.0, az = 0.0, phi = 0.0;
  int next = valid ? 1 : ncells;
  int c = group_min<GROUP>(next);
  const double2* cr = reinterpret_cast<const double2*>(cells + c);
  double2 c01 = cr[0], c23 = cr[1], c45 = cr[2];
  // every iteration moves the group's smallest pending cell strictly forward, so a walk
  // ends within ncells iterations; the bound only guards the loop
  for (int guard = 0; guard <= ncells; ++guard) {
    const double Mc = c23.y;
    const int sk = __double2loint(c45.y), kind = __double2hiint(c45.y);
    const double dx = c01.x - xi, dy = c01.y - yi, dz = c23.x - zi;
    const double r2 = fused(dz, dz, fused(dy, dy, rounded_product(dx, dx)));
    const bool mine = next == c;
    const bool acts = mine && r2 > c45.x;
    const bool list = mine && !acts && kind == kCellList;
    const int own = c;
    if (mine) next = acts || kind != kCellOpen ? sk : c + 1;
    // The next cell's record is on its way while this one's force is formed.  A group that is
    // done stays at the record behind the last cell, on which nothing acts.
    c = group_min<GROUP>(next);
    cr = reinterpret_cast<const double2*>(cells + c);
    c01 = cr[0];
    c23 = cr[1];
    c45 = cr[2];
    if (acts) {
      // 1/|r| and 1/sqrt(r^2 + s^2) from reciprocal square roots (the force is M/(r^2 + s^2) along
      // r/|r|, the potential -M/sqrt(r^2 + s^2)).
      const double rs = r2 + soft2;
      double inv = fast_rsqrt(r2), ri = fast_rsqrt(rs);
      double nx = dx*inv, ny = dy*inv, nz = dz*inv;
      if (!(r2 > 1.0e-100 && rs < 1.0e300)) {      // coincident with the cell, or out of the estimate's range
        const bool far = kind == kCellPoint || r2 > 1.0e-100;
        inv = far ? rsqrt(r2) : 0.0;
        ri = rsqrt(rs);
        nx = far ? dx*inv : 1.0;
        ny = dy*inv;
        nz = dz*inv;
      }
      const double f = DIM == 3 ? Mc*(ri*ri) : Mc*ri;
      ax = fused(f, nx, ax);
      ay = fused(f, ny, ay);
      az = fused(f, nz, az);
      phi = DIM == 3 ? fused(-Mc, ri, phi) : phi - Mc*(0.5*log(rs));
      if (COUNT) ++nCell;
    }
    if (COUNT && mine && own < ncells && !acts && kind == kCellPoint && r2 > self2) ++nPoint;
    if (list) {
      const int q1 = last[own];
      for (int q = first[own]; q <= q1; ++q) {
        const double2 pa = tp[2*(size_t)q], pb = tp[2*(size_t)q + 1];
        const double ex = pa.x - xi, ey = pa.y - yi, ez = pb.x - zi;
        const double q2 = fused(ez, ez, fused(ex, ex, rounded_product(ey, ey)));
        if (q2 > self2) {
          const double inv = rsqrt(q2);
          const double rs = q2 + soft2;
          const double mq = pb.y;
          const double ri = rsqrt(rs);
          const double f = DIM == 3 ? mq*(ri*ri) : mq*ri;
          ax = fused(f, ex*inv, ax);
          ay = fused(f, ey*inv, ay);
          az = fused(f, ez*inv, az);
          phi = DIM == 3 ? fused(-mq, ri, phi) : phi - mq*(0.5*log(rs));
          if (COUNT) ++nPoint;
        }
      }
    }
    if (__all(c >= ncells)) break;               // every group is done
  }
  if (valid) {
    const double amag = sqrt(ax*ax + ay*ay + az*az);
    if (amag > 0.0) dtv = sqrt(soft/amag);
    const uint32_t s = perm[p];
    acc0[s] = G*ax;
    acc1[s] = G*ay;
    acc2[s] = G*az;
    pot[s] = G*phi;
    if (COUNT) { counts[2*(size_t)p] = nCell; counts[2*(size_t)p + 1] = nPoint; }
  }
  __shared__ double red[kBlock];
  red[threadIdx.x] = dtv;
  __syncthreads();
  for (int s = kBlock/2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] = fmin(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) blockMin[blockIdx.x] = red[0];
}

__global__ void k_tree_dt(const double* blockMin, int nb, Scalars* sc, double G, double ftimestep) {
  __shared__ double red[kBlock];
  double m = 1.7976931348623157e308;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) m = fmin(m, blockMin[b]);
  red[threadIdx.x] = m;
  __syncthreads();
  for (int s = kBlock/2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] = fmin(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    sc->dtMinAcc = red[0]/sqrt(G);
    sc->gravDt = ftimestep*sc->dtMinAcc;
  }
}

class GravityTree {
 public:
  int D = 3;
  int64_t n = 0;
  hipStream_t stream = nullptr;
  bool active = false;
  std::vector<void*> allocs;
  int64_t bytes = 0;                // device memory the tree holds
  uint64_t *codes = nullptr, *keys = nullptr, *codesSorted = nullptr;
  uint32_t *idx = nullptr, *perm = nullptr;
  int2* slot = nullptr;
  uint64_t* splitKey = nullptr;
  uint32_t* splitId = nullptr;
  int *count = nullptr, *chunkTotal = nullptr, *chunkBefore = nullptr, *ncells = nullptr;
  TreeTop *top = nullptr, *topNext = nullptr;
  TreeOrder order{};                // points in tree order
  TreeBox* box = nullptr;
  int* cstart = nullptr;
  void* tmp = nullptr;
  size_t tmpBytes = 0;
  double* part = nullptr;
  double* zero = nullptr;           // 2-D: the z coordinate of every point
  double* sink = nullptr;           // 2-D: the walk's z acceleration
  int64_t cellCap = 0;
  TreeCell* cells = nullptr;        // the walk's cell records
  int *first = nullptr, *last = nullptr;
  int cellsAllocs = 0;              // how often they were allocated
  int npts = 0;                     // points of the tree (0: none yet)
  // opening^2 (< 0: none) and self-screen radius^2 that the cell records were formed for
  double cellsOpen2 = -1.0, cellsSelf2 = 0.0;

  template <typename T>
  T* alloc(size_t count) {
    void* p = nullptr;
    const size_t b = std::max<size_t>(count, 1)*sizeof(T);
    HIP_CHECK(hipMalloc(&p, b));
    allocs.push_back(p);
    bytes += (int64_t)b;
    return static_cast<T*>(p);
  }

  void init(int dim, int64_t n_, int ld, hipStream_t s, bool enabled) {
    D = dim;
    n = n_;
    stream = s;
    active = enabled;
    if (!active) return;
    if (D != 3 && D != 2) raise(SPX_ERR_UNSUPPORTED, "TreeGravity on the GPU is implemented for 2-D and 3-D");
    (void)ld;
    if (D == 2) {
      // z = 0 for every point (the quadtree as a flat octree), and a sink for the z acceleration
      zero = alloc<double>(n);
      HIP_CHECK(hipMemsetAsync(zero, 0, (size_t)std::max<int64_t>(n, 1)*sizeof(double), stream));
      sink = alloc<double>(n);
    }
    const int64_t small = std::min<int64_t>(n, kTreeOwnSort), nchunk = (n + kTreeChunk - 1)/kTreeChunk;
    codes = alloc<uint64_t>(n);
    keys = alloc<uint64_t>(small);
    codesSorted = alloc<uint64_t>(n);
    idx = alloc<uint32_t>(n);
    perm = alloc<uint32_t>(n);
    slot = alloc<int2>(small);
    splitKey = alloc<uint64_t>(kTreeBuckets);
    splitId = alloc<uint32_t>(kTreeBuckets);
    count = alloc<int>(kTreeBuckets);
    chunkTotal = alloc<int>(nchunk + 1);
    chunkBefore = alloc<int>(nchunk + 1);
    ncells = alloc<int>(1);
    top = alloc<TreeTop>((size_t)(kTreeBits + 1)*nchunk);
    topNext = alloc<TreeTop>((size_t)(kTreeBits + 1)*((nchunk + kTreeTopUnits - 1)/kTreeTopUnits));
    for (int a = 0; a < 3; ++a) order.x[a] = alloc<double>(n);
    order.m = alloc<double>(n);
    order.tp = alloc<double2>(2*(size_t)n);
    box = alloc<TreeBox>(1);
    cstart = alloc<int>(n + 1);
    part = alloc<double>(std::max<int64_t>((n + kBlock - 1)/kBlock, 6*kTreeBoxBlocks));
    ensureCells(kTreeBits*small + 2);               // the root, and the record behind the last cell
    if (n > kTreeOwnSort) {
      size_t t1 = 0, t2 = 0;
      HIP_CHECK(rocprim::radix_sort_pairs(nullptr, t1, codes, codesSorted, idx, perm, (size_t)n, 0, 60, stream));
      HIP_CHECK(rocprim::exclusive_scan(nullptr, t2, chunkTotal, chunkBefore, 0, (size_t)nchunk + 1, rocprim::plus<int>(),
                                        stream));
      tmpBytes = std::max(t1, t2);
      tmp = alloc<char>(tmpBytes);
      HIP_CHECK(hipMemsetAsync(chunkTotal, 0, (size_t)(nchunk + 1)*sizeof(int), stream));
    }
  }

  void release() {
    for (void* p : allocs) (void)hipFree(p);
    allocs.clear();
  }

  // Room for `need` cells.  The arrays that became too small are given back (the tree's launches on
  // them have been waited for), and cellsAllocs tells a captured step that its pointers are old.
  void ensureCells(int64_t need) {
    if (need <= cellCap) return;
    const int64_t cap = cellCap ? need + need/4 + 1024 : need;
    HIP_CHECK(hipStreamSynchronize(stream));
    for (void* p : {(void*)cells, (void*)first, (void*)last}) {
      if (!p) continue;
      allocs.erase(std::find(allocs.begin(), allocs.end(), p));
      HIP_CHECK(hipFree(p));
    }
    bytes -= cellCap*(int64_t)(sizeof(TreeCell) + 2*sizeof(int));
    cellCap = 0;
    cells = nullptr;
    first = last = nullptr;
    ++cellsAllocs;
    first = alloc<int>(cap);
    last = alloc<int>(cap);
    cells = alloc<TreeCell>(cap);
    cellCap = cap;
  }

  // The points in tree order and the number of cells per chunk.  Up to kTreeOwnSort points a build
  // is nine or ten launches and no wait: extent, splitters, buckets, scatter, bucket sorts, counts,
  // and the cells' (formCells).  Bound by the launches' latencies: 33k points 87 us, 250k 230 beside
  // the grad-h pass (extent 5, splitters 11 / 16, sort 15 / 40, cells 21 / 35, cells above 21 / 31).
  // The library's merge sort, one moments launch per level and three waits on the host took 500
  // and 870 us.  512 buckets instead of 1024 take 5 us off the splitters, and a bucket still fits a
  // block's registers up to kTreeFewer points.
  void build(double* const* xs, const double* m, int nn) {
    const int nb = (int)((nn + kBlock - 1)/kBlock), nbox = std::min(nb, kTreeBoxBlocks);
    const int nchunk = (nn + kTreeChunk - 1)/kTreeChunk;
    const bool own = nn <= kTreeOwnSort;
    const TreePoints pts{{xs[0], xs[1], D == 3 ? xs[2] : zero}};
    hipLaunchKernelGGL(k_tree_bbox, dim3(nbox), dim3(kBlock), 0, stream, pts, nn, part);
    const bool fewer = nn <= kTreeFewer;
    hipLaunchKernelGGL(fewer ? k_tree_split<kTreeBuckets/2> : k_tree_split<kTreeBuckets>, dim3(1),
                       dim3(fewer ? kTreeBuckets/2 : kTreeBuckets), 0, stream, pts, nn, (const double*)part, nbox, own, box,
                       splitKey, splitId, count);
    if (own) {
      const int buckets = fewer ? kTreeBuckets/2 : kTreeBuckets, block = fewer ? kBlock : 2*kBlock;
      const int room = std::max(kTreeBucketRoom*((nn + buckets - 1)/buckets), 2*kBlock);
      hipLaunchKernelGGL(fewer ? k_tree_rank<kTreeBuckets/2> : k_tree_rank<kTreeBuckets>, dim3(nb), dim3(kBlock), 0, stream,
                         pts, nn, (const TreeBox*)box, (const uint64_t*)splitKey, (const uint32_t*)splitId, count, codes,
                         slot);
      hipLaunchKernelGGL(fewer ? k_tree_scatter<kTreeBuckets/2> : k_tree_scatter<kTreeBuckets>, dim3(nb), dim3(kBlock), 0,
                         stream, nn, (const int*)count, (const uint64_t*)codes, (const int2*)slot, keys, idx);
      hipLaunchKernelGGL(fewer ? k_tree_sort<kBlock> : k_tree_sort<2*kBlock>, dim3(buckets), dim3(block),
                         room*(sizeof(uint64_t) + sizeof(uint32_t)), stream, (const int*)count, room, keys, idx, pts, m,
                         codesSorted, perm, order);
    } else {
      hipLaunchKernelGGL(k_tree_codes, dim3(nb), dim3(kBlock), 0, stream, pts, nn, (const TreeBox*)box, codes, idx);
      HIP_CHECK(hipGetLastError());
      size_t t = tmpBytes;
      HIP_CHECK(rocprim::radix_sort_pairs(tmp, t, codes, codesSorted, idx, perm, (size_t)nn, 0, 60, stream));
      hipLaunchKernelGGL(k_tree_gather, dim3(nb), dim3(kBlock), 0, stream, pts, m, (const uint32_t*)perm, nn, order);
    }
    hipLaunchKernelGGL(k_tree_count, dim3(nchunk), dim3(kTreeChunk), 0, stream, (const uint64_t*)codesSorted, nn,
                       chunkTotal);
    HIP_CHECK(hipGetLastError());
    if (!own) {
      size_t t = tmpBytes;
      HIP_CHECK(rocprim::exclusive_scan(tmp, t, chunkTotal, chunkBefore, 0, (size_t)nchunk + 1, rocprim::plus<int>(),
                                        stream));
      int total = 0;
      HIP_CHECK(hipMemcpyAsync(&total, chunkBefore + nchunk, sizeof(int), hipMemcpyDeviceToHost, stream));
      HIP_CHECK(hipStreamSynchronize(stream));
      ensureCells((int64_t)total + 1);
    }
    npts = nn;
    cellsOpen2 = -1.0;
  }

  // The largest r^2 that the softening's self screen r^2/soft^2 > 1e-10 excludes: the quotient is
  // monotone in r^2, so the walk compares r^2 with it instead of dividing at every visited leaf.
  static double selfRadius2(double soft2) {
    auto counts = [soft2](double r2) { return r2/soft2 > 1.0e-10; };
    if (!(soft2 < INFINITY)) return INFINITY;       // nothing counts
    double r = 1.0e-10*soft2;
    while (r > 0.0 && counts(r)) r = std::nextafter(r, 0.0);
    while (!counts(std::nextafter(r, INFINITY))) r = std::nextafter(r, INFINITY);
    return r;
  }

  // The cells and their walk records for this opening angle and self screen (once per tree and pair).
  void formCells(double opening, double self2) {
    const double open2 = opening*opening;
    if (cellsOpen2 == open2 && cellsSelf2 == self2) return;
    const int nchunk = (npts + kTreeChunk - 1)/kTreeChunk;
    const TreeShape shape{box, open2, self2, D, npts, cells, first, last};
    hipLaunchKernelGGL(k_tree_cells, dim3(nchunk), dim3(kTreeChunk), 0, stream, shape, (const uint64_t*)codesSorted, order,
                       (const int*)chunkTotal, npts <= kTreeOwnSort ? (const int*)nullptr : (const int*)chunkBefore, cstart,
                       ncells, top);
    TreeTop *from = top, *to = topNext;
    int64_t span = kTreeChunk;
    for (int units = nchunk; units > 1; span *= kTreeTopUnits) {
      const int groups = (units + kTreeTopUnits - 1)/kTreeTopUnits;
      hipLaunchKernelGGL(k_tree_top, dim3(groups), dim3(1024), 0, stream, shape, (const uint64_t*)codesSorted, order, units,
                         span, units == nchunk, (const int*)cstart, (const int*)ncells, (const TreeTop*)from, to);
      std::swap(from, to);
      units = groups;
    }
    HIP_CHECK(hipGetLastError());
    cellsOpen2 = open2;
    cellsSelf2 = self2;
  }

  // The tree now held was built and its cells formed by launches that were recorded earlier.
  void rebuilt(int nn, double opening, double soft) {
    npts = nn;
    cellsOpen2 = opening*opening;
    cellsSelf2 = selfRadius2(soft*soft);
  }
  bool buildsWithoutWait(int nn) const { return nn <= kTreeOwnSort; }
  void prepareWalk(double opening, double soft) { formCells(opening, selfRadius2(soft*soft)); }

  void evaluate(double* const* acc, double* pot, int nn, double G, double soft, double opening, Scalars* sc,
                double ftimestep) {
    const int nb = (nn + kBlock - 1)/kBlock;
    double* az = D == 3 ? acc[2] : sink;
    const double self2 = selfRadius2(soft*soft);
    formCells(opening, self2);
    auto walk = nn <= kTreeAlone ? (D == 3 ? k_tree_walk<1, false, 3> : k_tree_walk<1, false, 2>)
                                 : (D == 3 ? k_tree_walk<kTreeGroup, false, 3> : k_tree_walk<kTreeGroup, false, 2>);
    hipLaunchKernelGGL(walk, dim3(nb), dim3(kBlock), 0, stream, (const double*)order.x[0],
                       (const double*)order.x[1], (const double*)order.x[2], (const double2*)order.tp, (const TreeCell*)cells,
                       (const int*)first, (const int*)last, (const int*)ncells, npts, (const uint32_t*)perm, soft*soft,
                       self2, soft, G,
                       acc[0], acc[1], az, pot, part, (unsigned long long*)nullptr);
    hipLaunchKernelGGL(k_tree_dt, dim3(1), dim3(kBlock), 0, stream, part, nb, sc, G, ftimestep);
    HIP_CHECK(hipGetLastError());
  }

  // Interactions of one walk over the current tree (the counting variant of the walk, into
  // throw-away outputs): out[0] monopole (accepted cell) interactions, out[1] point-point
  // interactions, summed over the points.  A measurement aid: allocates, waits on the stream.
  void countInteractions(double soft, double opening, int64_t* out) {
    const int nn = npts;
    if (!active || nn <= 0) raise(SPX_ERR_STATE, "no TreeGravity evaluation to count");
    const int nb = (int)((nn + kBlock - 1)/kBlock);
    double* scratch = nullptr;
    unsigned long long* counts = nullptr;
    HIP_CHECK(hipMalloc(&scratch, (size_t)(4*(size_t)std::max(nn, 1) + nb)*sizeof(double)));
    HIP_CHECK(hipMalloc(&counts, 2*(size_t)std::max(nn, 1)*sizeof(unsigned long long)));
    double* a = scratch;
    formCells(opening, INFINITY);          // one-point cells keep their opening radius: told apart from points
    auto walk = D == 3 ? k_tree_walk<kTreeGroup, true, 3> : k_tree_walk<kTreeGroup, true, 2>;
    hipLaunchKernelGGL(walk, dim3(nb), dim3(kBlock), 0, stream, (const double*)order.x[0],
                       (const double*)order.x[1], (const double*)order.x[2], (const double2*)order.tp, (const TreeCell*)cells,
                       (const int*)first, (const int*)last, (const int*)ncells, npts, (const uint32_t*)perm, soft*soft,
                       selfRadius2(soft*soft), soft, 1.0, a, a + nn,
                       a + 2*(size_t)nn, a + 3*(size_t)nn, a + 4*(size_t)nn, counts);
    const hipError_t e = hipGetLastError();
    std::vector<unsigned long long> h(2*(size_t)nn);
    hipError_t e2 = hipSuccess;
    if (e == hipSuccess) {
      e2 = hipMemcpyAsync(h.data(), counts, h.size()*sizeof(unsigned long long), hipMemcpyDeviceToHost, stream);
      if (e2 == hipSuccess) e2 = hipStreamSynchronize(stream);
    }
    (void)hipFree(scratch);
    (void)hipFree(counts);
    HIP_CHECK(e);
    HIP_CHECK(e2);
    out[0] = out[1] = 0;
    for (int p = 0; p < nn; ++p) { out[0] += (int64_t)h[2*(size_t)p]; out[1] += (int64_t)h[2*(size_t)p + 1]; }
  }
};

}  // namespace spx
