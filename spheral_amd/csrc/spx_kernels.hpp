// spx_kernels.hpp -- neighbour build and the light pair passes of the SPH hot path.
//
// Every pair pass is a gather: one to four lanes per target particle walk its ELLPACK
// neighbour list and accumulate only its own sums, so no atomics touch the
// conserved quantities.  Where a pair term must agree from both sides (the pairwise
// acceleration and the compatible-energy partition) FP64 forms it by operations that
// commute in the two nodes; mixed precision evaluates the pair in one canonical (a, b)
// order: an image partner makes the gathering node "a" (the reference's internal-ghost
// pair), otherwise the lower slot is "a".
//
// A batch holds independent runs of one problem type; particle i belongs to run
// f.run[i] with its own cell grid (RunGrid) and time step (Scalars).  Pairs never
// cross runs.  R is the arithmetic type of the pair math (double, or float in the
// mixed-precision mode where positions are differenced in double first).
#pragma once

#include "spx_device.hpp"

namespace spx {

// ---------------------------------------------------------------------------
// Neighbour image of a slot: position and velocity transforms (PeriodicBoundary
// copies, ReflectingBoundary::reflectOperator flips the normal component:
// Boundary/ReflectingBoundary.cc:183-197).
// ---------------------------------------------------------------------------
template <int D>
__device__ __forceinline__ void image_pos(const Geo& g, int code, double* xj) {
#pragma unroll
  for (int a = 0; a < D; ++a) {
    const int c = (code >> (2*a)) & 3;
    if (c) xj[a] = image_coord<D>(((g.permask >> a) & 1) ? BC_PERIODIC : BC_REFLECTING, c, xj[a], g.xmin[a], g.xmax[a]);
  }
}
template <int D>
__device__ __forceinline__ double refl_sign(const Geo& g, int code, int a) {
  const int c = (code >> (2*a)) & 3;
  if (!c) return 1.0;
  return ((g.reflmask >> (2*a + c - 1)) & 1) ? -1.0 : 1.0;
}

template <int D>
__device__ __forceinline__ int cell_coord(const RunGrid& gr, int a, double x) {
  int c = (int)floor((x - gr.origin[a])*gr.inv_cell[a]);
  return c < 0 ? 0 : (c >= gr.nc[a] ? gr.nc[a] - 1 : c);
}

// ---------------------------------------------------------------------------
// Boundary enforcement + sort keys.  Periodic violators are mapped through the
// opposite plane, reflecting violators mirrored with their velocity
// (Boundary/PlanarBoundary.cc:153-200, ReflectingBoundary.cc:465-473).  Keys order
// the particles of active runs by (run, cell Morton code), then the finished runs
// (kept whole, behind the active ones), then removed runs (largest key).  Active runs
// that keep their candidate list (build[run] == 0) get no Morton bits: the sort is
// stable, so they keep their order.
// ---------------------------------------------------------------------------
// Node i's coordinate xa along axis a with the boundaries enforced (periodic: moved back into the
// box; reflecting: mirrored, the velocity too).
template <int D>
__device__ __forceinline__ double enforce_axis(const Fields& f, const Geo& g, int a, int i, double xa) {
  for (int side = 1; side <= 2; ++side) {
    const int bc = side == 1 ? (((g.permask >> a) & 1) ? BC_PERIODIC : (((g.reflmask >> (2*a)) & 1) ? BC_REFLECTING : BC_NONE))
                             : (((g.permask >> a) & 1) ? BC_PERIODIC : (((g.reflmask >> (2*a + 1)) & 1) ? BC_REFLECTING : BC_NONE));
    if (bc == BC_NONE) continue;
    const double thpt = side == 1 ? (xa - g.xmin[a]) : -(xa - g.xmax[a]);
    const bool fuzzy0 = fabs(thpt) <= 1.0e-15*fmax(1.0, fabs(thpt));
    if (!fuzzy0 && thpt < 0.0) {
      if (bc == BC_PERIODIC) {
        xa = image_coord<D>(bc, side == 1 ? 2 : 1, xa, g.xmin[a], g.xmax[a]);
      } else {
        xa = image_coord<D>(bc, side, xa, g.xmin[a], g.xmax[a]);
        f.v[a][i] = -f.v[a][i];
      }
    }
  }
  return xa;
}

template <int D>
__global__ void __launch_bounds__(kBlock) k_keys(Fields f, Geo g, const RunGrid* grids, const int* rstate,
                                                 const int* rorder, const int* build, int n, int enforce, int withKeys,
                                                 int mortonBits, int runBits, uint64_t* keys, uint32_t* vals, int* flags,
                                                 const int* sub, uint64_t* skeys, uint32_t* spos) {
  const int i = blockIdx.x*blockDim.x + threadIdx.x;
  if (enforce && i == 0) flags[kFlagWrap] = 0;
  if (i >= n) return;
  const int r = f.run[i];
  uint64_t key = 0;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    double xa = f.x[a][i];
    if (enforce) {
      xa = enforce_axis<D>(f, g, a, i, xa);
      f.x[a][i] = xa;
    }
    if (withKeys && build[r]) key |= spread_bits((uint64_t)cell_coord<D>(grids[r], a, xa), D) << a;
  }
  if (withKeys && sub) {
    // only the rebuilding runs' nodes, compacted: run r's go to [sub[3r+1], +n) in position order,
    // keyed [its segment index | Morton] (sub: per run segment start, compacted start, segment index)
    if (build[r]) {
      const int k = sub[3*r + 1] + (i - sub[3*r]);
      skeys[k] = ((uint64_t)sub[3*r + 2] << mortonBits) | key;
      spos[k] = (uint32_t)i;
    }
  } else if (withKeys) {
    // layout: [rank | run | Morton], rank 0 active (runs by their place rorder), 1 done (by
    // slot); removed runs take the maximum key
    const int st = rstate[r];
    const int shift = mortonBits + runBits;
    keys[i] = st == RUN_ACTIVE ? (((uint64_t)rorder[r] << mortonBits) | key)
            : (st == RUN_DONE ? ((1ull << shift) | ((uint64_t)r << mortonBits)) : ~0ull);
    vals[i] = (uint32_t)i;
  }
}

// Gather a set of arrays through a permutation (dst[p] = src[perm[p]]).
struct GatherSet {
  const double* src[64];
  double* dst[64];
  int count;
};
__global__ void __launch_bounds__(kBlock) k_gather(GatherSet s, const uint32_t* perm, int n) {
  const int p = blockIdx.x*blockDim.x + threadIdx.x;
  if (p >= n) return;
  const uint32_t q = perm[p];
  for (int k = 0; k < s.count; ++k) s.dst[k][p] = s.src[k][q];
}
// State transfer between the engine's arrays (one per component, particle order) and the boundary's
// Field records (NC doubles per node, the run's node order), through a staging buffer that holds the
// records of nodes [c0, c1): one strided pass on the device and one copy per field instead of a copy
// and a host loop per component.  Slot p holds node (oid[p] & low 40 bits); oid null: node p - slot0.
struct RecordSet {
  double* a[9];
  int nc;          // components per record
};
__device__ __forceinline__ int64_t node_of(const int64_t* oid, int64_t slot0, int64_t k) {
  return oid ? oid[slot0 + k] & (((int64_t)1 << 40) - 1) : k;
}
__global__ void __launch_bounds__(kBlock) k_to_records(RecordSet s, double* __restrict__ stage,
                                                       const int64_t* __restrict__ oid, int64_t slot0, int64_t n,
                                                       int64_t c0, int64_t c1) {
  const int64_t k = (int64_t)blockIdx.x*blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int64_t node = node_of(oid, slot0, k);
  if (node < c0 || node >= c1) return;
  double* out = stage + (node - c0)*s.nc;
  for (int c = 0; c < s.nc; ++c) out[c] = s.a[c][slot0 + k];
}
__global__ void __launch_bounds__(kBlock) k_from_records(RecordSet s, const double* __restrict__ stage,
                                                         const int64_t* __restrict__ oid, int64_t slot0, int64_t n,
                                                         int64_t c0, int64_t c1) {
  const int64_t k = (int64_t)blockIdx.x*blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int64_t node = node_of(oid, slot0, k);
  if (node < c0 || node >= c1) return;
  const double* in = stage + (node - c0)*s.nc;
  for (int c = 0; c < s.nc; ++c) s.a[c][slot0 + k] = in[c];
}
// Ids and run slots of a newly admitted run's nodes, at the slots from slot0.
__global__ void __launch_bounds__(kBlock) k_new_ids(int64_t* oid, int32_t* run, int64_t slot0, int64_t n, int slot) {
  const int64_t k = (int64_t)blockIdx.x*blockDim.x + threadIdx.x;
  if (k >= n) return;
  oid[slot0 + k] = ((int64_t)slot << 40) | k;
  run[slot0 + k] = slot;
}
// a[c][slot0 .. slot0 + n) = value for each of the set's arrays.
struct FillSet {
  double* a[40];
  int count;
};
__global__ void __launch_bounds__(kBlock) k_fill(FillSet s, int64_t slot0, int64_t n, double value) {
  const int64_t k = (int64_t)blockIdx.x*blockDim.x + threadIdx.x;
  if (k >= n) return;
  for (int c = 0; c < s.count; ++c) s.a[c][slot0 + k] = value;
}
__global__ void __launch_bounds__(kBlock) k_gather_ids(const int64_t* src, int64_t* dst, const int32_t* rsrc, int32_t* rdst,
                                                       const uint32_t* perm, int n) {
  const int p = blockIdx.x*blockDim.x + threadIdx.x;
  if (p < n) { dst[p] = src[perm[p]]; rdst[p] = rsrc[perm[p]]; }
}

template <int D>
__device__ __forceinline__ int lin_cell(const RunGrid& g, const int* c) {
  int l = c[D - 1];
  for (int a = D - 2; a >= 0; --a) l = l*g.nc[a] + c[a];
  return g.cellBase + l;
}
template <int D>
__device__ __forceinline__ void unspread(uint64_t key, int mortonBits, int* c) {
  for (int a = 0; a < D; ++a) {
    uint64_t v = 0;
    for (int b = 0; b < 21 && D*b + a < mortonBits; ++b) v |= ((key >> (D*b + a)) & 1ull) << b;
    c[a] = (int)v;
  }
}

// Cell ranges of the sorted keys of the runs that build candidate lists: start[cell],
// end[cell] (both 0 when empty).  The low mortonBits of a key are the cell's Morton code;
// a run's particles are one contiguous segment (run[] tells where it ends).
// With cell levels, each level's table: a level-l cell is the key prefix above the low
// D*(levels-1-l) bits, one contiguous range of the sorted particles.
template <int D>
__device__ __forceinline__ int level_cells(const RunGrid& g, int l, int* ncl) {
  const int sh = g.levels - 1 - l;
  int t = 1;
  for (int a = 0; a < D; ++a) { ncl[a] = ((g.nc[a] - 1) >> sh) + 1; t *= ncl[a]; }
  return t;
}
template <int D>
__device__ __forceinline__ int lin_level_cell(const RunGrid& g, int l, const int* ncl, const int* c) {
  int q = c[D - 1];
  for (int a = D - 2; a >= 0; --a) q = q*ncl[a] + c[a];
  return g.levelBase[l] + q;
}
template <int D>
__global__ void __launch_bounds__(kBlock) k_cell_bounds(const uint64_t* keys, const int32_t* run, int n,
                                                        const RunGrid* grids, const int* build, int mortonBits,
                                                        int* start, int* end) {
  const int p = blockIdx.x*blockDim.x + threadIdx.x;
  if (p >= n) return;
  const int r = run[p];
  if (!build[r]) return;
  const uint64_t mask = (1ull << mortonBits) - 1ull;
  const uint64_t k = keys[p] & mask;
  const RunGrid& gr = grids[r];
  const bool first = p == 0 || run[p - 1] != r, last = p == n - 1 || run[p + 1] != r;
  int c[3];
  if (gr.levels <= 1) {
    if (first || (keys[p - 1] & mask) != k) { unspread<D>(k, mortonBits, c); start[lin_cell<D>(gr, c)] = p; }
    if (last || (keys[p + 1] & mask) != k) { unspread<D>(k, mortonBits, c); end[lin_cell<D>(gr, c)] = p + 1; }
    return;
  }
  const uint64_t kp = first ? 0 : (keys[p - 1] & mask), kn = last ? 0 : (keys[p + 1] & mask);
  for (int l = 0; l < gr.levels; ++l) {
    const int sh = D*(gr.levels - 1 - l);
    const uint64_t q = k >> sh;
    int ncl[3] = {1, 1, 1};
    level_cells<D>(gr, l, ncl);
    if (first || (kp >> sh) != q) { unspread<D>(q, mortonBits, c); start[lin_level_cell<D>(gr, l, ncl, c)] = p; }
    if (last || (kn >> sh) != q) { unspread<D>(q, mortonBits, c); end[lin_level_cell<D>(gr, l, ncl, c)] = p + 1; }
  }
}

// Gather over a list of positions: dst[a][pos[k]] = src[a][from ? from[k] : pos[k]], oid alike;
// with sortedKeys, keysOut[pos[k]] = sortedKeys[k].
__global__ void __launch_bounds__(kBlock) k_gather_list(GatherSet s, const uint32_t* pos, const uint32_t* from,
                                                        const int64_t* oidSrc, int64_t* oidDst,
                                                        const uint64_t* sortedKeys, uint64_t* keysOut, int nsub) {
  const int k = blockIdx.x*blockDim.x + threadIdx.x;
  if (k >= nsub) return;
  const uint32_t p = pos[k], q = from ? from[k] : p;
  for (int a = 0; a < s.count; ++a) s.dst[a][p] = s.src[a][q];
  oidDst[p] = oidSrc[q];
  if (sortedKeys) keysOut[p] = sortedKeys[k];
}

// Running per-run minimum of a positive double: one atomic per wavefront when its lanes share a run.
__device__ __forceinline__ void run_min(Scalars* sc, int r, double v, bool valid) {
  const int r0 = __shfl(r, 0);
  const bool uniform = __all(!valid || r == r0);
  if (uniform) {
    double m = valid ? v : 1.7976931348623157e308;
    for (int off = 32; off > 0; off >>= 1) m = fmin(m, __shfl_xor(m, off));
    // most waves do not lower the running minimum: read first, then update atomically
    const unsigned long long b = ord_bits(m);
    if ((threadIdx.x & 63) == 0 && __any(valid) && b < sc[r0].dtBits) atomicMin(&sc[r0].dtBits, b);
  } else if (valid) {
    const unsigned long long b = ord_bits(v);
    if (b < sc[r].dtBits) atomicMin(&sc[r].dtBits, b);
  }
}

// Packed neighbour records (Fields::xh, Fields::vmr) of the current state, and nodeScale =
// 1/(lambda_max(H) nPerh) of each node (GenericHydro::dt, Physics/GenericHydro.cc:142-150).
template <int D>
__device__ __forceinline__ void pack_node(const Fields& f, const Phys& ph, int i) {
  const double h = f.hinv[i];
  double2* P = reinterpret_cast<double2*>(f.xh) + 2*(size_t)i;
  P[0] = make_double2(f.x[0][i], D >= 2 ? f.x[1 % D][i] : 0.0);
  P[1] = make_double2(D >= 3 ? f.x[2 % D][i] : 0.0, h);
  double2* V = reinterpret_cast<double2*>(f.vmr) + 2*(size_t)i;
  V[0] = make_double2(f.v[0][i], D >= 2 ? f.v[1 % D][i] : 0.0);
  V[1] = make_double2(D >= 3 ? f.v[2 % D][i] : 0.0, f.m[i]);
  f.ns[i] = 1.0/max_eigen_iso<D>(h)/ph.nperh;
}
template <int D>
__global__ void __launch_bounds__(kBlock) k_pack(Fields f, Phys ph, int n) {
  const int i = blockIdx.x*blockDim.x + threadIdx.x;
  if (i < n) pack_node<D>(f, ph, i);
}
constexpr unsigned long long kNoVote = 0xfff0000000000000ull;   // ord_bits(+inf)
// The start of a steady step in one launch: boundaries enforced where the last step left that
// pending, records packed, the dt votes and the filter's overflow flag cleared.
template <int D>
__global__ void __launch_bounds__(kBlock) k_prepare(Fields f, Geo g, Phys ph, int nTotal, int n, Scalars* sc, int nruns,
                                                    int* flags) {
  const int i = blockIdx.x*blockDim.x + threadIdx.x;
  if (i < nruns) sc[i].dtBits = kNoVote;
  if (i == 0) flags[kFlagOverflow] = 0;
  if (i >= nTotal) return;
  if (flags[kFlagWrap])
#pragma unroll
    for (int a = 0; a < D; ++a) f.x[a][i] = enforce_axis<D>(f, g, a, i, f.x[a][i]);
  if (i < n) pack_node<D>(f, ph, i);
}

// Position and h^-1 of node j from a 4-double (x, h^-1) record array.
template <int D>
__device__ __forceinline__ void load_xh(const double* xh, int j, double* x, double& h) {
  const double2* P = reinterpret_cast<const double2*>(xh) + 2*(size_t)j;
  const double2 a = P[0], b = P[1];
  x[0] = a.x;
  if (D >= 2) x[1 % D] = a.y;
  if (D >= 3) x[2 % D] = b.x;
  h = b.y;
}
// Velocity and mass of node j from a 4-double (v, m) record array.
template <int D>
__device__ __forceinline__ void load_vm(const double* vm, int j, double* v, double& m) {
  const double2* P = reinterpret_cast<const double2*>(vm) + 2*(size_t)j;
  const double2 a = P[0], b = P[1];
  v[0] = a.x;
  if (D >= 2) v[1 % D] = a.y;
  if (D >= 3) v[2 % D] = b.x;
  m = b.y;
}

// ---------------------------------------------------------------------------
// ConnectivityMap::computeConnectivity (Neighbor/ConnectivityMap.cc:905-947): j is a
// neighbour of i iff |Hi rij|^2 <= ext^2 or |Hj rij|^2 <= ext^2, i != j (an image of i
// itself counts, as the reference's ghost of i does), evaluated with the reference's
// rounding (no contraction) so the sets match exactly.
//
// Two stages.  k_candidates builds, for the runs whose list is stale, a candidate list
// with the criterion widened to ext (1 + skin): a few lanes per particle walk the cells its
// widened support reaches.  It records the positions and h^-1 the list was built from.  The
// filtering pass (k_density_dt) applies the exact criterion to the candidates every step.  The candidates stay complete while no pair can have closed in from beyond the
// widened radius: with D = max |x - xb| hb/ext and G = max hb/h^-1 over the run's nodes,
// |rij(now)| <= max(Si, Sj)(now) implies |rij(built)| <= max(Si, Sj)(built) (G + 2D), so a
// list is valid while G + 2D <= 1 + skin (the full update measures both after every step).
// Reflecting images are isometries of the node, and periodic images are re-chosen as the
// nearest copy each step (the box spans >= 3 widened supports), so both obey the bound.
// ---------------------------------------------------------------------------
// Image code of the same pair seen from the other node: a periodic image flips side, a
// reflecting image is its own inverse.
__device__ __forceinline__ int inverse_image(const Geo& g, int code) {
  int out = code;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int c = (code >> (2*a)) & 3;
    if (c && ((g.permask >> a) & 1)) out = (out & ~(3 << (2*a))) | ((3 - c) << (2*a));
  }
  return out;
}

// Candidate lists of the runs that rebuild: each node gathers the j within its own widened
// support (|Hi rij|^2 <= ext^2 (1 + skin)^2); see k_candidates for the cells it scans.
//
// The rebuilding runs' segments, listed as (first position, first index in the compacted
// range [0, nBuild)) in increasing order of both: compacted index k -> particle position, and
// (with seg_of) the segment that holds it.
__device__ __forceinline__ int seg_of(const int2* seg, int nseg, int k) {
  int lo = 0, hi = nseg - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (seg[mid].y <= k) lo = mid; else hi = mid - 1;
  }
  return lo;
}
__device__ __forceinline__ int build_pos(const int2* seg, int nseg, int k) {
  const int s = seg_of(seg, nseg, k);
  return seg[s].x + (k - seg[s].y);
}

// Launched over the rebuilding runs' particles only (seg, nBuild): a step that rebuilds a few
// small runs of a large batch neither walks the others nor leaves the work to the one XCD whose
// index range holds those runs.
//
// Cells.  A run whose h is near uniform has one grid of cells at least as wide as the widest
// widened support, and each node scans the 3^D cells around its own (image cells through
// periodic and reflecting planes).  Where h varies by 2x or more:
//  * open boundaries: levels.  Level-l cells are at least support/2^(l+2) wide (l = 0..levels-1;
//    the grid is that of the finest level, level-l cells are 2^(levels-1-l) finest cells per
//    axis, so each is one contiguous range of the Morton-sorted particles, with a table per
//    level).  A node works at the finest level l with support/2^l >= its widened support, whose
//    cells are at least a quarter of that support, and scans the 3 to 9 cells per axis the
//    support reaches: dense regions scan cells of their own size, sparse ones cells of theirs.
//  * periodic or reflecting axes: one grid, cells shrunk toward the smaller supports (by up to
//    4x while the grid stays within ~8 cells per node), and each node scans the cells its own
//    support reaches.
// Every node collects each j within its own widened support; where j's support does not reach
// i, i hands j the mirrored entry (tlist, merged by k_candidates_merge).  Together each list
// holds exactly the j with |Hi rij| or |Hj rij| within the widened extent.
//
// kSearchLanes lanes per node.  The stencil's cells are taken kSearchCells at a time, two consecutive
// ones per lane; a scan of their particle counts lays their particles out as one list (in cell order,
// then slot order, as one lane alone would meet them), which the lanes test kSearchLanes at a time,
// each finding its particle's cell by bisection of the scan in LDS.  Accepted entries keep the list's
// order by a ballot, so the candidate lists are the same for any lane count.  One lane per node left
// small runs with a few blocks walking up to a thousand candidates in turn, and where h varies most
// cells of a node's level hold no or few particles.  Per rebuild, one lane -> 16: KH 2-D 4096 245 ->
// 32 us, 65536 253 -> 91, Sod 3-D 25k 1879 -> 256, Evrard 250k 3030 -> 1599; Taylor-Green 128^3 3003 ->
// 3041 (instruction issue: 8 waves per SIMD and the test's ~80 instructions per candidate; at 79
// VGPRs and 6 waves 3167).  8 lanes: Sod 451, Evrard 2494, Taylor-Green 4245.
constexpr int kSearchLanes = 16, kSearchCells = 32;
// The largest capacity that a pass with too short lists asks for.  Read first: where most nodes
// overflow, as in a run's first build, an atomic per wavefront of 4 or 16 nodes queued at one word
// (KH 2-D 262144, first build: search 770 -> 215 us, filter 206 -> 48).
__device__ __forceinline__ void ask_capacity(int* need, int v) {
  if (v > __hip_atomic_load(need, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(need, v);
}
template <int D>
__global__ void __launch_bounds__(kBlock, 8) k_candidates(Fields f, Geo g, const RunGrid* grids, const int2* seg, int nseg,
                                                       int nBuild, const int* cstart, const int* cend, uint32_t* tlist,
                                                       int* tcnt, int tcap, int* overflow) {
  constexpr int C = kSearchLanes, Q = kSearchCells/C;
  __shared__ int sEnd[kBlock/C][kSearchCells];         // particles up to and including the cell
  __shared__ uint32_t sFirst[kBlock/C][kSearchCells];  // the cell's first slot minus those before it, image code on top
  const int gl = xcd_block()*blockDim.x + threadIdx.x;
  const int k = gl/C, sub = gl & (C - 1), grp = threadIdx.x/C;
  if (k >= nBuild) return;                             // a node's lanes leave together
  const int sg = seg_of(seg, nseg, k);
  const int i = seg[sg].x + (k - seg[sg].y);
  const RunGrid& gr = grids[f.run[i]];
  double xi[D];
  int ci[3] = {0, 0, 0};
#pragma unroll
  for (int a = 0; a < D; ++a) {
    xi[a] = f.x[a][i];
    ci[a] = cell_coord<D>(gr, a, xi[a]);
    if (sub == 0) f.xb[a][i] = xi[a];
  }
  const double hi = f.hinv[i];
  if (sub == 0) f.hb[i] = hi;
  const double ext2c = gr.ext2c;
  const double reach = gr.extc*fast_rcp(hi);
  // FP32 distance pre-filter with a 1e-4 relative margin (far above its own rounding): only the
  // FP64 criterion decides membership
  const float reach2 = (float)(reach*reach*(1.0 + 1.0e-4));
  const size_t ld = (size_t)f.ld;
  const int cap = f.ccap;
  // the stencil: the cells of the node's level that its own widened support reaches (with one grid,
  // at least the 3^D cells around its own)
  const bool levels = gr.levels > 1;
  int lv = 0, cl[3] = {0, 0, 0}, ncl[3] = {1, 1, 1}, kw[3] = {0, 0, 0};
  if (levels) {
    // the finest l with support/2^l >= its reach; those cells are at least support/2^(l+2) wide, a
    // quarter of the reach or more, so it scans 3 to 9 cells per axis
    double w = 0.5*gr.support;
    while (lv + 1 < gr.levels && w >= reach) { ++lv; w *= 0.5; }
    const int sh = gr.levels - 1 - lv;
    level_cells<D>(gr, lv, ncl);
#pragma unroll
    for (int a = 0; a < D; ++a) {
      cl[a] = ci[a] >> sh;
      kw[a] = max(1, (int)ceil(reach*gr.inv_cell[a]/(double)(1 << sh)*(1.0 + 1.0e-12)));
    }
  } else {
#pragma unroll
    for (int a = 0; a < D; ++a) {
      cl[a] = ci[a];
      ncl[a] = gr.nc[a];
      kw[a] = max(1, (int)ceil(reach*gr.inv_cell[a]*(1.0 + 1.0e-12)));
    }
  }
  const int wx = 2*kw[0] + 1, wy = D >= 2 ? 2*kw[1] + 1 : 1, wz = D >= 3 ? 2*kw[2] + 1 : 1;
  const int ncells = wx*wy*wz;
  bool inside = true;                                  // no cell of the stencil leaves the grid
#pragma unroll
  for (int a = 0; a < D; ++a) inside &= cl[a] >= kw[a] && cl[a] + kw[a] < ncl[a];
  // the particle range and image code of the cell at offset (dx, dy, dz); false: nothing there
  auto cell_range = [&](const int* off, int& first, int& last, int& code) -> bool {
    int cc[3] = {0, 0, 0};
    code = 0;
#pragma unroll
    for (int a = 0; a < D; ++a) cc[a] = cl[a] + off[a];
    if (!inside) {
      bool skip = false;
#pragma unroll
      for (int a = 0; a < D; ++a) {
        const bool per = !levels && ((g.permask >> a) & 1);
        const int refl = levels ? 0 : (g.reflmask >> (2*a)) & 3;
        int c = cc[a];
        if (c < 0) {
          if (per) { c += ncl[a]; code |= 1 << (2*a); }
          else if (refl & 1) { c = -c - 1; code |= 1 << (2*a); skip |= c >= ncl[a]; }
          else skip = true;
        } else if (c >= ncl[a]) {
          if (per) { c -= ncl[a]; code |= 2 << (2*a); }
          else if (refl & 2) { c = 2*ncl[a] - 1 - c; code |= 2 << (2*a); skip |= c < 0; }
          else skip = true;
        }
        cc[a] = c;
      }
      if (skip) return false;
    }
    const int cell = levels ? lin_level_cell<D>(gr, lv, ncl, cc) : lin_cell<D>(gr, cc);
    first = cstart[cell];
    last = cend[cell];
    return last > first;
  };
  int count = 0;
  for (int b0 = 0; b0 < ncells; b0 += kSearchCells) {
    // this lane's Q consecutive cells
    int len[Q], first[Q], codes[Q], sum = 0;
    int c = b0 + Q*sub;
    int off[3] = {c % wx, 0, 0};
    { const int t = c/wx; off[1] = t % wy; off[2] = t/wy; }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      len[q] = 0;
      first[q] = codes[q] = 0;
      if (c + q < ncells) {
        const int o[3] = {off[0] - kw[0], off[1] - kw[1], off[2] - kw[2]};
        int last = 0;
        if (cell_range(o, first[q], last, codes[q])) len[q] = last - first[q];
      }
      sum += len[q];
      if (++off[0] == wx) { off[0] = 0; if (++off[1] == wy) { off[1] = 0; ++off[2]; } }
    }
    int before = sum;
#pragma unroll
    for (int d = 1; d < C; d <<= 1) {
      const int o = __shfl_up(before, d, C);
      if (sub >= d) before += o;
    }
    const int total = __shfl(before, C - 1, C);
    before -= sum;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      sFirst[grp][Q*sub + q] = ((uint32_t)(first[q] - before) & kIdxMask) | ((uint32_t)codes[q] << kImgShift);
      before += len[q];
      sEnd[grp][Q*sub + q] = before;
    }
    // only this node's lanes, of one wavefront, read what they wrote
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int t0 = 0; t0 < total; t0 += C) {
      const int t = t0 + sub;
      bool acc = t < total;
      int j = i, code = 0;
      if (acc) {
        int m = 0;                                     // the first cell whose count exceeds t
#pragma unroll
        for (int s = kSearchCells/2; s > 0; s >>= 1) m += sEnd[grp][m + s - 1] <= t ? s : 0;
        const uint32_t e = sFirst[grp][m];
        j = (int)((e + (uint32_t)t) & kIdxMask);
        code = (int)(e >> kImgShift);
        acc = !(j == i && code == 0);
      }
      double rr[D];
      if (acc) {
        double xj[D];
#pragma unroll
        for (int a = 0; a < D; ++a) xj[a] = f.x[a][j];
        if (code) image_pos<D>(g, code, xj);
        float r2 = 0.0f;
#pragma unroll
        for (int a = 0; a < D; ++a) {
          rr[a] = dsub(xi[a], xj[a]);
          const float d = (float)rr[a];
          r2 += d*d;
        }
        acc = r2 <= reach2;
      }
      if (acc) {
        acc = eta2<D>(hi, rr) <= ext2c;
        if (acc) {
          const double hj = f.hinv[j];
          if (!(eta2<D>(hj, rr) <= ext2c)) {
            // j's own support does not reach i: j receives the pair from here
            const int slot = atomicAdd(&tcnt[j], 1);
            if (slot < tcap) tlist[ell_at(slot, j, ld)] = (uint32_t)i | ((uint32_t)inverse_image(g, code) << kImgShift);
          }
        }
      }
      const unsigned q = (unsigned)(__ballot(acc) >> (threadIdx.x & 63 & ~(C - 1))) & ((1u << C) - 1u);
      const int place = count + __popc(q & ((1u << sub) - 1u));
      if (acc && place < cap) f.cand[ell_at(place, i, ld)] = (uint32_t)j | ((uint32_t)code << kImgShift);
      count += __popc(q);
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (sub == 0) {
    f.ccnt[i] = count;
    if (count > cap) ask_capacity(overflow, count);
  }
}

// Number of the row's 16 lanes whose v is below e (row rotations by DPP).
template <int S = 15>
__device__ __forceinline__ int row_below(uint32_t v, uint32_t e) {
  if constexpr (S == 0) {
    return v < e ? 1 : 0;
  } else {
    const uint32_t o = (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x120 + S, 0xf, 0xf, false);   // row_ror:S
    return (o < e ? 1 : 0) + row_below<S - 1>(v, e);
  }
}

// Appends each rebuilding node's handed-over entries (tlist) to its candidate list, in
// ascending entry order (the order they arrived in is not deterministic).  Over the rebuilding
// runs' particles (seg, nBuild), 16 lanes (a DPP row) per node: each lane ranks an entry against all
// the node's entries, 16 at a time, and entry k goes to c0 + (number of smaller entries), entries
// being distinct.  Batches whose h is uniform hand nothing over and only read their counts.
// overflow[0]: the candidate capacity needed, overflow[1]: the handed-over capacity needed.
// A wavefront per 64 nodes, one node after the other, was bound by the latency of each node's reads:
// KH 2-D 58.7 us per rebuild, Sod 3-D 25k 135 us, Evrard 250k 865 us.
constexpr int kMergeLanes = 16;
__global__ void __launch_bounds__(kBlock) k_candidates_merge(Fields f, const int2* seg, int nseg, int nBuild,
                                                             const uint32_t* tlist, const int* tcnt, int tcap,
                                                             int* overflow) {
  const int gl = xcd_block()*blockDim.x + threadIdx.x;
  const int k = gl/kMergeLanes, sub = gl & (kMergeLanes - 1);
  if (k >= nBuild) return;                     // a node's lanes leave together
  const int i = build_pos(seg, nseg, k);
  const int t = tcnt[i];
  if (t == 0) return;
  if (t > tcap) {
    if (sub == 0) ask_capacity(&overflow[1], t);
    return;
  }
  const int c0 = f.ccnt[i];
  if (c0 + t > f.ccap) {
    if (sub == 0) ask_capacity(&overflow[0], c0 + t);
    return;
  }
  const size_t ld = (size_t)f.ld;
  for (int kb = 0; kb < t; kb += kMergeLanes) {
    const uint32_t e = kb + sub < t ? tlist[ell_at(kb + sub, i, ld)] : ~0u;
    int rank = 0;
    for (int cb = 0; cb < t; cb += kMergeLanes) {
      const uint32_t v = cb == kb ? e : (cb + sub < t ? tlist[ell_at(cb + sub, i, ld)] : ~0u);
      rank += row_below(v, e);
    }
    if (kb + sub < t) f.cand[ell_at(c0 + rank, i, ld)] = e;
  }
  if (sub == 0) f.ccnt[i] = c0 + t;
}

// Per-run maximum of an order-preserving double key: a wavefront whose lanes share a run
// reduces first, and an atomic is issued only when it would raise the running maximum
// (most wavefronts do not: reading first keeps them off the contended word).
__device__ __forceinline__ void run_max_bits(unsigned long long* word, size_t stride, int r, unsigned long long b,
                                             bool valid) {
  const int r0 = __shfl(r, 0);
  if (__all(!valid || r == r0)) {
    unsigned long long m = valid ? b : 0ull;
    for (int off = 32; off > 0; off >>= 1) {
      const unsigned long long o = __shfl_xor(m, off);
      m = o > m ? o : m;
    }
    unsigned long long* w = word + (size_t)r0*stride;
    if ((threadIdx.x & 63) == 0 && __any(valid) && m > __atomic_load_n(w, __ATOMIC_RELAXED)) atomicMax(w, m);
  } else if (valid) {
    unsigned long long* w = word + (size_t)r*stride;
    if (b > __atomic_load_n(w, __ATOMIC_RELAXED)) atomicMax(w, b);
  }
}

// Moves the candidate lists of runs whose particle segment shifted in a reorder (a run
// that keeps its list keeps its order, so old slot = new slot - delta):
// dst row p = src row p - delta with every index shifted by delta.  delta[run] ==
// kNoRemap marks runs whose rows are not moved.
constexpr int kNoRemap = INT32_MIN;
__global__ void __launch_bounds__(kBlock) k_remap_candidates(const uint32_t* src, const int32_t* srcCnt, uint32_t* dst,
                                                             int32_t* dstCnt, const int32_t* run, const int* delta,
                                                             size_t ld, int n) {
  const int p = blockIdx.x*blockDim.x + threadIdx.x;
  if (p >= n) return;
  const int d = delta[run[p]];
  if (d == kNoRemap) return;
  const int q = p - d;
  const int cnt = srcCnt[q];
  dstCnt[p] = cnt;
  for (int c = 0; c < cnt; c += 8) {
    const uint4* s = reinterpret_cast<const uint4*>(src + ell_at(c, q, ld));
    uint4* t = reinterpret_cast<uint4*>(dst + ell_at(c, p, ld));
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint4 v = s[h];
      v.x += (uint32_t)d; v.y += (uint32_t)d; v.z += (uint32_t)d; v.w += (uint32_t)d;
      t[h] = v;
    }
  }
}

// ---------------------------------------------------------------------------
// computeSPHSumMassDensity (SPH/computeSPHSumMassDensity.cc:35-85) in gather form
// -- node i receives m_j W(|Hj ri - Hj rj|, det Hj) -- fused with the GenericHydro::dt
// vote (Physics/GenericHydro.cc:112-381): per-node limits on the new density and the
// pairwise velocity-difference limit, min-reduced per run.
// FILT: the pass walks the candidate lists instead, applies the neighbour criterion to each
// candidate and writes the ELL neighbour list as it goes, so the connectivity filter and the first
// pair pass of the step read the neighbours once.  Without DENS and DT it only filters.
//
// Bound by the latency and the rate of the records' gathers (the L1 takes a 64-lane gather of 16
// bytes at about 1.4 lanes per clock).  kNodeLanes lanes per node: KH 2-D 4096 mixed 70.7 -> 26.5 us,
// 65536 FP64 80 -> 46 us, Sod 3-D 25k mixed 232 -> 92 us, Evrard 250k mixed 478 -> 417 us,
// Taylor-Green 96^3 mixed 494 -> 449 us, 128^3 FP64 1137 -> 1077 us (one lane per node before).
// ---------------------------------------------------------------------------
//
// The neighbour criterion: |Hi rij|^2 <= ext^2 or |Hj rij|^2 <= ext^2 in the reference's rounding.
// (h r)^2 with each product and sum rounded is non-decreasing in h, so the test with the smaller
// h^-1 decides both.  half[a]: half the box on a periodic axis (the nearest copy of j is taken),
// otherwise larger than any separation; only a pair that needs an image pays for one.  Returns
// whether j is a neighbour; code and rr = xi - xj are those of the image taken.
template <int D>
__device__ __forceinline__ bool neighbor_test(const Geo& g, double ext2, const double* half, const double* xi, double hi,
                                              const double* xj, double hj, bool self, int& code, double* rr) {
  code &= ~(((g.permask & 1) ? 3 : 0) | ((g.permask & 2) ? 12 : 0) | ((g.permask & 4) ? 48 : 0));
  bool far = code != 0;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    rr[a] = dsub(xi[a], xj[a]);
    far |= fabs(rr[a]) > half[a];
  }
  if (far) {
    double xk[D];
#pragma unroll
    for (int a = 0; a < D; ++a) {
      xk[a] = xj[a];
      if ((g.permask >> a) & 1) code |= (rr[a] < -half[a] ? 1 : (rr[a] > half[a] ? 2 : 0)) << (2*a);
    }
    image_pos<D>(g, code, xk);
#pragma unroll
    for (int a = 0; a < D; ++a) rr[a] = dsub(xi[a], xk[a]);
  }
  return eta2<D>(fmin(hi, hj), rr) <= ext2 && !(self && code == 0);
}

// U: entries in flight per lane.
template <int D, bool DENS, bool DT, typename R, int U, bool FILT, typename CP>
__device__ __forceinline__ void density_dt_node(const Fields& f, const Geo& g, const Phys& ph, const DevTable& tab,
                                                CP coef, int n, Scalars* sc, int* overflow) {
  constexpr int L = kNodeLanes;
  const int gl = xcd_block()*blockDim.x + threadIdx.x;
  const int i = gl/L, sub = gl & (L - 1);
  double dtmin = 1.7976931348623157e308;
  const bool valid = i < n;
  int r = 0;
  if (valid) {
    if (DT) r = f.run[i];
    double xi[D], vi[D], half[D];
#pragma unroll
    for (int a = 0; a < D; ++a) {
      xi[a] = f.x[a][i];
      vi[a] = DT ? f.v[a][i] : 0.0;
      half[a] = ((g.permask >> a) & 1) ? 0.5*(g.xmax[a] - g.xmin[a]) : 1.7976931348623157e308;
    }
    // pairwise limit min(ns_i, ns_j)/|v_ij| (GenericHydro.cc:196-210).  For isotropic H the
    // nodeScale is 1/(h^-1 nPerh) (lambda_max(h^-1 I) = h^-1; the reference's eigen-solver may
    // differ from it in the last bits), so the largest |v_ij|^2/min(ns)^2 is tracked as
    // max |v_ij|^2 max(h_i^-1, h_j^-1)^2, scaled by nPerh^2 at the end: no per-pair division
    // and no nodeScale read per neighbour
    const double hiD = f.hinv[i];
    double vmaxh = 0.0, rho0 = 0.0;
    if (DENS) {
      R w, gw, graw;
      kernel_wgw_c<R>(coef, tab, (R)0, hdet_iso<D, R>((R)hiD), w, gw, graw);   // self term W(|Hi ri - Hi ri|) = W(0)
      rho0 = f.m[i]*(double)w;
    }
    NodeSum<L, sizeof(R) == sizeof(float)> rhos(rho0, sub);
    const size_t ld = (size_t)f.ld;
    const int nn = FILT ? f.ccnt[i] : f.cnt[i];
    int count = 0;
    for (int k0 = 0; k0 < nn; k0 += U*L) {
      int js[U], codes[U];
      bool acc[U];
      lane_entries<U, L>(FILT ? f.cand : f.nbr, ld, k0, sub, i, nn, js, codes, acc);
      double xj[U][D], rr[U][D], vj[U][D], hj[U], mj[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        load_xh<D>(f.xh, js[u], xj[u], hj[u]);
        mj[u] = 0.0;
        if (!FILT) load_vm<D>(f.vmr, js[u], vj[u], mj[u]);
      }
      // the candidates are tested first; velocities and masses are then read for the accepted
      // ones only.  Accepted entries keep the candidates' order: a lane's place is the count so
      // far plus the accepted lanes of its quad below it
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (FILT) {
          acc[u] = acc[u] && neighbor_test<D>(g, ph.ext2, half, xi, hiD, xj[u], hj[u], js[u] == i, codes[u], rr[u]);
          const unsigned q = (unsigned)(__ballot(acc[u]) >> (threadIdx.x & 63 & ~(L - 1))) & ((1u << L) - 1u);
          const int place = count + __popc(q & ((1u << sub) - 1u));
          if (acc[u] && place < f.cap)
            f.nbr[ell_at(place, i, ld)] = (uint32_t)js[u] | ((uint32_t)codes[u] << kImgShift);
          count += __popc(q);
        } else if (acc[u]) {
          if (codes[u]) image_pos<D>(g, codes[u], xj[u]);
#pragma unroll
          for (int a = 0; a < D; ++a) rr[u][a] = xi[a] - xj[u][a];
        }
      }
      if (!DENS && !DT) continue;
      if (FILT) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (acc[u]) load_vm<D>(f.vmr, js[u], vj[u], mj[u]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        R w = (R)0;
        if (acc[u]) {
          if (DENS) {
            R d[D], gw, graw;
#pragma unroll
            for (int a = 0; a < D; ++a) d[a] = (R)hj[u]*(R)rr[u][a];
            // (in mixed precision the package-level sum starts most chains from the second axis:
            // the last FP32 bit it has always had)
            const R s = !FILT && sizeof(R) == sizeof(float) && !(D == 3 && sub == 0) ? norm2_second<D>(d) : norm2<D>(d);
            kernel_wgw_c<R>(coef, tab, sqrt(s), hdet_iso<D, R>((R)hj[u]), w, gw, graw);
          }
          if (DT) {
            double d[D];
#pragma unroll
            for (int a = 0; a < D; ++a)
              d[a] = vi[a] - (codes[u] ? refl_sign<D>(g, codes[u], a)*vj[u][a] : vj[u][a]);
            const double hm = fmax(hiD, hj[u]);
            vmaxh = fmax(vmaxh, norm2<D>(d)*(hm*hm));
          }
        }
        if (DENS) rhos.add(mj[u], w);
      }
    }
    if (FILT && sub == 0) {
      f.cnt[i] = count;
      if (count > f.cap) ask_capacity(overflow, count);
    }
    double rho = rhos.total();
    if (DT) {
      vmaxh = fmax(vmaxh, quad_swap<0xB1>(vmaxh));
      vmaxh = fmax(vmaxh, quad_swap<0x4E>(vmaxh));
    }
    if (sub == 0 && (DENS || DT)) {
      if (DENS) f.rho[i] = rho; else rho = f.rho[i];
      if (DT) {
        const double nsi = f.ns[i];
        const double tiny = 2.220446049250313e-16;
        // min(ns_i, ns_j)/max(tiny, |v_ij|) minimised over the pairs
        const double vmax2 = vmaxh*(ph.nperh*ph.nperh);
        if (vmax2 > 0.0) dtmin = fmin(dtmin, 1.0/sqrt(vmax2));
        dtmin = fmin(dtmin, nsi/(f.cs[i] + tiny));
        const double csq = sqrt(f.maxQ[i]/rho);
        dtmin = fmin(dtmin, nsi/(csq + tiny));
        double tr = 0.0;
#pragma unroll
        for (int a = 0; a < D; ++a) tr += f.DvDx[(a*D + a)*(size_t)f.ld + i];
        dtmin = fmin(dtmin, 1.0/(fabs(tr) + tiny));
        double ai[D];
#pragma unroll
        for (int a = 0; a < D; ++a) ai[a] = f.DvDt[a][i];
        const double vmag = sqrt(norm2_second<D>(vi));
        dtmin = fmin(dtmin, 0.1*fmax(nsi/(vmag + tiny), vmag/(sqrt(norm2_second<D>(ai)) + tiny)));
        if (ph.useVmagDt) dtmin = fmin(dtmin, nsi/(vmag + 1.0e-10));
      }
    }
  }
  if (DT) run_min(sc, r, dtmin, valid && sub == 0);
}

template <int D, bool DENS, bool DT, typename R, int U, bool FILT = false>
__global__ void __launch_bounds__(kBlock) k_density_dt(Fields f, Geo g, Phys ph, DevTable tab, int n, Scalars* sc,
                                                       int* overflow, int ldsTable) {
  with_table<R>(tab, DENS ? ldsTable : 0, [&](auto coef) {
    density_dt_node<D, DENS, DT, R, U, FILT>(f, g, ph, tab, coef, n, sc, overflow);
  });
}

// Integrator::selectDt (Integrator/Integrator.cc:116-169), one thread per run.
struct DtLimits { double lo, hi, growth; };
// Integrator::selectDt from the run's votes.
__device__ __forceinline__ double choose_dt(const Scalars& s, double hydro, const DtLimits& lim, int useGravity) {
  const double lo = fmin(lim.lo, s.tEnd - s.t), hi = fmin(lim.hi, s.tEnd - s.t);
  double dt = hi;
  if (hydro > 0.0 && hydro < dt) dt = hydro;
  if (useGravity) {
    const double gd = s.gravDt;
    if (gd > 0.0 && gd < dt) dt = gd;
  }
  dt = fmin(dt, lim.growth*s.lastDt);
  return fmin(hi, fmax(lo, dt));
}
__device__ __forceinline__ void store_dt(Scalars& s, const Phys& ph, const DtLimits& lim, int useGravity) {
  s.skinD = 0ull;
  s.skinG = 0ull;
  if (!s.active) { s.dt = 0.0; s.hdt = 0.0; return; }
  const double hydro = ord_value(s.dtBits)*ph.cfl;
  const double dt = choose_dt(s, hydro, lim, useGravity);
  s.hydroDt = hydro;
  s.dt = dt;
  s.hdt = 0.5*dt;
}
__global__ void k_select_dt(Scalars* sc, int nruns, Phys ph, DtLimits lim, int useGravity) {
  const int r = blockIdx.x*blockDim.x + threadIdx.x;
  if (r < nruns) store_dt(sc[r], ph, lim, useGravity);
}
__global__ void k_reset_dt(Scalars* sc, int nruns) {
  const int r = blockIdx.x*blockDim.x + threadIdx.x;
  if (r < nruns) sc[r].dtBits = kNoVote;
}

// End of the step: time advance (a run is done when it reaches its end time), and the runs' scalars and the overflow flag into the host's memory,
// then the number of the step, which tells a host that polls for it that all of it is there (one
// block writes them; with more than one, the host waits for the stream).
__global__ void k_advance_time(Scalars* sc, int nruns, Scalars* host, int* flags, int* hostFlags) {
  const int r = blockIdx.x*blockDim.x + threadIdx.x;
  if (r == 0) {
    flags[kFlagWrap] = 1;
    hostFlags[kFlagOverflow] = flags[kFlagOverflow];
  }
  if (r < nruns) {
    Scalars& s = sc[r];
    if (s.active) {
      s.t = s.t + s.dt;
      s.lastDt = s.dt;
      s.cycle = s.cycle + 1;
    }
    host[r] = s;
  }
  if (gridDim.x > 1) return;
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) {
    const int step = flags[kFlagStep] + 1;
    flags[kFlagStep] = step;
    __hip_atomic_store(&hostFlags[kFlagStep], step, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// ---------------------------------------------------------------------------
// CheapSynchronousRK2 mid-step: state.update with timeAdvanceOnly (increments with
// the previous step's derivatives), then the EOS policies
// (Integrator/CheapSynchronousRK2.cc:74-77; DataBase/IncrementStateInline.hh:42-80,
// IncrementBoundedStateInline.hh; ReplaceBoundedState::updateAsIncrement; GammaLawGas),
// preceded by the dt selection.
// ---------------------------------------------------------------------------
template <int D>
__global__ void __launch_bounds__(kBlock) k_midstep(Fields f, Phys ph, Scalars* sc, int nruns, DtLimits lim, int n) {
  const int i = blockIdx.x*blockDim.x + threadIdx.x;
  // dt selection: thread r stores run r's, and each node forms its run's from the fields that no
  // thread stores (one launch instead of two, 5 us of a small run's step)
  if (i < nruns) store_dt(sc[i], ph, lim, ph.gravity);
  if (i >= n) return;
  const Scalars& s = sc[f.run[i]];
  const double hdt = 0.5*choose_dt(s, ord_value(s.dtBits)*ph.cfl, lim, ph.gravity);
#pragma unroll
  for (int a = 0; a < D; ++a) {
    f.xm[a][i] = f.x[a][i] + hdt*f.DxDt[a][i];
    double va = f.v[a][i] + hdt*f.DvDt[a][i];
    if (ph.gravity) va = va + hdt*f.DvDtG[a][i];
    f.vm[a][i] = va;
  }
  const double rho = fmin(ph.rho_max, fmax(ph.rho_min, f.rho[i] + hdt*f.DrhoDt[i]));
  const double eps = f.eps[i] + hdt*f.DepsDt[i];
  const double h = fmin(ph.hminInv, fmax(ph.hmaxInv, f.hinv[i] + hdt*f.DHDt[i]));
  const double cs = sqrt(fmax(0.0, ph.gamma*ph.g1*eps));
  f.rhom[i] = rho;
  f.epsm[i] = eps;
  f.hinvm[i] = h;
  f.Pm[i] = ph.g1*rho*eps;
  f.csm[i] = cs;
  double2* P = reinterpret_cast<double2*>(f.xhm) + 2*(size_t)i;
  P[0] = make_double2(f.xm[0][i], D >= 2 ? f.xm[1 % D][i] : 0.0);
  P[1] = make_double2(D >= 3 ? f.xm[2 % D][i] : 0.0, h);
}

// Per-node pressure term Prho = safeInv(omega)*P/rho^2 of the midpoint state (SPH.cc:425-426),
// written with the rest of node i's midpoint record (Fields::pkm), which also carries 1/rho
// (the viscous pressure Q/rho of every pair the node takes part in is formed with it).
template <int D>
__device__ __forceinline__ void write_mid_record(const Fields& f, int i, double om) {
  const double rho = f.rhom[i];
  const double prho = (om/(om*om + 1.0e-30))*f.Pm[i]/(rho*rho);
  f.prhom[i] = prho;
  double2* P = reinterpret_cast<double2*>(f.pkm) + 4*(size_t)i;
  P[0] = make_double2(f.vm[0][i], D >= 2 ? f.vm[1 % D][i] : 0.0);
  P[1] = make_double2(D >= 3 ? f.vm[2 % D][i] : 0.0, f.m[i]);
  P[2] = make_double2(rho, f.csm[i]);
  P[3] = make_double2(prho, 1.0/rho);
}

// The midpoint records (Fields::xhm, Fields::pkm) from the midpoint arrays.  keepOmega: the
// midpoint grad-h correction is the state's (no grad-h pass: gradhCorrection off, where it
// stays at its initial 1).
template <int D>
__global__ void __launch_bounds__(kBlock) k_pack_mid(Fields f, int n, int keepOmega) {
  const int i = blockIdx.x*blockDim.x + threadIdx.x;
  if (i >= n) return;
  double2* P = reinterpret_cast<double2*>(f.xhm) + 2*(size_t)i;
  P[0] = make_double2(f.xm[0][i], D >= 2 ? f.xm[1 % D][i] : 0.0);
  P[1] = make_double2(D >= 3 ? f.xm[2 % D][i] : 0.0, f.hinvm[i]);
  double om = f.omegam[i];
  if (keepOmega) { om = f.omega[i]; f.omegam[i] = om; }
  write_mid_record<D>(f, i, om);
}

// EOS policies on the state arrays (PressurePolicy, SoundSpeedPolicy; GammaLawGas.cc:185-245).
__global__ void __launch_bounds__(kBlock) k_eos(Fields f, Phys ph, int n) {
  const int i = blockIdx.x*blockDim.x + threadIdx.x;
  if (i >= n) return;
  f.P[i] = ph.g1*f.rho[i]*f.eps[i];
  f.cs[i] = sqrt(fmax(0.0, ph.gamma*ph.g1*f.eps[i]));
}

// ---------------------------------------------------------------------------
// computeSPHOmegaGradhCorrection (SPH/computeSPHOmegaGradhCorrection.cc:136-204), gather form.
// Positions and h^-1 come from an (x, h^-1) record array.  MID: the midpoint pass, which
// also writes node i's midpoint record for the SPH pass (write_mid_record).  runMask
// (optional): only nodes of runs with a non-zero entry are updated.
// ---------------------------------------------------------------------------
// L lanes per node, U entries in flight per lane; the sums are in list order for either L, so the
// choice by particle count (omega_wide_nodes) changes no bit.
template <int D, typename R, bool MID, int U, int L, typename CP>
__device__ __forceinline__ void omega_node(const Fields& f, const Geo& g, const DevTable& tab, CP coef, int n,
                                           const double* xh, double* omega, const int* runMask) {
  const int gl = xcd_block()*blockDim.x + threadIdx.x;
  const int i = gl/L, sub = gl & (L - 1);
  if (i >= n) return;                       // the lanes of a node leave together
  if (runMask && !runMask[f.run[i]]) return;
  double xi[D], hid;
  load_xh<D>(xh, i, xi, hid);
  const R hi = (R)hid;
  const R hdeti = hdet_iso<D, R>(hi);
  NodeSum<L, true> ws(0.0, sub), gs(0.0, sub);
  const int nn = f.cnt[i];
  for (int k0 = 0; k0 < nn; k0 += U*L) {
    int js[U], codes[U];
    bool in[U];
    lane_entries<U, L>(f.nbr, (size_t)f.ld, k0, sub, i, nn, js, codes, in);
    double xj[U][D], hjunk[U];
#pragma unroll
    for (int u = 0; u < U; ++u) load_xh<D>(xh, js[u], xj[u], hjunk[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      R w = (R)0, t = (R)0;
      if (in[u]) {
        if (codes[u]) image_pos<D>(g, codes[u], xj[u]);
        R d[D], gw, graw;
#pragma unroll
        for (int a = 0; a < D; ++a) d[a] = hi*(R)(xi[a] - xj[u][a]);
        const R eta = sqrt(norm2<D>(d));
        kernel_wgw_c<R>(coef, tab, eta, hdeti, w, gw, graw);
        t = rounded_product(eta, gw);
      }
      ws.add(w);
      gs.add(t);
    }
  }
  double wsum = ws.total();
  const double gsum = gs.total();
  if (sub) return;
  double om;
  if (nn == 0) {
    om = 1.0;
  } else {
    wsum += (double)hdeti*tab.W0;
    om = fmax(1.0e-30, -gsum/(double(D)*wsum));
  }
  omega[i] = om;
  if (MID) write_mid_record<D>(f, i, om);
}
template <int D, typename R, bool MID, int U, int L>
__global__ void __launch_bounds__(kBlock) k_omega(Fields f, Geo g, DevTable tab, int n, const double* xh,
                                                  double* omega, const int* runMask, int ldsTable) {
  with_table<R>(tab, ldsTable,
                [&](auto coef) { omega_node<D, R, MID, U, L>(f, g, tab, coef, n, xh, omega, runMask); });
}

// SynchronousRK2 with TreeGravity as the only package (Integrator/SynchronousRK2.cc:40-135): the
// half step with the start-of-step derivatives (DxDt = v, DvDt = the tree acceleration), then the
// full step from the start state with the midpoint ones (TreeGravity.cc:303-316 sets DxDt = v).
template <int D>
__global__ void __launch_bounds__(kBlock) k_grav_mid(Fields f, const Scalars* sc, int n) {
  const int i = xcd_block()*blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double hdt = sc[f.run[i]].hdt;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    const double v = f.v[a][i];
    f.xm[a][i] = f.x[a][i] + hdt*v;
    f.vm[a][i] = v + hdt*f.DvDtG[a][i];
  }
}
template <int D>
__global__ void __launch_bounds__(kBlock) k_grav_full(Fields f, const Scalars* sc, int n) {
  const int i = xcd_block()*blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double dt = sc[f.run[i]].dt;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    const double vm = f.vm[a][i];
    f.x[a][i] = f.x[a][i] + dt*vm;
    f.v[a][i] = f.v[a][i] + dt*f.DvDtG[a][i];
    f.DxDt[a][i] = vm;
  }
}

// One pass of iterateIdealH (Utilities/iterateIdealH.cc:118-176) with the SPHSmoothingScale
// package alone (SmoothingScale/SPHSmoothingScale.cc:154-245) on the connectivity state: the
// zeroth moment of kernelValueSPH over the node's neighbours (images included) gives the ideal h;
// a node not yet converged takes it, and is flagged done once its H moved by at most tol.  The
// flags are indexed by the node's run-local id, so they survive the reorders between passes.
template <int D>
__global__ void __launch_bounds__(kBlock) k_ideal_h(Fields f, Geo g, Phys ph, DevTable tab, int n, double tol,
                                                    int* done, unsigned long long* maxDelta) {
  const int i = xcd_block()*blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t id = f.oid[i] & (((int64_t)1 << 40) - 1);
  if (done[id]) return;
  const double* coef = table_coef<double>(tab);
  double xi[D], hi;
  load_xh<D>(f.xh, i, xi, hi);
  const size_t ld = (size_t)f.ld;
  double m0 = 0.0;
  const int nn = f.cnt[i];
  for (int k = 0; k < nn; ++k) {
    const uint32_t e = f.nbr[ell_at(k, i, ld)];
    const int j = (int)(e & kIdxMask), code = (int)(e >> kImgShift);
    double xj[D], hj;
    load_xh<D>(f.xh, j, xj, hj);
    if (code) image_pos<D>(g, code, xj);
    double s = 0.0;
#pragma unroll
    for (int a = 0; a < D; ++a) { const double r = hi*(xi[a] - xj[a]); s += r*r; }
    double w, gw, graw;
    kernel_wgw_c<double>(coef, tab, sqrt(s), hdet_iso<D, double>(hi), w, gw, graw);
    m0 += fabs(graw);
  }
  m0 = rootnu<D>(fmax(0.0, m0));
  const double cur = (fabs(m0) <= 1.0e-15*fmax(1.0, fabs(m0))) ? 0.5*ph.nperh : nperh_lookup(tab, m0);
  const double sr = fmin(4.0, fmax(0.25, ph.nperh/(cur + 1.0e-30)));
  const double aa = sr < 1.0 ? 0.4*(1.0 + sr*sr) : 0.4*(1.0 + 1.0/(sr*sr*sr));
  const double hi1 = fmin(ph.hmax, fmax(ph.hmin, (1.0/hi)*(1.0 - aa + aa*sr)));
  const double H1 = 1.0/hi1;
  // eigenvalues of H1^1/2 H^-1 H1^1/2 (isotropic: one value)
  const double sq = sqrt(H1);
  const double dH = fabs((sq*(1.0/hi))*sq - 1.0);
  if (dH <= tol) done[id] = 1;
  const unsigned long long b = (unsigned long long)__double_as_longlong(dH);
  if (b > *maxDelta) atomicMax(maxDelta, b);
  f.hinv[i] = H1;
}

// Per-run extents for the next grid: min and max hinv and the bounding box, as ordered bits.
// One block per tile (run, begin, end) of a run's contiguous particle segment; a block
// reduces its tile and adds one set of atomics.
// ext layout per run (kExt values): [hinv_min, xmin0, xmax0, xmin1, xmax1, xmin2, xmax2, hinv_max].
constexpr int kExt = 8;
__host__ __device__ __forceinline__ bool ext_is_min(int q) { return q == 0 || (q < 7 && (q & 1)); }
template <int D>
__global__ void __launch_bounds__(kBlock) k_extent(Fields f, const int* tiles, unsigned long long* ext) {
  __shared__ unsigned long long red[kExt][kBlock/64];
  const int r = tiles[3*blockIdx.x], b = tiles[3*blockIdx.x + 1], e = tiles[3*blockIdx.x + 2];
  unsigned long long v[kExt];
#pragma unroll
  for (int q = 0; q < kExt; ++q) v[q] = ext_is_min(q) ? ~0ull : 0ull;
  for (int i = b + threadIdx.x; i < e; i += blockDim.x) {
    const unsigned long long h = ord_bits(f.hinv[i]);
    v[0] = h < v[0] ? h : v[0];
    v[7] = h > v[7] ? h : v[7];
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const unsigned long long x = ord_bits(f.x[a][i]);
      v[1 + 2*a] = x < v[1 + 2*a] ? x : v[1 + 2*a];
      v[2 + 2*a] = x > v[2 + 2*a] ? x : v[2 + 2*a];
    }
  }
#pragma unroll
  for (int q = 0; q < kExt; ++q) {
    unsigned long long x = v[q];
    for (int o = 32; o > 0; o >>= 1) {
      const unsigned long long y = __shfl_xor(x, o);
      x = ext_is_min(q) ? (y < x ? y : x) : (y > x ? y : x);
    }
    if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = x;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long* out = ext + (size_t)r*kExt;
    for (int q = 0; q < kExt; ++q) {
      if (q >= 1 + 2*D && q < 7) continue;
      unsigned long long x = red[q][0];
      for (int w = 1; w < kBlock/64; ++w) {
        const unsigned long long y = red[q][w];
        x = ext_is_min(q) ? (y < x ? y : x) : (y > x ? y : x);
      }
      if (ext_is_min(q)) atomicMin(&out[q], x);
      else atomicMax(&out[q], x);
    }
  }
}

// A candidate build's small host arrays into device memory in one launch, read from the host's pinned
// memory (each copy by itself was 5 to 10 us of a small run's build), and the extents cleared.
struct FetchSet {
  const int* src[6];
  int* dst[6];
  int n[6];
  int count;
};
__global__ void __launch_bounds__(kBlock) k_fetch(FetchSet s, unsigned long long* ext, int next) {
  const int i = blockIdx.x*kBlock + threadIdx.x;
  for (int k = 0; k < s.count; ++k)
    if (i < s.n[k]) s.dst[k][i] = s.src[k][i];
  if (i < next) ext[i] = ext_is_min(i % kExt) ? ~0ull : 0ull;
}
// Its cell tables, handed-over counts and overflow counts cleared, the grids fetched.
__global__ void __launch_bounds__(kBlock) k_begin_build(FetchSet grids, int* start, int* end, int64_t cells, int* tcnt,
                                                        int n, int* overflow) {
  const int64_t i = (int64_t)blockIdx.x*kBlock + threadIdx.x;
  if (i < grids.n[0]) grids.dst[0][i] = grids.src[0][i];
  if (i < cells) start[i] = end[i] = 0;
  if (i < n) tcnt[i] = 0;
  if (i < 2) overflow[i] = 0;
}

// Non-finite guard on the state (NaN/Inf -> per-run status word).
template <int D>
__global__ void __launch_bounds__(kBlock) k_finite(Fields f, int n, Scalars* sc) {
  const int i = blockIdx.x*blockDim.x + threadIdx.x;
  if (i >= n) return;
  bool ok = isfinite(f.rho[i]) && isfinite(f.eps[i]) && isfinite(f.hinv[i]);
  for (int a = 0; a < D; ++a) ok = ok && isfinite(f.x[a][i]) && isfinite(f.v[a][i]);
  if (!ok) atomicOr(&sc[f.run[i]].nonfinite, 1);
}

// `rows` arrays of n doubles, ld apart (a kernel: a captured graph holds no copies).
__global__ void __launch_bounds__(kBlock) k_copy_rows(const double* __restrict__ src, double* __restrict__ dst, int64_t n,
                                                      int64_t ld, int rows) {
  const int64_t i = (int64_t)blockIdx.x*kBlock + threadIdx.x;
  if (i < n)
    for (int c = 0; c < rows; ++c) dst[c*ld + i] = src[c*ld + i];
}
// dst[0..n) = src[0..n) (doubles): the velocities of the finished runs behind the active ones,
// which the update does not write, carried into the other velocity buffer.
__global__ void __launch_bounds__(kBlock) k_copy_doubles(const double* __restrict__ src, double* __restrict__ dst,
                                                         int64_t n) {
  const int64_t i = (int64_t)blockIdx.x*blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

// Unique-pair count of the neighbour lists (ConnectivityMap::nodePairList().size(),
// Neighbor/ConnectivityMap.cc:925-927): an entry (i, j) is i's pair when j is an image or a later
// slot (calculatePairInteraction, ConnectivityMapInline.hh:305-307).  One partial count per block
// (no atomics), summed by k_sum_partials.
__global__ void __launch_bounds__(kBlock) k_count_pairs(const uint32_t* nbr, const int32_t* cnt, size_t ld, int n,
                                                        unsigned long long* partial) {
  __shared__ unsigned long long red[kBlock/64];
  const int i = blockIdx.x*blockDim.x + threadIdx.x;
  unsigned long long c = 0;
  if (i < n) {
    const int nn = cnt[i];
    for (int k = 0; k < nn; ++k) {
      const uint32_t e = nbr[ell_at(k, i, ld)];
      c += ((e >> kImgShift) != 0u || (int)(e & kIdxMask) > i) ? 1ull : 0ull;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_down(c, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += red[w];
    partial[blockIdx.x] = t;
  }
}

// out[0] = sum of partial[0..nb); one block.
__global__ void __launch_bounds__(kBlock) k_sum_partials(const unsigned long long* partial, int nb,
                                                         unsigned long long* out) {
  __shared__ unsigned long long red[kBlock/64];
  unsigned long long c = 0;
  for (int k = threadIdx.x; k < nb; k += blockDim.x) c += partial[k];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_down(c, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += red[w];
    out[0] = t;
  }
}

}  // namespace spx
