// Morton-key octree and interaction lists on gfx950.
//
// The reference builds its adaptive octree by inserting sites one at a time and splitting a
// cell when it reaches ncrit sites (src/core/fmm/tree.cc:134-237). The resulting set of cells
// does not depend on insertion order: a cell exists iff it is a non-empty octant of a split
// cell, and a cell is split iff its region holds >= ncrit sites. This file builds that same
// set in parallel:
//   1. root centre = mean of the positions summed in index order, half-width = 1.001 * max
//      deviation (tree.cc:157-189) -- on the host, the sum sequential to keep its rounding;
//   2. per site, the octant path of 21 levels, replaying the reference's FP64 cell-centre
//      arithmetic child = parent + (r/2) * (+-1) and the strict '>' octant tests
//      (tree.cc:99-102,119-120,196-198), packed 3 bits per level into a 63-bit Morton key;
//   3. stable radix sort of (key, index): leaf contents keep increasing site index, as in
//      the reference (its leaf lists are filled in insertion order);
//   4. leaf level of each site = first level whose prefix range holds < ncrit sites;
//   5. cells per level (level order, Morton order inside a level), centres re-derived from
//      the prefix path with the same arithmetic, rmax = sqrt(3 r r) (tree.cc:17);
//   6. dual-tree traversal (fmm/calculate.cc:74-127) level-synchronously over a frontier of
//      (target, source) cell pairs with the reference's MAC R*theta > rmaxA + rmaxB and split
//      rule; lists are then sorted by (target, source) into per-target CSR (owner computes).
// Cell identity (level, centre) and list membership are bit-identical to the reference; only
// the cell numbering differs (level order here, creation order there).
//
// Forests: a system may hold several independent snapshots ("segments", contiguous site ranges
// with their own ncrit). Each gets its own root (steps 1-2 per segment), the sort is segmented,
// cell ranges never cross a segment boundary, and the traversal starts from every (root, root)
// pair, so no list entry joins two snapshots. A segment whose ncrit exceeds its size is a single
// leaf whose near list is itself: its far field is empty and its near field is the exact direct
// sum. One segment with the system's ncrit is the reference's tree.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <climits>
#include <cmath>

#include "system.hh"

namespace cppe_dev {

constexpr int kMaxLevel = 21;

// ---------------------------------------------------------------------------------------------
// Root cell of every snapshot (sites [off[g], off[g+1]) of the caller's positions): centre and
// half-width (tree.cc:157-189). On the host: the mean is a chain of additions in index order, which one
// lane walks at 23 cycles a site (2.9 ms at 300,000 sites) and a host core at 4, beside the copy of the
// positions to the device.
static std::vector<double> host_roots(const double* pos, const std::vector<int>& off) {
  const int ns = (int)off.size() - 1;
  std::vector<double> root(4 * (size_t)ns);
  for (int g = 0; g < ns; ++g) {
    const int n = off[g + 1] - off[g];
    const double* p = pos + 3 * (size_t)off[g];
    double s[3] = {0.0, 0.0, 0.0}, m[3] = {0.0, 0.0, 0.0};
    for (int k = 0; k < n; ++k)
      for (int c = 0; c < 3; ++c) s[c] = s[c] + p[3 * (size_t)k + c];
    for (int c = 0; c < 3; ++c) s[c] = s[c] / (double)n;
    for (int k = 0; k < n; ++k)
      for (int c = 0; c < 3; ++c) {
        const double d = std::fabs(p[3 * (size_t)k + c] - s[c]);
        m[c]           = d > m[c] ? d : m[c];
      }
    for (int c = 0; c < 3; ++c) root[4 * (size_t)g + c] = s[c];
    root[4 * (size_t)g + 3] = (m[0] > m[1] ? (m[0] > m[2] ? m[0] : m[2]) : (m[1] > m[2] ? m[1] : m[2])) * 1.001;
  }
  return root;
}

// child centre update of add_child (tree.cc:99-102); r is the parent's half-width
__device__ __forceinline__ void child_centre(int oct, double& cx, double& cy, double& cz, double& r) {
#pragma clang fp contract(off)
  double rc = r / 2.0;
  cx = cx + rc * (double)((oct & 1) * 2 - 1);
  cy = cy + rc * (double)((oct & 2) - 1);
  cz = cz + rc * (double)((oct & 4) / 2 - 1);
  r  = rc;
}

__global__ __launch_bounds__(256) void k_keys(int n, const double* __restrict__ x,
                                              const double* __restrict__ y,
                                              const double* __restrict__ z,
                                              const double* __restrict__ root, const int* __restrict__ seg_of,
                                              uint64_t* __restrict__ keys, int* __restrict__ idx) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double* rt = root + 4 * seg_of[i];
  double cx = rt[0], cy = rt[1], cz = rt[2], r = rt[3];
  const double px = x[i], py = y[i], pz = z[i];
  uint64_t key = 0;
  for (int l = 0; l < kMaxLevel; ++l) {
    int oct = (px > cx) + ((py > cy) << 1) + ((pz > cz) << 2);
    key     = (key << 3) | (uint64_t)oct;
    child_centre(oct, cx, cy, cz, r);
  }
  keys[i] = key;
  idx[i]  = i;
}

__device__ __forceinline__ int lower_bound_u64(const uint64_t* a, int lo, int hi, uint64_t v) {
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    if (a[mid] < v)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

__device__ __forceinline__ uint64_t prefix_of(uint64_t key, int L) {
  return L == 0 ? 0ull : (key >> (3 * (kMaxLevel - L)));
}

// range end (exclusive) of the level-L cell holding sorted position i, searched in [i, hi)
__device__ __forceinline__ int cell_end(const uint64_t* keys, int i, int hi, int L) {
  if (L == 0) return hi;
  uint64_t p    = prefix_of(keys[i], L);
  uint64_t next = (p + 1) << (3 * (kMaxLevel - L));
  if (L == 1 && p == 7) return hi;
  return lower_bound_u64(keys, i, hi, next);
}

// Leaf level of each sorted site: the first level whose cell holds < ncrit sites.
__global__ __launch_bounds__(256) void k_leaf_level(int n, const int* __restrict__ seg_of,
                                                    const int* __restrict__ seg_off,
                                                    const int* __restrict__ seg_ncrit,
                                                    const uint64_t* __restrict__ keys,
                                                    int* __restrict__ leaf_level, int* __restrict__ err) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int g     = seg_of[i];
  const int ncrit = seg_ncrit[g];
  int lo = seg_off[g], hi = seg_off[g + 1];
  for (int L = 0; L <= kMaxLevel; ++L) {
    if (L > 0) {
      uint64_t p = prefix_of(keys[i], L);
      uint64_t a = p << (3 * (kMaxLevel - L));
      lo         = lower_bound_u64(keys, lo, hi, a);
      hi         = (L == 1 && p == 7) ? hi : lower_bound_u64(keys, lo, hi, (p + 1) << (3 * (kMaxLevel - L)));
    }
    if (hi - lo < ncrit) {
      leaf_level[i] = L;
      return;
    }
  }
  leaf_level[i] = kMaxLevel;
  atomicExch(err, 1);  // >= ncrit sites share one finest cell (coincident sites)
}

__global__ __launch_bounds__(256) void k_heads(int n, int L, const uint64_t* __restrict__ keys,
                                               const int* __restrict__ seg_of, const int* __restrict__ seg_off,
                                               const int* __restrict__ leaf_level, int* __restrict__ flag) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int f = 0;
  if (leaf_level[i] >= L)
    f = (i == seg_off[seg_of[i]]) || (prefix_of(keys[i], L) != prefix_of(keys[i - 1], L));
  flag[i] = f;
}

__global__ __launch_bounds__(256) void k_fill_cells(
      int n, int L, int cell0, int prev0, int prev_n, const uint64_t* __restrict__ keys,
      const int* __restrict__ seg_of, const int* __restrict__ seg_off,
      const int* __restrict__ leaf_level, const int* __restrict__ flag, const int* __restrict__ rank,
      const double* __restrict__ root, double* cx, double* cy, double* cz, double* cr, double* crmax,
      int* start, int* count, int* parent, int* level) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !flag[i]) return;
  const int c    = cell0 + rank[i];
  const int g    = seg_of[i];
  uint64_t key   = keys[i];
  const double* rt = root + 4 * g;
  double x = rt[0], y = rt[1], z = rt[2], r = rt[3];
  for (int l = 1; l <= L; ++l) {
    int oct = (int)((key >> (3 * (kMaxLevel - l))) & 7ull);
    child_centre(oct, x, y, z, r);
  }
  cx[c]    = x;
  cy[c]    = y;
  cz[c]    = z;
  cr[c]    = r;
  crmax[c] = sqrt(3 * r * r);
  start[c] = i;
  count[c] = cell_end(keys, i, seg_off[g + 1], L) - i;
  level[c] = L;
  if (L == 0) {
    parent[c] = c;  // a root (one per snapshot) is its own parent
  } else {
    // parent = last cell of the previous level whose start <= i
    int lo = 0, hi = prev_n;
    while (lo < hi) {
      int mid = (lo + hi) >> 1;
      if (start[prev0 + mid] <= i)
        lo = mid + 1;
      else
        hi = mid;
    }
    parent[c] = prev0 + lo - 1;
  }
}

__global__ __launch_bounds__(256) void k_link(int ncells, const int* __restrict__ parent,
                                              const int* __restrict__ level, const int* __restrict__ start,
                                              const double* __restrict__ cx, const double* __restrict__ cy,
                                              const double* __restrict__ cz, int* child_first, int* nchild,
                                              int* octmask) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncells || level[c] == 0) return;
  const int p = parent[c];
  atomicMin(&child_first[p], c);
  atomicAdd(&nchild[p], 1);
  int oct = (cx[c] > cx[p]) + ((cy[c] > cy[p]) << 1) + ((cz[c] > cz[p]) << 2);
  atomicOr(&octmask[p], 1 << oct);
}

__global__ void k_fill_int(int* a, int n, int v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = v;
}

__global__ __launch_bounds__(256) void k_gather_sorted(int n, const int* __restrict__ idx,
                                                       const double* __restrict__ xin,
                                                       const double* __restrict__ yin,
                                                       const double* __restrict__ zin, double* xo,
                                                       double* yo, double* zo, int* iperm) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int j = idx[i];
  xo[i]       = xin[j];
  yo[i]       = yin[j];
  zo[i]       = zin[j];
  iperm[j]    = i;
}

__global__ void k_leaf_flags(int ncells, const int* nchild, int* flag) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < ncells) flag[c] = nchild[c] == 0;
}

// one block per leaf
__global__ void k_leaf_of(const int* __restrict__ leaf_ids, const int* __restrict__ start,
                          const int* __restrict__ count, int* __restrict__ leaf_of) {
  const int c = leaf_ids[blockIdx.x], i1 = start[c] + count[c];
  for (int i = start[c] + threadIdx.x; i < i1; i += blockDim.x) leaf_of[i] = c;
}

__global__ void k_scatter_ids(int n, const int* flag, const int* rank, int* out) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < n && flag[c]) out[rank[c]] = c;
}

template <typename T>
static void exclusive_scan(const T* in, T* out, int n, hipStream_t s, dbuf<char>& tmp) {
  size_t bytes = 0;
  CPPE_HIP_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, in, out, n, s));
  tmp.alloc(bytes + 16);
  CPPE_HIP_CHECK(hipcub::DeviceScan::ExclusiveSum(tmp.p, bytes, in, out, n, s));
}

void device_scan(System& S, const int* in, int* out, int n) {
  dbuf<char> tmp;
  exclusive_scan(in, out, n, S.stream, tmp);
  CPPE_HIP_CHECK(hipStreamSynchronize(S.stream));  // before the scratch is released
}

// Builds the octree over the positions held in S.x/y/z and, on the host, in pos (caller order); on return
// S.x/y/z, S.perm and S.iperm are in device (sorted) order.
void build_octree(System& S, const double* pos) {
  const int n       = S.n;
  hipStream_t st    = S.stream;
  const int nseg    = S.nseg;
  Octree& T         = S.tree;
  dbuf<double> root;
  root.alloc(4 * (size_t)nseg);
  const std::vector<double> h_root = host_roots(pos, S.h_seg_off);
  CPPE_HIP_CHECK(hipMemcpyAsync(root.p, h_root.data(), sizeof(double) * h_root.size(), hipMemcpyHostToDevice, st));
  dbuf<uint64_t> keys_in, keys;
  dbuf<int> idx_in, idx;
  keys_in.alloc(n);
  keys.alloc(n);
  idx_in.alloc(n);
  idx.alloc(n);
  hipLaunchKernelGGL(k_keys, dim3(ceil_div(n, 256)), dim3(256), 0, st, n, S.x.p, S.y.p, S.z.p, root.p,
                     S.seg_of.p, keys_in.p, idx_in.p);
  dbuf<char> tmp;
  size_t bytes = 0;
  if (nseg == 1) {
    CPPE_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, keys_in.p, keys.p, idx_in.p, idx.p, n,
                                                      0, 3 * kMaxLevel, st));
    tmp.alloc(bytes + 16);
    CPPE_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(tmp.p, bytes, keys_in.p, keys.p, idx_in.p, idx.p, n, 0,
                                                      3 * kMaxLevel, st));
  } else {
    // snapshots stay where they are; each is sorted by key on its own (stable)
    CPPE_HIP_CHECK(hipcub::DeviceSegmentedRadixSort::SortPairs(nullptr, bytes, keys_in.p, keys.p, idx_in.p,
                                                               idx.p, n, nseg, S.seg_off.p, S.seg_off.p + 1, 0,
                                                               3 * kMaxLevel, st));
    tmp.alloc(bytes + 16);
    CPPE_HIP_CHECK(hipcub::DeviceSegmentedRadixSort::SortPairs(tmp.p, bytes, keys_in.p, keys.p, idx_in.p, idx.p,
                                                               n, nseg, S.seg_off.p, S.seg_off.p + 1, 0,
                                                               3 * kMaxLevel, st));
  }
  // sorted positions, permutation
  dbuf<double> xs, ys, zs;
  xs.alloc(n);
  ys.alloc(n);
  zs.alloc(n);
  S.perm.alloc(n);
  S.iperm.alloc(n);
  hipLaunchKernelGGL(k_gather_sorted, dim3(ceil_div(n, 256)), dim3(256), 0, st, n, idx.p, S.x.p, S.y.p,
                     S.z.p, xs.p, ys.p, zs.p, S.iperm.p);
  CPPE_HIP_CHECK(hipMemcpyAsync(S.perm.p, idx.p, sizeof(int) * n, hipMemcpyDeviceToDevice, st));
  S.x.swap(xs);
  S.y.swap(ys);
  S.z.swap(zs);

  dbuf<int> leaf_level, err;
  leaf_level.alloc(n);
  err.alloc(1);
  err.zero(st);
  hipLaunchKernelGGL(k_leaf_level, dim3(ceil_div(n, 256)), dim3(256), 0, st, n, S.seg_of.p, S.seg_off.p,
                     S.seg_ncrit.p, keys.p, leaf_level.p, err.p);
  int h_err = 0;
  CPPE_HIP_CHECK(hipMemcpyAsync(&h_err, err.p, sizeof(int), hipMemcpyDeviceToHost, st));
  CPPE_HIP_CHECK(hipStreamSynchronize(st));
  if (h_err) throw std::runtime_error("octree: more than ncrit sites share one cell of the finest level");

  // cells level by level; capacity grows as needed
  dbuf<int> flag, rank;
  flag.alloc(n);
  rank.alloc(n);
  std::vector<int> level_off{0};
  size_t cap = std::max(64, n / 4);
  auto ensure = [&](size_t need) {
    if (need <= T.cx.n && T.cx.p) return;
    size_t nc = std::max(need, (size_t)(T.cx.n * 2));
    auto grow_d = [&](dbuf<double>& b) {
      dbuf<double> nb;
      nb.alloc(nc);
      if (b.p) CPPE_HIP_CHECK(hipMemcpyAsync(nb.p, b.p, sizeof(double) * b.n, hipMemcpyDeviceToDevice, st));
      CPPE_HIP_CHECK(hipStreamSynchronize(st));
      b.swap(nb);
    };
    auto grow_i = [&](dbuf<int>& b) {
      dbuf<int> nb;
      nb.alloc(nc);
      if (b.p) CPPE_HIP_CHECK(hipMemcpyAsync(nb.p, b.p, sizeof(int) * b.n, hipMemcpyDeviceToDevice, st));
      CPPE_HIP_CHECK(hipStreamSynchronize(st));
      b.swap(nb);
    };
    grow_d(T.cx);
    grow_d(T.cy);
    grow_d(T.cz);
    grow_d(T.cr);
    grow_d(T.crmax);
    grow_i(T.start);
    grow_i(T.count);
    grow_i(T.parent);
    grow_i(T.level);
    CPPE_HIP_CHECK(hipStreamSynchronize(st));
  };
  ensure(cap);
  int ncells = 0;
  int L      = 0;
  for (; L <= kMaxLevel; ++L) {
    hipLaunchKernelGGL(k_heads, dim3(ceil_div(n, 256)), dim3(256), 0, st, n, L, keys.p, S.seg_of.p,
                       S.seg_off.p, leaf_level.p, flag.p);
    exclusive_scan(flag.p, rank.p, n, st, tmp);
    int last_rank = 0, last_flag = 0;
    CPPE_HIP_CHECK(hipMemcpyAsync(&last_rank, rank.p + n - 1, sizeof(int), hipMemcpyDeviceToHost, st));
    CPPE_HIP_CHECK(hipMemcpyAsync(&last_flag, flag.p + n - 1, sizeof(int), hipMemcpyDeviceToHost, st));
    CPPE_HIP_CHECK(hipStreamSynchronize(st));
    const int nl = last_rank + last_flag;
    if (nl == 0) break;
    ensure((size_t)ncells + nl);
    const int prev0 = L > 0 ? level_off[L - 1] : 0;
    const int prevn = L > 0 ? level_off[L] - level_off[L - 1] : 0;
    hipLaunchKernelGGL(k_fill_cells, dim3(ceil_div(n, 256)), dim3(256), 0, st, n, L, ncells, prev0, prevn,
                       keys.p, S.seg_of.p, S.seg_off.p, leaf_level.p, flag.p, rank.p, root.p, T.cx.p, T.cy.p, T.cz.p, T.cr.p,
                       T.crmax.p, T.start.p, T.count.p, T.parent.p, T.level.p);
    ncells += nl;
    level_off.push_back(ncells);
  }
  T.ncells       = ncells;
  T.max_level    = (int)level_off.size() - 2;
  T.level_offset = level_off;
  T.child_first.alloc(ncells);
  T.nchild.alloc(ncells);
  T.octmask.alloc(ncells);
  hipLaunchKernelGGL(k_fill_int, dim3(ceil_div(ncells, 256)), dim3(256), 0, st, T.child_first.p, ncells,
                     INT_MAX);
  T.nchild.zero(st);
  T.octmask.zero(st);
  hipLaunchKernelGGL(k_link, dim3(ceil_div(ncells, 256)), dim3(256), 0, st, ncells, T.parent.p, T.level.p,
                     T.start.p, T.cx.p, T.cy.p, T.cz.p, T.child_first.p, T.nchild.p, T.octmask.p);
  // leaf ids
  dbuf<int> lf, lr;
  lf.alloc(ncells);
  lr.alloc(ncells);
  hipLaunchKernelGGL(k_leaf_flags, dim3(ceil_div(ncells, 256)), dim3(256), 0, st, ncells, T.nchild.p, lf.p);
  exclusive_scan(lf.p, lr.p, ncells, st, tmp);
  int lrank = 0, lflag = 0;
  CPPE_HIP_CHECK(hipMemcpyAsync(&lrank, lr.p + ncells - 1, sizeof(int), hipMemcpyDeviceToHost, st));
  CPPE_HIP_CHECK(hipMemcpyAsync(&lflag, lf.p + ncells - 1, sizeof(int), hipMemcpyDeviceToHost, st));
  CPPE_HIP_CHECK(hipStreamSynchronize(st));
  T.nleaves = lrank + lflag;
  T.leaf_ids.alloc(T.nleaves);
  hipLaunchKernelGGL(k_scatter_ids, dim3(ceil_div(ncells, 256)), dim3(256), 0, st, ncells, lf.p, lr.p,
                     T.leaf_ids.p);
  T.leaf_of.alloc(n);
  hipLaunchKernelGGL(k_leaf_of, dim3(T.nleaves), dim3(n / T.nleaves > 256 ? 1024 : 64), 0, st, T.leaf_ids.p,
                     T.start.p, T.count.p, T.leaf_of.p);
  // host copies of the leaves' ranges, for the work items of the near-field kernels
  T.h_leaf_ids.resize(T.nleaves);
  T.h_start.resize(ncells);
  T.h_count.resize(ncells);
  auto down = [&](std::vector<int>& h, const dbuf<int>& d) {
    CPPE_HIP_CHECK(hipMemcpyAsync(h.data(), d.p, sizeof(int) * h.size(), hipMemcpyDeviceToHost, st));
  };
  down(T.h_leaf_ids, T.leaf_ids);
  down(T.h_start, T.start);
  down(T.h_count, T.count);
  CPPE_HIP_CHECK(hipStreamSynchronize(st));
  T.built = true;
}

// ---------------------------------------------------------------------------------------------
// Dual-tree traversal (fmm/calculate.cc:74-127), one generation of the frontier per launch. A
// generation reads its length from the counters, so the generations follow each other without the
// host: a pair splits one of its cells per generation, 2 max_level + 1 of them empty the frontier.
// A list that is full is reported in the generation's own word, and a generation looks only at the word of the one
// before it, which no launch still writes: every wavefront of a block takes the same way to the barriers. (A word that
// other blocks set meanwhile let some wavefronts of a block leave, the rest then counted LDS nobody had written.)
// Slots are taken once per block, list and kTravTile pairs (classify, block prefix sums, one atomic per
// list, classify again and write): atomics on one address complete one after another, and a slot per pair
// or per wavefront made the traversal the longest set-up kernel (0.84 ms at 120,000 sites, 7.6 ms at
// 300,000; now 0.16 ms and 0.57 ms).
// ---------------------------------------------------------------------------------------------
constexpr int kTravGen = 2 * kMaxLevel + 1;
enum TravCount { TC_M2L = 0, TC_P2P, TC_FRONT, TC_OVER = TC_FRONT + kTravGen + 1, TC_COUNT = TC_OVER + kTravGen + 1 };
struct TravOut {
  int2* next;
  unsigned long long* m2l;  // (target << 32) | source
  unsigned long long* p2p;  // (target << 32) | source
  // TravCount: list lengths; per generation the frontier's length, and whether a list was full before it
  unsigned long long* counters;
  long long cap_next, cap_m2l, cap_p2p;
};

struct TravCells {
  const double *cx, *cy, *cz, *rmax;
  const int *nchild, *child_first;
  double theta;
};

// One pair: 0 far (M2L), 1 near (P2P), 2 split the target, 3 split the source; k children of that cell from c0 on.
__device__ __forceinline__ int trav_kind(const TravCells& c, int A, int B, int& k, int& c0) {
#pragma clang fp contract(off)
  const double dx = c.cx[A] - c.cx[B];
  const double dy = c.cy[A] - c.cy[B];
  const double dz = c.cz[A] - c.cz[B];
  const double R  = sqrt(dx * dx + dy * dy + dz * dz);
  const int na = c.nchild[A], nb = c.nchild[B];
  k = c0 = 0;
  if (R * c.theta > (c.rmax[A] + c.rmax[B])) return 0;
  if (na == 0 && nb == 0) return 1;
  const bool sa = nb == 0 || (c.rmax[A] >= c.rmax[B] && na != 0);
  k  = sa ? na : nb;
  c0 = c.child_first[sa ? A : B];
  return sa ? 2 : 3;
}

constexpr int kTravPer = 8, kTravTile = 256 * kTravPer;
__global__ __launch_bounds__(256) void k_traverse(int gen, const int2* __restrict__ front, TravOut o, TravCells c) {
  __shared__ int part[3][4];
  __shared__ long long base[3];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (o.counters[TC_OVER + gen]) {  // (final since the last launch: uniform over the grid)
    if (blockIdx.x == 0 && tid == 0) o.counters[TC_OVER + gen + 1] = 1;
    return;
  }
  const long long nfront = o.counters[TC_FRONT + gen];  // (within the capacity, else the word above is set)
  for (long long t0 = (long long)blockIdx.x * kTravTile; t0 < nfront; t0 += (long long)gridDim.x * kTravTile) {
    // (thread tid takes the pairs t0 + tid + 256 q: coalesced reads; the lists are sorted afterwards)
    int num[3] = {0, 0, 0}, k, c0;
    for (int q = 0; q < kTravPer; ++q) {
      const long long t = t0 + 256 * q + tid;
      if (t >= nfront) break;
      const int2 p = front[t];
      const int kd = trav_kind(c, p.x, p.y, k, c0);
      num[0] += kd == 0;
      num[1] += kd == 1;
      num[2] += k;
    }
    long long at[3];
    __syncthreads();  // (the previous tile's reads of part and base are done)
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      const int incl = wave_scan_incl(num[l], lane);
      if (lane == 63) part[l][wv] = incl;
      at[l] = incl - num[l];
    }
    __syncthreads();
    if (tid < 3) {
      const int total = part[tid][0] + part[tid][1] + part[tid][2] + part[tid][3];
      unsigned long long* counter = &o.counters[tid == 0 ? TC_M2L : tid == 1 ? TC_P2P : TC_FRONT + gen + 1];
      base[tid] = total ? (long long)atomicAdd(counter, (unsigned long long)total) : 0;
    }
    __syncthreads();
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      at[l] += base[l];
      for (int w = 0; w < wv; ++w) at[l] += part[l][w];
    }
    const long long cap[3] = {o.cap_m2l, o.cap_p2p, o.cap_next};
#pragma unroll
    for (int l = 0; l < 3; ++l)
      if (num[l] && at[l] + num[l] > cap[l]) {
        atomicExch(&o.counters[TC_OVER + gen + 1], 1ull);
        num[0] = num[1] = num[2] = -1;
      }
    if (num[0] < 0) continue;  // (no barrier before the next tile's first)
    for (int q = 0; q < kTravPer; ++q) {
      const long long t = t0 + 256 * q + tid;
      if (t >= nfront) break;
      const int2 p                  = front[t];
      const int kd                  = trav_kind(c, p.x, p.y, k, c0);
      const unsigned long long pair = ((unsigned long long)p.x << 32) | (unsigned)p.y;
      if (kd == 0)
        o.m2l[at[0]++] = pair;
      else if (kd == 1)
        o.p2p[at[1]++] = pair;
      else
        for (int i = 0; i < k; ++i) o.next[at[2]++] = kd == 2 ? make_int2(c0 + i, p.y) : make_int2(p.x, c0 + i);
    }
  }
}

// CSR offsets of target-sorted pair keys: off[c] = first entry with target >= c
__global__ void k_csr_offsets(int ncells, long long npairs, const unsigned long long* __restrict__ keys,
                              int* __restrict__ off) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c > ncells) return;
  unsigned long long v = (unsigned long long)c << 32;
  long long lo = 0, hi = npairs;
  while (lo < hi) {
    long long mid = (lo + hi) >> 1;
    if (keys[mid] < v)
      lo = mid + 1;
    else
      hi = mid;
  }
  off[c] = (int)lo;
}

__global__ void k_low_words(long long n, const unsigned long long* __restrict__ keys, int* __restrict__ out) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (int)(keys[i] & 0xffffffffull);
}

__global__ __launch_bounds__(256) void k_pair_sites(long long n, const unsigned long long* __restrict__ keys,
                                                    const int* __restrict__ count,
                                                    unsigned long long* __restrict__ acc) {
  __shared__ unsigned long long red[4];
  unsigned long long v = 0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const int A = (int)(keys[i] >> 32), B = (int)(keys[i] & 0xffffffffull);
    v += (unsigned long long)count[A] * (unsigned long long)count[B];
  }
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(acc, red[0] + red[1] + red[2] + red[3]);
}

static void sort_keys(dbuf<unsigned long long>& keys, long long n, int ncells, hipStream_t st,
                      dbuf<char>& tmp) {
  if (n == 0) return;
  dbuf<unsigned long long> out;
  out.alloc(n);
  int bits = 32;
  while ((1ll << (bits - 32)) <= ncells && bits < 64) ++bits;
  size_t bytes = 0;
  CPPE_HIP_CHECK(hipcub::DeviceRadixSort::SortKeys(nullptr, bytes, keys.p, out.p, (int)n, 0, bits, st));
  tmp.alloc(bytes + 16);
  CPPE_HIP_CHECK(hipcub::DeviceRadixSort::SortKeys(tmp.p, bytes, keys.p, out.p, (int)n, 0, bits, st));
  CPPE_HIP_CHECK(hipStreamSynchronize(st));
  keys.swap(out);
}

// Expanded near lists (one entry per near source site of each target leaf) for the slotted
// near-field kernel.
__global__ void k_xcount(int ncells, const int* __restrict__ off, const int* __restrict__ src,
                         const int* __restrict__ count, long long* __restrict__ xcnt) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncells) return;
  long long t = 0;
  for (int k = off[c]; k < off[c + 1]; ++k) t += count[src[k]];
  xcnt[c] = t;
}

// Entry of leaf A in the near list of leaf B (sorted by source leaf); without one, where it would stand.
__device__ __forceinline__ int near_entry(const int* __restrict__ off, const int* __restrict__ src, int B, int A) {
  int lo = off[B], hi = off[B + 1];
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (src[mid] < A)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// Whether site e is among the exclusion partners eidx[eoff[i] ..] of site i.
__device__ __forceinline__ bool lists_partner(const int* __restrict__ eoff, const int* __restrict__ eidx, int i, int e) {
  for (int k = eoff[i]; k < eoff[i + 1]; ++k)
    if (eidx[k] == e) return true;
  return false;
}

// Skip lists: per site the partners a near field leaves out, from either side's exclusions. A site's exclusions
// count for the field at that site alone (fmm/calculate.cc:205-225); a partner that only lists the site from its
// own side is marked kSkipKeep: the field at the site keeps that pair. Thread per site, cur[e] the entries
// of site e so far: with ent null they are counted. one_way is set when a partner is marked.
__global__ __launch_bounds__(256) void k_pair_skips(int n, const int* __restrict__ eoff, const int* __restrict__ eidx,
                                                    int* __restrict__ cur, unsigned* __restrict__ ent,
                                                    int* __restrict__ one_way) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int k = eoff[i]; k < eoff[i + 1]; ++k) {
    const int e = eidx[k];
    if (e < 0 || e == i) continue;
    bool again = false;
    for (int q = eoff[i]; q < k; ++q) again = again || eidx[q] == e;
    if (again) continue;
    const int at = atomicAdd(&cur[i], 1);
    if (ent) ent[at] = (unsigned)e;
    if (lists_partner(eoff, eidx, e, i)) continue;
    *one_way     = 1;
    const int to = atomicAdd(&cur[e], 1);
    if (ent) ent[to] = (unsigned)i | kSkipKeep;
  }
}

void build_pair_skips(System& S) {
  PairSkips& K = S.skips;
  if (K.built || !S.excl_off.p) return;
  hipStream_t st = S.stream;
  const dim3 g(ceil_div(S.n, 256)), b(256);
  dbuf<int> cur, flag;
  cur.alloc((size_t)S.n + 1);
  flag.alloc(1);
  CPPE_HIP_CHECK(hipMemsetAsync(cur.p, 0, sizeof(int) * ((size_t)S.n + 1), st));
  CPPE_HIP_CHECK(hipMemsetAsync(flag.p, 0, sizeof(int), st));
  K.off.alloc((size_t)S.n + 1);
  hipLaunchKernelGGL(k_pair_skips, g, b, 0, st, S.n, S.excl_off.p, S.excl_idx.p, cur.p, nullptr, flag.p);
  int one_way = 0, total = 0;
  CPPE_HIP_CHECK(hipMemcpyAsync(&one_way, flag.p, sizeof(int), hipMemcpyDeviceToHost, st));
  device_scan(S, cur.p, K.off.p, S.n + 1);
  CPPE_HIP_CHECK(hipMemcpyAsync(&total, K.off.p + S.n, sizeof(int), hipMemcpyDeviceToHost, st));
  CPPE_HIP_CHECK(hipMemcpyAsync(cur.p, K.off.p, sizeof(int) * (size_t)S.n, hipMemcpyDeviceToDevice, st));
  CPPE_HIP_CHECK(hipStreamSynchronize(st));
  K.ent.alloc((size_t)std::max(total, 1));
  hipLaunchKernelGGL(k_pair_skips, g, b, 0, st, S.n, S.excl_off.p, S.excl_idx.p, cur.p, K.ent.p, flag.p);
  CPPE_HIP_CHECK(hipStreamSynchronize(st));  // before the scratch is released
  K.one_way = one_way != 0;
  K.built   = true;
}

// Every entry of a cell's expanded near list in near-list order, one block per cell: the source site with
// its class in the top bits. XC_OWN: the leaf's own sites. XC_PARTNER: sites of other leaves that the skip list of an
// own site names. The others by the smallest Thole argument v = damping s_i s_j R_ij
// over the leaf's own sites i (exact, FP64): XC_NEAR: v < 18, XC_MID: 18 <= v < 25, XC_WIDE: 25 <= v < 40,
// XC_FAR: v >= 40 (a small margin above each bound). Undamped sites (s = 0) are XC_NEAR without the search, so are one-leaf
// (direct-summation) systems, all of whose sites are own, and cost O(n) here. The near
// leaves are taken 256 at a time (prefix sums of their sizes in LDS), the entries 64 at a time by the
// block's wavefronts, with the leaf's sites in LDS; a wavefront leaves the search once all its entries
// are of class XC_NEAR. The ends of the classes (totals over the cell) go to ends.
enum XClass : unsigned { XC_OWN = 0, XC_PARTNER, XC_NEAR, XC_MID, XC_WIDE, XC_FAR, XC_COUNT };
constexpr int kXclsShift = 29;
constexpr unsigned kXclsSite = (1u << kXclsShift) - 1u;
// ends of the classes XC_OWN, XC_PARTNER, XC_NEAR, XC_MID and XC_WIDE in the ordered list
struct XEnds {
  long long *own, *spec, *s32, *mid, *s64;
};
__global__ __launch_bounds__(256) void k_xclass(const int* __restrict__ off, const int* __restrict__ src,
                                                const int* __restrict__ start, const int* __restrict__ count,
                                                const int* __restrict__ leaf_of, const double* __restrict__ x,
                                                const double* __restrict__ y, const double* __restrict__ z,
                                                const double* __restrict__ s, double damping, SkipLists sk,
                                                const long long* __restrict__ xoff, unsigned* __restrict__ ent,
                                                XEnds ends) {
  __shared__ double4 own[256];
  __shared__ int pre[256], st[256], part[4], num[XC_COUNT];
  const int c = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int o0 = off[c], o1 = off[c + 1];
  if (o0 == o1) {
    if (tid == 0) ends.own[c] = ends.spec[c] = ends.s32[c] = ends.mid[c] = ends.s64[c] = xoff[c];
    return;
  }
  const int i0 = start[c], ni = count[c];
  if (damping > 0.0 && tid < ni) own[tid] = make_double4(x[i0 + tid], y[i0 + tid], z[i0 + tid], s[i0 + tid] * s[i0 + tid]);
  if (tid < XC_COUNT) num[tid] = 0;
  long long pos = xoff[c];
  for (int g0 = o0; g0 < o1; g0 += 256) {
    const int gn  = min(256, o1 - g0);
    const int B   = tid < gn ? src[g0 + tid] : -1;
    const int nb  = B >= 0 ? count[B] : 0;
    int incl      = wave_scan_incl(nb, lane);
    __syncthreads();
    if (lane == 63) part[wv] = incl;
    __syncthreads();
    for (int w = 0; w < wv; ++w) incl += part[w];
    pre[tid] = incl - nb;
    st[tid]  = B >= 0 ? start[B] : 0;
    const int total = part[0] + part[1] + part[2] + part[3];
    __syncthreads();
    for (int q0 = 64 * wv; q0 < total; q0 += 256) {
      const int q = q0 + lane;
      int j = 0;
      unsigned cl = XC_COUNT;
      if (q < total) {
        int lo = 0, hi = gn;  // last leaf whose first entry is at or before q
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (pre[mid] <= q)
            lo = mid;
          else
            hi = mid;
        }
        j  = st[lo] + (q - pre[lo]);
        cl = j >= i0 && j < i0 + ni ? XC_OWN : XC_NEAR;
      }
      const double sj = cl == XC_NEAR && damping > 0.0 ? s[j] : 0.0;
      double m        = 1e300;
      if (sj > 0.0) {
        const double xj = x[j], yj = y[j], zj = z[j];
        const double m18 = kFarClass32 * (1.0 + 1e-9) / (damping * sj), stop = 0.999 * m18 * m18;
        for (int i = 0; i < ni; ++i) {
          const double4 p = i < 256 ? own[i] : make_double4(x[i0 + i], y[i0 + i], z[i0 + i], s[i0 + i] * s[i0 + i]);
          const double dx = xj - p.x, dy = yj - p.y, dz = zj - p.z;
          m = fmin(m, p.w * (dx * dx + dy * dy + dz * dz));
          if ((i & 7) == 7 && __all(m < stop)) break;  // (of the lanes still searching)
        }
        const double v = damping * sj * sqrt(m);
        cl = v < kFarClass32 * (1.0 + 1e-9)      ? XC_NEAR
             : v < kTholeCutoff32 * (1.0 + 1e-9) ? XC_MID
             : v < kTholeCutoff * (1.0 + 1e-9)   ? XC_WIDE
                                                 : XC_FAR;
      }
      if (q < total) ent[pos + q] = (unsigned)j | (cl << kXclsShift);
#pragma unroll
      for (unsigned k : {XC_OWN, XC_NEAR, XC_MID, XC_WIDE}) {
        const int n = __popcll(__ballot(cl == k));
        if (lane == 0 && n) atomicAdd(&num[k], n);
      }
    }
    if (sk.off) {  // partners among this group's leaves (each entry moves to XC_PARTNER once)
      __threadfence();
      __syncthreads();
      for (int i = i0 + tid; i < i0 + ni; i += 256)
        for (int k = sk.off[i]; k < sk.off[i + 1]; ++k) {
          const int e = (int)(sk.ent[k] & kSkipSite);
          if (e >= i0 && e < i0 + ni) continue;
          const int L = near_entry(off, src, c, leaf_of[e]) - g0;
          if (L < 0 || L >= gn || src[g0 + L] != leaf_of[e]) continue;  // in another group, or not near
          const unsigned was =
              atomicMin(&ent[pos + pre[L] + (e - st[L])], (unsigned)e | ((unsigned)XC_PARTNER << kXclsShift));
          if (was >> kXclsShift == XC_PARTNER) continue;
          atomicAdd(&num[XC_PARTNER], 1);
          atomicAdd(&num[was >> kXclsShift], -1);
        }
    }
    pos += total;
  }
  __syncthreads();
  if (tid == 0) {
    long long e  = xoff[c];
    ends.own[c]  = e += num[XC_OWN];  // (a theta far above 1 can make a leaf far from itself: none)
    ends.spec[c] = e += num[XC_PARTNER];
    ends.s32[c]  = e += num[XC_NEAR];
    ends.mid[c]  = e += num[XC_MID];
    ends.s64[c]  = e + num[XC_WIDE];
  }
}

// One wavefront per cell: its entries written class by class, each class in near-list order (one pass,
// compaction with a ballot per class and 64 entries).
__global__ __launch_bounds__(256) void k_xfill(int ncells, const unsigned* __restrict__ ent,
                                               const long long* __restrict__ xoff, XEnds ends, int* __restrict__ xsrc) {
  const int c = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (c >= ncells) return;
  const unsigned long long below = (1ull << lane) - 1ull;
  const long long e0 = xoff[c], e1 = xoff[c + 1];
  long long pos[XC_COUNT] = {e0, ends.own[c], ends.spec[c], ends.s32[c], ends.mid[c], ends.s64[c]};
  for (long long e = e0; e < e1; e += 64) {
    const unsigned v = e + lane < e1 ? ent[e + lane] : 0xffffffffu;
    const unsigned k = v >> kXclsShift;
#pragma unroll
    for (unsigned cl = 0; cl < XC_COUNT; ++cl) {
      const unsigned long long m = __ballot(k == cl);
      if (k == cl) xsrc[pos[cl] + __popcll(m & below)] = (int)(v & kXclsSite);
      pos[cl] += __popcll(m);
    }
  }
}

void build_near_expanded(System& S) {
  Octree& T = S.tree;
  if (T.nx >= 0) return;
  hipStream_t st = S.stream;
  const int nc   = T.ncells;
  dbuf<long long> cnt;
  cnt.alloc(nc + 1);
  hipLaunchKernelGGL(k_xcount, dim3(ceil_div(nc, 256)), dim3(256), 0, st, nc, T.p2p_off.p, T.p2p_src.p, T.count.p,
                     cnt.p);
  long long zero = 0;
  CPPE_HIP_CHECK(hipMemcpyAsync(cnt.p + nc, &zero, sizeof(long long), hipMemcpyHostToDevice, st));
  T.xoff.alloc(nc + 1);
  dbuf<char> tmp;
  exclusive_scan(cnt.p, T.xoff.p, nc + 1, st, tmp);
  long long total = 0;
  CPPE_HIP_CHECK(hipMemcpyAsync(&total, T.xoff.p + nc, sizeof(long long), hipMemcpyDeviceToHost, st));
  CPPE_HIP_CHECK(hipStreamSynchronize(st));
  T.xsrc.alloc(std::max<long long>(total, 1));
  T.xspec.alloc(nc);
  T.xsplit[0].alloc(nc);
  T.xsplit[1].alloc(nc);
  T.xsplit[2].alloc(nc);
  build_pair_skips(S);
  dbuf<long long> xown;
  xown.alloc(nc);
  const XEnds ends{xown.p, T.xspec.p, T.xsplit[1].p, T.xsplit[2].p, T.xsplit[0].p};
  // (site indices below 2^29: a system of more sites has no room for its lists on the device)
  dbuf<unsigned> ent;
  ent.alloc(std::max<long long>(total, 1));
  hipLaunchKernelGGL(k_xclass, dim3(nc), dim3(256), 0, st, T.p2p_off.p, T.p2p_src.p, T.start.p, T.count.p, T.leaf_of.p,
                     S.x.p, S.y.p, S.z.p, S.s.p, S.s.p ? S.opts.damping : 0.0, S.skips.lists(), T.xoff.p, ent.p, ends);
  hipLaunchKernelGGL(k_xfill, dim3(ceil_div(nc, 4)), dim3(256), 0, st, nc, ent.p, T.xoff.p, ends, T.xsrc.p);
  CPPE_HIP_CHECK(hipStreamSynchronize(st));
  T.nx    = total;
  T.xdamp = S.opts.damping;
}

// ---- lists of the symmetric near field (near_sym.hh) -------------------------------------------
// One wavefront per cell, lanes over its near list: *one_sided set if a leaf near it does not have it as near
// leaf, or if it is a leaf that is not near itself.
__global__ __launch_bounds__(256) void k_near_one_sided(int ncells, const int* __restrict__ nchild,
                                                        const int* __restrict__ off, const int* __restrict__ src,
                                                        int* __restrict__ one_sided) {
  const int A = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (A >= ncells) return;
  if (nchild[A] == 0) {
    const int e = near_entry(off, src, A, A);
    if (e == off[A + 1] || src[e] != A) *one_sided = 1;
  }
  for (int k = off[A] + (threadIdx.x & 63); k < off[A + 1]; k += 64) {
    const int B = src[k], e = near_entry(off, src, B, A);
    if (e == off[B + 1] || src[e] != A) *one_sided = 1;
  }
}

// Whether B near A always comes with A near B, and every leaf is near itself. The walk splits the target first in a pair of equal cells, so at a
// theta where a cell touches the acceptance bound it may take a pair as far from one side only (at theta = 1
// 69 of the 84,595 near pairs of 60,000 sites).
bool near_lists_symmetric(System& S) {
  Octree& T = S.tree;
  if (T.near_symmetric < 0) {
    dbuf<int> one_sided;
    one_sided.alloc(1);
    int h = 0;
    CPPE_HIP_CHECK(hipMemcpyAsync(one_sided.p, &h, sizeof(int), hipMemcpyHostToDevice, S.stream));
    hipLaunchKernelGGL(k_near_one_sided, dim3(ceil_div(T.ncells, 4)), dim3(256), 0, S.stream, T.ncells, T.nchild.p,
                       T.p2p_off.p, T.p2p_src.p, one_sided.p);
    CPPE_HIP_CHECK(hipMemcpyAsync(&h, one_sided.p, sizeof(int), hipMemcpyDeviceToHost, S.stream));
    CPPE_HIP_CHECK(hipStreamSynchronize(S.stream));
    T.near_symmetric = h == 0;
  }
  return T.near_symmetric != 0;
}

// One wavefront per cell B (cell ncells: the scans' last entry), lanes over its near list (sorted
// by source leaf): the number of chunks of the leaves A < B before each entry (block index of A's
// first chunk among B's incoming reverse blocks) and in total; the upper-list length (own sites +
// sites of near leaves above B) and the reverse slots B receives (incoming blocks x 3 |B|).
__global__ __launch_bounds__(256) void k_sym_sizes(int ncells, const int* __restrict__ off,
                                                   const int* __restrict__ src, const int* __restrict__ count,
                                                   const int* __restrict__ nq, int* __restrict__ pre,
                                                   int* __restrict__ nin, long long* __restrict__ ucnt,
                                                   long long* __restrict__ rsz) {
  const int B = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (B > ncells) return;
  const int o0 = B < ncells ? off[B] : 0, o1 = B < ncells ? off[B + 1] : 0;
  int run = 0, up = 0;
  for (int k0 = o0; k0 < o1; k0 += 64) {
    const int k  = k0 + lane;
    const int A  = k < o1 ? src[k] : B;
    const int q  = A < B ? nq[A] : 0;
    const int in = wave_scan_incl(q, lane);
    if (k < o1) pre[k] = run + in - q;
    run += __shfl(in, 63);
    if (A > B) up += count[A];
  }
  for (int o = 32; o > 0; o >>= 1) up += __shfl_xor(up, o);
  if (lane == 0) {  // (cells without a near list: 0)
    const int nb = o1 > o0 ? count[B] : 0;
    ucnt[B]      = o1 > o0 ? (long long)nb + up : 0;
    rsz[B]       = (long long)run * 3 * nb;
    if (B < ncells) nin[B] = run;
  }
}

// Upper lists in near-list order, straight from the leaf lists (no classes: the FP64 pair decides
// its damping per stage): one wavefront per leaf A. 64 near leaves at a time, a lane per leaf finds
// the reverse slot of A's block in its receiver; then the lanes expand the leaves above A into
// their sites, 64 entries at a time.
__global__ __launch_bounds__(64) void k_sym_fill_leaf(const int* __restrict__ start, const int* __restrict__ count,
                                                      const int* __restrict__ p2p_off,
                                                      const int* __restrict__ p2p_src, const int* __restrict__ pre,
                                                      const long long* __restrict__ rev_off,
                                                      const long long* __restrict__ uoff, int* __restrict__ usrc,
                                                      int2* __restrict__ udst) {
  __shared__ int s_pre[64], s_j0[64], s_slot[64], s_nb[64];
  const int A = blockIdx.x, lane = threadIdx.x;
  const long long u0 = uoff[A];
  if (uoff[A + 1] == u0) return;
  const int na = count[A];
  for (int u = lane; u < na; u += 64) {
    usrc[u0 + u] = start[A] + u;
    udst[u0 + u] = make_int2(0, 0);
  }
  long long pos = u0 + na;
  const int o0 = p2p_off[A], o1 = p2p_off[A + 1];
  for (int k0 = o0; k0 < o1; k0 += 64) {
    const int B  = k0 + lane < o1 ? p2p_src[k0 + lane] : 0;
    const int nb = B > A ? count[B] : 0;
    int slot     = 0;
    if (nb) {
      slot = (int)(rev_off[B] + (long long)pre[near_entry(p2p_off, p2p_src, B, A)] * 3 * nb);
    }
    const int incl  = wave_scan_incl(nb, lane);
    const int total = __shfl(incl, 63);
    __syncthreads();
    s_pre[lane]  = incl - nb;
    s_j0[lane]   = nb ? start[B] : 0;
    s_slot[lane] = slot;
    s_nb[lane]   = nb;
    __syncthreads();
    for (int q = lane; q < total; q += 64) {
      int lo = 0, hi = 64;  // last leaf whose first entry is at or before q
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (s_pre[mid] <= q)
          lo = mid;
        else
          hi = mid;
      }
      const int u   = q - s_pre[lo];
      usrc[pos + q] = s_j0[lo] + u;
      udst[pos + q] = make_int2(s_slot[lo] + u, s_nb[lo]);
    }
    pos += total;
  }
}

// One wavefront per leaf A: its own sites, then the entries of its expanded near list whose leaf
// is above A (order kept, compaction by ballot), each with its reverse slot; usplit: position of
// the first kept entry at or after the FP32 far split of the expanded list.
__global__ __launch_bounds__(64) void k_sym_fill(const long long* __restrict__ xoff, const int* __restrict__ xsrc,
                                                 const long long* __restrict__ xs32, const int* __restrict__ leaf_of,
                                                 const int* __restrict__ start, const int* __restrict__ count,
                                                 const int* __restrict__ p2p_off, const int* __restrict__ p2p_src,
                                                 const int* __restrict__ pre, const long long* __restrict__ rev_off,
                                                 const long long* __restrict__ uoff, int* __restrict__ usrc,
                                                 int2* __restrict__ udst, long long* __restrict__ usplit) {
  const int A = blockIdx.x, lane = threadIdx.x;
  const long long u0 = uoff[A], u1 = uoff[A + 1];
  if (u1 == u0) {
    if (lane == 0) usplit[A] = u1;
    return;
  }
  const int na = count[A];
  for (int u = lane; u < na; u += 64) {
    usrc[u0 + u] = start[A] + u;
    udst[u0 + u] = make_int2(0, 0);
  }
  long long pos   = u0 + na;
  const long long x0 = xoff[A], x1 = xoff[A + 1];
  const long long split = xs32 ? xs32[A] : x1;
  long long usp   = -1;
  for (long long e0 = x0; e0 < x1; e0 += 64) {
    const long long e = e0 + lane;
    const bool valid  = e < x1;
    const int j       = valid ? xsrc[e] : 0;
    const int B       = valid ? leaf_of[j] : -1;
    const bool keep   = valid && B > A;
    const unsigned long long m = __ballot(keep);
    if (usp < 0 && split < e0 + 64) usp = pos + __popcll(__ballot(keep && e < split));
    if (keep) {
      const long long idx = pos + __popcll(m & ((1ull << lane) - 1ull));
      const int k         = near_entry(p2p_off, p2p_src, B, A);
      const long long slot = rev_off[B] + (long long)pre[k] * 3 * count[B] + (j - start[B]);
      usrc[idx] = j;
      udst[idx] = make_int2((int)slot, count[B]);
    }
    pos += __popcll(m);
  }
  if (usp < 0) usp = pos;
  if (lane == 0) usplit[A] = usp;
}

SymLists& build_sym_lists(System& S, int prec, int ts) {
  Octree& T    = S.tree;
  SymLists& Y  = T.sym[prec][sym_slot(ts)];
  if (Y.ts == ts) return Y;
  if (!near_lists_symmetric(S))
    throw hip_error("symmetric near field: the near lists of this tree are not symmetric");
  const bool classed = prec == 1;  // FP32: entries in the class order of the expanded near list
  if (classed) build_near_expanded(S);
  hipStream_t st = S.stream;
  const int nc   = T.ncells;
  std::vector<int> nq(nc, 0);
  const std::vector<int>&ids = T.h_leaf_ids, &cnt = T.h_count;
  std::vector<int4> items;
  items.reserve(T.nleaves + T.nleaves / 4);
  for (int c : ids) {
    nq[c] = (cnt[c] + ts - 1) / ts;
    for (int q = 0; q < nq[c]; ++q) items.push_back(make_int4(c, q * ts, std::min(ts, cnt[c] - q * ts), q));
  }
  dbuf<int> d_nq, pre;
  d_nq.alloc(nc);
  pre.alloc(std::max<long long>(T.n_p2p, 1));
  Y.nin.alloc(nc);
  CPPE_HIP_CHECK(hipMemcpyAsync(d_nq.p, nq.data(), sizeof(int) * nc, hipMemcpyHostToDevice, st));
  dbuf<long long> ucnt, rsz;
  ucnt.alloc(nc + 1);
  rsz.alloc(nc + 1);
  hipLaunchKernelGGL(k_sym_sizes, dim3(ceil_div(nc + 1, 4)), dim3(256), 0, st, nc, T.p2p_off.p, T.p2p_src.p, T.count.p,
                     d_nq.p, pre.p, Y.nin.p, ucnt.p, rsz.p);
  Y.uoff.alloc(nc + 1);
  Y.rev_off.alloc(nc + 1);
  dbuf<char> tmp;
  exclusive_scan(ucnt.p, Y.uoff.p, nc + 1, st, tmp);
  exclusive_scan(rsz.p, Y.rev_off.p, nc + 1, st, tmp);
  long long tot[2] = {0, 0};
  CPPE_HIP_CHECK(hipMemcpyAsync(&tot[0], Y.uoff.p + nc, sizeof(long long), hipMemcpyDeviceToHost, st));
  CPPE_HIP_CHECK(hipMemcpyAsync(&tot[1], Y.rev_off.p + nc, sizeof(long long), hipMemcpyDeviceToHost, st));
  CPPE_HIP_CHECK(hipStreamSynchronize(st));
  if (tot[1] >= (1ll << 31) - 1)
    throw hip_error("symmetric near field: more reverse slots than a 32-bit index addresses");
  Y.usrc.alloc(std::max<long long>(tot[0], 1));
  Y.udst.alloc(std::max<long long>(tot[0], 1));
  if (classed) {
    Y.usplit.alloc(nc);
    const long long* xs = S.opts.damping >= T.xdamp ? T.xsplit[1].p : nullptr;
    hipLaunchKernelGGL(k_sym_fill, dim3(nc), dim3(64), 0, st, T.xoff.p, T.xsrc.p, xs, T.leaf_of.p, T.start.p,
                       T.count.p, T.p2p_off.p, T.p2p_src.p, pre.p, Y.rev_off.p, Y.uoff.p, Y.usrc.p, Y.udst.p,
                       Y.usplit.p);
  } else {
    hipLaunchKernelGGL(k_sym_fill_leaf, dim3(nc), dim3(64), 0, st, T.start.p, T.count.p, T.p2p_off.p, T.p2p_src.p,
                       pre.p, Y.rev_off.p, Y.uoff.p, Y.usrc.p, Y.udst.p);
  }
  Y.items.alloc(std::max<size_t>(items.size(), 1));
  CPPE_HIP_CHECK(hipMemcpyAsync(Y.items.p, items.data(), sizeof(int4) * items.size(), hipMemcpyHostToDevice, st));
  CPPE_HIP_CHECK(hipStreamSynchronize(st));
  Y.nitems = (int)items.size();
  Y.nrev   = tot[1];
  Y.ts     = ts;
  return Y;
}

void build_lists(System& S) {
  Octree& T      = S.tree;
  hipStream_t st = S.stream;
  const double theta = S.opts.theta;
  long long cap_m2l  = 512ll * T.ncells + 4096;
  long long cap_p2p  = 256ll * T.nleaves + 4096;
  long long cap_next = std::max<long long>(cap_m2l, T.level_offset[1]);
  dbuf<unsigned long long> counters;
  counters.alloc(TC_COUNT);
  for (int attempt = 0; attempt < 6; ++attempt) {
    dbuf<int2> fa, fb;
    dbuf<unsigned long long> m2l, p2p;
    fa.alloc(cap_next);
    fb.alloc(cap_next);
    m2l.alloc(cap_m2l);
    p2p.alloc(cap_p2p);
    // one traversal per snapshot, all started together from the (root, root) pairs
    const int nroots = T.level_offset[1];
    std::vector<int2> seed(nroots);
    for (int c = 0; c < nroots; ++c) seed[c] = make_int2(c, c);
    CPPE_HIP_CHECK(hipMemcpyAsync(fa.p, seed.data(), sizeof(int2) * nroots, hipMemcpyHostToDevice, st));
    unsigned long long h_cnt[TC_COUNT] = {};
    h_cnt[TC_FRONT]                    = nroots;
    CPPE_HIP_CHECK(hipMemcpyAsync(counters.p, h_cnt, sizeof(h_cnt), hipMemcpyHostToDevice, st));
    const dim3 grid(std::min(2048, ceil_div(cap_next, kTravTile)));
    const TravCells cells{T.cx.p, T.cy.p, T.cz.p, T.crmax.p, T.nchild.p, T.child_first.p, theta};
    const int ngen = 2 * T.max_level + 1;
    for (int g = 0; g < ngen; ++g) {
      TravOut o{g % 2 ? fa.p : fb.p, m2l.p, p2p.p, counters.p, cap_next, cap_m2l, cap_p2p};
      hipLaunchKernelGGL(k_traverse, grid, dim3(256), 0, st, g, g % 2 ? fb.p : fa.p, o, cells);
    }
    CPPE_HIP_CHECK(hipMemcpyAsync(h_cnt, counters.p, sizeof(h_cnt), hipMemcpyDeviceToHost, st));
    CPPE_HIP_CHECK(hipStreamSynchronize(st));
    const bool overflow = h_cnt[TC_OVER + ngen] != 0;
    if (!overflow && h_cnt[TC_FRONT + ngen] != 0) throw std::runtime_error("octree: the traversal did not end");
    if (overflow) {
      cap_m2l *= 2;
      cap_p2p *= 2;
      cap_next *= 2;
      continue;
    }
    T.n_m2l = (long long)h_cnt[TC_M2L];
    T.n_p2p = (long long)h_cnt[TC_P2P];
    if (T.n_m2l > INT_MAX || T.n_p2p > INT_MAX)
      throw std::runtime_error("octree: more interaction pairs than a 32-bit index addresses");
    dbuf<char> tmp;
    sort_keys(m2l, T.n_m2l, T.ncells, st, tmp);
    sort_keys(p2p, T.n_p2p, T.ncells, st, tmp);
    T.m2l_off.alloc(T.ncells + 1);
    T.p2p_off.alloc(T.ncells + 1);
    T.m2l_src.alloc(std::max<long long>(T.n_m2l, 1));
    T.p2p_src.alloc(std::max<long long>(T.n_p2p, 1));
    hipLaunchKernelGGL(k_csr_offsets, dim3(ceil_div(T.ncells + 1, 256)), dim3(256), 0, st, T.ncells, T.n_m2l,
                       m2l.p, T.m2l_off.p);
    hipLaunchKernelGGL(k_csr_offsets, dim3(ceil_div(T.ncells + 1, 256)), dim3(256), 0, st, T.ncells, T.n_p2p,
                       p2p.p, T.p2p_off.p);
    if (T.n_m2l)
      hipLaunchKernelGGL(k_low_words, dim3(ceil_div(T.n_m2l, 256)), dim3(256), 0, st, T.n_m2l, m2l.p,
                         T.m2l_src.p);
    if (T.n_p2p)
      hipLaunchKernelGGL(k_low_words, dim3(ceil_div(T.n_p2p, 256)), dim3(256), 0, st, T.n_p2p, p2p.p,
                         T.p2p_src.p);
    dbuf<unsigned long long> acc;
    acc.alloc(1);
    acc.zero(st);
    if (T.n_p2p)
      hipLaunchKernelGGL(k_pair_sites, dim3(std::min(1024, ceil_div(T.n_p2p, 256))), dim3(256), 0, st, T.n_p2p, p2p.p,
                         T.count.p, acc.p);
    unsigned long long h_acc = 0;
    CPPE_HIP_CHECK(hipMemcpyAsync(&h_acc, acc.p, sizeof(h_acc), hipMemcpyDeviceToHost, st));
    CPPE_HIP_CHECK(hipStreamSynchronize(st));
    T.p2p_site_pairs = (long long)h_acc;
    return;
  }
  throw std::runtime_error("octree: interaction lists exceed the traversal capacity");
}

}  // namespace cppe_dev
