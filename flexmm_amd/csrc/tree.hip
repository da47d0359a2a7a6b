// Adaptive quadtree of the reference (flexmm/tree.py), built on the device.
//
// Every point gets a 31-level Morton key from the reference's own FP64
// midpoint recurrence (tree.py:169-176, 301-304: xmid = xmin + w/2, children
// start at xmid - w/2 or xmid, class 2*(x > xmid) + (y > ymid), tree.py:32-34),
// so the classification of every point at every level is the reference's
// bit for bit.  After a segmented MSD radix sort by key, the tree is three sets
// of cells:
//   S_d   cells of depth d that are split (refinement: > ncut points,
//         tree.py:204; plus the minimal corner 2:1 balance, tree.py:529-541);
//   X_d   real leaves with a split same-level neighbour (tree.py:542-553,
//         385-397), which get four fake children;
//   P_d   = S_d u X_d, the nodes of depth d that have children.
// Level d+1 holds the children of P_d in Morton order.  The sets are one bitmap
// per depth in trees of up to kBmLevels levels and sorted code lists in deeper
// ones; colleagues, parents, point ranges and M2L partners are lookups in them.
#include "tree.h"
#include "point_key.h"

#include <cstring>

namespace fmm {

namespace {

constexpr int BS = 256;

__device__ __forceinline__ int clz64(uint64_t v) { return v ? __clzll((long long)v) : 64; }

__device__ __forceinline__ int64_t bsearch_u64(const uint64_t* __restrict__ a, int64_t n,
                                               uint64_t v) {
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    int64_t mid = (lo + hi) >> 1;
    uint64_t am = a[mid];
    if (am < v)
      lo = mid + 1;
    else
      hi = mid;
  }
  return (lo < n && a[lo] == v) ? lo : -1;
}

__device__ __forceinline__ int64_t lower_bound_u64(const uint64_t* __restrict__ a, int64_t n,
                                                   uint64_t v) {
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    int64_t mid = (lo + hi) >> 1;
    if (a[mid] < v)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// --- points ----------------------------------------------------------------
// Morton keys of the points and an interleaved copy of their coordinates
// (the gather into tree order then reads one 16-byte record per point).
// One block of 1024 threads per chunk of kSortChunk points (4 per thread,
// strided by the block size; every load is issued before the first key is
// formed).  The key
// comes from the scaled-coordinate form where it provably equals the
// reference's recurrence (point_key.h) and from the recurrence itself for the
// few points within rounding reach of a midpoint.  With fr (more points than
// the sort's threshold) the block also counts its keys' top 8 bits for the
// sort's first round, and keys / vals are the sort's spare buffers.
constexpr int KEY_BS = 1024;
constexpr int kKeyPer = kSortChunk / KEY_BS;
static_assert(kKeyLevels == kMaxDepth, "keys cover every depth");
__global__ __launch_bounds__(KEY_BS) void k_point_keys(const double* __restrict__ x,
                                                   const double* __restrict__ y, int n,
                                                   double xmin0, double ymin0, double w0,
                                                   KeyScale ks, uint64_t* __restrict__ keys,
                                                   uint32_t* __restrict__ vals,
                                                   double2* __restrict__ xy,
                                                   int* __restrict__ bad_blk,
                                                   int* __restrict__ cnt, int ncnt,
                                                   SortFirstRound fr, int with_hist) {
  static_assert(kKeyPer * KEY_BS == kSortChunk, "one chunk per block");
  __shared__ int hist[256];
  if (with_hist && threadIdx.x < 256) hist[threadIdx.x] = 0;
  const int i0 = blockIdx.x * kSortChunk + threadIdx.x;
  double px[kKeyPer], py[kKeyPer];
#pragma unroll
  for (int u = 0; u < kKeyPer; ++u) {
    const int i = i0 + u * KEY_BS;
    px[u] = i < n ? x[i] : 0.0;
    py[u] = i < n ? y[i] : 0.0;
  }
  if (with_hist) __syncthreads();
  bool bad = false;
#pragma unroll
  for (int u = 0; u < kKeyPer; ++u) {
    const int i = i0 + u * KEY_BS;
    if (i < n) {
      xy[i] = make_double2(px[u], py[u]);
      bad |= !(__builtin_isfinite(px[u]) && __builtin_isfinite(py[u]));
      bool ok;
      uint64_t key = point_key_fast(px[u], py[u], xmin0, ymin0, ks, &ok);
      if (!ok) key = point_key_recurrence(px[u], py[u], xmin0, ymin0, w0);
      keys[i] = key;
      vals[i] = (uint32_t)i;
      if (with_hist) atomicAdd(&hist[(int)(key >> 56)], 1);
    }
  }
  // every block writes its own flag (no zeroed counter to race with), and
  // block 0 zeroes the build's counters, which only later kernels touch
  const int any_bad = __syncthreads_or(bad);
  if (threadIdx.x == 0) bad_blk[blockIdx.x] = any_bad;
  if (blockIdx.x == 0)
    for (int j = threadIdx.x; j < ncnt; j += KEY_BS) cnt[j] = 0;
  if (with_hist) sort_first_round_block(fr, blockIdx.x, hist);
}

// --- refinement: split cells from the sorted keys ----------------------------
// Position i starts the cells of depths s(i)+1.. (s = common depth with key
// i-1); such a cell has more than ncut points iff key i+ncut is still inside
// it, i.e. depth <= c(i) (common depth with key i+ncut).
// The same kernel counts the split cells per depth (position i starts one at
// each depth d with s < d <= c) and the split positions: each wave writes its
// ballot counts to its own LDS row, the block adds the rows and adds them to
// row b mod kSplitRows of `rows` ([kSplitRows][kMaxLevels + 1], zeroed; the
// host adds the rows): a thousand blocks adding to one set of counters
// serialised on those addresses (10 us of a 15 us kernel at 1M points).
// (Having the last block add the rows costs every block an agent-scope fence,
// which writes back its L2: 8.4 -> 32 us.)  A complete tree needs nothing
// more from the split positions.
constexpr int kSplitRows = 64;
// It also gathers the points into tree order (sx, sy from the interleaved
// copy xy through perm: one 16-byte gather per point), its loads in flight
// with the keys'.
__global__ __launch_bounds__(1024) void k_split_pos(const uint64_t* __restrict__ keys, int n,
                                                    int ncut, int2* __restrict__ sc,
                                                    int* __restrict__ rows,
                                                    const uint32_t* __restrict__ perm,
                                                    const double2* __restrict__ xy,
                                                    double* __restrict__ sx,
                                                    double* __restrict__ sy) {
  __shared__ int lc[1024 / 64][kMaxLevels + 1];
  const int i = blockIdx.x * 1024 + threadIdx.x;
  int s = 0, c = -1;
  if (i < n) {
    // the three keys are loaded together (clamped indices): behind their
    // conditions each load waited for the one before
    const int ip = i > 0 ? i - 1 : 0;
    const int ic = (int)min((int64_t)i + ncut, (int64_t)n - 1);
    const double2 pt = xy[perm[i]];
    const uint64_t k = keys[i], kp = keys[ip], kc = keys[ic];
    sx[i] = pt.x;
    sy[i] = pt.y;
    s = (i == 0) ? -1 : min(clz64(k ^ kp) >> 1, kMaxDepth);
    c = ((int64_t)i + ncut < n) ? min(clz64(k ^ kc) >> 1, kMaxDepth - 1) : -1;
    sc[i] = make_int2(s, c);
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const unsigned long long fm = __ballot(s < c);
  if (fm) {   // wave-uniform: most waves hold no split position
    for (int d = 0; d < kMaxLevels; ++d) {
      const int cnt = (int)__popcll(__ballot(s < d && d <= c));
      if (lane == 0) lc[wv][d] = cnt;
    }
    if (lane == 0) lc[wv][kMaxLevels] = (int)__popcll(fm);
  } else if (lane <= kMaxLevels) {
    lc[wv][lane] = 0;
  }
  __syncthreads();
  if (threadIdx.x <= kMaxLevels) {
    int t = 0;
#pragma unroll
    for (int w = 0; w < 1024 / 64; ++w) t += lc[w][threadIdx.x];
    if (t != 0)
      atomicAdd(&rows[(blockIdx.x % kSplitRows) * (kMaxLevels + 1) + threadIdx.x], t);
  }
}

// The host's share of the split counts: per depth d <= kMaxLevels the sum of
// the kSplitRows rows, and the non-finite flag, into words 0 .. kMaxLevels + 1
// of the host mailbox.  With gate: *gate = whether they describe the complete
// tree of depth D (every cell of depths < D split, none deeper, all points
// finite), the test the host makes once it has the words.
__global__ __launch_bounds__(64) void k_split_counts(const int* __restrict__ rows,
                                                     const int* __restrict__ bad_blk, int nblk,
                                                     uint64_t* __restrict__ mbox, uint32_t seq,
                                                     int D, int* __restrict__ gate) {
  const int d = threadIdx.x;
  int sum = 0;
  if (d <= kMaxLevels)
    for (int r = 0; r < kSplitRows; ++r) sum += rows[r * (kMaxLevels + 1) + d];
  // the key kernel's per-block non-finite flags, or-ed over the wave
  int b = 0;
  for (int j = d; j < nblk; j += 64) b |= bad_blk[j];
  const int any_bad = __ballot(b != 0) != 0ull;
  if (d == kMaxLevels + 1) sum = any_bad;
  if (d <= kMaxLevels + 1) mailbox_put(mbox, d, seq, sum);
  if (gate) {
    bool ok = true;
    if (d < D) ok = sum == (1 << (2 * d));
    else if (d < kMaxLevels || d == kMaxLevels + 1) ok = sum == 0;
    const bool all = __ballot(!ok) == 0ull;
    if (d == 0) *gate = all ? 1 : 0;
  }
}

// 1 at the split positions (those that start a split cell), for the scan
__global__ __launch_bounds__(BS) void k_split_flags(const int2* __restrict__ sc, int n,
                                                    int* __restrict__ flag) {
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i < n) flag[i] = sc[i].x < sc[i].y;
}

__global__ __launch_bounds__(BS) void k_compact_pos(const int* __restrict__ flag,
                                                    const int* __restrict__ rank,
                                                    const int2* __restrict__ sc, int n,
                                                    int* __restrict__ ppos, int2* __restrict__ psc) {
  int i = blockIdx.x * BS + threadIdx.x;
  if (i >= n || !flag[i]) return;
  int r = rank[i];
  ppos[r] = i;
  psc[r] = sc[i];
}

__global__ __launch_bounds__(1024) void k_depth_lists(const int* __restrict__ ppos,
                                                     const int2* __restrict__ psc, int np,
                                                     const uint64_t* __restrict__ keys,
                                                     const int64_t* __restrict__ soff,
                                                     uint64_t* __restrict__ sref) {
  __shared__ int lds[1024 / 64];
  __shared__ int tot;
  const int d = blockIdx.x;
  uint64_t* out = sref + soff[d];
  int carry = 0;
  for (int base = 0; base < np; base += 1024) {
    int j = base + threadIdx.x;
    int pred = 0;
    uint64_t code = 0;
    if (j < np) {
      int2 v = psc[j];
      pred = (v.x < d) && (d <= v.y);
      if (pred && d > 0) code = keys[ppos[j]] >> (64 - 2 * d);
    }
    int ex = block_exclusive_scan<1024>(pred, lds, &tot);
    if (pred) out[carry + ex] = code;
    __syncthreads();
    carry += tot;
    __syncthreads();
  }
}

// --- 2:1 balance ---------------------------------------------------------------
// A leaf at depth d is split iff a same-level neighbour has a grandchild; the
// minimal balanced refinement is S_d = Sref_d u N(parents(S_{d+1})), with
// N the 3x3 neighbourhood.  This kernel counts neighbours missing from Sref,
// which is zero exactly when the refinement tree is already balanced.
__global__ __launch_bounds__(BS) void k_balance_check(const uint64_t* __restrict__ sref,
                                                      const int64_t* __restrict__ soff, int L,
                                                      int* __restrict__ rcount) {
  int64_t e = soff[2] + (int64_t)blockIdx.x * BS + threadIdx.x;
  if (e >= soff[L - 1]) return;
  int D = 2;
  while (e >= soff[D + 1]) ++D;
  uint64_t s = sref[e];
  if (e > soff[D] && (sref[e - 1] >> 2) == (s >> 2)) return;
  const int d = D - 1;
  uint64_t pc = s >> 2;
  uint32_t ix, iy;
  demorton(pc, &ix, &iy);
  const int64_t lim = (int64_t)1 << d;
  const uint64_t* lst = sref + soff[d];
  const int64_t nl = soff[d + 1] - soff[d];
  int miss = 0;
  for (int k = 0; k < 9; ++k) {
    int64_t nx = (int64_t)ix + k / 3 - 1, ny = (int64_t)iy + k % 3 - 1;
    if (nx < 0 || ny < 0 || nx >= lim || ny >= lim) continue;
    if (bsearch_u64(lst, nl, morton((uint32_t)nx, (uint32_t)ny)) < 0) ++miss;
  }
  if (miss) atomicAdd(rcount, miss);
}

__global__ __launch_bounds__(BS) void k_bal_candidates(const uint64_t* __restrict__ sref_d,
                                                       int64_t nref,
                                                       const uint64_t* __restrict__ s_next,
                                                       int64_t nnext, int d,
                                                       uint64_t* __restrict__ cand,
                                                       uint32_t* __restrict__ vals) {
  int64_t i = (int64_t)blockIdx.x * BS + threadIdx.x;
  const int sh = 64 - 2 * d;
  if (i < nref) {
    cand[i] = sref_d[i] << sh;
    vals[i] = 0;
    return;
  }
  int64_t j = i - nref;
  if (j >= 9 * nnext) return;
  int64_t e = j / 9;
  int k = (int)(j % 9);
  uint64_t s = s_next[e];
  uint64_t out = ~0ull;
  if (e == 0 || (s_next[e - 1] >> 2) != (s >> 2)) {
    uint32_t ix, iy;
    demorton(s >> 2, &ix, &iy);
    int64_t lim = (int64_t)1 << d;
    int64_t nx = (int64_t)ix + k / 3 - 1, ny = (int64_t)iy + k % 3 - 1;
    if (nx >= 0 && ny >= 0 && nx < lim && ny < lim) out = morton((uint32_t)nx, (uint32_t)ny) << sh;
  }
  cand[i] = out;
  vals[i] = 0;
}

__global__ __launch_bounds__(BS) void k_unique_flags(const uint64_t* __restrict__ cand, int64_t n,
                                                     int* __restrict__ flag) {
  int64_t i = (int64_t)blockIdx.x * BS + threadIdx.x;
  if (i >= n) return;
  uint64_t c = cand[i];
  flag[i] = (c != ~0ull) && (i == 0 || cand[i - 1] != c);
}

__global__ __launch_bounds__(BS) void k_unique_scatter(const uint64_t* __restrict__ cand,
                                                       const int* __restrict__ flag,
                                                       const int* __restrict__ rank, int64_t n,
                                                       int d, uint64_t* __restrict__ out) {
  int64_t i = (int64_t)blockIdx.x * BS + threadIdx.x;
  if (i >= n || !flag[i]) return;
  out[rank[i]] = cand[i] >> (64 - 2 * d);
}

// Balance on bitmaps: bit c of depth d's bitmap is cell c (the depth-d Morton
// code); each depth's words start at a multiple of BS, so a block of BS words
// lies in one depth.  Marking is an idempotent OR, so the union needs neither
// sort nor unique, and the bitmap order is the code order.
constexpr int kBmDepth = 13;   // 4^13 bits = 8 MB at the deepest bitmap depth
struct BmOffsets {
  int64_t wo[kMaxLevels + 1];  // first word of depth d (depths 1 .. dmax)
};
__device__ __forceinline__ int bm_depth(const BmOffsets& o, int dmax, int64_t w) {
  int d = 1;
  while (d < dmax && w >= o.wo[d + 1]) ++d;
  return d;
}
__device__ __forceinline__ void bm_set(uint32_t* bm, uint64_t c) {
  atomicOr(bm + (c >> 5), 1u << (c & 31));
}
// the 3x3 neighbourhood (clipped to the domain) of parent cell pc at depth d;
// bits that fall in one word go out in one atomic (a neighbourhood spans at
// most four words)
__device__ __forceinline__ void bm_mark_nbrs(uint32_t* bm, uint64_t pc, int d) {
  uint32_t ix, iy;
  demorton(pc, &ix, &iy);
  const int64_t lim = (int64_t)1 << d;
  uint64_t wd[9];
  uint32_t bit[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const int64_t nx = (int64_t)ix + k / 3 - 1, ny = (int64_t)iy + k % 3 - 1;
    const bool in = nx >= 0 && ny >= 0 && nx < lim && ny < lim;
    const uint64_t c = in ? morton((uint32_t)nx, (uint32_t)ny) : 0;
    wd[k] = c >> 5;
    bit[k] = in ? 1u << (c & 31) : 0u;
  }
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    bool first = true;
#pragma unroll
    for (int j = 0; j < k; ++j) first = first && !(bit[j] && wd[j] == wd[k]);
    if (!first || !bit[k]) continue;
    uint32_t m = bit[k];
#pragma unroll
    for (int j = k + 1; j < 9; ++j) m |= wd[j] == wd[k] ? bit[j] : 0u;
    atomicOr(bm + wd[k], m);
  }
}
// Sref_d for depths 1 .. dmax into their bitmaps
__global__ __launch_bounds__(BS) void k_bm_mark(const uint64_t* __restrict__ sref,
                                                const int64_t* __restrict__ soff, int dmax,
                                                BmOffsets o, uint32_t* __restrict__ bm) {
  const int64_t e = soff[1] + (int64_t)blockIdx.x * BS + threadIdx.x;
  if (e >= soff[dmax + 1]) return;
  int d = 1;
  while (e >= soff[d + 1]) ++d;
  bm_set(bm + o.wo[d], sref[e]);
}
// N(parents) of the depth-(d+1) cells in bitmap bm1 into depth d's bitmap bm0,
// one thread per depth-d parent cell pc: its 4 children are bits
// 4(pc mod 8) .. +3 of word pc / 8
__global__ __launch_bounds__(BS) void k_bm_spread(const uint32_t* __restrict__ bm1, int d,
                                                  uint32_t* __restrict__ bm0) {
  const int64_t pc = (int64_t)blockIdx.x * BS + threadIdx.x;
  if (pc >= (int64_t)1 << (2 * d)) return;
  if (!((bm1[pc >> 3] >> (4 * (pc & 7))) & 0xFu)) return;
  bm_mark_nbrs(bm0, (uint64_t)pc, d);
}
// the same with one thread per word of bm1 (8 parents), for the deep and
// sparse bitmaps where a thread per cell would mostly find nothing
__global__ __launch_bounds__(BS) void k_bm_spread_w(const uint32_t* __restrict__ bm1, int d,
                                                    uint32_t* __restrict__ bm0) {
  const int64_t w = (int64_t)blockIdx.x * BS + threadIdx.x;
  if (w >= ((int64_t)1 << (2 * d)) / 8) return;
  const uint32_t v = bm1[w];
  if (!v) return;
  for (int q = 0; q < 8; ++q)
    if ((v >> (4 * q)) & 0xFu) bm_mark_nbrs(bm0, (uint64_t)w * 8 + q, d);
}
// the same from a sorted list of depth-(d+1) codes
__global__ __launch_bounds__(BS) void k_bm_spread_list(const uint64_t* __restrict__ lst,
                                                       int64_t n, int d,
                                                       uint32_t* __restrict__ bm0) {
  const int64_t i = (int64_t)blockIdx.x * BS + threadIdx.x;
  if (i >= n) return;
  const uint64_t c = lst[i];
  if (i > 0 && (lst[i - 1] >> 2) == (c >> 2)) return;
  bm_mark_nbrs(bm0, c >> 2, d);
}
// popcount per word (for the scan) and per depth
__global__ __launch_bounds__(BS) void k_bm_count(const uint32_t* __restrict__ bm, BmOffsets o,
                                                 int dmax, int* __restrict__ pc,
                                                 int* __restrict__ dcnt) {
  __shared__ int red[BS / 64];
  const int64_t w = (int64_t)blockIdx.x * BS + threadIdx.x;
  const int c = __popc(bm[w]);
  pc[w] = c;
  int v = c;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    for (int i = 0; i < BS / 64; ++i) t += red[i];
    if (t) atomicAdd(dcnt + bm_depth(o, dmax, (int64_t)blockIdx.x * BS), t);
  }
}
// set bits in word order -> codes, at out[pos[w] ...]
__global__ __launch_bounds__(BS) void k_bm_scatter(const uint32_t* __restrict__ bm, BmOffsets o,
                                                   int dmax, const int* __restrict__ pos,
                                                   uint64_t* __restrict__ out) {
  const int64_t w = (int64_t)blockIdx.x * BS + threadIdx.x;
  uint32_t v = bm[w];
  if (!v) return;
  const int d = bm_depth(o, dmax, w);
  const uint64_t base = (uint64_t)(w - o.wo[d]) * 32;
  int p = pos[w];
  while (v) {
    const int b = __builtin_ctz(v);
    out[p++] = base + (uint64_t)b;
    v &= v - 1;
  }
}

// --- nodes with children (split or X-list) -----------------------------------
// Real nodes of level d are the children of S_{d-1} (the root for d = 0).
__device__ __forceinline__ void real_flags_one(const uint64_t* __restrict__ s_all,
                                               const int64_t* __restrict__ soff,
                                               const int64_t* __restrict__ roff, int L, int64_t r,
                                               uint64_t* __restrict__ rcode, int* __restrict__ hasc,
                                               int* __restrict__ kind, int* lc) {
  int d = 0;
  while (r >= roff[d + 1]) ++d;
  int64_t k = r - roff[d];
  uint64_t code = d == 0 ? 0 : ((s_all[soff[d - 1] + k / 4] << 2) | (uint64_t)(k & 3));
  int inS = 0, isX = 0;
  if (d <= L - 2) {
    const uint64_t* lst = s_all + soff[d];
    const int64_t nl = soff[d + 1] - soff[d];
    inS = bsearch_u64(lst, nl, code) >= 0;
    if (!inS && d >= 1) {
      uint32_t ix, iy;
      demorton(code, &ix, &iy);
      const int64_t lim = (int64_t)1 << d;
      for (int q = 0; q < 9 && !isX; ++q) {
        if (q == 4) continue;
        int64_t nx = (int64_t)ix + q / 3 - 1, ny = (int64_t)iy + q % 3 - 1;
        if (nx < 0 || ny < 0 || nx >= lim || ny >= lim) continue;
        isX = bsearch_u64(lst, nl, morton((uint32_t)nx, (uint32_t)ny)) >= 0;
      }
    }
  }
  rcode[r] = code;
  hasc[r] = inS || isX;
  kind[r] = isX;
  if (inS || isX) atomicAdd(&lc[d], 1);
}

__global__ __launch_bounds__(BS) void k_real_flags(const uint64_t* __restrict__ s_all,
                                                   const int64_t* __restrict__ soff,
                                                   const int64_t* __restrict__ roff, int L,
                                                   uint64_t* __restrict__ rcode,
                                                   int* __restrict__ hasc, int* __restrict__ kind,
                                                   int* __restrict__ pcount) {
  __shared__ int lc[kMaxLevels];
  if (threadIdx.x < kMaxLevels) lc[threadIdx.x] = 0;
  __syncthreads();
  int64_t r = (int64_t)blockIdx.x * BS + threadIdx.x;
  if (r < roff[L]) real_flags_one(s_all, soff, roff, L, r, rcode, hasc, kind, lc);
  __syncthreads();
  if (threadIdx.x < kMaxLevels && lc[threadIdx.x]) atomicAdd(&pcount[threadIdx.x], lc[threadIdx.x]);
}

__global__ __launch_bounds__(BS) void k_p_scatter(const uint64_t* __restrict__ rcode,
                                                  const int* __restrict__ hasc,
                                                  const int* __restrict__ kind,
                                                  const int* __restrict__ rank, int64_t nr,
                                                  uint64_t* __restrict__ p_code,
                                                  int* __restrict__ p_kind) {
  int64_t r = (int64_t)blockIdx.x * BS + threadIdx.x;
  if (r >= nr || !hasc[r]) return;
  int q = rank[r];
  p_code[q] = rcode[r];
  p_kind[q] = kind[r];
}

// --- trees of at most kBmLevels levels: cells as bitmaps ------------------------
// Split cells down to depth kBmMaxD (every tree but those of points clustered
// to 2^-12 of the box) are one bitmap per depth: bit c of depth d is cell c
// (its Morton code), so a word is a block of 4 x 8 cells and the 3x3
// neighbourhoods of the 2:1 balance and of the X-list are shifts and masks of
// nine words, a cell's children a nibble, its rank among the nodes with
// children a popcount.  The lists below (sorted codes, binary searches, sorted
// scans) did the same work in 45 launches, copies and fills, most of them
// bound by their launch or by a chain of dependent loads, and two more
// counts read by the host: 270 us after the sort for 1M clustered points (58
// thousand nodes), the bitmaps 95.  The lists stay for the deeper trees, whose
// bitmaps would no longer fit in L2 (4^12 cells are 2 MB per bitmap and 4 MB
// with the index).
// Each depth's words start at a multiple of BS, so a block of BS words lies
// in one depth.
constexpr int kBmLevels = kBmMaxD + 2;
static_assert(BS == kBmBlock, "the bitmap kernels take a block of words each");
__host__ __device__ constexpr int bm_words(int d) { return d <= 2 ? 1 : 1 << (2 * d - 5); }
constexpr int kBmWords = bm_wo(kBmMaxD + 1);
constexpr int kBmBlocks = kBmWords / BS;
static_assert(bm_wo(8) == bm_wo(7) + bm_words(7) && kBmBlocks < 1024,
              "k_bm_sums scans the blocks' counts in one pass of 1024 threads");
__device__ __forceinline__ int bm_depth_of(int w, int dmax) {
  int d = 0;
  while (d < dmax && w >= bm_wo(d + 1)) ++d;
  return d;
}

// The split cells of the refinement: position i starts those of depths
// s(i)+1 .. c(i).  Depths below kBmMaxD are left out (the lists take such a
// tree).
__global__ __launch_bounds__(BS) void k_bm_mark_points(const uint64_t* __restrict__ keys,
                                                       const int2* __restrict__ sc, int n,
                                                       uint32_t* __restrict__ bm) {
  const int i = xcd_block(blockIdx.x, gridDim.x, 0) * BS + threadIdx.x;
  if (i >= n) return;
  const int2 v = sc[i];
  if (v.x >= v.y) return;
  const uint64_t k = keys[i];
  for (int d = v.x + 1; d <= min(v.y, kBmMaxD); ++d)
    bm_set(bm + bm_wo(d), d == 0 ? 0 : k >> (64 - 2 * d));
}

// nibble j of v nonzero -> bit j; and back, bit j -> nibble j all ones
__device__ __forceinline__ uint32_t nibbles_any(uint32_t v) {
  v |= v >> 1;
  v = (v | v >> 2) & 0x11111111u;
  v = (v | v >> 3) & 0x03030303u;
  v = (v | v >> 6) & 0x000F000Fu;
  return (v | v >> 12) & 0xFFu;
}
__device__ __forceinline__ uint32_t nibbles_all(uint32_t b) {
  b = (b | b << 12) & 0x000F000Fu;
  b = (b | b << 6) & 0x03030303u;
  b = (b | b << 3) & 0x11111111u;
  return b * 15u;
}
// The cells of word w and their neighbours above and below in y; wm and wp
// are the words at y - 8 and y + 8.  y's bits are bits 0, 2, 4 of the cell's
// place in its word, x's bits 1 and 3: a step in y moves a cell by 1, 3 or 11
// places by where the carry ends, and by 21 into the next word.
__device__ __forceinline__ uint32_t bm_dilate_y(uint32_t wm, uint32_t w, uint32_t wp) {
  const uint32_t up = (w & 0x55555555u) << 1 | (w & 0x0A0A0A0Au) << 3 | (w & 0x0000A0A0u) << 11;
  const uint32_t dn = (w & 0xAAAAAAAAu) >> 1 | (w & 0x50505050u) >> 3 | (w & 0x05050000u) >> 11;
  return w | up | dn | (wm & 0xA0A00000u) >> 21 | (wp & 0x00000505u) << 21;
}
// Word W of the 3x3 dilation of depth d's bitmap (d >= 1), whose word V is
// word(V): words interleave the low bit of x before that of y.
template <class F>
__device__ __forceinline__ uint32_t bm_dilate(int d, int W, F word) {
  if (d <= 2) {
    const uint32_t y0 = bm_dilate_y(0, word(0), 0);
    const uint32_t v = y0 | (y0 & 0x33333333u) << 2 | (y0 & 0x00CC00CCu) << 6 |
                       (y0 & 0xCCCCCCCCu) >> 2 | (y0 & 0x33003300u) >> 6;
    return v & (d == 1 ? 0xFu : 0xFFFFu);
  }
  uint32_t wx, wy;
  demorton((uint64_t)W, &wy, &wx);
  const int nx = 1 << (d - 2), ny = 1 << (d - 3);
  uint32_t c[3][3], y[3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      const int x = (int)wx + a - 1, yy = (int)wy + b - 1;
      const bool in = x >= 0 && yy >= 0 && x < nx && yy < ny;
      c[a][b] = in ? word((int)morton((uint32_t)yy, (uint32_t)x)) : 0u;
    }
#pragma unroll
  for (int a = 0; a < 3; ++a) y[a] = bm_dilate_y(c[a][0], c[a][1], c[a][2]);
  const uint32_t v = y[1];
  return v | (v & 0x33333333u) << 2 | (v & 0x00CC00CCu) << 6 | (v & 0xCCCCCCCCu) >> 2 |
         (v & 0x33003300u) >> 6 | (y[0] & 0xCC00CC00u) >> 10 | (y[2] & 0x00330033u) << 10;
}

// 2:1 balance: S_d |= N(parents(S_{d+1})), one thread per word of depth d,
// from the deepest depth up.  An already balanced tree keeps its cells.
__global__ __launch_bounds__(BS) void k_bm_balance(int d, uint32_t* __restrict__ bm) {
  const int w = blockIdx.x * BS + threadIdx.x;
  if (w >= bm_words(d)) return;
  const uint4* next = reinterpret_cast<const uint4*>(bm + bm_wo(d + 1));
  bm[bm_wo(d) + w] |= bm_dilate(d, w, [&](int V) {
    const uint4 v = next[V];
    return nibbles_any(v.x) | nibbles_any(v.y) << 8 | nibbles_any(v.z) << 16 |
           nibbles_any(v.w) << 24;
  });
}
// The depths dtop <= kBmLowD .. 1 in one block, their words (and those of
// depth dtop + 1) in LDS: a launch per depth cost more than its work.  Depth 7
// is the last whose words are at most one per thread; the loads of all depths
// are in flight together (a loop over the depths took 23 us instead of 10).
constexpr int kBmLowD = 7;
__host__ __device__ constexpr int bm_lo(int d) {   // first LDS word of depth d >= 1
  return d <= 2 ? d - 1 : 2 + 2 * (((1 << (2 * (d - 3))) - 1) / 3);
}
__global__ __launch_bounds__(1024) void k_bm_balance_low(int dtop, uint32_t* __restrict__ bm) {
  constexpr int kLds = bm_lo(kBmLowD + 2), kPer = (kLds + 1023) / 1024;
  __shared__ uint32_t sh[kLds];
  const int ntop = bm_lo(dtop + 2);
  int src[kPer];
  uint32_t v[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = j * 1024 + threadIdx.x;
    int d = 1;
#pragma unroll
    for (int e = 2; e <= kBmLowD + 1; ++e) d += i >= bm_lo(e) ? 1 : 0;
    src[j] = bm_wo(d) + i - bm_lo(d);
    v[j] = i < ntop ? bm[src[j]] : 0u;
  }
#pragma unroll
  for (int j = 0; j < kPer; ++j)
    if (j * 1024 + threadIdx.x < ntop) sh[j * 1024 + threadIdx.x] = v[j];
  __syncthreads();
  for (int d = dtop; d >= 1; --d) {
    const uint32_t* next = sh + bm_lo(d + 1);
    const int nn = bm_words(d + 1), w = threadIdx.x;
    if (w < bm_words(d))
      sh[bm_lo(d) + w] |= bm_dilate(d, w, [&](int V) {
        uint32_t q = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (4 * V + j < nn) q |= nibbles_any(next[4 * V + j]) << (8 * j);
        return q;
      });
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = j * 1024 + threadIdx.x;
    if (i < bm_lo(dtop + 1)) bm[src[j]] = sh[i];
  }
}

// Nodes with children, P_d = the real cells (children of S_{d-1}) in S_d or
// next to one of it: word and popcount prefix within the block of BS words
// (pp), and the block's count.
__global__ __launch_bounds__(BS) void k_bm_parents(const uint32_t* __restrict__ bm, int dmax,
                                                   uint2* __restrict__ pp,
                                                   int* __restrict__ bsum) {
  __shared__ int lds[BS / 64];
  __shared__ int tot;
  const int i = blockIdx.x * BS + threadIdx.x;
  const int d = bm_depth_of(blockIdx.x * BS, dmax);
  const int w = i - bm_wo(d);
  uint32_t v = 0;
  if (d == 0) {
    v = bm[i];
  } else if (w < bm_words(d)) {
    const uint32_t* s = bm + bm_wo(d);
    const uint32_t up = bm[bm_wo(d - 1) + (w >> 2)];
    v = bm_dilate(d, w, [&](int V) { return s[V]; }) & nibbles_all((up >> (8 * (w & 3))) & 0xFFu);
  }
  const int ex = block_exclusive_scan<BS>(__popc(v), lds, &tot);
  pp[i] = make_uint2(v, (uint32_t)ex);
  if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}
// Exclusive scan of the blocks' counts; the ranks that start the depths
// 0 .. dmax and their end to the host (words 0 .. dmax + 1 of the mailbox).
__global__ __launch_bounds__(1024) void k_bm_sums(int* __restrict__ bsum, int dmax,
                                                  uint64_t* __restrict__ mbox, uint32_t seq) {
  __shared__ int lds[1024 / 64];
  const int t = threadIdx.x, nblk = bm_wo(dmax + 1) / BS;
  const int ex = block_exclusive_scan<1024>(t < nblk ? bsum[t] : 0, lds, nullptr);
  if (t < nblk) bsum[t] = ex;
  for (int d = 0; d <= dmax + 1; ++d)
    if (t == bm_wo(d) / BS) mailbox_put(mbox, d, seq, ex);
}

// --- final node arrays ---------------------------------------------------------
struct LevOff {
  int lo[kMaxLevels + 1];   // node offset of each level, and the end
};
__device__ __forceinline__ int level_of(const LevOff& lv, int L, int g) {
  int d = 0;
  for (int j = 1; j < L; ++j) d += g >= lv.lo[j] ? 1 : 0;   // uniform loads
  return d;
}

// Neighbour cells without taking a code apart: x sits on its odd bits and y on
// its even ones, so adding a spread offset with the other bits set carries
// within one coordinate; a step out of the level's 4^d cells leaves bits above
// 2 d.  (With each neighbour's code formed from its coordinates k_node_slots
// took 23 us for 115 thousand nodes, with the steps 20.)
constexpr uint64_t kXBits = 0xAAAAAAAAAAAAAAAAull, kYBits = 0x5555555555555555ull;
__device__ __forceinline__ uint64_t cell_step(uint64_t c, uint64_t dx, uint64_t dy) {
  return (((c | kYBits) + dx) & kXBits) | (((c | kXBits) + dy) & kYBits);
}
__device__ __forceinline__ bool on_level(uint64_t c, int d) { return (c >> (2 * d)) == 0; }
// colleague q = 3 (dx + 1) + dy + 1 of cell c
__device__ __forceinline__ uint64_t colleague_cell(uint64_t c, int q) {
  return cell_step(c, morton((uint32_t)(q / 3 - 1), 0), morton(0, (uint32_t)(q % 3 - 1)));
}

// M2L partners: children of the parent's colleagues, outside the 3x3
// (tree.py:399-435).  For child position (cx, cy) the parent's 3x3 covers
// offsets [-2-cx, 3-cx] x [-2-cy, 3-cy].
struct SlotOffsets {
  int ox[kNumM2L], oy[kNumM2L];
  uint64_t dx[kNumM2L], dy[kNumM2L];   // the same as steps of a code
};
__constant__ SlotOffsets c_slot_off;
// whether slot s of cell c of level d names a cell, and that cell
__device__ __forceinline__ bool slot_cell(uint64_t c, int d, int s, uint64_t* e) {
  const int cx = (int)(c >> 1) & 1, cy = (int)c & 1;
  const int ox = c_slot_off.ox[s], oy = c_slot_off.oy[s];
  *e = cell_step(c, c_slot_off.dx[s], c_slot_off.dy[s]);
  return ox >= -2 - cx && ox <= 3 - cx && oy >= -2 - cy && oy <= 3 - cy && on_level(*e, d);
}

// Node lookups by cell: node(d, c) is the node index of the level-d cell with
// Morton code c or -1; kids(d, c, &xl) the first child of that node or -1, xl
// whether it is an X-list node.
struct BmCells {
  BmIndex ix;
  const uint32_t* bm;
  __device__ __forceinline__ int node(int d, uint64_t c) const { return ix.node(d, c); }
  __device__ __forceinline__ int kids(int d, uint64_t c, bool* xl) const {
    const uint32_t s = bm[bm_wo(d) + (int)(c >> 5)];
    const int r = ix.rank(d, c);
    *xl = r >= 0 && !((s >> (c & 31)) & 1u);
    return r >= 0 ? 1 + 4 * r : -1;
  }
};
// Of the deeper trees: direct on a full level, a table lookup on the other
// levels up to depth kIdxDepth (one int per cell of the level, -1 where no
// node), else a binary search in the level's sorted codes.
constexpr int kIdxDepth = 11;   // tables of at most 4^12/3 ints (22 MB)
struct ListCells {
  const uint64_t* code;
  LevOff lv;
  const int* tab;
  int64_t off[kMaxLevels];      // level d's table in tab, or -1
  const uint64_t* p_code;       // nodes with children and their kinds
  const int* p_kind;
  __device__ __forceinline__ int node(int d, uint64_t c) const {
    const int64_t nl = lv.lo[d + 1] - lv.lo[d];
    if (d < 16 && nl == ((int64_t)1 << (2 * d))) return lv.lo[d] + (int)c;
    if (off[d] >= 0) return tab[off[d] + (int64_t)c];
    const int64_t pos = bsearch_u64(code + lv.lo[d], nl, c);
    return pos >= 0 ? lv.lo[d] + (int)pos : -1;
  }
  __device__ __forceinline__ int kids(int d, uint64_t c, bool* xl) const {
    const int p0 = (lv.lo[d + 1] - 1) / 4;   // rank of the depth's first
    const int64_t pos = bsearch_u64(p_code + p0, (lv.lo[d + 2] - lv.lo[d + 1]) / 4, c);
    *xl = pos >= 0 && p_kind[p0 + pos] == 1;
    return pos >= 0 ? lv.lo[d + 1] + 4 * (int)pos : -1;
  }
};

// Codes, levels and fake flags of all nodes, their point ranges not yet set
// (-1; the root's are).  From the bitmaps: a thread per nibble of P, which
// writes the children of its cells; one thread also writes the root.
__global__ __launch_bounds__(BS) void k_bm_nodes(BmCells cells, int dmax, int npts,
                                                 uint64_t* __restrict__ code,
                                                 int* __restrict__ nlev, int* __restrict__ flags,
                                                 int* __restrict__ rb, int* __restrict__ rt) {
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i == 0) {
    code[0] = 0;
    nlev[0] = 0;
    flags[0] = 0;
    rb[0] = 0;
    rt[0] = npts;
  }
  const int w = i >> 3, q = 4 * (i & 7);
  if (w >= bm_wo(dmax + 1)) return;
  const uint2 v = cells.ix.pp[w];
  uint32_t m = (v.x >> q) & 0xFu;
  if (!m) return;
  const uint32_t sp = cells.bm[w] >> q;
  const int d = bm_depth_of((int)(blockIdx.x * (BS / 8)), dmax);
  const uint64_t c0 = (uint64_t)(w - bm_wo(d)) * 32 + (uint64_t)q;
  int g = 1 + 4 * (cells.ix.boff[w / BS] + (int)v.y + __popc(v.x & ((1u << q) - 1u)));
  for (; m; m &= m - 1, g += 4) {
    const int b = __builtin_ctz(m);
    const int f = (sp >> b) & 1u ? 0 : NF_FAKE;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      code[g + k] = ((c0 + (uint64_t)b) << 2) | (uint64_t)k;
      nlev[g + k] = d + 1;
      flags[g + k] = f;
      rb[g + k] = -1;
      rt[g + k] = -1;
    }
  }
}
// From the lists, with the entries of the level tables.
__global__ __launch_bounds__(BS) void k_list_nodes(ListCells cells, int L, int npts,
                                                   uint64_t* __restrict__ code,
                                                   int* __restrict__ nlev,
                                                   int* __restrict__ flags, int* __restrict__ rb,
                                                   int* __restrict__ rt, int* __restrict__ tab) {
  const int g = blockIdx.x * BS + threadIdx.x;
  if (g >= cells.lv.lo[L]) return;
  const int d = level_of(cells.lv, L, g);
  uint64_t c = 0;
  int fake = 0;
  if (d > 0) {
    const int pj = (g - 1) / 4;
    c = (cells.p_code[pj] << 2) | (uint64_t)((g - 1) & 3);
    fake = cells.p_kind[pj] == 1;
  }
  code[g] = c;
  nlev[g] = d;
  flags[g] = fake ? NF_FAKE : 0;
  rb[g] = g == 0 ? 0 : -1;
  rt[g] = g == 0 ? npts : -1;
  if (cells.off[d] >= 0) tab[cells.off[d] + (int64_t)c] = g;
}

// Source ranges of the nodes with points from the sorted keys: point i starts
// its cells of depths s(i)+1.. and ends those of depths s(i+1)+1.. (s = common
// depth with the previous key).  A cell exists only below an existing parent,
// so each walk stops at the first depth without one.
template <class Cells>
__global__ __launch_bounds__(BS) void k_cell_ranges(const uint64_t* __restrict__ keys,
                                                    const int2* __restrict__ sc, int n,
                                                    Cells cells, int L, int* __restrict__ rb,
                                                    int* __restrict__ rt) {
  const int i = xcd_block(blockIdx.x, gridDim.x, 0) * BS + threadIdx.x;
  if (i >= n) return;
  const int s0 = sc[i].x;
  const int s1 = i + 1 < n ? sc[i + 1].x : -1;
  if (s0 >= L - 1 && s1 >= L - 1) return;
  const uint64_t k = keys[i];
  for (int d = max(1, min(s0, s1) + 1); d <= L - 1; ++d) {
    const int g = cells.node(d, k >> (64 - 2 * d));
    if (g < 0) break;
    if (d > s0) rb[g] = i;
    if (d > s1) rt[g] = i + 1;
  }
}

// The kinds of the nodes that the lists below count, as lane masks of a wave:
// evaluation boxes, S2M boxes (compute_upwards nodes that own a multipole
// row), and the sibling groups (levels >= 2, from node g0) holding a source,
// which own four multipole rows.  Lane j of wave w holds node 64 w + j - 63,
// so a group is four lanes of one wave (the root alone fills wave 0).
struct NodeKinds {
  unsigned long long ev, up, grp;
};
__device__ __forceinline__ int wave_node(int v) { return v - 63; }
inline int64_t wave_slots(int64_t nn) { return nn + 63; }
__device__ __forceinline__ NodeKinds node_kinds(int f, int g, int g0) {
  NodeKinds k;
  k.ev = __ballot((f & NF_LEAF) != 0);
  k.up = __ballot((f & NF_UP) != 0 && g >= g0);
  unsigned long long m = __ballot((f & NF_SOURCE) != 0 && g >= g0);
  m |= m >> 1;
  m |= m >> 2;
  k.grp = m & 0x1111111111111111ull;
  return k;
}

// Everything of a node but its lists, and each wave's counts of the kinds
// (planes of nw ints).  A cell without points sits where its keys would be:
// behind the nearest sibling before it that has points, else at its parent's
// start, found the same way.
template <class Cells>
__global__ __launch_bounds__(64) void k_nodes(
    Cells cells, LevOff lv, int L, const int* __restrict__ rb, const int* __restrict__ rt,
    double xmin0, double ymin0, double w0, const uint64_t* __restrict__ code,
    int* __restrict__ flags, int* __restrict__ bot, int* __restrict__ top,
    int* __restrict__ parent, int* __restrict__ child, int* __restrict__ coll,
    double* __restrict__ xmid, double* __restrict__ ymid, int g0, int nw,
    int* __restrict__ wcnt) {
  const int g = wave_node(blockIdx.x * 64 + threadIdx.x);
  const bool act = g >= 0 && g < lv.lo[L];
  int f = 0;
  if (act) {
    const int d = level_of(lv, L, g);
    const uint64_t c = code[g];
    const int fake = flags[g] & NF_FAKE;
    bool xl = false;
    const int ch = !fake && d <= L - 2 ? cells.kids(d, c, &xl) : -1;
    const int leaf = !fake && (ch < 0 || xl);
    int b = rb[g], t = rt[g];
    int cg = g, cd = d;
    while (b < 0) {
      const int k = (cg - 1) & 3, sib = cg - k;
      const int t0 = rt[sib], t1 = rt[sib + 1], t2 = rt[sib + 2];
      if (k > 0) b = t0;
      if (k > 1 && t1 >= 0) b = t1;
      if (k > 2 && t2 >= 0) b = t2;
      if (b < 0) {
        --cd;
        cg = cells.node(cd, c >> (2 * (d - cd)));
        b = rb[cg];
      }
      t = b;
    }
    const int has_src = t > b;
    if (fake) f |= NF_FAKE;
    if (leaf) f |= NF_LEAF;
    if (xl) f |= NF_XLIST;
    if (ch >= 0) f |= NF_CHILDREN;
    if (has_src) f |= NF_SOURCE;
    if (((leaf && !xl) || fake) && has_src) f |= NF_UP;   // tree.py:557-560
    if ((!leaf || xl) && !fake) f |= NF_DOWN;             // tree.py:562 (fake nodes have leaf=False)
    flags[g] = f;
    bot[g] = b;
    top[g] = t;
    child[g] = ch;
    // centre by the reference recurrence
    double xm0 = xmin0, ym0 = ymin0, w = w0;
    for (int l = 1; l <= d; ++l) {
      const double h = 0.5 * w;
      const double xm = xm0 + h, ym = ym0 + h;
      const int dig = (int)((c >> (2 * (d - l))) & 3);
      xm0 = (dig & 2) ? xm : xm - h;
      ym0 = (dig & 1) ? ym : ym - h;
      w = h;
    }
    xmid[g] = xm0 + 0.5 * w;
    ymid[g] = ym0 + 0.5 * w;
    // colleagues and parent
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      const uint64_t e = colleague_cell(c, q);
      coll[(int64_t)g * 9 + q] = q == 4 ? g : on_level(e, d) ? cells.node(d, e) : -1;
    }
    parent[g] = d > 0 ? cells.node(d - 1, c >> 2) : -1;
  }
  const NodeKinds k = node_kinds(f, g, g0);
  if (threadIdx.x == 0) {
    wcnt[blockIdx.x] = (int)__popcll(k.ev);
    wcnt[nw + blockIdx.x] = (int)__popcll(k.up);
    wcnt[2 * nw + blockIdx.x] = (int)__popcll(k.grp);
  }
}

// Evaluation boxes, S2M boxes and multipole rows from the waves' counts.  Up
// to kSumWaves waves each block adds the counts of the waves before it itself
// (scanned = 0; a scan of its own would cost three launches); above, wcnt
// holds their exclusive prefixes.  The totals and the first row of each level
// >= 2 go to the host's mailbox: boxes, S2M boxes, row groups, then the levels.
constexpr int64_t kSumWaves = 8192;   // three 21-bit sums fit in 64 bits
__global__ __launch_bounds__(1024) void k_node_lists(const int* __restrict__ flags, LevOff lv,
                                                     int L, int g0, int nw,
                                                     const int* __restrict__ wcnt, int scanned,
                                                     int* __restrict__ evalid,
                                                     int* __restrict__ evalnode,
                                                     int* __restrict__ upnodes,
                                                     int* __restrict__ row,
                                                     uint64_t* __restrict__ mbox, uint32_t seq) {
  __shared__ unsigned long long part[16];
  __shared__ int wv[3][16];
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  const int w0 = blockIdx.x * 16;   // the block's first wave, < nw
  const int g = wave_node(blockIdx.x * 1024 + t);
  const bool act = g >= 0 && g < lv.lo[L];
  const int f = act ? flags[g] : 0;
  const NodeKinds k = node_kinds(f, g, g0);
  if (lane == 0) {
    wv[0][wid] = (int)__popcll(k.ev);
    wv[1][wid] = (int)__popcll(k.up);
    wv[2][wid] = (int)__popcll(k.grp);
  }
  unsigned long long acc = 0;
  if (!scanned) {
    for (int j = t; j < w0; j += 1024)
      acc += (unsigned long long)wcnt[j] | (unsigned long long)wcnt[nw + j] << 21 |
             (unsigned long long)wcnt[2 * nw + j] << 42;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if (lane == 0) part[wid] = acc;
  }
  __syncthreads();
  int base[3];
  if (scanned) {
    for (int q = 0; q < 3; ++q) base[q] = wcnt[(int64_t)q * nw + w0];
  } else {
    acc = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) acc += part[w];
    for (int q = 0; q < 3; ++q) base[q] = (int)(acc >> (21 * q)) & 0x1FFFFF;
  }
  for (int w = 0; w < wid; ++w)
    for (int q = 0; q < 3; ++q) base[q] += wv[q][w];
  if (blockIdx.x == gridDim.x - 1 && wid == 15 && lane < 3) {
    const int b = lane == 0 ? base[0] : lane == 1 ? base[1] : base[2];
    mailbox_put(mbox, lane, seq, b + wv[lane][15]);
  }
  if (!act) return;
  const unsigned long long below = (1ull << lane) - 1ull;
  const int e = base[0] + (int)__popcll(k.ev & below);
  const bool ev = (k.ev >> lane) & 1ull;
  evalid[g] = ev ? e : -1;
  if (ev) evalnode[e] = g;
  if ((k.up >> lane) & 1ull) upnodes[base[1] + (int)__popcll(k.up & below)] = g;
  const int lead = lane & ~3;
  const int r = 4 * (base[2] + (int)__popcll(k.grp & ((1ull << lead) - 1ull)));
  row[g] = (k.grp >> lead) & 1ull ? r + (lane & 3) : -1;
  for (int d = 2; d < L; ++d)
    if (g == lv.lo[d]) mailbox_put(mbox, 3 + d - 2, seq, r);
}

// The lists that read other nodes' records: the multipole rows of the M2L
// partners (levels >= 2), the source ranges of the nine colleagues (one load
// per colleague for the evaluation kernels instead of its index and then its
// range), and per multipole row the row of its node's first child (-1 without
// children) with the node's flags, one record for the upward pass.  Sixteen
// lanes per node, its 40 partner slots j, j + 16, j + 32 on lane j: bound by
// the chain of dependent loads, which three slots share, and then by the
// stores (a thread per slot took 24 us for 58 thousand nodes, this 16).
constexpr int kSlotLanes = 16;
template <class Cells>
__global__ __launch_bounds__(BS) void k_node_slots(
    Cells cells, LevOff lv, int L, const uint64_t* __restrict__ code,
    const int* __restrict__ nlev, const int* __restrict__ flags, const int* __restrict__ row,
    const int* __restrict__ child,
    const int* __restrict__ coll, const int* __restrict__ bot, const int* __restrict__ top,
    int* __restrict__ m2l, uint64_t* __restrict__ m2lmask, int2* __restrict__ crange,
    int2* __restrict__ rowinfo) {
  const int64_t tid = (int64_t)xcd_block(blockIdx.x, gridDim.x, 0) * BS + threadIdx.x;
  const int g = (int)(tid / kSlotLanes);
  const int j = (int)(tid % kSlotLanes);
  if (g >= lv.lo[L]) return;
  const int f = flags[g], d = nlev[g];
  const uint64_t cg = code[g];
  if (j < 9) {
    const int c = coll[(int64_t)g * 9 + j];
    crange[(int64_t)g * 9 + j] = c >= 0 ? make_int2(bot[c], top[c]) : make_int2(0, 0);
  } else if (j == 9) {
    const int r = row[g];
    if (r >= 0) rowinfo[r] = make_int2((f & NF_CHILDREN) ? row[child[g]] : -1, f);
  }
  if (L < 3 || g < lv.lo[2]) return;
  constexpr int kPer = (kNumM2L + kSlotLanes - 1) / kSlotLanes;
  int q[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int s = j + u * kSlotLanes;
    uint64_t e;
    q[u] = s < kNumM2L && !(f & NF_FAKE) && slot_cell(cg, d, s, &e) ? cells.node(d, e) : -1;
  }
  uint64_t mask = 0;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int s = j + u * kSlotLanes;
    const int r = q[u] >= 0 ? row[q[u]] : -1;
    if (s < kNumM2L) m2l[(int64_t)g * kNumM2L + s] = r;
    const unsigned long long b = __ballot(r >= 0) >> (threadIdx.x & (64 - kSlotLanes));
    mask |= (uint64_t)(b & ((1u << kSlotLanes) - 1u)) << (u * kSlotLanes);
  }
  if (j == 0) m2lmask[g] = mask;
}

__global__ __launch_bounds__(BS) void k_locate(const double* __restrict__ tx,
                                               const double* __restrict__ ty, int64_t nt,
                                               const int* __restrict__ flags,
                                               const int* __restrict__ child,
                                               const double* __restrict__ xmid,
                                               const double* __restrict__ ymid,
                                               int* __restrict__ out) {
  int64_t i = (int64_t)blockIdx.x * BS + threadIdx.x;
  if (i >= nt) return;
  const double x = tx[i], y = ty[i];
  int g = 0;
  for (int it = 0; it < kMaxLevels && !(flags[g] & NF_LEAF); ++it)
    g = child[g] + 2 * (x > xmid[g]) + (y > ymid[g]);   // tree.py:720-725
  out[i] = g;
}

inline unsigned grid_for(int64_t n) { return (unsigned)(n <= 0 ? 1 : ceil_div(n, BS)); }

// --- complete trees --------------------------------------------------------------
// When the split cells of every depth d < D are all 4^d cells of that depth
// and no cell of depth D splits, the reference's refinement (split iff more
// than ncut points, tree.py:204) has built the complete quadtree of depth D:
// its leaves all sit on level D, so no 2:1 balance split and no X-list node
// exists (both need leaves on different levels), and every sibling group of
// the levels >= 2 holds a source (its parent has more than ncut).  Uniform
// data give such trees.  After the sort and the split-cell counts that every
// build reads back, such a tree takes closed forms of all node arrays in one
// kernel instead of the split lists, their scans and the two further read-backs.
constexpr int kFullMaxDepth = 15;   // depth-D cell index tables of at most 4^15 ints

// first sorted point of each nonempty depth-D cell, -1 for the empty ones:
// the point that starts a cell also marks the empty cells between the
// previous point's cell and its own (and the last point those after it).  In
// a complete tree every depth D-1 cell has points, so such a run is at most
// six cells.
__global__ __launch_bounds__(BS) void k_full_starts(const uint64_t* __restrict__ keys,
                                                    const int2* __restrict__ sc, int n, int D,
                                                    int* __restrict__ start,
                                                    const int* __restrict__ gate) {
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i >= n || (gate && *gate == 0)) return;
  const int2 si = sc[i];
  // loaded with sc, not behind its test
  const uint64_t k = keys[i], kp = keys[i > 0 ? i - 1 : 0];
  const int64_t cell = (int64_t)(k >> (64 - 2 * D));
  if (si.x < D) {
    for (int64_t e = i > 0 ? (int64_t)(kp >> (64 - 2 * D)) + 1 : 0; e < cell; ++e) start[e] = -1;
    start[cell] = i;
  }
  if (i == n - 1)
    for (int64_t e = cell + 1; e < ((int64_t)1 << (2 * D)); ++e) start[e] = -1;
}

// points of a depth-d cell c: [bot, top) from the depth-D starts (a cell
// without points sits where its keys would be)
__device__ __forceinline__ int full_pos(const int* __restrict__ start,
                                        const uint64_t* __restrict__ keys, int n, int D, int d,
                                        uint64_t c) {
  const uint64_t leaf = c << (2 * (D - d));
  if (leaf >= ((uint64_t)1 << (2 * D))) return n;
  const int v = start[leaf];
  return v >= 0 ? v : (int)lower_bound_u64(keys, n, leaf << (64 - 2 * D));
}

__host__ __device__ __forceinline__ int full_levoff(int d) { return (int)((((int64_t)1 << (2 * d)) - 1) / 3); }

// Every node array of the complete tree of depth D (levels 0 .. D, level d =
// the 4^d cells in Morton order from levoff(d) = (4^d - 1) / 3).  Sixteen
// lanes per node: lane 0 writes the node's own fields, lanes 0..8 its nine
// colleague slots and all sixteen its 40 M2L slots (j, j + 16, j + 32), so
// the per-node arrays are written in contiguous runs.
constexpr int kFullLanes = 16;
__global__ __launch_bounds__(BS) void k_full_nodes(
    int D, int nn, const int* __restrict__ start, const uint64_t* __restrict__ keys, int npts,
    double xmin0, double ymin0, double w0, uint64_t* __restrict__ code, int* __restrict__ nlev,
    int* __restrict__ flags, int* __restrict__ bot, int* __restrict__ top,
    int* __restrict__ parent, int* __restrict__ child, int* __restrict__ coll,
    int2* __restrict__ crange, double* __restrict__ xmid, double* __restrict__ ymid,
    int* __restrict__ row, int* __restrict__ m2l, int* __restrict__ evalid,
    int* __restrict__ evalnode, int* __restrict__ upnodes, int2* __restrict__ rowinfo,
    const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  const int64_t tid = (int64_t)blockIdx.x * BS + threadIdx.x;
  const int g = (int)(tid / kFullLanes), j = (int)(tid % kFullLanes);
  if (g >= nn) return;
  int d = 0;
  while (d < D && g >= full_levoff(d + 1)) ++d;
  const int lo = full_levoff(d);
  const uint64_t c = (uint64_t)(g - lo);
  const bool leaf = d == D;
  const int g0 = full_levoff(2);
  if (j == 0) {
    const int b = full_pos(start, keys, npts, D, d, c), t = full_pos(start, keys, npts, D, d, c + 1);
    int f = leaf ? NF_LEAF : (NF_CHILDREN | NF_DOWN);   // tree.py:557-562
    if (t > b) f |= NF_SOURCE | (leaf ? NF_UP : 0);
    code[g] = c;
    nlev[g] = d;
    flags[g] = f;
    bot[g] = b;
    top[g] = t;
    parent[g] = d > 0 ? full_levoff(d - 1) + (int)(c >> 2) : -1;
    const int ch = leaf ? -1 : full_levoff(d + 1) + 4 * (int)c;
    child[g] = ch;
    // centre by the reference recurrence (as k_nodes)
    double xm0 = xmin0, ym0 = ymin0, w = w0;
    for (int l = 1; l <= d; ++l) {
      const double h = 0.5 * w;
      const double xm = xm0 + h, ym = ym0 + h;
      const int dig = (int)((c >> (2 * (d - l))) & 3);
      xm0 = (dig & 2) ? xm : xm - h;
      ym0 = (dig & 1) ? ym : ym - h;
      w = h;
    }
    xmid[g] = xm0 + 0.5 * w;
    ymid[g] = ym0 + 0.5 * w;
    // rows: every sibling group of levels >= 2 holds sources, so row = g - g0
    const int r = d >= 2 ? g - g0 : -1;
    row[g] = r;
    if (r >= 0) rowinfo[r] = make_int2(ch >= 0 ? ch - g0 : -1, f);
    evalid[g] = leaf ? (int)c : -1;
    if (leaf) {
      evalnode[c] = g;
      upnodes[c] = g;   // every leaf: an empty one has S2M check values 0 (no sources)
    }
  }
  if (j < 9) {
    const uint64_t cc = colleague_cell(c, j);
    int r = -1;
    int2 rg = make_int2(0, 0);
    if (on_level(cc, d)) {
      r = lo + (int)cc;
      rg = make_int2(full_pos(start, keys, npts, D, d, cc),
                     full_pos(start, keys, npts, D, d, cc + 1));
    }
    coll[(int64_t)g * 9 + j] = r;
    crange[(int64_t)g * 9 + j] = rg;
  }
  if (d >= 2)
    for (int s = j; s < kNumM2L; s += kFullLanes) {
      uint64_t e;
      m2l[(int64_t)g * kNumM2L + s] = slot_cell(c, d, s, &e) ? lo + (int)e - g0 : -1;
    }
}

}  // namespace

// Node arrays of a complete tree of depth D from the sorted points (keys and
// the common depths sc of neighbouring keys); see k_full_nodes.
// The complete tree of depth D, in three parts: its buffers, its node arrays
// (k_full_starts, k_full_nodes; with gate, the kernels do nothing unless
// *gate is set when they run) and the host's level tables.
static void tree_full_buffers(Tree& t, int D) {
  const int NN = full_levoff(D + 1);
  const int64_t n_eval = (int64_t)1 << (2 * D);
  const int64_t n_rows = NN - full_levoff(2);
  t.w_flag.ensure((n_eval + 1) * sizeof(int));
  t.code.ensure(NN * sizeof(uint64_t));
  t.nlevel.ensure(NN * sizeof(int));
  t.bot.ensure(NN * sizeof(int));
  t.top.ensure(NN * sizeof(int));
  t.parent.ensure(NN * sizeof(int));
  t.child.ensure(NN * sizeof(int));
  t.flags.ensure(NN * sizeof(int));
  t.coll.ensure(NN * 9 * sizeof(int));
  t.crange.ensure(((int64_t)NN * 9 + 1) * sizeof(int2));
  t.xmid.ensure(NN * sizeof(double));
  t.ymid.ensure(NN * sizeof(double));
  t.row.ensure(NN * sizeof(int));
  t.m2l.ensure((int64_t)NN * kNumM2L * sizeof(int));
  t.evalid.ensure(NN * sizeof(int));
  t.evalnode.ensure((n_eval + 1) * sizeof(int));
  t.upnodes.ensure((n_eval + 1) * sizeof(int));
  t.rowinfo.ensure((n_rows + 1) * sizeof(int2));
}

static void tree_full_kernels(Tree& t, int D, int npts, hipStream_t s, const int* gate) {
  const int NN = full_levoff(D + 1);
  int* start = t.w_flag.as<int>();
  hipLaunchKernelGGL(k_full_starts, dim3(grid_for(npts)), dim3(BS), 0, s, t.keys.as<uint64_t>(),
                     t.w_a.as<int2>(), npts, D, start, gate);
  FMM_LAUNCH_CHECK();
  // levels 0 and 1 have no M2L lists (their entries are never read), as in
  // the general build
  hipLaunchKernelGGL(k_full_nodes, dim3(grid_for((int64_t)NN * kFullLanes)), dim3(BS), 0, s, D, NN,
                     start,
                     t.keys.as<uint64_t>(), npts, t.xmin, t.ymin, t.w0, t.code.as<uint64_t>(),
                     t.nlevel.as<int>(), t.flags.as<int>(), t.bot.as<int>(), t.top.as<int>(),
                     t.parent.as<int>(), t.child.as<int>(), t.coll.as<int>(), t.crange.as<int2>(),
                     t.xmid.as<double>(), t.ymid.as<double>(), t.row.as<int>(), t.m2l.as<int>(),
                     t.evalid.as<int>(), t.evalnode.as<int>(), t.upnodes.as<int>(),
                     t.rowinfo.as<int2>(), gate);
  FMM_LAUNCH_CHECK();
}

static void tree_full_host(Tree& t, int D) {
  const int L = D + 1;
  t.L = L;
  t.lev.assign(L, TreeLevel());
  for (int d = 0; d < L; ++d) {
    t.lev[d].node_off = full_levoff(d);
    t.lev[d].n_nodes = (int64_t)1 << (2 * d);
    t.lev[d].width = std::ldexp(t.w0, -d);
  }
  const int NN = full_levoff(L);
  t.n_nodes = NN;
  const int g0 = full_levoff(2);
  t.n_rows = NN - g0;
  t.row_off.assign(L + 1, 0);
  for (int d = 0; d <= L; ++d) t.row_off[d] = d <= 2 ? 0 : full_levoff(d) - g0;
  t.n_eval = (int64_t)1 << (2 * D);
  t.n_up = t.n_eval;
  t.nidx_off.assign(kMaxLevels, -1);
  t.bm_index = false;
  t.complete = true;
  t.full_D = D;
  ++t.build_id;
  t.built = true;
}

// Device counters c[0 .. n) into the host mailbox, for read_counts.
__global__ __launch_bounds__(128) void k_counts_to_mailbox(const int* __restrict__ c, int n,
                                                           uint64_t* __restrict__ mbox,
                                                           uint32_t seq) {
  for (int i = threadIdx.x; i < n; i += 128) mailbox_put(mbox, i, seq, c[i]);
}

// host[0 .. n) = the device counters dev[0 .. n) once the work queued on s
// before this call has run, without draining s (HostMailbox).
static void read_counts(Tree& t, const int* dev, int n, int* host, hipStream_t s) {
  HostMailbox& mb = t.pw.mbox;
  mb.ensure();
  const uint32_t seq = mb.next();
  hipLaunchKernelGGL(k_counts_to_mailbox, dim3(1), dim3(128), 0, s, dev, n, mb.dev, seq);
  FMM_LAUNCH_CHECK();
  int64_t v[HostMailbox::kWords];
  mb.take(n, seq, s, v);
  for (int i = 0; i < n; ++i) host[i] = (int)v[i];
}

// Device counters of a build.
enum { CNT_R = 0, CNT_UNIQ = 1, CNT_PC = 2, CNT_BAL = CNT_PC + kMaxLevels,
       CNT_SPLIT = CNT_BAL + kMaxLevels, CNT_ALL = CNT_SPLIT + kSplitRows * (kMaxLevels + 1) };

// Nodes with children (p_code, p_kind, p_off) of a tree of more than kBmLevels
// levels: sorted code lists per depth, dcount[d] of them split and np split
// positions.
static void tree_split_lists(Tree& t, const int64_t* dcount, int np, hipStream_t s) {
  const int L = t.L, nn = (int)t.n;
  const int64_t n = t.n;
  const uint64_t* keys = t.keys.as<uint64_t>();
  const int2* sc = t.w_a.as<int2>();
  int* cnt = t.w_cnt.as<int>();
  int hc[CNT_SPLIT] = {};
  // Small host->device uploads go through distinct regions of a pinned buffer
  // so that the host never rewrites memory a queued copy still reads.
  constexpr int kUpRegion = kMaxLevels + 2;
  t.h_up.ensure(4 * kUpRegion * sizeof(int64_t));
  int64_t* hup = t.h_up.as<int64_t>();
  int up_region = 0;
  auto upload = [&](void* dst, const void* src, size_t bytes) {
    FMM_REQUIRE(up_region < 4 && bytes <= kUpRegion * sizeof(int64_t), FMM_E_INTERNAL,
                "tree: upload staging exhausted");
    int64_t* slot = hup + (int64_t)up_region * kUpRegion;
    ++up_region;
    std::memcpy(slot, src, bytes);
    FMM_HIP(hipMemcpyAsync(dst, slot, bytes, hipMemcpyHostToDevice, s));
  };

  // compacted split positions and the split-cell lists per depth (S_ref)
  t.w_flag.ensure(n * sizeof(int));
  t.w_rank.ensure(n * sizeof(int));
  int* flag = t.w_flag.as<int>();
  int* rank = t.w_rank.as<int>();
  hipLaunchKernelGGL(k_split_flags, dim3(grid_for(n)), dim3(BS), 0, s, sc, nn, flag);
  FMM_LAUNCH_CHECK();
  exclusive_scan_i32(flag, rank, n, nullptr, t.pw, s);
  t.w_c.ensure((int64_t)(n + 2) * (sizeof(int) + sizeof(int2)) + 16);
  int* ppos = t.w_c.as<int>();
  int2* psc = reinterpret_cast<int2*>(ppos + n + (n & 1));
  hipLaunchKernelGGL(k_compact_pos, dim3(grid_for(n)), dim3(BS), 0, s, flag, rank, sc, nn, ppos,
                     psc);
  FMM_LAUNCH_CHECK();
  t.s_off.assign(L + 1, 0);
  for (int d = 0; d < L; ++d) t.s_off[d + 1] = t.s_off[d] + (d <= L - 2 ? dcount[d] : 0);
  const int64_t ns_total = t.s_off[L];
  t.w_b.ensure((L + 1) * sizeof(int64_t) * 2 + 64);
  int64_t* d_soff = t.w_b.as<int64_t>();
  t.sref_all.ensure((ns_total + 1) * sizeof(uint64_t));
  if (np > 0) {
    upload(d_soff, t.s_off.data(), (L + 1) * sizeof(int64_t));
    hipLaunchKernelGGL(k_depth_lists, dim3(L - 1), dim3(1024), 0, s, ppos, psc, np, keys, d_soff,
                       t.sref_all.as<uint64_t>());
    FMM_LAUNCH_CHECK();
  }

  // -- 2:1 balance ---------------------------------------------------------------
  bool balanced = true;
  if (L >= 4) {
    int64_t ne = t.s_off[L - 1] - t.s_off[2];
    // the check looks for neighbours of split cells' parents (depths 1 .. L-3)
    // that are not split themselves; with every cell of those depths split
    // there is none
    bool full = true;
    for (int d = 1; d <= L - 3 && full; ++d)
      full = d < 31 && t.s_off[d + 1] - t.s_off[d] == ((int64_t)1 << (2 * d));
    if (ne > 0 && !full) {
      hipLaunchKernelGGL(k_balance_check, dim3(grid_for(ne)), dim3(BS), 0, s,
                         t.sref_all.as<uint64_t>(), d_soff, L, cnt + CNT_R);
      FMM_LAUNCH_CHECK();
      read_counts(t, cnt + CNT_R, 1, hc + CNT_R, s);
      balanced = hc[CNT_R] == 0;
    }
  }
  std::vector<int64_t> soff = t.s_off;
  if (balanced) {
    t.s_all.ensure((ns_total + 1) * sizeof(uint64_t));
    if (ns_total > 0)
      FMM_HIP(hipMemcpyAsync(t.s_all.ptr, t.sref_all.ptr, ns_total * sizeof(uint64_t),
                             hipMemcpyDeviceToDevice, s));
  } else {
    // Bottom-up: S_d = Sref_d u N(parents(S_{d+1})) for d = L-3 .. 1, with
    // S_0 = Sref_0 and S_{L-2} = Sref_{L-2}.  Depths above kBmDepth (very deep
    // trees) build sorted candidate lists; the others are bitmaps.
    const int DM = std::min(L - 3, kBmDepth);
    std::vector<int64_t> sz(L, 0);
    for (int d = 0; d < L; ++d) sz[d] = t.s_off[d + 1] - t.s_off[d];
    const uint64_t* sref = t.sref_all.as<uint64_t>();
    std::vector<DevBuf>& lists = t.bal_lists;
    if ((int)lists.size() < L) lists.resize(L);
    for (int d = L - 3; d > DM; --d) {
      const uint64_t* nxt = d + 1 == L - 2 ? sref + t.s_off[L - 2] : lists[d + 1].as<uint64_t>();
      const int64_t nref = sz[d];
      const int64_t nnext = sz[d + 1];
      const int64_t nc = nref + 9 * nnext;
      t.bal_k.ensure((nc + 1) * sizeof(uint64_t));
      t.bal_v.ensure((nc + 1) * sizeof(uint32_t));
      t.bal_f.ensure((nc + 1) * 2 * sizeof(int));
      uint64_t* candk = t.bal_k.as<uint64_t>();
      int* fl = t.bal_f.as<int>();
      int* rk = fl + (nc + 1);
      hipLaunchKernelGGL(k_bal_candidates, dim3(grid_for(nc)), dim3(BS), 0, s,
                         sref + t.s_off[d], nref, nxt, nnext, d, candk, t.bal_v.as<uint32_t>());
      FMM_LAUNCH_CHECK();
      sort_pairs_u64(candk, t.bal_v.as<uint32_t>(), nc, 1024, t.pw, s, 2 * d);
      hipLaunchKernelGGL(k_unique_flags, dim3(grid_for(nc)), dim3(BS), 0, s, candk, nc, fl);
      FMM_LAUNCH_CHECK();
      exclusive_scan_i32(fl, rk, nc, cnt + CNT_UNIQ, t.pw, s);
      read_counts(t, cnt + CNT_UNIQ, 1, hc + CNT_UNIQ, s);
      sz[d] = hc[CNT_UNIQ];
      lists[d].ensure((sz[d] + 1) * sizeof(uint64_t));
      hipLaunchKernelGGL(k_unique_scatter, dim3(grid_for(nc)), dim3(BS), 0, s, candk, fl, rk, nc,
                         d, lists[d].as<uint64_t>());
      FMM_LAUNCH_CHECK();
    }
    BmOffsets bo{};
    int64_t nwords = 0;
    for (int d = 1; d <= DM; ++d) {
      bo.wo[d] = nwords;
      const int64_t w = std::max<int64_t>(1, ((int64_t)1 << (2 * d)) / 32);
      nwords += ceil_div(w, BS) * BS;
    }
    bo.wo[DM + 1] = nwords;
    if (DM >= 1) {
      t.bal_bm.ensure(nwords * sizeof(uint32_t));
      t.bal_pc.ensure(nwords * sizeof(int));
      uint32_t* bm = t.bal_bm.as<uint32_t>();
      FMM_HIP(hipMemsetAsync(bm, 0, nwords * sizeof(uint32_t), s));
      const int64_t nmark = t.s_off[DM + 1] - t.s_off[1];
      if (nmark > 0) {
        hipLaunchKernelGGL(k_bm_mark, dim3(grid_for(nmark)), dim3(BS), 0, s, sref, d_soff, DM, bo,
                           bm);
        FMM_LAUNCH_CHECK();
      }
      for (int d = DM; d >= 1; --d) {
        if (d + 1 <= DM) {
          const int64_t npar = (int64_t)1 << (2 * d);   // depth-d cells
          if (npar <= ((int64_t)1 << 22))
            hipLaunchKernelGGL(k_bm_spread, dim3(grid_for(npar)), dim3(BS), 0, s,
                               bm + bo.wo[d + 1], d, bm + bo.wo[d]);
          else
            hipLaunchKernelGGL(k_bm_spread_w, dim3(grid_for(npar / 8)), dim3(BS), 0, s,
                               bm + bo.wo[d + 1], d, bm + bo.wo[d]);
        } else {
          const uint64_t* lst =
              d + 1 == L - 2 ? sref + t.s_off[L - 2] : lists[d + 1].as<uint64_t>();
          if (sz[d + 1] == 0) continue;
          hipLaunchKernelGGL(k_bm_spread_list, dim3(grid_for(sz[d + 1])), dim3(BS), 0, s, lst,
                             sz[d + 1], d, bm + bo.wo[d]);
        }
        FMM_LAUNCH_CHECK();
      }
      hipLaunchKernelGGL(k_bm_count, dim3(nwords / BS), dim3(BS), 0, s, bm, bo, DM,
                         t.bal_pc.as<int>(), cnt + CNT_BAL);
      FMM_LAUNCH_CHECK();
      exclusive_scan_i32(t.bal_pc.as<int>(), t.bal_pc.as<int>(), nwords, nullptr, t.pw, s);
      read_counts(t, cnt + CNT_BAL, kMaxLevels, hc + CNT_BAL, s);
    }
    for (int d = 1; d <= DM; ++d) sz[d] = hc[CNT_BAL + d];
    soff.assign(L + 1, 0);
    for (int d = 0; d < L; ++d) soff[d + 1] = soff[d] + (d <= L - 2 ? sz[d] : 0);
    t.s_all.ensure((soff[L] + 1) * sizeof(uint64_t));
    uint64_t* sall = t.s_all.as<uint64_t>();
    if (sz[0] > 0)
      FMM_HIP(hipMemcpyAsync(sall, sref, sz[0] * sizeof(uint64_t), hipMemcpyDeviceToDevice, s));
    if (DM >= 1 && soff[DM + 1] > soff[1]) {
      hipLaunchKernelGGL(k_bm_scatter, dim3(nwords / BS), dim3(BS), 0, s, t.bal_bm.as<uint32_t>(),
                         bo, DM, t.bal_pc.as<int>(), sall + soff[1]);
      FMM_LAUNCH_CHECK();
    }
    for (int d = DM + 1; d <= L - 3; ++d)
      if (sz[d] > 0)
        FMM_HIP(hipMemcpyAsync(sall + soff[d], lists[d].ptr, sz[d] * sizeof(uint64_t),
                               hipMemcpyDeviceToDevice, s));
    if (L - 2 >= 1 && sz[L - 2] > 0)
      FMM_HIP(hipMemcpyAsync(sall + soff[L - 2], sref + t.s_off[L - 2],
                             sz[L - 2] * sizeof(uint64_t), hipMemcpyDeviceToDevice, s));
  }

  // -- nodes with children (P_d = S_d u X_d) ----------------------------------------
  std::vector<int64_t> roff(L + 1, 0);
  roff[1] = 1;
  for (int d = 1; d < L; ++d) roff[d + 1] = roff[d] + 4 * (soff[d] - soff[d - 1]);
  const int64_t nr = roff[L];
  int64_t* d_soff2 = d_soff;
  int64_t* d_roff = d_soff + (L + 1);
  upload(d_soff2, soff.data(), (L + 1) * sizeof(int64_t));
  upload(d_roff, roff.data(), (L + 1) * sizeof(int64_t));
  t.w_c.ensure(nr * (sizeof(uint64_t) + 3 * sizeof(int)) + 64);
  uint64_t* rcode = t.w_c.as<uint64_t>();
  int* hasc = reinterpret_cast<int*>(rcode + nr);
  int* kind = hasc + nr;
  int* rrank = kind + nr;
  hipLaunchKernelGGL(k_real_flags, dim3(grid_for(nr)), dim3(BS), 0, s, t.s_all.as<uint64_t>(),
                     d_soff2, d_roff, L, rcode, hasc, kind, cnt + CNT_PC);
  FMM_LAUNCH_CHECK();
  exclusive_scan_i32(hasc, rrank, nr, nullptr, t.pw, s);
  read_counts(t, cnt + CNT_PC, kMaxLevels, hc + CNT_PC, s);
  t.p_off.assign(L + 1, 0);
  for (int d = 0; d < L; ++d) t.p_off[d + 1] = t.p_off[d] + hc[CNT_PC + d];
  FMM_REQUIRE(hc[CNT_PC + L - 1] == 0, FMM_E_INTERNAL, "tree: deepest level has children");
  const int64_t np_total = t.p_off[L];
  t.p_code.ensure((np_total + 1) * sizeof(uint64_t));
  t.p_kind.ensure((np_total + 1) * sizeof(int));
  hipLaunchKernelGGL(k_p_scatter, dim3(grid_for(nr)), dim3(BS), 0, s, rcode, hasc, kind, rrank, nr,
                     t.p_code.as<uint64_t>(), t.p_kind.as<int>());
  FMM_LAUNCH_CHECK();
}

// The node arrays of the levels lv from the cells' lookups (codes, levels and
// fake flags of the nodes are set): point ranges, records, lists, and the
// host's counts, which it reads while the last kernel runs.
template <class Cells>
static void node_arrays(Tree& t, const Cells& cells, const LevOff& lv, int g0, int nw, int* rb,
                        int* rt, int* wcnt, hipStream_t s) {
  const int L = t.L, NN = (int)t.n_nodes;
  hipLaunchKernelGGL(k_cell_ranges<Cells>, dim3(grid_for(t.n)), dim3(BS), 0, s,
                     t.keys.as<uint64_t>(), t.w_a.as<int2>(), (int)t.n, cells, L, rb, rt);
  FMM_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_nodes<Cells>, dim3(nw), dim3(64), 0, s, cells, lv, L, rb, rt, t.xmin, t.ymin,
                     t.w0, t.code.as<uint64_t>(), t.flags.as<int>(), t.bot.as<int>(),
                     t.top.as<int>(), t.parent.as<int>(), t.child.as<int>(), t.coll.as<int>(),
                     t.xmid.as<double>(), t.ymid.as<double>(), g0, nw, wcnt);
  FMM_LAUNCH_CHECK();
  const bool scanned = nw > kSumWaves;
  if (scanned)
    for (int q = 0; q < 3; ++q)
      exclusive_scan_i32(wcnt + (int64_t)q * nw, wcnt + (int64_t)q * nw, nw, nullptr, t.pw, s);
  HostMailbox& mb = t.pw.mbox;
  const uint32_t seq = mb.next();
  hipLaunchKernelGGL(k_node_lists, dim3((unsigned)ceil_div(nw, 16)), dim3(1024), 0, s,
                     t.flags.as<int>(), lv, L, g0, nw, wcnt, scanned ? 1 : 0, t.evalid.as<int>(),
                     t.evalnode.as<int>(), t.upnodes.as<int>(), t.row.as<int>(), mb.dev, seq);
  FMM_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_node_slots<Cells>, dim3(grid_for((int64_t)NN * kSlotLanes)), dim3(BS), 0, s,
                     cells, lv, L, t.code.as<uint64_t>(), t.nlevel.as<int>(), t.flags.as<int>(),
                     t.row.as<int>(), t.child.as<int>(), t.coll.as<int>(), t.bot.as<int>(), t.top.as<int>(),
                     t.m2l.as<int>(), t.m2lmask.as<uint64_t>(), t.crange.as<int2>(),
                     t.rowinfo.as<int2>());
  FMM_LAUNCH_CHECK();
  int64_t v[3 + kMaxLevels];
  mb.take(3 + std::max(0, L - 2), seq, s, v);
  t.n_eval = v[0];
  t.n_up = v[1];
  t.n_rows = 4 * v[2];
  t.row_off.assign(L + 1, 0);
  for (int d = 2; d < L; ++d) t.row_off[d] = v[3 + d - 2];
  t.row_off[L] = t.n_rows;
}

// ---------------------------------------------------------------------------
void tree_build(Tree& t, const double* x, const double* y, int64_t n, double xmin, double ymin,
                double w0, int ncut, hipStream_t s) {
  FMM_REQUIRE(n >= 1 && n < ((int64_t)1 << 31) - 1, FMM_E_LIMIT,
              "tree: number of sources %lld outside [1, 2^31-2]", (long long)n);
  FMM_REQUIRE(ncut >= 1, FMM_E_ARG, "tree: Ncutoff must be >= 1 (got %d)", ncut);
  FMM_REQUIRE(w0 > 0.0 && std::isfinite(w0), FMM_E_ARG, "tree: root width must be positive");
  t.built = false;
  t.complete = false;
  t.n = n;
  t.ncut = ncut;
  t.xmin = xmin;
  t.ymin = ymin;
  t.w0 = w0;
  const int nn = (int)n;

  // -- sorted points ----------------------------------------------------------
  t.keys.ensure(n * sizeof(uint64_t));
  t.perm.ensure(n * sizeof(uint32_t));
  t.sx.ensure(n * sizeof(double));
  t.sy.ensure(n * sizeof(double));
  uint64_t* keys = t.keys.as<uint64_t>();
  uint32_t* perm = t.perm.as<uint32_t>();
  t.xy.ensure(n * sizeof(double2));
  // -- counters (zeroed by the first kernel)
  t.w_cnt.ensure(CNT_ALL * sizeof(int));
  int* cnt = t.w_cnt.as<int>();
  const int nkey_blk = (int)ceil_div(n, kSortChunk);
  t.w_bad.ensure(nkey_blk * sizeof(int));
  const int sort_T = ncut < kLocalSortMax ? ncut : kLocalSortMax;
  const bool first_round = n > sort_T;
  const SortFirstRound fr = first_round ? sort_first_round(t.pw, n) : SortFirstRound{};
  hipLaunchKernelGGL(k_point_keys, dim3((unsigned)ceil_div(n, kSortChunk)), dim3(KEY_BS), 0, s, x, y,
                     nn, xmin, ymin, w0, key_scale(xmin, ymin, w0),
                     first_round ? fr.keys : keys, first_round ? fr.vals : perm,
                     t.xy.as<double2>(), t.w_bad.as<int>(), cnt, (int)CNT_ALL, fr,
                     first_round ? 1 : 0);
  FMM_LAUNCH_CHECK();
  // Segments of at most Ncutoff points that end in the last radix round sit
  // at the deepest radix depth D, which no cell of the tree goes below (2:1
  // balance splits lie at least two levels above the deepest leaf, X-list
  // children at most at depth D): the radix order within them stands.
  // Segments that end earlier are sorted, since balance and X-list children
  // can split their cells further.
  sort_pairs_u64(keys, perm, n, sort_T, t.pw, s, 64, true, first_round);

  // -- split cells of the refinement --------------------------------------------
  t.w_a.ensure(n * sizeof(int2));
  int2* sc = t.w_a.as<int2>();
  hipLaunchKernelGGL(k_split_pos, dim3((unsigned)ceil_div(n, 1024)), dim3(1024), 0, s, keys, nn,
                     ncut, sc, cnt + CNT_SPLIT, perm, t.xy.as<double2>(), t.sx.as<double>(),
                     t.sy.as<double>());
  FMM_LAUNCH_CHECK();
  // per depth, then the split positions; then the non-finite flag
  int64_t dcount[kMaxLevels + 2];
  // A complete tree of the previous build's depth is built at once, gated on
  // the device by the split counts (its kernels then follow without waiting
  // for the host to read them).  Otherwise the split cells go into the bitmaps
  // of an adaptive tree meanwhile.
  const int specD = t.full_D;
  const bool spec = t.allow_full && specD >= 2 && specD <= kFullMaxDepth;
  auto mark_split_cells = [&] {
    t.bm.ensure(kBmWords * sizeof(uint32_t));
    fill_i32(t.bm.as<int>(), kBmWords, 0, s);
    hipLaunchKernelGGL(k_bm_mark_points, dim3(grid_for(n)), dim3(BS), 0, s, keys, sc, nn,
                       t.bm.as<uint32_t>());
    FMM_LAUNCH_CHECK();
  };
  {
    HostMailbox& mb = t.pw.mbox;
    mb.ensure();
    const uint32_t seq = mb.next();
    int* gate = nullptr;
    if (spec) {
      t.w_gate.ensure(sizeof(int));
      gate = t.w_gate.as<int>();
      tree_full_buffers(t, specD);
    }
    hipLaunchKernelGGL(k_split_counts, dim3(1), dim3(64), 0, s, cnt + CNT_SPLIT,
                       t.w_bad.as<int>(), nkey_blk, mb.dev, seq, specD, gate);
    FMM_LAUNCH_CHECK();
    if (spec) tree_full_kernels(t, specD, nn, s, gate);
    else mark_split_cells();
    mb.take(kMaxLevels + 2, seq, s, dcount);
  }
  FMM_REQUIRE(dcount[kMaxLevels + 1] == 0, FMM_E_ARG,
              "tree: the source coordinates hold a NaN or infinite value");
  const int np = (int)dcount[kMaxLevels];
  int maxd = -1;
  for (int d = 0; d < kMaxLevels; ++d)
    if (dcount[d] > 0) maxd = d;
  const int L = maxd + 2;   // deepest split depth + children level + 1
  t.L = L;
  FMM_REQUIRE(L <= kMaxLevels, FMM_E_INTERNAL, "tree: %d levels exceed the depth cap", L);

  // a complete tree (every cell of the depths above the deepest split cells
  // split): closed forms of the node arrays (k_full_nodes)
  if (t.allow_full && L >= 3 && L - 1 <= kFullMaxDepth) {
    bool complete = true;
    for (int d = 0; d <= L - 2 && complete; ++d) complete = dcount[d] == ((int64_t)1 << (2 * d));
    if (complete) {
      if (!(spec && L - 1 == specD)) {   // else built already
        tree_full_buffers(t, L - 1);
        tree_full_kernels(t, L - 1, nn, s, nullptr);
      }
      tree_full_host(t, L - 1);
      return;
    }
  }
  t.full_D = 0;

  // -- nodes with children (P_d = S_d u X_d) ----------------------------------------
  t.bm_index = L <= kBmLevels;
  if (t.bm_index) {
    if (spec) mark_split_cells();   // else marked already
    t.p_off.assign(L + 1, 0);
    t.bm_pp.ensure(kBmWords * sizeof(uint2));
    t.bm_boff.ensure(kBmBlocks * sizeof(int));
    uint32_t* bm = t.bm.as<uint32_t>();
    for (int d = L - 3; d > kBmLowD; --d) {
      hipLaunchKernelGGL(k_bm_balance, dim3(grid_for(bm_words(d))), dim3(BS), 0, s, d, bm);
      FMM_LAUNCH_CHECK();
    }
    if (L >= 4) {
      hipLaunchKernelGGL(k_bm_balance_low, dim3(1), dim3(1024), 0, s, std::min(L - 3, kBmLowD), bm);
      FMM_LAUNCH_CHECK();
    }
    if (L >= 2) {
      HostMailbox& mb = t.pw.mbox;
      const uint32_t seq = mb.next();
      hipLaunchKernelGGL(k_bm_parents, dim3(bm_wo(L - 1) / BS), dim3(BS), 0, s, bm, L - 2,
                         t.bm_pp.as<uint2>(), t.bm_boff.as<int>());
      FMM_LAUNCH_CHECK();
      hipLaunchKernelGGL(k_bm_sums, dim3(1), dim3(1024), 0, s, t.bm_boff.as<int>(), L - 2, mb.dev,
                         seq);
      FMM_LAUNCH_CHECK();
      mb.take(L, seq, s, t.p_off.data());
      t.p_off[L] = t.p_off[L - 1];
    }
  } else {
    tree_split_lists(t, dcount, np, s);
  }

  // -- final node arrays ------------------------------------------------------------
  t.lev.assign(L, TreeLevel());
  LevOff lv{};
  int64_t off = 0;
  for (int d = 0; d < L; ++d) {
    int64_t nd = d == 0 ? 1 : 4 * (t.p_off[d] - t.p_off[d - 1]);
    t.lev[d].node_off = off;
    t.lev[d].n_nodes = nd;
    t.lev[d].width = std::ldexp(w0, -d);
    lv.lo[d] = (int)off;
    off += nd;
    FMM_REQUIRE(off < ((int64_t)1 << 31) / kNumM2L, FMM_E_LIMIT, "tree: too many nodes (%lld)",
                (long long)off);
  }
  lv.lo[L] = (int)off;
  t.n_nodes = off;
  t.nidx_off.assign(kMaxLevels, -1);
  const int NN = (int)off;
  const int g0 = L > 2 ? lv.lo[2] : NN;
  const int ngroups = (NN - g0) / 4;
  const int nw = (int)ceil_div(wave_slots(NN), 64);
  t.code.ensure(off * sizeof(uint64_t));
  t.nlevel.ensure(off * sizeof(int));
  t.bot.ensure(off * sizeof(int));
  t.top.ensure(off * sizeof(int));
  t.parent.ensure(off * sizeof(int));
  t.child.ensure(off * sizeof(int));
  t.flags.ensure(off * sizeof(int));
  t.coll.ensure(off * 9 * sizeof(int));
  t.crange.ensure((off * 9 + 1) * sizeof(int2));
  t.xmid.ensure(off * sizeof(double));
  t.ymid.ensure(off * sizeof(double));
  t.row.ensure(off * sizeof(int));
  t.rowinfo.ensure((4 * (int64_t)ngroups + 1) * sizeof(int2));
  t.m2l.ensure(off * kNumM2L * sizeof(int));
  t.m2lmask.ensure(off * sizeof(uint64_t));
  t.evalid.ensure(off * sizeof(int));
  t.evalnode.ensure(off * sizeof(int));
  t.upnodes.ensure(off * sizeof(int));
  t.w_rng.ensure(2 * off * sizeof(int));
  t.w_wave.ensure(3 * (int64_t)nw * sizeof(int));
  int* rb = t.w_rng.as<int>();
  int* rt = rb + off;
  int* wcnt = t.w_wave.as<int>();
  if (t.bm_index) {
    const BmCells cells{t.index(), t.bm.as<uint32_t>()};
    hipLaunchKernelGGL(k_bm_nodes, dim3(grid_for(8 * (int64_t)bm_wo(L - 1))), dim3(BS), 0, s,
                       cells, L - 2, nn, t.code.as<uint64_t>(), t.nlevel.as<int>(),
                       t.flags.as<int>(), rb, rt);
    FMM_LAUNCH_CHECK();
    node_arrays(t, cells, lv, g0, nw, rb, rt, wcnt, s);
  } else {
    ListCells cells{};
    int64_t ntab = 0;
    for (int d = 0; d < kMaxLevels; ++d) cells.off[d] = -1;
    for (int d = 1; d < L && d <= kIdxDepth; ++d) {
      if (t.lev[d].n_nodes == ((int64_t)1 << (2 * d))) continue;   // full: direct
      cells.off[d] = ntab;
      ntab += (int64_t)1 << (2 * d);
    }
    t.nidx_off.assign(cells.off, cells.off + kMaxLevels);
    t.nidx.ensure(ntab * sizeof(int));
    fill_i32(t.nidx.as<int>(), ntab, -1, s);
    cells.code = t.code.as<uint64_t>();
    cells.lv = lv;
    cells.tab = t.nidx.as<int>();
    cells.p_code = t.p_code.as<uint64_t>();
    cells.p_kind = t.p_kind.as<int>();
    hipLaunchKernelGGL(k_list_nodes, dim3(grid_for(off)), dim3(BS), 0, s, cells, L, nn,
                       t.code.as<uint64_t>(), t.nlevel.as<int>(), t.flags.as<int>(), rb, rt,
                       t.nidx.as<int>());
    FMM_LAUNCH_CHECK();
    node_arrays(t, cells, lv, g0, nw, rb, rt, wcnt, s);
  }
  ++t.build_id;
  t.built = true;
}

void tree_init_device() {
  SlotOffsets so;
  for (int q = 0; q < kNumM2L; ++q) {
    m2l_slot_offset(q, &so.ox[q], &so.oy[q]);
    so.dx[q] = morton((uint32_t)so.ox[q], 0);
    so.dy[q] = morton(0, (uint32_t)so.oy[q]);
  }
  FMM_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_slot_off), &so, sizeof so));
}

void tree_locate(const Tree& t, const double* tx, const double* ty, int64_t nt, int* out_node,
                 hipStream_t s) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_locate, dim3(grid_for(nt)), dim3(BS), 0, s, tx, ty, nt, t.flags.as<int>(),
                     t.child.as<int>(), t.xmid.as<double>(), t.ymid.as<double>(), out_node);
  FMM_LAUNCH_CHECK();
}

}  // namespace fmm
