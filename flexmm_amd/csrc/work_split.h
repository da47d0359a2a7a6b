// How work is cut into pieces: plain index arithmetic, for the device and the
// host (tests compile it with the host compiler).
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define FMM_SPLIT_HD __host__ __device__ __forceinline__
#else
#define FMM_SPLIT_HD inline
#endif

namespace fmm {

struct Span {
  int b, e;
};
// Part `part` of PARTS of the range [b, e), empty if e <= b.  The product is
// formed in 64 bits: a range may hold up to 2^31 - 2 sources.
template <int PARTS>
FMM_SPLIT_HD Span part_of(int b, int e, int part) {
  const int64_t n = e > b ? e - b : 0;
  return Span{b + (int)(n * part / PARTS), b + (int)(n * (part + 1) / PARTS)};
}

// XCD-aware block order.  MI355X dispatches consecutive workgroups round-robin
// to its 8 XCDs, each with its own L2.  These bijections of [0, n) keep
// neighbouring logical blocks, which share source data, on one XCD (blocks b
// with b % 8 == x): chunk = 0 gives XCD x one contiguous range, chunk > 0
// deals chunks of that many logical blocks to the XCDs in turn (for blocks of
// unequal cost), the remainder past a whole turn in natural order.
constexpr int kNumXcd = 8;
constexpr int kNumCUs = 256;   // MI355X compute units (launch-shape heuristics only)
FMM_SPLIT_HD int xcd_block(int b, int n, int chunk) {
  const int xcd = b % kNumXcd, local = b / kNumXcd;
  if (chunk > 0) {
    if (b >= n / (kNumXcd * chunk) * (kNumXcd * chunk)) return b;
    return (local / chunk * kNumXcd + xcd) * chunk + local % chunk;
  }
  const int per = n / kNumXcd, rem = n % kNumXcd;
  return xcd * per + (xcd < rem ? xcd : rem) + local;
}

// Work items of the evaluation kernels: kEvalWaves waves per block, ns waves
// (1 or kEvalWaves) per item.  chunk = 0: XCD x takes the x-th contiguous
// eighth of the items; chunk > 0 (a multiple of kEvalWaves): chunks of that
// many items go to the XCDs in turn.
constexpr int kEvalWaves = 4;   // waves per block of the evaluation and S2M kernels
// the item of wave `wave` of block `block` among ni, or -1
FMM_SPLIT_HD int xcd_item(unsigned block, int wave, int ni, int chunk, int ns) {
  const int x = block % kNumXcd;
  const int j = ((int)(block / kNumXcd) * kEvalWaves + wave) / ns;
  int first = (int)((int64_t)ni * x / kNumXcd) + j;
  int last = (int)((int64_t)ni * (x + 1) / kNumXcd);
  if (chunk > 0) {
    first = (j / chunk * kNumXcd + x) * chunk + j % chunk;
    last = ni;
  }
  return first < last ? first : -1;
}
// blocks for at most icap items
inline int eval_grid(int64_t icap, int chunk, int ns) {
  const int64_t per_xcd =
      chunk > 0 ? (icap + (int64_t)kNumXcd * chunk - 1) / ((int64_t)kNumXcd * chunk) * chunk
                : (icap + kNumXcd - 1) / kNumXcd + 1;
  return (int)((per_xcd * ns + kEvalWaves - 1) / kEvalWaves * kNumXcd);
}

// Whether boxes with sources (n_up of them) cover a fifth of the root box, each
// counted as one of the deepest level: a uniform set in a root box of up to
// twice its size.
inline bool broad_sources(int levels, int64_t n_up) {
  return levels <= 16 && 5 * n_up >= (int64_t)1 << (2 * (levels - 1));
}

// Whether so few boxes lie above the deepest level that a contiguous eighth of
// the items costs about an eighth.  The boxes come level by level and those
// above hold four times the targets, all in the first eighth: where m boxes of
// the deepest level are missing it costs about 1 + 8m/ne of another.  Measured,
// eighths against chunks: a 1400th missing 199 and 239 us (250K points, mixed,
// self), a 200th 220 and 225, a 93rd 224 and 213, a 16th 335 and 220 (1M points,
// FP64, self).
inline bool even_items(int levels, int64_t ne) {
  return levels <= 16 && 128 * ne >= (int64_t)127 << (2 * (levels - 1));
}

// Few items: the kEvalWaves waves of a block share one; each takes a quarter of
// the L2T terms and of every colleague's sources, and the sums are added in
// wave order through LDS.  One wave per item leaves such a launch bound by its
// load and table latencies (50K points at Ncutoff 500, one item per SIMD: 180 ->
// 81 us; 2,003 points 27 -> 11).  With more items, up to 16 per SIMD, that pays
// only where they hold many sources, since a block's start-up per item (its copy
// of the log table) then costs more than it hides.  Lines in sources per box,
// and shared against not (Laplace; K0, the Stokeslet and the black-box form lie
// around it):
//   self-evaluations kSplitSelf: 100K points of a curve, 54 sources: 0.74; 60K in
//   clusters, 15: 0.65; 30K uniform, 7: 1.08; 64K uniform, 4: 1.6;
//   up to 4 items per SIMD, and broad sources in boxes of several levels (a few
//   items then hold most sources) kSplitUneven: 46K uniform, 27: 0.51; 60K, 16:
//   0.54; 100K, 7: 1.6;
//   where most boxes hold sources kSplitMost: 250K uniform, 61: 0.46; 200K in
//   clusters, 44: 0.74; 100K uniform, 24: 1.0; 300K in clusters, 25: 1.2;
//   elsewhere kSplitAny, as most targets lie beside no sources: 100K on a curve,
//   113: 0.63; 54: 1.4.
// Where most boxes hold few targets or none (a box per 0.5 targets: 15 -> 42
// us), never.  FP32 near fields keep one wave per item (their FP32 runs stay
// whole).
constexpr int64_t kSplitItems = 16 * 4 * kNumCUs;
constexpr int64_t kSplitTargets = 4;   // targets per evaluation box at least
constexpr int64_t kSplitSelf = 9, kSplitUneven = 16, kSplitMost = 32, kSplitAny = 96;
// waves per item: icap items at most, nt targets in ne boxes, n sources in n_up
// S2M boxes of a tree of so many levels
inline int item_waves(int64_t icap, int64_t nt, int64_t ne, int64_t n, int64_t n_up, int levels,
                      bool self) {
  if (nt < kSplitTargets * ne || icap > kSplitItems) return 1;
  int64_t least = kSplitAny;
  if (icap <= kSplitItems / 8) least = 0;
  else if (self) least = kSplitSelf;
  else if (icap <= kSplitItems / 4 || (broad_sources(levels, n_up) && !even_items(levels, ne)))
    least = kSplitUneven;
  else if (2 * n_up >= ne) least = kSplitMost;
  // S2M boxes can outnumber the leaves (their parts beside smaller boxes)
  return n >= least * (n_up < ne ? n_up : ne) ? kEvalWaves : 1;
}

}  // namespace fmm
