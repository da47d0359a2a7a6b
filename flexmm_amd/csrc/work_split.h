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

}  // namespace fmm
