// bwl_metro_alone.hip -- small chains of the parallel Metropolis sampler, one
// site per lane in one workgroup.
//
// k_metro_nat gives a lane a whole pair: both sites' gathers, 2 z of them, in
// one lane, while a round of a small box has too few pairs to fill a CU's
// SIMDs.  Here lane i gathers the grid-1 site of pair i and lane i + 32 its
// grid-2 site, a wavefront takes 32 pairs, and each lane stores its own site's
// new species (no pair's neighbours hold another pair's sites, so a round needs
// one barrier).  The next round's sites and random numbers are formed behind
// the swaps.  The chain of a round's steps bounds it: fcc 8^3, 2 shells, 74 ->
// 60 us a sweep; fcc 10^3, 4 shells, 183 -> 117; bcc 12^3, 3 shells, 58 -> 47.
// The chain is that of k_metro_nat bit for bit, as in bwl_metro_split.hip.
#include "bwl_metro_split.h"

namespace bwl {

namespace {

template <int LAT, int R, typename CW, int NC, int FIELD>
__global__ __launch_bounds__(kSplitThreads) void k_metro_alone(const ParArgs *__restrict__ chains) {
  extern __shared__ __align__(16) uint8_t smem[];
  metro_split<LAT, R, CW, NC, FIELD, true>(chains[blockIdx.x], 0, smem);
}

template <int LAT, int R>
const void *alone_of(int words) {
  if (words == 0) return (const void *)k_metro_alone<LAT, R, uint32_t, kFixedPitch, 8>;
  if (words == 1) return (const void *)k_metro_alone<LAT, R, uint32_t, kFixedPitch, 6>;
  return (const void *)k_metro_alone<LAT, R, uint64_t, kFixedPitch, 8>;
}

}  // namespace

const void *par_alone_kernel(const Geo &g, bool fixed) {
  const int words = par_count_words(g, true);
  // the shape with its own pitch has no other layout in lattice coordinates;
  // 400 sweeps of fcc 8^3 take 23.0 ms so, 24.6 at the fixed pitch
  if (!fixed)
    return words == 0 && g.lattice == 1 && g.R == 2 && g.n[0] == 8 ? (const void *)k_metro_alone<1, 2, uint32_t, 8, 8>
                                                                  : nullptr;
  switch (g.lattice * 8 + g.R) {
    case 8 + 1: return alone_of<1, 1>(words);
    case 8 + 2: return alone_of<1, 2>(words);
    case 8 + 3: return alone_of<1, 3>(words);
    case 8 + 4: return alone_of<1, 4>(words);
    case 16 + 1: return alone_of<2, 1>(words);
    case 16 + 2: return alone_of<2, 2>(words);
    case 16 + 3: return alone_of<2, 3>(words);
    case 16 + 4: return alone_of<2, 4>(words);
  }
  return nullptr;
}

int par_alone_threads(int threads, int passes) {
  const int units = 2 * (threads / 64) * passes;
  return units <= kUnits ? 64 * units : 0;
}

}  // namespace bwl
