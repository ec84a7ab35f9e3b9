// bwl_metro_split.hip -- one chain of the parallel Metropolis sampler run by
// several workgroups (CUs), for lattices held at the fixed pitch or at a
// shape's own compile-time pitch.
//
// A round of k_metro_nat is bound by one CU's instruction issue (24
// wavefronts of pairs on four SIMDs): 5.2 us for bcc 32^3 with four shells,
// 2.4 here in 16 parts, of which the evaluation takes 1.0 (58 gathers from
// LDS a site), the exchange 1.0 and the swaps 0.35; the anneal of 1200 sweep
// rounds goes from 47.4 to 20.5 ms, fcc 24^3 with three shells from 12.3 to
// 7.4.  Here every part (workgroup) of a chain
// holds the whole lattice in its LDS, evaluates its share of a round's pairs
// and publishes the swaps it accepted, one 64-bit record each, in device
// memory; every part then makes all of the round's swaps on its own copy.
// A record holds both sites' natural coordinates and species beside a tag
// that counts the rounds, and each half row of pairs has a header with its
// tag and count, so a reader polls the data themselves: the exchange is one
// store and one load deep, with no barrier and no flag of its own.  Parts on
// one XCD share its L2, where a plain store is seen by the others' loads past
// L1: 0.49 us a round for 8 parts, a workgroup barrier included, against 0.71
// with stores at device scope (0.90 across XCDs), which are used when the
// parts find themselves on different XCDs; an atomic counter with acquire and
// release took 1.4 us.  A part packs its records side by side, so a wavefront
// reads a whole part's, or two parts', at once.
// While the records travel, each wavefront forms its next pairs' sites and
// random numbers, which depend on no state.
//
// The chain is that of k_metro_nat bit for bit: pairs belong to the same
// threads (virtual thread q mod nthr takes pairs q, q + nthr, ...), draw the
// same numbers, and the accepted energy changes are summed per virtual thread
// in the order of rounds and pairs, the sums of 64 virtual threads by the same
// tree, and those in order.  All pairs of 64 consecutive virtual threads (a
// row) belong to one part: row w to part w mod parts.  One wavefront
// evaluates half a row's pass, 32 pairs, one site per lane: lane i the grid-1
// site of pair i, lane i + 32 its grid-2 site.
//
// The parts wait for each other, so all of a chain's parts have to be on the
// device at once: the host asks for no more parts than this process's calls in
// flight leave CUs, every wait ends after a time, that for the parts' arrival
// soonest (the chain is then given up, its configuration untouched, and the
// host runs it undivided), and parts of one chain get block indices that fall
// on one XCD.
#include "bwl_metro_split.h"

namespace bwl {

namespace {

template <int LAT, int R, typename CW, int NC, int FIELD>
__global__ __launch_bounds__(kSplitThreads) void k_metro_split(const ParArgs *__restrict__ chains,
                                                              const int2 *__restrict__ map) {
  extern __shared__ __align__(16) uint8_t smem[];
  const int2 me = map[blockIdx.x];
  if (me.x < 0) return;
  metro_split<LAT, R, CW, NC, FIELD, false>(chains[me.x], me.y, smem);
}

template <int LAT, int R>
const void *split_of(int words) {
  if (words == 0) return (const void *)k_metro_split<LAT, R, uint32_t, kFixedPitch, 8>;
  if (words == 1) return (const void *)k_metro_split<LAT, R, uint32_t, kFixedPitch, 6>;
  return (const void *)k_metro_split<LAT, R, uint64_t, kFixedPitch, 8>;
}

}  // namespace

size_t par_split_lds_bytes(const Geo &g, const NatGeo &nat) {
  const int words = par_count_words(g, true);
  const size_t S1P = words == 0 ? 3 : (words == 1 ? 4 : 7);  // as in fill_tables
  const size_t tables = (size_t)((nat.lds_bytes + 15) & ~15) + sizeof(double) * g.S * g.S * ((g.R * S1P) | 1) +
                        sizeof(double) * g.S * g.R * g.S;
  return ((tables + 15) & ~(size_t)15) + sizeof(SplitRound) * kRoundBatch + sizeof(unsigned long long) * g.S * g.S * g.R +
         sizeof(double) * (3 * 32 * kUnits + 32) + sizeof(uint32_t) * 4 + 16;
}

size_t par_split_mail_words(const Geo &g, int threads, int parts) {
  return 4 * (size_t)parts * kRoundWords + 2 * 2 * (size_t)(threads / 64) + 2 * (size_t)parts * mail_end_words(g.S, g.R) +
         (size_t)parts + 1;
}

bool par_split_fits(const NatGeo &nat, int threads, int parts, int passes) {
  const int rows = threads / 64;
  // coordinates have 7 bits of a record; a wavefront takes one half row
  return nat.D[0] <= 128 && nat.D[1] <= 128 && nat.D[2] <= 128 && rows <= 16 && parts >= 2 && parts <= rows &&
         2 * ((rows + parts - 1) / parts) * passes <= kUnits;
}

hipError_t launch_metro_split(const void *fn, const ParArgs *args_dev, const int2 *map_dev, int blocks, size_t lds,
                              hipStream_t s) {
  void *kargs[] = {(void *)&args_dev, (void *)&map_dev};
  return launch_dynamic(fn, dim3(blocks), kSplitThreads, kargs, lds, s);
}

const void *par_split_kernel(const Geo &g, bool fixed) {
  const int words = par_count_words(g, true);
  if (!fixed) {
    // the shape with its own pitch that has rounds worth dividing: 200 sweeps
    // of bcc 32^3 in 16 parts 19.7 ms so, 21.4 at the fixed pitch
    return words == 0 && g.lattice == 2 && g.R == 4 && g.n[0] == 32
               ? (const void *)k_metro_split<2, 4, uint32_t, 32, 8>
               : nullptr;
  }
  switch (g.lattice * 8 + g.R) {
    case 8 + 1: return split_of<1, 1>(words);
    case 8 + 2: return split_of<1, 2>(words);
    case 8 + 3: return split_of<1, 3>(words);
    case 8 + 4: return split_of<1, 4>(words);
    case 16 + 1: return split_of<2, 1>(words);
    case 16 + 2: return split_of<2, 2>(words);
    case 16 + 3: return split_of<2, 3>(words);
    case 16 + 4: return split_of<2, 4>(words);
  }
  return nullptr;
}

}  // namespace bwl
