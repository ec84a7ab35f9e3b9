// bwl_seq_batches.h -- device code of the bit-exact Metropolis chain in
// speculative batches: in bwl_kernels.hip without the trials taken singly, in
// bwl_seq_singly.hip with them (apart, so that neither's registers are
// allotted beside the other's).
#pragma once

#include "bwl_kernels.h"
#include "bwl_spec.h"

namespace bwl {

// ------------------------------------------------------------------
// Bit-exact Metropolis in speculative batches (bwl_spec.h).  A trial draws its sites'
// numbers and one more when the swap would raise the energy, so where the
// next trial starts is known only with the energy: every lane takes the trial
// that would start at its own place in the stream (64 places), forms its
// energy change and its decision on the lattice as it is, and the batch is
// the chain of 8 trials found by hopping from place to place, cut at the
// first that an accepted swap before it reaches.
//
// On small boxes at high acceptance nearly every batch is cut after a trial or
// two, and a batch costs 1.2 to 3 trials taken one by one (64 places' energies
// in place of one's).  So while batches come out shorter than that, trials are
// taken singly, both sites' neighbours over the lanes and each shell's sum in
// a lane of its own, and a batch is tried again every kSingly of them (SINGLY:
// boxes large enough have a kernel without, see metro_seq_singly_kernel).
//
// A batch takes, one to four shells, 0.8, 1.6, 2.0 and 2.6 us on fcc (0.7,
// 1.2, 1.6 and 3.1 on bcc), a single trial 0.9, 0.9, 1.2 and 1.2 (0.8, 0.8, 1.0
// and 1.2).  20,000 trials at 10^6 K (nothing rejected) of fcc 3^3 with four
// shells: 61.5 ms in batches, 24.1 so (26.7 by k_metro_seq); of bcc 4^3 with
// three 31.9 -> 19.6 (21.0).
// ------------------------------------------------------------------
constexpr int kSingly = 16;
// 8 times the mean length of a batch that is as fast as single trials
template <int KEY>
constexpr uint32_t kBatchPays = KEY % 16 == 4 ? 24 : 17;

template <int KEY>
struct SingleDims {
  using D = SpecDims<KEY>;
  static constexpr int P = (2 * D::Z + 63) / 64;        // entries per lane
  static constexpr int ST = D::ML | 1, NC = 4 * D::R;   // a shell's sum: its slots, and how many sums
  static constexpr int kBytes = 8 * ST * NC;
};

// A lane's entries of a single trial: list positions 0..z-1 of the first
// site's neighbours, then the second's.
template <int KEY>
struct SingleLane {
  int off[SingleDims<KEY>::P];   // of the entry in a sublattice's offsets
  int slot[SingleDims<KEY>::P];  // in the sums' buffer, before the swap
  int row[SingleDims<KEY>::P];   // of the shell in V_ex
  __device__ __forceinline__ void init(int S) {
    using D = SpecDims<KEY>;
#pragma unroll
    for (int k = 0; k < SingleDims<KEY>::P; ++k) {
      const int t = 64 * k + ((int)threadIdx.x & 63), tt = t < D::Z ? t : t - D::Z;
      int n = 0, first = 0;
#pragma unroll
      for (int q = 1; q < D::R; ++q)
        if (tt >= shell_first<D::LAT>(q)) {
          n = q;
          first = shell_first<D::LAT>(q);
        }
      off[k] = n * D::ML + tt - first;
      slot[k] = ((t < D::Z ? 0 : D::R) + n) * SingleDims<KEY>::ST + tt - first;
      row[k] = n * S * S;
    }
  }
};

// Energy change of exchanging the species of sites a and b (LDS addresses,
// unequal codes), on every lane: the order of additions is pair_energy's, as
// in fixed_pair_sum2_chains.  The slots of `buf` past a shell's length stay 0.
template <int KEY>
__device__ __forceinline__ double single_delta(const SpecLds &L, const SeqGeo &g, uint32_t inv_S,
                                               const SingleLane<KEY> &sl, double *buf, SiteXYZ sa, SiteXYZ sb,
                                               int addr_a, int addr_b, int ca, int cb) {
  using D = SpecDims<KEY>;
  using N = SingleDims<KEY>;
  const int lane = threadIdx.x & 63;
  const int at_a = neighbour_index<KEY>(L, g, sa, sb), at_b = neighbour_index<KEY>(L, g, sb, sa);
  const int va = (int)(__umul24((uint32_t)ca, inv_S) >> 16), vb = (int)(__umul24((uint32_t)cb, inv_S) >> 16);
  const int oa = spec_sub<D::LAT>(sa) * D::R * D::ML, ob = spec_sub<D::LAT>(sb) * D::R * D::ML;
#pragma unroll
  for (int k = 0; k < N::P; ++k) {
    const int t = 64 * k + lane;
    if (t < 2 * D::Z) {
      const bool first = t < D::Z;
      const int code = L.lat[(first ? addr_a : addr_b) + L.off[(first ? oa : ob) + sl.off[k]]];
      // after the swap the other site, seen as a neighbour, has this site's species
      const int after = (first ? t == at_a : t - D::Z == at_b) ? (first ? ca : cb) : code;
      buf[sl.slot[k]] = L.vex[sl.row[k] + (first ? va : vb) + code];
      buf[sl.slot[k] + 2 * D::R * N::ST] = L.vex[sl.row[k] + (first ? vb : va) + after];
    }
  }
  wave_lds_order();
  const double *c = buf + (lane < N::NC ? lane : N::NC - 1) * N::ST;
  double b = 0.0;
#pragma unroll
  for (int j = 0; j < D::ML; ++j) b = b + c[j];
  wave_lds_order();
  double e[4];
#pragma unroll
  for (int w = 0; w < 4; ++w) {  // (before, A), (before, B), (after, A), (after, B)
    e[w] = readlane_d(b, w * D::R);
#pragma unroll
    for (int n = 1; n < D::R; ++n) e[w] = e[w] + readlane_d(b, w * D::R + n);
  }
  return (e[2] + e[3]) - (e[0] + e[1]);
}

template <int KEY, bool SINGLY>
__device__ __forceinline__ void metro_seq_spec_run(const SeqArgs &A, uint8_t *smem) {
  using D = SpecDims<KEY>;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = wave_uniform(tid >> 6);
  const SeqGeo g = seq_geo(A.g);
  const int S = g.S, n_atoms = A.g.n_atoms;
  const uint32_t inv_S = inverse_of(S);
  uint8_t *p = smem;
  auto take = [&](size_t bytes) {
    uint8_t *at = p;
    p += (bytes + 15) & ~(size_t)15;
    return at;
  };
  int8_t *lat = (int8_t *)take(A.g.lds_bytes);
  uint32_t *raw = (uint32_t *)take(4 * 624);
  uint32_t *tem = (uint32_t *)take(4 * kRingWords);
  uint2 *rsite = (uint2 *)take(8 * kRingWords);
  volatile int32_t *cmd = (volatile int32_t *)take(16);
  double *vex = (double *)take(sizeof(double) * S * S * D::R);
  double *ebuf = (double *)take(sizeof(double) * 2 * kEnergyChunk);
  double *sums = nullptr;
  if constexpr (SINGLY) {
    sums = (double *)take(SingleDims<KEY>::kBytes);
    for (int i = tid; i < SingleDims<KEY>::kBytes / 8; i += kSpecThreads) sums[i] = 0.0;
  }
  int32_t *offp = (int32_t *)take(4 * D::NSUB * D::R * D::ML);
  uint8_t *adj = take(D::TS * D::TS * D::TS);
  for (int i = tid; i < 624; i += kSpecThreads) raw[i] = A.mt[i];
  for (int i = tid; i < S * S * D::R; i += kSpecThreads) vex[i] = A.vex[i];
  stage_spec_tables<KEY>(offp, adj, A.off);
  stage_codes(lat, A.compact, g, D::NSUB, S);
  __syncthreads();
  ring_start<D::LAT>(g, raw, tem, rsite);
  const SpecLds L{lat, offp, vex, adj};
  if (wave != 0) {
    spec_helper<D::LAT>(g, raw, tem, rsite, cmd,
                        [&](int) { (void)spec_total_energy<KEY>(L, g, n_atoms, S, inv_S, ebuf); });
  } else {
    MtRing ring{raw, tem, rsite, cmd, 0, wave_uniform(A.mt_index[0]), false};
    const int trial = lane >> 3, w = (lane >> 2) & 1;
    const bool nbr_swap = A.nbr_swap != 0;
    const int drawn = nbr_swap ? 4 : 6;  // by a trial's sites
    const bool sampling = A.energies != nullptr && A.sample_every > 0;
    const double beta = A.beta;
    long long left = A.n_trials, to_sample = A.sample_every, sample_k = 0, accepted = 0;
    uint32_t length = 8 * kBatch;  // 8 times that of the last batches
    while (left > 0) {
      if (SINGLY && length < kBatchPays<KEY>) {
        SingleLane<KEY> sl;
        sl.init(S);
        for (int k = 0; k < kSingly && left > 0; ++k) {
          ring_ensure(ring, 9);
          const uint2 s1 = *ring_at(ring, rsite, 0);
          const SiteXYZ sa = unpack_xyz(s1.x);
          uint2 s2;
          if (nbr_swap) {
            const SiteXYZ sn = nbr_of_draw(g, sa, *ring_at(ring, tem, 3));
            s2 = make_uint2(pack_xyz(sn), (uint32_t)spec_addr<D::LAT>(g, sn));
          } else {
            s2 = *ring_at(ring, rsite, 3);
          }
          const uint32_t ru = *ring_at(ring, tem, drawn);
          const SiteXYZ sb = unpack_xyz(s2.x);
          const int ca = wave_uniform(lat[s1.y]), cb = wave_uniform(lat[s2.y]);
          ring.q += drawn;
          bool acc = true;
          if (ca != cb) {
            const double de = single_delta<KEY>(L, g, inv_S, sl, sums, sa, sb, (int)s1.y, (int)s2.y, ca, cb);
            if (wave_uniform(!(de < 0.0))) {
              ++ring.q;
              acc = wave_uniform(lt_exp_dev((double)ru * (1.0 / 4294967296.0), -(beta * de))) != 0;
            }
            if (acc) batch_write<D::LAT>(lat, g, lane < 8, w ? sb : sa, w ? ca : cb);
          }
          accepted += acc ? 1 : 0;
          left -= 1;
          if (sampling && --to_sample == 0) {
            to_sample = A.sample_every;
            spec_command(ring, kCmdEnergy);
            const double e = spec_total_energy<KEY>(L, g, n_atoms, S, inv_S, ebuf);
            if (lane == 0) A.energies[sample_k] = e;
            sample_k++;
          }
        }
        if (left <= 0) break;
      }
      ring_ensure(ring, 64 + 10);
      const uint2 s1 = *ring_at(ring, rsite, lane);
      const SiteXYZ sa = unpack_xyz(s1.x);
      uint2 s2;
      if (nbr_swap) {
        const SiteXYZ sn = nbr_of_draw(g, sa, *ring_at(ring, tem, lane + 3));
        s2 = make_uint2(pack_xyz(sn), (uint32_t)spec_addr<D::LAT>(g, sn));
      } else {
        s2 = *ring_at(ring, rsite, lane + 3);
      }
      const uint32_t ru = *ring_at(ring, tem, lane + drawn);
      const SiteXYZ sb = unpack_xyz(s2.x);
      const int ca = lat[s1.y], cb = lat[s2.y];
      const bool same = ca == cb;
      double ba, aa, bb, ab;
      spec_site_energies<KEY>(L, g, S, inv_S, sa, sb, (int)s1.y, ca, cb, ba, aa);
      spec_site_energies<KEY>(L, g, S, inv_S, sb, sa, (int)s2.y, cb, ca, bb, ab);
      const double de = (aa + ab) - (ba + bb);
      // equal species are accepted without a draw (metropolis.F90:774-777)
      const bool draws = !same && !(de < 0.0);
      bool acc = true;
      if (draws) acc = lt_exp_dev((double)ru * (1.0 / 4294967296.0), -(beta * de));
      const int next = lane + drawn + (draws ? 1 : 0);
      // the 8 trials' places: at most 49, so every hop stays in sight
      int my = 0, at = 0;
#pragma unroll
      for (int t = 1; t < kBatch; ++t) {
        at = __builtin_amdgcn_readlane(next, at);
        my = trial >= t ? at : my;
      }
      const uint32_t pa = (uint32_t)__shfl((int)s1.x, my), pb = (uint32_t)__shfl((int)s2.x, my);
      // code of A, code of B, accepted, exchanged
      const int what = __shfl(ca | (cb << 8) | (acc ? 1 << 16 : 0) | (acc && !same ? 1 << 17 : 0), my);
      const bool moved = (what >> 17) & 1;
      const bool reach = batch_conflict(g, D::RC, pa, pb);  // (on all lanes: it reads other lanes' sites)
      unsigned long long conf = __ballot(reach && moved && trial < (lane & 7));
      int n = kBatch;
      conf |= conf >> 32;
      conf |= conf >> 16;
      conf |= conf >> 8;
      if (conf & 0xffu) n = __ffs((int)(conf & 0xffu)) - 1;
      if constexpr (SINGLY) length = (uint32_t)wave_uniform((int)(length - length / 8 + n));
      n = n < left ? n : (int)left;
      if (sampling && n > to_sample) n = (int)to_sample;
      const unsigned long long upto = n < kBatch ? (1ull << (8 * n)) - 1ull : ~0ull;
      accepted += __popcll(__ballot((what >> 16) & 1) & upto & 0x0101010101010101ull);
      batch_write<D::LAT>(lat, g, moved && trial < n, unpack_xyz(w ? pb : pa), w ? what & 0xff : (what >> 8) & 0xff);
      ring.q = wave_uniform(ring.q + __shfl(next, __builtin_amdgcn_readlane(my, 8 * (n - 1))));
      left -= n;
      if (sampling) {
        to_sample -= n;
        if (to_sample == 0) {
          to_sample = A.sample_every;
          spec_command(ring, kCmdEnergy);
          const double e = spec_total_energy<KEY>(L, g, n_atoms, S, inv_S, ebuf);
          if (lane == 0) A.energies[sample_k] = e;
          sample_k++;
        }
      }
    }
    spec_command(ring, kCmdExit);
    ring_finish(ring, A.mt, A.mt_index);
    if (lane == 0) A.accepted[0] = accepted;
  }
  __syncthreads();
  unstage_codes(lat, A.compact, g, D::NSUB, inv_S);
}

}  // namespace bwl
