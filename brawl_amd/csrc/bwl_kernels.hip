// bwl_kernels.hip -- gfx950 kernels of the lattice-sampling path.
//
//   k_pack / k_unpack      reference doubled-grid layout <-> compact
//                          per-sublattice layout (HBM)
//   k_histogram            integer pair-count histogram, a part of one plane
//                          of cells per workgroup
//   k_site_energy          one site's energy in the reference's FP64 order
//   k_metro_seq            bit-exact sequential Metropolis driven by the
//                          reference's MT19937 stream: one trial at a time in
//                          one wavefront, or in speculative batches in a
//                          workgroup (k_metro_seq_spec); _batch: many chains
// (the parallel Metropolis sampler is in bwl_metro_kernels.h)
#include <hip/hip_runtime.h>

#include "bwl_kernels.h"
#include "bwl_spec.h"

namespace bwl {


// ------------------------------------------------------------------
// layout conversion
// ------------------------------------------------------------------
// Eight cells of the reference layout a thread, in one access: `ref` may be
// pinned host memory, where each access is a transfer of its own.  (The cells
// of a lattice are a multiple of 8: every extent is even.)
struct RefWalk {  // cells of the doubled grid in memory order
  int x, y, z;
};
__device__ inline RefWalk ref_walk(const Geo &g, int idx) {
  const int r = idx / g.m[0], z = r / g.m[1];
  return RefWalk{idx - r * g.m[0], r - z * g.m[1], z};
}
__device__ inline void ref_step(const Geo &g, RefWalk &w) {
  if (++w.x < g.m[0]) return;
  w.x = 0;
  if (++w.y < g.m[1]) return;
  w.y = 0;
  ++w.z;
}
__device__ inline bool ref_site(const Geo &g, const RefWalk &w) {
  return g.lattice == 1 ? ((w.x + w.y + w.z) & 1) == 0 : ((w.x ^ w.y) & 1) == 0 && ((w.y ^ w.z) & 1) == 0;
}
__device__ inline int ref_to_compact(const Geo &g, const RefWalk &w) {
  return compact_addr(g, sub_of(g.lattice, w.x & 1, w.y & 1), w.x >> 1, w.y >> 1, w.z >> 1);
}

__global__ void k_pack(const int8_t *__restrict__ ref, int8_t *__restrict__ compact, Geo g) {
  const int total = g.m[0] * g.m[1] * g.m[2];
  for (int idx = 8 * (blockIdx.x * blockDim.x + threadIdx.x); idx < total; idx += 8 * gridDim.x * blockDim.x) {
    const uint64_t v = *(const uint64_t *)(ref + idx);
    RefWalk w = ref_walk(g, idx);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (ref_site(g, w)) compact[ref_to_compact(g, w)] = (int8_t)(v >> (8 * k));
      ref_step(g, w);
    }
  }
}

__global__ void k_unpack(const int8_t *__restrict__ compact, int8_t *__restrict__ ref, Geo g) {
  const int total = g.m[0] * g.m[1] * g.m[2];
  for (int idx = 8 * (blockIdx.x * blockDim.x + threadIdx.x); idx < total; idx += 8 * gridDim.x * blockDim.x) {
    RefWalk w = ref_walk(g, idx);
    uint64_t v = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (ref_site(g, w)) v |= (uint64_t)(uint8_t)compact[ref_to_compact(g, w)] << (8 * k);
      ref_step(g, w);
    }
    *(uint64_t *)(ref + idx) = v;
  }
}

// ------------------------------------------------------------------
// pair-count histogram: H[n][b][a] += number of shell-n neighbours of
// species b around sites of species a (Fortran H(a,b,n) layout).
// A block counts part of one plane of cells (all sublattices) on the planes
// within the halo's reach, staged in LDS; the staging of the lattice bounded
// it when every block held it whole (bcc 32^3, four shells: 122 us in 32
// blocks, 21 here in 256).  The block's counts go to its own part of the
// output, which the host adds up: integers, so the split does not show.
// ------------------------------------------------------------------
constexpr int kHistThreads = 256;

__global__ __launch_bounds__(kHistThreads) void k_histogram(HistArgs A, int per_plane) {
  extern __shared__ __align__(16) uint8_t smem[];
  const Geo &g = A.g;
  int8_t *lat = (int8_t *)smem;
  const int hsize = g.S * g.S * g.R;
  constexpr int nw = kHistThreads / 64;
  const int plane = g.P[0] * g.P[1], planes = 2 * g.h + 1, slab = plane * planes;
  uint32_t *hw = (uint32_t *)(smem + ((g.nsub * slab + 15) & ~15));
  int32_t *offl = (int32_t *)(hw + hsize * nw);
  for (int i = threadIdx.x; i < hsize * nw; i += kHistThreads) hw[i] = 0;
  // offsets (ds * sub_stride + rest, |rest| < sub_stride / 2) in the slab's
  // shorter sublattices
  for (int i = threadIdx.x; i < g.nsub * g.z; i += kHistThreads) {
    const int o = A.off[i] + g.nsub * g.sub_stride + g.sub_stride / 2;
    const int ds = o / g.sub_stride - g.nsub;
    offl[i] = A.off[i] + ds * (slab - g.sub_stride);
  }
  const int cz = blockIdx.x / per_plane, part = blockIdx.x - cz * per_plane;
  for (int i = threadIdx.x; i < g.nsub * slab; i += kHistThreads) {
    const int s = i / slab;
    int r = i - s * slab;
    const int pz = r / plane;
    r -= pz * plane;
    const int py = r / g.P[0], px = r - py * g.P[0];
    lat[i] = A.compact[compact_addr(g, s, pmod(px - g.h, g.n[0]), pmod(py - g.h, g.n[1]), pmod(cz + pz - g.h, g.n[2]))];
  }
  __syncthreads();
  uint32_t *mine = hw + (threadIdx.x >> 6) * hsize;
  const int cells = g.n[0] * g.n[1], nsites = g.nsub * cells;
  for (int i = part * kHistThreads + threadIdx.x; i < nsites; i += per_plane * kHistThreads) {
    const int s = i / cells, r = i - s * cells;
    const int cy = r / g.n[0], cx = r - cy * g.n[0];
    const int addr = s * slab + g.h * plane + (cy + g.h) * g.P[0] + cx + g.h;
    const int a = lat[addr];
    if (a <= 0) continue;
    const int32_t *off = offl + s * g.z;
    for (int n = 0; n < g.R; ++n) {
      // 8-bit packed counts per species (a shell has at most 32 entries)
      uint64_t c = 0;
      for (int t = g.shell_start[n]; t < g.shell_start[n + 1]; ++t)
        c += (uint64_t)1 << (8 * (lat[addr + off[t]] - 1));
      for (int b = 0; b < g.S; ++b) {
        const uint32_t k = (uint32_t)(c >> (8 * b)) & 0xffu;
        if (k) atomicAdd(&mine[(a - 1) + g.S * (b + g.S * n)], k);
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < hsize; i += kHistThreads) {
    uint32_t t = 0;
    for (int w = 0; w < nw; ++w) t += hw[w * hsize + i];
    A.parts[(size_t)blockIdx.x * hsize + i] = t;
  }
}

// Energies of two sites, one wavefront: each lane gathers its neighbours from
// the lattice as it lies in memory (2 z bytes of it are wanted, so none is
// staged), then the entries are added in the reference's order.
__global__ __launch_bounds__(64) void k_site_energy(SiteArgs A) {
  const Geo &g = A.g;
  PairLanes pl;
  init_pair_lanes(g, pl);
  auto at = [&](int x, int y, int z) {
    return (int)A.compact[compact_addr(g, sub_of(g.lattice, x & 1, y & 1), x >> 1, y >> 1, z >> 1)];
  };
  const int sp0 = at(A.x[0], A.y[0], A.z[0]), sp1 = at(A.x[1], A.y[1], A.z[1]);
  double vals[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    vals[k] = 0.0;
    const int t = 64 * k + (int)threadIdx.x;
    if (k < pl.passes && t < 2 * g.z) {
      const int w = t < g.z ? 0 : 1;
      // the offset mod the box is below the extent: one subtraction wraps
      int x = A.x[w] + (pl.dmod[k] & 1023), y = A.y[w] + ((pl.dmod[k] >> 10) & 1023), z = A.z[w] + (pl.dmod[k] >> 20);
      x -= x >= g.m[0] ? g.m[0] : 0;
      y -= y >= g.m[1] ? g.m[1] : 0;
      z -= z >= g.m[2] ? g.m[2] : 0;
      vals[k] = A.vex[((w ? sp1 : sp0) - 1) + g.S * ((at(x, y, z) - 1) + g.S * pl.shell[k])];
    }
  }
  double eA = 0.0;
  const double e = pair_sum(g, pl, vals, &eA);
  if (threadIdx.x == 0) {
    A.out[0] = eA;
    A.out[1] = e;
  }
}

// ------------------------------------------------------------------
// Bit-exact sequential Metropolis (metropolis.F90:751-891), one wavefront.
// All lanes run the same control flow; the MT19937 state is in LDS.
// ------------------------------------------------------------------
template <int KEY>
__device__ __forceinline__ void metro_seq_run(const SeqArgs &A, uint8_t *smem) {
  const Geo &g = A.g;
  const int lane = threadIdx.x;
  int8_t *lat = (int8_t *)smem;
  size_t o = (g.lds_bytes + 15) & ~15;
  uint32_t *st = (uint32_t *)(smem + o);
  o += 624 * 4;
  double *sumbuf = (double *)(smem + o);
  clear_sum_buf(sumbuf);
  o += kSumBufBytes;
  double *vex = (double *)(smem + o);
  o += sizeof(double) * g.S * g.S * g.R;
  int32_t *offl = (int32_t *)(smem + o);
  o += sizeof(int32_t) * g.nsub * g.z;
  // the trial loop's geometry and swap mode (see put_seq_geo)
  int32_t *gw = (int32_t *)(smem + ((o + 15) & ~(size_t)15));

  for (int i = lane; i < 624; i += 64) st[i] = A.mt[i];
  for (int i = lane; i < g.S * g.S * g.R; i += 64) vex[i] = A.vex[i];
  put_seq_geo(gw, g);
  if (lane == 0) {
    gw[kSeqGeoWords] = A.nbr_swap;
    gw[kSeqGeoWords + 1] = A.energies != nullptr && A.sample_every > 0;
  }
  put_loop64(gw, 2, (unsigned long long)A.n_trials);
  put_loop64(gw, 4, (unsigned long long)A.sample_every);
  put_loop64(gw, 6, (unsigned long long)__double_as_longlong(A.beta));
  stage_offsets(offl, A.off, g);
  PairLanes pl;
  init_pair_lanes(g, pl);
  stage_lattice(lat, A.compact, g, 0);
  __syncthreads();
  int mti = A.mt_index[0];
  MtWin win{0u, kMtWinEmpty};
  long long accepted = 0;
  long long sample_k = 0;
  const SeqGeo sg = get_seq_geo(gw);
  const int nbr_swap = gw[kSeqGeoWords];
  const bool sampling = gw[kSeqGeoWords + 1] != 0;
  const long long n_trials = (long long)get_loop64(gw, 2), sample_every = (long long)get_loop64(gw, 4);
  const double beta = __longlong_as_double((long long)get_loop64(gw, 6));

  long long to_sample = sample_every;  // trial % sample_every == 0, counted down
  for (long long trial = 1; trial <= n_trials; ++trial) {
    SiteXYZ s1 = random_site_dev(sg, st, mti, win);
    SiteXYZ s2 = nbr_swap ? random_nbr_dev(sg, s1, st, mti, win) : random_site_dev(sg, st, mti, win);
    int addr1 = padded_addr_xyz(sg, s1.x, s1.y, s1.z);
    int addr2 = padded_addr_xyz(sg, s2.x, s2.y, s2.z);
    int sub1 = sub_of(sg.lattice, s1.x & 1, s1.y & 1);
    int sub2 = sub_of(sg.lattice, s2.x & 1, s2.y & 1);
    int sp1 = lat[addr1], sp2 = lat[addr2];
    bool acc;
    if (sp1 == sp2) {
      acc = true;  // metropolis.F90:774-777: counted as accepted, no draw
    } else {
      // energies before and after the swap from one gather of the unswapped lattice
      double e_un, e_sw;
      pair_energy_swap_lanes<KEY>(lat, sg, offl, vex, pl, addr1, sub1, s1, addr2, sub2, s2, sp1, sp2, sumbuf, e_un,
                                  e_sw);
      double de = e_sw - e_un;
      if (de < 0.0) {
        acc = true;
      } else {
        uint32_t r = mt_next(st, mti, win);
        double u = (double)r * (1.0 / 4294967296.0);
        acc = lt_exp_dev(u, -(beta * de));
      }
      if (acc) put_pair(lat, sg, s1, sub1, (int8_t)sp2, s2, sub2, (int8_t)sp1);
    }
    if (acc) accepted++;
    if (sampling && --to_sample == 0) {
      to_sample = sample_every;
      const double e = ref_total_energy(lat, g, offl, vex);
      if (lane == 0) A.energies[sample_k] = e;
      sample_k++;
    }
  }
  __syncthreads();
  unstage_lattice(lat, A.compact, g, 0);
  for (int i = lane; i < 624; i += 64) A.mt[i] = st[i];
  if (lane == 0) {
    A.mt_index[0] = mti;
    A.accepted[0] = accepted;
  }
}

// ------------------------------------------------------------------
// The same in speculative batches (bwl_spec.h).  A trial draws its sites'
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
// boxes large enough have a kernel without, see BWL_KERNEL_SINGLY).
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
    // n trials have been made
    auto count = [&](int n) {
      left -= n;
      if (!sampling) return;
      to_sample -= n;
      if (to_sample == 0) {
        to_sample = A.sample_every;
        spec_command(ring, kCmdEnergy);
        const double e = spec_total_energy<KEY>(L, g, n_atoms, S, inv_S, ebuf);
        if (lane == 0) A.energies[sample_k] = e;
        sample_k++;
      }
    };
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
          count(1);
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
      count(n);
    }
    spec_command(ring, kCmdExit);
    ring_finish(ring, A.mt, A.mt_index);
    if (lane == 0) A.accepted[0] = accepted;
  }
  __syncthreads();
  unstage_codes(lat, A.compact, g, D::NSUB, inv_S);
}

// ------------------------------------------------------------------
// Proposal draws (rdm_site, rdm_nbr, mc_select) from the reference stream,
// one wavefront (the MT19937 twist is wavefront-wide); lane 0 writes.
// ------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_draw_sites(DrawArgs A) {
  __shared__ uint32_t st[624];
  const int lane = threadIdx.x;
  for (int i = lane; i < 624; i += 64) st[i] = A.mt[i];
  __syncthreads();
  int mti = A.mt_index[0];
  const Geo &g = A.g;
  auto put = [&](int32_t *o, SiteXYZ s) {
    if (lane == 0) {
      o[0] = 1;
      o[1] = s.x + 1;
      o[2] = s.y + 1;
      o[3] = s.z + 1;
    }
  };
  if (A.mode == 1) {
    SiteXYZ s;
    s.x = A.site[1] - 1;
    s.y = A.site[2] - 1;
    s.z = A.site[3] - 1;
    put(A.out, random_nbr_dev(g, s, st, mti));
  } else {
    for (int q = 0; q < A.n; ++q) {
      SiteXYZ s1 = random_site_dev(g, st, mti);
      if (A.mode == 0) {
        put(A.out + 4 * q, s1);
        continue;
      }
      SiteXYZ s2 = A.mode == 3 ? random_nbr_dev(g, s1, st, mti) : random_site_dev(g, st, mti);
      put(A.out + 8 * q, s1);
      put(A.out + 8 * q + 4, s2);
    }
  }
  __syncthreads();
  for (int i = lane; i < 624; i += 64) A.mt[i] = st[i];
  if (lane == 0) A.mt_index[0] = mti;
}

hipError_t launch_draw_sites(const DrawArgs &a, hipStream_t s) {
  hipLaunchKernelGGL(k_draw_sites, dim3(1), dim3(64), 0, s, a);
  return hipGetLastError();
}

// ------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------
hipError_t launch_pack(const int8_t *ref, int8_t *compact, const Geo &g, hipStream_t s) {
  int total = g.m[0] * g.m[1] * g.m[2] / 8;
  int blocks = (total + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_pack, dim3(blocks), dim3(256), 0, s, ref, compact, g);
  return hipGetLastError();
}

hipError_t launch_unpack(const int8_t *compact, int8_t *ref, const Geo &g, hipStream_t s) {
  int total = g.m[0] * g.m[1] * g.m[2] / 8;
  int blocks = (total + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_unpack, dim3(blocks), dim3(256), 0, s, compact, ref, g);
  return hipGetLastError();
}

size_t hist_lds_bytes(const Geo &g, int threads) {
  return (size_t)((g.lds_bytes + 15) & ~15) + sizeof(uint32_t) * g.S * g.S * g.R * (threads / 64) +
         sizeof(int32_t) * g.nsub * g.z;
}

// blocks of about 256 sites, at most 8 to a plane of cells
static int hist_per_plane(const Geo &g) {
  const int q = (g.nsub * g.n[0] * g.n[1] + kHistThreads - 1) / kHistThreads;
  return q < 8 ? q : 8;
}

int hist_blocks(const Geo &g) { return hist_per_plane(g) * g.n[2]; }

hipError_t launch_histogram(const HistArgs &a, int blocks, hipStream_t s) {
  const Geo &g = a.g;
  const size_t lds = (size_t)((g.nsub * g.P[0] * g.P[1] * (2 * g.h + 1) + 15) & ~15) +
                     sizeof(uint32_t) * g.S * g.S * g.R * (kHistThreads / 64) + sizeof(int32_t) * g.nsub * g.z;
  HistArgs arg = a;
  int per_plane = hist_per_plane(g);
  void *kargs[] = {(void *)&arg, (void *)&per_plane};
  return launch_dynamic((const void *)k_histogram, dim3(blocks), kHistThreads, kargs, lds, s);
}

size_t site_lds_bytes(const Geo &g) {
  return (size_t)((g.lds_bytes + 15) & ~15) + sizeof(double) * g.S * g.S * g.R +
         sizeof(int32_t) * g.nsub * g.z;
}

hipError_t launch_site_energy(const SiteArgs &a, hipStream_t s) {
  hipLaunchKernelGGL(k_site_energy, dim3(1), dim3(64), 0, s, a);
  return hipGetLastError();
}

// One chain (the context's), its arguments in the kernel arguments.
template <int KEY>
__global__ __launch_bounds__(64) void k_metro_seq(SeqArgs A) {
  extern __shared__ __align__(16) uint8_t smem[];
  metro_seq_run<KEY>(A, smem);
}

// Many independent chains, one wavefront each (block b runs args[b]): the
// reference's replica ensemble, every chain on its own MT19937 stream.
template <int KEY>
__global__ __launch_bounds__(64) void k_metro_seq_batch(const SeqArgs *__restrict__ args) {
  extern __shared__ __align__(16) uint8_t smem[];
  metro_seq_run<KEY>(args[blockIdx.x], smem);
}

size_t seq_lds_bytes(const Geo &g) {
  return seq_geo_region((size_t)((g.lds_bytes + 15) & ~15) + 624 * 4 + kSumBufBytes +
                        sizeof(double) * g.S * g.S * g.R + sizeof(int32_t) * g.nsub * g.z) +
         64;
}

template <int KEY>
__global__ __launch_bounds__(kSpecThreads) void k_metro_seq_spec(SeqArgs A) {
  extern __shared__ __align__(16) uint8_t smem[];
  metro_seq_spec_run<KEY, false>(A, smem);
}

template <int KEY>
__global__ __launch_bounds__(kSpecThreads) void k_metro_seq_spec_batch(const SeqArgs *__restrict__ args) {
  extern __shared__ __align__(16) uint8_t smem[];
  metro_seq_spec_run<KEY, false>(args[blockIdx.x], smem);
}

template <int KEY>
__global__ __launch_bounds__(kSpecThreads) void k_metro_seq_singly(SeqArgs A) {
  extern __shared__ __align__(16) uint8_t smem[];
  metro_seq_spec_run<KEY, true>(A, smem);
}

template <int KEY>
__global__ __launch_bounds__(kSpecThreads) void k_metro_seq_singly_batch(const SeqArgs *__restrict__ args) {
  extern __shared__ __align__(16) uint8_t smem[];
  metro_seq_spec_run<KEY, true>(args[blockIdx.x], smem);
}

namespace {
const void *metro_seq_kernel(int key) { BWL_KERNEL_FOR_PAIR_SUM_KEY(k_metro_seq, key) }
const void *metro_seq_batch_kernel(int key) { BWL_KERNEL_FOR_PAIR_SUM_KEY(k_metro_seq_batch, key) }
// The kernel of template family `kern` that can take trials singly, nullptr if
// none is needed.  It takes 0 to 4 % longer where it does not (fcc 8^3, two
// shells, 8192 trials 2.08 ms -> 2.15), so boxes that are large enough for
// batches to be as fast with nothing rejected have one without: against one
// trial at a time 1.4x and 1.5x on fcc and bcc 6^3 with two shells (reach
// 0.29), 1.4x on fcc 8^3 with three (0.12; 0.95x on 6^3), 1.18x on fcc 8^3 with
// four and 1.02x on bcc 10^3 (0.17; 0.80x on 8^3).
#define BWL_KERNEL_SINGLY(kern, pick)                          \
  if (pick.reach > (pick.key % 16 == 2 ? 0.3 : 0.18)) {        \
    switch (pick.key) {                                        \
      case 16 + 2: return (const void *)kern<16 + 2>;          \
      case 16 + 3: return (const void *)kern<16 + 3>;          \
      case 16 + 4: return (const void *)kern<16 + 4>;          \
      case 32 + 2: return (const void *)kern<32 + 2>;          \
      case 32 + 3: return (const void *)kern<32 + 3>;          \
      case 32 + 4: return (const void *)kern<32 + 4>;          \
    }                                                          \
  }
const void *metro_seq_spec_kernel(const SeqPick &pick) {
  BWL_KERNEL_SINGLY(k_metro_seq_singly, pick)
  BWL_KERNEL_FOR_SPEC_KEY(k_metro_seq_spec, pick.key)
}
const void *metro_seq_spec_batch_kernel(const SeqPick &pick) {
  BWL_KERNEL_SINGLY(k_metro_seq_singly_batch, pick)
  BWL_KERNEL_FOR_SPEC_KEY(k_metro_seq_spec_batch, pick.key)
}
}  // namespace

size_t seq_spec_lds_bytes(const Geo &g) {
  // SingleDims::kBytes, whether the launch's kernel uses them or not
  const size_t sums = 8 * 4 * (size_t)g.R * (shell_max(g.lattice, g.R) | 1);
  return spec_table_bytes(g) + spec_ring_bytes() + spec_energy_bytes() + spec_align(sums);
}

bool spec_pays(const void *fn, int n, const SeqPick &pick, double far) {
  if (!fn) return false;
  int dev = 0, n_cu = 0, resident = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return false;
  if (n <= n_cu) return true;
  if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)pick.lds_spec) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&resident, fn, kSpecThreads, pick.lds_spec) != hipSuccess)
    return false;
  const long long room = (long long)n_cu * resident;
  return n <= room || (pick.reach <= far && n <= 2 * room);
}

hipError_t launch_metro_seq(const SeqArgs &a, const SeqPick &pick, hipStream_t s) {
  SeqArgs arg = a;
  void *kargs[] = {(void *)&arg};
  if (pick.spec) return launch_dynamic(metro_seq_spec_kernel(pick), dim3(1), kSpecThreads, kargs, pick.lds_spec, s);
  return launch_dynamic(metro_seq_kernel(pick.key), dim3(1), 64, kargs, pick.lds, s);
}

hipError_t launch_metro_seq_batch(const SeqArgs *args_dev, int n, const SeqPick &pick, hipStream_t s) {
  void *kargs[] = {(void *)&args_dev};
  const void *fn = pick.spec ? metro_seq_spec_batch_kernel(pick) : nullptr;
  // (a batch here is 64 places' energies: the more shells, the sooner too much)
  if (spec_pays(fn, n, pick, pick.key % 16 <= 2 ? 0.05 : 0.0))
    return launch_dynamic(fn, dim3(n), kSpecThreads, kargs, pick.lds_spec, s);
  return launch_dynamic(metro_seq_batch_kernel(pick.key), dim3(n), 64, kargs, pick.lds, s);
}

// ------------------------------------------------------------------
// LDS read bandwidth probe (measurement only): each block fills 64 KiB of
// LDS, then every lane streams 16-byte reads, a wavefront reading 1 KiB of
// consecutive addresses per step (no bank conflicts).  The index is made
// opaque to the compiler each step so no read can be merged away; the
// folded values are written only if they hit one improbable pattern.
// ------------------------------------------------------------------
__global__ __launch_bounds__(1024) void k_lds_bandwidth(int iters, uint32_t *sink) {
  __shared__ uint4 buf[4096];
  const int t = threadIdx.x;
  for (int i = t; i < 4096; i += blockDim.x) buf[i] = make_uint4(i, 3u * i, 5u * i, 7u * i);
  __syncthreads();
  uint32_t acc = 0;
  int idx = t & 4095;
  for (int k = 0; k < iters; ++k) {
    const uint4 v = buf[idx];
    acc ^= v.x ^ v.y ^ v.z ^ v.w;
    idx = (idx + 1024) & 4095;
    asm volatile("" : "+v"(idx));
  }
  if (acc == 0x9e3779b9u) sink[blockIdx.x] = acc;
}

hipError_t launch_lds_bandwidth(int blocks, int iters, uint32_t *sink, hipStream_t s) {
  hipLaunchKernelGGL(k_lds_bandwidth, dim3(blocks), dim3(1024), 0, s, iters, sink);
  return hipGetLastError();
}

}  // namespace bwl
