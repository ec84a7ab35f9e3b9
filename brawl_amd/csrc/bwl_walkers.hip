// bwl_walkers.hip -- sequential walkers on the device: nested-sampling runs,
// Wang-Landau walker sweeps and window entry, and the windowed pair-count
// histogram behind the radial densities.
//
// Each nested-sampling run and each Wang-Landau walker is one workgroup
// that consumes its own MT19937 stream exactly as the reference's serial
// code does (one MPI rank per walker there), with site and pair energies in
// the reference's FP64 order, so every walker's trajectory is bit-identical
// to the reference's: four wavefronts that take trials in speculative batches
// (k_ns_spec, k_wl_sweeps_spec; see bwl_spec.h), or, where spec_pays says so
// and for window entry, one wavefront and one trial at a time.  Throughput
// comes from running many walkers in one launch.
#include <hip/hip_runtime.h>

#include "bwl_kernels.h"
#include "bwl_spec.h"

namespace bwl {

namespace {

// bin_index (wang-landau.F90:515-523): truncation toward zero, +1.
__device__ inline int wl_bin_index(double e, const double *edges, int bins) {
  const double range = edges[bins] - edges[0];
  return (int)(((e - edges[0]) / range) * (double)bins) + 1;
}

// bin_index with its constants in registers, for an energy that every lane
// holds alike (the result is wavefront-uniform).  x = ((e - e0) * (1/range)) *
// bins differs from the reference's ((e - e0) / range) * bins by at most a
// few units in the last place (under 1e-15 |x|); when x is further than
// 1e-9 max(1, |x|) from every integer both truncate to the same integer, and
// otherwise the reference's expression is evaluated.  The result is always
// that of wl_bin_index.
struct BinMap {
  double e0, range, rinv, nb;
};

__device__ inline BinMap bin_map(const double *edges, int bins) {
  BinMap b;
  b.e0 = edges[0];
  b.range = edges[bins] - edges[0];
  b.rinv = 1.0 / b.range;
  b.nb = (double)bins;
  return b;
}

__device__ inline int wl_bin_index(double e, const BinMap &b) {
  const double a = e - b.e0;
  const double x = (a * b.rinv) * b.nb;
  const double t = trunc(x);
  const double f = fabs(x - t);
  const double tol = 1e-9 * fmax(1.0, fabs(x));
  if (wave_uniform(f > tol && 1.0 - f > tol)) return wave_uniform((int)t + 1);
  return wave_uniform((int)((a / b.range) * b.nb) + 1);
}

__device__ inline double genrand_dev(uint32_t *st, int &mti) {
  return (double)mt_next(st, mti) * (1.0 / 4294967296.0);
}

__device__ inline double genrand_dev(uint32_t *st, int &mti, MtWin &win) {
  return (double)mt_next(st, mti, win) * (1.0 / 4294967296.0);
}

}  // namespace

// ------------------------------------------------------------------
// Initial walker energies of nested-sampling runs, all walkers of all runs
// at once (block (w, run)): total_energy + genrand()*1e-8
// (nested_sampling.f90:95; 1e-8 is a REAL(4) literal there), the total in
// the reference's summation order.
// ------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_ns_energies(const NsArgs *__restrict__ args) {
  extern __shared__ __align__(16) uint8_t smem[];
  const NsArgs &A = args[blockIdx.y];
  const int w = blockIdx.x;
  if (w >= A.n_walkers) return;
  const Geo &g = A.g;
  int8_t *lat = (int8_t *)smem;
  size_t o = (g.lds_bytes + 15) & ~15;
  double *vex = (double *)(smem + o);
  o += sizeof(double) * g.S * g.S * g.R;
  int32_t *offl = (int32_t *)(smem + o);
  for (int i = threadIdx.x; i < g.S * g.S * g.R; i += 64) vex[i] = A.vex[i];
  stage_offsets(offl, A.off, g);
  stage_lattice(lat, A.walkers + (size_t)g.compact_bytes * w, g, 0);
  __syncthreads();
  const double e = ref_total_energy(lat, g, offl, vex);
  if (threadIdx.x == 0) A.E[w] = e + A.rnde[w] * (double)1e-8f;
}

// ------------------------------------------------------------------
// Nested sampling: the whole serial loop of nested_sampling.f90:78-200 for
// one run.  Walker lattices stay in HBM; the walker being walked is staged
// in LDS.  Walker energies live in LDS.
// ------------------------------------------------------------------
template <int KEY>
__global__ __launch_bounds__(64) void k_ns(const NsArgs *__restrict__ args) {
  extern __shared__ __align__(16) uint8_t smem[];
  const NsArgs &A = args[blockIdx.x];
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
  double *E = (double *)(smem + o);
  o += sizeof(double) * A.n_walkers;
  int32_t *offl = (int32_t *)(smem + o);
  o += sizeof(int32_t) * g.nsub * g.z;
  // the trial loop's geometry (see put_seq_geo)
  int32_t *gw = (int32_t *)(smem + ((o + 15) & ~(size_t)15));

  for (int i = lane; i < 624; i += 64) st[i] = A.mt[i];
  for (int i = lane; i < g.S * g.S * g.R; i += 64) vex[i] = A.vex[i];
  put_seq_geo(gw, g);
  if (lane == 0) gw[kSeqGeoWords] = A.n_steps;
  put_loop64(gw, 2, (unsigned long long)A.max_redraws);
  stage_offsets(offl, A.off, g);
  PairLanes pl;
  init_pair_lanes(g, pl);
  int mti = A.mt_index[0];
  MtWin win{0u, kMtWinEmpty};
  const int nw = A.n_walkers;
  const size_t cb = (size_t)g.compact_bytes;

  // walker energies, computed beforehand by k_ns_energies
  for (int w = lane; w < nw; w += 64) E[w] = A.E[w];
  __syncthreads();

  long long trials = 0, accepted = 0;
  int status = 0;
  int extra = 0, n_acc = 0;
  const int half = (int)((float)nw / 2.0f);
  const SeqGeo sg = get_seq_geo(gw);
  const ImageLanes il = image_lanes(sg);
  const int n_steps = gw[kSeqGeoWords];
  const long long max_redraws = (long long)get_loop64(gw, 2);
  for (int it = 1; it <= A.n_iter && status == 0; ++it) {
    // maxloc: the first maximum (nested_sampling.f90:117)
    double best = -INFINITY;
    int bi = 0x7fffffff;  // no walker seen
    for (int w = lane; w < nw; w += 64)
      if (bi == 0x7fffffff || E[w] > best) {
        best = E[w];
        bi = w;
      }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) {
      const double ob = __shfl_xor(best, m);
      const int oi = __shfl_xor(bi, m);
      if (oi != 0x7fffffff && (bi == 0x7fffffff || ob > best || (ob == best && oi < bi))) {
        best = ob;
        bi = oi;
      }
    }
    const int imax = bi;
    const double limit = best;
    if (lane == 0) A.e_limits[it - 1] = limit;
    // walk-length adaptation (nested_sampling.f90:129-144)
    if (it % half == 0) {
      if (((float)n_acc < (float)A.n_at * 0.05f) && (extra < n_steps * 100)) extra += n_steps;
    }
    // clone a random walker over the discarded one (nested_sampling.f90:149-152)
    const double rnd = genrand_dev(st, mti, win);
    int irnd = (int)ceil(rnd * (double)nw);
    if (irnd < 1) irnd = 1;
    const int src = irnd - 1;
    __syncthreads();
    stage_lattice_walk(lat, A.walkers + cb * src, g);
    __syncthreads();
    double ecur = E[src];
    n_acc = 0;
    // the walk (nested_sampling.f90:157-192)
    for (int stp = 1; stp <= n_steps + extra; ++stp) {
      // rdm2 is redrawn while its species equals rdm1's; the first rdm2 is
      // drawn before either species is read, so both reads go out together
      const SiteXYZ r1 = random_site_dev(sg, st, mti, win);
      SiteXYZ r2 = random_site_dev(sg, st, mti, win);
      const int a1 = padded_addr_xyz(sg, r1.x, r1.y, r1.z);
      int a2 = padded_addr_xyz(sg, r2.x, r2.y, r2.z);
      const int s1 = lat[a1];
      int s2 = lat[a2];
      long long redraws = 0;
      while (s1 == s2 && ++redraws < max_redraws) {
        r2 = random_site_dev(sg, st, mti, win);
        a2 = padded_addr_xyz(sg, r2.x, r2.y, r2.z);
        s2 = lat[a2];
      }
      if (s1 == s2) {
        status = 1;
        break;
      }
      const int sub1 = sub_of(sg.lattice, r1.x & 1, r1.y & 1);
      const int sub2 = sub_of(sg.lattice, r2.x & 1, r2.y & 1);
      // energies before and after the swap from one gather of the unswapped lattice
      double eu, es;
      pair_energy_swap_lanes<KEY>(lat, sg, offl, vex, pl, a1, sub1, r1, a2, sub2, r2, s1, s2, sumbuf, eu, es);
      const double de = es - eu;
      ++trials;
      const bool acc = ecur + de < limit;
      if (acc) {
        ecur = ecur + de;
        ++n_acc;
        ++accepted;
      }
      if (acc) put_pair(lat, sg, il, r1, sub1, (int8_t)s2, r2, sub2, (int8_t)s1);
    }
    __syncthreads();
    if (lane == 0) E[imax] = ecur;
    unstage_lattice_walk(lat, A.walkers + cb * imax, g);
    __syncthreads();
  }
  for (int w = lane; w < nw; w += 64) A.E[w] = E[w];
  for (int i = lane; i < 624; i += 64) A.mt[i] = st[i];
  if (lane == 0) {
    A.mt_index[0] = mti;
    A.counters[0] = trials;
    A.counters[1] = accepted;
    A.counters[2] = status;
  }
}

// ------------------------------------------------------------------
// Nested sampling in speculative batches (bwl_spec.h); the run and its
// results are those of k_ns.  A walk's trial draws three numbers for its
// first site, then three per candidate second site until one holds another
// species, so with the lattice as it is the whole run of trials is fixed by
// the species of the next 64 triples' sites: lane l holds triple l, finds the
// first later triple of another species from the ballots per species, and
// the trials follow by hopping from a trial's last triple to the next.
//
// Four trials at a time: trial g = lane >> 4, and within its 16 lanes the
// shell (lane & 3), the site (lane & 4) and before or after the swap (lane &
// 8), one chain of ordered additions each.  Early in a run nearly every trial
// is accepted and on the small lattices of such runs a swap reaches a
// quarter of the others, so the trials are foreseen to end as most of the
// last ones did: foreseen accepted, a trial's swap is written before the next
// trial's neighbours are read (one wavefront's LDS accesses complete in
// program order), and taken back if the decision falls otherwise.
// ------------------------------------------------------------------
template <int KEY>
__global__ __launch_bounds__(kSpecThreads) void k_ns_spec(const NsArgs *__restrict__ args) {
  using D = SpecDims<KEY>;
  constexpr int ML = D::ML, R = D::R;
  extern __shared__ __align__(16) uint8_t smem[];
  const NsArgs &A = args[blockIdx.x];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = wave_uniform(tid >> 6);
  const SeqGeo g = seq_geo(A.g);
  const int S = g.S;
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
  // command, walker to clone, walker discarded, walker discarded before
  volatile int32_t *sh = (volatile int32_t *)take(16);
  double *vex = (double *)take(sizeof(double) * S * S * R);
  double *E = (double *)take(sizeof(double) * A.n_walkers);
  int32_t *offp = (int32_t *)take(4 * D::NSUB * R * ML);
  uint8_t *adj = take(D::TS * D::TS * D::TS);

  const int nw = A.n_walkers;
  const size_t cb = (size_t)A.g.compact_bytes;
  for (int i = tid; i < 624; i += kSpecThreads) raw[i] = A.mt[i];
  for (int i = tid; i < S * S * R; i += kSpecThreads) vex[i] = A.vex[i];
  for (int w = tid; w < nw; w += kSpecThreads) E[w] = A.E[w];
  stage_spec_tables<KEY>(offp, adj, A.off);
  __syncthreads();
  ring_start<D::LAT>(g, raw, tem, rsite);
  const SpecLds L{lat, offp, vex, adj};
  // the walked lattice over the discarded walker, then the next clone
  auto turn = [&](int cmd) {
    const int src = sh[1], last = sh[3];
    if (cmd != kCmdLoad) {
      unstage_codes(lat, A.walkers + cb * last, g, D::NSUB, inv_S);
      __syncthreads();
    }
    if (cmd != kCmdStore) {
      stage_codes(lat, A.walkers + cb * src, g, D::NSUB, S);
      __syncthreads();
    }
  };
  if (wave != 0) {
    spec_helper<D::LAT>(g, raw, tem, rsite, sh, turn);
    return;
  }

  MtRing ring{raw, tem, rsite, sh, 0, wave_uniform(A.mt_index[0]), false};
  const int grp = lane >> 4, w = (lane >> 2) & 1, shell = (lane & 3) < R ? lane & 3 : R - 1;
  const bool after = (lane & 8) != 0;
  int first, len;
  lane_shell<KEY>(shell, first, len);
  const int row = shell * S * S;
  const unsigned long long later = lane == 63 ? 0ull : ~0ull << (lane + 1);
  long long trials = 0, accepted = 0;
  int extra = 0, n_acc = 0, status = 0;
  bool foresee = true;  // trials foreseen accepted
  const int half = (int)((float)nw / 2.0f);
  int it = 1;
  for (; it <= A.n_iter && status == 0; ++it) {
    // maxloc: the first maximum (nested_sampling.f90:117)
    double best = -INFINITY;
    int bi = 0x7fffffff;  // no walker seen
    for (int k = lane; k < nw; k += 64)
      if (bi == 0x7fffffff || E[k] > best) {
        best = E[k];
        bi = k;
      }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) {
      const double ob = __shfl_xor(best, m);
      const int oi = __shfl_xor(bi, m);
      if (oi != 0x7fffffff && (bi == 0x7fffffff || ob > best || (ob == best && oi < bi))) {
        best = ob;
        bi = oi;
      }
    }
    const double limit = best;
    const int imax = wave_uniform(bi);
    if (lane == 0) A.e_limits[it - 1] = limit;
    // walk-length adaptation (nested_sampling.f90:129-144)
    if (it % half == 0) {
      if (((float)n_acc < (float)A.n_at * 0.05f) && (extra < A.n_steps * 100)) extra += A.n_steps;
    }
    // clone a random walker over the discarded one (nested_sampling.f90:149-152)
    ring_ensure(ring, 1);
    const double rnd = (double)*ring_at(ring, tem, 0) * (1.0 / 4294967296.0);
    ring.q += 1;
    int irnd = (int)ceil(rnd * (double)nw);
    if (irnd < 1) irnd = 1;
    const int src = wave_uniform(irnd - 1);
    if (lane == 0) {
      sh[3] = sh[2];
      sh[1] = src;
      sh[2] = imax;
    }
    const int cmd = it == 1 ? kCmdLoad : kCmdTurn;
    spec_command(ring, cmd);
    turn(cmd);
    double ecur = E[src];
    n_acc = 0;
    // the walk (nested_sampling.f90:157-192)
    int left = A.n_steps + extra;
    while (left > 0 && status == 0) {
      ring_ensure(ring, 194);
      uint2 site = *ring_at(ring, rsite, 3 * lane);
      int code = lat[site.y];
      unsigned long long same = 0;
      for (int s = 0; s < S; ++s) {
        const unsigned long long m = __ballot(code == s * S);
        same = code == s * S ? m : same;
      }
      const unsigned long long differ = ~same & later;
      const int second = differ ? __ffsll((long long)differ) - 1 : 64;
      int j = 0;  // first triple of the next trial
      if (__builtin_amdgcn_readlane(second, 0) == 64) {
        // no site of another species in sight: the first site is kept (lane
        // 0) and the stream searched on, 64 candidates at a time
        const int c0 = __builtin_amdgcn_readlane(code, 0);
        long long seen = 63;
        for (;;) {
          ring.q += 192;
          if (seen >= A.max_redraws) {
            status = 1;
            break;
          }
          ring_ensure(ring, 194);
          const uint2 s2 = *ring_at(ring, rsite, 3 * lane);
          const int c2 = lat[s2.y];
          const unsigned long long m = __ballot(c2 != c0);
          if (m) {
            // as if the two had been triples 0 and 1, with the position after them
            const int k = __ffsll((long long)m) - 1;
            const uint32_t x1 = (uint32_t)__builtin_amdgcn_readlane((int)s2.x, k);
            const uint32_t y1 = (uint32_t)__builtin_amdgcn_readlane((int)s2.y, k);
            const int c1 = __builtin_amdgcn_readlane(c2, k);
            if (lane == 1) {
              site = make_uint2(x1, y1);
              code = c1;
            }
            ring.q += 3 * (k + 1) - 6;
            break;
          }
          seen += 64;
        }
        if (status) break;
        j = -1;  // one trial of triples 0 and 1, then a new window
      }
      const bool lone = j < 0;
      if (lone) j = 0;
      bool stale = false;
      while (!stale) {
        // the next trials' triples (j: first site, k: second), each lane
        // hopping to its own trial's
        const int most = lone ? 1 : (left < 4 ? left : 4);
        int my_j = j, my_k = __shfl(second, j);
        if (lone) my_k = 1;
#pragma unroll
        for (int t = 1; t < 4; ++t) {
          const int k = __shfl(second, (my_k + 1) & 63);
          const bool hop = grp >= t;
          my_j = hop ? my_k + 1 : my_j;
          my_k = hop ? (my_j < 64 ? k : 64) : my_k;
        }
        // trials in sight: those before the first without a second site
        const unsigned long long out = __ballot(my_k >= 64);
        int ng = out ? (__ffsll((long long)out) - 1) >> 4 : 4;
        ng = ng < most ? ng : most;
        if (ng == 0) break;
        my_j &= 63;
        my_k &= 63;
        const uint32_t pa = (uint32_t)__shfl((int)site.x, my_j), pb = (uint32_t)__shfl((int)site.x, my_k);
        const int aa = __shfl((int)site.y, my_j), ab = __shfl((int)site.y, my_k);
        const int ca = __shfl(code, my_j), cb2 = __shfl(code, my_k);
        // Row trial grp against column trial lane & 3, one pair of their
        // sites per lane: the same site, or a site the column's trial passed
        // over (the first two are looked at; a trial that passed over more
        // counts as equal to any), or within reach.
        const int col = (lane & 3) * 16;
        const uint32_t qa = (uint32_t)__shfl((int)pa, col), qb = (uint32_t)__shfl((int)pb, col);
        const int cj = __shfl(my_j, col), ck = __shfl(my_k, col);
        const uint32_t r1 = (uint32_t)__shfl((int)site.x, (cj + 1) & 63), r2 = (uint32_t)__shfl((int)site.x, (cj + 2) & 63);
        const uint32_t rp = (lane & 4) ? pb : pa, cp = (lane & 8) ? qb : qa;
        bool equal = rp == cp;
        if (!lone) equal = equal || (ck > cj + 1 && rp == r1) || (ck > cj + 2 && rp == r2) || ck > cj + 3;
        const bool reach = box_gap(unpack_xyz(rp), unpack_xyz(cp), g, D::RC) <= 2u * D::RC;
        unsigned long long eq = __ballot(equal && grp < (lane & 3));
        const unsigned long long conf = __ballot(reach);
        if (eq) {
          eq |= eq >> 32;
          eq |= eq >> 16;
          eq |= eq >> 8;
          eq |= eq >> 4;
          const int c = __ffs((int)(eq & 0xeu)) - 1;
          ng = c < ng ? c : ng;
        }
        // triples of the sites that these trials may exchange: once passed, a
        // later one's species is out of date
        bool touched = false;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          touched |= q < ng && (site.x == (uint32_t)__builtin_amdgcn_readlane((int)pa, 16 * q) ||
                                site.x == (uint32_t)__builtin_amdgcn_readlane((int)pb, 16 * q));
        const unsigned long long hit = __ballot(touched);
        const SiteXYZ own = unpack_xyz(w ? pb : pa), oth = unpack_xyz(w ? pa : pb);
        const int c_own = w ? cb2 : ca, c_oth = w ? ca : cb2;
        // images of both sites over the trial's 16 lanes
        const SiteXYZ ws = unpack_xyz(after ? pb : pa);
        const int wat = image_addr<D::LAT>(g, ws, lane & 7);
        const int wold = after ? cb2 : ca, wnew = after ? ca : cb2;
        const int addr = w ? ab : aa;
        const int at = neighbour_index<KEY>(L, g, own, oth) - first;
        // the shell's cells are read half by the lane before the swap, half
        // by its partner after it, and exchanged
        constexpr int MH = ML / 2;
        int mh[MH];
        int2 o[MH / 2];
        {
          const int2 *op = (const int2 *)(offp + (spec_sub<D::LAT>(own) * R + shell) * ML) + (after ? MH / 2 : 0);
#pragma unroll
          for (int q = 0; q < MH / 2; ++q) o[q] = op[q];
        }
        if (foresee) {
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            wave_lds_order();
            if (grp == t) {
#pragma unroll
              for (int q = 0; q < MH / 2; ++q) {
                mh[2 * q] = lat[addr + o[q].x];
                mh[2 * q + 1] = lat[addr + o[q].y];
              }
              wave_lds_order();
              if (t < ng && wat >= 0) lat[wat] = (int8_t)wnew;
            }
          }
          wave_lds_order();
        } else {
#pragma unroll
          for (int q = 0; q < MH / 2; ++q) {
            mh[2 * q] = lat[addr + o[q].x];
            mh[2 * q + 1] = lat[addr + o[q].y];
          }
        }
        int cd[ML];
#pragma unroll
        for (int q = 0; q < MH; ++q) {
          const int other = __builtin_amdgcn_update_dpp(0, mh[q], kRowRotate8, 0xf, 0xf, true);
          cd[q] = after ? other : mh[q];
          cd[MH + q] = after ? mh[q] : other;
        }
        const double *vr = vex + row + (int)(__umul24((uint32_t)(after ? c_oth : c_own), inv_S) >> 16);
        double v[ML];
#pragma unroll
        for (int i = 0; i < ML; ++i) v[i] = vr[cd[i]];
        // after the swap the other site, seen as a neighbour, has this site's species
        const bool fix = after && at >= 0 && at < len;
        if (__ballot(fix) != 0) {
          const double f = vr[c_own];
#pragma unroll
          for (int i = 0; i < ML; ++i) v[i] = fix && i == at ? f : v[i];
        }
        double e = quad_sum<R>(shell_chain<ML>(v, len));
        e = e + dpp_d<kRowHalfMirror>(e);
        const double de = dpp_d<kRowRotate8>(e) - e;  // lanes before: after - before
        // The decisions, in order and without branches: a trial counts until
        // one is reached by an earlier one that went otherwise than foreseen
        // (it was read from the wrong lattice).
        int swaps = 0, off_course = 0, t = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          uint32_t c = (uint32_t)(conf >> (16 * q)) & 0xffffu;
          c |= c >> 8;
          c = (c | c >> 4) & 0xfu & (0xeu << q);
          const bool counts = q < ng && t == q && !((off_course >> q) & 1);
          const double en = ecur + readlane_d(de, 16 * q);
          const bool acc = counts && en < limit;
          ecur = acc ? en : ecur;
          swaps |= acc ? 1 << q : 0;
          off_course |= counts && acc != foresee ? (int)c : 0;
          t += counts ? 1 : 0;
        }
        swaps = wave_uniform(swaps);
        t = wave_uniform(t);
        const bool mine = ((swaps >> grp) & 1u) != 0;
        wave_lds_order();
        if (grp < ng && mine != foresee && wat >= 0) lat[wat] = (int8_t)(mine ? wnew : wold);
        wave_lds_order();
        const int got = __popc((unsigned)swaps);
        foresee = 2 * got > t;
        const int next = __builtin_amdgcn_readlane(my_k, 16 * (t - 1)) + 1;
        left -= t;
        trials += t;
        n_acc += got;
        j = next;
        stale = lone || left <= 0 || j >= 64 || (hit >> j) != 0;
      }
      ring.q += 3 * j;
    }
    accepted += n_acc;
    if (lane == 0) E[imax] = ecur;
    wave_lds_order();
  }
  if (lane == 0) sh[3] = sh[2];
  spec_command(ring, kCmdStore);
  turn(kCmdStore);
  spec_command(ring, kCmdExit);
  for (int k = lane; k < nw; k += 64) A.E[k] = E[k];
  ring_finish(ring, A.mt, A.mt_index);
  if (lane == 0) {
    A.counters[0] = trials;
    A.counters[1] = accepted;
    A.counters[2] = status;
  }
}

// ------------------------------------------------------------------
// Wang-Landau `sweeps` (wang-landau.F90:539-632) for one walker, without the
// window average (a separate kernel does that after every walker's call).
// The walker's ln g and visit histogram are staged in LDS.  KEY is the
// pair-sum variant of every walker of the launch (pair_sum_key), or -1 when
// the launch mixes lattices: a kernel for one variant carries only that
// sum's code, which leaves the registers to the rest of the trial.
// ------------------------------------------------------------------
template <int KEY>
__global__ __launch_bounds__(64) void k_wl_sweeps(const WlArgs *__restrict__ args) {
  extern __shared__ __align__(16) uint8_t smem[];
  const WlArgs &A = args[blockIdx.x];
  const Geo &g = A.g;
  const int lane = threadIdx.x;
  const int hb = A.end_idx - A.start_idx + 1;
  int8_t *lat = (int8_t *)smem;
  size_t o = (g.lds_bytes + 15) & ~15;
  uint32_t *st = (uint32_t *)(smem + o);
  o += 624 * 4;
  double *sumbuf = (double *)(smem + o);
  clear_sum_buf(sumbuf);
  o += kSumBufBytes;
  double *vex = (double *)(smem + o);
  o += sizeof(double) * g.S * g.S * g.R;
  double *lng = (double *)(smem + o);
  o += sizeof(double) * A.bins;
  double *edges = (double *)(smem + o);
  o += sizeof(double) * (A.bins + 1);
  double *hist = (double *)(smem + o);
  o += sizeof(double) * hb;
  int32_t *offl = (int32_t *)(smem + o);
  o += sizeof(int32_t) * g.nsub * g.z;
  // the trial loop's geometry and window (see put_seq_geo)
  int32_t *gw = (int32_t *)(smem + ((o + 15) & ~(size_t)15));

  for (int i = lane; i < 624; i += 64) st[i] = A.mt[i];
  for (int i = lane; i < g.S * g.S * g.R; i += 64) vex[i] = A.vex[i];
  put_seq_geo(gw, g);
  if (lane == 0) {
    gw[kSeqGeoWords + 0] = A.bins;
    gw[kSeqGeoWords + 1] = A.start_idx;
    gw[kSeqGeoWords + 2] = A.end_idx;
    gw[kSeqGeoWords + 3] = A.nbr_swap;
  }
  stage_offsets(offl, A.off, g);
  PairLanes pl;
  init_pair_lanes(g, pl);
  for (int i = lane; i < A.bins; i += 64) lng[i] = A.lng[i];
  for (int i = lane; i <= A.bins; i += 64) edges[i] = A.bin_edges[i];
  for (int i = lane; i < hb; i += 64) hist[i] = A.hist[i];
  stage_lattice(lat, A.compact, g, 0);
  __syncthreads();
  int mti = A.mt_index[0];
  MtWin win{0u, kMtWinEmpty};
  const SeqGeo sg = get_seq_geo(gw);
  const ImageLanes il = image_lanes(sg);
  const int bins = gw[kSeqGeoWords + 0], start_idx = gw[kSeqGeoWords + 1];
  const int end_idx = gw[kSeqGeoWords + 2], nbr_swap = gw[kSeqGeoWords + 3];
  const double wl_f = A.wl_f;
  const long long cadence = (long long)(int)(0.02 * (double)(float)g.n_atoms);
  double e_un = ref_total_energy(lat, g, offl, vex);
  const BinMap bmap = bin_map(edges, bins);
  int ibin = wl_bin_index(e_un, edges, bins);  // bin of e_un, kept with it
  // ln g of ibin (0 outside 1..bins), kept with it: lane 0 is the only
  // writer of lng and writes this value back after every trial
  double lcur = (ibin >= 1 && ibin <= bins) ? lng[ibin - 1] : 0.0;
  long long accepted = 0;
  const long long total = (long long)A.mc_sweeps * g.n_atoms;
  // trials until the next histogram update: i % cadence == 0, counted down
  // (a 64-bit remainder per trial costs more than the rest of the decision)
  long long to_hit = cadence;
  for (long long i = 1; i <= total; ++i) {
    const SiteXYZ r1 = random_site_dev(sg, st, mti, win);
    const SiteXYZ r2 =
        nbr_swap ? random_nbr_dev(sg, r1, st, mti, win) : random_site_dev(sg, st, mti, win);
    const int a1 = padded_addr_xyz(sg, r1.x, r1.y, r1.z);
    const int a2 = padded_addr_xyz(sg, r2.x, r2.y, r2.z);
    const int sub1 = sub_of(sg.lattice, r1.x & 1, r1.y & 1);
    const int sub2 = sub_of(sg.lattice, r2.x & 1, r2.y & 1);
    const int s1 = wave_uniform(lat[a1]), s2 = wave_uniform(lat[a2]);
    // The reference also evaluates pair_energy and swaps when the species
    // are equal; neither changes the state, so both are skipped here.
    double e_sw = e_un;
    if (s1 != s2) {
      // energies before and after the swap from one gather of the unswapped lattice
      double pu, ps;
      pair_energy_swap_lanes<KEY>(lat, sg, offl, vex, pl, a1, sub1, r1, a2, sub2, r2, s1, s2, sumbuf, pu, ps);
      e_sw = e_un - pu + ps;
    }
    bool acc = false;
    // e_sw == e_un when the species are equal (no swap): same bin
    int jbin = s1 != s2 ? wl_bin_index(e_sw, bmap) : ibin;
    const bool hit = cadence > 0 && --to_hit == 0;
    if (hit) to_hit = cadence;
    if (jbin > start_idx - 1 && jbin < end_idx + 1) {
      const double lj = lng[jbin - 1];
      const double u = genrand_dev(st, mti, win);
      if (log_lt_dev_uniform(u, lcur - lj)) {
        acc = true;
        ++accepted;
        e_un = e_sw;
        ibin = jbin;
        lcur = lj;
      } else {
        jbin = ibin;
      }
    } else {
      jbin = ibin;
    }
    if (s1 != s2 && acc) put_pair(lat, sg, il, r1, sub1, (int8_t)s2, r2, sub2, (int8_t)s1);
    // a walker outside its window would index outside the reference's
    // arrays; such updates are dropped
    const bool in_range = jbin >= 1 && jbin <= bins;
    if (in_range) lcur = lcur + wl_f;
    if (lane == 0) {
      if (hit && jbin >= start_idx && jbin <= end_idx) hist[jbin - start_idx] += 1.0;
      if (in_range) lng[jbin - 1] = lcur;
    }
    wave_lds_order();  // one wavefront: the next trial's LDS reads follow these writes
  }
  __syncthreads();
  unstage_lattice(lat, A.compact, g, 0);
  for (int i = lane; i < A.bins; i += 64) A.lng[i] = lng[i];
  for (int i = lane; i < hb; i += 64) A.hist[i] = hist[i];
  for (int i = lane; i < 624; i += 64) A.mt[i] = st[i];
  if (lane == 0) {
    A.mt_index[0] = mti;
    A.accepted[0] = accepted;
  }
}

// ------------------------------------------------------------------
// `sweeps` in speculative batches (bwl_spec.h); the call and its results are
// those of k_wl_sweeps.  A trial whose new energy lies inside the window
// draws one number after its sites', so trial t of a batch is foreseen to
// start t * len draws on, len by whether the walker is inside its window; a
// trial that goes otherwise ends its batch.  The energies of the batch's 8
// trials are formed together (8 lanes each); the decisions too, from one
// trial that changes the walker to the next (a decision at a time on the
// scalar unit costs a round trip of about 60 cycles for every branch on a
// vector result).
// ------------------------------------------------------------------
template <int KEY>
__global__ __launch_bounds__(kSpecThreads) void k_wl_sweeps_spec(const WlArgs *__restrict__ args) {
  using D = SpecDims<KEY>;
  extern __shared__ __align__(16) uint8_t smem[];
  const WlArgs &A = args[blockIdx.x];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = wave_uniform(tid >> 6);
  const SeqGeo g = seq_geo(A.g);
  const int S = g.S, n_atoms = A.g.n_atoms;
  const uint32_t inv_S = inverse_of(S);
  const int bins = A.bins, start_idx = A.start_idx, end_idx = A.end_idx;
  const int hb = end_idx - start_idx + 1;
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
  double *lng = (double *)take(sizeof(double) * bins);
  double *hist = (double *)take(sizeof(double) * hb);
  double *ebuf = (double *)take(sizeof(double) * 2 * kEnergyChunk);
  int32_t *offp = (int32_t *)take(4 * D::NSUB * D::R * D::ML);
  uint8_t *adj = take(D::TS * D::TS * D::TS);

  for (int i = tid; i < 624; i += kSpecThreads) raw[i] = A.mt[i];
  for (int i = tid; i < S * S * D::R; i += kSpecThreads) vex[i] = A.vex[i];
  for (int i = tid; i < bins; i += kSpecThreads) lng[i] = A.lng[i];
  for (int i = tid; i < hb; i += kSpecThreads) hist[i] = A.hist[i];
  stage_spec_tables<KEY>(offp, adj, A.off);
  stage_codes(lat, A.compact, g, D::NSUB, S);
  __syncthreads();
  ring_start<D::LAT>(g, raw, tem, rsite);
  const SpecLds L{lat, offp, vex, adj};
  double e_un = spec_total_energy<KEY>(L, g, n_atoms, S, inv_S, ebuf);
  if (wave != 0) {
    spec_helper<D::LAT>(g, raw, tem, rsite, cmd, [](int) {});
  } else {
    MtRing ring{raw, tem, rsite, cmd, 0, wave_uniform(A.mt_index[0]), false};
    const int trial = lane >> 3, w = (lane >> 2) & 1, shell = lane & 3;
    const bool nbr_swap = A.nbr_swap != 0;
    const int drawn = nbr_swap ? 4 : 6;  // by a trial's sites
    const double wl_f = A.wl_f;
    const int cadence = wave_uniform((int)(0.02 * (double)(float)n_atoms));
    const BinMap bmap = bin_map(A.bin_edges, bins);
    // x = (e - e0) / range * bins as one multiply-add, good to 1e-9 while
    // |e0 / range * bins| and |x| stay below 1e6: the bin is its truncation
    // unless x lies within 1e-6 of an integer (then the reference's form)
    const double slope = bmap.rinv * bmap.nb, shift = -(bmap.e0 * slope);
    // ... and while no ln g reaches 1e10 in this call (see below)
    bool small = true;
    const double grown = fabs(wl_f) * ((double)A.mc_sweeps * (double)n_atoms);
    for (int i = lane; i < bins; i += 64) small = small && fabs(lng[i]) + grown < 1e10;
    const bool quick = wave_uniform(fabs(shift) < 1e6) != 0 && __ballot(!small) == 0;
    int ibin = wave_uniform(wl_bin_index(e_un, A.bin_edges, bins));  // bin of e_un, kept with it
    auto in_range = [&](int b) { return b >= 1 && b <= bins; };
    auto in_window = [&](int b) { return b >= start_idx && b <= end_idx; };
    // ln g of ibin, kept here and written back when the walker leaves the bin
    double lcur = in_range(ibin) ? lng[ibin - 1] : 0.0;
    long long accepted = 0;
    long long left = (long long)wave_uniform(A.mc_sweeps) * n_atoms;
    int to_hit = cadence;
    auto count_visits = [&](int n) {  // the cadence-th trials among the next n, all ending in ibin
      if (cadence <= 0) return;
      while (__builtin_expect(n >= to_hit, 0)) {
        n -= to_hit;
        to_hit = cadence;
        if (in_window(ibin) && lane == 0) hist[ibin - start_idx] += 1.0;
      }
      to_hit -= n;
    };
    while (left > 0) {
      const bool inside = wave_uniform(in_window(ibin)) != 0;  // trials foreseen to draw for the decision
      const int len = drawn + (inside ? 1 : 0);
      ring_ensure(ring, 7 * kBatch + 2);
      const uint2 s1 = *ring_at(ring, rsite, len * trial);
      const SiteXYZ sa = unpack_xyz(s1.x);
      uint2 s2;
      if (nbr_swap) {
        const SiteXYZ sn = nbr_of_draw(g, sa, *ring_at(ring, tem, len * trial + 3));
        s2 = make_uint2(pack_xyz(sn), (uint32_t)spec_addr<D::LAT>(g, sn));
      } else {
        s2 = *ring_at(ring, rsite, len * trial + 3);
      }
      const uint32_t ru = *ring_at(ring, tem, len * trial + drawn);
      const SiteXYZ sb = unpack_xyz(s2.x);
      const int ca = lat[s1.y], cb = lat[s2.y];
      const bool differ = ca != cb;
      const unsigned long long same = __ballot(!differ);
      const SiteXYZ own = w ? sb : sa, oth = w ? sa : sb;
      const int c_own = w ? cb : ca, c_oth = w ? ca : cb;
      double pu, ps;
      spec_pair_energies<KEY>(L, g, S, inv_S, shell, own, oth, (int)(w ? s2.y : s1.y), c_own, c_oth, pu, ps);
      const unsigned long long conf = __ballot(batch_conflict(g, D::RC, s1.x, s2.x));
      // the float logarithm decides when clear of its threshold by 1e-4
      // (its error is below 1e-5); a drawn 0 goes to the full comparison
      const double lf = ru ? (double)__logf((float)((double)ru * (1.0 / 4294967296.0))) : NAN;
      const double surely = lf + 1e-4, hardly = lf - 1e-4;
      int nt = wave_uniform(left < kBatch ? (int)left : kBatch);
      int t0 = 0, off = 0;
      uint32_t swaps = 0;
      // The decisions, as far at a time as the next trial that changes the
      // walker: until then every trial sees the same energy, and a ln g that
      // has grown by wl_f per trial since (as a product here, which is near
      // enough for a decision that is clear by 1e-4: below 1e10 a sum of 8
      // rounds by less than 1e-5; added up trial by trial where it is kept).
      for (;;) {
        t0 = wave_uniform(t0);
        nt = wave_uniform(nt);
        ibin = wave_uniform(ibin);
        to_hit = wave_uniform(to_hit);
        const double e_sw = e_un - pu + ps;
        const double x = __builtin_fma(e_sw, slope, shift);
        const int xi = (int)x;
        const double f = fabs(x - (double)xi);
        const int jbin = differ ? xi + 1 : ibin;  // equal species: nothing moves
        const bool inw = in_window(jbin);
        const double lmem = lng[inw ? jbin - 1 : 0];
        const double grow = in_range(ibin) ? wl_f : 0.0;
        const double th = jbin == ibin ? 0.0 : __builtin_fma((double)(trial - t0), grow, lcur - lmem);
        const bool acc = surely < th;
        // trials for the full path below: another number of draws than
        // foreseen, or a bin or a decision too close to call here
        const bool close = differ & !((fabs(x) < 1e6) & (f > 1e-6) & (f < 1.0 - 1e-6));
        const bool full = !quick | (inw != inside) | close | (inside & !acc & !(hardly > th));
        const unsigned long long live = (~0ull << (8 * t0)) & (nt < 8 ? (1ull << (8 * nt)) - 1ull : ~0ull);
        const unsigned long long fulls = __ballot(full) & live;
        const unsigned long long events = fulls | (__ballot(acc & inw & differ) & live);
        const int te = events ? (__ffsll((long long)events) - 1) >> 3 : nt;
        // trials t0 .. te-1: rejected, or accepted without a change
        if (te > t0) {
          if (inside) accepted += __popcll(same & live & (te < 8 ? (1ull << (8 * te)) - 1ull : ~0ull) & 0x0101010101010101ull);
          const int n = te - t0;
          if (n & 1) lcur = lcur + grow;
          if (n & 2) lcur = (lcur + grow) + grow;
          if (n & 4) lcur = (((lcur + grow) + grow) + grow) + grow;
          if (n & 8) lcur = (((((((lcur + grow) + grow) + grow) + grow) + grow) + grow) + grow) + grow;
          count_visits(te - t0);
        }
        t0 = te;
        if (te >= nt) break;
        const int l = 8 * te;
        ++t0;
        if (__builtin_expect((fulls >> l) & 1ull, 0)) {
          // one trial in the reference's own terms; it ends the batch
          bool in1 = in_window(ibin), acc1 = in1;  // equal species: accepted (log u < 0) when it draws
          if (!((same >> l) & 1ull)) {
            const double e1 = readlane_d(e_sw, l);
            const int b1 = wave_uniform((int)(((e1 - bmap.e0) / bmap.range) * bmap.nb) + 1);
            in1 = in_window(b1);
            acc1 = false;
            if (in1) {
              const double l1 = b1 == ibin ? lcur : lng[b1 - 1];
              const uint32_t r = (uint32_t)__builtin_amdgcn_readlane((int)ru, l);
              acc1 = wave_uniform(log_lt_dev((double)r * (1.0 / 4294967296.0), lcur - l1)) != 0;
              if (acc1) {
                if (lane == 0 && in_range(ibin)) lng[ibin - 1] = lcur;
                wave_lds_order();
                e_un = e1;
                ibin = b1;
                lcur = l1;
                swaps |= 1u << te;
              }
            }
          }
          accepted += acc1 ? 1 : 0;
          if (in_range(ibin)) lcur = lcur + wl_f;
          count_visits(1);
          off = (in1 ? 1 : 0) - (inside ? 1 : 0);
          break;
        }
        ++accepted;
        if (lane == 0 && in_range(ibin)) lng[ibin - 1] = lcur;
        wave_lds_order();
        e_un = readlane_d(e_sw, l);
        const int to = __builtin_amdgcn_readlane(jbin, l);
        lcur = (to == ibin ? lcur : readlane_d(lmem, l)) + wl_f;
        ibin = to;
        count_visits(1);
        swaps |= 1u << te;
        // the first later trial that the swap reaches ends the batch
        const uint32_t reached = (uint32_t)(conf >> l) & 0xffu & (0xffu << t0);
        if (reached) nt = min(nt, __ffs((int)reached) - 1);
        if (t0 >= nt) break;
      }
      t0 = wave_uniform(t0);
      batch_write<D::LAT>(lat, g, ((swaps >> trial) & 1u) != 0, own, c_oth);
      ring.q = wave_uniform(ring.q + len * t0 + off);
      left -= t0;
    }
    if (lane == 0) {
      if (in_range(ibin)) lng[ibin - 1] = lcur;
      A.accepted[0] = accepted;
    }
    spec_command(ring, kCmdExit);
    ring_finish(ring, A.mt, A.mt_index);
  }
  __syncthreads();
  unstage_codes(lat, A.compact, g, D::NSUB, inv_S);
  for (int i = tid; i < bins; i += kSpecThreads) A.lng[i] = lng[i];
  for (int i = tid; i < hb; i += kSpecThreads) A.hist[i] = hist[i];
}

// Window average after `sweeps` (wang-landau.F90:628-631): ln g and the
// visit histogram summed over a window's walkers in walker order, divided
// by the number of walkers, and written back to every walker of the window.
// One thread per (window, bin).
__global__ void k_wl_average(double *lng, double *hist, int n_windows, int wpw, int bins,
                             int hist_stride) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int per = bins + hist_stride;
  if (t >= n_windows * per) return;
  const int w = t / per;
  const int b = t - w * per;
  double *base;
  int stride;
  if (b < bins) {
    base = lng + (size_t)w * wpw * bins + b;
    stride = bins;
  } else {
    base = hist + (size_t)w * wpw * hist_stride + (b - bins);
    stride = hist_stride;
  }
  double s = base[0];
  for (int k = 1; k < wpw; ++k) s = s + base[(size_t)k * stride];
  s = s / (double)wpw;
  for (int k = 0; k < wpw; ++k) base[(size_t)k * stride] = s;
}

// ------------------------------------------------------------------
// replica_exchange (wang-landau.F90:1392-1501).
// k_wl_energies: e_unswapped = full_energy(config) of every walker
// (bw_hamiltonian.f90:58-81 order), one wavefront per walker.
// ------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_wl_energies(const WlArgs *__restrict__ args, double *E) {
  extern __shared__ __align__(16) uint8_t smem[];
  const WlArgs &A = args[blockIdx.x];
  const Geo &g = A.g;
  int8_t *lat = (int8_t *)smem;
  size_t o = (g.lds_bytes + 15) & ~15;
  double *vex = (double *)(smem + o);
  o += sizeof(double) * g.S * g.S * g.R;
  int32_t *offl = (int32_t *)(smem + o);
  for (int i = threadIdx.x; i < g.S * g.S * g.R; i += 64) vex[i] = A.vex[i];
  stage_offsets(offl, A.off, g);
  stage_lattice(lat, A.compact, g, 0);
  __syncthreads();
  const double e = ref_total_energy(lat, g, offl, vex);
  if (threadIdx.x == 0) E[blockIdx.x] = e;
}

// Reference-order total energies of walkers by whole workgroups
// (spec_total_energy): block w is Wang-Landau walker w, or walker w of
// nested-sampling run blockIdx.y with its energy jitter.  (No table of list
// positions, which took longer than a small box's energy: 8 walkers of bcc
// 4^3 with four shells 58 us with it, 35 by one wavefront each.)
template <int KEY>
__device__ __forceinline__ double walker_energy(const Geo &geo, const int8_t *compact, const int32_t *off,
                                                const double *v, uint8_t *smem) {
  using D = SpecDims<KEY>;
  const SeqGeo g = seq_geo(geo);
  const int S = g.S;
  uint8_t *p = smem;
  auto take = [&](size_t bytes) {
    uint8_t *at = p;
    p += (bytes + 15) & ~(size_t)15;
    return at;
  };
  int8_t *lat = (int8_t *)take(geo.lds_bytes);
  double *vex = (double *)take(sizeof(double) * S * S * D::R);
  double *ebuf = (double *)take(sizeof(double) * 2 * kEnergyChunk);
  int32_t *offp = (int32_t *)take(4 * D::NSUB * D::R * D::ML);
  for (int i = threadIdx.x; i < S * S * D::R; i += kSpecThreads) vex[i] = v[i];
  stage_spec_offsets<KEY>(offp, off);
  stage_codes(lat, compact, g, D::NSUB, S);
  __syncthreads();
  return spec_total_energy<KEY>(SpecLds{lat, offp, vex, nullptr}, g, geo.n_atoms, S, inverse_of(S), ebuf);
}

template <int KEY>
__global__ __launch_bounds__(kSpecThreads) void k_wl_energies_spec(const WlArgs *__restrict__ args, double *E) {
  extern __shared__ __align__(16) uint8_t smem[];
  const WlArgs &A = args[blockIdx.x];
  const double e = walker_energy<KEY>(A.g, A.compact, A.off, A.vex, smem);
  if (threadIdx.x == 0) E[blockIdx.x] = e;
}

template <int KEY>
__global__ __launch_bounds__(kSpecThreads) void k_ns_energies_spec(const NsArgs *__restrict__ args) {
  extern __shared__ __align__(16) uint8_t smem[];
  const NsArgs &A = args[blockIdx.y];
  const int w = blockIdx.x;
  if (w >= A.n_walkers) return;
  const double e = walker_energy<KEY>(A.g, A.walkers + (size_t)A.g.compact_bytes * w, A.off, A.vex, smem);
  if (threadIdx.x == 0) A.E[w] = e + A.rnde[w] * (double)1e-8f;
}

// The exchange decisions, one wavefront for the whole walker set (a few
// hundred random numbers at most).  Each walker's overlap location comes
// from the bin of its energy (:1406-1431).  For each pair of neighbouring
// windows (i, i+1), rank 0's stream (walker 0) shuffles the candidate rows
// of both windows (shuffle_rows, :1513-1524), the rows are matched greedily
// in shuffled order (:1447-1468), and each matched pair (a in window i, b in
// window i+1), in order, draws genrand() from a's stream and exchanges iff
// it is below exp(lng_a(bin_a) - lng_a(bin_b)) (:1476-1497).  All lanes
// follow the same control flow (the MT19937 helpers are whole-wavefront);
// lane 0 writes the shared rows and the outputs.
__global__ __launch_bounds__(64) void k_wl_exchange(WlExchangeArgs A) {
  extern __shared__ __align__(16) uint8_t smem[];
  const int lane = threadIdx.x;
  const int W = A.W, wpw = A.wpw, nwin = A.num_windows;
  uint32_t *st0 = (uint32_t *)smem;       // walker 0's stream
  uint32_t *st1 = st0 + 624;              // the deciding walker's stream
  int32_t *ibin = (int32_t *)(st1 + 624); // W
  int32_t *loc = ibin + W;                // W
  int32_t *lo = loc + W;                  // rows (walker, location) of window i
  int32_t *up = lo + 2 * wpw;             // rows of window i+1
  int32_t *pr = up + 2 * wpw;             // matched pairs, then their count
  for (int k = lane; k < W; k += 64) {
    const int b = wl_bin_index(A.E[k], A.bin_edges, A.bins);
    const int m = k / wpw + 1;  // the rank's window, 1-based
    bool lower = false, upper = false;
    if (m > 1) lower = b < A.windows[2 * (m - 2) + 1] + 1 && b > A.windows[2 * (m - 1)] - 1;
    if (m < nwin) upper = b > A.windows[2 * m] - 1 && b < A.windows[2 * (m - 1) + 1] + 1;
    ibin[k] = b;
    loc[k] = upper ? m : (lower ? m - 1 : 0);
    A.partner[k] = -1;
    A.accepted[k] = 0;
  }
  for (int i = lane; i < 624; i += 64) st0[i] = A.mt[i];
  int mti0 = A.mt_index[0];
  int nsw = 0;
  __syncthreads();
  for (int i = 1; i < nwin; ++i) {
    for (int j = lane; j < wpw; j += 64) {
      lo[2 * j] = (i - 1) * wpw + j;
      lo[2 * j + 1] = loc[(i - 1) * wpw + j];
      up[2 * j] = i * wpw + j;
      up[2 * j + 1] = loc[i * wpw + j];
    }
    __syncthreads();
    for (int side = 0; side < 2; ++side) {
      int32_t *rows = side ? up : lo;
      for (int t = wpw; t >= 2; --t) {
        const double u = genrand_dev(st0, mti0);
        int r = 1 + (int)(u * (double)t);
        if (r > wpw) r = wpw;
        if (lane == 0) {
          const int32_t a0 = rows[2 * (t - 1)], a1 = rows[2 * (t - 1) + 1];
          rows[2 * (t - 1)] = rows[2 * (r - 1)];
          rows[2 * (t - 1) + 1] = rows[2 * (r - 1) + 1];
          rows[2 * (r - 1)] = a0;
          rows[2 * (r - 1) + 1] = a1;
        }
        __syncthreads();
      }
    }
    if (lane == 0) {
      int np = 0;
      for (int j = 0; j < wpw; ++j) {
        if (lo[2 * j + 1] == 0) continue;
        for (int k = 0; k < wpw; ++k) {
          if (up[2 * k + 1] == 0) continue;
          if (lo[2 * j + 1] == up[2 * k + 1]) {
            pr[2 * np] = lo[2 * j];
            pr[2 * np + 1] = up[2 * k];
            ++np;
            lo[2 * j] = lo[2 * j + 1] = 0;
            up[2 * k] = up[2 * k + 1] = 0;
          }
        }
      }
      pr[2 * wpw] = np;
    }
    __syncthreads();
    const int np = pr[2 * wpw];
    for (int j = 0; j < np; ++j) {
      const int a = pr[2 * j], b = pr[2 * j + 1];
      double u;
      const int mti_a = a == 0 ? 0 : A.mt_index[a];
      if (a == 0) {
        u = genrand_dev(st0, mti0);
      } else if (mti_a < 624) {
        // no twist due: the draw is the next stored word, tempered
        u = (double)mt_temper(A.mt[(size_t)624 * a + mti_a]) * (1.0 / 4294967296.0);
        __syncthreads();  // every lane has read the index before lane 0 moves it
        if (lane == 0) A.mt_index[a] = mti_a + 1;
      } else {
        for (int q = lane; q < 624; q += 64) st1[q] = A.mt[(size_t)624 * a + q];
        int m1 = A.mt_index[a];
        __syncthreads();
        u = genrand_dev(st1, m1);
        __syncthreads();
        for (int q = lane; q < 624; q += 64) A.mt[(size_t)624 * a + q] = st1[q];
        if (lane == 0) A.mt_index[a] = m1;
        __syncthreads();
      }
      // ibin of a matched walker lies inside both windows' bins
      const double x = A.lng[(size_t)A.bins * a + ibin[a] - 1] - A.lng[(size_t)A.bins * a + ibin[b] - 1];
      const bool acc = x >= 0.0 || lt_exp_dev(u, x);  // u < 1 <= exp(x) when x >= 0
      if (lane == 0) {
        A.partner[a] = b;
        A.partner[b] = a;
        A.accepted[a] = A.accepted[b] = acc ? 1 : 0;
        if (acc) {
          A.swaps[2 * nsw] = a;
          A.swaps[2 * nsw + 1] = b;
        }
      }
      nsw += acc ? 1 : 0;
    }
    __syncthreads();
  }
  for (int i = lane; i < 624; i += 64) A.mt[i] = st0[i];
  if (lane == 0) {
    A.mt_index[0] = mti0;
    A.n_swaps[0] = nsw;
  }
}

// Exchange the configurations of the accepted pairs: block j swaps pair j.
__global__ void k_wl_swap_configs(int8_t *walkers, long long bytes, const int32_t *swaps,
                                  const int32_t *n_swaps) {
  const int j = blockIdx.x;
  if (j >= n_swaps[0]) return;
  int8_t *a = walkers + bytes * swaps[2 * j];
  int8_t *b = walkers + bytes * swaps[2 * j + 1];
  for (long long i = threadIdx.x; i < bytes; i += blockDim.x) {
    const int8_t t = a[i];
    a[i] = b[i];
    b[i] = t;
  }
}

// ------------------------------------------------------------------
// enter_energy_window (wang-landau.F90:643-741) for one walker.
// ------------------------------------------------------------------
template <int KEY>
__global__ __launch_bounds__(64) void k_wl_enter(const WlEnterArgs *__restrict__ args) {
  extern __shared__ __align__(16) uint8_t smem[];
  const WlEnterArgs &A = args[blockIdx.x];
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
  // the trial loop's geometry (see put_seq_geo)
  int32_t *gw = (int32_t *)(smem + ((o + 15) & ~(size_t)15));

  for (int i = lane; i < 624; i += 64) st[i] = A.mt[i];
  for (int i = lane; i < g.S * g.S * g.R; i += 64) vex[i] = A.vex[i];
  put_seq_geo(gw, g);
  put_loop64(gw, 0, (unsigned long long)__double_as_longlong(A.min_e));
  put_loop64(gw, 2, (unsigned long long)__double_as_longlong(A.max_e));
  put_loop64(gw, 4, (unsigned long long)__double_as_longlong(A.denom));
  put_loop64(gw, 6, (unsigned long long)A.period);
  put_loop64(gw, 8, (unsigned long long)A.budget);
  stage_offsets(offl, A.off, g);
  PairLanes pl;
  init_pair_lanes(g, pl);
  stage_lattice(lat, A.compact, g, 0);
  __syncthreads();
  int mti = A.mt_index[0];
  MtWin win{0u, kMtWinEmpty};
  const double min_e = __longlong_as_double((long long)get_loop64(gw, 0));
  const double max_e = __longlong_as_double((long long)get_loop64(gw, 2));
  const double denom = __longlong_as_double((long long)get_loop64(gw, 4));
  const long long period = (long long)get_loop64(gw, 6), budget = (long long)get_loop64(gw, 8);
  const double target = (min_e + max_e) / 2.0;
  const double cond = fabs(max_e - min_e) * 0.1;
  double e_un = A.init_e ? ref_total_energy(lat, g, offl, vex) : A.e_unswapped[0];
  long long isteps = A.i_steps[0];
  long long trials = A.trials[0];
  long long made = 0;
  bool skip = A.resume[0] != 0;
  int status = 0;
  const SeqGeo sg = get_seq_geo(gw);
  const ImageLanes il = image_lanes(sg);
  // iterations until isteps is next a multiple of period, counted down
  long long to_period = period - isteps % period;
  for (;;) {
    if (!skip) {
      ++isteps;
      if (--to_period == 0) {
        isteps = 0;
        status = 1;  // the host re-runs initial_setup, then resumes here
        break;
      }
    }
    skip = false;
    if (e_un < max_e - cond && e_un > min_e + cond) {
      e_un = ref_total_energy(lat, g, offl, vex);
      if (e_un < max_e - cond && e_un > min_e + cond) {
        status = 0;
        break;
      }
      continue;
    }
    if (made >= budget) {
      status = 2;
      skip = true;  // resume before this iteration's trial
      break;
    }
    ++made;
    ++trials;
    const SiteXYZ r1 = random_site_dev(sg, st, mti, win);
    const SiteXYZ r2 = random_site_dev(sg, st, mti, win);
    const int a1 = padded_addr_xyz(sg, r1.x, r1.y, r1.z);
    const int a2 = padded_addr_xyz(sg, r2.x, r2.y, r2.z);
    const int s1 = lat[a1], s2 = lat[a2];
    if (s1 != s2) {
      const int sub1 = sub_of(sg.lattice, r1.x & 1, r1.y & 1);
      const int sub2 = sub_of(sg.lattice, r2.x & 1, r2.y & 1);
      // energies before and after the swap from one gather of the unswapped lattice
      double pu, ps;
      pair_energy_swap_lanes<KEY>(lat, sg, offl, vex, pl, a1, sub1, r1, a2, sub2, r2, s1, s2, sumbuf, pu, ps);
      const double e_sw = e_un - pu + ps;
      const double de = ((e_sw - target) * (e_sw - target) - (e_un - target) * (e_un - target)) /
                        denom;
      const double u = genrand_dev(st, mti, win);
      const bool acc = log_lt_dev(u, -de);
      if (acc) e_un = e_sw;
      if (acc) put_pair(lat, sg, il, r1, sub1, (int8_t)s2, r2, sub2, (int8_t)s1);
    }
  }
  __syncthreads();
  unstage_lattice(lat, A.compact, g, 0);
  for (int i = lane; i < 624; i += 64) A.mt[i] = st[i];
  if (lane == 0) {
    A.mt_index[0] = mti;
    A.e_unswapped[0] = e_un;
    A.i_steps[0] = isteps;
    A.trials[0] = trials;
    A.resume[0] = (status == 1 || status == 2) ? 1 : 0;
    A.status[0] = status;
  }
}

// ------------------------------------------------------------------
// Windowed pair counts of radial_densities: for every occupied site of
// species a and every window offset whose minimum-image distance falls on
// shell l, the species b at that offset: H(a, b, l) += 1.  The lattice is
// read from HBM (it is small and stays in L2); counts are packed 8 bits per
// species per shell and flushed to a per-block LDS histogram, which goes to
// the block's part of the output (the host adds the parts up: integers, so
// the split does not show).
// ------------------------------------------------------------------
template <bool NEAR>
__global__ __launch_bounds__(256) void k_asro(AsroArgs A) {
  __shared__ unsigned int lh[kMaxSpecies * kMaxSpecies * kMaxAsroShells];
  const Geo &g = A.g;
  const int S = g.S;
  const int hsize = S * S * A.wc;
  for (int i = threadIdx.x; i < hsize; i += blockDim.x) lh[i] = 0;
  __syncthreads();
  const int cells = g.n[0] * g.n[1] * g.n[2];
  const int nsites = g.nsub * cells;
  for (int idx = blockIdx.x * blockDim.x + threadIdx.x; idx < nsites;
       idx += gridDim.x * blockDim.x) {
    const int s = idx / cells;
    int r = idx - s * cells;
    const int cz = r / (g.n[0] * g.n[1]);
    r -= cz * g.n[0] * g.n[1];
    const int cy = r / g.n[0];
    const int cx = r - cy * g.n[0];
    int bx, by, bz;
    sub_bits(g.lattice, s, bx, by, bz);
    const int x = 2 * cx + bx, y = 2 * cy + by, z = 2 * cz + bz;
    const int a = A.compact[idx];
    if (a <= 0) continue;
    for (int l = 0; l < A.wc; ++l) {
      uint64_t c = 0;
      int k = 0;
      for (int t = A.shell_start[l]; t < A.shell_start[l + 1]; ++t) {
        const int32_t d = NEAR ? A.near[t] : A.off[t];
        int xx = x + (int8_t)d, yy = y + (int8_t)(d >> 8), zz = z + (int8_t)(d >> 16);
        xx = xx < 0 ? xx + g.m[0] : (xx >= g.m[0] ? xx - g.m[0] : xx);
        yy = yy < 0 ? yy + g.m[1] : (yy >= g.m[1] ? yy - g.m[1] : yy);
        zz = zz < 0 ? zz + g.m[2] : (zz >= g.m[2] ? zz - g.m[2] : zz);
        const int b = A.compact[compact_addr(g, sub_of(g.lattice, xx & 1, yy & 1), xx >> 1, yy >> 1,
                                             zz >> 1)];
        c += (uint64_t)1 << (8 * (b - 1));
        if (++k == 255 || t + 1 == A.shell_start[l + 1]) {
          for (int bb = 0; bb < S; ++bb) {
            const unsigned q = (unsigned)(c >> (8 * bb)) & 0xffu;
            if (q) atomicAdd(&lh[(a - 1) + S * (bb + S * l)], q);
          }
          c = 0;
          k = 0;
        }
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < hsize; i += blockDim.x)
    A.parts[(size_t)blockIdx.x * hsize + i] = lh[i];
}

// ------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------
namespace {
const void *wl_sweeps_kernel(int key) { BWL_KERNEL_FOR_PAIR_SUM_KEY(k_wl_sweeps, key) }
const void *ns_kernel(int key) { BWL_KERNEL_FOR_PAIR_SUM_KEY(k_ns, key) }
const void *wl_enter_kernel(int key) { BWL_KERNEL_FOR_PAIR_SUM_KEY(k_wl_enter, key) }
const void *wl_sweeps_spec_kernel(int key) { BWL_KERNEL_FOR_SPEC_KEY(k_wl_sweeps_spec, key) }
const void *ns_spec_kernel(int key) { BWL_KERNEL_FOR_SPEC_KEY(k_ns_spec, key) }
const void *wl_energies_spec_kernel(int key) { BWL_KERNEL_FOR_SPEC_KEY(k_wl_energies_spec, key) }
const void *ns_energies_spec_kernel(int key) { BWL_KERNEL_FOR_SPEC_KEY(k_ns_energies_spec, key) }

}  // namespace

size_t ns_spec_lds_bytes(const Geo &g, int n_walkers) {
  return spec_table_bytes(g) + spec_ring_bytes() + spec_align(sizeof(double) * (size_t)n_walkers);
}

size_t wl_spec_lds_bytes(const Geo &g, int bins, int window_bins) {
  return spec_table_bytes(g) + spec_ring_bytes() + spec_align(sizeof(double) * (size_t)bins) +
         spec_align(sizeof(double) * (size_t)window_bins) + spec_energy_bytes();
}

size_t energies_spec_lds_bytes(const Geo &g) { return spec_table_bytes(g) + spec_energy_bytes(); }

size_t ns_lds_bytes(const Geo &g, int n_walkers) {
  return seq_geo_region((size_t)((g.lds_bytes + 15) & ~15) + 624 * 4 + kSumBufBytes +
                        sizeof(double) * g.S * g.S * g.R + sizeof(double) * (size_t)n_walkers +
                        sizeof(int32_t) * g.nsub * g.z);
}

constexpr double kWalkersFar = 0.125;  // see spec_pays

hipError_t launch_ns(const NsArgs *args_dev, int n, const SeqPick &pick, int max_walkers, const SeqPick &energies,
                     hipStream_t s) {
  void *kargs[] = {(void *)&args_dev};
  const dim3 walkers(max_walkers, n);
  const void *fn = pick.spec ? ns_spec_kernel(pick.key) : nullptr;
  const bool spec = spec_pays(fn, n, pick, kWalkersFar);
  // (energies in workgroups of one wavefront before runs of one: 1024 runs
  // after workgroups of four were spread unevenly over the SIMDs, fcc 3^3 with
  // four shells 2.34 ms against 1.81)
  const hipError_t e =
      energies.spec && spec
          ? launch_dynamic(ns_energies_spec_kernel(energies.key), walkers, kSpecThreads, kargs, energies.lds_spec, s)
          : launch_dynamic((const void *)k_ns_energies, walkers, 64, kargs, energies.lds, s);
  if (e != hipSuccess) return e;
  if (spec) return launch_dynamic(fn, dim3(n), kSpecThreads, kargs, pick.lds_spec, s);
  return launch_dynamic(ns_kernel(pick.key), dim3(n), 64, kargs, pick.lds, s);
}

size_t ns_energies_lds_bytes(const Geo &g) {
  return (size_t)((g.lds_bytes + 15) & ~15) + sizeof(double) * g.S * g.S * g.R +
         sizeof(int32_t) * g.nsub * g.z;
}

size_t wl_lds_bytes(const Geo &g, int bins, int window_bins) {
  return seq_geo_region((size_t)((g.lds_bytes + 15) & ~15) + 624 * 4 + kSumBufBytes +
                        sizeof(double) * g.S * g.S * g.R +
                        sizeof(double) * (size_t)(2 * bins + 1 + window_bins) + sizeof(int32_t) * g.nsub * g.z);
}

hipError_t launch_wl_sweeps(const WlArgs *args_dev, int n, const SeqPick &pick, hipStream_t s) {
  void *kargs[] = {(void *)&args_dev};
  const void *fn = pick.spec ? wl_sweeps_spec_kernel(pick.key) : nullptr;
  if (spec_pays(fn, n, pick, kWalkersFar)) return launch_dynamic(fn, dim3(n), kSpecThreads, kargs, pick.lds_spec, s);
  return launch_dynamic(wl_sweeps_kernel(pick.key), dim3(n), 64, kargs, pick.lds, s);
}

hipError_t launch_wl_average(double *lng, double *hist, int n_windows, int wpw, int bins,
                             int hist_stride, hipStream_t s) {
  const int total = n_windows * (bins + hist_stride);
  hipLaunchKernelGGL(k_wl_average, dim3((total + 255) / 256), dim3(256), 0, s, lng, hist,
                     n_windows, wpw, bins, hist_stride);
  return hipGetLastError();
}

hipError_t launch_wl_energies(const WlArgs *args_dev, int n, double *E, const SeqPick &pick, hipStream_t s) {
  void *kargs[] = {(void *)&args_dev, (void *)&E};
  if (pick.spec)
    return launch_dynamic(wl_energies_spec_kernel(pick.key), dim3(n), kSpecThreads, kargs, pick.lds_spec, s);
  return launch_dynamic((const void *)k_wl_energies, dim3(n), 64, kargs, pick.lds, s);
}

size_t wl_exchange_lds_bytes(int W, int wpw) {
  return 2 * 624 * 4 + sizeof(int32_t) * (size_t)(2 * W + 6 * wpw + 1);
}

hipError_t launch_wl_exchange(const WlExchangeArgs &a, size_t lds, hipStream_t s) {
  hipError_t e = hipFuncSetAttribute((const void *)k_wl_exchange,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_wl_exchange, dim3(1), dim3(64), lds, s, a);
  return hipGetLastError();
}

hipError_t launch_wl_swap_configs(int8_t *walkers, long long bytes, const int32_t *swaps,
                                  const int32_t *n_swaps, int max_pairs, hipStream_t s) {
  hipLaunchKernelGGL(k_wl_swap_configs, dim3(max_pairs > 0 ? max_pairs : 1), dim3(256), 0, s,
                     walkers, bytes, swaps, n_swaps);
  return hipGetLastError();
}

size_t wl_enter_lds_bytes(const Geo &g) {
  return seq_geo_region((size_t)((g.lds_bytes + 15) & ~15) + 624 * 4 + kSumBufBytes +
                        sizeof(double) * g.S * g.S * g.R + sizeof(int32_t) * g.nsub * g.z);
}

hipError_t launch_wl_enter(const WlEnterArgs *args_dev, int n, size_t lds, hipStream_t s, int key) {
  const void *fn = wl_enter_kernel(key);
  hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  void *kargs[] = {(void *)&args_dev};
  return hipLaunchKernel(fn, dim3(n), dim3(64), kargs, lds, s);
}

// blocks of 256 sites or more, at most 1024 with at most 2^18 counts between
// them
int asro_blocks(const Geo &g, int wc) {
  const int b = (g.nsub * g.n[0] * g.n[1] * g.n[2] + 255) / 256, most = (1 << 18) / (g.S * g.S * wc);
  return b < most ? (b < 1024 ? b : 1024) : (most < 1024 ? most : 1024);
}

hipError_t launch_asro(const AsroArgs &a, int blocks, hipStream_t s) {
  if (a.off)
    hipLaunchKernelGGL(k_asro<false>, dim3(blocks), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(k_asro<true>, dim3(blocks), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace bwl
