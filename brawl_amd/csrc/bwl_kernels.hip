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
#include "bwl_seq_batches.h"

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

namespace {
const void *metro_seq_kernel(int key) { BWL_KERNEL_FOR_PAIR_SUM_KEY(k_metro_seq, key) }
const void *metro_seq_batch_kernel(int key) { BWL_KERNEL_FOR_PAIR_SUM_KEY(k_metro_seq_batch, key) }
const void *metro_seq_spec_kernel(int key) { BWL_KERNEL_FOR_SPEC_KEY(k_metro_seq_spec, key) }
const void *metro_seq_spec_batch_kernel(int key) { BWL_KERNEL_FOR_SPEC_KEY(k_metro_seq_spec_batch, key) }
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
  if (pick.spec) {
    const void *singly = metro_seq_singly_kernel(pick, false);
    return launch_dynamic(singly ? singly : metro_seq_spec_kernel(pick.key), dim3(1), kSpecThreads, kargs, pick.lds_spec, s);
  }
  return launch_dynamic(metro_seq_kernel(pick.key), dim3(1), 64, kargs, pick.lds, s);
}

hipError_t launch_metro_seq_batch(const SeqArgs *args_dev, int n, const SeqPick &pick, hipStream_t s) {
  void *kargs[] = {(void *)&args_dev};
  const void *fn = nullptr;
  if (pick.spec) fn = metro_seq_singly_kernel(pick, true);
  if (pick.spec && !fn) fn = metro_seq_spec_batch_kernel(pick.key);
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
