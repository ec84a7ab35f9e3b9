// bwl_spec.h -- the sequential samplers' trials in speculative batches.
//
// A sequential chain (bit-exact Metropolis, a nested-sampling walk, a
// Wang-Landau walker) is a dependent sequence of trials, and one trial at a
// time leaves a wavefront waiting: its site draws, its neighbour gather, its
// ordered sums and its decision follow each other, each a few LDS round
// trips, on lanes that mostly idle.  Here the wavefront looks a few trials
// ahead in the random stream: it takes their sites, reads their neighbours
// from the lattice as it is (or as it will be if they are accepted) and
// forms their energies side by side, then makes the decisions in order.  A
// later trial of the batch stands as long as no swap before it that went
// otherwise than foreseen touched a site within its reach (every pair of
// trials is tested at once) and its place in the stream was foreseen rightly;
// at the first that does not stand, the batch ends and the next begins
// there.  Every value and every order of addition is that of one trial at a
// time, so the chains are bit-identical.
//
// What bounds it is still latency, now of a batch: on this part a dependent
// vector instruction follows after 9 cycles (5 when independent), an LDS read
// or a shuffle after 57 to 65, and a branch on a vector result costs 60 to 75;
// so the per-trial control flow is kept on the scalar unit or in lanes, and
// decisions are taken several at a time.
//
// For lattices of up to 4 shells whose box is longer than twice the
// interaction range on every axis, so that a site sees another through at
// most one offset and never itself.  One workgroup of kSpecThreads per
// chain: wavefront 0 runs the trials; wavefront 1 keeps the stream ahead of
// it (draws and the sites they make, which depend on no state); all four
// stage the lattice and recount energies.
#pragma once

#include "bwl_seq.h"

namespace bwl {

constexpr int kSpecThreads = 256;
constexpr int kBatch = 8;

template <int KEY>
struct SpecDims {
  static constexpr int LAT = KEY / 16, R = KEY % 16;
  static constexpr int Z = shell_first<LAT>(R);
  static constexpr int ML = shell_max(LAT, R);  // a multiple of 4
  static constexpr int NSUB = LAT == 1 ? 4 : 2;
  static constexpr int RC = spec_rcut(LAT, R);
  static constexpr int TS = 2 * RC + 1;
};

template <int LAT>
__host__ __device__ constexpr int shell_len(int n) {
  return LAT == 1 ? kFccShellSize[n] : kBccShellSize[n];
}

// LDS tables of a speculative kernel beside the lattice.
//   off  [nsub][R][ML]: padded-layout neighbour offsets, each shell padded
//        with zeros to ML entries (read four at a time)
//   vex  V_ex as the reference lays it out
//   adj  [TS][TS][TS]: list position of the neighbour at an offset, 255 none
struct SpecLds {
  int8_t *lat;
  const int32_t *off;
  const double *vex;
  const uint8_t *adj;
};

template <int KEY>
__device__ inline void stage_spec_offsets(int32_t *offp, const int32_t *__restrict__ off) {
  using D = SpecDims<KEY>;
  for (int i = threadIdx.x; i < D::NSUB * D::R * D::ML; i += blockDim.x) {
    const int k = i % D::ML, n = (i / D::ML) % D::R, s = i / (D::ML * D::R);
    int first = 0, len = 0;
    for (int q = 0; q <= n; ++q) {
      first += len;
      len = shell_len<D::LAT>(q);
    }
    offp[i] = k < len ? off[s * D::Z + first + k] : 0;
  }
}

template <int KEY>
__device__ inline void stage_spec_tables(int32_t *offp, uint8_t *adj, const int32_t *__restrict__ off) {
  using D = SpecDims<KEY>;
  stage_spec_offsets<KEY>(offp, off);
  for (int i = threadIdx.x; i < D::TS * D::TS * D::TS; i += blockDim.x) {
    const int dx = i % D::TS - D::RC, dy = (i / D::TS) % D::TS - D::RC, dz = i / (D::TS * D::TS) - D::RC;
    int at = 255;
    for (int t = 0; t < D::Z; ++t) {
      const int8_t *v = D::LAT == 1 ? kFccOffsets[t] : kBccOffsets[t];
      if (v[0] == dx && v[1] == dy && v[2] == dz) at = t;
    }
    adj[i] = (uint8_t)at;
  }
}

// ------------------------------------------------------------------
// The stream as a ring of tempered draws and of the sites they make: the
// current block of 624 in one half, the next in the other, so that a window
// of draws never stops at a block's end.  Entry i of `site` is the site of
// draws i, i+1, i+2 (packed coordinates, LDS address).  While wavefront 0
// uses the current block, wavefront 1 makes the next one; the two meet at
// barriers (all wavefronts take part: the helpers wait for a command, see
// spec_helper): one when the current block is used up and its half may be
// overwritten, one before the first use of the new block.
// ------------------------------------------------------------------
constexpr int kRingWords = 2 * 624 + 8;  // the last 8 repeat the first 8

struct MtRing {
  uint32_t *raw, *tem;  // raw: the state after the newest block's twist
  uint2 *site;
  volatile int32_t *cmd;
  int half;    // 0 or 624: the current block's draws
  int q;       // draws of the current block consumed
  bool ready;  // the other half holds the next block
};

enum SpecCommand { kCmdExit, kCmdBlock, kCmdEnergy, kCmdLoad, kCmdStore, kCmdTurn };

__device__ inline uint32_t mt_untemper(uint32_t y) {
  y ^= y >> 18;
  y ^= (y << 15) & 0xefc60000u;
  uint32_t x = y;
#pragma unroll
  for (int i = 0; i < 5; ++i) x = y ^ ((x << 7) & 0x9d2c5680u);
  y = x;
#pragma unroll
  for (int i = 0; i < 3; ++i) x = y ^ (x >> 11);
  return x;
}

// The next block's state (in place, in three runs of words that depend only
// on earlier ones) and draws, by one wavefront.
__device__ inline void ring_twist(uint32_t *st, uint32_t *tem, int half) {
  const int lane = threadIdx.x & 63;
  uint32_t *out = tem + (624 - half);
  const bool first = half != 0;  // the next block goes to the first half
#pragma unroll
  for (int run = 0; run < 3; ++run) {
    const int lo = 227 * run, hi = run == 2 ? 623 : lo + 227;
    uint32_t v[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int k = lo + 64 * c + lane;
      v[c] = 0;
      if (k < hi) {
        const uint32_t y = (st[k] & 0x80000000u) | (st[k + 1] & 0x7fffffffu);
        v[c] = st[run == 0 ? k + 397 : k - 227] ^ (y >> 1) ^ ((y & 1u) ? 0x9908b0dfu : 0u);
      }
    }
    wave_lds_order();
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int k = lo + 64 * c + lane;
      if (k < hi) {
        const uint32_t d = mt_temper(v[c]);
        st[k] = v[c];
        out[k] = d;
        if (first && k < 8) out[1248 + k] = d;
      }
    }
    wave_lds_order();
  }
  if (lane == 0) {
    const uint32_t y = (st[623] & 0x80000000u) | (st[0] & 0x7fffffffu);
    const uint32_t v = st[396] ^ (y >> 1) ^ ((y & 1u) ? 0x9908b0dfu : 0u);
    st[623] = v;
    out[623] = mt_temper(v);
  }
  wave_lds_order();
}

// Address of entry `k` past the position in a ring array (entries k .. k+7
// follow it).
template <class T>
__device__ __forceinline__ const T *ring_at(const MtRing &g, const T *a, int k) {
  const uint32_t i = (uint32_t)(g.half + g.q + k);
  return a + min(i, i - 1248u);
}

// Makes the next `need` draws, and the sites of all but the last two of
// them, readable (wavefront 0).
__device__ __forceinline__ void ring_ensure(MtRing &g, int need) {
  if (g.q > 624) {
    if ((threadIdx.x & 63) == 0) *g.cmd = kCmdBlock;
    __syncthreads();
    g.q -= 624;
    g.half = 624 - g.half;
    g.ready = false;
  }
  if (!g.ready && g.q + need > 622) {
    __syncthreads();
    g.ready = true;
  }
}

// Has the helpers take up a command with wavefront 0.
__device__ __forceinline__ void spec_command(MtRing &g, int cmd) {
  if (!g.ready) {
    __syncthreads();
    g.ready = true;
  }
  if ((threadIdx.x & 63) == 0) *g.cmd = cmd;
  __syncthreads();
}

// The reference's state array and index at the position (after the helpers
// have finished; the newest block is the next one, so the current block's
// words come back from its draws).
__device__ inline void ring_finish(const MtRing &g, uint32_t *mt, int32_t *mt_index) {
  const int lane = threadIdx.x & 63;
  const int half = g.q > 624 ? 624 - g.half : g.half;
  for (int k = lane; k < 624; k += 64) mt[k] = mt_untemper(g.tem[half + k]);
  if (lane == 0) mt_index[0] = g.q > 624 ? g.q - 624 : g.q;
}

// ------------------------------------------------------------------
// sites
// ------------------------------------------------------------------
__device__ __forceinline__ uint32_t pack_xyz(SiteXYZ s) {
  return (uint32_t)s.x | ((uint32_t)s.y << 10) | ((uint32_t)s.z << 20);
}

__device__ __forceinline__ SiteXYZ unpack_xyz(uint32_t p) {
  return SiteXYZ{(int)(p & 1023u), (int)((p >> 10) & 1023u), (int)(p >> 20)};
}

// site_of_draws with the lattice known at compile time.
template <int LAT>
__device__ __forceinline__ SiteXYZ spec_site(const SeqGeo &g, uint32_t r1, uint32_t r2, uint32_t r3) {
  const int z = (int)__umulhi(r1, (uint32_t)g.m[2]);
  SiteXYZ s;
  s.z = z;
  if (LAT == 2) {
    s.x = 2 * (int)__umulhi(r2, (uint32_t)g.n[0]) + (z & 1);
    s.y = 2 * (int)__umulhi(r3, (uint32_t)g.n[1]) + (z & 1);
  } else {
    s.x = (int)__umulhi(r2, (uint32_t)g.m[0]);
    s.y = 2 * (int)__umulhi(r3, (uint32_t)g.n[1]) + ((s.x + z) & 1);
  }
  return s;
}

template <int LAT>
__device__ __forceinline__ int spec_sub(SiteXYZ s) {
  return LAT == 1 ? 2 * (s.x & 1) + (s.y & 1) : (s.x & 1);
}

// padded_addr_xyz with 24-bit multiplies (LDS addresses are far below 2^24).
template <int LAT>
__device__ __forceinline__ int spec_addr(const SeqGeo &g, SiteXYZ s) {
  const uint32_t row = __umul24((uint32_t)((s.z >> 1) + g.h), (uint32_t)g.P[1]) + (uint32_t)((s.y >> 1) + g.h);
  return (int)(__umul24((uint32_t)spec_sub<LAT>(s), (uint32_t)g.sub_stride) + __umul24(row, (uint32_t)g.P[0]) +
               (uint32_t)((s.x >> 1) + g.h));
}

// Ring entries of the sites at draws from, from + 1, ..., count of them
// (first + step * i for thread i of `step`).
template <int LAT>
__device__ inline void ring_sites(const SeqGeo &g, const uint32_t *tem, uint2 *site, int from, int count, int first,
                                  int step) {
  for (int i = first; i < count; i += step) {
    uint32_t k = (uint32_t)(from + i);
    k = min(k, k - 1248u);
    const SiteXYZ s = spec_site<LAT>(g, tem[k], tem[k + 1], tem[k + 2]);
    const uint2 v = make_uint2(pack_xyz(s), (uint32_t)spec_addr<LAT>(g, s));
    site[k] = v;
    if (k < 8) site[1248 + k] = v;
  }
}

// The first block's draws and sites from the state in `raw`, by the whole
// workgroup.
template <int LAT>
__device__ inline void ring_start(const SeqGeo &g, uint32_t *raw, uint32_t *tem, uint2 *site) {
  for (int k = threadIdx.x; k < 624; k += blockDim.x) {
    const uint32_t v = mt_temper(raw[k]);
    tem[k] = v;
    if (k < 8) tem[1248 + k] = v;
  }
  __syncthreads();
  ring_sites<LAT>(g, tem, site, 0, 622, threadIdx.x, blockDim.x);
  __syncthreads();
}

// What wavefronts 1-3 do while wavefront 0 runs the trials: wavefront 1
// makes the next block, then all wait for a command.  `other` serves the
// commands beyond blocks and the end (with barriers of its own, matched by
// wavefront 0).
template <int LAT, class F>
__device__ __forceinline__ void spec_helper(const SeqGeo &g, uint32_t *raw, uint32_t *tem, uint2 *site,
                                            volatile int32_t *cmd, F other) {
  const int wave = wave_uniform(threadIdx.x >> 6);
  int half = 0;
  for (;;) {
    if (wave == 1) {
      ring_twist(raw, tem, half);
      ring_sites<LAT>(g, tem, site, half + 622, 624, threadIdx.x & 63, 64);
    }
    half = 624 - half;
    __syncthreads();
    for (;;) {
      __syncthreads();
      const int c = wave_uniform(*cmd);
      if (c == kCmdExit) return;
      if (c == kCmdBlock) break;
      other(c);
    }
  }
}

// (a - b + rc) mod m for coordinates in [0, m), m > 2 rc: at most 2 rc
// exactly when a and b are within rc of each other through the period.
__device__ __forceinline__ uint32_t axis_gap(int a, int b, int m, int rc) {
  const int t = a - b + rc;
  return min(min((uint32_t)t, (uint32_t)(t + m)), (uint32_t)(t - m));
}

__device__ __forceinline__ uint32_t box_gap(SiteXYZ a, SiteXYZ b, const SeqGeo &g, int rc) {
  return max(max(axis_gap(a.x, b.x, g.m[0], rc), axis_gap(a.y, b.y, g.m[1], rc)), axis_gap(a.z, b.z, g.m[2], rc));
}

// List position of site b among a's neighbours, 255 if it is none.
template <int KEY>
__device__ __forceinline__ int neighbour_index(const SpecLds &L, const SeqGeo &g, SiteXYZ a, SiteXYZ b) {
  using D = SpecDims<KEY>;
  const uint32_t ux = axis_gap(b.x, a.x, g.m[0], D::RC), uy = axis_gap(b.y, a.y, g.m[1], D::RC),
                 uz = axis_gap(b.z, a.z, g.m[2], D::RC);
  int at = 255;
  if (max(max(ux, uy), uz) <= 2u * D::RC) at = L.adj[(uz * D::TS + uy) * D::TS + ux];
  return at;
}

// ------------------------------------------------------------------
// energies
// ------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (long long)(uint32_t)lo);
}

// First list entry and length of shell n, for a lane's own n.
template <int KEY>
__device__ __forceinline__ void lane_shell(int n, int &first, int &len) {
  using D = SpecDims<KEY>;
  first = 0;
  len = shell_len<D::LAT>(0);
#pragma unroll
  for (int q = 1; q < D::R; ++q)
    if (n >= q) {
      first = shell_first<D::LAT>(q);
      len = shell_len<D::LAT>(q);
    }
}

// Neighbour codes of the site at LDS address `addr` in shell n (ML of them;
// past the shell's length the site itself).
template <int KEY>
__device__ __forceinline__ void lane_codes(const SpecLds &L, int addr, int sub, int n, int (&code)[SpecDims<KEY>::ML]) {
  using D = SpecDims<KEY>;
  const int4 *op = (const int4 *)(L.off + (sub * D::R + n) * D::ML);
#pragma unroll
  for (int q = 0; q < D::ML / 4; ++q) {
    const int4 o = op[q];
    code[4 * q + 0] = L.lat[addr + o.x];
    code[4 * q + 1] = L.lat[addr + o.y];
    code[4 * q + 2] = L.lat[addr + o.z];
    code[4 * q + 3] = L.lat[addr + o.w];
  }
}

// A shell's sum in list order from 0.0; shells shorter than ML stop at their
// length (6, 8 or 12 entries).
template <int ML, int LO, int HI>
__device__ __forceinline__ void add_run(const double (&v)[ML], double &b) {
#pragma unroll
  for (int i = LO; i < HI; ++i)
    if (i < ML) b = b + v[i];
}

template <int ML>
__device__ __forceinline__ double shell_chain(const double (&v)[ML], int len) {
  double b = 0.0;
  add_run<ML, 0, 6>(v, b);
  if (len > 6) {
    add_run<ML, 6, 8>(v, b);
    if (ML > 8 && len > 8) {
      add_run<ML, 8, 12>(v, b);
      if (ML > 12 && len > 12) add_run<ML, 12, 24>(v, b);
    }
  }
  return b;
}

// The site energy from its shells' sums in the quad's lanes: left to right.
template <int R>
__device__ __forceinline__ double quad_sum(double b) {
  double s = dpp_d<0x00>(b);
  if constexpr (R > 1) s = s + dpp_d<0x55>(b);
  if constexpr (R > 2) s = s + dpp_d<0xaa>(b);
  if constexpr (R > 3) s = s + dpp_d<0xff>(b);
  return s;
}

constexpr int kRowHalfMirror = 0x141;  // lane i of 8 takes lane 7 - i
constexpr int kRowRotate8 = 0x128;     // lane i of 16 takes lane (i + 8) mod 16

// pair_energy before and after the swap of a trial's two sites, on all 8 of
// its lanes: lane & 3 is the shell n and own / oth the lane's site and the
// other one (sites of lanes 0-3 and 4-7), with their codes.
template <int KEY>
__device__ __forceinline__ void spec_pair_energies(const SpecLds &L, const SeqGeo &g, int S, uint32_t inv_S, int n,
                                                   SiteXYZ own, SiteXYZ oth, int addr, int code_own, int code_oth,
                                                   double &e_before, double &e_after) {
  using D = SpecDims<KEY>;
  constexpr int ML = D::ML, R = D::R;
  const int nn = n < R ? n : R - 1;
  int code[ML];
  lane_codes<KEY>(L, addr, spec_sub<D::LAT>(own), nn, code);
  int first, len;
  lane_shell<KEY>(nn, first, len);
  const int at = neighbour_index<KEY>(L, g, own, oth) - first;  // the other site in this lane's shell
  const int row = (int)__umul24((uint32_t)nn, (uint32_t)(S * S));
  const double *vo = L.vex + row + (int)((__umul24((uint32_t)code_own, inv_S)) >> 16);
  const double *vt = L.vex + row + (int)((__umul24((uint32_t)code_oth, inv_S)) >> 16);
  double vb[ML], va[ML];
#pragma unroll
  for (int i = 0; i < ML; ++i) {
    vb[i] = vo[code[i]];
    va[i] = vt[code[i]];
  }
  // after the swap the other site, seen as a neighbour, has this site's species
  if (__ballot(at >= 0 && at < len) != 0) {
    const double f = vt[code_own];
#pragma unroll
    for (int i = 0; i < ML; ++i) va[i] = i == at ? f : va[i];
  }
  const double sb = quad_sum<R>(shell_chain<ML>(vb, len)), sa = quad_sum<R>(shell_chain<ML>(va, len));
  // the other site's sum from the mirrored lane of the 8
  e_before = sb + dpp_d<kRowHalfMirror>(sb);
  e_after = sa + dpp_d<kRowHalfMirror>(sa);
}

// One site's energy before and after its trial's swap, by one lane: the
// shells in list order from 0.0, added left to right.
template <int KEY>
__device__ __forceinline__ void spec_site_energies(const SpecLds &L, const SeqGeo &g, int S, uint32_t inv_S,
                                                   SiteXYZ own, SiteXYZ oth, int addr, int code_own, int code_oth,
                                                   double &eb, double &ea) {
  using D = SpecDims<KEY>;
  constexpr int ML = D::ML, R = D::R;
  const int32_t *ob = L.off + spec_sub<D::LAT>(own) * R * ML;
  const int at = neighbour_index<KEY>(L, g, own, oth);
  const double *vo = L.vex + (int)((__umul24((uint32_t)code_own, inv_S)) >> 16);
  const double *vt = L.vex + (int)((__umul24((uint32_t)code_oth, inv_S)) >> 16);
#pragma unroll
  for (int n = 0; n < R; ++n) {
    double b = 0.0, a = 0.0;
    const double *von = vo + n * S * S, *vtn = vt + n * S * S;
#pragma unroll
    for (int i = 0; i < shell_len<D::LAT>(n); ++i) {
      const int code = L.lat[addr + ob[n * ML + i]];
      const int after = shell_first<D::LAT>(n) + i == at ? code_own : code;
      b = b + von[code];
      a = a + vtn[after];
    }
    eb = n == 0 ? b : eb + b;
    ea = n == 0 ? a : ea + a;
  }
}

// total_energy in the reference's order (ref_total_energy) by the whole
// workgroup: wavefronts 1-3 form the energies of 192 sites at a time while
// wavefront 0 adds the 192 before them in order.  The result is wavefront
// 0's.  buf: 2 x 192 doubles.
constexpr int kEnergyChunk = kSpecThreads - 64;

template <int KEY>
__device__ inline double spec_total_energy(const SpecLds &L, const SeqGeo &g, int n_atoms, int S, uint32_t inv_S,
                                           double *buf) {
  using D = SpecDims<KEY>;
  const int wave = wave_uniform(threadIdx.x >> 6);
  const int hx = g.m[0] >> 1, hy = g.m[1] >> 1;
  const int chunks = (n_atoms + kEnergyChunk - 1) / kEnergyChunk;
  double e = 0.0;
  for (int c = 0; c <= chunks; ++c) {
    if (wave > 0) {
      const int idx = c * kEnergyChunk + (int)threadIdx.x - 64;
      double v = 0.0;
      if (idx < n_atoms) {
        const int row = idx / hx;
        const int xh = idx - row * hx;
        SiteXYZ s;
        if (D::LAT == 1) {
          s.z = row / g.m[1];
          s.y = row - s.z * g.m[1];
          s.x = 2 * xh + ((s.y + s.z) & 1);
        } else {
          s.z = row / hy;
          s.y = 2 * (row - s.z * hy) + (s.z & 1);
          s.x = 2 * xh + (s.z & 1);
        }
        const int addr = spec_addr<D::LAT>(g, s);
        const int32_t *ob = L.off + spec_sub<D::LAT>(s) * D::R * D::ML;
        const double *vo = L.vex + (int)((__umul24((uint32_t)L.lat[addr], inv_S)) >> 16);
#pragma unroll
        for (int n = 0; n < D::R; ++n) {
          double b = 0.0;
#pragma unroll
          for (int i = 0; i < shell_len<D::LAT>(n); ++i) b = b + vo[n * S * S + L.lat[addr + ob[n * D::ML + i]]];
          v = n == 0 ? b : v + b;
        }
      }
      buf[(c & 1) * kEnergyChunk + threadIdx.x - 64] = v;
    } else if (c > 0) {
      // entries past the last site are +0.0, which changes no sum begun at +0.0
      const double2 *p = (const double2 *)(buf + ((c - 1) & 1) * kEnergyChunk);
#pragma unroll 16
      for (int i = 0; i < kEnergyChunk / 2; ++i) {
        const double2 v = p[i];
        e = e + v.x;
        e = e + v.y;
      }
    }
    __syncthreads();
  }
  return 0.5 * e;
}

// ------------------------------------------------------------------
// conflicts and writes of a batch
// ------------------------------------------------------------------
// Whether a swap of the lane's row trial (lane >> 3) reaches a site of the
// lane's column trial (lane & 7): any two of their sites within the
// interaction range.  pa / pb: the packed sites of the trial lane >> 3.
__device__ __forceinline__ bool batch_conflict(const SeqGeo &g, int rc, uint32_t pa, uint32_t pb) {
  const int col = 8 * (threadIdx.x & 7);
  const SiteXYZ a = unpack_xyz(pa), b = unpack_xyz(pb);
  const SiteXYZ c = unpack_xyz((uint32_t)__shfl((int)pa, col)), d = unpack_xyz((uint32_t)__shfl((int)pb, col));
  const uint32_t u = min(min(box_gap(a, c, g, rc), box_gap(a, d, g, rc)), min(box_gap(b, c, g, rc), box_gap(b, d, g, rc)));
  return u <= 2u * (uint32_t)rc;
}

// LDS address of one of a site's 8 possible images (bits of `image`: x, y,
// z), -1 if that image does not exist.
template <int LAT>
__device__ __forceinline__ int image_addr(const SeqGeo &g, SiteXYZ s, int image) {
  auto first = [](int c, int h, int n) {
    const int p = c + h;
    return p >= n ? p - n : p;
  };
  const int px = first(s.x >> 1, g.h, g.n[0]) + ((image & 1) ? g.n[0] : 0);
  const int py = first(s.y >> 1, g.h, g.n[1]) + ((image & 2) ? g.n[1] : 0);
  const int pz = first(s.z >> 1, g.h, g.n[2]) + ((image & 4) ? g.n[2] : 0);
  const int at = (int)(__umul24((uint32_t)spec_sub<LAT>(s), (uint32_t)g.sub_stride) +
                       __umul24(__umul24((uint32_t)pz, (uint32_t)g.P[1]) + (uint32_t)py, (uint32_t)g.P[0]) + (uint32_t)px);
  return px < g.P[0] && py < g.P[1] && pz < g.P[2] ? at : -1;
}

// Writes `code` at the lane's site and its periodic images, the 8 possible
// images over the site's 4 lanes.  The accepted trials of a batch touch
// different sites, so all of them are written at once.
template <int LAT>
__device__ __forceinline__ void batch_write(int8_t *lat, const SeqGeo &g, bool doit, SiteXYZ s, int code) {
  const int v = threadIdx.x & 3;
  const int a0 = image_addr<LAT>(g, s, v), a1 = image_addr<LAT>(g, s, v | 4);
  wave_lds_order();
  if (doit) {
    if (a0 >= 0) lat[a0] = (int8_t)code;
    if (a1 >= 0) lat[a1] = (int8_t)code;
  }
  wave_lds_order();
}

// Staging by the whole workgroup, the digits of each thread's walk carried
// (stage_lattice_walk) and 8 cells in flight per thread; cells as codes
// S * (species - 1).
__device__ inline void stage_codes(int8_t *lat, const int8_t *__restrict__ compact, const SeqGeo &g, int nsub, int S) {
  const int total = nsub * g.sub_stride;
  BoxWalk w = box_walk(threadIdx.x, blockDim.x, g.P[0], g.P[1], g.P[2]);
  for (int idx = threadIdx.x; idx < total; idx += 8 * blockDim.x) {
    int v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      v[q] = 1;
      if (idx + q * (int)blockDim.x < total) {
        const int cx = unpad(w.x, g.h, g.n[0]), cy = unpad(w.y, g.h, g.n[1]), cz = unpad(w.z, g.h, g.n[2]);
        v[q] = compact[(int)(__umul24(__umul24(__umul24((uint32_t)w.s, (uint32_t)g.n[2]) + (uint32_t)cz, (uint32_t)g.n[1]) +
                                         (uint32_t)cy, (uint32_t)g.n[0])) + cx];
      }
      box_step(w, g.P[0], g.P[1], g.P[2]);
    }
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (idx + q * (int)blockDim.x < total) lat[idx + q * blockDim.x] = (int8_t)(S * (v[q] - 1));
  }
}

__device__ inline void unstage_codes(const int8_t *lat, int8_t *__restrict__ compact, const SeqGeo &g, int nsub,
                                     uint32_t inv_S) {
  const int total = nsub * g.n[0] * g.n[1] * g.n[2];
  BoxWalk w = box_walk(threadIdx.x, blockDim.x, g.n[0], g.n[1], g.n[2]);
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int v = lat[padded_addr(g, w.s, w.x, w.y, w.z)];
    compact[idx] = (int8_t)((__umul24((uint32_t)v, inv_S) >> 16) + 1);
    box_step(w, g.n[0], g.n[1], g.n[2]);
  }
}

// LDS of the speculative kernels: lattice and tables, the stream's ring, the
// energy recount's buffer (the carves round every part up to 16 bytes).
inline size_t spec_align(size_t v) { return (v + 15) & ~(size_t)15; }
inline size_t spec_ring_bytes() {
  return spec_align(4 * 624) + spec_align(4 * kRingWords) + spec_align(8 * kRingWords) + 16;
}
inline size_t spec_energy_bytes() { return spec_align(sizeof(double) * 2 * kEnergyChunk); }
inline size_t spec_table_bytes(const Geo &g) {
  const size_t ts = 2 * (size_t)g.rcut + 1;
  return spec_align((size_t)g.lds_bytes) + spec_align(sizeof(double) * g.S * g.S * g.R) +
         spec_align(4 * (size_t)g.nsub * g.R * shell_max(g.lattice, g.R)) + spec_align(ts * ts * ts);
}

// code / S for codes S * (0..7) as a multiply and a shift by 16.
__device__ __forceinline__ uint32_t inverse_of(int S) { return 65536u / (uint32_t)S + 1u; }

__device__ __forceinline__ SeqGeo seq_geo(const Geo &g) {
  SeqGeo s;
  s.lattice = g.lattice;
  for (int a = 0; a < 3; ++a) {
    s.n[a] = g.n[a];
    s.m[a] = g.m[a];
    s.P[a] = g.P[a];
  }
  s.h = g.h;
  s.sub_stride = g.sub_stride;
  s.S = g.S;
  s.R = g.R;
  s.z = g.z;
  return s;
}

}  // namespace bwl
