// bwl_metro_split.h -- the device code of a chain of the parallel Metropolis
// sampler at one site per lane, in several workgroups (bwl_metro_split.hip) or
// in one (bwl_metro_alone.hip).
#pragma once

#include "bwl_metro_kernels.h"

namespace bwl {

namespace {

constexpr int kSplitThreads = 512;  // 8 wavefronts with up to 256 registers each: no spills
constexpr int kSplitWaves = kSplitThreads / 64;
// Ticks of 10 ns (1 s) that a wait for another part's word may take once all
// have arrived: they are resident then, so only a device taken away for that
// long ends one.  Arriving they wait ParArgs::patience.
constexpr long long kSplitPatience = 100000000LL;

// Mailbox, in 64-bit words.  Per round (4 slots in turn) and part: a header
// per half row, then the records; then the sums of the rows (2 slots), the
// temperature step's counts (2 slots), the parts' XCDs, and the word that
// gives a chain up.
constexpr int kUnits = kSplitWaves;         // half rows a part may have
constexpr int kRecords = 32 * kUnits;
constexpr int kRoundWords = kUnits + kRecords;

__host__ __device__ inline size_t mail_end_words(int S, int R) { return (size_t)(S * S * R) + 2; }

__device__ __forceinline__ unsigned long long mail_load(const unsigned long long *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void mail_store(unsigned long long *p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Whether a wait has lasted too long or the chain has been given up; called
// once per poll.
struct Patience {
  long long limit = kSplitPatience;
  uint32_t between = 1023;  // polls, less one, from one look at the clock to the next
  uint32_t tries = 0;
  long long since = 0;
  __device__ __forceinline__ bool over(unsigned long long *gone) {
    if ((++tries & between) != 0) return false;
    const long long now = wall_clock64();
    if (since == 0) since = now;
    if (mail_load(gone) != 0) return true;
    if (now - since <= limit) return false;
    if ((threadIdx.x & 63) == 0) mail_store(gone, 1);
    return true;
  }
};

// Polls the lanes' words until each (of the lanes that want one) carries
// `tag` in its upper half; false when the chain has been given up.
__device__ __forceinline__ bool mail_wait(const unsigned long long *p, bool want, uint32_t tag, unsigned long long *gone,
                                          unsigned long long &v, Patience wait = Patience()) {
  for (;;) {
    v = (unsigned long long)tag << 32;
    if (want) v = mail_load(p);
    if (__ballot((uint32_t)(v >> 32) != tag) == 0) return true;
    if (wait.over(gone)) return false;
  }
}

// A round's parameters as the lanes use them (see NatAffine), formed 64
// rounds ahead, one thread each.
struct __align__(16) SplitRound {
  int32_t a[2], b[2], c[2];  // biased bases of grids 1 and 2
  int32_t aj, au, av, bj, bu, bv, cj, cu, cv;
  int32_t nL1, al, ab, ac;
  int32_t n2, bfast, full, rest, pad;  // full, rest: n2 by and mod the virtual threads
};

// nat_put without branches: where a cell has no image along an axis the step
// is 0 and the store repeats one already made.
__device__ __forceinline__ void put_images(int8_t *lat, const ND &N, int a, int b, int c, int8_t v) {
  const int row = N.P0, plane = (int)__umul24((uint32_t)N.P0, (uint32_t)N.P1);
  const int da = a < N.h0 ? N.D0 : (a >= N.D0 - N.h0 ? -N.D0 : 0);
  const int db = b < N.h1 ? N.D1 * row : (b >= N.D1 - N.h1 ? -N.D1 * row : 0);
  const int dc = c < N.h2 ? N.D2 * plane : (c >= N.D2 - N.h2 ? -N.D2 * plane : 0);
  const int p = nat_addr(N, a, b, c), pb = p + db, pc = p + dc, pbc = pb + dc;
  lat[p] = v;
  lat[p + da] = v;
  lat[pb] = v;
  lat[pb + da] = v;
  lat[pc] = v;
  lat[pc + da] = v;
  lat[pbc] = v;
  lat[pbc + da] = v;
}

// A record: natural coordinates (7 bits each) and species - 1 (3 bits) of
// both sites, 16 bits of tag (the round mod 65536, or 65535 where that is 0,
// which no other round within reach has).  Slots are cleared before their tags
// come around again.
__device__ __forceinline__ uint32_t record_tag(uint32_t round) {
  const uint32_t t = round & 0xffffu;
  return t ? t : 0xffffu;
}

// ALONE: the chain has one part, in a workgroup of as many wavefronts as it
// has half rows of pairs (see bwl_metro_alone.hip): no mailbox, each lane
// makes its own site's swap.
template <int LAT, int R, typename CW, int NC, int FIELD, bool ALONE>
__device__ __forceinline__ void metro_split(const ParArgs &C, const int part, uint8_t *smem) {
  static_assert(NC != 0, "compile-time neighbour offsets");
  const int parts = ALONE ? 1 : C.parts;
  const int n_threads = ALONE ? (int)blockDim.x : kSplitThreads, n_waves = ALONE ? n_threads >> 6 : kSplitWaves;
  const Geo &g = C.g;
  constexpr NatGeo KG = nat_geo_c<LAT, R, NC>();
  ND N = NC > 0 ? nd_of(KG) : nd_of(C.nat);
  if constexpr (NC == kFixedPitch) {
    N.P0 = KG.P[0];
    N.P1 = KG.P[1];
    N.h0 = KG.h[0];
    N.h1 = KG.h[1];
    N.h2 = KG.h[2];
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = uni(tid >> 6);
  const int nthr = C.threads, rows = nthr >> 6;           // virtual threads, rows of 64
  const int my_rows = (rows - part + parts - 1) / parts;  // rows part, part + parts, ...
  const int passes = C.passes;
  const int units = 2 * my_rows * passes;                 // this part's half rows, pass after pass
  const int S = g.S;
  constexpr int RSTR = kRowStride<R, CW, FIELD>;
  int8_t *lat = (int8_t *)smem;
  size_t o = ((N.P0 * N.P1 * N.P2) + 15) & ~15;
  double *dtab = (double *)(smem + o);
  o += sizeof(double) * S * S * RSTR;
  double *vrow = (double *)(smem + o);
  o += sizeof(double) * S * R * S;
  o = (o + 15) & ~(size_t)15;
  SplitRound *rps = (SplitRound *)(smem + o);
  o += sizeof(SplitRound) * kRoundBatch;
  unsigned long long *hacc = (unsigned long long *)(smem + o);
  o += sizeof(unsigned long long) * S * S * R;
  // accepted energy changes of the passes after the first, by round parity;
  // the sums of the rows' virtual threads; the rows' sums
  double *late = (double *)(smem + o);
  o += sizeof(double) * 2 * 32 * kUnits;
  double *vsum = (double *)(smem + o);
  o += sizeof(double) * 32 * kUnits;
  double *red = (double *)(smem + o);
  o += sizeof(double) * 32;
  // records packed so far, by round
  uint32_t *packed = (uint32_t *)(smem + o);
  o += sizeof(uint32_t) * 4;
  // the round (from 1) in which a wait of this part ended without its word;
  // compared with the round at hand, so that every wavefront leaves at the
  // same barrier
  volatile uint32_t *dead = (volatile uint32_t *)(smem + o);

  unsigned long long *mail = C.mail;
  unsigned long long *msum = mail + 4 * (size_t)parts * kRoundWords;
  unsigned long long *mend = msum + 2 * 2 * (size_t)rows;
  const int end_words = (int)mail_end_words(S, R);
  unsigned long long *mxcd = mend + 2 * (size_t)parts * end_words;
  unsigned long long *gone = mxcd + parts;

  for (int i = tid; i < S * S * R; i += n_threads) hacc[i] = 0ull;
  if (tid < 4) packed[tid] = 0;
  if (tid == 0) *dead = 0;
  fill_tables<R, CW, FIELD>(dtab, vrow, C.vex, S);
  nat_stage<LAT>(lat, C.compact, g, N, FIELD);
  __syncthreads();

  const int Kq = C.K[0];
  const float invKK = 1.0f / (float)(Kq * Kq), invK = 1.0f / (float)Kq;
  const float invD1 = 1.0f / (float)N.D1, invD2 = 1.0f / (float)N.D2;
  unsigned long long phase = C.phase0;
  long long acc_total = 0, trials_total = 0;
  uint32_t round_tag = 0, sum_tag = 0;
  int off[1] = {0};
  // (asked once per batch of rounds: after a wait has ended without its word
  // the following ones end soon)
  auto given_up = [&]() {
    const uint32_t d = *dead;
    return d != 0 && d <= round_tag + 1;
  };

  // whether all parts are on this XCD (every part sees the same words)
  bool one_xcd = true;
  if constexpr (!ALONE) {
    uint32_t xcd;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcd));
    if (tid == 0) mail_store(&mxcd[part], (1ull << 32) | xcd);
    unsigned long long v = 0;
    if (!mail_wait(&mxcd[lane < parts ? lane : 0], lane < parts, 1, gone, v, Patience{C.patience, 15}) ||
        mail_load(gone) != 0)
      *dead = 1;
    one_xcd = __ballot(lane < parts && (uint32_t)v != xcd) == 0;
  }
  auto post = [&](unsigned long long *p, unsigned long long v) {
    if (one_xcd)
      __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else
      mail_store(p, v);
  };

  // This wavefront's half row: unit `wave` is pass wave / (2 my_rows) of row
  // (wave >> 1) mod my_rows, half wave & 1.
  const bool evaluates = wave < units;
  const int e = evaluates ? wave : 0;
  const int my_pass = e / (2 * my_rows);
  const int vt = 64 * (part + parts * ((e >> 1) - my_pass * my_rows)) + 32 * (e & 1) + (lane & 31);
  const int q = vt + my_pass * nthr;  // the lane's pair
  const bool first = my_pass == 0;    // the pass that keeps the virtual thread's sum
  const bool isA = lane < 32;
  // q in grid indices (the same every round; see k_metro_nat)
  int q_jl, q_ks, q_kf;
  {
    uint32_t j, rem, ks, kf;
    divmod_small((uint32_t)q, (uint32_t)(Kq * Kq), invKK, j, rem);
    divmod_small(rem, (uint32_t)Kq, invK, ks, kf);
    q_jl = (int)j;
    q_ks = (int)ks;
    q_kf = (int)kf;
  }
  double sum = 0.0;  // accepted energy changes of the virtual thread in this sweep
  uint32_t draws = 0, have = 0xffffffffu;  // draws of this batch before the round, Philox block held
  U4 rnd = {0, 0, 0, 0};
  // the coming round: whether the lane has a pair, its site, its number
  bool valid = false;
  int sa = 0, sb = 0, sc = 0, addr = 0;
  uint32_t ru = 0;
  int n2 = 0;
  auto prepare = [&](int r) {
    const SplitRound &P = rps[r];
    n2 = uni(P.n2);
    if (!evaluates) return;
    const int nL1 = P.nL1;
    valid = q < n2;
    // random number of the pair: draw `draws + pass` of the virtual thread
    const uint32_t d = draws + (uint32_t)my_pass;
    if ((d >> 2) != have) {
      have = d >> 2;
      rnd = philox4x32(U4{(uint32_t)phase, (uint32_t)(phase >> 32), (uint32_t)vt | (have << 12), C.chain_id}, C.seed_lo,
                       C.seed_hi);
    }
    ru = (d & 3) == 0 ? rnd.x : (d & 3) == 1 ? rnd.y : (d & 3) == 2 ? rnd.z : rnd.w;
    // draws made by the end of this round
    draws += (uint32_t)(P.full + (vt < P.rest ? 1 : 0));
    // lanes 0-31: grid-1 site (A), the partner by (al, ab, ac) in grid
    // indices; lanes 32-63: grid-2 site (B)
    int j = q_jl + (isA ? P.al : 0), kb = (P.bfast ? q_kf : q_ks) + (isA ? P.ab : 0),
        kc = (P.bfast ? q_ks : q_kf) + (isA ? P.ac : 0);
    if (isA) {
      if (j >= nL1) j -= nL1;
      if (kb >= Kq) kb -= Kq;
      if (kc >= Kq) kc -= Kq;
    }
    const int gr = isA ? 0 : 1;
    const uint32_t va = (uint32_t)(P.a[gr] + __mul24(j, P.aj) + __mul24(kb, P.au) + __mul24(kc, P.av));
    sa = (int)min(va, va - (uint32_t)N.D0);
    sb = mod_pos(P.b[gr] + __mul24(j, P.bj) + __mul24(kb, P.bu) + __mul24(kc, P.bv), N.D1, invD1);
    sc = mod_pos(P.c[gr] + __mul24(j, P.cj) + __mul24(kb, P.cu) + __mul24(kc, P.cv), N.D2, invD2);
    addr = valid ? nat_addr(N, sa, sb, sc) : nat_addr(N, 0, 0, 0);
  };

  // The sums of the rows in order, from every row's 64 values (vsum of its
  // part): each part reduces its rows, the first adds them all.  Returns the
  // total on the first part's thread 0.
  auto total_of_rows = [&]() -> double {
    ++sum_tag;
    __syncthreads();
    if constexpr (ALONE) {
      for (int r = wave; r < rows; r += n_waves) {
        double v = vsum[64 * r + lane];
#pragma unroll
        for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
        if (lane == 0) red[r] = v;
      }
      __syncthreads();
      double t = 0.0;
      if (tid == 0)
        for (int r = 0; r < rows; ++r) t += red[r];
      __syncthreads();
      return t;
    }
    unsigned long long *slot = msum + (size_t)(sum_tag & 1u) * 2 * rows;
    for (int r = wave; r < my_rows; r += kSplitWaves) {
      double v = vsum[64 * r + lane];
#pragma unroll
      for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
      const unsigned long long b = (unsigned long long)__double_as_longlong(v);
      if (lane < 2)
        mail_store(&slot[2 * (part + parts * r) + lane],
                   ((unsigned long long)sum_tag << 32) | (lane ? b >> 32 : b & 0xffffffffull));
    }
    double t = 0.0;
    if (part == 0) {
      if (wave == 0) {
        // 2 words for each of at most 16 rows: one per lane
        unsigned long long v = 0;
        if (!mail_wait(&slot[lane], lane < 2 * rows, sum_tag, gone, v)) *dead = round_tag + 1;
        const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)v, (2 * lane) & 63);
        const uint32_t hi = (uint32_t)__shfl((int)(uint32_t)v, (2 * lane + 1) & 63);
        if (lane < rows) red[lane] = __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
      }
      __syncthreads();
      if (tid == 0)
        for (int r = 0; r < rows; ++r) t += red[r];
    }
    __syncthreads();
    return t;
  };

  // Energy of the lattice recounted from its shell counts: virtual thread v
  // takes sites v, v + nthr, ...  (on the first part's thread 0)
  auto recount = [&]() -> double {
    const int nsites = N.D0 * N.D1 * N.D2;
    for (int r = wave; r < my_rows; r += n_waves) {
      double s = 0.0;
      for (int i = 64 * (part + parts * r) + lane; i < nsites; i += nthr)
        add_site_energy<LAT, R, CW, NC, FIELD>(lat, N, off, vrow, S, i, s);
      vsum[64 * r + lane] = s;
    }
    return 0.5 * total_of_rows();
  };
  double E = recount();

  for (int t = 0; t < C.T_steps && !given_up(); ++t) {
    const double temp = C.T0 + (double)t * C.dT;
    const double sim_temp = temp * kKbInRyPar;
    const double beta = 1.0 / sim_temp;
    double step_E = 0.0, step_Esq = 0.0;
    unsigned long long acc_local = 0;
    long long trials_sampled = 0;
    const int nsw = C.burn_sweeps + C.n_sweeps;
    for (int sw = 0; sw < nsw && !given_up(); ++sw) {
      const bool sampled = sw >= C.burn_sweeps;
      sum = 0.0;
      const int want = (int)C.min_trials_per_sweep;
      int done = 0;
      while (done < want) {
        if (tid < kRoundBatch) {
          const RoundP P = round_params(C, phase + (unsigned long long)tid);
          const NatAffine F = nat_affine<LAT>(P.ax, C.L, C.stride, g.n[0], P.oA1, P.oB1, P.oC1, P.oA2, P.oB2, P.oC2);
          SplitRound &Q = rps[tid];
          Q.a[0] = F.a1; Q.a[1] = F.a2;
          Q.b[0] = F.b1; Q.b[1] = F.b2;
          Q.c[0] = F.c1; Q.c[1] = F.c2;
          Q.aj = F.aj; Q.au = F.au; Q.av = F.av;
          Q.bj = F.bj; Q.bu = F.bu; Q.bv = F.bv;
          Q.cj = F.cj; Q.cu = F.cu; Q.cv = F.cv;
          Q.nL1 = P.nL1; Q.al = P.al; Q.ab = P.ab; Q.ac = P.ac;
          Q.n2 = P.n2;
          Q.full = P.n2 / nthr;
          Q.rest = P.n2 - Q.full * nthr;
          Q.bfast = (KG.lane_order >> P.ax) & 1;
        }
        __syncthreads();
        draws = 0;
        have = 0xffffffffu;
        prepare(0);
        int r = 0;
        double mine = 0.0;  // the lane's accepted energy change of the round
        // sums of the virtual threads, passes in order (of the round before
        // this one: its last reader is past the barrier, its next writer two
        // rounds away)
        auto add_round = [&](uint32_t round) {
          if (!(evaluates && first)) return;
          sum += mine;
          for (int pass = 1; pass < passes; ++pass)
            sum += late[((round & 1u) * kUnits + e + 2 * my_rows * pass) * 32 + (lane & 31)];
        };
        for (; r < kRoundBatch && done < want; ++r) {
          ++round_tag;
          const uint32_t rtag = record_tag(round_tag);
          unsigned long long *slot = mail + __umul24((round_tag & 3u) * (uint32_t)parts, (uint32_t)kRoundWords);
          unsigned long long *my_slot = slot + (uint32_t)(part * kRoundWords);

          // ---- this part's pairs
          double fresh = 0.0;
          if (evaluates) {
            uint32_t swaps = 0, base = 0;
            if (__ballot(valid) != 0) {
              const int code = lat[addr];
              CW cnt[R];
              count_c<LAT, R, CW, NC>(lat, addr, cnt);
              __builtin_amdgcn_sched_barrier(0);
              // both halves of the wavefront get both sites' counts
              auto both = [](uint32_t x, uint32_t &va, uint32_t &vb) {
                const auto s = __builtin_amdgcn_permlane32_swap(x, x, false, false);
                va = s[0];
                vb = s[1];
              };
              CW ca[R], cb[R];
              uint32_t codeA, codeB;
              both((uint32_t)code, codeA, codeB);
#pragma unroll
              for (int n = 0; n < R; ++n) {
                uint32_t x, y;
                both((uint32_t)cnt[n], x, y);
                ca[n] = x;
                cb[n] = y;
                if constexpr (sizeof(CW) > 4) {
                  both((uint32_t)((uint64_t)cnt[n] >> 32), x, y);
                  ca[n] |= (CW)((uint64_t)x << 32);
                  cb[n] |= (CW)((uint64_t)y << 32);
                }
              }
              const double dE = pair_delta<R, CW, FIELD>(dtab, S, (int)codeA, (int)codeB, ca, cb);
              const bool same = codeA == codeB;
              bool acc = same || dE < 0.0;
              if (!acc) acc = metropolis_accept((double)ru * (1.0 / 4294967296.0), -(beta * dE));
              acc = acc && valid;
              const bool moves = acc && !same;
              fresh = moves ? dE : 0.0;
              if (sampled && acc && isA) acc_local++;
              // its swaps, packed behind those of the part's other half rows
              if constexpr (ALONE) {
                // (no pair's neighbours hold another pair's sites)
                if (moves) put_images(lat, N, sa, sb, sc, (int8_t)(isA ? codeB : codeA));
              } else {
                swaps = (uint32_t)__ballot(moves);
              }
              if (swaps) {
                if (lane == 0) base = atomicAdd(&packed[round_tag & 3u], (uint32_t)__popc(swaps));
                base = (uint32_t)uni((int)base);
                // lane i (A) completes its record with its partner's half
                const uint32_t half = (uint32_t)sa | ((uint32_t)sb << 7) | ((uint32_t)sc << 14) | (((uint32_t)code / FIELD) << 21);
                uint32_t ha, hb;
                both(half, ha, hb);
                const uint32_t at = base + (uint32_t)__builtin_amdgcn_mbcnt_lo(swaps, 0);
                if (moves && isA)
                  post(&my_slot[kUnits + at],
                       ((unsigned long long)rtag << 48) | ((unsigned long long)hb << 24) | (unsigned long long)ha);
              }
            }
            if (!ALONE && lane == 0) post(&my_slot[e], ((unsigned long long)round_tag << 32) | (base + (uint32_t)__popc(swaps)));
            // the passes after the first hand their energy changes to the first
            if (!first && isA) late[((round_tag & 1u) * kUnits + e) * 32 + lane] = fresh;
          }
          if (!ALONE && tid == 0) packed[(round_tag + 2) & 3u] = 0;
          // record tags come around every 65535 rounds: well before, each of
          // the 4 slots is cleared once, two rounds ahead of its use
          if (!ALONE && (round_tag & 0x7fffu) < 4u) {
            for (int i = tid; i < kRecords; i += kSplitThreads)
              post(mail + (size_t)((round_tag + 2) & 3u) * parts * kRoundWords + (size_t)part * kRoundWords + kUnits + i, 0);
            __threadfence();  // done before any wavefront's later record
          }

          // meanwhile: the last round's sums, the next round's sites and numbers
          if (r > 0) add_round(round_tag - 1);
          mine = fresh;
          done += n2;
          if (r + 1 < kRoundBatch && done < want) prepare(r + 1);

          // ---- all of the round's swaps on this part's lattice: a wavefront
          // reads one part's records, or two parts' with half its lanes each
          const int per = parts > kSplitWaves ? 32 : 64;  // lanes per part
          const int idx = lane & (per - 1);
          for (int k0 = wave; !ALONE && k0 < parts; k0 += kSplitWaves * (64 / per)) {
            const int k = k0 + kSplitWaves * (lane / per);
            const bool there = k < parts;
            const unsigned long long *box = slot + (uint32_t)((there ? k : 0) * kRoundWords);
            const int k_units = there ? 2 * ((rows - k + parts - 1) / parts) * passes : 0;
            Patience wait;
            uint32_t total = 0;
            unsigned long long rec = 0;
            for (bool ok = false; !ok;) {
              const unsigned long long h = idx < k_units ? mail_load(&box[idx]) : (unsigned long long)round_tag << 32;
              rec = mail_load(&box[kUnits + idx]);
              // a half row without swaps says 0; otherwise where its end is
              int m = (int)(uint32_t)h;
              m = max(m, __builtin_amdgcn_update_dpp(0, m, 0xb1, 0xf, 0xf, true));   // lane ^ 1
              m = max(m, __builtin_amdgcn_update_dpp(0, m, 0x4e, 0xf, 0xf, true));   // lane ^ 2
              m = max(m, __builtin_amdgcn_update_dpp(0, m, 0x141, 0xf, 0xf, true));  // 7 - lane of 8
              const uint32_t t0 = (uint32_t)__builtin_amdgcn_readlane(m, 0), t1 = (uint32_t)__builtin_amdgcn_readlane(m, 32);
              total = per == 32 && lane >= 32 ? t1 : t0;
              ok = __ballot((uint32_t)(h >> 32) != round_tag || ((uint32_t)idx < total && (uint32_t)(rec >> 48) != rtag)) == 0;
              if (!ok && wait.over(gone)) {
                *dead = round_tag + 1;
                total = 0;
                break;
              }
            }
            for (uint32_t i = (uint32_t)idx;; i += (uint32_t)per) {
              if (i < total) {
                const uint32_t ha = (uint32_t)rec & 0xffffffu, hb = (uint32_t)(rec >> 24) & 0xffffffu;
                const int aA = (int)(ha & 127u), bA = (int)((ha >> 7) & 127u), cA = (int)((ha >> 14) & 127u);
                const int aB = (int)(hb & 127u), bB = (int)((hb >> 7) & 127u), cB = (int)((hb >> 14) & 127u);
                put_images(lat, N, aA, bA, cA, (int8_t)(FIELD * (hb >> 21)));
                put_images(lat, N, aB, bB, cB, (int8_t)(FIELD * (ha >> 21)));
              }
              const bool more = i + (uint32_t)per < total;
              if (__ballot(more) == 0) break;
              // the records that did not fit
              Patience again;
              for (;;) {
                rec = more ? mail_load(&box[kUnits + i + (uint32_t)per]) : 0;
                if (__ballot(more && (uint32_t)(rec >> 48) != rtag) == 0) break;
                if (again.over(gone)) {
                  *dead = round_tag + 1;
                  total = 0;
                  break;
                }
              }
            }
          }
          __syncthreads();
        }
        add_round(round_tag);
        phase += (unsigned long long)r;
        if (given_up()) break;
      }
      trials_total += done;
      // the sweep's accepted energy changes
      if (evaluates && first && isA) vsum[32 * e + lane] = sum;
      E += total_of_rows();
      if (sampled) {
        trials_sampled += done;
        if (part == 0 && tid == 0) {
          step_E = step_E + E;
          step_Esq = step_Esq + E * E;
          if (C.e_trace) C.e_trace[(long long)t * C.n_sweeps + (sw - C.burn_sweeps)] = E;
        }
        if (C.asro_every > 0 && (sw - C.burn_sweeps + 1) % C.asro_every == 0)
          asro_sample<LAT, R, CW, NC, FIELD>(lat, N, nullptr, S, part * n_threads + tid, parts * n_threads, true,
                                             hacc);
      }
    }
    // the step's accepted trials and shell pair counts
    if constexpr (ALONE) {
      __syncthreads();
      unsigned long long v = acc_local;
#pragma unroll
      for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
      unsigned long long *accs = (unsigned long long *)late;
      if (lane == 0) accs[wave] = v;
      __syncthreads();
      if (C.asro_every > 0) write_rho<LAT, R>(C, hacc, S, t);
      if (tid == 0) {
        unsigned long long s = 0;
        for (int k = 0; k < n_waves; ++k) s += accs[k];
        write_step(C, t, temp, sim_temp, step_E, step_Esq, s, trials_sampled);
        acc_total += (long long)s;
      }
      __syncthreads();
      for (int i = tid; i < S * S * R; i += n_threads) hacc[i] = 0ull;
    } else {
      // every part's to the first
      __syncthreads();
      unsigned long long v = acc_local;
#pragma unroll
      for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
      unsigned long long *ends = mend + (size_t)(t & 1) * parts * end_words;
      unsigned long long *mine = ends + (size_t)part * end_words;
      unsigned long long *accs = (unsigned long long *)late;
      if (lane == 0) accs[wave] = v;
      __syncthreads();
      if (tid == 0) {
        unsigned long long s = 0;
        for (int k = 0; k < kSplitWaves; ++k) s += accs[k];
        mail_store(&mine[0], s);
      }
      for (int i = tid; i < S * S * R; i += kSplitThreads) {
        mail_store(&mine[1 + i], hacc[i]);
        hacc[i] = 0ull;
      }
      __threadfence();
      __syncthreads();
      if (tid == 0) mail_store(&mine[end_words - 1], (unsigned long long)(uint32_t)(t + 1) << 32);
      if (part == 0) {
        if (wave == 0) {
          unsigned long long w = 0;
          if (!mail_wait(&ends[(size_t)(lane < parts ? lane : 0) * end_words + end_words - 1], lane < parts,
                         (uint32_t)(t + 1), gone, w))
            *dead = round_tag + 1;
        }
        __syncthreads();
        __threadfence();
        for (int i = tid; i < S * S * R; i += kSplitThreads) {
          unsigned long long s = 0;
          for (int k = 0; k < parts; ++k) s += mail_load(&ends[(size_t)k * end_words + 1 + i]);
          hacc[i] = s;
        }
        __syncthreads();
        if (C.asro_every > 0) write_rho<LAT, R>(C, hacc, S, t);
        if (tid == 0) {
          unsigned long long s = 0;
          for (int k = 0; k < parts; ++k) s += mail_load(&ends[(size_t)k * end_words]);
          write_step(C, t, temp, sim_temp, step_E, step_Esq, s, trials_sampled);
          acc_total += (long long)s;
        }
        __syncthreads();
        for (int i = tid; i < S * S * R; i += kSplitThreads) hacc[i] = 0ull;
      }
    }
    const double Er = recount();
    if (part == 0 && tid == 0) {
      C.e_drift[t] = E - Er;
      C.e_drift[C.T_steps + t] = Er;
    }
    E = Er;
  }
  __syncthreads();
  // (a part that gave up said so before its last words, which this one has read)
  if (ALONE || (part == 0 && !given_up() && mail_load(gone) == 0)) {
    nat_unstage<LAT>(lat, C.compact, g, N, FIELD);
    if (tid == 0) {
      C.counters[0] = (long long)phase;
      C.counters[1] += acc_total;
      C.counters[2] += trials_total;
      C.counters[3] = 1;  // the chain is complete
    }
  }
}

}  // namespace

}  // namespace bwl
