// bwl_setup.hip -- initial configurations (initial_setup, initialise.F90:
// 434-617) of many walkers on the device, each drawn from its stream exactly
// as the host's initial_setup_host draws it.
//
// The rule: sites are filled in a fixed order; a site takes draws until one
// names a species with atoms left.  A draw is therefore taken exactly when
// fewer than count(s) earlier draws of the walker named its species s, and
// the site it fills is the number of draws taken before it: both are prefix
// counts, so a wavefront settles 64 draws at once with one ballot a species.
// A draw that lies on the bound of two species (the bounds are inclusive on
// both sides) goes to the first of them with atoms left; such a draw is
// settled alone.
//
// One workgroup follows one stream: wavefront 0 places the walkers one after
// another (where a walker starts in the stream depends on the one before it),
// wavefront 1 makes the stream's next 624 draws meanwhile.  Wavefront 0's
// instructions bound it.  128 walkers of 864 sites, 5 species: 1.8 ms on the
// host, 1.6 ms here, but the streams of a batch run side by side: 32 such runs
// 64 ms on the host, 1.6 ms here.
#include <hip/hip_runtime.h>

#include "bwl_kernels.h"
#include "bwl_spec.h"

namespace bwl {

namespace {

constexpr long long kSetupDraws = 1LL << 26;  // a walker's; its mean is at most 10^4 a species beyond the sites
constexpr int kAtOnce = 4;                    // groups of 64 draws

__global__ __launch_bounds__(128) void k_setup(const SetupArgs *__restrict__ args) {
  __shared__ uint32_t raw[624];
  __shared__ uint32_t tem[kRingWords];
  __shared__ volatile int32_t last;  // the barrier after which wavefront 1 leaves, counted from 1
  const SetupArgs &A = args[blockIdx.x];
  if (A.made || A.n_walkers < 1) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = wave_uniform(tid >> 6);
  if (tid == 0) last = 0;
  for (int i = tid; i < 624; i += 128) {
    const uint32_t v = A.mt[i];
    raw[i] = v;
    tem[i] = mt_temper(v);
  }
  __syncthreads();
  int half = 0, turn = 0;
  if (wave != 0) {
    for (;;) {
      ring_twist(raw, tem, half);
      __syncthreads();
      if (last == ++turn) return;
      half = 624 - half;
    }
  }
  int pos = wave_uniform(A.mt_index[0]);
  const int n_atoms = A.g.n_atoms, S = A.g.S, n_walkers = A.n_walkers;
  int status = 0;
  auto refill = [&]() {
    if (pos < 624) return;
    __syncthreads();
    ++turn;
    half = 624 - half;
    pos = 0;
  };
  uint32_t lo[kMaxSpecies], hi[kMaxSpecies];
  int count[kMaxSpecies];
#pragma unroll
  for (int s = 0; s < kMaxSpecies; ++s) {
    lo[s] = (uint32_t)wave_uniform((int)A.rule.lo[s]);
    hi[s] = (uint32_t)wave_uniform((int)A.rule.hi[s]);
    count[s] = wave_uniform(A.rule.count[s]);
  }
  int8_t *const orders = A.order;
  double *const rnde = A.rnde;
  for (int w = 0; w < n_walkers; ++w) {
    int8_t *out = orders + (size_t)w * n_atoms;
    int room[kMaxSpecies];
#pragma unroll
    for (int s = 0; s < kMaxSpecies; ++s) room[s] = s < S ? count[s] : 0;
    int filled = 0;
    long long draws = 0;
    while (filled < n_atoms) {
      refill();
      // up to 256 draws at once while no species runs out among them
      {
        const int ahead = 624 - pos;
        uint32_t k[kAtOnce];
        unsigned long long any[kAtOnce], twice = 0;
        int mine[kAtOnce], left[kMaxSpecies];
        bool fits = true;
#pragma unroll
        for (int j = 0; j < kAtOnce; ++j) {
          k[j] = tem[half + min(pos + 64 * j + lane, 623)];
          any[j] = 0;
          mine[j] = 0;
        }
#pragma unroll
        for (int s = 0; s < kMaxSpecies; ++s) {
          left[s] = room[s];
          if (s < S) {
#pragma unroll
            for (int j = 0; j < kAtOnce; ++j) {
              const bool in = k[j] - lo[s] <= hi[s] - lo[s] && lo[s] <= hi[s] && 64 * j + lane < ahead;
              const unsigned long long b = __ballot(in);
              twice |= any[j] & b;
              any[j] |= b;
              left[s] -= __popcll(b);
              if (in) mine[j] = s + 1;
            }
            fits = fits && left[s] >= 0;
          }
        }
        if (fits && !twice) {
#pragma unroll
          for (int j = 0; j < kAtOnce; ++j) {
            if (mine[j])
              out[filled + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(any[j] >> 32),
                                                          __builtin_amdgcn_mbcnt_lo((uint32_t)any[j], 0))] = (int8_t)mine[j];
            filled += __popcll(any[j]);
          }
#pragma unroll
          for (int s = 0; s < kMaxSpecies; ++s) room[s] = left[s];
          // (the last site's draw is the last one taken)
          int used = min(64 * kAtOnce, ahead);
          if (filled == n_atoms) {
            used = 0;
#pragma unroll
            for (int j = 0; j < kAtOnce; ++j)
              if (any[j]) used = 64 * j + 64 - __clzll((long long)any[j]);
          }
          pos += used;
          draws += used;
          continue;
        }
      }
      int n = min(64, 624 - pos);
      const uint32_t k = tem[half + pos + min(lane, n - 1)];
      const unsigned long long inside = n < 64 ? (1ull << n) - 1ull : ~0ull;
      unsigned long long named[kMaxSpecies], any = 0, twice = 0;
#pragma unroll
      for (int s = 0; s < kMaxSpecies; ++s) {
        named[s] = s < S ? __ballot(k >= lo[s] && k <= hi[s]) & inside : 0ull;
        twice |= any & named[s];
        any |= named[s];
      }
      if (twice) {
        const int at = __ffsll((long long)twice) - 1;
        n = at > 0 ? at : 1;
        const unsigned long long keep = (1ull << n) - 1ull;
        bool open = true;
#pragma unroll
        for (int s = 0; s < kMaxSpecies; ++s) {
          named[s] &= keep;
          if (at == 0) {
            if (!open || room[s] == 0) named[s] = 0;
            if (named[s]) open = false;
          }
        }
      }
      unsigned long long taken = 0;
      int mine = 0;
#pragma unroll
      for (int s = 0; s < kMaxSpecies; ++s) {
        int c = __popcll(named[s]);
        if (c > room[s]) {
          const bool first = ((named[s] >> lane) & 1) != 0 &&
                             (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(named[s] >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)named[s], 0)) < room[s];
          named[s] = __ballot(first);
          c = room[s];
        }
        room[s] -= c;
        taken |= named[s];
        if ((named[s] >> lane) & 1) mine = s + 1;
      }
      if (mine)
        out[filled + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(taken >> 32),
                                                    __builtin_amdgcn_mbcnt_lo((uint32_t)taken, 0))] = (int8_t)mine;
      filled += __popcll(taken);
      pos += filled == n_atoms ? 64 - __clzll((long long)taken) : n;
      draws += n;
      if (draws > kSetupDraws) {
        // (every site gets a species: the kernels after this one read them all)
        for (int i = filled + lane; i < n_atoms; i += 64) out[i] = 1;
        filled = n_atoms;
        status = 1;
      }
    }
    if (rnde) {
      refill();
      if (lane == 0) rnde[w] = (double)tem[half + pos] * (1.0 / 4294967296.0);
      ++pos;
    }
  }
  // the state is the block in use; it lies in the other half of the draws
  // than the one wavefront 1 is making
  for (int i = lane; i < 624; i += 64) A.mt[i] = mt_untemper(tem[half + i]);
  if (lane == 0) {
    A.mt_index[0] = pos;
    *A.status = status;
    last = turn + 1;
  }
  __syncthreads();
}

// From the order of set-up to the compact layout.
__global__ void k_order_to_compact(const SetupArgs *__restrict__ args, int max_walkers) {
  const SetupArgs &A = args[blockIdx.z];
  const Geo &g = A.g;
  const int n0 = g.n[0], plane = g.n[0] * g.n[1], cells = plane * g.n[2];
  for (int w = blockIdx.y; w < max_walkers; w += gridDim.y) {
    if (w >= A.n_walkers) return;
    const int8_t *from = A.order + (size_t)w * g.n_atoms;
    int8_t *to = A.walkers + (size_t)w * g.compact_bytes;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < g.n_atoms; i += gridDim.x * blockDim.x) {
      const int s = i / cells;
      int r = i - s * cells;
      const int cz = r / plane;
      r -= cz * plane;
      int bx, by, bz;
      sub_bits(g.lattice, s, bx, by, bz);
      const int z = 2 * cz + bz;
      if (g.lattice == 1) {
        const int cy = r / n0, cx = r - cy * n0;
        to[i] = from[(z * g.m[1] + 2 * cy + by) * n0 + cx];
      } else {
        to[i] = from[z * plane + r];
      }
    }
  }
}

}  // namespace

hipError_t launch_setup(const SetupArgs *args_dev, int n, int max_walkers, int max_atoms, bool any_drawn, hipStream_t s) {
  for (int first = 0; first < n; first += 65535) {
    const int m = n - first < 65535 ? n - first : 65535;
    if (any_drawn) hipLaunchKernelGGL(k_setup, dim3(m), dim3(128), 0, s, args_dev + first);
    const int blocks = (max_atoms + 1023) / 1024;
    hipLaunchKernelGGL(k_order_to_compact, dim3(blocks < 64 ? blocks : 64, max_walkers < 65535 ? max_walkers : 65535, m),
                       dim3(256), 0, s, args_dev + first, max_walkers);
  }
  return hipGetLastError();
}

}  // namespace bwl
