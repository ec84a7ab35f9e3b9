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
// One workgroup follows one stream in a pipeline of blocks of 624 draws:
// wavefront 1 makes a block's draws, wavefronts 2 and 3 then the species that
// each names and, per 64 draws, the mask of those that name a species, and
// wavefront 0 places the walkers one after another from those (where a walker
// starts in the stream depends on the one before it); the four meet at one
// barrier a block.  The chain of wavefront 0's steps bounds it.  128 walkers
// of 864 sites, 5 species: 1.8 ms on the host, 1.6 ms with the masks formed in
// the chain, 0.76 ms so; the streams of a batch run side by side (32 of them: 64 ms
// on the host).
#include <hip/hip_runtime.h>

#include "bwl_kernels.h"
#include "bwl_spec.h"

namespace bwl {

namespace {

constexpr int kSetupThreads = 256;
constexpr int kGroups = 10;        // of 64 draws in a block, the last of 48
constexpr int kAny = kMaxSpecies;  // masks of a group: per species, of all that name one,
constexpr int kTwice = kAny + 1;   // of those that name two
constexpr int kMasks = kTwice + 1;

__device__ __forceinline__ unsigned long long lane_mask(unsigned long long v, int l) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), l);
  return ((unsigned long long)hi << 32) | lo;
}

__global__ __launch_bounds__(kSetupThreads) void k_setup(const SetupArgs *__restrict__ args) {
  __shared__ uint32_t raw[624];
  __shared__ uint32_t tem[3][624];
  __shared__ uint8_t code[2][64 * kGroups];
  __shared__ unsigned long long masks[2][kGroups][kMasks];
  __shared__ volatile int32_t last;  // the barrier after which the helpers leave, counted from 1
  const SetupArgs &A = args[blockIdx.x];
  if (A.made || A.n_walkers < 1) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = wave_uniform(tid >> 6);
  const int S = A.g.S;
  if (tid == 0) last = 0;
  for (int i = tid; i < 624; i += kSetupThreads) {
    const uint32_t v = A.mt[i];
    raw[i] = v;
    tem[0][i] = mt_temper(v);
  }
  __syncthreads();
  // block b's draws lie in tem[b mod 3], what they name in slot b mod 2
  auto classify = [&](int b) {
    const uint32_t *t = tem[b % 3];
    for (int j = wave - 2; j < kGroups; j += 2) {
      const bool there = 64 * j + lane < 624;
      const uint32_t k = t[there ? 64 * j + lane : 623];
      unsigned long long any = 0, twice = 0, mine = 0;
      int names = 0;
      for (int s = 0; s < S; ++s) {
        const bool in = there && k >= A.rule.lo[s] && k <= A.rule.hi[s];
        const unsigned long long m = __ballot(in);
        twice |= any & m;
        any |= m;
        if (in) names = s + 1;
        if (lane == s) mine = m;
      }
      if (lane == kAny) mine = any;
      if (lane == kTwice) mine = twice;
      code[b & 1][64 * j + lane] = (uint8_t)names;
      if (lane < kMasks) masks[b & 1][j][lane] = mine;
    }
  };
  auto twist = [&](int b) { ring_twist(raw, tem[b % 3] - 624, 0); };  // (to tem[b mod 3])
  if (wave == 1) twist(1);
  if (wave >= 2) classify(0);
  __syncthreads();
  int turn = 0;  // barriers since, and the block that wavefront 0 uses
  if (wave != 0) {
    for (;;) {
      if (wave == 1)
        twist(turn + 2);
      else
        classify(turn + 1);
      __syncthreads();
      if (last == ++turn) return;
    }
  }
  int pos = wave_uniform(A.mt_index[0]);
  const int n_atoms = A.g.n_atoms, n_walkers = A.n_walkers;
  // lane s keeps species s
  const uint32_t lo = lane < S ? A.rule.lo[lane] : 1u, hi = lane < S ? A.rule.hi[lane] : 0u;
  const int count = lane < S ? A.rule.count[lane] : 0;
  int8_t *const orders = A.order;
  double *const rnde = A.rnde;
  int status = 0;
  auto refill = [&]() {
    if (pos < 624) return;
    __syncthreads();
    ++turn;
    pos = 0;
  };
  for (int w = 0; w < n_walkers; ++w) {
    int8_t *out = orders + (size_t)w * n_atoms;
    int room = count, filled = 0;
    long long draws = 0;
    while (filled < n_atoms) {
      refill();
      const int j = pos >> 6, off = pos & 63;
      const unsigned long long *M = masks[turn & 1][j];
      const unsigned long long m = M[lane < kMasks ? lane : 0];
      const int names = code[turn & 1][64 * j + lane];
      unsigned long long window = ~0ull << off;
      int end = min(64, 624 - 64 * j);
      const unsigned long long twice = lane_mask(m, kTwice) & window;
      if (twice) {
        const int at = __ffsll((long long)twice) - 1;
        if (at == off) {
          const uint32_t k = tem[turn % 3][pos];
          const unsigned long long b = __ballot(k >= lo && k <= hi && room > 0);
          if (b) {
            const int s = __ffsll((long long)b) - 1;
            if (lane == s) {
              --room;
              out[filled] = (int8_t)(s + 1);
            }
            ++filled;
          }
          ++pos;
          ++draws;
          continue;
        }
        window &= (1ull << at) - 1ull;
        end = at;
      }
      const int c = lane < kMaxSpecies ? __popcll(m & window) : 0;
      unsigned long long taken = lane_mask(m, kAny) & window;
      if (__ballot(c > room && lane < kMaxSpecies)) {
        // a species runs out: its first draws are taken
        const unsigned long long own = M[names ? names - 1 : 0] & window;
        const int before = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(own >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)own, 0));
        const int open = __shfl(room, names ? names - 1 : 0);
        taken = __ballot(((taken >> lane) & 1) != 0 && before < open);
      }
      room -= min(c, room);
      if ((taken >> lane) & 1)
        out[filled + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(taken >> 32),
                                                    __builtin_amdgcn_mbcnt_lo((uint32_t)taken, 0))] = (int8_t)names;
      filled += __popcll(taken);
      draws += end - off;
      // (the last site's draw is the last one taken)
      pos = 64 * j + (filled == n_atoms ? 64 - __clzll((long long)taken) : end);
      if (draws > kSetupDraws && filled < n_atoms) {
        // (every site gets a species: the kernels after this one read them all)
        for (int i = filled + lane; i < n_atoms; i += 64) out[i] = 1;
        filled = n_atoms;
        status = 1;
      }
    }
    if (rnde) {
      refill();
      if (lane == 0) rnde[w] = (double)tem[turn % 3][pos] * (1.0 / 4294967296.0);
      ++pos;
    }
  }
  // the state is that of the block in use
  for (int i = lane; i < 624; i += 64) A.mt[i] = mt_untemper(tem[turn % 3][i]);
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
    if (any_drawn) hipLaunchKernelGGL(k_setup, dim3(m), dim3(kSetupThreads), 0, s, args_dev + first);
    const int blocks = (max_atoms + 1023) / 1024;
    hipLaunchKernelGGL(k_order_to_compact, dim3(blocks < 64 ? blocks : 64, max_walkers < 65535 ? max_walkers : 65535, m),
                       dim3(256), 0, s, args_dev + first, max_walkers);
  }
  return hipGetLastError();
}

}  // namespace bwl
