// bwl_seq_singly.hip -- the bit-exact Metropolis kernels in speculative batches
// that take trials singly where batches are cut short (bwl_seq_batches.h).
#include <hip/hip_runtime.h>

#include "bwl_seq_batches.h"

namespace bwl {

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

template <int KEY>
const void *singly_of(bool batch) {
  return batch ? (const void *)k_metro_seq_singly_batch<KEY> : (const void *)k_metro_seq_singly<KEY>;
}

}  // namespace

const void *metro_seq_singly_kernel(const SeqPick &pick, bool batch) {
  if (pick.reach <= (pick.key % 16 == 2 ? 0.3 : 0.18)) return nullptr;
  switch (pick.key) {
    case 16 + 2: return singly_of<16 + 2>(batch);
    case 16 + 3: return singly_of<16 + 3>(batch);
    case 16 + 4: return singly_of<16 + 4>(batch);
    case 32 + 2: return singly_of<32 + 2>(batch);
    case 32 + 3: return singly_of<32 + 3>(batch);
    case 32 + 4: return singly_of<32 + 4>(batch);
  }
  return nullptr;
}

}  // namespace bwl
