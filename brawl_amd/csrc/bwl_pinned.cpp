// bwl_pinned.cpp -- the pool behind bwl_pinned.h.
#include "bwl_pinned.h"

#include <map>
#include <mutex>
#include <vector>

namespace bwl {

namespace {

struct Pool {
  std::mutex mu;
  std::map<size_t, std::vector<void *>> kept;  // by size
  size_t bytes = 0;                            // kept
  int users = 0;
};

// (never destroyed: the HIP runtime may be gone by then)
Pool &pool() {
  static Pool *p = new Pool;
  return *p;
}

size_t block_size(size_t n) {
  size_t s = 4096;
  while (s < n) s *= 2;
  return s;
}

}  // namespace

void pinned_hold() {
  Pool &P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  ++P.users;
}

void pinned_drop() {
  Pool &P = pool();
  std::vector<void *> gone;
  {
    std::lock_guard<std::mutex> lock(P.mu);
    if (--P.users > 0) return;
    for (auto &k : P.kept) gone.insert(gone.end(), k.second.begin(), k.second.end());
    P.kept.clear();
    P.bytes = 0;
  }
  for (void *p : gone) (void)hipHostFree(p);
}

bool pinned_ready(size_t bytes) {
  Pool &P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  const auto it = P.kept.find(block_size(bytes));
  return it != P.kept.end() && !it->second.empty();
}

bool Pinned::take(size_t bytes, hipStream_t stream) {
  const size_t n = block_size(bytes);
  Pool &P = pool();
  {
    std::lock_guard<std::mutex> lock(P.mu);
    auto it = P.kept.find(n);
    if (it != P.kept.end() && !it->second.empty()) {
      p = (char *)it->second.back();
      it->second.pop_back();
      P.bytes -= n;
    }
  }
  if (!p && hipHostMalloc((void **)&p, n, hipHostMallocPortable) != hipSuccess) {
    p = nullptr;
    return false;
  }
  size_ = n;
  stream_ = stream;
  busy_ = true;
  return true;
}

Pinned::~Pinned() {
  if (!p) return;
  if (busy_) (void)hipStreamSynchronize(stream_);
  Pool &P = pool();
  {
    std::lock_guard<std::mutex> lock(P.mu);
    if (P.users > 0 && P.bytes + size_ <= kPinnedKept) {
      P.kept[size_].push_back(p);
      P.bytes += size_;
      return;
    }
  }
  (void)hipHostFree(p);
}

}  // namespace bwl
