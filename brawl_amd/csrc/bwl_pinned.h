// bwl_pinned.h -- pinned host memory that kernels read and write in place.
//
// The calls that move little (a trial's random stream, an energy, a
// configuration) were bound by their copies: each hipMemcpyAsync to or from
// ordinary memory is a launch of its own and a wait (5-15 us).  Their kernels
// now read their inputs from a block of pinned memory and write their results
// to it, one launch and one wait a call: a pair energy 46 -> 18 us, one
// bound Monte Carlo trial with the configuration up and down 106 -> 60 us.
//
// Blocks come from a pool for the process.  A call holds its block until its
// kernels have ended.  The pool keeps returned blocks, at most kPinnedKept
// bytes of them, while any context or server lives, and frees them with the
// last.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace bwl {

constexpr size_t kPinnedKept = size_t(32) << 20;

// A context or server lives (hold) or has gone (drop).
void pinned_hold();
void pinned_drop();

// Whether the pool holds a block for that many bytes.
bool pinned_ready(size_t bytes);

// A block of pinned memory for work on `stream`.  It goes back to the pool
// when the object does, after the stream's work unless settled() said that
// the work has ended.
class Pinned {
 public:
  Pinned() = default;
  ~Pinned();
  Pinned(const Pinned &) = delete;
  Pinned &operator=(const Pinned &) = delete;
  bool take(size_t bytes, hipStream_t stream);
  void settled() { busy_ = false; }
  char *p = nullptr;

 private:
  size_t size_ = 0;
  hipStream_t stream_ = nullptr;
  bool busy_ = false;
};

}  // namespace bwl
