// bwl_ctx.h -- the context behind the C-ABI's opaque bwl_ctx handle, and
// the error plumbing shared by the C-ABI source files.
#pragma once

#include <hip/hip_runtime.h>
#include <string.h>

#include <string>
#include <vector>

#include "../../include/brawl_hip.h"
#include "bwl_host.h"
#include "bwl_kernels.h"
#include "bwl_pinned.h"

namespace bwl {
// message of the last failure on this thread (bwl_last_error)
extern thread_local std::string g_err;

inline int fail(int code, const std::string &msg) {
  g_err = msg;
  return code;
}
}  // namespace bwl

#define HIP_OK(call)                                                                    \
  do {                                                                                  \
    hipError_t e_ = (call);                                                             \
    if (e_ != hipSuccess)                                                               \
      return bwl::fail(BWL_ERR_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

struct bwl_ctx {
  bwl_lattice_desc desc;
  bwl::Geo g;
  std::vector<int32_t> off;
  std::vector<double> vex;
  hipStream_t stream = nullptr;
  int device = 0;
  int8_t *d_compact = nullptr;
  int8_t *d_ref = nullptr;
  int32_t *d_off = nullptr;
  double *d_vex = nullptr;
  void *d_scratch = nullptr;  // small per-call outputs
  size_t scratch_bytes = 0;
  bool has_config = false;
  bwl::MT19937 mt;
  unsigned long long phase = 0;  // parallel-sampler round counter
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  std::vector<hipStream_t> side;  // further streams of the context's batches
  bool held = false;      // counted by pinned_hold
  bool borrowed = false;  // device memory and stream belong to someone else
  int32_t layout = 0;     // parallel-sampler layout: 0 by rule, else BWL_LAYOUT_*
  int32_t threads = 0;    // parallel-sampler threads per chain: 0 by rule
  // how the last anneal ran: workgroups, whether its division was given up,
  // whether it took one site per lane in one workgroup
  int32_t ran[3] = {0, 0, 0};
  bool give_up = false;  // the parts of a divided anneal find it given up
};

namespace bwl {

// Most bytes of streams and results that a call keeps in pinned memory.
constexpr size_t kPinnedSeries = size_t(4) << 20;
// Largest configuration (reference layout) that goes through pinned memory.
// Beyond, allocating the block makes a first call slower (8 MB up: 4.7 ms
// against 2.0) and later ones are no faster (1.9 ms both ways).
constexpr size_t kPinnedConfig = size_t(1) << 20;
// Most bytes of a request's configuration, and of a launch's final ones at a
// time, that the request server passes through pinned memory.
constexpr size_t kPinnedServed = size_t(16) << 20;

inline int ensure_scratch(bwl_ctx *c, size_t bytes) {
  if (bytes <= c->scratch_bytes) return BWL_OK;
  if (c->d_scratch) HIP_OK(hipFree(c->d_scratch));
  c->d_scratch = nullptr;
  c->scratch_bytes = 0;
  if (hipMalloc(&c->d_scratch, bytes) != hipSuccess) return fail(BWL_ERR_NOMEM, "device allocation failed");
  c->scratch_bytes = bytes;
  return BWL_OK;
}

inline int check_ctx(bwl_ctx *c, bool need_config) {
  if (!c) return fail(BWL_ERR_ARG, "null context");
  if (need_config && !c->has_config) return fail(BWL_ERR_STATE, "no configuration uploaded");
  HIP_OK(hipSetDevice(c->device));
  return BWL_OK;
}

inline int lds_limit() {
  int dev = 0, v = 0;
  if (hipGetDevice(&dev) != hipSuccess) return kLdsBytes;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeSharedMemPerBlockOptin, dev) == hipSuccess && v > 0)
    return v;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess && v > 0)
    return v;
  return kLdsBytes;
}

// A context whose device buffers live in caller-provided memory (`bytes` >=
// ctx_device_bytes) and whose uploads go on `stream`; bwl_destroy frees
// neither.
size_t ctx_device_bytes(const bwl_lattice_desc &d);
// tables: ctx_tables_bytes of (pinned) memory for the upload, kept until it
// has ended
size_t ctx_tables_bytes(const Geo &g);
int ctx_create_borrowed(const bwl_lattice_desc &d, const double *v_ex, char *mem, size_t bytes,
                        hipStream_t stream, char *tables, bwl_ctx **out);

// Workgroups of divided chains on each XCD of a device.
struct SplitLanes {
  int parts[8] = {0, 0, 0, 0, 0, 0, 0, 0};
};

// The undivided workgroups of a call or launch while it is in flight, a CU
// each (a device's at most): those CUs are not offered to chains that could be
// divided.  Calls of one short kernel (an energy, a configuration) are not
// counted; the parts of a chain wait that long for their CUs.
class CuUse {
 public:
  CuUse(int device, long long workgroups);
  ~CuUse();
  CuUse(const CuUse &) = delete;
  CuUse &operator=(const CuUse &) = delete;

 private:
  int device_ = -1, n_ = 0;
};

// A batch of anneals prepared on the host (anneal_plan), its arguments and
// buffers placed in caller-provided device memory (anneal_upload), its
// launches enqueued one group per stream (anneal_launch), and its outputs
// copied out after completion (anneal_collect).
struct AnnealPlan {
  struct Item {
    int idx = 0;
    const void *fn = nullptr;
    int threads = 0;
    size_t lds = 0;
    ParArgs a;
    ParPlan plan;
    size_t T = 0, off_muls = 0, off_out = 0, off_cnt = 0, off_rho = 0, rho_n = 0;
    size_t off_mail = 0, mail_n = 0;  // mailbox of a divided chain, in words
    const void *split_fn = nullptr;   // kernel that can divide the chain, if any
    bool natural = false;             // held in lattice coordinates
    bool split_fixed = false;         // ... at the fixed pitch
    bool alone = false;               // runs k_metro_alone
    int chunks = 0, passes = 0;       // most pairs of a round, in 64s and per thread
    int lane = 0;                     // XCD of a divided chain's parts
    double rounds = 0.0;              // rounds of the whole anneal, about
    double work = 0.0;
  };
  struct Group {
    const void *fn;
    int threads;
    size_t lds;
    std::vector<int> members;
    size_t off_args;
    bool split;                 // a divided group: block b runs map[b]
    std::vector<int2> map;
    size_t off_map;
  };
  std::vector<Item> items;
  std::vector<Group> groups;
  std::vector<char> image;  // what goes up, kept alive until the upload has ended
  size_t out_bytes = 0, up_bytes = 0, scratch_bytes = 0;
  char *base = nullptr;
  SplitLanes split;  // workgroups of its divided chains
};
// The parallel-sampler kernel variant, block size and LDS for a lattice:
// layout 0 takes the first that fits of fixed pitch, own pitch, per
// sublattice; a BWL_LAYOUT_* value takes only that one.  threads_req > 0
// asks for that many threads per chain instead of the rule's count (layout
// 0 then takes the first layout that can run them).
int anneal_kernel(const Geo &g, ParPlan &plan, NatGeo &nat, const void *&fn, int &threads,
                  size_t &lds, bool *natural = nullptr, int layout = 0, int threads_req = 0);
// About how long a chain takes in one workgroup, in us.
double anneal_estimate_us(const Geo &g, const ParPlan &plan, const bwl_anneal_params &p);
// split: the workgroups that chains may be divided into (none: no chain is
// divided); AnnealPlan::split says how many the divided chains take.
int anneal_plan(int n, bwl_ctx *const *ctxs, const bwl_anneal_params *params, AnnealPlan &P,
                const SplitLanes *split = nullptr);
// image: up_bytes of (pinned) memory for what goes up, else the plan's own.
// No memset unless chains are divided.
int anneal_upload(AnnealPlan &P, char *scratch_dev, hipStream_t s, char *image = nullptr);
int anneal_launch(const AnnealPlan &P, const hipStream_t *streams);
int anneal_collect(const AnnealPlan &P, bwl_ctx *const *ctxs, double *const *energies_of_T,
                   double *const *C_of_T, double *const *acceptance_of_T, bwl_run_stats *stats,
                   double kernel_ms, hipStream_t s, double *const *rho_of_T = nullptr,
                   std::vector<int> *again = nullptr, char *host = nullptr);
// The whole call: plan (dividing chains over idle CUs), upload, launch, wait,
// collect.
int anneal_run(int n, bwl_ctx *const *ctxs, const bwl_anneal_params *params, double *const *energies_of_T,
               double *const *C_of_T, double *const *acceptance_of_T, bwl_run_stats *stats, double *makespan_ms,
               double *const *rho_of_T, bool divide = true);

// Device buffer freed at scope exit.
struct DevBuf {
  void *p = nullptr;
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
};

}  // namespace bwl

// bwl_ctx::ran, for the tests and the benchmark's labels, and bwl_ctx::give_up,
// for the tests (neither is part of include/brawl_hip.h).
extern "C" {
int bwl_test_anneal_ran(const bwl_ctx *c, int32_t *ran3);
int bwl_test_give_up(bwl_ctx *c, int32_t on);
}
