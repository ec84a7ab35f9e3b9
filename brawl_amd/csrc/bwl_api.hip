// bwl_api.hip -- the C-ABI (include/brawl_hip.h) over the gfx950 kernels.
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>
#include <unistd.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "bwl_ctx.h"

using namespace bwl;

namespace bwl {
thread_local std::string g_err;
}

extern "C" {

const char *bwl_last_error(void) { return g_err.c_str(); }

int bwl_device_count(int32_t *count) {
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess) n = 0;
  if (count) *count = n;
  return e == hipSuccess ? BWL_OK : fail(BWL_ERR_DEVICE, hipGetErrorString(e));
}

int bwl_lds_bandwidth(int32_t iters, double *bytes_per_s, int32_t *cus) {
  if (iters < 1 || !bytes_per_s || !cus) return fail(BWL_ERR_ARG, "bad argument");
  int dev = 0, n_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      n_cu < 1)
    return fail(BWL_ERR_DEVICE, "no HIP device");
  // two 64 KiB, 1024-thread blocks per CU run at once; 8 blocks per CU in all
  const int blocks = 8 * n_cu;
  DevBuf sink;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  bool ok = hipMalloc(&sink.p, sizeof(uint32_t) * blocks) == hipSuccess &&
            hipEventCreate(&e0) == hipSuccess && hipEventCreate(&e1) == hipSuccess &&
            launch_lds_bandwidth(blocks, 16, (uint32_t *)sink.p, 0) == hipSuccess &&  // warm-up
            hipEventRecord(e0, 0) == hipSuccess &&
            launch_lds_bandwidth(blocks, iters, (uint32_t *)sink.p, 0) == hipSuccess &&
            hipEventRecord(e1, 0) == hipSuccess && hipEventSynchronize(e1) == hipSuccess;
  float ms = 0.0f;
  if (ok) ok = hipEventElapsedTime(&ms, e0, e1) == hipSuccess && ms > 0.0f;
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (!ok) return fail(BWL_ERR_DEVICE, "LDS bandwidth probe failed");
  *bytes_per_s = (double)blocks * 1024.0 * (double)iters * 16.0 / ((double)ms * 1e-3);
  *cus = n_cu;
  return BWL_OK;
}

int bwl_create(const bwl_lattice_desc *desc, const double *v_ex, bwl_ctx **out) {
  if (!desc || !v_ex || !out) return fail(BWL_ERR_ARG, "null argument");
  *out = nullptr;
  bwl_ctx *c = new bwl_ctx();
  c->desc = *desc;
  int rc = make_geo(*desc, c->g, c->off, g_err);
  if (rc) {
    delete c;
    return rc;
  }
  const Geo &g = c->g;
  c->vex.assign(v_ex, v_ex + (size_t)g.S * g.S * g.R);
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n < 1) {
    delete c;
    return fail(BWL_ERR_DEVICE, "no HIP device available");
  }
  if (hipGetDevice(&c->device) != hipSuccess) c->device = 0;
  size_t ref_bytes = (size_t)g.m[0] * g.m[1] * g.m[2];
  bool ok = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) == hipSuccess &&
            hipMalloc(&c->d_compact, g.compact_bytes) == hipSuccess &&
            hipMalloc(&c->d_ref, ref_bytes) == hipSuccess &&
            hipMalloc(&c->d_off, sizeof(int32_t) * c->off.size()) == hipSuccess &&
            hipMalloc(&c->d_vex, sizeof(double) * c->vex.size()) == hipSuccess &&
            hipEventCreate(&c->ev0) == hipSuccess && hipEventCreate(&c->ev1) == hipSuccess;
  if (!ok) {
    bwl_destroy(c);
    return fail(BWL_ERR_NOMEM, "device allocation failed");
  }
  if (hipMemcpy(c->d_off, c->off.data(), sizeof(int32_t) * c->off.size(), hipMemcpyHostToDevice) !=
          hipSuccess ||
      hipMemcpy(c->d_vex, c->vex.data(), sizeof(double) * c->vex.size(), hipMemcpyHostToDevice) !=
          hipSuccess) {
    bwl_destroy(c);
    return fail(BWL_ERR_DEVICE, "upload failed");
  }
  pinned_hold();
  c->held = true;
  c->mt.seed(110179u);  // f90_init_genrand static seed, rank 0 (mt19937ar.c:138)
  *out = c;
  return BWL_OK;
}

int bwl_destroy(bwl_ctx *c) {
  if (!c) return BWL_OK;
  (void)hipSetDevice(c->device);
  if (c->stream && !c->borrowed) (void)hipStreamSynchronize(c->stream);
  for (hipStream_t s : c->side) {
    (void)hipStreamSynchronize(s);
    (void)hipStreamDestroy(s);
  }
  if (!c->borrowed) {
    (void)hipFree(c->d_compact);
    (void)hipFree(c->d_ref);
    (void)hipFree(c->d_off);
    (void)hipFree(c->d_vex);
  }
  if (c->d_scratch) (void)hipFree(c->d_scratch);
  if (c->ev0) (void)hipEventDestroy(c->ev0);
  if (c->ev1) (void)hipEventDestroy(c->ev1);
  if (c->stream && !c->borrowed) (void)hipStreamDestroy(c->stream);
  if (c->held) pinned_drop();
  delete c;
  return BWL_OK;
}

int bwl_n_atoms(const bwl_ctx *c, int32_t *n_atoms) {
  if (!c || !n_atoms) return fail(BWL_ERR_ARG, "null argument");
  *n_atoms = c->g.n_atoms;
  return BWL_OK;
}

int bwl_set_config(bwl_ctx *c, const int8_t *config) {
  int rc = check_ctx(c, false);
  if (rc) return rc;
  if (!config) return fail(BWL_ERR_ARG, "null config");
  rc = check_config(c->g, config, g_err);
  if (rc) return rc;
  size_t ref_bytes = (size_t)c->g.m[0] * c->g.m[1] * c->g.m[2];
  Pinned pin;
  const int8_t *from = c->d_ref;
  // (no block is allocated for a context's first configuration: a program that
  // creates a context, sets its configuration and destroys it took 192 us
  // against 162 by copy)
  if (ref_bytes <= kPinnedConfig && (c->has_config || pinned_ready(ref_bytes))) {
    if (!pin.take(ref_bytes, c->stream)) return fail(BWL_ERR_NOMEM, "pinned memory allocation failed");
    memcpy(pin.p, config, ref_bytes);
    from = (const int8_t *)pin.p;
  } else {
    HIP_OK(hipMemcpyAsync(c->d_ref, config, ref_bytes, hipMemcpyHostToDevice, c->stream));
  }
  HIP_OK(launch_pack(from, c->d_compact, c->g, c->stream));
  HIP_OK(hipStreamSynchronize(c->stream));
  pin.settled();
  c->has_config = true;
  return BWL_OK;
}

int bwl_get_config(bwl_ctx *c, int8_t *config) {
  int rc = check_ctx(c, true);
  if (rc) return rc;
  if (!config) return fail(BWL_ERR_ARG, "null config");
  size_t ref_bytes = (size_t)c->g.m[0] * c->g.m[1] * c->g.m[2];
  if (ref_bytes > kPinnedConfig) {
    HIP_OK(launch_unpack(c->d_compact, c->d_ref, c->g, c->stream));
    HIP_OK(hipMemcpyAsync(config, c->d_ref, ref_bytes, hipMemcpyDeviceToHost, c->stream));
    HIP_OK(hipStreamSynchronize(c->stream));
    return BWL_OK;
  }
  Pinned pin;
  if (!pin.take(ref_bytes, c->stream)) return fail(BWL_ERR_NOMEM, "pinned memory allocation failed");
  HIP_OK(launch_unpack(c->d_compact, (int8_t *)pin.p, c->g, c->stream));
  HIP_OK(hipStreamSynchronize(c->stream));
  pin.settled();
  memcpy(config, pin.p, ref_bytes);
  return BWL_OK;
}

int bwl_pair_histogram(bwl_ctx *c, int64_t *hist) {
  int rc = check_ctx(c, true);
  if (rc) return rc;
  if (!hist) return fail(BWL_ERR_ARG, "null hist");
  const Geo &g = c->g;
  const int threads = 512;
  if (hist_lds_bytes(g, threads) > (size_t)lds_limit())
    return fail(BWL_ERR_UNSUPPORTED, "lattice does not fit in LDS");
  const int hsize = g.S * g.S * g.R, blocks = hist_blocks(g);
  Pinned pin;
  if (!pin.take(sizeof(uint32_t) * (size_t)hsize * (size_t)blocks, c->stream))
    return fail(BWL_ERR_NOMEM, "pinned memory allocation failed");
  HistArgs a;
  a.g = g;
  a.compact = c->d_compact;
  a.off = c->d_off;
  a.parts = (uint32_t *)pin.p;
  HIP_OK(launch_histogram(a, blocks, c->stream));
  HIP_OK(hipStreamSynchronize(c->stream));
  pin.settled();
  for (int i = 0; i < hsize; ++i) hist[i] = 0;
  for (int k = 0; k < blocks; ++k)
    for (int i = 0; i < hsize; ++i) hist[i] += a.parts[(size_t)k * hsize + i];
  return BWL_OK;
}

int bwl_total_energy(bwl_ctx *c, double *energy) {
  if (!c || !energy) return fail(BWL_ERR_ARG, "null argument");
  std::vector<int64_t> h((size_t)c->g.S * c->g.S * c->g.R);
  int rc = bwl_pair_histogram(c, h.data());
  if (rc) return rc;
  const int S = c->g.S;
  double e = 0.0;
  for (int n = 0; n < c->g.R; ++n)
    for (int b = 0; b < S; ++b)
      for (int a = 0; a < S; ++a) {
        size_t i = a + (size_t)S * (b + (size_t)S * n);
        e += (double)h[i] * c->vex[i];
      }
  *energy = 0.5 * e;
  return BWL_OK;
}

static int site_pair(bwl_ctx *c, const int32_t *s1, const int32_t *s2, double *out2) {
  int rc = check_ctx(c, true);
  if (rc) return rc;
  const Geo &g = c->g;
  if (site_lds_bytes(g) > (size_t)lds_limit())
    return fail(BWL_ERR_UNSUPPORTED, "lattice does not fit in LDS");
  const int32_t *sites[2] = {s1, s2};
  SiteArgs a;
  a.g = g;
  for (int w = 0; w < 2; ++w) {
    const int32_t *s = sites[w];
    if (s[0] != 1) return fail(BWL_ERR_ARG, "basis index must be 1");
    int x = s[1] - 1, y = s[2] - 1, z = s[3] - 1;
    if (x < 0 || y < 0 || z < 0 || x >= g.m[0] || y >= g.m[1] || z >= g.m[2])
      return fail(BWL_ERR_ARG, "site index out of range");
    bool occ = g.lattice == BWL_FCC ? (((x + y + z) & 1) == 0)
                                    : ((x & 1) == (y & 1) && (y & 1) == (z & 1));
    if (!occ) return fail(BWL_ERR_ARG, "site is not a lattice site");
    a.x[w] = x; a.y[w] = y; a.z[w] = z;
  }
  Pinned pin;
  if (!pin.take(2 * sizeof(double), c->stream)) return fail(BWL_ERR_NOMEM, "pinned memory allocation failed");
  a.compact = c->d_compact;
  a.vex = c->d_vex;
  a.out = (double *)pin.p;
  HIP_OK(launch_site_energy(a, c->stream));
  HIP_OK(hipStreamSynchronize(c->stream));
  pin.settled();
  memcpy(out2, pin.p, 2 * sizeof(double));
  return BWL_OK;
}

int bwl_site_energy(bwl_ctx *c, int32_t site_b, int32_t site_i, int32_t site_j, int32_t site_k,
                    double *energy) {
  if (!energy) return fail(BWL_ERR_ARG, "null energy");
  int32_t s[4] = {site_b, site_i, site_j, site_k};
  double o[2];
  int rc = site_pair(c, s, s, o);
  if (rc) return rc;
  *energy = o[0];
  return BWL_OK;
}

int bwl_pair_energy(bwl_ctx *c, const int32_t *site1, const int32_t *site2, double *energy) {
  if (!energy || !site1 || !site2) return fail(BWL_ERR_ARG, "null argument");
  double o[2];
  int rc = site_pair(c, site1, site2, o);
  if (rc) return rc;
  *energy = o[1];
  return BWL_OK;
}

int bwl_genrand_seed(bwl_ctx *c, uint32_t seed) {
  if (!c) return fail(BWL_ERR_ARG, "null context");
  c->mt.seed(seed);
  return BWL_OK;
}

int bwl_genrand_get_state(bwl_ctx *c, uint32_t *mt, int32_t *mti) {
  if (!c || !mt || !mti) return fail(BWL_ERR_ARG, "null argument");
  memcpy(mt, c->mt.mt, sizeof(c->mt.mt));
  *mti = c->mt.mti;
  return BWL_OK;
}

int bwl_genrand_set_state(bwl_ctx *c, const uint32_t *mt, int32_t mti) {
  if (!c || !mt) return fail(BWL_ERR_ARG, "null argument");
  if (mti < 0 || mti > 625) return fail(BWL_ERR_ARG, "mti out of range");
  memcpy(c->mt.mt, mt, sizeof(c->mt.mt));
  c->mt.mti = mti;
  return BWL_OK;
}

// A lattice site of the context given as (b, i, j, k), 1-based.
static int check_site(const Geo &g, const int32_t *s) {
  if (s[0] != 1) return fail(BWL_ERR_ARG, "basis index must be 1");
  const int x = s[1] - 1, y = s[2] - 1, z = s[3] - 1;
  if (x < 0 || y < 0 || z < 0 || x >= g.m[0] || y >= g.m[1] || z >= g.m[2])
    return fail(BWL_ERR_ARG, "site index out of range");
  const bool occ = g.lattice == BWL_FCC ? (((x + y + z) & 1) == 0)
                                        : ((x & 1) == (y & 1) && (y & 1) == (z & 1));
  if (!occ) return fail(BWL_ERR_ARG, "site is not a lattice site");
  return BWL_OK;
}

// Proposal draws on the device from the context's MT19937 stream: the
// state goes up, the draws are made by one wavefront, the state comes back.
static int draw_sites(bwl_ctx *c, int mode, int32_t n, const int32_t *site, int32_t *out) {
  int rc = check_ctx(c, false);
  if (rc) return rc;
  if (!out || n < 1 || n > (1 << 20)) return fail(BWL_ERR_ARG, "bad count or null output");
  if (mode == 1) {
    if (!site) return fail(BWL_ERR_ARG, "null site");
    rc = check_site(c->g, site);
    if (rc) return rc;
  }
  if (c->mt.mti == 625) c->mt.seed(5489u);
  const size_t vals = (size_t)n * (mode >= 2 ? 8 : 4);
  rc = ensure_scratch(c, 624 * 4 + 64 + sizeof(int32_t) * vals);
  if (rc) return rc;
  char *base = (char *)c->d_scratch;
  DrawArgs a;
  memset(&a, 0, sizeof(a));
  a.g = c->g;
  a.mt = (uint32_t *)base;
  a.mt_index = (int32_t *)(base + 624 * 4);
  a.out = (int32_t *)(base + 624 * 4 + 64);
  a.mode = mode;
  a.n = mode == 1 ? 1 : n;
  if (site) memcpy(a.site, site, sizeof(a.site));
  int32_t mti = c->mt.mti;
  HIP_OK(hipMemcpyAsync(a.mt, c->mt.mt, 624 * 4, hipMemcpyHostToDevice, c->stream));
  HIP_OK(hipMemcpyAsync(a.mt_index, &mti, 4, hipMemcpyHostToDevice, c->stream));
  HIP_OK(launch_draw_sites(a, c->stream));
  HIP_OK(hipMemcpyAsync(c->mt.mt, a.mt, 624 * 4, hipMemcpyDeviceToHost, c->stream));
  HIP_OK(hipMemcpyAsync(&mti, a.mt_index, 4, hipMemcpyDeviceToHost, c->stream));
  HIP_OK(hipMemcpyAsync(out, a.out, sizeof(int32_t) * vals, hipMemcpyDeviceToHost, c->stream));
  HIP_OK(hipStreamSynchronize(c->stream));
  c->mt.mti = mti;
  return BWL_OK;
}

int bwl_random_site(bwl_ctx *c, int32_t n, int32_t *sites) {
  return draw_sites(c, 0, n, nullptr, sites);
}

int bwl_random_nbr(bwl_ctx *c, const int32_t *site, int32_t *nbr) {
  return draw_sites(c, 1, 1, site, nbr);
}

int bwl_select_sites(bwl_ctx *c, int32_t nbr_swap, int32_t n, int32_t *sites) {
  return draw_sites(c, nbr_swap ? 3 : 2, n, nullptr, sites);
}

int bwl_initial_setup(bwl_ctx *c, const int64_t *species_numbers, const double *concentrations) {
  int rc = check_ctx(c, false);
  if (rc) return rc;
  std::vector<int8_t> cfg((size_t)c->g.m[0] * c->g.m[1] * c->g.m[2]);
  rc = initial_setup_host(c->g, species_numbers, concentrations, c->mt, cfg.data(), g_err);
  if (rc) return rc;
  return bwl_set_config(c, cfg.data());
}

int bwl_mc_steps(bwl_ctx *c, double beta, int32_t nbr_swap, int64_t n_trials, int64_t sample_every,
                 double *energies, int64_t *accepted) {
  int rc = check_ctx(c, true);
  if (rc) return rc;
  if (n_trials < 0) return fail(BWL_ERR_ARG, "negative trial count");
  if (energies && sample_every <= 0) return fail(BWL_ERR_ARG, "sample_every must be positive");
  const Geo &g = c->g;
  SeqPick pick;
  pick.add(g, seq_lds_bytes(g), seq_spec_lds_bytes(g));
  const int limit = lds_limit();
  if (pick.lds > (size_t)limit) return fail(BWL_ERR_UNSUPPORTED, "lattice does not fit in LDS");
  pick.settle(limit);
  if (2 * g.R > 64) return fail(BWL_ERR_UNSUPPORTED, "too many shells");
  // the MT state must be initialised (mti == 625 means "seed with 5489")
  if (c->mt.mti == 625) c->mt.seed(5489u);
  const long long n_samples = energies ? n_trials / sample_every : 0;
  // the stream and the results lie in pinned memory, but for long series of
  // energies
  const size_t e_bytes = sizeof(double) * (size_t)n_samples;
  const bool e_pinned = e_bytes <= kPinnedSeries;
  Pinned pin;
  if (!pin.take(624 * 4 + 64 + (e_pinned ? e_bytes : 0), c->stream))
    return fail(BWL_ERR_NOMEM, "pinned memory allocation failed");
  if (!e_pinned) {
    rc = ensure_scratch(c, e_bytes);
    if (rc) return rc;
  }
  SeqArgs a;
  a.g = g;
  a.compact = c->d_compact;
  a.off = c->d_off;
  a.vex = c->d_vex;
  a.mt = (uint32_t *)pin.p;
  a.mt_index = (int32_t *)(pin.p + 624 * 4);
  a.accepted = (long long *)(pin.p + 624 * 4 + 16);
  a.energies = !n_samples ? nullptr : e_pinned ? (double *)(pin.p + 624 * 4 + 64) : (double *)c->d_scratch;
  a.beta = beta;
  a.nbr_swap = nbr_swap ? 1 : 0;
  a.n_trials = n_trials;
  a.sample_every = energies ? sample_every : 0;
  memcpy(a.mt, c->mt.mt, 624 * 4);
  *a.mt_index = c->mt.mti;
  const CuUse use(c->device, 1);
  HIP_OK(launch_metro_seq(a, pick, c->stream));
  if (n_samples && !e_pinned)
    HIP_OK(hipMemcpyAsync(energies, a.energies, e_bytes, hipMemcpyDeviceToHost, c->stream));
  HIP_OK(hipStreamSynchronize(c->stream));
  pin.settled();
  memcpy(c->mt.mt, a.mt, 624 * 4);
  c->mt.mti = *a.mt_index;
  if (n_samples && e_pinned) memcpy(energies, a.energies, e_bytes);
  if (accepted) *accepted = *a.accepted;
  return BWL_OK;
}

int bwl_mc_steps_batch(int32_t n, bwl_ctx *const *ctxs, const double *beta, int32_t nbr_swap,
                       int64_t n_trials, int64_t sample_every, double *const *energies,
                       int64_t *accepted, double *kernel_ms) {
  if (n < 1 || !ctxs || !beta) return fail(BWL_ERR_ARG, "null argument or empty batch");
  if (n_trials < 0) return fail(BWL_ERR_ARG, "negative trial count");
  if (energies && sample_every <= 0) return fail(BWL_ERR_ARG, "sample_every must be positive");
  SeqPick pick;
  for (int i = 0; i < n; ++i) {
    bwl_ctx *c = ctxs[i];
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if (c->device != ctxs[0]->device) return fail(BWL_ERR_ARG, "all chains of a batch must be on one device");
    if (2 * c->g.R > 64) return fail(BWL_ERR_UNSUPPORTED, "too many shells");
    pick.add(c->g, seq_lds_bytes(c->g), seq_spec_lds_bytes(c->g));
  }
  const int limit = lds_limit();
  if (pick.lds > (size_t)limit) return fail(BWL_ERR_UNSUPPORTED, "lattice does not fit in LDS");
  pick.settle(limit);
  HIP_OK(hipSetDevice(ctxs[0]->device));
  // per chain: MT state, index, accepted count, sampled energies
  const long long n_samples = energies ? n_trials / sample_every : 0;
  const size_t stride = ((624 * 4 + 64 + sizeof(double) * (size_t)n_samples) + 255) & ~(size_t)255;
  const size_t args_bytes = (sizeof(SeqArgs) * (size_t)n + 255) & ~(size_t)255, io_bytes = stride * (size_t)n;
  hipStream_t s = ctxs[0]->stream;
  // the chains' arguments on the device; their streams and results in pinned
  // memory unless there are many
  const bool io_pinned = io_bytes <= kPinnedSeries;
  Pinned pin;
  if (!pin.take(args_bytes + (io_pinned ? io_bytes : 0), s)) return fail(BWL_ERR_NOMEM, "pinned memory allocation failed");
  int rc_s = ensure_scratch(ctxs[0], args_bytes + (io_pinned ? 0 : io_bytes));
  if (rc_s) return rc_s;
  char *base = (char *)ctxs[0]->d_scratch;
  std::vector<char> far(io_pinned ? 0 : io_bytes);
  char *const host = io_pinned ? pin.p + args_bytes : far.data();  // the streams and results here,
  char *const io = io_pinned ? host : base + args_bytes;           // and where the kernel finds them
  SeqArgs *args = (SeqArgs *)pin.p;
  for (int i = 0; i < n; ++i) {
    bwl_ctx *c = ctxs[i];
    if (c->mt.mti == 625) c->mt.seed(5489u);
    if (i > 0) HIP_OK(hipStreamSynchronize(c->stream));  // the chain's own earlier work
    char *h = host + stride * (size_t)i;
    memcpy(h, c->mt.mt, 624 * 4);
    memcpy(h + 624 * 4, &c->mt.mti, 4);
    char *d = io + stride * (size_t)i;
    SeqArgs &a = args[(size_t)i];
    a.g = c->g;
    a.compact = c->d_compact;
    a.off = c->d_off;
    a.vex = c->d_vex;
    a.mt = (uint32_t *)d;
    a.mt_index = (int32_t *)(d + 624 * 4);
    a.accepted = (long long *)(d + 624 * 4 + 16);
    a.energies = n_samples ? (double *)(d + 624 * 4 + 64) : nullptr;
    a.beta = beta[i];
    a.nbr_swap = nbr_swap ? 1 : 0;
    a.n_trials = n_trials;
    a.sample_every = energies ? sample_every : 0;
  }
  HIP_OK(hipMemcpyAsync(base, args, sizeof(SeqArgs) * (size_t)n, hipMemcpyHostToDevice, s));
  if (!io_pinned) HIP_OK(hipMemcpyAsync(io, host, io_bytes, hipMemcpyHostToDevice, s));
  const CuUse use(ctxs[0]->device, n);
  HIP_OK(hipEventRecord(ctxs[0]->ev0, s));
  HIP_OK(launch_metro_seq_batch((const SeqArgs *)base, n, pick, s));
  HIP_OK(hipEventRecord(ctxs[0]->ev1, s));
  if (!io_pinned) HIP_OK(hipMemcpyAsync(host, io, io_bytes, hipMemcpyDeviceToHost, s));
  HIP_OK(hipStreamSynchronize(s));
  pin.settled();
  float ms = 0.f;
  (void)hipEventElapsedTime(&ms, ctxs[0]->ev0, ctxs[0]->ev1);
  if (kernel_ms) *kernel_ms = ms;
  for (int i = 0; i < n; ++i) {
    bwl_ctx *c = ctxs[i];
    const char *h = host + stride * (size_t)i;
    memcpy(c->mt.mt, h, 624 * 4);
    memcpy(&c->mt.mti, h + 624 * 4, 4);
    long long acc = 0;
    memcpy(&acc, h + 624 * 4 + 16, sizeof(acc));
    if (accepted) accepted[i] = acc;
    if (n_samples && energies[i]) memcpy(energies[i], h + 624 * 4 + 64, sizeof(double) * n_samples);
  }
  return BWL_OK;
}

int bwl_set_layout(bwl_ctx *c, int32_t layout) {
  if (!c) return fail(BWL_ERR_ARG, "null context");
  if (layout < BWL_LAYOUT_AUTO || layout > BWL_LAYOUT_FIXED) return fail(BWL_ERR_ARG, "unknown layout");
  c->layout = layout;
  return BWL_OK;
}

int bwl_set_threads(bwl_ctx *c, int32_t threads) {
  if (!c) return fail(BWL_ERR_ARG, "null context");
  if (threads < 0 || threads > kMaxNatThreads || threads % 64 != 0)
    return fail(BWL_ERR_ARG, "threads per chain must be 0 (by rule) or a multiple of 64 up to 1024");
  c->threads = threads;
  return BWL_OK;
}

int bwl_layout_info(bwl_ctx *c, int32_t layout, int32_t *threads, int64_t *lds_bytes) {
  if (!c) return fail(BWL_ERR_ARG, "null context");
  if (layout < BWL_LAYOUT_AUTO || layout > BWL_LAYOUT_FIXED) return fail(BWL_ERR_ARG, "unknown layout");
  ParPlan plan;
  NatGeo nat;
  const void *fn = nullptr;
  int t = 0;
  size_t lds = 0;
  int rc = anneal_kernel(c->g, plan, nat, fn, t, lds, nullptr, layout);
  if (rc) return rc;
  if (threads) *threads = t;
  if (lds_bytes) *lds_bytes = (int64_t)lds;
  return BWL_OK;
}

int bwl_layouts(bwl_ctx *c, int32_t *mask) {
  if (!c || !mask) return fail(BWL_ERR_ARG, "null argument");
  *mask = 0;
  for (int layout = BWL_LAYOUT_COMPACT; layout <= BWL_LAYOUT_FIXED; ++layout)
    if (bwl_layout_info(c, layout, nullptr, nullptr) == BWL_OK) *mask |= 1 << (layout - 1);
  bwl::g_err.clear();
  return BWL_OK;
}

int bwl_metropolis_anneal(bwl_ctx *c, const bwl_anneal_params *p, double *energies_of_T,
                          double *C_of_T, double *acceptance_of_T, bwl_run_stats *stats) {
  if (!p) return fail(BWL_ERR_ARG, "null argument");
  bwl_anneal_params q = *p;
  q.asro_every = 0;
  bwl_ctx *cs[1] = {c};
  double *e[1] = {energies_of_T}, *cv[1] = {C_of_T}, *ac[1] = {acceptance_of_T};
  return bwl_metropolis_anneal_batch(1, cs, &q, e, cv, ac, stats, nullptr);
}

int bwl_metropolis_anneal_rho(bwl_ctx *c, const bwl_anneal_params *p, double *energies_of_T,
                              double *C_of_T, double *acceptance_of_T, double *rho_of_T,
                              bwl_run_stats *stats) {
  if (!c || !p || !energies_of_T || !C_of_T || !acceptance_of_T || !rho_of_T)
    return fail(BWL_ERR_ARG, "null argument");
  if (p->asro_every < 1) return fail(BWL_ERR_ARG, "asro_every must be positive");
  bwl_ctx *cs[1] = {c};
  double *e[1] = {energies_of_T}, *cv[1] = {C_of_T}, *ac[1] = {acceptance_of_T}, *rh[1] = {rho_of_T};
  return anneal_run(1, cs, p, e, cv, ac, stats, nullptr, rh);
}

}  // extern "C"

namespace bwl {

size_t ctx_device_bytes(const bwl_lattice_desc &d) {
  Geo g;
  std::vector<int32_t> off;
  std::string err;
  if (make_geo(d, g, off, err)) return 0;
  const size_t ref = (size_t)g.m[0] * g.m[1] * g.m[2];
  auto a = [](size_t v) { return (v + 255) & ~(size_t)255; };
  return a((size_t)g.compact_bytes) + a(ref) + a(sizeof(int32_t) * off.size()) +
         a(sizeof(double) * (size_t)g.S * g.S * g.R);
}

size_t ctx_tables_bytes(const Geo &g) {
  auto a = [](size_t v) { return (v + 255) & ~(size_t)255; };
  return a(sizeof(int32_t) * (size_t)g.nsub * g.z) + sizeof(double) * (size_t)g.S * g.S * g.R;
}

int ctx_create_borrowed(const bwl_lattice_desc &d, const double *v_ex, char *mem, size_t bytes,
                        hipStream_t stream, char *tables, bwl_ctx **out) {
  *out = nullptr;
  bwl_ctx *c = new bwl_ctx();
  c->desc = d;
  int rc = make_geo(d, c->g, c->off, g_err);
  if (rc) {
    delete c;
    return rc;
  }
  if (bytes < ctx_device_bytes(d)) {
    delete c;
    return fail(BWL_ERR_ARG, "borrowed block too small for the lattice");
  }
  const Geo &g = c->g;
  c->vex.assign(v_ex, v_ex + (size_t)g.S * g.S * g.R);
  c->borrowed = true;
  if (hipGetDevice(&c->device) != hipSuccess) c->device = 0;
  auto a = [](size_t v) { return (v + 255) & ~(size_t)255; };
  char *q = mem;
  c->d_compact = (int8_t *)q;
  q += a((size_t)g.compact_bytes);
  c->d_ref = (int8_t *)q;
  q += a((size_t)g.m[0] * g.m[1] * g.m[2]);
  c->d_off = (int32_t *)q;
  q += a(sizeof(int32_t) * c->off.size());
  c->d_vex = (double *)q;
  c->stream = stream;
  // the offset table and V_ex, which follow each other in the block
  memcpy(tables, c->off.data(), sizeof(int32_t) * c->off.size());
  memcpy(tables + ((char *)c->d_vex - (char *)c->d_off), c->vex.data(), sizeof(double) * c->vex.size());
  const bool ok = hipEventCreate(&c->ev0) == hipSuccess && hipEventCreate(&c->ev1) == hipSuccess &&
                  hipMemcpyAsync(c->d_off, tables, ctx_tables_bytes(g), hipMemcpyHostToDevice, stream) == hipSuccess;
  if (!ok) {
    bwl_destroy(c);
    return fail(BWL_ERR_DEVICE, "borrowed context set-up failed");
  }
  c->mt.seed(110179u);
  *out = c;
  return BWL_OK;
}

}  // namespace bwl

// ----------------------------------------------------------------------
// Batched anneal in three steps (used by bwl_metropolis_anneal_batch and by
// the request server): plan on the host, upload + launch on streams, collect
// after completion.
// ----------------------------------------------------------------------
namespace bwl {

int anneal_kernel(const Geo &g, ParPlan &plan, NatGeo &nat, const void *&fn, int &threads,
                  size_t &lds, bool *natural, int layout, int threads_req) {
  const int lim = lds_limit();
  int rc = plan_parallel(g, plan, g_err);
  if (rc) return rc;
  int max_pairs = 0;
  for (const RoundVar &v : plan.vars) max_pairs = v.n2 > max_pairs ? v.n2 : max_pairs;
  // fewest passes over a round's pairs, then the fewest threads for that;
  // with two or more passes on the 1024-thread kernels, all their threads:
  // the extra wavefronts hide the gathers' latency (bcc 32^3 anneal 2.68 ->
  // 2.43 s, 256-chain batch 165 -> 157 ms)
  auto block_size = [&](int cap) {
    const int passes = (max_pairs + cap - 1) / cap;
    int t = (((max_pairs + passes - 1) / passes + 63) / 64) * 64;
    if (cap == kMaxNatThreads && passes > 1) t = cap;
    if (t > cap) t = cap;
    return t < 64 ? 64 : t;
  };
  // Layouts in order of preference: the fixed-pitch natural layout (one
  // kernel with compile-time offsets for all sizes of a lattice and shell
  // count), unless the shape has a kernel of its own; the natural layout
  // with this size's own pitch; the per-sublattice layout.  Packed counts
  // (par_count_words): 32-bit words with 8-bit fields up to 4 species,
  // 6-bit fields for 5, else 64-bit words.
  NatGeo per{}, fix{};
  const bool nat_ok = make_nat(g, per);
  const bool fix_ok = nat_ok && !par_specialised(g) && make_nat_fixed(g, fix) &&
                      par_fixed_kernel(g.lattice, g.R, par_count_words(g, true)) != nullptr;
  const int modes[3] = {fix_ok ? 2 : -1, nat_ok ? 1 : -1, 0};
  // BWL_LAYOUT_COMPACT / _NATURAL / _FIXED are modes 0 / 1 / 2
  for (int mode : modes) {
    if (mode < 0 || (layout != 0 && mode != layout - 1)) continue;
    const bool use_nat = mode != 0, fixed = mode == 2;
    const NatGeo *ng = fixed ? &fix : (use_nat ? &per : nullptr);
    const int cap = par_max_threads(g, use_nat, fixed);
    if (threads_req > cap) continue;
    threads = threads_req > 0 ? threads_req : block_size(cap);
    lds = par_lds_bytes(g, ng, threads);
    if (lds > (size_t)lim) continue;
    if (ng) nat = *ng;
    else memset(&nat, 0, sizeof(nat));
    fn = par_kernel_for(g, use_nat, fixed);
    if (!fn) return fail(BWL_ERR_UNSUPPORTED, "no kernel for this lattice");
    if (natural) *natural = use_nat;
    return BWL_OK;
  }
  if (threads_req > 0)
    return fail(BWL_ERR_UNSUPPORTED, "no layout of this lattice runs the requested threads per chain");
  if (layout != 0) return fail(BWL_ERR_UNSUPPORTED, "the requested layout is not available for this lattice");
  return fail(BWL_ERR_UNSUPPORTED, "lattice does not fit in LDS");
}

// Estimated time of a chain's rounds (us), undivided and divided: fitted to
// runs of 19 shapes with 1-24 chunks of 64 pairs a round and 8-54 gathers a
// site (z); a divided round takes 2.2-2.6 us whatever its size.
static double undivided_us(const AnnealPlan::Item &it) {
  return it.rounds * (0.7 + 0.135 * sqrt((double)it.chunks * (double)it.a.g.z));
}
double anneal_estimate_us(const Geo &g, const ParPlan &plan, const bwl_anneal_params &p) {
  int pairs = 1;
  for (const RoundVar &v : plan.vars) pairs = std::max(pairs, (int)v.n2);
  const double rounds = (double)p.T_steps * ((double)p.n_sweeps + p.burn_in_sweeps) * g.n_atoms / pairs;
  return rounds * (0.7 + 0.135 * sqrt((double)((pairs + 63) / 64) * (double)g.z));
}
static double divided_us(const AnnealPlan::Item &it) { return it.rounds * 2.4; }

// Divides the longest chains over workgroups (a.parts, lane of their items)
// where the device would end the whole batch sooner than such a chain alone.
//
// A chain is worth dividing from chunks * z = 192 on: 1.10x at 252 (fcc 18^3, 3
// shells), 1.19x at 196 (bcc 24^3, 2), 1.6x at 588 (fcc 24^3, 3), 2.0x at 1200
// (bcc 32^3, 4), against 0.99x at 144 (fcc 20^3, 2) and 1.00x at 150 (bcc 16^3,
// 4).  Two kinds of chains from there on are not: those that k_metro_alone
// takes whole (fcc 15^3 to 17^3 and bcc 18^3, 4 shells, in 2 parts: 0.77-0.97x,
// 1.01x at best), and, with 64-bit count words, whose pairs cost more, chains of
// less than 8 chunks unless z makes up for it (fcc 18^3, 3 shells, 0.95x; bcc
// 19^3, 4 shells, 0.89x; fcc 20^3, 3 shells, 1.07x; fcc 18^3, 4 shells, 1.26x).
// One wavefront per SIMD and part (4 half rows) is best where the CUs are there
// (bcc 32^3: 16 parts 5.1 ms, 8 parts 5.7; fcc 24^3: 7 parts 7.4, 4 parts 7.7),
// else two.
//
// With more than one shell that holds from the first sweep on, since the
// recounts of the energy are divided too.  With one shell they are short, and
// 16 wavefronts stage the lattice in 40 to 60 us less than the 8 of a part: fcc
// 16^3 196 us for one sweep (divided 223) and 596 for twelve (533), bcc 18^3
// 183 (211) and 447 (373), so such a chain has to be some 6 sweeps long.
//
// The parts of a chain go to one XCD (lane), which has n_cu / 8 CUs: as many
// as this process's calls in flight (CuUse, SplitShare) and the call's other
// chains leave free, but half an XCD in any case: the parts are launched
// before those other chains (200 fcc 16^3 and one bcc 32^3, 16 parts: 20.0 ms,
// undivided 30.5).  Parts and undivided chains together have a CU each: a
// batch of 256 uneven chains, eight of them fcc 24^3, took 184 ms with those
// eight divided (smaller chains then share CUs with parts that all the others
// wait for) and 144 with none.  Equally free XCDs are taken from one on that
// differs by process, since processes that share a device do not see each
// other's.
static void divide_chains(AnnealPlan &P, const SplitLanes &free_parts, int n_cu, int lim) {
  const int n = (int)P.items.size();
  const int cap = std::max(n_cu / 8 - (n + 7) / 8, n_cu / 16), first = (int)((unsigned)getpid() % 8u);
  int lanes[8], blocks = n;
  bool any = false;
  for (int x = 0; x < 8; ++x) {
    lanes[x] = std::min(free_parts.parts[x], cap);
    any = any || lanes[x] >= 2;
  }
  if (!any) return;
  double load = 0.0;  // CU time
  auto share = [&](const AnnealPlan::Item &it) {  // of a CU, undivided
    return std::min(1.0, std::max((double)it.lds / (double)lim, (double)it.threads / (double)kMaxNatThreads));
  };
  std::vector<AnnealPlan::Item *> by_time;
  for (AnnealPlan::Item &it : P.items) {
    load += undivided_us(it) * share(it);
    by_time.push_back(&it);
  }
  std::stable_sort(by_time.begin(), by_time.end(), [](const AnnealPlan::Item *x, const AnnealPlan::Item *y) {
    return undivided_us(*x) > undivided_us(*y);
  });
  auto divide = [&](AnnealPlan::Item &it) {
    if (!it.split_fn || it.chunks * it.a.g.z < 192 || par_split_lds_bytes(it.a.g, it.a.nat) > (size_t)lim) return false;
    if (par_alone_kernel(it.a.g, it.split_fixed) && par_alone_threads(it.threads, it.passes) > 0) return false;
    if (par_count_words(it.a.g, true) == 2 && it.chunks < 8 && it.chunks * it.a.g.z < 320) return false;
    if (it.a.g.R == 1 && undivided_us(it) < 160.0) return false;
    const int rows = it.threads / 64;
    for (int units = 4; units <= 8; units += 4) {
      const int rows_each = std::max(1, units / (2 * it.passes));
      const int parts = (rows + rows_each - 1) / rows_each;
      if (!par_split_fits(it.a.nat, it.threads, parts, it.passes)) continue;
      const double load_then = load + parts * divided_us(it) - undivided_us(it) * share(it);
      int to = first;
      for (int x = 1; x < 8; ++x)
        if (lanes[(first + x) % 8] > lanes[to]) to = (first + x) % 8;
      if (parts > lanes[to] || blocks + parts - 1 > n_cu || load_then > n_cu * undivided_us(it)) continue;
      blocks += parts - 1;
      load = load_then;
      lanes[to] -= parts;
      it.a.parts = parts;
      it.lane = to;
      // CUs that other processes hold may keep some of the parts from
      // arriving; the others wait for a quarter of what the division saves,
      // 0.2 to 5 ms, then the chain runs undivided (bcc 32^3, 40 sweeps, while
      // another process's chains had 200 CUs: 11 to 18 ms, 1029 with 1 s of
      // patience)
      const double wait_us = std::min(5000.0, std::max(200.0, 0.25 * (undivided_us(it) - divided_us(it))));
      it.a.patience = (int32_t)(100.0 * wait_us);
      return true;
    }
    return false;
  };
  for (AnnealPlan::Item *it : by_time)
    if (!divide(*it)) break;
  // a division that leaves the batch waiting for chains as long is undone
  double longest = 0.0;
  for (const AnnealPlan::Item &it : P.items)
    longest = std::max(longest, it.a.parts > 1 ? divided_us(it) : undivided_us(it));
  const bool gains = longest < 0.95 * undivided_us(*by_time[0]);
  for (AnnealPlan::Item &it : P.items)
    if (!gains || undivided_us(it) <= longest) it.a.parts = 1;
}

int anneal_plan(int n, bwl_ctx *const *ctxs, const bwl_anneal_params *params, AnnealPlan &P,
                const SplitLanes *split) {
  P.items.assign((size_t)n, AnnealPlan::Item());
  P.groups.clear();
  P.split = SplitLanes();
  size_t total = 0;
  const int lim = lds_limit();
  for (int i = 0; i < n; ++i) {
    bwl_ctx *c = ctxs[i];
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if (i > 0 && c->device != ctxs[0]->device)
      return fail(BWL_ERR_ARG, "all chains of a batch must be on one device");
    const bwl_anneal_params *p = &params[i];
    if (p->T_steps < 1 || p->n_sweeps < 1 || p->burn_in_sweeps < 0)
      return fail(BWL_ERR_ARG, "T_steps and n_sweeps must be positive");
    AnnealPlan::Item &it = P.items[(size_t)i];
    it.idx = i;
    const Geo &g = c->g;
    NatGeo nat;
    int threads = 0;
    size_t lds = 0;
    bool natural = false;
    rc = anneal_kernel(g, it.plan, nat, it.fn, threads, lds, &natural, c->layout, c->threads);
    if (rc) return rc;
    if (p->asro_every < 0 || p->asro_every > p->n_sweeps)
      return fail(BWL_ERR_ARG, "asro_every must be in 0..n_sweeps");
    if (p->asro_every > 0) {
      if (!natural)
        return fail(BWL_ERR_UNSUPPORTED,
                    "radial densities in the anneal need a cubic supercell held in lattice coordinates");
      const int w = std::min(std::min(g.n[0], g.n[1]), std::min(g.n[2], 5));
      if (g.rcut > w)
        return fail(BWL_ERR_UNSUPPORTED,
                    "an interaction shell reaches outside the radial-density window (supercell too small)");
    }
    it.threads = threads;
    it.lds = lds;
    it.natural = natural;
    int max_pairs = 0;
    for (const RoundVar &v : it.plan.vars) max_pairs = std::max(max_pairs, (int)v.n2);
    it.chunks = (max_pairs + 63) / 64;
    it.passes = (max_pairs + threads - 1) / threads;
    it.rounds = (double)p->T_steps * (double)(p->n_sweeps + p->burn_in_sweeps) * (double)g.n_atoms / (double)max_pairs;
    // (a layout other than the rule's, where the caller asked for one, has
    // run-time neighbour offsets or none in lattice coordinates)
    it.split_fixed = natural && it.fn == par_fixed_kernel(g.lattice, g.R, par_count_words(g, true));
    if (natural) it.split_fn = par_split_kernel(g, it.split_fixed);
    if (natural && it.split_fn && it.fn != par_fixed_kernel(g.lattice, g.R, par_count_words(g, true)) && !par_specialised(g))
      it.split_fn = nullptr;
    ParArgs &a = it.a;
    memset(&a, 0, sizeof(a));
    a.g = g;
    a.nat = nat;
    a.compact = c->d_compact;
    a.off = c->d_off;
    a.vex = c->d_vex;
    a.stride = it.plan.stride;
    a.L = it.plan.L;
    for (int k = 0; k < 3; ++k) {
      a.K[k] = it.plan.K[k];
      a.n_units[k] = it.plan.n_units[k];
      for (int u = 0; u < 16; ++u) a.units[k][u] = it.plan.units[k][u];
    }
    a.n_var = (int32_t)it.plan.vars.size();
    for (size_t k = 0; k < it.plan.vars.size(); ++k) a.var[k] = it.plan.vars[k];
    a.fast_halo = it.plan.fast_halo ? 1 : 0;
    a.min_trials_per_sweep = g.n_atoms;
    a.threads = threads;
    a.T0 = p->T;
    a.dT = p->delta_T;
    a.T_steps = p->T_steps;
    a.n_sweeps = p->n_sweeps;
    a.burn_sweeps = p->burn_in_sweeps;
    a.seed_lo = (uint32_t)p->seed;
    a.seed_hi = (uint32_t)(p->seed >> 32);
    a.chain_id = 0;  // the stream depends on the seed and position only, not on the batch
    a.phase0 = c->phase;
    a.e_trace = nullptr;
    a.asro_every = p->asro_every;
    a.rho_of_T = nullptr;
    it.T = (size_t)p->T_steps;
    it.off_out = total;
    total += 256 * ((5 * it.T * sizeof(double) + 255) / 256);
    it.off_cnt = total;
    total += 256;
    it.rho_n = p->asro_every > 0 ? (size_t)g.S * g.S * (g.R + 1) * it.T : 0;
    it.off_rho = total;
    total += 256 * ((it.rho_n * sizeof(double) + 255) / 256);
    it.work = (double)g.n_atoms * (double)p->T_steps * (double)(p->n_sweeps + p->burn_in_sweeps);
    a.parts = 1;
    a.passes = it.passes;
  }
  int n_cu = 0;
  if (hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, ctxs[0]->device) != hipSuccess) n_cu = 0;
  if (split) divide_chains(P, *split, n_cu, lim);
  // The scratch: the chains' results (copied down in one piece), what goes up
  // (counters among the results, then multipliers, arguments and maps, copied
  // in one piece), and the divided chains' mailboxes (cleared in one piece).
  P.out_bytes = total;
  for (AnnealPlan::Item &it : P.items) {
    it.off_muls = total;
    total += 256 * ((it.plan.muls.size() * 4 + 255) / 256);
  }
  int blocks = 0;
  for (AnnealPlan::Item &it : P.items) {
    if (it.a.parts > 1) {
      it.fn = it.split_fn;
      it.lds = par_split_lds_bytes(it.a.g, it.a.nat);
      P.split.parts[it.lane] += it.a.parts;
    }
    blocks += it.a.parts;
  }
  // group chains that run the same kernel (one launch each, the block size
  // of its largest member; each chain loops over its own pairs with the
  // threads it has), largest work first inside a group.  Few groups keep
  // every launch on its own hardware queue, so all groups run at once.
  std::vector<int> order((size_t)n);
  for (int i = 0; i < n; ++i) order[(size_t)i] = i;
  std::sort(order.begin(), order.end(), [&](int x, int y) {
    const AnnealPlan::Item &A = P.items[(size_t)x], &B = P.items[(size_t)y];
    // divided chains first: all of their workgroups have to be on the device
    if ((A.a.parts > 1) != (B.a.parts > 1)) return A.a.parts > 1;
    if (A.fn != B.fn) return A.fn < B.fn;
    return A.work > B.work;
  });
  for (int i : order) {
    const AnnealPlan::Item &it = P.items[(size_t)i];
    if (P.groups.empty() || P.groups.back().fn != it.fn)
      P.groups.push_back(AnnealPlan::Group{it.fn, it.threads, 0, {}, 0, it.a.parts > 1, {}, 0});
    AnnealPlan::Group &gr = P.groups.back();
    gr.members.push_back(i);
    if (it.threads > gr.threads) gr.threads = it.threads;
  }
  // Groups of small chains take the kernel with one site per lane, all of a
  // group's chains or none: no more launches than before (past 4
  // the launches of a batch wait for each other).  Up to 8 wavefronts of 32
  // pairs it was faster on every shape tried, from 1.54x (fcc 10^3, 4 shells: 1
  // row of pairs) to 1.03x (fcc 16^3, 4 shells: 4 rows).
  for (AnnealPlan::Group &gr : P.groups) {
    if (gr.split) continue;
    const void *fn = nullptr;
    int threads = 0;
    bool all = true;
    for (int i : gr.members) {
      const AnnealPlan::Item &it = P.items[(size_t)i];
      const Geo &g = it.a.g;
      const bool fixed = it.natural && it.fn == par_fixed_kernel(g.lattice, g.R, par_count_words(g, true));
      fn = fixed || (it.natural && par_specialised(g) && it.fn == par_kernel_for(g, true, false)) ? par_alone_kernel(g, fixed)
                                                                                                 : nullptr;
      const int t = par_alone_threads(it.threads, it.passes);
      all = all && fn && t > 0 && par_split_lds_bytes(g, it.a.nat) <= (size_t)lim;
      threads = std::max(threads, t);
    }
    if (!all) continue;
    gr.fn = fn;
    gr.threads = threads;
    for (int i : gr.members) {
      AnnealPlan::Item &it = P.items[(size_t)i];
      it.lds = par_split_lds_bytes(it.a.g, it.a.nat);
      it.fn = fn;
      it.alone = true;
    }
  }
  // LDS per launch: the largest member's need at the group's block size
  for (AnnealPlan::Group &gr : P.groups)
    for (int i : gr.members) {
      const AnnealPlan::Item &it = P.items[(size_t)i];
      const size_t need = it.lds + (gr.threads > it.threads && !gr.split ? sizeof(double) * (size_t)(gr.threads - it.threads) / 64 : 0);
      if (need > gr.lds) gr.lds = need;
    }
  // With no more chains than compute units, give every chain a CU of its
  // own: ask each block for more than half the LDS so no two share a CU
  // (the largest chains set the makespan; sharing a CU would halve them).
  const size_t exclusive = (size_t)lim / 2 + 1024;
  for (AnnealPlan::Group &gr : P.groups)
    if (gr.split || blocks <= n_cu)
      if (gr.lds < exclusive && exclusive <= (size_t)lim) gr.lds = exclusive;
  for (AnnealPlan::Group &gr : P.groups) {
    gr.off_args = total;
    total += 256 * ((sizeof(ParArgs) * gr.members.size() + 255) / 256);
    // Workgroups go to the 8 XCDs in turn, so block b lands on XCD b mod 8:
    // the parts of a chain take blocks of one residue.
    if (gr.split) {
      std::vector<int2> lane[8];
      for (size_t k = 0; k < gr.members.size(); ++k) {
        const AnnealPlan::Item &it = P.items[(size_t)gr.members[k]];
        for (int p = 0; p < it.a.parts; ++p) lane[it.lane].push_back(make_int2((int)k, p));
      }
      size_t rows = 0;
      for (const auto &l : lane) rows = std::max(rows, l.size());
      gr.map.assign(8 * rows, make_int2(-1, 0));
      for (size_t x = 0; x < 8; ++x)
        for (size_t k = 0; k < lane[x].size(); ++k) gr.map[8 * k + x] = lane[x][k];
      gr.off_map = total;
      total += 256 * ((sizeof(int2) * gr.map.size() + 255) / 256);
    }
  }
  P.up_bytes = total;
  for (AnnealPlan::Item &it : P.items) {
    it.mail_n = it.a.parts > 1 ? par_split_mail_words(it.a.g, it.threads, it.a.parts) : 0;
    it.off_mail = total;
    total += 256 * ((it.mail_n * sizeof(unsigned long long) + 255) / 256);
  }
  P.scratch_bytes = total;
  return BWL_OK;
}

int anneal_upload(AnnealPlan &P, char *base, hipStream_t s, char *image) {
  P.base = base;
  if (!image) {
    P.image.resize(P.up_bytes);
    image = P.image.data();
  }
  memset(image, 0, P.up_bytes);  // the counters start at 0
  for (AnnealPlan::Item &it : P.items) {
    it.a.muls = (const uint32_t *)(base + it.off_muls);
    it.a.energies_of_T = (double *)(base + it.off_out);
    it.a.C_of_T = it.a.energies_of_T + it.T;
    it.a.acc_of_T = it.a.C_of_T + it.T;
    it.a.e_drift = it.a.acc_of_T + it.T;
    it.a.counters = (long long *)(base + it.off_cnt);
    it.a.rho_of_T = it.rho_n ? (double *)(base + it.off_rho) : nullptr;
    it.a.mail = it.mail_n ? (unsigned long long *)(base + it.off_mail) : nullptr;
    memcpy(image + it.off_muls, it.plan.muls.data(), it.plan.muls.size() * 4);
  }
  for (AnnealPlan::Group &gr : P.groups) {
    char *to = image + gr.off_args;
    for (int i : gr.members) {
      memcpy(to, &P.items[(size_t)i].a, sizeof(ParArgs));
      to += sizeof(ParArgs);
    }
    if (gr.split) memcpy(image + gr.off_map, gr.map.data(), sizeof(int2) * gr.map.size());
  }
  HIP_OK(hipMemcpyAsync(base, image, P.up_bytes, hipMemcpyHostToDevice, s));
  if (P.scratch_bytes > P.up_bytes) HIP_OK(hipMemsetAsync(base + P.up_bytes, 0, P.scratch_bytes - P.up_bytes, s));
  return BWL_OK;
}

int anneal_launch(const AnnealPlan &P, const hipStream_t *streams) {
  for (size_t k = 0; k < P.groups.size(); ++k) {
    const AnnealPlan::Group &gr = P.groups[k];
    if (gr.split) {
      HIP_OK(launch_metro_split(gr.fn, (const ParArgs *)(P.base + gr.off_args), (const int2 *)(P.base + gr.off_map),
                                (int)gr.map.size(), gr.lds, streams[k]));
      continue;
    }
    HIP_OK(launch_metro_par_fn(gr.fn, (const ParArgs *)(P.base + gr.off_args),
                               (int)gr.members.size(), gr.lds, gr.threads, streams[k]));
  }
  return BWL_OK;
}

int anneal_collect(const AnnealPlan &P, bwl_ctx *const *ctxs, double *const *energies_of_T,
                   double *const *C_of_T, double *const *acceptance_of_T, bwl_run_stats *stats,
                   double kernel_ms, hipStream_t s, double *const *rho_of_T, std::vector<int> *again,
                   char *host) {
  const size_t n = P.items.size();
  std::vector<char> own;
  if (!host) {
    own.resize(P.out_bytes);
    host = own.data();
  }
  HIP_OK(hipMemcpyAsync(host, P.base, P.out_bytes, hipMemcpyDeviceToHost, s));
  HIP_OK(hipStreamSynchronize(s));
  std::vector<const double *> out(n);
  std::vector<long long> cnt(4 * n);
  for (size_t i = 0; i < n; ++i) {
    const AnnealPlan::Item &it = P.items[i];
    out[i] = (const double *)(host + it.off_out);
    memcpy(&cnt[4 * i], host + it.off_cnt, 4 * sizeof(long long));
  }
  for (size_t i = 0; i < n; ++i) {
    const size_t T = P.items[i].T;
    if (P.items[i].a.parts > 1 && cnt[4 * i + 3] == 0) {
      // a divided chain whose parts did not all get onto the device in time:
      // its configuration and stream are as they were
      if (!again) return fail(BWL_ERR_DEVICE, "a divided chain was given up");
      again->push_back((int)i);
      continue;
    }
    if (energies_of_T && energies_of_T[i]) memcpy(energies_of_T[i], out[i], T * sizeof(double));
    if (C_of_T && C_of_T[i]) memcpy(C_of_T[i], out[i] + T, T * sizeof(double));
    if (acceptance_of_T && acceptance_of_T[i]) memcpy(acceptance_of_T[i], out[i] + 2 * T, T * sizeof(double));
    if (rho_of_T && rho_of_T[i] && P.items[i].rho_n)
      memcpy(rho_of_T[i], host + P.items[i].off_rho, P.items[i].rho_n * sizeof(double));
    if (stats) {
      stats[i].trials = cnt[4 * i + 2];
      stats[i].accepted = cnt[4 * i + 1];
      stats[i].kernel_ms = kernel_ms;
      // largest difference between the carried energy and its recount over
      // the T steps, absolute (Ry) and relative to the recounted energy
      double da = 0.0, dr = 0.0;
      for (size_t t = 0; t < T; ++t) {
        const double d = fabs(out[i][3 * T + t]), e = fabs(out[i][4 * T + t]);
        da = d > da ? d : da;
        if (e > 0.0 && d / e > dr) dr = d / e;
      }
      stats[i].e_drift_abs = da;
      stats[i].e_drift_rel = dr;
    }
    ctxs[i]->phase = (unsigned long long)cnt[4 * i];
  }
  return BWL_OK;
}

}  // namespace bwl

extern "C" {

int bwl_metropolis_anneal_batch(int32_t n, bwl_ctx *const *ctxs, const bwl_anneal_params *params,
                                double *const *energies_of_T, double *const *C_of_T,
                                double *const *acceptance_of_T, bwl_run_stats *stats,
                                double *makespan_ms) {
  return anneal_run(n, ctxs, params, energies_of_T, C_of_T, acceptance_of_T, stats, makespan_ms, nullptr);
}

}  // extern "C"

namespace {

// The workgroups of divided chains on each of a device's XCDs, and the
// undivided ones on the whole device (they go to the XCDs in turn), over all
// calls in this process: the parts of a chain wait for each other, so together
// they must not outnumber the CUs.  A call takes what is free, keeps what its
// plan uses and gives it back when its launches have ended.
constexpr int kMaxSplitDevices = 64;
std::mutex g_split_mu;
SplitLanes g_split_used[kMaxSplitDevices];
long long g_undivided[kMaxSplitDevices];

struct SplitShare {
  int device = -1;
  SplitLanes held;
  SplitShare(int dev, int n_cu) {
    if (dev < 0 || dev >= kMaxSplitDevices) return;
    std::lock_guard<std::mutex> lock(g_split_mu);
    device = dev;
    for (int x = 0; x < 8; ++x) {
      held.parts[x] = (int)std::max(0LL, n_cu / 8 - g_split_used[dev].parts[x] - (g_undivided[dev] + 7) / 8);
      g_split_used[dev].parts[x] += held.parts[x];
    }
  }
  void keep(const SplitLanes &used) {
    if (device < 0) return;
    std::lock_guard<std::mutex> lock(g_split_mu);
    for (int x = 0; x < 8; ++x) g_split_used[device].parts[x] -= held.parts[x] - used.parts[x];
    held = used;
  }
  ~SplitShare() { keep(SplitLanes()); }
  SplitShare(const SplitShare &) = delete;
  SplitShare &operator=(const SplitShare &) = delete;
};

}  // namespace

namespace bwl {

CuUse::CuUse(int device, long long workgroups) {
  if (device < 0 || device >= kMaxSplitDevices || workgroups < 1) return;
  int n_cu = 0;
  if (hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return;
  device_ = device;
  n_ = (int)std::min(workgroups, (long long)n_cu);
  std::lock_guard<std::mutex> lock(g_split_mu);
  g_undivided[device_] += n_;
}

CuUse::~CuUse() {
  if (device_ < 0) return;
  std::lock_guard<std::mutex> lock(g_split_mu);
  g_undivided[device_] -= n_;
}

int anneal_run(int n, bwl_ctx *const *ctxs, const bwl_anneal_params *params, double *const *energies_of_T,
               double *const *C_of_T, double *const *acceptance_of_T, bwl_run_stats *stats, double *makespan_ms,
               double *const *rho_of_T, bool divide) {
  if (n < 1 || !ctxs || !params || !energies_of_T || !C_of_T || !acceptance_of_T)
    return fail(BWL_ERR_ARG, "null argument");
  for (int i = 0; i < n; ++i)
    if (!energies_of_T[i] || !C_of_T[i] || !acceptance_of_T[i]) return fail(BWL_ERR_ARG, "null output");
  AnnealPlan P;
  int n_cu = 0;
  if (divide && ctxs[0] &&
      hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, ctxs[0]->device) != hipSuccess)
    n_cu = 0;
  SplitShare share(ctxs[0] ? ctxs[0]->device : -1, n_cu);
  int rc = anneal_plan(n, ctxs, params, P, &share.held);
  if (rc) return rc;
  share.keep(P.split);
  bwl_ctx *c0 = ctxs[0];
  const CuUse rest(c0->device, std::count_if(P.items.begin(), P.items.end(),
                                             [](const AnnealPlan::Item &it) { return it.a.parts == 1; }));
  rc = ensure_scratch(c0, P.scratch_bytes);
  if (rc) return rc;
  char *const scratch = (char *)c0->d_scratch;
  // every group on its own stream so groups overlap on the device; the
  // context keeps the streams (as many as a batch has kernel variants)
  std::vector<hipStream_t> streams(1, c0->stream);
  for (size_t k = 1; k < P.groups.size(); ++k) {
    if (c0->side.size() < k) {
      hipStream_t s = nullptr;
      HIP_OK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
      c0->side.push_back(s);
    }
    streams.push_back(c0->side[k - 1]);
  }
  hipEvent_t ready = nullptr;
  HIP_OK(hipEventCreateWithFlags(&ready, hipEventDisableTiming));
  struct EventFreer {
    hipEvent_t e;
    ~EventFreer() { (void)hipEventDestroy(e); }
  } efree{ready};
  Pinned pin;
  const bool pinned = P.up_bytes <= kPinnedSeries;
  if (pinned && !pin.take(P.up_bytes, c0->stream)) return fail(BWL_ERR_NOMEM, "pinned memory allocation failed");
  // what is queued when the call ends early reads the scratch and the pinned
  // block and holds CUs: it is waited for before any of these is given back
  struct Waits {
    const std::vector<hipStream_t> *streams;
    ~Waits() {
      if (streams)
        for (hipStream_t s : *streams) (void)hipStreamSynchronize(s);
    }
  } waits{&streams};
  HIP_OK(hipEventRecord(c0->ev0, c0->stream));
  rc = anneal_upload(P, scratch, c0->stream, pin.p);
  if (rc) return rc;
  static const unsigned long long kGone = 1;
  for (int i = 0; i < n; ++i) {
    const AnnealPlan::Item &it = P.items[(size_t)i];
    ctxs[i]->ran[0] = it.a.parts;
    ctxs[i]->ran[1] = 0;
    ctxs[i]->ran[2] = it.alone ? 1 : 0;
    if (it.mail_n && ctxs[i]->give_up)  // (the mailbox ends with the word that gives a chain up)
      HIP_OK(hipMemcpyAsync(it.a.mail + it.mail_n - 1, &kGone, sizeof(kGone), hipMemcpyHostToDevice, c0->stream));
  }
  HIP_OK(hipEventRecord(ready, c0->stream));
  for (size_t k = 1; k < streams.size(); ++k) HIP_OK(hipStreamWaitEvent(streams[k], ready, 0));
  rc = anneal_launch(P, streams.data());
  if (rc) return rc;
  for (size_t k = 1; k < streams.size(); ++k) {
    hipEvent_t done = nullptr;
    HIP_OK(hipEventCreateWithFlags(&done, hipEventDisableTiming));
    HIP_OK(hipEventRecord(done, streams[k]));
    HIP_OK(hipStreamWaitEvent(c0->stream, done, 0));
    (void)hipEventDestroy(done);
  }
  HIP_OK(hipEventRecord(c0->ev1, c0->stream));
  HIP_OK(hipStreamSynchronize(c0->stream));
  waits.streams = nullptr;
  float ms = 0.f;
  (void)hipEventElapsedTime(&ms, c0->ev0, c0->ev1);
  if (makespan_ms) *makespan_ms = ms;
  std::vector<int> again;
  rc = anneal_collect(P, ctxs, energies_of_T, C_of_T, acceptance_of_T, stats, ms, c0->stream, rho_of_T, &again, pin.p);
  pin.settled();
  if (rc || again.empty()) return rc;
  // chains whose division was given up run undivided, with the same results
  std::vector<bwl_ctx *> cs;
  std::vector<bwl_anneal_params> ps;
  std::vector<double *> e, cv, ac, rh;
  for (int i : again) {
    cs.push_back(ctxs[i]);
    ps.push_back(params[i]);
    e.push_back(energies_of_T[i]);
    cv.push_back(C_of_T[i]);
    ac.push_back(acceptance_of_T[i]);
    rh.push_back(rho_of_T ? rho_of_T[i] : nullptr);
  }
  std::vector<bwl_run_stats> st(again.size());
  double more_ms = 0.0;
  rc = anneal_run((int)again.size(), cs.data(), ps.data(), e.data(), cv.data(), ac.data(), st.data(), &more_ms,
                  rho_of_T ? rh.data() : nullptr, false);
  if (rc) return rc;
  for (size_t k = 0; k < again.size(); ++k) {
    if (stats) stats[again[k]] = st[k];
    cs[k]->ran[1] = 1;
  }
  if (makespan_ms) *makespan_ms = ms + more_ms;
  return BWL_OK;
}

}  // namespace bwl

extern "C" {

int bwl_test_anneal_ran(const bwl_ctx *c, int32_t *ran3) {
  memcpy(ran3, c->ran, sizeof(c->ran));
  return BWL_OK;
}

int bwl_test_give_up(bwl_ctx *c, int32_t on) {
  c->give_up = on != 0;
  return BWL_OK;
}

}  // extern "C"
