// C ABI of librdmce.so (declared in include/rdmce.h): host graph handling,
// generators, and the device plan that uploads a graph once and runs the
// enumeration kernels on it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "capi_internal.hpp"
#include "generators.hpp"
#include "mce_device.hpp"
#include "parallel.hpp"
#include "rng.hpp"

using namespace rdmce;

namespace {
thread_local std::string g_err;
}  // namespace

void rdmce::set_last_error(const std::string &msg) { g_err = msg; }

namespace {
mce_status fail(mce_status s, const std::string &msg) {
  g_err = msg;
  return s;
}

#define HIP_TRY(expr)                                                                            \
  do {                                                                                           \
    hipError_t e_ = (expr);                                                                      \
    if (e_ != hipSuccess)                                                                        \
      return fail(MCE_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_));            \
  } while (0)

double ms_since(std::chrono::steady_clock::time_point t0) {
  return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

template <class F>
mce_status guarded(F &&f) {
  try {
    return f();
  } catch (const std::bad_alloc &) {
    return fail(MCE_ERR_NOMEM, "host allocation failed");
  } catch (const std::exception &e) {
    return fail(MCE_ERR_INTERNAL, e.what());
  }
}

mce_status new_graph(mce_graph **out) {
  if (!out) return fail(MCE_ERR_ARG, "null output pointer");
  *out = new mce_graph();
  return MCE_OK;
}

// Canonical roots: edge roots (v0 << 32 | v1), v0 < v1, ascending; vertex
// roots v ascending.
void build_roots(const HostGraph &g, int mode, std::vector<uint64_t> &roots, uint64_t &max_out) {
  std::vector<uint64_t> first(g.n + 1, 0), outdeg(g.n + 1, 0);
  max_out = 0;
  for (uint64_t v = 0; v < g.n; ++v) {
    const uint32_t *b = g.col.data() + g.rowoff[v], *e = g.col.data() + g.rowoff[v + 1];
    first[v] = (uint64_t)(std::upper_bound(b, e, (uint32_t)v) - b);
    outdeg[v] = (uint64_t)(e - b) - first[v];
    max_out = std::max(max_out, outdeg[v]);
  }
  if (mode == MCE_ROOT_VERTEX) {
    roots.resize(g.n);
    for (uint64_t v = 0; v < g.n; ++v) roots[v] = v;
    return;
  }
  std::vector<uint64_t> off(g.n + 1, 0);
  for (uint64_t v = 0; v < g.n; ++v) off[v + 1] = off[v] + outdeg[v];
  roots.resize(off[g.n]);
  parallel_chunks(g.n, [&](int, uint64_t b, uint64_t e) {
    for (uint64_t v = b; v < e; ++v) {
      const uint32_t *nb = g.col.data() + g.rowoff[v] + first[v];
      for (uint64_t k = 0; k < outdeg[v]; ++k) roots[off[v] + k] = (v << 32) | nb[k];
    }
  });
}
}  // namespace

extern "C" {

const char *mce_last_error(void) { return g_err.c_str(); }
const char *mce_version(void) { return "rdmce-mi355x 0.1"; }

// ---------------------------------------------------------------------------
// Graph
// ---------------------------------------------------------------------------
mce_status mce_graph_load_coo_text(const char *path, mce_graph **out) {
  return guarded([&] {
    if (!path) return fail(MCE_ERR_ARG, "null path");
    mce_status s = new_graph(out);
    if (s) return s;
    std::string err;
    if (!load_coo_text((*out)->g, path, &err)) {
      delete *out;
      *out = nullptr;
      return fail(MCE_ERR_IO, err);
    }
    return MCE_OK;
  });
}

mce_status mce_graph_load_bin(const char *path, mce_graph **out) {
  return guarded([&] {
    if (!path) return fail(MCE_ERR_ARG, "null path");
    mce_status s = new_graph(out);
    if (s) return s;
    std::string err;
    if (!load_bin((*out)->g, path, &err)) {
      delete *out;
      *out = nullptr;
      return fail(MCE_ERR_IO, err);
    }
    return MCE_OK;
  });
}

mce_status mce_graph_store_bin(const mce_graph *g, const char *path) {
  return guarded([&] {
    if (!g || !path) return fail(MCE_ERR_ARG, "null argument");
    std::string err;
    if (!store_bin(g->g, path, &err)) return fail(MCE_ERR_IO, err);
    return MCE_OK;
  });
}

mce_status mce_graph_bin_path(const char *input_path, char *buf, uint64_t buf_len) {
  if (!input_path || !buf) return fail(MCE_ERR_ARG, "null argument");
  std::string s = bin_path_for(input_path);
  if (s.size() + 1 > buf_len) return fail(MCE_ERR_ARG, "buffer too small");
  std::memcpy(buf, s.c_str(), s.size() + 1);
  return MCE_OK;
}

mce_status mce_graph_from_pairs(const uint32_t *u, const uint32_t *v, uint64_t count, mce_graph **out) {
  return guarded([&] {
    if ((!u || !v) && count) return fail(MCE_ERR_ARG, "null endpoint array");
    mce_status s = new_graph(out);
    if (s) return s;
    graph_from_pairs((*out)->g, u, v, count);
    return MCE_OK;
  });
}

mce_status mce_graph_from_csr(uint64_t n, const uint64_t *rowoff, const uint32_t *col, const uint32_t *labels,
                              uint64_t degeneracy, mce_graph **out) {
  return guarded([&] {
    if (!rowoff || (!col && rowoff[n])) return fail(MCE_ERR_ARG, "null CSR array");
    if (n >= (1ull << 32)) return fail(MCE_ERR_UNSUPPORTED, "more than 2^32-1 vertices");
    if (rowoff[0] != 0) return fail(MCE_ERR_ARG, "rowoff[0] is not 0");
    for (uint64_t v = 0; v < n; ++v) {
      if (rowoff[v + 1] < rowoff[v]) return fail(MCE_ERR_ARG, "row offsets decrease");
      for (uint64_t i = rowoff[v]; i < rowoff[v + 1]; ++i) {
        if (col[i] >= n || col[i] == v) return fail(MCE_ERR_ARG, "column id out of range or self loop");
        if (i > rowoff[v] && col[i] <= col[i - 1]) return fail(MCE_ERR_ARG, "row not strictly ascending");
      }
    }
    if (rowoff[n] % 2) return fail(MCE_ERR_ARG, "odd number of adjacency entries");
    // Symmetry: the kernels build P from out-lists and X from in-lists, so an
    // edge listed in one direction only would change the results silently.
    // Rows are sorted (checked above): a binary search per entry.
    std::atomic<int64_t> bad{-1};
    parallel_chunks(n, [&](int, uint64_t b, uint64_t e) {
      for (uint64_t v = b; v < e && bad.load(std::memory_order_relaxed) < 0; ++v)
        for (uint64_t i = rowoff[v]; i < rowoff[v + 1]; ++i) {
          const uint32_t u = col[i];
          if (!std::binary_search(col + rowoff[u], col + rowoff[u + 1], (uint32_t)v)) {
            bad.store((int64_t)v, std::memory_order_relaxed);
            break;
          }
        }
    });
    if (bad.load() >= 0)
      return fail(MCE_ERR_ARG, "CSR is not symmetric: row " + std::to_string(bad.load()) +
                                   " lists a neighbour whose row does not list it");
    mce_status s = new_graph(out);
    if (s) return s;
    HostGraph &g = (*out)->g;
    g.n = n;
    g.m = rowoff[n] / 2;
    g.rowoff.assign(rowoff, rowoff + n + 1);
    g.col.assign(col, col + rowoff[n]);
    g.labels.resize(n);
    for (uint64_t v = 0; v < n; ++v) g.labels[v] = labels ? labels[v] : (uint32_t)v;
    g.recompute_max_degree();
    g.degeneracy = degeneracy ? degeneracy : g.max_degree;
    return MCE_OK;
  });
}

mce_status mce_graph_order(mce_graph *g, int32_t order) {
  return guarded([&] {
    if (!g) return fail(MCE_ERR_ARG, "null graph");
    if (order < MCE_ORDER_UNCHANGED || order > MCE_ORDER_DEG) return fail(MCE_ERR_ARG, "unknown order");
    apply_order(g->g, (Order)order);
    return MCE_OK;
  });
}

mce_status mce_graph_get_info(const mce_graph *g, mce_graph_info *info) {
  if (!g || !info) return fail(MCE_ERR_ARG, "null argument");
  info->n = g->g.n;
  info->m = g->g.m;
  info->max_degree = g->g.max_degree;
  info->degeneracy = g->g.degeneracy;
  return MCE_OK;
}

mce_status mce_graph_get_csr(const mce_graph *g, const uint64_t **rowoff, const uint32_t **col,
                             const uint32_t **labels) {
  if (!g) return fail(MCE_ERR_ARG, "null graph");
  if (rowoff) *rowoff = g->g.rowoff.data();
  if (col) *col = g->g.col.data();
  if (labels) *labels = g->g.labels.data();
  return MCE_OK;
}

mce_status mce_graph_get_core(mce_graph *g, const uint32_t **core) {
  return guarded([&] {
    if (!g || !core) return fail(MCE_ERR_ARG, "null argument");
    if (g->g.core.size() != g->g.n) {
      std::vector<uint32_t> order, c;
      degeneracy_order(g->g, order, c);
      g->g.core.swap(c);
    }
    *core = g->g.core.data();
    return MCE_OK;
  });
}

mce_status mce_graph_write_coo_text(const mce_graph *g, const char *path) {
  return guarded([&] {
    if (!g || !path) return fail(MCE_ERR_ARG, "null argument");
    std::string err;
    if (!write_coo_text(g->g, path, &err)) return fail(MCE_ERR_IO, err.empty() ? "write failed" : err);
    return MCE_OK;
  });
}

void mce_graph_free(mce_graph *g) { delete g; }

// ---------------------------------------------------------------------------
// Generators
// ---------------------------------------------------------------------------
mce_status mce_gen_er(uint32_t n, double p, uint64_t seed, mce_graph **out) {
  return guarded([&] {
    if (!(p >= 0.0 && p <= 1.0)) return fail(MCE_ERR_ARG, "p outside [0, 1]");
    std::vector<uint64_t> keys;
    gen_er(n, p, seed, keys);
    mce_status s = new_graph(out);
    if (s) return s;
    graph_from_keys((*out)->g, std::move(keys));
    return MCE_OK;
  });
}

mce_status mce_gen_rmat(int32_t scale, uint64_t edge_factor, double a, double b, double c, uint64_t seed,
                        mce_graph **out) {
  return guarded([&] {
    if (scale < 1 || scale > 31) return fail(MCE_ERR_ARG, "scale outside [1, 31]");
    if (a < 0 || b < 0 || c < 0 || a + b + c > 1.0) return fail(MCE_ERR_ARG, "bad quadrant probabilities");
    std::vector<uint64_t> keys;
    gen_rmat(scale, edge_factor, a, b, c, seed, keys);
    mce_status s = new_graph(out);
    if (s) return s;
    graph_from_keys((*out)->g, std::move(keys));
    return MCE_OK;
  });
}

mce_status mce_gen_chung_lu_planted(uint64_t n, double gamma, double mean_degree, uint32_t n_comm, uint32_t cmin,
                                    uint32_t cmax, double p_in, uint64_t seed, mce_graph **out) {
  return guarded([&] {
    if (n == 0 || n >= (1ull << 32) || gamma <= 1.0 || mean_degree <= 0 || cmin > cmax || p_in < 0 || p_in > 1)
      return fail(MCE_ERR_ARG, "bad Chung-Lu parameters");
    std::vector<uint64_t> keys;
    gen_chung_lu_planted(n, gamma, mean_degree, n_comm, cmin, cmax, p_in, seed, keys);
    mce_status s = new_graph(out);
    if (s) return s;
    graph_from_keys((*out)->g, std::move(keys));
    return MCE_OK;
  });
}

mce_status mce_gen_batch_params(uint64_t seed, uint64_t index, uint32_t nmin, uint32_t nmax, double pmin,
                                double pmax, uint32_t *n, double *p, uint64_t *edge_seed) {
  if (!n || !p || !edge_seed || nmin > nmax || pmin > pmax) return fail(MCE_ERR_ARG, "bad batch parameters");
  BatchGraphParams bp = batch_graph_params(seed, index, nmin, nmax, pmin, pmax);
  *n = bp.n;
  *p = bp.p;
  *edge_seed = bp.seed;
  return MCE_OK;
}

void mce_options_init(mce_options *opt) {
  if (!opt) return;
  std::memset(opt, 0, sizeof(*opt));
  opt->device = 0;
  opt->root_mode = MCE_ROOT_EDGE;
  opt->waves_per_cu = 0;
  opt->share_bound = 0;
  opt->schedule = MCE_SCHED_PLAIN;
  opt->lds_tier = 1;
}

mce_status mce_copy_probe(int32_t device, uint64_t bytes, int32_t iters, double *ms_per_copy) {
  if (bytes < 16 || iters <= 0 || !ms_per_copy) return fail(MCE_ERR_ARG, "bad copy probe arguments");
  HIP_TRY(hipSetDevice(device));
  void *src = nullptr, *dst = nullptr;
  HIP_TRY(hipMalloc(&src, bytes));
  if (hipMalloc(&dst, bytes) != hipSuccess) {
    (void)hipFree(src);
    return fail(MCE_ERR_NOMEM, "copy probe allocation failed");
  }
  hipEvent_t e0, e1;
  hipError_t e = hipMemset(src, 1, bytes);
  if (e == hipSuccess) e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  if (e == hipSuccess) e = launch_copy_probe(src, dst, bytes, nullptr);
  if (e == hipSuccess) e = hipEventRecord(e0, nullptr);
  for (int i = 0; i < iters && e == hipSuccess; ++i) e = launch_copy_probe(src, dst, bytes, nullptr);
  if (e == hipSuccess) e = hipEventRecord(e1, nullptr);
  if (e == hipSuccess) e = hipEventSynchronize(e1);
  float ms = 0;
  if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  (void)hipFree(src);
  (void)hipFree(dst);
  if (e != hipSuccess) return fail(MCE_ERR_DEVICE, hipGetErrorString(e));
  *ms_per_copy = ms / iters;
  return MCE_OK;
}

mce_status mce_device_sync(int32_t device) {
  HIP_TRY(hipSetDevice(device));
  HIP_TRY(hipDeviceSynchronize());
  return MCE_OK;
}

int32_t mce_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Plan: one graph, or a batch of disjoint graphs concatenated, resident in
// HBM with its roots and per-wave scratch.
// ---------------------------------------------------------------------------
// What the packed search of a plan needs in device memory.
struct PackNeed {
  uint64_t stack = 0;       // words of a wave's record stack
  uint32_t waves = 0;       // waves with a stack (and clique-list ids in plans with lists)
  uint32_t mail_waves = 0;  // waves with mail (0: nothing is ever given away)
  uint32_t lists = 0;       // lists of roots too wide for a variant: one less than the launches
  uint64_t pool = 0;        // words for kept vertex bitmaps
  bool covers(const PackNeed &o) const {
    return stack >= o.stack && waves >= o.waves && mail_waves >= o.mail_waves && lists >= o.lists &&
           (pool > 0 || o.pool == 0);
  }
};

struct mce_plan {
  mce_options opt{};
  int device = 0;
  int cus = 0;
  uint64_t n = 0;
  uint64_t n_roots = 0;
  uint64_t n_dispatch = 0;
  uint32_t hist_len = 0;
  // launch configuration (the autotuner may change it between runs)
  int waves_per_cu = 16;
  uint32_t waves = 0;
  uint32_t max_waves = 0;
  uint32_t lds_bytes = 0;
  uint32_t lds_per_cu = kCuLds;
  uint32_t lds_per_block_max = 64u << 10;
  int share_bound = 24;
  int lds_tier = 1;
  uint64_t slot_bytes = 0;
  uint64_t stack_bytes = 0;
  uint64_t deferred_cap = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
  uint8_t *d_inputs = nullptr;      // the inputs below, d_rowoff .. d_eager and the packed search's, in one allocation
  uint64_t *d_rowoff = nullptr;
  uint64_t *d_outoff = nullptr;
  uint32_t *d_col = nullptr;
  uint64_t *d_lhash = nullptr;
  uint32_t *d_labels = nullptr;
  uint64_t *d_roots = nullptr;
  uint64_t *d_perm = nullptr;
  uint8_t *d_eager = nullptr;
  uint8_t *d_slots = nullptr;
  uint8_t *d_stacks = nullptr;
  ShareRec *d_recs = nullptr;
  unsigned int *d_users = nullptr;
  unsigned long long *d_has_work = nullptr;
  unsigned long long *d_ctr = nullptr;  // see Ctr
  unsigned long long *d_work = nullptr; // see kWorkWords
  unsigned long long *d_hist = nullptr;
  unsigned long long *d_root_nodes = nullptr;
  unsigned long long *d_root_cycles = nullptr;
  uint32_t *d_list = nullptr;
  uint64_t list_cap = 0;
  uint64_t *d_deferred = nullptr;
  uint64_t *d_deferred2 = nullptr;
  uint8_t *d_slots2 = nullptr;
  uint64_t slots2_bytes = 0;
  uint8_t *d_stacks2 = nullptr;
  uint64_t stacks2_bytes = 0;
  // batches
  uint64_t n_graphs = 0;
  uint32_t g_hist_stride = 0;
  uint32_t *d_root_graph = nullptr;
  unsigned long long *d_gcount = nullptr;
  unsigned long long *d_ghash = nullptr;
  unsigned long long *d_ghist = nullptr;
  // packed search (pack_kernel.hip): settings and arenas, allocated at its
  // first run
  uint64_t max_out = 0;              // largest out-degree: bounds |P0| and the search depth
  uint64_t max_deg = 0;              // largest degree: bounds |X0'|
  int pack = 0;
  uint32_t pack_slots = 4;
  int pack_wpc = 16;
  uint64_t pool_bound = 0;           // words that every vertex's bitmap would take
  PackNeed pk;                       // what the arenas below hold
  uint8_t *d_pack = nullptr;         // all of them, in one allocation
  uint64_t *d_pk_stack = nullptr;
  uint32_t *d_pk_plist = nullptr;
  uint64_t *d_wide[kPackVariants] = {};  // roots too wide for variant v, in the order met
  uint64_t *d_mail = nullptr;       // packed search: per-wave mail (work handed to idle waves)
  unsigned long long *d_pk_idle = nullptr;
  uint64_t *d_wide_h[2] = {};       // per entry of list v (in turn): its kept vertex bitmap in d_pool
  uint64_t *d_pool = nullptr;
  std::vector<uint64_t> h_rfirst;    // edge roots: canonical id of the first root of each vertex, + m
  uint64_t *d_rfirst = nullptr;
  uint64_t *d_gstart = nullptr;      // runs of the plan's dispatch list sharing their first vertex
  uint64_t n_groups = 0;
  std::vector<uint64_t> h_runs;      // host copy of d_gstart
  // captured run (hipGraph)
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
};

struct mce_batch {
  mce_plan *plan = nullptr;
};

namespace {
// Words of d_ctr: the collected sums (Sum), then the others.
enum Ctr { kCount = sCount, kHash = sHash, kNodes = sNodes, kWords = sWords, kBuild = sBuild, kShared = sShared,
           kPublished = sPublished, kOwnerTasks = sOwner, kListCursor = kNumSums, kNDeferred, kDeferNeed,
           kDeferStackNeed, kErr, kNWide0, kPoolUsed = kNWide0 + kPackVariants, kNumCtr };
// Words of d_work, the per-run counters kept in copies: dispatch counters and
// work state of each launch of a run, the sums and the clique sizes.
constexpr uint64_t kLaunches = kPackVariants + 1;
constexpr uint64_t kNextWords = (uint64_t)kShards * kShardWords;
constexpr uint64_t kStateWords = (uint64_t)kStateShards * kShardWords;
constexpr uint64_t kStateAt = kLaunches * kNextWords, kSumsAt = kStateAt + kLaunches * kStateWords,
                   kHistAt = kSumsAt + (uint64_t)kShards * kShardWords,
                   kWorkWords = kHistAt + (uint64_t)kShards * kLdsHist;

template <class T>
hipError_t dalloc(T **p, uint64_t count) {
  return hipMalloc((void **)p, std::max<uint64_t>(count, 1) * sizeof(T));
}

void drop_graph(mce_plan *p) {
  if (p->graph_exec) (void)hipGraphExecDestroy(p->graph_exec);
  if (p->graph) (void)hipGraphDestroy(p->graph);
  p->graph_exec = nullptr;
  p->graph = nullptr;
}

void plan_release(mce_plan *p) {
  if (!p) return;
  (void)hipSetDevice(p->device);
  drop_graph(p);
  void *ptrs[] = {p->d_inputs,      p->d_slots,       p->d_ctr,     p->d_root_nodes, p->d_root_cycles, p->d_list,
                  p->d_deferred,    p->d_deferred2,   p->d_slots2,  p->d_stacks,     p->d_stacks2,     p->d_recs,
                  p->d_users,       p->d_has_work,    p->d_gcount,  p->d_ghash,      p->d_ghist,       p->d_work};
  for (void *q : ptrs)
    if (q) (void)hipFree(q);
  if (p->d_pack) (void)hipFree(p->d_pack);
  for (auto &e : p->ev)
    if (e) (void)hipEventDestroy(e);
  if (p->stream) (void)hipStreamDestroy(p->stream);
  delete p;
}

uint64_t align_up(uint64_t x, uint64_t a) { return (x + a - 1) / a * a; }

// Scratch of the largest possible root: candidates c <= max degree,
// |P| <= max out-degree.  Data region: candidate list + bitmap + label
// hashes; stack: (|P| + 1) level records.
uint64_t worst_data(uint64_t maxdeg, uint64_t maxout) {
  uint64_t p = std::min(maxdeg, maxout), c = maxdeg;
  uint64_t W = (p + 63) / 64;
  return align_up(4 * c, 256) + align_up(8 * W * align_up(c, 64), 256) + align_up(8 * p, 256);
}
uint64_t worst_stack(uint64_t maxdeg, uint64_t maxout) {
  uint64_t p = std::min(maxdeg, maxout), x = maxdeg;
  uint64_t W = (p + 63) / 64, Wx = (x + 63) / 64;
  return (p + 1) * (4 * W + Wx + 4) * 8;
}

uint32_t lds_for(const mce_plan *p, int wpc, uint32_t override_bytes) {
  if (override_bytes) return std::min<uint32_t>(override_bytes, p->lds_per_block_max);
  uint64_t per_wave = p->lds_per_cu / (uint64_t)std::max(1, wpc);
  per_wave = per_wave > 1024 ? per_wave - 1024 : 0;  // the LDS histogram (kLdsHist words) + slack
  per_wave = std::min<uint64_t>(per_wave, p->lds_per_block_max);
  return (uint32_t)(per_wave / 256 * 256);
}

void set_config(mce_plan *p, int wpc, int share_bound, int lds_tier) {
  p->waves_per_cu = wpc;
  p->waves = (uint32_t)std::min<uint64_t>(p->max_waves, std::max<uint64_t>(1, (uint64_t)p->cus * wpc));
  p->share_bound = share_bound;
  p->lds_tier = lds_tier;
  p->lds_bytes = lds_for(p, wpc, p->opt.lds_bytes);
  drop_graph(p);
}

// Runs of consecutive dispatch entries that are edge roots of one first
// vertex (the packed search builds that vertex's bitmap once per run):
// run r covers dispatch entries [out[r], out[r + 1]).  disp(i) gives the
// canonical root id of dispatch entry i.
template <class F>
std::vector<uint64_t> dispatch_runs(const std::vector<uint64_t> &rfirst, uint64_t n_disp, F disp) {
  std::vector<uint64_t> out;
  out.push_back(0);
  uint64_t lo = 1, hi = 0;  // canonical ids of the current first vertex: [lo, hi)
  for (uint64_t i = 0; i < n_disp; ++i) {
    const uint64_t r = disp(i);
    if (r >= lo && r < hi) continue;
    const uint64_t v0 = (uint64_t)(std::upper_bound(rfirst.begin(), rfirst.end(), r) - rfirst.begin()) - 1;
    lo = rfirst[v0];
    hi = rfirst[v0 + 1];
    if (i) out.push_back(i);
  }
  if (n_disp) out.push_back(n_disp);
  return out;
}

// A plan's input arrays: one device allocation, each array aligned to 256
// bytes, filled by one copy when they are small (a copy costs 12 us however
// short; ten of them were a third of a solve of G(200, 0.1)) and by one each
// when gathering them on the host first would cost more (1 MB takes 93 us to
// copy).
struct Inputs {
  struct Item {
    void **dst;
    const void *src;
    uint64_t bytes, at;
  };
  std::vector<Item> items;
  uint64_t total = 0;
  // `src` has to stay until upload(); *dst is set there.
  template <class T>
  void add(T **dst, const T *src, uint64_t count) {
    items.push_back({(void **)dst, src, count * sizeof(T), total});
    total += (std::max<uint64_t>(count, 1) * sizeof(T) + 255) / 256 * 256;
  }
  hipError_t upload(uint8_t **base) const {
    hipError_t e = hipMalloc((void **)base, std::max<uint64_t>(total, 256));
    if (e != hipSuccess) return e;
    for (const Item &it : items) *it.dst = *base + it.at;
    if (total <= (1u << 20)) {
      std::vector<uint8_t> stage(total);
      for (const Item &it : items)
        if (it.bytes) std::memcpy(stage.data() + it.at, it.src, it.bytes);
      return total ? hipMemcpy(*base, stage.data(), total, hipMemcpyHostToDevice) : hipSuccess;
    }
    for (const Item &it : items)
      if (it.bytes && e == hipSuccess) e = hipMemcpy(*base + it.at, it.src, it.bytes, hipMemcpyHostToDevice);
    return e;
  }
};

// What a plan is built from: a (possibly concatenated) graph, and for
// batches the graph index of every vertex range.
struct PlanSpec {
  const HostGraph *g;
  const std::vector<uint64_t> *graph_vstart = nullptr;  // batches: first vertex of each graph, + total
};

mce_status plan_create_impl(const PlanSpec &spec, const mce_options &opt, mce_plan **out) {
  const HostGraph &g = *spec.g;
  auto p = new mce_plan();
  p->opt = opt;
  p->device = opt.device;
  auto bail = [&](mce_status s) {
    plan_release(p);
    return s;
  };
#define PTRY(expr)                                                                                   \
  do {                                                                                               \
    hipError_t e_ = (expr);                                                                          \
    if (e_ != hipSuccess)                                                                            \
      return bail(fail(e_ == hipErrorOutOfMemory ? MCE_ERR_NOMEM : MCE_ERR_DEVICE,                   \
                       std::string(#expr) + ": " + hipGetErrorString(e_)));                          \
  } while (0)
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return bail(fail(MCE_ERR_DEVICE, "no HIP device"));
  if (opt.device < 0 || opt.device >= ndev) return bail(fail(MCE_ERR_ARG, "device ordinal out of range"));
  PTRY(hipSetDevice(opt.device));
  hipDeviceProp_t prop;
  PTRY(hipGetDeviceProperties(&prop, opt.device));
  p->cus = prop.multiProcessorCount;
  p->lds_per_cu = lds_of_cu(prop.sharedMemPerMultiprocessor);
  if (prop.sharedMemPerBlock) p->lds_per_block_max = (uint32_t)prop.sharedMemPerBlock - 1024;
  PTRY(hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking));
  for (auto &e : p->ev) PTRY(hipEventCreate(&e));

  const int mode = opt.root_mode == MCE_ROOT_VERTEX ? MCE_ROOT_VERTEX : MCE_ROOT_EDGE;
  p->opt.root_mode = mode;
  std::vector<uint64_t> roots;
  uint64_t max_out = 0;
  build_roots(g, mode, roots, max_out);
  p->max_out = max_out;
  p->pack = opt.pack > 0 ? 1 : 0;
  p->pack_slots = opt.pack_slots ? std::min<uint32_t>(std::max<uint32_t>(opt.pack_slots, 1), kPackMaxSlots) : 4;
  p->pack_wpc = opt.pack_waves_per_cu ? (int)std::min<uint32_t>(std::max<uint32_t>(opt.pack_waves_per_cu, 1), 32) : 16;
  p->n = g.n;
  p->n_roots = roots.size();
  p->n_dispatch = p->n_roots;
  p->hist_len = (uint32_t)std::min<uint64_t>(max_out + 3, 1ull << 20);
  if (p->hist_len < kLdsHist) p->hist_len = kLdsHist;

  Inputs in;
  std::vector<uint64_t> lhash(g.n);
  for (uint64_t v = 0; v < g.n; ++v) lhash[v] = splitmix64_mix(g.labels[v]);

  std::vector<uint64_t> outoff(g.n + 1, 0);
  {
    parallel_chunks(g.n, [&](int, uint64_t b, uint64_t e) {
      for (uint64_t v = b; v < e; ++v) {
        const uint32_t *rb = g.col.data() + g.rowoff[v], *re = g.col.data() + g.rowoff[v + 1];
        outoff[v] = g.rowoff[v] + (uint64_t)(std::upper_bound(rb, re, (uint32_t)v) - rb);
      }
    });
    outoff[g.n] = g.rowoff[g.n];
    // words of one kept vertex bitmap per vertex with 2 to 1024 edge roots
    // (the packed search's pool bound)
    for (uint64_t v = 0; v < g.n; ++v) {
      const uint64_t d = g.rowoff[v + 1] - outoff[v], x = outoff[v] - g.rowoff[v];
      p->max_deg = std::max(p->max_deg, d + x);
      if (d >= 2 && d <= 1024) p->pool_bound += 8 + (d + 63) / 64 * (align_up(d + x, 64) + 1) + d;
    }
  }
  in.add(&p->d_rowoff, g.rowoff.data(), g.n + 1);
  in.add(&p->d_outoff, outoff.data(), g.n + 1);
  in.add(&p->d_col, g.col.data(), g.col.size());
  in.add(&p->d_lhash, lhash.data(), g.n);
  in.add(&p->d_labels, g.labels.data(), g.n);
  in.add(&p->d_roots, roots.data(), p->n_roots);
  if (opt.schedule == MCE_SCHED_CUSTOM) {
    if (!opt.roots) return bail(fail(MCE_ERR_ARG, "custom schedule without a root list"));
    if (opt.n_roots > p->n_roots) return bail(fail(MCE_ERR_ARG, "custom root list longer than the root set"));
    // The list holds distinct canonical root ids (all of them, or a subset:
    // then the results cover exactly the cliques of the listed roots).
    std::vector<uint8_t> seen(p->n_roots, 0);
    for (uint64_t i = 0; i < opt.n_roots; ++i) {
      if (opt.roots[i] >= p->n_roots || seen[opt.roots[i]])
        return bail(fail(MCE_ERR_ARG, "root list has an out-of-range or repeated id"));
      seen[opt.roots[i]] = 1;
    }
    p->n_dispatch = opt.n_roots;
    in.add(&p->d_perm, opt.roots, opt.n_roots);
  }
  if (mode == MCE_ROOT_EDGE) {
    p->h_rfirst.assign(g.n + 1, 0);
    uint64_t r = 0;
    for (uint64_t v = 0; v < g.n; ++v) {
      p->h_rfirst[v] = r;
      while (r < p->n_roots && (roots[r] >> 32) == v) ++r;
    }
    p->h_rfirst[g.n] = r;
    in.add(&p->d_rfirst, p->h_rfirst.data(), g.n + 1);
    const uint64_t nd = p->n_dispatch;
    const uint64_t *cr = opt.schedule == MCE_SCHED_CUSTOM ? opt.roots : nullptr;
    std::vector<uint64_t> runs;
    if (opt.runs && cr) {
      // caller runs: boundaries ascending from 0 to n_roots, one first vertex each
      if (opt.runs[0] != 0 || opt.runs[opt.n_runs] != nd)
        return bail(fail(MCE_ERR_ARG, "runs must start at 0 and end at the root count"));
      for (uint64_t r = 0; r < opt.n_runs; ++r) {
        if (opt.runs[r] >= opt.runs[r + 1]) return bail(fail(MCE_ERR_ARG, "runs must be strictly ascending"));
        const uint64_t lo = p->h_rfirst[(uint64_t)(roots[cr[opt.runs[r]]] >> 32)];
        const uint64_t hi = p->h_rfirst[(uint64_t)(roots[cr[opt.runs[r]]] >> 32) + 1];
        for (uint64_t i = opt.runs[r]; i < opt.runs[r + 1]; ++i)
          if (cr[i] < lo || cr[i] >= hi) return bail(fail(MCE_ERR_ARG, "a run mixes first vertices"));
      }
      runs.assign(opt.runs, opt.runs + opt.n_runs + 1);
    } else {
      runs = dispatch_runs(p->h_rfirst, nd, [&](uint64_t i) { return cr ? cr[i] : nd - 1 - i; });
    }
    p->n_groups = runs.size() - 1;
    p->h_runs = std::move(runs);
    in.add(&p->d_gstart, p->h_runs.data(), p->h_runs.size());
  }
  if (opt.eager) in.add(&p->d_eager, opt.eager, p->n_dispatch);
  std::vector<uint32_t> rg;
  if (spec.graph_vstart) {
    const auto &vs = *spec.graph_vstart;
    p->n_graphs = vs.size() - 1;
    p->g_hist_stride = std::max<uint32_t>(p->hist_len, kLdsHist);
    rg.resize(p->n_roots);
    for (uint64_t r = 0; r < p->n_roots; ++r) {
      uint64_t v0 = mode == MCE_ROOT_EDGE ? (roots[r] >> 32) : roots[r];
      rg[r] = (uint32_t)(std::upper_bound(vs.begin(), vs.end(), v0) - vs.begin() - 1);
    }
    in.add(&p->d_root_graph, rg.data(), p->n_roots);
    PTRY(dalloc(&p->d_gcount, p->n_graphs));
    PTRY(dalloc(&p->d_ghash, p->n_graphs));
    PTRY(dalloc(&p->d_ghist, p->n_graphs * p->g_hist_stride));
  }

  PTRY(in.upload(&p->d_inputs));

  const int wpc = opt.waves_per_cu > 0 ? opt.waves_per_cu : 16;
  p->max_waves = (uint32_t)std::min<uint64_t>(16384, (uint64_t)p->cus * std::max(wpc, 32));
  size_t free_b = 0, total_b = 0;
  PTRY(hipMemGetInfo(&free_b, &total_b));
  // Each wave gets a data region and a stack; both are sized for the largest
  // root when that fits in ~45% of free HBM, else capped (larger roots go to
  // the deferred pass).  slot_bytes, when given, is split evenly.
  uint64_t cap = std::min<uint64_t>(32ull << 20, (uint64_t)(free_b * 0.22) / p->max_waves);
  uint64_t want_d = opt.slot_bytes ? opt.slot_bytes / 2 : std::min(worst_data(g.max_degree, max_out), cap);
  uint64_t want_s = opt.slot_bytes ? opt.slot_bytes / 2 : std::min(worst_stack(g.max_degree, max_out), cap);
  p->slot_bytes = align_up(std::max<uint64_t>(want_d, 2048), 256);
  p->stack_bytes = align_up(std::max<uint64_t>(want_s, 2048), 256);
  PTRY(dalloc(&p->d_slots, p->slot_bytes * p->max_waves));
  PTRY(dalloc(&p->d_stacks, p->stack_bytes * p->max_waves));
  PTRY(dalloc(&p->d_recs, p->max_waves));
  PTRY(dalloc(&p->d_users, p->max_waves + 2));  // zeroed in whole 8-byte words
  PTRY(dalloc(&p->d_has_work, (p->max_waves + 63) / 64));
  PTRY(dalloc(&p->d_work, kWorkWords));
  set_config(p, wpc, opt.share_bound == 0 ? 24 : opt.share_bound, opt.lds_tier ? 1 : 0);

  PTRY(dalloc(&p->d_ctr, kNumCtr + (uint64_t)p->hist_len));
  p->d_hist = p->d_ctr + kNumCtr;  // read back with the counters
  if (opt.want_root_stats) {
    PTRY(dalloc(&p->d_root_nodes, p->n_roots));
    PTRY(dalloc(&p->d_root_cycles, p->n_roots));
  }
  if (opt.want_list) {
    p->list_cap = opt.list_capacity ? opt.list_capacity : (1ull << 24);
    PTRY(dalloc(&p->d_list, p->list_cap));
  }
  p->deferred_cap = std::max<uint64_t>(1, std::min<uint64_t>(p->n_roots, 1ull << 24));
  PTRY(dalloc(&p->d_deferred, p->deferred_cap));
  PTRY(hipStreamSynchronize(p->stream));
  *out = p;
  return MCE_OK;
#undef PTRY
}

KArgs make_args(const mce_plan *p) {
  KArgs a{};
  a.rowoff = p->d_rowoff;
  a.outoff = p->d_outoff;
  a.col = p->d_col;
  a.label_hash = p->d_lhash;
  a.labels = p->d_labels;
  a.n = p->n;
  a.roots = p->d_roots;
  a.n_roots_canon = p->n_roots;
  a.perm = p->d_perm;
  a.eager = p->d_eager;
  a.n_dispatch = p->n_dispatch;
  a.reverse = p->d_perm ? 0 : 1;
  a.root_mode = p->opt.root_mode;
  a.next_root = p->d_work;
  a.state = p->d_work + kStateAt;
  a.sums = p->d_work + kSumsAt;
  a.hist_sh = p->d_work + kHistAt;
  a.list_cursor = p->d_ctr + kListCursor;
  a.n_deferred = p->d_ctr + kNDeferred;
  a.deferred_need = p->d_ctr + kDeferNeed;
  a.deferred_stack_need = p->d_ctr + kDeferStackNeed;
  a.err = (unsigned int *)(p->d_ctr + kErr);
  a.hist = p->d_hist;
  a.hist_len = p->hist_len;
  a.root_nodes = p->d_root_nodes;
  a.root_cycles = p->d_root_cycles;
  a.list = p->d_list;
  a.list_cap = p->list_cap;
  a.slots = p->d_slots;
  a.slot_bytes = p->slot_bytes;
  a.stacks = p->d_stacks;
  a.stack_bytes = p->stack_bytes;
  a.recs = p->d_recs;
  a.users = p->d_users;
  a.has_work = p->d_has_work;
  a.share_bound = p->share_bound;
  a.n_waves = p->waves;
  a.lds_tier = p->lds_tier;
  a.lds_bytes = p->lds_bytes;
  a.word_path = p->opt.word_path >= 0;
  a.deferred = p->d_deferred;
  a.deferred_cap = p->deferred_cap;
  a.root_graph = p->d_root_graph;
  a.g_count = p->d_gcount;
  a.g_hash = p->d_ghash;
  a.g_hist = p->d_ghist;
  a.g_hist_stride = p->g_hist_stride;
  a.rfirst = p->d_rfirst;
  a.pk_gstart = p->d_gstart;
  a.pk_ngroups = p->n_groups;
  return a;
}

// Packed search: records per wave and the depth above which only the top
// record is expanded, for variant (nw, nx).  A record's depth is at most
// |R| <= |P0| <= min(64 nw, largest out-degree); expanding only the top record
// adds at most 64 records per depth level, so pk_thr + 64 (depth + 3) records
// always suffice.
constexpr uint64_t kPackThr = 256;
uint64_t pack_need_records(const mce_plan *p, uint32_t nw) {
  return kPackThr + 64 * (std::min<uint64_t>(64ull * nw, p->max_out) + 3);
}

// Whether a level can ever be exposed, or records given away: |P| >=
// share_bound takes a root with that many candidates (at most the largest
// out-degree), or an eager root.
bool can_share(const mce_plan *p, const KArgs &a) {
  return a.share_bound > 0 && ((uint64_t)a.share_bound <= p->max_out || a.eager);
}

// Launches of a packed run: its variants up to the first one that no root of
// this graph is too wide for (|P0| is at most the largest out-degree, |X0'| the
// largest degree), else all of them and the one-root-per-wave kernel, which
// also takes the eager roots.
int pack_launches(const mce_plan *p, const KArgs &a) {
  for (int v = 0; v < kPackVariants; ++v)
    if (p->max_out <= 64 * kPackNW[v] && p->max_deg <= 64 * kPackNX[v] && !a.eager) return v + 1;
  return kPackVariants + 1;
}

// Slots and waves of variant v's launch.
struct PackShape {
  uint32_t slots, waves;
};
PackShape pack_shape(const mce_plan *p, const KArgs &a, int v) {
  const uint32_t nw = kPackNW[v], nx = kPackNX[v];
  const bool batch = a.root_graph != nullptr;
  // the wider variants' slots are 3.5 and 5.5 times larger: half and a
  // quarter as many; and no more than let the requested waves per CU all be
  // resident in its LDS (a wave that waited for LDS started late)
  uint32_t slots = std::max<uint32_t>(1, p->pack_slots >> v);
  while (slots > 1 && (pack_lds_bytes(nw, nx, slots, batch) > p->lds_per_block_max ||
                       pack_lds_bytes(nw, nx, slots, batch) * (uint64_t)p->pack_wpc > p->lds_per_cu))
    --slots;
  // Waves: those that fit a CU's LDS and the registers of the variant that
  // launch_pack picks (a wave that has to wait starts late); without sharing,
  // no more than the runs the first launch hands out (the others' list lengths
  // are not known here).
  uint64_t fit = std::max<uint64_t>(1, p->lds_per_cu / pack_lds_bytes(nw, nx, slots, batch));
  if (v == 2 || (v == 1 && p->pack_wpc <= 16)) fit = std::min<uint64_t>(fit, 12);
  uint64_t waves = std::min<uint64_t>({(uint64_t)p->max_waves, (uint64_t)p->cus * 32, fit * p->cus,
                                       std::max<uint64_t>(1, (uint64_t)p->cus * p->pack_wpc)});
  if (v == 0 && !can_share(p, a))
    waves = std::min<uint64_t>(waves, std::max<uint64_t>(a.pk_gstart ? a.pk_ngroups : a.n_dispatch, 1));
  return {slots, (uint32_t)waves};
}

// What a run with these arguments and the plan's present settings needs: the
// variants and waves that it launches, not the widest and most there could be.
// A solve allocates and frees this in every call, and what is freed has to be
// cleared before it is handed out again, at some 30 GB/s.  Solves one after the
// other, with arenas for 8,192 waves of the widest variant against this:
// G(91, 0.157), 1.1 GB, 32.1 ms a call against 0.26; G(3854, 0.0038), 1.5 GB, 33
// to 49 against 6.6.
PackNeed pack_need(const mce_plan *p, const KArgs &a) {
  PackNeed n;
  const int launches = pack_launches(p, a);
  for (int v = 0; v < launches && v < kPackVariants; ++v) {
    n.stack = std::max(n.stack, pack_need_records(p, kPackNW[v]) * pack_rec_words(kPackNW[v], kPackNX[v]));
    n.waves = std::max(n.waves, pack_shape(p, a, v).waves);
  }
  if (can_share(p, a)) n.mail_waves = n.waves;
  n.lists = (uint32_t)launches - 1;
  if (n.lists) n.pool = p->pool_bound;
  return n;
}

// Allocates the packed search's arenas for a run with these arguments, again
// when settings or arguments ask for more: one allocation, so they are all
// there or none is.
mce_status ensure_pack(mce_plan *p, const KArgs &a) {
  const PackNeed need = pack_need(p, a);
  if (p->d_pack && p->pk.covers(need)) return MCE_OK;
  PackNeed n = p->pk;
  n.stack = std::max(n.stack, need.stack);
  n.waves = std::max(n.waves, need.waves);
  n.mail_waves = std::max(n.mail_waves, need.mail_waves);
  n.lists = std::max(n.lists, need.lists);
  n.pool = std::max(n.pool, need.pool);
  drop_graph(p);  // (it would launch with the old ones)
  if (p->d_pack) (void)hipFree(p->d_pack);
  p->d_pack = nullptr;
  p->pk = PackNeed{};
  uint64_t bytes = 0;
  auto take = [&](uint64_t b) {
    const uint64_t at = bytes;
    bytes = align_up(bytes + b, 256);
    return at;
  };
  const uint64_t list = 8 * std::max<uint64_t>(p->n_dispatch, 1);
  const uint64_t o_stack = take(8 * n.stack * n.waves), o_mail = take(8ull * kPackMailWords * n.mail_waves),
                 o_idle = take((n.mail_waves + 63) / 64 * 8), o_wide = take(n.lists * list),
                 o_wide_h = take(2 * list),
                 o_ids = take(p->opt.want_list ? 4ull * kPackMaxSlots * kPackMaxP * n.waves : 0);
  // Kept vertex bitmaps: room for one per vertex with two or more edge roots,
  // within a quarter of the free device memory (a run that was split keeps one
  // per part; what finds no room is built again).
  size_t free_b = 0, total_b = 0;
  if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) free_b = 0;
  n.pool = std::min<uint64_t>(n.pool, free_b > bytes ? (free_b - bytes) / 4 / 8 : 0);
#ifdef RDMCE_PACK_POOL_MAX  // test builds: a pool that runs out after a few bitmaps
  n.pool = std::min<uint64_t>(n.pool, RDMCE_PACK_POOL_MAX);
#endif
  const uint64_t o_pool = take(8 * n.pool);
  const hipError_t e = hipMalloc((void **)&p->d_pack, bytes);
  if (e != hipSuccess) {
    p->d_pack = nullptr;
    (void)hipGetLastError();  // or the next launch would report it
    return fail(MCE_ERR_DEVICE, std::string("packed search memory: ") + hipGetErrorString(e));
  }
  auto at = [&](bool has, uint64_t o) { return has ? p->d_pack + o : nullptr; };
  p->d_pk_stack = (uint64_t *)at(true, o_stack);
  p->d_mail = (uint64_t *)at(n.mail_waves, o_mail);
  p->d_pk_idle = (unsigned long long *)at(n.mail_waves, o_idle);
  for (uint32_t v = 0; v < (uint32_t)kPackVariants; ++v) p->d_wide[v] = (uint64_t *)at(v < n.lists, o_wide + v * list);
  for (int k = 0; k < 2; ++k) p->d_wide_h[k] = (uint64_t *)at(true, o_wide_h + k * list);
  p->d_pk_plist = (uint32_t *)at(p->opt.want_list, o_ids);
  p->d_pool = (uint64_t *)at(n.pool, o_pool);
  p->pk = n;
  return MCE_OK;
}

// Ranges zeroed before a run: counters and results ...
void result_fills(const mce_plan *p, FillList &f) {
  f.add(p->d_ctr, kNumCtr);
  f.add(p->d_hist, p->hist_len);
  if (p->d_gcount) f.add(p->d_gcount, p->n_graphs);
  if (p->d_ghash) f.add(p->d_ghash, p->n_graphs);
  if (p->d_ghist) f.add(p->d_ghist, p->n_graphs * p->g_hist_stride);
}
// ... and before each launch of the one-root-per-wave kernel: its sharing
// words.
void share_fills(const mce_plan *p, uint64_t waves, FillList &f) {
  f.add(p->d_recs, sizeof(ShareRec) / 8 * waves);
  f.add(p->d_users, (waves + 1) / 2);
  f.add(p->d_has_work, (waves + 63) / 64);
}

hipError_t collect(const mce_plan *p, hipStream_t s) {
  return launch_collect(p->d_work + kSumsAt, p->d_work + kHistAt, p->d_ctr, p->d_hist, p->hist_len, s);
}

// Waves of the one-root-per-wave kernel: those beyond the root count could
// only take shared tasks.
uint32_t mce_waves(const mce_plan *p, KArgs &a) {
  if (can_share(p, a)) return p->waves;
  a.share_bound = -1;
  return (uint32_t)std::min<uint64_t>(p->waves, std::max<uint64_t>(a.n_dispatch, 1));
}

// Resets every counter, result and sharing word of a run with one fill kernel
// (graph-capturable; one launch per buffer took 11 launches, 2 us each) and
// launches the enumeration kernels: with the packed search on, its variants
// in turn, the first over the dispatch list, each next one over the roots the
// one before found too wide (derived from the vertex bitmaps the first one
// kept for them), and the one-root-per-wave kernel over the rest (each
// later launch reads its list length from the counter the earlier one
// filled, so the sequence needs no host round trip).
hipError_t enqueue_run(const mce_plan *p, const KArgs &a0, hipStream_t s) {
  KArgs a = a0;
  FillList f;
  result_fills(p, f);
  share_fills(p, p->waves, f);
  f.add(p->d_work, kWorkWords);
  if (p->d_root_nodes) f.add(p->d_root_nodes, p->n_roots);
  if (p->d_root_cycles) f.add(p->d_root_cycles, p->n_roots);
  if (p->pack && p->d_pk_idle) f.add(p->d_pk_idle, (p->pk.mail_waves + 63) / 64);
  hipError_t e = launch_fill_zero(f, s);
  if (e != hipSuccess) return e;
  if (!p->pack) {
    e = launch_mce(a, mce_waves(p, a), (uint32_t)p->waves_per_cu, s);
    return e == hipSuccess ? collect(p, s) : e;
  }
  const bool share = can_share(p, a);
  const int launches = pack_launches(p, a);
  for (int v = 0; v < launches && v < kPackVariants && e == hipSuccess; ++v) {
    const PackShape sh = pack_shape(p, a, v);
    const uint32_t nw = kPackNW[v], nx = kPackNX[v];
    KArgs b = a;
    b.pk_stack = p->d_pk_stack;
    b.pk_cap = p->pk.stack / pack_rec_words(nw, nx);
    b.pk_thr = (uint32_t)(b.pk_cap - 64 * (std::min<uint64_t>(64ull * nw, p->max_out) + 3));
#ifdef RDMCE_PACK_THR_MAX  // test builds: reach the depth-first expansion on small graphs
    b.pk_thr = std::min<uint32_t>(b.pk_thr, RDMCE_PACK_THR_MAX);
#endif
    b.pk_slots = sh.slots;
    b.pk_plist = p->d_pk_plist;
    b.wide = p->d_wide[v];
    b.n_wide = p->d_ctr + kNWide0 + v;
    b.heavy = p->d_wide[kPackVariants - 1];
    b.n_heavy = p->d_ctr + kNWide0 + kPackVariants - 1;
    b.pk_pool = p->d_pool;
    b.pk_pool_words = p->pk.pool;
    b.pk_pool_used = p->d_ctr + kPoolUsed;
    // wide roots leave with a copy of their vertex bitmap, from which the
    // next launches derive them
    b.wide_h = v + 1 < kPackVariants ? p->d_wide_h[v & 1] : nullptr;
    if (v) {
      b.eager = nullptr;
      b.pk_gstart = nullptr;
      b.pk_whandle = p->d_wide_h[(v - 1) & 1];
      b.perm = p->d_wide[v - 1];
      b.reverse = 0;
      b.n_dispatch_dev = p->d_ctr + kNWide0 + v - 1;
      b.next_root = p->d_work + v * kNextWords;
    }
    b.state = p->d_work + kStateAt + v * kStateWords;
    b.pk_share = share;
    b.pk_nwaves = sh.waves;
    b.pk_idle = p->d_pk_idle;
    b.pk_mail = p->d_mail;
    e = launch_pack(b, v, sh.waves, (uint32_t)p->pack_wpc, s);
  }
  if (e != hipSuccess) return e;
  if (launches <= kPackVariants) return collect(p, s);
  KArgs c = a;
  c.perm = p->d_wide[kPackVariants - 1];
  c.reverse = 0;
  c.eager = nullptr;
  c.n_dispatch_dev = p->d_ctr + kNWide0 + kPackVariants - 1;
  c.next_root = p->d_work + kPackVariants * kNextWords;
  c.state = p->d_work + kStateAt + kPackVariants * kStateWords;
  if (!can_share(p, c)) c.share_bound = -1;
  e = launch_mce(c, p->waves, (uint32_t)p->waves_per_cu, s);
  return e == hipSuccess ? collect(p, s) : e;
}

struct RunOut {
  unsigned long long ctr[kNumCtr];
  std::vector<unsigned long long> hist;  // of the last pass
  float kernel_ms = 0;
  int passes = 0;
  bool replay = false;
};

// Counters and clique sizes, which follow each other, in one copy.
hipError_t read_back(const mce_plan *p, RunOut &ro) {
  std::vector<unsigned long long> buf(kNumCtr + (uint64_t)p->hist_len);
  hipError_t e = hipMemcpy(buf.data(), p->d_ctr, buf.size() * 8, hipMemcpyDeviceToHost);
  std::copy(buf.begin(), buf.begin() + kNumCtr, ro.ctr);
  ro.hist.assign(buf.begin() + kNumCtr, buf.end());
  return e;
}

// One enumeration (plus the deferred pass when needed).  `a` may carry a
// dispatch list other than the plan's (autotuner samples).
mce_status run_core(mce_plan *p, const KArgs &a0, bool allow_graph, RunOut &ro) {
  hipStream_t s = p->stream;
  KArgs a = a0;
  ro.passes = 0;
  ro.kernel_ms = 0;
  if (a.n_dispatch == 0) {
    FillList f;
    result_fills(p, f);
    HIP_TRY(launch_fill_zero(f, s));
    HIP_TRY(hipStreamSynchronize(s));
    std::memset(ro.ctr, 0, sizeof(ro.ctr));
    ro.hist.assign(p->hist_len, 0);
    return MCE_OK;
  }
  if (p->pack) {
    mce_status st = ensure_pack(p, a);
    if (st) return st;
  }
  const bool use_graph = allow_graph && p->opt.use_graph;
  if (use_graph && !p->graph_exec) {
    HIP_TRY(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    hipError_t e = enqueue_run(p, a, s);
    hipGraph_t gr = nullptr;
    hipError_t e2 = hipStreamEndCapture(s, &gr);
    if (e != hipSuccess || e2 != hipSuccess) {
      if (gr) (void)hipGraphDestroy(gr);
      return fail(MCE_ERR_DEVICE, std::string("graph capture failed: ") + hipGetErrorString(e ? e : e2));
    }
    p->graph = gr;
    HIP_TRY(hipGraphInstantiate(&p->graph_exec, p->graph, nullptr, nullptr, 0));
  }
  HIP_TRY(hipEventRecord(p->ev[0], s));
  if (use_graph) {
    HIP_TRY(hipGraphLaunch(p->graph_exec, s));
    ro.replay = true;
  } else {
    HIP_TRY(enqueue_run(p, a, s));
  }
  HIP_TRY(hipEventRecord(p->ev[1], s));
  HIP_TRY(hipEventSynchronize(p->ev[1]));
  float ms = 0;
  HIP_TRY(hipEventElapsedTime(&ms, p->ev[0], p->ev[1]));
  ro.kernel_ms += ms;
  ro.passes = 1;
  HIP_TRY(read_back(p, ro));
  uint64_t nd = ro.ctr[kNDeferred];
  if (nd > p->deferred_cap) return fail(MCE_ERR_NOMEM, "deferred-root list overflow");
  if (nd) {
    // Second pass: the deferred roots with scratch sized to the largest need.
    uint64_t slot2 = align_up(std::max<uint64_t>(ro.ctr[kDeferNeed], 2048), 256);
    uint64_t stack2 = align_up(std::max<uint64_t>(ro.ctr[kDeferStackNeed], 2048), 256);
    size_t free_b = 0, total_b = 0;
    HIP_TRY(hipMemGetInfo(&free_b, &total_b));
    uint64_t fit = (uint64_t)(free_b * 0.8) / (slot2 + stack2);
    uint64_t waves2 = std::min<uint64_t>({(uint64_t)p->waves, nd, fit});
    if (waves2 == 0) return fail(MCE_ERR_NOMEM, "a root needs " + std::to_string(slot2 + stack2) + " bytes of scratch");
    if (p->slots2_bytes < slot2 * waves2) {
      if (p->d_slots2) (void)hipFree(p->d_slots2);
      p->d_slots2 = nullptr;
      p->slots2_bytes = 0;
      HIP_TRY(dalloc(&p->d_slots2, slot2 * waves2));
      p->slots2_bytes = slot2 * waves2;
    }
    if (p->stacks2_bytes < stack2 * waves2) {
      if (p->d_stacks2) (void)hipFree(p->d_stacks2);
      p->d_stacks2 = nullptr;
      p->stacks2_bytes = 0;
      HIP_TRY(dalloc(&p->d_stacks2, stack2 * waves2));
      p->stacks2_bytes = stack2 * waves2;
    }
    if (!p->d_deferred2) HIP_TRY(dalloc(&p->d_deferred2, p->deferred_cap));
    HIP_TRY(hipMemcpyAsync(p->d_deferred2, p->d_deferred, nd * 8, hipMemcpyDeviceToDevice, s));
    FillList f;
    f.add(p->d_ctr + kNDeferred, 3);
    f.add(p->d_work, kSumsAt);
    share_fills(p, waves2, f);
    HIP_TRY(launch_fill_zero(f, s));
    KArgs b = a;
    b.perm = p->d_deferred2;
    b.eager = nullptr;
    b.n_dispatch = nd;
    b.reverse = 0;
    b.slots = p->d_slots2;
    b.slot_bytes = slot2;
    b.stacks = p->d_stacks2;
    b.stack_bytes = stack2;
    b.n_waves = (uint32_t)waves2;
    HIP_TRY(hipEventRecord(p->ev[2], s));
    HIP_TRY(launch_mce(b, (uint32_t)waves2, (uint32_t)p->waves_per_cu, s));
    HIP_TRY(collect(p, s));
    HIP_TRY(hipEventRecord(p->ev[3], s));
    HIP_TRY(hipEventSynchronize(p->ev[3]));
    HIP_TRY(hipEventElapsedTime(&ms, p->ev[2], p->ev[3]));
    ro.kernel_ms += ms;
    ro.passes = 2;
    uint64_t deferred_first = ro.ctr[kNDeferred];
    HIP_TRY(read_back(p, ro));
    if (ro.ctr[kNDeferred]) return fail(MCE_ERR_INTERNAL, "root deferred twice");
    ro.ctr[kNDeferred] = deferred_first;
  }
  uint32_t err = (uint32_t)ro.ctr[kErr];
  if (err & kErrPTooLarge) return fail(MCE_ERR_UNSUPPORTED, "a root has more than 4096 candidates");
  if (err & kErrHistOverflow) return fail(MCE_ERR_INTERNAL, "clique size beyond histogram");
  if (err & kErrListFull) return fail(MCE_ERR_NOMEM, "clique list capacity exceeded");
  if (err & kErrDeferFull) return fail(MCE_ERR_NOMEM, "deferred-root list overflow");
  if (err & kErrPackStack) return fail(MCE_ERR_INTERNAL, "packed search: record stack full");
  return MCE_OK;
}

mce_status plan_run_impl(mce_plan *p, mce_result **out) {
  auto t0 = std::chrono::steady_clock::now();
  HIP_TRY(hipSetDevice(p->device));
  RunOut ro;
  mce_status st = run_core(p, make_args(p), true, ro);
  if (st) return st;
  auto res = new mce_result();
  std::memset(res, 0, sizeof(*res));
  auto bail = [&](mce_status s) {
    mce_result_free(res);
    return s;
  };
#define RTRY(expr)                                                                          \
  do {                                                                                      \
    hipError_t e_ = (expr);                                                                 \
    if (e_ != hipSuccess) return bail(fail(MCE_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_))); \
  } while (0)
  res->passes = ro.passes;
  res->waves = (int32_t)p->waves;
  res->deferred_roots = ro.ctr[kNDeferred];
  res->count = ro.ctr[kCount];
  res->hash = ro.ctr[kHash];
  res->total_nodes = ro.ctr[kNodes];
  res->shared_tasks = ro.ctr[kShared];
  res->published_levels = ro.ctr[kPublished];
  res->owner_tasks = ro.ctr[kOwnerTasks];
  res->search_bytes = ro.ctr[kWords] * 8;
  res->build_bytes = ro.ctr[kBuild];
  if (p->d_list) {
    res->list_len = ro.ctr[kListCursor];
    res->list = (uint32_t *)std::malloc(std::max<uint64_t>(res->list_len, 1) * 4);
    if (res->list_len) RTRY(hipMemcpy(res->list, p->d_list, res->list_len * 4, hipMemcpyDeviceToHost));
  }
  res->hist_len = p->hist_len;
  res->hist = (uint64_t *)std::calloc(p->hist_len, 8);
  std::copy(ro.hist.begin(), ro.hist.end(), res->hist);
  res->n_roots = p->n_roots;
  if (p->d_root_nodes) {
    res->root_nodes = (uint64_t *)std::malloc(std::max<uint64_t>(p->n_roots, 1) * 8);
    res->root_cycles = (uint64_t *)std::malloc(std::max<uint64_t>(p->n_roots, 1) * 8);
    if (p->n_roots) {
      RTRY(hipMemcpy(res->root_nodes, p->d_root_nodes, p->n_roots * 8, hipMemcpyDeviceToHost));
      RTRY(hipMemcpy(res->root_cycles, p->d_root_cycles, p->n_roots * 8, hipMemcpyDeviceToHost));
    }
  }
  res->kernel_ms = ro.kernel_ms;
  res->total_ms = ms_since(t0);
  *out = res;
  return MCE_OK;
#undef RTRY
}

mce_status autotune_impl(mce_plan *p, uint64_t stride, mce_tune_result *out) {
  HIP_TRY(hipSetDevice(p->device));
  if (stride == 0) stride = 1;
  // Sample: every stride-th run of edge roots sharing a first vertex, whole
  // (runs share a build in the packed search), or every stride-th root.
  std::vector<uint64_t> disp(p->n_dispatch);
  if (p->d_perm) HIP_TRY(hipMemcpy(disp.data(), p->d_perm, p->n_dispatch * 8, hipMemcpyDeviceToHost));
  else
    for (uint64_t i = 0; i < p->n_dispatch; ++i) disp[i] = p->n_dispatch - 1 - i;
  std::vector<uint64_t> sample, sruns;
  if (!p->h_runs.empty()) {
    sruns.push_back(0);
    for (uint64_t r = 0; r + 1 < p->h_runs.size(); r += stride) {
      for (uint64_t i = p->h_runs[r]; i < p->h_runs[r + 1]; ++i) sample.push_back(disp[i]);
      sruns.push_back(sample.size());
    }
  } else {
    for (uint64_t i = 0; i < disp.size(); i += stride) sample.push_back(disp[i]);
  }
  uint64_t *d_sample = nullptr, *d_sruns = nullptr;
  HIP_TRY(dalloc(&d_sample, sample.size()));
  if (!sample.empty()) HIP_TRY(hipMemcpy(d_sample, sample.data(), sample.size() * 8, hipMemcpyHostToDevice));
  const uint64_t n_sruns = sruns.empty() ? 0 : sruns.size() - 1;
  if (n_sruns) {
    HIP_TRY(dalloc(&d_sruns, sruns.size()));
    HIP_TRY(hipMemcpy(d_sruns, sruns.data(), sruns.size() * 8, hipMemcpyHostToDevice));
  }
  // Waves per CU first (LDS tier on), then the sharing bound at the best
  // occupancy, then waves per CU again when the bound changed, then the LDS
  // tier off at the best pair.
  const int wpcs[] = {8, 12, 16, 20, 24, 28, 32};
  const int taus[] = {16, 24, 48, -1};
  const int base_wpc = p->waves_per_cu, base_tau = p->share_bound, base_lds = p->lds_tier;
  double best = 1e30, base_ms = 0;
  int best_wpc = base_wpc, best_tau = base_tau, best_lds = base_lds, trials = 0;
  unsigned long long ref_count = 0, ref_hash = 0;
  auto trial = [&](int wpc, int tau, int lds, double &ms) -> mce_status {
    set_config(p, wpc, tau, lds);
    KArgs a = make_args(p);
    a.perm = d_sample;
    a.eager = nullptr;
    a.n_dispatch = sample.size();
    a.reverse = 0;
    a.pk_gstart = d_sruns;
    a.pk_ngroups = n_sruns;
    a.eager = nullptr;
    RunOut ro;
    mce_status s = run_core(p, a, false, ro);
    if (s) return s;
    ms = ro.kernel_ms;
    if (trials == 0) {
      ref_count = ro.ctr[kCount];
      ref_hash = ro.ctr[kHash];
    } else if (ro.ctr[kCount] != ref_count || ro.ctr[kHash] != ref_hash) {
      return fail(MCE_ERR_INTERNAL, "autotuner settings disagree on the result");
    }
    ++trials;
    return MCE_OK;
  };
  mce_status st = MCE_OK;
  double ms = 0;
  // default setting first (warm-up run, then the timed one)
  st = trial(base_wpc, base_tau, base_lds, ms);
  if (!st) st = trial(base_wpc, base_tau, base_lds, base_ms);
  if (!st) best = base_ms;
  if (p->pack) {
    // Packed plans: subproblems per wave (the LDS tile width), packed waves
    // per CU, then the default sharing bound if the plan has another.  Sharing
    // is never turned off: a sample holds few of the heavy roots that it is for
    // (Chung-Lu 4M: the sample took 34.6 ms without against 36.4, and the
    // vertex roots then 3,077 ms against 32).  Sample runs vary by a few percent
    // from run to run, so the default is timed twice more and a setting replaces
    // the best one only when the better of two runs beats it by kPackTuneMargin.
    constexpr double kPackTuneMargin = 0.97;
    if (!st) st = trial(base_wpc, base_tau, base_lds, ms);
    if (!st) best = base_ms = std::min(base_ms, ms);
    auto challenge = [&](int tau, bool &better) -> mce_status {
      better = false;
      double m1 = 0, m2 = 0;
      mce_status s = trial(base_wpc, tau, base_lds, m1);
      if (s || m1 >= best * kPackTuneMargin) return s;
      s = trial(base_wpc, tau, base_lds, m2);
      if (s) return s;
      const double m = std::min(m1, m2);
      if (m < best * kPackTuneMargin) {
        best = m;
        better = true;
      }
      return MCE_OK;
    };
    const uint32_t base_slots = p->pack_slots;
    const int base_pwpc = p->pack_wpc;
    uint32_t best_slots = base_slots;
    int best_pwpc = base_pwpc;
    bool better = false;
    for (uint32_t sl : {1u, 2u, 4u, 8u}) {
      if (st || sl == base_slots) continue;
      p->pack_slots = sl;
      st = challenge(base_tau, better);
      if (!st && better) best_slots = sl;
    }
    p->pack_slots = best_slots;
    for (int pw : {12, 16, 20, 24}) {
      if (st || pw == base_pwpc) continue;
      p->pack_wpc = pw;
      st = challenge(base_tau, better);
      if (!st && better) best_pwpc = pw;
    }
    p->pack_wpc = best_pwpc;
    if (!st && base_tau != 24) {
      st = challenge(24, better);
      if (!st && better) best_tau = 24;
    }
    (void)hipFree(d_sample);
    if (d_sruns) (void)hipFree(d_sruns);
    if (st) {
      p->pack_slots = base_slots;
      p->pack_wpc = base_pwpc;
      set_config(p, base_wpc, base_tau, base_lds);
      return st;
    }
    set_config(p, base_wpc, best_tau, base_lds);
    if (out) {
      std::memset(out, 0, sizeof(*out));
      out->waves_per_cu = base_wpc;
      out->share_bound = best_tau;
      out->lds_tier = base_lds;
      out->trials = trials;
      out->best_ms = best;
      out->base_ms = base_ms;
      out->pack_slots = p->pack_slots;
      out->pack_waves_per_cu = (uint32_t)p->pack_wpc;
    }
    return MCE_OK;
  }
  for (int wpc : wpcs) {
    if ((uint64_t)p->cus * wpc > p->max_waves || st || (wpc == base_wpc && base_lds == 1)) continue;
    st = trial(wpc, base_tau, 1, ms);
    if (!st && ms < best) {
      best = ms;
      best_wpc = wpc;
      best_lds = 1;
      best_tau = base_tau;
    }
  }
  for (int tau : taus) {
    if (st) break;
    if (tau == best_tau) continue;
    st = trial(best_wpc, tau, best_lds, ms);
    if (!st && ms < best) {
      best = ms;
      best_tau = tau;
    }
  }
  // Occupancy again at the chosen sharing bound: without sharing (or with a
  // different bound) the best number of resident waves can differ.
  if (!st && best_tau != base_tau) {
    const int wpc0 = best_wpc;
    for (int wpc : wpcs) {
      if ((uint64_t)p->cus * wpc > p->max_waves || st || wpc == wpc0) continue;
      st = trial(wpc, best_tau, best_lds, ms);
      if (!st && ms < best) {
        best = ms;
        best_wpc = wpc;
      }
    }
  }
  if (!st && best_lds == 1) {
    st = trial(best_wpc, best_tau, 0, ms);
    if (!st && ms < best) {
      best = ms;
      best_lds = 0;
    }
  }
  (void)hipFree(d_sample);
  if (d_sruns) (void)hipFree(d_sruns);
  if (st) {
    set_config(p, base_wpc, base_tau, base_lds);
    return st;
  }
  set_config(p, best_wpc, best_tau, best_lds);
  if (out) {
    std::memset(out, 0, sizeof(*out));
    out->waves_per_cu = best_wpc;
    out->share_bound = best_tau;
    out->lds_tier = best_lds;
    out->trials = trials;
    out->best_ms = best;
    out->base_ms = base_ms;
    out->pack_slots = p->pack_slots;
    out->pack_waves_per_cu = (uint32_t)p->pack_wpc;
  }
  return MCE_OK;
}
}  // namespace

extern "C" {

mce_status mce_plan_create(const mce_graph *g, const mce_options *opt, mce_plan **out) {
  return guarded([&] {
    if (!g || !out) return fail(MCE_ERR_ARG, "null argument");
    mce_options o;
    mce_options_init(&o);
    if (opt) o = *opt;
    PlanSpec spec;
    spec.g = &g->g;
    return plan_create_impl(spec, o, out);
  });
}

mce_status mce_plan_run(mce_plan *p, mce_result **out) {
  return guarded([&] {
    if (!p || !out) return fail(MCE_ERR_ARG, "null argument");
    return plan_run_impl(p, out);
  });
}

mce_status mce_plan_autotune(mce_plan *p, uint64_t stride, mce_tune_result *out) {
  return guarded([&] {
    if (!p) return fail(MCE_ERR_ARG, "null plan");
    return autotune_impl(p, stride, out);
  });
}

void mce_plan_free(mce_plan *p) { plan_release(p); }

mce_status mce_plan_roots(const mce_graph *g, int32_t root_mode, uint64_t *out, uint64_t cap, uint64_t *count) {
  return guarded([&] {
    if (!g || !count) return fail(MCE_ERR_ARG, "null argument");
    std::vector<uint64_t> roots;
    uint64_t max_out;
    build_roots(g->g, root_mode == MCE_ROOT_VERTEX ? MCE_ROOT_VERTEX : MCE_ROOT_EDGE, roots, max_out);
    *count = roots.size();
    if (out) {
      if (cap < roots.size()) return fail(MCE_ERR_ARG, "root buffer too small");
      std::memcpy(out, roots.data(), roots.size() * 8);
    }
    return MCE_OK;
  });
}

mce_status mce_solve(const mce_graph *g, const mce_options *opt, mce_result **out) {
  return guarded([&] {
    if (!g || !out) return fail(MCE_ERR_ARG, "null argument");
    auto t0 = std::chrono::steady_clock::now();
    mce_plan *p = nullptr;
    mce_status s = mce_plan_create(g, opt, &p);
    if (s) return s;
    s = mce_plan_run(p, out);
    mce_plan_free(p);
    if (s == MCE_OK) (*out)->total_ms = ms_since(t0);
    return s;
  });
}

mce_status mce_solve_csr(uint64_t n, const uint64_t *rowoff, const uint32_t *col, const uint32_t *labels,
                         uint64_t degeneracy, const mce_options *opt, mce_result **out) {
  mce_graph *g = nullptr;
  mce_status s = mce_graph_from_csr(n, rowoff, col, labels, degeneracy, &g);
  if (s) return s;
  s = mce_solve(g, opt, out);
  mce_graph_free(g);
  return s;
}

void mce_result_free(mce_result *r) {
  if (!r) return;
  std::free(r->hist);
  std::free(r->list);
  std::free(r->root_nodes);
  std::free(r->root_cycles);
  delete r;
}

// ---------------------------------------------------------------------------
// Batches
// ---------------------------------------------------------------------------
mce_status mce_batch_create(const mce_graph *const *graphs, uint64_t count, const mce_options *opt,
                            mce_batch **out) {
  return guarded([&] {
    if (!graphs || !out || count == 0) return fail(MCE_ERR_ARG, "empty batch");
    mce_options o;
    mce_options_init(&o);
    if (opt) o = *opt;
    if (o.schedule == MCE_SCHED_CUSTOM && !o.roots) return fail(MCE_ERR_ARG, "custom schedule without a root list");
    if (o.want_list) return fail(MCE_ERR_UNSUPPORTED, "clique lists are per-graph solves only");
    // Concatenate: graph i's vertices become [vstart[i], vstart[i+1]).
    HostGraph cat;
    std::vector<uint64_t> vstart(count + 1, 0);
    uint64_t nnz = 0;
    for (uint64_t i = 0; i < count; ++i) {
      if (!graphs[i]) return fail(MCE_ERR_ARG, "null graph in batch");
      vstart[i + 1] = vstart[i] + graphs[i]->g.n;
      nnz += graphs[i]->g.col.size();
    }
    if (vstart[count] >= (1ull << 32)) return fail(MCE_ERR_UNSUPPORTED, "batch has more than 2^32-1 vertices");
    cat.n = vstart[count];
    cat.m = nnz / 2;
    cat.rowoff.resize(cat.n + 1);
    cat.col.resize(nnz);
    cat.labels.resize(cat.n);
    uint64_t at = 0;
    for (uint64_t i = 0; i < count; ++i) {
      const HostGraph &g = graphs[i]->g;
      const uint32_t base = (uint32_t)vstart[i];
      for (uint64_t v = 0; v < g.n; ++v) {
        cat.rowoff[base + v] = at + g.rowoff[v];
        cat.labels[base + v] = g.labels[v];
      }
      for (uint64_t k = 0; k < g.col.size(); ++k) cat.col[at + k] = g.col[k] + base;
      at += g.col.size();
      cat.max_degree = std::max(cat.max_degree, g.max_degree);
      cat.degeneracy = std::max(cat.degeneracy, g.degeneracy);
    }
    cat.rowoff[cat.n] = at;
    auto b = new mce_batch();
    PlanSpec spec;
    spec.g = &cat;
    spec.graph_vstart = &vstart;
    mce_status s = plan_create_impl(spec, o, &b->plan);
    if (s) {
      delete b;
      return s;
    }
    *out = b;
    return MCE_OK;
  });
}

mce_status mce_batch_run(mce_batch *b, mce_batch_result **out) {
  return guarded([&] {
    if (!b || !out) return fail(MCE_ERR_ARG, "null argument");
    auto t0 = std::chrono::steady_clock::now();
    mce_plan *p = b->plan;
    HIP_TRY(hipSetDevice(p->device));
    RunOut ro;
    mce_status st = run_core(p, make_args(p), true, ro);
    if (st) return st;
    auto r = new mce_batch_result();
    std::memset(r, 0, sizeof(*r));
    r->n_graphs = p->n_graphs;
    r->hist_stride = p->g_hist_stride;
    r->count = (uint64_t *)std::calloc(std::max<uint64_t>(p->n_graphs, 1), 8);
    r->hash = (uint64_t *)std::calloc(std::max<uint64_t>(p->n_graphs, 1), 8);
    r->hist = (uint64_t *)std::calloc(std::max<uint64_t>(p->n_graphs * p->g_hist_stride, 1), 8);
    hipError_t e = hipMemcpy(r->count, p->d_gcount, p->n_graphs * 8, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(r->hash, p->d_ghash, p->n_graphs * 8, hipMemcpyDeviceToHost);
    if (e == hipSuccess)
      e = hipMemcpy(r->hist, p->d_ghist, p->n_graphs * p->g_hist_stride * 8, hipMemcpyDeviceToHost);
    if (e != hipSuccess) {
      mce_batch_result_free(r);
      return fail(MCE_ERR_DEVICE, hipGetErrorString(e));
    }
    for (uint64_t i = 0; i < p->n_graphs; ++i) r->total_count += r->count[i];
    r->total_nodes = ro.ctr[kNodes];
    r->kernel_ms = ro.kernel_ms;
    r->total_ms = ms_since(t0);
    r->graph_replay = ro.replay ? 1 : 0;
    r->passes = ro.passes;
    *out = r;
    return MCE_OK;
  });
}

mce_status mce_batch_autotune(mce_batch *b, uint64_t stride, mce_tune_result *out) {
  return guarded([&] {
    if (!b) return fail(MCE_ERR_ARG, "null batch");
    return autotune_impl(b->plan, stride, out);
  });
}

void mce_batch_result_free(mce_batch_result *r) {
  if (!r) return;
  std::free(r->count);
  std::free(r->hash);
  std::free(r->hist);
  delete r;
}

void mce_batch_free(mce_batch *b) {
  if (!b) return;
  plan_release(b->plan);
  delete b;
}

}  // extern "C"
