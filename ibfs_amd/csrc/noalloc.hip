// Allocation-free traversal: one group of up to 128 sources with every
// scratch buffer (status snapshots, queues, control blocks, hub cache,
// changed flags, lane table, masks, edge counter) in one file-scope device
// array, and levels enqueued eight at a time on the null stream (direction
// decided on the device, the host reading the control blocks in between).  For callers that
// cannot allocate: code under HIP graph capture, tight serving loops,
// harnesses that forbid allocation.
#include <hip/hip_runtime.h>

#include <cstring>
#include <mutex>
#include <vector>

#include "common.h"
#include "graph_dev.h"
#include "kernels.h"

using namespace ibfs;

namespace {

// Limits of the scratch array (each GPU holds one copy until the process
// ends): up to 128 lanes (two status words), 2^18 vertices with an edge
// (R-MAT scale 18), 2^24 adjacency entries, the default hub cache (131,072
// hubs), 8 ring snapshots, top-down chunks of at least 2,048 edges.
constexpr int NA_W = 2;
constexpr int NA_K = 64 * NA_W;
constexpr int64_t NA_VT = int64_t(1) << 18;
constexpr int64_t NA_E = int64_t(1) << 24;
constexpr int64_t NA_H = 131072;
constexpr int NA_R = 8;       // at the vertex limit and 128 lanes; smaller graphs keep more
constexpr int NA_RMAX = 32;
constexpr int NA_MIN_CHUNK_SHIFT = 11;

constexpr size_t up256(size_t x) { return (x + 255) & ~size_t(255); }

// byte offsets of each buffer inside the array
constexpr size_t OFF_RING = 0;
constexpr size_t SZ_RING = size_t(NA_R) * NA_VT * NA_W * sizeof(u64);
constexpr size_t OFF_CTL = OFF_RING + up256(SZ_RING);
constexpr size_t SZ_CTL = ctl_ring_bytes(NA_RMAX);
constexpr size_t OFF_Q = OFF_CTL + up256(SZ_CTL);
constexpr size_t SZ_Q1 = up256(queue_entries(NA_VT) * sizeof(int32_t));
constexpr size_t OFF_CHUNKS = OFF_Q + (NQ - 1) * SZ_Q1;
constexpr size_t SZ_CHUNKS = chunk_entries(NA_VT, NA_E, NA_MIN_CHUNK_SHIFT) * sizeof(int2);
constexpr size_t OFF_HS = OFF_CHUNKS + up256(SZ_CHUNKS);
constexpr size_t SZ_HS = size_t(NA_H) * NA_W * sizeof(u64);
constexpr size_t OFF_FLAGS = OFF_HS + up256(SZ_HS);
constexpr size_t SZ_FLAGS = size_t(NA_VT);
constexpr size_t OFF_MASKS = OFF_FLAGS + up256(SZ_FLAGS);
constexpr size_t SZ_MASKS = size_t(2 + NA_RMAX + 1) * NA_W * sizeof(u64);
constexpr size_t OFF_LANES = OFF_MASKS + up256(SZ_MASKS);
constexpr size_t SZ_LANES = size_t(NA_K) * sizeof(LaneOut);
constexpr size_t OFF_COUNT = OFF_LANES + up256(SZ_LANES);
constexpr size_t NA_BYTES = OFF_COUNT + 256;
static_assert(NA_BYTES == IBFS_NOALLOC_SCRATCH_BYTES, "scratch size in ibfs.h");

// The scratch array.  In host code its name is a host-side stand-in, not a
// device address: host code uses only the per-device address from
// hipGetSymbolAddress (scratch_ptr below).
static __device__ __align__(256) unsigned char scratch[NA_BYTES];

std::mutex g_mu;  // one traversal at a time per process (the array is shared)
std::vector<unsigned char *> g_ptr;  // per device: the array's device address

// Device address of the scratch array on the current device `dev`, looked
// up once per device.
int scratch_ptr(int dev, unsigned char **out) {
  if ((size_t)dev >= g_ptr.size()) g_ptr.resize((size_t)dev + 1, nullptr);
  if (!g_ptr[(size_t)dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(IBFS_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev,
                  hipGetErrorString(e));
    g_ptr[(size_t)dev] = static_cast<unsigned char *>(p);
  }
  *out = g_ptr[(size_t)dev];
  return IBFS_OK;
}

#define NA_TRY(expr)                                                                   \
  do {                                                                                 \
    hipError_t _e = (expr);                                                            \
    if (_e != hipSuccess)                                                              \
      return fail(IBFS_ERR_HIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e), \
                  __FILE__, __LINE__);                                                 \
  } while (0)

// Waits for the null stream within the library's wait limit.
int wait_null_stream() {
  WaitClock clk;
  for (;;) {
    const hipError_t q = hipStreamQuery(nullptr);
    if (q == hipSuccess) return IBFS_OK;
    if (q != hipErrorNotReady) return fail(IBFS_ERR_HIP, "stream error: %s", hipGetErrorString(q));
    if (clk.expired())
      return fail(IBFS_ERR_STATE, "traversal did not finish within the wait limit (%.1f s)",
                  wait_timeout_s());
  }
}

int run(ibfs_graph_s *g, const ibfs_config &cfg, const int32_t *src, int k, int32_t *dout,
        int64_t *edges) {
  int dev = 0;
  NA_TRY(hipGetDevice(&dev));
  unsigned char *base = nullptr;
  if (int rc = scratch_ptr(dev, &base)) return rc;
  const int W = k <= 64 ? 1 : 2;
  const int64_t V = g->V, Vt = g->Vt;
  const int R = (int)std::min<int64_t>(
      NA_RMAX, (int64_t)(SZ_RING / sizeof(u64)) / std::max<int64_t>(Vt * W, 1));
  u64 *ring = reinterpret_cast<u64 *>(base + OFF_RING);
  LevelCtl *ctl = reinterpret_cast<LevelCtl *>(base + OFF_CTL);
  Queues q{};
  for (int i = 0, j = 0; i < NQ; ++i)
    if (i != Q_TD_L) q.q[i] = reinterpret_cast<int32_t *>(base + OFF_Q + (size_t)(j++) * SZ_Q1);
  q.chunks = reinterpret_cast<int2 *>(base + OFF_CHUNKS);
  u64 *hs = reinterpret_cast<u64 *>(base + OFF_HS);
  uint8_t *flags = base + OFF_FLAGS;
  u64 *masks = reinterpret_cast<u64 *>(base + OFF_MASKS);
  LaneOut *lanes = reinterpret_cast<LaneOut *>(base + OFF_LANES);
  u64 *count = reinterpret_cast<u64 *>(base + OFF_COUNT);
  const HubCut hc = hub_cut(g, cfg.hybrid_hubs);
  const GraphDev gd = graph_dev(g, cfg, hc);
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus <= 0)
    cus = 256;
  const int grid = cfg.dd_grid > 0 ? cfg.dd_grid : cus * 4;  // as the engine's levels enqueued ahead
  hipStream_t st = nullptr;  // the null stream: nothing to create

  // the previous call's contents stay in the array: clear what starts at zero
  SourceList sl;
  sl.k = k;
  int iso = 0;
  for (int i = 0; i < k; ++i) {
    sl.src[i] = src[i];
    iso |= g->h_cid[src[i]] < 0;
  }
  NA_TRY(launch_group_start(W, sl, g->d_cid, dout, V, Vt, ring, flags,
                            reinterpret_cast<u64 *>(ctl), (int64_t)(ctl_ring_bytes(R) / 8), lanes,
                            masks, R, count, st));
  CtlSpread *spread = ctl_spread(ctl, R);
  auto dec = [&](int L) {
    return Decide{2, L, cfg.policy, cfg.sw_level, cfg.alpha, cfg.beta, cfg.hybrid_gamma, hc.rho_q10,
                  (u64)V};
  };
  auto slot = [&](int L) { return ring + (int64_t)(L % R) * Vt * W; };
  auto inspect = [&](int L) {
    InspectArgs a{};
    a.full_diff = 1;
    a.prev = L > 0 ? slot(L - 1) : nullptr;
    a.cur = slot(L);
    a.next = slot(L + 1);
    a.ctl = ctl + L % R;
    a.ctl_zero = ctl + (L + 1) % R;
    a.ctl_prev = L > 0 ? ctl + (L - 1) % R : nullptr;
    a.lam_prev = L > 0 ? a.ctl_prev->lam : masks;
    a.dec = dec(L);
    a.deg = g->d_deg;
    a.V = Vt;
    a.q = q;
    a.sml = cfg.sml_shed;
    a.lrg = cfg.lrg_shed;
    a.chunk_shift = gd.chunk_shift;
    a.chunk_extra = (unsigned)(g->E >> gd.chunk_shift) + 1;
    a.hubs = g->d_hubs;
    a.H = g->H;
    a.hs = hs;
    a.flags = flags;
    a.vpt = cfg.inspect_vpt;
    a.nw = cfg.wg_size / 64;
    a.hsplit = gd.hsp;
    a.spread = spread + (L & 1);
    return launch_inspect(W, a, st);
  };
  auto expand = [&](int L) {
    NextArgs n{};
    n.dec = dec(L - 1);
    n.spread = spread + ((L - 1) & 1);
    n.spread_old = spread + (L & 1);
    n.ctl = ctl + (L - 1) % R;
    n.ctl_prev = L > 1 ? ctl + (L - 2) % R : nullptr;
    return launch_expand_next(W, gd, slot(L - 1), slot(L), hs, flags, n, q, grid, st);
  };
  NA_TRY(inspect(0));

  const EmitSpace sp{g->d_cid, V, Vt, g->d_deg};
  const int vec4 = (V % 4 == 0) && ((uintptr_t)dout % 16 == 0);
  int level = 1, lo = 0;  // next level to enqueue, base of the emission window
  for (;;) {
    int B = std::min(8, R - 1 - (level - lo));
    if (B < 1) {  // the next levels would overwrite S_lo: emit [lo, level-1]
      NA_TRY(launch_emit(W, cfg.emit_mode, vec4, ring, R, sp, lo, level - 1, lanes, masks + 2 * W,
                         masks + W, k, nullptr, iso, st));
      lo = level - 1;
      B = std::min(8, R - 1 - (level - lo));
    }
    for (int i = 0; i < B; ++i, ++level) {
      NA_TRY(expand(level));
      NA_TRY(inspect(level));
    }
    if (int rc = wait_null_stream()) return rc;
    // the expansion of level-1 folded the counters of level-2: whether a level
    // up to that one changed nothing, and the first that did
    LevelCtl h[NA_RMAX];
    NA_TRY(hipMemcpy(h, ctl, sizeof(LevelCtl) * (size_t)R, hipMemcpyDeviceToHost));
    if (h[(level - 2) % R].next_dir < 0) {
      int end = level - 2;
      while (end > 0 && end > level - 1 - B && h[(end - 1) % R].next_dir < 0) --end;
      const int last = end > 0 ? end - 1 : 0;
      if (last >= lo)
        NA_TRY(launch_emit(W, cfg.emit_mode, vec4, ring, R, sp, lo, last, lanes, masks + 2 * W,
                           masks + W, k, edges ? count : nullptr, iso, st));
      else if (edges)  // no final window: count over S_last
        NA_TRY(launch_count_edges(W, slot(last), g->d_deg, Vt, masks, count, st));
      if (int rc = wait_null_stream()) return rc;
      if (edges) {
        u64 c = 0;
        NA_TRY(hipMemcpy(&c, count, sizeof c, hipMemcpyDeviceToHost));
        // sources without a status word reach themselves, degree 0: nothing to add
        *edges = (int64_t)c;
      }
      return IBFS_OK;
    }
    if (level > Vt + 2 + B) return fail(IBFS_ERR_STATE, "traversal exceeded V+2 levels");
  }
}

}  // namespace

extern "C" {

int ibfs_traversal_noalloc(ibfs_graph_t g, const ibfs_config *cfg_in, const int32_t *src,
                           int32_t k, int32_t *depth_out, int64_t *traversed_edges) {
  if (!g) return fail(IBFS_ERR_ARG, "ibfs_traversal_noalloc: null graph");
  if (k < 1 || k > NA_K) return fail(IBFS_ERR_ARG, "k=%d outside [1, %d]", k, NA_K);
  if (!src || !depth_out) return fail(IBFS_ERR_ARG, "null sources or output");
  if (g->Vt > NA_VT || g->E > NA_E || g->H > NA_H)
    return fail(IBFS_ERR_ARG,
                "graph beyond the scratch limits: %lld vertices with an edge (max %lld), %lld "
                "adjacency entries (max %lld), %lld hubs (max %lld)",
                (long long)g->Vt, (long long)NA_VT, (long long)g->E, (long long)NA_E,
                (long long)g->H, (long long)NA_H);
  ibfs_config cfg;
  if (cfg_in) cfg = *cfg_in;
  else ibfs_config_default(&cfg);
  if (cfg.sml_shed < 1 || cfg.lrg_shed < cfg.sml_shed)
    return fail(IBFS_ERR_ARG, "need 1 <= sml_shed <= lrg_shed");
  if (int rc = check_direction_config(cfg)) return rc;
  if (cfg.td_chunk < (1 << NA_MIN_CHUNK_SHIFT) || (cfg.td_chunk & (cfg.td_chunk - 1)))
    return fail(IBFS_ERR_ARG, "td_chunk must be a power of two >= %d here (got %d)",
                1 << NA_MIN_CHUNK_SHIFT, cfg.td_chunk);
  if (cfg.emit_mode < 0 || cfg.emit_mode > 3) return fail(IBFS_ERR_ARG, "bad emit_mode");
  if (!valid_inspect_vpt(cfg.inspect_vpt)) return fail(IBFS_ERR_ARG, "bad inspect_vpt");
  if (!valid_wg_size(cfg.wg_size)) return fail(IBFS_ERR_ARG, "wg_size must be 256, 512 or 1024");
  const int64_t V = g->V;
  for (int i = 0; i < k; ++i)
    if (src[i] < 0 || src[i] >= V)
      return fail(IBFS_ERR_ARG, "source %d = %d out of range [0,%lld)", i, src[i], (long long)V);
  std::lock_guard<std::mutex> lk(g_mu);
  int cur = 0;
  NA_TRY(hipGetDevice(&cur));
  NA_TRY(hipSetDevice(g->device));
  HeadsUse heads;
  heads.take(g->heads);
  const int rc = run(g, cfg, src, k, depth_out, traversed_edges);
  (void)hipSetDevice(cur);
  return rc;
}

}  // extern "C"
