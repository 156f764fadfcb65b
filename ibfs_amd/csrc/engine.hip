// Engine: device graph, per-group traversal driver (level loop, direction
// switch, snapshot ring, depth emission) and GroupBy, behind the C ABI.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "common.h"
#include "graph_dev.h"
#include "host_copy.h"
#include "kernels.h"

using namespace ibfs;

#define HIP_TRY(expr)                                                                  \
  do {                                                                                 \
    hipError_t _e = (expr);                                                            \
    if (_e != hipSuccess)                                                              \
      return fail(IBFS_ERR_HIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e), \
                  __FILE__, __LINE__);                                                 \
  } while (0)

struct ibfs_engine_s {
  ibfs_graph_s *g = nullptr;
  ibfs_config cfg{};
  // K: lanes per group (lane_bits); W: status words per vertex of the current
  // traversal, the narrowest power of two that holds its sources (at most
  // Wmax = lane_bits / 64, which sizes the buffers)
  int K = 128, W = 2, Wmax = 2, R = 32, chunk_shift = 12;
  int hy_grid = 8192, next_grid = 8192;  // workgroups of a hybrid level, of one enqueued ahead
  HubCut hc;           // hubs a hybrid level pulls through
  HeadsUse heads;
  hipStream_t st = nullptr;
  hipEvent_t ev_wait = nullptr;  // behind a failed call's work (poll_stream)
  u64 *ring = nullptr;
  LevelCtl *d_ctl = nullptr;
  // coherent pinned: control blocks posted by the inspector (level l into
  // entry l % POSTS with tag post_seq base + l), the end of a group
  CtlPost *post = nullptr;
  GroupPost *post_end = nullptr;
  u64 post_seq = 0;
  Queues q{};
  u64 *d_masks = nullptr;     // [0,W) lanes_all, [W,2W) sel, [2W, 2W+(R+1)W) level masks
  LaneOut *d_lanes = nullptr;
  int32_t *d_out = nullptr;   // staging for host-placed output
  size_t d_out_cap = 0;
  u64 *d_count = nullptr;     // edges, start clock; work model at [2], [3]
  u64 *h_count = nullptr;     // work model, pinned
  double clock_khz = 1e5;     // of the device clock in d_count and post_end
  u64 *hs = nullptr;          // hub cache, H * W words
  uint8_t *flags = nullptr;   // changed-at-this-level byte per traversal vertex
  int emit_vec4 = 0;          // every lane output of this traversal is 16-byte aligned
  int iso = 0;                // some source of this traversal is isolated
  std::vector<ibfs_level_info> log;
  std::vector<hipEvent_t> ev;  // event pool
  size_t ev_used = 0;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> emit_ev;  // emission timings of a traversal
  // a traversal failed with work possibly still enqueued on st (a wait past
  // the limit): the next one drains it first, since its set-up rewrites the
  // pinned blocks that work may still copy into
  bool unsettled = false;
};

namespace {

constexpr int POSTS = 8;  // > levels enqueued ahead
// Levels enqueued ahead of the host, and the largest S_L (64-bit words) for
// it.  Waiting for the host costs 5 to 8 us a level; a fixed grid instead of
// one sized by the queues costs more once levels are long.  128 lanes, enqueued
// ahead against not: R-MAT s18 303 / 344 us, s20 (1.3M words) 666 / 676, s21
// (2.5M) 1,296 / 1,238, s22 1,993 / 1,923.
constexpr int AHEAD = 2;
constexpr int64_t AHEAD_WORDS = (int64_t)1 << 21;

size_t masks_words(const ibfs_engine_s *e) { return (size_t)(2 + (e->R + 1)) * e->W; }

// Waits for the work enqueued so far by polling an event recorded behind it
// (an earlier call's work after a failure; a group's levels and end are waited
// for on their posts).
// Past the wait limit (ibfs_set_wait_timeout) it fails with IBFS_ERR_STATE.
int poll_stream(hipStream_t st, hipEvent_t ev) {
  const hipError_t r = hipEventRecord(ev, st);
  if (r != hipSuccess) return fail(IBFS_ERR_HIP, "hipEventRecord: %s", hipGetErrorString(r));
  WaitClock clk;
  for (;;) {
    const hipError_t q = hipEventQuery(ev);
    if (q == hipSuccess) return IBFS_OK;
    if (q != hipErrorNotReady) return fail(IBFS_ERR_HIP, "stream error: %s", hipGetErrorString(q));
    if (clk.expired())
      return fail(IBFS_ERR_STATE, "group did not finish within the wait limit (%.1f s)",
                  wait_timeout_s());
  }
}

// Waits until *tag is seq (a spin; every 1,024 reads the stream is queried, so
// an error, or an idle stream without the tag, ends the wait with an error).
int wait_tag(hipStream_t st, const u64 *tag, u64 seq, const char *what) {
  WaitClock clk;
  for (unsigned i = 1;; ++i) {
    if (__atomic_load_n(tag, __ATOMIC_ACQUIRE) == seq) return IBFS_OK;
    if ((i & 1023) == 0) {
      const hipError_t q = hipStreamQuery(st);
      if (q == hipErrorNotReady) {
        if (clk.expired())
          return fail(IBFS_ERR_STATE, "%s did not finish within the wait limit (%.1f s)", what,
                      wait_timeout_s());
        continue;
      }
      if (q != hipSuccess) return fail(IBFS_ERR_HIP, "stream error: %s", hipGetErrorString(q));
      if (__atomic_load_n(tag, __ATOMIC_ACQUIRE) == seq) return IBFS_OK;
      return fail(IBFS_ERR_STATE, "%s: post did not arrive", what);
    }
  }
}

// Elapsed time between two events the device has passed.  A posted control
// block can reach the host before the runtime has seen the completion of the
// events enqueued ahead of it, so each is queried until it reports completion.
// Past the wait limit it returns hipErrorNotReady (reported by HIP_TRY).
hipError_t elapsed_ms(float *ms, hipEvent_t a, hipEvent_t b) {
  for (hipEvent_t x : {a, b}) {
    hipError_t q;
    WaitClock clk;
    while ((q = hipEventQuery(x)) == hipErrorNotReady) {
      if (clk.expired()) return hipErrorNotReady;
    }
    if (q != hipSuccess) return q;
  }
  return hipEventElapsedTime(ms, a, b);
}

hipEvent_t next_event(ibfs_engine_s *e) {
  if (e->ev_used == e->ev.size()) {
    hipEvent_t x;
    if (hipEventCreate(&x) != hipSuccess) return nullptr;
    e->ev.push_back(x);
  }
  return e->ev[e->ev_used++];
}

int check_device(int dev) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= 0)
    return fail(IBFS_ERR_NODEVICE, "no HIP device available");
  if (dev < 0 || dev >= n) return fail(IBFS_ERR_ARG, "device %d out of range [0,%d)", dev, n);
  if (hipSetDevice(dev) != hipSuccess) return fail(IBFS_ERR_HIP, "hipSetDevice(%d) failed", dev);
  return IBFS_OK;
}

// One non-blocking stream per device for the library's synchronous copies
// (created on first use, kept until the process ends).
int copy_stream(int dev, hipStream_t *out) {
  static std::mutex mu;
  static std::vector<hipStream_t> streams;
  std::lock_guard<std::mutex> lk(mu);
  if (dev < 0) return fail(IBFS_ERR_ARG, "bad device %d", dev);
  if ((size_t)dev >= streams.size()) streams.resize((size_t)dev + 1, nullptr);
  if (!streams[(size_t)dev]) {
    int cur = 0;
    HIP_TRY(hipGetDevice(&cur));
    HIP_TRY(hipSetDevice(dev));
    const hipError_t r = hipStreamCreateWithFlags(&streams[(size_t)dev], hipStreamNonBlocking);
    (void)hipSetDevice(cur);
    if (r != hipSuccess) {
      streams[(size_t)dev] = nullptr;
      return fail(IBFS_ERR_HIP, "copy stream: %s", hipGetErrorString(r));
    }
  }
  *out = streams[(size_t)dev];
  return IBFS_OK;
}

template <class T>
void dfree(T *&p) {
  if (p) (void)hipFree((void *)p);
  p = nullptr;
}

template <class T>
void hfree(T *&p) {
  if (p) (void)hipHostFree((void *)p);
  p = nullptr;
}

void engine_release(ibfs_engine_s *e) {
  if (!e) return;
  if (e->g) (void)hipSetDevice(e->g->device);
  if (e->st) (void)hipStreamSynchronize(e->st);
  dfree(e->ring);
  dfree(e->d_ctl);
  hfree(e->post);
  hfree(e->post_end);
  for (int i = 0; i < NQ; ++i) dfree(e->q.q[i]);
  dfree(e->q.chunks);
  dfree(e->d_masks);
  dfree(e->d_lanes);
  dfree(e->d_out);
  dfree(e->d_count);
  hfree(e->h_count);
  dfree(e->hs);
  dfree(e->flags);
  for (auto x : e->ev) (void)hipEventDestroy(x);
  e->ev.clear();
  if (e->ev_wait) (void)hipEventDestroy(e->ev_wait);
  e->ev_wait = nullptr;
  if (e->st) (void)hipStreamDestroy(e->st);
  e->st = nullptr;
}

// The engine's stream, event and buffers, for its settings.
hipError_t engine_alloc(ibfs_engine_s *e) {
  const ibfs_graph_s *g = e->g;
  const int64_t Vt = std::max<int64_t>(g->Vt, 1);
  hipError_t err = hipStreamCreateWithFlags(&e->st, hipStreamNonBlocking);
  if (err == hipSuccess) err = hipEventCreateWithFlags(&e->ev_wait, hipEventDisableTiming);
  auto A = [&](void **p, size_t bytes) {
    if (err == hipSuccess) err = hipMalloc(p, bytes ? bytes : 1);
  };
  auto H = [&](void **p, size_t bytes) {
    if (err == hipSuccess) err = hipHostMalloc(p, bytes ? bytes : 1, hipHostMallocDefault);
  };
  A((void **)&e->ring, (size_t)e->R * (size_t)Vt * (size_t)e->W * sizeof(u64));
  A((void **)&e->d_ctl, ctl_ring_bytes(e->R));
  if (err == hipSuccess) err = hipHostMalloc((void **)&e->post, POSTS * sizeof(CtlPost), hipHostMallocCoherent);
  if (err == hipSuccess) std::memset(e->post, 0, POSTS * sizeof(CtlPost));
  if (err == hipSuccess) err = hipHostMalloc((void **)&e->post_end, sizeof(GroupPost), hipHostMallocCoherent);
  if (err == hipSuccess) std::memset(e->post_end, 0, sizeof(GroupPost));
  for (int i = 0; i < NQ; ++i)
    if (i != Q_TD_L) A((void **)&e->q.q[i], sizeof(int32_t) * queue_entries((size_t)Vt));
  A((void **)&e->q.chunks, sizeof(int2) * chunk_entries((size_t)Vt, (size_t)g->E, e->chunk_shift));
  A((void **)&e->d_masks, sizeof(u64) * masks_words(e));
  A((void **)&e->d_lanes, sizeof(LaneOut) * (size_t)e->K);
  A((void **)&e->hs, sizeof(u64) * (size_t)e->W * (size_t)std::max<int64_t>(g->H, 1));
  A((void **)&e->flags, sizeof(u64) * (size_t)((Vt + 7) / 8));
  A((void **)&e->d_count, 4 * sizeof(u64));
  H((void **)&e->h_count, 4 * sizeof(u64));
  return err;
}

u64 *slot(ibfs_engine_s *e, int L) {
  return e->ring + (size_t)(L % e->R) * (size_t)e->g->Vt * (size_t)e->W;
}

EmitSpace emit_space(const ibfs_graph_s *g) { return EmitSpace{g->d_cid, g->V, g->Vt, g->d_deg}; }

// Distinct sources without a status word (isolated vertices): they change
// at their admission level like any source, but outside the status words.
int64_t isolated_sources(const ibfs_graph_s *g, const int32_t *src, int k) {
  std::vector<int32_t> iso;
  for (int i = 0; i < k; ++i)
    if (g->h_cid[src[i]] < 0) iso.push_back(src[i]);
  std::sort(iso.begin(), iso.end());
  return (int64_t)(std::unique(iso.begin(), iso.end()) - iso.begin());
}

// Arguments of the inspection of level L (the pass also refreshes the hub
// cache from S_L for the next bottom-up level).  With `on` 1 it decides level
// L+1 into its control block and posts that with tag `tag` (Decide::on).
InspectArgs inspect_args(ibfs_engine_s *e, int L, int on, u64 tag) {
  const ibfs_config &k = e->cfg;
  InspectArgs a{};
  a.full_diff = 1;  // of level 0; later levels derive it
  a.prev = L > 0 ? slot(e, L - 1) : nullptr;
  a.cur = slot(e, L);
  a.next = slot(e, L + 1);
  a.ctl = &e->d_ctl[L % e->R];
  a.ctl_zero = &e->d_ctl[(L + 1) % e->R];
  a.ctl_prev = L > 0 ? &e->d_ctl[(L - 1) % e->R] : nullptr;
  a.lam_prev = L > 0 ? a.ctl_prev->lam : e->d_masks;
  a.dec = Decide{on, L, k.policy, k.sw_level, k.alpha, k.beta, k.hybrid_gamma, e->hc.rho_q10,
                 (u64)e->g->V};
  a.deg = e->g->d_deg;
  a.V = e->g->Vt;
  a.q = e->q;
  a.sml = e->cfg.sml_shed;
  a.lrg = e->cfg.lrg_shed;
  a.chunk_shift = e->chunk_shift;
  a.chunk_extra = (unsigned)(e->g->E >> e->chunk_shift) + 1;
  a.hubs = e->g->d_hubs;
  a.H = e->g->H;
  a.hs = e->hs;
  a.flags = e->flags;
  a.vpt = e->cfg.inspect_vpt;
  a.nw = e->cfg.wg_size / 64;
  a.hsplit = hub_split(e->hc);
  a.spread = ctl_spread(e->d_ctl, e->R) + (on == 2 ? L & 1 : 0);
  if (on == 1) {
    a.post = &e->post[L % POSTS];
    a.post_tag = tag;
  }
  return a;
}

// Emits the window [b, en] for the group's lanes.
// edges (final window only, or null): the pass also adds the TEPS numerator.
int emit_window(ibfs_engine_s *e, int b, int en, int k, ibfs_stats *stats, u64 *edges) {
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (e->cfg.kernel_timing) {
    e0 = next_event(e);
    HIP_TRY(hipEventRecord(e0, e->st));
  }
  HIP_TRY(launch_emit(e->W, e->cfg.emit_mode, e->emit_vec4, e->ring, e->R, emit_space(e->g), b,
                      en, e->d_lanes, e->d_masks + 2 * e->W, e->d_masks + e->W, k, edges,
                      e->iso, e->st));
  if (e->cfg.kernel_timing) {
    e1 = next_event(e);
    HIP_TRY(hipEventRecord(e1, e->st));
    e->emit_ev.emplace_back(e0, e1);  // read after the traversal's last wait
  }
  if (stats) stats->n_emit_launches++;
  return IBFS_OK;
}

// One group of k sources (lanes 0..k-1), depths into dout (device, k*V).
//
// The host enqueues `ahead` levels beyond the last one whose control block it
// has read: expansions take their direction on the device from the counters
// of the level before, and once a level has changed nothing the kernels of
// later ones return at once.  The device then does not wait for the host
// between levels, and the levels enqueued too many cost about 5 us each at the
// end.  ahead 0 (kernel events, work model, and graphs whose levels are long:
// AHEAD_WORDS) launches the direction's own kernel, sized by the counters that
// the host has read.
int traverse(ibfs_engine_s *e, const int32_t *src, int k, int32_t *dout, ibfs_stats *stats) {
  ibfs_graph_s *g = e->g;
  const int64_t V = g->V, Vt = g->Vt;
  // a partial group streams only the status words its lanes need
  e->W = 1;
  while (e->W * 64 < k && e->W < e->Wmax) e->W *= 2;
  const int W = e->W;
  const GraphDev gd = graph_dev(g, e->cfg, e->hc);
  e->ev_used = 0;
  e->emit_ev.clear();
  e->log.clear();
  clear_hip_error();
  const bool timing = e->cfg.kernel_timing != 0;
  const bool small = Vt * W <= AHEAD_WORDS;
  const int ahead = (timing || e->cfg.work_model || !small) ? 0 : AHEAD;

  SourceList sl;
  sl.k = k;
  e->iso = 0;
  for (int i = 0; i < k; ++i) {
    sl.src[i] = src[i];
    e->iso |= g->h_cid[src[i]] < 0;
  }
  e->emit_vec4 = (V % 4 == 0) && ((uintptr_t)dout % 16 == 0);
  // level 0: S_0 = source bits; inspection builds the level-1 queues
  HIP_TRY(launch_group_start(W, sl, g->d_cid, dout, V, Vt, slot(e, 0), e->flags,
                             reinterpret_cast<u64 *>(e->d_ctl), (int64_t)(ctl_ring_bytes(e->R) / 8),
                             e->d_lanes, e->d_masks, e->R, e->d_count, e->st));
  const u64 seq0 = e->post_seq + 1;  // tag of level 0

  // events of the level in flight (timing only)
  hipEvent_t x0 = nullptr, x1 = nullptr, y0 = nullptr, y1 = nullptr;
  auto mark = [&](hipEvent_t *x) -> hipError_t {
    *x = next_event(e);
    return hipEventRecord(*x, e->st);
  };
  auto inspect = [&](int L) -> hipError_t {
    e->post_seq = seq0 + (u64)L;
    return launch_inspect(W, inspect_args(e, L, ahead ? 2 : 1, e->post_seq), e->st);
  };
  if (timing) HIP_TRY(mark(&y0));
  HIP_TRY(inspect(0));
  if (timing) HIP_TRY(mark(&y1));

  int known = -1, dir = -1;  // last level whose block was read, and its direction
  LevelCtl c{};              // that block
  // Reads the control block of level known+1: counters, level log.
  auto learn = [&]() -> int {
    const int l = known + 1;
    const CtlPost *p = &e->post[l % POSTS];
    if (int rc = wait_tag(e->st, &p->tag, seq0 + (u64)l, "level")) return rc;
    if (l > 0) dir = c.next_dir;
    std::memcpy(&c, &p->c, sizeof c);
    known = l;
    float ems = 0, ims = 0;
    if (timing) {
      if (l > 0) HIP_TRY(elapsed_ms(&ems, x0, x1));
      HIP_TRY(elapsed_ms(&ims, y0, y1));
    }
    if (stats) {
      stats->n_inspect_launches++;
      stats->inspect_ms += ims;
      if (l > 0) {
        (dir == 0 ? stats->n_td_launches : dir == 2 ? stats->n_hy_launches : stats->n_bu_launches)++;
        (dir == 0 ? stats->expand_td_ms : dir == 2 ? stats->expand_hy_ms : stats->expand_bu_ms) += ems;
      }
    }
    ibfs_level_info li{};
    li.level = l;
    li.direction = l > 0 ? dir : -1;
    li.n_changed = (int64_t)c.n_changed + (l == 0 ? isolated_sources(g, src, k) : 0);
    li.n_frontier = (int64_t)c.n_front;
    li.m_frontier = (int64_t)c.m_front;
    li.n_unvisited = (int64_t)c.n_cand;
    li.m_unvisited = (int64_t)c.m_cand;
    for (int i = 0; i < 3; ++i) {
      li.q_td[i] = c.q[i];
      li.q_bu[i] = c.cls[i];
    }
    li.expand_ms = ems;
    li.inspect_ms = ims;
    li.m_frontier_nonhub = (int64_t)c.m_front_nh;
    if (e->cfg.work_model && dir == 1) {
      li.bu_work = (int64_t)e->h_count[0];
      li.bu_prefix = (int64_t)e->h_count[1];
    }
    e->log.push_back(li);
    return IBFS_OK;
  };

  int base = 0;
  for (int L = 1;; ++L) {
    auto learn_to = [&](int l) -> int {
      while (known < l && !(known >= 0 && c.n_changed == 0))
        if (int rc = learn()) return rc;
      return IBFS_OK;
    };
    if (int rc = learn_to(L - 1 - ahead)) return rc;
    if (known >= 0 && c.n_changed == 0) break;
    if (L > 1 << 20) return fail(IBFS_ERR_STATE, "level limit exceeded");
    const LevelCtl *cp = e->d_ctl + (L - 1) % e->R;
    if (timing) HIP_TRY(mark(&x0));
    if (ahead) {
      CtlSpread *sp = ctl_spread(e->d_ctl, e->R);
      NextArgs n;
      n.dec = inspect_args(e, L - 1, 2, 0).dec;
      n.spread = sp + ((L - 1) & 1);
      n.spread_old = sp + (L & 1);
      n.ctl = e->d_ctl + (L - 1) % e->R;
      n.ctl_prev = L > 1 ? e->d_ctl + (L - 2) % e->R : nullptr;
      n.post = &e->post[(L - 1) % POSTS];
      n.post_tag = seq0 + (u64)(L - 1);
      HIP_TRY(launch_expand_next(W, gd, slot(e, L - 1), slot(e, L), e->hs, e->flags, n, e->q,
                                 e->next_grid, e->st));
    } else if (c.next_dir == 0) {
      HIP_TRY(launch_expand_td(W, gd, slot(e, L - 1), slot(e, L), cp, e->q, c.q[Q_TD_S],
                               c.q[Q_TD_M], c.q[Q_TD_L], c.next_flag ? e->flags : nullptr, e->st));
    } else if (c.next_dir == 2) {
      HIP_TRY(launch_expand_hy(W, gd, slot(e, L - 1), e->hs, slot(e, L), cp, e->q, e->hy_grid,
                               e->st));
    } else {
      if (e->cfg.work_model) {  // instrumentation: exact early-termination prefixes
        HIP_TRY(hipMemsetAsync(e->d_count + 2, 0, 2 * sizeof(u64), e->st));
        HIP_TRY(launch_bu_model(W, g->d_beg, g->d_tadj, slot(e, L - 1), e->hs, cp->lam, Vt,
                                e->d_count + 2, e->st));
        HIP_TRY(hipMemcpyAsync(e->h_count, e->d_count + 2, 2 * sizeof(u64), hipMemcpyDeviceToHost,
                               e->st));
        if (timing) HIP_TRY(hipEventRecord(x0, e->st));
      }
      HIP_TRY(launch_expand_bu(W, gd, slot(e, L - 1), e->hs, slot(e, L), e->flags, cp, e->q,
                               c.bu_queued ? (int64_t)c.q[Q_BU] : Vt, (int)c.bu_queued, e->st));
    }
    if (timing) HIP_TRY(mark(&x1));
    // the inspection's start event is the expansion's end event unless a
    // window flush runs in between
    y0 = x1;
    if ((L + 1) - base >= e->R) {  // the next copy would overwrite S_base
      // a level that is known to run (a no-op for ahead 0)
      int rc = learn_to(L - 1);
      if (rc) return rc;
      if (c.n_changed == 0) break;
      rc = emit_window(e, base, L, k, stats, nullptr);
      if (rc) return rc;
      if (stats) stats->emit_windows++;
      base = L;
      if (timing) HIP_TRY(mark(&y0));
    }
    HIP_TRY(inspect(L));
    if (timing) HIP_TRY(mark(&y1));
  }
  const int last = known > 0 ? known - 1 : 0;
  // the final window also counts the TEPS numerator (over S_last, which its
  // pass reads anyway)
  if (last >= base) {
    int rc = emit_window(e, base, last, k, stats, stats ? e->d_count : nullptr);
    if (rc) return rc;
    if (stats) stats->emit_windows++;
  } else if (stats) {  // no final window (the last flush ended at last + 1)
    HIP_TRY(launch_count_edges(W, slot(e, last), g->d_deg, Vt, e->d_masks, e->d_count, e->st));
  }
  // one wait for the group, on its end
  const u64 end = ++e->post_seq;
  HIP_TRY(launch_group_end(e->d_count, e->post_end, end, e->st));
  if (int rc = wait_tag(e->st, &e->post_end->tag, end, "group")) return rc;
  if (stats) {
    stats->total_ms += (double)(e->post_end->t1 - e->post_end->t0) / e->clock_khz;
    for (const auto &x : e->emit_ev) {
      float ms = 0;
      HIP_TRY(elapsed_ms(&ms, x.first, x.second));
      stats->emit_ms += ms;
    }
    stats->levels = std::max(stats->levels, last + 1);
    stats->traversed_edges += (int64_t)e->post_end->edges;
  }
  return IBFS_OK;
}

int ensure_out(ibfs_engine_s *e, size_t elems) {
  if (e->d_out_cap >= elems) return IBFS_OK;
  dfree(e->d_out);
  e->d_out_cap = 0;
  hipError_t err = hipMalloc((void **)&e->d_out, elems * sizeof(int32_t));
  if (err == hipErrorOutOfMemory && e->heads.drop())
    err = hipMalloc((void **)&e->d_out, elems * sizeof(int32_t));
  HIP_TRY(err);
  e->d_out_cap = elems;
  return IBFS_OK;
}

// The device's GroupBy workspaces (null without host memory for them: GroupBy
// then takes the form of large source sets).
std::shared_ptr<GroupbyPool> groupby_pool(int device) {
  static std::mutex mu;
  static std::vector<std::weak_ptr<GroupbyPool>> of;
  try {
    std::lock_guard<std::mutex> lk(mu);
    if ((size_t)device >= of.size()) of.resize((size_t)device + 1);
    auto w = of[(size_t)device].lock();
    if (!w) of[(size_t)device] = w = std::make_shared<GroupbyPool>();
    return w;
  } catch (...) {
    return nullptr;
  }
}

// A workspace for one call, in *out.
int groupby_take(GroupbyPool &p, GroupbyWork **out) {
  for (WaitClock clk;;) {
    {
      std::lock_guard<std::mutex> lk(p.mu);
      for (GroupbyWork **at = &p.late; *at;) {
        GroupbyWork *w = *at;
        if (hipStreamQuery((hipStream_t)w->st) == hipSuccess) {
          *at = w->next;
          --p.n_late;
          w->next = p.idle;
          p.idle = w;
          ++p.n_idle;
        } else {
          at = &w->next;
        }
      }
      if (p.idle) {
        *out = p.idle;
        p.idle = p.idle->next;
        --p.n_idle;
        return IBFS_OK;
      }
      if (p.n_late < GroupbyPool::KEEP) break;
    }
    if (clk.expired())
      return fail(IBFS_ERR_STATE, "groupby: earlier calls did not finish within the wait limit (%.1f s)",
                  wait_timeout_s());
  }
  GroupbyWork *w = new (std::nothrow) GroupbyWork();
  if (!w) return fail(IBFS_ERR_NOMEM, "groupby workspace");
  hipStream_t st = nullptr;
  hipError_t err = hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
  w->st = st;
  if (err == hipSuccess) err = hipHostMalloc(&w->post, sizeof(GroupbyPost), hipHostMallocCoherent);
  if (err == hipSuccess) err = hipMalloc((void **)&w->comp, sizeof(u64) * (GROUPBY_WORDS + 1));
  if (err == hipSuccess) err = launch_fill_u64(w->comp + GROUPBY_WORDS, 1, 0ull, st);
  if (err != hipSuccess) {
    delete w;
    return fail(err == hipErrorOutOfMemory ? IBFS_ERR_NOMEM : IBFS_ERR_HIP,
                "groupby workspace: %s", hipGetErrorString(err));
  }
  std::memset(w->post, 0, sizeof(GroupbyPost));
  w->ticket = w->comp + GROUPBY_WORDS;
  *out = w;
  return IBFS_OK;
}

// Gives a workspace back; of (or null): the graph that its kernel may still read.
void groupby_put(GroupbyPool &p, GroupbyWork *w, const void *of) {
  w->graph = of;
  {
    std::lock_guard<std::mutex> lk(p.mu);
    if (of || p.n_idle < GroupbyPool::KEEP) {
      GroupbyWork *&list = of ? p.late : p.idle;
      w->next = list;
      list = w;
      ++(of ? p.n_late : p.n_idle);
      return;
    }
  }
  delete w;  // more calls at once than are kept
}

}  // namespace

ibfs::GroupbyWork::~GroupbyWork() {
  if (st) {
    (void)hipStreamSynchronize((hipStream_t)st);
    (void)hipStreamDestroy((hipStream_t)st);
  }
  if (post) (void)hipHostFree(post);
  if (comp) (void)hipFree(comp);
}

ibfs::GroupbyPool::~GroupbyPool() {
  for (GroupbyWork *list : {idle, late})
    while (list) {
      GroupbyWork *w = list;
      list = w->next;
      delete w;
    }
}

ibfs::HeadsUse::~HeadsUse() {
  if (!h_) return;
  std::lock_guard<std::mutex> lk(h_->mu);
  --h_->users;
}

void ibfs::HeadsUse::take(const std::shared_ptr<GraphHeads> &h) {
  h_ = h;
  std::lock_guard<std::mutex> lk(h_->mu);
  ++h_->users;
}

bool ibfs::HeadsUse::drop() {
  std::lock_guard<std::mutex> lk(h_->mu);
  if (!h_->d || h_->users > 1) return false;
  dfree(h_->d);
  clear_hip_error();
  return true;
}

HubCut hub_cut(const ibfs_graph_s *g, int64_t r) {
  HubCut c;
  const int64_t H = g->H;
  if (r <= 0 || r > H) r = H;
  c.cut = (int32_t)r;
  if (r > 0) {
    c.deg = g->h_hub_deg[(size_t)r - 1];
    c.tie = g->h_hub_id[(size_t)r - 1];
  }
  c.rho_q10 = g->E > 0 ? (int32_t)((g->h_hub_entries[(size_t)r] * 1024) / g->E) : 0;
  return c;
}

extern "C" {

int ibfs_config_default(ibfs_config *cfg) {
  if (!cfg) return fail(IBFS_ERR_ARG, "null config");
  std::memset(cfg, 0, sizeof *cfg);
  cfg->lane_bits = 128;
  // wave64: a top-down vertex with fewer than 64 edges would leave lanes of its
  // wave idle, so it takes a row of 16 lanes (the reference's 32 matches a
  // 32-wide warp)
  cfg->sml_shed = 64;
  cfg->lrg_shed = 512;
  cfg->policy = IBFS_POLICY_ALPHA_BETA;
  cfg->sw_level = 2;
  // With 128 concurrent lanes a bottom-up vertex rarely covers every active
  // lane early, so top-down stays cheaper far longer than for one source:
  // switch when the frontier's edges exceed half of the candidates' edges.
  cfg->alpha = 2;
  cfg->beta = 48;
  // A top-down level whose frontier edges mostly leave the top 4,096 hubs
  // runs hybrid: the candidates pull through those hubs (a pulled entry
  // costs about a quarter of a pushed edge), the rest of the frontier pushes.
  // Measured on R-MAT s22: plain 7.5K -> 7.85K GTEPS (128 lanes), batched
  // 9.7K -> 10.4K.
  cfg->hybrid_gamma = 16;
  cfg->hybrid_hubs = 4096;
  // batched runs group sources by two-hop size: lanes that start slowly (a
  // degree-1 source next to low-degree vertices) no longer keep every
  // bottom-up candidate of a fast group scanning its whole list (R-MAT s22,
  // 256 lanes x 2 contexts: 10.3K -> 11.7K GTEPS)
  cfg->pack_sources = 1;
  cfg->split_cov = 0;
  cfg->phase_offsets = 0;
  // batched runs: the last levels (frontier under V/32 vertices and E/32
  // edges) run as sparse tail levels (R-MAT s22, 1,024 sources in 256-lane
  // groups: 10.23 -> 10.00 ms per batch)
  cfg->tail_div = 32;
  cfg->wg_size = 512;
  cfg->td_chunk = 2048;
  cfg->ring_levels = 32;
  cfg->kernel_timing = 0;
  cfg->device = 0;
  cfg->emit_mode = 0;
  return IBFS_OK;
}

int ibfs_device_count(int *n) {
  if (!n) return fail(IBFS_ERR_ARG, "null argument");
  int c = 0;
  if (hipGetDeviceCount(&c) != hipSuccess) c = 0;
  *n = c;
  return IBFS_OK;
}

int ibfs_device_alloc(int device, size_t bytes, void **dptr) {
  if (!dptr) return fail(IBFS_ERR_ARG, "null argument");
  int rc = check_device(device);
  if (rc) return rc;
  if (hipMalloc(dptr, bytes ? bytes : 1) != hipSuccess)
    return fail(IBFS_ERR_NOMEM, "hipMalloc(%zu) failed", bytes);
  return IBFS_OK;
}

int ibfs_device_free(void *dptr) {
  if (dptr) HIP_TRY(hipFree(dptr));
  return IBFS_OK;
}

int ibfs_memcpy_d2h(void *dst, const void *src, size_t bytes) {
  if (bytes && (!dst || !src)) return fail(IBFS_ERR_ARG, "ibfs_memcpy_d2h: null pointer");
  if (!bytes) return IBFS_OK;
  // on a library stream of the source's device, as ibfs_memcpy_d2d
  hipPointerAttribute_t pa{};
  HIP_TRY(hipPointerGetAttributes(&pa, src));
  int cur = 0;
  HIP_TRY(hipGetDevice(&cur));
  const int dev = pa.device >= 0 ? pa.device : cur;
  hipStream_t st = nullptr;
  if (int rc = copy_stream(dev, &st)) return rc;
  HIP_TRY(hipSetDevice(dev));
  const D2HPiece pc{dst, src, bytes};
  const int rc = copy_to_host(&pc, 1, st);
  (void)hipSetDevice(cur);
  return rc;
}

int ibfs_memcpy_h2d(void *dst, const void *src, size_t bytes) {
  HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
  return IBFS_OK;
}

int ibfs_memcpy_d2d(void *dst, const void *src, size_t bytes) {
  if (bytes && (!dst || !src)) return fail(IBFS_ERR_ARG, "null device pointer");
  if (!bytes) return IBFS_OK;
  // on a library stream of the destination's device, waiting for that
  // stream only: engines, batches and servers on the device keep running
  hipPointerAttribute_t pa{};
  HIP_TRY(hipPointerGetAttributes(&pa, dst));
  int dev = pa.device;
  if (dev < 0) HIP_TRY(hipGetDevice(&dev));
  hipStream_t st = nullptr;
  if (int rc = copy_stream(dev, &st)) return rc;
  HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, st));
  HIP_TRY(hipStreamSynchronize(st));
  return IBFS_OK;
}

int ibfs_graph_opts_default(ibfs_graph_opts *o) {
  if (!o) return fail(IBFS_ERR_ARG, "null options");
  std::memset(o, 0, sizeof *o);
  o->hub_count = 131072;
  o->nthreads = 0;
  return IBFS_OK;
}

int ibfs_graph_create(const int64_t *beg, int64_t V, const int32_t *adj, int64_t E, int device,
                      ibfs_graph_t *out) {
  return ibfs_graph_create_ex(beg, V, adj, E, device, nullptr, out);
}

int ibfs_graph_create_ex(const int64_t *beg, int64_t V, const int32_t *adj, int64_t E, int device,
                         const ibfs_graph_opts *opts_in, ibfs_graph_t *out) {
  ibfs_graph_opts opts;
  if (opts_in) opts = *opts_in;
  else ibfs_graph_opts_default(&opts);
  if (opts.hub_count < 0) return fail(IBFS_ERR_ARG, "hub_count must be >= 0");
  if (!out || !beg || V < 1 || E < 0 || (E > 0 && !adj))
    return fail(IBFS_ERR_ARG, "ibfs_graph_create: bad arguments (V=%lld, E=%lld)", (long long)V,
                (long long)E);
  if (V > 0x7fffffffLL) return fail(IBFS_ERR_ARG, "vertex count exceeds int32 ids");
  if (beg[0] != 0 || beg[V] != E)
    return fail(IBFS_ERR_FORMAT, "beg_pos[0]=%lld, beg_pos[V]=%lld, expected 0 and %lld",
                (long long)beg[0], (long long)beg[V], (long long)E);
  std::vector<int32_t> deg((size_t)V);
  int64_t maxd = 0;
  for (int64_t v = 0; v < V; ++v) {
    const int64_t d = beg[v + 1] - beg[v];
    if (d < 0) return fail(IBFS_ERR_FORMAT, "beg_pos decreases at vertex %lld", (long long)v);
    if (d > 0x7fffffffLL) return fail(IBFS_ERR_FORMAT, "degree exceeds int32");
    deg[v] = (int32_t)d;
    maxd = std::max(maxd, d);
  }
  for (int64_t i = 0; i < E; ++i)
    if (adj[i] < 0 || adj[i] >= V)
      return fail(IBFS_ERR_FORMAT, "adjacency entry %lld = %d out of range", (long long)i, adj[i]);
  int rc = check_device(device);
  if (rc) return rc;
  int nthreads = opts.nthreads > 0 ? opts.nthreads : (int)std::thread::hardware_concurrency();
  nthreads = std::max(1, std::min(nthreads, 64));
  // Traversal vertex space: vertices with an out- or in-edge, original order.
  std::vector<uint8_t> has_in((size_t)V, 0);
  struct MarkCtx {
    const int32_t *adj;
    uint8_t *has_in;
    int64_t E;
    int nt;
  } mx{adj, has_in.data(), E, nthreads};
  parallel_for_threads(nthreads, [](int t, void *p) {
    MarkCtx &c = *(MarkCtx *)p;
    const int64_t lo = c.E * t / c.nt, hi = c.E * (t + 1) / c.nt;
    for (int64_t j = lo; j < hi; ++j) __atomic_store_n(&c.has_in[c.adj[j]], 1, __ATOMIC_RELAXED);
  }, &mx);
  std::vector<int32_t> cid((size_t)V, -1);
  int64_t Vt = 0;
  for (int64_t v = 0; v < V; ++v)
    if (deg[v] > 0 || has_in[v]) cid[v] = (int32_t)Vt++;
  std::vector<int64_t> tbeg((size_t)Vt + 1);
  std::vector<int32_t> tdeg((size_t)std::max<int64_t>(Vt, 1));
  for (int64_t v = 0; v < V; ++v)
    if (cid[v] >= 0) {
      tbeg[cid[v]] = beg[v];
      tdeg[cid[v]] = deg[v];
    }
  tbeg[Vt] = E;
  // Hubs: the H highest-degree traversal vertices (ties by id).  Traversal
  // adjacency: each list ordered by descending neighbour degree (ties by
  // id), hub neighbours encoded as 0x80000000 | hub slot.
  const int64_t H = std::min<int64_t>(opts.hub_count, Vt);
  std::vector<int32_t> order((size_t)Vt);
  for (int64_t v = 0; v < Vt; ++v) order[v] = (int32_t)v;
  std::stable_sort(order.begin(), order.end(),
                   [&](int32_t a, int32_t b) { return tdeg[a] > tdeg[b]; });
  std::vector<int32_t> slot_of((size_t)std::max<int64_t>(Vt, 1), -1);
  for (int64_t i = 0; i < H; ++i) slot_of[order[i]] = (int32_t)i;
  std::vector<int32_t> xadj((size_t)std::max<int64_t>(E, 1)), tadj((size_t)std::max<int64_t>(E, 1));
  struct Ctx {
    const int64_t *beg;
    const int32_t *adj, *deg, *slot_of, *cid;
    int32_t *xadj, *tadj;
    int64_t Vt;
    int nt;
  } cx{tbeg.data(), adj, tdeg.data(), slot_of.data(), cid.data(), xadj.data(), tadj.data(), Vt,
       nthreads};
  parallel_for_threads(cx.nt, [](int t, void *p) {
    Ctx &c = *(Ctx *)p;
    for (int64_t v = t; v < c.Vt; v += c.nt) {
      const int64_t s = c.beg[v], e = c.beg[v + 1];
      for (int64_t j = s; j < e; ++j) c.xadj[j] = c.cid[c.adj[j]];
      int32_t *a = c.tadj + s, *ae = c.tadj + e;
      std::copy(c.xadj + s, c.xadj + e, a);
      std::sort(a, ae, [&](int32_t x, int32_t y) {
        return c.deg[x] != c.deg[y] ? c.deg[x] > c.deg[y] : x < y;
      });
      for (int32_t *x = a; x < ae; ++x)
        if (c.slot_of[*x] >= 0) *x = (int32_t)(0x80000000u | (uint32_t)c.slot_of[*x]);
    }
  }, &cx);
  auto *g = new ibfs_graph_s;
  g->device = device;
  g->V = V;
  g->E = E;
  g->Vt = Vt;
  g->H = H;
  g->max_deg = maxd;
  g->h_hub_deg.resize((size_t)H);
  g->h_hub_id.resize((size_t)H);
  for (int64_t i = 0; i < H; ++i) {
    g->h_hub_id[i] = order[i];
    g->h_hub_deg[i] = tdeg[order[i]];
  }
  {  // entries per hub slot, then the prefix over slots
    std::vector<int64_t> per((size_t)H + 1, 0);
    for (int64_t j = 0; j < E; ++j)
      if (tadj[j] < 0) ++per[(size_t)(tadj[j] & 0x7fffffff) + 1];
    for (int64_t i = 1; i <= H; ++i) per[i] += per[i - 1];
    g->h_hub_entries = std::move(per);
  }
  const size_t eb = sizeof(int32_t) * (size_t)std::max<int64_t>(E, 1);
  const size_t vtb = sizeof(int32_t) * (size_t)std::max<int64_t>(Vt, 1);
  // the heads are made where memory holds them beside the rest
  int32_t *&head = g->heads->d;
  hipError_t err = hipSuccess;
  auto A = [&](void **p, size_t bytes) {
    if (err != hipSuccess) return;
    err = hipMalloc(p, bytes);
    if (err == hipErrorOutOfMemory && head) {
      dfree(head);
      err = hipMalloc(p, bytes);
    }
  };
  A((void **)&g->d_beg, sizeof(int64_t) * (size_t)(Vt + 1));
  A((void **)&g->d_adj, eb);
  A((void **)&g->d_tadj, eb);
  if (err == hipSuccess &&
      hipMalloc((void **)&head, sizeof(int4) * 2 * (size_t)std::max<int64_t>(Vt, 1)) != hipSuccess)
    head = nullptr;
  A((void **)&g->d_deg, vtb);
  A((void **)&g->d_hubs, sizeof(int32_t) * (size_t)std::max<int64_t>(H, 1));
  A((void **)&g->d_cid, sizeof(int32_t) * (size_t)V);
  A((void **)&g->d_vid, vtb);
  clear_hip_error();
  if (err == hipSuccess) err = hipMemcpy(g->d_beg, tbeg.data(), sizeof(int64_t) * (size_t)(Vt + 1), hipMemcpyHostToDevice);
  if (err == hipSuccess && E > 0) err = hipMemcpy(g->d_adj, xadj.data(), sizeof(int32_t) * (size_t)E, hipMemcpyHostToDevice);
  if (err == hipSuccess && E > 0) err = hipMemcpy(g->d_tadj, tadj.data(), sizeof(int32_t) * (size_t)E, hipMemcpyHostToDevice);
  if (err == hipSuccess && head) err = launch_build_head(g->d_beg, g->d_tadj, Vt, reinterpret_cast<int4 *>(head), nullptr);
  if (err == hipSuccess && Vt > 0) err = hipMemcpy(g->d_deg, tdeg.data(), sizeof(int32_t) * (size_t)Vt, hipMemcpyHostToDevice);
  if (err == hipSuccess && H > 0) err = hipMemcpy(g->d_hubs, order.data(), sizeof(int32_t) * (size_t)H, hipMemcpyHostToDevice);
  if (err == hipSuccess) err = hipMemcpy(g->d_cid, cid.data(), sizeof(int32_t) * (size_t)V, hipMemcpyHostToDevice);
  if (err == hipSuccess && Vt > 0) {
    std::vector<int32_t> vid((size_t)Vt);
    for (int64_t v = 0; v < V; ++v)
      if (cid[v] >= 0) vid[(size_t)cid[v]] = (int32_t)v;
    err = hipMemcpy(g->d_vid, vid.data(), sizeof(int32_t) * (size_t)Vt, hipMemcpyHostToDevice);
  }
  if (err == hipSuccess) g->h_cid = std::move(cid);
  if (err != hipSuccess) {
    dfree(g->d_beg);
    dfree(g->d_adj);
    dfree(g->d_tadj);
    dfree(head);
    dfree(g->d_deg);
    dfree(g->d_hubs);
    dfree(g->d_cid);
    dfree(g->d_vid);
    delete g;
    return fail(err == hipErrorOutOfMemory ? IBFS_ERR_NOMEM : IBFS_ERR_HIP,
                "graph upload failed: %s", hipGetErrorString(err));
  }
  g->gb = groupby_pool(device);
  *out = g;
  return IBFS_OK;
}

int ibfs_graph_from_host(ibfs_hostcsr_t h, int device, ibfs_graph_t *out) {
  if (!h) return fail(IBFS_ERR_ARG, "null host csr");
  return ibfs_graph_create(h->csr.beg.data(), h->csr.V, h->csr.adj.data(), h->csr.E, device, out);
}

int ibfs_graph_load_files(const char *beg_path, const char *csr_path, int device,
                          ibfs_graph_t *out) {
  ibfs_hostcsr_t h = nullptr;
  int rc = ibfs_hostcsr_load(beg_path, csr_path, &h);
  if (rc) return rc;
  rc = ibfs_graph_from_host(h, device, out);
  ibfs_hostcsr_free(h);
  return rc;
}

int ibfs_graph_info(ibfs_graph_t g, int64_t *V, int64_t *E) {
  if (!g) return fail(IBFS_ERR_ARG, "null graph");
  if (V) *V = g->V;
  if (E) *E = g->E;
  return IBFS_OK;
}

int ibfs_graph_layout(ibfs_graph_t g, int64_t *traversal_vertices, int64_t *hubs) {
  if (!g) return fail(IBFS_ERR_ARG, "null graph");
  if (traversal_vertices) *traversal_vertices = g->Vt;
  if (hubs) *hubs = g->H;
  return IBFS_OK;
}

int ibfs_graph_hub_entries(ibfs_graph_t g, int64_t top, int64_t *entries) {
  if (!g || !entries) return fail(IBFS_ERR_ARG, "ibfs_graph_hub_entries: null argument");
  if (top <= 0 || top > g->H) top = g->H;
  *entries = g->h_hub_entries[(size_t)top];
  return IBFS_OK;
}

int ibfs_graph_destroy(ibfs_graph_t g) {
  if (!g) return IBFS_OK;
  (void)hipSetDevice(g->device);
  if (g->gb) {  // a failed call's kernel may still read the graph
    GroupbyWork *mine = nullptr;
    {
      std::lock_guard<std::mutex> lk(g->gb->mu);
      for (GroupbyWork **at = &g->gb->late; *at;) {
        GroupbyWork *w = *at;
        if (w->graph == g) {
          *at = w->next;
          --g->gb->n_late;
          w->next = mine;
          mine = w;
        } else {
          at = &w->next;
        }
      }
    }
    while (mine) {  // waits for its stream
      GroupbyWork *w = mine;
      mine = w->next;
      delete w;
    }
  }
  dfree(g->d_beg);
  dfree(g->d_adj);
  dfree(g->d_tadj);
  dfree(g->heads->d);
  dfree(g->d_deg);
  dfree(g->d_hubs);
  dfree(g->d_cid);
  dfree(g->d_vid);
  delete g;
  return IBFS_OK;
}

}  // extern "C"

// GroupBy through a workspace of the device (n <= GROUPBY_SMALL).
static int groupby_small(ibfs_graph_s *g, const int32_t *src, int n, int32_t *out) {
  GroupbyWork *w = nullptr;
  if (int rc = groupby_take(*g->gb, &w)) return rc;
  hipStream_t st = (hipStream_t)w->st;
  auto *post = static_cast<GroupbyPost *>(w->post);
  std::memcpy(post->src, src, sizeof(int32_t) * (size_t)n);
  const u64 tag = ++w->seq;
  clear_hip_error();
  const hipError_t err = launch_groupby_small(g->d_beg, g->d_adj, g->d_deg, g->d_cid, n, post,
                                              w->comp, reinterpret_cast<unsigned *>(w->ticket),
                                              tag, st);
  int rc = IBFS_OK;
  if (err != hipSuccess)
    rc = fail(IBFS_ERR_HIP, "groupby launch: %s", hipGetErrorString(err));
  else
    rc = wait_tag(st, &post->tag, tag, "groupby");
  if (rc == IBFS_OK) std::memcpy(out, post->out, sizeof(int32_t) * (size_t)n);
  groupby_put(*g->gb, w, rc == IBFS_OK ? nullptr : g);
  return rc;
}

extern "C" {

int ibfs_groupby(ibfs_graph_t g, const int32_t *src, int64_t n, int32_t *out) {
  if (!g || (n > 0 && (!src || !out)) || n < 0) return fail(IBFS_ERR_ARG, "ibfs_groupby: bad arguments");
  if (n == 0) return IBFS_OK;
  for (int64_t i = 0; i < n; ++i)
    if (src[i] < 0 || src[i] >= g->V)
      return fail(IBFS_ERR_ARG, "source %lld = %d out of range", (long long)i, src[i]);
  int rc = check_device(g->device);
  if (rc) return rc;
  if (n <= GROUPBY_SMALL && g->gb) return groupby_small(g, src, (int)n, out);
  int32_t *d = nullptr;
  void *ws = nullptr;
  const size_t wsb = groupby_workspace_bytes(n);
  HIP_TRY(hipMalloc((void **)&d, sizeof(int32_t) * (size_t)n * 3));
  hipError_t err = hipMalloc(&ws, wsb);
  if (err == hipSuccess) err = hipMemcpy(d, src, sizeof(int32_t) * (size_t)n, hipMemcpyHostToDevice);
  if (err == hipSuccess)
    err = launch_groupby(g->d_beg, g->d_adj, g->d_deg, g->d_cid, d, n, d + n, d + 2 * n, ws, wsb,
                         nullptr);
  if (err == hipSuccess)
    err = hipMemcpy(out, d + 2 * n, sizeof(int32_t) * (size_t)n, hipMemcpyDeviceToHost);
  (void)hipFree(ws);
  (void)hipFree(d);
  if (err != hipSuccess) return fail(IBFS_ERR_HIP, "groupby failed: %s", hipGetErrorString(err));
  return IBFS_OK;
}

int ibfs_engine_create(ibfs_graph_t g, const ibfs_config *cfg_in, ibfs_engine_t *out) {
  if (!g || !out) return fail(IBFS_ERR_ARG, "ibfs_engine_create: null argument");
  ibfs_config cfg;
  if (cfg_in) cfg = *cfg_in;
  else ibfs_config_default(&cfg);
  if (cfg.lane_bits != 64 && cfg.lane_bits != 128 && cfg.lane_bits != 256 && cfg.lane_bits != 512)
    return fail(IBFS_ERR_ARG, "lane_bits must be 64, 128, 256 or 512 (got %d)", cfg.lane_bits);
  if (cfg.sml_shed < 1 || cfg.lrg_shed < cfg.sml_shed)
    return fail(IBFS_ERR_ARG, "need 1 <= sml_shed <= lrg_shed (got %d, %d)", cfg.sml_shed, cfg.lrg_shed);
  if (int rc = check_direction_config(cfg)) return rc;
  if (cfg.td_chunk < 256 || (cfg.td_chunk & (cfg.td_chunk - 1)))
    return fail(IBFS_ERR_ARG, "td_chunk must be a power of two >= 256 (got %d)", cfg.td_chunk);
  if (cfg.emit_mode < 0 || cfg.emit_mode > 3)
    return fail(IBFS_ERR_ARG, "emit_mode must be 0, 1, 2 or 3 (got %d)", cfg.emit_mode);
  if (cfg.ring_levels < 4 || cfg.ring_levels > 255)
    return fail(IBFS_ERR_ARG, "ring_levels must be in [4, 255] (got %d)", cfg.ring_levels);
  if (!valid_inspect_vpt(cfg.inspect_vpt))
    return fail(IBFS_ERR_ARG, "inspect_vpt must be 0, 1, 2, 4, 8 or 16 (got %d)", cfg.inspect_vpt);
  if (!valid_wg_size(cfg.wg_size))
    return fail(IBFS_ERR_ARG, "wg_size must be 256, 512 or 1024 (got %d)", cfg.wg_size);
  if (cfg.device != g->device)
    return fail(IBFS_ERR_ARG, "config device %d differs from the graph's device %d", cfg.device, g->device);
  int rc = check_device(g->device);
  if (rc) return rc;
  auto *e = new ibfs_engine_s;
  e->g = g;
  e->cfg = cfg;
  e->K = cfg.lane_bits;
  e->W = e->Wmax = cfg.lane_bits / 64;
  e->chunk_shift = __builtin_ctz((unsigned)cfg.td_chunk);
  {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, g->device) !=
            hipSuccess || cus <= 0)
      cus = 256;
    e->hy_grid = cfg.dd_grid > 0 ? cfg.dd_grid : cus * 32;
    // each of its workgroups folds the level's counters, so no more than start
    // together: 512 x 512 grid 24.3 us per level at 1,024 workgroups, 25.5 at
    // 2,048, 27.6 at 512, 34.8 at 8,192
    e->next_grid = cfg.dd_grid > 0 ? cfg.dd_grid : cus * 4;
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, g->device) == hipSuccess &&
        khz > 0)
      e->clock_khz = khz;
  }
  e->hc = hub_cut(g, cfg.hybrid_hubs);
  const int64_t Vt = std::max<int64_t>(g->Vt, 1);
  // ring: at most 8 GiB of snapshots, at least 4 levels
  const size_t slot_bytes = (size_t)Vt * (size_t)e->W * sizeof(u64);
  int R = cfg.ring_levels;
  const size_t budget = (size_t)8 << 30;
  while (R > 4 && (size_t)R * slot_bytes > budget) --R;
  e->R = R;
  e->heads.take(g->heads);
  hipError_t err = engine_alloc(e);
  if (err == hipErrorOutOfMemory && e->heads.drop()) {
    engine_release(e);
    err = engine_alloc(e);
  }
  if (err != hipSuccess) {
    engine_release(e);
    delete e;
    return fail(err == hipErrorOutOfMemory ? IBFS_ERR_NOMEM : IBFS_ERR_HIP,
                "engine allocation failed: %s", hipGetErrorString(err));
  }
  *out = e;
  return IBFS_OK;
}

int ibfs_engine_destroy(ibfs_engine_t e) {
  if (!e) return IBFS_OK;
  engine_release(e);
  delete e;
  return IBFS_OK;
}

int ibfs_traversal(ibfs_engine_t e, const int32_t *src, int32_t k, int32_t *depth_out,
                   int32_t out_place, ibfs_stats *stats) {
  if (!e) return fail(IBFS_ERR_ARG, "null engine");
  if (k < 0 || k > e->K) return fail(IBFS_ERR_ARG, "k=%d outside [0, %d]", k, e->K);
  if (k > 0 && (!src || !depth_out)) return fail(IBFS_ERR_ARG, "null sources or output");
  if (out_place != IBFS_OUT_HOST && out_place != IBFS_OUT_DEVICE)
    return fail(IBFS_ERR_ARG, "bad out_place %d", out_place);
  const int64_t V = e->g->V;
  for (int i = 0; i < k; ++i)
    if (src[i] < 0 || src[i] >= V)
      return fail(IBFS_ERR_ARG, "source %d = %d out of range [0,%lld)", i, src[i], (long long)V);
  if (stats) std::memset(stats, 0, sizeof *stats);
  if (k == 0) return IBFS_OK;
  int rc = check_device(e->g->device);
  if (rc) return rc;
  if (e->unsettled) {
    rc = poll_stream(e->st, e->ev_wait);
    if (rc) return rc;
    e->unsettled = false;
  }
  int32_t *dout = depth_out;
  if (out_place == IBFS_OUT_HOST) {
    rc = ensure_out(e, (size_t)k * (size_t)V);
    if (rc) return rc;
    dout = e->d_out;
  }
  rc = traverse(e, src, k, dout, stats);
  if (rc == IBFS_OK && out_place == IBFS_OUT_HOST) {
    const D2HPiece pc{depth_out, dout, sizeof(int32_t) * (size_t)k * (size_t)V};
    rc = copy_to_host(&pc, 1, e->st);
  }
  if (rc) e->unsettled = true;
  return rc;
}

int ibfs_run_groups(ibfs_engine_t e, const int32_t *src, int64_t n, int32_t *depth_out,
                    int32_t out_place, ibfs_stats *stats) {
  if (!e || n < 0 || (n > 0 && (!src || !depth_out))) return fail(IBFS_ERR_ARG, "ibfs_run_groups: bad arguments");
  if (stats) std::memset(stats, 0, sizeof *stats);
  const int64_t V = e->g->V;
  for (int64_t g0 = 0; g0 < n; g0 += e->K) {
    const int k = (int)std::min<int64_t>(e->K, n - g0);
    ibfs_stats s{};
    int rc = ibfs_traversal(e, src + g0, k, depth_out + (size_t)g0 * (size_t)V, out_place,
                            stats ? &s : nullptr);
    if (rc) return rc;
    if (stats) {
      stats->levels = std::max(stats->levels, s.levels);
      stats->emit_windows += s.emit_windows;
      stats->traversed_edges += s.traversed_edges;
      stats->total_ms += s.total_ms;
      stats->init_ms += s.init_ms;
      stats->expand_td_ms += s.expand_td_ms;
      stats->expand_bu_ms += s.expand_bu_ms;
      stats->inspect_ms += s.inspect_ms;
      stats->emit_ms += s.emit_ms;
      stats->n_td_launches += s.n_td_launches;
      stats->n_bu_launches += s.n_bu_launches;
      stats->n_inspect_launches += s.n_inspect_launches;
      stats->n_emit_launches += s.n_emit_launches;
      stats->expand_hy_ms += s.expand_hy_ms;
      stats->n_hy_launches += s.n_hy_launches;
    }
  }
  return IBFS_OK;
}

int ibfs_engine_level_log(ibfs_engine_t e, ibfs_level_info *out, int32_t cap, int32_t *n) {
  if (!e || !n || cap < 0 || (cap > 0 && !out)) return fail(IBFS_ERR_ARG, "bad arguments");
  *n = (int32_t)e->log.size();
  for (int32_t i = 0; i < cap && i < *n; ++i) out[i] = e->log[i];
  return IBFS_OK;
}

}  // extern "C"
