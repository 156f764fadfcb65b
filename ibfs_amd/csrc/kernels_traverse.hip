// Traversal kernels (gfx950, wave64): lane init, inspector, top-down and
// bottom-up expanders (host-driven and device-driven), bottom-up work model.
#include <hip/hip_runtime.h>

#include "../../include/ibfs.h"
#include "device_util.h"

namespace ibfs {
namespace {

using namespace dev;

__global__ void k_fill_u64(u64 *p, int64_t n, u64 value) {
  for (int64_t i = (int64_t)blockIdx.x * BS + threadIdx.x; i < n; i += (int64_t)gridDim.x * BS)
    p[i] = value;
}

// Three ranges filled with zeros in one launch (a group's first snapshot,
// changed flags and control blocks), over their concatenated index space.
__global__ void k_zero3_u64(u64 *p0, int64_t n0, u64 *p1, int64_t n1, u64 *p2, int64_t n2) {
  const int64_t n01 = n0 + n1, n = n01 + n2;
  for (int64_t i = (int64_t)blockIdx.x * BS + threadIdx.x; i < n; i += (int64_t)gridDim.x * BS) {
    if (i < n0) p0[i] = 0;
    else if (i < n01) p1[i - n0] = 0;
    else p2[i - n01] = 0;
  }
}

// Group start (launch_group_start): a workgroup zeroes the words and flags of
// its share of the vertices and sets there the bits of the sources that fall
// into it, so one launch replaces three copies and two fills.  Bound by
// writing S_0 (9 us at R-MAT s22, 128 lanes).
template <int W>
__global__ __launch_bounds__(BS) void k_group_start(SourceList sl, const int32_t *__restrict__ cid,
                                                    int32_t *dout, int64_t V, int64_t Vt, u64 *S0,
                                                    uint8_t *flags, u64 *ctl, int64_t ctl_words,
                                                    LaneOut *lanes, u64 *masks, int R,
                                                    u64 *counters) {
  const int t = threadIdx.x;
  // shares of a multiple of 16 vertices: whole 64-bit words of flags
  const int64_t share = ((Vt + gridDim.x - 1) / gridDim.x + 15) & ~(int64_t)15;
  const int64_t v0 = blockIdx.x * share, v1 = v0 + share < Vt ? v0 + share : Vt;
  for (int64_t i = v0 * W + t; i < v1 * W; i += BS) S0[i] = 0;
  u64 *f = reinterpret_cast<u64 *>(flags);  // padded to whole words
  for (int64_t i = v0 / 8 + t; i < (v1 + 7) / 8; i += BS) f[i] = 0;
  if (blockIdx.x == 0) {
    if (t == 0) {
      counters[0] = 0;
      counters[1] = (u64)wall_clock64();
    }
    for (int64_t i = t; i < ctl_words; i += BS) ctl[i] = 0;
    for (int i = t; i < (2 + R + 1) * W; i += BS) {
      u64 m = ~0ull;
      if (i < 2 * W) {
        const int n = sl.k - (i % W) * 64;
        m = n >= 64 ? ~0ull : (n <= 0 ? 0ull : (1ull << n) - 1);
      }
      masks[i] = m;
    }
    for (int i = t; i < sl.k; i += BS) {
      lanes[i].out = dout + (int64_t)i * V;
      lanes[i].admit = 0;
      lanes[i].src = sl.src[i];
    }
  }
  __syncthreads();
  for (int i = t; i < sl.k; i += BS) {
    const int32_t v = cid[sl.src[i]];
    if (v >= v0 && v < v1) {  // (an isolated source has no word)
      atomicOr(&S0[(int64_t)v * W + (i >> 6)], 1ull << (i & 63));
      flags[v] = 1;
    }
  }
}

// Start of a device-planned traversal (launch_plan_start), shared out like
// k_group_start, with one word of the set-up block per thread of the first
// workgroups.  Bound by its launch on small graphs: in place of a copy, a fill
// and a set-up kernel, 42 -> 10 us from the set-up's first command to the first
// inspection on R-MAT s16 (closeness of 4,096 sources on s18 3.59 -> 3.51 ms, of
// 8,192 on s14 3.84 -> 3.76); a server's cohort had three copies more.  The
// host's memory is read past the caches, which may hold the block of the
// traversal before.
template <int W>
__global__ __launch_bounds__(BS) void k_plan_start(SourceList sl, int64_t Vt, u64 *S0,
                                                   uint8_t *flags, u64 *ctl, int64_t ctl_words,
                                                   const u64 *host, u64 *dev, int64_t words) {
  const int t = threadIdx.x;
  const int64_t at = (int64_t)blockIdx.x * BS + t, all = (int64_t)gridDim.x * BS;
  for (int64_t i = at; i < words; i += all)
    dev[i] = __hip_atomic_load(&host[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  for (int64_t i = at; i < ctl_words; i += all) ctl[i] = 0;
  const int64_t share = ((Vt + gridDim.x - 1) / gridDim.x + 15) & ~(int64_t)15;
  const int64_t v0 = blockIdx.x * share, v1 = v0 + share < Vt ? v0 + share : Vt;
  for (int64_t i = v0 * W + t; i < v1 * W; i += BS) S0[i] = 0;
  u64 *f = reinterpret_cast<u64 *>(flags);  // padded to whole words
  for (int64_t i = v0 / 8 + t; i < (v1 + 7) / 8; i += BS) f[i] = 0;
  __syncthreads();
  for (int i = t; i < sl.k; i += BS) {
    const int32_t v = sl.src[i];
    if (v >= v0 && v < v1) {
      atomicOr(&S0[(int64_t)v * W + (i >> 6)], 1ull << (i & 63));
      flags[v] = 1;
    }
  }
}

__global__ void k_group_end(const u64 *counters, GroupPost *post, u64 tag) {
  const int t = threadIdx.x;
  if (t < 3)
    __hip_atomic_store(&(&post->edges)[t],
                       t == 2 ? (u64)wall_clock64() : atomic_read(&counters[t]),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (t == 0) __hip_atomic_store(&post->tag, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Admission: bit lane[i] set in S[src[i]] (lanes of any position).  OR, so
// duplicate sources keep their bit.  src[i] < 0 is an isolated source: it
// has no status word and its depth array is -1 except 0 at the source (the
// reference stores and skips zero-degree sources, expander.cu:63,70-71).
template <int W>
__global__ void k_admit(const int32_t *src, const int32_t *lane, int n, u64 *S, uint8_t *flags) {
  int i = blockIdx.x * BS + threadIdx.x;
  if (i >= n || src[i] < 0) return;
  const int k = lane[i];
  atomicOr(&S[(int64_t)src[i] * W + (k >> 6)], 1ull << (k & 63));
  flags[src[i]] = 1;
}

// Admission into a device-driven traversal between the expansion and the
// inspection of level L = plan->level: when the posted list is tagged for L,
// lane lane[i] (clean in every snapshot so far) gets its bit at src[i] in
// S_L, the vertex is flagged, and the lanes join lam_{L-1} so that the
// inspection of L counts a vertex that misses one of them as a bottom-up
// candidate of L+1 (lam_{L-1} is not read again after that).  A lane whose
// source is isolated gains nothing in any status word and stays out of
// lam.  One workgroup; nothing to do when the plan is done or the list is
// for another level.  The lanes meet in LDS: a thread per word that read the
// whole list took 34 us of 200 sources (now 5).
template <int W>
__global__ void k_admit_dd(const AdmitList *al, const Plan *plan, u64 *ring, int R, int64_t V,
                           LevelCtl *ctl_ring, uint8_t *flags) {
  const int L = plan->level;
  if (plan->done || plan->tail_start || L < 1 || al->level != L) return;
  const int n = al->n;
  u64 *S = ring + (int64_t)(L % R) * V * W;
  __shared__ u64 lam[W];
  if (threadIdx.x < W) lam[threadIdx.x] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int32_t v = al->src[i];
    const int k = al->lane[i];
    if (v >= 0) {
      const u64 bit = 1ull << (k & 63);
      atomicOr(&S[(int64_t)v * W + (k >> 6)], bit);
      atomicOr(&lam[k >> 6], bit);
      flags[v] = 1;
    }
  }
  __syncthreads();
  if (threadIdx.x < W && lam[threadIdx.x])
    atomicOr(&ctl_ring[(L - 1) % R].lam[threadIdx.x], lam[threadIdx.x]);
}

// Progress of the sparse tail, and the direction of level L+1 from the
// counters of level L (same rule as the host-driven driver): fixed switch
// level, or alpha/beta; or the entry into the sparse tail (Plan::tail_div).
__device__ void plan_tail(Plan *p, int L) {
  // sparse tail level L: the records it appended are the next frontier; none
  // ends the traversal, an overflowing log ends it for a dense rerun
  const u64 cnt = atomic_read(&p->tail_count);
  if (cnt > p->tail_cap || cnt == p->tail_hi) {
    p->done = 1;
    p->last = L - 1;
    return;
  }
  p->tail_lo = p->tail_hi;
  p->tail_hi = cnt;
  p->dirlog[(L + 1) & 255] = 4;
  p->level = L + 1;
}

__device__ void plan_decide(Plan *p, const LevelCtl &c, int L) {
  const u64 nch = c.n_changed, nf = c.n_front, mf = c.m_front;
  const u64 mc = c.m_cand, nc = c.n_cand, mfn = c.m_front_nh;
  if (nch == 0 && L >= p->hold) {
    p->done = 1;
    // level 0 always ends a window: lanes whose source is isolated change
    // nothing in the status words but still have depth 0 at the source
    p->last = L > 0 ? L - 1 : 0;
    return;
  }
  const int Ln = L + 1;
  // the candidates bound what the tail can still append (every record holds
  // a bit one of them gains): on a long-diameter graph (a grid, a path) most
  // vertices still miss some lane when the frontier is small, and their
  // records would overflow the log and cost a dense rerun
  if (p->tail_div > 0 && L >= 2 && L >= p->hold && nf <= p->nf_prev &&
      nf * (u64)p->tail_div <= p->V && mf * (u64)p->tail_div <= p->E &&
      nc * (u64)p->tail_div <= p->V) {
    p->tail_start = Ln;
    p->tail_lo = p->tail_hi = 0;
    p->nf_prev = nf;
    p->dir = 4;
    p->td_flag = 0;
    p->dirlog[Ln & 255] = 4;
    p->level = Ln;
    return;
  }
  const int dir_prev = (L == 0) ? -1 : p->dir;
  const int dir = choose_direction(p->policy, p->sw_level, p->alpha, p->beta, p->gamma, p->rho,
                                   p->V, Ln, dir_prev, p->nf_prev, nf, mf, mc, mfn);
  p->nf_prev = nf;
  p->dir = dir;
  p->td_flag = dir == 0 && flag_top_down(mf, p->V);
  p->dirlog[Ln & 255] = dir;
  p->level = Ln;
}

// ---------------------------------------------------------------------------
// Inspector of level L: one pass over the traversal vertices.  Copies S_L
// (cur) into S_{L+1} (next, the slot the expanders of L+1 update), refreshes
// the hub cache from S_L, diffs S_L against S_{L-1} and accumulates the lanes
// that advanced (lam of L).  After a bottom-up or a sparse top-down level only
// the vertices the expander (or the source admission) flagged are diffed
// (prev is read only for them); after other levels and at level 0 every
// vertex is.  Flags are cleared as they are read.  It compacts, per degree
// class, the top-down frontier of L+1 (changed, degree > 0), counts the
// bottom-up candidates (degree > 0 and missing a lane of lam_prev) and, once
// they are few (candidates_queued), compacts them too.  Replaces
// td/sw_frontier_count + insp_scan + td/sw_frontier_gather + extract_depth
// of inspector.cu:37-500 and scan.cuh:455-904 with a single kernel.
//
// A workgroup of NW waves takes tiles of NW*64*VPT consecutive vertices;
// lane l of wave w handles vertex (w*VPT + i)*64 + l in round i.  A wave
// issues all loads of its rounds before any store, classifies in registers,
// and the waves' class totals meet in LDS, so each tile reserves its queue
// ranges with at most two 64-bit atomics (two queues each): same-address
// device atomics serialize, so their number per level is what this layout
// keeps small.  Entries go to ballot prefix positions, ascending vertex order
// within a tile.  Device-driven mode: the level and its slots come from the
// plan, and the last workgroup picks the next direction.
//
// Bound by its streams (88 to 127 MB per pass of R-MAT s22 at 128 lanes, about
// 30 to 40 us) and, on small graphs, by its chain of dependent accesses
// (7 us).  Queues and tickets of one counter each: 36 us on average at s22
// against 32, and 14.6 against 9 us per pass of a 512 x 512 grid.
__device__ __forceinline__ unsigned lanes_below(u64 m) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

template <int W, int VPT, int NW>
__global__ __launch_bounds__(NW * 64) void k_inspect(InspectArgs a) {
  constexpr int IBS = NW * 64;
  __shared__ unsigned wsum[2][NW][NQ];   // per-wave queue totals, double-buffered by tile parity
  __shared__ unsigned wbase[2][NW][NQ];  // per-wave queue bases
  __shared__ u64 red[NW][7 + W];
  __shared__ u64 fold[CTL_COPIES][16];
  __shared__ LevelCtl fin;
  __shared__ int last_s;

  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const u64 *prev = a.prev, *cur = a.cur;
  u64 *next = a.next;
  const u64 *lam_prev = a.lam_prev;
  LevelCtl *ctl = a.ctl, *ctl_zero = a.ctl_zero;
  int full = a.full_diff;
  bool queue_bu = a.queue_bu != 0;
  // the hub cache's indexes are level-independent: loaded ahead of the plan's chain
  const int64_t hub0 = (int64_t)blockIdx.x * IBS + t;
  int32_t hubv = hub0 < a.H ? a.hubs[hub0] : -1;
  if (a.plan) {
    if (a.plan->done) return;
    const int L = a.plan->level;
    if (a.plan->tail_start) {  // sparse tail levels skip the pass
      if (a.decide && blockIdx.x == 0 && t == 0) plan_tail(a.plan, L);
      return;
    }
    full = (L == 0 || !(a.plan->dir == 1 || (a.plan->dir == 0 && a.plan->td_flag)));
    const int64_t slot = a.V * W;
    prev = L > 0 ? a.ring + (int64_t)((L - 1) % a.R) * slot : nullptr;
    cur = a.ring + (int64_t)(L % a.R) * slot;
    next = a.ring + (int64_t)((L + 1) % a.R) * slot;
    ctl = a.ctl_ring + L % a.R;
    ctl_zero = a.ctl_ring + (L + 1) % a.R;
    lam_prev = L > 0 ? a.ctl_ring[(L - 1) % a.R].lam : a.lanes_all;
    queue_bu = L > 0 && candidates_queued(L, a.ctl_ring[(L - 1) % a.R].n_cand, (u64)a.V);
  }
  if (a.dec.on) {
    const LevelCtl *cp = a.ctl_prev;
    if (cp) {
      const int dir = cp->next_dir;
      if (dir < 0) return;  // ended before this level (its counters stay zero)
      full = !(dir == 1 || (dir == 0 && cp->next_flag));
      queue_bu = candidates_queued(a.dec.level, cp->n_cand, (u64)a.V);
    }
  }
  if (blockIdx.x == 0 && ctl_zero && t < (int)(sizeof(LevelCtl) / 8))
    reinterpret_cast<u64 *>(ctl_zero)[t] = 0;

  u64 lp[W], keep[W], nand[W], lamacc[W];
#pragma unroll
  for (int w = 0; w < W; ++w) {
    lp[w] = lam_prev[w];
    keep[w] = a.prev_keep ? a.prev_keep[w] : ~0ull;
    nand[w] = a.next_and ? a.next_and[w] : ~0ull;
    lamacc[w] = 0;
  }
  unsigned n_changed = 0, n_front = 0, n_cs = 0, n_cm = 0, n_cl = 0;  // of the wave
  u64 m_front = 0, m_cand = 0, m_front_nh = 0;      // of the lane
  const HubSplit hsp = a.hsplit;
  const int64_t V = a.V;
  const int sml = a.sml, lrg = a.lrg, cs = a.chunk_shift;
  uint8_t *flags = a.flags;
  const u64 *__restrict__ curp = cur;
  const u64 *__restrict__ prevp = prev;
  const int32_t *__restrict__ degp = a.deg;
  CtlSpread *sp = a.spread;

  constexpr int TILE = IBS * VPT;
  static_assert(TILE <= MAX_TILE, "queue arrays");
  const int64_t ntiles = (V + TILE - 1) / TILE;
  // segments of the queues: tile k fills segment k % QSEG
  const unsigned segcap = (unsigned)((ntiles + QSEG - 1) / QSEG) * TILE;
  const unsigned chunkcap = segcap + a.chunk_extra;
  int par = 0;
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x, par ^= 1) {
    const int64_t c0 = tile * TILE + (int64_t)wv * 64 * VPT;
    // every load of the wave's rounds first, so that none waits behind a store
    uint8_t fl[VPT];
    int dgv[VPT];
    u64 cw[VPT][W], pw[VPT][W];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int64_t v = c0 + i * 64 + lane;
      fl[i] = 0;
      dgv[i] = 0;
#pragma unroll
      for (int w = 0; w < W; ++w) cw[i][w] = pw[i][w] = 0;
      if (v < V) {
        fl[i] = flags[v];
        dgv[i] = degp[v];
        load_word<W>(curp + v * W, cw[i]);
      }
    }
    // the workgroup's first share of the hub cache, stored below
    u64 hubx[W];
    if (hubv >= 0) load_word<W>(curp + (int64_t)hubv * W, hubx);
    if (prevp) {
#pragma unroll
      for (int i = 0; i < VPT; ++i)
        if ((full || fl[i]) && c0 + i * 64 + lane < V)
          load_word<W>(prevp + (c0 + i * 64 + lane) * W, pw[i]);
    }
    uint8_t code[VPT];  // bits 0-1 top-down class, bits 2-3 bottom-up class
    unsigned tot[NQ] = {0, 0, 0, 0};  // wave totals (uniform)
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int64_t v = c0 + i * 64 + lane;
      int tc = 0, bc = 0, nck = 0;
      bool ch = false;
      if (v < V) {
        bool cover = true;
        u64 n[W];
        if (fl[i]) flags[v] = 0;
        if (full || fl[i]) {
#pragma unroll
          for (int w = 0; w < W; ++w) {
            const u64 d = cw[i][w] & ~(pw[i][w] & keep[w]);
            lamacc[w] |= d;
            ch |= (d != 0);
          }
        }
#pragma unroll
        for (int w = 0; w < W; ++w) {
          n[w] = cw[i][w] & nand[w];
          cover &= ((cw[i][w] & lp[w]) == lp[w]);
        }
        store_word<W>(next + v * W, n);
        const int dg = dgv[i];
        if (ch) {
          if (dg > 0) {
            m_front += (u64)dg;
            if (!is_hub(hsp, v, dg)) m_front_nh += (u64)dg;
            tc = degree_class(dg, sml, lrg);
            if (tc == 3) nck = (dg + (1 << cs) - 1) >> cs;
          }
        }
        if (dg > 0 && !cover) {
          m_cand += (u64)dg;
          bc = degree_class(dg, sml, lrg);
        }
      }
      code[i] = (uint8_t)(tc | (bc << 2));
      n_changed += (unsigned)__popcll(__ballot(ch));
      tot[Q_TD_S] += (unsigned)__popcll(__ballot(tc == 1));
      tot[Q_TD_M] += (unsigned)__popcll(__ballot(tc == 2));
      if (const u64 m3 = __ballot(tc == 3)) {
        n_front += (unsigned)__popcll(m3);
        tot[Q_TD_L] += (unsigned)wave_sum((u64)nck);
      }
      const unsigned cs1 = (unsigned)__popcll(__ballot(bc == 1));
      const unsigned cm1 = (unsigned)__popcll(__ballot(bc == 2));
      const unsigned cl1 = (unsigned)__popcll(__ballot(bc == 3));
      n_cs += cs1;
      n_cm += cm1;
      n_cl += cl1;
      if (queue_bu) tot[Q_BU] += cs1 + cm1 + cl1;
    }
    if (hubv >= 0) {
      store_word<W>(a.hs + hub0 * W, hubx);
      hubv = -1;
    }
    n_front += tot[Q_TD_S] + tot[Q_TD_M];
    if (lane == 0) {
#pragma unroll
      for (int k = 0; k < NQ; ++k) wsum[par][wv][k] = tot[k];
    }
    __syncthreads();
    // reservation for the tile: thread j < 2 adds queues 2j, 2j+1 in one
    // 64-bit atomic and lays out the waves' bases in wave order
    if (t < NQ / 2) {
      unsigned lo = 0, hi = 0;
      for (int w = 0; w < NW; ++w) {
        lo += wsum[par][w][2 * t];
        hi += wsum[par][w][2 * t + 1];
      }
      const unsigned long long add = (unsigned long long)lo | ((unsigned long long)hi << 32);
      const unsigned seg = (unsigned)(tile % QSEG);
      const unsigned long long got = add ? atomicAdd(&sp->qseg[seg][t], add) : 0ull;
      unsigned blo = (unsigned)got + seg * (t == 0 ? segcap : chunkcap);
      unsigned bhi = (unsigned)(got >> 32) + seg * segcap;
      for (int w = 0; w < NW; ++w) {
        wbase[par][w][2 * t] = blo;
        wbase[par][w][2 * t + 1] = bhi;
        blo += wsum[par][w][2 * t];
        bhi += wsum[par][w][2 * t + 1];
      }
    }
    __syncthreads();
    unsigned base[NQ];
#pragma unroll
    for (int k = 0; k < NQ; ++k) base[k] = wbase[par][wv][k];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int tc = code[i] & 3, bc = code[i] >> 2;
      const int32_t v = (int32_t)(c0 + i * 64 + lane);
      u64 m = __ballot(tc == 1);
      if (tc == 1) a.q.q[Q_TD_S][base[Q_TD_S] + lanes_below(m)] = v;
      base[Q_TD_S] += (unsigned)__popcll(m);
      m = __ballot(tc == 2);
      if (tc == 2) a.q.q[Q_TD_M][base[Q_TD_M] + lanes_below(m)] = v;
      base[Q_TD_M] += (unsigned)__popcll(m);
      if (__ballot(tc == 3)) {  // hub frontier vertices: (vertex, chunk) pairs
        const int nck = (tc == 3) ? (dgv[i] + (1 << cs) - 1) >> cs : 0;
        const unsigned inc = wave_incl_scan((unsigned)nck, lane);
        if (tc == 3) {
          const unsigned p0 = base[Q_TD_L] + inc - (unsigned)nck;
          for (int c = 0; c < nck; ++c) a.q.chunks[p0 + c] = make_int2(v, c);
        }
        base[Q_TD_L] += (unsigned)__shfl((int)inc, 63, 64);
      }
      if (queue_bu) {
        m = __ballot(bc != 0);
        if (bc) a.q.q[Q_BU][base[Q_BU] + lanes_below(m)] = v;
        base[Q_BU] += (unsigned)__popcll(m);
      }
    }
  }
  // the rest of the hub cache (more hubs than threads; none on the first pass)
  for (int64_t i = hub0 + (hubv < 0 ? (int64_t)gridDim.x * IBS : 0); i < a.H;
       i += (int64_t)gridDim.x * IBS) {
    u64 x[W];
    load_word<W>(curp + (int64_t)a.hubs[i] * W, x);
    store_word<W>(a.hs + i * W, x);
  }

  // The level's counters: waves, then the workgroup, then one atomic each
  // into the workgroup's copy.
  const unsigned n_cand = n_cs + n_cm + n_cl;
  u64 vals[7 + W] = {n_changed, n_front, 0, n_cand, 0, 0};
  if (n_front) {
    vals[2] = wave_sum(m_front);
    vals[5] = wave_sum(m_front_nh);
  }
  if (n_cand) vals[4] = wave_sum(m_cand);
#pragma unroll
  for (int w = 0; w < W; ++w) vals[6 + w] = n_changed ? wave_or(lamacc[w]) : 0;
  vals[6 + W] = (u64)n_cs | ((u64)n_cm << 32);
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < 7 + W; ++i) red[wv][i] = vals[i];
  }
  __syncthreads();
  const int copy = blockIdx.x % CTL_COPIES;
  if (t < 7 + W) {
    const bool add = t < 6 || t == 6 + W;
    u64 s = 0;
    for (int w = 0; w < NW; ++w) s = add ? s + red[w][t] : s | red[w][t];
    u64 *d = &sp->v[copy][t == 6 + W ? SPREAD_CLS : t];
    if (s && add) atomicAdd(d, s);
    else if (s) atomicOr(d, s);
  }
  if (a.dec.on == 2) {  // the next expansion folds
    if (blockIdx.x == 0 && t == 0) {
      ctl->segcap = segcap;
      ctl->chunkcap = chunkcap;
      ctl->bu_queued = queue_bu;
    }
    return;
  }
  // Measured against one set of counters and a launch of its own that posted
  // or decided: 512 x 512 grid, 128 lanes, 35.1 -> 31.0 us per level; R-MAT
  // s18 closeness 310 -> 291 ms; R-MAT s22, 8 groups of 128, 15.0 -> 14.6 ms.
  // The last workgroup to take a ticket folds the copies.  What it reads was
  // written by device atomics alone, and each workgroup has waited for the
  // completion of its own before its ticket: no cache is written back or
  // invalidated in the middle of the pass, as an agent-scope fence would do
  // on this multi-XCD part.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (t == 0) {
    const unsigned n = gridDim.x, copies = n < CTL_COPIES ? n : CTL_COPIES;
    const unsigned of_copy = n / CTL_COPIES + ((unsigned)copy < n % CTL_COPIES ? 1 : 0);
    last_s = atomicAdd(&sp->ticket[copy][0], 1u) == of_copy - 1 &&
             atomicAdd(&sp->top, 1u) == copies - 1;
  }
  __syncthreads();
  if (!last_s) return;
  if (t < CTL_COPIES * 16) {
    u64 *d = &sp->v[t >> 4][t & 15];
    fold[t >> 4][t & 15] = atomic_read(d);
    __hip_atomic_store(d, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (t < (int)CTL_WORDS) reinterpret_cast<u64 *>(&fin)[t] = 0;
  __shared__ u64 segn[QSEG][NQ / 2];
  if (t < QSEG * NQ / 2) {
    u64 *d = &sp->qseg[t / (NQ / 2)][t % (NQ / 2)];
    segn[t / (NQ / 2)][t % (NQ / 2)] = atomic_read(d);
    __hip_atomic_store(d, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else if (t >= 64 && t < 64 + CTL_COPIES) {
    __hip_atomic_store(&sp->ticket[t - 64][0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else if (t == 128) {
    __hip_atomic_store(&sp->top, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (t < 6 + W) {
    u64 s = 0;
    for (int c = 0; c < CTL_COPIES; ++c) s = t < 6 ? s + fold[c][t] : s | fold[c][t];
    if (t < 6) (&ctl->n_changed)[t] = (&fin.n_changed)[t] = s;
    else ctl->lam[t - 6] = fin.lam[t - 6] = s;
  } else if (t >= 32 && t < 32 + NQ) {
    const int c = t - 32;
    unsigned n = 0;
    for (int k = 0; k < QSEG; ++k) {
      ctl->pre[c][k] = fin.pre[c][k] = n;
      n += (unsigned)(segn[k][c / 2] >> (32 * (c & 1)));
    }
    ctl->q[c] = fin.q[c] = n;
  } else if (t == 48) {
    ctl->segcap = fin.segcap = segcap;
    ctl->chunkcap = fin.chunkcap = chunkcap;
    u64 s = 0, nc = 0;
    for (int c = 0; c < CTL_COPIES; ++c) {
      s += fold[c][SPREAD_CLS];
      nc += fold[c][3];
    }
    ctl->cls[0] = fin.cls[0] = (unsigned)s;
    ctl->cls[1] = fin.cls[1] = (unsigned)(s >> 32);
    ctl->cls[2] = fin.cls[2] = (unsigned)(nc - (s >> 32) - (s & 0xffffffffull));
    ctl->bu_queued = fin.bu_queued = queue_bu;
  }
  __syncthreads();
  if (a.dec.on && t == 0) {
    const Decide &d = a.dec;
    const LevelCtl *cp = a.ctl_prev;
    int dir = -1;
    if (fin.n_changed)
      dir = choose_direction(d.policy, d.sw_level, d.alpha, d.beta, d.gamma, d.rho, d.V,
                             d.level + 1, cp ? cp->next_dir : -1, cp ? cp->n_front : ~0ull,
                             fin.n_front, fin.m_front, fin.m_cand, fin.m_front_nh);
    ctl->next_dir = fin.next_dir = dir;
    ctl->next_flag = fin.next_flag = dir == 0 && flag_top_down(fin.m_front, d.V);
  }
  __syncthreads();  // the decision is in the block that other lanes copy
  if (a.post) {  // one wave: the block's words arrive at the host before the tag
    if (t < (int)CTL_WORDS)
      __hip_atomic_store(&reinterpret_cast<u64 *>(&a.post->c)[t], reinterpret_cast<u64 *>(&fin)[t],
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (t == 0)
      __hip_atomic_store(&a.post->tag, a.post_tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  if (a.plan && a.decide && t == 0) plan_decide(a.plan, fin, a.plan->level);
}

// Device-driven decision after the inspection of plan->level, as a launch of
// its own: the split rule reads hub-cache words that other workgroups of the
// inspector stored, which they see only past a kernel boundary.
// Thread 0 applies the direction rule.  A bottom-up choice with split_cov > 0
// then samples 64 of the top `hubs` hubs in the hub cache hs (S_L words, W per
// hub; wave w takes word w): an active lane set in at least split_cov % of
// the sample is dense and stays bottom-up, the other active lanes push
// top-down.  The level splits (dir 3) when both kinds are active.  A lane
// that holds few hubs has reached little of the graph: its candidates would
// scan their whole lists without covering it, while its own frontier is small.
__global__ __launch_bounds__(512) void k_plan_decide(Plan *plan, const LevelCtl *ctl_ring, int R,
                                                     const u64 *hs, int W, int hubs) {
  __shared__ int dir_s;
  __shared__ u64 dense[MAX_W];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int L = plan->level, done = plan->done, cov = plan->split_cov;
  __syncthreads();  // every wave has read the plan before thread 0 changes it
  if (done) return;
  if (t == 0) {
    if (plan->tail_start) plan_tail(plan, L);
    else plan_decide(plan, ctl_ring[L % R], L);
    dir_s = plan->done ? -1 : plan->dir;
  }
  __syncthreads();
  if (dir_s != 1 || cov <= 0 || hubs <= 0 || R < 3) return;  // (hubs > 0: 64 * W threads)
  const int ns = hubs < 64 ? hubs : 64, step = hubs / ns;
  if (wv < W) {
    const u64 x = lane < ns ? hs[(int64_t)lane * step * W + wv] : 0;
    u64 d = 0;
    for (int b = 0; b < 64; ++b) {
      const u64 m = __ballot((x >> b) & 1);
      if (__popcll(m) * 100 >= cov * ns) d |= 1ull << b;
    }
    if (lane == 0) dense[wv] = d;
  }
  __syncthreads();
  if (t == 0) {
    const LevelCtl *c = ctl_ring + L % R;
    u64 dn = 0, sp = 0;
    for (int w = 0; w < W; ++w) {
      const u64 lw = atomic_read(&c->lam[w]);
      dn |= lw & dense[w];
      sp |= lw & ~dense[w];
    }
    if (dn && sp) {
      for (int w = 0; w < W; ++w) plan->split[w] = dense[w];
      plan->dir = 3;
      plan->dirlog[(L + 1) & 255] = 3;
    }
  }
}

// ---------------------------------------------------------------------------
// Top-down: a frontier vertex u pushes S_{L-1}[u] & lam_{L-1} into S_L of its
// neighbours with 64-bit atomic ORs, skipping neighbours that already hold
// the bits (expander.cu:100-252).
// A dense top-down level flags nothing: its changes are scattered, and a byte
// store per changed vertex costs a partial-line write once the line is
// evicted; the inspector diffs every vertex after it instead.  A sparse one
// (flag_top_down) flags the vertices it changes.
// NEW (split levels): only the bits u gained at L-1 (S_{L-1} & ~S_{L-2}, pp
// = S_{L-2} or null) are pushed, and u is skipped when none is in lam.
template <int W, bool NEW = false>
__device__ __forceinline__ bool td_bits(const u64 *__restrict__ prev, const u64 *__restrict__ pp,
                                        const u64 (&lam)[W], int32_t u, u64 (&p)[W]) {
  load_word<W>(prev + (int64_t)u * W, p);
  u64 any = 0;
  if (NEW && pp) {
    u64 o[W];
    load_word<W>(pp + (int64_t)u * W, o);
#pragma unroll
    for (int w = 0; w < W; ++w) p[w] &= ~o[w];
  }
#pragma unroll
  for (int w = 0; w < W; ++w) {
    p[w] &= lam[w];
    any |= p[w];
  }
  return !NEW || any != 0;
}

// Edges [j0, j1) of u, every stride-th: four neighbours per step, their
// entries and words loaded before any atomic, so a step costs one chain of
// dependent accesses for four neighbours.  An entry past the end reads u's own
// word, which holds every bit u pushes.
template <int W, bool NEW = false>
__device__ __forceinline__ void td_push(const int32_t *__restrict__ adj,
                                        const u64 *__restrict__ prev, u64 *cur,
                                        const u64 (&lam)[W], int32_t u, int64_t j0, int64_t j1,
                                        int stride, const u64 *pp = nullptr,
                                        uint8_t *flags = nullptr) {
  u64 p[W];
  if (!td_bits<W, NEW>(prev, pp, lam, u, p)) return;
  for (int64_t j = j0; j < j1; j += 4 * stride) {
    int64_t v[4];
    u64 c[4][W];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = j + r * stride < j1 ? adj[j + r * stride] : u;
#pragma unroll
    for (int r = 0; r < 4; ++r) load_word<W>(cur + v[r] * W, c[r]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      bool ch = false;
#pragma unroll
      for (int w = 0; w < W; ++w)
        if (p[w] & ~c[r][w]) {
          atomicOr(&cur[v[r] * W + w], p[w]);
          ch = true;
        }
      if (flags && ch) flags[v[r]] = 1;
    }
  }
}

// Lanes per vertex of the small class (degree below sml): a list of up to 64
// neighbours is one step.  One thread per vertex walked it in up to 16 steps
// of dependent accesses, which was the time of a sparse level; the wider
// classes took one neighbour per lane and step.  Top-down of one s16 group
// 37 -> 16 us (4 lanes: 19), of 1,024 s22 sources 1.05 -> 0.92 ms, of a dense
// level on 300K Chung-Lu vertices 9% less; bound there by the random reads of
// the targets' words.
constexpr int TD_SMALL = 16;

// Positions of a level's queue entries (LevelCtl::pre).
struct QIndex {
  unsigned pre[QSEG];
  unsigned cap;
  __device__ __forceinline__ QIndex(const LevelCtl *c, int cls)
      : cap(cls == Q_TD_L ? c->chunkcap : c->segcap) {
#pragma unroll
    for (int s = 0; s < QSEG; ++s) pre[s] = c->pre[cls][s];
  }
  __device__ __forceinline__ int64_t operator()(int64_t i) const {
    unsigned at = (unsigned)i;
#pragma unroll
    for (int s = 1; s < QSEG; ++s)
      if ((unsigned)i >= pre[s]) at = (unsigned)i - pre[s] + (unsigned)s * cap;
    return at;
  }
};

// chunk i of a large top-down vertex: edges [lo, hi)
__device__ __forceinline__ void td_chunk_range(const int64_t *__restrict__ beg, int2 e, int cs,
                                               int64_t &lo, int64_t &hi) {
  lo = beg[e.x] + ((int64_t)e.y << cs);
  const int64_t end = beg[e.x + 1];
  hi = (lo + (1ll << cs)) < end ? (lo + (1ll << cs)) : end;
}

// Result of a bottom-up candidate: x (= x0 | new bits) into cur.  A plain
// store and a flag for the inspector's flagged diff; a hybrid level ORs the
// changed words in atomically instead (pushes may target the same vertex).
template <int W, bool HY>
__device__ __forceinline__ void bu_commit(u64 *cur, uint8_t *flags, int64_t v, const u64 (&x)[W],
                                          const u64 (&x0)[W]) {
  if (!differs<W>(x, x0)) return;
  if (HY) {
#pragma unroll
    for (int w = 0; w < W; ++w)
      if (x[w] != x0[w]) atomicOr(&cur[v * W + w], x[w]);
  } else {
    store_word<W>(cur + v * W, x);
    flags[v] = 1;
  }
}

// Bottom-up: a candidate v ORs S_{L-1} of its neighbours (restricted to
// lam_{L-1}, the only lanes that can still be new) in traversal-adjacency
// order (descending degree, hubs first) and stops as soon as its word
// covers lam_{L-1} (bitwise early termination, expander.cu:258-359).
// MODE 0: bottom-up level.  MODE 1 (hybrid level): only the prefix of hub
// entries with slot < cut is read (from the hub cache).  MODE 2 (split
// level): the whole list, for the dense lanes in lam.  In modes 1 and 2 new
// bits go in with atomic ORs (frontier vertices push into the same words
// concurrently) and nothing is flagged.
//
// A workgroup takes 256 vertices, one per thread.  Each reads its first eight
// entries from the head array, which is in vertex order: where vertices are
// consecutive, words and heads stream, and a vertex that is covered by then
// (most are, in a dense level) touches neither its offsets nor its list.  The
// others go on by degree: up to lrg one vertex per row of 16 lanes, above, one
// per workgroup.
__device__ __forceinline__ bool pulled(int32_t a, int cut) {
  return a < 0 && (a & 0x7fffffff) < cut;
}

// ORs four entries into x; false once the list or the pulled prefix has
// ended or x covers lam.  own: the vertex's word, read in place of an entry
// that is not taken (its bits are in x already, or on their way there).
template <int W, int MODE>
__device__ __forceinline__ bool bu_four(const Gather &gs, const int32_t (&a)[4], const u64 *own,
                                        const u64 (&lam)[W], int cut, u64 (&x)[W]) {
  u64 s[4][W];
  bool end = false;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const bool ok = MODE == 1 ? pulled(a[r], cut) : a[r] != NO_NBR;
    const u64 *p = a[r] < 0 ? gs.hs + (int64_t)(a[r] & 0x7fffffff) * W : gs.prev + (int64_t)a[r] * W;
    load_word<W>(ok ? p : own, s[r]);
    end |= !ok;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int w = 0; w < W; ++w) x[w] |= s[r][w] & lam[w];
  return !end && !covers<W>(x, lam);
}

// Entries 4 * part to 4 * part + 3 of v's traversal adjacency.
__device__ __forceinline__ int4 list_head(const int64_t *__restrict__ beg,
                                          const int32_t *__restrict__ tadj, int64_t v, int part) {
  const int64_t j = beg[v] + 4 * part, e = beg[v + 1];
  return make_int4(j < e ? tadj[j] : NO_NBR, j + 1 < e ? tadj[j + 1] : NO_NBR,
                   j + 2 < e ? tadj[j + 2] : NO_NBR, j + 3 < e ? tadj[j + 3] : NO_NBR);
}

__device__ __forceinline__ int4 head_entries(const GraphDev &g, int64_t v, int part) {
  return g.head ? g.head[part * g.V + v] : list_head(g.beg, g.tadj, v, part);
}

constexpr int BU_ROW = 4;   // entries per lane and step of the row class
constexpr int BU_BIG = 16;  // vertices of the workgroup class staged at a time

template <int W>
struct BuShared {
  int64_t j[BU_BIG], e[BU_BIG];  // entries left of each
  u64 x[BU_BIG][W];              // its word
  u64 part[2][BS / 64][W];       // waves' partial ORs, by step parity
  int stop[2][BS / 64];          // a wave met the end of the pulled prefix
  int n;
};

// N entries per lane of [r, e), stride apart from r + i.
template <int N>
__device__ __forceinline__ void bu_entries(const int32_t *__restrict__ tadj, int64_t r, int64_t e,
                                           int i, int stride, int32_t (&a)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int64_t j = r + i + (int64_t)k * stride;
    a[k] = j < e ? tadj[j] : NO_NBR;
  }
}

// ORs N entries' words into acc; returns whether one of the entries lies
// past the pulled prefix (MODE 1).
template <int W, int MODE, int N>
__device__ __forceinline__ bool bu_gather(const Gather &gs, const int32_t (&a)[N], int cut,
                                          u64 (&acc)[W]) {
  bool past = false;
  u64 y[N][W];
#pragma unroll
  for (int k = 0; k < N; ++k) {
#pragma unroll
    for (int w = 0; w < W; ++w) y[k][w] = 0;
    if (MODE == 1) {
      past |= a[k] != NO_NBR && !pulled(a[k], cut);
      if (pulled(a[k], cut)) load_nbr<W>(gs, a[k], y[k]);
    } else if (a[k] != NO_NBR) {
      load_nbr<W>(gs, a[k], y[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < N; ++k)
#pragma unroll
    for (int w = 0; w < W; ++w) acc[w] |= y[k][w];
  return past;
}

// The whole workgroup calls it, each thread with its vertex v (-1: none).
// What bounds it: random 16- to 64-byte reads of neighbour words (L2 misses),
// and for a graph that does not fill the chip the chain of the slowest wave.
// R-MAT s22, 128 lanes, against one queue per degree class with 4, 64 or 256
// list entries at a time: a group's dense level 290 -> 140 us, bottom-up of
// 1,024 sources 5.0 -> 4.1 ms; batched 1M Chung-Lu 2.32 -> 1.90 ms.
// Rows of 16 lanes against one vertex per thread below 64 neighbours and one
// per wave above: a row reads its list in lines where a thread reads 16 bytes,
// a wave has four lists in flight where it had one, and an average list fills
// it.  s22 at 256 lanes, first two dense levels 295 + 270 -> 269 + 245 us;
// closeness of 4,096 sources on s18 3.76 -> 3.60 ms, with 512 lanes
// 3.51 -> 3.24, on a power-law graph of 1M vertices 8.9 -> 8.6.  Slower or
// alike: 2, 3 or 6 entries per lane for 4, the next four vertices' entries
// loaded ahead, the first hubs' words in LDS.
template <int W, int MODE>
__device__ __forceinline__ void bu_tile(const GraphDev &g, const Gather &gs, u64 *cur,
                                        uint8_t *flags, const u64 (&lam)[W], int64_t v,
                                        BuShared<W> &sh) {
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int cut = g.hsp.cut;
  const int32_t *__restrict__ tadj = g.tadj;
  u64 x[W], x0[W];
#pragma unroll
  for (int w = 0; w < W; ++w) x[w] = 0;
  int64_t j = 0, e = 0;
  int64_t deg = 0;
  bool pend = false;
  const u64 *own = cur + v * W;
  if (v >= 0) {
    const int4 h = head_entries(g, v, 0);
    load_word<W>(own, x);
#pragma unroll
    for (int w = 0; w < W; ++w) x0[w] = x[w];
    if (!covers<W>(x, lam)) {
      const int32_t a[4] = {h.x, h.y, h.z, h.w};
      pend = bu_four<W, MODE>(gs, a, own, lam, cut, x);
      if (pend) {
        const int4 h1 = head_entries(g, v, 1);
        const int32_t a1[4] = {h1.x, h1.y, h1.z, h1.w};
        pend = bu_four<W, MODE>(gs, a1, own, lam, cut, x);
      }
      if (pend) {
        j = g.beg[v];
        e = g.beg[v + 1];
        deg = e - j;
        j += 8;
        pend = j < e;
      }
    }
  } else {
#pragma unroll
    for (int w = 0; w < W; ++w) x0[w] = 0;
  }
  // row class: four vertices at a time, one per row of 16 lanes
  const bool big = pend && deg > g.lrg;
  u64 m = __ballot(pend && !big);
  while (m) {
    int from = -1, back = -1;  // the lane this row works for, the row that works for this lane
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (m) {
        const int b = __builtin_ctzll(m);
        m &= m - 1;
        if (lane >> 4 == k) from = b;
        if (lane == b) back = 16 * k;
      }
    }
    int64_t r = __shfl(j, from & 63, 64);
    const int64_t er = __shfl(e, from & 63, 64);
    u64 y[W];
#pragma unroll
    for (int w = 0; w < W; ++w) y[w] = __shfl(x[w], from & 63, 64);
    bool more = from >= 0;
    while (more) {
      int32_t a[BU_ROW];
      bu_entries<BU_ROW>(tadj, r, er, lane & 15, 16, a);
      u64 acc[W];
#pragma unroll
      for (int w = 0; w < W; ++w) acc[w] = 0;
      const bool past = bu_gather<W, MODE, BU_ROW>(gs, a, cut, acc);
#pragma unroll
      for (int w = 0; w < W; ++w) y[w] |= row_or(acc[w] & lam[w]);
      r += 16 * BU_ROW;
      more = r < er && !covers<W>(y, lam);
      if (MODE == 1 && ((__ballot(past) >> (lane & 48)) & 0xffff)) more = false;
    }
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const u64 z = __shfl(y[w], back & 63, 64);
      if (back >= 0) x[w] = z;
    }
  }
  // workgroup class: BU_BIG vertices at a time through LDS, 1,024 entries
  // per step (a vertex of 160,000 neighbours is one workgroup's chain)
  if (__syncthreads_or(big)) {
    if (t == 0) sh.n = 0;
    __syncthreads();
    const int at = big ? atomicAdd(&sh.n, 1) : -1;
    __syncthreads();
    const int n = sh.n;
    for (int i0 = 0; i0 < n; i0 += BU_BIG) {
      const bool mine = big && at >= i0 && at < i0 + BU_BIG;
      if (mine) {
        sh.j[at - i0] = j;
        sh.e[at - i0] = e;
#pragma unroll
        for (int w = 0; w < W; ++w) sh.x[at - i0][w] = x[w];
      }
      __syncthreads();
      int par = 0;
      for (int i = 0; i < BU_BIG && i0 + i < n; ++i) {
        const int64_t eb = sh.e[i];
        u64 y[W];
#pragma unroll
        for (int w = 0; w < W; ++w) y[w] = sh.x[i][w];
        for (int64_t r = sh.j[i]; r < eb; r += 4 * BS, par ^= 1) {
          u64 acc[W];
#pragma unroll
          for (int w = 0; w < W; ++w) acc[w] = 0;
          int32_t a[4];
          bu_entries<4>(tadj, r, eb, t, BS, a);
          const bool past = bu_gather<W, MODE, 4>(gs, a, cut, acc);
#pragma unroll
          for (int w = 0; w < W; ++w) acc[w] = wave_or(acc[w] & lam[w]);
          const int wpast = MODE == 1 && __ballot(past) != 0;
          if (lane == 0) {
#pragma unroll
            for (int w = 0; w < W; ++w) sh.part[par][wv][w] = acc[w];
            sh.stop[par][wv] = wpast;
          }
          // one barrier per step: the other parity is written next, and a
          // wave reaches that step's barrier only after reading this one
          __syncthreads();
          int stop = 0;
#pragma unroll
          for (int k = 0; k < BS / 64; ++k) {
#pragma unroll
            for (int w = 0; w < W; ++w) y[w] |= sh.part[par][k][w];
            stop |= sh.stop[par][k];
          }
          if (covers<W>(y, lam) || stop) {
            par ^= 1;
            break;
          }
        }
        if (t == 0) {  // every wave has read x[i] before the step's barrier, or alike now
#pragma unroll
          for (int w = 0; w < W; ++w) sh.x[i][w] |= y[w];
        }
      }
      __syncthreads();
      if (mine) {
#pragma unroll
        for (int w = 0; w < W; ++w) x[w] = sh.x[at - i0][w];
      }
      __syncthreads();
    }
  }
  if (v >= 0) bu_commit<W, MODE != 0>(cur, flags, v, x, x0);
}

// vertices per wave of bu_level
__host__ __device__ inline int bu_per_wave(int64_t n) {
  int pw = 64;
  while (pw > 8 && n < (int64_t)4 * pw * 2048) pw /= 2;
  return pw;
}

// Every candidate (the n of the queue, or every vertex), grid-strided in tiles
// of 4 waves.  A wave takes 64 vertices, or only 32, 16 or 8 where that keeps
// the number of workgroups near 2,048 (8 per CU): a wave works off its
// vertices of the row class four by four, and with few vertices that chain, not
// the chip, is the level's time.
template <int W, int MODE>
__device__ __forceinline__ void bu_level(const GraphDev &g, const Gather &gs, u64 *cur,
                                         uint8_t *flags, const u64 (&lam)[W],
                                         const LevelCtl *ctl, const int32_t *__restrict__ queue,
                                         int64_t n, BuShared<W> &sh) {
  const QIndex qi(ctl, Q_BU);
  const int pw = bu_per_wave(n), lane = threadIdx.x & 63;
  const int64_t tile = 4 * pw;
  for (int64_t i0 = blockIdx.x * tile; i0 < n; i0 += gridDim.x * tile) {
    const int64_t i = i0 + (threadIdx.x >> 6) * pw + lane;
    const bool on = lane < pw && i < n;
    bu_tile<W, MODE>(g, gs, cur, flags, lam, on ? (queue ? queue[qi(i)] : i) : -1, sh);
  }
}

__global__ void k_build_head(const int64_t *__restrict__ beg, const int32_t *__restrict__ tadj,
                             int64_t V, int4 *__restrict__ head) {
  for (int64_t i = (int64_t)blockIdx.x * BS + threadIdx.x; i < 2 * V; i += (int64_t)gridDim.x * BS) {
    head[i] = list_head(beg, tadj, i < V ? i : i - V, i < V ? 0 : 1);
  }
}

// Host-driven top-down: workgroups [0, nbs) take small vertices one per row of
// TD_SMALL lanes, [nbs, nbs+nbm) mid vertices one per wave, the rest one chunk
// of 2^chunk_shift edges of a large vertex per workgroup.
template <int W>
__global__ __launch_bounds__(BS) void k_expand_td(GraphDev g, const u64 *__restrict__ prev,
                                                  u64 *cur, const LevelCtl *__restrict__ ctl,
                                                  Queues q, int64_t ns, int64_t nm, int64_t nl,
                                                  int64_t nbs, int64_t nbm, uint8_t *flags) {
  const int64_t *__restrict__ beg = g.beg;
  const int32_t *__restrict__ adj = g.adj;
  const int cs = g.chunk_shift;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int64_t b = blockIdx.x;
  u64 lam[W];
#pragma unroll
  for (int w = 0; w < W; ++w) lam[w] = ctl->lam[w];
  if (b < nbs) {
    const int64_t i = (b * BS + t) / TD_SMALL;
    if (i >= ns) return;
    const int32_t u = q.q[Q_TD_S][QIndex(ctl, Q_TD_S)(i)];
    td_push<W>(adj, prev, cur, lam, u, beg[u] + t % TD_SMALL, beg[u + 1], TD_SMALL, nullptr, flags);
  } else if (b < nbs + nbm) {
    const int64_t i = (b - nbs) * 4 + wv;
    if (i >= nm) return;
    const int32_t u = q.q[Q_TD_M][QIndex(ctl, Q_TD_M)(i)];
    td_push<W>(adj, prev, cur, lam, u, beg[u] + lane, beg[u + 1], 64, nullptr, flags);
  } else {
    const int64_t i = b - nbs - nbm;
    if (i >= nl) return;
    const int2 e = q.chunks[QIndex(ctl, Q_TD_L)(i)];
    int64_t lo, hi;
    td_chunk_range(beg, e, cs, lo, hi);
    td_push<W>(adj, prev, cur, lam, e.x, lo + t, hi, BS, nullptr, flags);
  }
}

// Host-driven bottom-up: the n candidates of the queue, or every vertex.
template <int W>
__global__ __launch_bounds__(BS) void k_expand_bu(GraphDev g, Gather gs, u64 *cur, uint8_t *flags,
                                                  const LevelCtl *__restrict__ ctl,
                                                  const int32_t *queue, int64_t n) {
  __shared__ BuShared<W> sh;
  u64 lam[W];
#pragma unroll
  for (int w = 0; w < W; ++w) lam[w] = ctl->lam[w];
  bu_level<W, 0>(g, gs, cur, flags, lam, ctl, queue, n, sh);
}

// Hybrid level from the queues of ctl (the control block of the level
// before), grid-strided: the bottom-up candidates pull through their prefix
// of pulled hubs (the top hsp.cut), then the other top-down frontier
// vertices push.  A pulled-hub frontier vertex u reaches every candidate
// neighbour v through that prefix of v's traversal-adjacency list; a
// neighbour that is no candidate already holds every lane u can bring.
template <int W>
__device__ __forceinline__ void expand_hybrid(const GraphDev &g, const Gather &gs, u64 *cur,
                                              const u64 (&lam)[W], const LevelCtl *ctl,
                                              const Queues &q, BuShared<W> &sh) {
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int64_t G = gridDim.x;
  const int64_t *__restrict__ beg = g.beg;
  const int32_t *__restrict__ adj = g.adj;
  const int cs = g.chunk_shift;
  const HubSplit hsp = g.hsp;
  const bool queued = ctl->bu_queued != 0;
  bu_level<W, 1>(g, gs, cur, nullptr, lam, ctl, queued ? q.q[Q_BU] : nullptr,
                 queued ? (int64_t)ctl->q[Q_BU] : g.V, sh);
  const QIndex is(ctl, Q_TD_S), im(ctl, Q_TD_M), il(ctl, Q_TD_L);
  const int64_t ts = ctl->q[Q_TD_S], tm = ctl->q[Q_TD_M], tl = ctl->q[Q_TD_L];
  for (int64_t i = ((int64_t)blockIdx.x * BS + t) / TD_SMALL; i < ts; i += G * (BS / TD_SMALL)) {
    const int32_t u = q.q[Q_TD_S][is(i)];
    const int64_t b0 = beg[u], b1 = beg[u + 1];
    if (!is_hub(hsp, u, (int)(b1 - b0)))
      td_push<W>(adj, gs.prev, cur, lam, u, b0 + t % TD_SMALL, b1, TD_SMALL);
  }
  for (int64_t i = (int64_t)blockIdx.x * 4 + wv; i < tm; i += G * 4) {
    const int32_t u = q.q[Q_TD_M][im(i)];
    const int64_t b0 = beg[u], b1 = beg[u + 1];
    if (!is_hub(hsp, u, (int)(b1 - b0))) td_push<W>(adj, gs.prev, cur, lam, u, b0 + lane, b1, 64);
  }
  for (int64_t i = blockIdx.x; i < tl; i += G) {
    const int2 e = q.chunks[il(i)];
    if (is_hub(hsp, e.x, (int)(beg[e.x + 1] - beg[e.x]))) continue;
    int64_t lo, hi;
    td_chunk_range(beg, e, cs, lo, hi);
    td_push<W>(adj, gs.prev, cur, lam, e.x, lo + t, hi, BS);
  }
}

// Host-driven hybrid level (queue lengths read on the device from ctl).
template <int W>
__global__ __launch_bounds__(BS) void k_expand_hy(GraphDev g, Gather gs, u64 *cur,
                                                  const LevelCtl *__restrict__ ctl, Queues q) {
  __shared__ BuShared<W> sh;
  u64 lam[W];
#pragma unroll
  for (int w = 0; w < W; ++w) lam[w] = ctl->lam[w];
  expand_hybrid<W>(g, gs, cur, lam, ctl, q, sh);
}

// Sparse tail level L >= T = plan->tail_start: the frontier items push their
// bits along their adjacency ranges into the cumulative slot of level T.  At
// L = T the items are the top-down queues of level T-1 (small vertices one
// per thread, mid vertices and large-vertex chunks one per wave) with the
// bits S_{T-1} & ~S_{T-2}; after that they are the records of level L-1
// (vertices of degree < 64 one per thread, the others one per wave).  A
// neighbour word the push changes gains the bits that were absent from the
// atomic OR's previous value; each gain is appended as a record of level L
// (one 64-bit reservation per wave and step; records past the capacity are
// dropped and the plan ends the run for a dense rerun).  A bit is gained
// once, so each lane's arrival at a vertex is in exactly one record.
template <int W>
__device__ __forceinline__ bool tail_visit(const int32_t *__restrict__ adj, u64 *cum,
                                           const u64 (&p)[W], int64_t j, int32_t &v,
                                           u64 (&g)[W]) {
  v = adj[j];
  u64 c[W];
  load_word<W>(cum + (int64_t)v * W, c);
  bool any = false;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    g[w] = 0;
    if (p[w] & ~c[w]) {
      g[w] = p[w] & ~atomicOr(&cum[(int64_t)v * W + w], p[w]);
      any |= g[w] != 0;
    }
  }
  return any;
}

// Appends the gains of the active lanes (any: this lane gained g at v); the
// lowest active lane reserves the wave's records.  Called in divergent code:
// the ballots see the active lanes only.
template <int W>
__device__ __forceinline__ void tail_append(const Plan *plan, const TailLog &tl, u64 cap, int L,
                                            bool any, int32_t v, const u64 (&g)[W]) {
  const u64 m = __ballot(any);
  if (!m) return;
  const int lane = threadIdx.x & 63;
  const int leader = __builtin_ctzll(__ballot(1));
  u64 base = 0;
  // the plan's only field written during the level
  if (lane == leader) base = atomicAdd(const_cast<u64 *>(&plan->tail_count), (u64)__popcll(m));
  base = __shfl(base, leader, 64);
  if (any) {
    const u64 pos = base + lanes_below(m);
    if (pos < cap) {
      tl.v[pos] = v;
      tl.lev[pos] = L;
      store_word<W>(tl.bits + pos * W, g);
    }
  }
}

// One item's range [lo, hi) pushed by one wave (64 neighbours per step).
template <int W>
__device__ __forceinline__ void tail_wave(const int32_t *__restrict__ adj, u64 *cum,
                                          const Plan *plan, const TailLog &tl, u64 cap, int L,
                                          const u64 (&p)[W], int64_t lo, int64_t hi) {
  const int lane = threadIdx.x & 63;
  for (int64_t j0 = lo; j0 < hi; j0 += 64) {
    u64 g[W];
    int32_t v = -1;
    bool any = false;
    if (j0 + lane < hi) any = tail_visit<W>(adj, cum, p, j0 + lane, v, g);
    tail_append<W>(plan, tl, cap, L, any, v, g);
  }
}

// One item's range [lo, hi) pushed by one thread.
template <int W>
__device__ __forceinline__ void tail_thread(const int32_t *__restrict__ adj, u64 *cum,
                                            const Plan *plan, const TailLog &tl, u64 cap, int L,
                                            const u64 (&p)[W], int64_t lo, int64_t hi) {
  for (int64_t j = lo; j < hi; ++j) {
    u64 g[W];
    int32_t v;
    const bool any = tail_visit<W>(adj, cum, p, j, v, g);
    tail_append<W>(plan, tl, cap, L, any, v, g);
  }
}

constexpr int TAIL_THREAD_DEG = 64;  // records of smaller degree: one thread each

template <int W>
__device__ void tail_level(const int64_t *__restrict__ beg, const int32_t *__restrict__ adj,
                           u64 *ring, int R, int64_t V, const LevelCtl *ctl_ring,
                           const Plan *__restrict__ plan, const Queues &q, int cs,
                           const TailLog &tl) {
  const int L = plan->level, T = plan->tail_start;
  const int64_t slot = V * W;
  u64 *cum = ring + (int64_t)(T % R) * slot;
  const int64_t nthreads = (int64_t)gridDim.x * BS, nwaves = nthreads / 64;
  const int64_t tid = (int64_t)blockIdx.x * BS + threadIdx.x, wid = tid >> 6;
  const u64 cap = plan->tail_cap;
  if (L == T) {
    const LevelCtl *c = ctl_ring + (T - 1) % R;
    const int64_t ns = c->q[Q_TD_S], nm = c->q[Q_TD_M], nl = c->q[Q_TD_L];
    const QIndex is(c, Q_TD_S), im(c, Q_TD_M), il(c, Q_TD_L);
    const u64 *s1 = ring + (int64_t)((T - 1) % R) * slot;
    const u64 *s2 = ring + (int64_t)((T - 2) % R) * slot;
    auto bits = [&](int32_t u, u64(&p)[W]) {
      u64 o[W];
      load_word<W>(s1 + (int64_t)u * W, p);
      load_word<W>(s2 + (int64_t)u * W, o);
#pragma unroll
      for (int w = 0; w < W; ++w) p[w] &= ~o[w];
    };
    for (int64_t i = tid; i < ns; i += nthreads) {
      const int32_t u = q.q[Q_TD_S][is(i)];
      u64 p[W];
      bits(u, p);
      tail_thread<W>(adj, cum, plan, tl, cap, L, p, beg[u], beg[u + 1]);
    }
    for (int64_t i = wid; i < nm + nl; i += nwaves) {
      int32_t u;
      int64_t lo, hi;
      if (i < nm) {
        u = q.q[Q_TD_M][im(i)];
        lo = beg[u];
        hi = beg[u + 1];
      } else {
        const int2 e = q.chunks[il(i - nm)];
        u = e.x;
        td_chunk_range(beg, e, cs, lo, hi);
      }
      u64 p[W];
      bits(u, p);
      tail_wave<W>(adj, cum, plan, tl, cap, L, p, lo, hi);
    }
    return;
  }
  const int64_t r0 = (int64_t)plan->tail_lo, n = (int64_t)plan->tail_hi - r0;
  for (int64_t i = tid; i < n; i += nthreads) {
    const int32_t u = tl.v[r0 + i];
    const int64_t lo = beg[u], hi = beg[u + 1];
    if (hi - lo >= TAIL_THREAD_DEG) continue;
    u64 p[W];
    load_word<W>(tl.bits + (r0 + i) * W, p);
    tail_thread<W>(adj, cum, plan, tl, cap, L, p, lo, hi);
  }
  for (int64_t i = wid; i < n; i += nwaves) {
    const int32_t u = tl.v[r0 + i];
    const int64_t lo = beg[u], hi = beg[u + 1];
    if (hi - lo < TAIL_THREAD_DEG) continue;
    u64 p[W];
    load_word<W>(tl.bits + (r0 + i) * W, p);
    tail_wave<W>(adj, cum, plan, tl, cap, L, p, lo, hi);
  }
}

// One level in direction dir (0 top-down, tf: flags of what it changes or
// null; 1 bottom-up; 2 hybrid): a fixed grid strides over the queues, or the
// vertices, that the inspection of the level before left in c.
template <int W>
__device__ __forceinline__ void expand_level(const GraphDev &g, const u64 *prev, u64 *cur,
                                             const u64 *hs, uint8_t *flags, uint8_t *tf,
                                             const LevelCtl *__restrict__ c, const Queues &q,
                                             int dir, BuShared<W> &sh) {
  const int64_t *__restrict__ beg = g.beg;
  const int32_t *__restrict__ adj = g.adj;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int64_t G = gridDim.x;
  u64 lam[W];
#pragma unroll
  for (int w = 0; w < W; ++w) lam[w] = c->lam[w];
  if (dir == 0) {
    const QIndex is(c, Q_TD_S), im(c, Q_TD_M), il(c, Q_TD_L);
    const int64_t ns = c->q[Q_TD_S], nm = c->q[Q_TD_M], nl = c->q[Q_TD_L];
    for (int64_t i = ((int64_t)blockIdx.x * BS + t) / TD_SMALL; i < ns; i += G * (BS / TD_SMALL)) {
      const int32_t u = q.q[Q_TD_S][is(i)];
      td_push<W>(adj, prev, cur, lam, u, beg[u] + t % TD_SMALL, beg[u + 1], TD_SMALL, nullptr, tf);
    }
    for (int64_t i = (int64_t)blockIdx.x * 4 + wv; i < nm; i += G * 4) {
      const int32_t u = q.q[Q_TD_M][im(i)];
      td_push<W>(adj, prev, cur, lam, u, beg[u] + lane, beg[u + 1], 64, nullptr, tf);
    }
    for (int64_t i = blockIdx.x; i < nl; i += G) {
      const int2 e = q.chunks[il(i)];
      int64_t lo, hi;
      td_chunk_range(beg, e, g.chunk_shift, lo, hi);
      td_push<W>(adj, prev, cur, lam, e.x, lo + t, hi, BS, nullptr, tf);
    }
  } else if (dir == 2) {
    const Gather gs{prev, hs};
    expand_hybrid<W>(g, gs, cur, lam, c, q, sh);
  } else {
    const Gather gs{prev, hs};
    const bool queued = c->bu_queued != 0;
    bu_level<W, 0>(g, gs, cur, flags, lam, c, queued ? q.q[Q_BU] : nullptr,
                   queued ? (int64_t)c->q[Q_BU] : g.V, sh);
  }
}

// Levels enqueued ahead of the host: every workgroup folds the inspection's
// counters for itself (16 cache lines) and comes to the same decision; the
// first writes it to the control block and to the host.  The inspection ends
// without a ticket, a fold and a wait for the host's memory, 3 us of its 11 on
// a 512 x 512 grid.
template <int W>
__global__ __launch_bounds__(BS) void k_expand_next(GraphDev g, const u64 *prev, u64 *cur,
                                                    const u64 *hs, uint8_t *flags, NextArgs n,
                                                    Queues q) {
  __shared__ BuShared<W> sh;
  __shared__ u64 fold[CTL_COPIES][16];
  __shared__ u64 segn[QSEG][NQ / 2];
  __shared__ LevelCtl c;
  const int t = threadIdx.x;
  static_assert(CTL_COPIES * 16 == BS, "one counter per thread");
  const int dir_prev = n.ctl_prev ? n.ctl_prev->next_dir : -1;
  const u64 nf_prev = n.ctl_prev ? n.ctl_prev->n_front : ~0ull;
  fold[t >> 4][t & 15] = n.spread->v[t >> 4][t & 15];
  if (t < QSEG * NQ / 2) segn[t / (NQ / 2)][t % (NQ / 2)] = n.spread->qseg[t / (NQ / 2)][t % (NQ / 2)];
  if (t < (int)CTL_WORDS) reinterpret_cast<u64 *>(&c)[t] = 0;
  __syncthreads();
  if (t < 6 + W) {
    u64 s = 0;
#pragma unroll
    for (int k = 0; k < CTL_COPIES; ++k) s = t < 6 ? s + fold[k][t] : s | fold[k][t];
    if (t < 6) (&c.n_changed)[t] = s;
    else c.lam[t - 6] = s;
  } else if (t >= 64 && t < 64 + NQ) {
    const int k = t - 64;
    unsigned m = 0;
#pragma unroll
    for (int i = 0; i < QSEG; ++i) {
      c.pre[k][i] = m;
      m += (unsigned)(segn[i][k / 2] >> (32 * (k & 1)));
    }
    c.q[k] = m;
  } else if (t == 128) {
    u64 s = 0, nc = 0;
#pragma unroll
    for (int k = 0; k < CTL_COPIES; ++k) {
      s += fold[k][SPREAD_CLS];
      nc += fold[k][3];
    }
    c.cls[0] = (unsigned)s;
    c.cls[1] = (unsigned)(s >> 32);
    c.cls[2] = (unsigned)(nc - (s >> 32) - (s & 0xffffffffull));
  } else if (t == 192) {
    c.segcap = n.ctl->segcap;
    c.chunkcap = n.ctl->chunkcap;
    c.bu_queued = n.ctl->bu_queued;
  }
  __syncthreads();
  if (t == 0) {
    const Decide &d = n.dec;
    int dir = -1;
    if (c.n_changed)
      dir = choose_direction(d.policy, d.sw_level, d.alpha, d.beta, d.gamma, d.rho, d.V,
                             d.level + 1, dir_prev, nf_prev, c.n_front, c.m_front, c.m_cand,
                             c.m_front_nh);
    c.next_dir = dir;
    c.next_flag = dir == 0 && flag_top_down(c.m_front, d.V);
  }
  __syncthreads();
  if (blockIdx.x == 0) {
    u64 *old = reinterpret_cast<u64 *>(n.spread_old);
    for (int i = t; i < (int)(sizeof(CtlSpread) / 8); i += BS) old[i] = 0;
    if (t < (int)CTL_WORDS) {
      const u64 x = reinterpret_cast<const u64 *>(&c)[t];
      reinterpret_cast<u64 *>(n.ctl)[t] = x;
      if (n.post) {
        __hip_atomic_store(&reinterpret_cast<u64 *>(&n.post->c)[t], x, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (t == 0)
          __hip_atomic_store(&n.post->tag, n.post_tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
  if (c.next_dir < 0) return;
  expand_level<W>(g, prev, cur, hs, flags, c.next_flag ? flags : nullptr, &c, q, c.next_dir, sh);
}

// Device-driven expansion of level plan->level, or of the frontier of a
// sparse tail level.
template <int W>
__global__ __launch_bounds__(BS) void k_expand_dd(GraphDev g, u64 *ring, uint8_t *flags, int R,
                                                  const LevelCtl *__restrict__ ctl_ring,
                                                  const Plan *__restrict__ plan,
                                                  const u64 *__restrict__ hs, Queues q,
                                                  TailLog tl) {
  __shared__ BuShared<W> sh;
  const int64_t *__restrict__ beg = g.beg;
  const int32_t *__restrict__ adj = g.adj;
  const int64_t V = g.V;
  const int cs = g.chunk_shift;
  if (plan->done || plan->level < 1) return;
  if (plan->tail_start) {
    tail_level<W>(beg, adj, ring, R, V, ctl_ring, plan, q, cs, tl);
    return;
  }
  const int L = plan->level, dir = plan->dir;
  const LevelCtl *c = ctl_ring + (L - 1) % R;
  const int64_t slot = V * W;
  const u64 *prev = ring + (int64_t)((L - 1) % R) * slot;
  u64 *cur = ring + (int64_t)(L % R) * slot;
  if (dir != 3) {
    expand_level<W>(g, prev, cur, hs, flags, plan->td_flag ? flags : nullptr, c, q, dir, sh);
    return;
  }
  // split level: the dense lanes pull over whole lists, the sparse lanes
  // push the bits their frontier vertices gained at L-1
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int64_t G = gridDim.x;
  const Gather gs{prev, hs};
  const u64 *pp = L >= 2 ? ring + (int64_t)((L - 2) % R) * slot : nullptr;
  u64 ld[W], ls[W];
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const u64 lw = c->lam[w];
    ld[w] = lw & plan->split[w];
    ls[w] = lw & ~plan->split[w];
  }
  const bool queued = c->bu_queued != 0;
  bu_level<W, 2>(g, gs, cur, nullptr, ld, c, queued ? q.q[Q_BU] : nullptr,
                 queued ? (int64_t)c->q[Q_BU] : V, sh);
  const QIndex is(c, Q_TD_S), im(c, Q_TD_M), il(c, Q_TD_L);
  const int64_t ns = c->q[Q_TD_S], nm = c->q[Q_TD_M], nl = c->q[Q_TD_L];
  for (int64_t i = ((int64_t)blockIdx.x * BS + t) / TD_SMALL; i < ns; i += G * (BS / TD_SMALL)) {
    const int32_t u = q.q[Q_TD_S][is(i)];
    td_push<W, true>(adj, prev, cur, ls, u, beg[u] + t % TD_SMALL, beg[u + 1], TD_SMALL, pp);
  }
  for (int64_t i = (int64_t)blockIdx.x * 4 + wv; i < nm; i += G * 4) {
    const int32_t u = q.q[Q_TD_M][im(i)];
    td_push<W, true>(adj, prev, cur, ls, u, beg[u] + lane, beg[u + 1], 64, pp);
  }
  for (int64_t i = blockIdx.x; i < nl; i += G) {
    const int2 e = q.chunks[il(i)];
    int64_t lo, hi;
    td_chunk_range(beg, e, cs, lo, hi);
    td_push<W, true>(adj, prev, cur, ls, e.x, lo + t, hi, BS, pp);
  }
}

// Depth patch after a sparse tail (launch_tail_patch): one thread per
// record; record i of level lev > T writes lev - admit into the row of every
// selected lane it holds, or adds lev - T to that lane's closeness sum.  Each
// (vertex, lane) arrival is in one record, so no two threads write the same
// entry.
template <int W>
__global__ __launch_bounds__(BS) void k_tail_patch(TailLog tl, int64_t n, int T,
                                                   const int32_t *__restrict__ vid,
                                                   const LaneOut *__restrict__ lanes,
                                                   const u64 *__restrict__ sel, int k_lanes,
                                                   u64 *sum_out) {
  for (int64_t i = (int64_t)blockIdx.x * BS + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * BS) {
    const int lev = tl.lev[i];
    if (lev <= T) continue;
    const int32_t v = vid[tl.v[i]];
#pragma unroll
    for (int w = 0; w < W; ++w) {
      u64 b = tl.bits[i * W + w] & sel[w];
      while (b) {
        const int k = w * 64 + __builtin_ctzll(b);
        b &= b - 1;
        if (k >= k_lanes) break;
        if (sum_out) {
          atomicAdd(&sum_out[k], (u64)(lev - T));
        } else {
          int32_t *out = lanes[k].out;
          if (out) out[v] = lev - lanes[k].admit;
        }
      }
    }
  }
}

// Work model of a bottom-up level (instrumentation, not on the timed path):
// out[0] = vertices of degree > 0 whose S_{L-1} word misses a lane of
// lam_{L-1}; out[1] = sum over them of the sequential traversal-adjacency
// prefix after which the word covers lam_{L-1} (the whole list if never).
template <int W>
__global__ __launch_bounds__(BS) void k_bu_model(const int64_t *__restrict__ beg,
                                                 const int32_t *__restrict__ tadj,
                                                 const u64 *__restrict__ prev,
                                                 const u64 *__restrict__ hs,
                                                 const u64 *__restrict__ lam_prev, int64_t V,
                                                 u64 *out) {
  __shared__ u64 red[2][4];
  u64 lam[W];
#pragma unroll
  for (int w = 0; w < W; ++w) lam[w] = lam_prev[w];
  const Gather gs{prev, hs};
  u64 nv = 0, pref = 0;
  for (int64_t v = (int64_t)blockIdx.x * BS + threadIdx.x; v < V; v += (int64_t)gridDim.x * BS) {
    const int64_t s = beg[v], e = beg[v + 1];
    if (s == e) continue;
    u64 x[W];
    load_word<W>(prev + v * W, x);
    if (covers<W>(x, lam)) continue;
    ++nv;
    for (int64_t j = s; j < e; ++j) {
      u64 y[W];
      load_nbr<W>(gs, tadj[j], y);
#pragma unroll
      for (int w = 0; w < W; ++w) x[w] |= y[w] & lam[w];
      ++pref;
      if (covers<W>(x, lam)) break;
    }
  }
  nv = wave_sum(nv);
  pref = wave_sum(pref);
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = nv;
    red[1][threadIdx.x >> 6] = pref;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    const u64 s = red[threadIdx.x][0] + red[threadIdx.x][1] + red[threadIdx.x][2] +
                  red[threadIdx.x][3];
    if (s) atomicAdd(&out[threadIdx.x], s);
  }
}

#define IBFS_DISPATCH_W(W, STMT)             \
  switch (W) {                               \
    case 1: { constexpr int WW = 1; STMT; break; } \
    case 2: { constexpr int WW = 2; STMT; break; } \
    case 4: { constexpr int WW = 4; STMT; break; } \
    case 8: { constexpr int WW = 8; STMT; break; } \
    default: return hipErrorInvalidValue;    \
  }

}  // namespace

// ---------------------------------------------------------------------------
hipError_t launch_fill_u64(u64 *p, int64_t n, u64 value, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_u64, dim3(grid_for(n, BS * 8, 8192)), dim3(BS), 0, st, p, n, value);
  return hipGetLastError();
}

hipError_t launch_zero3_u64(u64 *p0, int64_t n0, u64 *p1, int64_t n1, u64 *p2, int64_t n2,
                            hipStream_t st) {
  if (n0 < 0 || n1 < 0 || n2 < 0) return hipErrorInvalidValue;
  const int64_t n = n0 + n1 + n2;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_zero3_u64, dim3(grid_for(n, BS * 8, 8192)), dim3(BS), 0, st, p0, n0, p1, n1,
                     p2, n2);
  return hipGetLastError();
}

hipError_t launch_group_start(int W, const SourceList &sl, const int32_t *cid, int32_t *dout,
                              int64_t V, int64_t Vt, u64 *S0, uint8_t *flags, u64 *ctl,
                              int64_t ctl_words, LaneOut *lanes, u64 *masks, int R, u64 *counters,
                              hipStream_t st) {
  dim3 g(grid_for(Vt * W, BS * 8, 8192)), blk(BS);
  IBFS_DISPATCH_W(W, hipLaunchKernelGGL(k_group_start<WW>, g, blk, 0, st, sl, cid, dout, V, Vt, S0,
                                        flags, ctl, ctl_words, lanes, masks, R, counters));
  return hipGetLastError();
}

hipError_t launch_plan_start(int W, const SourceList &sl, int64_t Vt, u64 *S0, uint8_t *flags,
                             u64 *ctl, int64_t ctl_words, const u64 *host, u64 *dev, int64_t words,
                             hipStream_t st) {
  dim3 g(std::max(grid_for(Vt * W, BS * 8, 8192), grid_for(words, BS, 64))), blk(BS);
  IBFS_DISPATCH_W(W, hipLaunchKernelGGL(k_plan_start<WW>, g, blk, 0, st, sl, Vt, S0, flags, ctl,
                                        ctl_words, host, dev, words));
  return hipGetLastError();
}

hipError_t launch_group_end(const u64 *counters, GroupPost *post, u64 tag, hipStream_t st) {
  hipLaunchKernelGGL(k_group_end, dim3(1), dim3(64), 0, st, counters, post, tag);
  return hipGetLastError();
}

hipError_t launch_admit_dd(int W, const AdmitList *al, const Plan *plan, u64 *ring, int R,
                           int64_t V, LevelCtl *ctl_ring, uint8_t *flags, hipStream_t st) {
  IBFS_DISPATCH_W(W, hipLaunchKernelGGL(k_admit_dd<WW>, dim3(1), dim3(BS), 0, st, al, plan, ring,
                                        R, V, ctl_ring, flags));
  return hipGetLastError();
}

hipError_t launch_admit(int W, const int32_t *src, const int32_t *lane, int n, u64 *S,
                        uint8_t *flags, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  dim3 g(grid_for(n, BS, 1 << 20)), blk(BS);
  IBFS_DISPATCH_W(W, hipLaunchKernelGGL(k_admit<WW>, g, blk, 0, st, src, lane, n, S, flags));
  return hipGetLastError();
}

// Vertices per lane and round set: 8/W, at least 2 (8 for 64-lane words, 4
// for 128, 2 for 256 and 512: chunk registers within 8 words per lane, and
// tiles large enough that the per-tile reservation atomics stay rare), or
// less while the graph has fewer than 512 such tiles.  1,024-thread
// workgroups have half the registers per lane, so their words per lane are
// halved.  a.vpt overrides within the same register caps.
int inspect_vpt(const InspectArgs &a, int W, int NW) {
  const int cap = NW >= 16 ? 4 : 8;  // status words of chunk registers per lane
  int v;
  if (a.vpt == 1 || a.vpt == 2 || a.vpt == 4 || a.vpt == 8 || a.vpt == 16) {
    v = a.vpt > 8 ? 8 : a.vpt;
    while (v > 1 && v * W > 2 * cap) v /= 2;
    return v;
  }
  v = cap / W < 2 ? (NW >= 16 ? 1 : 2) : cap / W;
  while (v > 1 && a.V < (int64_t)64 * NW * v * 512) v /= 2;
  return v;
}

// A grid of 512 workgroups (two per CU) strides over the tiles: with one
// workgroup per tile the last round of tiles runs on a half-empty part.
#ifndef IBFS_INSPECT_GRID_CAP
#define IBFS_INSPECT_GRID_CAP 512
#endif

template <int W, int VPT, int NW>
static void inspect_launch(const InspectArgs &a, hipStream_t st) {
  const int64_t tiles = (a.V + 64 * NW * VPT - 1) / (64 * NW * VPT);
  hipLaunchKernelGGL((k_inspect<W, VPT, NW>), dim3(grid_for(tiles, 1, IBFS_INSPECT_GRID_CAP)),
                     dim3(64 * NW), 0, st, a);
}

template <int W, int NW>
static void inspect_nw(const InspectArgs &a, hipStream_t st) {
  switch (inspect_vpt(a, W, NW)) {
    case 8: inspect_launch<W, 8, NW>(a, st); break;
    case 4: inspect_launch<W, 4, NW>(a, st); break;
    case 2: inspect_launch<W, 2, NW>(a, st); break;
    default: inspect_launch<W, 1, NW>(a, st); break;
  }
}

template <int W>
static void inspect_w(const InspectArgs &a, hipStream_t st) {
  // 1,024-thread workgroups are not used for 512-lane words (register spills)
  const int nw = (a.nw == 16 && W < 8) ? 16 : (a.nw == 4 ? 4 : 8);
  if (nw == 16) inspect_nw<W, 16>(a, st);
  else if (nw == 4) inspect_nw<W, 4>(a, st);
  else inspect_nw<W, 8>(a, st);
}

// A graph without an edge (V == 0) still runs one workgroup: the pass also
// posts the control block and decides the next level.
hipError_t launch_inspect(int W, const InspectArgs &a, hipStream_t st) {
  IBFS_DISPATCH_W(W, inspect_w<WW>(a, st));
  return hipGetLastError();
}

hipError_t launch_expand_td(int W, const GraphDev &g, const u64 *prev, u64 *cur,
                            const LevelCtl *ctl_prev, Queues q, int64_t ns, int64_t nm, int64_t nl,
                            uint8_t *flags, hipStream_t st) {
  const int64_t nbs = (ns * TD_SMALL + BS - 1) / BS, nbm = (nm + 3) / 4;
  const int64_t nb = nbs + nbm + nl;
  if (nb == 0) return hipSuccess;
  if (nb > 0x7fffffffLL) return hipErrorInvalidValue;
  dim3 gr((unsigned)nb), blk(BS);
  IBFS_DISPATCH_W(W, hipLaunchKernelGGL(k_expand_td<WW>, gr, blk, 0, st, g, prev, cur, ctl_prev, q,
                                        ns, nm, nl, nbs, nbm, flags));
  return hipGetLastError();
}

hipError_t launch_expand_bu(int W, const GraphDev &g, const u64 *prev, const u64 *hs, u64 *cur,
                            uint8_t *flags, const LevelCtl *ctl_prev, Queues q, int64_t n,
                            int queued, hipStream_t st) {
  const Gather gs{prev, hs};
  if (n <= 0) return hipSuccess;
  dim3 gr(grid_for(n, 4 * bu_per_wave(n), 0x7fffffff)), blk(BS);
  const int32_t *queue = queued ? q.q[Q_BU] : nullptr;
  IBFS_DISPATCH_W(W, hipLaunchKernelGGL(k_expand_bu<WW>, gr, blk, 0, st, g, gs, cur, flags,
                                        ctl_prev, queue, n));
  return hipGetLastError();
}

hipError_t launch_expand_next(int W, const GraphDev &g, const u64 *prev, u64 *cur, const u64 *hs,
                              uint8_t *flags, const NextArgs &n, Queues q, int grid,
                              hipStream_t st) {
  dim3 gr(grid > 0 ? grid : 1), blk(BS);
  IBFS_DISPATCH_W(W, hipLaunchKernelGGL(k_expand_next<WW>, gr, blk, 0, st, g, prev, cur, hs, flags,
                                        n, q));
  return hipGetLastError();
}

hipError_t launch_expand_dd(int W, const GraphDev &g, u64 *ring, uint8_t *flags, int R,
                            const LevelCtl *ctl_ring, Plan *plan, const u64 *hs, Queues q,
                            TailLog tl, int grid, hipStream_t st) {
  dim3 gr(grid > 0 ? grid : 1), blk(BS);
  IBFS_DISPATCH_W(W, hipLaunchKernelGGL(k_expand_dd<WW>, gr, blk, 0, st, g, ring, flags, R,
                                        ctl_ring, plan, hs, q, tl));
  return hipGetLastError();
}

hipError_t launch_build_head(const int64_t *beg, const int32_t *tadj, int64_t V, int4 *head,
                             hipStream_t st) {
  if (V <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_build_head, dim3(grid_for(2 * V, BS, 65536)), dim3(BS), 0, st, beg, tadj, V,
                     head);
  return hipGetLastError();
}

hipError_t launch_tail_patch(int W, TailLog tl, int64_t n, int T, const int32_t *vid,
                             const LaneOut *lanes, const u64 *sel, int k_lanes, u64 *sum_out,
                             hipStream_t st) {
  if (n <= 0) return hipSuccess;
  dim3 g(grid_for(n, BS, 4096)), blk(BS);
  IBFS_DISPATCH_W(W, hipLaunchKernelGGL(k_tail_patch<WW>, g, blk, 0, st, tl, n, T, vid, lanes,
                                        sel, k_lanes, sum_out));
  return hipGetLastError();
}

hipError_t launch_expand_hy(int W, const GraphDev &g, const u64 *prev, const u64 *hs, u64 *cur,
                            const LevelCtl *ctl_prev, Queues q, int grid, hipStream_t st) {
  dim3 gr(grid > 0 ? grid : 1), blk(BS);
  const Gather gs{prev, hs};
  IBFS_DISPATCH_W(W, hipLaunchKernelGGL(k_expand_hy<WW>, gr, blk, 0, st, g, gs, cur, ctl_prev, q));
  return hipGetLastError();
}

hipError_t launch_plan_decide(Plan *plan, const LevelCtl *ctl_ring, int R, const u64 *hs, int W,
                              int hubs, hipStream_t st) {
  // one wave without the split rule: a wider workgroup waits longer for a CU
  // while another context's expansion fills the device
  hipLaunchKernelGGL(k_plan_decide, dim3(1), dim3(hubs > 0 ? 64 * W : 64), 0, st, plan, ctl_ring,
                     R, hs, W, hubs);
  return hipGetLastError();
}

hipError_t launch_bu_model(int W, const int64_t *beg, const int32_t *tadj, const u64 *prev,
                           const u64 *hs, const u64 *lam_prev, int64_t V, u64 *out,
                           hipStream_t st) {
  if (V <= 0) return hipSuccess;
  dim3 g(grid_for(V, BS, 8192)), blk(BS);
  IBFS_DISPATCH_W(W, hipLaunchKernelGGL(k_bu_model<WW>, g, blk, 0, st, beg, tadj, prev, hs,
                                        lam_prev, V, out));
  return hipGetLastError();
}

}  // namespace ibfs
