// Plain and multi-source BFS over one resident CSR.
//
// Replaces the BFS.cu:124-148 level loop, in which every level costs an
// O(V) host fill + H2D of the accumulators (oliver.h:66, grd.h:90-97), a
// 4V-byte memset of the flag frontier, the push kernel K1
// (oliverKernel.h:45-83), a full O(V) scan in K2 (oliverKernel.h:85-141) and
// two device syncs.
//
// Here a level is two kernels, expand and compact, and the loop control
// lives on the device (BfsCtl): expand reads the level number, direction and
// queue length the previous compact wrote; compact reads the level's
// counters, takes the direction decision, writes the next level's state and
// -- when the next step is top-down -- turns the next-frontier bitmap into
// the queue.  The host enqueues levels in chunks without waiting and checks
// the done flag once per chunk; surplus levels return at once.  The whole
// sequence is capturable in a hipGraph (olv_plan_*).  A kernel boundary costs
// about 3 us on MI355X (1.8 us inside a hipGraph), less than a grid barrier
// (6-34 us), so this beats one persistent kernel; the persistent variant is
// kept behind OLV_PERSISTENT for comparison.
//
// A graph of many small levels (meshes, road networks) is bound by those two
// launches, about 7.7 us a level whatever the level holds.  For such graphs a
// third kernel precedes every few pairs: one workgroup that keeps the frontier
// in LDS and runs level after level until the frontier outgrows it
// (bfs_narrow_kernel; 1.5 us a level of 150 vertices, 2.4 us of 340).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstddef>
#include <cstring>
#include <memory>
#include <mutex>
#include <type_traits>
#include <vector>

#include "bfs_core.hpp"
#include "internal.hpp"

namespace olv {

constexpr int kBlock = 256;
constexpr uint32_t kSpinLimit = 1u << 24;
// Workgroups per CU of the per-level kernels come from the graph's tuning
// (Tuning::bfs_*_per_cu).  Defaults: expansion in the graph's own numbering
// 8 (full occupancy; 4 and 16 measured slower); on the renumbered twin 6
// (RMAT-22 0.148 ms; 7: 0.148, 5: 0.150, 4: 0.154, 8: 0.160, 3: 0.165);
// compaction 8 (insensitive).

struct BfsState {              // per level parity
  unsigned long long mu;       // unexplored out-edges before this level
  uint32_t mode;               // 0 = top-down, 1 = bottom-up
  uint32_t nbu;                // bottom-up levels before this one
};

struct BfsCtl {
  uint32_t done;       // traversal finished
  uint32_t skip;       // the narrow kernel has expanded the level: the next expand launch passes
  uint32_t level;      // next level to expand (written by compact)
  uint32_t level_e;    // level being compacted (written by expand)
  uint32_t pairs;      // result: expand/compact launch pairs that had work
  uint32_t nlevels;    // result: levels run by the narrow kernel
  uint32_t levels;     // result: levels run, the final empty one included
  uint32_t nbu;        // result: bottom-up levels
  uint32_t overflow;   // result: level cap (n + 1) reached
  uint32_t qfill[2];   // frontier queue length of level L, slot L & 1
  uint32_t hfill[2];   // hub items of level L, slot L & 1
  uint32_t pad;
  unsigned long long inspected;  // result: edges read
  BfsState st[2];
  CtrSet cnt[3];       // level counters, slot L % 3
};
constexpr size_t kBfsCtlHead = offsetof(BfsCtl, st);  // what the host reads back

struct BfsWork {
  uint32_t n = 0, nw = 0, nwp = 0;  // vertices, bitmap words, padded words
  uint8_t *visited = nullptr;       // one byte per vertex, nwp * 32 bytes
  uint32_t *snap = nullptr;         // claims as of the last frontier extraction (bitmap)
  uint32_t *bms = nullptr;          // 2 frontier bitmaps of nwp words
  uint32_t *queue = nullptr;
  uint2 *hubs = nullptr;
  BfsCtl *ctl = nullptr;
  BfsCtl *h_ctl = nullptr;          // pinned mirror
  GridBar *bar = nullptr;           // persistent mode
  unsigned long long *stat = nullptr;
  // launch pairs that the last runs take (first chunk = their maximum) and
  // whether the last one had many small levels: narrow launches from the start.
  // Of runs that could launch the narrow kernel only
  uint32_t recent[4] = {0, 0, 0, 0};
  bool deep = false;
  // the same of the last run, whatever its flags (for a plan's capture)
  uint32_t last_pairs = 0;
  bool last_narrow = true;
  bool force_bu = false;            // OLV_FORCE_BOTTOM_UP of the current run
};

static void release_bfs_work(BfsWork *w) {
  void *ps[] = {w->visited, w->snap, w->bms, w->queue, w->hubs, w->ctl, w->bar, w->stat};
  for (void *p : ps)
    if (p) (void)hipFree(p);
  if (w->h_ctl) (void)hipHostFree(w->h_ctl);
  delete w;
}

void free_bfs_work(olv_graph *g) {
  if (!g->bfs) return;
  release_bfs_work(g->bfs);
  g->bfs = nullptr;
}

static int alloc_bfs_work(BfsWork *w, const olv_graph *g) {
  w->n = g->n;
  w->nw = (g->n + 31) / 32;
  w->nwp = (w->nw + 63) / 64 * 64;
  OLV_HIP(hipMalloc(reinterpret_cast<void **>(&w->visited), (size_t)w->nwp * 32));
  OLV_HIP(hipMalloc(reinterpret_cast<void **>(&w->snap), (size_t)w->nwp * 4));
  OLV_HIP(hipMalloc(reinterpret_cast<void **>(&w->bms), (size_t)w->nwp * 4 * 2));
  OLV_HIP(hipMalloc(reinterpret_cast<void **>(&w->queue), (size_t)g->n * 4));
  OLV_HIP(hipMalloc(reinterpret_cast<void **>(&w->hubs), hub_capacity(g->m) * sizeof(uint2)));
  OLV_HIP(hipMalloc(reinterpret_cast<void **>(&w->ctl), sizeof(BfsCtl)));
  OLV_HIP(hipMalloc(reinterpret_cast<void **>(&w->bar), sizeof(GridBar)));
  OLV_HIP(hipMalloc(reinterpret_cast<void **>(&w->stat), 2 * sizeof(unsigned long long)));
  OLV_HIP(hipHostMalloc(reinterpret_cast<void **>(&w->h_ctl), sizeof(BfsCtl), hipHostMallocDefault));
  return OLV_OK;
}

// The graph's work buffers, allocated on first use; published to the graph
// only once every allocation has succeeded.
static int get_work(const olv_graph *cg, BfsWork **out) {
  olv_graph *g = const_cast<olv_graph *>(cg);
  if (!g->bfs) {
    BfsWork *w = new BfsWork();
    const int rc = alloc_bfs_work(w, g);
    if (rc != OLV_OK) {
      release_bfs_work(w);
      return rc;
    }
    g->bfs = w;
  }
  *out = g->bfs;
  return OLV_OK;
}

// ------------------------------------------------------------- kernels
// levels = INF, bitmaps/control/barrier = 0; the vertices without in-edges
// are pre-claimed (visited byte and snapshot bit) when bottom-up steps may
// run -- no parent can claim them, so bottom-up steps skip them;
// bfs_seed_kernel releases the seeds among them -- else nothing is.
// With a single seed (seed1; ~0: none) the seeding is done here as well:
// the seed's level, visited byte and snapshot bit are written by the lanes
// that own them, and workgroup 0 builds the level-0 frontier after clearing
// the control block -- one launch instead of two, and no copy of the seed.
__global__ void bfs_reset_kernel(int32_t *__restrict__ levels, uint32_t n, uint8_t *__restrict__ visited,
                                 uint32_t *__restrict__ snap, const uint32_t *__restrict__ no_in,
                                 uint32_t *__restrict__ bms, uint32_t nwp, BfsCtl *__restrict__ ctl,
                                 GridBar *__restrict__ bar, uint32_t seed1, BfsArgs a,
                                 unsigned long long m) {
  const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  const size_t nw = ((size_t)n + 31) / 32;
  const uint32_t s = seed1;
  const uint32_t so = (s != 0xffffffffu && a.omap) ? a.omap[s] : s;  // the seed's levels index
  for (size_t i = tid; i < n; i += stride) levels[i] = i == so ? 0 : kInf;
  for (size_t i = tid; i < nwp; i += stride) {
    uint32_t d = (no_in && i < nw) ? no_in[i] : 0u;
    if (s != 0xffffffffu && i == (s >> 5)) d |= 1u << (s & 31);  // the seed is claimed
    snap[i] = d;
    uint32_t b[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t nib = (d >> (4 * k)) & 0xfu;
      b[k] = (nib & 1u) | ((nib & 2u) << 7) | ((nib & 4u) << 14) | ((nib & 8u) << 21);
    }
    uint4 *o = reinterpret_cast<uint4 *>(visited + i * 32);
    o[0] = make_uint4(b[0], b[1], b[2], b[3]);
    o[1] = make_uint4(b[4], b[5], b[6], b[7]);
  }
  for (size_t i = tid; i < (size_t)nwp * 2; i += stride) bms[i] = 0u;
  if (blockIdx.x != 0) return;
  for (uint32_t i = threadIdx.x; i < sizeof(BfsCtl) / 4; i += blockDim.x) reinterpret_cast<uint32_t *>(ctl)[i] = 0u;
  for (uint32_t i = threadIdx.x; i < sizeof(GridBar) / 4; i += blockDim.x) reinterpret_cast<uint32_t *>(bar)[i] = 0u;
  if (s == 0xffffffffu) return;
  __syncthreads();
  unsigned long long deg = 0;
  seed_frontier(nullptr, 1u, a.row_ptr, a.hub_thr, a.queue, &ctl->qfill[0], a.hubs, &ctl->hfill[0],
                [&](uint32_t) -> uint32_t { return s; }, IdRow(), &deg);
  if (threadIdx.x == 0) {
    ctl->st[0].mu = m > deg ? m - deg : 0ull;
    ctl->st[0].mode = 0;
    ctl->st[0].nbu = 0;
  }
}

// One workgroup: distinct seeds become level 0 and the level-0 frontier.
__global__ void bfs_seed_kernel(const uint32_t *__restrict__ seeds, uint32_t k, BfsArgs a, unsigned long long m,
                                BfsCtl *__restrict__ ctl) {
  for (uint32_t i = threadIdx.x; i < k; i += blockDim.x) {
    const uint32_t s = seeds[i];
    atomicAnd(&a.snap[s >> 5], ~(1u << (s & 31)));
  }
  __syncthreads();
  // the snapshot bit decides between duplicate seeds (level 0 is not a next
  // frontier, so seeds stay in the snapshot)
  auto claim = [&](uint32_t i) -> uint32_t {
    const uint32_t s = seeds[i];
    const uint32_t old = atomicOr(&a.snap[s >> 5], 1u << (s & 31));
    if (old & (1u << (s & 31))) return 0xffffffffu;
    a.visited[s] = 1;
    if (a.omap) a.set_level<true>(s, 0);
    else a.set_level<false>(s, 0);
    return s;
  };
  unsigned long long deg = 0;
  seed_frontier(seeds, k, a.row_ptr, a.hub_thr, a.queue, &ctl->qfill[0], a.hubs, &ctl->hfill[0], claim, IdRow(),
                &deg);
  if (threadIdx.x == 0) {
    ctl->st[0].mu = m > deg ? m - deg : 0ull;
    ctl->st[0].mode = 0;
    ctl->st[0].nbu = 0;
  }
}

struct BfsDir {
  uint32_t can_bu;
  uint32_t force_bu;  // every level after the first bottom-up (OLV_FORCE_BOTTOM_UP)
  float alpha, beta;
};

// Level L = ctl->level: claim the vertices of level L + 1, top-down from
// the level's queue and hub items or bottom-up against frontier bitmap
// L & 1; reset the next level's fill counters.
template <bool Mapped>
__global__ void __launch_bounds__(kBlock) bfs_expand_kernel(BfsArgs a, BfsCtl *ctl, uint32_t *bms, uint32_t nwp) {
  // (both written by earlier launches; loaded together, one after the other
  // would cost a level another trip to the cache)
  if ((ctl->done | ctl->skip) != 0) return;
  const uint32_t L = ctl->level;
  const BfsState st = ctl->st[L & 1];
  const uint32_t qsize = ctl->qfill[L & 1], nhubs = ctl->hfill[L & 1];
  const uint32_t *front = bms + (size_t)(L & 1) * nwp;
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) {
      ctl->level_e = L;
      ctl->qfill[(L + 1) & 1] = 0;
      ctl->hfill[(L + 1) & 1] = 0;
    }
    ctr_clear(&ctl->cnt[(L + 1) % 3]);
  }
  uint32_t nf = 0;
  unsigned long long mf = 0, insp = 0;
  if (st.mode == 0)
    td_step<kBlock, Mapped>(a, qsize, nhubs, (int32_t)(L + 1), blockIdx.x, gridDim.x, nf, mf, insp);
  else
    bu_step<kBlock, Mapped>(a, front, (int32_t)(L + 1), blockIdx.x, gridDim.x, nf, mf, insp);
  flush_counters<kBlock>(&ctl->cnt[L % 3], nf, mf, insp);
}

// Level L = ctl->level_e: decide the next direction and extract level
// L + 1's frontier (bitmap (L + 1) & 1; also queue and hub items if the
// next step is top-down).  Workgroup 0 publishes the next level's state.
__global__ void __launch_bounds__(kBlock) bfs_compact_kernel(BfsArgs a, BfsCtl *ctl, uint32_t *bms, uint32_t nw,
                                                             uint32_t nwp, unsigned long long m, BfsDir dir) {
  const uint32_t w0 = blockIdx.x * kBlock + threadIdx.x;
  const WordLoad pre = w0 < nw ? load_word(a, w0) : WordLoad{};
  if (__hip_atomic_load(&ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const uint32_t L = ctl->level_e;
  const CtrSum c = ctr_total(&ctl->cnt[L % 3]);
  const BfsState st = ctl->st[L & 1];
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  const uint32_t nbu = st.nbu + st.mode;
  if (lead) {
    ctl->inspected += c.inspected;
    ctl->pairs += 1;
    ctl->skip = 0;
  }
  if (c.nf == 0 || L + 1 > a.n) {
    if (lead) {
      ctl->levels = L + 1;
      ctl->nbu = nbu;
      ctl->overflow = c.nf != 0;
      ctl->done = 1u;
    }
    return;
  }
  const unsigned long long mu = st.mu > c.mf ? st.mu - c.mf : 0ull;
  const bool next_bu =
      dir.force_bu != 0 || choose_bottom_up(st.mode != 0, dir.can_bu != 0, c.nf, c.mf, mu, a.n, dir.alpha, dir.beta);
  if (lead) {
    BfsState ns;
    ns.mu = mu;
    ns.mode = next_bu ? 1u : 0u;
    ns.nbu = nbu;
    ctl->st[(L + 1) & 1] = ns;
    ctl->level = L + 1;
  }
  frontier_words<kBlock>(a, bms + (size_t)((L + 1) & 1) * nwp, nw, !next_bu, &ctl->qfill[(L + 1) & 1],
                         &ctl->hfill[(L + 1) & 1], blockIdx.x, gridDim.x, pre);
}

// Top-down levels of a small frontier, one after another, in one workgroup.
// Returns at once unless the level's frontier is a queue of at most kNarrowQ
// vertices with at most kNarrowEdges out-edges.  A level is bound by its chain:
// the column loads, the claims in LDS, the claimed vertices' rows, a barrier.
// So a row is dealt to a group of lanes about as wide as the frontier's mean
// degree (a lane holds one edge where the level has few: four claims one after
// another by a lane cost more than the loads), and what the claims go by
// depends on the vertex count:
//   Bits   a bitmap of the visited vertices in LDS, read from the visited
//          bytes on entry (up to kNarrowBitsN vertices).  Nothing that a level
//          stores to memory is read by the next, so the barrier waits for LDS
//          only.
//   else   the visited bytes, read beside the rows; a hash set of the level's
//          claims in LDS, at most half full, tells apart lanes that find a
//          vertex unvisited at once.  The barrier waits for the stores.
// A vertex whose level the kernel expands itself gets visited byte 3, not 1:
// frontier_words takes it for an old claim (setting its snapshot bit here would
// take an atomic, about 1 us of the level's chain).
// The direction rule is not asked: a bottom-up level reads every unvisited
// vertex's state in two launches, so at these sizes it costs several times a
// level here (the last 38 levels of a 200 x 150 grid: 10 us each).
// The level whose claims no longer fit ends as the expand kernel would leave
// it, its claims in the visited bytes and its totals in the counters, and
// `skip` makes the next expand launch pass: the compact launch then takes the
// direction decision and extracts the frontier.
// Traversals of grids from an inner vertex, before and with it: 200 x 150 2.14
// and 0.31 ms, 601 x 389 7.6 and 1.65 ms, 1200 x 900 (more than kNarrowBitsN
// vertices) 22.1 and 11.6 ms, 30 x 8000 (6134 levels) 63.7 and 9.6 ms.
constexpr int kNarrowBlock = 1024;
constexpr uint32_t kNarrowQ = 2048;
constexpr uint32_t kNarrowEdges = 4096;
constexpr uint32_t kNarrowHashBits = 13;  // twice kNarrowEdges slots
constexpr uint32_t kNarrowBitsN = 24576 * 32;  // 96 KB of bitmap
constexpr uint32_t kNarrowLevels = 8192;  // levels per launch, at most
constexpr uint32_t kNarrowEvery = 16;     // launch pairs between narrow launches

template <bool Mapped, bool Bits>
__global__ void __launch_bounds__(kNarrowBlock) bfs_narrow_kernel(BfsArgs a, BfsCtl *ctl) {
  constexpr uint32_t kSlots = 1u << kNarrowHashBits;
  __shared__ uint32_t s_v[2][kNarrowQ], s_beg[2][kNarrowQ], s_deg[2][kNarrowQ];  // frontier L in [L & 1]
  __shared__ uint32_t s_claim[Bits ? kNarrowBitsN / 32 : 2 * kSlots];  // bitmap, or two hash sets (~0 = free)
  __shared__ uint16_t s_slot[2][Bits ? 1 : kNarrowQ];                  // the frontier's places in its hash set
  __shared__ uint32_t s_cnt[3], s_mf[3];  // level L's claims and their out-degrees, slot L % 3
  __shared__ unsigned long long s_red[kNarrowBlock / kWave];
  if (__hip_atomic_load(&ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const uint32_t t = threadIdx.x, lane = lane_id();
  const uint32_t L0 = ctl->level;
  uint32_t L = L0, qs = ctl->qfill[L & 1];
  const BfsState st = ctl->st[L & 1];
  if (st.mode != 0 || ctl->hfill[L & 1] != 0 || qs == 0 || qs > kNarrowQ) return;
  unsigned long long insp = 0;
  for (uint32_t i = t; i < qs; i += kNarrowBlock) {
    const uint32_t v = a.queue[i], b = a.row_ptr[v], d = a.row_ptr[v + 1] - b;
    s_v[L & 1][i] = v;
    s_beg[L & 1][i] = b;
    s_deg[L & 1][i] = d;
    if (!Bits) s_slot[L & 1][i] = 0;
    insp += d;
  }
  if (t < 3) s_cnt[t] = s_mf[t] = 0;
  insp = block_sum<kNarrowBlock, unsigned long long>(insp, s_red);
  if (insp > kNarrowEdges) return;
  uint32_t qe = (uint32_t)insp;  // edges of the frontier
  if (Bits) {
    const uint32_t nw = (a.n + 31) / 32;
    for (uint32_t i = t; i < nw; i += kNarrowBlock) {
      const uint4 *p = reinterpret_cast<const uint4 *>(a.visited + (size_t)i * 32u);
      s_claim[i] = byte_flags(p[0], p[1], 0);
    }
  } else {
    for (uint32_t i = t; i < 2 * kSlots; i += kNarrowBlock) s_claim[i] = 0xffffffffu;
  }
  __syncthreads();
  unsigned long long mu = st.mu;
  uint32_t nf = 0, mf = 0;
  insp = 0;
  for (;;) {
    const uint32_t cur = L & 1, nxt = cur ^ 1, c3 = L % 3;
    if (t == 0) s_cnt[(L + 1) % 3] = s_mf[(L + 1) % 3] = 0;  // last read before the previous level's barrier
    uint32_t lmf = 0;
    // the unvisited targets among U edges of a lane
    auto visit = [&](const auto &e, const auto &in) {
      constexpr int U = sizeof(in);
      uint32_t v[U], h[U];
      uint2 r[U];
      bool mine[U];
#pragma unroll
      for (int j = 0; j < U; ++j) v[j] = in[j] ? a.col[e[j]] : 0u;
      if (Bits) {
#pragma unroll
        for (int j = 0; j < U; ++j) {
          const uint32_t bit = 1u << (v[j] & 31);
          mine[j] = in[j] && !(atomicOr(&s_claim[v[j] >> 5], bit) & bit);
        }
      } else {
#pragma unroll
        for (int j = 0; j < U; ++j) mine[j] = in[j] && a.visited[v[j]] == 0;
      }
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const bool ld = Bits ? mine[j] : in[j];
        r[j] = make_uint2(0u, 0u);
        if (ld) __builtin_memcpy(&r[j], a.row_ptr + v[j], 8);  // begin and end in one load
      }
      if (!Bits) {
#pragma unroll
        for (int j = 0; j < U; ++j) {
          if (!mine[j]) continue;
          uint32_t *set = s_claim + nxt * kSlots, old;
          h[j] = (v[j] * 2654435761u) >> (32 - kNarrowHashBits);
          while ((old = atomicCAS(&set[h[j]], 0xffffffffu, v[j])) != 0xffffffffu && old != v[j])
            h[j] = (h[j] + 1) & (kSlots - 1);
          mine[j] = old != v[j];  // else another edge's claim
        }
      }
      uint32_t before[U], total = 0;  // the wave's claims, counted by one atomic
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const uint64_t w = ballot(mine[j]);
        before[j] = total + lane_rank(w);
        total += (uint32_t)__popcll(w);
      }
      if (total == 0) return;
      uint32_t base = 0;
      if (lane == 0) base = atomicAdd(&s_cnt[c3], total);
      base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
      for (int j = 0; j < U; ++j) {
        if (!mine[j]) continue;
        const uint32_t pos = base + before[j];
        lmf += r[j].y - r[j].x;
        if (!Bits) a.visited[v[j]] = 1;
        if (pos < kNarrowQ) {
          s_v[nxt][pos] = v[j];
          s_beg[nxt][pos] = r[j].x;
          s_deg[nxt][pos] = r[j].y - r[j].x;
          if (!Bits) s_slot[nxt][pos] = (uint16_t)h[j];
        } else {
          if (Bits) a.visited[v[j]] = 1;
          a.template set_level<Mapped>(v[j], (int32_t)(L + 1));
        }
      }
    };
    // lanes per row: the mean degree rounded up to a power of two, a lane
    // visiting one edge at a time; where the frontier has more rows than that
    // allows at once, fewer lanes, each visiting two edges at a time (four:
    // 601 x 389 grid 1.70 ms, two 1.65; one, in more rounds: 1.78)
    uint32_t lg = 0;
    while (lg < 6 && (qs << lg) < qe) ++lg;
    const bool one = (qs << lg) <= kNarrowBlock;
    while (lg > 0 && (qs << lg) > kNarrowBlock) --lg;
    const uint32_t gl = 1u << lg, sub = t & (gl - 1);
    auto edges = [&](uint32_t first, uint32_t count, uint32_t sub_, uint32_t gl_, auto U) {
      for (uint32_t q = 0; ballot(q < count); q += U * gl_) {
        uint32_t e[U];
        bool in[U];
#pragma unroll
        for (uint32_t j = 0; j < U; ++j) {
          e[j] = first + q + j * gl_ + sub_;
          in[j] = q + j * gl_ + sub_ < count;
        }
        visit(e, in);
      }
    };
    for (uint32_t i = t >> lg; i - (lane >> lg) < qs; i += kNarrowBlock >> lg) {  // the same rounds for the whole wave
      uint32_t beg = 0, deg = 0, u = 0, o = 0;
      const bool put = L != L0 && sub == 0 && i < qs;  // the vertex's level is stored beside the visits
      if (i < qs) {
        beg = s_beg[cur][i];
        deg = s_deg[cur][i];
        if (put) {
          u = s_v[cur][i];
          o = Mapped ? a.omap[u] : u;
        }
        if (sub == 0) {
          insp += deg;
          if (!Bits) s_claim[cur * kSlots + s_slot[cur][i]] = 0xffffffffu;  // free for the claims of the next level
        }
      }
      const bool wide = deg > 8 * gl;
      if (one)
        edges(beg, wide ? 0u : deg, sub, gl, std::integral_constant<uint32_t, 1>());
      else
        edges(beg, wide ? 0u : deg, sub, gl, std::integral_constant<uint32_t, 2>());
      for (uint64_t w = ballot(wide && sub == 0); w; w &= w - 1) {  // rows of many edges: the wave's lanes on each
        const int from = __ffsll((unsigned long long)w) - 1;
        edges(__shfl(beg, from, kWave), __shfl(deg, from, kWave), lane, kWave, std::integral_constant<uint32_t, 4>());
      }
      if (put) {
        a.levels[o] = (int32_t)L;
        a.visited[u] = 3;
      }
    }
    lmf = wave_sum_last(lmf);  // 64 lanes' atomics on one word would take longer than the loads
    if (lane == kWave - 1 && lmf) atomicAdd(&s_mf[c3], lmf);
    if (Bits) {
      lds_barrier();
    } else {
      __syncthreads();
    }
    nf = s_cnt[c3];
    mf = s_mf[c3];
    if (nf == 0 || L + 1 > a.n || nf > kNarrowQ || mf > kNarrowEdges) break;
    mu = mu > mf ? mu - mf : 0ull;
    qs = nf;
    qe = mf;
    nf = 0;
    ++L;
    if (L - L0 == kNarrowLevels) break;
  }
  const bool more = L - L0 == kNarrowLevels;  // level L's frontier is whole and has its row in LDS
  const uint32_t last = more ? L : L + 1;     // the frontier not expanded here
  for (uint32_t i = t; i < min(more ? qs : nf, kNarrowQ); i += kNarrowBlock) {
    const uint32_t v = s_v[last & 1][i];
    a.template set_level<Mapped>(v, (int32_t)last);
    a.visited[v] = more ? 3 : 1;
    if (more) a.queue[i] = v;
  }
  ctr_clear(&ctl->cnt[L % 3]);
  ctr_clear(&ctl->cnt[(L + 1) % 3]);
  insp = block_sum<kNarrowBlock, unsigned long long>(insp, s_red);  // (and a barrier)
  if (t != 0) return;
  ctl->nlevels += L - L0 + (more ? 0u : 1u);
  if (!more && nf == 0) {
    ctl->levels = L + 1;
    ctl->nbu = st.nbu;
    ctl->inspected += insp;
    ctl->done = 1u;
    return;
  }
  BfsState ns;
  ns.mu = mu;
  ns.mode = 0;
  ns.nbu = st.nbu;
  ctl->st[L & 1] = ns;
  ctl->level = L;
  if (more) {
    ctl->inspected += insp;
    ctl->qfill[L & 1] = qs;
    ctl->hfill[L & 1] = 0;
    return;
  }
  ctl->level_e = L;
  ctl->qfill[(L + 1) & 1] = 0;
  ctl->hfill[(L + 1) & 1] = 0;
  BfsCtr &c = ctl->cnt[L % 3].s[0];
  c.nf = nf;
  c.mf = mf;
  c.inspected = insp;
  ctl->skip = 1;
}

// All levels in one cooperative launch with the XCD-aware grid barrier
// (OLV_PERSISTENT).  Same steps and decisions as the pipeline.
template <bool Mapped>
__global__ void __launch_bounds__(kBlock) bfs_persistent_kernel(BfsArgs a, BfsCtl *ctl, uint32_t *bms, uint32_t nw,
                                                                uint32_t nwp, BfsDir dir, GridBar *bar) {
  GridBarLocal gb;
  if (!gbar_init(bar, gb, gridDim.x, kSpinLimit)) return;
  const uint32_t vb = blockIdx.x, nvb = gridDim.x;
  const bool lead = vb == 0 && threadIdx.x == 0;
  BfsState st = ctl->st[0];
  unsigned long long insp_all = 0;
  uint32_t L = 0;
  for (;;) {
    const uint32_t *front = bms + (size_t)(L & 1) * nwp;
    const uint32_t qsize = __hip_atomic_load(&ctl->qfill[L & 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t nhubs = __hip_atomic_load(&ctl->hfill[L & 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (vb == 0) {
      if (threadIdx.x == 0) {
        ctl->qfill[(L + 1) & 1] = 0;
        ctl->hfill[(L + 1) & 1] = 0;
      }
      ctr_clear(&ctl->cnt[(L + 1) % 3]);
    }
    uint32_t nf = 0;
    unsigned long long mf = 0, insp = 0;
    if (st.mode == 0)
      td_step<kBlock, Mapped>(a, qsize, nhubs, (int32_t)(L + 1), vb, nvb, nf, mf, insp);
    else
      bu_step<kBlock, Mapped>(a, front, (int32_t)(L + 1), vb, nvb, nf, mf, insp);
    flush_counters<kBlock>(&ctl->cnt[L % 3], nf, mf, insp);
    if (!grid_barrier(bar, gb, kSpinLimit)) break;
    const CtrSum c = ctr_total(&ctl->cnt[L % 3]);
    insp_all += c.inspected;
    const uint32_t nbu = st.nbu + st.mode;
    if (c.nf == 0 || L + 1 > a.n) {
      if (lead) {
        ctl->levels = L + 1;
        ctl->nbu = nbu;
        ctl->overflow = c.nf != 0;
        ctl->inspected = insp_all;
        ctl->done = 1u;
      }
      break;
    }
    const unsigned long long mu = st.mu > c.mf ? st.mu - c.mf : 0ull;
    const bool next_bu =
        dir.force_bu != 0 || choose_bottom_up(st.mode != 0, dir.can_bu != 0, c.nf, c.mf, mu, a.n, dir.alpha, dir.beta);
    st.mu = mu;
    st.mode = next_bu ? 1u : 0u;
    st.nbu = nbu;
    const uint32_t wp = vb * kBlock + threadIdx.x;
    frontier_words<kBlock>(a, bms + (size_t)((L + 1) & 1) * nwp, nw, !next_bu, &ctl->qfill[(L + 1) & 1],
                           &ctl->hfill[(L + 1) & 1], vb, nvb, wp < nw ? load_word(a, wp) : WordLoad{});
    if (!grid_barrier(bar, gb, kSpinLimit)) break;
    ++L;
  }
}

// Reached vertices and the sum of their out-degrees (E_r of the byte model).
__global__ void bfs_stat_kernel(const int32_t *__restrict__ levels, const uint32_t *__restrict__ row_ptr,
                                uint32_t n, unsigned long long *__restrict__ stat) {
  __shared__ unsigned long long s_red[kBlock / kWave];
  unsigned long long vr = 0, er = 0;
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x)
    if (levels[v] != kInf) {
      vr += 1;
      er += row_ptr[v + 1] - row_ptr[v];
    }
  vr = block_sum<kBlock, unsigned long long>(vr, s_red);
  er = block_sum<kBlock, unsigned long long>(er, s_red);
  if (threadIdx.x == 0) {
    atomicAdd(&stat[0], vr);
    atomicAdd(&stat[1], er);
  }
}

// ------------------------------------------------------------- drivers
static BfsArgs make_args(const olv_graph *g, BfsWork *w, int32_t *levels) {
  BfsArgs a;
  a.row_ptr = g->row_ptr;
  a.col = g->col;
  a.in_row_ptr = g->in_row_ptr;
  a.in_col = g->in_col;
  a.in_head = g->in_head;
  a.levels = levels;
  a.omap = g->out_map;
  a.visited = w->visited;
  a.snap = w->snap;
  a.queue = w->queue;
  a.hubs = w->hubs;
  a.n = g->n;
  a.wave_thr = g->tune.td_wave_thr;
  a.block_thr = g->tune.td_block_thr;
  a.hub_thr = g->tune.hub_thr;
  return a;
}

static unsigned grid_for(size_t items, size_t per_block, size_t per_cu) {
  size_t b = (items + per_block - 1) / per_block;
  size_t cap = (size_t)cu_count() * per_cu;
  return (unsigned)std::max<size_t>(1, std::min(b, cap));
}

static BfsDir make_dir(const olv_graph *g, const BfsWork *w, bool can_bu) {
  BfsDir d;
  d.can_bu = (can_bu && g->in_row_ptr) ? 1u : 0u;
  d.force_bu = (d.can_bu && w->force_bu) ? 1u : 0u;
  d.alpha = g->tune.alpha;
  d.beta = g->tune.beta;
  return d;
}

// Transpose (for bottom-up steps) and work buffers of g.
int bfs_prepare(const olv_graph *g, bool can_bu, BfsWork **w) {
  if (can_bu && !g->in_row_ptr) OLV_TRY(olv_graph_build_transpose(const_cast<olv_graph *>(g)));
  if (can_bu) OLV_TRY(ensure_in_head(const_cast<olv_graph *>(g)));
  return get_work(g, w);
}

// Stream-ordered, capturable: reset and seeding from k seeds d_seeds
// (device), or from the one seed `seed1` by value (k == 1).
int bfs_enqueue_init(const olv_graph *g, BfsWork *w, const uint32_t *d_seeds, uint32_t k, uint32_t seed1,
                     int32_t *levels, bool can_bu) {
  const uint32_t *no_in = can_bu ? g->no_in_bm : nullptr;
  const BfsArgs a = make_args(g, w, levels);
  hipLaunchKernelGGL(bfs_reset_kernel, dim3(grid_for(std::max<size_t>(g->n, (size_t)w->nwp * 2), 256, 8)), dim3(256),
                     0, stream(), levels, g->n, w->visited, w->snap, no_in, w->bms, w->nwp, w->ctl, w->bar,
                     k == 1 ? seed1 : 0xffffffffu, a, (unsigned long long)g->m);
  if (k != 1)
    hipLaunchKernelGGL(bfs_seed_kernel, dim3(1), dim3(256), 0, stream(), d_seeds, k, a, (unsigned long long)g->m,
                       w->ctl);
  OLV_HIP(hipGetLastError());
  return OLV_OK;
}

// Stream-ordered, capturable: `count` launch pairs (expand + compact, a level
// each), with a narrow launch ahead of every kNarrowEvery of them if `narrow`.
int bfs_enqueue_levels(const olv_graph *g, BfsWork *w, int32_t *levels, bool can_bu, uint32_t count, bool narrow) {
  const BfsArgs a = make_args(g, w, levels);
  const BfsDir dir = make_dir(g, w, can_bu);
  const unsigned ge = (unsigned)cu_count() * (a.omap ? g->tune.bfs_expand_per_cu_twin : g->tune.bfs_expand_per_cu);
  const unsigned gc = grid_for(w->nw, kBlock, g->tune.bfs_compact_per_cu);
  for (uint32_t i = 0; i < count; ++i) {
    if (narrow && !dir.force_bu && i % kNarrowEvery == 0) {
      const bool bits = g->n <= kNarrowBitsN;
      auto *kern = a.omap ? (bits ? bfs_narrow_kernel<true, true> : bfs_narrow_kernel<true, false>)
                          : (bits ? bfs_narrow_kernel<false, true> : bfs_narrow_kernel<false, false>);
      hipLaunchKernelGGL(kern, dim3(1), dim3(kNarrowBlock), 0, stream(), a, w->ctl);
    }
    if (a.omap)
      hipLaunchKernelGGL(bfs_expand_kernel<true>, dim3(ge), dim3(kBlock), 0, stream(), a, w->ctl, w->bms, w->nwp);
    else
      hipLaunchKernelGGL(bfs_expand_kernel<false>, dim3(ge), dim3(kBlock), 0, stream(), a, w->ctl, w->bms, w->nwp);
    hipLaunchKernelGGL(bfs_compact_kernel, dim3(gc), dim3(kBlock), 0, stream(), a, w->ctl, w->bms, w->nw, w->nwp,
                       (unsigned long long)g->m, dir);
  }
  OLV_HIP(hipGetLastError());
  return OLV_OK;
}

static int enqueue_persistent(const olv_graph *g, BfsWork *w, int32_t *levels, bool can_bu) {
  BfsArgs a = make_args(g, w, levels);
  const void *kern = a.omap ? reinterpret_cast<const void *>(bfs_persistent_kernel<true>)
                            : reinterpret_cast<const void *>(bfs_persistent_kernel<false>);
  int per_cu = 0;
  OLV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kBlock, 0));
  if (per_cu <= 0) return fail(OLV_EUNSUPPORTED, "persistent BFS kernel does not fit on a CU");
  const int grid = cu_count();  // one workgroup per CU: cheapest barrier (measured)
  BfsCtl *ctl = w->ctl;
  uint32_t *bms = w->bms;
  uint32_t nw = w->nw, nwp = w->nwp;
  BfsDir dir = make_dir(g, w, can_bu);
  GridBar *bar = w->bar;
  void *args[] = {&a, &ctl, &bms, &nw, &nwp, &dir, &bar};
  OLV_HIP(hipLaunchCooperativeKernel(kern, dim3(grid), dim3(kBlock), args, 0, stream()));
  return OLV_OK;
}

// Wait for the stream, then read the head of the control block.
int bfs_result(BfsWork *w, uint32_t *levels_run, uint32_t *bu_levels) {
  OLV_HIP(hipMemcpyAsync(w->h_ctl, w->ctl, kBfsCtlHead, hipMemcpyDeviceToHost, stream()));
  OLV_HIP(hipStreamSynchronize(stream()));
  if (levels_run) *levels_run = w->h_ctl->levels;
  if (bu_levels) *bu_levels = w->h_ctl->nbu;
  return OLV_OK;
}

bool bfs_done(BfsWork *w) { return w->h_ctl->done != 0; }
// Launch pairs that a run like the last one takes, and whether it begins with
// a narrow launch (so it does where no run went through launch pairs: a graph
// for bfs_small).
uint32_t bfs_pairs_hint(const BfsWork *w) { return std::max(1u, w->last_pairs); }
bool bfs_deep_hint(const BfsWork *w) { return w->last_narrow; }

// Enqueue launch pairs in growing chunks until the device reports done; one
// host round trip per level if `host_loop`.  The narrow kernel joins from the
// second chunk on, or from the first where the last run on this graph ran
// kDeepLevels levels in it: on a shallow graph a launch that finds a wide
// frontier costs 2 us for nothing.  A first chunk without it has kShallowPairs
// pairs at most, so that no run of many levels ends before the kernel has been
// asked: one that did would leave the next run without it as well.  The stop
// event of `t` follows the last enqueued level, ahead of the control block
// read-back, so host latency after the last kernel is not timed (the gaps
// between chunks are).
constexpr uint32_t kDeepLevels = 8;
constexpr uint32_t kShallowPairs = 32;

static int run_pipeline(const olv_graph *g, BfsWork *w, int32_t *levels, bool can_bu, uint32_t chunk0, bool host_loop,
                        Timer *t) {
  const bool may_narrow = !host_loop && !w->force_bu;
  bool narrow = may_narrow && w->deep;
  uint32_t chunk = host_loop ? 1u : (narrow || !may_narrow ? chunk0 : std::min(chunk0, kShallowPairs));
  uint32_t rest = host_loop ? 0u : chunk0 - chunk, more = 4;
  uint64_t enq = 0;
  for (;;) {
    OLV_TRY(bfs_enqueue_levels(g, w, levels, can_bu, chunk, narrow));
    if (t) t->stop();
    enq += chunk;
    OLV_TRY(bfs_result(w, nullptr, nullptr));
    if (w->h_ctl->done) break;
    if (enq > (uint64_t)g->n + 2) return fail(OLV_EINTERNAL, "olv_bfs: level loop did not terminate");
    if (rest) chunk = rest, rest = 0;
    else if (!host_loop) chunk = more = std::min(more * 2, 256u);
    narrow = may_narrow;
  }
  w->last_narrow = may_narrow && w->h_ctl->nlevels >= kDeepLevels;
  // a run that begins without the narrow kernel needs a pair for every level
  w->last_pairs = w->last_narrow ? w->h_ctl->pairs : w->h_ctl->levels;
  if (!may_narrow) return OLV_OK;
  w->deep = w->last_narrow;
  for (int i = 3; i > 0; --i) w->recent[i] = w->recent[i - 1];
  w->recent[0] = w->last_pairs;
  return OLV_OK;
}

static int collect_stats(const olv_graph *g, BfsWork *w, const int32_t *levels, olv_stats *st) {
  if (!st) return OLV_OK;
  OLV_HIP(hipMemsetAsync(w->stat, 0, 2 * sizeof(unsigned long long), stream()));
  hipLaunchKernelGGL(bfs_stat_kernel, dim3(grid_for(g->n, kBlock, 8)), dim3(kBlock), 0, stream(), levels, g->row_ptr,
                     g->n, w->stat);
  unsigned long long h[2];
  OLV_HIP(hipMemcpyAsync(h, w->stat, sizeof(h), hipMemcpyDeviceToHost, stream()));
  OLV_HIP(hipStreamSynchronize(stream()));
  st->vertices_reached = h[0];
  st->edges_traversed = h[1];
  return OLV_OK;
}

// ------------------------------------------------------------- small graphs
// A graph of at most 16,384 vertices whose out-lists are short runs its
// whole traversal in one workgroup: the row offsets, the visited bits and
// both frontier queues sit in LDS (~130 KB), so a level costs the column
// loads (L2 hits after the first level), LDS claims and one barrier -- not
// two kernel launches.  A small frontier is dealt to lanes by edges (2^lg
// lanes a row, lg from the graph's mean degree), a large one by rows, four
// edges of a lane in flight; a wave counts its claims by one LDS atomic.  The
// 128 x 128 grid (from an inner vertex, 200 levels of at most 128 vertices):
// 254 us by rows with a lane's claims one by one and two barriers a level,
// 174 us so.
constexpr uint32_t kSmallN = 16384;
constexpr uint32_t kSmallMaxDeg = 256;
constexpr int kSmallBlock = 1024;

// Seeds: k of them at `seeds` (device), or the one seed `seed1` (k == 1).
// out (nullptr: not wanted): [0] = levels run (the deepest level + 1), [1] =
// edges read (= the out-degree sum of reached vertices), [2] = vertices reached.
__global__ void __launch_bounds__(kSmallBlock) bfs_small_kernel(const uint32_t *__restrict__ rp,
                                                                const uint32_t *__restrict__ col, uint32_t n,
                                                                uint32_t lg, const uint32_t *__restrict__ seeds,
                                                                uint32_t k, uint32_t seed1,
                                                                int32_t *__restrict__ levels,
                                                                unsigned long long *__restrict__ out) {
  __shared__ uint32_t s_rp[kSmallN + 1];
  __shared__ uint32_t s_vis[kSmallN / 32];
  __shared__ uint16_t s_q[2][kSmallN];
  __shared__ uint32_t s_cnt[3];  // frontier L's size, slot L % 3
  __shared__ unsigned long long s_red[kSmallBlock / kWave];
  const uint32_t t = threadIdx.x, lane = lane_id();
  for (uint32_t i = t; i <= n; i += kSmallBlock) s_rp[i] = rp[i];
  for (uint32_t i = t; i < kSmallN / 32; i += kSmallBlock) s_vis[i] = 0u;
  for (uint32_t v = t; v < n; v += kSmallBlock) levels[v] = kInf;
  if (t < 3) s_cnt[t] = 0u;
  __syncthreads();
  for (uint32_t i = t; i < k; i += kSmallBlock) {
    const uint32_t v = k == 1 ? seed1 : seeds[i], bit = 1u << (v & 31);
    if (!(atomicOr(&s_vis[v >> 5], bit) & bit)) {
      s_q[0][atomicAdd(&s_cnt[0], 1u)] = (uint16_t)v;
      levels[v] = 0;
    }
  }
  __syncthreads();
  uint32_t L = 0;
  unsigned long long insp = 0, reached = 0;
  for (;; ++L) {
    const uint32_t qs = s_cnt[L % 3], cur = L & 1, nxt = cur ^ 1, c3 = (L + 1) % 3;
    if (qs == 0 || L > n) break;
    if (t == 0) s_cnt[(L + 2) % 3] = 0u;  // last read before the previous level's barrier
    reached += t < qs ? (qs - t + kSmallBlock - 1) / kSmallBlock : 0u;
    // the unvisited among U targets of a lane (~0: none)
    auto visit = [&](const auto &v) {
      constexpr int U = sizeof(v) / 4;
      bool mine[U];
      uint32_t before[U], total = 0;
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const uint32_t bit = 1u << (v[j] & 31);
        mine[j] = v[j] != 0xffffffffu && !(s_vis[v[j] >> 5] & bit) && !(atomicOr(&s_vis[v[j] >> 5], bit) & bit);
      }
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const uint64_t w = ballot(mine[j]);
        before[j] = total + lane_rank(w);
        total += (uint32_t)__popcll(w);
      }
      if (total == 0) return;
      uint32_t base = 0;
      if (lane == 0) base = atomicAdd(&s_cnt[c3], total);
      base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
      for (int j = 0; j < U; ++j)
        if (mine[j]) {
          levels[v[j]] = (int32_t)(L + 1);
          s_q[nxt][base + before[j]] = (uint16_t)v[j];
        }
    };
    const bool by_edge = (qs << lg) <= kSmallBlock;
    const uint32_t g = by_edge ? lg : 0u;
    for (uint32_t i = t >> g; i - (lane >> g) < qs; i += kSmallBlock >> g) {  // the same rounds for the whole wave
      uint32_t x = 0, e = 0;
      if (i < qs) {
        const uint32_t u = s_q[cur][i];
        x = s_rp[u] + (t & ((1u << g) - 1));
        e = s_rp[u + 1];
        if ((t & ((1u << g) - 1)) == 0) insp += e - x;
      }
      if (by_edge) {
        for (; ballot(x < e); x += 1u << g) {
          const uint32_t v[1] = {x < e ? col[x] : 0xffffffffu};
          visit(v);
        }
      } else {
        for (; ballot(x < e); x += 4) {
          uint32_t v[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = x + j < e ? col[x + j] : 0xffffffffu;
          visit(v);
        }
      }
    }
    lds_barrier();
  }
  if (!out) return;
  const unsigned long long ti = block_sum<kSmallBlock, unsigned long long>(insp, s_red);
  const unsigned long long tr = block_sum<kSmallBlock, unsigned long long>(reached, s_red);
  if (t == 0) {
    out[0] = L;
    out[1] = ti;
    out[2] = tr;
  }
}

static bool small_bfs_fits(const olv_graph *g, unsigned flags) {
  return g->n <= kSmallN && g->max_outdeg <= kSmallMaxDeg &&
         !(flags & (OLV_PERSISTENT | OLV_HOST_LOOP | OLV_FORCE_BOTTOM_UP));
}

static int bfs_small(const olv_graph *g, const std::vector<uint32_t> &seeds, int32_t *levels, bool host,
                     olv_stats *st) {
  const uint32_t k = (uint32_t)seeds.size();
  DevBuf d_seeds, d_out, d_levels;
  if (k > 1) {
    OLV_TRY(d_seeds.alloc((size_t)k * 4));
    OLV_HIP(hipMemcpyAsync(d_seeds.p, seeds.data(), (size_t)k * 4, hipMemcpyHostToDevice, stream()));
  }
  if (st) OLV_TRY(d_out.alloc(3 * sizeof(unsigned long long)));
  int32_t *outl = levels;
  if (host) {
    OLV_TRY(d_levels.alloc((size_t)g->n * 4));
    outl = d_levels.as<int32_t>();
  }
  uint32_t lg = 0;  // lanes per row: the mean degree rounded up to a power of two
  while (lg < 6 && ((uint64_t)g->n << lg) < g->m) ++lg;
  std::unique_ptr<Timer> t(st ? new Timer() : nullptr);
  if (t) t->start();
  hipLaunchKernelGGL(bfs_small_kernel, dim3(1), dim3(kSmallBlock), 0, stream(), g->row_ptr, g->col, g->n, lg,
                     d_seeds.as<uint32_t>(), k, seeds[0], outl, d_out.as<unsigned long long>());
  OLV_HIP(hipGetLastError());
  if (t) t->stop();
  unsigned long long h[3];
  if (st) OLV_HIP(hipMemcpyAsync(h, d_out.p, sizeof(h), hipMemcpyDeviceToHost, stream()));
  OLV_HIP(hipStreamSynchronize(stream()));
  if (host) OLV_HIP(hipMemcpy(levels, outl, (size_t)g->n * 4, hipMemcpyDeviceToHost));
  if (st) {
    std::memset(st, 0, sizeof(*st));
    st->elapsed_ms = t->ms();
    st->iterations = (uint32_t)h[0];
    st->edges_inspected = h[1];
    st->edges_traversed = h[1];
    st->vertices_reached = h[2];
  }
  return OLV_OK;
}

// Multi-source BFS on g (levels = distance to the nearest seed).
// seeds_host: seeds is a host array (levels follow OLV_PTR_HOST in flags).
// Direction-optimising runs go to g's twin -- g renumbered by descending
// in-degree, so hubs and their visited bytes sit together, and in-lists
// start with the hubs -- whose level stores go through the twin's out_map
// straight to g's numbering.  BFS levels do not depend on the numbering, so
// they are the same values.  OLV_GRAPH_ORDER (or OLV_NO_DIRECTION_OPT) runs
// on g itself.
int bfs_multisource(const olv_graph *g0, const uint32_t *seeds, uint32_t k, bool seeds_host, int32_t *levels,
                    unsigned flags, olv_stats *st) {
  if (!g0 || !seeds || !levels) return fail(OLV_EINVAL, "olv_bfs: NULL argument");
  if (k == 0) return fail(OLV_EINVAL, "olv_bfs: no source");
  const bool host = (flags & OLV_PTR_HOST) != 0;
  std::vector<uint32_t> h_seeds(k);
  if (seeds_host) std::memcpy(h_seeds.data(), seeds, (size_t)k * 4);
  else OLV_HIP(hipMemcpy(h_seeds.data(), seeds, (size_t)k * 4, hipMemcpyDeviceToHost));
  for (uint32_t i = 0; i < k; ++i)
    if (h_seeds[i] >= g0->n) return fail(OLV_EINVAL, "olv_bfs: source %u out of range (n=%u)", h_seeds[i], g0->n);
  const bool can_bu = !(flags & OLV_NO_DIRECTION_OPT);
  if (!can_bu && (flags & OLV_FORCE_BOTTOM_UP))
    return fail(OLV_EINVAL, "olv_bfs: OLV_FORCE_BOTTOM_UP and OLV_NO_DIRECTION_OPT together");
  if (small_bfs_fits(g0, flags)) return bfs_small(g0, h_seeds, levels, host, st);
  const bool twin = can_bu && !(flags & OLV_GRAPH_ORDER);
  const olv_graph *g = g0;
  if (twin) {
    olv_graph *gm = const_cast<olv_graph *>(g0);
    OLV_TRY(ensure_twin(gm));
    gm->twin->tune = gm->tune;
    for (uint32_t &s : h_seeds) s = gm->h_rl_pi[s];
    g = gm->twin;
  }
  BfsWork *w = nullptr;
  OLV_TRY(bfs_prepare(g, can_bu, &w));
  w->force_bu = (flags & OLV_FORCE_BOTTOM_UP) != 0;
  DevBuf d_seeds, d_levels;
  if (k > 1) {
    OLV_TRY(d_seeds.alloc((size_t)k * 4));
    OLV_HIP(hipMemcpyAsync(d_seeds.p, h_seeds.data(), (size_t)k * 4, hipMemcpyHostToDevice, stream()));
  }
  int32_t *out = levels;
  if (host) {
    OLV_TRY(d_levels.alloc((size_t)g->n * 4));
    out = d_levels.as<int32_t>();
  }
  std::unique_ptr<Timer> t(st ? new Timer() : nullptr);
  if (t) t->start();
  OLV_TRY(bfs_enqueue_init(g, w, d_seeds.as<uint32_t>(), k, h_seeds[0], out, can_bu));
  if (flags & OLV_PERSISTENT) {
    OLV_TRY(enqueue_persistent(g, w, out, can_bu));
    if (t) t->stop();
    OLV_TRY(bfs_result(w, nullptr, nullptr));
    GridBar hb;
    OLV_HIP(hipMemcpy(&hb, w->bar, sizeof(hb), hipMemcpyDeviceToHost));
    if (hb.err || !w->h_ctl->done) return fail(OLV_EINTERNAL, "olv_bfs: grid barrier timed out (co-residency lost)");
  } else {
    // first chunk: the most launch pairs of the last few runs (traversals of
    // one graph from different sources have similar depths); longer runs
    // continue in doubling chunks after one host check
    const uint32_t recent_max = std::max(std::max(w->recent[0], w->recent[1]), std::max(w->recent[2], w->recent[3]));
    OLV_TRY(run_pipeline(g, w, out, can_bu, std::max(w->deep ? 1u : 4u, recent_max), (flags & OLV_HOST_LOOP) != 0,
                         t.get()));
  }
  const uint32_t levels_run = w->h_ctl->levels, bu_levels = w->h_ctl->nbu;
  const double ms = t ? t->ms() : 0.0;
  if (w->h_ctl->overflow) return fail(OLV_EINTERNAL, "olv_bfs: more than n levels");
  if (host) OLV_HIP(hipMemcpy(levels, out, (size_t)g->n * 4, hipMemcpyDeviceToHost));
  if (st) {
    std::memset(st, 0, sizeof(*st));
    st->elapsed_ms = ms;
    st->iterations = levels_run;
    st->bottom_up_levels = bu_levels;
    st->edges_inspected = w->h_ctl->inspected;
    OLV_TRY(collect_stats(g0, w, out, st));  // levels are in g0's numbering
  }
  return OLV_OK;
}

}  // namespace olv

using namespace olv;

extern "C" int olv_bfs(const olv_graph *g, uint32_t src, int32_t *levels, unsigned flags, olv_stats *st) {
  if (!g) return fail(OLV_EINVAL, "olv_bfs: NULL graph");
  if (src >= g->n) return fail(OLV_EINVAL, "olv_bfs: source %u out of range (n=%u)", src, g->n);
  return bfs_multisource(g, &src, 1, true, levels, flags, st);
}

// ------------------------------------------------ allocation-free entry point
// olv_bfs_noalloc keeps every work buffer of a traversal (visited bytes,
// snapshot and frontier bitmaps, queue, hub items, control block, barrier,
// statistics) in one static device array per GPU instead of
// buffers allocated with the graph.  The host code only ever uses the array's
// device address, obtained once per device with hipGetSymbolAddress.
namespace olv {
constexpr size_t kNoAllocScratchBytes = size_t(32) << 20;
}  // namespace olv

static __device__ __align__(256) unsigned char scratch[olv::kNoAllocScratchBytes];

namespace olv {
namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned char *g_scratch_ptr[kMaxDevices] = {};

struct NoAllocLayout {
  size_t visited, snap, bms, queue, hubs, ctl, bar, stat, total;
  uint32_t nw, nwp;
};

NoAllocLayout noalloc_layout(uint32_t n, uint64_t m) {
  auto al = [](size_t x) { return (x + 255) / 256 * 256; };
  NoAllocLayout L;
  L.nw = (n + 31) / 32;
  L.nwp = (L.nw + 63) / 64 * 64;
  size_t o = 0;
  L.visited = o;
  o += al((size_t)L.nwp * 32);
  L.snap = o;
  o += al((size_t)L.nwp * 4);
  L.bms = o;
  o += al((size_t)L.nwp * 8);
  L.queue = o;
  o += al(std::max<size_t>(n, 1) * 4);
  L.hubs = o;
  o += al(hub_capacity(m) * sizeof(uint2));
  L.ctl = o;
  o += al(sizeof(BfsCtl));
  L.bar = o;
  o += al(sizeof(GridBar));
  L.stat = o;
  o += al(2 * sizeof(unsigned long long));
  L.total = o;
  return L;
}
}  // namespace

// The current device's copy of `scratch` (its address looked up once per
// device, with that device current).
int noalloc_scratch(unsigned char **out) {
  const int dev = current_device();
  if (dev < 0 || dev >= kMaxDevices) return fail(OLV_EUNSUPPORTED, "device %d beyond the %d supported", dev, kMaxDevices);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      (void)hipGetLastError();
      return fail(OLV_EHIP, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
    }
    g_scratch_ptr[dev] = static_cast<unsigned char *>(p);
  }
  *out = g_scratch_ptr[dev];
  return OLV_OK;
}

}  // namespace olv

extern "C" int olv_bfs_noalloc(const olv_graph *g, uint32_t src, int32_t *levels, unsigned flags, olv_stats *st) {
  if (!g || !levels) return fail(OLV_EINVAL, "olv_bfs_noalloc: NULL argument");
  if (src >= g->n) return fail(OLV_EINVAL, "olv_bfs_noalloc: source %u out of range (n=%u)", src, g->n);
  if (flags & OLV_PTR_HOST) return fail(OLV_EINVAL, "olv_bfs_noalloc: levels must be a device pointer");
  if (flags & OLV_PERSISTENT) return fail(OLV_EINVAL, "olv_bfs_noalloc: OLV_PERSISTENT is not supported");
  const bool can_bu = !(flags & OLV_NO_DIRECTION_OPT);
  if (!can_bu && (flags & OLV_FORCE_BOTTOM_UP))
    return fail(OLV_EINVAL, "olv_bfs_noalloc: OLV_FORCE_BOTTOM_UP and OLV_NO_DIRECTION_OPT together");
  if (can_bu && (!g->in_row_ptr || !g->in_head))
    return fail(OLV_EINVAL,
                "olv_bfs_noalloc: the graph has no in-edge CSR with in-list heads (create it with "
                "OLV_BUILD_TRANSPOSE and run olv_bfs on it once, or pass OLV_NO_DIRECTION_OPT)");
  const NoAllocLayout L = noalloc_layout(g->n, g->m);
  if (L.total > kNoAllocScratchBytes)
    return fail(OLV_ERANGE, "olv_bfs_noalloc: the graph needs %zu bytes of work memory, the static scratch holds %zu "
                            "(n=%u, m=%u)",
                L.total, kNoAllocScratchBytes, g->n, g->m);
  unsigned char *base = nullptr;
  OLV_TRY(noalloc_scratch(&base));
  BfsWork w;  // views into the scratch array; nothing here is freed
  BfsCtl hctl;
  w.n = g->n;
  w.nw = L.nw;
  w.nwp = L.nwp;
  w.visited = base + L.visited;
  w.snap = reinterpret_cast<uint32_t *>(base + L.snap);
  w.bms = reinterpret_cast<uint32_t *>(base + L.bms);
  w.queue = reinterpret_cast<uint32_t *>(base + L.queue);
  w.hubs = reinterpret_cast<uint2 *>(base + L.hubs);
  w.ctl = reinterpret_cast<BfsCtl *>(base + L.ctl);
  w.bar = reinterpret_cast<GridBar *>(base + L.bar);
  w.stat = reinterpret_cast<unsigned long long *>(base + L.stat);
  w.h_ctl = &hctl;
  w.force_bu = (flags & OLV_FORCE_BOTTOM_UP) != 0;
  const auto t0 = std::chrono::steady_clock::now();
  OLV_TRY(bfs_enqueue_init(g, &w, nullptr, 1, src, levels, can_bu));
  OLV_TRY(run_pipeline(g, &w, levels, can_bu, 8u, (flags & OLV_HOST_LOOP) != 0, nullptr));
  const uint32_t levels_run = hctl.levels, bu_levels = hctl.nbu;
  const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  if (hctl.overflow) return fail(OLV_EINTERNAL, "olv_bfs_noalloc: more than n levels");
  if (st) {
    std::memset(st, 0, sizeof(*st));
    st->elapsed_ms = ms;
    st->iterations = levels_run;
    st->bottom_up_levels = bu_levels;
    st->edges_inspected = hctl.inspected;
    OLV_TRY(collect_stats(g, &w, levels, st));
  }
  return OLV_OK;
}
