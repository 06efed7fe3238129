// Single- and multi-source shortest paths over int32 weights: frontier
// relaxation.
//
// The reference SSSP (SSSP.cu:146-163) alternates edgeFilter (reset every
// accumulator to INF, gather dist[u] + w, atomicMin into acc[v], flag v;
// oliver.h:56-83) and vertexFilter (if dist[v] > acc[v]: dist[v] = acc[v],
// enqueue v; oliver.h:92-113) until the queue is empty, capped at n rounds
// (negative-cycle guard, SSSP.cu:153-157).  Shortest distances are unique,
// so relaxing straight into dist with atomicMin -- no accumulator array, no
// per-round O(V) reset -- reaches the same fixed point: a vertex whose
// distance dropped this round is marked and expanded next round.
//
// Near-far ordering (Davidson et al., IPDPS'14): with a split distance T, an
// improved vertex joins the next round's frontier only if its new distance
// is below T; otherwise it stays marked.  When the near frontier runs dry, T
// moves to the smallest marked distance + delta and the marked vertices below
// it form the next frontier.  Vertices are then mostly expanded once with
// their final distance instead of once per improvement, and the fixed point --
// hence every distance -- is the same.
// Negative weights turn the ordering off (plain rounds, so the reference's
// n-round negative-cycle rule applies unchanged).
//
// A vertex whose distance dropped is marked with a plain byte store: the
// bitmap atomics that marked it before cost as much as the distance atomics
// and serialised on the words of an RMAT graph's hubs, and extracting a
// frontier from them took a lane per 32 vertices (RMAT 250K x 4M: 16-28 us per
// large round; 5-7 from the bytes).
//
// k sources run as k instances over one shared CSR: instance s owns virtual
// vertices s*n .. s*n+n-1 (dist row s), so one launch per round relaxes all
// k frontiers together.  Rounds are a relax kernel and a compact kernel
// whose control lives on the device (as for BFS); OLV_PERSISTENT runs all
// rounds (plain, without the near-far split) in one cooperative kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstddef>
#include <cstring>
#include <type_traits>
#include <vector>

#include "bfs_core.hpp"
#include "internal.hpp"

namespace olv {

constexpr int kSBlock = 256;
constexpr uint32_t kSSpin = 1u << 24;

// A marked vertex has a distance not expanded yet: kMarkNew, lowered since the
// last compaction; kMarkFar, at or above the split then.
constexpr uint8_t kMarkNew = 1, kMarkFar = 2;

// Candidate copies.  A relaxation probes dist and lowers a candidate kept
// apart from it: an atomic is performed at the memory side and takes the line
// from the caches that the other relaxations probe.  Atomics to one address
// also serialise there (about 12 ns each), and in a large round of an RMAT
// graph many relaxations improve on the same hub, so workgroup b lowers copy
// b % kCopies; the compaction, a launch later, takes the smallest of a marked
// vertex's copies.  RMAT 250K x 4M: 601 us lowering dist itself, 502, 474, 452,
// 455 with 1, 2, 4, 8 copies; RMAT 1M x 8M 605 and 582.  Past 1M vertices the
// copies no longer stay cached (RMAT 2M x 16M: 1458 and 1418; 4M x 32M: 1532 and
// 2040), and without hubs they gain nothing from 600K on (uniform, 8 edges a
// vertex: 500K 743 and 674 us, 700K 780 and 765, 800K 769 and 788, 1M 882 and
// 947), so relaxations lower dist there.
constexpr uint32_t kCopies = 4;
constexpr uint64_t kCopiesHubs = 1u << 20, kCopiesNoHubs = 600000;  // vertices, at most
constexpr uint32_t kWideWords = 4;  // words of mark bytes a lane compacts without copies
static bool with_copies(const olv_graph *g, uint64_t nv) {
  return nv <= (g->max_outdeg >= g->tune.hub_thr ? kCopiesHubs : kCopiesNoHubs);
}

template <bool Multi>
struct SsspVisitor {
  using P = typename std::conditional<Multi, unsigned long long, int32_t>::type;
  const uint32_t *col;
  const int32_t *w;
  const int32_t *dist;
  int32_t *low;  // what relaxations lower: dist, or this workgroup's copy of the candidates
  uint8_t *mark;
  uint32_t n;
  __device__ SsspVisitor(const uint32_t *c, const int32_t *ww, const int32_t *d, int32_t *lo, uint8_t *mk, uint32_t nn)
      : col(c), w(ww), dist(d), low(lo), mark(mk), n(nn) {}
  __device__ __forceinline__ uint32_t row(uint32_t q) const { return Multi ? q % n : q; }
  __device__ __forceinline__ P load(uint32_t q) const {
    if constexpr (Multi)
      return ((unsigned long long)(q - q % n) << 32) | (unsigned long long)(uint32_t)dist[q];
    else
      return dist[q];
  }
  // target of edge e: (vertex, candidate distance)
  __device__ __forceinline__ uint2 tgt(uint32_t e, P pl) const {
    int32_t du;
    uint32_t base;
    if constexpr (Multi) {
      du = (int32_t)(uint32_t)pl;
      base = (uint32_t)(pl >> 32);
    } else {
      du = pl;
      base = 0;
    }
    return make_uint2(base + col[e], (uint32_t)du + (uint32_t)w[e]);
  }
  __device__ __forceinline__ int32_t state(uint2 t) const { return dist[t.x]; }
  // Relax: lower v and mark it.  No lane waits on the atomic: a relaxation
  // that loses a race to a lower distance still marks v, which only re-expands
  // v with its final distance.
  __device__ __forceinline__ void apply(uint2 t, int32_t cur, P) {
    const int32_t cand = (int32_t)t.y;
    if (cand >= cur) return;
    __hip_atomic_fetch_min(&low[t.x], cand, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    mark[t.x] = kMarkNew;
  }
};

enum : uint32_t { kModeNear = 0, kModeResplit = 1, kModeDone = 2 };

// Smallest marked distance at or above the split, one copy per 128-byte line
// (workgroup b updates copy b % kCtrSlots).  Exact after a round that moved the
// split; until the next one it may stand for a vertex that has since been
// lowered below the split, and a re-split from it then promotes less, at worst
// nothing, and leaves the exact one.
struct alignas(128) MinSlot {
  int32_t v;
  uint32_t pad[31];
};

struct SsspCtl {
  uint32_t done;
  uint32_t rounds;    // result
  uint32_t capped;    // result: max_rounds without convergence
  uint32_t round;     // next round to relax (written by compact)
  uint32_t round_e;   // round being compacted (written by relax)
  uint32_t pad;
  unsigned long long relax;  // result: edges read
  uint32_t mode[2];   // mode of round R, slot R & 1
  int32_t split[2];   // split that the frontier of round R was built with
  uint32_t qfill[2];  // frontier queue length of round R, slot R & 1
  uint32_t hfill[2];  // hub items of round R, slot R & 1
  MinSlot minfar[2][kCtrSlots];
  CtrSet cnt[2];      // edges read by round R, slot R & 1
};
constexpr size_t kSsspCtlHead = offsetof(SsspCtl, mode);  // what the host reads back

struct SsspParams {
  const uint32_t *row_ptr;
  const uint32_t *col;
  const int32_t *w;
  int32_t *dist;     // ninst x n
  uint32_t *queue;   // virtual ids
  uint2 *hubs;       // hub items (virtual id, chunk)
  uint8_t *mark;     // one byte per vertex (padded to 4): kMarkNew, kMarkFar or 0
  int32_t *cand;     // kCopies x nv candidates, or nullptr: relaxations lower dist
  SsspCtl *ctl;
  GridBar *bar;
  int32_t delta;     // near-far step (0: plain rounds)
  uint32_t n, ninst, nv;
  uint32_t wave_thr, block_thr, hub_thr;
  uint32_t max_rounds;
};

// Virtual id -> CSR row.
struct ModRow {
  uint32_t n;
  __device__ __forceinline__ uint32_t operator()(uint32_t v) const { return v % n; }
};

template <bool Multi, bool Copies>
__device__ __forceinline__ void sssp_round(const SsspParams &p, uint32_t qsize, uint32_t nhubs, uint32_t vb,
                                           uint32_t nvb, unsigned long long &insp) {
  SsspVisitor<Multi> vis(p.col, p.w, p.dist, Copies ? p.cand + (size_t)(vb % kCopies) * p.nv : p.dist, p.mark, p.n);
  push_expand<kSBlock>(p.queue, qsize, p.hubs, nhubs, p.row_ptr, p.wave_thr, p.block_thr, p.hub_thr, vb, nvb, vis,
                       insp);
}

// Marked vertices with a distance below `split` -> queue and hub items (their
// marks cleared); the smallest other marked distance -> *minfar.  Where the
// split has not moved (`all` false) vertices marked far stay so, and only those
// lowered since are looked at.  A lane takes W consecutive words of four mark
// bytes.  W = 1 with candidate copies, where a vertex costs five loads and lanes
// are few; else W = kWideWords, and a workgroup collects its vertices in LDS:
// its place in the queue comes from an atomic, and one for every 1024 vertices,
// 12 ns each after another, made a compaction of 16.7M vertices 195 us whatever
// it found (85 to 110 with W = 4, 25 to 50 collected and without the far ones).
// Relaxed directly, 16.7M vertices with 67M edges 8.4 -> 4.8 ms a call, 5M with
// 40M 3.33 -> 2.46.
template <int BLOCK, uint32_t W>
__device__ void sssp_take(const SsspParams &p, int32_t split, bool all, uint32_t *qcount, uint32_t *hcount,
                          int32_t *minfar, uint32_t vb, uint32_t nvb) {
  const uint32_t look = all ? 0xffffffffu : 0x01010101u * kMarkNew;
  constexpr uint32_t kHold = W > 1 ? BLOCK * 4 * W : 1;
  __shared__ uint32_t s_hold[kHold];
  uint32_t held = 0;  // entries in s_hold
  auto flush = [&]() {
    __shared__ uint32_t s_at;
    __syncthreads();
    if (threadIdx.x == 0) s_at = atomicAdd(qcount, held);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < held; i += BLOCK) p.queue[s_at + i] = s_hold[i];
    __syncthreads();
    held = 0;
  };
  __shared__ uint32_t s_scan[BLOCK / kWave + 1];
  __shared__ uint32_t s_base;
  __shared__ int32_t s_mf[BLOCK / kWave];
  const ModRow row{p.n};
  const uint32_t nw = (p.nv + 3) / 4;
  uint32_t *words = reinterpret_cast<uint32_t *>(p.mark);
  int32_t mf = kInf;
  for (uint64_t w0 = (uint64_t)vb * BLOCK * W; w0 < nw; w0 += (uint64_t)nvb * BLOCK * W) {
    const uint32_t wl = (uint32_t)w0 + threadIdx.x * W;  // this lane's first word
    uint32_t word[W], take = 0;  // take: bit b, vertex 4 wl + b goes to the queue
#pragma unroll
    for (uint32_t i = 0; i < W; ++i) word[i] = wl + i < nw ? words[wl + i] : 0u;
#pragma unroll
    for (uint32_t i = 0; i < W; ++i) {
      const uint32_t seen = word[i] & look;
      if (!seen) continue;
      const uint32_t w = wl + i;
      uint32_t keep = word[i];
      int32_t d[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) d[b] = (seen >> (8 * b)) & 0xffu ? p.dist[w * 4u + b] : kInf;
      if (p.cand) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          if (!((seen >> (8 * b)) & kMarkNew)) continue;
          int32_t c[kCopies], m = d[b];
#pragma unroll
          for (uint32_t x = 0; x < kCopies; ++x) c[x] = p.cand[(size_t)x * p.nv + w * 4u + b];
#pragma unroll
          for (uint32_t x = 0; x < kCopies; ++x) m = c[x] < m ? c[x] : m;
          if (m < d[b]) p.dist[w * 4u + b] = d[b] = m;
        }
      }
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        if (!((seen >> (8 * b)) & 0xffu)) continue;
        keep &= ~(0xffu << (8 * b));
        if (d[b] >= split) {
          mf = d[b] < mf ? d[b] : mf;
          keep |= (uint32_t)kMarkFar << (8 * b);
          continue;
        }
        const uint32_t x = w * 4u + b, u = p.ninst > 1 ? row(x) : x;
        const uint32_t deg = p.row_ptr[u + 1] - p.row_ptr[u];
        if (deg >= p.hub_thr) {
          const uint32_t k = (deg + p.hub_thr - 1) / p.hub_thr;
          const uint32_t hb = atomicAdd(hcount, k);
          for (uint32_t j = 0; j < k; ++j) p.hubs[hb + j] = make_uint2(x, j);
        } else {
          take |= 1u << (4 * i + b);
        }
      }
      if (keep != word[i]) words[w] = keep;
    }
    uint32_t total;
    const uint32_t off = block_exclusive_scan<BLOCK>((uint32_t)__popc(take), s_scan, &total);
    if constexpr (W > 1) {
      if (held + total > kHold) flush();
      uint32_t pos = held + off;
      for (uint32_t x = take; x; x &= x - 1) s_hold[pos++] = wl * 4u + __ffs(x) - 1;
      held += total;
    } else {
      if (threadIdx.x == 0) s_base = total ? atomicAdd(qcount, total) : 0u;
      __syncthreads();
      uint32_t pos = s_base + off;
      for (uint32_t x = take; x; x &= x - 1) p.queue[pos++] = wl * 4u + __ffs(x) - 1;
      __syncthreads();
    }
  }
  if (held) flush();
  mf = wave_min(mf);
  if (lane_id() == 0) s_mf[threadIdx.x / kWave] = mf;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < BLOCK / kWave; ++i) mf = s_mf[i] < mf ? s_mf[i] : mf;
    if (mf < kInf) atomicMin(minfar, mf);
  }
}

// Round R: decide from the frontier that the last compaction built (its
// vertices, or none: re-split past the smallest marked distance, or done) and
// relax it.
template <bool Multi, bool Copies>
__global__ void __launch_bounds__(kSBlock) sssp_relax_kernel(SsspParams p) {
  SsspCtl *ctl = p.ctl;
  if (__hip_atomic_load(&ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const uint32_t R = ctl->round, t = threadIdx.x;
  const uint32_t qsize = ctl->qfill[R & 1], nhubs = ctl->hfill[R & 1];
  if (blockIdx.x == 0) {
    __shared__ int32_t s_mf;
    const int32_t far = t < kCtrSlots ? ctl->minfar[R & 1][t].v : kInf;
    if (t < kWave) {
      const int32_t mf = wave_min(far);
      if (t == 0) s_mf = mf;
    }
    __syncthreads();
    const uint32_t mode = (qsize + nhubs) ? kModeNear : (s_mf < kInf ? kModeResplit : kModeDone);
    if (t == 0) {
      const int32_t split = ctl->split[R & 1];
      ctl->round_e = R;
      ctl->mode[R & 1] = mode;
      ctl->split[(R + 1) & 1] = mode == kModeNear ? split : (s_mf > kInf - p.delta ? kInf : s_mf + p.delta);
      ctl->qfill[(R + 1) & 1] = 0;
      ctl->hfill[(R + 1) & 1] = 0;
      if (mode == kModeDone || R >= p.max_rounds) {
        ctl->rounds = R;
        ctl->capped = mode != kModeDone;
        ctl->done = 1u;
      }
    }
    if (t < kCtrSlots) ctl->minfar[(R + 1) & 1][t].v = mode == kModeNear ? far : kInf;
  }
  if (qsize + nhubs == 0 || R >= p.max_rounds) return;
  unsigned long long insp = 0;
  sssp_round<Multi, Copies>(p, qsize, nhubs, blockIdx.x, gridDim.x, insp);
  flush_counters<kSBlock>(&ctl->cnt[R & 1], 0u, 0ull, insp);
}

template <uint32_t W>
__global__ void __launch_bounds__(kSBlock) sssp_compact_kernel(SsspParams p) {
  SsspCtl *ctl = p.ctl;
  if (__hip_atomic_load(&ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const uint32_t R = ctl->round_e;
  if (blockIdx.x == 0) {
    const CtrSum c = ctr_total(&ctl->cnt[R & 1]);
    if (threadIdx.x == 0) {
      ctl->relax += c.inspected;
      ctl->round = R + 1;
    }
    ctr_clear(&ctl->cnt[(R + 1) & 1]);
  }
  sssp_take<kSBlock, W>(p, ctl->split[(R + 1) & 1], ctl->mode[R & 1] != kModeNear, &ctl->qfill[(R + 1) & 1],
                        &ctl->hfill[(R + 1) & 1], &ctl->minfar[(R + 1) & 1][blockIdx.x % kCtrSlots].v, blockIdx.x,
                        gridDim.x);
}

// All rounds (plain: every marked vertex is expanded) in one cooperative
// launch.
template <bool Multi>
__global__ void __launch_bounds__(kSBlock) sssp_persistent_kernel(SsspParams p) {
  GridBarLocal gb;
  if (!gbar_init(p.bar, gb, gridDim.x, kSSpin)) return;
  SsspCtl *ctl = p.ctl;
  const uint32_t vb = blockIdx.x, nvb = gridDim.x;
  const bool lead = vb == 0 && threadIdx.x == 0;
  unsigned long long insp = 0;
  for (uint32_t R = 0;; ++R) {
    const uint32_t qsize = __hip_atomic_load(&ctl->qfill[R & 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t nhubs = __hip_atomic_load(&ctl->hfill[R & 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (qsize + nhubs == 0 || R >= p.max_rounds) {
      if (lead) {
        ctl->rounds = R;
        ctl->capped = qsize + nhubs != 0;
        ctl->done = 1u;
      }
      break;
    }
    if (lead) {
      ctl->qfill[(R + 1) & 1] = 0;
      ctl->hfill[(R + 1) & 1] = 0;
    }
    sssp_round<Multi, false>(p, qsize, nhubs, vb, nvb, insp);
    if (!grid_barrier(p.bar, gb, kSSpin)) break;
    sssp_take<kSBlock, 1>(p, kInf, true, &ctl->qfill[(R + 1) & 1], &ctl->hfill[(R + 1) & 1],
                          &ctl->minfar[0][vb % kCtrSlots].v, vb, nvb);
    if (!grid_barrier(p.bar, gb, kSSpin)) break;
  }
  __shared__ unsigned long long s_red[kSBlock / kWave];
  const unsigned long long total = block_sum<kSBlock, unsigned long long>(insp, s_red);
  if (threadIdx.x == 0 && total) atomicAdd(&ctl->relax, total);
}

// dist and candidates = INF, marks/control/barrier = 0, minfar = INF, split = delta.  With a
// single source (k == 1: src) the seeding is done here as well -- its
// distance by the lane that owns it, the frontier by workgroup 0 after
// clearing the control block -- one launch instead of two.
__global__ void sssp_reset_kernel(SsspParams p, uint32_t src) {
  const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  const bool one = p.ninst == 1;
  for (size_t i = tid; i < p.nv; i += stride) p.dist[i] = one && i == src ? 0 : kInf;
  for (size_t i = tid; i < ((size_t)p.nv + 3) / 4; i += stride) reinterpret_cast<uint32_t *>(p.mark)[i] = 0u;
  if (p.cand)
    for (size_t i = tid; i < (size_t)p.nv * kCopies; i += stride) p.cand[i] = kInf;
  if (blockIdx.x != 0) return;
  for (uint32_t i = threadIdx.x; i < sizeof(SsspCtl) / 4; i += blockDim.x) reinterpret_cast<uint32_t *>(p.ctl)[i] = 0u;
  for (uint32_t i = threadIdx.x; i < sizeof(GridBar) / 4; i += blockDim.x) reinterpret_cast<uint32_t *>(p.bar)[i] = 0u;
  __syncthreads();
  if (threadIdx.x < 2 * kCtrSlots) p.ctl->minfar[threadIdx.x / kCtrSlots][threadIdx.x % kCtrSlots].v = kInf;
  if (threadIdx.x == 0) p.ctl->split[0] = p.delta > 0 ? p.delta : kInf;
  if (!one) return;
  unsigned long long deg;
  seed_frontier(&src, 1u, p.row_ptr, p.hub_thr, p.queue, &p.ctl->qfill[0], p.hubs, &p.ctl->hfill[0],
                [&](uint32_t) -> uint32_t { return src; }, ModRow{p.n}, &deg);
}

// One workgroup: instance s starts from virtual vertex s*n + srcs[s].
__global__ void sssp_seed_kernel(const uint32_t *__restrict__ srcs, uint32_t k, SsspParams p) {
  auto claim = [&](uint32_t s) -> uint32_t {
    const uint32_t x = s * p.n + srcs[s];
    p.dist[x] = 0;
    return x;
  };
  unsigned long long deg;
  seed_frontier(srcs, k, p.row_ptr, p.hub_thr, p.queue, &p.ctl->qfill[0], p.hubs, &p.ctl->hfill[0], claim,
                ModRow{p.n}, &deg);
}

// Work arrays for up to k instances, kept on the graph for the next call
// (allocating them took 0.35 ms of every call).
struct SsspWork {
  uint32_t k = 0;
  uint64_t cand_nv = 0;  // virtual vertices that the candidate copies have room for
  size_t bytes = 0;      // of queue, marks and hub items
  uint32_t *queue = nullptr;
  uint8_t *mark = nullptr;
  int32_t *cand = nullptr;
  uint2 *hubs = nullptr;
  SsspCtl *ctl = nullptr, *h_ctl = nullptr;
  GridBar *bar = nullptr;
  ~SsspWork() {
    void *ps[] = {queue, mark, cand, hubs, ctl, bar};
    for (void *p : ps)
      if (p) (void)hipFree(p);
    if (h_ctl) (void)hipHostFree(h_ctl);
  }
  int alloc(uint64_t nv, uint32_t kk, uint64_t m) {
    k = kk;
    const size_t hb = hub_capacity(m) * k * sizeof(uint2);
    bytes = (size_t)nv * 5 + hb;
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&queue), (size_t)nv * 4));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&mark), ((size_t)nv + 3) / 4 * 4));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&hubs), hb));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&ctl), sizeof(SsspCtl)));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&bar), sizeof(GridBar)));
    OLV_HIP(hipHostMalloc(reinterpret_cast<void **>(&h_ctl), sizeof(SsspCtl), hipHostMallocDefault));
    return OLV_OK;
  }
  int alloc_copies(uint64_t nv) {
    if (nv <= cand_nv) return OLV_OK;
    if (cand) (void)hipFree(cand);
    cand = nullptr;
    cand_nv = 0;
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&cand), (size_t)nv * kCopies * 4));
    cand_nv = nv;
    return OLV_OK;
  }
};
// Larger work is freed after the call: its allocation is little beside
// relaxing that many vertices.
constexpr size_t kSsspKeepBytes = size_t(4) << 30;

void free_sssp_work(olv_graph *g) { delete g->sssp.exchange(nullptr); }

static unsigned sgrid(size_t items, size_t per) {
  size_t b = (items + per - 1) / per;
  return (unsigned)std::max<size_t>(1, std::min(b, (size_t)cu_count() * 8));
}

// Minimum and mean of the int32 weights (one reduction, read back).
__global__ void wstat_kernel(const int32_t *__restrict__ w, uint32_t m, long long *__restrict__ out) {
  __shared__ long long s_red[256 / kWave];
  long long mn = LLONG_MAX, sum = 0;
  for (uint32_t e = blockIdx.x * blockDim.x + threadIdx.x; e < m; e += gridDim.x * blockDim.x) {
    const long long x = w[e];
    mn = x < mn ? x : mn;
    sum += x;
  }
  for (int o = kWave / 2; o > 0; o >>= 1) {
    const long long y = __shfl_xor(mn, o, kWave);
    mn = y < mn ? y : mn;
  }
  if (lane_id() == 0) s_red[threadIdx.x / kWave] = mn;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < 256 / kWave; ++i) mn = s_red[i] < mn ? s_red[i] : mn;
    atomicMin(&out[0], mn);
  }
  __syncthreads();
  sum = block_sum<256, long long>(sum, s_red);
  if (threadIdx.x == 0) atomicAdd(reinterpret_cast<unsigned long long *>(&out[1]), (unsigned long long)sum);
}

static int weight_stats(const int32_t *w, uint32_t m, int32_t *wmin, double *wmean) {
  long long h[2] = {LLONG_MAX, 0};
  DevBuf b;
  OLV_TRY(b.alloc(sizeof(h)));
  OLV_HIP(hipMemcpyAsync(b.p, h, sizeof(h), hipMemcpyHostToDevice, stream()));
  hipLaunchKernelGGL(wstat_kernel, dim3(sgrid(m, 256)), dim3(256), 0, stream(), w, m, b.as<long long>());
  OLV_HIP(hipMemcpyAsync(h, b.p, sizeof(h), hipMemcpyDeviceToHost, stream()));
  OLV_HIP(hipStreamSynchronize(stream()));
  *wmin = m ? (int32_t)h[0] : 0;
  *wmean = m ? (double)h[1] / m : 0.0;
  return OLV_OK;
}

// Near-far step: mean weight x the graph's sssp_delta_num (32 unless tuned)
// / mean out-degree; 0 (plain rounds) when a weight is negative.
static int sssp_delta(const olv_graph *g, const int32_t *w, int32_t *delta) {
  *delta = 0;
  if (!g->m || !g->n) return OLV_OK;
  int32_t wmin = 0;
  double wmean = 0.0;
  olv_graph *mg = const_cast<olv_graph *>(g);
  if (w == g->weights && mg->wstat_ready) {
    wmin = mg->wmin;
    wmean = mg->wmean;
  } else {
    OLV_TRY(weight_stats(w, g->m, &wmin, &wmean));
    if (w == g->weights) {
      mg->wmin = wmin;
      mg->wmean = wmean;
      mg->wstat_ready = true;
    }
  }
  if (wmin < 0) return OLV_OK;
  const double deg = (double)g->m / g->n;
  const double d = wmean * g->tune.sssp_delta_num / (deg > 1.0 ? deg : 1.0);
  *delta = d < 1.0 ? 1 : (d > 1e9 ? 1000000000 : (int32_t)(d + 0.5));
  return OLV_OK;
}

static int sssp_read(SsspWork &w) {
  OLV_HIP(hipMemcpyAsync(w.h_ctl, w.ctl, kSsspCtlHead, hipMemcpyDeviceToHost, stream()));
  OLV_HIP(hipStreamSynchronize(stream()));
  return OLV_OK;
}

// k instances from the host sources srcs[0..k); dist is k x n.
static int sssp_run(const olv_graph *g, const uint32_t *srcs, uint32_t k, const int32_t *weights, int32_t *dist,
                    unsigned flags, olv_stats *st) {
  const uint64_t nv = (uint64_t)k * g->n;
  if (nv >= (1ull << 32)) return fail(OLV_ERANGE, "sssp: %u sources x %u vertices exceed 2^32 ids", k, g->n);
  const bool multi = k > 1;
  olv_graph *gm = const_cast<olv_graph *>(g);
  hipStream_t s = stream();
  int32_t delta = 0;
  if (!(flags & OLV_PERSISTENT)) OLV_TRY(sssp_delta(g, weights, &delta));
  const bool binned = delta > 0 && !(flags & (OLV_PERSISTENT | OLV_SSSP_DIRECT)) && sssp_bin_fits(g, k);
  DevBuf ds;  // the sources, when they do not travel as an argument
  if (multi || binned) {
    OLV_TRY(ds.alloc((size_t)k * 4));
    OLV_HIP(hipMemcpyAsync(ds.p, srcs, (size_t)k * 4, hipMemcpyHostToDevice, s));
  }
  // destination binning (sssp_bin.hip) unless asked to relax directly
  if (binned) return sssp_bin_run(g, ds.as<uint32_t>(), k, weights, dist, delta, flags, st);
  WorkLease<SsspWork> lease(gm->sssp);
  const bool copies = with_copies(g, nv);
  if (!lease.w || lease.w->k < k) {
    lease.renew();
    OLV_TRY(lease.w->alloc(nv, k, g->m));
  }
  if (copies) OLV_TRY(lease.w->alloc_copies(nv));
  SsspWork *w = lease.w;
  SsspParams p;
  p.row_ptr = g->row_ptr;
  p.col = g->col;
  p.w = weights;
  p.dist = dist;
  p.queue = w->queue;
  p.hubs = w->hubs;
  p.mark = w->mark;
  p.cand = copies && !(flags & OLV_PERSISTENT) ? w->cand : nullptr;
  p.ctl = w->ctl;
  p.bar = w->bar;
  p.n = g->n;
  p.ninst = k;
  p.nv = (uint32_t)nv;
  p.wave_thr = g->tune.td_wave_thr;
  p.block_thr = g->tune.td_block_thr;
  p.hub_thr = g->tune.hub_thr;
  p.delta = delta;
  // plain rounds keep the reference's negative-cycle rule (n rounds); with
  // non-negative weights the cap only guards against a runaway loop
  p.max_rounds = delta ? (uint32_t)std::min<uint64_t>(4ull * g->n + 1024, 0xffffffffull) : g->n;
  Timer t;
  t.start();
  hipLaunchKernelGGL(sssp_reset_kernel, dim3(sgrid((size_t)nv * (p.cand ? kCopies : 1u), 256)), dim3(256), 0, s, p,
                     srcs[0]);
  if (multi) hipLaunchKernelGGL(sssp_seed_kernel, dim3(1), dim3(256), 0, s, ds.as<uint32_t>(), k, p);
  OLV_HIP(hipGetLastError());
  if (flags & OLV_PERSISTENT) {
    const void *fn = multi ? reinterpret_cast<const void *>(sssp_persistent_kernel<true>)
                           : reinterpret_cast<const void *>(sssp_persistent_kernel<false>);
    int per_cu = 0;
    OLV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, kSBlock, 0));
    if (per_cu <= 0) return fail(OLV_EUNSUPPORTED, "persistent SSSP kernel does not fit on a CU");
    void *args[] = {&p};
    OLV_HIP(hipLaunchCooperativeKernel(fn, dim3(cu_count()), dim3(kSBlock), args, 0, s));
    t.stop();
    OLV_TRY(sssp_read(*w));
    GridBar hb;
    OLV_HIP(hipMemcpy(&hb, w->bar, sizeof(hb), hipMemcpyDeviceToHost));
    if (hb.err || !w->h_ctl->done) return fail(OLV_EINTERNAL, "olv_sssp: grid barrier timed out (co-residency lost)");
  } else {
    // relax workgroups per CU: the graph's tuning
    const unsigned gr = (unsigned)cu_count() * g->tune.sssp_relax_per_cu;
    const bool wide = !p.cand;
    const unsigned gc = sgrid(((size_t)nv + 3) / 4, (size_t)kSBlock * (wide ? kWideWords : 1));
    // first chunk: the longest of the last few runs on this graph (8 at
    // first; a run of r rounds takes r + 1 launch pairs, and two runs may
    // differ by a round or two); longer runs continue in chunks of 8, 16, ...
    // after a host check
    uint32_t hist = 8;
    for (uint32_t r : gm->sssp_rounds) hist = std::max(hist, std::min(r + 3, 4096u));
    uint32_t chunk = (flags & OLV_HOST_LOOP) ? 1u : hist;
    uint32_t more = 4;
    uint64_t enq = 0;
    for (;;) {
      for (uint32_t i = 0; i < chunk; ++i) {
        if (p.cand && multi)
          hipLaunchKernelGGL((sssp_relax_kernel<true, true>), dim3(gr), dim3(kSBlock), 0, s, p);
        else if (p.cand)
          hipLaunchKernelGGL((sssp_relax_kernel<false, true>), dim3(gr), dim3(kSBlock), 0, s, p);
        else if (multi)
          hipLaunchKernelGGL((sssp_relax_kernel<true, false>), dim3(gr), dim3(kSBlock), 0, s, p);
        else
          hipLaunchKernelGGL((sssp_relax_kernel<false, false>), dim3(gr), dim3(kSBlock), 0, s, p);
        if (wide)
          hipLaunchKernelGGL(sssp_compact_kernel<kWideWords>, dim3(gc), dim3(kSBlock), 0, s, p);
        else
          hipLaunchKernelGGL(sssp_compact_kernel<1>, dim3(gc), dim3(kSBlock), 0, s, p);
      }
      OLV_HIP(hipGetLastError());
      t.stop();  // ahead of the read-back: host latency after the last round is not timed
      enq += chunk;
      OLV_TRY(sssp_read(*w));
      if (w->h_ctl->done) break;
      // the device stops by itself after p.max_rounds rounds (capped)
      if (enq > (uint64_t)p.max_rounds + 2) return fail(OLV_EINTERNAL, "olv_sssp: round loop did not terminate");
      if (!(flags & OLV_HOST_LOOP)) chunk = more = std::min(more * 2, 256u);
    }
  }
  for (int i = 3; i > 0; --i) gm->sssp_rounds[i] = gm->sssp_rounds[i - 1];
  gm->sssp_rounds[0] = w->h_ctl->rounds;
  if (st) {
    std::memset(st, 0, sizeof(*st));
    st->elapsed_ms = t.ms();
    st->iterations = w->h_ctl->rounds;
    st->edges_inspected = w->h_ctl->relax;
  }
  const bool capped = w->h_ctl->capped != 0;
  // (the stream is idle: the control block has been read back)
  if (w->bytes <= kSsspKeepBytes) lease.keep();
  if (capped) return fail(OLV_ENOCONV, "olv_sssp: still relaxing after n=%u rounds (negative cycle)", g->n);
  return OLV_OK;
}

__global__ void reach_stat_kernel(const int32_t *__restrict__ d, const uint32_t *__restrict__ rp, uint32_t n,
                                  size_t total, unsigned long long *__restrict__ out) {
  __shared__ unsigned long long s_red[256 / kWave];
  unsigned long long vr = 0, er = 0;
  for (size_t x = (size_t)blockIdx.x * blockDim.x + threadIdx.x; x < total; x += (size_t)gridDim.x * blockDim.x)
    if (d[x] != kInf) {
      const uint32_t v = (uint32_t)(x % n);
      vr += 1;
      er += rp[v + 1] - rp[v];
    }
  vr = block_sum<256, unsigned long long>(vr, s_red);
  er = block_sum<256, unsigned long long>(er, s_red);
  if (threadIdx.x == 0) {
    atomicAdd(&out[0], vr);
    atomicAdd(&out[1], er);
  }
}

// Reached (vertex, source) pairs and the sum of their out-degrees.
int reach_stats(const olv_graph *g, const int32_t *d, uint32_t k, olv_stats *st) {
  DevBuf b;
  OLV_TRY(b.alloc(16));
  OLV_HIP(hipMemsetAsync(b.p, 0, 16, stream()));
  const size_t total = (size_t)k * g->n;
  hipLaunchKernelGGL(reach_stat_kernel, dim3(sgrid(total, 256)), dim3(256), 0, stream(), d, g->row_ptr, g->n, total,
                     b.as<unsigned long long>());
  unsigned long long h[2];
  OLV_HIP(hipMemcpyAsync(h, b.p, 16, hipMemcpyDeviceToHost, stream()));
  OLV_HIP(hipStreamSynchronize(stream()));
  st->vertices_reached = h[0];
  st->edges_traversed = h[1];
  return OLV_OK;
}

static int sssp_entry(const olv_graph *g, const uint32_t *srcs, uint32_t k, const int32_t *weights, int32_t *dist,
                      unsigned flags, olv_stats *st) {
  if (!g || !dist || !srcs) return fail(OLV_EINVAL, "olv_sssp: NULL argument");
  if (k == 0) return fail(OLV_EINVAL, "olv_sssp: no source");
  const bool host = (flags & OLV_PTR_HOST) != 0;
  for (uint32_t i = 0; i < k; ++i)
    if (srcs[i] >= g->n) return fail(OLV_EINVAL, "olv_sssp: source %u out of range (n=%u)", srcs[i], g->n);
  DevBuf dw, dd;
  const int32_t *w = weights;
  if (!w) {
    if (g->wdtype != OLV_W_I32) return fail(OLV_EINVAL, "olv_sssp: graph has no int32 weights and none were given");
    w = static_cast<const int32_t *>(g->weights);
  } else if (host) {
    OLV_TRY(dw.alloc((size_t)g->m * 4));
    if (g->m) OLV_HIP(hipMemcpy(dw.p, weights, (size_t)g->m * 4, hipMemcpyHostToDevice));
    w = dw.as<int32_t>();
  }
  const size_t total = (size_t)k * g->n;
  int32_t *out = dist;
  if (host) {
    OLV_TRY(dd.alloc(total * 4));
    out = dd.as<int32_t>();
  }
  OLV_TRY(sssp_run(g, srcs, k, w, out, flags, st));
  if (st) OLV_TRY(reach_stats(g, out, k, st));
  if (host) OLV_HIP(hipMemcpy(dist, out, total * 4, hipMemcpyDeviceToHost));
  return OLV_OK;
}

}  // namespace olv

using namespace olv;

extern "C" int olv_sssp(const olv_graph *g, uint32_t src, const int32_t *weights, int32_t *dist, unsigned flags,
                        olv_stats *st) {
  if (!g) return fail(OLV_EINVAL, "olv_sssp: NULL graph");
  return sssp_entry(g, &src, 1, weights, dist, flags, st);
}

extern "C" int olv_sssp_batched(const olv_graph *g, const uint32_t *srcs, uint32_t k, const int32_t *weights,
                                int32_t *dist, unsigned flags, olv_stats *st) {
  return sssp_entry(g, srcs, k, weights, dist, flags, st);
}
