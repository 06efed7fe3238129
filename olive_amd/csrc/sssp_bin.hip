// SSSP by destination binning, for large graphs without hub vertices: each
// round's relaxations are scattered into per-partition regions, then applied
// partition by partition in LDS.
//
// Same fixed point as the frontier relaxation of SSSP.cu:146-163 (and the
// direct path in sssp.hip): every vertex whose distance drops is expanded
// again with its new distance until nothing drops, and shortest distances
// are unique, so the order of relaxations changes no output.  What changes is
// where the min-reductions happen.  A relaxation in the direct path is a
// random 4-byte probe of dist and, when it improves, a device-scope atomicMin.
// On MI355X those atomics are performed at the memory side, and binning the
// probes by the XCD that owns the destination does not help them: 20M random
// relaxations into a 16 MB array cost about 735 us either way; scattering the
// pairs into per-partition bins and applying each partition in LDS takes
// about 90 + 35 us.
//
// Near-far order (Davidson et al., IPDPS'14) is kept with one "dirty" bit per
// vertex: the distance dropped since the vertex was last expanded.  With
// split T, the frontier is {dirty, dist < T}; when it is empty the next round
// re-splits at (smallest dirty far distance) + delta -- no empty promotion,
// the split always lands past at least one vertex -- and when nothing is
// dirty the run is done.
//
// k sources run as k instances over virtual vertices s*n + v (as in
// sssp.hip); partitions cover virtual ranges, so one launch serves all.
//
// A workgroup owns a slice of consecutive vertices, so a graph whose edges
// crowd on some vertices leaves most of the chip idle, and small graphs have
// too few slices: those take the direct path.
//
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstring>
#include <memory>
#include <vector>

#include "bfs_core.hpp"
#include "internal.hpp"

namespace olv {

__device__ __forceinline__ int32_t add_clamp(int32_t t, int32_t d) { return t > kInf - d ? kInf : t + d; }

// ------------------------------------------------------------------ rounds
// One kernel per round: workgroup q owns
// partition q (2^14 virtual vertices) and, in launch R,
//   1. applies the pairs that every partition sent it in launch R-1 (region
//      p -> q of the pair store, one count per region) to its dist slice in
//      LDS,
//   2. updates its dirty bits and picks its frontier {dirty, dist < T},
//   3. expands that frontier at once: the pairs for partition q' go to region
//      q -> q' of the other pair store, at offsets this workgroup counts in
//      LDS -- each region has a single writer, so no device-scope atomic is
//      needed to place them (region capacities are the edge counts between
//      the two slices, fixed per graph).
// The split T of launch R comes from the previous launch's totals (striped
// counters): frontier non-empty -> same split; empty -> re-split at the
// smallest dirty far distance + delta; nothing dirty -> done.
// Slices of 2^14 vertices (64 KB of dist; ~135 KB of LDS, one workgroup per
// CU) up to 16M virtual vertices.  (2^13-vertex slices fit two workgroups per
// CU by LDS, but the second ones started up to 120 us late on MI355X and a
// 4M-vertex run took 1.78 ms against 1.30 ms.)
constexpr uint32_t kFSb = 14, kFS = 1u << kFSb;  // vertices of a slice
constexpr uint32_t kFParts = 1024;               // slices at most (16M virtual vertices)
constexpr int kFB = 1024;                        // workgroup

struct alignas(128) FusedSlot {
  uint32_t nnear;  // frontier vertices chosen (and expanded) in the launch
  int32_t mf;      // smallest dirty distance left at or above the split
  unsigned long long edges;
  uint32_t pad[28];
};

struct FusedCtl {
  uint32_t done, rounds, capped, err, resplits, pad[3];
  int32_t split[2];  // split of launch R in slot R & 1
  unsigned long long relax;
  FusedSlot slot[3][kCtrSlots];  // totals of launch R in slot R % 3
};

struct FusedArgs {
  const uint32_t *row_ptr;
  const uint32_t *col;
  const int32_t *w;
  int32_t *dist;
  uint32_t *dirty;
  uint2 *pairs[2];        // pair store written by launch R in pairs[(R + 1) & 1]
  const uint32_t *base;   // [q * nparts + p]: start of region p -> q; base[nparts^2] = total
  uint32_t *cnt[2];       // [q * nparts + p]: pairs in region p -> q (written by p, read as a row by q)
  FusedCtl *ctl;
  uint32_t n, k, nv, nw, nparts;
  int32_t delta;
  uint32_t max_rounds;
};

// Exclusive prefix over the workgroup with one barrier: every wave reads the
// kFB / 64 wave totals itself (no serial pass by one lane).  `wt` holds
// kFB / 64 words and must not be reused before the next barrier.
__device__ __forceinline__ uint32_t fused_scan(uint32_t v, uint32_t *wt, uint32_t *total) {
  const uint32_t lane = lane_id(), wid = threadIdx.x / kWave;
  const uint32_t inc = wave_inclusive_scan(v);
  if (lane == kWave - 1) wt[wid] = inc;
  __syncthreads();
  uint32_t before = 0, tot = 0;
#pragma unroll
  for (uint32_t i = 0; i < kFB / kWave; ++i) {
    const uint32_t x = wt[i];
    before += i < wid ? x : 0u;
    tot += x;
  }
  *total = tot;
  return before + inc - v;
}

__global__ void __launch_bounds__(kFB) ssspf_round_kernel(FusedArgs a, uint32_t R) {
  constexpr uint32_t kFV = kFS / kFB;  // consecutive vertices per lane
  FusedCtl *ctl = a.ctl;
  const uint32_t t = threadIdx.x, lane = lane_id();
  const uint32_t q = blockIdx.x;
  const uint32_t P = a.nparts;
  __shared__ int4 s_d4[kFS / 4];
  int32_t *s_d = reinterpret_cast<int32_t *>(s_d4);
  __shared__ uint16_t s_near[kFS];
  __shared__ uint32_t s_in[kFParts + 1], s_base[kFParts];  // incoming regions: scan, start
  __shared__ uint32_t s_obase[kFParts], s_ocap[kFParts];   // outgoing regions: start, capacity
  __shared__ uint32_t s_run[kFParts];  // pairs placed in region q -> q'
  constexpr uint32_t kNW = kFB / kWave;
  __shared__ uint32_t s_wo[kNW][kWave + 1], s_wb[kNW][kWave], s_wx[kNW][kWave];  // per-wave items
  __shared__ int32_t s_wd[kNW][kWave];
  __shared__ uint32_t s_scan[2][kNW];
  __shared__ int32_t s_mfw[kFB / kWave];
  __shared__ int32_t s_T;
  __shared__ uint32_t s_stop;
  // Everything this launch reads that does not depend on the round decision
  // is requested first: the slice (16 consecutive values per lane), its dirty
  // word, the region counts and offsets of this partition.
  const uint32_t x0 = q << kFSb;
  const uint32_t cv = min(kFS, a.nv - x0);
  const uint32_t o0 = t * kFV;  // this lane's first vertex in the slice
  int32_t old[kFV];
  if (o0 + kFV <= cv) {
    const int4 *src = reinterpret_cast<const int4 *>(a.dist + x0 + o0);
#pragma unroll
    for (uint32_t i = 0; i < kFV / 4; ++i) {
      const int4 v = src[i];
      old[4 * i] = v.x;
      old[4 * i + 1] = v.y;
      old[4 * i + 2] = v.z;
      old[4 * i + 3] = v.w;
    }
  } else {
#pragma unroll
    for (uint32_t i = 0; i < kFV; ++i) old[i] = o0 + i < cv ? a.dist[x0 + o0 + i] : kInf;
  }
  const uint32_t wd = (x0 + o0) >> 5;  // dirty word holding this lane's 16 bits
  const uint32_t dw = o0 < cv ? a.dirty[wd] : 0u;
  uint32_t cin = 0, bin = 0, ob = 0, oe = 0;
  if (t < P) {
    if (R > 0) cin = a.cnt[R & 1][q * P + t];
    bin = a.base[q * P + t];
    ob = a.base[t * P + q];
    oe = a.base[t * P + q + 1];
  }
  // round decision (identical in every workgroup)
  if (t < kWave) {
    uint32_t nn = 0;
    int32_t mf = kInf;
    unsigned long long ed = 0;
    if (R > 0 && t < kCtrSlots) {
      const FusedSlot &sl = ctl->slot[(R - 1) % 3][t];
      nn = sl.nnear;
      mf = sl.mf;
      ed = sl.edges;
    }
    nn = wave_sum(nn);
    ed = wave_sum(ed);
    for (int o = kWave / 2; o > 0; o >>= 1) {
      const int32_t y = __shfl_xor(mf, o, kWave);
      mf = y < mf ? y : mf;
    }
    if (t == 0) {
      int32_t T;
      uint32_t stop = __hip_atomic_load(&ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ? 3u : 0u;
      if (R == 0) {
        T = a.delta;
      } else if (nn > 0) {
        T = ctl->split[(R - 1) & 1];
      } else if (mf < kInf) {
        T = add_clamp(mf, a.delta);
      } else {
        T = kInf;
        if (!stop) stop = 1;  // nothing dirty: done
      }
      if (!stop && R >= a.max_rounds) stop = 2;
      s_T = T;
      s_stop = stop;
      if (q == 0 && stop != 3) {
        ctl->relax += ed;
        if (stop) {
          ctl->rounds = R;
          ctl->capped = stop == 2;
          ctl->done = 1u;
        } else {
          ctl->split[R & 1] = T;
          if (R > 0 && nn == 0) ctl->resplits += 1;
        }
      }
    }
  }
  __syncthreads();
  if (s_stop) return;
  if (q == 0 && t < kCtrSlots) {
    FusedSlot &z = ctl->slot[(R + 1) % 3][t];
    z.nnear = 0;
    z.mf = kInf;
    z.edges = 0;
  }
  const int32_t T = s_T;
#pragma unroll
  for (uint32_t i = 0; i < kFV / 4; ++i)
    s_d4[t * (kFV / 4) + i] = make_int4(old[4 * i], old[4 * i + 1], old[4 * i + 2], old[4 * i + 3]);
  // 1. incoming pairs
  uint32_t tin;
  const uint32_t ein = fused_scan(cin, s_scan[0], &tin);
  if (t < P) {
    s_in[t] = ein;
    s_base[t] = bin;
    s_obase[t] = ob;
    s_ocap[t] = oe - ob;
    s_run[t] = 0;
  }
  if (t == 0) s_in[P] = tin;
  __syncthreads();
  {
    const uint2 *src = a.pairs[R & 1];
    auto pair_at = [&](uint32_t i) -> uint2 {
      uint32_t lo = 0, hi = P;  // s_in[lo] <= i < s_in[hi]
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (s_in[mid] <= i)
          lo = mid;
        else
          hi = mid;
      }
      return src[s_base[lo] + (i - s_in[lo])];
    };
    constexpr int UA = 8;  // pairs in flight per lane
    for (uint32_t i0 = 0; i0 < tin; i0 += UA * kFB) {
      uint2 pp[UA];
#pragma unroll
      for (int u = 0; u < UA; ++u) {
        const uint32_t i = i0 + u * kFB + t;
        pp[u] = i < tin ? pair_at(i) : make_uint2(0xffffffffu, 0u);
      }
#pragma unroll
      for (int u = 0; u < UA; ++u)
        if (pp[u].x != 0xffffffffu) atomicMin(&s_d[(pp[u].x - x0) & (kFS - 1)], (int32_t)pp[u].y);
    }
  }
  __syncthreads();
  // 2. dirty' = dirty | improved; frontier = dirty' & dist < T (expanded
  // now, so it leaves the dirty set); far minimum over the rest
  int32_t nv[kFV];
#pragma unroll
  for (uint32_t i = 0; i < kFV / 4; ++i) {
    const int4 v = s_d4[t * (kFV / 4) + i];
    nv[4 * i] = v.x;
    nv[4 * i + 1] = v.y;
    nv[4 * i + 2] = v.z;
    nv[4 * i + 3] = v.w;
  }
  const uint32_t was = (dw >> (o0 & 31)) & ((1u << kFV) - 1u);
  uint32_t imp = 0, rest = 0, nr = 0;
  int32_t mf = kInf;
#pragma unroll
  for (uint32_t i = 0; i < kFV; ++i) {
    const bool improved = nv[i] < old[i];  // (vertices past cv hold INF on both sides)
    const bool dirty = ((was >> i) & 1u) || improved;
    const bool near = dirty && nv[i] < T;
    imp |= (uint32_t)improved << i;
    nr |= (uint32_t)near << i;
    rest |= (uint32_t)(dirty && !near) << i;
    if (dirty && !near) mf = nv[i] < mf ? nv[i] : mf;
  }
  // write back the 128-byte lines (lane pairs) that changed
  uint32_t lim = imp;
#pragma unroll
  for (uint32_t o = 1; o < 32 / kFV; o <<= 1) lim |= __shfl_xor(lim, o, kWave);
  const bool line = lim != 0;
  if (line) {
    if (o0 + kFV <= cv) {
      int4 *dst = reinterpret_cast<int4 *>(a.dist + x0 + o0);
#pragma unroll
      for (uint32_t i = 0; i < kFV / 4; ++i) dst[i] = make_int4(nv[4 * i], nv[4 * i + 1], nv[4 * i + 2], nv[4 * i + 3]);
    } else {
#pragma unroll
      for (uint32_t i = 0; i < kFV; ++i)
        if (o0 + i < cv) a.dist[x0 + o0 + i] = nv[i];
    }
  }
  // lanes sharing a dirty word combine their bits; the first one stores it
  constexpr uint32_t kLW = 32 / kFV;  // lanes per word
  uint32_t word = rest << (o0 & 31);
#pragma unroll
  for (uint32_t o = 1; o < kLW; o <<= 1) word |= __shfl_xor(word, o, kWave);
  if ((t % kLW) == 0 && o0 < cv) a.dirty[wd] = word;
  uint32_t N;
  const uint32_t nb = fused_scan((uint32_t)__popc(nr), s_scan[1], &N);
  {
    uint32_t pos = nb;
    for (uint32_t x = nr; x; x &= x - 1) s_near[pos++] = (uint16_t)(o0 + __ffs(x) - 1);
  }
  for (int o = kWave / 2; o > 0; o >>= 1) {
    const int32_t y = __shfl_xor(mf, o, kWave);
    mf = y < mf ? y : mf;
  }
  if (lane == 0) s_mfw[t / kWave] = mf;
  __syncthreads();
  // 3. expand the frontier into the regions q -> q'.  Each wave takes 64
  // frontier vertices at a time and deals their out-edges to its lanes (a
  // wave-local prefix of the degrees); a pair's place in its region is an
  // LDS atomic on the region's counter (one writer per region: this
  // workgroup), so no barrier stands between reading an edge and storing its
  // pair.  Lines of a region fill from consecutive claims and merge in L2.
  uint2 *dst = a.pairs[(R + 1) & 1];
  unsigned long long edges = 0;
  {
    const uint32_t wv = t / kWave;
    constexpr int U = 8;  // edges in flight per lane
    // a lane's frontier vertex of chunk cb: out-list start, degree, instance
    // base, distance (the next chunk's are requested before this one's edges)
    auto item = [&](uint32_t i, uint32_t &beg, uint32_t &deg, uint32_t &xb, int32_t &du) {
      beg = deg = xb = 0;
      du = 0;
      if (i < N) {
        const uint32_t o = s_near[i];
        const uint32_t x = x0 + o;
        const uint32_t row = a.k > 1 ? x % a.n : x;
        beg = a.row_ptr[row];
        deg = a.row_ptr[row + 1] - beg;
        xb = x - row;
        du = s_d[o];
      }
    };
    uint32_t beg, deg, xb;
    int32_t du;
    item(wv * kWave + lane, beg, deg, xb, du);
    for (uint32_t cb = wv * kWave; cb < N; cb += kNW * kWave) {
      uint32_t nbeg, ndeg, nxb;
      int32_t ndu;
      item(cb + kNW * kWave + lane, nbeg, ndeg, nxb, ndu);
      const uint32_t inc = wave_inclusive_scan(deg);
      const uint32_t E = __shfl(inc, kWave - 1, kWave);
      s_wo[wv][lane] = inc - deg;
      s_wb[wv][lane] = beg;
      s_wx[wv][lane] = xb;
      s_wd[wv][lane] = du;
      if (lane == 0) s_wo[wv][kWave] = E;
      edges += deg;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      for (uint32_t s0 = 0; s0 < E; s0 += kWave * U) {
        uint32_t e[U], xbv[U];
        int32_t duv[U];
        bool ok[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t slot = s0 + u * kWave + lane;
          ok[u] = slot < E;
          uint32_t lo = 0, hi = kWave;  // s_wo[lo] <= slot < s_wo[hi]
          if (ok[u])
            while (hi - lo > 1) {
              const uint32_t mid = (lo + hi) >> 1;
              if (s_wo[wv][mid] <= slot)
                lo = mid;
              else
                hi = mid;
            }
          e[u] = ok[u] ? s_wb[wv][lo] + (slot - s_wo[wv][lo]) : 0u;
          xbv[u] = s_wx[wv][lo];
          duv[u] = s_wd[wv][lo];
        }
        uint32_t cv_[U], wv_[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          cv_[u] = ok[u] ? a.col[e[u]] : 0u;
          wv_[u] = ok[u] ? (uint32_t)a.w[e[u]] : 0u;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (ok[u]) {
            const uint32_t v = xbv[u] + cv_[u];
            const uint32_t p = v >> kFSb;
            const uint32_t pos = atomicAdd(&s_run[p], 1u);
            if (pos < s_ocap[p]) dst[s_obase[p] + pos] = make_uint2(v, (uint32_t)duv[u] + wv_[u]);
          }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();  // the wave's item arrays are rewritten next
      beg = nbeg;
      deg = ndeg;
      xb = nxb;
      du = ndu;
    }
  }
  __syncthreads();
  if (t < P && s_run[t] > s_ocap[t]) __hip_atomic_store(&ctl->err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // counts of the regions q -> q' filled in this launch (zeros included)
  if (t < P) a.cnt[(R + 1) & 1][t * P + q] = min(s_run[t], s_ocap[t]);
  // totals
  __shared__ unsigned long long s_red[kFB / kWave];
  const unsigned long long te = block_sum<kFB, unsigned long long>(edges, s_red);
  if (t == 0) {
    int32_t m = kInf;
    for (int i = 0; i < kFB / kWave; ++i) m = s_mfw[i] < m ? s_mfw[i] : m;
    FusedSlot &sl = ctl->slot[R % 3][q % kCtrSlots];
    if (N) atomicAdd(&sl.nnear, N);
    if (m < kInf) atomicMin(&sl.mf, m);
    if (te) atomicAdd(&sl.edges, te);
  }
}

// Edges from slice p to slice q (virtual): cap[q * nparts + p]; one
// workgroup per source slice.
__global__ void ssspf_cap_kernel(const uint32_t *rp, const uint32_t *col, uint32_t n, uint32_t k, uint32_t nv,
                                 uint32_t nparts, uint32_t *cap) {
  __shared__ uint32_t s_h[kFParts];
  const uint32_t p = blockIdx.x;
  for (uint32_t i = threadIdx.x; i < nparts; i += blockDim.x) s_h[i] = 0;
  __syncthreads();
  const uint32_t x0 = p << kFSb, x1 = min(nv, x0 + kFS);
  // one wave per source vertex
  const uint32_t lane = lane_id(), wv = threadIdx.x / kWave, nwv = blockDim.x / kWave;
  for (uint32_t x = x0 + wv; x < x1; x += nwv) {
    const uint32_t row = k > 1 ? x % n : x, xb = x - row;
    for (uint32_t e = rp[row] + lane; e < rp[row + 1]; e += kWave) atomicAdd(&s_h[(xb + col[e]) >> kFSb], 1u);
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < nparts; i += blockDim.x)
    if (s_h[i]) cap[i * nparts + p] = s_h[i];
}

// dist = INF, dirty = 0, counts of parity 0 = 0, control zero (slots: mf =
// INF), then the seeds: dist 0 and dirty.
__global__ void ssspf_reset_kernel(FusedArgs a) {
  const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = tid; i < a.nv; i += stride) a.dist[i] = kInf;
  for (size_t i = tid; i < a.nw; i += stride) a.dirty[i] = 0u;
  for (size_t i = tid; i < (size_t)a.nparts * a.nparts; i += stride) a.cnt[0][i] = 0u;
  uint32_t *c = reinterpret_cast<uint32_t *>(a.ctl);
  for (size_t i = tid; i < sizeof(FusedCtl) / 4; i += stride) c[i] = 0u;
}

__global__ void ssspf_seed_kernel(const uint32_t *srcs, FusedArgs a) {
  if (threadIdx.x < 3 * kCtrSlots) a.ctl->slot[threadIdx.x / kCtrSlots][threadIdx.x % kCtrSlots].mf = kInf;
  for (uint32_t s = threadIdx.x; s < a.k; s += blockDim.x) {
    const uint32_t x = s * a.n + srcs[s];
    a.dist[x] = 0;
    atomicOr(&a.dirty[x >> 5], 1u << (x & 31));
  }
}

// --------------------------------------------------------------------- host
struct SsspBinWork {
  uint32_t k = 0, nparts = 0, nw = 0, nwp = 0;
  uint64_t nv = 0;
  uint32_t *dirty = nullptr;
  uint2 *pairs[2] = {nullptr, nullptr};
  uint32_t *base = nullptr, *cnt[2] = {nullptr, nullptr};
  FusedCtl *fctl = nullptr, *h_fctl = nullptr;
  ~SsspBinWork() {
    void *ps[] = {dirty, pairs[0], pairs[1], base, cnt[0], cnt[1], fctl};
    for (void *q : ps)
      if (q) (void)hipFree(q);
    if (h_fctl) (void)hipHostFree(h_fctl);
  }
};

void free_sssp_bin(olv_graph *g) {
  delete g->sssp_bin;
  g->sssp_bin = nullptr;
}

static unsigned bgrid(size_t items, size_t per) {
  size_t b = (items + per - 1) / per;
  return (unsigned)std::max<size_t>(1, std::min(b, (size_t)cu_count() * 8));
}

// Work for the fused rounds: region capacities (edges between every pair of
// slices), their offsets, two pair stores and two count matrices.  Published to
// the graph only once the offsets are on the device: the rounds store pairs by
// them.
static int fused_work(olv_graph *g, uint32_t k, SsspBinWork **out) {
  if (g->sssp_bin && g->sssp_bin->k == k) {
    *out = g->sssp_bin;
    return OLV_OK;
  }
  free_sssp_bin(g);
  std::unique_ptr<SsspBinWork> w(new SsspBinWork());
  w->k = k;
  w->nv = (uint64_t)k * g->n;
  w->nparts = (uint32_t)((w->nv + kFS - 1) >> kFSb);
  w->nw = (uint32_t)((w->nv + 31) / 32);
  w->nwp = (w->nw + 63) / 64 * 64;
  const size_t P2 = (size_t)w->nparts * w->nparts;
  const size_t npairs = std::max<uint64_t>((uint64_t)k * g->m, 1);
  if (hipMalloc(reinterpret_cast<void **>(&w->dirty), (size_t)w->nwp * 4) != hipSuccess ||
      hipMalloc(reinterpret_cast<void **>(&w->pairs[0]), npairs * sizeof(uint2)) != hipSuccess ||
      hipMalloc(reinterpret_cast<void **>(&w->pairs[1]), npairs * sizeof(uint2)) != hipSuccess ||
      hipMalloc(reinterpret_cast<void **>(&w->base), (P2 + 1) * 4) != hipSuccess ||
      hipMalloc(reinterpret_cast<void **>(&w->cnt[0]), P2 * 4) != hipSuccess ||
      hipMalloc(reinterpret_cast<void **>(&w->cnt[1]), P2 * 4) != hipSuccess ||
      hipMalloc(reinterpret_cast<void **>(&w->fctl), sizeof(FusedCtl)) != hipSuccess ||
      hipHostMalloc(reinterpret_cast<void **>(&w->h_fctl), sizeof(FusedCtl), hipHostMallocDefault) != hipSuccess)
    return fail(OLV_ENOMEM, "olv_sssp: device allocation for the fused rounds failed");
  DevBuf cap;
  OLV_TRY(cap.alloc(P2 * 4));
  OLV_HIP(hipMemsetAsync(cap.p, 0, P2 * 4, stream()));
  hipLaunchKernelGGL(ssspf_cap_kernel, dim3(w->nparts), dim3(1024), 0, stream(), g->row_ptr, g->col, g->n, k,
                     (uint32_t)w->nv, w->nparts, cap.as<uint32_t>());
  OLV_HIP(hipGetLastError());
  std::vector<uint32_t> hc(P2), hb(P2 + 1);
  OLV_HIP(hipMemcpyAsync(hc.data(), cap.p, P2 * 4, hipMemcpyDeviceToHost, stream()));
  OLV_HIP(hipStreamSynchronize(stream()));
  uint64_t run = 0;
  for (size_t i = 0; i < P2; ++i) {
    hb[i] = (uint32_t)run;
    run += hc[i];
  }
  hb[P2] = (uint32_t)run;
  if (run != (uint64_t)k * g->m)
    return fail(OLV_EINTERNAL, "olv_sssp: region capacities %llu != %llu edges", (unsigned long long)run,
                (unsigned long long)k * g->m);
  OLV_HIP(hipMemcpy(w->base, hb.data(), (P2 + 1) * 4, hipMemcpyHostToDevice));
  *out = g->sssp_bin = w.release();
  return OLV_OK;
}

static int fused_run(const olv_graph *g, const uint32_t *d_srcs, uint32_t k, const int32_t *weights, int32_t *dist,
                     int32_t delta, unsigned flags, olv_stats *st) {
  olv_graph *gm = const_cast<olv_graph *>(g);
  SsspBinWork *w = nullptr;
  OLV_TRY(fused_work(gm, k, &w));
  FusedArgs a;
  a.row_ptr = g->row_ptr;
  a.col = g->col;
  a.w = weights;
  a.dist = dist;
  a.dirty = w->dirty;
  a.pairs[0] = w->pairs[0];
  a.pairs[1] = w->pairs[1];
  a.base = w->base;
  a.cnt[0] = w->cnt[0];
  a.cnt[1] = w->cnt[1];
  a.ctl = w->fctl;
  a.n = g->n;
  a.k = k;
  a.nv = (uint32_t)w->nv;
  a.nw = w->nw;
  a.nparts = w->nparts;
  a.delta = delta;
  a.max_rounds = (uint32_t)std::min<uint64_t>(4ull * g->n + 1024, 0xffffffffull);
  hipStream_t s = stream();
  Timer t;
  t.start();
  hipLaunchKernelGGL(ssspf_reset_kernel,
                     dim3(bgrid(std::max<uint64_t>(w->nv, (uint64_t)w->nparts * w->nparts), 256)), dim3(256), 0, s, a);
  hipLaunchKernelGGL(ssspf_seed_kernel, dim3(1), dim3(256), 0, s, d_srcs, a);
  OLV_HIP(hipGetLastError());
  uint32_t hist = 8;
  for (uint32_t r : gm->sssp_rounds) hist = std::max(hist, std::min(r + 3, 4096u));
  uint32_t chunk = (flags & OLV_HOST_LOOP) ? 1u : hist;
  uint32_t more = 4;
  uint64_t enq = 0;
  for (;;) {
    for (uint32_t i = 0; i < chunk; ++i)
      hipLaunchKernelGGL(ssspf_round_kernel, dim3(w->nparts), dim3(kFB), 0, s, a, (uint32_t)(enq + i));
    OLV_HIP(hipGetLastError());
    t.stop();
    enq += chunk;
    OLV_HIP(hipMemcpyAsync(w->h_fctl, w->fctl, sizeof(FusedCtl), hipMemcpyDeviceToHost, s));
    OLV_HIP(hipStreamSynchronize(s));
    if (w->h_fctl->done) break;
    if (enq > (uint64_t)a.max_rounds + 2) return fail(OLV_EINTERNAL, "olv_sssp: round loop did not terminate");
    if (!(flags & OLV_HOST_LOOP)) chunk = more = std::min(more * 2, 256u);
  }
  const FusedCtl &c = *w->h_fctl;
  for (int i = 3; i > 0; --i) gm->sssp_rounds[i] = gm->sssp_rounds[i - 1];
  gm->sssp_rounds[0] = c.rounds;
  if (st) {
    std::memset(st, 0, sizeof(*st));
    st->elapsed_ms = t.ms();
    st->iterations = c.rounds;
    st->edges_inspected = c.relax;
  }
  if (c.err) return fail(OLV_EINTERNAL, "olv_sssp: a pair region overflowed its capacity");
  if (c.capped) return fail(OLV_ENOCONV, "olv_sssp: still relaxing after %u rounds", c.rounds);
  return OLV_OK;
}

// Where binning beats direct relaxation on graphs without hubs: from
// kBinMinVertices virtual vertices, or from kBinMinSparse where a vertex has at
// most kBinSparse edges.  In between, the direct rounds have the cheaper edges
// and the binned ones, whose slices leave CUs idle, the cheaper vertices (us,
// binned / direct; d: edges a vertex):
//   vertices  d 2.5      d 4        d 8         d 16
//   800K      785/774    777/747    902/769    1203/841
//   1M        755/797    825/845    962/882    1256/942
//   1.2M      881/913    857/885    940/885    1286/1059
//   1.5M      824/908    894/920   1006/1012   1391/1202
//   4.2M                           1640/2200
//   16.7M                5150/4800 7350/7480  11330/11910
// Past 16M vertices (two slices per lane of a workgroup) direct is the faster
// one up to 8 edges a vertex and, beyond, slower by up to a fifth than binning
// with a launch of its own for the apply step was, which went by queues in
// memory (17M vertices: d 4 7.5 ms binned, 5.1 direct; d 8 8.65 and 7.4; d 16
// 11.7 and 12.4; d 24 16.5 and 20.0).
constexpr uint64_t kBinMinVertices = 1250000, kBinMinSparse = 900000, kBinSparse = 5;

// Whether k instances of g go through the binned rounds: no out-list long
// enough to be split, slices for most of the chip, and at most 16M vertices
// and 2^32 pairs.
bool sssp_bin_fits(const olv_graph *g, uint32_t k) {
  const uint64_t nv = (uint64_t)k * g->n;
  if (!g->m || (uint64_t)k * g->m >= (1ull << 32) || nv >= (1ull << 32)) return false;
  if (g->max_outdeg >= g->tune.hub_thr || g->n > ((uint64_t)kFParts << kFSb)) return false;
  return nv >= kBinMinVertices || (nv >= kBinMinSparse && g->m <= kBinSparse * g->n);
}

// Binned SSSP for k instances (sources d_srcs[0..k), on the device; the
// graph fits) with near-far step delta > 0.  More instances than 16M virtual
// vertices run in groups of as many as fit.
int sssp_bin_run(const olv_graph *g, const uint32_t *d_srcs, uint32_t k, const int32_t *weights, int32_t *dist,
                 int32_t delta, unsigned flags, olv_stats *st) {
  const uint32_t gk = (uint32_t)std::min<uint64_t>(k, ((uint64_t)kFParts << kFSb) / g->n);
  if (gk == k) return fused_run(g, d_srcs, k, weights, dist, delta, flags, st);
  olv_stats tot;
  std::memset(&tot, 0, sizeof(tot));
  for (uint32_t s0 = 0; s0 < k; s0 += gk) {
    const uint32_t kk = std::min(gk, k - s0);
    olv_stats one;
    OLV_TRY(fused_run(g, d_srcs + s0, kk, weights, dist + (size_t)s0 * g->n, delta, flags, &one));
    tot.elapsed_ms += one.elapsed_ms;
    tot.iterations += one.iterations;
    tot.edges_inspected += one.edges_inspected;
  }
  if (st) *st = tot;
  return OLV_OK;
}

}  // namespace olv
