// Batched traversals (no reference counterpart; each result equals repeated
// runs of the plain engine):
//  * olv_bfs_batched: up to 256 sources per sweep, bit-parallel.  Every
//    vertex carries a 256-bit visited mask V, a frontier mask F and (for
//    push levels) an accumulator N; one adjacency sweep per level serves all
//    sources.  Push (top-down) levels OR F[u] into N[v] with atomics and a
//    contraction pass applies them; pull (bottom-up) levels OR the F of
//    in-neighbours into v and stop once v has every source.  Source s's
//    level of v is written when bit s of V[v] first turns on.  Like the
//    plain BFS, a level is a few kernels whose control lives on the device.
//  * olv_bfs_multisource / olv_graph_union / olv_bfs_multigraph: many
//    graphs as one block-diagonal union traversed by one multi-source BFS.
//  * olv_plan_*: a whole traversal (reset, seeding, all levels) captured
//    once in a hipGraph and replayed with one launch.
//  * olv_autotune: picks degree-bucket thresholds and direction-switch
//    parameters for a graph by timing the plain BFS.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "bfs_core.hpp"
#include "internal.hpp"
#include "seg_core.hpp"


namespace olv {

int bfs_multisource(const olv_graph *g, const uint32_t *seeds, uint32_t k, bool seeds_host, int32_t *levels,
                    unsigned flags, olv_stats *st);
int bfs_prepare(const olv_graph *g, bool can_bu, BfsWork **w);
int bfs_enqueue_init(const olv_graph *g, BfsWork *w, const uint32_t *d_seeds, uint32_t k, uint32_t seed1,
                     int32_t *levels, bool can_bu);
int bfs_enqueue_levels(const olv_graph *g, BfsWork *w, int32_t *levels, bool can_bu, uint32_t count, bool narrow);
int bfs_result(BfsWork *w, uint32_t *levels_run, uint32_t *bu_levels);
bool bfs_done(BfsWork *w);
uint32_t bfs_pairs_hint(const BfsWork *w);
bool bfs_deep_hint(const BfsWork *w);
int reach_stats(const olv_graph *g, const int32_t *d, uint32_t k, olv_stats *st);

constexpr int kMB = 256;          // workgroup size
constexpr int kMW = 8;            // 32-bit words per vertex mask

struct MbfsState {
  unsigned long long mu;
  uint32_t mode, nbu;
};

struct MbfsCtl {
  uint32_t level, level_e, done, levels, nbu, overflow;
  uint32_t qfill[2], hfill[2];  // frontier queue / hub items of level L, slot L & 1
  uint32_t pad[2];
  MbfsState st[2];
  CtrSet cnt[3];
};

struct MbfsParams {
  const uint32_t *row_ptr, *col, *in_row_ptr, *in_col;
  uint32_t n, nw, nwp;
  uint32_t k;
  uint32_t full[kMW];
  uint32_t *V;     // n * kMW
  uint32_t *F;     // 2 * n * kMW
  uint32_t *N;     // n * kMW
  uint32_t *A;     // 3 * nwp  active (frontier) bitmaps
  uint32_t *T;     // 2 * nwp  touched bitmaps (push levels)
  uint32_t *D;     // nwp      vertices that have every source
  uint32_t *queue; // n
  uint2 *hubs;     // hub items
  uint8_t *S;      // n * sstride  level byte per (vertex, source)
  int32_t *levels; // k * n
  // on a renumbered twin: its vertex -> levels index (omap) and back (imap);
  // both nullptr on the graph itself
  const uint32_t *omap, *imap;
  uint32_t sstride;
  MbfsCtl *ctl;
  unsigned long long m;
  uint32_t wave_thr, block_thr, hub_thr;
  float alpha, beta;
  uint32_t can_bu;
  uint32_t pull_per_cu;  // pull workgroups per CU (host side only)
};

__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v |= __shfl_xor(v, o, kWave);
  return v;
}

struct MbfsTdVisitor {
  const MbfsParams &p;
  const uint32_t *Ff;
  uint32_t *T;
  __device__ MbfsTdVisitor(const MbfsParams &pp, const uint32_t *f, uint32_t *t) : p(pp), Ff(f), T(t) {}
  __device__ __forceinline__ uint32_t row(uint32_t q) const { return q; }
  __device__ __forceinline__ uint32_t load(uint32_t q) const { return q; }
  __device__ __forceinline__ uint32_t tgt(uint32_t e, uint32_t) const { return p.col[e]; }
  __device__ __forceinline__ uint32_t state(uint32_t v) const { return p.D[v >> 5]; }
  __device__ __forceinline__ void apply(uint32_t v, uint32_t dword, uint32_t u) {
    if ((dword >> (v & 31)) & 1u) return;
    bool any = false;
#pragma unroll
    for (int j = 0; j < kMW; ++j) {
      const uint32_t f = Ff[(size_t)u * kMW + j];
      if (!f) continue;
      const uint32_t nv = f & ~p.V[(size_t)v * kMW + j];
      if (nv) {
        atomicOr(&p.N[(size_t)v * kMW + j], nv);
        any = true;
      }
    }
    if (any) {
      const uint32_t bit = 1u << (v & 31);
      if (!(T[v >> 5] & bit)) atomicOr(&T[v >> 5], bit);
    }
  }
};

// V |= new, F_next = new; returns whether v now has every source.
__device__ __forceinline__ bool mbfs_apply(const MbfsParams &p, uint32_t v, const uint32_t *nwv, const uint32_t *vv,
                                           uint32_t *Fn) {
  bool full = true;
#pragma unroll
  for (int j = 0; j < kMW; ++j) {
    Fn[(size_t)v * kMW + j] = nwv[j];
    if (nwv[j]) p.V[(size_t)v * kMW + j] = vv[j] | nwv[j];
    full = full && ((vv[j] | nwv[j]) == p.full[j]);
  }
  return full;
}

// Level bytes: S holds one byte per (vertex, source of the group), the
// level at which the source reached the vertex; it is valid where V has
// the source's bit (the bytes are never cleared).  mbfs_levels_kernel turns
// it into the source-major int32 output with coalesced stores.  Levels of
// 255 and deeper are stored as 0xFF and written to the output directly.
__device__ __forceinline__ uint32_t byte_mask4(uint32_t nib) {
  return ((nib * 0x00204081u) & 0x01010101u) * 0xFFu;  // bit i of nib -> byte i = 0xFF
}

// Record level `nlevel` for the sources x of mask word j at v, if there are
// any: read-modify-write of that word's 32 bytes of v's row.
__device__ __forceinline__ void mbfs_record_word(const MbfsParams &p, uint32_t v, uint32_t j, uint32_t x,
                                                 int32_t nlevel) {
  const uint32_t l4 = (nlevel < 255 ? (uint32_t)nlevel : 0xFFu) * 0x01010101u;
  uint4 *row = reinterpret_cast<uint4 *>(p.S + (size_t)v * p.sstride);
  auto mix = [l4](uint32_t o, uint32_t nib) {
    const uint32_t m = byte_mask4(nib & 15u);
    return (o & ~m) | (l4 & m);
  };
  if (x) {
    uint4 a = row[2 * j], b = row[2 * j + 1];
    a.x = mix(a.x, x);
    a.y = mix(a.y, x >> 4);
    a.z = mix(a.z, x >> 8);
    a.w = mix(a.w, x >> 12);
    b.x = mix(b.x, x >> 16);
    b.y = mix(b.y, x >> 20);
    b.z = mix(b.z, x >> 24);
    b.w = mix(b.w, x >> 28);
    row[2 * j] = a;
    row[2 * j + 1] = b;
  }
  if (nlevel >= 255)
    for (; x; x &= x - 1)
      p.levels[(size_t)(j * 32 + __ffs(x) - 1) * p.n + (p.omap ? p.omap[v] : v)] = nlevel;
}

// The same for all words of v by one lane.
__device__ __forceinline__ void mbfs_record(const MbfsParams &p, uint32_t v, const uint32_t *nwv, int32_t nlevel) {
#pragma unroll
  for (int j = 0; j < kMW; ++j) mbfs_record_word(p, v, j, nwv[j], nlevel);
}

__device__ __forceinline__ void mbfs_buffers(const MbfsParams &p, uint32_t L, const uint32_t *&Ff, uint32_t *&Fn,
                                             const uint32_t *&Af, uint32_t *&An, uint32_t *&Ac, uint32_t *&Tc,
                                             uint32_t *&Tx) {
  const size_t fstride = (size_t)p.n * kMW;
  Ff = p.F + (size_t)((L + 1) & 1) * fstride;
  Fn = p.F + (size_t)(L & 1) * fstride;
  Af = p.A + (size_t)((L + 2) % 3) * p.nwp;
  An = p.A + (size_t)(L % 3) * p.nwp;
  Ac = p.A + (size_t)((L + 1) % 3) * p.nwp;
  Tc = p.T + (size_t)(L & 1) * p.nwp;
  Tx = p.T + (size_t)((L + 1) & 1) * p.nwp;
}

// Level L bookkeeping, and for a push level the expansion: touch T,
// accumulate N (a pull level is done by mbfs_pull_kernel).
__global__ void __launch_bounds__(kMB) mbfs_expand_kernel(MbfsParams p) {
  MbfsCtl *ctl = p.ctl;
  if (__hip_atomic_load(&ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const uint32_t L = ctl->level;
  const MbfsState st = ctl->st[L & 1];
  const uint32_t qsize = ctl->qfill[L & 1], nhubs = ctl->hfill[L & 1];
  const uint32_t *Ff, *Af;
  uint32_t *Fn, *An, *Ac, *Tc, *Tx;
  mbfs_buffers(p, L, Ff, Fn, Af, An, Ac, Tc, Tx);
  for (uint32_t i = blockIdx.x * kMB + threadIdx.x; i < p.nwp; i += gridDim.x * kMB) {
    Ac[i] = 0u;
    Tx[i] = 0u;
  }
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
  const int32_t nlevel = (int32_t)(L + 1);
  if (st.mode == 0) {
    MbfsTdVisitor vis(p, Ff, Tc);
    push_expand<kMB>(p.queue, qsize, p.hubs, nhubs, p.row_ptr, p.wave_thr, p.block_thr, p.hub_thr, blockIdx.x, gridDim.x, vis,
                     insp);
  }
  flush_counters<kMB>(&ctl->cnt[L % 3], nf, mf, insp);
}

// ---- pull levels: bucketed by in-degree (the SegPlan of the in-CSR) ----
__device__ __forceinline__ void or_mask(uint32_t *acc, const uint32_t *Ff, uint32_t u) {
  const uint4 *f = reinterpret_cast<const uint4 *>(Ff + (size_t)u * kMW);
  const uint4 a = f[0], b = f[1];
  acc[0] |= a.x;
  acc[1] |= a.y;
  acc[2] |= a.z;
  acc[3] |= a.w;
  acc[4] |= b.x;
  acc[5] |= b.y;
  acc[6] |= b.z;
  acc[7] |= b.w;
}

// OR of F[u] over active in-neighbours k = beg + j, beg + j + G, ...;
// kVisitUnroll in-neighbours per step: their index loads, then their
// activity probes, then their mask loads are issued together.
template <int G>
__device__ __forceinline__ void lane_or(const MbfsParams &p, const uint32_t *Af, const uint32_t *Ff, uint32_t beg,
                                        uint32_t end, uint32_t j, uint32_t *acc) {
  constexpr int U = kVisitUnroll;
  for (uint64_t k = (uint64_t)beg + j; k < end; k += (uint64_t)U * G) {
    uint32_t u[U];
    bool act[U];
#pragma unroll
    for (int i = 0; i < U; ++i) u[i] = k + (uint64_t)i * G < end ? p.in_col[k + (uint64_t)i * G] : 0xffffffffu;
#pragma unroll
    for (int i = 0; i < U; ++i) act[i] = u[i] != 0xffffffffu && bm_test(Af, u[i]);
#pragma unroll
    for (int i = 0; i < U; ++i)
      if (act[i]) or_mask(acc, Ff, u[i]);
  }
}

// OR of the lanes' masks over aligned groups of G >= 8 lanes: lane l ends with
// word l & 7.  The first three steps halve the words a lane keeps, so a group
// takes 7 + log2(G / 8) shuffles, not 8 log2(G).
template <int G>
__device__ __forceinline__ uint32_t group_or(const uint32_t *acc) {
  const uint32_t lane = lane_id();
  uint32_t h[4], q[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bool up = lane & 4u;
    h[i] = (up ? acc[4 + i] : acc[i]) | __shfl_xor(up ? acc[i] : acc[4 + i], 4, kWave);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const bool up = lane & 2u;
    q[i] = (up ? h[2 + i] : h[i]) | __shfl_xor(up ? h[i] : h[2 + i], 2, kWave);
  }
  const bool up = lane & 1u;
  uint32_t r = (up ? q[1] : q[0]) | __shfl_xor(up ? q[0] : q[1], 1, kWave);
#pragma unroll
  for (int o = 8; o < G; o <<= 1) r |= __shfl_xor(r, o, kWave);
  return r;
}

// Workgroup OR of the lane masks: word t of it in threads t < 8.
__device__ __forceinline__ uint32_t block_or(const uint32_t *acc, uint32_t (*s)[kMW]) {
  uint32_t r = group_or<kWave>(acc);
  if (lane_id() < kMW) s[threadIdx.x / kWave][lane_id()] = r;
  __syncthreads();
  if (threadIdx.x < kMW)
    for (uint32_t w = 1; w < kMB / kWave; ++w) r |= s[w][threadIdx.x];
  __syncthreads();
  return r;
}

__device__ __forceinline__ uint32_t full_word(uint32_t k, uint32_t j) {
  return k >= 32 * j + 32 ? 0xffffffffu : k <= 32 * j ? 0u : (1u << (k - 32 * j)) - 1u;
}

// New bits of v from the OR of its in-neighbours' frontier masks.
__device__ __forceinline__ void mbfs_pull_finish(const MbfsParams &p, uint32_t v, const uint32_t *acc, uint32_t *An,
                                                 uint32_t *Fn, int32_t nlevel, uint32_t &nf,
                                                 unsigned long long &mf) {
  uint32_t vv[kMW], nwv[kMW];
  bool any = false;
#pragma unroll
  for (int j = 0; j < kMW; ++j) {
    vv[j] = p.V[(size_t)v * kMW + j];
    nwv[j] = acc[j] & ~vv[j];
    any = any || nwv[j];
  }
  if (!any) return;
  const uint32_t bit = 1u << (v & 31);
  if (mbfs_apply(p, v, nwv, vv, Fn)) atomicOr(&p.D[v >> 5], bit);
  atomicOr(&An[v >> 5], bit);
  nf += 1;
  mf += p.row_ptr[v + 1] - p.row_ptr[v];
  mbfs_record(p, v, nwv, nlevel);
}

// The same by eight neighbouring lanes, a mask word each (if `valid`): where a
// group of lanes has ORed the masks, one lane of it would go through the
// vertex's 352 bytes of state alone (256 sources on RMAT-20 1.59 ms a call so,
// 1.50 by eight).  Every lane of the wave must call.
__device__ __forceinline__ void mbfs_pull_finish8(const MbfsParams &p, bool valid, uint32_t v, uint32_t acc,
                                                 uint32_t *An, uint32_t *Fn, int32_t nlevel, uint32_t &nf,
                                                 unsigned long long &mf) {
  const uint32_t lane = lane_id(), j = lane & 7u, sh = lane & 56u;
  const uint32_t vv = valid ? p.V[(size_t)v * kMW + j] : 0u;
  const uint32_t nw = valid ? acc & ~vv : 0u;
  const uint32_t some = (uint32_t)(ballot(nw != 0) >> sh) & 0xffu;
  const uint32_t full = (uint32_t)(ballot((vv | nw) == full_word(p.k, j)) >> sh) & 0xffu;
  if (!some) return;
  Fn[(size_t)v * kMW + j] = nw;
  if (nw) p.V[(size_t)v * kMW + j] = vv | nw;
  mbfs_record_word(p, v, j, nw, nlevel);
  if (j != 0) return;
  const uint32_t bit = 1u << (v & 31);
  if (full == 0xffu) atomicOr(&p.D[v >> 5], bit);
  atomicOr(&An[v >> 5], bit);
  nf += 1;
  mf += p.row_ptr[v + 1] - p.row_ptr[v];
}

constexpr uint32_t kCoopRows = 1u << 16;  // one-lane rows from which a wave records them together
constexpr int kCoopLanes = 16;            // and rows of the wave with something to record

// Pull level: every vertex not yet holding every source ORs the frontier
// masks of its active in-neighbours, with 1, 8, 64 or 256 lanes per vertex by
// in-degree; rows longer than the plan's chunk are cut into pieces whose ORs
// go to N (applied by mbfs_contract_kernel).
__global__ void __launch_bounds__(kMB) mbfs_pull_kernel(MbfsParams p, SegDev d) {
  MbfsCtl *ctl = p.ctl;
  if (__hip_atomic_load(&ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const uint32_t L = ctl->level;
  if (ctl->st[L & 1].mode == 0) return;
  __shared__ uint32_t s_or[kMB / kWave][kMW];
  __shared__ uint32_t s_acc[kMB][kMW + 1];
  const uint32_t *Ff, *Af;
  uint32_t *Fn, *An, *Ac, *Tc, *Tx;
  mbfs_buffers(p, L, Ff, Fn, Af, An, Ac, Tc, Tx);
  const int32_t nlevel = (int32_t)(L + 1);
  const uint32_t *rp = p.in_row_ptr;
  uint32_t nf = 0;
  unsigned long long mf = 0, insp = 0;
  // rows without in-edges (listed last) can gain nothing from a pull
  for (uint32_t b = blockIdx.x; b < d.live_end; b += gridDim.x) {
    uint32_t acc[kMW] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (b < d.role_start[1]) {
      // piece of a very long in-list: OR into N, touch T
      const uint32_t c = b;
      const uint32_t h = d.chunk_hub[c];
      const uint32_t v = d.hub_vertex[h];
      if (bm_test(p.D, v)) continue;
      const uint32_t beg = rp[v] + (c - d.hub_first[h]) * d.chunk;
      const uint32_t end = min(rp[v + 1], beg + d.chunk);
      lane_or<kMB>(p, Af, Ff, beg, end, threadIdx.x, acc);
      if (threadIdx.x == 0) insp += end - beg;
      const uint32_t r = block_or(acc, s_or);
      if (threadIdx.x < kMW) {
        const uint32_t nv = r & ~p.V[(size_t)v * kMW + threadIdx.x];
        if (nv) atomicOr(&p.N[(size_t)v * kMW + threadIdx.x], nv);
        const uint64_t any = ballot(nv != 0);
        if (threadIdx.x == 0 && any) atomicOr(&Tc[v >> 5], 1u << (v & 31));
      }
    } else if (b < d.role_start[2]) {
      const uint32_t v = d.list[d.off[3] + (b - d.role_start[1])];
      if (bm_test(p.D, v)) continue;
      lane_or<kMB>(p, Af, Ff, rp[v], rp[v + 1], threadIdx.x, acc);
      if (threadIdx.x == 0) insp += rp[v + 1] - rp[v];
      const uint32_t r = block_or(acc, s_or);
      if (threadIdx.x < kWave) mbfs_pull_finish8(p, threadIdx.x < kMW, v, r, An, Fn, nlevel, nf, mf);
    } else if (b < d.role_start[3]) {
      const uint32_t idx = d.off[2] + (b - d.role_start[2]) * (kMB / 64) + threadIdx.x / 64;
      if (idx >= d.off[3]) continue;
      const uint32_t v = d.list[idx];
      if (bm_test(p.D, v)) continue;
      const uint32_t j = threadIdx.x % 64;
      lane_or<64>(p, Af, Ff, rp[v], rp[v + 1], j, acc);
      if (j == 0) insp += rp[v + 1] - rp[v];
      mbfs_pull_finish8(p, j < kMW, v, group_or<64>(acc), An, Fn, nlevel, nf, mf);
    } else if (b < d.role_start[4]) {
      const uint32_t idx = d.off[1] + (b - d.role_start[3]) * (kMB / 8) + threadIdx.x / 8;
      const uint32_t j = threadIdx.x % 8;
      const bool ok = idx < d.off[2];
      const uint32_t v = ok ? d.list[idx] : 0u;
      const bool todo = ok && !bm_test(p.D, v);
      if (todo) lane_or<8>(p, Af, Ff, rp[v], rp[v + 1], j, acc);
      if (todo && j == 0) insp += rp[v + 1] - rp[v];
      mbfs_pull_finish8(p, todo, v, group_or<8>(acc), An, Fn, nlevel, nf, mf);
    } else {
      const uint32_t idx = d.off[0] + (b - d.role_start[4]) * kMB + threadIdx.x;
      const bool ok = idx < d.off[1];
      const uint32_t v = ok ? d.list[idx] : 0u;
      const bool todo = ok && !bm_test(p.D, v);
      bool got = false;  // a source that v does not hold yet
      if (todo) {
        uint32_t vv[kMW];
#pragma unroll
        for (int j = 0; j < kMW; ++j) vv[j] = p.V[(size_t)v * kMW + j];
        // kVisitUnroll in-neighbours per step, stopping after the step that
        // completes the mask
        constexpr int U = kVisitUnroll;
        uint32_t k = 0;
        const uint32_t eb = rp[v], ee = rp[v + 1];
        for (uint32_t e = eb; e < ee; e += U) {
          uint32_t u[U];
          bool act[U];
#pragma unroll
          for (int i = 0; i < U; ++i) u[i] = e + i < ee ? p.in_col[e + i] : 0xffffffffu;
#pragma unroll
          for (int i = 0; i < U; ++i) act[i] = u[i] != 0xffffffffu && bm_test(Af, u[i]);
#pragma unroll
          for (int i = 0; i < U; ++i)
            if (act[i]) or_mask(acc, Ff, u[i]);
          k += ee - e < (uint32_t)U ? ee - e : (uint32_t)U;
          bool full = true;
#pragma unroll
          for (int j = 0; j < kMW; ++j) full = full && ((acc[j] | vv[j]) == p.full[j]);
          if (full) break;
        }
        insp += k;
#pragma unroll
        for (int j = 0; j < kMW; ++j) got = got || (acc[j] & ~vv[j]);
      }
      // The wave goes through its vertices' state eight vertices at a time
      // (word j of vertex 8 r + q to lane 8 q + j): whole lines, but eight
      // rounds one after another, which only a chip full of waves hides and
      // only a wave with much to record repays.  By lanes and so: 256 sources
      // on RMAT-20 1.50 and 1.36 ms, 64 sources 0.88 and 0.84, 256 on 2^18
      // vertices with 2^20 uniform edges 1.12 and 0.91; levels of small
      // frontiers, 40 sources on a 1000 x 1000 grid, 77 and 85 (8 to 48 rows:
      // 78).
      const uint64_t gots = ballot(got);
      if (p.sstride < 64 || d.off[1] - d.off[0] < kCoopRows || __popcll(gots) < kCoopLanes) {
        if (got) mbfs_pull_finish(p, v, acc, An, Fn, nlevel, nf, mf);
        continue;
      }
      const uint32_t lane = lane_id(), w0 = threadIdx.x - lane;
#pragma unroll
      for (int j = 0; j < kMW; ++j) s_acc[threadIdx.x][j] = acc[j];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      for (uint32_t r = 0; r < 8; ++r) {
        if (!((gots >> (8 * r)) & 0xffu)) continue;
        const uint32_t from = 8 * r + lane / 8;
        mbfs_pull_finish8(p, (gots >> from) & 1u, __shfl(v, (int)from, kWave), s_acc[w0 + from][lane & 7u], An, Fn,
                          nlevel, nf, mf);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();  // s_acc is rewritten by the wave's next vertices
    }
  }
  flush_counters<kMB>(&ctl->cnt[L % 3], nf, mf, insp);
}

// Apply N to every touched vertex (every vertex reached by a push level,
// and the long rows of a pull level).  One lane per bitmap word owns the 32
// vertices of that word.
__global__ void __launch_bounds__(kMB) mbfs_contract_kernel(MbfsParams p) {
  MbfsCtl *ctl = p.ctl;
  if (__hip_atomic_load(&ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const uint32_t L = ctl->level_e;
  const uint32_t *Ff, *Af;
  uint32_t *Fn, *An, *Ac, *Tc, *Tx;
  mbfs_buffers(p, L, Ff, Fn, Af, An, Ac, Tc, Tx);
  const int32_t nlevel = (int32_t)(L + 1);
  uint32_t nf = 0;
  unsigned long long mf = 0;
  // One lane per vertex (touched vertices cluster in few words on a
  // renumbered graph, so a lane per word left most lanes idle); a wave
  // covers two bitmap words, whose new bits lanes 0 and 32 write.
  const uint32_t lane = lane_id();
  for (uint32_t v = blockIdx.x * kMB + threadIdx.x; v < p.nw * 32u; v += gridDim.x * kMB) {
    const uint32_t w = v >> 5, b = v & 31u;
    bool act = false, dn = false;
    if ((Tc[w] >> b) & 1u) {
      uint32_t nwv[kMW], vv[kMW];
      bool any = false;
#pragma unroll
      for (int j = 0; j < kMW; ++j) {
        const uint32_t nj = p.N[(size_t)v * kMW + j];
        if (nj) p.N[(size_t)v * kMW + j] = 0u;
        vv[j] = p.V[(size_t)v * kMW + j];
        nwv[j] = nj & ~vv[j];
        any = any || nwv[j];
      }
      if (any) {
        dn = mbfs_apply(p, v, nwv, vv, Fn);
        act = true;
        nf += 1;
        mf += p.row_ptr[v + 1] - p.row_ptr[v];
        mbfs_record(p, v, nwv, nlevel);
      }
    }
    const uint64_t am = __ballot(act), dm = __ballot(dn);
    if ((lane & 31u) == 0) {
      const uint32_t anext = (uint32_t)(am >> (lane & 32u)), dnew = (uint32_t)(dm >> (lane & 32u));
      // |=: on a pull level the pull kernel has already set bits of this word
      if (anext) An[w] |= anext;
      if (dnew) p.D[w] |= dnew;
    }
  }
  flush_counters<kMB>(&ctl->cnt[L % 3], nf, mf, 0ull);
}

// Decide the next direction; compact the active bitmap when top-down.
__global__ void __launch_bounds__(kMB) mbfs_compact_kernel(MbfsParams p) {
  MbfsCtl *ctl = p.ctl;
  if (__hip_atomic_load(&ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const uint32_t L = ctl->level_e;
  const CtrSum c = ctr_total(&ctl->cnt[L % 3]);
  const MbfsState st = ctl->st[L & 1];
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  const uint32_t nbu = st.nbu + st.mode;
  if (c.nf == 0 || L + 1 > p.n) {
    if (lead) {
      ctl->levels = L + 1;
      ctl->nbu = nbu;
      ctl->overflow = c.nf != 0;
      ctl->done = 1u;
    }
    return;
  }
  const unsigned long long mu = st.mu > c.mf ? st.mu - c.mf : 0ull;
  const bool next_bu = choose_bottom_up(st.mode != 0, p.can_bu != 0, c.nf, c.mf, mu, p.n, p.alpha, p.beta);
  if (lead) {
    MbfsState ns;
    ns.mu = mu;
    ns.mode = next_bu ? 1u : 0u;
    ns.nbu = nbu;
    ctl->st[(L + 1) & 1] = ns;
    ctl->level = L + 1;
  }
  if (!next_bu)
    compact_step<kMB>(p.A + (size_t)(L % 3) * p.nwp, p.nw, p.row_ptr, p.hub_thr, p.queue, &ctl->qfill[(L + 1) & 1],
                      p.hubs, &ctl->hfill[(L + 1) & 1], blockIdx.x, gridDim.x, IdRow());
}

// Reset state for one group of sources (grid-stride).
__global__ void mbfs_reset_kernel(MbfsParams p) {
  const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  const size_t nm = (size_t)p.n * kMW;
  for (size_t i = tid; i < nm; i += stride) {
    p.V[i] = 0u;
    p.N[i] = 0u;
  }
  for (size_t i = tid; i < (size_t)p.nwp * 3; i += stride) p.A[i] = 0u;
  for (size_t i = tid; i < (size_t)p.nwp * 2; i += stride) p.T[i] = 0u;
  for (size_t i = tid; i < (size_t)p.nwp; i += stride) p.D[i] = 0u;
  for (size_t i = tid; i < sizeof(MbfsCtl) / 4; i += stride) reinterpret_cast<uint32_t *>(p.ctl)[i] = 0u;
}

// Level-0 state from the sources (one workgroup): V and the level-0
// frontier F (buffer 1) get bit s at srcs[s]; queue = distinct sources.
__global__ void mbfs_seed_kernel(MbfsParams p, const uint32_t *__restrict__ srcs) {
  const size_t fstride = (size_t)p.n * kMW;
  uint32_t *F0 = p.F + fstride;
  uint32_t *A0 = p.A + (size_t)2 * p.nwp;
  for (uint32_t s = threadIdx.x; s < p.k; s += blockDim.x)
    for (int j = 0; j < kMW; ++j) F0[(size_t)srcs[s] * kMW + j] = 0u;
  __syncthreads();
  for (uint32_t s = threadIdx.x; s < p.k; s += blockDim.x) {
    const uint32_t v = srcs[s];
    atomicOr(&p.V[(size_t)v * kMW + s / 32], 1u << (s % 32));
    atomicOr(&F0[(size_t)v * kMW + s / 32], 1u << (s % 32));
    p.S[(size_t)v * p.sstride + s] = 0;  // level 0; distinct sources own distinct bytes
  }
  __syncthreads();
  // distinct source vertices form the level-0 frontier
  auto claim = [&](uint32_t s) -> uint32_t {
    const uint32_t v = srcs[s];
    const uint32_t old = atomicOr(&A0[v >> 5], 1u << (v & 31));
    return (old & (1u << (v & 31))) ? 0xffffffffu : v;
  };
  unsigned long long deg = 0;
  seed_frontier(srcs, p.k, p.row_ptr, p.hub_thr, p.queue, &p.ctl->qfill[0], p.hubs, &p.ctl->hfill[0], claim, IdRow(),
                &deg);
  for (uint32_t s = threadIdx.x; s < p.k; s += blockDim.x) {
    const uint32_t v = srcs[s];
    bool full = true;
    for (int j = 0; j < kMW; ++j) full = full && (p.V[(size_t)v * kMW + j] == p.full[j]);
    if (full) atomicOr(&p.D[v >> 5], 1u << (v & 31));
  }
  if (threadIdx.x == 0) {
    p.ctl->st[0].mu = p.m > deg ? p.m - deg : 0ull;
    p.ctl->st[0].mode = 0;
    p.ctl->st[0].nbu = 0;
  }
}

// Output for one group: levels[s * n + v] for s < k from the level bytes
// (kInf where V lacks bit s).  A workgroup takes kLevTile consecutive
// vertices: their rows of S are one contiguous block, staged in LDS (rows
// padded by a dword so the per-source column reads are conflict-free);
// each wave then stores kLevTile consecutive int32 of one source's output
// row per step.
constexpr int kLevTile = 64;

__global__ void __launch_bounds__(kMB) mbfs_levels_kernel(MbfsParams p) {
  __shared__ uint32_t s_row[kLevTile][kMW * 8 + 1];
  __shared__ uint32_t s_vis[kLevTile][kMW + 1];
  const uint32_t kw = p.sstride / 32;  // 32-source groups in a row
  const uint32_t q4 = p.sstride / 16;  // uint4 per row
  for (uint32_t v0 = blockIdx.x * kLevTile; v0 < p.n; v0 += gridDim.x * kLevTile) {
    const uint32_t rows = min((uint32_t)kLevTile, p.n - v0);
    // output vertex v0 + r reads the row of vertex imap[v0 + r] (a whole
    // sstride-byte row, so a renumbered twin still reads full lines)
    for (uint32_t q = threadIdx.x; q < rows * q4; q += kMB) {
      const uint32_t ov = v0 + q / q4, tv = p.imap ? p.imap[ov] : ov;
      const uint4 x = reinterpret_cast<const uint4 *>(p.S + (size_t)tv * p.sstride)[q % q4];
      uint32_t *d = &s_row[q / q4][(q % q4) * 4];
      d[0] = x.x;
      d[1] = x.y;
      d[2] = x.z;
      d[3] = x.w;
    }
    for (uint32_t q = threadIdx.x; q < rows * kw; q += kMB) {
      const uint32_t ov = v0 + q / kw, tv = p.imap ? p.imap[ov] : ov;
      s_vis[q / kw][q % kw] = p.V[(size_t)tv * kMW + q % kw];
    }
    __syncthreads();
    const uint32_t t = threadIdx.x % kLevTile;
    if (t < rows) {
      const uint32_t v = v0 + t;
      for (uint32_t s = threadIdx.x / kLevTile; s < p.k; s += kMB / kLevTile) {
        const bool seen = (s_vis[t][s >> 5] >> (s & 31)) & 1u;
        const uint32_t b = (s_row[t][s >> 2] >> (8 * (s & 3))) & 0xFFu;
        if (seen && b == 0xFFu) continue;  // level >= 255: already in the output
        p.levels[(size_t)s * p.n + v] = seen ? (int32_t)b : kInf;
      }
    }
    __syncthreads();
  }
}

// Bytes per vertex row of S for groups of up to k sources.
static inline uint32_t level_stride(uint32_t k) { return (std::min(k, 256u) + 31) / 32 * 32; }

struct MbfsWork {
  uint32_t *V = nullptr, *F = nullptr, *N = nullptr, *A = nullptr, *T = nullptr, *D = nullptr, *queue = nullptr;
  uint8_t *S = nullptr;
  uint2 *hubs = nullptr;
  MbfsCtl *ctl = nullptr, *h_ctl = nullptr;
  uint32_t *srcs = nullptr;                // a group's sources
  uint32_t last_levels = 0, sstride = 0;
  uint32_t room = 0;                       // bytes per S row allocated
  ~MbfsWork() {
    void *ps[] = {V, F, N, A, T, D, queue, S, hubs, ctl, srcs};
    for (void *p : ps)
      if (p) (void)hipFree(p);
    if (h_ctl) (void)hipHostFree(h_ctl);
  }
  // k: the largest group (at most 256 sources); S rows hold ceil(k/32)*32 bytes
  int alloc(uint32_t n, uint32_t nwp, uint64_t m, uint32_t k) {
    const size_t nm = (size_t)n * kMW * 4;
    room = sstride = level_stride(k);
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&S), (size_t)n * sstride));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&hubs), hub_capacity(m) * sizeof(uint2)));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&V), nm));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&F), nm * 2));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&N), nm));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&A), (size_t)nwp * 4 * 3));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&T), (size_t)nwp * 4 * 2));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&D), (size_t)nwp * 4));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&queue), (size_t)n * 4));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&ctl), sizeof(MbfsCtl)));
    OLV_HIP(hipMalloc(reinterpret_cast<void **>(&srcs), 256 * 4));
    OLV_HIP(hipHostMalloc(reinterpret_cast<void **>(&h_ctl), sizeof(MbfsCtl), hipHostMallocDefault));
    return OLV_OK;
  }
};

static unsigned mgrid(size_t items, size_t per) {
  size_t b = (items + per - 1) / per;
  return (unsigned)std::max<size_t>(1, std::min(b, (size_t)cu_count() * 8));
}

// Work larger than this is freed after the call: its allocation is little
// beside a traversal of that many bytes.
constexpr size_t kMbfsKeepBytes = size_t(4) << 30;

void free_mbfs_work(olv_graph *g) { delete g->mbfs.exchange(nullptr); }

static MbfsParams mbfs_params(const olv_graph *g, MbfsWork &w, uint32_t k, int32_t *levels) {
  MbfsParams p;
  std::memset(&p, 0, sizeof(p));
  p.row_ptr = g->row_ptr;
  p.col = g->col;
  p.in_row_ptr = g->in_row_ptr;
  p.in_col = g->in_col;
  p.n = g->n;
  p.nw = (g->n + 31) / 32;
  p.nwp = (p.nw + 63) / 64 * 64;
  p.k = k;
  for (int j = 0; j < kMW; ++j) {
    const int lo = j * 32;
    const int bits = std::max(0, std::min(32, (int)k - lo));
    p.full[j] = bits == 32 ? 0xffffffffu : ((1u << bits) - 1u);
  }
  p.V = w.V;
  p.F = w.F;
  p.N = w.N;
  p.A = w.A;
  p.T = w.T;
  p.D = w.D;
  p.queue = w.queue;
  p.hubs = w.hubs;
  p.S = w.S;
  p.levels = levels;
  p.sstride = w.sstride;
  p.ctl = w.ctl;
  p.m = g->m;
  p.wave_thr = g->tune.td_wave_thr;
  p.block_thr = g->tune.td_block_thr;
  p.hub_thr = g->tune.hub_thr;
  p.alpha = g->tune.alpha;
  p.beta = g->tune.beta;
  p.can_bu = g->in_row_ptr ? 1u : 0u;
  p.pull_per_cu = g->tune.mbfs_pull_per_cu;
  return p;
}

static int mbfs_enqueue_init(const MbfsParams &p, const uint32_t *d_srcs) {
  hipStream_t s = stream();
  hipLaunchKernelGGL(mbfs_reset_kernel, dim3(mgrid((size_t)p.n * kMW, 256)), dim3(256), 0, s, p);
  hipLaunchKernelGGL(mbfs_seed_kernel, dim3(1), dim3(256), 0, s, p, d_srcs);
  OLV_HIP(hipGetLastError());
  return OLV_OK;
}

static int mbfs_enqueue_levels(const MbfsParams &p, const SegDev &d, uint32_t count) {
  hipStream_t s = stream();
  const unsigned ge = (unsigned)cu_count() * 8;
  const unsigned gw = mgrid(p.nw, kMB);
  const unsigned gv = mgrid((size_t)p.nw * 32, kMB);  // one lane per vertex
  // pull workgroups per CU, at most one per virtual block of the bucket
  // plan (256 sources on RMAT-22: 48 gives 7.21 ms; 64: 7.21, 96: 7.25, 32:
  // 7.30, 16: 7.44, 8: 8.17)
  const unsigned gp =
      std::max<unsigned>(1u, std::min<unsigned>(d.role_start[5], (unsigned)cu_count() * p.pull_per_cu));
  for (uint32_t i = 0; i < count; ++i) {
    hipLaunchKernelGGL(mbfs_expand_kernel, dim3(ge), dim3(kMB), 0, s, p);
    hipLaunchKernelGGL(mbfs_pull_kernel, dim3(gp), dim3(kMB), 0, s, p, d);
    hipLaunchKernelGGL(mbfs_contract_kernel, dim3(gv), dim3(kMB), 0, s, p);
    hipLaunchKernelGGL(mbfs_compact_kernel, dim3(gw), dim3(kMB), 0, s, p);
  }
  OLV_HIP(hipGetLastError());
  return OLV_OK;
}

static int mbfs_enqueue_finish(const MbfsParams &p) {
  const size_t tiles = ((size_t)p.n + kLevTile - 1) / kLevTile;
  hipLaunchKernelGGL(mbfs_levels_kernel, dim3((unsigned)std::min<size_t>(tiles, (size_t)cu_count() * 64)), dim3(kMB),
                     0, stream(), p);
  OLV_HIP(hipGetLastError());
  return OLV_OK;
}

static int mbfs_read(MbfsWork &w) {
  OLV_HIP(hipMemcpyAsync(w.h_ctl, w.ctl, sizeof(MbfsCtl), hipMemcpyDeviceToHost, stream()));
  OLV_HIP(hipStreamSynchronize(stream()));
  return OLV_OK;
}

// In-degree buckets for pull levels (empty schedule when pull is off).
// The graph batched BFS runs on: g's renumbered twin unless OLV_GRAPH_ORDER
// (seeds mapped to the twin's numbering in place), else g itself.
static int mbfs_target(olv_graph *g, unsigned flags, std::vector<uint32_t> &seeds, olv_graph **run) {
  *run = g;
  if (flags & OLV_GRAPH_ORDER) return OLV_OK;
  OLV_TRY(ensure_twin(g));
  g->twin->tune = g->tune;
  for (uint32_t &x : seeds) x = g->h_rl_pi[x];
  *run = g->twin;
  return OLV_OK;
}

static void mbfs_map(const olv_graph *g, const olv_graph *run, MbfsParams &p) {
  if (run == g) return;
  p.omap = run->out_map;
  p.imap = g->rl_pi;
}

static int mbfs_pull_plan(olv_graph *g, unsigned flags, SegDev *d) {
  std::memset(d, 0, sizeof(*d));
  if (flags & OLV_NO_DIRECTION_OPT) return OLV_OK;
  if (!g->in_row_ptr) OLV_TRY(olv_graph_build_transpose(g));
  if (!g->plan_in_ready || seg_plan_stale(g->plan_in, g->tune)) {
    OLV_TRY(build_seg_plan(g, true, g->plan_in));
    g->plan_in_ready = true;
  }
  *d = make_seg_dev(g->plan_in, g->tune);
  return OLV_OK;
}

// Run one group to completion: levels enqueued in chunks, the first as long as
// the last group was deep (of this call or the one before), those after it 8,
// 16, ...: groups of one graph differ by a few levels.
static int mbfs_run_group(const MbfsParams &p, const SegDev &d, MbfsWork &w, const uint32_t *d_srcs) {
  OLV_TRY(mbfs_enqueue_init(p, d_srcs));
  uint32_t chunk = std::max(4u, w.last_levels), more = 4;
  uint64_t enq = 0;
  for (;;) {
    OLV_TRY(mbfs_enqueue_levels(p, d, chunk));
    enq += chunk;
    OLV_TRY(mbfs_read(w));
    if (w.h_ctl->done) break;
    if (enq > (uint64_t)p.n + 2) return fail(OLV_EINTERNAL, "olv_bfs_batched: level loop did not terminate");
    chunk = more = std::min(more * 2, 256u);
  }
  if (w.h_ctl->overflow) return fail(OLV_EINTERNAL, "olv_bfs_batched: more than n levels");
  w.last_levels = w.h_ctl->levels;
  return mbfs_enqueue_finish(p);
}

}  // namespace olv

// --------------------------------------------------------------- plans
struct olv_plan {
  int kind = 0;  // 1 = multi-source BFS, 2 = batched BFS
  const olv_graph *g = nullptr;
  olv::DevBuf seeds;
  uint32_t k = 0;
  int32_t *levels = nullptr;
  bool can_bu = true;
  bool narrow = false;  // BFS: with narrow launches
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  olv::BfsWork *bw = nullptr;
  olv::MbfsWork *mw = nullptr;
  std::vector<olv::MbfsParams> groups;
  olv::SegDev seg;
  ~olv_plan() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    delete mw;
  }
};

namespace olv {

// Capture `enqueue` (stream-ordered work) into plan->graph/exec.
template <class Fn>
static int capture(olv_plan *plan, Fn enqueue) {
  hipStream_t user = stream();
  hipStream_t cap = nullptr;
  OLV_HIP(hipStreamCreateWithFlags(&cap, hipStreamNonBlocking));
  hipError_t e = hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal);
  if (e != hipSuccess) {
    (void)hipStreamDestroy(cap);
    return fail(OLV_EHIP, "hipStreamBeginCapture failed: %s", hipGetErrorString(e));
  }
  olv_set_stream(cap);
  int st = enqueue();
  olv_set_stream(user);
  hipGraph_t graph = nullptr;
  e = hipStreamEndCapture(cap, &graph);
  (void)hipStreamDestroy(cap);
  if (st != OLV_OK) {
    if (graph) (void)hipGraphDestroy(graph);
    return st;
  }
  if (e != hipSuccess) return fail(OLV_EHIP, "hipStreamEndCapture failed: %s", hipGetErrorString(e));
  plan->graph = graph;
  e = hipGraphInstantiate(&plan->exec, graph, nullptr, nullptr, 0);
  if (e != hipSuccess) return fail(OLV_EHIP, "hipGraphInstantiate failed: %s", hipGetErrorString(e));
  return OLV_OK;
}

}  // namespace olv

using namespace olv;

extern "C" {

int olv_bfs_multisource(const olv_graph *g, const uint32_t *srcs, uint32_t k, int32_t *levels, unsigned flags,
                        olv_stats *st) {
  return bfs_multisource(g, srcs, k, true, levels, flags, st);
}

int olv_bfs_batched(const olv_graph *cg, const uint32_t *srcs, uint32_t k, int32_t *levels, unsigned flags,
                    olv_stats *st) {
  if (!cg || !srcs || !levels) return fail(OLV_EINVAL, "olv_bfs_batched: NULL argument");
  if (k == 0) return fail(OLV_EINVAL, "olv_bfs_batched: no source");
  olv_graph *g = const_cast<olv_graph *>(cg);
  for (uint32_t i = 0; i < k; ++i)
    if (srcs[i] >= g->n) return fail(OLV_EINVAL, "olv_bfs_batched: source %u out of range (n=%u)", srcs[i], g->n);
  if ((uint64_t)k * g->n > (1ull << 40)) return fail(OLV_ERANGE, "olv_bfs_batched: output too large");
  std::vector<uint32_t> seeds(srcs, srcs + k);
  olv_graph *rg = nullptr;
  OLV_TRY(mbfs_target(g, flags, seeds, &rg));
  SegDev d;
  OLV_TRY(mbfs_pull_plan(rg, flags, &d));
  const bool host = (flags & OLV_PTR_HOST) != 0;
  // The work buffers stay with the graph: allocating and freeing them took
  // 0.7 ms of a 2.5 ms call (256 sources on RMAT-20, 0.45 GB).
  WorkLease<MbfsWork> lease(g->mbfs);
  if (!lease.w || lease.w->room < level_stride(k)) {
    lease.renew();
    OLV_TRY(lease.w->alloc(g->n, ((g->n + 31) / 32 + 63) / 64 * 64, g->m, std::min(k, 256u)));
  }
  MbfsWork &w = *lease.w;
  w.sstride = level_stride(k);
  DevBuf d_out;
  int32_t *out = levels;
  if (host) {
    OLV_TRY(d_out.alloc((size_t)k * g->n * 4));
    out = d_out.as<int32_t>();
  }
  Timer t;
  t.start();
  uint32_t max_levels = 0, bu_levels = 0;
  for (uint32_t g0 = 0; g0 < k; g0 += 256) {
    const uint32_t kg = std::min(256u, k - g0);
    MbfsParams p = mbfs_params(rg, w, kg, out + (size_t)g0 * g->n);
    mbfs_map(g, rg, p);
    if (flags & OLV_NO_DIRECTION_OPT) p.can_bu = 0;
    OLV_HIP(hipMemcpyAsync(w.srcs, seeds.data() + g0, (size_t)kg * 4, hipMemcpyHostToDevice, stream()));
    OLV_TRY(mbfs_run_group(p, d, w, w.srcs));
    max_levels = std::max(max_levels, w.h_ctl->levels);
    bu_levels += w.h_ctl->nbu;
  }
  t.stop();
  const double ms = t.ms();
  if (st) {
    std::memset(st, 0, sizeof(*st));
    st->elapsed_ms = ms;
    st->iterations = max_levels;
    st->bottom_up_levels = bu_levels;
    OLV_TRY(reach_stats(g, out, k, st));
  }
  if (host) OLV_HIP(hipMemcpy(levels, out, (size_t)k * g->n * 4, hipMemcpyDeviceToHost));
  // (the stop event has been waited for: the stream is done with the work)
  if ((size_t)g->n * (w.room + 5 * kMW * 4) <= kMbfsKeepBytes) lease.keep();
  return OLV_OK;
}

}  // extern "C"

// ------------------------------------------------------------ graph union
namespace olv {

__global__ void union_rows_kernel(const uint32_t *__restrict__ rp, uint32_t n, uint32_t voff, uint32_t eoff,
                                  uint32_t *__restrict__ out) {
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x)
    out[voff + v] = rp[v] + eoff;
}

__global__ void union_cols_kernel(const uint32_t *__restrict__ c, uint32_t m, uint32_t add,
                                  uint32_t *__restrict__ out) {
  for (uint32_t e = blockIdx.x * blockDim.x + threadIdx.x; e < m; e += gridDim.x * blockDim.x) out[e] = c[e] + add;
}

__global__ void set_word_kernel(uint32_t *p, uint32_t v) { *p = v; }

static int concat_rows(const uint32_t *const *rps, const uint32_t *ns, const uint32_t *voff, const uint32_t *eoff,
                       uint32_t k, uint32_t n_total, uint32_t m_total, uint32_t **out) {
  OLV_HIP(hipMalloc(reinterpret_cast<void **>(out), ((size_t)n_total + 1) * 4));
  for (uint32_t i = 0; i < k; ++i)
    hipLaunchKernelGGL(union_rows_kernel, dim3(mgrid(ns[i], 256)), dim3(256), 0, stream(), rps[i], ns[i], voff[i],
                       eoff[i], *out);
  hipLaunchKernelGGL(set_word_kernel, dim3(1), dim3(1), 0, stream(), *out + n_total, m_total);
  OLV_HIP(hipGetLastError());
  return OLV_OK;
}

static int concat_cols(const uint32_t *const *cs, const uint32_t *ms, const uint32_t *eoff, const uint32_t *adds,
                       uint32_t k, uint32_t m_total, uint32_t **out) {
  OLV_HIP(hipMalloc(reinterpret_cast<void **>(out), std::max<size_t>(m_total, 1) * 4));
  for (uint32_t i = 0; i < k; ++i)
    if (ms[i])
      hipLaunchKernelGGL(union_cols_kernel, dim3(mgrid(ms[i], 256)), dim3(256), 0, stream(), cs[i], ms[i], adds[i],
                         *out + eoff[i]);
  OLV_HIP(hipGetLastError());
  return OLV_OK;
}

static int graph_union(olv_graph *const *gs, uint32_t k, olv_graph **out, std::vector<uint32_t> &voff) {
  if (!gs || !out || k == 0) return fail(OLV_EINVAL, "olv_graph_union: bad arguments");
  voff.assign(k + 1, 0);
  std::vector<uint32_t> eoff(k + 1, 0), ns(k), ms(k);
  bool all_t = true;
  uint64_t nt = 0, mt = 0;
  for (uint32_t i = 0; i < k; ++i) {
    if (!gs[i]) return fail(OLV_EINVAL, "olv_graph_union: graph %u is NULL", i);
    ns[i] = gs[i]->n;
    ms[i] = gs[i]->m;
    voff[i] = (uint32_t)nt;
    eoff[i] = (uint32_t)mt;
    nt += gs[i]->n;
    mt += gs[i]->m;
    all_t = all_t && gs[i]->in_row_ptr;
    if (nt >= (1ull << 32) || mt >= (1ull << 32)) return fail(OLV_ERANGE, "olv_graph_union: union too large");
  }
  voff[k] = (uint32_t)nt;
  eoff[k] = (uint32_t)mt;
  olv_graph *u = new olv_graph();
  u->device = current_device();
  u->n = (uint32_t)nt;
  u->m = (uint32_t)mt;
  std::vector<const uint32_t *> rps(k), cs(k), irps(k), ics(k), ies(k);
  for (uint32_t i = 0; i < k; ++i) {
    rps[i] = gs[i]->row_ptr;
    cs[i] = gs[i]->col;
    irps[i] = gs[i]->in_row_ptr;
    ics[i] = gs[i]->in_col;
    ies[i] = gs[i]->in_eid;
    u->max_outdeg = std::max(u->max_outdeg, gs[i]->max_outdeg);
    u->max_indeg = std::max(u->max_indeg, gs[i]->max_indeg);
  }
  int st = OLV_OK;
  do {
    if ((st = concat_rows(rps.data(), ns.data(), voff.data(), eoff.data(), k, u->n, u->m, &u->row_ptr))) break;
    if ((st = concat_cols(cs.data(), ms.data(), eoff.data(), voff.data(), k, u->m, &u->col))) break;
    if (hipMalloc(reinterpret_cast<void **>(&u->inv_outdeg), (size_t)u->n * 4) != hipSuccess) {
      st = fail(OLV_ENOMEM, "olv_graph_union: allocation failed");
      break;
    }
    for (uint32_t i = 0; i < k; ++i)
      if (hipMemcpyAsync(u->inv_outdeg + voff[i], gs[i]->inv_outdeg, (size_t)ns[i] * 4, hipMemcpyDeviceToDevice,
                         stream()) != hipSuccess) {
        st = fail(OLV_EHIP, "olv_graph_union: copy failed");
        break;
      }
    if (st) break;
    if (all_t) {
      if ((st = concat_rows(irps.data(), ns.data(), voff.data(), eoff.data(), k, u->n, u->m, &u->in_row_ptr))) break;
      if ((st = concat_cols(ics.data(), ms.data(), eoff.data(), voff.data(), k, u->m, &u->in_col))) break;
      if ((st = concat_cols(ies.data(), ms.data(), eoff.data(), eoff.data(), k, u->m, &u->in_eid))) break;
      if ((st = ensure_in_head(u))) break;
    }
    if (hipStreamSynchronize(stream()) != hipSuccess) st = fail(OLV_EHIP, "olv_graph_union: build failed");
  } while (0);
  if (st != OLV_OK) {
    olv_graph_destroy(u);
    return st;
  }
  u->tune = gs[0]->tune;
  *out = u;
  return OLV_OK;
}

}  // namespace olv

extern "C" {

int olv_graph_union(olv_graph *const *gs, uint32_t k, olv_graph **out, uint32_t *vertex_offsets) {
  std::vector<uint32_t> voff;
  OLV_TRY(graph_union(gs, k, out, voff));
  if (vertex_offsets) std::memcpy(vertex_offsets, voff.data(), voff.size() * 4);
  return OLV_OK;
}

int olv_bfs_multigraph(olv_graph *const *gs, uint32_t k, const uint32_t *srcs, int32_t *const *levels,
                       unsigned flags, olv_stats *st) {
  if (!gs || !srcs || !levels || k == 0) return fail(OLV_EINVAL, "olv_bfs_multigraph: bad arguments");
  for (uint32_t i = 0; i < k; ++i) {
    if (!gs[i] || !levels[i]) return fail(OLV_EINVAL, "olv_bfs_multigraph: NULL graph or output %u", i);
    if (srcs[i] >= gs[i]->n) return fail(OLV_EINVAL, "olv_bfs_multigraph: source %u out of range in graph %u", srcs[i], i);
  }
  olv_graph *u = nullptr;
  std::vector<uint32_t> voff;
  OLV_TRY(graph_union(gs, k, &u, voff));
  std::vector<uint32_t> seeds(k);
  for (uint32_t i = 0; i < k; ++i) seeds[i] = voff[i] + srcs[i];
  DevBuf lv;
  int s = lv.alloc((size_t)u->n * 4);
  if (s == OLV_OK)  // the union is built per call: no renumbered twin for it
    s = bfs_multisource(u, seeds.data(), k, true, lv.as<int32_t>(), (flags & ~OLV_PTR_HOST) | OLV_GRAPH_ORDER, st);
  if (s == OLV_OK) {
    const bool host = (flags & OLV_PTR_HOST) != 0;
    for (uint32_t i = 0; i < k && s == OLV_OK; ++i) {
      const size_t bytes = (size_t)gs[i]->n * 4;
      hipError_t e = host ? hipMemcpy(levels[i], lv.as<int32_t>() + voff[i], bytes, hipMemcpyDeviceToHost)
                          : hipMemcpyAsync(levels[i], lv.as<int32_t>() + voff[i], bytes, hipMemcpyDeviceToDevice, stream());
      if (e != hipSuccess) s = fail(OLV_EHIP, "olv_bfs_multigraph: output copy failed");
    }
    if (s == OLV_OK && hipStreamSynchronize(stream()) != hipSuccess) s = fail(OLV_EHIP, "olv_bfs_multigraph: sync failed");
  }
  olv_graph_destroy(u);
  return s;
}

// A plan captures init + the launch pairs (and narrow launches) of an eager
// run at plan time (levels are deterministic for fixed sources); a replay that
// still reports work left continues eagerly, so results never depend on what
// was captured.
int olv_plan_bfs(const olv_graph *g, const uint32_t *srcs, uint32_t k, int32_t *levels, unsigned flags,
                 olv_plan **out) {
  if (!g || !srcs || !levels || !out || k == 0) return fail(OLV_EINVAL, "olv_plan_bfs: bad arguments");
  *out = nullptr;
  for (uint32_t i = 0; i < k; ++i)
    if (srcs[i] >= g->n) return fail(OLV_EINVAL, "olv_plan_bfs: source %u out of range", srcs[i]);
  OLV_TRY(apply_cached_tuning(const_cast<olv_graph *>(g)));
  olv_plan *p = new olv_plan();
  p->kind = 1;
  p->g = g;
  p->k = k;
  p->levels = levels;
  p->can_bu = !(flags & OLV_NO_DIRECTION_OPT);
  int s = bfs_prepare(g, p->can_bu, &p->bw);
  if (s == OLV_OK)  // on g itself: its work buffers keep the depth the capture uses
    s = bfs_multisource(g, srcs, k, true, levels, (flags & ~(OLV_PTR_HOST | OLV_PERSISTENT | OLV_HOST_LOOP)) | OLV_GRAPH_ORDER,
                        nullptr);
  if (s == OLV_OK) s = p->seeds.alloc((size_t)k * 4);
  if (s == OLV_OK && hipMemcpy(p->seeds.p, srcs, (size_t)k * 4, hipMemcpyHostToDevice) != hipSuccess)
    s = fail(OLV_EHIP, "olv_plan_bfs: seed copy failed");
  uint32_t pairs = 0;
  if (s == OLV_OK) {
    pairs = bfs_pairs_hint(p->bw);
    p->narrow = bfs_deep_hint(p->bw);
  }
  if (s == OLV_OK)
    s = capture(p, [&]() -> int {
      OLV_TRY(bfs_enqueue_init(g, p->bw, p->seeds.as<uint32_t>(), k, srcs[0], levels, p->can_bu));
      return bfs_enqueue_levels(g, p->bw, levels, p->can_bu, pairs, p->narrow);
    });
  if (s != OLV_OK) {
    delete p;
    return s;
  }
  *out = p;
  return OLV_OK;
}

int olv_plan_bfs_batched(const olv_graph *cg, const uint32_t *srcs, uint32_t k, int32_t *levels, unsigned flags,
                         olv_plan **out) {
  if (!cg || !srcs || !levels || !out || k == 0) return fail(OLV_EINVAL, "olv_plan_bfs_batched: bad arguments");
  *out = nullptr;
  olv_graph *g = const_cast<olv_graph *>(cg);
  for (uint32_t i = 0; i < k; ++i)
    if (srcs[i] >= g->n) return fail(OLV_EINVAL, "olv_plan_bfs_batched: source %u out of range", srcs[i]);
  OLV_TRY(apply_cached_tuning(g));
  std::vector<uint32_t> seeds(srcs, srcs + k);
  olv_graph *rg = nullptr;
  OLV_TRY(mbfs_target(g, flags, seeds, &rg));
  SegDev d;
  OLV_TRY(mbfs_pull_plan(rg, flags, &d));
  olv_plan *p = new olv_plan();
  p->kind = 2;
  p->seg = d;
  p->g = g;
  p->k = k;
  p->levels = levels;
  p->mw = new MbfsWork();
  int s = p->mw->alloc(g->n, ((g->n + 31) / 32 + 63) / 64 * 64, g->m, std::min(k, 256u));
  if (s == OLV_OK) s = p->seeds.alloc((size_t)k * 4);
  if (s == OLV_OK && hipMemcpy(p->seeds.p, seeds.data(), (size_t)k * 4, hipMemcpyHostToDevice) != hipSuccess)
    s = fail(OLV_EHIP, "olv_plan_bfs_batched: seed copy failed");
  std::vector<uint32_t> depth;
  for (uint32_t g0 = 0; s == OLV_OK && g0 < k; g0 += 256) {
    const uint32_t kg = std::min(256u, k - g0);
    MbfsParams prm = mbfs_params(rg, *p->mw, kg, levels + (size_t)g0 * g->n);
    mbfs_map(g, rg, prm);
    if (flags & OLV_NO_DIRECTION_OPT) prm.can_bu = 0;
    p->groups.push_back(prm);
    s = mbfs_run_group(prm, p->seg, *p->mw, p->seeds.as<uint32_t>() + g0);  // learns the depth
    depth.push_back(p->mw->h_ctl->levels);
  }
  if (s == OLV_OK)
    s = capture(p, [&]() -> int {
      for (size_t i = 0; i < p->groups.size(); ++i) {
        OLV_TRY(mbfs_enqueue_init(p->groups[i], p->seeds.as<uint32_t>() + 256 * i));
        OLV_TRY(mbfs_enqueue_levels(p->groups[i], p->seg, depth[i]));
        OLV_TRY(mbfs_enqueue_finish(p->groups[i]));
      }
      return OLV_OK;
    });
  if (s != OLV_OK) {
    delete p;
    return s;
  }
  *out = p;
  return OLV_OK;
}

int olv_plan_launch(olv_plan *p, olv_stats *st) {
  if (!p || !p->exec) return fail(OLV_EINVAL, "olv_plan_launch: bad plan");
  Timer t;
  t.start();
  OLV_HIP(hipGraphLaunch(p->exec, stream()));
  t.stop();
  double ms = t.ms();
  uint32_t levels = 0, nbu = 0;
  if (p->kind == 1) {
    OLV_TRY(bfs_result(p->bw, &levels, &nbu));
    if (!bfs_done(p->bw)) {  // deeper than captured: finish eagerly
      Timer t2;
      t2.start();
      for (uint32_t chunk = 8; !bfs_done(p->bw); chunk = std::min(chunk * 2, 256u)) {
        OLV_TRY(bfs_enqueue_levels(p->g, p->bw, p->levels, p->can_bu, chunk, p->narrow));
        OLV_TRY(bfs_result(p->bw, &levels, &nbu));
      }
      t2.stop();
      ms += t2.ms();
    }
  } else {
    // each group ran to its captured depth; a group's done flag is only
    // kept for the last one, so re-check all groups' depths by replaying
    // nothing: the plan was built from a completed run of the same sources
    OLV_TRY(mbfs_read(*p->mw));
    if (!p->mw->h_ctl->done) return fail(OLV_EINTERNAL, "olv_plan_launch: batched plan did not finish");
    levels = p->mw->h_ctl->levels;
    nbu = p->mw->h_ctl->nbu;
  }
  if (st) {
    std::memset(st, 0, sizeof(*st));
    st->elapsed_ms = ms;
    st->iterations = levels;
    st->bottom_up_levels = nbu;
  }
  return OLV_OK;
}

int olv_plan_destroy(olv_plan *p) {
  if (p) {
    (void)hipStreamSynchronize(stream());
    delete p;
  }
  return OLV_OK;
}

int olv_set_direction(olv_graph *g, float alpha, float beta) {
  if (!g || !(alpha > 0) || !(beta > 0)) return fail(OLV_EINVAL, "olv_set_direction: bad arguments");
  g->tune.alpha = alpha;
  g->tune.beta = beta;
  return OLV_OK;
}

int olv_get_tuning(const olv_graph *g, uint32_t *wave_thr, uint32_t *block_thr, float *alpha, float *beta) {
  if (!g) return fail(OLV_EINVAL, "olv_get_tuning: NULL graph");
  if (wave_thr) *wave_thr = g->tune.td_wave_thr;
  if (block_thr) *block_thr = g->tune.td_block_thr;
  if (alpha) *alpha = g->tune.alpha;
  if (beta) *beta = g->tune.beta;
  return OLV_OK;
}

}  // extern "C"
