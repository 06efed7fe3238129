// Device construction of the source-segmented pull plan (blocked.hpp).
//
// The entries are sorted by the segment of their source (one or two radix
// passes; rows stay ascending inside a segment), cut into pieces, and the
// pieces are sorted twice: by row, which gives the combine its term lists,
// and by (segment, class), which gives the segment pass its layout.  Only
// the per-segment and per-(segment, class) counts come to the host, which
// deals the tasks out to the workgroups.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "blocked.hpp"
#include "radix.hpp"

namespace olv {

namespace {

unsigned pgrid(size_t items) {
  const size_t b = (items + 255) / 256;
  return (unsigned)std::max<size_t>(1, std::min(b, (size_t)cu_count() * 16));
}

constexpr uint32_t kDirectKeyBits = 4;  // class field of a piece's layout key

// Device binary search: first i in [0, m) with a[i] >= key (a ascending in
// `at`), m if none.
template <class At>
__device__ __forceinline__ uint32_t first_ge(uint32_t m, uint32_t key, At at) {
  uint32_t lo = 0, hi = m;
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (at(mid) < key) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ uint32_t row_of(const uint32_t *v, uint32_t i) { return v[i]; }
__device__ __forceinline__ uint32_t row_of(const uint2 *v, uint32_t i) { return v[i].x; }
__device__ __forceinline__ uint32_t slot_of(const uint32_t *, uint32_t) { return 0u; }
__device__ __forceinline__ uint32_t slot_of(const uint2 *v, uint32_t i) { return v[i].y; }

// flag[i] = 1 where entry i (sorted by segment, then row) starts a new
// (segment, row).
template <class V>
__global__ void piece_head_kernel(const uint32_t *__restrict__ key, const V *__restrict__ val, uint32_t m,
                                  uint32_t *__restrict__ flag) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (size_t)gridDim.x * blockDim.x)
    flag[i] = i == 0 || (key[i - 1] >> kSegBits) != (key[i] >> kSegBits) ||
              row_of(val, (uint32_t)i - 1) != row_of(val, (uint32_t)i);
}

// Cuts inside the (segment, row) groups that start at the flags of `scan`:
// every kPieceMax entries, and the tail at half its capacity when it would
// leave a quarter or more of that unused.
__global__ void piece_cut_kernel(const uint32_t *__restrict__ start, const uint32_t *__restrict__ count,
                                 uint32_t *__restrict__ flag) {
  const uint32_t groups = *count;
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < groups; p += gridDim.x * blockDim.x) {
    uint32_t a = start[p];
    const uint32_t end = start[p + 1];
    for (; end - a > kPieceMax; a += kPieceMax) flag[a + kPieceMax] = 1u;
    const uint32_t len = end - a;
    if (len <= kCutCap / 2) continue;
    const uint32_t cap = 1u << (32 - __clz(len - 1));
    if (len <= cap / 4 * 3) flag[a + cap / 2] = 1u;
  }
}

// out[0] = pieces, out[1] = rows up to the last one with entries, out[2 + s]
// = entries of segment s.
__global__ void seg_stat_kernel(const uint32_t *__restrict__ key, const uint32_t *__restrict__ scan, uint32_t m,
                                const uint32_t *__restrict__ rp, uint32_t n, uint32_t nseg,
                                uint32_t *__restrict__ out) {
  for (uint32_t s = blockIdx.x * blockDim.x + threadIdx.x; s < nseg; s += gridDim.x * blockDim.x) {
    const uint32_t a = first_ge(m, s, [&](uint32_t i) { return key[i] >> kSegBits; });
    const uint32_t b = first_ge(m, s + 1, [&](uint32_t i) { return key[i] >> kSegBits; });
    out[2 + s] = b - a;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    out[0] = scan[m];
    out[1] = first_ge(n, m, [&](uint32_t v) { return rp[v]; });
  }
}

__global__ void live_rows_kernel(const uint32_t *__restrict__ rp, uint32_t n, uint32_t m, uint32_t *__restrict__ out) {
  out[0] = first_ge(n, m, [&](uint32_t v) { return rp[v]; });
}

// pstart[p] = first entry of piece p (a flag of the scan); pstart[pieces] = m.
__global__ void piece_start_kernel(const uint32_t *__restrict__ scan, uint32_t m, uint32_t *__restrict__ pstart) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (size_t)gridDim.x * blockDim.x) {
    const uint32_t p = scan[i];
    if (scan[i + 1] != p) pstart[p] = (uint32_t)i;
    if (i + 1 == m) pstart[scan[m]] = m;
  }
}

template <class V>
__global__ void piece_row_kernel(const V *__restrict__ val, const uint32_t *__restrict__ pstart, uint32_t pieces,
                                 uint32_t *__restrict__ prow) {
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < pieces; p += gridDim.x * blockDim.x)
    prow[p] = row_of(val, pstart[p]);
}

// The layout key of every piece: (segment, class), or nseg << 4 for a piece
// whose entries the combine reads directly.
__global__ void piece_key_kernel(const uint32_t *__restrict__ key, const uint32_t *__restrict__ pstart,
                                 uint32_t pieces, const uint32_t *__restrict__ entries, uint32_t nseg, uint32_t *__restrict__ lkey) {
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < pieces; p += gridDim.x * blockDim.x) {
    const uint32_t a = pstart[p], len = pstart[p + 1] - a, s = key[a] >> kSegBits;
    uint32_t k = nseg << kDirectKeyBits;
    if (entries[s] >= kSegMinEntries) k = (s << kDirectKeyBits) | (len <= 1 ? 0u : 32u - __clz(len - 1));
    lkey[p] = k;
  }
}

// terms[j] = combine terms of the j-th piece in row order.
__global__ void piece_terms_kernel(const uint32_t *__restrict__ by_row, const uint32_t *__restrict__ pstart,
                                   const uint32_t *__restrict__ lkey, uint32_t pieces, uint32_t nseg,
                                   uint32_t *__restrict__ terms) {
  for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < pieces; j += gridDim.x * blockDim.x) {
    const uint32_t p = by_row[j];
    terms[j] = lkey[p] == nseg << kDirectKeyBits ? pstart[p + 1] - pstart[p] : 1u;
  }
}

// cofs[p] = the piece's first combine term; cmb_rp[v] = row v's first term.
__global__ void combine_rows_kernel(const uint32_t *__restrict__ by_row, const uint32_t *__restrict__ row_sorted,
                                    const uint32_t *__restrict__ term_scan, uint32_t pieces, uint32_t n,
                                    uint32_t *__restrict__ cofs, uint32_t *__restrict__ cmb_rp) {
  const uint32_t stride = gridDim.x * blockDim.x, t = blockIdx.x * blockDim.x + threadIdx.x;
  for (uint32_t j = t; j < pieces; j += stride) cofs[by_row[j]] = term_scan[j];
  for (size_t v = t; v <= n; v += stride)
    cmb_rp[v] = term_scan[first_ge(pieces, (uint32_t)v, [&](uint32_t i) { return row_sorted[i]; })];
}

__device__ __forceinline__ uint32_t tier_of(uint32_t terms) {
  return terms > kCmbBig ? 3u : (terms > kCmbMid ? 2u : (terms > kCmbLight ? 1u : 0u));
}

__global__ void tier_kernel(const uint32_t *__restrict__ cmb_rp, uint32_t n, uint32_t *__restrict__ tier) {
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x)
    tier[v] = tier_of(cmb_rp[v + 1] - cmb_rp[v]);
}

// out[g] = first position of key g in the sorted keys, g < count.
__global__ void group_start_kernel(const uint32_t *__restrict__ sorted, uint32_t items, uint32_t count,
                                   uint32_t *__restrict__ out) {
  for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < count; g += gridDim.x * blockDim.x)
    out[g] = first_ge(items, g, [&](uint32_t i) { return sorted[i]; });
}

// The j-th piece in layout order: its partial or direct terms go to the
// combine list, epos[p] = its first entry's position (~0: direct).
template <class V>
__global__ void piece_place_kernel(const uint32_t *__restrict__ by_key, const uint32_t *__restrict__ key_sorted,
                                   const uint32_t *__restrict__ gstart, const uint32_t *__restrict__ gtask,
                                   const uint32_t *__restrict__ gpart, const uint32_t *__restrict__ pstart,
                                   const uint32_t *__restrict__ cofs, const uint32_t *__restrict__ key,
                                   const V *__restrict__ val, const uint32_t *__restrict__ eid, uint32_t pieces,
                                   uint32_t nseg, uint32_t *__restrict__ cmb_pos, uint32_t *__restrict__ wcmb_eid,
                                   size_t *__restrict__ epos) {
  for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < pieces; j += gridDim.x * blockDim.x) {
    const uint32_t p = by_key[j], g = key_sorted[j], c = cofs[p];
    if (g == nseg << kDirectKeyBits) {
      const uint32_t a = pstart[p], len = pstart[p + 1] - a;
      for (uint32_t e = 0; e < len; ++e) {
        cmb_pos[c + e] = key[a + e];
        if (wcmb_eid) wcmb_eid[c + e] = eid[slot_of(val, a + e)];
      }
      epos[p] = ~(size_t)0;
    } else {
      const uint32_t r = j - gstart[g], cls = g & ((1u << kDirectKeyBits) - 1);
      cmb_pos[c] = kIsPartial | (gpart[g] + r);
      if (wcmb_eid) wcmb_eid[c] = kEidOne;
      epos[p] = (size_t)gtask[g] * kTask + (r << cls);
    }
  }
}

// Every entry of a staged piece into its place.
template <class V>
__global__ void entry_place_kernel(const uint32_t *__restrict__ key, const V *__restrict__ val,
                                   const uint32_t *__restrict__ scan, uint32_t m, const uint32_t *__restrict__ pstart,
                                   const size_t *__restrict__ epos, const uint32_t *__restrict__ eid,
                                   uint16_t *__restrict__ lidx, uint32_t *__restrict__ went_eid) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (size_t)gridDim.x * blockDim.x) {
    const uint32_t p = scan[i + 1] - 1;
    const size_t ep = epos[p];
    if (ep == ~(size_t)0) continue;
    const size_t pos = ep + ((uint32_t)i - pstart[p]);
    lidx[pos] = (uint16_t)(key[i] & (kSegSize - 1));
    if (went_eid) went_eid[pos / kTask * kTask + wpos((uint32_t)(pos % kTask))] = eid[slot_of(val, (uint32_t)i)];
  }
}

// Descriptors of the tasks of every (segment, class) group; one workgroup a
// group.
__global__ void task_desc_kernel(const uint32_t *__restrict__ gtask, const uint32_t *__restrict__ gpart,
                                 uint2 *__restrict__ desc) {
  const uint32_t g = blockIdx.x, cls = g & ((1u << kDirectKeyBits) - 1);
  const uint32_t a = gtask[g], b = gtask[g + 1];
  for (uint32_t t = a + threadIdx.x; t < b; t += blockDim.x) desc[t] = make_uint2(cls, gpart[g] + (t - a) * (kTask >> cls));
}

// Time of a task by class and of a segment's slice, in 1/16 of a middling
// task, fitted to per-workgroup clocks of RMAT-20 passes.
constexpr uint32_t kSliceCost = 800;
inline uint32_t task_cost(uint32_t g) {
  constexpr uint32_t kCost[1u << kDirectKeyBits] = {22, 17, 16, 16, 16, 16, 16, 18, 18, 18};
  return kCost[g & ((1u << kDirectKeyBits) - 1)];
}

// Device memory in one block, cut into 256-byte aligned arrays.
struct Arena {
  size_t size = 0;
  size_t take(size_t bytes) {
    const size_t at = size;
    size += (bytes + 255) / 256 * 256;
    return at;
  }
};

int to_host(void *h, const void *d, size_t bytes) {
  OLV_HIP(hipMemcpyAsync(h, d, bytes, hipMemcpyDeviceToHost, stream()));
  OLV_HIP(hipStreamSynchronize(stream()));
  return OLV_OK;
}

// Rows by tier (bp.cmb_rp built): the mid, big and huge rows, each ascending,
// into `rows` (n words at least); counts to the host.
int list_tiers(BlockedPlan &bp, uint32_t *rows) {
  ScratchBuf tier, start;
  OLV_TRY(tier.alloc((size_t)bp.n * 4));
  OLV_TRY(start.alloc(5 * 4));
  hipLaunchKernelGGL(tier_kernel, dim3(pgrid(bp.n)), dim3(256), 0, stream(), bp.cmb_rp, bp.n, tier.as<uint32_t>());
  SortBufs b;
  OLV_TRY(radix_sort<uint32_t>(tier.as<uint32_t>(), LoadIndex{}, bp.n, 2, b));
  hipLaunchKernelGGL(group_start_kernel, dim3(1), dim3(64), 0, stream(), b.keys(), bp.n, 5u, start.as<uint32_t>());
  OLV_HIP(hipGetLastError());
  uint32_t h[5];
  OLV_TRY(to_host(h, start.p, sizeof(h)));
  bp.n_mid = h[2] - h[1];
  bp.n_big = h[3] - h[2];
  bp.n_huge = h[4] - h[3];
  if (h[4] > h[1])
    OLV_HIP(hipMemcpyAsync(rows, b.vals<uint32_t>() + h[1], (size_t)(h[4] - h[1]) * 4, hipMemcpyDeviceToDevice, stream()));
  bp.cmb_rows = rows;
  return OLV_OK;
}

// No segment pass: the rows' entries are the combine's terms.
int build_solo(const uint32_t *rp, const uint32_t *col, const uint32_t *eid, BlockedPlan &bp) {
  const uint32_t n = bp.n, m = bp.m;
  Arena ar;
  const size_t o_rp = ar.take(((size_t)n + 1) * 4), o_pos = ar.take((size_t)m * 4),
               o_rows = ar.take((size_t)n * 4), o_w = ar.take(eid ? (size_t)m * 4 : 0);
  OLV_HIP(hipMalloc(&bp.mem, std::max<size_t>(ar.size, 256)));
  char *base = static_cast<char *>(bp.mem);
  bp.cmb_rp = reinterpret_cast<uint32_t *>(base + o_rp);
  bp.cmb_pos = reinterpret_cast<uint32_t *>(base + o_pos);
  OLV_HIP(hipMemcpyAsync(bp.cmb_rp, rp, ((size_t)n + 1) * 4, hipMemcpyDeviceToDevice, stream()));
  if (m) OLV_HIP(hipMemcpyAsync(bp.cmb_pos, col, (size_t)m * 4, hipMemcpyDeviceToDevice, stream()));
  if (eid) {
    bp.weid = reinterpret_cast<uint32_t *>(base + o_w);
    if (m) OLV_HIP(hipMemcpyAsync(bp.weid, eid, (size_t)m * 4, hipMemcpyDeviceToDevice, stream()));
  }
  bp.ncmb = m;
  bp.nweights = eid ? m : 0;
  return list_tiers(bp, reinterpret_cast<uint32_t *>(base + o_rows));
}

template <class V>
int build_segmented(const uint32_t *rp, const uint32_t *col, const uint32_t *eid, uint32_t groups, BlockedPlan &bp) {
  const uint32_t n = bp.n, m = bp.m;
  const uint32_t nseg = ((n - 1) >> kSegBits) + 1;
  hipStream_t s = stream();
  // 1. entries by segment, rows ascending inside
  SortBufs ent;
  {
    ScratchBuf erow;
    OLV_TRY(erow.alloc((size_t)m * 4));
    OLV_TRY(slot_rows(rp, n, m, erow.as<uint32_t>()));
    if constexpr (sizeof(V) == 8) OLV_TRY((radix_sort<V>(col, LoadAndIndex{erow.as<uint32_t>()}, m, bits_for(nseg), ent, kSegBits)));
    else OLV_TRY((radix_sort<V>(col, LoadArr{erow.as<uint32_t>()}, m, bits_for(nseg), ent, kSegBits)));
  }
  const uint32_t *key = ent.keys();
  const V *val = ent.vals<V>();
  // 2. pieces
  ScratchBuf scan, stat;
  OLV_TRY(scan.alloc(((size_t)m + 1) * 4));
  OLV_TRY(stat.alloc(((size_t)nseg + 2) * 4));
  {
    ScratchBuf flag, gstart;
    OLV_TRY(flag.alloc((size_t)m * 4));
    OLV_TRY(gstart.alloc(((size_t)m + 1) * 4));
    hipLaunchKernelGGL(piece_head_kernel<V>, dim3(pgrid(m)), dim3(256), 0, s, key, val, m, flag.as<uint32_t>());
    OLV_TRY(exclusive_scan(flag.as<uint32_t>(), scan.as<uint32_t>(), m));
    hipLaunchKernelGGL(piece_start_kernel, dim3(pgrid(m)), dim3(256), 0, s, scan.as<uint32_t>(), m,
                       gstart.as<uint32_t>());
    hipLaunchKernelGGL(piece_cut_kernel, dim3(pgrid(m)), dim3(256), 0, s, gstart.as<uint32_t>(),
                       scan.as<uint32_t>() + m, flag.as<uint32_t>());
    OLV_TRY(exclusive_scan(flag.as<uint32_t>(), scan.as<uint32_t>(), m));
  }
  hipLaunchKernelGGL(seg_stat_kernel, dim3(pgrid(nseg)), dim3(256), 0, s, key, scan.as<uint32_t>(), m, rp, n, nseg,
                     stat.as<uint32_t>());
  OLV_HIP(hipGetLastError());
  std::vector<uint32_t> h_stat((size_t)nseg + 2);
  OLV_TRY(to_host(h_stat.data(), stat.p, h_stat.size() * 4));
  const uint32_t pieces = h_stat[0];
  bp.n_live = h_stat[1];
  // 3. the combine's term lists: pieces by row
  ScratchBuf pbuf;
  Arena pa;
  const size_t pw = ((size_t)pieces + 1) * 4;
  const size_t o_start = pa.take(pw), o_row = pa.take(pw), o_key = pa.take(pw), o_terms = pa.take(pw),
               o_cofs = pa.take(pw), o_epos = pa.take(2 * pw);
  OLV_TRY(pbuf.alloc(pa.size));
  auto parr = [&](size_t o) { return reinterpret_cast<uint32_t *>(pbuf.as<char>() + o); };
  uint32_t *pstart = parr(o_start), *prow = parr(o_row), *lkey = parr(o_key), *terms = parr(o_terms),
           *cofs = parr(o_cofs);
  size_t *epos = reinterpret_cast<size_t *>(parr(o_epos));
  hipLaunchKernelGGL(piece_start_kernel, dim3(pgrid(m)), dim3(256), 0, s, scan.as<uint32_t>(), m, pstart);
  hipLaunchKernelGGL(piece_row_kernel<V>, dim3(pgrid(pieces)), dim3(256), 0, s, val, pstart, pieces, prow);
  hipLaunchKernelGGL(piece_key_kernel, dim3(pgrid(pieces)), dim3(256), 0, s, key, pstart, pieces,
                     stat.as<uint32_t>() + 2, nseg, lkey);
  OLV_HIP(hipGetLastError());
  ScratchBuf crp;
  OLV_TRY(crp.alloc(((size_t)n + 1) * 4));
  {
    SortBufs by;
    OLV_TRY(radix_sort<uint32_t>(prow, LoadIndex{}, pieces, bits_for(n), by));
    hipLaunchKernelGGL(piece_terms_kernel, dim3(pgrid(pieces)), dim3(256), 0, s, by.vals<uint32_t>(), pstart, lkey,
                       pieces, nseg, terms);
    OLV_TRY(exclusive_scan(terms, terms, pieces));
    hipLaunchKernelGGL(combine_rows_kernel, dim3(pgrid(std::max(n, pieces))), dim3(256), 0, s, by.vals<uint32_t>(),
                       by.keys(), terms, pieces, n, cofs, crp.as<uint32_t>());
    OLV_HIP(hipGetLastError());
  }
  // 4. the segment pass's layout: pieces by (segment, class)
  const uint32_t ngr = nseg << kDirectKeyBits;  // groups; key ngr: direct pieces
  SortBufs by;
  OLV_TRY(radix_sort<uint32_t>(lkey, LoadIndex{}, pieces, bits_for(ngr + 1), by));
  ScratchBuf gbuf;  // gstart (ngr + 2, the last the terms in all), gtask (ngr + 1), gpart (ngr + 1)
  OLV_TRY(gbuf.alloc(((size_t)ngr * 3 + 4) * 4));
  uint32_t *gstart = gbuf.as<uint32_t>(), *gtask = gstart + ngr + 2, *gpart = gtask + ngr + 1;
  hipLaunchKernelGGL(group_start_kernel, dim3(pgrid(ngr + 1)), dim3(256), 0, s, by.keys(), pieces, ngr + 1, gstart);
  OLV_HIP(hipGetLastError());
  OLV_HIP(hipMemcpyAsync(gstart + ngr + 1, terms + pieces, 4, hipMemcpyDeviceToDevice, s));
  std::vector<uint32_t> hg((size_t)ngr + 2), ht((size_t)ngr * 2 + 2);
  OLV_TRY(to_host(hg.data(), gstart, hg.size() * 4));
  bp.ncmb = hg[ngr + 1];
  uint64_t task = 0, part = 0;
  for (uint32_t g = 0; g < ngr; ++g) {
    const uint32_t cls = g & ((1u << kDirectKeyBits) - 1);
    if (cls == 0) part = (part + kTask - 1) / kTask * kTask;  // 16-byte stores in the first classes
    ht[g] = (uint32_t)task;
    ht[ngr + 1 + g] = (uint32_t)part;
    if (cls >= kClasses) continue;
    const uint64_t ppt = kTask >> cls, nt = (hg[g + 1] - hg[g] + ppt - 1) / ppt;
    task += nt;
    part += nt * ppt;
  }
  ht[ngr] = (uint32_t)task;
  ht[2 * (size_t)ngr + 1] = (uint32_t)part;
  if (part >= kIsPartial) return build_solo(rp, col, eid, bp);  // beyond a term's 31 bits
  bp.ntasks = (uint32_t)task;
  bp.nparts = (uint32_t)part;
  // Tasks to workgroups: consecutive runs of about equal cost, a task
  // task_cost (classes of short pieces store more) and a segment's slice
  // kSliceCost (its 128 KB load between two barriers, and the ring's restart).
  std::vector<uint4> first, items;
  {
    uint64_t total = 0;
    for (uint32_t g = 0; g < ngr; ++g) total += (uint64_t)(ht[g + 1] - ht[g]) * task_cost(g);
    for (uint32_t g = 0; g < nseg; ++g)
      total += ht[(g + 1) << kDirectKeyBits] > ht[g << kDirectKeyBits] ? kSliceCost : 0;
    uint64_t share = std::max<uint64_t>((total + (uint64_t)kSliceCost * groups + groups - 1) / groups,
                                        kSliceCost + kBlkWaves * task_cost(kClasses - 1));
    for (;; share += share / 64 + 1) {  // until no more than `groups` workgroups come out
      first.clear();
      items.clear();
      uint64_t room = 0;                // what the current workgroup may still take
      uint32_t cur = 0xffffffffu;       // its current item's segment
      for (uint32_t g = 0; g < ngr; ++g) {
        const uint32_t sg = g >> kDirectKeyBits, c = task_cost(g);
        for (uint32_t t = ht[g]; t < ht[g + 1];) {
          if (first.empty() || room < (cur == sg ? 0u : kSliceCost) + kBlkWaves * c / 2 ||
              (first.back().w & 0xfffu) == 0xfffu) {
            first.push_back(make_uint4(0, 0, 0, (uint32_t)items.size() << 12));
            room = share;
            cur = 0xffffffffu;
          }
          uint4 &f = first.back();
          const bool add = cur != sg;
          if (add) {
            room -= kSliceCost;
            cur = sg;
            if (f.w & 0xfffu) items.push_back(make_uint4(sg, t, t, 0));
            else f = make_uint4(sg, t, t, f.w);
            ++f.w;
          }
          const uint32_t take = (uint32_t)std::min<uint64_t>(ht[g + 1] - t, std::max<uint64_t>(1, room / c));
          t += take;
          ((f.w & 0xfffu) == 1 ? f : items.back()).z = t;
          room -= std::min<uint64_t>(room, (uint64_t)take * c);
        }
      }
      if (first.size() <= groups || nseg > (uint64_t)groups * 4000) break;
    }
    // Workgroup b runs on XCD b % kXcds: neighbours in the list, which share a
    // slice, go to one XCD and load it through one L2.
    constexpr size_t kXcds = 8;
    const size_t per = (first.size() + kXcds - 1) / kXcds;
    std::vector<uint4> order(per * kXcds, make_uint4(0, 0, 0, 0));
    for (size_t b = 0; b < order.size(); ++b) {
      const size_t l = b % kXcds * per + b / kXcds;
      if (l < first.size()) order[b] = first[l];
    }
    first.swap(order);
    if (items.size() >= (1u << 20)) return fail(OLV_ERANGE, "pull plan: %zu segment items", items.size());
  }
  bp.ngroups = (uint32_t)first.size();  // (some may have no items)
  // 5. the plan's arrays
  Arena ar;
  const size_t o_first = ar.take(first.size() * sizeof(uint4)), o_items = ar.take((items.size() + 1) * sizeof(uint4)),
               o_desc = ar.take((size_t)task * sizeof(uint2)), o_lidx = ar.take((size_t)task * kTask * 2),
               o_rp = ar.take(((size_t)n + 1) * 4), o_pos = ar.take((size_t)bp.ncmb * 4),
               o_rows = ar.take((size_t)n * 4), o_part = ar.take((size_t)part * 4),
               o_w = ar.take(eid ? ((size_t)task * kTask + bp.ncmb) * 4 : 0);
  OLV_HIP(hipMalloc(&bp.mem, std::max<size_t>(ar.size, 256)));
  char *base = static_cast<char *>(bp.mem);
  bp.wg_first = reinterpret_cast<uint4 *>(base + o_first);
  bp.wg_items = reinterpret_cast<uint4 *>(base + o_items);
  bp.desc = reinterpret_cast<uint2 *>(base + o_desc);
  bp.lidx = reinterpret_cast<uint16_t *>(base + o_lidx);
  bp.cmb_rp = reinterpret_cast<uint32_t *>(base + o_rp);
  bp.cmb_pos = reinterpret_cast<uint32_t *>(base + o_pos);
  bp.partial = reinterpret_cast<float *>(base + o_part);
  if (eid) {
    bp.weid = reinterpret_cast<uint32_t *>(base + o_w);
    bp.nweights = (size_t)task * kTask + bp.ncmb;
  }
  OLV_HIP(hipMemcpyAsync(gtask, ht.data(), ht.size() * 4, hipMemcpyHostToDevice, s));
  if (!first.empty())
    OLV_HIP(hipMemcpyAsync(bp.wg_first, first.data(), first.size() * sizeof(uint4), hipMemcpyHostToDevice, s));
  if (!items.empty())
    OLV_HIP(hipMemcpyAsync(bp.wg_items, items.data(), items.size() * sizeof(uint4), hipMemcpyHostToDevice, s));
  OLV_HIP(hipMemcpyAsync(bp.cmb_rp, crp.p, ((size_t)n + 1) * 4, hipMemcpyDeviceToDevice, s));
  OLV_TRY(fill_u32(reinterpret_cast<uint32_t *>(bp.lidx), kSegSize | kSegSize << 16, (size_t)task * kTask / 2));
  if (eid) OLV_TRY(fill_u32(bp.weid, kEidZero, (size_t)task * kTask));
  hipLaunchKernelGGL(task_desc_kernel, dim3(ngr), dim3(256), 0, s, gtask, gpart, bp.desc);
  uint32_t *wcmb_eid = eid ? bp.weid + (size_t)task * kTask : nullptr;
  hipLaunchKernelGGL(piece_place_kernel<V>, dim3(pgrid(pieces)), dim3(256), 0, s, by.vals<uint32_t>(), by.keys(),
                     gstart, gtask, gpart, pstart, cofs, key, val, eid, pieces, nseg, bp.cmb_pos, wcmb_eid, epos);
  hipLaunchKernelGGL(entry_place_kernel<V>, dim3(pgrid(m)), dim3(256), 0, s, key, val, scan.as<uint32_t>(), m, pstart,
                     epos, eid, bp.lidx, bp.weid);
  OLV_HIP(hipGetLastError());
  OLV_TRY(list_tiers(bp, reinterpret_cast<uint32_t *>(base + o_rows)));
  OLV_HIP(hipStreamSynchronize(s));  // the uploads read this function's vectors
  return OLV_OK;
}

}  // namespace

int build_blocked_plan(const uint32_t *rp, const uint32_t *col, const uint32_t *eid, uint32_t n, uint32_t m,
                       uint32_t max_row, uint32_t groups, BlockedPlan &bp) {
  bp.release();
  if (n == 0 || n >= kIsPartial) return fail(OLV_ERANGE, "pull plan: %u vertices", n);
  bp.n = n;
  bp.m = m;
  int rc = OLV_OK;
  if (m < kPassMinEntries && max_row <= kDirectRowMax) {
    ScratchBuf w;
    rc = w.alloc(4);
    if (rc == OLV_OK) {
      hipLaunchKernelGGL(live_rows_kernel, dim3(1), dim3(1), 0, stream(), rp, n, m, w.as<uint32_t>());
      rc = to_host(&bp.n_live, w.p, 4);
    }
    if (rc == OLV_OK) rc = build_solo(rp, col, eid, bp);
  } else if (eid) {
    rc = build_segmented<uint2>(rp, col, eid, std::max(1u, groups), bp);
  } else {
    rc = build_segmented<uint32_t>(rp, col, eid, std::max(1u, groups), bp);
  }
  if (rc != OLV_OK) {
    bp.release();
    return rc;
  }
  bp.ready = true;
  return OLV_OK;
}

}  // namespace olv
