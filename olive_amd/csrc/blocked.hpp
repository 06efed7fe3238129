// Source-segmented pull for the PageRank iteration (CSR segmenting: Zhang,
// Kiriansky, Mendis, Amarasinghe, Zaharia, Matei, "Making Caches Work for
// Graph Analytics", IEEE BigData 2017, restated for a GPU with a 160 KB LDS
// per CU).
//
// The iterate's source vector is cut into segments of kSegSize consecutive
// vertices (128 KB of fp32, one LDS slice).  The in-edges of every
// destination are grouped by the segment of their source into "pieces"
// (destination, segment) of at most kPieceMax entries.  One iteration is two
// launches:
//
//   segment pass  sums every piece from the staged slice and stores one
//                 partial per piece;
//   combine       adds, per destination, its terms -- partials, in segment
//                 order -- and applies the vertex update.
//
// A term may also be a single source, read straight from the vector.  That
// gather is random, so it costs about 2.4 partials (180 against 420 G/s on a
// uniform graph: the partials of neighbouring rows are neighbours), and it is
// used only where the pass does not pay: for the entries of a segment too
// small to be worth a slice (kSegMinEntries), and for a whole CSR of few
// edges (kPassMinEntries), which then takes one launch per iteration.
//
// Layout of the segment pass.  A piece of c entries is padded to a capacity
// of 1, 2, 4, ..., 512 entries (its class) with the slice's zero slot, and the
// pieces of one (segment, class) are stored back to back, so a task -- 512
// consecutive 16-bit entries, 1 KB -- holds 512 pieces of class 0 down to one
// piece of class 9 and every lane of a wave reads its 8 entries with one
// 16-byte load.  A lane holds 8 pieces (class 0), 4, 2, one (class 3), or a
// 2^i-th of one (the group's sum is taken with DPP moves).  All tasks have the
// same shape, so a wave streams its tasks through a ring of registers kBlkRing
// deep with no LDS staging and no barrier inside a segment; weighted passes
// read 8 fp32 weights per lane beside the entries.
//
// Pieces of more than kPieceMax entries are cut, and so is the tail of one
// that would fill at most 3/4 of its capacity (from kCutCap on), at half the
// capacity: RMAT-20's padding falls from 27 to 10 % for 5 % more partials.
//
// What bounds it (RMAT-20, 16.8 M edges, 1.83 M partials): plain, the segment
// pass takes 14.0 us -- 4 us until the workgroups' first slices are in LDS,
// then 6-7 us of LDS gathers over 37 MB of entries, the rest launch and
// imbalance -- and the combine 9.7 us, 4 of them its launch and the others
// its gathered partials; 24.5 us per iteration against 32.4 when every unit
// of entries was staged in LDS with 16K-source slices.  Weighted, the pass
// reads 118 MB in 22.5 us (28 before), 5.2 TB/s: the rate of the caches behind L2.
//
// A piece's terms are summed in a fixed order and the terms of a row in
// segment order, so an iteration is bit-reproducible from run to run.
#pragma once
#include <type_traits>

#include "device.hpp"
#include "internal.hpp"
#include "seg_core.hpp"

namespace olv {

constexpr uint32_t kSegBits = 15;
constexpr uint32_t kSegSize = 1u << kSegBits;  // sources per LDS slice (128 KB of fp32), plus a zero slot
static_assert(kSegSize <= 0xffff, "entries hold a slice offset or the zero slot in 16 bits");
constexpr int kBlkThreads = 1024;              // segment-pass workgroup (one per CU: 128 KB of LDS)
constexpr uint32_t kBlkWaves = kBlkThreads / kWave;
constexpr uint32_t kClasses = 10;              // class c: pieces of up to 1 << c entries
constexpr uint32_t kPieceMax = 1u << (kClasses - 1);
constexpr uint32_t kCutCap = 32;               // capacities cut in two when at most 3/4 full
constexpr uint32_t kTask = 512;                // entries of a task: 64 lanes x 8
static_assert(kPieceMax == kTask, "the longest piece fills one task");
// Tasks in flight per wave (1 KB each, weighted 3 KB): 64 and 96 KB per CU
// cover the latency of the stream; a deeper weighted ring spills registers
// (4 tasks: 41 against 22 us per RMAT-20 pass).
template <bool kW>
constexpr int kBlkRing = kW ? 2 : 4;
constexpr uint32_t kSegMinEntries = 2048;      // entries of a staged segment, at least
// Edges of a CSR with a segment pass, at least: one launch of m random gathers
// against two launches.  20 iterations, one launch / two (us), uniform edges at
// 6, 16, 32 a vertex, then RMAT: 500K edges 197/232, 197/220, 180/218 and
// 200/231, 220/228, 215/227; 850K 228/247, 231/228, 192/228 and 219/238,
// 242/228, 251/240; 1.2M 268/279, 252/242, 214/241 and 256/256, 267/243,
// 268/242.  Weighted solves cross at the same sizes.
constexpr uint32_t kPassMinEntries = 700000;
constexpr uint32_t kDirectRowMax = 16384;      // without a segment pass: entries per row, at most
constexpr uint32_t kIsPartial = 0x80000000u;   // combine term: a partial's index, else a source
constexpr uint32_t kEidZero = 0xffffffffu;     // weight source of a padding entry: 0
constexpr uint32_t kEidOne = 0xfffffffeu;      // weight source of a partial in the combine: 1
constexpr uint32_t kCmbLight = 16;             // terms of a row combined by one lane, at most
constexpr uint32_t kCmbMid = 128;              // by kCmbMidLanes lanes, at most
constexpr uint32_t kCmbMidLanes = 8;
constexpr uint32_t kCmbBig = 1024;             // by a wave, at most; a workgroup beyond
constexpr uint32_t kCmbPer = 16;               // terms in flight per lane

// Device arrays of a segmented pull over one CSR (one allocation).
struct BlockedPlan {
  uint32_t n = 0, m = 0, n_live = 0;         // vertices, entries, rows up to the last one with entries
  uint32_t n_mid = 0, n_big = 0, n_huge = 0; // rows with more than kCmbLight / kCmbMid / kCmbBig terms
  uint32_t ntasks = 0, ngroups = 0;          // tasks, segment-pass workgroups (0: no segment pass)
  uint32_t nparts = 0, ncmb = 0;             // partials (with class padding), combine terms
  size_t nweights = 0;                       // weighted: ntasks * kTask + ncmb
  void *mem = nullptr;
  uint4 *wg_first = nullptr;     // ngroups: each workgroup's first item (segment, first task, end task,
                                 // items | index of its second item in wg_items << 12)
  uint4 *wg_items = nullptr;     // the workgroups' further items (segment, first task, end task, -)
  uint2 *desc = nullptr;         // ntasks: class, first partial
  uint16_t *lidx = nullptr;      // ntasks * kTask: source offset in the segment (kSegSize: padding)
  uint32_t *cmb_rp = nullptr;    // n + 1: each row's range in cmb_pos
  uint32_t *cmb_pos = nullptr;   // ncmb: kIsPartial | partial, or a source; by row, in segment order
  uint32_t *cmb_rows = nullptr;  // rows of the mid, big and huge tiers, each ascending
  float *partial = nullptr;      // nparts
  // weighted plans: where the weight of every entry (in the order the segment
  // pass reads them, see wpos) and then of every combine term comes from: an
  // edge id, kEidZero or kEidOne
  uint32_t *weid = nullptr;      // nweights
  bool ready = false;
  void release() {
    if (mem) (void)hipFree(mem);
    *this = BlockedPlan();
  }
};

// Builds the plan on the device for the CSR rp (n + 1), col (m, source ids
// < n).  eid (not null: a weighted plan): the edge id of every slot.
// max_row: the longest row.  groups: workgroups of the segment pass.
int build_blocked_plan(const uint32_t *rp, const uint32_t *col, const uint32_t *eid, uint32_t n, uint32_t m,
                       uint32_t max_row, uint32_t groups, BlockedPlan &bp);

struct BlkDev {
  const uint4 *wg_first;
  const uint4 *wg_items;
  const uint2 *desc;
  const uint16_t *lidx;
  const uint32_t *cmb_rp;
  const uint32_t *cmb_pos;
  const uint32_t *cmb_mid, *cmb_big, *cmb_huge;
  float *partial;
  const float *went;  // weights of the entries, kTask per task (weighted passes)
  const float *wcmb;  // weights of the combine terms
  uint32_t n, n_live, n_mid, n_big, n_huge;
};

inline BlkDev make_blk_dev(const BlockedPlan &p, const float *weights = nullptr) {
  BlkDev d;
  d.wg_first = p.wg_first;
  d.wg_items = p.wg_items;
  d.desc = p.desc;
  d.lidx = p.lidx;
  d.cmb_rp = p.cmb_rp;
  d.cmb_pos = p.cmb_pos;
  d.cmb_mid = p.cmb_rows;
  d.cmb_big = p.cmb_rows + p.n_mid;
  d.cmb_huge = p.cmb_rows + p.n_mid + p.n_big;
  d.partial = p.partial;
  d.went = weights;
  d.wcmb = weights ? weights + (size_t)p.ntasks * kTask : nullptr;
  d.n = p.n;
  d.n_live = p.n_live;
  d.n_mid = p.n_mid;
  d.n_big = p.n_big;
  d.n_huge = p.n_huge;
  return d;
}

// Where the weight of entry x of a task sits among the task's kTask weights:
// lane x / 8 reads its 8 weights with two 16-byte loads, each contiguous over
// the wave.
__host__ __device__ __forceinline__ uint32_t wpos(uint32_t x) {
  return ((x >> 2) & 1u) * (kTask / 2) + (x >> 3) * 4 + (x & 3u);
}

// DPP move of x (rows of 16 lanes outside RowMask receive 0)
template <int Ctrl, int RowMask = 0xf>
__device__ __forceinline__ float blk_dpp(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), Ctrl, RowMask, 0xf, false));
}

// Sum over aligned groups of G lanes with DPP moves (no LDS round trip):
// inside rows of 16 lanes every lane of the group ends with the sum; 32
// lanes add the lower row's sum into the upper row (row_bcast:15), so there
// the upper row holds it; for the whole wave the four row sums are read by
// lane and every lane holds the sum.  Lane G - 1 of a group always does.
template <int G>
__device__ __forceinline__ float blk_group_sum(float v) {
  static_assert(G == 1 || G == 2 || G == 4 || G == 8 || G == 16 || G == 32 || G == kWave, "group of 2^i lanes");
  if constexpr (G == 1) return v;
  v += blk_dpp<0xb1>(v);                          // quad_perm [1,0,3,2]: lane ^ 1
  if constexpr (G >= 4) v += blk_dpp<0x4e>(v);    // quad_perm [2,3,0,1]: lane ^ 2
  if constexpr (G >= 8) v += blk_dpp<0x141>(v);   // row_half_mirror: lane 7 - i of 8
  if constexpr (G >= 16) v += blk_dpp<0x140>(v);  // row_mirror: lane 15 - i of 16
  if constexpr (G == 32) v += blk_dpp<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  if constexpr (G == kWave) {
    const float r0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 15));
    const float r1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 31));
    const float r2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 47));
    const float r3 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
    v = (r0 + r1) + (r2 + r3);
  }
  return v;
}

// One task: the 8 terms of this lane, summed by class into partials from
// `part` on.
__device__ __forceinline__ void blk_task(uint32_t cls, float *__restrict__ part, const float *v) {
  const uint32_t lane = lane_id();
  const float a0 = v[0] + v[1], a1 = v[2] + v[3], a2 = v[4] + v[5], a3 = v[6] + v[7];
  if (cls == 1) {
    reinterpret_cast<float4 *>(part)[lane] = make_float4(a0, a1, a2, a3);
    return;
  }
  if (cls == 0) {
    float4 *p = reinterpret_cast<float4 *>(part) + 2 * lane;
    p[0] = make_float4(v[0], v[1], v[2], v[3]);
    p[1] = make_float4(v[4], v[5], v[6], v[7]);
    return;
  }
  if (cls == 2) {
    reinterpret_cast<float2 *>(part)[lane] = make_float2(a0 + a1, a2 + a3);
    return;
  }
  const float s = (a0 + a1) + (a2 + a3);
  auto store = [&](float x, uint32_t lg) {  // groups of 2^lg lanes; the last one stores
    const uint32_t g = (1u << lg) - 1;
    if ((lane & g) == g) part[lane >> lg] = x;
  };
  switch (cls) {
    case 3: part[lane] = s; break;
    case 4: store(blk_group_sum<2>(s), 1); break;
    case 5: store(blk_group_sum<4>(s), 2); break;
    case 6: store(blk_group_sum<8>(s), 3); break;
    case 7: store(blk_group_sum<16>(s), 4); break;
    case 8: store(blk_group_sum<32>(s), 5); break;
    default: store(blk_group_sum<kWave>(s), 6); break;
  }
}

// Segment pass of iteration k over `src`.  It first applies the stop rule of
// the iteration loop: returns at once when done; workgroup 0 alone sets done
// when iteration k - 1 left an L1 residual below eps (the other workgroups'
// partials of that pass are then unused: the combine launch returns on done)
// and clears the residual slots of iteration k + 1.
// kW: every entry's value is multiplied by its weight (d.went).
template <bool kW>
__global__ void __launch_bounds__(kBlkThreads) blk_segment_kernel(BlkDev d, const float *__restrict__ src,
                                                                   IterCtl *ctl, uint32_t k) {
  __shared__ __align__(16) float slice[kSegSize + 4];  // slice[kSegSize] is the zero slot of the padding entries
  constexpr int R = kBlkRing<kW>;
  const uint32_t tid = threadIdx.x, lane = lane_id();
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  uint4 item = d.wg_first[blockIdx.x];  // in flight during the checks
  if (__hip_atomic_load(&ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  if (blockIdx.x == 0) {
    if (k > 0) {
      const double res = err_total(ctl, (k - 1) % 3);
      if (res < ctl->eps) {
        if (threadIdx.x == 0) {
          ctl->iters = k;
          ctl->residual = res;
          __hip_atomic_store(&ctl->done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return;
      }
    }
    double *z = &ctl->errs[(k + 1) % 3][0].v;
    for (uint32_t i = threadIdx.x; i < kErrSlots * (sizeof(ErrSlot) / sizeof(double)); i += kBlkThreads) z[i] = 0.0;
  }
  const uint32_t nitems = __builtin_amdgcn_readfirstlane(item.w & 0xfffu);
  const uint32_t inext = __builtin_amdgcn_readfirstlane(item.w >> 12);
  if (tid == 0) slice[kSegSize] = 0.f;  // read after the first barrier
  constexpr uint32_t kSl = kSegSize / (4 * kBlkThreads);
  for (uint32_t it = 0; it < nitems; ++it) {
    if (it) {
      item = d.wg_items[inext + it - 1];
      __syncthreads();  // the previous segment's sums are done with the slice
    }
    const uint32_t seg = __builtin_amdgcn_readfirstlane(item.x);
    const uint32_t t0 = __builtin_amdgcn_readfirstlane(item.y) + wave;
    const uint32_t t1 = __builtin_amdgcn_readfirstlane(item.z);
    // this wave's tasks: t0, t0 + kBlkWaves, ...; lane i holds the
    // descriptor of the i-th of up to 64 of them
    uint32_t nt = t0 < t1 ? (t1 - t0 + kBlkWaves - 1) / kBlkWaves : 0u;
    uint4 e[R];
    float4 wa[kW ? R : 1], wb[kW ? R : 1];
    auto load = [&](int j, uint32_t t) {
      e[j] = reinterpret_cast<const uint4 *>(d.lidx + (size_t)t * kTask)[lane];
      if constexpr (kW) {
        const float4 *w = reinterpret_cast<const float4 *>(d.went + (size_t)t * kTask);
        wa[j] = w[lane];
        wb[j] = w[kWave + lane];
      }
    };
    float4 sl[kSl];  // the slice first: the ring's loads then stay in flight behind it
    const uint32_t base = seg << kSegBits, cnt = d.n - base;
    if (cnt >= kSegSize) {
#pragma unroll
      for (uint32_t j = 0; j < kSl; ++j)
        sl[j] = *reinterpret_cast<const float4 *>(src + base + (tid + j * kBlkThreads) * 4);
    } else {  // the last, partial segment (element by element it took a pass of 1 M edges 4.5 us longer)
#pragma unroll
      for (uint32_t j = 0; j < kSl; ++j) {
        const uint32_t i = (tid + j * kBlkThreads) * 4;
        sl[j] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (i + 4 <= cnt) {
          sl[j] = *reinterpret_cast<const float4 *>(src + base + i);
        } else {
          if (i < cnt) sl[j].x = src[base + i];
          if (i + 1 < cnt) sl[j].y = src[base + i + 1];
          if (i + 2 < cnt) sl[j].z = src[base + i + 2];
        }
      }
    }
    uint2 ds = make_uint2(0, 0);
    if (nt) {
      if (lane < nt) ds = d.desc[t0 + lane * kBlkWaves];
#pragma unroll
      for (int j = 0; j < R; ++j) load(j, t0 + min((uint32_t)j, nt - 1) * kBlkWaves);
    }
#pragma unroll
    for (uint32_t j = 0; j < kSl; ++j)
      *reinterpret_cast<float4 *>(&slice[(tid + j * kBlkThreads) * 4]) = sl[j];
    __syncthreads();
    for (uint32_t i0 = 0; i0 < nt; i0 += kWave) {  // 64 tasks per batch of descriptors
      if (i0 && lane < nt - i0) ds = d.desc[t0 + (i0 + lane) * kBlkWaves];
      const uint32_t i1 = min(nt, i0 + kWave);
      for (uint32_t i = i0; i < i1; i += R) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
          if (i + j < i1) {
            const uint32_t x[4] = {e[j].x, e[j].y, e[j].z, e[j].w};
            float v[8];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              v[2 * q] = slice[x[q] & 0xffffu];
              v[2 * q + 1] = slice[x[q] >> 16];
            }
            if constexpr (kW) {
              v[0] *= wa[j].x;
              v[1] *= wa[j].y;
              v[2] *= wa[j].z;
              v[3] *= wa[j].w;
              v[4] *= wb[j].x;
              v[5] *= wb[j].y;
              v[6] *= wb[j].z;
              v[7] *= wb[j].w;
            }
            const uint32_t cls = __builtin_amdgcn_readlane(ds.x, i + j - i0);
            float *part = d.partial + __builtin_amdgcn_readlane(ds.y, i + j - i0);
            load(j, t0 + min(i + j + R, nt - 1) * kBlkWaves);
            blk_task(cls, part, v);
          }
        }
      }
    }
  }
}

// Combine of iteration k: row v's terms added in a fixed order, then
// fin.finish(v, sum, err, fin.pre(v)) (pre: the row's other inputs, loaded
// ahead); the residual goes to errs[k % 3].  A term is a partial of the
// segment pass or an element of `src`; kW: times its weight (1 for a partial).
// Rows by their number of terms: more than kCmbBig a workgroup each (the
// first huge_blocks workgroups), more than kCmbMid a wave, more than
// kCmbLight kCmbMidLanes lanes, each lane with kCmbPer terms in flight and the
// lanes' sums added with DPP moves; every other row a lane, its terms all in
// flight and added in order, 256 consecutive rows per workgroup in the rest.
// Rows past n_live get a constant update: iterations 0 and 1 write it into
// both ping-pong buffers, later iterations skip them.
// kSolo: there is no segment pass, so this launch applies the stop rule
// (every workgroup reads the residual of iteration k - 1).
// kMany: a lane has four rows and more (a kernel of its own: with their code in
// it a weighted forward on RMAT-20 took 1.142 ms, without 1.132).
template <class Fin, bool kW, bool kSolo, bool kMany>
__global__ void __launch_bounds__(256) blk_combine_kernel(BlkDev d, Fin fin, const float *__restrict__ src,
                                                          IterCtl *ctl, uint32_t k, uint32_t huge_blocks,
                                                          uint32_t big_blocks, uint32_t mid_blocks) {
  if (__hip_atomic_load(&ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  if constexpr (kSolo) {
    if (k > 0) {
      const double res = err_total(ctl, (k - 1) % 3);
      if (res < ctl->eps) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
          ctl->iters = k;
          ctl->residual = res;
          __hip_atomic_store(&ctl->done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return;
      }
    }
    if (blockIdx.x == 0) {
      double *z = &ctl->errs[(k + 1) % 3][0].v;
      for (uint32_t i = threadIdx.x; i < kErrSlots * (sizeof(ErrSlot) / sizeof(double)); i += 256) z[i] = 0.0;
    }
  }
  __shared__ float s_red[256 / kWave];
  const uint32_t nv = k >= 2 ? d.n_live : d.n;
  float err = 0.f;
  const uint32_t lane = threadIdx.x % kWave;
  // U terms, all in flight: term t at cmb_pos[at(t)] where in(t), else 0
  auto gather = [&](auto u, auto at, auto in, float *p) {
    constexpr uint32_t U = decltype(u)::value;
    uint32_t ix[U];
    float w[kW ? U : 1];
#pragma unroll
    for (uint32_t t = 0; t < U; ++t) ix[t] = in(t) ? d.cmb_pos[at(t)] : 0u;
    if constexpr (kW) {  // beside a segment pass nearly every term is a partial: no weight to load
#pragma unroll
      for (uint32_t t = 0; t < U; ++t) {
        const bool has = kSolo ? in(t) : (in(t) && !(ix[t] & kIsPartial));
        w[t] = has ? d.wcmb[at(t)] : 1.f;
      }
    }
#pragma unroll
    for (uint32_t t = 0; t < U; ++t) {
      const float *b = (ix[t] & kIsPartial) ? d.partial : src;
      p[t] = in(t) ? b[ix[t] & ~kIsPartial] : 0.f;
    }
    if constexpr (kW) {
#pragma unroll
      for (uint32_t t = 0; t < U; ++t) p[t] *= w[t];
    }
  };
  // those of a range from q on, `stride` apart
  auto terms = [&](auto u, uint32_t q, uint32_t stride, uint32_t end, float *p) {
    gather(u, [&](uint32_t t) { return q + t * stride; }, [&](uint32_t t) { return q + t * stride < end; }, p);
  };
  using Per = std::integral_constant<uint32_t, kCmbPer>;
  uint32_t blk = blockIdx.x;
  if (blk < huge_blocks) {
    for (uint32_t i = blk; i < d.n_huge; i += huge_blocks) {
      const uint32_t v = d.cmb_huge[i];
      const uint32_t b = d.cmb_rp[v + 1];
      float s = 0.f;
      for (uint32_t q = d.cmb_rp[v] + threadIdx.x; q < b; q += kCmbPer * 256) {
        float p[kCmbPer];
        terms(Per{}, q, 256, b, p);
#pragma unroll
        for (uint32_t w = kCmbPer / 2; w > 0; w >>= 1)
#pragma unroll
          for (uint32_t t = 0; t < w; ++t) p[t] += p[t + w];
        s += p[0];
      }
      s = block_sum<256, float>(s, s_red);
      if (threadIdx.x == 0) fin.finish(v, s, err, fin.pre(v));
    }
  } else if ((blk -= huge_blocks) < big_blocks) {
    for (uint32_t i = (blk * 256 + threadIdx.x) / kWave; i < d.n_big; i += big_blocks * (256 / kWave)) {
      const uint32_t v = d.cmb_big[i];  // the same for the whole wave
      float p[kCmbPer];
      terms(Per{}, d.cmb_rp[v] + lane, kWave, d.cmb_rp[v + 1], p);
#pragma unroll
      for (uint32_t w = kCmbPer / 2; w > 0; w >>= 1)
#pragma unroll
        for (uint32_t t = 0; t < w; ++t) p[t] += p[t + w];
      const float s = blk_group_sum<kWave>(p[0]);
      if (lane == 0) fin.finish(v, s, err, fin.pre(v));
    }
  } else if ((blk -= big_blocks) < mid_blocks) {
    constexpr uint32_t G = kCmbMidLanes;
    const uint32_t j = threadIdx.x % G;
    for (uint32_t i = (blk * 256 + threadIdx.x) / G; i < d.n_mid; i += mid_blocks * (256 / G)) {
      const uint32_t v = d.cmb_mid[i];  // the same for the group's lanes (inside one DPP row)
      float p[kCmbPer];
      terms(Per{}, d.cmb_rp[v] + j, G, d.cmb_rp[v + 1], p);
#pragma unroll
      for (uint32_t w = kCmbPer / 2; w > 0; w >>= 1)
#pragma unroll
        for (uint32_t t = 0; t < w; ++t) p[t] += p[t + w];
      const float s = blk_group_sum<G>(p[0]);
      if (j == 0) fin.finish(v, s, err, fin.pre(v));
    }
  } else {
    blk -= mid_blocks;
    const uint32_t nlb = gridDim.x - huge_blocks - big_blocks - mid_blocks;
    auto one = [&](uint32_t v) {
      const uint32_t a = d.cmb_rp[v], b = d.cmb_rp[v + 1];
      if (b - a > kCmbLight) return;  // a listed row
      const auto pre = fin.pre(v);
      // the wave takes 4, 8 or 16 terms a lane by its longest row
      const bool over4 = ballot(b - a > 4) != 0, over8 = ballot(b - a > 8) != 0;
      float s = 0.f;
      auto run = [&](auto u) {
        constexpr uint32_t U = decltype(u)::value;
        float p[U];
        terms(u, a, 1, b, p);
#pragma unroll
        for (uint32_t t = 0; t < U; ++t) s += p[t];
      };
      if (over8) run(std::integral_constant<uint32_t, 16>{});
      else if (over4) run(std::integral_constant<uint32_t, 8>{});
      else run(std::integral_constant<uint32_t, 4>{});
      fin.finish(v, s, err, pre);
    };
    // R rows of the lane, `step` apart, of at most T terms each, all in flight.
    // Where a lane has many short rows (millions of vertices of low degree) its
    // rows one after another are a chain of offsets, places, terms and stores
    // that does not keep HBM busy: an iteration on a path of 10 M vertices 109
    // us row by row, 94 so; a 3000 x 3000 grid 111 and 98; the adjoint on 40 M
    // vertices with 1 M edges 83 and 58.
    const uint32_t step = nlb * 256;
    auto rows = [&](auto r, auto per, uint32_t v, const uint32_t *a, const uint32_t *b) {
      constexpr uint32_t R = decltype(r)::value, T = decltype(per)::value;
      typename Fin::Pre pre[R];
#pragma unroll
      for (uint32_t i = 0; i < R; ++i) pre[i] = fin.pre(v + i * step);
      float p[R * T];
      gather(std::integral_constant<uint32_t, R * T>{}, [&](uint32_t t) { return a[t / T] + t % T; },
             [&](uint32_t t) { return a[t / T] + t % T < b[t / T]; }, p);
#pragma unroll
      for (uint32_t i = 0; i < R; ++i) {
        float s = 0.f;
#pragma unroll
        for (uint32_t t = 0; t < T; ++t) s += p[i * T + t];
        fin.finish(v + i * step, s, err, pre[i]);
      }
    };
    using R2 = std::integral_constant<uint32_t, 2>;
    using R4 = std::integral_constant<uint32_t, 4>;
    uint32_t v = blk * 256 + threadIdx.x;
    if constexpr (kMany) {
      for (; nv > 3 * step && v < nv - 3 * step; v += 4 * step) {
        uint32_t a[4], b[4], most = 0;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) a[i] = d.cmb_rp[v + i * step], b[i] = d.cmb_rp[v + i * step + 1];
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) most = max(most, b[i] - a[i]);
        if (!ballot(most > 2)) {
          rows(R4{}, R2{}, v, a, b);
        } else if (!ballot(most > 4)) {
          rows(R2{}, R4{}, v, a, b);
          rows(R2{}, R4{}, v + 2 * step, a + 2, b + 2);
        } else {
          for (uint32_t i = 0; i < 4; ++i) one(v + i * step);
        }
      }
    }
    for (; v < nv; v += step) one(v);
  }
  err = block_sum<256, float>(err, s_red);
  if (threadIdx.x == 0 && err != 0.f) atomicAdd(&ctl->errs[k % 3][blockIdx.x % kErrSlots].v, (double)err);
}

}  // namespace olv
