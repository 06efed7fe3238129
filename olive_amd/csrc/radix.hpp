// Stable LSD radix sort of 32-bit keys on the device (8 bits per pass),
// shared by the ingest (COO -> CSR, transposes), the in-degree numbering and
// the PageRank plans.
#pragma once
#include <algorithm>

#include "device.hpp"
#include "internal.hpp"

namespace olv {
namespace {

constexpr int kIB = 256;                     // workgroup size of the sort and scan kernels
constexpr int kIItems = 16;                  // items per lane in a tile
constexpr uint32_t kITile = kIB * kIItems;   // 4096 items per tile
constexpr int kRBits = 8;                    // radix digit width
constexpr int kRDigits = 1 << kRBits;
constexpr int kIWaves = kIB / kWave;

// ------------------------------------------------------------------ scans
// Exclusive prefix of x over the workgroup; `total` gets the workgroup sum.
__device__ __forceinline__ uint32_t block_excl_sum(uint32_t x, uint32_t &total) {
  __shared__ uint32_t s_w[kIWaves];
  const uint32_t incl = wave_inclusive_scan(x);
  const uint32_t w = threadIdx.x / kWave;
  if (lane_id() == kWave - 1) s_w[w] = incl;
  __syncthreads();
  uint32_t off = 0, tot = 0;
#pragma unroll
  for (uint32_t i = 0; i < (uint32_t)kIWaves; ++i) {
    const uint32_t v = s_w[i];
    off += i < w ? v : 0u;
    tot += v;
  }
  __syncthreads();
  total = tot;
  return off + incl - x;
}

// ---------------------------------------------------------- rows of slots
// Last row r in [0, n) with rp[r] <= slot, found by the calling wave 64
// probes at a time (rp[0] = 0 <= slot < rp[n]).
__device__ __forceinline__ uint32_t wave_row_of(const uint32_t *__restrict__ rp, uint32_t n, uint32_t slot) {
  uint32_t lo = 0, hi = n;  // rp[lo] <= slot < rp[hi]
  while (hi - lo > 1) {
    const uint32_t step = (hi - lo + kWave) / (kWave + 1);
    const uint64_t at = (uint64_t)lo + (uint64_t)step * (lane_id() + 1);
    const uint64_t le = ballot(at < hi && rp[at < hi ? (uint32_t)at : lo] <= slot);  // a prefix of the lanes
    const uint32_t k = (uint32_t)__popcll(le);
    const uint64_t nhi = (uint64_t)lo + (uint64_t)step * (k + 1);
    lo += step * k;
    hi = nhi < hi ? (uint32_t)nhi : hi;
  }
  return lo;
}

// Rows of the slots base .. base + cnt - 1 (0 < cnt <= kITile) of a CSR for a
// workgroup of kIB lanes: slot base + j lies in row first + s_row[j].  Returns
// `first`.  Rows that start in the tile are marked in LDS -- the empty ones
// aside, so no two at one slot -- and spread by a running maximum, so hub rows
// cost no more than any others.  A tile over a long run of empty rows (a block
// of ids without edges) does not walk it: every lane searches the row of the
// first of its kIItems consecutive slots, then those of the others up to the
// next lane's.
constexpr uint32_t kIWalk = 8;           // rows in flight per lane
constexpr uint32_t kIWalkRows = 1u << 16;  // rows between a tile's first and last that are walked, at most
__device__ __forceinline__ uint32_t tile_rows(const uint32_t *__restrict__ rp, uint32_t n, uint32_t base, uint32_t cnt,
                                              uint32_t *s_row) {
  __shared__ uint32_t s_ends[2], s_w[kIWaves];
  const uint32_t t = threadIdx.x, w = t / kWave;
  if (w < 2) {
    const uint32_t r = wave_row_of(rp, n, w ? base + cnt - 1 : base);
    if (lane_id() == 0) s_ends[w] = r;
  }
  for (uint32_t j = t; j < kITile; j += kIB) s_row[j] = 0u;
  __syncthreads();
  const uint32_t first = s_ends[0], last = s_ends[1];
  if (last - first > kIWalkRows) {
    const uint32_t j0 = t * kIItems;
    uint32_t r0 = first;
    for (uint32_t len = last - first + 1; len > 1; len -= len / 2)  // the row is in r0 .. r0 + len - 1
      if (rp[r0 + len / 2] <= base + min(j0, cnt - 1)) r0 += len / 2;
    s_row[j0] = r0 - first;
    __syncthreads();
    uint32_t r[kIItems];
#pragma unroll
    for (int i = 1; i < kIItems; ++i) r[i] = r0;
    for (uint32_t len = (j0 + kIItems < kITile ? first + s_row[j0 + kIItems] : last) - r0 + 1; len > 1; len -= len / 2) {
#pragma unroll
      for (int i = 1; i < kIItems; ++i)
        if (rp[r[i] + len / 2] <= base + min(j0 + i, cnt - 1)) r[i] += len / 2;
    }
#pragma unroll
    for (int i = 1; i < kIItems; ++i) s_row[j0 + i] = r[i] - first;
    __syncthreads();
    return first;
  }
  const uint32_t span = last - first;  // counted from `first`: ids of rows reach 2^32 - 2
  for (uint32_t q = 1 + t; q <= span; q += kIWalk * kIB) {
    uint32_t at[kIWalk], end[kIWalk];
#pragma unroll
    for (uint32_t i = 0; i < kIWalk; ++i) {
      const uint32_t r = first + min(q + i * kIB, span);
      at[i] = rp[r];
      end[i] = rp[(size_t)r + 1];
    }
#pragma unroll
    for (uint32_t i = 0; i < kIWalk; ++i)
      if (end[i] > at[i] && q + i * kIB <= span) s_row[at[i] - base] = q + i * kIB;
  }
  __syncthreads();
  uint32_t v[kIItems], run = 0;
#pragma unroll
  for (int i = 0; i < kIItems; ++i) {
    run = max(run, s_row[t * kIItems + i]);
    v[i] = run;
  }
  uint32_t inc = run;  // running maximum over the wave, then over the waves before
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t x = __shfl_up(inc, o, kWave);
    if (lane_id() >= (uint32_t)o) inc = max(inc, x);
  }
  if (lane_id() == kWave - 1) s_w[w] = inc;
  uint32_t before = __shfl_up(inc, 1, kWave);
  if (lane_id() == 0) before = 0;
  __syncthreads();
  for (uint32_t i = 0; i < w; ++i) before = max(before, s_w[i]);
#pragma unroll
  for (int i = 0; i < kIItems; ++i) s_row[t * kIItems + i] = max(v[i], before);
  __syncthreads();
  return first;
}

// ------------------------------------------------------------- radix sort
// counts[d * ntiles + t] = keys of tile t whose digit at `shift` is d.
__global__ void __launch_bounds__(kIB) radix_count_kernel(const uint32_t *__restrict__ keys, uint32_t m,
                                                          uint32_t shift, uint32_t ntiles,
                                                          uint32_t *__restrict__ counts) {
  __shared__ uint32_t h[kIWaves][kRDigits];
  for (uint32_t i = threadIdx.x; i < (uint32_t)(kIWaves * kRDigits); i += kIB) (&h[0][0])[i] = 0u;
  __syncthreads();
  const uint32_t w = threadIdx.x / kWave;
  const size_t base = (size_t)blockIdx.x * kITile;
#pragma unroll
  for (int i = 0; i < kIItems; ++i) {
    const size_t k = base + (size_t)i * kIB + threadIdx.x;
    if (k < m) atomicAdd(&h[w][(keys[k] >> shift) & (kRDigits - 1)], 1u);
  }
  __syncthreads();
  for (uint32_t d = threadIdx.x; d < (uint32_t)kRDigits; d += kIB) {
    uint32_t c = 0;
#pragma unroll
    for (int x = 0; x < kIWaves; ++x) c += h[x][d];
    counts[(size_t)d * ntiles + blockIdx.x] = c;
  }
}

// Value sources of the first pass (later passes read the previous output).
struct LoadIndex {
  __device__ uint32_t operator()(size_t k) const { return (uint32_t)k; }
};
struct LoadArr {
  const uint32_t *a;
  __device__ uint32_t operator()(size_t k) const { return a[k]; }
};
struct LoadPair {
  const uint32_t *a, *b;
  __device__ uint2 operator()(size_t k) const { return make_uint2(a[k], b[k]); }
};
struct LoadIndexAnd {
  const uint32_t *b;
  __device__ uint2 operator()(size_t k) const { return make_uint2((uint32_t)k, b[k]); }
};
struct LoadAndIndex {
  const uint32_t *a;
  __device__ uint2 operator()(size_t k) const { return make_uint2(a[k], (uint32_t)k); }
};
template <class V>
struct LoadPrev {
  const V *a;
  __device__ V operator()(size_t k) const { return a[k]; }
};

// Stable scatter of one pass.  Wave w of tile t owns items
// t*kITile + w*kITile/kIWaves + i*64 + lane (i = 0..kIItems-1): in that order
// each item's rank among equal digits comes from 8 ballots (lanes with the
// same digit) plus the wave's running digit count in LDS; waves of a tile
// follow each other, tiles follow the scanned digit-major offsets.  The tile
// is first reordered by digit in LDS, so the stores of each digit's run go
// out as consecutive addresses.
static_assert(kIB == kRDigits, "one lane per digit in the offset step");
template <class V, class Load>
__global__ void __launch_bounds__(kIB) radix_scatter_kernel(const uint32_t *__restrict__ kin, Load load,
                                                            uint32_t *__restrict__ kout, V *__restrict__ vout,
                                                            uint32_t m, uint32_t shift, uint32_t ntiles,
                                                            const uint32_t *__restrict__ offs) {
  __shared__ uint32_t s_cnt[kIWaves][kRDigits];
  __shared__ uint32_t s_delta[kRDigits];
  __shared__ uint32_t s_key[kITile];
  __shared__ V s_val[kITile];
  for (uint32_t i = threadIdx.x; i < (uint32_t)(kIWaves * kRDigits); i += kIB) (&s_cnt[0][0])[i] = 0u;
  __syncthreads();
  const uint32_t w = threadIdx.x / kWave, l = lane_id();
  const size_t base = (size_t)blockIdx.x * kITile + (size_t)w * (kITile / kIWaves);
  const uint64_t below_mask = (1ull << l) - 1ull;
  uint32_t key[kIItems], rank[kIItems];
  V val[kIItems];
#pragma unroll
  for (int i = 0; i < kIItems; ++i) {
    const size_t k = base + (size_t)i * kWave + l;
    const bool ok = k < m;
    key[i] = ok ? kin[k] : 0u;
    val[i] = ok ? load(k) : V{};
    const uint32_t d = (key[i] >> shift) & (kRDigits - 1);
    uint64_t peers = __ballot(ok);
#pragma unroll
    for (int b = 0; b < kRBits; ++b) {
      const bool bit = (d >> b) & 1u;
      const uint64_t bb = __ballot(bit);
      peers &= bit ? bb : ~bb;
    }
    uint32_t r = 0;
    if (ok) {
      const uint32_t below = (uint32_t)__popcll(peers & below_mask);
      const uint32_t c0 = s_cnt[w][d];
      r = c0 + below;
      if (below == 0) s_cnt[w][d] = c0 + (uint32_t)__popcll(peers);  // first lane of the digit
    }
    rank[i] = r;
  }
  __syncthreads();
  {
    // lane d: tile-local start of digit d, each wave's start inside it, and
    // the shift from tile position to output position
    const uint32_t d = threadIdx.x;
    uint32_t c[kIWaves], tot = 0;
#pragma unroll
    for (int x = 0; x < kIWaves; ++x) {
      c[x] = s_cnt[x][d];
      tot += c[x];
    }
    uint32_t all;
    const uint32_t start = block_excl_sum(tot, all);
    uint32_t run = start;
#pragma unroll
    for (int x = 0; x < kIWaves; ++x) {
      s_cnt[x][d] = run;
      run += c[x];
    }
    s_delta[d] = offs[(size_t)d * ntiles + blockIdx.x] - start;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kIItems; ++i) {
    const size_t k = base + (size_t)i * kWave + l;
    if (k < m) {
      const uint32_t lp = s_cnt[w][(key[i] >> shift) & (kRDigits - 1)] + rank[i];
      s_key[lp] = key[i];
      s_val[lp] = val[i];
    }
  }
  __syncthreads();
  const uint32_t cnt = (uint32_t)min((size_t)kITile, (size_t)m - (size_t)blockIdx.x * kITile);
  for (uint32_t j = threadIdx.x; j < cnt; j += kIB) {
    const uint32_t k = s_key[j];
    const uint32_t pos = s_delta[(k >> shift) & (kRDigits - 1)] + j;
    kout[pos] = k;
    vout[pos] = s_val[j];
  }
}

struct SortBufs {
  ScratchBuf k[2], v[2], counts;
  int cur = 0;
  uint32_t *keys() const { return k[cur].as<uint32_t>(); }
  template <class V>
  V *vals() const { return v[cur].as<V>(); }
};

// Stable sort of items 0..m-1 by keys_in >> low (which is < 2^key_bits),
// carrying a value of type V read by load0(k) in the first pass.  keys_in is
// left unchanged; the result is b.keys() / b.vals<V>().
template <class V, class Load0>
int radix_sort(const uint32_t *keys_in, Load0 load0, uint32_t m, uint32_t key_bits, SortBufs &b, uint32_t low = 0) {
  const uint32_t ntiles = (uint32_t)(((size_t)m + kITile - 1) / kITile);
  for (int i = 0; i < 2; ++i) {
    OLV_TRY(b.k[i].alloc((size_t)m * 4));
    OLV_TRY(b.v[i].alloc((size_t)m * sizeof(V)));
  }
  OLV_TRY(b.counts.alloc(((size_t)kRDigits * ntiles + 1) * 4));
  const uint32_t passes = std::max(1u, (key_bits + kRBits - 1) / kRBits);
  hipStream_t s = stream();
  uint32_t *counts = b.counts.as<uint32_t>();
  for (uint32_t p = 0; p < passes && ntiles; ++p) {
    const int out = (int)(p & 1u);
    const uint32_t shift = low + p * kRBits;
    const uint32_t *kin = p == 0 ? keys_in : b.k[out ^ 1].as<uint32_t>();
    hipLaunchKernelGGL(radix_count_kernel, dim3(ntiles), dim3(kIB), 0, s, kin, m, shift, ntiles, counts);
    OLV_HIP(hipGetLastError());
    OLV_TRY(exclusive_scan(counts, counts, (size_t)kRDigits * ntiles));
    if (p == 0)
      hipLaunchKernelGGL((radix_scatter_kernel<V, Load0>), dim3(ntiles), dim3(kIB), 0, s, kin, load0,
                         b.k[out].as<uint32_t>(), b.v[out].as<V>(), m, shift, ntiles, counts);
    else
      hipLaunchKernelGGL((radix_scatter_kernel<V, LoadPrev<V>>), dim3(ntiles), dim3(kIB), 0, s, kin,
                         LoadPrev<V>{b.v[out ^ 1].as<V>()}, b.k[out].as<uint32_t>(), b.v[out].as<V>(), m, shift,
                         ntiles, counts);
    OLV_HIP(hipGetLastError());
    b.cur = out;
  }
  return OLV_OK;
}

inline uint32_t bits_for(uint32_t n) {  // bits of the largest id n - 1
  uint32_t b = 0;
  while (b < 32 && ((uint64_t)(n - 1) >> b) != 0) ++b;
  return b;
}

}  // namespace
}  // namespace olv
