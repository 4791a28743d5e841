// One-pass partition of both relations of a fused join.
//
// A join of medium size spends its time on launches and on reading its inputs
// for a histogram, one relation after the other.  Here both relations share
// every launch:
//   1. k_one_count: the digit counts — of a sample (one 128-byte line in 16, as
//      the two-pass partitions take) of a relation of kGapMinRows or more, of
//      every tuple of a smaller one — and, by the workgroup that finishes a
//      relation last, the layout of its partitions and cursors;
//   2. k_one_scatter: one workgroup per 16K-tuple tile of either relation, its
//      runs reserved from the partition cursors;
//   3. k_one_plan: the partitions' ends, the probe's tiles and their scan.
// The sampled buffers are sized for any line clumping (a line holds 16 tuples,
// so a sampled count's variance is at most 16 times its mean): sorted or
// grouped keys only widen the margins.  A partition that proves too small all
// the same raises kErrCapacity and the caller redoes the join exactly.
#include <algorithm>

#include "device.hpp"
#include "kernels.hpp"
#include "tile_kernels.hpp"

namespace eo {
namespace {

using tile::kFastNT;

constexpr int kOneNT = tile::kGapSampleNT;           // 512
constexpr uint32_t kOneTiles = tile::kGapSampleUnroll;  // tiles one workgroup samples
constexpr int kOnePlanNT = 1024;

// A counter's kOneCopies copies, one_hs_words apart, are added to by different
// XCDs' workgroups (atomics on one word queue up) and summed by the layout.
__device__ __forceinline__ uint32_t sum_copies(const uint32_t *p, uint32_t stride) {
  uint32_t v[kOneCopies], sum = 0;
#pragma unroll
  for (uint32_t x = 0; x < kOneCopies; ++x) v[x] = ld_agent(p + x * stride);
#pragma unroll
  for (uint32_t x = 0; x < kOneCopies; ++x) sum += v[x];
  return sum;
}

// The layout of relation r from the copies of its counts hs[0, F), clumping
// sum hs[F] and lines measured hs[F + 1]; clears them.  All threads of the
// workgroup.
template <int BITS>
__device__ __forceinline__ void one_layout(const OneRel &r, uint32_t *hs, uint32_t *err) {
  constexpr uint32_t F = 1u << BITS, BPT = F > (uint32_t)kOneNT ? F / kOneNT : 1, HW = one_hs_words(BITS);
  __shared__ uint64_t red[kOneNT / kWave + 1];
  const uint32_t b0 = threadIdx.x * BPT;
  uint32_t sv[BPT];
  uint64_t loc = 0, sq = 0;
#pragma unroll
  for (uint32_t k = 0; k < BPT; ++k) {
    sv[k] = b0 + k < F ? sum_copies(hs + b0 + k, HW) : 0u;
    loc += sv[k];
    sq += (uint64_t)sv[k] * sv[k];
  }
  const uint32_t qs = sum_copies(hs + F, HW), m = sum_copies(hs + F + 1, HW);
  const uint64_t ns = block_sum<kOneNT, uint64_t>(loc, red);
  const uint64_t ns2 = block_sum<kOneNT, uint64_t>(sq, red);
  const double f = ns ? (double)r.n / (double)ns : 0.0;
  // groups of lines the sample draws from (as the two-pass layout counts them)
  const uint64_t T = (r.n + tile::kFastTile - 1) / tile::kFastTile;
  const uint64_t tail = r.n - (T - 1) * tile::kFastTile;
  const double g = (double)(T - 1) * tile::kGapLinesPerTile +
                   (double)((tail + tile::kGapLineTuples * tile::kGapGroup - 1) / (tile::kGapLineTuples * tile::kGapGroup));
  const float kap = (r.sampled && ns && m) ? tile::gap_kappa((double)ns, (double)ns2, (double)qs * g / m, g) : 1.0f;
  uint64_t c[BPT];
  uint64_t sum = 0;
#pragma unroll
  for (uint32_t k = 0; k < BPT; ++k) {
    c[k] = b0 + k >= F ? 0
           : !r.sampled ? (sv[k] + tile::kGapLineTuples - 1) / tile::kGapLineTuples * tile::kGapLineTuples
           : ns ? tile::gap_cap(sv[k], kap, f) : 0;
    sum += c[k];
  }
  uint64_t tot;
  uint64_t at = block_excl_scan<kOneNT, uint64_t>(sum, red, &tot);
  if (threadIdx.x == 0 && (ns == 0 || tot > r.budget)) atomic_or_agent(err, kErrCapacity);
#pragma unroll
  for (uint32_t k = 0; k < BPT; ++k) {
    if (b0 + k < F) {
      const uint32_t a = (uint32_t)min(at, r.budget), e = (uint32_t)min(at + c[k], r.budget);
      r.start[b0 + k] = a;
      r.cur[tile::cursor_slot<BITS>(b0 + k)] = a;
      r.end[b0 + k] = e;  // the region's end, until the plan sets the filled one
    }
    at += c[k];
  }
  for (uint32_t i = threadIdx.x; i < kOneCopies * HW; i += kOneNT) hs[i] = 0;  // (every read is behind a barrier)
}

template <int BITS>
__global__ __launch_bounds__(kOneNT) void k_one_count(OneArgs a, uint32_t *err) {
  constexpr uint32_t F = 1u << BITS;
  constexpr int U = tile::kGapSampleUnroll;
  static_assert(kOneNT / kWave == U && F <= 0x8000u, "one wave per unrolled tile; digits packed two to a word");
  __shared__ uint32_t hist[F];
  __shared__ uint32_t s_last;
  const uint32_t rel = blockIdx.x < a.rel[0].units ? 0u : 1u;
  const OneRel &r = a.rel[rel];
  const uint32_t u = rel ? blockIdx.x - a.rel[0].units : blockIdx.x;
  uint32_t *const hs0 = a.hs + rel * kOneCopies * one_hs_words(BITS);  // this relation's copies
  uint32_t *const hs = hs0 + blockIdx.x % kOneCopies * one_hs_words(BITS);
  for (uint32_t d = threadIdx.x; d < F; d += kOneNT) hist[d] = 0;
  __syncthreads();
  if (r.sampled) {
    const uint32_t T = (uint32_t)((r.n + tile::kFastTile - 1) / tile::kFastTile), t0 = u * kOneTiles;
    const uint64_t npairs = r.n / 2;
    const uint4 *in4 = reinterpret_cast<const uint4 *>(r.in);
    const uint32_t j = threadIdx.x >> 3, q = threadIdx.x & 7;
    uint4 v[U];
    bool ok[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const uint32_t t = t0 + (uint32_t)k;
      const uint64_t p =
          (uint64_t)t * (tile::kFastTile / 2) + (uint64_t)tile::gap_line(t, j) * (tile::kGapLineTuples / 2) + q;
      ok[k] = t < T && p < npairs;
      v[k] = ok[k] ? ld_stream(in4 + p) : make_uint4(0u, 0u, 0u, 0u);
    }
    uint32_t qsum = 0, lines = 0;
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const uint32_t d0 = v[k].x & (F - 1), d1 = v[k].z & (F - 1);
      if (k == (int)(threadIdx.x / kWave)) {  // wave-uniform: the tile whose clumping this wave measures
        uint32_t c0, c1;
        tile::line_same_counts(ok[k] ? d0 | d1 << 16 : ~0u, c0, c1);
        qsum = ok[k] ? c0 + c1 : 0u;
        lines = (uint32_t)__popcll(__ballot(ok[k] && q == 0));
      }
      if (!ok[k]) continue;
      atomicAdd(&hist[d0], 1u);
      atomicAdd(&hist[d1], 1u);
    }
    qsum = wave_sum(qsum);
    if (lane_id() == 0 && lines) {
      atomic_add_agent(hs + F, qsum);
      atomic_add_agent(hs + F + 1, lines);
    }
  } else {
    const uint64_t beg = (uint64_t)u * tile::kFastTile;
    tile::hist_stripe<BITS, kOneNT, true>(hist, r.in, beg, min(beg + tile::kFastTile, r.n), 0, 0u);
  }
  __syncthreads();
  for (uint32_t d = threadIdx.x; d < F; d += kOneNT)
    if (hist[d]) atomic_add_agent(hs + d, hist[d]);
  // The relation's last workgroup lays it out, from counts that are device-scope
  // atomics like the ticket.  (A release fence at device scope would also write
  // the XCD's whole L2 back, once per workgroup: 15 M tuples 39 instead of 28
  // us; one counter copy instead of kOneCopies: 28 instead of 13 us.)
  wait_atomics();
  __syncthreads();
  if (threadIdx.x == 0) s_last = atomic_add_agent(a.ticket + rel, 1u) == r.units - 1;
  __syncthreads();
  if (!s_last) return;
  one_layout<BITS>(r, hs0, err);
  if (threadIdx.x == 0) a.ticket[rel] = 0;
}

// Blocks [0, round8(tiles of R)) scatter R, the rest S; consecutive tiles of a
// relation on one XCD.  Also clears the left outer probe's words.
template <int BITS>
__global__ __launch_bounds__(kFastNT) void k_one_scatter(OneArgs a, uint32_t *err) {
  __shared__ tile::ScatterShared<BITS> sh;
  for (uint32_t i = blockIdx.x * kFastNT + threadIdx.x; i < a.nzero; i += gridDim.x * kFastNT) a.zero[i] = 0;
  const uint32_t g0 = (a.rel[0].tiles + kXcds - 1) / kXcds * kXcds;
  const uint32_t rel = blockIdx.x < g0 ? 0u : 1u;
  const OneRel &r = a.rel[rel];
  const uint32_t t = rel ? xcd_local_index(blockIdx.x - g0, gridDim.x - g0) : xcd_local_index(blockIdx.x, g0);
  const uint64_t beg = (uint64_t)t * tile::kFastTile;
  if (beg >= r.n) return;
  const uint64_t end = min(beg + tile::kFastTile, r.n);
  __shared__ uint32_t s_err;  // raised: the caller redoes the join, nothing is moved (as k_tile_scatter)
  if (threadIdx.x == 0) s_err = __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int d = threadIdx.x; d < (1 << BITS); d += kFastNT) {
    sh.cursor[d] = r.end[d];
    sh.clear_count(d);
  }
  tile::scatter_stripe<BITS, false, true>(sh, r.in, beg, end, r.n, 0, 0u, r.out, err, r.cur, &s_err);
}

// One workgroup: every partition's filled end, its probe tiles (R chunks of
// `cap`, outer: at least one, x S spans) and their scan.
template <int BITS>
__global__ __launch_bounds__(kOnePlanNT) void k_one_plan(OneArgs a, uint32_t s_span, uint32_t cap, int outer,
                                                          uint32_t *__restrict__ tile_start, uint64_t *n_tiles) {
  constexpr uint32_t F = 1u << BITS, BPT = F > (uint32_t)kOnePlanNT ? F / kOnePlanNT : 1;
  __shared__ uint64_t red[kOnePlanNT / kWave + 1];
  const uint32_t b0 = threadIdx.x * BPT;
  uint64_t cnt[BPT], sum = 0;
#pragma unroll
  for (uint32_t k = 0; k < BPT; ++k) {
    cnt[k] = 0;
    const uint32_t p = b0 + k;
    if (p < F) {
      uint32_t n[2];
#pragma unroll
      for (int rel = 0; rel < 2; ++rel) {
        const OneRel &r = a.rel[rel];
        const uint32_t e = min(r.cur[tile::cursor_slot<BITS>(p)], r.end[p]);
        r.end[p] = e;
        n[rel] = e - r.start[p];
      }
      // (products in 64 bits: a sum of 2^31 or more is refused by the probe)
      const uint32_t spans = (n[1] + s_span - 1) / s_span, chunks = (n[0] + cap - 1) / cap;
      cnt[k] = (uint64_t)(outer ? max(chunks, 1u) : chunks) * spans;
    }
    sum += cnt[k];
  }
  uint64_t tot;
  uint64_t at = block_excl_scan<kOnePlanNT, uint64_t>(sum, red, &tot);
#pragma unroll
  for (uint32_t k = 0; k < BPT; ++k) {
    if (b0 + k < F) tile_start[b0 + k] = (uint32_t)at;
    at += cnt[k];
  }
  if (threadIdx.x == 0) {
    tile_start[F] = (uint32_t)tot;
    *n_tiles = tot;
  }
}

}  // namespace

OneRel one_pass_rel(const eo_tuple *in, uint64_t n, int bits, eo_tuple *out, uint32_t *start, uint32_t *end,
                    uint32_t *cur) {
  OneRel r{};
  r.in = reinterpret_cast<const uint2 *>(in);
  r.out = reinterpret_cast<uint2 *>(out);
  r.n = n;
  r.sampled = n >= kGapMinRows;
  r.tiles = (uint32_t)((n + tile::kFastTile - 1) / tile::kFastTile);
  r.units = r.sampled ? (r.tiles + kOneTiles - 1) / kOneTiles : r.tiles;
  r.budget = one_pass_rows(n, bits);
  r.start = start;
  r.end = end;
  r.cur = cur;
  return r;
}

namespace {

template <int BITS>
hipError_t launch_one(const OneArgs &a, uint32_t s_span, uint32_t cap, bool outer, uint32_t *tile_start,
                      uint64_t *n_tiles, uint32_t *err, hipStream_t stream) {
  EO_TIMED("part_sample", stream,
           hipLaunchKernelGGL(k_one_count<BITS>, dim3(a.rel[0].units + a.rel[1].units), dim3(kOneNT), 0, stream, a,
                              err));
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const uint32_t grid =
      (a.rel[0].tiles + kXcds - 1) / kXcds * kXcds + (a.rel[1].tiles + kXcds - 1) / kXcds * kXcds;
  EO_TIMED("part_scatter", stream,
           hipLaunchKernelGGL(k_one_scatter<BITS>, dim3(grid), dim3(kFastNT), 0, stream, a, err));
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_one_plan<BITS>, dim3(1), dim3(kOnePlanNT), 0, stream, a, s_span, cap, (int)outer, tile_start,
                     n_tiles);
  return hipGetLastError();
}

}  // namespace

hipError_t one_pass_partition(const OneArgs &a, int bits, uint32_t s_span, uint32_t cap, bool outer,
                              uint32_t *tile_start, uint64_t *n_tiles, uint32_t *err, hipStream_t stream) {
  for (const OneRel &r : a.rel)
    if (((uintptr_t)r.in & 15) || ((uintptr_t)r.out & 7)) return hipErrorInvalidValue;
  switch (bits) {
#define EO_ONE_CASE(B) \
  case B:              \
    return launch_one<B>(a, s_span, cap, outer, tile_start, n_tiles, err, stream);
    EO_ONE_CASE(1) EO_ONE_CASE(2) EO_ONE_CASE(3) EO_ONE_CASE(4) EO_ONE_CASE(5) EO_ONE_CASE(6)
    EO_ONE_CASE(7) EO_ONE_CASE(8) EO_ONE_CASE(9) EO_ONE_CASE(10)
#undef EO_ONE_CASE
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace eo
