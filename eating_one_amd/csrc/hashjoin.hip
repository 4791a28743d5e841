// Per-partition join of a radix-partitioned R and S.
//
// The reference's probe (count / join, joins/hashJoin_gpu/main_street/
// join_gpu.cu:9-113) holds a <=256-tuple S chunk in shared memory and compares
// every R tuple of the partition against all of it — a partitioned nested
// loop, run twice (count, then write).  Here each work tile
//   (partition p, R-chunk c of <= the LDS table's tuples, S span j)
// builds a bucketised table of its R chunk in LDS (tile::probe_tile: LDS
// counting sort by a multiplicative hash) and streams its S span past it.
// Default order: one fused pass per tile that reserves its rows with one
// atomic per S batch.  Deterministic order (the reference's count -> presum ->
// join): a count pass stores one total per tile, a u64 scan turns them into
// tile offsets, and a write pass re-probes with a table order fixed by the
// inputs and writes each tile's rows from its offset on.
#include <algorithm>

#include "device.hpp"
#include "kernels.hpp"
#include "plan.hpp"
#include "tile_kernels.hpp"

namespace eo {
namespace {

// Fused probe, one pass over S.  A tile is (partition p, R-chunk c, S span j):
// the R chunk (<= 16384 tuples) is built once into an LDS table and the whole S
// span (up to s_span tuples) streams past it in batches of NT*SPT tuples held
// in VGPRs, the next batch's loads in flight while the current one probes.
//
// LDS table (SoA, 144 KB): keys[16384] and pays[16384] grouped by bucket,
// u16 bucket offsets off[8192 + 1].  Built in three steps without a cursor
// array: (1) every R tuple takes its rank inside its bucket from an LDS
// atomic on a u32 counter array that lives in the (still empty) keys region,
// (2) a workgroup scan turns the counters into u16 offsets, (3) each tuple is
// stored at off[h] + rank.
//
// Per batch, every S tuple is probed once (match count and first payload kept
// in registers), output positions are numbered register-major (so a wave's
// store instruction writes one contiguous run), and one 64-bit atomic per
// batch reserves the output range.  Pairs at positions >= out_cap are counted
// but not written.
using namespace tile;

// Partition p of R is [r_start[p], r_end[p]) (r_end = r_start + 1 for
// contiguous partitions), of S [s_start[p], s_end[p]).
__device__ __forceinline__ bool resolve_span(uint32_t t, const uint32_t *tile_start, uint32_t P,
                                             const uint32_t *r_start, const uint32_t *r_end,
                                             const uint32_t *s_start, const uint32_t *s_end, uint32_t s_span,
                                             uint32_t cap, SpanRef *ref, uint32_t *part = nullptr) {
  if (t >= tile_start[P]) return false;
  const uint32_t p = wave_find(tile_start, P, t);
  if (part) *part = p;
  const uint32_t local = t - tile_start[p];
  const uint32_t rb = r_start[p], rn = r_end[p] - rb;
  const uint32_t sb = s_start[p], sn = s_end[p] - sb;
  const uint32_t nc = max(1u, (rn + cap - 1) / cap);
  const uint32_t c = local % nc, j = local / nc;
  ref->r_beg = rb + c * cap;
  ref->r_n = min(cap, rn - c * cap);
  ref->s_beg = sb + j * s_span;
  ref->s_n = min(s_span, sn - j * s_span);
  return true;
}

// The half-size table variant is limited to 64 VGPRs so that two 16-wave
// workgroups fit on a CU (8 waves per SIMD).
//
// The grid is sized on the host without knowing the tile count (no readback
// between planning and probing): block b runs tiles b, b + grid, ... below the
// planned total *n_tiles, so a grid of one block per partition covers the
// usual one-tile partitions exactly and the extra span tiles of skewed
// partitions go to the blocks that started first.
template <typename C>
__global__ __launch_bounds__(kFNT) __attribute__((amdgpu_waves_per_eu(C::Cap <= 8704 ? 8 : 1)))
void k_join_fused(const uint2 *__restrict__ R, const uint32_t *__restrict__ r_start,
                  const uint32_t *__restrict__ r_end, const uint2 *__restrict__ S,
                  const uint32_t *__restrict__ s_start, const uint32_t *__restrict__ s_end,
                  const uint32_t *__restrict__ tile_start, uint32_t P,
                                                     uint32_t s_span, uint2 *__restrict__ out, uint64_t out_cap,
                                                     uint64_t *out_cursor, int wide, uint32_t *matched,
                                                     const uint64_t *__restrict__ n_tiles, uint32_t *err,
                                                     int swapped) {
  __shared__ tile::ProbeShared<C> sh;
  const uint64_t nt = *n_tiles;
  if (nt >= (1ull << 31)) {  // tile ids are 32-bit: report, probe nothing
    if (blockIdx.x == 0 && threadIdx.x == 0) atomic_or_agent(err, kErrOverflow);
    return;
  }
  // round-robin over the XCDs: the span tiles of one hot (skewed) partition
  // are consecutive and must not all land on one XCD
  for (uint32_t t = blockIdx.x; t < (uint32_t)nt; t += gridDim.x) {
    if (t != blockIdx.x) __syncthreads();  // the previous tile's LDS reads are done
    SpanRef ref;
    if (!resolve_span(t, tile_start, P, r_start, r_end, s_start, s_end, s_span, C::Cap, &ref)) return;
    tile::probe_tile<C>(sh, R, S, ref, out, out_cap, out_cursor, wide != 0, matched, 0, swapped != 0);
  }
}

// Null rows of the S tuples of a span whose bit (over S positions) is clear.
// LDS is free for use; all threads of the workgroup.
template <typename C>
__device__ __forceinline__ void null_rows(tile::ProbeShared<C> &sh, const uint2 *__restrict__ S, const SpanRef &ref,
                                          const uint32_t *bits, uint2 *__restrict__ out, uint64_t out_cap,
                                          uint64_t *cursor, bool wide) {
  for (uint32_t b0 = 0; b0 < ref.s_n; b0 += C::Batch) {
    uint32_t mask = 0;
#pragma unroll
    for (int u = 0; u < C::SPT; ++u) {
      const uint32_t i = b0 + u * C::NT + threadIdx.x, pos = ref.s_beg + i;
      if (i < ref.s_n && !((ld_agent(bits + pos / 32) >> (pos % 32)) & 1u)) mask |= 1u << u;
    }
    uint32_t tot;
    const uint32_t ex = block_excl_scan<C::NT, uint32_t>((uint32_t)__popc(mask), sh.scan_tmp, &tot);
    if (threadIdx.x == 0) sh.base_sh[0] = tot ? atomic_add_agent(cursor, (uint64_t)tot) : 0ull;
    __syncthreads();
    uint64_t pos = sh.base_sh[0] + ex;
    for (; mask; mask &= mask - 1u, ++pos) {
      const uint2 t = S[ref.s_beg + b0 + ((uint32_t)__ffs(mask) - 1u) * C::NT + threadIdx.x];
      if (pos < out_cap) emit_null(out, pos, t.y, t.x, wide);
    }
    __syncthreads();
  }
}

// Left outer join of one-pass partitions.  A partition whose R side is one
// chunk (the usual case) writes its null rows with the others.  The chunks of a
// larger one run beside each other, mark the matches of their span in bits
// (over S positions, zero on entry), and the last of them (done: a ticket per
// span, zero on entry) writes the null rows.  (One workgroup per span taking
// the chunks in turn needed neither, and 5 ms instead of 0.1 where one
// partition held all of 2^22 R tuples.)
template <typename C>
__global__ __launch_bounds__(kFNT) __attribute__((amdgpu_waves_per_eu(C::Cap <= 8704 ? 8 : 1)))
void k_join_outer(const uint2 *__restrict__ R, const uint32_t *__restrict__ r_start,
                  const uint32_t *__restrict__ r_end, const uint2 *__restrict__ S,
                  const uint32_t *__restrict__ s_start, const uint32_t *__restrict__ s_end,
                  const uint32_t *__restrict__ tile_start, uint32_t P, uint32_t s_span, uint2 *__restrict__ out,
                  uint64_t out_cap, uint64_t *cursor, int wide, uint32_t *bits, uint32_t *done,
                  const uint64_t *__restrict__ n_tiles, uint32_t *err) {
  __shared__ tile::ProbeShared<C> sh;
  __shared__ uint32_t s_last;
  const uint64_t nt = *n_tiles;
  if (nt >= (1ull << 31)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) atomic_or_agent(err, kErrOverflow);
    return;
  }
  for (uint32_t t = blockIdx.x; t < (uint32_t)nt; t += gridDim.x) {
    if (t != blockIdx.x) __syncthreads();
    SpanRef ref;
    uint32_t p = 0;
    if (!resolve_span(t, tile_start, P, r_start, r_end, s_start, s_end, s_span, C::Cap, &ref, &p)) return;
    const uint32_t nc = (r_end[p] - r_start[p] + C::Cap - 1) / C::Cap;
    tile::probe_tile<C, tile::kProbeFused, true>(sh, R, S, ref, out, out_cap, cursor, wide != 0,
                                                 nc > 1 ? bits : nullptr);
    if (nc <= 1) continue;
    wait_atomics();
    __syncthreads();
    // (spans have a ticket each: a partition's lie one s_span apart)
    if (threadIdx.x == 0) s_last = atomic_add_agent(done + p + ref.s_beg / s_span, 1u) == nc - 1;
    __syncthreads();
    if (s_last) null_rows<C>(sh, S, ref, bits, out, out_cap, cursor, wide != 0);
  }
}

// An unpartitioned left outer join whose R side is one chunk: one S span per
// workgroup, the null rows with the others.  WRITE = false counts only.
template <typename C, bool WRITE>
__global__ __launch_bounds__(C::NT) __attribute__((amdgpu_waves_per_eu(C::Cap <= 8704 ? 8 : 1)))
void k_join_direct_outer(const uint2 *__restrict__ R, uint32_t nR, const uint2 *__restrict__ S, uint32_t nS,
                         uint32_t span, uint2 *__restrict__ out, uint64_t out_cap, uint64_t *cursor, int wide) {
  __shared__ tile::ProbeShared<C> sh;
  SpanRef ref;
  ref.r_beg = 0;
  ref.r_n = nR;
  ref.s_beg = blockIdx.x * span;
  ref.s_n = min(span, nS - ref.s_beg);
  if (WRITE) {
    tile::probe_tile<C, tile::kProbeFused, true>(sh, R, S, ref, out, out_cap, cursor, wide != 0);
  } else {
    const uint64_t n = tile::probe_tile<C, tile::kProbeCount, true>(sh, R, S, ref, nullptr, 0, nullptr);
    if (threadIdx.x == 0 && n) atomic_add_agent(cursor, n);
  }
}

// An unpartitioned join: tile t is R chunk t % chunks against S span t /
// chunks, so nothing is planned on the device and the join is this launch.
// WRITE = false counts only.  matched: as probe_tile's.
template <typename C, bool WRITE>
__global__ __launch_bounds__(C::NT) __attribute__((amdgpu_waves_per_eu(C::Cap <= 8704 ? 8 : 1)))
void k_join_direct(const uint2 *__restrict__ R, uint64_t nR, const uint2 *__restrict__ S, uint64_t nS, uint32_t chunk,
                   uint32_t chunks, uint32_t span, uint2 *__restrict__ out, uint64_t out_cap, uint64_t *cursor,
                   int wide, uint32_t *matched, int swapped) {
  __shared__ tile::ProbeShared<C> sh;
  const uint32_t c = blockIdx.x % chunks, j = blockIdx.x / chunks;
  SpanRef ref;
  ref.r_beg = c * chunk;
  ref.r_n = (uint32_t)min((uint64_t)chunk, nR - ref.r_beg);
  ref.s_beg = j * span;
  ref.s_n = (uint32_t)min((uint64_t)span, nS - ref.s_beg);
  if (WRITE) {
    tile::probe_tile<C>(sh, R, S, ref, out, out_cap, cursor, wide != 0, matched, 0, swapped != 0);
  } else {
    const uint64_t n = tile::probe_tile<C, tile::kProbeCount>(sh, R, S, ref, nullptr, 0, nullptr, false, matched);
    if (threadIdx.x == 0 && n) atomic_add_agent(cursor, n);
  }
}

// Deterministic order on the fused probe's tiles: a count pass (one count per
// tile, and the matched bits of a left outer join), a scan of the counts, and
// a write pass whose tiles write from their scanned offsets with a table
// order fixed by the inputs (kProbeOrdered).
template <typename C>
__global__ __launch_bounds__(kFNT) __attribute__((amdgpu_waves_per_eu(C::Cap <= 8704 ? 8 : 1)))
void k_span_count(const uint2 *__restrict__ R, const uint32_t *__restrict__ r_start, const uint2 *__restrict__ S,
                  const uint32_t *__restrict__ s_start, const uint32_t *__restrict__ tile_start, uint32_t P,
                  uint32_t s_span, uint64_t *__restrict__ tile_count, uint32_t n, uint32_t *matched,
                  const uint64_t *__restrict__ n_tiles) {
  __shared__ tile::ProbeShared<C> sh;
  // 2^31 tiles or more: tile_start may have wrapped, and the host, which reads
  // *n_tiles, refuses the join
  const bool too_many = *n_tiles >= (1ull << 31);
  for (uint32_t t = blockIdx.x; t < n; t += gridDim.x) {  // a grid below the tile count loops
    if (t != blockIdx.x) __syncthreads();
    SpanRef ref;
    if (too_many ||
        !resolve_span(t, tile_start, P, r_start, r_start + 1, s_start, s_start + 1, s_span, C::Cap, &ref)) {
      if (threadIdx.x == 0) tile_count[t] = 0;  // past the last tile (uniform)
      continue;
    }
    const uint64_t n = tile::probe_tile<C, tile::kProbeCount>(sh, R, S, ref, nullptr, 0, nullptr, false, matched);
    if (threadIdx.x == 0) tile_count[t] = n;
  }
}

template <typename C>
__global__ __launch_bounds__(kFNT) __attribute__((amdgpu_waves_per_eu(C::Cap <= 8704 ? 8 : 1)))
void k_span_write(const uint2 *__restrict__ R, const uint32_t *__restrict__ r_start, const uint2 *__restrict__ S,
                  const uint32_t *__restrict__ s_start, const uint32_t *__restrict__ tile_start, uint32_t P,
                  uint32_t s_span, const uint64_t *__restrict__ tile_off, uint2 *__restrict__ out, uint64_t out_cap,
                  int wide) {
  __shared__ tile::ProbeShared<C> sh;
  for (uint32_t t = blockIdx.x;; t += gridDim.x) {  // a grid below the tile count loops
    if (t != blockIdx.x) __syncthreads();
    SpanRef ref;
    if (!resolve_span(t, tile_start, P, r_start, r_start + 1, s_start, s_start + 1, s_span, C::Cap, &ref)) return;
    tile::probe_tile<C, tile::kProbeOrdered>(sh, R, S, ref, out, out_cap, nullptr, wide != 0, nullptr, tile_off[t]);
  }
}

// tiles[p] of every partition (R chunks x S spans), and their 64-bit sum added
// to *n_tiles: a sum of 2^31 or more is refused by the kernels that read it,
// since the 32-bit tile numbers scanned from tiles[] may then have wrapped.
constexpr int kPlanNT = 256;
__global__ __launch_bounds__(kPlanNT) void k_plan_spans(const uint32_t *r_start, const uint32_t *r_end,
                                                        const uint32_t *s_start, const uint32_t *s_end, uint32_t P,
                                                        uint32_t s_span, uint32_t cap, uint32_t *tiles,
                                                        uint64_t *n_tiles) {
  __shared__ uint64_t red[kPlanNT / kWave + 1];
  const uint32_t p = blockIdx.x * kPlanNT + threadIdx.x;
  uint64_t n = 0;
  if (p < P)  // (below 2^31 tuples and spans below 2^31: the quotients fit 32 bits, their product need not)
    n = (uint64_t)((r_end[p] - r_start[p] + cap - 1) / cap) * ((s_end[p] - s_start[p] + s_span - 1) / s_span);
  if (p <= P) tiles[p] = (uint32_t)n;
  const uint64_t sum = block_sum<kPlanNT, uint64_t>(n, red);
  if (threadIdx.x == 0 && sum) atomic_add_agent(n_tiles, sum);
}

}  // namespace

size_t outer_words(uint64_t s_rows, uint32_t parts, uint32_t s_span) {
  return matched_words(s_rows) + parts + s_rows / s_span + 1;
}

size_t join_plan_scratch_bytes(uint32_t parts) { return scan_scratch_bytes_u32((uint64_t)parts + 1); }

}  // namespace eo

namespace eo {

static_assert(tile::ProbeBig::Cap == kFusedTableFull && tile::ProbeSmall::Cap == kFusedTableHalf &&
                  tile::ProbeQuarter::Cap == kFusedTableQuarter,
              "the planner's table sizes are the probe's");

uint32_t join_fused_cap(uint32_t lds_cap) {
  return lds_cap <= 8192 ? (uint32_t)tile::ProbeSmall::Cap : (uint32_t)tile::ProbeBig::Cap;
}

hipError_t join_fused_plan(uint32_t parts, uint32_t s_span, uint32_t cap, const uint32_t *r_start,
                           const uint32_t *r_end, const uint32_t *s_start, const uint32_t *s_end,
                           uint32_t *tile_start, uint64_t *n_tiles_dev, void *scan_scratch, uint32_t *err,
                           hipStream_t stream) {
  const uint32_t n = parts + 1;
  hipLaunchKernelGGL(k_plan_spans, dim3((n + kPlanNT - 1) / kPlanNT), dim3(kPlanNT), 0, stream, r_start, r_end,
                     s_start, s_end, parts, s_span, cap, tile_start, n_tiles_dev);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return scan_u32(tile_start, tile_start, n, nullptr, scan_scratch, err, stream);
}

// Largest grid of 1024-thread blocks one dispatch takes (2^32 work-items),
// in whole rounds over the 8 XCDs.
constexpr uint64_t kMaxFNTBlocks = (0xffffffffull / kFNT) / kXcds * kXcds;

// One block per tile, up to the dispatch limit (the kernels loop beyond it).
static uint32_t exact_grid(uint32_t n_tiles) {
  return (uint32_t)std::min<uint64_t>(((uint64_t)n_tiles + kXcds - 1) / kXcds * kXcds, kMaxFNTBlocks);
}

uint32_t join_fused_grid(uint32_t parts, uint64_t nR, uint64_t nS, uint64_t tiles_est, int cus) {
  // one block per partition that can hold a tile (the common one tile per
  // partition; a tile needs an R and an S tuple, so at most min(|R|, |S|)
  // partitions have one), at least two blocks per CU, never more than the
  // estimated tile count, and within the dispatch limit of 2^32 work-items
  uint64_t g = std::min<uint64_t>(parts, std::min(nR, nS));
  g = std::max<uint64_t>(g, 2ull * (uint64_t)cus);
  g = std::min<uint64_t>(g, std::max<uint64_t>(tiles_est, 1));
  g = (g + kXcds - 1) / kXcds * kXcds;
  return (uint32_t)std::min(g, kMaxFNTBlocks);
}

hipError_t join_fused(uint32_t parts, uint32_t s_span, uint32_t cap, uint32_t grid, const uint64_t *n_tiles_dev,
                      const eo_tuple *R, const uint32_t *r_start, const uint32_t *r_end, const eo_tuple *S,
                      const uint32_t *s_start, const uint32_t *s_end, const uint32_t *tile_start, eo_pair *out,
                      uint64_t out_cap, uint64_t *out_cursor, bool wide, uint32_t *matched, uint32_t *err,
                      hipStream_t stream, bool swapped) {
  if (grid == 0) return hipSuccess;
  const uint2 *vR = reinterpret_cast<const uint2 *>(R), *vS = reinterpret_cast<const uint2 *>(S);
  uint2 *vout = reinterpret_cast<uint2 *>(out);
#define EO_FUSED(C)                                                                                                \
  EO_TIMED("probe", stream,                                                                                        \
           hipLaunchKernelGGL(k_join_fused<tile::C>, dim3(grid), dim3(kFNT), 0, stream, vR, r_start, r_end, vS,     \
                              s_start, s_end, tile_start, parts, s_span, vout, out_cap, out_cursor, (int)wide,     \
                              matched, n_tiles_dev, err, (int)swapped))
  if (cap == (uint32_t)tile::ProbeSmall::Cap) EO_FUSED(ProbeSmall);
  else if (cap == (uint32_t)tile::ProbeBig::Cap) EO_FUSED(ProbeBig);
  else return hipErrorInvalidValue;
#undef EO_FUSED
  return hipGetLastError();
}

hipError_t join_outer(uint32_t parts, uint32_t s_span, uint32_t cap, uint32_t grid, const uint64_t *n_tiles_dev,
                      const eo_tuple *R, const uint32_t *r_start, const uint32_t *r_end, const eo_tuple *S,
                      const uint32_t *s_start, const uint32_t *s_end, const uint32_t *tile_start, eo_pair *out,
                      uint64_t out_cap, uint64_t *out_cursor, bool wide, uint64_t s_rows, uint32_t *words, uint32_t *err,
                      hipStream_t stream) {
  if (grid == 0) return hipSuccess;
  const uint2 *vR = reinterpret_cast<const uint2 *>(R), *vS = reinterpret_cast<const uint2 *>(S);
  uint2 *vout = reinterpret_cast<uint2 *>(out);
  uint32_t *done = words + matched_words(s_rows);
#define EO_OUTER(C)                                                                                                \
  EO_TIMED("probe", stream,                                                                                        \
           hipLaunchKernelGGL(k_join_outer<tile::C>, dim3(grid), dim3(kFNT), 0, stream, vR, r_start, r_end, vS,     \
                              s_start, s_end, tile_start, parts, s_span, vout, out_cap, out_cursor, (int)wide,     \
                              words, done, n_tiles_dev, err))
  if (cap == (uint32_t)tile::ProbeSmall::Cap) EO_OUTER(ProbeSmall);
  else if (cap == (uint32_t)tile::ProbeBig::Cap) EO_OUTER(ProbeBig);
  else return hipErrorInvalidValue;
#undef EO_OUTER
  return hipGetLastError();
}

template <typename C>
static hipError_t launch_direct(const DirectPlan &d, const uint2 *R, uint64_t nR, const uint2 *S, uint64_t nS,
                                uint2 *out, uint64_t out_cap, uint64_t *cursor, bool wide, uint32_t *matched,
                                bool outer, bool swapped, const char *name, hipStream_t stream) {
  const uint64_t grid = (uint64_t)d.chunks * d.spans;
  if (grid > 0xffffffffull / C::NT) return hipErrorInvalidValue;  // 2^32 work-items a dispatch
  if (outer && !matched && out)
    EO_TIMED(name, stream,
             hipLaunchKernelGGL((k_join_direct_outer<C, true>), dim3((uint32_t)grid), dim3(C::NT), 0, stream, R,
                                (uint32_t)nR, S, (uint32_t)nS, d.span, out, out_cap, cursor, (int)wide));
  else if (outer && !matched)
    EO_TIMED(name, stream,
             hipLaunchKernelGGL((k_join_direct_outer<C, false>), dim3((uint32_t)grid), dim3(C::NT), 0, stream, R,
                                (uint32_t)nR, S, (uint32_t)nS, d.span, nullptr, 0ull, cursor, 0));
  else if (out)
    EO_TIMED(name, stream,
             hipLaunchKernelGGL((k_join_direct<C, true>), dim3((uint32_t)grid), dim3(C::NT), 0, stream, R, nR, S, nS,
                                d.chunk, d.chunks, d.span, out, out_cap, cursor, (int)wide, matched, (int)swapped));
  else
    EO_TIMED(name, stream,
             hipLaunchKernelGGL((k_join_direct<C, false>), dim3((uint32_t)grid), dim3(C::NT), 0, stream, R, nR, S, nS,
                                d.chunk, d.chunks, d.span, nullptr, 0ull, cursor, 0, matched, 0));
  return hipGetLastError();
}

hipError_t join_direct(const DirectPlan &d, const eo_tuple *R, uint64_t nR, const eo_tuple *S, uint64_t nS,
                       eo_pair *out, uint64_t out_cap, uint64_t *out_cursor, bool wide, uint32_t *outer,
                       bool swapped, const char *name, hipStream_t stream) {
  if (nS == 0 || (nR == 0 && !outer)) return hipSuccess;
  const uint2 *vR = reinterpret_cast<const uint2 *>(R), *vS = reinterpret_cast<const uint2 *>(S);
  uint2 *vout = reinterpret_cast<uint2 *>(out);
  // several R chunks: all tiles beside each other, the null rows from the
  // matches they marked
  uint32_t *matched = outer && d.chunks > 1 ? outer : nullptr;
  hipError_t e = matched ? fill_u32(matched, 0u, matched_words(nS), stream) : hipSuccess;
  if (e != hipSuccess) return e;
#define EO_DIRECT(C) \
  launch_direct<tile::C>(d, vR, nR, vS, nS, vout, out_cap, out_cursor, wide, matched, outer, swapped, name, stream)
  switch (d.table) {
    case kFusedTableFull: e = EO_DIRECT(ProbeBig); break;
    case kFusedTableHalf: e = EO_DIRECT(ProbeSmall); break;
    case kFusedTableQuarter: e = EO_DIRECT(ProbeQuarter); break;
    default: return hipErrorInvalidValue;
  }
#undef EO_DIRECT
  if (e == hipSuccess && matched) e = emit_unmatched(S, nS, matched, out_cursor, out, out_cap, wide, stream);
  return e;
}

hipError_t span_count(uint32_t parts, uint32_t s_span, uint32_t cap, uint32_t n_tiles, const uint64_t *n_tiles_dev,
                      const eo_tuple *R, const uint32_t *r_start, const eo_tuple *S, const uint32_t *s_start,
                      const uint32_t *tile_start, uint32_t *matched, uint64_t *tile_count, hipStream_t stream) {
  if (n_tiles == 0) return hipSuccess;
  const uint32_t grid = exact_grid(n_tiles);
  const uint2 *vR = reinterpret_cast<const uint2 *>(R), *vS = reinterpret_cast<const uint2 *>(S);
  if (cap == (uint32_t)tile::ProbeSmall::Cap)
    EO_TIMED("probe_count", stream,
             hipLaunchKernelGGL(k_span_count<tile::ProbeSmall>, dim3(grid), dim3(kFNT), 0, stream, vR, r_start, vS,
                                s_start, tile_start, parts, s_span, tile_count, n_tiles, matched, n_tiles_dev));
  else if (cap == (uint32_t)tile::ProbeBig::Cap)
    EO_TIMED("probe_count", stream,
             hipLaunchKernelGGL(k_span_count<tile::ProbeBig>, dim3(grid), dim3(kFNT), 0, stream, vR, r_start, vS,
                                s_start, tile_start, parts, s_span, tile_count, n_tiles, matched, n_tiles_dev));
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t span_write(uint32_t parts, uint32_t s_span, uint32_t cap, uint32_t n_tiles, const eo_tuple *R,
                      const uint32_t *r_start, const eo_tuple *S, const uint32_t *s_start, const uint32_t *tile_start,
                      const uint64_t *tile_off, eo_pair *out, uint64_t out_cap, bool wide, hipStream_t stream) {
  if (n_tiles == 0) return hipSuccess;
  const uint32_t grid = exact_grid(n_tiles);
  const uint2 *vR = reinterpret_cast<const uint2 *>(R), *vS = reinterpret_cast<const uint2 *>(S);
  uint2 *vout = reinterpret_cast<uint2 *>(out);
  if (cap == (uint32_t)tile::ProbeSmall::Cap)
    EO_TIMED("probe_write", stream,
             hipLaunchKernelGGL(k_span_write<tile::ProbeSmall>, dim3(grid), dim3(kFNT), 0, stream, vR, r_start, vS,
                                s_start, tile_start, parts, s_span, tile_off, vout, out_cap, (int)wide));
  else if (cap == (uint32_t)tile::ProbeBig::Cap)
    EO_TIMED("probe_write", stream,
             hipLaunchKernelGGL(k_span_write<tile::ProbeBig>, dim3(grid), dim3(kFNT), 0, stream, vR, r_start, vS,
                                s_start, tile_start, parts, s_span, tile_off, vout, out_cap, (int)wide));
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

namespace {

// Left outer join: one row (null R side) per S tuple whose bit in `matched`
// is clear.  Each workgroup (256 words = 8192 positions) reserves its rows
// from *cursor with one atomic, or, with block_off, writes them at
// base + block_off[workgroup] (S order: deterministic).  out == NULL: only
// counts.
__global__ __launch_bounds__(256) void k_emit_unmatched(const uint2 *__restrict__ S, uint64_t n,
                                                        const uint32_t *__restrict__ matched, uint64_t *cursor,
                                                        const uint64_t *__restrict__ block_off, uint64_t base,
                                                        uint2 *__restrict__ out, uint64_t out_cap, int wide) {
  __shared__ uint64_t red[256 / kWave + 1];
  __shared__ uint64_t base_sh;
  const uint64_t wd = (uint64_t)blockIdx.x * 256 + threadIdx.x;  // one 32-position word per thread
  uint32_t unm = 0;
  if (wd * 32 < n) {
    const uint64_t left = n - wd * 32;
    const uint32_t valid = left >= 32 ? ~0u : ((1u << left) - 1u);
    unm = ~matched[wd] & valid;
  }
  uint64_t tot;
  const uint64_t excl = block_excl_scan<256, uint64_t>((uint64_t)__popc(unm), red, &tot);
  if (threadIdx.x == 0) {
    if (block_off) base_sh = base + block_off[blockIdx.x];
    else base_sh = tot ? atomic_add_agent(cursor, tot) : 0ull;
  }
  __syncthreads();
  if (!out) return;
  uint64_t pos = base_sh + excl;
  while (unm) {
    const uint32_t b = (uint32_t)__ffs(unm) - 1u;
    unm &= unm - 1u;
    const uint2 t = S[wd * 32 + b];
    if (pos < out_cap) emit_null(out, pos, t.y, t.x, wide != 0);
    ++pos;
  }
}

// Unmatched S positions per 256-word block (the counts k_emit_unmatched's
// deterministic mode scans into block offsets).
__global__ __launch_bounds__(256) void k_count_unmatched(uint64_t n, const uint32_t *__restrict__ matched,
                                                         uint64_t *__restrict__ block_cnt) {
  __shared__ uint64_t red[256 / kWave + 1];
  const uint64_t wd = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  uint32_t unm = 0;
  if (wd * 32 < n) {
    const uint64_t left = n - wd * 32;
    const uint32_t valid = left >= 32 ? ~0u : ((1u << left) - 1u);
    unm = ~matched[wd] & valid;
  }
  const uint64_t tot = block_sum<256, uint64_t>((uint64_t)__popc(unm), red);
  if (threadIdx.x == 0) block_cnt[blockIdx.x] = tot;
}

}  // namespace

size_t matched_words(uint64_t n) { return (n + 31) / 32; }

uint64_t unmatched_blocks(uint64_t n) { return (matched_words(n) + 255) / 256; }

hipError_t count_unmatched(uint64_t n, const uint32_t *matched, uint64_t *block_cnt, hipStream_t stream) {
  const uint64_t blocks = unmatched_blocks(n);
  if (blocks == 0) return hipSuccess;
  if (blocks >= (1ull << 31)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_count_unmatched, dim3((uint32_t)blocks), dim3(256), 0, stream, n, matched, block_cnt);
  return hipGetLastError();
}

hipError_t emit_unmatched_at(const eo_tuple *S, uint64_t n, const uint32_t *matched, const uint64_t *block_off,
                             uint64_t base, eo_pair *out, uint64_t out_cap, bool wide, hipStream_t stream) {
  const uint64_t blocks = unmatched_blocks(n);
  if (blocks == 0) return hipSuccess;
  if (blocks >= (1ull << 31)) return hipErrorInvalidValue;
  EO_TIMED("outer_rows", stream,
           hipLaunchKernelGGL(k_emit_unmatched, dim3((uint32_t)blocks), dim3(256), 0, stream,
                              reinterpret_cast<const uint2 *>(S), n, matched, nullptr, block_off, base,
                              reinterpret_cast<uint2 *>(out), out_cap, (int)wide));
  return hipGetLastError();
}

hipError_t emit_unmatched(const eo_tuple *S, uint64_t n, const uint32_t *matched, uint64_t *cursor, eo_pair *out,
                          uint64_t out_cap, bool wide, hipStream_t stream) {
  const uint64_t words = matched_words(n);
  if (words == 0) return hipSuccess;
  const uint64_t blocks = (words + 255) / 256;
  if (blocks >= (1ull << 31)) return hipErrorInvalidValue;
  EO_TIMED("outer_rows", stream,
           hipLaunchKernelGGL(k_emit_unmatched, dim3((uint32_t)blocks), dim3(256), 0, stream,
                              reinterpret_cast<const uint2 *>(S), n, matched, cursor, nullptr, 0ull,
                              reinterpret_cast<uint2 *>(out), out_cap, (int)wide));
  return hipGetLastError();
}

}  // namespace eo
