// Block nested-loop equi-join in the deterministic order, and the distance
// join.  (The default order's block nested-loop join looks its inner blocks up
// in LDS hash tables: join_direct in hashjoin.hip, 2^18 x 2^18 tuples in
// 0.05 ms where comparing every pair, at 0.88 of the compare loop's rate, took
// 3.23 ms.)
//
// The reference (joins/blockJoin_gpu/main_street/join_gpu.cu:28-118) holds
// 512 R tuples in shared memory per block and one S tuple per thread, writes
// one count per (thread, R slice) — 2^27 counts for a 2^18 x 2^18 tile — and
// repeats every compare in the write kernel.  Here a workgroup of 4 waves
// keeps an R tile of 4096 keys in LDS and 8 S keys per lane in VGPRs
// (a 2048-tuple S tile), and reads R keys from LDS four at a time with one
// wave-uniform (broadcast) load.  Each (R key, S register) compare is one
// VALU compare whose 64-lane ballot is OR-ed into a scalar accumulator; only
// a group of 8 R keys whose accumulator shows a hit is recounted exactly.
// Counts are kept per wave, so the write pass (same loop, same order) writes
// every pair at its wave's scanned offset in a deterministic order.
#include <algorithm>

#include "device.hpp"
#include "kernels.hpp"

namespace eo {
namespace {

constexpr int kNljNT = 256;
constexpr int kNljNW = kNljNT / kWave;
constexpr int kNljK = 8;                     // S keys per lane
constexpr int kNljSTile = kNljNT * kNljK;    // 2048
constexpr int kNljRTile = 4096;
constexpr int kNljGroup = 8;                 // R keys per OR-accumulated group

struct SRegs {
  int32_t key[kNljK];
  int32_t pay[kNljK];
  uint64_t valid[kNljK];  // ballot of lanes holding a real S tuple in register k
};

__device__ __forceinline__ void load_s(const uint2 *__restrict__ S, uint64_t nS, uint64_t s0, SRegs &sr,
                                       bool need_pay) {
  const int w = threadIdx.x / kWave, lane = lane_id();
#pragma unroll
  for (int k = 0; k < kNljK; ++k) {
    // wave w owns S[s0 + w*64*K, +64*K); register k holds element k*64 + lane of it
    const uint64_t i = s0 + (uint64_t)w * kWave * kNljK + (uint64_t)k * kWave + lane;
    const bool ok = i < nS;
    uint2 t = ok ? S[i] : make_uint2(0u, 0u);
    sr.key[k] = (int32_t)t.x;
    sr.pay[k] = need_pay ? (int32_t)t.y : 0;
    sr.valid[k] = __ballot(ok);
  }
}

// matched (count pass, optional): bitmap over S positions; this wave's S
// register k covers positions s_wave + k*64 + lane.
template <bool WRITE>
__device__ __forceinline__ void nlj_tile(const int32_t *rkey, const int32_t *rpay, uint32_t rn, const SRegs &sr,
                                         uint64_t *count, uint64_t base, uint2 *out, uint64_t out_cap, bool wide,
                                         uint32_t *matched = nullptr, uint64_t s_wave = 0) {
  const uint64_t lt = lanemask_lt();
  uint64_t running = 0;
  uint64_t hitk[kNljK];
#pragma unroll
  for (int k = 0; k < kNljK; ++k) hitk[k] = 0;
  uint32_t g = 0;
  for (; g + kNljGroup <= rn; g += kNljGroup) {
    int32_t rk[kNljGroup];
    const int4 *q = reinterpret_cast<const int4 *>(rkey + g);
    const int4 a = q[0], b = q[1];
    rk[0] = a.x; rk[1] = a.y; rk[2] = a.z; rk[3] = a.w;
    rk[4] = b.x; rk[5] = b.y; rk[6] = b.z; rk[7] = b.w;
    uint64_t acc = 0;
#pragma unroll
    for (int q2 = 0; q2 < kNljGroup; ++q2)
#pragma unroll
      for (int k = 0; k < kNljK; ++k) acc |= __ballot(sr.key[k] == rk[q2]);
    if (acc) {
#pragma unroll
      for (int q2 = 0; q2 < kNljGroup; ++q2) rk[q2] = opaque(rk[q2]);  // recompute, do not keep the ballots
#pragma unroll
      for (int q2 = 0; q2 < kNljGroup; ++q2)
#pragma unroll
        for (int k = 0; k < kNljK; ++k) {
          const uint64_t m = __ballot(sr.key[k] == rk[q2]) & sr.valid[k];
          hitk[k] |= m;
          if (m) {
            if (WRITE && sr.key[k] == rk[q2] && ((sr.valid[k] >> lane_id()) & 1)) {
              const uint64_t pos = base + running + __popcll(m & lt);
              if (pos < out_cap) emit_pair(out, pos, (uint32_t)rpay[g + q2], (uint32_t)sr.pay[k], (uint32_t)rk[q2], wide);
            }
            running += __popcll(m);
          }
        }
    }
  }
  for (; g < rn; ++g) {  // tail of the R tile
    const int32_t r = rkey[g];
#pragma unroll
    for (int k = 0; k < kNljK; ++k) {
      const uint64_t m = __ballot(sr.key[k] == r) & sr.valid[k];
      hitk[k] |= m;
      if (m) {
        if (WRITE && sr.key[k] == r && ((sr.valid[k] >> lane_id()) & 1)) {
          const uint64_t pos = base + running + __popcll(m & lt);
          if (pos < out_cap) emit_pair(out, pos, (uint32_t)rpay[g], (uint32_t)sr.pay[k], (uint32_t)r, wide);
        }
        running += __popcll(m);
      }
    }
  }
  if (!WRITE && lane_id() == 0) *count = running;
  if (!WRITE && matched) {
#pragma unroll
    for (int k = 0; k < kNljK; ++k) mark_bits(matched, s_wave + (uint64_t)k * kWave, hitk[k]);
  }
}

template <bool WRITE>
__global__ __launch_bounds__(kNljNT) void k_nlj(const uint2 *__restrict__ R, uint64_t nR, const uint2 *__restrict__ S,
                                                uint64_t nS, uint32_t s_tiles, uint64_t *wave_count,
                                                const uint64_t *__restrict__ wave_off, uint2 *__restrict__ out,
                                                uint64_t out_cap, int wide, uint32_t *matched) {
  __shared__ __attribute__((aligned(16))) int32_t rkey[kNljRTile];
  __shared__ int32_t rpay[WRITE ? kNljRTile : 1];
  const uint32_t b = blockIdx.x;
  const uint32_t st = b % s_tiles, rt = b / s_tiles;
  const uint64_t r0 = (uint64_t)rt * kNljRTile;
  const uint32_t rn = (uint32_t)std::min<uint64_t>(kNljRTile, nR - r0);
  for (uint32_t i = threadIdx.x; i < rn; i += kNljNT) {
    const uint2 t = R[r0 + i];
    rkey[i] = (int32_t)t.x;
    if (WRITE) rpay[i] = (int32_t)t.y;
  }
  SRegs sr;
  load_s(S, nS, (uint64_t)st * kNljSTile, sr, WRITE);
  __syncthreads();
  const uint64_t slot = (uint64_t)b * kNljNW + threadIdx.x / kWave;
  if (WRITE)
    nlj_tile<true>(rkey, rpay, rn, sr, nullptr, wave_off[slot], out, out_cap, wide != 0);
  else
    nlj_tile<false>(rkey, rpay, rn, sr, wave_count + slot, 0, nullptr, 0, false, matched,
                    (uint64_t)st * kNljSTile + (uint64_t)(threadIdx.x / kWave) * kWave * kNljK);
}

// ---- distance predicate (FP64) ---------------------------------------------------
// The multi-attribute predicate of joins/CPU_JOIN/3d_cpu/nestLoopJoin.cc:73-81:
// a pair matches when (r0-s0)^2 + (r1-s1)^2 + (r2-s2)^2 < d2, accumulated in
// that order with every subtraction, product and sum rounded on its own
// (__dsub_rn / __dmul_rn / __dadd_rn: no fused multiply-add), which makes each
// decision bit-identical to the reference's unfused x86-64 arithmetic.  One
// fused pass: an R tile (up to 1024 points) in LDS, 8 S points per lane, OR-accumulated ballots per group of 8 R points,
// per-wave hit-group list, one output reservation per wave.
//
// The exact predicate takes 9 FP64 instructions per pair.  Every pair first
// passes a filter of 4 (three FMAs and a compare) that never rejects a match:
//   |r|^2 - 2 r.s < d2 - |s|^2,   both sides widened by kDistSlack of the terms
// and only the S registers of a group in which it holds for some pair evaluate
// the predicate (on coordinates read again, so that the loop keeps only the
// filter's registers).  8 S points per lane, because the R point that they
// share is a 32-byte LDS broadcast: with 4 the CU's LDS port is as busy as its
// four FP64 pipes.
// Rounding: with u = 2^-53 the filter's left side is off by at most 3u |r|^2
// (the squares' sum) + 3u (|r|^2 + 2 |r||s|) (the FMAs) <= 9u (|r|^2 + |s|^2),
// the right side by 4u (|s|^2 + d2), and the reference's own sum is within 8u
// of the real squared distance, at most 8u d2 at the threshold: together
// under 16u (|r|^2 + |s|^2 + d2); kDistSlack is 128u.  A point whose squared
// length is not below 2^1000 (infinities and NaN included) makes every pair
// of it pass.  FP64 issue bound (0.89 of the VALU's cycles): 2^17 x 2^17 points
// in 3.69 ms with the exact predicate on every pair, 2.27 ms with the filter
// (4 S points per lane 2.35, a running minimum instead of the compares 2.33).
constexpr int kDistNT = 256;
constexpr int kDistNW = kDistNT / kWave;
constexpr int kDistK = 8;
constexpr int kDistSTile = kDistNT * kDistK;  // 2048
constexpr int kDistRTile = 1024;
constexpr int kDistGroup = 8;
constexpr double kDistSlack = 0x1p-46;
constexpr double kDistHuge = 0x1p1000;
constexpr double kDistTiny = 0x1p-1060;  // covers squares that round to a multiple of 2^-1074

struct Point3 {
  int32_t id, pad;
  double v[3];
};

__device__ __forceinline__ bool dist_lt(double sx, double sy, double sz, double rx, double ry, double rz, double d2) {
  const double t0 = __dsub_rn(rx, sx), t1 = __dsub_rn(ry, sy), t2 = __dsub_rn(rz, sz);
  double acc = __dmul_rn(t0, t0);
  acc = __dadd_rn(acc, __dmul_rn(t1, t1));
  acc = __dadd_rn(acc, __dmul_rn(t2, t2));
  return acc < d2;
}

// An R point as the filter reads it: c = |r|^2 lowered by the slack, or -inf.
struct alignas(16) DistPoint {
  double x, y, z, c;
};

template <bool WRITE>
__global__ __launch_bounds__(kDistNT) __attribute__((amdgpu_waves_per_eu(4))) void k_nlj_dist(const Point3 *__restrict__ R, uint64_t nR,
                                                      const Point3 *__restrict__ S, uint64_t nS, uint32_t s_tiles,
                                                      uint32_t r_tile, double d2, uint64_t *cursor,
                                                      uint2 *__restrict__ out, uint64_t out_cap) {
  __shared__ DistPoint rp[kDistRTile];
  __shared__ uint16_t hits[WRITE ? kDistNW : 1][WRITE ? kDistRTile / kDistGroup : 1];
  const uint32_t b = blockIdx.x;
  const uint32_t st = b % s_tiles, rt = b / s_tiles;
  const uint64_t r0 = (uint64_t)rt * r_tile;
  const uint32_t rn = (uint32_t)std::min<uint64_t>(r_tile, nR - r0);
  for (uint32_t i = threadIdx.x; i < rn; i += kDistNT) {
    const Point3 &p = R[r0 + i];
    const double x = p.v[0], y = p.v[1], z = p.v[2], q = x * x + y * y + z * z;
    rp[i] = DistPoint{x, y, z, q < kDistHuge ? q - kDistSlack * q : -__builtin_inf()};
  }
  // the last group is filled with points that pass no pair
  for (uint32_t i = rn + threadIdx.x; i < (rn + kDistGroup - 1) / kDistGroup * kDistGroup; i += kDistNT)
    rp[i] = DistPoint{0.0, 0.0, 0.0, __builtin_inf()};
  const int w = threadIdx.x / kWave;
  const int lane = lane_id();
  const uint64_t s0 = (uint64_t)st * kDistSTile + (uint64_t)w * kWave * kDistK;
  double mx[kDistK], my[kDistK], mz[kDistK], thr[kDistK];
#pragma unroll
  for (int k = 0; k < kDistK; ++k) {
    const uint64_t i = s0 + (uint64_t)k * kWave + lane;
    const bool ok = i < nS;
    const double x = ok ? S[i].v[0] : 0.0, y = ok ? S[i].v[1] : 0.0, z = ok ? S[i].v[2] : 0.0;
    const double q = x * x + y * y + z * z;
    const bool h = !(q < kDistHuge);
    mx[k] = h ? 0.0 : -2.0 * x;
    my[k] = h ? 0.0 : -2.0 * y;
    mz[k] = h ? 0.0 : -2.0 * z;
    // (a lane past the end of S passes nothing but huge R points)
    thr[k] = h ? __builtin_inf() : ok ? d2 - q + (kDistSlack * (q + d2) + kDistTiny) : -__builtin_inf();
  }
  __syncthreads();
  const uint64_t lt = lanemask_lt();
  const uint32_t ngroups = (rn + kDistGroup - 1) / kDistGroup;
  uint64_t total = 0;
  uint32_t nh = 0;
  for (uint32_t gi = 0; gi < ngroups; ++gi) {
    const uint32_t g = gi * kDistGroup;
    const uint32_t gn = rn - g < (uint32_t)kDistGroup ? rn - g : (uint32_t)kDistGroup;  // wave-uniform
    uint64_t acc[kDistK] = {};
#pragma unroll
    for (int q = 0; q < kDistGroup; ++q) {
      const DistPoint p = rp[g + q];
      double v[kDistK];  // coordinate by coordinate: kDistK independent FMAs in a row
#pragma unroll
      for (int k = 0; k < kDistK; ++k) v[k] = __builtin_fma(mz[k], p.z, p.c);
#pragma unroll
      for (int k = 0; k < kDistK; ++k) v[k] = __builtin_fma(my[k], p.y, v[k]);
#pragma unroll
      for (int k = 0; k < kDistK; ++k) v[k] = __builtin_fma(mx[k], p.x, v[k]);
#pragma unroll
      for (int k = 0; k < kDistK; ++k) acc[k] |= __ballot(!(v[k] >= thr[k]));  // (not "less": a NaN passes)
    }
    uint32_t pass = 0;  // S registers with a pair that passes
#pragma unroll
    for (int k = 0; k < kDistK; ++k) pass |= acc[k] ? 1u << k : 0u;
    if (!pass) continue;
    uint64_t cnt = 0;
    uint32_t hit = 0;
    for (uint32_t left = pass; left; left &= left - 1) {  // wave-uniform
      const uint32_t k = (uint32_t)__ffs(left) - 1u;
      const uint64_t i = s0 + (uint64_t)k * kWave + lane;
      const Point3 &sp = S[min(i, nS - 1)];
      const double x = sp.v[0], y = sp.v[1], z = sp.v[2];
      uint64_t c = 0;
      for (uint32_t q = 0; q < gn; ++q) {
        const DistPoint p = rp[g + q];
        c += __popcll(__ballot(i < nS && dist_lt(x, y, z, p.x, p.y, p.z, d2)));
      }
      cnt += c;
      hit |= c ? 1u << k : 0u;
    }
    if (cnt) {
      total += cnt;
      if (WRITE) {
        if (lane == 0) hits[w][nh] = (uint16_t)(gi << 8 | hit);
        ++nh;
      }
    }
  }
  uint64_t base = 0;
  if (total) {
    if (lane == 0) base = atomic_add_agent(cursor, total);
    base = read_lane(base, 0);
  }
  if (!WRITE || total == 0) return;
  uint64_t running = 0;
  for (uint32_t h = 0; h < nh; ++h) {
    const uint32_t rec = (uint32_t)__builtin_amdgcn_readfirstlane((int)hits[w][h]);
    const uint32_t g = (rec >> 8) * kDistGroup;
    const uint32_t gn = rn - g < (uint32_t)kDistGroup ? rn - g : (uint32_t)kDistGroup;
    for (uint32_t left = rec & 0xffu; left; left &= left - 1) {
      const uint32_t k = (uint32_t)__ffs(left) - 1u;
      const uint64_t i = s0 + (uint64_t)k * kWave + lane;
      const Point3 &sp = S[min(i, nS - 1)];
      const double x = sp.v[0], y = sp.v[1], z = sp.v[2];
      for (uint32_t q = 0; q < gn; ++q) {
        const DistPoint p = rp[g + q];
        const bool eq = i < nS && dist_lt(x, y, z, p.x, p.y, p.z, d2);
        const uint64_t m = __ballot(eq);
        if (m) {
          if (eq) {
            const uint64_t pos = base + running + __popcll(m & lt);
            if (pos < out_cap) out[pos] = make_uint2((uint32_t)R[r0 + g + q].id, (uint32_t)sp.id);
          }
          running += __popcll(m);
        }
      }
    }
  }
}

static_assert(kDistK <= 8 && kDistRTile / kDistGroup <= 256, "a hit record: group << 8 | S registers");

}  // namespace

NljPlan plan_nlj(uint64_t nR, uint64_t nS) {
  NljPlan p{};
  p.nR = nR;
  p.nS = nS;
  p.r_tile = kNljRTile;
  p.s_tile = kNljSTile;
  p.r_tiles = (uint32_t)((nR + kNljRTile - 1) / kNljRTile);
  p.s_tiles = (uint32_t)((nS + kNljSTile - 1) / kNljSTile);
  return p;
}

uint64_t nlj_count_slots(const NljPlan &p) { return (uint64_t)p.r_tiles * p.s_tiles * kNljNW; }

hipError_t nlj_count(const NljPlan &p, const eo_tuple *R, const eo_tuple *S, uint64_t *wave_count,
                     hipStream_t stream, uint32_t *matched) {
  const uint64_t grid = (uint64_t)p.r_tiles * p.s_tiles;
  if (grid == 0) return hipSuccess;
  if (grid >= (1ull << 31)) return hipErrorInvalidValue;
  EO_TIMED("nlj_count", stream, hipLaunchKernelGGL(k_nlj<false>, dim3((uint32_t)grid), dim3(kNljNT), 0, stream, reinterpret_cast<const uint2 *>(R),
                     p.nR, reinterpret_cast<const uint2 *>(S), p.nS, p.s_tiles, wave_count, nullptr, nullptr, 0, 0,
                     matched));
  return hipGetLastError();
}

hipError_t nlj_write(const NljPlan &p, const eo_tuple *R, const eo_tuple *S, const uint64_t *wave_off, eo_pair *out,
                     uint64_t out_cap, bool wide, hipStream_t stream) {
  const uint64_t grid = (uint64_t)p.r_tiles * p.s_tiles;
  if (grid == 0) return hipSuccess;
  if (grid >= (1ull << 31)) return hipErrorInvalidValue;
  EO_TIMED("nlj_write", stream, hipLaunchKernelGGL(k_nlj<true>, dim3((uint32_t)grid), dim3(kNljNT), 0, stream, reinterpret_cast<const uint2 *>(R),
                     p.nR, reinterpret_cast<const uint2 *>(S), p.nS, p.s_tiles, nullptr, wave_off,
                     reinterpret_cast<uint2 *>(out), out_cap, (int)wide, nullptr));
  return hipGetLastError();
}

// R tuples per tile: `full`, or fewer (whole groups, at least 64) while the
// grid has less than four workgroups of 256 threads per CU: a small join is
// bound by the length of one workgroup's loop (2^12 x 2^12 points in 16 tile
// pairs of 1024 x 1024: 279 us; in 128 of 64 x 2048, with the filter: 58 us).
static uint32_t nlj_r_tile(uint64_t nR, uint64_t s_tiles, uint32_t full, uint32_t group, int cus) {
  const uint64_t want = 4ull * (uint64_t)std::max(cus, 8) / std::max<uint64_t>(s_tiles, 1);  // R tiles
  uint64_t t = want > 1 ? (nR + want - 1) / want : full;
  t = (t + group - 1) / group * group;
  return (uint32_t)std::min<uint64_t>(std::max<uint64_t>(t, 64), full);
}

hipError_t nlj_dist(const eo_point3 *R, uint64_t nR, const eo_point3 *S, uint64_t nS, double d2, uint64_t *cursor,
                    eo_pair *out, uint64_t out_cap, int cus, hipStream_t stream) {
  const uint64_t s_tiles = (nS + kDistSTile - 1) / kDistSTile;
  const uint32_t r_tile = nlj_r_tile(nR, s_tiles, kDistRTile, kDistGroup, cus);
  const uint64_t grid = (nR + r_tile - 1) / r_tile * s_tiles;
  if (grid == 0) return hipSuccess;
  if (grid >= (1ull << 31)) return hipErrorInvalidValue;
  const Point3 *vR = reinterpret_cast<const Point3 *>(R), *vS = reinterpret_cast<const Point3 *>(S);
  if (out)
    EO_TIMED("nlj_dist", stream,
             hipLaunchKernelGGL(k_nlj_dist<true>, dim3((uint32_t)grid), dim3(kDistNT), 0, stream, vR, nR, vS, nS,
                                (uint32_t)s_tiles, r_tile, d2, cursor, reinterpret_cast<uint2 *>(out), out_cap));
  else
    EO_TIMED("nlj_dist_count", stream,
             hipLaunchKernelGGL(k_nlj_dist<false>, dim3((uint32_t)grid), dim3(kDistNT), 0, stream, vR, nR, vS, nS,
                                (uint32_t)s_tiles, r_tile, d2, cursor, nullptr, 0));
  return hipGetLastError();
}

}  // namespace eo
