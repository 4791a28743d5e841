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
// fused pass: R tiles of up to 1024 points in LDS against the workgroup's 2048 S points in
// registers, rows reserved per workgroup.
//
// The exact predicate takes 9 FP64 instructions per pair.  Every pair first
// passes a filter that never rejects a match:
//   |r|^2 - 2 r.s + |s|^2 - d2 < 0,  lowered by a bound on the filter's error
// and only pairs that pass it evaluate the predicate, on the coordinates as
// given.  There are two filters: a workgroup takes the matrix filter up to its
// first R tile with a point outside that filter's range (none, if its S tile has
// one) and the FP64 filter from there on.
//
// Matrix filter (dist_matrix).  The sum is a contraction: coordinates about a
// common origin o (a mean of the S tile's points, subtracted in FP64) as two
// bf16 words, h = bf16(x), m = bf16(x - h), and the squared lengths as three:
//   hh' + hm' + mh' for each coordinate (9 products), c_r 1 (3), 1 t_s (3)
// 15 of the 16 products that one 32x32x16 MFMA sums per pair; a sign test of
// its 32-bit result is the filter.  Error, with N = |r - o|^2 + |s - o|^2: a
// bf16 word rounds off at most 2^-8 of its number, so hh' + hm' + mh' misses
// 3.03 2^-16 2 |x x'| per coordinate, in all 12.1 2^-18 N; 16 additions of terms
// whose magnitudes sum to 2 N + d2, each off by 2^-22 of that sum at most even
// if the unit cuts instead of rounding: 2^-18 (2 N + d2); the third words of c
// and t and the FP64 steps stay below 2^-22 (N + d2).  Together under 14.2
// 2^-18 (N + d2); kMatSlack is 16 2^-18.  (Measured over 2^24 pairs each in
// boxes of 4 to 100, near each other or not: 6.9 2^-18 (N + d2) at most; 0.04
// where the coordinates are bf16 numbers, which is what the unit's additions are
// off by.)  It is used where every N stays within 2^15 d2, so that
// the slack is 2 d2 at the corners and few pairs pass that do not match, and
// d2 is within 2^-60 .. 2^60 (no bf16 or 32-bit word overflows, and what is
// flushed to zero is far below the slack).
//
// FP64 filter (dist_fp64), else: three FMAs and a compare,
//   |r|^2 - 2 r.s < d2 - |s|^2,   both sides widened by kDistSlack of the terms
// 8 S points per lane, because the R point that they share is a 32-byte LDS
// broadcast: with 4 the CU's LDS port is as busy as its four FP64 pipes.
// Rounding: with u = 2^-53 the filter's left side is off by at most 3u |r|^2
// (the squares' sum) + 3u (|r|^2 + 2 |r||s|) (the FMAs) <= 9u (|r|^2 + |s|^2),
// the right side by 4u (|s|^2 + d2), and the reference's own sum is within 8u
// of the real squared distance, at most 8u d2 at the threshold: together
// under 16u (|r|^2 + |s|^2 + d2); kDistSlack is 128u.  A point whose squared
// length is not below 2^1000 (infinities and NaN included) makes every pair
// of it pass.
//
// 2^17 x 2^17 points: 3.69 ms with the exact predicate on every pair, 2.27 ms
// with the FP64 filter (issue bound, 0.89 of the VALU's cycles), 0.54 ms with
// the matrix filter: a SIMD's MFMAs (0.44 of its cycles) and VALU (0.62) do not
// run beside each other, so the signs cost as much as the products.  (Each MFMA
// issued before the signs of the tile before it, four tiles to a test: 0.66
// ms, registers spilled.)
constexpr int kDistNT = 256;
constexpr int kDistNW = kDistNT / kWave;
constexpr int kDistK = 8;
constexpr int kDistSTile = kDistNT * kDistK;  // 2048
constexpr int kDistRTile = 1024;                // R points in LDS at a time
constexpr int kDistRFull = 8 * kDistRTile;      // R points of a workgroup, at most: its S side is prepared once
constexpr int kDistGroup = 8;
constexpr int kMatTiles = kDistSTile / kDistNW / 32;  // 32-point S tiles per wave
constexpr int kMatList = 384;                         // rows a wave collects before it writes them
constexpr double kMatSlack = 0x1p-14;
constexpr double kMatMaxN = 0x1p14;  // squared length of a point, in units of d2
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

// Rows of one R tile in LDS with the FP64 filter.
template <bool WRITE>
__device__ __forceinline__ void dist_fp64(DistPoint *rp, uint16_t (*hits)[WRITE ? kDistRTile / kDistGroup : 1],
                                          const Point3 *__restrict__ R, uint64_t r0, uint32_t rn,
                                          const Point3 *__restrict__ S, uint64_t nS, uint32_t st, double d2,
                                          uint64_t *cursor, uint2 *__restrict__ out, uint64_t out_cap) {
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

// A number as the sum of its first two or three bf16 words (round to nearest).
struct Bf16Words {
  __bf16 h, m, l;
};
__device__ __forceinline__ Bf16Words bf16_words(double v) {
  const float f = (float)v;
  Bf16Words r;
  r.h = (__bf16)f;
  const float f1 = f - (float)r.h;
  r.m = (__bf16)f1;
  r.l = (__bf16)(f1 - (float)r.m);
  return r;
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Collected rows of a wave, (R point of the workgroup) << 11 | (S point of its
// tile), to out.
__device__ __forceinline__ void dist_flush(const uint32_t *list, uint32_t n, uint64_t base, const Point3 *__restrict__ R,
                                           uint64_t r_base, const Point3 *__restrict__ S, uint64_t s_base,
                                           uint2 *__restrict__ out, uint64_t out_cap) {
  for (uint32_t k = lane_id(); k < n; k += kWave) {
    const uint32_t e = list[k];
    if (base + k < out_cap)
      out[base + k] = make_uint2((uint32_t)R[r_base + (e >> 11)].id, (uint32_t)S[s_base + (e & 2047u)].id);
  }
}

// A workgroup: S points [2048 st, + 2048) against r_tile R points, 1024 at a
// time in LDS (as bf16 words, 32 bytes each, or as DistPoints).  A wave's 512 S
// points stay in registers as 16 MFMA operands; each 32 R points are read once
// (16 bytes per lane) for 16 MFMAs.  Per 1024 pairs one MFMA of 8 passes (32
// cycles) and 8 three-operand ORs (32 cycles of VALU) on the signs of its
// results.
template <bool WRITE>
__global__ __launch_bounds__(kDistNT) __attribute__((amdgpu_waves_per_eu(4))) void k_nlj_dist(
    const Point3 *__restrict__ R, uint64_t nR, const Point3 *__restrict__ S, uint64_t nS, uint32_t s_tiles,
    uint32_t r_tile, double d2, uint64_t *cursor, uint2 *__restrict__ out, uint64_t out_cap) {
  __shared__ DistPoint rp[kDistRTile];
  __shared__ uint16_t hits[WRITE ? kDistNW : 1][WRITE ? kDistRTile / kDistGroup : 1];
  __shared__ uint32_t list[WRITE ? kDistNW : 1][WRITE ? kMatList : 1];
  __shared__ uint32_t unfit;  // some point so far is outside the matrix filter's range
  __shared__ uint32_t wave_rows[kDistNW];
  __shared__ uint64_t wg_base;
  bf16x8 *const frag = reinterpret_cast<bf16x8 *>(rp);  // [half][point]: products 0..7 and 8..15
  static_assert(sizeof(rp) == 2 * kDistRTile * sizeof(bf16x8), "the two forms of an R tile take the same LDS");
  const uint32_t st = blockIdx.x % s_tiles, rt = blockIdx.x / s_tiles;
  const uint64_t r_base = (uint64_t)rt * r_tile, s_base = (uint64_t)st * kDistSTile;
  const uint64_t r_last = std::min<uint64_t>(nR, r_base + r_tile);
  const int w = threadIdx.x / kWave, lane = lane_id();
  const uint32_t half = lane >> 5, col = lane & 31;
  if (threadIdx.x == 0) unfit = d2 >= 0x1p-60 && d2 <= 0x1p60 ? 0u : 1u;
  // the origin: the mean of 64 points spread over the S tile (the same in
  // every wave: the same loads and sums)
  const uint64_t sn = std::min<uint64_t>(kDistSTile, nS - s_base);
  const Point3 &op = S[s_base + (uint64_t)lane * sn / kWave];
  const double ox = wave_sum<double>(op.v[0]) / kWave, oy = wave_sum<double>(op.v[1]) / kWave,
               oz = wave_sum<double>(op.v[2]) / kWave;
  const double max_n = kMatMaxN * d2;
  const __bf16 zero = (__bf16)0.0f, one = (__bf16)1.0f;
  __syncthreads();
  bf16x8 b[kMatTiles];
#pragma unroll
  for (int t = 0; t < kMatTiles; ++t) {
    const uint32_t i = (uint32_t)(w * kMatTiles + t) * 32 + col;
    const bool ok = i < sn;
    const Point3 &p = S[s_base + (ok ? i : 0u)];
    const double x = p.v[0] - ox, y = p.v[1] - oy, z = p.v[2] - oz, n = x * x + y * y + z * z;
    if (!(n <= max_n)) unfit = 1;
    const Bf16Words bx = bf16_words(-2.0 * x), by = bf16_words(-2.0 * y), bz = bf16_words(-2.0 * z);
    // (a lane past the end of S passes nothing)
    const Bf16Words bt = bf16_words(ok ? n - d2 - kMatSlack * (n + d2) : 4.0 * max_n);
    b[t] = half ? bf16x8{bz.h, one, one, one, bt.h, bt.m, bt.l, zero}
                : bf16x8{bx.h, bx.m, bx.h, by.h, by.m, by.h, bz.h, bz.m};
  }
  uint64_t total = 0;
  uint32_t nl = 0;  // rows in this wave's list
  uint64_t r0 = r_base;
  for (; r0 < r_last; r0 += kDistRTile) {
    const uint32_t rn = (uint32_t)std::min<uint64_t>(kDistRTile, r_last - r0), rows = (rn + 31) / 32 * 32;
    __syncthreads();  // the last R tile is read, every S point tested
    if (!unfit) {
      for (uint32_t i = threadIdx.x; i < rows; i += kDistNT) {
        const bool ok = i < rn;
        const Point3 &p = R[r0 + (ok ? i : 0u)];
        const double x = p.v[0] - ox, y = p.v[1] - oy, z = p.v[2] - oz, n = x * x + y * y + z * z;
        if (!(n <= max_n)) unfit = 1;
        const Bf16Words ax = bf16_words(x), ay = bf16_words(y), az = bf16_words(z);
        const Bf16Words ac = bf16_words(ok ? n - kMatSlack * n : 8.0 * max_n);  // (a row past the end: no pair)
        frag[i] = bf16x8{ax.h, ax.h, ax.m, ay.h, ay.h, ay.m, az.h, az.h};
        frag[kDistRTile + i] = bf16x8{az.m, ac.h, ac.m, ac.l, one, one, one, zero};
      }
    }
    __syncthreads();
    if (unfit) break;
    for (uint32_t g = 0; g < rows; g += 32) {
      const bf16x8 a = frag[half * kDistRTile + g + col];
#pragma unroll
      for (int t = 0; t < kMatTiles; t += 2) {
        const f32x16 c0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[t], f32x16{}, 0, 0, 0);
        const f32x16 c1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[t + 1], f32x16{}, 0, 0, 0);
        uint32_t sign = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) sign |= __float_as_uint(c0[i]);
#pragma unroll
        for (int i = 0; i < 16; ++i) sign |= __float_as_uint(c1[i]);
        if (__ballot((int32_t)sign < 0) == 0) continue;
        uint32_t cand = 0;  // bit i: result i of the first S tile, bit 16 + i: of the second
#pragma unroll
        for (int i = 0; i < 16; ++i)
          cand |= (__float_as_uint(c0[i]) >> 31) << i | (__float_as_uint(c1[i]) >> 31) << (16 + i);
        while (__ballot(cand != 0)) {
          // result i: R point (i & 3) + 8 (i >> 2 & 3) + 4 half of the 32, S point col of tile t or t + 1
          const uint32_t i = (uint32_t)__ffs(cand) - 1u;
          const uint32_t r = g + (i & 3u) + 8u * (i >> 2 & 3u) + 4u * half;
          const uint32_t sp = (uint32_t)(w * kMatTiles + t + (i >> 4 & 1u)) * 32 + col;
          bool eq = cand != 0 && r < rn && sp < sn;
          if (eq) {
            const Point3 &p = R[r0 + r], &q = S[s_base + sp];
            eq = dist_lt(q.v[0], q.v[1], q.v[2], p.v[0], p.v[1], p.v[2], d2);
          }
          cand &= cand - 1u;
          const uint64_t m = __ballot(eq);
          const uint32_t n = (uint32_t)__popcll(m);
          if (!n) continue;
          total += n;
          if (!WRITE) continue;
          if (eq) list[w][nl + (uint32_t)__popcll(m & lanemask_lt())] = (uint32_t)(r0 - r_base + r) << 11 | sp;
          nl += n;
          if (nl > kMatList - kWave) {
            uint64_t base = 0;
            if (lane == 0) base = atomic_add_agent(cursor, (uint64_t)nl);
            dist_flush(list[w], nl, read_lane(base, 0), R, r_base, S, s_base, out, out_cap);
            total -= nl;
            nl = 0;
          }
        }
      }
    }
  }
  for (; r0 < r_last; r0 += kDistRTile) {  // from the first R tile outside the matrix filter's range on
    __syncthreads();
    dist_fp64<WRITE>(rp, hits, R, r0, (uint32_t)std::min<uint64_t>(kDistRTile, r_last - r0), S, nS, st, d2, cursor,
                     out, out_cap);
  }
  // the rows not yet counted, with one reservation per workgroup
  if (lane == 0) wave_rows[w] = (uint32_t)total;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t n = 0;
    for (int v = 0; v < kDistNW; ++v) n += wave_rows[v];
    wg_base = n ? atomic_add_agent(cursor, n) : 0ull;
  }
  if (!WRITE) return;
  __syncthreads();
  uint64_t base = wg_base;
  for (int v = 0; v < w; ++v) base += wave_rows[v];
  dist_flush(list[w], nl, base, R, r_base, S, s_base, out, out_cap);
}

static_assert(kDistRFull << 11 > 0 && kDistSTile == 2048, "a collected row: R point << 11 | S point");
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
// pairs of 1024 x 1024: 279 us; in 128 of 64 x 2048 58 us, with the matrix filter 25 us a call).
static uint32_t nlj_r_tile(uint64_t nR, uint64_t s_tiles, uint32_t full, uint32_t group, int cus) {
  const uint64_t want = 4ull * (uint64_t)std::max(cus, 8) / std::max<uint64_t>(s_tiles, 1);  // R tiles
  uint64_t t = want > 1 ? (nR + want - 1) / want : full;
  t = (t + group - 1) / group * group;
  return (uint32_t)std::min<uint64_t>(std::max<uint64_t>(t, 64), full);
}

hipError_t nlj_dist(const eo_point3 *R, uint64_t nR, const eo_point3 *S, uint64_t nS, double d2, uint64_t *cursor,
                    eo_pair *out, uint64_t out_cap, int cus, hipStream_t stream) {
  const uint64_t s_tiles = (nS + kDistSTile - 1) / kDistSTile;
  const uint32_t r_tile = nlj_r_tile(nR, s_tiles, kDistRFull, 32, cus);
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
