#include "plan.hpp"

#include <algorithm>
#include <cmath>

#include "kernels.hpp"

namespace eo {

namespace {
int ceil_log2(uint64_t x) {
  int b = 0;
  while ((1ull << b) < x) ++b;
  return b;
}
bool valid_cap(int c) { return c == 4096 || c == 8192 || c == 16384; }
}  // namespace

eo_status plan_hash_join(uint64_t nR, uint64_t nS, const eo_join_opts *o, HashPlan *out, int cus) {
  HashPlan p;
  const int cap_opt = o ? o->lds_tuples : 0;
  if (cap_opt != 0 && !valid_cap(cap_opt)) return EO_EINVAL;
  p.lds_cap = cap_opt ? (uint32_t)cap_opt : 16384u;

  const int bits_opt = o ? o->radix_bits : 0;
  if (bits_opt < -1 || bits_opt > kMaxJoinBits) return EO_EINVAL;
  // A join that needs two partition passes anyway takes half tables: the
  // extra radix bit lands in the second pass (which moves the same bytes),
  // and two probe workgroups per CU hide each other's barrier and atomic
  // round trips (C2, 2^27 x 2^28: probe 1.32 -> 1.08 ms, join 5.09 -> 4.93 ms;
  // deterministic order 7.35 -> 6.86 ms).
  if (!cap_opt && !bits_opt && nR > 16384 && ceil_log2((nR + 16383) / 16384) > kMaxPassBits) p.lds_cap = 8192u;
  if (bits_opt == -1) {
    p.bits = 0;
  } else if (bits_opt > 0) {
    p.bits = bits_opt;
  } else if (nR <= p.lds_cap) {
    p.bits = 0;
  } else if (!cap_opt && (nR + fused_table_tuples(p.lds_cap) - 1) / fused_table_tuples(p.lds_cap) <=
                             kUnpartitionedChunks &&
             (nR + fused_table_tuples(p.lds_cap) - 1) / fused_table_tuples(p.lds_cap) * nS <=
                 kUnpartitionedSReads) {
    // A build side of a few LDS tables beside a small S: no partitioning;
    // every S tile streams past each R chunk (S read up to four times), which
    // costs less than partitioning both sides (measured: 2^16 x 2^20 0.071 ms
    // against 0.089 partitioned, 2^15 x 2^20 0.064 against 0.096; 2^17 x
    // 2^20, 8 chunks, and 2^16 x 2^22, 2^24 S reads, are faster partitioned)
    p.bits = 0;
  } else {
    // Mean R partition at most lds_cap tuples, so that each partition is one
    // LDS table (the table holds 17408: a full 16K partition plus binomial
    // spread).  Up to 2^11 digits in one pass (each digit's run per 16K-tuple
    // staging tile stays near 64 bytes, so writes coalesce); beyond that two
    // passes, high digit first.
    p.bits = ceil_log2((nR + p.lds_cap - 1) / p.lds_cap);
    if (p.bits > kMaxJoinBits) p.bits = kMaxJoinBits;
  }

  const int passes_opt = o ? o->passes : 0;
  if (passes_opt < 0 || passes_opt > 2) return EO_EINVAL;
  if (p.bits == 0) {
    p.passes = 0;
  } else if (passes_opt) {
    p.passes = passes_opt;
  } else {
    p.passes = p.bits <= kMaxPassBits ? 1 : 2;
  }
  if (p.passes == 1) {
    if (p.bits > kMaxPassBits) return EO_EINVAL;
    p.bits_pass1 = p.bits;
  } else if (p.passes == 2) {
    if (p.bits < 2 || p.bits > 2 * kMaxPassBits) return EO_EINVAL;
    p.bits_pass1 = p.bits / 2;
    p.bits_pass2 = p.bits - p.bits_pass1;
  }

  const int st_opt = o ? o->s_tile : 0;
  if (st_opt < 0) return EO_EINVAL;
  p.s_tile = st_opt ? (uint32_t)st_opt : 16384u;
  p.s_span = st_opt ? std::max<uint32_t>(8192, (uint32_t)st_opt) : plan_span(nR, nS, p.lds_cap, p.bits, nS, cus);
  *out = p;
  return EO_OK;
}

namespace {
// Time model of a probe tile in microseconds, fitted to joins of 300 to 131072
// by 4000 to 2^24 tuples on each table: a workgroup's fixed cost, per R tuple
// built, per S tuple probed; and every S batch's output reservation, an
// atomic on one word of the whole device (about 100 million a second).
// 2^16 x 2^20 unpartitioned: full tables 22 us, half 35, quarter 108; 1000 x
// 4000: 3.1, 1.8, 1.2 (each beside 18.5 of launches and the readback).
struct ProbeTable {
  uint32_t cap, batch, per_cu;  // tuples, S tuples per batch, workgroups per CU
  double fixed, build, probe;
  double tile(double r, double s) const { return fixed + build * r + probe * s; }
};
constexpr double kAtomicUs = 0.010;
constexpr uint64_t kDirectTiles = (1ull << 22) - 1;  // of up to 1024 threads each
constexpr ProbeTable kProbeTables[] = {{kFusedTableFull, 8192, 1, 2.0, 1.5e-4, 6e-4},
                                       {kFusedTableHalf, 4096, 2, 1.2, 2e-4, 1e-3},
                                       {kFusedTableQuarter, 2048, 4, 0.8, 2e-4, 7e-4}};
}  // namespace

DirectPlan plan_direct(uint64_t nR, uint64_t nS, const eo_join_opts *o, int cus, bool outer) {
  const int cap_opt = o ? o->lds_tuples : 0, span_opt = o ? o->s_tile : 0;
  const uint64_t n_cu = (uint64_t)std::max(cus, 8);
  DirectPlan best;
  for (const ProbeTable &t : kProbeTables) {
    if (cap_opt && fused_table_tuples((uint32_t)cap_opt, true) != t.cap) continue;
    DirectPlan d;
    d.table = t.cap;
    d.chunks = (uint32_t)std::max<uint64_t>(1, (nR + t.cap - 1) / t.cap);
    d.chunk = (uint32_t)std::max<uint64_t>(1, (nR + d.chunks - 1) / d.chunks);  // chunks of equal length
    d.chunks = (uint32_t)std::max<uint64_t>(1, (nR + d.chunk - 1) / d.chunk);
    const uint64_t slots = n_cu * t.per_cu, batches = std::max<uint64_t>(1, (nS + t.batch - 1) / t.batch);
    // as many S spans as fill the chip once, of whole batches
    uint64_t spans = std::min(batches, std::max<uint64_t>(1, slots / d.chunks));
    uint64_t span = (batches + spans - 1) / spans * t.batch;
    if (span_opt) span = std::max<uint64_t>(t.batch, (uint64_t)span_opt);
    // (a dispatch holds fewer than 2^32 work-items: a shorter span from the
    // caller is lengthened until the tiles fit one launch)
    const uint64_t most = std::max<uint64_t>(1, kDirectTiles / d.chunks);
    span = std::max(span, (batches + most - 1) / most * t.batch);
    span = std::min<uint64_t>(span, 1u << 30);
    spans = std::max<uint64_t>(1, (nS + span - 1) / span);
    d.span = (uint32_t)span;
    d.spans = (uint32_t)spans;
    const double waves = (double)((d.chunks * spans + slots - 1) / slots);
    d.us = waves * t.tile(d.chunk, (double)std::min(span, nS)) + kAtomicUs * (double)d.chunks * (double)batches;
    // several chunks: the match bitmap is cleared before and read after the tiles
    if (outer && d.chunks > 1) d.us += 10 + 2e-6 * (double)nS;
    if (!best.table || d.us < best.us) best = d;
  }
  return best;
}

double plan_one_pass(uint64_t nR, uint64_t nS, int cus, HashPlan *p) {
  // launches: counts, scatter, tile plan (measured at 3.4 M to 50 M tuples of 5
  // to 10 bits: 9 to 21 us, 18 to 227 us, 5 us); more digits cut the scatter's
  // runs short
  const double n = (double)nR + (double)nS, fixed = 9 + 0.25e-6 * n + 5;
  const uint64_t n_cu = (uint64_t)std::max(cus, 8);
  double best = 0;
  for (const ProbeTable &t : kProbeTables) {
    if (t.cap == kFusedTableQuarter) continue;  // unpartitioned joins only
    const uint32_t lds = t.cap == kFusedTableFull ? 16384 : 8192;
    const int b0 = std::max(1, ceil_log2((nR + lds - 1) / lds));
    for (int b = b0; b <= std::min(b0 + 5, kOneMaxBits); ++b) {
      const double scatter = 8 + 3.7e-6 * n * (b <= 8 ? 1.0 : b == 9 ? 1.07 : 1.22);
      const uint64_t P = 1ull << b, slots = n_cu * t.per_cu;
      const double r = (double)nR / P, s = (double)nS / P;
      for (uint64_t k = 1; k <= 16; k *= 2) {  // spans per partition
        if (k > 1 && s / k < t.batch) break;
        // tiles a little over the mean: a partition's length varies
        const double us = fixed + scatter + (double)((P * k + slots - 1) / slots) * t.tile(r, s / k) +
                          kAtomicUs * P * k * std::max(1.0, s / k / t.batch);
        if (best == 0 || us < best) {
          best = us;
          p->bits = p->bits_pass1 = b;
          p->bits_pass2 = 0;
          p->passes = 1;
          p->lds_cap = lds;
          // half as long again as the mean share, so that ordinary partitions
          // stay k tiles and one grown by skewed keys still splits; whole
          // batches, at least one (a left outer join's S may hold fewer
          // tuples than there are partitions)
          const uint64_t batches = std::max<uint64_t>(1, ((uint64_t)(1.5 * s / k) + t.batch - 1) / t.batch);
          p->s_span = (uint32_t)std::min<uint64_t>(batches * t.batch, 1u << 20);
        }
      }
    }
  }
  return best;
}

// Tuples a relation of n needs in a buffer of P sampled regions (the first
// pass's 8 2^bh, the final 2^(bh+bl)) for any sample whose clumping ratios
// are at most K.  A region of sampled count s and ratio kappa gets f kappa m w^3
// with m = s / kappa + 1, and w <= 1 + z/(3 sqrt(m)) gives m w^3 <= m + z
// sqrt(m) + z^2/3 + z^3/27, so its capacity is at most f (s + kappa + z
// sqrt(kappa (s + kappa)) + kappa (z^2/3 + z^3/27)) + pad + line; over the P
// regions, with kappa <= K and sum(sqrt(s_b + K)) <= sqrt(P (ns + K P))
// (Cauchy-Schwarz), at most f (ns + K P (1 + z^2/3 + z^3/27) + z sqrt(K P (ns
// + K P))) + P (pad + line + 1), and f ns = n; f = n / ns falls as the sample
// grows, so the smallest sample (full tiles only) bounds it.  A layout whose
// ratios pass K may not fit: it raises kErrCapacity before any tuple moves.
uint64_t gap_rows(uint64_t n, uint64_t P, double K) {
  const uint64_t full = n / kPartTile;
  const double ns = (double)full * (kPartTile / kGapGroup);
  if (ns <= 0.0) return ~0ull;
  const double f = (double)n / ns, z = kGapZ, p = (double)P;
  const double extra = f * (K * p * (1.0 + z * z / 3.0 + z * z * z / 27.0) + z * std::sqrt(K * p * (ns + K * p)));
  return n + (uint64_t)std::ceil(extra) + P * (kGapPad + kGapLineTuples + 2);
}

uint64_t one_pass_rows(uint64_t n, int bits) {
  const uint64_t P = 1ull << bits;
  if (n < kGapMinRows) return n + P * kGapLineTuples;
  // the largest variance ratio that a line of 16 tuples allows
  return gap_rows(n, P, kGapLineTuples);
}

// 32-bit cursors start below the buffer size and grow by at most n.
bool one_pass_supported(uint64_t nR, uint64_t nS, int bits) {
  return bits >= 1 && bits <= kOneMaxBits && nR && nS && one_pass_rows(nR, bits) + nR < (1ull << 32) &&
         one_pass_rows(nS, bits) + nS < (1ull << 32);
}

void plan_fused(uint64_t nR, uint64_t nS, int cus, bool outer, HashPlan *p) {
  if (p->bits > kOneMaxBits) {
    // 11 bits: where both relations' partitions are sampled two passes of the
    // half table's 12 bits, since a tile's runs of 2048 digits are 64 bytes
    // (one counted pass, two sampled: 17 M x 34 M tuples 0.68 and 0.68 ms, 30 M
    // x 60 M 1.14 and 1.00; counted either way, 17 M x 34 M take 0.68 and
    // 0.75, left outer 0.71 and 0.77)
    eo_join_opts half{};
    half.lds_tuples = 8192;
    if (!outer) (void)plan_hash_join(nR, nS, &half, p, cus);
    return;
  }
  HashPlan one = *p;
  const double us = plan_one_pass(nR, nS, cus, &one);
  if (us == 0) return;
  // (the model of the unpartitioned join is some 15 % low: 2^16 x 2^20 22.5
  // us for 19.4, 100000 x 2^20 38.5 for 32, partitioned 31)
  if (us >= 1.2 * plan_direct(nR, nS, nullptr, cus, outer).us) p->bits = p->bits_pass1 = p->passes = 0;
  else if (one_pass_supported(nR, nS, one.bits)) *p = one;
  // (else relations of nearly 2^31 tuples: their counted pass, which takes any
  // size; unpartitioned, 2^24 x (2^31 - 1) would read S 964 times)
}

std::vector<PlanChoice> tune_candidates(uint64_t nR, uint64_t nS, int cus) {
  std::vector<PlanChoice> v;
  // per LDS table (a full table, one 1024-thread workgroup per CU, or a half
  // table with two): bits b0-1 .. b0+2 around the planner's for that table,
  // passes 1 (bits <= 11) or 2, span auto / x2 / x0.5
  for (int lds : {16384, 8192}) {
    eo_join_opts lo{};
    lo.lds_tuples = lds;
    HashPlan base;
    if (plan_hash_join(nR, nS, &lo, &base, cus) != EO_OK) continue;
    for (int b = std::max(0, base.bits - 1); b <= std::min(kMaxJoinBits, base.bits + 2); ++b) {
      for (int p = 1; p <= 2; ++p) {
        if (b == 0 && p == 2) continue;
        if (b > 0 && p == 1 && b > kMaxPassBits) continue;
        if (p == 2 && (b < 2 || b > 2 * kMaxPassBits)) continue;
        HashPlan hp;
        eo_join_opts o{};
        o.radix_bits = b ? b : -1;
        o.passes = b ? p : 0;
        o.lds_tuples = lds;
        if (plan_hash_join(nR, nS, &o, &hp, cus) != EO_OK) continue;
        for (int k = 0; k < 3; ++k) {
          uint32_t span = hp.s_span;
          if (k == 1) span = std::min<uint32_t>(span * 2, 1u << 18);
          if (k == 2) span = std::max<uint32_t>(span / 2, 8192u);
          if (k > 0 && span == hp.s_span) continue;
          v.push_back({b, b ? p : 0, lds, k == 0 ? 0 : (int)span});
        }
        if (b == 0) break;
      }
    }
  }
  // the untuned join's own plan (built on the smaller side), whose bits, table
  // and span may be none of those
  const uint64_t r = std::min(nR, nS), s = std::max(nR, nS);
  HashPlan own;
  if (r && plan_hash_join(r, s, nullptr, &own, cus) == EO_OK && own.passes <= 1) {
    plan_fused(r, s, cus, false, &own);
    const DirectPlan d = plan_direct(r, s, nullptr, cus);
    const PlanChoice c = own.passes
                             ? PlanChoice{own.bits, own.passes, (int)own.lds_cap, (int)std::max(own.s_span, 8192u)}
                             : PlanChoice{0, 0, (int)table_lds(d.table), 0};
    v.push_back(c);
  }
  return v;
}

uint32_t plan_span(uint64_t nR, uint64_t nS, uint32_t lds_cap, int bits, uint64_t s_pool, int cus) {
  // Fused probe: S spans short enough to give every CU a few tiles of the
  // s_pool S tuples that share the GPU (this join's, or a whole batch's), and
  // at most twice the mean S partition, so that a partition grown by skewed
  // keys splits into tiles no longer than the others (a long tile late in the
  // grid would hold the whole join up); long enough to amortise the LDS build.
  const uint64_t parts = 1ull << bits;
  const uint64_t want_tiles = (uint64_t)std::max(cus, 8) * 4;
  const uint64_t chunks = (nR + lds_cap - 1) / std::max<uint32_t>(lds_cap, 1);
  uint64_t span = std::max(s_pool, nS) * chunks / want_tiles;
  span = std::min<uint64_t>(span, 2 * ((nS + parts - 1) / parts));
  uint32_t s2 = 8192;
  while (s2 < span && s2 < (1u << 18)) s2 <<= 1;
  return s2;
}

}  // namespace eo
