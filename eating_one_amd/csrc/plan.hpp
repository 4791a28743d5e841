// Host-only planning for the hash join: radix bits, passes, LDS table size
// and S tile, per input size.  Pure functions (no HIP calls), so they run and
// are tested without a GPU.
//
// The reference plans at joins/hashJoin_gpu/main_street/hj.cc:378-436:
// p_num = |R| / PART_STANDARD(64) rounded to a power of 64 or of 2, then
// 6 bits per pass.  Here partitions are sized to the LDS table instead, so
// that each R partition is built once in LDS and probed by its S partition.
#pragma once

#include <stdint.h>

#include <vector>

#include "eojoin.h"

namespace eo {

struct HashPlan {
  int bits = 0;        // total radix bits (0 = single partition)
  int passes = 0;      // 0 (no partitioning), 1 or 2
  int bits_pass1 = 0;  // LSD: first pass takes the low bits
  int bits_pass2 = 0;
  uint32_t lds_cap = 0;
  uint32_t s_tile = 0;  // S tuples per tile of the deterministic count/write path
  uint32_t s_span = 0;  // S tuples per tile of the fused probe
  uint32_t stable_stripes = 0;  // stripes of a stable partition pass at most (0 = the pass's bound)
};

constexpr int kMaxJoinBits = 22;

// R tuples one fused-probe LDS table holds for a planned lds_cap: the full
// table (lds_cap 16384) 17408, the half table (lds_cap <= 8192) 8704.
constexpr uint32_t kFusedTableFull = 17408, kFusedTableHalf = 8704;
// An unpartitioned join (every S tile probes each R chunk of one LDS table)
// when R fills at most this many tables and the S tuples read across them stay
// within kUnpartitionedSReads.
constexpr uint64_t kUnpartitionedChunks = 4;
constexpr uint64_t kUnpartitionedSReads = 1ull << 22;

// Tables of an unpartitioned join's tiles, by lds_cap: the full one (16384), the
// half one (8192) and, in unpartitioned joins only, a quarter one (4096).
constexpr uint32_t kFusedTableQuarter = 4352;
inline uint32_t fused_table_tuples(uint32_t lds_cap, bool direct = false) {
  if (direct && lds_cap <= 4096) return kFusedTableQuarter;
  return lds_cap <= 8192 ? kFusedTableHalf : kFusedTableFull;
}

// The tiles of an unpartitioned join: `chunks` R chunks of `chunk` tuples (the
// last one shorter) by `spans` S spans of `span` tuples.
struct DirectPlan {
  uint32_t table = 0;  // LDS table: kFusedTableFull, Half or Quarter
  uint32_t chunk = 0, chunks = 0;
  uint32_t span = 0, spans = 0;
  double us = 0;  // the time model's estimate of the launch
};
// opts: lds_tuples and s_tile overrides (0: chosen here).  outer: a left outer
// join, which adds two launches to tiles of several chunks.
DirectPlan plan_direct(uint64_t nR, uint64_t nS, const eo_join_opts *opts, int cus, bool outer = false);

// The plan of a fused join of one pass that partitions both relations together
// (kernels.hpp, OneArgs): fills bits, table and span of *p and returns the time
// model's estimate of the whole join in microseconds.
double plan_one_pass(uint64_t nR, uint64_t nS, int cus, HashPlan *p);

// The plan of a fused join that no option, tuned entry or misaligned input
// fixes, from plan_hash_join's *p of at most one pass: unpartitioned or both
// relations together, as the time model has it, or *p as it is where the model's
// one pass does not take the sizes.
void plan_fused(uint64_t nR, uint64_t nS, int cus, bool outer, HashPlan *p);

// lds_tuples of an LDS table of `table` tuples (fused_table_tuples' inverse).
inline uint32_t table_lds(uint32_t table) {
  return table == kFusedTableQuarter ? 4096u : table == kFusedTableHalf ? 8192u : 16384u;
}

// Plans the autotuner times for a join of these sizes (radix_bits 0:
// unpartitioned), the one that an untuned join takes among them.
struct PlanChoice {
  int radix_bits, passes, lds_tuples, s_tile;
};
std::vector<PlanChoice> tune_candidates(uint64_t nR, uint64_t nS, int cus);

// Returns EO_OK and fills *out, or EO_EINVAL for inconsistent overrides.
eo_status plan_hash_join(uint64_t nR, uint64_t nS, const eo_join_opts *opts, HashPlan *out, int cus = 256);

// S tuples per fused-probe tile of a join of nR x nS planned with lds_cap and
// bits, when s_pool S tuples (>= nS: the join's own, or a batch's) share the
// GPU: a power of two in [8192, 2^18].
uint32_t plan_span(uint64_t nR, uint64_t nS, uint32_t lds_cap, int bits, uint64_t s_pool, int cus);

}  // namespace eo
