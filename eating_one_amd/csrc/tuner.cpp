// Autotuner for the hash join plan.
//
// The reference fixes its plan with compile-time tables (PART_STANDARD,
// per-size `#define`s; joins/hashJoin_gpu/main_street/hj.cc:378-436 derives
// p_num from |R| / 64 and 6 bits per pass).  Here the planner's choice
// (plan.cpp: partitions sized to one LDS table) is a starting point: for one
// size class (ceil log2 |R|, ceil log2 |S|) eo_tune_hash_join times every
// candidate on the device (plan.cpp: tune_candidates, the planner's own choice
// among them) and keeps the fastest in the context's table.  Joins and batches that leave radix_bits, passes,
// lds_tuples and s_tile at 0 then use the table's entry for their class.
// Every candidate computes the same result (tested), so tuning only changes
// speed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <vector>

#include "ctx.hpp"
#include "eojoin.h"
#include "plan.hpp"

using namespace eo;

extern "C" {

eo_status eo_tune_hash_join(eo_ctx *c, const eo_tuple *R, uint64_t nR, const eo_tuple *S, uint64_t nS, eo_pair *out,
                            uint64_t out_cap, int reps, eo_tune_result *res) {
  if (!c || !res || nR == 0 || nS == 0 || !R || !S || (out_cap && !out) || nR > kMaxRows || nS > kMaxRows)
    return EO_EINVAL;
  reps = std::max(1, std::min(reps, 16));
  std::memset(res, 0, sizeof(*res));
  eo_status st = EO_OK;
  const std::vector<PlanChoice> cands = tune_candidates(nR, nS, c->props.cus);
  c->tuned.erase(tune_key(nR, nS));  // the baseline below is the untuned planner
  eo_join_stats stats;
  auto time_plan = [&](const eo_join_opts &o, double *best) -> eo_status {
    *best = 1e30;
    for (int r = 0; r <= reps; ++r) {  // first run warms the arena
      uint64_t n = 0;
      eo_status s2 = eo_hash_join(c, R, nR, S, nS, out, out_cap, &n, &o);
      if (s2 != EO_OK && s2 != EO_ECAPACITY) return s2;
      if (r > 0) *best = std::min(*best, stats.ms_total);
    }
    return EO_OK;
  };
  eo_join_opts o{};
  o.struct_size = sizeof(o);
  o.where = EO_DEVICE;
  o.stats = &stats;
  // the untuned planner
  double def_ms = 0;
  st = time_plan(o, &def_ms);
  if (st != EO_OK) return st;
  TunedPlan best{0, 0, 0, 0, 1e30};
  for (const PlanChoice &cd : cands) {
    o.radix_bits = cd.radix_bits ? cd.radix_bits : -1;
    o.passes = cd.passes;
    o.lds_tuples = cd.lds_tuples;
    o.s_tile = cd.s_tile;
    double ms = 0;
    st = time_plan(o, &ms);
    if (st != EO_OK) return st;
    if (ms < best.ms) best = {cd.radix_bits, cd.passes, cd.lds_tuples, cd.s_tile, ms};
  }
  c->tuned[tune_key(nR, nS)] = best;
  res->radix_bits = best.radix_bits;
  res->passes = best.passes;
  res->lds_tuples = best.lds_tuples;
  res->s_tile = best.s_tile;
  res->ms = best.ms;
  res->default_ms = def_ms;
  res->candidates = (uint32_t)cands.size();
  return EO_OK;
}

}  // extern "C"
