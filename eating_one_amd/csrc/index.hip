// Resident indexes on R and their probe kernels.
//
// Every index holds its (key, payload) entries as an array of 8-byte pairs,
// so that the line a search ends in also holds the payload of the row to
// write: a probe of an index larger than the caches pays for one line of
// entries instead of one of keys and one of payloads.
//
// Hash index (reference: CPU counting sort into NB_BUCKET buckets,
// joins/innerJoin_gpu/main_street/inner-idx-bnlj.cc:149-180, probed by one
// thread per S tuple in count.cu:15-48 / join_gpu.cu:8-86).  Here the build is
// on the device: bucket b = multiplicative hash of the key (NB = power of two
// >= |R|), histogram with global atomics that also return every tuple's rank
// in its bucket, exclusive scan, placement at bucket start + rank; the index
// is the entries grouped by bucket plus off[NB+1].
//
// Sorted index (reference: CPU quicksort of {val, adr},
// joins/innerJoin_gpu/sort_index/main_street/inner-idx-bnlj.cc:175-216, probed
// by a device binary search and expansion over equal keys, join_gpu.cu:9-113).
// Here: stable LSD radix sort of the R tuples by key on the device
// (partition.hip, four 8-bit passes on the sign-flipped key), whose last pass
// writes the entries (the payload itself instead of the reference's row
// address adr; the joined pairs are the same), and a directory over them:
// level 1 holds the largest key of every 16 entries (one 128-byte line),
// each further level the largest of every 32 of the level below (one line),
// up to a level of at most 4096 keys, which every workgroup keeps in LDS.  A
// search is a binary search in LDS and then one line per level, where a plain
// binary search over 2^24 keys takes 24 dependent loads of as many lines.
//
// Learned sorted index: a 2-stage model over the sorted keys.
//   root: piecewise-linear CDF through K1 = 256 knots at equal-count
//         positions (knot i = (keys[i*n/K1], i*n/K1)); a key's segment is found
//         by binary search over the knots (in LDS), the position interpolated
//         in FP32 and mapped to leaf = pred * L / n, L = 4096;
//   leaf: FP32 linear model pos = a + b * (key - k0) fit by least squares
//         (FP64 sums) on the keys the root routes to it; err_lo / err_hi = the
//         largest under- / over-prediction of the first position of any key
//         routed to the leaf, measured with this same inference code.
// A learned lookup is the lower bound within [pred - err_hi, pred + err_lo]
// (clamped), found by searching that window alone: every key present in R lies
// in its window, so results equal the plain search exactly; absent keys find no
// equal key in any window.  A learned index's join searches the directory like
// any sorted index's: the rows are the same, and it writes them at once.
//
// The deterministic order is count -> scan -> write: per tile of 2048 S tuples
// a count, a u64 scan of those, then the write kernel re-probes and writes at
// tile offset + workgroup-scanned thread offsets.
#include <algorithm>

#include "device.hpp"
#include "kernels.hpp"

namespace eo {
namespace {

constexpr int kIdxNT = 256;
constexpr int kIdxU = 8;                      // probes per thread of a deterministic tile
constexpr int kIdxTile = kIdxNT * kIdxU;
constexpr int kIdxFNT = 512, kIdxFU = 4;       // the fused order's workgroup and probes per thread
constexpr int kNodeLanes = 8;                // lanes that read a node together, 16 bytes each
constexpr uint32_t kEntNode = kNodeLanes * 2; // entries of a node
constexpr uint32_t kDirNode = kNodeLanes * 4; // directory keys of a node
constexpr uint32_t kDirTop = 4096;            // keys of the level searched in LDS (16 KB)
constexpr uint32_t kPadKey = 0x7fffffffu;     // fills the last line of every level

// ---- hash index build ---------------------------------------------------------

// cnt[b] = tuples of bucket b; rank[i] = tuple i's place among them (the count
// its own increment found, so that the placement needs no second atomic).
// Also clears the state of the scan that follows (nzero words).
__global__ void k_hidx_count(const uint2 *__restrict__ R, uint64_t n, int log2nb, uint32_t *cnt,
                             uint32_t *__restrict__ rank, uint64_t *__restrict__ zero, uint32_t nzero) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nzero; i += gridDim.x * blockDim.x) zero[i] = 0ull;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    rank[i] = atomicAdd(&cnt[bucket_hash((int32_t)R[i].x, log2nb)], 1u);
}

__global__ void k_hidx_place(const uint2 *__restrict__ R, uint64_t n, int log2nb, const uint32_t *__restrict__ off,
                             const uint32_t *__restrict__ rank, uint2 *__restrict__ ent) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint2 t = R[i];
    ent[off[bucket_hash((int32_t)t.x, log2nb)] + rank[i]] = t;
  }
}

// ---- sorted index helpers --------------------------------------------------------

__global__ void k_split_soa(const uint2 *__restrict__ T, uint64_t n, uint32_t *keys, uint32_t *pays) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint2 t = T[i];
    keys[i] = t.x;
    pays[i] = t.y;
  }
}

// The directory levels of n entries: level l (0-based) holds cnt[l] keys at
// dir + off[l], key i the largest of its kEntNode * kDirNode^l entries; every
// level is padded to whole lines.
struct DirGeo {
  int levels;
  uint32_t cnt[8], off[8];
  uint32_t total;  // words of the whole directory
};

DirGeo dir_geo(uint64_t n) {
  DirGeo g{};
  uint64_t c = (std::max<uint64_t>(n, 1) + kEntNode - 1) / kEntNode;
  for (;;) {
    g.cnt[g.levels] = (uint32_t)c;
    g.off[g.levels] = g.total;
    g.total += (uint32_t)((c + kDirNode - 1) / kDirNode * kDirNode);
    ++g.levels;
    if (c <= kDirTop) return g;
    c = (c + kDirNode - 1) / kDirNode;
  }
}

// Fills the entries' padding and every level of the directory (one launch:
// each level reads the sorted entries themselves).
__global__ void k_dir_build(uint2 *__restrict__ ent, uint64_t n, DirGeo g, uint32_t *__restrict__ dir) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < kEntNode && n + i < (n + kEntNode - 1) / kEntNode * kEntNode) ent[n + i] = make_uint2(kPadKey, 0u);
  if (i >= g.total) return;
  int l = 0;
  uint64_t span = kEntNode;
  while (l + 1 < g.levels && i >= g.off[l + 1]) {
    ++l;
    span *= kDirNode;
  }
  const uint32_t k = i - g.off[l];
  const uint64_t last = (uint64_t)(k + 1) * span - 1;
  dir[i] = k < g.cnt[l] ? ent[last < n ? last : n - 1].x : kPadKey;
}

// ---- learned model ----------------------------------------------------------------

constexpr int kKnots = 256;     // root segments
constexpr int kLeaves = 4096;   // stage-2 linear models

struct LeafModel {
  float a, b;        // pos ~= a + b * (key - k0)
  int32_t k0;        // first key routed to the leaf
  uint32_t pad;
  int32_t err_lo;    // max (true - pred), >= 0
  int32_t err_hi;    // max (pred - true), >= 0
  uint32_t first, last;  // position range of the leaf's keys [first, last)
};

// Root: position estimate from the knot table (knot_key[K+1], knot_pos[K+1]).
__device__ __forceinline__ float root_pred(const int32_t *knot_key, const float *knot_pos, int32_t k) {
  int lo = 0, hi = kKnots;  // knot_key[lo] <= k < knot_key[hi] (clamped at the ends)
  if (k <= knot_key[0]) return knot_pos[0];
  if (k >= knot_key[kKnots]) return knot_pos[kKnots];
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (knot_key[mid] <= k) lo = mid; else hi = mid;
  }
  const float dk = (float)((int64_t)knot_key[hi] - (int64_t)knot_key[lo]);
  const float t = dk > 0.f ? (float)((int64_t)k - (int64_t)knot_key[lo]) / dk : 0.f;
  return knot_pos[lo] + t * (knot_pos[hi] - knot_pos[lo]);
}

__device__ __forceinline__ uint32_t leaf_of(float root, uint64_t n) {
  const float l = root * (float)kLeaves / (float)n;
  const int li = (int)l;
  return (uint32_t)min(max(li, 0), kLeaves - 1);
}

__device__ __forceinline__ int64_t leaf_pred(const LeafModel &m, int32_t k) {
  const float x = (float)((int64_t)k - (int64_t)m.k0);
  return (int64_t)floorf(m.a + m.b * x);
}

__global__ void k_knots(const uint2 *__restrict__ ent, uint64_t n, int32_t *knot_key, float *knot_pos) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i > kKnots) return;
  uint64_t p = (uint64_t)((double)i * (double)(n - 1) / kKnots);
  knot_key[i] = (int32_t)ent[p].x;
  knot_pos[i] = (float)p;
}

// leaf id of every position (monotone in position because the root is)
__global__ void k_leaf_ids(const uint2 *__restrict__ ent, uint64_t n, const int32_t *knot_key, const float *knot_pos,
                           uint16_t *leaf) {
  __shared__ int32_t kk[kKnots + 1];
  __shared__ float kp[kKnots + 1];
  for (int i = threadIdx.x; i <= kKnots; i += blockDim.x) {
    kk[i] = knot_key[i];
    kp[i] = knot_pos[i];
  }
  __syncthreads();
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    leaf[i] = (uint16_t)leaf_of(root_pred(kk, kp, (int32_t)ent[i].x), n);
}

// One workgroup per leaf: locate its position range, least-squares fit in FP64,
// then the error bounds with the FP32 inference code.
__global__ __launch_bounds__(256) void k_fit_leaves(const uint2 *__restrict__ ent, uint64_t n,
                                                    const uint16_t *__restrict__ leaf, LeafModel *models) {
  __shared__ double red[256 / kWave + 1];
  __shared__ uint64_t range[2];
  __shared__ float ab[2];
  const uint32_t l = blockIdx.x;
  if (threadIdx.x == 0) {
    uint64_t lo = 0, hi = n;  // first position with leaf >= l
    while (lo < hi) {
      const uint64_t mid = (lo + hi) >> 1;
      if (leaf[mid] < l) lo = mid + 1; else hi = mid;
    }
    const uint64_t first = lo;
    hi = n;
    while (lo < hi) {
      const uint64_t mid = (lo + hi) >> 1;
      if (leaf[mid] <= l) lo = mid + 1; else hi = mid;
    }
    range[0] = first;
    range[1] = lo;
  }
  __syncthreads();
  const uint64_t first = range[0], last = range[1];
  LeafModel m{};
  m.first = (uint32_t)first;
  m.last = (uint32_t)last;
  if (first == last) {
    if (threadIdx.x == 0) {
      m.k0 = 0;
      m.a = (float)first;
      m.b = 0.f;
      m.err_lo = m.err_hi = 0;
      models[l] = m;
    }
    return;
  }
  const int32_t k0 = (int32_t)ent[first].x;
  double sx = 0, sy = 0, sxx = 0, sxy = 0;
  for (uint64_t i = first + threadIdx.x; i < last; i += blockDim.x) {
    const double x = (double)((int64_t)(int32_t)ent[i].x - (int64_t)k0);
    const double y = (double)i;
    sx += x;
    sy += y;
    sxx += x * x;
    sxy += x * y;
  }
  sx = block_sum<256, double>(sx, red);
  sy = block_sum<256, double>(sy, red);
  sxx = block_sum<256, double>(sxx, red);
  sxy = block_sum<256, double>(sxy, red);
  if (threadIdx.x == 0) {
    const double cnt = (double)(last - first);
    const double den = cnt * sxx - sx * sx;
    double b = den > 0 ? (cnt * sxy - sx * sy) / den : 0.0;
    double a = (sy - b * sx) / cnt;
    ab[0] = (float)a;
    ab[1] = (float)b;
  }
  __syncthreads();
  m.k0 = k0;
  m.a = ab[0];
  m.b = ab[1];
  // error bounds against the first position of each key (lower_bound)
  int32_t elo = 0, ehi = 0;
  for (uint64_t i = first + threadIdx.x; i < last; i += blockDim.x) {
    if (i > 0 && ent[i - 1].x == ent[i].x) continue;  // not the first occurrence
    const int64_t pred = leaf_pred(m, (int32_t)ent[i].x);
    const int64_t d = (int64_t)i - pred;
    elo = max(elo, (int32_t)min<int64_t>(d, 1 << 30));
    ehi = max(ehi, (int32_t)min<int64_t>(-d, 1 << 30));
  }
  __shared__ int32_t er[2];
  if (threadIdx.x == 0) er[0] = er[1] = 0;
  __syncthreads();
  atomicMax(&er[0], elo);
  atomicMax(&er[1], ehi);
  __syncthreads();
  if (threadIdx.x == 0) {
    m.err_lo = er[0];
    m.err_hi = er[1];
    models[l] = m;
  }
}

// ---- probes -------------------------------------------------------------------------

struct IndexView {
  uint64_t n;
  int log2nb;
  const uint2 *ent;       // entries (sorted kinds: padded to whole lines)
  const uint32_t *off;    // hash: bucket offsets; sorted kinds: the directory
  DirGeo dir;
  const int32_t *knot_key;
  const float *knot_pos;
  const LeafModel *leaves;
};

// Sum of x over the lanes that share a node, in all of them.
__device__ __forceinline__ uint32_t node_sum(uint32_t x) {
  x += dpp_u32<0xb1, 0xf>(x);   // quad_perm 1,0,3,2
  x += dpp_u32<0x4e, 0xf>(x);   // quad_perm 2,3,0,1
  if constexpr (kNodeLanes == 8) x += dpp_u32<0x141, 0xf>(x);  // row_half_mirror
  return x;
}
// v of the group's lane i in r[i]
template <int IT = 0>
__device__ __forceinline__ void node_spread(uint32_t v, uint32_t (&r)[kNodeLanes]) {
  if constexpr (IT < kNodeLanes) {
    r[IT] = (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, (0x1f & ~(kNodeLanes - 1)) | (IT << 5));
    node_spread<IT + 1>(v, r);
  }
}
// The byte of this lane's probe in the group's packed sums (4 probes a word).
__device__ __forceinline__ uint32_t own_byte(const uint32_t (&sum)[kNodeLanes / 4]) {
  const uint32_t lane = (uint32_t)lane_id();
  uint32_t w = sum[0];
  if constexpr (kNodeLanes == 8) w = (lane & 4u) ? sum[1] : sum[0];
  return (w >> (8u * (lane & 3u))) & 0xffu;
}

// Sorted kinds, one probe per lane of a full wave: pos = lower bound of key
// among the n entries, m = entries equal to it, pay = the first one's payload.
// Each level's line is read by 8 lanes together (16 bytes each), the lines of
// a group's 8 probes in flight at once: one instruction reads 8 whole lines,
// where one lane reading its own line takes 8 instructions of 64 lines each.
// A lane counts the smaller keys among its 4 of every line; the counts of 4
// probes are summed over the 8 lanes together, one byte each.
// Bound by the lines that miss L2 (2^25 probes of 2^24 entries: 47 M lines of
// 128 bytes in 0.90 ms, 6.7 TB/s; the binary search over keys, or the model's
// windows, and the payload gather before it: 9 and 2.2 ms).  Nodes of half a
// line, read by 4 lanes, take as many lines of entries and more of level 1
// (54 M, 1.02 ms): the memory side fetches whole lines.
__device__ __forceinline__ void sorted_locate(const IndexView &ix, const int32_t *top, int32_t key, uint32_t &pos,
                                              uint32_t &m, uint32_t &pay) {
  const uint32_t T = ix.dir.cnt[ix.dir.levels - 1];
  uint32_t node = 0;  // keys of the top level below `key`
  for (uint32_t b = 1u << (31 - __clz(T)); b; b >>= 1)
    if (node + b <= T && top[node + b - 1] < key) node += b;
  node = min(node, T - 1);
  constexpr int G = kNodeLanes, GW = G / 4;
  const uint32_t lane = (uint32_t)lane_id(), part = (lane & (G - 1)) * 16u;  // this lane's bytes of a node
  uint32_t kb[G], nb[G];
  node_spread((uint32_t)key, kb);
  uint4 v[G];
  for (int l = ix.dir.levels - 2; l >= 0; --l) {
    const char *lvl = reinterpret_cast<const char *>(ix.off + ix.dir.off[l]);
    node_spread(node, nb);
#pragma unroll
    for (int i = 0; i < G; ++i) v[i] = *reinterpret_cast<const uint4 *>(lvl + (nb[i] * (kDirNode * 4u) + part));
    uint32_t c[GW] = {};
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int32_t k = (int32_t)kb[i];
      c[i / 4] += ((uint32_t)((int32_t)v[i].x < k) + (uint32_t)((int32_t)v[i].y < k) +
                   (uint32_t)((int32_t)v[i].z < k) + (uint32_t)((int32_t)v[i].w < k)) << (8 * (i & 3));
    }
#pragma unroll
    for (int w = 0; w < GW; ++w) c[w] = node_sum(c[w]);
    node = min(node * kDirNode + own_byte(c), ix.dir.cnt[l] - 1);
  }
  node_spread(node, nb);
  const char *ent = reinterpret_cast<const char *>(ix.ent);
#pragma unroll
  for (int i = 0; i < G; ++i)
    v[i] = *reinterpret_cast<const uint4 *>(ent + ((uint64_t)nb[i] * (kEntNode * 8u) + part));
  uint32_t cl[GW] = {}, ce[GW] = {};
#pragma unroll
  for (int i = 0; i < G; ++i) {
    const int32_t k = (int32_t)kb[i];
    cl[i / 4] += ((uint32_t)((int32_t)v[i].x < k) + (uint32_t)((int32_t)v[i].z < k)) << (8 * (i & 3));
    ce[i / 4] += ((uint32_t)((int32_t)v[i].x == k) + (uint32_t)((int32_t)v[i].z == k)) << (8 * (i & 3));
  }
#pragma unroll
  for (int w = 0; w < GW; ++w) {
    cl[w] = node_sum(cl[w]);
    ce[w] = node_sum(ce[w]);
  }
  const uint32_t lt = own_byte(cl), eq = own_byte(ce);
  // the payload at each probe's lower bound, from the lane that holds it: the
  // node was read whole, and reading 8 bytes of it again costs as much as the
  // node did (2^25 probes of 2^24 entries: 0.92 against 1.12 ms)
#pragma unroll
  for (int i = 0; i < G; ++i) {
    const uint32_t at = (cl[i / 4] >> (8 * (i & 3))) & 0xffu;
    const uint32_t p =
        (uint32_t)__shfl((int)((at & 1u) ? v[i].w : v[i].y), (int)((lane & ~(uint32_t)(G - 1)) + ((at >> 1) & (G - 1))));
    if ((lane & (G - 1)) == (uint32_t)i) pay = p;
  }
  // (the padding of the last line may equal a probe's key: not entries)
  const uint32_t n = (uint32_t)ix.n;
  pos = min(node * kEntNode + lt, n);
  m = min(eq, n - pos);
  if (m && lt + eq == kEntNode)  // equal entries may go on past the line
    while (pos + m < n && (int32_t)ix.ent[pos + m].x == key) ++m;
}

// Hash kind: [b, e) is the bucket of key; m equal entries, pay the first one's.
// PAIRS (the deterministic order's few long tiles): buckets of many duplicates
// two entries a load (2^20 entries, 1024 of each key, 2^14 probes: 10.6 -> 8.2
// ms; the fused order's kernel loses occupancy by it, 2^22 probes 152 -> 172 us).
constexpr uint32_t kLongBucket = 16;
template <bool PAIRS>
__device__ __forceinline__ void hash_count(const IndexView &ix, uint32_t key, uint32_t b, uint32_t e, uint32_t &m,
                                           uint32_t &pay) {
  m = 0;
  auto see = [&](uint32_t k, uint32_t p) {
    if (k == key) {
      if (m == 0) pay = p;
      ++m;
    }
  };
  uint32_t j = b;
  if (PAIRS && e - b >= kLongBucket) {
    if (j & 1) {
      see(ix.ent[j].x, ix.ent[j].y);
      ++j;
    }
    for (; j + 2 <= e; j += 2) {
      const uint4 q = *reinterpret_cast<const uint4 *>(ix.ent + j);
      see(q.x, q.y);
      see(q.z, q.w);
    }
  }
  for (; j < e; ++j) {
    const uint2 t = ix.ent[j];
    see(t.x, t.y);
  }
}

// Lookups by the learned model: the lower bound of each key within its leaf's
// window, searched there alone, so that a lookup shows what the model is worth.
// First the window's nodes by level 1 of the directory, then the node, one line
// of each for most probes.  Bound by the latency of those dependent loads and
// by the lines of entries that miss L2: one probe per thread, a workgroup per
// 256 probes (2^27 lookups of 2^26 lognormal keys 4.85 ms, the directory search
// 5.09; the window's keys in an array of their own 4.74; two and four probes
// per thread step by step 5.4 and 7.7, workgroups that walk the probes 5.1).
constexpr int kLookNT = 256;
__global__ __launch_bounds__(kLookNT) void k_learned_lookup(IndexView ix, const uint2 *__restrict__ S, uint64_t nS,
                                                            uint64_t *__restrict__ pos) {
  __shared__ int32_t kk[kKnots + 1];
  __shared__ float kp[kKnots + 1];
  for (int i = threadIdx.x; i <= kKnots; i += kLookNT) {
    kk[i] = ix.knot_key[i];
    kp[i] = ix.knot_pos[i];
  }
  __syncthreads();
  const uint32_t *const dir = ix.off + ix.dir.off[0];
  for (uint64_t i = (uint64_t)blockIdx.x * kLookNT + threadIdx.x; i < nS; i += (uint64_t)gridDim.x * kLookNT) {
    const int32_t key = (int32_t)S[i].x;
    const LeafModel m = ix.leaves[leaf_of(root_pred(kk, kp, key), ix.n)];
    const int64_t pred = leaf_pred(m, key), n = (int64_t)ix.n;
    const uint32_t lo = (uint32_t)min<int64_t>(max<int64_t>(0, pred - m.err_hi), n);
    const uint32_t hi = (uint32_t)max<int64_t>(lo, min<int64_t>(n, pred + m.err_lo + 1));  // (none: an empty window)
    // the first node of the window whose largest key is not below the probe's
    uint32_t a = lo / kEntNode, b = hi > lo ? (hi - 1) / kEntNode + 1 : a;
    while (a < b) {
      const uint32_t mid = (a + b) / 2;
      if ((int32_t)dir[mid] < key) a = mid + 1;
      else b = mid;
    }
    // and its first such entry within the window
    const uint64_t first = (uint64_t)a * kEntNode;
    b = (uint32_t)min<uint64_t>(hi, first + kEntNode);
    a = (uint32_t)min<uint64_t>(max<uint64_t>(lo, first), hi);
    while (a < b) {
      const uint32_t mid = (a + b) / 2;
      if ((int32_t)ix.ent[mid].x < key) a = mid + 1;
      else b = mid;
    }
    pos[i] = a;
  }
}

// KIND 0: hash; 1: sorted.  U probes per thread and tile; workgroups walk the
// tiles, so the top of the directory is read into LDS once per workgroup.
template <int KIND, bool WRITE, int U, int NT>
__global__ __launch_bounds__(NT) void k_index_probe(IndexView ix, const uint2 *__restrict__ S, uint64_t nS,
                                                        uint32_t tiles, uint64_t *__restrict__ tile_cnt,
                                                        uint64_t *cursor, uint2 *__restrict__ out, uint64_t out_cap,
                                                        uint64_t *__restrict__ lb_out, int wide, int outer) {
  constexpr int NW = NT / kWave;
  __shared__ int32_t top[KIND != 0 ? kDirTop : 1];
  __shared__ uint64_t red[NT / kWave + 1];
  __shared__ uint64_t wtot[U * NW];
  __shared__ uint64_t base_sh;
  if (KIND != 0) {
    const int l = ix.dir.levels - 1;
    for (uint32_t i = threadIdx.x; i < ix.dir.cnt[l]; i += NT) top[i] = (int32_t)ix.off[ix.dir.off[l] + i];
  }
  if (KIND != 0) __syncthreads();
  for (uint32_t t = blockIdx.x; t < tiles; t += gridDim.x) {
    const uint64_t s0 = (uint64_t)t * (NT * U);
    uint2 s[U];
    uint32_t b[U];       // first entry to compare with
    uint32_t e[KIND == 0 ? U : 1];
    uint32_t m[U], fp[U];  // matches (at most the index size, < 2^31), the first one's payload
    uint32_t nul = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t i = s0 + (uint64_t)u * NT + threadIdx.x;
      s[u] = i < nS ? S[i] : make_uint2(0u, 0u);
    }
    if constexpr (KIND == 0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t h = bucket_hash((int32_t)s[u].x, ix.log2nb);
        b[u] = ix.off[h];
        e[u] = ix.off[h + 1];
      }
    }
    uint64_t total = 0;  // a thread's matches can pass 2^32
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t i = s0 + (uint64_t)u * NT + threadIdx.x;
      fp[u] = 0;
      if constexpr (KIND == 0) hash_count<U == kIdxU>(ix, s[u].x, b[u], e[u], m[u], fp[u]);
      else sorted_locate(ix, top, (int32_t)s[u].x, b[u], m[u], fp[u]);
      if (i >= nS) m[u] = 0;
      if (lb_out && i < nS) lb_out[i] = b[u];
      if (outer && m[u] == 0 && i < nS) nul |= 1u << u;  // left outer join: one null-padded row
      total += (uint64_t)m[u] + ((nul >> u) & 1u);
    }
    if (!WRITE) {
      const uint64_t tot = block_sum<NT, uint64_t>(total, red);
      if (threadIdx.x == 0) {
        if (tile_cnt) tile_cnt[t] = tot;
        else if (cursor && tot) atomic_add_agent(cursor, tot);
      }
      continue;
    }
    uint64_t pos[U];
    if (tile_cnt) {  // deterministic: thread by thread from the tile's scanned offset
      uint64_t tile_total;
      uint64_t run = tile_cnt[t] + block_excl_scan<NT, uint64_t>(total, red, &tile_total);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        pos[u] = run;
        run += (uint64_t)m[u] + ((nul >> u) & 1u);
      }
    } else {
      // a range reserved with one atomic, slot by slot: the lanes of a wave
      // write consecutive rows
      const int w = threadIdx.x / kWave;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t c = m[u] + ((nul >> u) & 1u);
        uint64_t inc;
        if (__ballot(c >> 25) == 0) inc = wave_incl_scan(c);  // the wave's sum fits 32 bits
        else inc = wave_incl_scan((uint64_t)c);
        pos[u] = inc - c;
        if (lane_id() == kWave - 1) wtot[u * NW + w] = inc;
      }
      __syncthreads();
      if (w == 0) {
        static_assert(U * NW <= kWave, "one lane per (slot, wave)");
        const uint64_t x = lane_id() < U * NW ? wtot[lane_id()] : 0ull;
        const uint64_t inc = wave_incl_scan(x);
        if (lane_id() < U * NW) wtot[lane_id()] = inc - x;
        const uint64_t tot = read_lane(inc, kWave - 1);
        if (lane_id() == 0) base_sh = tot ? atomic_add_agent(cursor, tot) : 0ull;
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < U; ++u) pos[u] += base_sh + wtot[u * NW + w];
      __syncthreads();  // wtot and base_sh are written again by the next tile
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      uint64_t p = pos[u];
      if ((nul >> u) & 1u) {
        if (p < out_cap) emit_null(out, p, s[u].y, s[u].x, wide != 0);
      } else if (m[u] == 1) {
        if (p < out_cap) emit_pair(out, p, fp[u], s[u].y, s[u].x, wide != 0);
      } else if (m[u]) {
        uint32_t j = b[u];
        for (uint32_t c = 0; c < m[u]; ++j) {
          const uint2 r = ix.ent[j];
          if (KIND == 0 && r.x != s[u].x) continue;
          if (p < out_cap) emit_pair(out, p, r.y, s[u].y, s[u].x, wide != 0);
          ++p;
          ++c;
        }
      }
    }
  }
}

// The fused order takes 4 probes per thread in workgroups of 512 (measured on
// 2^25 probes of 2^24 entries: 0.90 ms; 2 probes 0.94, 8 probes 1.27 for their
// registers; workgroups of 256 and 1024 0.91 and 0.95), and one probe per
// thread while that leaves fewer than two workgroups per CU, so that a small S
// still spreads over the chip (2^18 probes of 2^18 entries: 128 workgroups of
// 8 probes a thread 57 us, 1024 of one 29 us).  The deterministic order keeps
// the tiles its row order follows.
template <int KIND, bool WRITE, int U, int NT>
hipError_t launch_probe_u(const IndexView &ix, const eo_tuple *S, uint64_t nS, uint64_t *tile_cnt, uint64_t *cursor,
                          eo_pair *out, uint64_t out_cap, uint64_t *lb_out, bool wide, bool outer, int cus,
                          hipStream_t stream) {
  const uint64_t tile = (uint64_t)NT * U, tiles = (nS + tile - 1) / tile;
  if (tiles >= (1ull << 31)) return hipErrorInvalidValue;
  // 2048 threads fill a CU (the top level takes 16 KB of LDS per workgroup)
  const uint32_t grid = (uint32_t)std::min<uint64_t>(tiles, (2048ull / NT) * (uint64_t)std::max(cus, 8));
  EO_TIMED(WRITE ? "index_write" : "index_probe", stream,
           hipLaunchKernelGGL((k_index_probe<KIND, WRITE, U, NT>), dim3(grid), dim3(NT), 0, stream, ix,
                              reinterpret_cast<const uint2 *>(S), nS, (uint32_t)tiles, tile_cnt, cursor,
                              reinterpret_cast<uint2 *>(out), out_cap, lb_out, (int)wide, (int)outer));
  return hipGetLastError();
}

template <int KIND, bool WRITE>
hipError_t launch_probe(const IndexView &ix, const eo_tuple *S, uint64_t nS, uint64_t *tile_cnt, uint64_t *cursor,
                        eo_pair *out, uint64_t out_cap, uint64_t *lb_out, bool wide, bool outer, int cus,
                        hipStream_t stream) {
  if (nS == 0) return hipSuccess;
#define EO_PROBE_U(U, NT) \
  launch_probe_u<KIND, WRITE, U, NT>(ix, S, nS, tile_cnt, cursor, out, out_cap, lb_out, wide, outer, cus, stream)
  if (tile_cnt) return EO_PROBE_U(kIdxU, kIdxNT);
  if (nS >= 2ull * kIdxFNT * kIdxFU * (uint64_t)std::max(cus, 8)) return EO_PROBE_U(kIdxFU, kIdxFNT);
  return EO_PROBE_U(1, kIdxNT);
#undef EO_PROBE_U
}

// *flag = 1 if some adjacent pair is out of (signed) key order.
__global__ void k_check_sorted(const uint2 *__restrict__ in, uint64_t n, uint32_t *flag) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i + 1 < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    if ((int32_t)in[i].x > (int32_t)in[i + 1].x) *flag = 1u;
}

uint32_t grid_for(uint64_t n) { return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((n + 255) / 256, 16384)); }

}  // namespace

uint64_t index_probe_tiles(uint64_t nS) { return (nS + kIdxTile - 1) / kIdxTile; }
int learned_leaves() { return kLeaves; }
int learned_knots() { return kKnots; }
size_t learned_model_bytes() {
  return (kKnots + 1) * (sizeof(int32_t) + sizeof(float)) + kLeaves * sizeof(LeafModel) + 64;
}

uint64_t index_entries(uint64_t n) { return (std::max<uint64_t>(n, 1) + kEntNode - 1) / kEntNode * kEntNode; }
uint64_t index_dir_words(uint64_t n) { return dir_geo(n).total; }

hipError_t hidx_build(const eo_tuple *R, uint64_t n, int log2nb, eo_tuple *ent, uint32_t *off, uint32_t *rank,
                      void *scan_scratch, uint32_t *err, hipStream_t stream) {
  const uint64_t nb = 1ull << log2nb;
  hipError_t e = fill_u32(off, 0u, nb + 1, stream);
  if (e != hipSuccess) return e;
  const uint2 *vR = reinterpret_cast<const uint2 *>(R);
  hipLaunchKernelGGL(k_hidx_count, dim3(grid_for(n)), dim3(256), 0, stream, vR, n, log2nb, off, rank,
                     (uint64_t *)scan_scratch, (uint32_t)scan_state_words_u32(nb + 1));
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if ((e = scan_u32_clean(off, off, nb + 1, nullptr, scan_scratch, err, stream)) != hipSuccess) return e;
  hipLaunchKernelGGL(k_hidx_place, dim3(grid_for(n)), dim3(256), 0, stream, vR, n, log2nb, off, rank,
                     reinterpret_cast<uint2 *>(ent));
  return hipGetLastError();
}

hipError_t index_dir_build(eo_tuple *ent, uint64_t n, uint32_t *dir, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  const DirGeo g = dir_geo(n);
  hipLaunchKernelGGL(k_dir_build, dim3((g.total + 255) / 256), dim3(256), 0, stream, reinterpret_cast<uint2 *>(ent), n,
                     g, dir);
  return hipGetLastError();
}

hipError_t check_sorted(const eo_tuple *in, uint64_t n, uint32_t *flag, hipStream_t stream) {
  hipError_t e = fill_u32(flag, 0u, 1, stream);
  if (e != hipSuccess || n < 2) return e;
  hipLaunchKernelGGL(k_check_sorted, dim3(grid_for(n)), dim3(256), 0, stream, reinterpret_cast<const uint2 *>(in), n,
                     flag);
  return hipGetLastError();
}

hipError_t index_split(const eo_tuple *ent, uint64_t n, uint32_t *keys, uint32_t *pays, hipStream_t stream) {
  hipLaunchKernelGGL(k_split_soa, dim3(grid_for(n)), dim3(256), 0, stream, reinterpret_cast<const uint2 *>(ent), n,
                     keys, pays);
  return hipGetLastError();
}

hipError_t learned_fit(const eo_tuple *entries, uint64_t n, void *model, uint16_t *leaf_scratch, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  const uint2 *ent = reinterpret_cast<const uint2 *>(entries);
  char *mp = (char *)model;
  int32_t *knot_key = (int32_t *)mp;
  float *knot_pos = (float *)(mp + (kKnots + 1) * sizeof(int32_t));
  LeafModel *leaves = (LeafModel *)(mp + ((kKnots + 1) * (sizeof(int32_t) + sizeof(float)) + 63) / 64 * 64);
  hipLaunchKernelGGL(k_knots, dim3(2), dim3(256), 0, stream, ent, n, knot_key, knot_pos);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_leaf_ids, dim3(grid_for(n)), dim3(256), 0, stream, ent, n, knot_key, knot_pos, leaf_scratch);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_fit_leaves, dim3(kLeaves), dim3(256), 0, stream, ent, n, leaf_scratch, leaves);
  return hipGetLastError();
}

hipError_t index_probe(int kind, bool write, uint64_t n, int log2nb, const eo_tuple *ent, const uint32_t *off,
                       const void *model, const eo_tuple *S, uint64_t nS, uint64_t *tile_cnt, uint64_t *cursor,
                       eo_pair *out, uint64_t out_cap, uint64_t *lb_out, bool wide, bool outer, int cus,
                       hipStream_t stream) {
  IndexView ix{};
  ix.n = n;
  ix.log2nb = log2nb;
  ix.ent = reinterpret_cast<const uint2 *>(ent);
  ix.off = off;
  if (kind != 0) ix.dir = dir_geo(n);
  if (kind == 2 && (!lb_out || n == 0)) kind = 1;  // the rows are the plain search's
  if (kind == 2) {
    if (write || tile_cnt || cursor) return hipErrorInvalidValue;  // lookups only
    if (nS == 0) return hipSuccess;
    const char *mp = (const char *)model;
    ix.knot_key = (const int32_t *)mp;
    ix.knot_pos = (const float *)(mp + (kKnots + 1) * sizeof(int32_t));
    ix.leaves = (const LeafModel *)(mp + ((kKnots + 1) * (sizeof(int32_t) + sizeof(float)) + 63) / 64 * 64);
    const uint32_t grid = (uint32_t)std::min<uint64_t>((nS + kLookNT - 1) / kLookNT, 1u << 20);
    EO_TIMED("index_probe", stream,
             hipLaunchKernelGGL(k_learned_lookup, dim3(grid), dim3(kLookNT), 0, stream, ix,
                                reinterpret_cast<const uint2 *>(S), nS, lb_out));
    return hipGetLastError();
  }
#define EO_PROBE(K, W) \
  launch_probe<K, W>(ix, S, nS, tile_cnt, cursor, out, out_cap, lb_out, wide, outer, cus, stream)
  switch (kind) {
    case 0: return write ? EO_PROBE(0, true) : EO_PROBE(0, false);
    case 1: return write ? EO_PROBE(1, true) : EO_PROBE(1, false);
    default: return hipErrorInvalidValue;
  }
#undef EO_PROBE
}

}  // namespace eo
