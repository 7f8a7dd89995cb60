// adaptive.hip — the adaptive-octree driver (OctreeGenerator, sources/scene/upsample.cpp) on the GPU.
//
// OctreeGenerator::generate (upsample.cpp:228-251) refines cells of the [-1, 1]^3 octree level by
// level: it projects every cell centre once onto the surface (one step, unbounded step length,
// find_stable_nodesGPU, upsample.cpp:317-346), keeps the cell enclosing each projection at the
// cell's own depth (the root when the projected normal is degenerate), subdivides those cells
// and adds the 26 neighbours of every new child (compute_leaves, upsample.cpp:274-287).  An
// outer loop restarts from the depth-0 neighbours of the cells reached and adapts the final
// depth to the extent of the depth-0 cells used (getRelativeDepth, upsample.cpp:146-161).
//
// Here the cell sets stay on the device as unique 64-bit keys whose unsigned order is the
// reference's node_comparator (octree.h:147-154: depth, then z, y, x, signed):
//   key = depth << 60 | (z + 2^19) << 40 | (y + 2^19) << 20 | (x + 2^19)
// The sets between two levels need no order (the queries are sorted along a curve before they are
// projected, and a query's projection depends on it alone), so the kernel that makes the cells of one
// (enclosing cells, children with their neighbours, ancestors) keeps the first of each through a hash
// table; the results are sorted by a rocPRIM radix sort / unique.  The projection is the library's own
// projection of the tree (its kernel, parameters, semantics, form and neighbourhood mode).  Only
// the handful of depth-0 cells of the outer loop live on the host.
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_select.hpp>

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <vector>

#include "mlod_internal.h"

namespace mlod {
namespace {

constexpr int BS = 256;
constexpr int kBias = 1 << 19;              // coordinates live in [-2^19, 2^19)
constexpr uint64_t kNone = ~(uint64_t)0;    // empty slot of an expansion
constexpr uint32_t kMaxGenDepth = 14;       // depth field: 4 bits, children at max_depth + 1

__host__ __device__ __forceinline__ uint64_t cell_key(int d, int x, int y, int z) {
  return ((uint64_t)d << 60) | ((uint64_t)(uint32_t)(z + kBias) << 40) | ((uint64_t)(uint32_t)(y + kBias) << 20) |
         (uint64_t)(uint32_t)(x + kBias);
}
__host__ __device__ __forceinline__ int key_depth(uint64_t k) { return (int)(k >> 60); }
__host__ __device__ __forceinline__ int key_x(uint64_t k) { return (int)(k & 0xfffffu) - kBias; }
__host__ __device__ __forceinline__ int key_y(uint64_t k) { return (int)((k >> 20) & 0xfffffu) - kBias; }
__host__ __device__ __forceinline__ int key_z(uint64_t k) { return (int)((k >> 40) & 0xfffffu) - kBias; }
__host__ __device__ __forceinline__ bool coord_ok(int v) { return v >= -kBias && v < kBias; }

// Error flags raised by kernels (bit 0: a coordinate left the key range).
enum { kFlagRange = 1 };

// ----------------------------------------------------------------------------- sets of cells
// What the kernels of one set operation leave for the host (one copy brings it).
struct GenState {
  uint64_t count;                // cells of the set
  unsigned long long nonfinite;  // projections that were not finite
  uint32_t flags;
};

// An open-addressing table of keys, empty slots kNone, twice as many slots as keys are offered (a probe so
// ends; with the list of those that enter, 24 bytes an offer, what sorting them takes); the keys that enter it first go to `out`, in no particular order.  Most offers are
// repeats (a cell's 64 slots hold some 10 new ones), which one load settles; sorting them all took up to
// 20 launches and four waits a set.  generate() on 1M points, ms with each set sorted / hashed: depth 5 5.7 /
// 4.3, 7 18.6 / 15.1, 8 36.4 / 31.1, 9 88 / 77, 10 294 / 260, 11 1086 / 967 (33M cells).
struct CellSet {
  uint64_t* table;
  uint64_t slots;  // even
  uint64_t* out;
  GenState* st;
};

__global__ __launch_bounds__(BS) void k_clear_set(CellSet set) {
  const uint64_t stride = (uint64_t)gridDim.x * BS;
  const uint64_t i0 = (uint64_t)blockIdx.x * BS + threadIdx.x;
  if (i0 == 0) set.st->count = 0;
  ulonglong2* t = reinterpret_cast<ulonglong2*>(set.table);
  for (uint64_t i = i0; i < set.slots / 2; i += stride) t[i] = make_ulonglong2(kNone, kNone);
}

// True for the one offer of `key` that enters it.
__device__ __forceinline__ bool set_enter(const CellSet& set, uint64_t key) {
  uint64_t h = __umul64hi(key * 0x9e3779b97f4a7c15ull, set.slots);
  for (;; h = h + 1 < set.slots ? h + 1 : 0) {
    unsigned long long* slot = reinterpret_cast<unsigned long long*>(set.table + h);
    // most offers find their key with a load (a stale one is settled by the exchange)
    const uint64_t seen = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (seen == key) return false;
    if (seen != kNone) continue;
    const uint64_t was = atomicCAS(slot, (unsigned long long)kNone, (unsigned long long)key);
    if (was == kNone) return true;
    if (was == key) return false;
  }
}

// Offers R keys a thread (kNone: no offer) and appends those that entered; every thread of the
// workgroup calls it.  A key that the lane before or the thread's last one has too is left to that one:
// ancestors come in long runs, and exchanges on one slot take 12 ns each (120k cells of one ancestor: 1.5
// ms without this).
template <int R>
__device__ __forceinline__ void set_add(const CellSet& set, const uint64_t (&key)[R]) {
  constexpr uint32_t W = BS / 64;
  __shared__ uint32_t sCount[R * W];
  __shared__ uint64_t sBase;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint64_t fresh[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint64_t left = __shfl_up(key[r], 1);
    const bool again = (lane != 0 && key[r] == left) || (r != 0 && key[r] == key[r ? r - 1 : 0]);
    const bool f = key[r] != kNone && !again && set_enter(set, key[r]);
    fresh[r] = __ballot(f);
    if (lane == 0) sCount[r * W + wave] = (uint32_t)__popcll(fresh[r]);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t sum = 0;
    for (uint32_t k = 0; k < R * W; ++k) {
      const uint32_t c = sCount[k];
      sCount[k] = sum;
      sum += c;
    }
    sBase = sum ? atomicAdd(reinterpret_cast<unsigned long long*>(&set.st->count), (unsigned long long)sum) : 0ull;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (fresh[r] >> lane & 1ull)
      set.out[sBase + sCount[r * W + wave] + (uint32_t)__popcll(fresh[r] & ((1ull << lane) - 1ull))] = key[r];
}

// aabb_octree::center over [-1, 1]^3 (octree.h:946-955): min + w p and min + w (p + 1) with
// w = 2 / 2^d, averaged.  Every one of those float operations is exact for |p| < 2^19 and
// d <= 14, so the centre is exactly (2p + 1) 2^-d - 1, which is what is computed.
__device__ __forceinline__ float cell_centre(int p, int d) {
  return __fadd_rn(__fmul_rn((float)(2 * p + 1), __builtin_ldexpf(1.0f, -d)), -1.0f);
}

__global__ __launch_bounds__(BS) void k_centres(const uint64_t* __restrict__ keys, uint32_t n, float* __restrict__ xyz) {
  const uint32_t i = blockIdx.x * BS + threadIdx.x;
  if (i >= n) return;
  const uint64_t k = keys[i];
  const int d = key_depth(k);
  xyz[3 * (size_t)i] = cell_centre(key_x(k), d);
  xyz[3 * (size_t)i + 1] = cell_centre(key_y(k), d);
  xyz[3 * (size_t)i + 2] = cell_centre(key_z(k), d);
}

// aabb_octree::enclosing (octree.h:957-965) over [-1, 1]^3: floor(((p - (-1)) / 2) / 2^-d).
// Returns false for a non-finite or out-of-int coordinate.
__device__ __forceinline__ bool enclose1(float p, int d, int& out) {
  const float t = __fdiv_rn(__fdiv_rn(__fsub_rn(p, -1.0f), 2.0f), __builtin_ldexpf(1.0f, -d));
  const float f = floorf(t);
  if (!(f >= -2147483648.0f && f < 2147483648.0f)) return false;
  out = (int)f;
  return true;
}

// find_stable_nodesGPU's cell assignment (upsample.cpp:336-343) for the projected queries in
// the tree's sorted order: slot j holds the projection of input cell perm[j].  A degenerate
// normal (|n|^2 < 0.5, glm::length2) or a non-finite projected position gives the root.
__device__ __forceinline__ uint64_t enclosing_key(const float4* __restrict__ q, const float4* __restrict__ qn,
                                                  const uint32_t* __restrict__ perm, const uint64_t* __restrict__ in,
                                                  uint32_t j, GenState* __restrict__ st) {
  const int d = key_depth(in[perm[j]]);
  const float4 nm = qn[j];
  const float l2 = __fadd_rn(__fadd_rn(__fmul_rn(nm.x, nm.x), __fmul_rn(nm.y, nm.y)), __fmul_rn(nm.z, nm.z));
  uint64_t key = cell_key(0, 0, 0, 0);
  if (!(l2 < 0.5f)) {
    const float4 p = q[j];
    int x, y, z;
    if (enclose1(p.x, d, x) && enclose1(p.y, d, y) && enclose1(p.z, d, z)) {
      if (coord_ok(x) && coord_ok(y) && coord_ok(z))
        key = cell_key(d, x, y, z);
      else
        atomicOr(&st->flags, (uint32_t)kFlagRange);
    } else {
      atomicAdd(&st->nonfinite, 1ull);
    }
  }
  return key;
}
__global__ __launch_bounds__(BS) void k_enclose_set(const float4* __restrict__ q, const float4* __restrict__ qn,
                                                    const uint32_t* __restrict__ perm, const uint64_t* __restrict__ in,
                                                    uint32_t n, CellSet set) {
  const uint32_t j = blockIdx.x * BS + threadIdx.x;
  const uint64_t key[1] = {j < n ? enclosing_key(q, qn, perm, in, j, set.st) : kNone};
  set_add<1>(set, key);
}

// add_children (upsample.cpp:348-358) followed by expand(current, depth + 1)
// (upsample.cpp:409-419): a cell at `depth` contributes the 4 x 4 x 4 block of depth + 1 cells
// made of its children and their neighbours; a shallower cell (the root and its descendants
// re-entered after a failed projection) contributes its 8 children only.  64 slots per cell.
__device__ __forceinline__ uint64_t expanded_key(const uint64_t* __restrict__ sub, uint64_t t, int depth,
                                                 GenState* __restrict__ st) {
  const uint32_t i = (uint32_t)(t >> 6), s = (uint32_t)(t & 63);
  const uint64_t k = sub[i];
  const int d = key_depth(k), x = key_x(k), y = key_y(k), z = key_z(k);
  int cx, cy, cz;
  if (d == depth) {
    cx = 2 * x - 1 + (int)(s & 3);
    cy = 2 * y - 1 + (int)((s >> 2) & 3);
    cz = 2 * z - 1 + (int)(s >> 4);
  } else if (s < 8) {
    cx = 2 * x + (int)(s & 1);
    cy = 2 * y + (int)((s >> 1) & 1);
    cz = 2 * z + (int)(s >> 2);
  } else {
    return kNone;
  }
  if (!coord_ok(cx) || !coord_ok(cy) || !coord_ok(cz)) {
    atomicOr(&st->flags, (uint32_t)kFlagRange);
    return kNone;
  }
  return cell_key(d + 1, cx, cy, cz);
}
constexpr int kExpandRun = 4;  // offers a thread
__global__ __launch_bounds__(BS) void k_expand_set(const uint64_t* __restrict__ sub, uint32_t n, int depth, CellSet set) {
  const uint64_t t0 = (uint64_t)blockIdx.x * (BS * kExpandRun) + threadIdx.x;
  uint64_t key[kExpandRun];
#pragma unroll
  for (int r = 0; r < kExpandRun; ++r) {
    const uint64_t t = t0 + r * BS;
    key[r] = t < (uint64_t)n * 64 ? expanded_key(sub, t, depth, set.st) : kNone;
  }
  set_add<kExpandRun>(set, key);
}

// ancestor_at_depth (octree.h:561-573): repeated floor halving, i.e. an arithmetic shift.
// Cells at or above `depth` are kept as they are (onlySetDepthNodes, upsample.cpp:163-173).
__device__ __forceinline__ uint64_t ancestor_key(uint64_t k, int depth) {
  const int sh = key_depth(k) - depth;
  return sh <= 0 ? k : cell_key(depth, key_x(k) >> sh, key_y(k) >> sh, key_z(k) >> sh);
}
__global__ __launch_bounds__(BS) void k_ancestor(const uint64_t* __restrict__ in, uint32_t n, int depth,
                                                 uint64_t* __restrict__ out) {
  const uint32_t i = blockIdx.x * BS + threadIdx.x;
  if (i < n) out[i] = ancestor_key(in[i], depth);
}
constexpr int kAncestorRun = 8;
__global__ __launch_bounds__(BS) void k_ancestor_set(const uint64_t* __restrict__ in, uint32_t n, int depth, CellSet set) {
  const uint32_t i0 = blockIdx.x * (BS * kAncestorRun) + threadIdx.x;
  uint64_t key[kAncestorRun];
#pragma unroll
  for (int r = 0; r < kAncestorRun; ++r) {
    const uint32_t i = i0 + r * BS;
    key[r] = i < n ? ancestor_key(in[i], depth) : kNone;
  }
  set_add<kAncestorRun>(set, key);
}

// generateFromPoints (upsample.cpp:128-144): the max_depth cell enclosing each point of the
// box (aabb_octree::enclosing, octree.h:957-965): floor(((p - min) / diag) / 2^-d).
__global__ __launch_bounds__(BS) void k_enclose_points(const float* __restrict__ xyz, uint32_t n, int d, float mnx,
                                                       float mny, float mnz, float dgx, float dgy, float dgz,
                                                       uint64_t* __restrict__ out, GenState* __restrict__ st) {
  const uint32_t i = blockIdx.x * BS + threadIdx.x;
  if (i >= n) return;
  const float w = __builtin_ldexpf(1.0f, -d);
  const float mn[3] = {mnx, mny, mnz}, dg[3] = {dgx, dgy, dgz};
  int c[3];
  bool fin = true;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float f = floorf(__fdiv_rn(__fdiv_rn(__fsub_rn(xyz[3 * (size_t)i + a], mn[a]), dg[a]), w));
    if (!(f >= -2147483648.0f && f < 2147483648.0f)) {
      fin = false;
      c[a] = 0;
    } else {
      c[a] = (int)f;
    }
  }
  if (!fin) {
    atomicAdd(&st->nonfinite, 1ull);
    out[i] = kNone;
    return;
  }
  if (!coord_ok(c[0]) || !coord_ok(c[1]) || !coord_ok(c[2])) {
    atomicOr(&st->flags, (uint32_t)kFlagRange);
    out[i] = kNone;
    return;
  }
  out[i] = cell_key(d, c[0], c[1], c[2]);
}

// aabb_octree::center of a general box (octree.h:946-955): w = diag / 2^d, then
// (min + w p + min + w (p + 1)) / 2 in float, without contraction.
__global__ __launch_bounds__(BS) void k_centres_box(const uint64_t* __restrict__ keys, uint32_t n, float mnx, float mny,
                                                    float mnz, float dgx, float dgy, float dgz, float* __restrict__ xyz) {
  const uint32_t i = blockIdx.x * BS + threadIdx.x;
  if (i >= n) return;
  const uint64_t k = keys[i];
  const int d = key_depth(k);
  const int p[3] = {key_x(k), key_y(k), key_z(k)};
  const float mn[3] = {mnx, mny, mnz}, dg[3] = {dgx, dgy, dgz};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float w = __fdiv_rn(dg[a], (float)(1 << d));
    const float lo = __fadd_rn(mn[a], __fmul_rn(w, (float)p[a]));
    const float hi = __fadd_rn(mn[a], __fmul_rn(w, (float)(p[a] + 1)));
    xyz[3 * (size_t)i + a] = __fdiv_rn(__fadd_rn(lo, hi), 2.0f);
  }
}

__global__ __launch_bounds__(BS) void k_decode(const uint64_t* __restrict__ keys, uint32_t n, int32_t* __restrict__ out) {
  const uint32_t i = blockIdx.x * BS + threadIdx.x;
  if (i >= n) return;
  const uint64_t k = keys[i];
  out[4 * (size_t)i] = key_depth(k);
  out[4 * (size_t)i + 1] = key_x(k);
  out[4 * (size_t)i + 2] = key_y(k);
  out[4 * (size_t)i + 3] = key_z(k);
}

inline uint32_t blocks(uint64_t n) { return (uint32_t)((n + BS - 1) / BS); }

// A growable device array of keys.  (A growth waits for the stream: the small levels share one size.)
constexpr size_t kKeyVecMin = (size_t)1 << 18;
struct KeyVec {
  uint64_t* p = nullptr;
  size_t n = 0, cap = 0;
  void release() {
    if (p) dev_free(p);
    p = nullptr;
    n = cap = 0;
  }
  // room for m keys, keeping the first `keep`
  int reserve(size_t m, size_t keep, hipStream_t s) {
    if (m <= cap) return MLOD_OK;
    const size_t nc = std::max({m, cap + cap / 2, kKeyVecMin});
    uint64_t* q = nullptr;
    if (dev_malloc(&q, nc * sizeof(uint64_t)) != hipSuccess)
      return fail(MLOD_ERR_OOM, "adaptive octree: hipMalloc failed for " + std::to_string(nc) + " cells");
    if (keep) MLOD_HIP(hipMemcpyAsync(q, p, keep * sizeof(uint64_t), hipMemcpyDeviceToDevice, s));
    MLOD_HIP(hipStreamSynchronize(s));
    if (p) dev_free(p);
    p = q;
    cap = nc;
    return MLOD_OK;
  }
};

}  // namespace
}  // namespace mlod

struct mlod_generator {
  mlod_tree* tree = nullptr;
  mlod::KeyVec leaves, total;   // results, sorted and unique
  mlod::KeyVec a, b, c;         // work sets
  mlod::KeyVec table;           // slots of the set that is being made, or a sort's temporary storage
  mlod::GenState* dState = nullptr;
  float* dXyz = nullptr;        // centres of the leaves (n x 3), valid after mlod_generator_centres
  size_t xyzCap = 0;
  float* dStage = nullptr;      // centres projected by the current level
  size_t stageCap = 0;
  uint32_t maxRel = 0;
  uint64_t projected = 0, calls = 0, nonfinite = 0;
  bool keepTotal = true;
  float box[6] = {-1.f, -1.f, -1.f, 1.f, 1.f, 1.f};  // frame of the leaves' centres
};

namespace mlod {
namespace {

int KeyVec_append(KeyVec& v, const uint64_t* src, size_t m, hipMemcpyKind kind, hipStream_t s) {
  if (!m) return MLOD_OK;
  if (int r = v.reserve(v.n + m, v.n, s)) return r;
  MLOD_HIP(hipMemcpyAsync(v.p + v.n, src, m * sizeof(uint64_t), kind, s));
  v.n += m;
  return MLOD_OK;
}

int ensure_sort_tmp(mlod_generator* g, size_t n, size_t* bytes, hipStream_t s) {
  size_t need = 0, need2 = 0;
  MLOD_HIP(rocprim::radix_sort_keys(nullptr, need, (uint64_t*)nullptr, (uint64_t*)nullptr, n, 0, 64, s));
  MLOD_HIP(rocprim::unique(nullptr, need2, (uint64_t*)nullptr, (uint64_t*)nullptr, (uint64_t*)nullptr, n,
                           rocprim::equal_to<uint64_t>(), s));
  need = std::max(need, need2);
  if (int r = g->table.reserve((need + 7) / 8, 0, s)) return r;
  *bytes = g->table.cap * 8;
  return MLOD_OK;
}

// The count, flags and non-finite projections of the operations so far (waits for the stream).
int read_state(mlod_generator* g, uint64_t* count, hipStream_t s) {
  GenState st;
  MLOD_HIP(hipMemcpyAsync(&st, g->dState, sizeof(st), hipMemcpyDeviceToHost, s));
  MLOD_HIP(hipStreamSynchronize(s));
  g->nonfinite = st.nonfinite;
  if (count) *count = st.count;
  if (st.flags & kFlagRange)
    return fail(MLOD_ERR_UNSUPPORTED, "adaptive octree: a cell coordinate left [-2^19, 2^19) (the surface reaches far "
                                      "outside [-1, 1]^3 at this depth)");
  return MLOD_OK;
}

// remove_duplicates (upsample.cpp:28-32) of the n keys in `in` (clobbered) into `out`, sorted; drops the
// empty-slot key.  Returns the unique count through *m (waits for the stream).
int sort_unique(mlod_generator* g, KeyVec& in, size_t n, KeyVec& out, size_t* m, hipStream_t s) {
  *m = 0;
  if (!n) {
    out.n = 0;
    return MLOD_OK;
  }
  if (n > 0xffffffffu) return fail(MLOD_ERR_UNSUPPORTED, "adaptive octree: more than 2^32 cells in one set");
  size_t tmp = 0;
  if (int r = ensure_sort_tmp(g, n, &tmp, s)) return r;
  if (int r = out.reserve(n, 0, s)) return r;
  size_t bytes = tmp;
  MLOD_HIP(rocprim::radix_sort_keys(g->table.p, bytes, in.p, out.p, n, 0, 64, s));
  bytes = tmp;
  MLOD_HIP(rocprim::unique(g->table.p, bytes, out.p, in.p, &g->dState->count, n, rocprim::equal_to<uint64_t>(), s));
  uint64_t cnt = 0, last = 0;
  const int flagged = read_state(g, &cnt, s);  // (the set is handed over all the same)
  if (flagged && flagged != MLOD_ERR_UNSUPPORTED) return flagged;
  if (cnt) {
    MLOD_HIP(hipMemcpyAsync(&last, in.p + cnt - 1, sizeof(last), hipMemcpyDeviceToHost, s));
    MLOD_HIP(hipStreamSynchronize(s));
    if (last == kNone) --cnt;
  }
  std::swap(in, out);  // the unique keys are in `in`'s storage: hand it to `out`
  out.n = cnt;
  in.n = 0;
  *m = cnt;
  return flagged;
}

// An empty set for `offers` keys, its cells to go to `out`.
int begin_set(mlod_generator* g, size_t offers, KeyVec& out, CellSet* set, hipStream_t s) {
  if (offers > 0xffffffffu) return fail(MLOD_ERR_UNSUPPORTED, "adaptive octree: more than 2^32 cells in one set");
  const uint64_t slots = 2 * std::max<uint64_t>(offers, 2048);
  if (int r = out.reserve(offers, 0, s)) return r;
  if (int r = g->table.reserve(slots, 0, s)) return r;
  *set = CellSet{g->table.p, slots, out.p, g->dState};
  k_clear_set<<<std::min<uint32_t>(blocks(slots / 2), 2048u), BS, 0, s>>>(*set);
  MLOD_HIP(hipGetLastError());
  return MLOD_OK;
}
int end_set(mlod_generator* g, KeyVec& out, hipStream_t s) {
  uint64_t n = 0;
  const int r = read_state(g, &n, s);
  out.n = n;
  return r;
}

// The tree's own projection of the n centres in g->dStage: one step, step bound FLT_MAX
// (upsample.cpp:331-333).  Results stay in the tree's sorted query arrays.
int project_centres(mlod_generator* g, uint32_t n, hipStream_t s) {
  mlod_tree* t = g->tree;
  if (int r = queries_set(t, g->dStage, n, true, s)) return r;
  int r = (t->mode == MLOD_MODE_KNN || t->mode == MLOD_MODE_BALL) ? launch_neighbors(t, n, 1, s)
                                                                   : launch_project(t, n, 1, FLT_MAX, s);
  g->projected += n;
  g->calls += 1;
  return r;
}

// find_stable_nodesGPU (upsample.cpp:317-346) on the cells in cur -> unique cells in sub
int find_stable(mlod_generator* g, KeyVec& cur, KeyVec& sub, hipStream_t s) {
  const size_t n = cur.n;
  if (!n) {
    sub.n = 0;
    return MLOD_OK;
  }
  if (n > g->stageCap) {
    if (g->dStage) dev_free(g->dStage);
    g->dStage = nullptr;
    g->stageCap = 0;
    if (dev_malloc(&g->dStage, n * 3 * sizeof(float)) != hipSuccess)
      return fail(MLOD_ERR_OOM, "adaptive octree: centre buffer");
    g->stageCap = n;
  }
  k_centres<<<blocks(n), BS, 0, s>>>(cur.p, (uint32_t)n, g->dStage);
  MLOD_HIP(hipGetLastError());
  if (int r = project_centres(g, (uint32_t)n, s)) return r;
  const QueryState& qs = g->tree->qs;
  CellSet set;
  if (int r = begin_set(g, n, sub, &set, s)) return r;
  k_enclose_set<<<blocks(n), BS, 0, s>>>(qs.q, qs.qn, qs.perm, cur.p, (uint32_t)n, set);
  MLOD_HIP(hipGetLastError());
  return end_set(g, sub, s);
}

// compute_leaves (upsample.cpp:274-287): cur in, the cells after the last level in cur
int compute_leaves(mlod_generator* g, uint32_t maxDepth, hipStream_t s) {
  KeyVec &cur = g->a, &sub = g->b;
  for (uint32_t depth = 0; depth < maxDepth + 1; ++depth) {
    if (int r = find_stable(g, cur, sub, s)) return r;
    const size_t ns = sub.n;
    cur.n = 0;
    if (ns) {
      CellSet set;
      if (int r = begin_set(g, ns * 64, cur, &set, s)) return r;
      k_expand_set<<<(uint32_t)((ns * 64 + BS * kExpandRun - 1) / (BS * kExpandRun)), BS, 0, s>>>(sub.p, (uint32_t)ns,
                                                                                                 (int)depth, set);
      MLOD_HIP(hipGetLastError());
      if (int r = end_set(g, cur, s)) return r;
    }
    if (g->keepTotal)
      if (int r = KeyVec_append(g->total, cur.p, cur.n, hipMemcpyDeviceToDevice, s)) return r;
  }
  return MLOD_OK;
}

// onlySetDepthNodes (upsample.cpp:163-173): ancestors at `depth` of deeper cells, sorted unique
int only_set_depth(mlod_generator* g, KeyVec& v, uint32_t depth, hipStream_t s) {
  if (!v.n) return MLOD_OK;
  KeyVec& tmp = g->c;
  if (int r = tmp.reserve(v.n, 0, s)) return r;
  k_ancestor<<<blocks(v.n), BS, 0, s>>>(v.p, (uint32_t)v.n, (int)depth, tmp.p);
  MLOD_HIP(hipGetLastError());
  size_t m = 0;
  return sort_unique(g, tmp, v.n, v, &m, s);
}

struct HostCell {
  int d, x, y, z;
};

// OctreeGenerator::generate (upsample.cpp:228-251)
int generate(mlod_generator* g, uint32_t maxDepth, hipStream_t s) {
  g->leaves.n = g->total.n = 0;
  g->projected = g->calls = g->nonfinite = 0;
  MLOD_HIP(hipMemsetAsync(g->dState, 0, sizeof(GenState), s));
  std::vector<uint64_t> depth0{cell_key(0, 0, 0, 0)}, old0;
  uint32_t maxRel = maxDepth;
  int mn[3] = {INT_MAX, INT_MAX, INT_MAX}, mx[3] = {-INT_MAX, -INT_MAX, -INT_MAX};
  while (!depth0.empty()) {
    if (g->keepTotal)
      if (int r = KeyVec_append(g->total, depth0.data(), depth0.size(), hipMemcpyHostToDevice, s)) return r;
    if (int r = g->a.reserve(depth0.size(), 0, s)) return r;
    MLOD_HIP(hipMemcpyAsync(g->a.p, depth0.data(), depth0.size() * sizeof(uint64_t), hipMemcpyHostToDevice, s));
    g->a.n = depth0.size();
    if (int r = compute_leaves(g, maxRel, s)) return r;
    KeyVec& cur = g->a;
    // depth0_ancestors(current) (upsample.cpp:360-368): a small set, brought to the host
    std::vector<uint64_t> anc;
    if (cur.n) {
      CellSet set;
      if (int r = begin_set(g, cur.n, g->c, &set, s)) return r;
      k_ancestor_set<<<(uint32_t)((cur.n + BS * kAncestorRun - 1) / (BS * kAncestorRun)), BS, 0, s>>>(
          cur.p, (uint32_t)cur.n, 0, set);
      MLOD_HIP(hipGetLastError());
      if (int r = end_set(g, g->c, s)) return r;
      const size_t m = g->c.n;
      anc.resize(m);
      if (m) {
        MLOD_HIP(hipMemcpyAsync(anc.data(), g->c.p, m * sizeof(uint64_t), hipMemcpyDeviceToHost, s));
        MLOD_HIP(hipStreamSynchronize(s));
      }
    }
    // getRelativeDepth (upsample.cpp:146-161); min / max persist across iterations
    int rd = 0;
    if (cur.n) {
      for (uint64_t k : anc) {
        const int p[3] = {key_x(k), key_y(k), key_z(k)};
        for (int a = 0; a < 3; ++a) mn[a] = std::min(mn[a], p[a]), mx[a] = std::max(mx[a], p[a]);
      }
      for (int a = 0; a < 3; ++a) rd = std::max(rd, (int)std::ceil(float(std::log2(mx[a] - mn[a] + 1))));
    }
    maxRel = (uint32_t)std::max(0, (int)maxDepth - rd);
    if (int r = KeyVec_append(g->leaves, cur.p, cur.n, hipMemcpyDeviceToDevice, s)) return r;
    old0.insert(old0.end(), depth0.begin(), depth0.end());
    std::sort(old0.begin(), old0.end());
    // expand(depth0) over all depths, minus every depth-0 cell already processed
    std::vector<uint64_t> nxt;
    for (uint64_t k : anc)
      for (int dz = -1; dz <= 1; ++dz)
        for (int dy = -1; dy <= 1; ++dy)
          for (int dx = -1; dx <= 1; ++dx) {
            const int x = key_x(k) + dx, y = key_y(k) + dy, z = key_z(k) + dz;
            if (!coord_ok(x) || !coord_ok(y) || !coord_ok(z))
              return fail(MLOD_ERR_UNSUPPORTED, "adaptive octree: depth-0 cell out of range");
            nxt.push_back(cell_key(0, x, y, z));
          }
    std::sort(nxt.begin(), nxt.end());
    nxt.erase(std::unique(nxt.begin(), nxt.end()), nxt.end());
    depth0.clear();
    for (uint64_t k : nxt)
      if (!std::binary_search(old0.begin(), old0.end(), k)) depth0.push_back(k);
  }
  // remove_duplicates(nodes) then onlySetDepthNodes(nodes / total_tree, max relative depth)
  if (int r = only_set_depth(g, g->leaves, maxRel, s)) return r;
  if (g->keepTotal)
    if (int r = only_set_depth(g, g->total, maxRel, s)) return r;
  g->maxRel = maxRel;
  for (int a = 0; a < 3; ++a) g->box[a] = -1.f, g->box[3 + a] = 1.f;
  return read_state(g, nullptr, s);
}

int leaf_centres(mlod_generator* g, hipStream_t s) {
  const size_t n = g->leaves.n;
  if (n > g->xyzCap) {
    if (g->dXyz) dev_free(g->dXyz);
    g->dXyz = nullptr;
    g->xyzCap = 0;
    if (dev_malloc(&g->dXyz, std::max<size_t>(n, 1) * 3 * sizeof(float)) != hipSuccess)
      return fail(MLOD_ERR_OOM, "adaptive octree: leaf centre buffer");
    g->xyzCap = n;
  }
  if (n) {
    const float* b = g->box;
    k_centres_box<<<blocks(n), BS, 0, s>>>(g->leaves.p, (uint32_t)n, b[0], b[1], b[2], b[3] - b[0], b[4] - b[1],
                                           b[5] - b[2], g->dXyz);
    MLOD_HIP(hipGetLastError());
  }
  return MLOD_OK;
}

}  // namespace
}  // namespace mlod

using namespace mlod;

extern "C" {

int mlod_generator_create(mlod_tree* t, mlod_generator** out) {
  if (!out) return fail(MLOD_ERR_INVALID, "out is NULL");
  *out = nullptr;
  mlod_generator* g = new mlod_generator();
  g->tree = t;
  if (dev_malloc(&g->dState, sizeof(GenState)) != hipSuccess) {
    mlod_generator_destroy(g);
    return fail(MLOD_ERR_OOM, "generator: hipMalloc failed");
  }
  *out = g;
  return MLOD_OK;
}

int mlod_generator_destroy(mlod_generator* g) {
  if (!g) return MLOD_OK;
  (void)hipDeviceSynchronize();
  g->leaves.release(), g->total.release(), g->a.release(), g->b.release(), g->c.release(), g->table.release();
  void* p[] = {g->dState, g->dXyz, g->dStage};
  dev_free(p, sizeof(p) / sizeof(p[0]));
  delete g;
  return MLOD_OK;
}

int mlod_generate(mlod_generator* g, uint32_t max_depth, int32_t keep_total, void* stream) {
  if (!g) return fail(MLOD_ERR_INVALID, "generator is NULL");
  if (!g->tree) return fail(MLOD_ERR_STATE, "generator has no tree (created for generate_from_points only)");
  if (max_depth + 1 >= kMaxGenDepth) return fail(MLOD_ERR_INVALID, "max_depth must be <= 12");
  if (!g->tree->kernel_set) return fail(MLOD_ERR_STATE, "no kernel set on the tree (mlod_set_kernel)");
  g->keepTotal = keep_total != 0;
  return generate(g, max_depth, (hipStream_t)stream);
}

int mlod_generate_from_points(mlod_generator* g, const float* xyz, uint32_t n, int32_t device_src, uint32_t max_depth,
                              const float* box6, void* stream) {
  if (!g || (!xyz && n)) return fail(MLOD_ERR_INVALID, "NULL argument");
  if (max_depth >= kMaxGenDepth) return fail(MLOD_ERR_INVALID, "max_depth must be <= 13");
  hipStream_t s = (hipStream_t)stream;
  float b[6] = {-1.f, -1.f, -1.f, 1.f, 1.f, 1.f};
  if (box6) {
    bool empty = false;  // Eigen's isEmpty: some min > max
    for (int a = 0; a < 3; ++a) empty |= box6[a] > box6[3 + a];
    if (!empty) std::memcpy(b, box6, sizeof(b));
  }
  g->leaves.n = g->total.n = 0;
  g->maxRel = max_depth;
  g->projected = g->calls = 0;
  std::memcpy(g->box, b, sizeof(b));
  if (n == 0) return MLOD_OK;  // upsample.cpp:130
  MLOD_HIP(hipMemsetAsync(g->dState, 0, sizeof(GenState), s));
  const float* src = xyz;
  if (!device_src) {
    if (n > g->stageCap) {
      if (g->dStage) dev_free(g->dStage);
      g->dStage = nullptr;
      g->stageCap = 0;
      if (dev_malloc(&g->dStage, (size_t)n * 3 * sizeof(float)) != hipSuccess)
        return fail(MLOD_ERR_OOM, "generator: point buffer");
      g->stageCap = n;
    }
    MLOD_HIP(hipMemcpyAsync(g->dStage, xyz, (size_t)n * 3 * sizeof(float), hipMemcpyHostToDevice, s));
    src = g->dStage;
  }
  if (int r = g->c.reserve(n, 0, s)) return r;
  k_enclose_points<<<blocks(n), BS, 0, s>>>(src, n, (int)max_depth, b[0], b[1], b[2], b[3] - b[0], b[4] - b[1],
                                            b[5] - b[2], g->c.p, g->dState);
  MLOD_HIP(hipGetLastError());
  size_t m = 0;
  return sort_unique(g, g->c, n, g->leaves, &m, s);
}

int mlod_generator_info(const mlod_generator* g, uint64_t* out6) {
  if (!g || !out6) return fail(MLOD_ERR_INVALID, "NULL argument");
  out6[0] = g->leaves.n;
  out6[1] = g->total.n;
  out6[2] = g->maxRel;
  out6[3] = g->projected;
  out6[4] = g->calls;
  out6[5] = g->nonfinite;
  return MLOD_OK;
}

int mlod_generator_cells(mlod_generator* g, int32_t which, int32_t* out_ids4, void* stream) {
  if (!g || !out_ids4) return fail(MLOD_ERR_INVALID, "NULL argument");
  const KeyVec& v = which ? g->total : g->leaves;
  if (!v.n) return MLOD_OK;
  hipStream_t s = (hipStream_t)stream;
  int32_t* d = nullptr;
  if (dev_malloc(&d, v.n * 4 * sizeof(int32_t)) != hipSuccess) return fail(MLOD_ERR_OOM, "cell download buffer");
  k_decode<<<blocks(v.n), BS, 0, s>>>(v.p, (uint32_t)v.n, d);
  hipError_t e = hipGetLastError();
  if (!e) e = hipMemcpyAsync(out_ids4, d, v.n * 4 * sizeof(int32_t), hipMemcpyDeviceToHost, s);
  if (!e) e = hipStreamSynchronize(s);
  dev_free(d);
  if (e) return hip_fail(e, "generator cells", __FILE__, __LINE__);
  return MLOD_OK;
}

int mlod_generator_centres(mlod_generator* g, float* out_xyz, const float** d_xyz, void* stream) {
  if (!g) return fail(MLOD_ERR_INVALID, "generator is NULL");
  hipStream_t s = (hipStream_t)stream;
  if (int r = leaf_centres(g, s)) return r;
  if (d_xyz) *d_xyz = g->dXyz;
  if (out_xyz && g->leaves.n) {
    MLOD_HIP(hipMemcpyAsync(out_xyz, g->dXyz, g->leaves.n * 3 * sizeof(float), hipMemcpyDeviceToHost, s));
    MLOD_HIP(hipStreamSynchronize(s));
  }
  return MLOD_OK;
}

}  // extern "C"
