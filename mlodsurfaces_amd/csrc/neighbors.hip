// neighbors.hip — kNN and ball APSS on the GPU (gfx950).
//
// Restates APSSOctree::projectAPSSCPU (sources/apss/CPUUtils.cpp:690-737), which the
// reference runs on the CPU only, over its kd-tree (kdTreeNN.h:416-493):
//   per step: the k nearest input points of the current position (kdTree::knearest) or all
//   points with d^2 <= r^2 (getInBall; r < 0 => 3 sigmas[0]); unit weights w(p_i, q) on the
//   raw points and normals; the sphere fit of projectOnAPSSStats called with q aliased to
//   the output (CPUUtils.cpp:735), so no step clamp applies and a NaN fit leaves a NaN
//   position (normal zeroed); an empty ball returns the step's starting query with a zero
//   normal and ends the iterations (CPUUtils.cpp:711-716).
// Neighbours are found by walking this library's octree with box-distance pruning instead of
// a kd-tree; distances use the kd-tree's arithmetic (float differences, squares summed in
// float, compared as double), so the neighbour sets are the same; the k nearest are ordered
// by (distance, point index).
//
// kNN: one lane per query.  Per depth level the lane keeps in LDS the first child and the
// children still to visit in increasing box distance (so the search reaches the query's own
// leaves first and the k-th distance bound tightens early); small subtrees are scanned as
// contiguous point ranges.  Candidates within the bound are buffered in LDS and merged, by all lanes
// of a wavefront together, into a sorted array of 64-bit keys in registers (distance bits << 32 |
// sorted point index).  The kernel is bound by vector instructions (VALU 93 % busy, k = 32): merging
// together runs the insertion about as often as the fullest lane needs it instead of once per point
// that any lane takes (k = 32, 5M points, 4M queries, FP32C: 12.0 ms a step with 64-bit integer
// compares, 7.7 with keys as doubles, 5.9 with the buffers).  Ball: one walk per wavefront over the union of
// its lanes' balls (k_ball_wave).
#include <cfloat>
#include <cmath>

#include "mlod_internal.h"
#include "weights.h"

namespace mlod {
namespace {

constexpr int NBS = 128;
constexpr int kLevels = kMaxDepth;

#define LAUNCH_CHECK()                                                           \
  do {                                                                           \
    hipError_t e_ = hipGetLastError();                                           \
    if (e_ != hipSuccess) return hip_fail(e_, "kernel launch", __FILE__, __LINE__); \
  } while (0)

template <class T>
struct V3 {
  T x, y, z;
};

// kdTreeNN distance arithmetic (kdTreeNN.h:421, 470): ((dx*dx + dy*dy) + dz*dz) in float.
// This file is compiled without multiply-add contraction.
__device__ __forceinline__ float kd_d2(float4 p, V3<float> q) {
  const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
  return (dx * dx + dy * dy) + dz * dz;
}

// A lower bound of the squared distance from q to the points of a node, from the node's centre (one
// 16-byte record) and the half extents of its depth: `h` holds the root's half extents over 2^depth,
// grown by what float rounding moves a cell's bounds and centre (HalfBox), so the box it spans
// contains the cell.  The cell's own bounds are 24 bytes in three loads (k = 32, 5M points, 4M
// queries: 7.7 ms a step with them, 7.4 with the centres).
struct HalfBox {
  float x, y, z, eps;  // the root's half extents; the rounding margin
};
__device__ __forceinline__ V3<float> half_at(HalfBox hb, uint32_t depth) {
  return V3<float>{ldexpf(hb.x, -(int)depth) + hb.eps, ldexpf(hb.y, -(int)depth) + hb.eps,
                   ldexpf(hb.z, -(int)depth) + hb.eps};
}
__device__ __forceinline__ float cell_d2(float4 g, V3<float> h, V3<float> q) {
  const float dx = fmaxf(fabsf(q.x - g.x) - h.x, 0.f);
  const float dy = fmaxf(fabsf(q.y - g.y) - h.y, 0.f);
  const float dz = fmaxf(fabsf(q.z - g.z) - h.z, 0.f);
  return (dx * dx + dy * dy) + dz * dz;
}

// Bound slack: box distances are float-rounded, so a node is kept while its bound is within
// a relative 1e-4 of the squared search radius (a superset of the exact test).
constexpr float kSlack = 1.0001f;

// kNN: subtrees of at most this many points are scanned rather than walked.
constexpr uint32_t kScanPointsKnn = 8;
// kNN: candidates within the bound are buffered in LDS and merged into the sorted keys by all lanes
// of a wavefront together, once one of them holds kBufFill; a lane scans at most kBufFill points
// between two merges.
constexpr uint32_t kBufFill = 8, kBufCap = 2 * kBufFill - 1;

// Weighted sums of the neighbours (CPUUtils.cpp:719-731): unit area, raw p and n.
struct SumF {  // plain FP32
  float w, px, py, pz, nx, ny, nz, pn, pp;
};
struct KSum {
  float s, c;
  __device__ __forceinline__ void add(float x) {
    const float y = x - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
  }
  __device__ __forceinline__ double val() const { return (double)s - (double)c; }
};
struct SumC {  // compensated, query frame
  KSum w, px, py, pz, nx, ny, nz, pn, pp;
};
struct SumD {
  double w, px, py, pz, nx, ny, nz, pn, pp;
};

template <int FORM>
struct Sums;
template <> struct Sums<0> { using S = SumF; };
template <> struct Sums<1> { using S = SumC; };
template <> struct Sums<2> { using S = SumD; };

template <int FORM, int KT>
__device__ __forceinline__ void add_nb(typename Sums<FORM>::S& s, const KParams& kp, float4 P, float4 N, V3<double> qd,
                                       V3<float> qf) {
  if constexpr (FORM == 0) {
    const float dx = qf.x - P.x, dy = qf.y - P.y, dz = qf.z - P.z;
    const float w = weight32<KT>(kp, (dx * dx + dy * dy) + dz * dz);
    s.pn += w * ((P.x * N.x + P.y * N.y) + P.z * N.z);
    s.pp += w * ((P.x * P.x + P.y * P.y) + P.z * P.z);
    s.px += w * P.x;
    s.py += w * P.y;
    s.pz += w * P.z;
    s.nx += w * N.x;
    s.ny += w * N.y;
    s.nz += w * N.z;
    s.w += w;
  } else if constexpr (FORM == 1) {
    const float dx = P.x - qf.x, dy = P.y - qf.y, dz = P.z - qf.z;
    const float d2 = (dx * dx + dy * dy) + dz * dz;
    const float w = weight32<KT>(kp, d2);
    s.w.add(w);
    s.px.add(w * dx);
    s.py.add(w * dy);
    s.pz.add(w * dz);
    s.nx.add(w * N.x);
    s.ny.add(w * N.y);
    s.nz.add(w * N.z);
    s.pn.add(w * ((dx * N.x + dy * N.y) + dz * N.z));
    s.pp.add(w * d2);
  } else {
    const double x = P.x, y = P.y, z = P.z;
    const double dx = qd.x - x, dy = qd.y - y, dz = qd.z - z;
    const double w = weight64<KT>(kp, dx * dx + dy * dy + dz * dz);
    s.pn += w * ((x * N.x + y * N.y) + z * N.z);
    s.pp += w * ((x * x + y * y) + z * z);
    s.px += w * x;
    s.py += w * y;
    s.pz += w * z;
    s.nx += w * N.x;
    s.ny += w * N.y;
    s.nz += w * N.z;
    s.w += w;
  }
}

template <class T>
__device__ __forceinline__ T dot3(V3<T> a, V3<T> b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

// projectOnAPSSStats with q aliased to the output (CPUUtils.cpp:735, 739-782): plane
// threshold 1e-12, normalize(0) = NaN, NaN positions kept with a zero normal, no step clamp.
// kind: 0 sphere, 1 plane, 2 invalid (NaN position kept, zero normal)
template <class T>
__device__ __forceinline__ void fit_aliased(T sw, V3<T> sp, V3<T> sn, T spn, T spp, V3<T> q, V3<T>& outP, V3<T>& outN,
                                            float& kind) {
  const T A = spn - dot3(sp, V3<T>{sn.x / sw, sn.y / sw, sn.z / sw});
  const T B = spp - dot3(sp, V3<T>{sp.x / sw, sp.y / sw, sp.z / sw});
  const T u4 = (T)((0.5 * (double)A) / (double)B);
  const T t2 = T(2) * u4;
  const V3<T> u{(sn.x - t2 * sp.x) / sw, (sn.y - t2 * sp.y) / sw, (sn.z - t2 * sp.z) / sw};
  const T u0 = -(dot3(sp, u) + u4 * spp) / sw;
  V3<T> p = q, n;
  kind = fabs((double)u4) < 0.000000000001 ? 1.f : 0.f;
  if (fabs((double)u4) < 0.000000000001) {
    const V3<T> nn{-u.x, -u.y, -u.z};
    const T lambda = (u0 - dot3(p, nn)) / dot3(nn, nn);
    p = V3<T>{p.x + lambda * nn.x, p.y + lambda * nn.y, p.z + lambda * nn.z};
    const T inv = T(1) / sqrt(dot3(sn, sn));
    n = V3<T>{sn.x * inv, sn.y * inv, sn.z * inv};
  } else {
    const T m2 = T(-2) * u4;
    const V3<T> c{u.x / m2, u.y / m2, u.z / m2};
    const T v = dot3(c, c) - u0 / u4;
    const T r = sqrt(v > T(0) ? v : T(0));
    const V3<T> d{p.x - c.x, p.y - c.y, p.z - c.z};
    const T inv = T(1) / sqrt(dot3(d, d));
    p = V3<T>{c.x + r * d.x * inv, c.y + r * d.y * inv, c.z + r * d.z * inv};
    const V3<T> g{u.x + t2 * p.x, u.y + t2 * p.y, u.z + t2 * p.z};
    const T ig = T(1) / sqrt(dot3(g, g));
    n = V3<T>{g.x * ig, g.y * ig, g.z * ig};
  }
  if (isnan(p.x) || isnan(p.y) || isnan(p.z)) {
    n = V3<T>{0, 0, 0};
    kind = 2.f;
  }
  outP = p;
  outN = n;
}

template <int FORM>
__device__ __forceinline__ void fit_step(const typename Sums<FORM>::S& s, V3<double>& qd, V3<float> qf, float4& nout) {
  if constexpr (FORM == 0) {
    V3<float> p, n;
    float kind;
    fit_aliased<float>(s.w, V3<float>{s.px, s.py, s.pz}, V3<float>{s.nx, s.ny, s.nz}, s.pn, s.pp, qf, p, n, kind);
    qd = V3<double>{p.x, p.y, p.z};
    nout = make_float4(n.x, n.y, n.z, kind);
  } else if constexpr (FORM == 1) {
    V3<double> p, n;
    float kind;
    fit_aliased<double>(s.w.val(), V3<double>{s.px.val(), s.py.val(), s.pz.val()},
                        V3<double>{s.nx.val(), s.ny.val(), s.nz.val()}, s.pn.val(), s.pp.val(), V3<double>{0, 0, 0}, p, n,
                        kind);
    qd = V3<double>{(double)qf.x + p.x, (double)qf.y + p.y, (double)qf.z + p.z};
    nout = make_float4((float)n.x, (float)n.y, (float)n.z, kind);
  } else {
    V3<double> p, n;
    float kind;
    fit_aliased<double>(s.w, V3<double>{s.px, s.py, s.pz}, V3<double>{s.nx, s.ny, s.nz}, s.pn, s.pp, qd, p, n, kind);
    qd = p;
    nout = make_float4((float)n.x, (float)n.y, (float)n.z, kind);
  }
}

// Sorted (ascending) candidate keys of the k nearest, in registers.  A key is
// (distance bits << 32) | (sorted point index + 1) held as a double: distance bits are those of a
// non-negative float (a NaN is cut to 0x7fc00000), so every key is a finite non-negative double and
// doubles order as the 64-bit integers do.  One slot of the insertion is then v_max_f64 and
// v_min_f64 (full rate on this chip) instead of two 64-bit integer compares and four selects: 64
// vector instructions an insertion at k = 32 against 192.  The first KMAX - k slots hold the
// sentinel 0, smaller than every real key and never displaced, so the k-th smallest real key is
// always the last slot (a static register index); empty slots hold +inf.  Both have a zero low word.
__device__ __forceinline__ double min_key(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double max_key(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double make_key(float d2, uint32_t j) {
  const uint32_t hi = min(__float_as_uint(d2) & 0x7fffffffu, 0x7fc00000u);
  return __hiloint2double((int)hi, (int)(j + 1u));
}

template <int KMAX>
struct TopK {
  double key[KMAX];
  __device__ __forceinline__ void clear(uint32_t k) {
#pragma unroll
    for (int j = 0; j < KMAX; ++j) key[j] = (uint32_t)j < KMAX - k ? 0.0 : (double)INFINITY;
  }
  __device__ __forceinline__ void insert(double x) {
    if (!(x < key[KMAX - 1])) return;
#pragma unroll
    for (int j = KMAX - 1; j > 0; --j) key[j] = min_key(key[j], max_key(key[j - 1], x));
    key[0] = min_key(key[0], x);
  }
  // squared distance of the k-th candidate, infinite while there are fewer
  __device__ __forceinline__ float bound() const {
    const uint32_t hi = (uint32_t)__double2hiint(key[KMAX - 1]);
    return hi == 0x7ff00000u ? INFINITY : __uint_as_float(hi);
  }
};

template <int FORM, int KT, int KMAX>
// The 32 sorted 64-bit keys take 64 VGPRs; the FP32 forms fit four waves per SIMD (119 VGPRs).
__global__ __launch_bounds__(NBS) __attribute__((amdgpu_waves_per_eu(FORM == 2 ? 1 : 3)))
void k_knn(TreeView tv, HalfBox hb, KParams kp,
                                             float4* __restrict__ q, float4* __restrict__ qn,
                                             const uint32_t* __restrict__ perm, uint32_t m, uint32_t limit, uint32_t nIter,
                                             uint32_t k) {
  // per lane: the search's stack (two words a level) and the buffered candidates, then the found
  // indices of the step
  constexpr int kStack = 2 * kLevels, kWords = KMAX > kStack + kBufCap ? KMAX : kStack + kBufCap;
  __shared__ uint32_t sWords[kWords][NBS];
  uint32_t (*sFirst)[NBS] = sWords;            // first child
  uint32_t (*sOrder)[NBS] = sWords + kLevels;  // waiting children, nearest first, 3 bits each; their
                                               // number << 24; their depth << 28
  uint32_t (*sBuf)[NBS] = sWords + kStack;
  const int tid = threadIdx.x;
  const uint32_t i = xcd_block() * NBS + tid;
  if (i >= m) return;
  if (limit < m && perm[i] >= limit) return;
  const float4 q4 = q[i];
  V3<double> qd{q4.x, q4.y, q4.z};
  float4 nout = make_float4(0.f, 0.f, 0.f, 0.f);
  for (uint32_t it = 0; it < nIter; ++it) {
    const V3<float> qf{(float)qd.x, (float)qd.y, (float)qd.z};
    TopK<KMAX> top;
    top.clear(k);
    float bound = INFINITY;  // squared distance of the k-th candidate when last merged
    uint32_t cnt = 0;        // buffered candidates
    // inserts the buffered candidates of every lane (their distances are computed again: the points
    // were just read)
    const auto merge = [&]() {
#pragma unroll 1
      for (uint32_t b = 0; b < cnt; ++b) {
        const uint32_t j = sBuf[b][tid];
        top.insert(make_key(kd_d2(tv.pts[j], qf), j));
      }
      cnt = 0;
      bound = top.bound();
    };
    int lvl = -1;
    uint32_t cur = 0;         // node to expand next (root first)
    uint32_t sa = 0, sb = 0;  // points still to scan
    bool have = true;
    while (true) {
      if (have) {
        const uint4 h = tv.hdr[cur];
        const uint2 sp = tv.span[cur];
        have = false;
        if (hdr_leaf(h.y) || sp.y - sp.x <= kScanPointsKnn) {
          // a leaf or a small subtree: every point is a candidate (the k nearest do not depend
          // on the order they are offered in)
          sa = sp.x;
          sb = sp.y;
        } else {
          // children whose box reaches the bound, visited nearest box first, so that the
          // first leaves reached are the query's own and the bound tightens at once
          const uint32_t first = h.x, nc = hdr_count(h.y);
          const V3<float> hc = half_at(hb, hdr_depth(h.y) + 1u);
          // keys: the box distance's bits (non-negative floats order as integers) with the child
          // slot in the low 3 bits, children beyond the bound last; an 8-input sorting network
          // (19 compare-exchanges) orders them.  The visiting order only steers the search: the
          // k nearest do not depend on it.  All eight centres are loaded before the first is used
          float4 g[8];
#pragma unroll
          for (uint32_t c = 0; c < 8; ++c) g[c] = tv.geo[first + min(c, nc - 1u)];
          uint32_t key[8], n = 0;
#pragma unroll
          for (uint32_t c = 0; c < 8; ++c) {
            const float d = cell_d2(g[c], hc, qf);
            const bool in = c < nc && d <= bound * kSlack;
            key[c] = in ? (__float_as_uint(d) & ~7u) | c : 0xffffffffu;
            n += in ? 1u : 0u;
          }
          const auto cx = [&](int a, int b) {
            const uint32_t lo = min(key[a], key[b]), hi = max(key[a], key[b]);
            key[a] = lo, key[b] = hi;
          };
          cx(0, 2), cx(1, 3), cx(4, 6), cx(5, 7), cx(0, 4), cx(1, 5), cx(2, 6), cx(3, 7), cx(0, 1), cx(2, 3);
          cx(4, 5), cx(6, 7), cx(2, 4), cx(3, 5), cx(1, 4), cx(3, 6), cx(1, 2), cx(3, 4), cx(5, 6);
          uint32_t order = (hdr_depth(h.y) + 1u) << 28 | n << 24;
#pragma unroll
          for (uint32_t r = 0; r < 8; ++r) order |= (key[r] & 7u) << (3u * r);
          if (n) {
            ++lvl;
            sFirst[lvl][tid] = first;
            sOrder[lvl][tid] = order;
          }
        }
      }
      // scan at most kBufFill points: those that the bound does not rule out are buffered
      for (uint32_t e = min(sb, sa + kBufFill); sa < e; ++sa) {
        if (!(kd_d2(tv.pts[sa], qf) > bound)) {
          sBuf[cnt][tid] = sa;
          ++cnt;
        }
      }
      if (__any(cnt >= kBufFill)) merge();
      if (sa < sb) continue;
      if (lvl < 0) break;
      const uint32_t w = sOrder[lvl][tid];
      const uint32_t c = sFirst[lvl][tid] + (w & 7u);
      const uint32_t rest = ((w & 0xffffffu) >> 3) + (w & 0xff000000u) - (1u << 24);
      sOrder[lvl][tid] = rest;
      if (!(rest & 0x0f000000u)) --lvl;
      if (cell_d2(tv.geo[c], half_at(hb, w >> 28), qf) <= bound * kSlack) {  // the bound may have shrunk since the push
        cur = c;
        have = true;
      }
    }
    merge();
    // the found indices through this lane's own LDS column (a rolled loop cannot index registers),
    // summed nearest first
#pragma unroll
    for (int j = 0; j < KMAX; ++j) sWords[j][tid] = (uint32_t)__double2loint(top.key[j]);
    typename Sums<FORM>::S s{};
#pragma unroll 1
    for (uint32_t j = KMAX - k; j < KMAX; ++j) {
      const uint32_t pj = sWords[j][tid];
      if (pj == 0u) break;  // fewer than k points (of a finite distance) found
      add_nb<FORM, KT>(s, kp, tv.pts[pj - 1u], tv.nrm[pj - 1u], qd, qf);
    }
    fit_step<FORM>(s, qd, qf, nout);
  }
  q[i] = make_float4((float)qd.x, (float)qd.y, (float)qd.z, 0.f);
  qn[i] = nout;
}

// Ball APSS, one wavefront at a time.  A wavefront's queries are neighbours on the curve, so their
// balls overlap almost entirely: the wavefront walks the octree once over the union of its
// balls (node boxes against its queries' box grown by r), takes the points of every
// reached subtree that is small enough as a contiguous range, and loads each range 64 points at a
// time with one coalesced load per lane; every query sums the points inside its own ball.  Ranges
// come in increasing point order, so a query sums exactly the points inside its ball, in increasing
// point order (the order of a walk over its own ball alone), whatever the wavefront's other queries.
__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float bcast(float v, uint32_t lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), (int)lane));
}

// squared distance between a node's box and the box [lo, hi]
__device__ __forceinline__ float box_box_d2(const float* __restrict__ box, uint32_t c, V3<float> lo, V3<float> hi) {
  const float2 a = *reinterpret_cast<const float2*>(box + 6 * (size_t)c);
  const float2 b = *reinterpret_cast<const float2*>(box + 6 * (size_t)c + 2);
  const float2 e = *reinterpret_cast<const float2*>(box + 6 * (size_t)c + 4);
  const float dx = fmaxf(fmaxf(a.x - hi.x, lo.x - b.y), 0.f);
  const float dy = fmaxf(fmaxf(a.y - hi.y, lo.y - e.x), 0.f);
  const float dz = fmaxf(fmaxf(b.x - hi.z, lo.z - e.y), 0.f);
  return (dx * dx + dy * dy) + dz * dz;
}

constexpr uint32_t kWaveScanPoints = 256;  // subtrees up to this size are taken as one range

// The plain FP32 form, and every form of a cloud with points that are not finite (see k_ball_sums): the form's own
// sums one after another, 64 queries a wavefront, each point broadcast lane to lane.
template <int FORM, int KT>
__global__ __launch_bounds__(NBS) void k_ball_wave(TreeView tv, const float* __restrict__ box, KParams kp,
                                                   float4* __restrict__ q, float4* __restrict__ qn,
                                                   const uint32_t* __restrict__ perm, uint32_t m, uint32_t limit,
                                                   uint32_t nIter, float r2f) {
  constexpr int kWaves = NBS / 64;
  __shared__ uint32_t sFirst[kLevels][kWaves];
  __shared__ uint32_t sMask[kLevels][kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const uint32_t i = xcd_block() * NBS + tid;
  const uint32_t i0 = i - (uint32_t)lane;  // the wavefront's first slot
  if (i0 >= m) return;                      // whole wavefront past the end
  const bool mine = i < m && !(limit < m && perm[i] >= limit);
  // lanes without a query of their own follow the wavefront's first query (never stored)
  const float4 q4 = q[i < m ? i : i0];
  V3<double> qd{q4.x, q4.y, q4.z};
  float4 nout = make_float4(0.f, 0.f, 0.f, 0.f);
  bool done = !mine;
  const float r = sqrtf(r2f) * kSlack;
  for (uint32_t it = 0; it < nIter; ++it) {
    const V3<float> qf{(float)qd.x, (float)qd.y, (float)qd.z};
    // the union of the live lanes' balls, bounded by their query box grown by r
    const float big = 3.0e38f;
    const V3<float> qlo{wave_min(done ? big : qf.x) - r, wave_min(done ? big : qf.y) - r, wave_min(done ? big : qf.z) - r};
    const V3<float> qhi{wave_max(done ? -big : qf.x) + r, wave_max(done ? -big : qf.y) + r, wave_max(done ? -big : qf.z) + r};
    if (qlo.x > qhi.x) break;  // every lane finished (uniform)
    typename Sums<FORM>::S s{};
    uint32_t cnt = 0;
    int lvl = -1;
    uint32_t cur = 0;
    bool have = true;
    while (true) {
      if (have) {
        const uint4 h = tv.hdr[cur];
        const uint2 sp = tv.span[cur];
        if (hdr_leaf(h.y) || sp.y - sp.x <= kWaveScanPoints) {
          // the range's points, 64 at a time: one coalesced load per lane, then each point
          // is broadcast and tested by every lane
          for (uint32_t base = sp.x; base < sp.y; base += 64) {
            const uint32_t nb = min(64u, sp.y - base);
            const uint32_t j = base + (uint32_t)lane;
            const float4 P = (uint32_t)lane < nb ? tv.pts[j] : make_float4(0.f, 0.f, 0.f, 0.f);
            const float4 N = (uint32_t)lane < nb ? tv.nrm[j] : make_float4(0.f, 0.f, 0.f, 0.f);
            for (uint32_t t = 0; t < nb; ++t) {
              const float4 Pt = make_float4(bcast(P.x, t), bcast(P.y, t), bcast(P.z, t), bcast(P.w, t));
              if (!done && kd_d2(Pt, qf) <= r2f) {
                const float4 Nt = make_float4(bcast(N.x, t), bcast(N.y, t), bcast(N.z, t), 0.f);
                add_nb<FORM, KT>(s, kp, Pt, Nt, qd, qf);
                ++cnt;
              }
            }
          }
        } else {
          const uint32_t first = __builtin_amdgcn_readfirstlane(h.x), nc = hdr_count(h.y);
          uint32_t mask = 0;
          for (uint32_t c = 0; c < nc; ++c)
            if (box_box_d2(box, first + c, qlo, qhi) <= 0.f) mask |= 1u << c;
          ++lvl;
          if (lane == 0) {
            sFirst[lvl][wv] = first;
            sMask[lvl][wv] = mask;
          }
        }
        have = false;
      }
      if (lvl < 0) break;
      const uint32_t mask = __builtin_amdgcn_readfirstlane(sMask[lvl][wv]);
      if (mask == 0) {
        --lvl;
        continue;
      }
      if (lane == 0) sMask[lvl][wv] = mask & (mask - 1u);
      cur = __builtin_amdgcn_readfirstlane(sFirst[lvl][wv]) + (uint32_t)__builtin_ctz(mask);
      have = true;
    }
    if (!done) {
      if (cnt == 0) {  // empty ball: the starting query, zero normal (CPUUtils.cpp:711-716)
        qd = V3<double>{q4.x, q4.y, q4.z};
        nout = make_float4(0.f, 0.f, 0.f, 0.f);
        done = true;
      } else {
        fit_step<FORM>(s, qd, qf, nout);
      }
    }
  }
  if (mine) {
    q[i] = make_float4((float)qd.x, (float)qd.y, (float)qd.z, 0.f);
    qn[i] = nout;
  }
}

// One step from FP64 sums over the neighbours (CPUUtils.cpp:719-735) about `o`, which is 0 in the FP64 form; the
// compensated form moves them to the query's frame.
template <int FORM>
__device__ __forceinline__ void fit_sums(const double* S, V3<float> o, V3<double>& qd, V3<float> qf, float4& nout) {
  V3<double> p, n;
  float kind;
  const V3<double> sp{S[1], S[2], S[3]}, sn{S[4], S[5], S[6]};
  if constexpr (FORM == 1) {
    const V3<double> q{(double)qf.x - o.x, (double)qf.y - o.y, (double)qf.z - o.z};
    fit_aliased<double>(S[0], V3<double>{sp.x - q.x * S[0], sp.y - q.y * S[0], sp.z - q.z * S[0]}, sn, S[7] - dot3(q, sn),
                        S[8] - 2.0 * dot3(q, sp) + dot3(q, q) * S[0], V3<double>{0, 0, 0}, p, n, kind);
    qd = V3<double>{(double)qf.x + p.x, (double)qf.y + p.y, (double)qf.z + p.z};
  } else {
    fit_aliased<double>(S[0], sp, sn, S[7], S[8], qd, p, n, kind);
    qd = p;
  }
  nout = make_float4((float)n.x, (float)n.y, (float)n.z, kind);
}

// Orders a wavefront's own LDS writes and reads (its LDS operations complete in order).
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

typedef double Acc4 __attribute__((ext_vector_type(4)));

// The compensated and FP64 forms: a wavefront walks the union of 16 queries' balls, the sums on the matrix cores. A
// range's points go to LDS 64 at a time with their nine moments {1, p, n, p.n, |p|^2} in FP64; then, four points a
// step and four steps at once, each lane weighs one (query lane % 16, point lane / 16) pair a step, a pair outside
// its ball with weight 0, and an FP64 16x16x4 matrix instruction adds the 64 weights times the points' moments. A
// pair so costs its distance, test and weight and none of the nine sums. The ranges and the steps within them are
// the tree's, whatever the queries, and a zero weight leaves a sum as it is: a query's sums do not depend on its
// wavefront's other queries. That holds for finite moments only (0 * NaN and 0 * infinity are NaN), so a cloud with
// a point that is not finite goes to k_ball_wave, which leaves out what a ball does not hold (adding such points
// apart in this kernel took 14 more registers, a wavefront a SIMD, and 7 % of every other cloud's time). The
// compensated form's sums are about a point of the cloud, the middle one in the tree's order, and moved to the
// query at the end: that costs 1e-16 of the squared distance between the two over the neighbourhood's, where the
// global frame costs it of the squared coordinates (a cloud 1e4 of its sizes from the origin, four sigmas of a
// twentieth: normals off by up to 1e-6, with the middle point 4e-8). Bound by the weights' vector instructions at high
// query counts (500k: 58 % of the SIMDs' cycles, the matrix instructions 18 %), by the walk's
// loads at low ones. r = 3 sigma0, 1M points (about 300 a ball), FP32C: 500k queries 4.8 -> 1.5 ms, 20k 1.0, 2k
// 1.3; FP64, 100k queries 1.6 (1.3 with weights.h's exponential). Wavefronts of 64 queries (unions of four times
// the surface, four times fewer wavefronts): 2.9, 3.1, 10.6, 4.6; of 32: 1.8, 1.5, 2.7, 2.5.
constexpr uint32_t kBallQ = 16;            // queries a wavefront
constexpr uint32_t kScanPointsBall = 512;  // subtrees up to this size are taken as one range (256: 1.65 ms, 1024: 1.57)

template <int FORM, int KT>
__global__ __launch_bounds__(NBS) void k_ball_sums(TreeView tv, const float* __restrict__ box, KParams kp,
                                                   float4* __restrict__ q, float4* __restrict__ qn,
                                                   const uint32_t* __restrict__ perm, uint32_t m, uint32_t limit,
                                                   uint32_t nIter, float r2f) {
  constexpr int kWaves = NBS / 64, U = 4;  // steps at once
  __shared__ uint32_t sFirst[kLevels][kWaves];
  __shared__ uint32_t sMask[kLevels][kWaves];
  __shared__ float4 sPts[kWaves][64];
  __shared__ double sMom[kWaves][64][9];  // then the wavefront's sums, 16 queries x 9
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t row = (uint32_t)lane & 15u, kk = (uint32_t)lane >> 4, col = min(row, 8u);
  const uint32_t i0 = (xcd_block() * kWaves + (uint32_t)wv) * kBallQ;  // the wavefront's first slot
  const uint32_t i = i0 + (uint32_t)lane;
  if (i0 >= m) return;  // whole wavefront past the end
  const bool mine = lane < (int)kBallQ && i < m && !(limit < m && perm[i] >= limit);
  // lanes without a query of their own follow the wavefront's first query (never stored)
  const float4 q4 = q[mine ? i : i0];
  V3<double> qd{q4.x, q4.y, q4.z};
  float4 nout = make_float4(0.f, 0.f, 0.f, 0.f);
  bool done = !mine;
  const float r = sqrtf(r2f) * kSlack;
  const float4 mid = tv.pts[tv.n >> 1];
  const V3<float> o = FORM == 1 ? V3<float>{mid.x, mid.y, mid.z} : V3<float>{0.f, 0.f, 0.f};  // the sums' origin
  float4* pts = sPts[wv];
  double (*mom)[9] = sMom[wv];
  for (uint32_t it = 0; it < nIter; ++it) {
    const V3<float> qf{(float)qd.x, (float)qd.y, (float)qd.z};
    // the union of the live lanes' balls, bounded by their query box grown by r
    const float big = 3.0e38f;
    const V3<float> qlo{wave_min(done ? big : qf.x) - r, wave_min(done ? big : qf.y) - r, wave_min(done ? big : qf.z) - r};
    const V3<float> qhi{wave_max(done ? -big : qf.x) + r, wave_max(done ? -big : qf.y) + r, wave_max(done ? -big : qf.z) + r};
    if (qlo.x > qhi.x) break;  // every lane finished (uniform)
    const V3<float> g{__shfl(qf.x, (int)row, 64), __shfl(qf.y, (int)row, 64), __shfl(qf.z, (int)row, 64)};  // the pairs' query
    V3<double> gd{0, 0, 0};
    if constexpr (FORM == 2)
      gd = V3<double>{__shfl(qd.x, (int)row, 64), __shfl(qd.y, (int)row, 64), __shfl(qd.z, (int)row, 64)};
    Acc4 acc{0, 0, 0, 0};
    bool some = false;
    int lvl = -1;
    uint32_t cur = 0;
    bool have = true;
    while (true) {
      if (have) {
        const uint4 h = tv.hdr[cur];
        const uint2 sp = tv.span[cur];
        if (hdr_leaf(h.y) || sp.y - sp.x <= kScanPointsBall) {
          const uint32_t a = __builtin_amdgcn_readfirstlane(sp.x), b = __builtin_amdgcn_readfirstlane(sp.y);
          for (uint32_t base = a; base < b; base += 64) {
            const uint32_t nb = min(64u, b - base);
            const bool in = (uint32_t)lane < nb;  // past the end: the first point with no moments
            const float4 P = tv.pts[base + (in ? (uint32_t)lane : 0u)], N = tv.nrm[base + (in ? (uint32_t)lane : 0u)];
            const double e = in ? 1.0 : 0.0, x = (double)P.x - o.x, y = (double)P.y - o.y, z = (double)P.z - o.z;
            const double nx = N.x, ny = N.y, nz = N.z;
            pts[lane] = P;
            mom[lane][0] = e;
            mom[lane][1] = e * x, mom[lane][2] = e * y, mom[lane][3] = e * z;
            mom[lane][4] = e * nx, mom[lane][5] = e * ny, mom[lane][6] = e * nz;
            mom[lane][7] = e * ((x * nx + y * ny) + z * nz);
            mom[lane][8] = e * ((x * x + y * y) + z * z);
            wave_order();
            for (uint32_t t0 = kk; t0 < nb + kk; t0 += 4 * U) {  // uniform
              float d2[U];
              bool hit[U], any = false;
#pragma unroll
              for (int v = 0; v < U; ++v) {
                d2[v] = kd_d2(pts[t0 + 4 * v], g);
                hit[v] = d2[v] <= r2f;
                any |= hit[v];
              }
              if (__builtin_amdgcn_ballot_w64(any) == 0ull) continue;  // uniform
              double w[U];
              if constexpr (FORM == 2) {
#pragma unroll
                for (int v = 0; v < U; ++v) {
                  const float4 Pt = pts[t0 + 4 * v];
                  const double dx = gd.x - (double)Pt.x, dy = gd.y - (double)Pt.y, dz = gd.z - (double)Pt.z;
                  w[v] = weight64<KT>(kp, dx * dx + dy * dy + dz * dz);
                }
              } else {
                float wf[U];
                weights32<KT, U>(kp, d2, wf);
#pragma unroll
                for (int v = 0; v < U; ++v) w[v] = (double)wf[v];
              }
#pragma unroll
              for (int v = 0; v < U; ++v)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(hit[v] ? w[v] : 0.0, mom[t0 + 4 * v][col], acc, 0, 0, 0);
              some |= any;
            }
            wave_order();
          }
        } else {
          const uint32_t first = __builtin_amdgcn_readfirstlane(h.x), nc = hdr_count(h.y);
          uint32_t mask = 0;
          for (uint32_t c = 0; c < nc; ++c)
            if (box_box_d2(box, first + c, qlo, qhi) <= 0.f) mask |= 1u << c;
          ++lvl;
          if (lane == 0) {
            sFirst[lvl][wv] = first;
            sMask[lvl][wv] = mask;
          }
        }
        have = false;
      }
      if (lvl < 0) break;
      const uint32_t mask = __builtin_amdgcn_readfirstlane(sMask[lvl][wv]);
      if (mask == 0) {
        --lvl;
        continue;
      }
      if (lane == 0) sMask[lvl][wv] = mask & (mask - 1u);
      cur = __builtin_amdgcn_readfirstlane(sFirst[lvl][wv]) + (uint32_t)__builtin_ctz(mask);
      have = true;
    }
    // register v of a lane holds query 4 v + lane / 16, moment lane % 16
    const uint64_t b = __builtin_amdgcn_ballot_w64(some);
    const uint32_t found = (uint32_t)(b | b >> 16 | b >> 32 | b >> 48) & 0xffffu;  // queries with a point in their ball
    if (row < 9u) {
#pragma unroll
      for (uint32_t v = 0; v < 4; ++v) mom[4u * v + kk][row] = acc[v];
    }
    wave_order();
    if (!done) {
      if (!((found >> lane) & 1u)) {  // empty ball: the starting query, zero normal (CPUUtils.cpp:711-716)
        qd = V3<double>{q4.x, q4.y, q4.z};
        nout = make_float4(0.f, 0.f, 0.f, 0.f);
        done = true;
      } else {
        double S[9];
#pragma unroll
        for (int c = 0; c < 9; ++c) S[c] = mom[lane][c];
        fit_sums<FORM>(S, o, qd, qf, nout);
      }
    }
    wave_order();
  }
  if (mine) {
    q[i] = make_float4((float)qd.x, (float)qd.y, (float)qd.z, 0.f);
    qn[i] = nout;
  }
}

// The root's half extents and the rounding margin of a cell's bounds.  Every bound of a cell is the
// root's or a split rounded to float, so it is within 2^-24 M of the exact halving of its own
// level's bounds (M: the largest |coordinate| of the root box); those errors halve from level to
// level, so an extent is within 4 * 2^-24 M of the root's over 2^depth, and the centre is rounded once
// more.  The products and sums here and in the kernel round too: 16 * 2^-24 M covers them all.
HalfBox half_box(const mlod_tree* t) {
  float m = 0.f, h[3];
  for (int a = 0; a < 3; ++a) {
    m = fmaxf(m, fmaxf(fabsf(t->bb[a]), fabsf(t->BB[a])));
    h[a] = 0.5f * (t->BB[a] - t->bb[a]);
  }
  return HalfBox{h[0], h[1], h[2], m * (16.f / 16777216.f)};
}

template <int FORM, int KT>
int launch_form(mlod_tree* t, const KParams& kp, uint32_t limit, uint32_t nIter, hipStream_t s) {
  const uint32_t m = t->qs.m;
  const uint32_t grid = (m + NBS - 1) / NBS;
  if (t->mode == MLOD_MODE_KNN) {
    const uint32_t k = t->knn < t->n ? t->knn : t->n;
    if (k <= 8)
      k_knn<FORM, KT, 8><<<grid, NBS, 0, s>>>(t->view(), half_box(t), kp, t->qs.q, t->qs.qn, t->qs.perm, m, limit, nIter, k);
    else if (k <= 16)
      k_knn<FORM, KT, 16><<<grid, NBS, 0, s>>>(t->view(), half_box(t), kp, t->qs.q, t->qs.qn, t->qs.perm, m, limit, nIter, k);
    else if (k <= 32)
      k_knn<FORM, KT, 32><<<grid, NBS, 0, s>>>(t->view(), half_box(t), kp, t->qs.q, t->qs.qn, t->qs.perm, m, limit, nIter, k);
    else if (k <= 64)
      k_knn<FORM, KT, 64><<<grid, NBS, 0, s>>>(t->view(), half_box(t), kp, t->qs.q, t->qs.qn, t->qs.perm, m, limit, nIter, k);
    else
      return fail(MLOD_ERR_UNSUPPORTED, "kNN supports k <= 64");
  } else {
    // getInBall(q, r) with r = sigmas[0] * 3 when r < 0 (CPUUtils.cpp:706-709), d^2 <= r*r in
    // double; r2f is the largest float not above r*r, so a float compare is the same test.
    float r = t->ball_radius;
    if (r < 0.f) {
      if (t->kernel.type != MLOD_KERNEL_GAUSSIAN_MULTIPLE || t->kernel.n_sigmas < 1)
        return fail(MLOD_ERR_INVALID, "ball radius < 0 needs a multi-Gaussian kernel (3 sigmas[0])");
      r = t->kernel.sigmas[0] * 3;
    }
    const double r2 = (double)r * (double)r;
    float r2f = (float)r2;
    if ((double)r2f > r2) r2f = nextafterf(r2f, 0.f);
    if (FORM == 0 || !t->finite)
      k_ball_wave<FORM, KT><<<grid, NBS, 0, s>>>(t->view(), t->box, kp, t->qs.q, t->qs.qn, t->qs.perm, m, limit, nIter, r2f);
    else
      k_ball_sums<FORM == 0 ? 1 : FORM, KT><<<(m + kBallQ * (NBS / 64) - 1) / (kBallQ * (NBS / 64)), NBS, 0, s>>>(t->view(), t->box, kp, t->qs.q, t->qs.qn, t->qs.perm, m, limit, nIter, r2f);
  }
  LAUNCH_CHECK();
  return MLOD_OK;
}

template <int FORM>
int launch_kt(mlod_tree* t, const KParams& kp, uint32_t limit, uint32_t nIter, hipStream_t s) {
  switch (kp.type) {
    case MLOD_KERNEL_GAUSSIAN: return launch_form<FORM, MLOD_KERNEL_GAUSSIAN>(t, kp, limit, nIter, s);
    case MLOD_KERNEL_SINGULAR: return launch_form<FORM, MLOD_KERNEL_SINGULAR>(t, kp, limit, nIter, s);
    default: return launch_form<FORM, MLOD_KERNEL_GAUSSIAN_MULTIPLE>(t, kp, limit, nIter, s);
  }
}

}  // namespace

int launch_neighbors(mlod_tree* t, uint32_t n, uint32_t n_iter, hipStream_t s) {
  const KParams kp = make_kparams(t->kernel);
  switch (t->precision) {
    case MLOD_PREC_FP32C: return launch_kt<1>(t, kp, n, n_iter, s);
    case MLOD_PREC_FP64: return launch_kt<2>(t, kp, n, n_iter, s);
    default: return launch_kt<0>(t, kp, n, n_iter, s);
  }
}

}  // namespace mlod
