// project.hip — MLoD and global APSS projection kernels (gfx950).
//
// One lane per query (queries sorted along a curve by queries.hip, so a wavefront's 64 lanes walk
// neighbouring parts of the tree).  The MLoD sum of the reference,
//   value(leaf)  = sum over its points of w(p_i) stats_i                (Fastapss.cu:189-200)
//   value(far)   = w(pbar) stats                                        (Fastapss.cu:214-237)
//   value(near)  = sum_c [ b_c value(c) + (1 - b_c) share_c w(pbar) stats ] (Fastapss.cu:238-299,
//                  CPUUtils.cpp:478-501; b_c = (1 - cos(pi t))/2, t = dP / (dP + dC))
//   value(depth < minDepth) = sum_c value(c)                            (Fastapss.cu:303-329)
// is linear in the stats, so it is evaluated top-down: each node carries the product m of
// the blend factors on its path and adds m * (its own term) to one accumulator.  That needs
// no per-depth accumulator stack (the reference keeps 12 of them per thread); the per-lane
// traversal state is, per depth level, the first child and a mask of children still to descend,
// held in LDS.  A near node
// loops over its contiguous children once: far children and leaves are summed right there, the
// parent's (1 - b_c) share is accumulated, and only near internal children are left in the mask.
//
// Arithmetic forms (template FORM):
//   0 plain FP32   — global-frame moments and the reference's FP32 sphere fit;
//   1 FP32C        — node-centred moments, contributions recentred on the query
//                    (sum w a (p - q), sum w a |p - q|^2, ...), Kahan-compensated FP32
//                    accumulation, FP64 sphere fit in the query frame;
//   2 plain FP64   — everything in double.
// Semantics (template SEM): 0 = REF_GPU (Fastapss.cu), 1 = REF_CPU (CPUUtils.cpp), see
// mlod.h.  Weight kernels (template KT): Kernel.h:37 numbering.
#include <cfloat>
#include <cmath>

#include "mlod_internal.h"
#include "weights.h"

namespace mlod {
namespace {

constexpr int PBS = 128;         // lanes per workgroup
// Levels of the LDS stack of waiting nodes.  A node waits only while it has more than one near
// child still to expand, and near children are internal nodes; internal nodes have depth
// 0..kMaxDepth - 1 and their children depth <= kMaxDepth, so a waiting node has depth at most
// kMaxDepth - 2 (its near children are internal, hence of depth <= kMaxDepth - 1): 11 levels.
constexpr int kLevels = kMaxDepth - 1;

#define LAUNCH_CHECK()                                                           \
  do {                                                                           \
    hipError_t e_ = hipGetLastError();                                           \
    if (e_ != hipSuccess) return hip_fail(e_, "kernel launch", __FILE__, __LINE__); \
  } while (0)

// Level blending (1 - cos(pi x)) / 2 (CPUUtils.cpp:400-408, Fastapss.cu:84-95).  The FP32
// form uses the hardware cosine, which takes revolutions: cos(pi x) = cos_rev(x / 2).
__device__ __forceinline__ float blend(float x) { return 0.5f - 0.5f * __builtin_amdgcn_cosf(0.5f * x); }
// In FP64 (x in [0, 1], 3.14159265 x as the reference has it): (1 + sin(u)) / 2 with u = 3.14159265 x - pi/2, the
// Taylor series of the sine to the 21st power (remainder 1.3e-18 at |u| = pi/2).  Exactly 1 at x = 1.
__device__ __forceinline__ double blend(double x) {
  const double u = fma(x, 3.14159265, -1.5707963267948966), z = u * u;
  double p = 1.9572941063391263e-20;
  p = fma(p, z, -8.22063524662433e-18);
  p = fma(p, z, 2.8114572543455206e-15);
  p = fma(p, z, -7.647163731819816e-13);
  p = fma(p, z, 1.6059043836821613e-10);
  p = fma(p, z, -2.505210838544172e-08);
  p = fma(p, z, 2.7557319223985893e-06);
  p = fma(p, z, -0.0001984126984126984);
  p = fma(p, z, 0.008333333333333333);
  p = fma(p, z, -0.16666666666666666);
  return fma(0.5, fma(u * z, p, u), 0.5);
}

__device__ __forceinline__ float fsqrt(float x) { return __builtin_sqrtf(x); }
__device__ __forceinline__ double fsqrt(double x) { return sqrt(x); }

// ----------------------------------------------------------------------------- accumulators
struct KSum {
  float s, c;
  __device__ __forceinline__ void init() { s = 0.f, c = 0.f; }
  __device__ __forceinline__ void add(float x) {
    const float y = __fsub_rn(x, c);
    const float t = __fadd_rn(s, y);
    c = __fsub_rn(__fsub_rn(t, s), y);
    s = t;
  }
  __device__ __forceinline__ double val() const { return (double)s - (double)c; }
};

template <class T>
struct V3 {
  T x, y, z;
};

// FORM 0: plain global-frame FP32 sums (apssStatsGPU, GPUUtils.cu:318-392)
struct AccP32 {
  float w, px, py, pz, nx, ny, nz, pn, pp;
  __device__ __forceinline__ void init() { w = px = py = pz = nx = ny = nz = pn = pp = 0.f; }
};
// FORM 1: compensated, query-frame.  Terms go by one FMA each into plain FP32 partial sums (the
// l* members), which are added into the Kahan-compensated sums every kFlush traversal iterations
// and at the end of a walk (flush()): the compensation is paid once per block of terms, and a
// block's rounding error is bounded by its few terms.
constexpr uint32_t kFlush = 8;
struct AccC32 {
  KSum w, px, py, pz, nx, ny, nz, pn, pp;
  float lw, lpx, lpy, lpz, lnx, lny, lnz, lpn, lpp;
  __device__ __forceinline__ void init() {
    w.init(), px.init(), py.init(), pz.init(), nx.init(), ny.init(), nz.init(), pn.init(), pp.init();
    lw = lpx = lpy = lpz = lnx = lny = lnz = lpn = lpp = 0.f;
  }
  __device__ __forceinline__ void flush() {
    w.add(lw), px.add(lpx), py.add(lpy), pz.add(lpz), nx.add(lnx), ny.add(lny), nz.add(lnz), pn.add(lpn), pp.add(lpp);
    lw = lpx = lpy = lpz = lnx = lny = lnz = lpn = lpp = 0.f;
  }
};
// FORM 2: plain FP64
struct AccP64 {
  double w, px, py, pz, nx, ny, nz, pn, pp;
  __device__ __forceinline__ void init() { w = px = py = pz = nx = ny = nz = pn = pp = 0.0; }
};

template <int FORM> struct FormT;
template <> struct FormT<0> { using T = float;  using Acc = AccP32; };
template <> struct FormT<1> { using T = float;  using Acc = AccC32; };
template <> struct FormT<2> { using T = double; using Acc = AccP64; };

struct Counters {
  uint32_t far_, leafPts, tested, nearN, iters;
};

// A point's mean position (a p) / a in the plain form.  EXACT: areas of any exponent (a subnormal one's reciprocal
// overflows, that of one above 2^126 is flushed), the compiler's division; see areas_normal.
template <bool EXACT>
__device__ __forceinline__ V3<float> point_mean(float4 P) {
  const float a = P.w, apx = a * P.x, apy = a * P.y, apz = a * P.z;
  if constexpr (EXACT)
    return V3<float>{apx / a, apy / a, apz / a};
  else
    return V3<float>{quot(apx, a), quot(apy, a), quot(apz, a)};
}
template <int KT, class KP>
__device__ __forceinline__ void add_point_plain(AccP32& acc, const KP& kp, float4 P, float4 N, V3<float> mean, V3<float> q,
                                                float f) {
  const float a = P.w;
  const float apx = a * P.x, apy = a * P.y, apz = a * P.z;
  const float dx = mean.x - q.x, dy = mean.y - q.y, dz = mean.z - q.z;
  const float w = f * weight32<KT>(kp, fmaf(dz, dz, fmaf(dx, dx, __fmul_rn(dy, dy))));
  acc.w = fmaf(w, a, acc.w);
  acc.px = fmaf(w, apx, acc.px);
  acc.py = fmaf(w, apy, acc.py);
  acc.pz = fmaf(w, apz, acc.pz);
  acc.nx = fmaf(w, a * N.x, acc.nx);
  acc.ny = fmaf(w, a * N.y, acc.ny);
  acc.nz = fmaf(w, a * N.z, acc.nz);
  acc.pn = fmaf(w, a * (P.x * N.x + P.y * N.y + P.z * N.z), acc.pn);
  acc.pp = fmaf(w, a * (P.x * P.x + P.y * P.y + P.z * P.z), acc.pp);
}

// Contribution of one point (leaf member) with multiplier f, weight at the point's mean
// position (a p) / a (Fastapss.cu:193; CPUUtils.cpp:455).
template <int FORM, int KT, bool EXACT, class KP>
__device__ __forceinline__ void add_point(typename FormT<FORM>::Acc& acc, const KP& kp, const TreeView& tv, uint32_t j,
                                          V3<typename FormT<FORM>::T> q, typename FormT<FORM>::T f) {
  const float4 P = tv.pts[j], N = tv.nrm[j];
  if constexpr (FORM == 0) {
    add_point_plain<KT>(acc, kp, P, N, point_mean<EXACT>(P), q, f);
  } else if constexpr (FORM == 1) {
    // the fused operations are written out: every kernel that adds a point rounds alike
    const float dx = P.x - q.x, dy = P.y - q.y, dz = P.z - q.z;
    const float d2 = fmaf(dz, dz, fmaf(dx, dx, __fmul_rn(dy, dy)));
    const float fw = __fmul_rn(f, weight32<KT>(kp, d2));
    const float fa = __fmul_rn(fw, P.w);
    acc.lw = fmaf(fw, P.w, acc.lw);
    acc.lpx = fmaf(fa, dx, acc.lpx);
    acc.lpy = fmaf(fa, dy, acc.lpy);
    acc.lpz = fmaf(fa, dz, acc.lpz);
    acc.lnx = fmaf(fa, N.x, acc.lnx);
    acc.lny = fmaf(fa, N.y, acc.lny);
    acc.lnz = fmaf(fa, N.z, acc.lnz);
    acc.lpn = fmaf(fa, fmaf(dz, N.z, fmaf(dx, N.x, __fmul_rn(dy, N.y))), acc.lpn);
    acc.lpp = fmaf(fa, d2, acc.lpp);
  } else {
    const double a = P.w, x = P.x, y = P.y, z = P.z;
    const double apx = a * x, apy = a * y, apz = a * z;
    const double ra = near_rcp(a);
    const double dx = quot_rcp(apx, a, ra) - q.x, dy = quot_rcp(apy, a, ra) - q.y, dz = quot_rcp(apz, a, ra) - q.z;
    const double w = f * weight64<KT>(kp, dx * dx + dy * dy + dz * dz);
    acc.w += w * a;
    acc.px += w * apx;
    acc.py += w * apy;
    acc.pz += w * apz;
    acc.nx += w * (a * N.x);
    acc.ny += w * (a * N.y);
    acc.nz += w * (a * N.z);
    acc.pn += w * (a * ((x * N.x + y * N.y) + z * N.z));
    acc.pp += w * (a * ((x * x + y * y) + z * z));
  }
}

// Moments of one node as loaded from HBM (node-centred FP32 for the compensated form,
// global-frame FP32 for the plain form, FP64 for the FP64 form).
template <int FORM> struct NodeMom { float4 m0, m1; };
template <> struct NodeMom<0> { float4 m0, m1; float rA; };  // rA = 1 / A, correctly rounded
template <> struct NodeMom<2> { double4 m0, m1; double A; };

template <int FORM>
__device__ __forceinline__ NodeMom<FORM> load_mom(const TreeView& tv, uint32_t c) {
  NodeMom<FORM> r;
  if constexpr (FORM == 0) {
    r.m0 = tv.recP[4 * (size_t)c + 2], r.m1 = tv.recP[4 * (size_t)c + 3];
    r.rA = tv.recP[4 * (size_t)c + 1].w;
  } else if constexpr (FORM == 1) {
    r.m0 = tv.recC[4 * (size_t)c + 2], r.m1 = tv.recC[4 * (size_t)c + 3];
  } else {
    r.m0 = tv.momD[2 * (size_t)c], r.m1 = tv.momD[2 * (size_t)c + 1];
    r.A = tv.AD[c];
  }
  return r;
}

// Contribution of a node's moments with multiplier f, weight at its mean point.
// n / A from the stored reciprocal of A.  EXACT (trees whose areas may be subnormal, see walk_short): the
// compiler's division.
template <bool EXACT>
__device__ __forceinline__ float quot_area(float n, float A, float rA) {
  return EXACT ? n / A : quot_rcp(n, A, rA);
}

template <int FORM, int KT, bool EXACT = false, class KP>
__device__ __forceinline__ void add_mom(typename FormT<FORM>::Acc& acc, const KP& kp, const NodeMom<FORM>& mm, float Af,
                                        V3<typename FormT<FORM>::T> q, typename FormT<FORM>::T f) {
  if constexpr (FORM == 0) {
    const float4 m0 = mm.m0, m1 = mm.m1;
    const float dx = quot_area<EXACT>(m0.x, Af, mm.rA) - q.x, dy = quot_area<EXACT>(m0.y, Af, mm.rA) - q.y,
                dz = quot_area<EXACT>(m0.z, Af, mm.rA) - q.z;
    const float w = f * weight32<KT>(kp, fmaf(dz, dz, fmaf(dx, dx, __fmul_rn(dy, dy))));
    acc.w = fmaf(w, Af, acc.w);
    acc.px = fmaf(w, m0.x, acc.px);
    acc.py = fmaf(w, m0.y, acc.py);
    acc.pz = fmaf(w, m0.z, acc.pz);
    acc.nx = fmaf(w, m1.x, acc.nx);
    acc.ny = fmaf(w, m1.y, acc.ny);
    acc.nz = fmaf(w, m1.z, acc.nz);
    acc.pn = fmaf(w, m0.w, acc.pn);
    acc.pp = fmaf(w, m1.w, acc.pp);
  } else if constexpr (FORM == 1) {
    const float4 m0 = mm.m0, m1 = mm.m1;
    const float dx = m0.x - q.x, dy = m0.y - q.y, dz = m0.z - q.z;
    const float d2 = fmaf(dz, dz, fmaf(dx, dx, __fmul_rn(dy, dy)));
    const float fw = __fmul_rn(f, weight32<KT>(kp, d2));
    const float fa = __fmul_rn(fw, Af);
    acc.lw = fmaf(fw, Af, acc.lw);
    acc.lpx = fmaf(fa, dx, acc.lpx);
    acc.lpy = fmaf(fa, dy, acc.lpy);
    acc.lpz = fmaf(fa, dz, acc.lpz);
    acc.lnx = fmaf(fw, m1.x, acc.lnx);
    acc.lny = fmaf(fw, m1.y, acc.lny);
    acc.lnz = fmaf(fw, m1.z, acc.lnz);
    acc.lpn = fmaf(fw, __fadd_rn(m0.w, fmaf(dz, m1.z, fmaf(dx, m1.x, __fmul_rn(dy, m1.y)))), acc.lpn);
    acc.lpp = fmaf(fw, fmaf(Af, d2, m1.w), acc.lpp);
  } else {
    const double4 m0 = mm.m0, m1 = mm.m1;
    const double A = mm.A;
    const double rA = near_rcp(A);
    const double dx = quot_rcp(m0.x, A, rA) - q.x, dy = quot_rcp(m0.y, A, rA) - q.y, dz = quot_rcp(m0.z, A, rA) - q.z;
    const double w = f * weight64<KT>(kp, dx * dx + dy * dy + dz * dz);
    acc.w += w * A;
    acc.px += w * m0.x;
    acc.py += w * m0.y;
    acc.pz += w * m0.z;
    acc.nx += w * m1.x;
    acc.ny += w * m1.y;
    acc.nz += w * m1.z;
    acc.pn += w * m0.w;
    acc.pp += w * m1.w;
  }
}

// add_mom as the (factor, value) pairs of its nine fused operations, in the order of the sums
// (FP32 forms; the same roundings).
template <int FORM, int KT, bool EXACT, class KP>
__device__ __forceinline__ void mom_pairs(float2* p, const KP& kp, const NodeMom<FORM>& mm, float Af, V3<float> q, float f) {
  const float4 m0 = mm.m0, m1 = mm.m1;
  if constexpr (FORM == 0) {
    const float dx = quot_area<EXACT>(m0.x, Af, mm.rA) - q.x, dy = quot_area<EXACT>(m0.y, Af, mm.rA) - q.y,
                dz = quot_area<EXACT>(m0.z, Af, mm.rA) - q.z;
    const float w = f * weight32<KT>(kp, fmaf(dz, dz, fmaf(dx, dx, __fmul_rn(dy, dy))));
    p[0] = make_float2(w, Af);
    p[1] = make_float2(w, m0.x), p[2] = make_float2(w, m0.y), p[3] = make_float2(w, m0.z);
    p[4] = make_float2(w, m1.x), p[5] = make_float2(w, m1.y), p[6] = make_float2(w, m1.z);
    p[7] = make_float2(w, m0.w), p[8] = make_float2(w, m1.w);
  } else {
    const float dx = m0.x - q.x, dy = m0.y - q.y, dz = m0.z - q.z;
    const float d2 = fmaf(dz, dz, fmaf(dx, dx, __fmul_rn(dy, dy)));
    const float fw = __fmul_rn(f, weight32<KT>(kp, d2));
    const float fa = __fmul_rn(fw, Af);
    p[0] = make_float2(fw, Af);
    p[1] = make_float2(fa, dx), p[2] = make_float2(fa, dy), p[3] = make_float2(fa, dz);
    p[4] = make_float2(fw, m1.x), p[5] = make_float2(fw, m1.y), p[6] = make_float2(fw, m1.z);
    p[7] = make_float2(fw, __fadd_rn(m0.w, fmaf(dz, m1.z, fmaf(dx, m1.x, __fmul_rn(dy, m1.y)))));
    p[8] = make_float2(fw, fmaf(Af, d2, m1.w));
  }
}

template <int FORM, int KT, bool EXACT = false, class KP>
__device__ __forceinline__ void add_node(typename FormT<FORM>::Acc& acc, const KP& kp, const TreeView& tv, uint32_t c,
                                         float Af, V3<typename FormT<FORM>::T> q, typename FormT<FORM>::T f) {
  add_mom<FORM, KT, EXACT>(acc, kp, load_mom<FORM>(tv, c), Af, q, f);
}

template <int FORM, int SEM, int KT, bool CNT, bool EXACT = false, class KP>
__device__ __forceinline__ void add_leaf(typename FormT<FORM>::Acc& acc, const KP& kp, const TreeView& tv, uint4 h,
                                         V3<typename FormT<FORM>::T> q, typename FormT<FORM>::T f, Counters& ct) {
  const uint32_t first = h.x, cnt = hdr_count(h.y);
  if constexpr (SEM == MLOD_SEM_REF_CPU) {
    // apssStats of a leaf is assigned, not summed, per point: only the last point stays
    // (CPUUtils.cpp:448-457).
    add_point<FORM, KT, EXACT>(acc, kp, tv, first + cnt - 1, q, f);
    if constexpr (CNT) ct.leafPts += 1;
  } else {
    for (uint32_t j = first; j < first + cnt; ++j) add_point<FORM, KT, EXACT>(acc, kp, tv, j, q, f);
    if constexpr (CNT) ct.leafPts += cnt;
  }
}

// Traversal arithmetic per form.  The plain forms keep correctly rounded division and square root
// (the reference's arithmetic); the compensated form, whose error budget is set by its FP64 fit and
// compensated sums, takes the hardware reciprocal and square root (1 ulp).
template <int FORM, bool EXACT = false>
__device__ __forceinline__ typename FormT<FORM>::T tdist(V3<typename FormT<FORM>::T> q, float4 g) {
  if constexpr (FORM != 2) {  // (the fused operations written out: every kernel rounds alike)
    const float dx = q.x - g.x, dy = q.y - g.y, dz = q.z - g.z;
    const float d2 = fmaf(dz, dz, fmaf(dx, dx, __fmul_rn(dy, dy)));
    return FORM == 1 ? __builtin_amdgcn_sqrtf(d2) : EXACT ? fsqrt(d2) : root(d2);
  } else {
    const double dx = q.x - (double)g.x, dy = q.y - (double)g.y, dz = q.z - (double)g.z;
    return root(dx * dx + dy * dy + dz * dz);
  }
}
template <int FORM, bool EXACT = false, class T>
__device__ __forceinline__ T tratio(T a, T b) {  // a / b
  if constexpr (FORM == 1)
    return a * __builtin_amdgcn_rcpf(b);
  else if constexpr (EXACT)
    return a / b;
  else
    return quot(a, b);
}

// A node with near children still to expand, per level and lane: its first child, and those children.
struct WalkStack {
  uint32_t (*first)[PBS];
  uint8_t (*mask)[PBS];
};

// Flattened traversal (the FP64 form's; traverse_staged is the FP32 forms').  The lane's current node
// (expanded: near, or above minDepth) has its children tested one per loop iteration; when they are done
// the node's own (1 - b_c) share is added and the next near node becomes the current one.  Either way an
// iteration handles exactly one node X: it loads X's cell and header and the moments of the node it
// contributes (X itself when testing, the finished node when moving on), computes X's distance, then
// either classifies X as a child (far / leaf / near) or makes it the current node, and ends in one shared
// node contribution.  Lanes of a wavefront therefore advance by one node per iteration whatever their
// position in their own tree walk, instead of waiting for the widest child loop of the wavefront at every
// level.  A near child's blend factor is exactly 1 (its t is dp / (dp + 0)), so the product of the factors
// on the path to any expanded node is 1 and is not kept.
//
// A finished node with near children leaves {first child, near children} in LDS for its depth (5 B per
// level and lane, a per-lane bit set marks the levels in use), and the first waiting child of the deepest
// such node is next.
//
// Bound by FP64 vector instructions (276 an iteration against 370: weights.h has the exponential, quotients and
// roots, blend() the cosine, and no multiplier), with the L1 72 % busy beside them.  1M points, 400k queries,
// two steps, six sigmas: 8.0 -> 4.75 ms; 1k queries 2.1 -> 1.3; a rational kernel, 400k queries, 7.4 -> 3.8.
constexpr double kNoBlend64 = 1e300;  // a distance term that makes every blend factor exactly 1 (above minDepth)
template <int FORM, int SEM, int KT, bool CNT, class KP>
__device__ __forceinline__ void traverse_loads(AccP64& acc, const KP& kp, const TreeView& tv, V3<double> q, double cutoff,
                                               uint32_t minDepth, WalkStack st, int tid, Counters& ct) {
  static_assert(FORM == 2, "the FP32 forms' walk is staged");
  const uint4 h0 = tv.hdr[0];
  if (hdr_leaf(h0.y)) {
    add_leaf<FORM, SEM, KT, CNT>(acc, kp, tv, h0, q, 1.0, ct);
    return;
  }
  const float4 g0 = tv.geo[0];
  double dp = kNoBlend64;  // the current node's distance term
  if (minDepth == 0) {
    const double over = tdist<FORM>(q, g0) - (double)g0.w * cutoff;
    if (over > 0.0) {
      add_node<FORM, KT>(acc, kp, tv, 0, __uint_as_float(h0.z), q, 1.0);
      if constexpr (CNT) ct.far_ += 1;
      return;
    }
    dp = fabs(over);
  }
  const int32_t blendKey = (int32_t)(min(minDepth, 15u) << 27);  // headers of internal nodes at or below minDepth
  // the current node: its children [x, xEnd) still to test, the near ones found
  uint32_t node = 0, first = h0.x, x = first, xEnd = first + hdr_count(h0.y), mask = 0, pend = 0;
  int lvl = 0;
  double A = __uint_as_float(h0.z), shareSum = 0.0;
  double scale = SEM == MLOD_SEM_REF_CPU ? tratio<FORM>(1.0, (double)hdr_count(h0.y)) : near_rcp(A);
  for (bool active = true; active;) {
    if constexpr (CNT) ct.iters += 1;
    const bool testing = x < xEnd;
    const uint32_t tgt = testing ? x : node;
    uint32_t nx = x;
    if (!testing) {
      if (mask) {
        st.first[lvl][tid] = first;
        st.mask[lvl][tid] = (uint8_t)mask;
        pend |= 1u << lvl;
      }
      active = pend != 0u;
      if (active) {
        const uint32_t L = 31u - (uint32_t)__builtin_clz(pend);
        const uint32_t bits = st.mask[L][tid], rest = bits & (bits - 1u);
        nx = st.first[L][tid] + (uint32_t)__builtin_ctz(bits);
        st.mask[L][tid] = (uint8_t)rest;
        if (!rest) pend ^= 1u << L;
        lvl = (int)L + 1;
      } else {
        nx = 0u;
      }
    }
    const float4* rec = tv.recP + 4 * (uint64_t)nx;
    const NodeMom<FORM> mm = load_mom<FORM>(tv, tgt);
    const float4 g = rec[0];
    const uint4 h = reinterpret_cast<const uint4*>(rec)[1];
    const double over = tdist<FORM>(q, g) - (double)g.w * cutoff;
    const double Ax = __uint_as_float(h.z);
    bool contrib;
    double f;
    if (testing) {
      // X's blend factor against its parent (CPUUtils.cpp:489-497); far: beyond its cutoff
      f = blend(tratio<FORM>(dp, dp + fmax(over, 0.0)));
      shareSum += (1.0 - f) * (SEM == MLOD_SEM_REF_CPU ? scale : quot_rcp(Ax, A, scale));
      const bool leaf = (int32_t)h.y < 0, single = h.y >= (kLeafBit | kSingleBit);
      const bool far = (int32_t)h.y >= blendKey && over > 0.0;
      mask |= (leaf || far ? 0u : 1u) << (x - first);
      if (leaf && !single) add_leaf<FORM, SEM, KT, CNT>(acc, kp, tv, h, q, f, ct);  // multi-point leaf
      if constexpr (CNT) {
        ct.tested += 1;
        ct.far_ += far ? 1u : 0u;
        ct.leafPts += single ? 1u : 0u;
      }
      ++x;
      contrib = far || single;
    } else {
      // the finished node's own share; X becomes the current node, its children to test
      f = shareSum;
      contrib = f != 0.0;
      if constexpr (CNT) ct.nearN += contrib ? 1u : 0u;
      node = nx;
      first = x = h.x;
      xEnd = first + (h.y & 15u);  // an internal node has at most 8 children
      mask = 0u;
      dp = (int32_t)h.y >= blendKey ? fabs(over) : kNoBlend64;
      A = Ax;
      scale = SEM == MLOD_SEM_REF_CPU ? tratio<FORM>(1.0, (double)(h.y & 15u)) : near_rcp(A);
      shareSum = 0.0;
    }
    if (contrib) add_mom<FORM, KT>(acc, kp, mm, 0.f, q, f);
  }
}

// ----------------------------------------------------------------------------- staged walk (FP32 forms)
// The same walk, one node per lane and iteration, with the node's 64-byte record (cell, header,
// moments: recP / recC) brought in by the four lanes of a quad together.  A lane that gathers its own
// record takes four 16-byte loads, and each of those costs the L1 cache one access per distinct
// segment of a quad: 41 accesses per load instruction of 64 lanes, 164 an iteration, one access every
// cycle of the launch (8M points and queries, FP32C).  Here load j brings the record of lane j of
// every quad, its four lanes fetching the 16-byte pieces of one segment: 16 accesses, 64 an
// iteration.  The loads go straight to LDS (load j to row j, 64 lanes x 16 B), from where each lane
// reads its own record back; a row is one 16-byte bank group longer than its data, which spreads those
// reads over all banks.  With the L1 out of the way the walk is bound by vector instructions (VALU
// 100 % busy, 131 an iteration against 152 before: no multiplier, reciprocals of A kept in the
// records, one stack access an iteration), and the smaller stacks let five waves run per SIMD against
// four.  8M points, 8M queries, six sigmas, FP32C: 20.6 -> 16.5 ms a step; 1M points and queries,
// rational kernel, plain FP32: 11.7 -> 10.0 (8.1 with the quotients and roots of weights.h).
// (Four waves per SIMD, with the stacks one word a level longer, left the step at 20.6 ms.)
// A launch that fills the chip less is bound by an iteration's round trip.  So a record serves both its
// visits: a node that becomes current comes through the stage like a child, its moments stay in
// registers until its own share is added, and the next record's loads are issued as soon as this one has
// been classified, before its terms are formed.  100k queries x 10 steps on 1M points: 5.5 -> 4.8 ms with
// the stage, 4.2 so (loading the cell of the node that becomes current apart, and the finished node's
// moments again, at the iteration's start); a burst of 20 requests served 29.3 -> 26.0.
constexpr uint32_t kStageRow = 1024 + 16;
constexpr uint32_t kStageBytes = 4 * kStageRow;  // per wavefront

template <int J>
__device__ __forceinline__ uint32_t quad_lane(uint32_t v) {  // lane J of this lane's quad
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, J * 0x55, 0xf, 0xf, true);
}
typedef const __attribute__((address_space(1))) void* GlobalPtr;
typedef __attribute__((address_space(3))) void* LdsPtr;

// WIDE: 2^26 nodes or more, whose byte offsets need more than 32 bits
template <int J, bool WIDE>
__device__ __forceinline__ void stage_row(const char* rec, uint32_t idx, uint32_t lane, unsigned char* stage) {
  const uint32_t piece = (lane & 3u) * 16u;
  const char* src = WIDE ? rec + piece + (uint64_t)quad_lane<J>(idx) * 64u : rec + (quad_lane<J>(idx << 6) + piece);
  __builtin_amdgcn_global_load_lds((GlobalPtr)src, (LdsPtr)(stage + J * kStageRow), 16, 0, 0);
}
// Starts the loads of record `idx` of every lane (all 64 lanes take part).
template <bool WIDE>
__device__ __forceinline__ void stage_issue(const float4* rec, uint32_t idx, uint32_t lane, unsigned char* stage) {
  const char* r = reinterpret_cast<const char*>(rec);
  stage_row<0, WIDE>(r, idx, lane, stage);
  stage_row<1, WIDE>(r, idx, lane, stage);
  stage_row<2, WIDE>(r, idx, lane, stage);
  stage_row<3, WIDE>(r, idx, lane, stage);
}

// Half a distance term that makes every blend factor 1 (a node above minDepth: no blending below it):
// kNoBlend / (2 kNoBlend + anything a cloud spans) is 1/2 to the last bit, and its shares are 0 (areas'
// reciprocals are held finite).  Not so over an infinite distance: walk_short.
constexpr float kNoBlend = 1e30f;

__device__ __forceinline__ void swap_regs(float& a, float& b) { asm("v_swap_b32 %0, %1" : "+v"(a), "+v"(b)); }
__device__ __forceinline__ void swap_regs(float4& a, float4& b) {
  swap_regs(a.x, b.x), swap_regs(a.y, b.y), swap_regs(a.z, b.z), swap_regs(a.w, b.w);
}
__device__ __forceinline__ bool any_lane(bool p) { return __builtin_amdgcn_ballot_w64(p) != 0ull; }

// Whether the areas of all points and nodes are from 2^-126 to 2^126, where they have normal reciprocals: a point's
// is its leaf's squared diagonal, at least 2^-12 of the root's (2 r), over the leaf's points; the points' sum is
// the root's.
__host__ __device__ __forceinline__ bool areas_normal(float radius, uint32_t points) {
  const float r2 = radius * radius, n = (float)points;
  return r2 >= n * 0x1p-104f && r2 * n <= 0x1p124f;
}
// Whether a wavefront's plain walk may take the short quotients and roots and the large distance term (uniform):
// the areas have normal reciprocals, and no query is so far away that its distances overflow and meets nodes
// without blending.  The other walk (EXACT) holds everywhere and gives the same bits.  The compensated form has one
// walk: it takes the hardware's reciprocals, and has no fit for such a query (its sum of squared offsets
// overflows too).
template <int FORM>
__device__ __forceinline__ bool walk_short(const TreeView& tv, V3<float> q, uint32_t minDepth, bool live) {
  if constexpr (FORM == 1) return true;
  bool ok = areas_normal(tv.geo[0].w, tv.n);
  if (minDepth) ok = ok && !any_lane(live && !(fmaxf(fmaxf(fabsf(q.x), fabsf(q.y)), fabsf(q.z)) < 1e18f));
  return ok;
}

// What the walk relies on.  A near child's blend factor is exactly 1 (its distance is within its
// cutoff, so t = dP / (dP + 0), at most one rounding off 1, and the hardware cosine at half a
// revolution, and one float to either side of it, is exactly -1): the product of the factors on
// the path to any expanded node is 1 and is not kept.  Terms are added in the order of the walk (a node's
// children in slot order, then its own (1 - b_c) share, then its first near child), and the
// compensated form's block flushes come every kFlush iterations of the loop, which all lanes start
// together, so a lane's sums depend on its own query only.
template <int FORM, int SEM, int KT, bool CNT, bool WIDE, bool EXACT, class KP>
__device__ __forceinline__ void traverse_staged(typename FormT<FORM>::Acc& acc, const KP& kp, const TreeView& tv,
                                                V3<float> q, float cutoff, uint32_t minDepth, bool live,
                                                WalkStack st, unsigned char* stage, int tid, Counters& ct) {
#pragma clang fp contract(off)  // the fused operations are written out
  const uint32_t lane = __lane_id();
  const float4* __restrict__ rec = FORM == 0 ? tv.recP : tv.recC;
  const uint4 h0 = tv.hdr[0];
  if (hdr_leaf(h0.y)) {  // a one-leaf tree (uniform)
    if (live) add_leaf<FORM, SEM, KT, CNT, EXACT>(acc, kp, tv, h0, q, 1.f, ct);
    if constexpr (FORM == 1) acc.flush();
    return;
  }
  const int32_t blendKey = (int32_t)(min(minDepth, 15u) << 27);  // headers of internal nodes at or below minDepth
  const float4 g0 = tv.geo[0];
  uint32_t active = live ? 1u : 0u;  // (a word: one compare makes the wavefront's mask of it)
  float dh = kNoBlend;  // half the current node's distance term
  if (minDepth == 0) {
    const float d0 = tdist<FORM, EXACT>(q, g0), rc = g0.w * cutoff;
    dh = 0.5f * fabsf(d0 - rc);
    if (d0 > rc) {
      if (live) {
        add_node<FORM, KT, EXACT>(acc, kp, tv, 0, __uint_as_float(h0.z), q, 1.f);
        if constexpr (CNT) ct.far_ += 1;
      }
      active = 0u;
    }
  }
  // the current node: its children [first, xEnd), the next one to test, the near ones found; its area and moments
  uint32_t first = h0.x, x = first, xEnd = active ? first + hdr_count(h0.y) : first, mask = 0, pend = 0;
  int lvl = 0;
  float Ai = __uint_as_float(h0.z), shareSum = 0.f;
  float scale = SEM == MLOD_SEM_REF_CPU ? tratio<FORM, EXACT>(1.f, (float)hdr_count(h0.y)) : rec[1].w;
  NodeMom<FORM> own = load_mom<FORM>(tv, 0);
  const unsigned char* mine = stage + (lane & 3u) * kStageRow + (lane >> 2) * 64u;
  stage_issue<WIDE>(rec, x, lane, stage);
  while (any_lane(active != 0u)) {
#pragma unroll 1
    for (uint32_t b = 0; b < kFlush && any_lane(active != 0u); ++b) {
      if constexpr (CNT) ct.iters += active ? 1u : 0u;
      // the record: a child of the current node, or the node that follows it
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const float4 g = *reinterpret_cast<const float4*>(mine);
      const uint4 h = *reinterpret_cast<const uint4*>(mine + 16);
      NodeMom<FORM> mm;
      mm.m0 = *reinterpret_cast<const float4*>(mine + 32);
      mm.m1 = *reinterpret_cast<const float4*>(mine + 48);
      if constexpr (FORM == 0) mm.rA = __uint_as_float(h.w);
      float At = __uint_as_float(h.z);
      const float over = tdist<FORM, EXACT>(q, g) - g.w * cutoff;
      bool contrib = false, multi = false;
      float f = 0.f;
      if (x < xEnd) {
        // X's blend factor against its parent (CPUUtils.cpp:489-497); far: beyond its cutoff
        const float dc = fmaxf(over, 0.f);
        f = fmaf(__builtin_amdgcn_cosf(tratio<FORM, EXACT>(dh, fmaf(2.f, dh, dc))), -0.5f, 0.5f);
        if constexpr (EXACT) f = dh == kNoBlend ? 1.f : f;
        const float share = SEM == MLOD_SEM_REF_CPU ? scale : (FORM == 1 ? At * scale : quot_area<EXACT>(At, Ai, scale));
        shareSum = fmaf(share, 1.f - f, shareSum);
        const bool leaf = (int32_t)h.y < 0;
        const bool single = h.y >= (kLeafBit | kSingleBit);
        const bool far = (int32_t)h.y >= blendKey && over > 0.f;
        mask |= (leaf || far ? 0u : 1u) << (x - first);
        multi = leaf && !single;
        if constexpr (CNT) {
          ct.tested += 1;
          ct.far_ += far ? 1u : 0u;
          ct.leafPts += single ? 1u : 0u;
        }
        ++x;
        contrib = far || single;
      } else if (active) {
        // the current node is finished: its own share is added, and X becomes current
        f = shareSum;
        contrib = f != 0.f;
        if constexpr (CNT) ct.nearN += contrib ? 1u : 0u;
        swap_regs(mm.m0, own.m0);
        swap_regs(mm.m1, own.m1);
        if constexpr (FORM == 0) swap_regs(mm.rA, own.rA);
        swap_regs(At, Ai);
        shareSum = 0.f;
        active = lvl >= 0 ? 1u : 0u;  // (none follows the last node)
        first = x = h.x;
        xEnd = active ? first + (h.y & 15u) : first;  // an internal node has at most 8 children
        dh = 0.5f * fabsf(over);
        if (blendKey) {
          asm volatile("");  // (a uniform branch, not a select)
          dh = (int32_t)h.y >= blendKey ? dh : kNoBlend;
        }
        scale = SEM == MLOD_SEM_REF_CPU ? tratio<FORM, EXACT>(1.f, (float)(h.y & 15u)) : __uint_as_float(h.w);
      }
      uint32_t idx = x;
      if (active && x == xEnd) {
        // the children are done: the first waiting child of the deepest node that has some follows
        if (mask) {
          st.first[lvl][tid] = first;
          st.mask[lvl][tid] = (uint8_t)mask;
          pend |= 1u << lvl;
          mask = 0u;
        }
        lvl = -1;
        idx = 0u;
        if (pend) {
          const uint32_t L = 31u - (uint32_t)__builtin_clz(pend);
          const uint32_t bits = st.mask[L][tid], from = st.first[L][tid];
          const uint32_t rest = bits & (bits - 1u);
          st.mask[L][tid] = (uint8_t)rest;
          if (!rest) pend ^= 1u << L;
          lvl = (int)L + 1;
          idx = from + (uint32_t)__builtin_ctz(bits);
        }
      }
      // the next record's loads go out before this one's terms are formed (it has been read by now)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      stage_issue<WIDE>(rec, idx, lane, stage);
      if (contrib) add_mom<FORM, KT, EXACT>(acc, kp, mm, At, q, f);
      if (any_lane(multi)) {  // a leaf of several points (at the last level, or by the build's option)
        if (multi) add_leaf<FORM, SEM, KT, CNT, EXACT>(acc, kp, tv, h, q, f, ct);
      }
    }
    if constexpr (FORM == 1) acc.flush();
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the stage may be used again)
  if constexpr (FORM == 1) acc.flush();
}

// ----------------------------------------------------------------------------- grouped walk (FP32 forms)
// The same walk with eight lanes a query, for batches too small to fill the chip with a lane each.
// There a step lasts as long as its longest walk: some 600 iterations of one dependent load each.
// Here the children of a node are tested by the group's lanes at once, so a node costs one round
// trip; what a near child needs to become the current node (its header and distance term) goes to the
// group's LDS stack when it is found near; and the next node's loads are issued before the sums of the
// last one are added.  The sums are the lane walk's to the bit: the children's terms go through LDS as
// (factor, value) pairs and are added in slot order by one fused operation each, lane a of the group
// adding sum a (and the even lanes the ninth), with the compensated form's block flushes after the same
// terms.
struct GroupNode {
  uint32_t fn;    // first child, #children << 27
  float dh, A;    // half its distance term; its area
  uint32_t node;
};
constexpr uint32_t kGroup = 8;                 // lanes a query
constexpr uint32_t kGroups = 64 / kGroup;      // queries a wavefront
struct GroupLds {  // one wavefront
  GroupNode wait[kLevels][64];                 // near children, per level: lane's slot
  float2 pair[64][10];                         // a child's terms: nine sums, then (share, 1 - blend)
  double sum[kGroups][9];
  uint8_t mask[kLevels][kGroups];              // the level's children still to expand
};

// The sums of one lane of a group: partial sum and Kahan pair of sum `lane % 8` and, in the even
// lanes, of the ninth.
struct GroupSums {
  float l0, l8;
  KSum k0, k8;
  uint32_t cnt;  // the walk's iterations since the last flush (compensated form)
  __device__ __forceinline__ void init() { l0 = l8 = 0.f, k0.init(), k8.init(), cnt = 0; }
  template <int FORM>
  __device__ __forceinline__ void flush() {
    if constexpr (FORM == 1) {
      k0.add(l0), k8.add(l8);
      l0 = l8 = 0.f;
      cnt = 0;
    }
  }
};

// The partial sums as an accumulator whose nine sums all hold l, and back: a term added to it by
// add_mom / add_point adds to every sum, of which the lane keeps its own.
template <int FORM>
__device__ __forceinline__ typename FormT<FORM>::Acc spread_sum(float l0, float l8) {
  typename FormT<FORM>::Acc a;
  if constexpr (FORM == 0) {
    a.w = a.px = a.py = a.pz = a.nx = a.ny = a.nz = a.pn = l0, a.pp = l8;
  } else {
    a.lw = a.lpx = a.lpy = a.lpz = a.lnx = a.lny = a.lnz = a.lpn = l0, a.lpp = l8;
  }
  return a;
}
template <int FORM>
__device__ __forceinline__ void pick_sum(const typename FormT<FORM>::Acc& a, uint32_t c, float& l0, float& l8) {
  float v[9];
  if constexpr (FORM == 0) {
    v[0] = a.w, v[1] = a.px, v[2] = a.py, v[3] = a.pz, v[4] = a.nx, v[5] = a.ny, v[6] = a.nz, v[7] = a.pn, v[8] = a.pp;
  } else {
    v[0] = a.lw, v[1] = a.lpx, v[2] = a.lpy, v[3] = a.lpz, v[4] = a.lnx, v[5] = a.lny, v[6] = a.lnz, v[7] = a.lpn,
    v[8] = a.lpp;
  }
  const float x = c & 1u ? v[1] : v[0], y = c & 1u ? v[3] : v[2], z = c & 1u ? v[5] : v[4], t = c & 1u ? v[7] : v[6];
  const float u = c & 2u ? y : x, r = c & 2u ? t : z;
  l0 = c & 4u ? r : u;
  l8 = v[8];
}

struct Record {
  float4 g;
  uint4 h;
  float4 m0, m1;
};
template <bool WIDE>
__device__ __forceinline__ Record load_record(const float4* rec, uint32_t idx) {
  const char* r = reinterpret_cast<const char*>(rec);
  const char* src = WIDE ? r + (uint64_t)idx * 64u : r + (idx << 6);
  return Record{reinterpret_cast<const float4*>(src)[0], reinterpret_cast<const uint4*>(src)[1],
                reinterpret_cast<const float4*>(src)[2], reinterpret_cast<const float4*>(src)[3]};
}

template <int FORM, int SEM, int KT, bool WIDE, bool EXACT, class KP>
__device__ __forceinline__ void traverse_group(GroupSums& gs, const KP& kp, const TreeView& tv, V3<float> q, float cutoff,
                                               uint32_t minDepth, bool live, GroupLds& lds) {
#pragma clang fp contract(off)  // the fused operations are written out
  const uint32_t lane = __lane_id(), c = lane & (kGroup - 1u), grp = lane / kGroup, base = lane & ~(kGroup - 1u);
  const float4* __restrict__ rec = FORM == 0 ? tv.recP : tv.recC;
  Counters ct{0, 0, 0, 0, 0};
  const uint4 h0 = tv.hdr[0];
  const float4 g0 = tv.geo[0];
  const float A0 = __uint_as_float(h0.z);
  const auto single_term = [&](auto&& add) {  // a term added outside the group's exchange
    auto a = spread_sum<FORM>(gs.l0, gs.l8);
    add(a);
    pick_sum<FORM>(a, c, gs.l0, gs.l8);
  };
  if (hdr_leaf(h0.y)) {  // a one-leaf tree (uniform)
    if (live) single_term([&](auto& a) { add_leaf<FORM, SEM, KT, false, EXACT>(a, kp, tv, h0, q, 1.f, ct); });
    gs.template flush<FORM>();
    return;
  }
  const int32_t blendKey = (int32_t)(min(minDepth, 15u) << 27);
  uint32_t active = live ? 1u : 0u;
  float dh = kNoBlend;
  if (minDepth == 0) {
    const float d0 = tdist<FORM, EXACT>(q, g0), rc = g0.w * cutoff;
    dh = 0.5f * fabsf(d0 - rc);
    if (d0 > rc) {
      if (live) single_term([&](auto& a) { add_node<FORM, KT, EXACT>(a, kp, tv, 0, A0, q, 1.f); });
      active = 0u;
    }
  }
  // the current node of the group
  uint32_t node = 0, first = h0.x, nc = active ? hdr_count(h0.y) : 0u, pend = 0, lvl = 0;
  float Ai = A0;
  Record next = load_record<WIDE>(rec, first + (c < nc ? c : 0u));  // the lane's child
  NodeMom<FORM> own = load_mom<FORM>(tv, node);
  float rA = rec[4 * (size_t)node + 1].w;  // the reciprocal of its area
  while (any_lane(active != 0u)) {
    const float4 g = next.g;
    const uint4 h = next.h;
    NodeMom<FORM> mm;
    mm.m0 = next.m0;
    mm.m1 = next.m1;
    if constexpr (FORM == 0) mm.rA = __uint_as_float(h.w);
    // the node that is summed below
    const uint32_t ncP = nc;
    const float AiP = Ai, dhP = dh, rAP = rA;
    const NodeMom<FORM> ownP = own;
    const bool mineP = c < ncP, activeP = active != 0u;
    // --- near children, and the next node
    const float over = tdist<FORM, EXACT>(q, g) - g.w * cutoff;
    const bool leaf = (int32_t)h.y < 0, single = h.y >= (kLeafBit | kSingleBit);
    const bool far = (int32_t)h.y >= blendKey && over > 0.f;
    const bool near = mineP && !leaf && !far;
    const float At = __uint_as_float(h.z);
    uint32_t bits = (uint32_t)(__builtin_amdgcn_ballot_w64(near) >> base) & 0xffu, L = lvl;
    if (near)
      lds.wait[lvl][lane] = GroupNode{h.x | (h.y & 15u) << 27, (int32_t)h.y >= blendKey ? 0.5f * fabsf(over) : kNoBlend, At,
                                      first + c};
    if (activeP) {
      if (bits) {
        if (bits & (bits - 1u)) pend |= 1u << lvl;
      } else if (pend) {
        L = 31u - (uint32_t)__builtin_clz(pend);
        bits = lds.mask[L][grp];
      } else {
        active = 0u;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // records read, near children written
    nc = 0u;
    if (active) {
      const uint32_t k = (uint32_t)__builtin_ctz(bits), rest = bits & (bits - 1u);
      const GroupNode e = lds.wait[L][base + k];
      lds.mask[L][grp] = (uint8_t)rest;
      if (!rest) pend &= ~(1u << L);
      node = e.node;
      first = e.fn & kCountMask;
      nc = e.fn >> 27;
      dh = e.dh;
      Ai = e.A;
      lvl = L + 1u;
    }
    next = load_record<WIDE>(rec, first + (c < nc ? c : 0u));
    own = load_mom<FORM>(tv, node);
    rA = rec[4 * (size_t)node + 1].w;
    // --- the sums of the node that was tested
    float f = fmaf(__builtin_amdgcn_cosf(tratio<FORM, EXACT>(dhP, fmaf(2.f, dhP, fmaxf(over, 0.f)))), -0.5f, 0.5f);
    if constexpr (EXACT) f = dhP == kNoBlend ? 1.f : f;
    float share;
    if constexpr (SEM == MLOD_SEM_REF_CPU)
      share = tratio<FORM, EXACT>(1.f, (float)ncP);
    else if constexpr (FORM == 1)
      share = At * rAP;
    else
      share = quot_area<EXACT>(At, AiP, rAP);
    const bool contrib = mineP && (far || single), multi = mineP && leaf && !single;
    {
      float2 p[10];
#pragma unroll
      for (int t = 0; t < 10; ++t) p[t] = make_float2(0.f, 0.f);
      if (contrib) mom_pairs<FORM, KT, EXACT>(p, kp, mm, At, q, f);
      if (mineP) p[9] = make_float2(share, 1.f - f);
      float4* out = reinterpret_cast<float4*>(lds.pair[lane]);
#pragma unroll
      for (int t = 0; t < 5; ++t) out[t] = make_float4(p[2 * t].x, p[2 * t].y, p[2 * t + 1].x, p[2 * t + 1].y);
    }
    float shareSum = 0.f;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    // the compensated form's flush falls before child `due` (after the last one when that is their number)
    const uint32_t terms = gs.cnt + ncP, due = terms >= kFlush ? kFlush - gs.cnt : ~0u;
    static_assert(kFlush == kGroup, "at most one flush among a node's children");
    if (!any_lane(multi)) {  // uniform
      // lane c's second chain is the ninth sum in even lanes, the share sum in odd ones
      const bool odd = c & 1u;
      float2 x[kGroup], y[kGroup];
#pragma unroll
      for (uint32_t j = 0; j < kGroup; ++j) {  // (children past the last hold zeros)
        x[j] = lds.pair[base + j][c];
        y[j] = lds.pair[base + j][8u + (c & 1u)];
      }
      float l0 = gs.l0, l1 = odd ? 0.f : gs.l8, b0 = 0.f, b1 = 0.f;  // b: the block that is complete, if one is
#pragma unroll
      for (uint32_t j = 0; j <= kGroup; ++j) {
        if constexpr (FORM == 1) {
          if (j > 0) {
            const bool full = j == due;
            b0 = full ? l0 : b0;
            l0 = full ? 0.f : l0;
            b1 = full ? l1 : b1;
            l1 = full && !odd ? 0.f : l1;
          }
        }
        if (j < kGroup) {
          l0 = fmaf(x[j].x, x[j].y, l0);
          l1 = fmaf(y[j].x, y[j].y, l1);
        }
      }
      shareSum = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(l1), 0xf5, 0xf, 0xf, true));  // lane | 1 of the quad
      gs.l0 = l0;
      gs.l8 = odd ? gs.l8 : l1;
      if constexpr (FORM == 1) {
        if (due != ~0u) gs.k0.add(b0), gs.k8.add(b1);
      }
    } else {  // a leaf of several points among the children (at the last level, or by the build's option)
#pragma unroll 1
      for (uint32_t j = 0; j < kGroup; ++j) {
        if constexpr (FORM == 1) {
          if (j > 0 && j == due) gs.template flush<FORM>();
        }
        const float2 x = lds.pair[base + j][c];
        const float4 y = *reinterpret_cast<const float4*>(lds.pair[base + j] + 8);
        gs.l0 = fmaf(x.x, x.y, gs.l0);
        gs.l8 = fmaf(y.x, y.y, gs.l8);
        shareSum = fmaf(y.z, y.w, shareSum);
        const uint4 hj = make_uint4((uint32_t)__shfl((int)h.x, (int)(base + j), 64), (uint32_t)__shfl((int)h.y, (int)(base + j), 64), 0u, 0u);
        const float fj = __shfl(f, (int)(base + j), 64);
        const bool mj = __shfl((int)multi, (int)(base + j), 64) != 0;
        if (mj) single_term([&](auto& t) { add_leaf<FORM, SEM, KT, false, EXACT>(t, kp, tv, hj, q, fj, ct); });
      }
      if constexpr (FORM == 1) {
        if (due == kGroup) gs.template flush<FORM>();
      }
    }
    if constexpr (FORM == 1) gs.cnt = terms >= kFlush ? terms - kFlush : terms;
    if (activeP) {
      if (shareSum != 0.f) single_term([&](auto& x) { add_mom<FORM, KT, EXACT>(x, kp, ownP, AiP, q, shareSum); });
      if constexpr (FORM == 1) {
        if (++gs.cnt == kFlush) gs.template flush<FORM>();
      }
    }
  }
  gs.template flush<FORM>();
}

// The LDS of one workgroup's walks: the stacks of waiting nodes (5 B a level and lane in the FP32
// forms) and the wavefronts' staging rows (15.4 KB: ten workgroups a CU, five waves per SIMD), or the
// FP64 form's stacks.
template <int FORM>
struct WalkLds {
  uint32_t first[kLevels][PBS];
  uint8_t mask[kLevels][PBS];
  alignas(16) unsigned char stage[PBS / 64][kStageBytes];
};
template <>
struct WalkLds<2> {
  uint32_t first[kLevels][PBS];
  uint8_t mask[kLevels][PBS];
};

// One walk of each live lane of the wavefront (every lane calls it).
template <int FORM, int SEM, int KT, bool CNT, class KP>
__device__ __forceinline__ void traverse(typename FormT<FORM>::Acc& acc, const KP& kp, const TreeView& tv,
                                         V3<typename FormT<FORM>::T> q, typename FormT<FORM>::T cutoff,
                                         uint32_t minDepth, bool live, WalkLds<FORM>& lds, int tid, Counters& ct) {
  if constexpr (FORM == 2) {
    if (live) traverse_loads<FORM, SEM, KT, CNT>(acc, kp, tv, q, cutoff, minDepth, WalkStack{lds.first, lds.mask}, tid, ct);
  } else {
    const WalkStack st{lds.first, lds.mask};
    unsigned char* stage = lds.stage[__builtin_amdgcn_readfirstlane(tid >> 6)];
    if (!walk_short<FORM>(tv, q, minDepth, live))
      traverse_staged<FORM, SEM, KT, CNT, true, FORM == 0>(acc, kp, tv, q, cutoff, minDepth, live, st, stage, tid, ct);
    else if (tv.nn < (1u << 26))
      traverse_staged<FORM, SEM, KT, CNT, false, false>(acc, kp, tv, q, cutoff, minDepth, live, st, stage, tid, ct);
    else
      traverse_staged<FORM, SEM, KT, CNT, true, false>(acc, kp, tv, q, cutoff, minDepth, live, st, stage, tid, ct);
  }
}

// ----------------------------------------------------------------------------- wave-shared walk
// The same MLoD sum, walked once per wavefront over the union of its lanes' walks.  The node
// being handled is wave-uniform, so its records come through scalar loads; each lane keeps
// its own multiplier, distance term, share sum and near-child bits and takes part only in the
// nodes its own walk visits (a lane is active at a child when it was active at the parent and
// found the child near).  The union walk is a depth-first walk in child order, like each lane's
// own walk, so every lane adds the same terms in the same order as walking alone, and it counts
// its own iterations (one per tested child and one per finished node), so the compensated
// form's block flushes fall where they fall in a lane's own walk.
struct WaveLevel {
  uint32_t first;  // the waiting node's first child
  uint32_t rest;   // its children still to expand (near for at least one lane)
  uint64_t act;    // the lanes active at the waiting node
};

template <class T>
struct WaveStack {
  WaveLevel (*lv)[PBS / 64];  // per level and wavefront
  T (*mul)[PBS];              // per level and lane: the waiting node's multiplier
  T (*dist)[PBS];             // its distance term (negative: no blending below it)
  uint8_t (*near)[PBS];       // its near children for this lane
};

// A wave-uniform record through the constant address space: the tree is not written while a
// projection runs, so the load is a scalar load into SGPRs (one per wavefront, through the
// scalar cache) instead of a vector load per lane.
template <class T>
__device__ __forceinline__ T ld_uni(const T* base, uint32_t idx) {
  static_assert(sizeof(T) % 4 == 0, "records are whole dwords");
  typedef uint32_t W __attribute__((ext_vector_type(sizeof(T) / 4)));
  const W w = *(const __attribute__((address_space(4))) W*)((const __attribute__((address_space(4))) char*)base +
                                                            (uint64_t)idx * sizeof(T));
  T r;
  __builtin_memcpy(&r, &w, sizeof(T));
  return r;
}

template <int FORM>
__device__ __forceinline__ NodeMom<FORM> load_mom_uni(const TreeView& tv, uint32_t c) {
  NodeMom<FORM> r;
  if constexpr (FORM == 0) {
    r.m0 = ld_uni(tv.recP, 4 * c + 2), r.m1 = ld_uni(tv.recP, 4 * c + 3);
    r.rA = ld_uni(tv.recP, 4 * c + 1).w;
  } else if constexpr (FORM == 1) {
    r.m0 = ld_uni(tv.recC, 4 * c + 2), r.m1 = ld_uni(tv.recC, 4 * c + 3);
  } else {
    r.m0 = ld_uni(tv.momD, 2 * c), r.m1 = ld_uni(tv.momD, 2 * c + 1);
    r.A = ld_uni(tv.AD, c);
  }
  return r;
}

template <int FORM, int SEM, int KT, bool CNT, bool EXACT>
__device__ __forceinline__ void traverse_wave(typename FormT<FORM>::Acc& acc, const KParams& kp, const TreeView& tv,
                                              V3<typename FormT<FORM>::T> q, typename FormT<FORM>::T cutoff,
                                              uint32_t minDepth, bool live, WaveStack<typename FormT<FORM>::T> st,
                                              int tid, int wv, Counters& ct, uint32_t& waveIters) {
  using T = typename FormT<FORM>::T;
  const uint32_t lane = __lane_id();
  uint32_t itc = 0;  // the lane's own iterations since the last block flush (compensated form)
  const uint4 h0 = ld_uni(tv.hdr, 0u);
  if (hdr_leaf(h0.y)) {
    if (live) add_leaf<FORM, SEM, KT, CNT, EXACT>(acc, kp, tv, h0, q, T(1), ct);
    return;
  }
  const float4 g0 = ld_uni(tv.geo, 0u);
  bool blendNode = minDepth == 0;
  bool act = live;
  T m = T(1), distP = T(-1), shareSum = T(0);
  uint32_t nearb = 0;
  if (act) {
    const T d0 = tdist<FORM, EXACT>(q, g0);
    if (minDepth == 0 && d0 > (T)g0.w * cutoff) {
      add_mom<FORM, KT, EXACT>(acc, kp, load_mom_uni<FORM>(tv, 0u), __uint_as_float(h0.z), q, T(1));
      if constexpr (CNT) ct.far_ += 1;
      act = false;
    } else {
      distP = blendNode ? fabs(d0 - (T)g0.w * cutoff) : T(-1);
    }
  }
  uint64_t actMask = __ballot(act);
  if (!actMask) return;
  // the current node X (wave-uniform)
  uint32_t first = h0.x, nc = hdr_count(h0.y), k = 0, un = 0, pend = 0;
  int lvl = 0;
  float Ai = __uint_as_float(h0.z);
  T shareScale = SEM == MLOD_SEM_REF_CPU ? tratio<FORM, EXACT>(T(1), (T)nc) : tratio<FORM, EXACT>(T(1), (T)Ai);
  NodeMom<FORM> momX = load_mom_uni<FORM>(tv, 0);
  while (true) {
    if constexpr (CNT) ++waveIters;
    // one iteration: test child k of X, or finish X (its own (1 - b_c) share); either way at
    // most one node term per lane, added at the one call site below
    const bool testing = k < nc;
    NodeMom<FORM> mm = momX;
    float At = Ai;
    T f = m * shareSum;
    bool contrib = false;
    if (testing) {
      const uint32_t x = __builtin_amdgcn_readfirstlane(first + k);
      const float4 gx = ld_uni(tv.geo, x);
      const uint4 hx = ld_uni(tv.hdr, x);
      mm = load_mom_uni<FORM>(tv, x);
      const float Ax = __uint_as_float(hx.z);
      const bool leaf = hdr_leaf(hx.y);
      const bool single = leaf && hdr_count(hx.y) == 1u;
      const bool deep = hdr_depth(hx.y) >= minDepth;
      bool nearc = false;
      if (act) {
        if constexpr (CNT) ct.iters += 1, ct.tested += 1;
        const T dxq = tdist<FORM, EXACT>(q, gx);
        const T rc = (T)gx.w * cutoff;
        const T dp = blendNode ? distP : T(-1);
        T beta = T(1);
        if (dp >= T(0)) {
          const T dc = fmax(dxq - rc, T(0));
          beta = blend(tratio<FORM, EXACT>(dp, dp + dc));
        }
        const T mx = m * beta;
        if (blendNode) {
          const T share = SEM == MLOD_SEM_REF_CPU ? shareScale : (FORM == 1 ? (T)Ax * shareScale : (T)Ax / (T)Ai);
          shareSum += (T(1) - beta) * share;
        }
        const bool far = !leaf && deep && dxq > rc;
        if (leaf && !single) add_leaf<FORM, SEM, KT, CNT, EXACT>(acc, kp, tv, hx, q, mx, ct);
        nearc = !leaf && !far;
        if (nearc) nearb |= 1u << k;
        if constexpr (CNT) {
          ct.far_ += far ? 1u : 0u;
          ct.leafPts += single ? 1u : 0u;
        }
        contrib = far || single;
        f = mx;
      }
      At = Ax;
      if (__ballot(nearc)) un |= 1u << k;
      ++k;
    } else if (act) {
      if constexpr (CNT) {
        ct.iters += 1;
        ct.nearN += (blendNode && shareSum != T(0)) ? 1u : 0u;
      }
      contrib = blendNode && shareSum != T(0);
    }
    if (contrib) add_mom<FORM, KT, EXACT>(acc, kp, mm, At, q, f);
    if constexpr (FORM == 1) {
      if (act && ++itc == kFlush) {
        acc.flush();
        itc = 0;
      }
    }
    if (testing) continue;
    // X is finished: the next node to expand
    uint32_t firstP, c, nbits;
    uint64_t actP;
    T mp, dp;
    if (un) {
      // X's first near child is next; the rest wait at this level
      c = __builtin_ctz(un);
      const uint32_t rest = un & (un - 1u);
      mp = m;
      dp = blendNode ? distP : T(-1);
      nbits = nearb;
      actP = actMask;
      firstP = first;
      if (rest) {
        if (lane == 0) st.lv[lvl][wv] = WaveLevel{first, rest, actMask};
        st.mul[lvl][tid] = mp;
        st.dist[lvl][tid] = dp;
        st.near[lvl][tid] = (uint8_t)nearb;
        pend |= 1u << lvl;
      }
      lvl = lvl + 1;
    } else if (pend) {
      // the deepest waiting node's next near child
      const int L = 31 - __builtin_clz(pend);
      const WaveLevel e = st.lv[L][wv];
      firstP = __builtin_amdgcn_readfirstlane(e.first);
      const uint32_t wm = __builtin_amdgcn_readfirstlane(e.rest);
      actP = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(e.act >> 32)) << 32) |
             (uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)e.act);
      c = __builtin_ctz(wm);
      const uint32_t rest = wm & (wm - 1u);
      if (rest) {
        if (lane == 0) st.lv[L][wv].rest = rest;
      } else {
        pend &= ~(1u << L);
      }
      mp = st.mul[L][tid];
      dp = st.dist[L][tid];
      nbits = st.near[L][tid];
      lvl = L + 1;
    } else {
      break;
    }
    // descend: the child becomes X for the lanes that found it near
    act = ((actP >> lane) & 1u) && ((nbits >> c) & 1u);
    actMask = __ballot(act);
    const uint32_t xn = __builtin_amdgcn_readfirstlane(firstP + c);
    const float4 gx = ld_uni(tv.geo, xn);
    const uint4 hx = ld_uni(tv.hdr, xn);
    momX = load_mom_uni<FORM>(tv, xn);
    if (act) {
      const T dxq = tdist<FORM, EXACT>(q, gx);
      const T rc = (T)gx.w * cutoff;
      T beta = T(1);
      if (dp >= T(0)) {
        const T dc = fmax(dxq - rc, T(0));
        beta = blend(tratio<FORM, EXACT>(dp, dp + dc));
      }
      m = mp * beta;
      distP = fabs(dxq - rc);
    }
    first = hx.x;
    nc = hdr_count(hx.y);
    k = 0;
    un = 0;
    nearb = 0;
    shareSum = T(0);
    blendNode = hdr_depth(hx.y) >= minDepth;
    Ai = __uint_as_float(hx.z);
    shareScale = SEM == MLOD_SEM_REF_CPU ? tratio<FORM, EXACT>(T(1), (T)nc) : tratio<FORM, EXACT>(T(1), (T)Ai);
  }
}

// ----------------------------------------------------------------------------- sphere fit
// Algebraic sphere fit and projection, Fastapss.cu:354-395 (REF_GPU: plane below |u4| 1e-6,
// normalize(0) = 0) and CPUUtils.cpp:739-782 (REF_CPU: plane below 1e-12, normalize(0) = NaN).
template <class T, int SEM>
__device__ __forceinline__ V3<T> nrmz(V3<T> v) {
  const T l2 = v.x * v.x + v.y * v.y + v.z * v.z;
  if (SEM == MLOD_SEM_REF_GPU && l2 == T(0)) return V3<T>{0, 0, 0};
  const T inv = T(1) / fsqrt(l2);
  return V3<T>{v.x * inv, v.y * inv, v.z * inv};
}

template <class T>
__device__ __forceinline__ T dot3(V3<T> a, V3<T> b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

// Sums in frame `o` (origin of the accumulated positions): q is the query in that frame.
// Returns the projection in that frame (NaN guard and step clamp applied).
// STABLE (query frame only, q = 0): the sphere point c + r (q - c)/|q - c| is computed as
// tau * u/|u| with tau = -2 u0 / (|u| + sqrt(|u|^2 - 4 u4 u0)), the small root of
// u0 + tau |u| + u4 tau^2 = 0 along the line through q and the centre.  It is the same point
// (|c| - r = 2 u0 / (|u| + sqrt(|u|^2 - 4 u4 u0)) up to sign) without the cancellation of c and
// r near planar fits (|u4| -> 0, |c| ~ 1/|u4|), and tends to the plane projection as u4 -> 0.
// kind: 0 sphere, 1 plane (|u4| below the threshold), 2 invalid (NaN: the query is kept)
template <class T, class TF, int SEM, bool STABLE = false>
__device__ __forceinline__ void fit(T sw, V3<T> sp, V3<T> sn, T spn, T spp, V3<T> q, T stepMax, V3<T>& outP, V3<T>& outN,
                                    float& kind) {
  const T A = spn - dot3(sp, V3<T>{sn.x / sw, sn.y / sw, sn.z / sw});
  const T B = spp - dot3(sp, V3<T>{sp.x / sw, sp.y / sw, sp.z / sw});
  const T u4 = (T)((0.5 * (double)A) / (double)B);
  const T two_u4 = T(2) * u4;
  const V3<T> u{(sn.x - two_u4 * sp.x) / sw, (sn.y - two_u4 * sp.y) / sw, (sn.z - two_u4 * sp.z) / sw};
  const T u0 = -(dot3(sp, u) + u4 * spp) / sw;
  V3<T> p = q, nr;
  const double tau = SEM == MLOD_SEM_REF_GPU ? 0.000001 : 0.000000000001;
  kind = fabs((double)u4) < tau ? 1.f : 0.f;
  if (fabs((double)u4) < tau) {
    const V3<T> nn{-u.x, -u.y, -u.z};
    const T lambda = (u0 - dot3(p, nn)) / dot3(nn, nn);
    p = V3<T>{p.x + lambda * nn.x, p.y + lambda * nn.y, p.z + lambda * nn.z};
    nr = nrmz<T, SEM>(sn);
  } else if constexpr (STABLE) {
    const T un2 = dot3(u, u);
    const T un = fsqrt(un2);
    const T disc = un2 - T(4) * u4 * u0;
    if (disc < T(0)) {  // r^2 < 0: the reference clamps r to 0, i.e. the centre
      const T m2 = T(-2) * u4;
      p = V3<T>{u.x / m2, u.y / m2, u.z / m2};
    } else {
      const T s = (T(-2) * u0 / (un + fsqrt(disc))) / un;
      p = V3<T>{s * u.x, s * u.y, s * u.z};
    }
    nr = nrmz<T, SEM>(V3<T>{u.x + two_u4 * p.x, u.y + two_u4 * p.y, u.z + two_u4 * p.z});
  } else {
    const T m2 = T(-2) * u4;
    const V3<T> c{u.x / m2, u.y / m2, u.z / m2};
    const T v = dot3(c, c) - u0 / u4;
    const T r = fsqrt(v > T(0) ? v : T(0));
    const V3<T> pc = nrmz<T, SEM>(V3<T>{p.x - c.x, p.y - c.y, p.z - c.z});
    p = V3<T>{c.x + r * pc.x, c.y + r * pc.y, c.z + r * pc.z};
    nr = nrmz<T, SEM>(V3<T>{u.x + two_u4 * p.x, u.y + two_u4 * p.y, u.z + two_u4 * p.z});
  }
  if (isnan(p.x) || isnan(p.y) || isnan(p.z)) {
    outP = q;
    outN = V3<T>{0, 0, 0};
    kind = 2.f;
    return;
  }
  const V3<T> dlt{p.x - q.x, p.y - q.y, p.z - q.z};
  const T step = fsqrt(dot3(dlt, dlt));
  if (step > stepMax) {
    const T s = stepMax / step;
    p = V3<T>{q.x + s * dlt.x, q.y + s * dlt.y, q.z + s * dlt.z};
  }
  outP = p;
  outN = nr;
}

// One projection step of query q (double carried between steps) from the nine sums: the global frame's
// for the plain forms, the query frame's for the compensated one.
template <int FORM, int SEM>
__device__ __forceinline__ void fit_total(const double* S, V3<double>& qd, V3<float> qf, float stepMax, float4& nout) {
  float kind;
  if constexpr (FORM == 0) {
    V3<float> p, n;
    fit<float, float, SEM>((float)S[0], V3<float>{(float)S[1], (float)S[2], (float)S[3]},
                           V3<float>{(float)S[4], (float)S[5], (float)S[6]}, (float)S[7], (float)S[8], qf, stepMax, p, n, kind);
    qd = V3<double>{p.x, p.y, p.z};
    nout = make_float4(n.x, n.y, n.z, kind);
  } else {
    V3<double> p, n;
    if constexpr (FORM == 1) {  // the query is the origin
      fit<double, double, SEM, true>(S[0], V3<double>{S[1], S[2], S[3]}, V3<double>{S[4], S[5], S[6]}, S[7], S[8],
                                     V3<double>{0, 0, 0}, (double)stepMax, p, n, kind);
      qd = V3<double>{(double)qf.x + p.x, (double)qf.y + p.y, (double)qf.z + p.z};
    } else {
      fit<double, double, SEM>(S[0], V3<double>{S[1], S[2], S[3]}, V3<double>{S[4], S[5], S[6]}, S[7], S[8], qd,
                               (double)stepMax, p, n, kind);
      qd = p;
    }
    nout = make_float4((float)n.x, (float)n.y, (float)n.z, kind);
  }
}
template <int FORM, int SEM>
__device__ __forceinline__ void fit_step(const typename FormT<FORM>::Acc& acc, V3<double>& qd, V3<float> qf, float stepMax,
                                         float4& nout) {
  if constexpr (FORM == 1) {
    const double S[9] = {acc.w.val(),  acc.px.val(), acc.py.val(), acc.pz.val(), acc.nx.val(),
                         acc.ny.val(), acc.nz.val(), acc.pn.val(), acc.pp.val()};
    fit_total<1, SEM>(S, qd, qf, stepMax, nout);
  } else {
    const double S[9] = {acc.w, acc.px, acc.py, acc.pz, acc.nx, acc.ny, acc.nz, acc.pn, acc.pp};
    fit_total<FORM, SEM>(S, qd, qf, stepMax, nout);
  }
}

// ----------------------------------------------------------------------------- kernels
// MLoD projection of the sorted queries q[0..m) in place (projectCuda, Fastapss.cu:398-437):
// n_iter steps per query, one lane per query; queries whose caller index perm[i] >= limit are
// skipped.  A wavefront's 64 lanes hold 64 consecutive (curve-ordered) queries, so they start
// their walks together and load the same nodes at the same iterations for much of them.
template <int FORM, int SEM, int KT, bool CNT>
__global__ __launch_bounds__(PBS) void k_project(TreeView tv, KParams kp, float4* __restrict__ q, float4* __restrict__ qn,
                                                 const uint32_t* __restrict__ perm, uint32_t m, uint32_t limit,
                                                 uint32_t nIter, float stepMax, float cutoff, uint32_t minDepth,
                                                 unsigned long long* __restrict__ counters) {
  using T = typename FormT<FORM>::T;
  __shared__ WalkLds<FORM> lds;
  const int tid = threadIdx.x;
  const uint32_t i = xcd_block() * PBS + tid;
  const bool live = i < m && !(limit < m && perm[i] >= limit);
  Counters ct{0, 0, 0, 0, 0};
  if (__any(live)) {  // uniform over a wavefront: its lanes load node records together
    const float4 q4 = live ? q[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    V3<double> qd{q4.x, q4.y, q4.z};
    float4 nout = make_float4(0.f, 0.f, 0.f, 0.f);
    for (uint32_t it = 0; it < nIter; ++it) {
      typename FormT<FORM>::Acc acc;
      acc.init();
      const V3<float> qf{(float)qd.x, (float)qd.y, (float)qd.z};
      V3<T> qt;
      if constexpr (FORM == 2)
        qt = V3<T>{qd.x, qd.y, qd.z};
      else
        qt = V3<T>{qf.x, qf.y, qf.z};
      traverse<FORM, SEM, KT, CNT>(acc, kp, tv, qt, (T)cutoff, minDepth, live, lds, tid, ct);
      fit_step<FORM, SEM>(acc, qd, qf, stepMax, nout);
    }
    if (live) {
      q[i] = make_float4((float)qd.x, (float)qd.y, (float)qd.z, 0.f);
      qn[i] = nout;
    }
  }
  if constexpr (CNT) {
    // lane slots: 64 x the longest loop of the wavefront (lanes wait for it)
    uint32_t wmax = ct.iters;
    for (int o = 32; o > 0; o >>= 1) wmax = max(wmax, (uint32_t)__shfl_xor((int)wmax, o));
    if (live) {
      atomicAdd(&counters[0], (unsigned long long)ct.far_);
      atomicAdd(&counters[1], (unsigned long long)ct.leafPts);
      atomicAdd(&counters[2], (unsigned long long)ct.tested);
      atomicAdd(&counters[3], (unsigned long long)ct.nearN);
      atomicAdd(&counters[4], (unsigned long long)ct.iters);
    }
    if (__lane_id() == 0) atomicAdd(&counters[5], (unsigned long long)wmax);
  }
}

// k_project with the grouped walk: a wavefront projects 8 queries, one wavefront a workgroup.  Bound by
// the latency of its own instructions (about 400 a node): 1k queries, three steps, 60k points: 1.77 -> 0.49
// ms.  With the records staged through LDS as in the lane walk it took 0.57: the compiler then holds the
// exchange back until the staging loads are in.
template <int FORM, int SEM, int KT>
__global__ __launch_bounds__(64) void k_project_group(TreeView tv, KParams kp, float4* __restrict__ q,
                                                      float4* __restrict__ qn, const uint32_t* __restrict__ perm,
                                                      uint32_t m, uint32_t limit, uint32_t nIter, float stepMax,
                                                      float cutoff, uint32_t minDepth) {
  __shared__ GroupLds lds;
  const uint32_t lane = threadIdx.x, c = lane & (kGroup - 1u), grp = lane / kGroup;
  const uint32_t i = xcd_block() * kGroups + grp;
  const bool live = i < m && !(limit < m && perm[i] >= limit);
  if (!any_lane(live)) return;
  const float4 q4 = live ? q[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  V3<double> qd{q4.x, q4.y, q4.z};
  float4 nout = make_float4(0.f, 0.f, 0.f, 0.f);
  for (uint32_t it = 0; it < nIter; ++it) {
    GroupSums gs;
    gs.init();
    const V3<float> qf{(float)qd.x, (float)qd.y, (float)qd.z};
    if (!walk_short<FORM>(tv, qf, minDepth, live))
      traverse_group<FORM, SEM, KT, true, FORM == 0>(gs, kp, tv, qf, cutoff, minDepth, live, lds);
    else if (tv.nn < (1u << 26))
      traverse_group<FORM, SEM, KT, false, false>(gs, kp, tv, qf, cutoff, minDepth, live, lds);
    else
      traverse_group<FORM, SEM, KT, true, false>(gs, kp, tv, qf, cutoff, minDepth, live, lds);
    lds.sum[grp][c] = FORM == 0 ? (double)gs.l0 : gs.k0.val();
    if (c == 0) lds.sum[grp][8] = FORM == 0 ? (double)gs.l8 : gs.k8.val();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    double S[9];
#pragma unroll
    for (int t = 0; t < 9; ++t) S[t] = lds.sum[grp][t];
    fit_total<FORM, SEM>(S, qd, qf, stepMax, nout);
  }
  if (live && c == 0) {
    q[i] = make_float4((float)qd.x, (float)qd.y, (float)qd.z, 0.f);
    qn[i] = nout;
  }
}

// k_project with the wave-shared walk: every lane of a wavefront calls the walk (lanes without a
// query take part in no node), so the walk's control flow stays wave-uniform.
template <int FORM, int SEM, int KT, bool CNT, bool EXACT>
__global__ __launch_bounds__(PBS) void k_project_wave(TreeView tv, KParams kp, float4* __restrict__ q,
                                                      float4* __restrict__ qn, const uint32_t* __restrict__ perm,
                                                      uint32_t m, uint32_t limit, uint32_t nIter, float stepMax,
                                                      float cutoff, uint32_t minDepth,
                                                      unsigned long long* __restrict__ counters) {
  using T = typename FormT<FORM>::T;
  __shared__ WaveLevel sLv[kLevels][PBS / 64];
  __shared__ T sMul[kLevels][PBS];
  __shared__ T sDist[kLevels][PBS];
  __shared__ uint8_t sNear[kLevels][PBS];
  const int tid = threadIdx.x;
  const int wv = tid >> 6;
  const uint32_t i = xcd_block() * PBS + tid;
  const bool live = i < m && !(limit < m && perm[i] >= limit);
  Counters ct{0, 0, 0, 0, 0};
  uint32_t waveIters = 0;
  const WaveStack<T> st{sLv, sMul, sDist, sNear};
  const float4 q4 = live ? q[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  V3<double> qd{q4.x, q4.y, q4.z};
  float4 nout = make_float4(0.f, 0.f, 0.f, 0.f);
  for (uint32_t it = 0; it < nIter; ++it) {
    typename FormT<FORM>::Acc acc;
    acc.init();
    const V3<float> qf{(float)qd.x, (float)qd.y, (float)qd.z};
    V3<T> qt;
    if constexpr (FORM == 2)
      qt = V3<T>{qd.x, qd.y, qd.z};
    else
      qt = V3<T>{qf.x, qf.y, qf.z};
    traverse_wave<FORM, SEM, KT, CNT, EXACT>(acc, kp, tv, qt, (T)cutoff, minDepth, live, st, tid, wv, ct, waveIters);
    if constexpr (FORM == 1) acc.flush();
    if (live) fit_step<FORM, SEM>(acc, qd, qf, stepMax, nout);
  }
  if (live) {
    q[i] = make_float4((float)qd.x, (float)qd.y, (float)qd.z, 0.f);
    qn[i] = nout;
  }
  if constexpr (CNT) {
    if (live) {
      atomicAdd(&counters[0], (unsigned long long)ct.far_);
      atomicAdd(&counters[1], (unsigned long long)ct.leafPts);
      atomicAdd(&counters[2], (unsigned long long)ct.tested);
      atomicAdd(&counters[3], (unsigned long long)ct.nearN);
      atomicAdd(&counters[4], (unsigned long long)ct.iters);
    }
    if (__lane_id() == 0) atomicAdd(&counters[5], (unsigned long long)waveIters);
  }
}

// ----------------------------------------------------------------------------- global APSS
// One projection step from the nine sums over all neighbours in FP64, {sum w, sum w p, sum w n, sum w p.n,
// sum w |p|^2}, about `o`, which is 0 in the FP64 form.  The compensated form takes them about a point of the cloud
// and moves them to the query's frame (that costs 1e-16 of the squared distance between the two against the
// kernel's width squared).
template <int FORM, int SEM>
__device__ __forceinline__ void fit_sums(const double* S, V3<float> o, V3<double>& qd, float stepMax, float4& nout) {
  const V3<float> qf{(float)qd.x, (float)qd.y, (float)qd.z};
  if constexpr (FORM == 1) {
    const V3<double> q{(double)qf.x - o.x, (double)qf.y - o.y, (double)qf.z - o.z}, sp{S[1], S[2], S[3]}, sn{S[4], S[5], S[6]};
    const double R[9] = {S[0], sp.x - q.x * S[0], sp.y - q.y * S[0], sp.z - q.z * S[0], sn.x, sn.y, sn.z, S[7] - dot3(q, sn),
                         S[8] - 2.0 * dot3(q, sp) + dot3(q, q) * S[0]};
    fit_total<1, SEM>(R, qd, qf, stepMax, nout);
  } else {
    fit_total<FORM, SEM>(S, qd, qf, stepMax, nout);
  }
}

typedef double Acc4 __attribute__((ext_vector_type(4)));

// Global APSS over all points (GlobalAPSS.cu:113-192 / APSSStats, CPUUtils.cpp:515-528), compensated and
// FP64 forms: the sums are a contraction, weights (queries x points) times moments (points x 9), and run on the matrix cores.
// A workgroup of W wavefronts takes 16 queries; in one step a wavefront takes 4 points, each lane the
// weight of one (query lane % 16, point lane / 16) pair, and one FP64 16x16x4 matrix instruction adds
// the 64 weights times the 4 points' nine moments (columns 9..15 hold copies that nobody reads).  So a
// pair costs its distance and weight and none of the nine sums, which the matrix cores add in FP64:
// the weights keep their form's precision, the sums gain.  Points are staged through LDS a tile at a time,
// their moments formed once per tile.
// Step g of a tile belongs to slice g % 16; a wavefront holds 16 / W slices apart, and the slices are
// added in order at the end, so the result does not depend on W.
// Bound by the weights' vector instructions and the FP64 products (56 % and 33 % of the SIMDs' cycles).  30k
// points, four sigmas, FP32C: 20k queries 6.0 -> 0.80 ms, 500 queries 6.0 -> 0.19 (one lane per query left the
// chip two thirds empty, and each pair paid nine compensated sums), 100k queries 6.4 -> 3.3; FP64, 8k queries:
// 20.1 -> 1.05.
// The fit uses the 1e-12 plane threshold of GlobalAPSS.cu:143 (the REF_CPU fit).
constexpr int kGlobalQ = 16;
constexpr int kSlices = 16;
template <int FORM, int KT, int W>
__global__ __launch_bounds__(W * 64) void k_global(TreeView tv, KParams kp, float4* __restrict__ q, float4* __restrict__ qn,
                                                   const uint32_t* __restrict__ perm, uint32_t m, uint32_t limit,
                                                   uint32_t nIter, float stepMax) {
  using T = typename FormT<FORM>::T;
  constexpr uint32_t TILE = W == 4 ? 256 : 512;
  constexpr int NA = kSlices / W;         // slices of a wavefront
  constexpr int U = 4;                    // steps of a round
  constexpr uint32_t ROUND = U * W * 4;   // points of a round (a multiple of the slices' 64)
  __shared__ float4 sP[TILE];
  __shared__ double sF[TILE][9];  // then the slices' sums: [16 slices][16 queries][9]
  __shared__ double sS[kGlobalQ][9], sQ[kGlobalQ][3];
  static_assert(sizeof(sF) >= sizeof(double) * kSlices * kGlobalQ * 9, "the slices' sums fit the moments' tile");
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, row = lane & 15u, kk = lane >> 4, col = min(row, 8u);
  const uint32_t i = blockIdx.x * kGlobalQ + tid;
  const bool active = tid < kGlobalQ && i < m && !(limit < m && perm[i] >= limit);
  const float4 mid = tv.pts[tv.n >> 1];
  const V3<float> o = FORM == 1 ? V3<float>{mid.x, mid.y, mid.z} : V3<float>{0.f, 0.f, 0.f};  // the sums' origin
  V3<double> qd{0, 0, 0};  // (of the first 16 threads)
  float4 nout = make_float4(0.f, 0.f, 0.f, 0.f);
  if (active) {
    const float4 q4 = q[i];
    qd = V3<double>{q4.x, q4.y, q4.z};
  }
  for (uint32_t it = 0; it < nIter; ++it) {
    if (tid < kGlobalQ) {
      sQ[tid][0] = FORM == 2 ? qd.x : (double)(float)qd.x;
      sQ[tid][1] = FORM == 2 ? qd.y : (double)(float)qd.y;
      sQ[tid][2] = FORM == 2 ? qd.z : (double)(float)qd.z;
    }
    __syncthreads();
    const T qx = (T)sQ[row][0], qy = (T)sQ[row][1], qz = (T)sQ[row][2];
    Acc4 acc[NA];
#pragma unroll
    for (int u = 0; u < NA; ++u) acc[u] = Acc4{0, 0, 0, 0};
    for (uint32_t base = 0; base < tv.n; base += TILE) {
      const uint32_t cnt = min(TILE, tv.n - base), end = (cnt + ROUND - 1u) / ROUND * ROUND;
      __syncthreads();
      for (uint32_t t = tid; t < end; t += W * 64) {
        const bool in = t < cnt;  // past the end: the tile's first point with no moments
        const float4 P = tv.pts[base + (in ? t : 0u)], N = tv.nrm[base + (in ? t : 0u)];
        const double a = in ? (double)P.w : 0.0, x = (double)P.x - o.x, y = (double)P.y - o.y, z = (double)P.z - o.z;
        sP[t] = P;
        sF[t][0] = a;
        sF[t][1] = a * x, sF[t][2] = a * y, sF[t][3] = a * z;
        sF[t][4] = a * N.x, sF[t][5] = a * N.y, sF[t][6] = a * N.z;
        sF[t][7] = a * ((x * N.x + y * N.y) + z * N.z);
        sF[t][8] = a * ((x * x + y * y) + z * z);
      }
      __syncthreads();
      for (uint32_t t0 = 4u * wave + kk; t0 < end; t0 += ROUND) {
        T d2[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float4 P = sP[t0 + u * 4 * W];
          const T dx = (T)P.x - qx, dy = (T)P.y - qy, dz = (T)P.z - qz;
          if constexpr (FORM == 2)
            d2[u] = dx * dx + dy * dy + dz * dz;
          else
            d2[u] = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
        }
        T w[U];
        if constexpr (FORM == 2) {
#pragma unroll
          for (int u = 0; u < U; ++u) w[u] = weight64<KT>(kp, d2[u]);
        } else {
          weights32<KT, U>(kp, d2, w);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
          acc[u % NA] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)w[u], sF[t0 + u * 4 * W][col], acc[u % NA], 0, 0, 0);
      }
    }
    // the slices' sums: register r of a lane holds query 4 r + lane / 16, moment lane % 16
    __syncthreads();
    double* red = &sF[0][0];
    if (row < 9u) {
#pragma unroll
      for (int u = 0; u < NA; ++u)
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r)
          red[((u * W + wave) * kGlobalQ + 4u * r + kk) * 9u + row] = acc[u][r];
    }
    __syncthreads();
    for (uint32_t t = tid; t < kGlobalQ * 9u; t += W * 64) {
      double x = 0.0;
      for (int sl = 0; sl < kSlices; ++sl) x += red[sl * kGlobalQ * 9 + t];
      sS[t / 9u][t % 9u] = x;
    }
    __syncthreads();
    if (tid < kGlobalQ) fit_sums<FORM, MLOD_SEM_REF_CPU>(sS[tid], o, qd, stepMax, nout);
  }
  if (active) {
    q[i] = make_float4((float)qd.x, (float)qd.y, (float)qd.z, 0.f);
    qn[i] = nout;
  }
}

// The plain FP32 form of global APSS: the reference's own sums, in FP32 and in point order, one lane per
// query over point tiles in LDS, a point's mean divided out once a tile.  Bound by vector instructions and, up to
// some 100k queries, by the chip being part empty: 20k queries, 30k points, four sigmas 5.3 ms (5.7 with the mean
// formed for every pair), rational kernel 8.1 (9.4).
template <int KT>
__global__ __launch_bounds__(PBS) void k_global_plain(TreeView tv, KParams kp, float4* __restrict__ q, float4* __restrict__ qn,
                                                const uint32_t* __restrict__ perm, uint32_t m, uint32_t limit,
                                                uint32_t nIter, float stepMax) {
  __shared__ float4 sP[PBS], sN[PBS];
  __shared__ V3<float> sM[PBS];
  const int tid = threadIdx.x;
  const uint32_t i = blockIdx.x * PBS + tid;
  const bool active = i < m && !(limit < m && perm[i] >= limit);
  const float4 q4 = active ? q[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  V3<double> qd{q4.x, q4.y, q4.z};
  float4 nout = make_float4(0.f, 0.f, 0.f, 0.f);
  for (uint32_t it = 0; it < nIter; ++it) {
    AccP32 acc;
    acc.init();
    const V3<float> qf{(float)qd.x, (float)qd.y, (float)qd.z};
    for (uint32_t base = 0; base < tv.n; base += PBS) {
      __syncthreads();
      if (base + tid < tv.n) {
        sP[tid] = tv.pts[base + tid];
        sN[tid] = tv.nrm[base + tid];
        sM[tid] = point_mean<true>(sP[tid]);
      }
      __syncthreads();
      const uint32_t cnt = min((uint32_t)PBS, tv.n - base);
      if (active)
        for (uint32_t j = 0; j < cnt; ++j) add_point_plain<KT>(acc, kp, sP[j], sN[j], sM[j], qf, 1.f);
    }
    fit_step<0, MLOD_SEM_REF_CPU>(acc, qd, qf, stepMax, nout);
  }
  if (active) {
    q[i] = make_float4((float)qd.x, (float)qd.y, (float)qd.z, 0.f);
    qn[i] = nout;
  }
}

// Serving step launch: workgroup b projects the kBatchWG pool slots of pool block blocks[b].y
// with the tree, kernel and parameters of run descriptor blocks[b].x, read by the workgroup from
// the launch table with wave-uniform (scalar) loads; per-lane work and results are those of
// k_project, so a query gives the same bits alone, in any mix, and whether its steps run in one
// launch or several (the FP64 form carries its FP64 position between launches in qdp, as
// k_project carries it between the steps of one launch).  A launch for interactive requests
// raises its wavefronts' issue priority (s_setprio), so they keep close to their unloaded speed
// beside bulk launches.  A run taking its last steps writes its results to the host staging and
// flags each of its workgroups done (system-scope release).
template <int FORM, int SEM, int KT>
__global__ __launch_bounds__(PBS) void k_project_batch(const ReqDesc* __restrict__ reqs, const uint2* __restrict__ blocks,
                                                       float4* __restrict__ q, float4* __restrict__ qn,
                                                       double4* __restrict__ qdp, BatchOut bo, uint32_t prio) {
  static_assert(PBS == kBatchWG, "one workgroup per pool block");
  using T = typename FormT<FORM>::T;
  __shared__ WalkLds<FORM> lds;
  if (prio) __builtin_amdgcn_s_setprio(3);
  const int tid = threadIdx.x;
  const uint32_t lb = xcd_block();
  const uint2 b = blocks[lb];
  const uint32_t r = __builtin_amdgcn_readfirstlane(b.x), pb = __builtin_amdgcn_readfirstlane(b.y);
  const ReqDesc& R = reqs[r];
  const uint32_t i = pb * PBS + tid, outOff = R.outOff;
  const bool live = i < R.pad0 + R.count;
  V3<double> qd{0, 0, 0};
  float4 nout = make_float4(0.f, 0.f, 0.f, 0.f);
  if (__any(live)) {  // uniform over a wavefront: its lanes load node records together
    const TreeView tv = R.tv;
    const KParams& kp = R.kp;
    const float cutoff = R.cutoff, stepMax = R.stepMax;
    const uint32_t minDepth = R.minDepth, nIter = R.nIter;
    if (live) {
      if constexpr (FORM == 2) {
        const double4 d4 = qdp[i];
        qd = V3<double>{d4.x, d4.y, d4.z};
      } else {
        const float4 q4 = q[i];
        qd = V3<double>{q4.x, q4.y, q4.z};
      }
    }
    Counters ct{0, 0, 0, 0, 0};
    for (uint32_t it = 0; it < nIter; ++it) {
      typename FormT<FORM>::Acc acc;
      acc.init();
      const V3<float> qf{(float)qd.x, (float)qd.y, (float)qd.z};
      V3<T> qt;
      if constexpr (FORM == 2)
        qt = V3<T>{qd.x, qd.y, qd.z};
      else
        qt = V3<T>{qf.x, qf.y, qf.z};
      traverse<FORM, SEM, KT, false>(acc, kp, tv, qt, (T)cutoff, minDepth, live, lds, tid, ct);
      fit_step<FORM, SEM>(acc, qd, qf, stepMax, nout);
    }
  }
  if (live) {
    const float4 p4 = make_float4((float)qd.x, (float)qd.y, (float)qd.z, 0.f);
    q[i] = p4;
    qn[i] = nout;
    if constexpr (FORM == 2) qdp[i] = make_double4(qd.x, qd.y, qd.z, 0.0);
    if (outOff != kNoOut) {
      const uint64_t d = outOff + bo.pidx[i], e = (uint64_t)bo.cap + d;
      bo.out[3 * d] = p4.x;
      bo.out[3 * d + 1] = p4.y;
      bo.out[3 * d + 2] = p4.z;
      bo.out[3 * e] = nout.x;
      bo.out[3 * e + 1] = nout.y;
      bo.out[3 * e + 2] = nout.z;
    }
  }
  if (outOff != kNoOut) {  // uniform over the workgroup
    __threadfence_system();
    __syncthreads();
    if (tid == 0) __hip_atomic_store(bo.flag + lb, bo.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

template <int FORM, int SEM>
void launch_batch_all(const ReqDesc* r, const uint2* blocks, uint32_t nblk, float4* q, float4* qn, double4* qd,
                      const BatchOut& bo, uint32_t prio, hipStream_t s) {
  k_project_batch<FORM, SEM, -1><<<nblk, PBS, 0, s>>>(r, blocks, q, qn, qd, bo, prio);
}

// Batches of at most this many queries take the grouped walk: it issues three times the instructions of
// the lane walk and is done in a third of its time while the chip has room for them.  Three steps on 1M
// points, four sigmas, FP32C, us with a lane / a group: 4k queries 1140 / 427, 16k 1178 / 537, 32k
// 1180 / 905, 48k 1271 / 1212, 64k 1289 / 1464; plain FP32, rational, cutoff 3, torus: 32k 5412 / 3097,
// 48k 5673 / 4314, 64k 5807 / 5470.  It is the uploaded queries that count, not those a call asks for: a few
// of a large upload are walked a lane each, beside lanes that have nothing to do (they lie anywhere along the
// curve, and wavefronts without one end at once).
constexpr uint32_t kGroupMax = 49152;

template <int FORM, int SEM, int KT, bool CNT>
int launch_one(const mlod_tree* t, const KParams& kp, uint32_t limit, uint32_t nIter, float stepMax,
               unsigned long long* counters, hipStream_t s) {
  const uint32_t m = t->qs.m;
  if (m == 0) return MLOD_OK;
  if (t->traversal == MLOD_TRAVERSAL_WAVE) {
    if (FORM != 0 || areas_normal(t->radius, t->n))
      k_project_wave<FORM, SEM, KT, CNT, false><<<(m + PBS - 1) / PBS, PBS, 0, s>>>(
          t->view(), kp, t->qs.q, t->qs.qn, t->qs.perm, m, limit, nIter, stepMax, t->cutoff, t->min_depth, counters);
    else
      k_project_wave<FORM, SEM, KT, CNT, FORM == 0><<<(m + PBS - 1) / PBS, PBS, 0, s>>>(
          t->view(), kp, t->qs.q, t->qs.qn, t->qs.perm, m, limit, nIter, stepMax, t->cutoff, t->min_depth, counters);
  } else if (FORM != 2 && !CNT && m <= kGroupMax) {
    k_project_group<FORM == 2 ? 1 : FORM, SEM, KT><<<(m + kGroups - 1) / kGroups, 64, 0, s>>>(
        t->view(), kp, t->qs.q, t->qs.qn, t->qs.perm, m, limit, nIter, stepMax, t->cutoff, t->min_depth);
  } else {
    k_project<FORM, SEM, KT, CNT><<<(m + PBS - 1) / PBS, PBS, 0, s>>>(t->view(), kp, t->qs.q, t->qs.qn, t->qs.perm, m,
                                                                       limit, nIter, stepMax, t->cutoff, t->min_depth,
                                                                       counters);
  }
  return MLOD_OK;
}

template <int FORM, int KT>
void launch_global(const mlod_tree* t, const KParams& kp, uint32_t limit, uint32_t nIter, float stepMax, hipStream_t s) {
  const uint32_t m = t->qs.m;
  if constexpr (FORM == 0) {
    k_global_plain<KT><<<(m + PBS - 1) / PBS, PBS, 0, s>>>(t->view(), kp, t->qs.q, t->qs.qn, t->qs.perm, m, limit, nIter,
                                                            stepMax);
  } else {
    // Four wavefronts a workgroup load the chip's 1024 SIMDs twice over from 512 workgroups on; below
    // that the points are split over sixteen (30k points, us with 4 / 16 wavefronts: 500 queries 276 /
    // 189, 4k 289 / 203, 8k 385 / 389, 12k 496 / 554, 20k 761 / 884).
    const uint32_t grid = (m + kGlobalQ - 1) / kGlobalQ;
    if (grid >= 512)
      k_global<FORM, KT, 4><<<grid, 4 * 64, 0, s>>>(t->view(), kp, t->qs.q, t->qs.qn, t->qs.perm, m, limit, nIter, stepMax);
    else
      k_global<FORM, KT, 16><<<grid, 16 * 64, 0, s>>>(t->view(), kp, t->qs.q, t->qs.qn, t->qs.perm, m, limit, nIter, stepMax);
  }
}

template <int FORM, int SEM>
int dispatch_kt(const mlod_tree* t, const KParams& kp, uint32_t limit, uint32_t nIter, float stepMax, hipStream_t s) {
  switch (kp.type) {
    case MLOD_KERNEL_GAUSSIAN: return launch_one<FORM, SEM, MLOD_KERNEL_GAUSSIAN, false>(t, kp, limit, nIter, stepMax, nullptr, s);
    case MLOD_KERNEL_SINGULAR: return launch_one<FORM, SEM, MLOD_KERNEL_SINGULAR, false>(t, kp, limit, nIter, stepMax, nullptr, s);
    default: return launch_one<FORM, SEM, MLOD_KERNEL_GAUSSIAN_MULTIPLE, false>(t, kp, limit, nIter, stepMax, nullptr, s);
  }
}

template <int FORM>
void dispatch_global(const mlod_tree* t, const KParams& kp, uint32_t limit, uint32_t nIter, float stepMax, hipStream_t s) {
  switch (kp.type) {
    case MLOD_KERNEL_GAUSSIAN: launch_global<FORM, MLOD_KERNEL_GAUSSIAN>(t, kp, limit, nIter, stepMax, s); break;
    case MLOD_KERNEL_SINGULAR: launch_global<FORM, MLOD_KERNEL_SINGULAR>(t, kp, limit, nIter, stepMax, s); break;
    default: launch_global<FORM, MLOD_KERNEL_GAUSSIAN_MULTIPLE>(t, kp, limit, nIter, stepMax, s); break;
  }
}

}  // namespace

KParams make_kparams(const mlod_kernel& k) {
  KParams p{};
  p.type = k.type;
  p.ns = k.type == MLOD_KERNEL_GAUSSIAN_MULTIPLE ? k.n_sigmas : 1;
  p.c = k.constant_shift;
  p.cp = k.constant_shift > 0.0001f ? k.constant_shift : 0.0001f;
  p.e = k.exponent;
  p.c4 = 0.25f * p.c;
  p.cp4 = 0.25f * p.cp;
  const double er = std::nearbyint((double)k.exponent);
  p.cpe = std::pow((double)p.cp, (double)p.e);
  p.eint = (er == (double)k.exponent && er >= 1.0 && er <= 16.0) ? (int)er : -1;
  const double log2e = 1.4426950408889634;
  if (k.type == MLOD_KERNEL_GAUSSIAN_MULTIPLE) {
    for (int s = 0; s < k.n_sigmas && s < MLOD_MAX_SIGMAS; ++s) {
      const double sg = k.sigmas[s];
      p.a[s] = (float)(-log2e / (2.0 * sg * sg));
      p.b[s] = (float)(1.0 / (sg * sg * sg));
      p.ad[s] = (double)(-1.44269504088896340736L / (2.0L * sg * sg));
      p.bd[s] = 1.0 / (sg * sg * sg);
    }
    // the weights are formed two or four terms at a time: a term past the last is the first's exponential times 0
    // (of a coefficient 0 it would be exp2(inf * 0), a NaN, where the squared distance overflows)
    for (int s = p.ns; s < MLOD_MAX_SIGMAS; ++s) p.a[s] = p.a[0];
    for (int s = p.ns; s < MLOD_MAX_SIGMAS + 1; ++s) p.ad[s] = p.ad[0];
  } else if (k.type == MLOD_KERNEL_GAUSSIAN) {
    const double sg = k.sigma;
    p.a[0] = (float)(-log2e / (2.0 * sg * sg));
    p.ad[0] = (double)(-1.44269504088896340736L / (2.0L * sg * sg));
  }
  return p;
}

int launch_project_batch(const ReqDesc* d_reqs, const uint2* d_blocks, uint32_t nblk, float4* d_q, float4* d_qn,
                         double4* d_qd, const BatchOut& bo, uint32_t prio, int semantics, int precision,
                         hipStream_t s) {
  if (nblk == 0) return MLOD_OK;
  const bool cpu = semantics == MLOD_SEM_REF_CPU;
  if (precision == MLOD_PREC_FP32C) {
    if (cpu) launch_batch_all<1, MLOD_SEM_REF_CPU>(d_reqs, d_blocks, nblk, d_q, d_qn, d_qd, bo, prio, s);
    else launch_batch_all<1, MLOD_SEM_REF_GPU>(d_reqs, d_blocks, nblk, d_q, d_qn, d_qd, bo, prio, s);
  } else if (precision == MLOD_PREC_FP32) {
    if (cpu) launch_batch_all<0, MLOD_SEM_REF_CPU>(d_reqs, d_blocks, nblk, d_q, d_qn, d_qd, bo, prio, s);
    else launch_batch_all<0, MLOD_SEM_REF_GPU>(d_reqs, d_blocks, nblk, d_q, d_qn, d_qd, bo, prio, s);
  } else {
    if (!d_qd) return fail(MLOD_ERR_INVALID, "the FP64 form needs the FP64 position pool");
    if (cpu) launch_batch_all<2, MLOD_SEM_REF_CPU>(d_reqs, d_blocks, nblk, d_q, d_qn, d_qd, bo, prio, s);
    else launch_batch_all<2, MLOD_SEM_REF_GPU>(d_reqs, d_blocks, nblk, d_q, d_qn, d_qd, bo, prio, s);
  }
  LAUNCH_CHECK();
  return MLOD_OK;
}

int launch_project(mlod_tree* t, uint32_t n, uint32_t n_iter, float step_max, hipStream_t s) {
  const KParams kp = make_kparams(t->kernel);
  const uint32_t limit = n;
  if (t->mode == MLOD_MODE_GLOBAL) {
    switch (t->precision) {
      case MLOD_PREC_FP32C: dispatch_global<1>(t, kp, limit, n_iter, step_max, s); break;
      case MLOD_PREC_FP64: dispatch_global<2>(t, kp, limit, n_iter, step_max, s); break;
      default: dispatch_global<0>(t, kp, limit, n_iter, step_max, s); break;
    }
    LAUNCH_CHECK();
    return MLOD_OK;
  }
  const bool cpu = t->semantics == MLOD_SEM_REF_CPU;
  int r;
  switch (t->precision) {
    case MLOD_PREC_FP32C:
      r = cpu ? dispatch_kt<1, MLOD_SEM_REF_CPU>(t, kp, limit, n_iter, step_max, s)
              : dispatch_kt<1, MLOD_SEM_REF_GPU>(t, kp, limit, n_iter, step_max, s);
      break;
    case MLOD_PREC_FP64:
      r = cpu ? dispatch_kt<2, MLOD_SEM_REF_CPU>(t, kp, limit, n_iter, step_max, s)
              : dispatch_kt<2, MLOD_SEM_REF_GPU>(t, kp, limit, n_iter, step_max, s);
      break;
    default:
      r = cpu ? dispatch_kt<0, MLOD_SEM_REF_CPU>(t, kp, limit, n_iter, step_max, s)
              : dispatch_kt<0, MLOD_SEM_REF_GPU>(t, kp, limit, n_iter, step_max, s);
      break;
  }
  if (r != MLOD_OK) return r;
  LAUNCH_CHECK();
  return MLOD_OK;
}

// Counter pass: one FP32C step with counting on; positions are not advanced (the step
// runs on a scratch copy of the queries).
int launch_count(mlod_tree* t, uint32_t n, unsigned long long* d_out4, hipStream_t s) {
  const KParams kp = make_kparams(t->kernel);
  const bool cpu = t->semantics == MLOD_SEM_REF_CPU;
  int r;
#define MLOD_CNT_CASE(SEMV)                                                                                  \
  switch (kp.type) {                                                                                         \
    case MLOD_KERNEL_GAUSSIAN: r = launch_one<1, SEMV, MLOD_KERNEL_GAUSSIAN, true>(t, kp, n, 1, t->radius, d_out4, s); break; \
    case MLOD_KERNEL_SINGULAR: r = launch_one<1, SEMV, MLOD_KERNEL_SINGULAR, true>(t, kp, n, 1, t->radius, d_out4, s); break; \
    default: r = launch_one<1, SEMV, MLOD_KERNEL_GAUSSIAN_MULTIPLE, true>(t, kp, n, 1, t->radius, d_out4, s); break;     \
  }
  if (cpu) {
    MLOD_CNT_CASE(MLOD_SEM_REF_CPU)
  } else {
    MLOD_CNT_CASE(MLOD_SEM_REF_GPU)
  }
#undef MLOD_CNT_CASE
  if (r != MLOD_OK) return r;
  LAUNCH_CHECK();
  return MLOD_OK;
}

}  // namespace mlod
