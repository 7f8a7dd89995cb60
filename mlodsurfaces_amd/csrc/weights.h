// weights.h — the weight kernels on the device, shared by the projection and neighbour kernels, and the
// correctly rounded division and square root they and the plain walk take.
#pragma once

#include "mlod_internal.h"

namespace mlod {
namespace {

// Correctly rounded FP32 quotients and square roots in fewer instructions than the compiler's own
// expansions (7 against 11, 3 where the reciprocal is at hand, and 8 against 16): the plain walk is bound by
// vector instructions, and a third of them were these (1M points and queries, rational kernel: 10.0 ->
// 8.1 ms a step, the same bits).  An approximation within an ulp, its residual by one fused operation,
// which is exact, and one fused correction (Markstein, "Computation of elementary functions on the IBM
// RISC System/6000 processor", 1990).  The expansions spend the rest on operands at the ends of the
// exponent range.  Here the divisor is zero, infinite, or from 2^-126 to 2^126 (a smaller one's reciprocal
// overflows, a larger one's is flushed), and the quotient is right where it and the residual are normal
// (above some 2^-100), and within an ulp below; zeros, infinities and NaN go through the hardware's
// fix-up.  The square root is right from 2^-100 on,
// checked for every float there; below it loses up to an ulp, and a subnormal argument (a distance
// under 1e-19) is returned as it is.  Where areas or distances may lie outside, the plain walk has a variant with
// the compiler's (walk_short in project.hip).
__device__ __forceinline__ float quot_rcp(float n, float d, float r) {  // n / d, r = 1 / d correctly rounded
  const float q = __fmul_rn(n, r);
  return fmaf(fmaf(-d, q, n), r, q);
}
__device__ __forceinline__ float near_rcp(float d) {  // 1 / d, right but for some last bits
  const float r = __builtin_amdgcn_rcpf(d);
  return fmaf(fmaf(-d, r, 1.f), r, r);
}
__device__ __forceinline__ float quot(float n, float d) {
  return __builtin_amdgcn_div_fixupf(quot_rcp(n, d, near_rcp(d)), d, n);
}
__device__ __forceinline__ float root(float x) {
  const float y = __builtin_amdgcn_rsqf(x), s = __fmul_rn(x, y);
  const float t = fmaf(fmaf(-s, s, x), __fmul_rn(0.5f, y), s);
  return __builtin_amdgcn_classf(x, 0x2e0) ? x : t;  // zero, subnormal, +infinity
}

// FP32 weights (Kernel.cpp:64-83 / GPUUtils.cu:243-257) from the squared distance.
// KT < 0: the kernel type is read at run time from the (wave-uniform) coefficients, so one
// launch serves workgroups of different kernel types with a scalar branch per evaluation.
template <int KT, class KP>
__device__ __forceinline__ float weight32(const KP& k, float d2) {
  if constexpr (KT < 0) {
    if (k.type == MLOD_KERNEL_GAUSSIAN_MULTIPLE) return weight32<MLOD_KERNEL_GAUSSIAN_MULTIPLE>(k, d2);
    if (k.type == MLOD_KERNEL_GAUSSIAN) return weight32<MLOD_KERNEL_GAUSSIAN>(k, d2);
    return weight32<MLOD_KERNEL_SINGULAR>(k, d2);
  } else if constexpr (KT == MLOD_KERNEL_GAUSSIAN_MULTIPLE) {
    // sum over s of sigma_s^-3 * 2^(a_s d2), in order of s.  Statically indexed, so the coefficients
    // sit in scalar registers; two terms between wave-uniform exits (a scalar compare and branch;
    // the empty asm keeps the compiler from hoisting the compares into lane masks), so that two
    // exponentials are in flight.  A term past the last adds 0 times the first's exponential (make_kparams)
    float w = k.b[0] * __builtin_amdgcn_exp2f(d2 * k.a[0]);
    w = fmaf(k.b[1], __builtin_amdgcn_exp2f(d2 * k.a[1]), w);
    int ns = k.ns;
#pragma unroll
    for (int s = 2; s < 8; s += 2) {
      asm volatile("" : "+s"(ns));
      if (s >= ns) break;
      const float e0 = __builtin_amdgcn_exp2f(d2 * k.a[s]), e1 = __builtin_amdgcn_exp2f(d2 * k.a[s + 1]);
      w = fmaf(k.b[s], e0, w);
      w = fmaf(k.b[s + 1], e1, w);
    }
    // more sigmas (the sample models' settings use up to 30): four at a time, each group's
    // coefficients fetched by two 16-byte scalar loads (the table is 16-byte aligned)
    for (int s0 = 8; s0 < ns; s0 += 4) {
      const float4 A4 = *reinterpret_cast<const float4*>(k.a + s0);
      const float4 B4 = *reinterpret_cast<const float4*>(k.b + s0);
      const float e0 = __builtin_amdgcn_exp2f(d2 * A4.x), e1 = __builtin_amdgcn_exp2f(d2 * A4.y);
      const float e2 = __builtin_amdgcn_exp2f(d2 * A4.z), e3 = __builtin_amdgcn_exp2f(d2 * A4.w);
      w = fmaf(B4.x, e0, w);
      w = fmaf(B4.y, e1, w);
      w = fmaf(B4.z, e2, w);
      w = fmaf(B4.w, e3, w);
    }
    // an all-underflowed sum falls back to constant_shift (Kernel.cpp:69-73); nothing to do for a zero
    // one (the empty asm keeps the uniform branch from becoming two selects)
    if (__float_as_uint(k.c) << 1) {
      asm volatile("");
      w = w == 0.f ? k.c : w;
    }
    return w;
  } else if constexpr (KT == MLOD_KERNEL_GAUSSIAN) {
    return __builtin_amdgcn_exp2f(d2 * k.a[0]) + k.c;
  } else {
    float base;
    if ((__float_as_uint(k.c) & 0x7fffffffu) > 0x0da24260u) {  // |c| > 1e-30: the divisor is no subnormal (uniform)
      asm volatile("");
      base = quot(k.cp4, fmaf(d2, 0.25f, k.c4));  // both a quarter: the largest divisor has a normal reciprocal too
    } else {
      asm volatile("");
      base = k.cp / (d2 + k.c);
    }
    if (k.eint > 0) {
      float r = 1.f, b = base;
      for (int e = k.eint; e; e >>= 1) {
        if (e & 1) r *= b;
        b *= b;
      }
      return r;
    }
    return __builtin_amdgcn_exp2f(k.e * __builtin_amdgcn_logf(base));
  }
}

// weight32 of U squared distances at once: the terms of one sigma for all of them before the next
// sigma's, so that U exponentials are in flight and the uniform exits are shared.
template <int KT, int U, class KP>
__device__ __forceinline__ void weights32(const KP& k, const float (&d2)[U], float (&w)[U]) {
  if constexpr (KT == MLOD_KERNEL_GAUSSIAN_MULTIPLE) {
#pragma unroll
    for (int u = 0; u < U; ++u) w[u] = k.b[0] * __builtin_amdgcn_exp2f(d2[u] * k.a[0]);
    int ns = k.ns;
#pragma unroll
    for (int s = 1; s < 8; ++s) {
      asm volatile("" : "+s"(ns));
      if (s >= ns) break;
#pragma unroll
      for (int u = 0; u < U; ++u) w[u] = fmaf(k.b[s], __builtin_amdgcn_exp2f(d2[u] * k.a[s]), w[u]);
    }
    for (int s = 8; s < ns; ++s) {
      const float A = k.a[s], B = k.b[s];
#pragma unroll
      for (int u = 0; u < U; ++u) w[u] = fmaf(B, __builtin_amdgcn_exp2f(d2[u] * A), w[u]);
    }
    if (__float_as_uint(k.c) << 1) {
      asm volatile("");
#pragma unroll
      for (int u = 0; u < U; ++u) w[u] = w[u] == 0.f ? k.c : w[u];
    }
  } else if constexpr (KT == MLOD_KERNEL_SINGULAR) {
    if ((__float_as_uint(k.c) & 0x7fffffffu) > 0x0da24260u) {  // as weight32's, for all of them at once
#pragma unroll
      for (int u = 0; u < U; ++u) w[u] = quot(k.cp4, fmaf(d2[u], 0.25f, k.c4));
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) w[u] = k.cp / (d2[u] + k.c);
    }
    if (k.eint > 0) {
      float r[U];
#pragma unroll
      for (int u = 0; u < U; ++u) r[u] = 1.f;
      for (int e = k.eint; e; e >>= 1) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (e & 1) r[u] *= w[u];
          w[u] *= w[u];
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) w[u] = r[u];
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) w[u] = __builtin_amdgcn_exp2f(k.e * __builtin_amdgcn_logf(w[u]));
    }
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u) w[u] = weight32<KT>(k, d2[u]);
  }
}

// The same in FP64.  An approximate reciprocal and two Newton steps; then as above.
__device__ __forceinline__ double quot_rcp(double n, double d, double r) {
  const double q = __dmul_rn(n, r);
  return fma(fma(-d, q, n), r, q);
}
__device__ __forceinline__ double near_rcp(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = fma(fma(-d, r, 1.0), r, r);
  return fma(fma(-d, r, 1.0), r, r);
}
__device__ __forceinline__ double quot(double n, double d) {
  return __builtin_amdgcn_div_fixup(quot_rcp(n, d, near_rcp(d)), d, n);
}
// (Goldschmidt's iteration; arguments here are zero or sums of squares of float differences, no subnormals)
__device__ __forceinline__ double root(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = __dmul_rn(x, y), h = __dmul_rn(0.5, y);
  const double e = fma(-h, g, 0.5);
  g = fma(g, e, g), h = fma(h, e, h);
  g = fma(fma(-g, g, x), h, g);
  g = fma(fma(-g, g, x), h, g);
  return __builtin_amdgcn_class(x, 0x260) ? x : g;  // zero, infinity
}

// 2^y: y = k + f with |f| <= 1/2, 2^f by the Taylor series of exp(f log 2) to the 13th power (remainder
// 4e-18), 0.86 ulp in all, as the library's exp, in 17 instructions against some 40.  y is finite (or NaN); a k out of range underflows in ldexp.
__device__ __forceinline__ double pow2(double y) {
#pragma clang fp contract(off)  // y is a product: f of the fused one is its rounding error, which is huge where y is
  const double t = __builtin_rint(y), f = y - t;
  double p = 1.3691488853904128e-12;
  p = fma(p, f, 2.5678435993488206e-11);
  p = fma(p, f, 4.4455382718708116e-10);
  p = fma(p, f, 7.054911620801123e-09);
  p = fma(p, f, 1.01780860092397e-07);
  p = fma(p, f, 1.321548679014431e-06);
  p = fma(p, f, 1.5252733804059841e-05);
  p = fma(p, f, 0.0001540353039338161);
  p = fma(p, f, 0.0013333558146428443);
  p = fma(p, f, 0.009618129107628477);
  p = fma(p, f, 0.05550410866482158);
  p = fma(p, f, 0.24022650695910072);
  p = fma(p, f, 0.6931471805599453);
  p = fma(p, f, 1.0);
  int k;
  asm("v_cvt_i32_f64 %0, %1" : "=v"(k) : "v"(t));  // (saturates)
  return __builtin_amdgcn_ldexp(p, k);
}

template <int KT>
__device__ __forceinline__ double weight64(const KParams& k, double d2) {
  if constexpr (KT < 0) {
    if (k.type == MLOD_KERNEL_GAUSSIAN_MULTIPLE) return weight64<MLOD_KERNEL_GAUSSIAN_MULTIPLE>(k, d2);
    if (k.type == MLOD_KERNEL_GAUSSIAN) return weight64<MLOD_KERNEL_GAUSSIAN>(k, d2);
    return weight64<MLOD_KERNEL_SINGULAR>(k, d2);
  } else if constexpr (KT == MLOD_KERNEL_GAUSSIAN_MULTIPLE) {
    d2 = d2 > 1e200 ? 1e200 : d2;  // (keeps a NaN; the exponents stay finite for every float sigma)
    double w = 0.0;
    for (int s = 0; s < k.ns; s += 2) {  // two in flight; bd is zero past ns
      const double e0 = pow2(d2 * k.ad[s]), e1 = pow2(d2 * k.ad[s + 1]);
      w = fma(e0, k.bd[s], w);
      w = fma(e1, k.bd[s + 1], w);
    }
    return w == 0.0 ? (double)k.c : w;
  } else if constexpr (KT == MLOD_KERNEL_GAUSSIAN) {
    return pow2((d2 > 1e200 ? 1e200 : d2) * k.ad[0]) + (double)k.c;
  } else {
    // small whole exponents by products: no more rounding than pow's own
    const double den = d2 + (double)k.c;
    if (k.eint >= 1 && k.eint <= 4 && k.c > 1e-15f) {  // (uniform; den^4 is no subnormal)
      const double d22 = den * den;
      return quot(k.cpe, k.eint == 1 ? den : k.eint == 2 ? d22 : k.eint == 3 ? d22 * den : d22 * d22);
    }
    return pow((double)k.cp, (double)k.e) / pow(den, (double)k.e);
  }
}

}  // namespace
}  // namespace mlod
