// weights.h — the weight kernels on the device, shared by the projection and neighbour kernels.
#pragma once

#include "mlod_internal.h"

namespace mlod {
namespace {

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
    // exponentials are in flight.  Coefficients past ns are zero: a term past the last adds 0 * 1
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
    const float base = k.cp / (d2 + k.c);
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
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u) w[u] = weight32<KT>(k, d2[u]);
  }
}

template <int KT>
__device__ __forceinline__ double weight64(const KParams& k, double d2) {
  if constexpr (KT < 0) {
    if (k.type == MLOD_KERNEL_GAUSSIAN_MULTIPLE) return weight64<MLOD_KERNEL_GAUSSIAN_MULTIPLE>(k, d2);
    if (k.type == MLOD_KERNEL_GAUSSIAN) return weight64<MLOD_KERNEL_GAUSSIAN>(k, d2);
    return weight64<MLOD_KERNEL_SINGULAR>(k, d2);
  } else if constexpr (KT == MLOD_KERNEL_GAUSSIAN_MULTIPLE) {
    double w = 0.0;
    for (int s = 0; s < k.ns; ++s) w += exp(d2 * k.ad[s]) * k.bd[s];
    return w == 0.0 ? (double)k.c : w;
  } else if constexpr (KT == MLOD_KERNEL_GAUSSIAN) {
    return exp(d2 * k.ad[0]) + (double)k.c;
  } else {
    return pow((double)k.cp, (double)k.e) / pow(d2 + (double)k.c, (double)k.e);
  }
}

}  // namespace
}  // namespace mlod
