// rsg_device.h -- device helpers shared by the per-step kernels (rsg_kernels.hip) and the
// resident multi-step kernel (rsg_resident.hip): the differences of the scheme, the Voigt
// update and the class-table reads.  The order of the floating-point operations here is the
// reference's; both kernels get bit-identical results because they share it.
#pragma once

#include <hip/hip_runtime.h>

#include "rsg_internal.h"

namespace rsg {
namespace {

__device__ __forceinline__ bool is_boxed(double v) { return __builtin_isnan(v); }
__device__ __forceinline__ bool is_boxed(float v) { return __builtin_isnan(v); }
__device__ __forceinline__ int unbox(double v) {
  return (int)(uint32_t)(__double_as_longlong(v) & 0xFFFFFFFFll);
}
__device__ __forceinline__ int unbox(float v) { return (int)(__float_as_uint(v) & 0x3FFFFFu); }

// RightHex slot patterns: forward and backward vertices (or cell slots) per axis.
//   x: fwd {1,2,5,6} bwd {0,3,4,7};  y: fwd {2,3,6,7} bwd {0,1,4,5};
//   z: fwd {4,5,6,7} bwd {0,1,2,3}
template <int AX>
__device__ __forceinline__ double diffsum(const double (&f)[8]) {
  double v = 0.0;
  if (AX == 0) {
    v += (f[1] - f[0]); v += (f[2] - f[3]); v += (f[5] - f[4]); v += (f[6] - f[7]);
  } else if (AX == 1) {
    v += (f[2] - f[0]); v += (f[3] - f[1]); v += (f[6] - f[4]); v += (f[7] - f[5]);
  } else {
    v += (f[4] - f[0]); v += (f[5] - f[1]); v += (f[6] - f[2]); v += (f[7] - f[3]);
  }
  return v;
}
template <int AX>
__device__ __forceinline__ float diffsum(const float (&f)[8]) {
  float v;
  if (AX == 0) {
    v = ((f[1] - f[0]) + (f[2] - f[3])) + ((f[5] - f[4]) + (f[6] - f[7]));
  } else if (AX == 1) {
    v = ((f[2] - f[0]) + (f[3] - f[1])) + ((f[6] - f[4]) + (f[7] - f[5]));
  } else {
    v = ((f[4] - f[0]) + (f[5] - f[1])) + ((f[6] - f[2]) + (f[7] - f[3]));
  }
  return v;
}
// Derivative from a difference sum: FP64 (value*0.25)/spacing, FP32 value*(0.25/spacing).
__device__ __forceinline__ double dscale(double v, double sp) { return v * 0.25 / sp; }
__device__ __forceinline__ float dscale(float v, float inv) { return v * inv; }

typedef double d2v __attribute__((ext_vector_type(2)));
typedef float f4v __attribute__((ext_vector_type(4)));

// One material row (16-byte aligned) as 16-byte loads through the caches: lanes of a
// wavefront that share a material read the same addresses, which coalesce.
template <int W>
__device__ __forceinline__ void load_row(const double* __restrict__ p, double (&out)[W]) {
  static_assert(W % 2 == 0, "row width");
  const d2v* q = reinterpret_cast<const d2v*>(p);
#pragma unroll
  for (int i = 0; i < W / 2; i++) {
    const d2v v = q[i];
    out[2 * i] = v.x;
    out[2 * i + 1] = v.y;
  }
}
template <int W>
__device__ __forceinline__ void load_row(const float* __restrict__ p, float (&out)[W]) {
  static_assert(W % 4 == 0, "row width");
  const f4v* q = reinterpret_cast<const f4v*>(p);
#pragma unroll
  for (int i = 0; i < W / 4; i++) {
    const f4v v = q[i];
    out[4 * i] = v.x;
    out[4 * i + 1] = v.y;
    out[4 * i + 2] = v.z;
    out[4 * i + 3] = v.w;
  }
}

// Material/spacing key of an entity, and its special index (or -1).
template <typename A>
__device__ __forceinline__ uint32_t resolve_key(const A& a, uint32_t key, int& sp) {
  if (key & kSpecialKey) {
    sp = (int)(key & ~kSpecialKey);
    return a.sp_key[sp];
  }
  sp = -1;
  return key;
}
template <typename P, typename T>
__device__ __forceinline__ void axis_spacings(P axis, uint32_t k, T& sx, T& sy, T& sz) {
  sx = axis[(k >> 14) & (kAxisClasses - 1)];
  sy = axis[kAxisClasses + ((k >> 7) & (kAxisClasses - 1))];
  sz = axis[2 * kAxisClasses + (k & (kAxisClasses - 1))];
}

// The class tables are written only by the host, so a wavefront-uniform read of them may go
// through the scalar cache: a pointer in the constant address space lets the compiler use
// scalar loads (reads only; nothing is ever stored through this path).
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T* as_const(const T* p) {
  return (const __attribute__((address_space(4))) T*)p;
}

// Index of C_(I,J) (0-based Voigt indices) in the 21-entry upper triangle.
__host__ __device__ constexpr int tri(int i, int j) {
  return (i <= j) ? (i * 6 - i * (i - 1) / 2 + (j - i)) : (j * 6 - j * (j - 1) / 2 + (i - j));
}

// Summed moment terms of a special cell, per Voigt component.
template <typename T>
__device__ __forceinline__ void cell_moments(const StressArgs<T>& a, int sp, double (&m)[6]) {
#pragma unroll
  for (int k = 0; k < 6; k++) m[k] = 0.0;
  if (sp < 0) return;
  const int* off = a.sp_off + 7 * (size_t)sp;
#pragma unroll
  for (int k = 0; k < 6; k++) {
    double acc = 0.0;
    for (int t = off[k]; t < off[k + 1]; t++) acc += a.amp[a.term[t]];
    m[k] = acc;
  }
}

// S += dt*(C : grad V + m) for one cell; cc[j] is the j-th of the 21 stored C (a class-table
// row or the cell's own array).
template <typename T, typename R>
__device__ __forceinline__ void voigt_update(T dt, R cc, const T (&d)[6], const double (&m)[6], int sp,
                                             T (&s)[6]) {
#pragma unroll
  for (int ks = 0; ks < 6; ks++) {
    T acc = cc[tri(ks, 0)] * d[0] + cc[tri(ks, 1)] * d[1] + cc[tri(ks, 2)] * d[2] +
            cc[tri(ks, 3)] * d[3] + cc[tri(ks, 4)] * d[4] + cc[tri(ks, 5)] * d[5];
    if constexpr (sizeof(T) == 8) {
      if (sp >= 0) acc = acc + (T)m[ks];
      s[ks] = s[ks] + dt * acc;  // C is plain C_IJ: S += dt*(C:gradV + m)
    } else {
      if (sp >= 0) acc = acc + (T)((double)dt * m[ks]);  // C holds dt*C_IJ
      s[ks] = s[ks] + acc;
    }
  }
}

// The velocity rates of a node before its sources, div S with the reference's order of
// operations.  pair(p, f, g) reads components 2p and 2p + 1 of (Sxx, Sxy, Sxz, Syy, Syz, Szz)
// at the node's 8 cells (0 at a missing one).
template <typename T, typename L>
__device__ __forceinline__ void node_rates(L&& pair, T sx, T sy, T sz, T (&r)[3]) {
  T f[8], g[8];
  pair(0, f, g);
  const T dx_sxx = dscale(diffsum<0>(f), sx);
  const T dx_sxy = dscale(diffsum<0>(g), sx);
  const T dy_sxy = dscale(diffsum<1>(g), sy);
  pair(1, f, g);
  const T dx_sxz = dscale(diffsum<0>(f), sx);
  const T dz_sxz = dscale(diffsum<2>(f), sz);
  const T dy_syy = dscale(diffsum<1>(g), sy);
  pair(2, f, g);
  const T dy_syz = dscale(diffsum<1>(f), sy);
  const T dz_syz = dscale(diffsum<2>(f), sz);
  const T dz_szz = dscale(diffsum<2>(g), sz);
  r[0] = (dx_sxx + dy_sxy) + dz_sxz;
  r[1] = (dx_sxy + dy_syy) + dz_syz;
  r[2] = (dx_sxz + dy_syz) + dz_szz;
}

// Strain-rate terms of one cell from its 8 vertices: the diagonal D_i V_i and the shear
// sums D_j V_k + D_k V_j, in the reference's order of operations.  xy(f, g) reads Vx and Vy at
// the vertices, z(f) reads Vz.
template <typename T, typename LXY, typename LZ>
__device__ __forceinline__ void strain_rates(LXY&& xy, LZ&& z, T sx, T sy, T sz, T (&d)[6]) {
  // dik = D_i V_k (i: derivative axis, k: velocity component)
  T f[8], g[8];
  xy(f, g);
  const T d00 = dscale(diffsum<0>(f), sx);
  const T d10 = dscale(diffsum<1>(f), sy);
  const T d20 = dscale(diffsum<2>(f), sz);
  const T d01 = dscale(diffsum<0>(g), sx);
  const T d11 = dscale(diffsum<1>(g), sy);
  const T d21 = dscale(diffsum<2>(g), sz);
  z(f);
  const T d02 = dscale(diffsum<0>(f), sx);
  const T d12 = dscale(diffsum<1>(f), sy);
  const T d22 = dscale(diffsum<2>(f), sz);
  d[0] = d00;
  d[1] = d11;
  d[2] = d22;
  d[3] = d12 + d21;
  d[4] = d02 + d20;
  d[5] = d01 + d10;
}

// Summed force terms of a special node, added to its rates.
template <typename T>
__device__ __forceinline__ void add_node_forces(const VelocityArgs<T>& a, int sp, T (&r)[3]) {
  const int* off = a.sp_off + 4 * (size_t)sp;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    double acc = 0.0;
    for (int t = off[d]; t < off[d + 1]; t++) acc += a.amp[a.term[t]];
    r[d] = r[d] + (T)acc;
  }
}

}  // namespace
}  // namespace rsg
