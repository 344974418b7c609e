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

// A spacing as the resident kernel divides by it.  FP32 multiplies by its inverse anyway; FP64 takes
// the same quotients as dscale, bit for bit, from the spacing's reciprocal: 4 fused operations
// each instead of the 11 of an IEEE division.  With r = RN(1/d) and e = RN((1 - d r) r),
// q = x r + x e is x/d to well under an ulp, so x - q d is exact and q + (x - q d) r rounds to the
// correctly rounded quotient (Markstein, IBM J. Res. Dev. 34, 1990), where nothing under- or
// overflows.
struct Recip {
  double d, r, e;
};
__device__ __forceinline__ void set_spacing(double d, Recip& s) {
  // a spacing of no usual size: every quotient comes out NaN and is taken by an IEEE division
  const bool usual = fabs(d) > 0x1p-60 && fabs(d) < 0x1p60;
  s.d = d;
  s.r = usual ? 1.0 / d : __builtin_nan("");
  s.e = __builtin_fma(-d, s.r, 1.0) * s.r;
}
__device__ __forceinline__ void set_spacing(float inv, float& s) { s = inv; }
__device__ __forceinline__ double quotient(double v, const Recip& s) {
  const double x = v * 0.25;
  const double q = __builtin_fma(x, s.r, x * s.e);
  return __builtin_fma(__builtin_fma(-q, s.d, x), s.r, q);
}
__device__ __forceinline__ float quotient(float v, float inv) { return v * inv; }
// Nonzero difference sums below 2^kTinySum go the long way: x - q d would underflow.  (A zero's
// exponent reads as 0.)  A wave's sums are rarely there but for the front of a pulse, long before
// it can be seen.
constexpr int kTinySum = -890;
__device__ __forceinline__ int least_exponent(const double (&v)[9]) {
  int e = __builtin_amdgcn_frexp_exp(v[0]);
#pragma unroll
  for (int i = 1; i < 9; i++) e = min(e, (int)__builtin_amdgcn_frexp_exp(v[i]));
  return e;
}

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

// The 21 stiffness entries of cell e from the per-cell arrays, AXIAL: nine of them and the row of the
// others.  load(p) reads one value.
template <bool AXIAL, typename T, typename L>
__device__ __forceinline__ void cell_constants(const StressArgs<T>& a, int e, L&& load, T (&cc)[21]) {
  // ldc > 0: [entries][ldc] arrays; ldc == 0: blocks of 64 cells, [n/64][entries][64], so one
  // wavefront's coefficients are a single contiguous run
  constexpr int N = AXIAL ? kAxialEntries : 21;
  const T* p = a.C + (a.ldc ? (int64_t)e : (int64_t)(e >> 6) * (N * 64) + (e & 63));
  const int64_t step = a.ldc ? a.ldc : 64;
#pragma unroll
  for (int j = 0; j < 21; j++) {
    const int q = AXIAL ? axial_entry(j) : j;
    cc[j] = q >= 0 ? load(p + q * step) : as_const(a.crow)[j];
  }
}
template <typename T>
__device__ __forceinline__ void cell_constants(const StressArgs<T>& a, int e, T (&cc)[21]) {
  auto plain = [](const T* p) { return *p; };
  if (a.crow)
    cell_constants<true>(a, e, plain, cc);
  else
    cell_constants<false>(a, e, plain, cc);
}

// Summed moment terms of a special cell, Voigt component k, taken where the update adds them: six
// sums kept for that cost the FP64 stress kernel 45 of 112 registers and three of seven waves per
// SIMD (a million cells 52.2 us a step against 50.2, FP32 31.0 against 30.1).
template <typename T>
__device__ __forceinline__ double cell_moment(const StressArgs<T>& a, int sp, int k) {
  const int* off = a.sp_off + 7 * (size_t)sp;
  double acc = 0.0;
  for (int t = off[k]; t < off[k + 1]; t++) acc += a.amp[a.term[t]];
  return acc;
}

// S += dt*(C : grad V + m) for one cell; cc[j] is the j-th of the 21 stored C (a class-table
// row or the cell's own array), m(k) a special cell's summed moment terms.
template <typename T, typename R, typename M>
__device__ __forceinline__ void voigt_update(T dt, R cc, const T (&d)[6], M&& m, int sp, T (&s)[6]) {
#pragma unroll
  for (int ks = 0; ks < 6; ks++) {
    T acc = cc[tri(ks, 0)] * d[0] + cc[tri(ks, 1)] * d[1] + cc[tri(ks, 2)] * d[2] +
            cc[tri(ks, 3)] * d[3] + cc[tri(ks, 4)] * d[4] + cc[tri(ks, 5)] * d[5];
    if constexpr (sizeof(T) == 8) {
      if (sp >= 0) acc = acc + (T)m(ks);
      s[ks] = s[ks] + dt * acc;  // C is plain C_IJ: S += dt*(C:gradV + m)
    } else {
      if (sp >= 0) acc = acc + (T)((double)dt * m(ks));  // C holds dt*C_IJ
      s[ks] = s[ks] + acc;
    }
  }
}

// The velocity rates of a node before its sources, div S with the reference's order of
// operations.  pair(p, f, g) reads components 2p and 2p + 1 of (Sxx, Sxy, Sxz, Syy, Syz, Szz)
// at the node's 8 cells (0 at a missing one).
template <typename T, typename D>
__device__ __forceinline__ void sum_rates(D&& div, const T (&v)[9], T (&r)[3]) {
  const T dx_sxx = div(v[0], 0), dx_sxy = div(v[1], 0), dx_sxz = div(v[2], 0);
  const T dy_sxy = div(v[3], 1), dy_syy = div(v[4], 1), dy_syz = div(v[5], 1);
  const T dz_sxz = div(v[6], 2), dz_syz = div(v[7], 2), dz_szz = div(v[8], 2);
  r[0] = (dx_sxx + dy_sxy) + dz_sxz;
  r[1] = (dx_sxy + dy_syy) + dz_syz;
  r[2] = (dx_sxz + dy_syz) + dz_szz;
}
template <typename T, typename L>
__device__ __forceinline__ void node_sums(L&& pair, T (&v)[9]) {
  T f[8], g[8];
  pair(0, f, g);
  v[0] = diffsum<0>(f);
  v[1] = diffsum<0>(g);
  v[3] = diffsum<1>(g);
  pair(1, f, g);
  v[2] = diffsum<0>(f);
  v[6] = diffsum<2>(f);
  v[4] = diffsum<1>(g);
  pair(2, f, g);
  v[5] = diffsum<1>(f);
  v[7] = diffsum<2>(f);
  v[8] = diffsum<2>(g);
}
template <typename T, typename L>
__device__ __forceinline__ void node_rates(L&& pair, T sx, T sy, T sz, T (&r)[3]) {
  T v[9];
  node_sums(pair, v);
  sum_rates([&](T x, int ax) { return dscale(x, ax == 0 ? sx : ax == 1 ? sy : sz); }, v, r);
}

// Strain-rate terms of one cell from its 8 vertices: the diagonal D_i V_i and the shear
// sums D_j V_k + D_k V_j, in the reference's order of operations.  xy(f, g) reads Vx and Vy at
// the vertices, z(f) reads Vz.
template <typename T, typename D>
__device__ __forceinline__ void sum_strains(D&& div, const T (&v)[9], T (&d)[6]) {
  // v[3 i + k]: the difference sum of D_i V_k (i: derivative axis, k: velocity component)
  d[0] = div(v[0], 0);
  d[1] = div(v[4], 1);
  d[2] = div(v[8], 2);
  const T d12 = div(v[5], 1), d21 = div(v[7], 2), d02 = div(v[2], 0), d20 = div(v[6], 2);
  const T d01 = div(v[1], 0), d10 = div(v[3], 1);
  d[3] = d12 + d21;
  d[4] = d02 + d20;
  d[5] = d01 + d10;
}
template <typename T, typename LXY, typename LZ>
__device__ __forceinline__ void cell_sums(LXY&& xy, LZ&& z, T (&v)[9]) {
  T f[8], g[8];
  xy(f, g);
  v[0] = diffsum<0>(f);
  v[3] = diffsum<1>(f);
  v[6] = diffsum<2>(f);
  v[1] = diffsum<0>(g);
  v[4] = diffsum<1>(g);
  v[7] = diffsum<2>(g);
  z(f);
  v[2] = diffsum<0>(f);
  v[5] = diffsum<1>(f);
  v[8] = diffsum<2>(f);
}
template <typename T, typename LXY, typename LZ>
__device__ __forceinline__ void strain_rates(LXY&& xy, LZ&& z, T sx, T sy, T sz, T (&d)[6]) {
  T v[9];
  cell_sums(xy, z, v);
  sum_strains([&](T x, int ax) { return dscale(x, ax == 0 ? sx : ax == 1 ? sy : sz); }, v, d);
}

// The same with quotients from reciprocals; what they may not give goes through dscale.
template <typename L>
__device__ __forceinline__ void node_rates(L&& pair, const Recip (&s)[3], double (&r)[3]) {
  double v[9];
  node_sums(pair, v);
  sum_rates([&](double x, int ax) { return quotient(x, s[ax]); }, v, r);
  if (__builtin_isnan((r[0] + r[1]) + r[2]) || least_exponent(v) < kTinySum) {
    asm volatile("" ::: "memory");  // read again rather than held in registers
    node_sums(pair, v);
    sum_rates([&](double x, int ax) { return dscale(x, s[ax].d); }, v, r);
  }
}
template <typename L>
__device__ __forceinline__ void node_rates(L&& pair, const float (&s)[3], float (&r)[3]) {
  node_rates(pair, s[0], s[1], s[2], r);
}
template <typename LXY, typename LZ>
__device__ __forceinline__ void strain_rates(LXY&& xy, LZ&& z, const Recip (&s)[3], double (&d)[6]) {
  double v[9];
  cell_sums(xy, z, v);
  sum_strains([&](double x, int ax) { return quotient(x, s[ax]); }, v, d);
  if (__builtin_isnan(((d[0] + d[1]) + (d[2] + d[3])) + (d[4] + d[5])) || least_exponent(v) < kTinySum) {
    asm volatile("" ::: "memory");
    cell_sums(xy, z, v);
    sum_strains([&](double x, int ax) { return dscale(x, s[ax].d); }, v, d);
  }
}
template <typename LXY, typename LZ>
__device__ __forceinline__ void strain_rates(LXY&& xy, LZ&& z, const float (&s)[3], float (&d)[6]) {
  strain_rates(xy, z, s[0], s[1], s[2], d);
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
