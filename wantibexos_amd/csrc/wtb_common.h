// Shared device/host helpers for the gfx950 BSE kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <string>
#include <type_traits>

// ---------------------------------------------------------------------------
// complex double with value semantics (interleaved re,im as in Fortran COMPLEX*16)
// ---------------------------------------------------------------------------
struct __attribute__((aligned(16))) zc {
  double re, im;
};

__host__ __device__ inline zc mkz(double r, double i) { zc z; z.re = r; z.im = i; return z; }
__host__ __device__ inline zc operator+(zc a, zc b) { return mkz(a.re + b.re, a.im + b.im); }
__host__ __device__ inline zc operator-(zc a, zc b) { return mkz(a.re - b.re, a.im - b.im); }
__host__ __device__ inline zc operator-(zc a) { return mkz(-a.re, -a.im); }
// (a.re*b.re - a.im*b.im) + i(a.re*b.im + a.im*b.re): the Fortran complex product
__host__ __device__ inline zc operator*(zc a, zc b) {
  return mkz(a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re);
}
__host__ __device__ inline zc operator*(double s, zc a) { return mkz(s * a.re, s * a.im); }
__host__ __device__ inline zc operator*(zc a, double s) { return mkz(a.re * s, a.im * s); }
__host__ __device__ inline zc conj(zc a) { return mkz(a.re, -a.im); }
__host__ __device__ inline double norm2(zc a) { return a.re * a.re + a.im * a.im; }
__host__ __device__ inline zc& operator+=(zc& a, zc b) { a.re += b.re; a.im += b.im; return a; }
__host__ __device__ inline zc& operator-=(zc& a, zc b) { a.re -= b.re; a.im -= b.im; return a; }
// complex float storage (COMPLEX*8) for the precision form; arithmetic stays in zc
struct __attribute__((aligned(8))) zf {
  float re, im;
};
__host__ __device__ inline zc ldz(const zc& v) { return v; }
__host__ __device__ inline zc ldz(const zf& v) { return mkz((double)v.re, (double)v.im); }
__host__ __device__ inline void stz(zc& d, zc v) { d = v; }
__host__ __device__ inline void stz(zf& d, zc v) {
  d.re = (float)v.re;
  d.im = (float)v.im;
}

// conj(a)*b accumulated with fused multiply-adds
__device__ inline zc fma_conj(zc a, zc b, zc acc) {
  acc.re = fma(a.re, b.re, fma(a.im, b.im, acc.re));
  acc.im = fma(a.re, b.im, fma(-a.im, b.re, acc.im));
  return acc;
}
__device__ inline zc fma_z(zc a, zc b, zc acc) {
  acc.re = fma(a.re, b.re, fma(-a.im, b.im, acc.re));
  acc.im = fma(a.re, b.im, fma(a.im, b.re, acc.im));
  return acc;
}

// x of another lane by a DPP lane permutation (within rows of 16 lanes); both halves of the
// double move
template <int CTRL>
__device__ inline double dpp_d(double x) {
  const long long v = __builtin_bit_cast(long long, x);
  const int lo = __builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(v >> 32), CTRL, 0xF, 0xF, false);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (long long)(unsigned)lo);
}
template <int CTRL>
__device__ inline zc dpp_z(zc v) { return mkz(dpp_d<CTRL>(v.re), dpp_d<CTRL>(v.im)); }

// Lane halves and 16-lane rows by the swap instructions (VALU, no LDS round trip): after
// swap32(a, b) lane l < 32 holds a(l) and a(l + 32), lane l >= 32 b(l - 32) and b(l); swap16
// does the same within each pair of 16-lane rows.  a + b is then a sum over that lane bit,
// of a in the lanes where the bit is clear and of b where it is set.
__device__ inline void swap32(double& a, double& b) {
  const unsigned long long x = __builtin_bit_cast(unsigned long long, a), y = __builtin_bit_cast(unsigned long long, b);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  a = __builtin_bit_cast(double, ((unsigned long long)hi[0] << 32) | lo[0]);
  b = __builtin_bit_cast(double, ((unsigned long long)hi[1] << 32) | lo[1]);
}
__device__ inline void swap16(double& a, double& b) {
  const unsigned long long x = __builtin_bit_cast(unsigned long long, a), y = __builtin_bit_cast(unsigned long long, b);
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  a = __builtin_bit_cast(double, ((unsigned long long)hi[0] << 32) | lo[0]);
  b = __builtin_bit_cast(double, ((unsigned long long)hi[1] << 32) | lo[1]);
}
__device__ inline double add32(double a, double b) {
  swap32(a, b);
  return a + b;
}
__device__ inline double add16(double a, double b) {
  swap16(a, b);
  return a + b;
}
__device__ inline float add32(float a, float b) {
  const auto v = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  const unsigned x = v[0], y = v[1];           // (bit_cast of a vector's element reads element 0)
  return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}
__device__ inline float add16(float a, float b) {
  const auto v = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  const unsigned x = v[0], y = v[1];
  return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}

// sum of p[b * stride] over b = b0, b0 + step, ... < b1, added in that order, with the loads
// issued eight at a time (a plain loop waits for each load before the next).  The last
// group loads from clamped indices (b1 - 1 is in range whenever the group runs) and adds
// only the terms below b1, so short sums keep their loads in flight too.
template <class V>
__device__ inline V strided_sum(const V* __restrict__ p, size_t stride, int b0, int b1, int step, V acc) {
  int b = b0;
  for (; b + 7 * step < b1; b += 8 * step) {
    V v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p[(size_t)(b + u * step) * stride];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc += v[u];
  }
  if (b < b1) {
    V v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int bu = b + u * step;
      v[u] = p[(size_t)(bu < b1 ? bu : b1 - 1) * stride];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (b + u * step < b1) acc += v[u];
  }
  return acc;
}

// ---------------------------------------------------------------------------
// MFMA lane layouts on gfx950 (measured with a lane probe):
//   v_mfma_f64_16x16x4_f64: lane l holds A[l%16][l/16] and B[l/16][l%16];
//     accumulator register r of lane l is D[(l/16) + 4*r][l%16].
//   v_mfma_f32_16x16x4_f32: same A and B; register r is D[4*(l/16) + r][l%16].
// ---------------------------------------------------------------------------
typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

__device__ inline d4 mfma16x16x4(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ inline f4 mfma16x16x4f32(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// host error plumbing
// ---------------------------------------------------------------------------
namespace wtb {
void set_error(const std::string& msg);
}

#define WTB_HIP(call)                                                        \
  do {                                                                       \
    hipError_t _e = (call);                                                  \
    if (_e != hipSuccess) {                                                  \
      wtb::set_error(std::string(#call) + ": " + hipGetErrorString(_e));     \
      return WTB_ERR_HIP;                                                    \
    }                                                                        \
  } while (0)

#define WTB_LAUNCH_CHECK()                                                   \
  do {                                                                       \
    hipError_t _e = hipGetLastError();                                       \
    if (_e != hipSuccess) {                                                  \
      wtb::set_error(std::string("kernel launch: ") + hipGetErrorString(_e)); \
      return WTB_ERR_HIP;                                                    \
    }                                                                        \
  } while (0)
