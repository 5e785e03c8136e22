// Stage (d1) in two stages: a Hermitian matrix (lower triangle, column-major, ld) is
// reduced first to a lower band of width b (dense -> band, blocked Householder on panels
// of b columns with MFMA two-sided updates), then to a real symmetric tridiagonal (band ->
// tridiagonal by bulge chasing), applying the conjugate transpose of every orthogonal
// factor to a few tracked vectors, so that X^T h = Z^T Q2^T Q1^T h needs no eigenvectors.
// The arithmetic is that of LAPACK's ZHETRD_HE2HB (ZGEQRF panels with ZLARFG reflectors,
// ZLARFT compact WY factor, the ZHER2K-form two-sided update) and ZHETRD_HB2ST (the
// bulge-chasing sweeps); the organisation into kernels is this file's own.
//
// Stage 1, panel p (columns c0 = p b .. c0 + b - 1, trailing rows r0 = c0 + b .. N - 1):
//   k_pqr_col(c), c = 0..k     one launch per column: finish reflector c - 1 from the
//                              previous launch's partial sums (every workgroup, in a fixed
//                              order), apply it to the panel columns right of it, and form
//                              the partial sums of column c (|x|^2 and x^H P(:, j))
//   k_pfin                     explicit V (unit diagonal) and R back into the matrix
//   k_gram, k_gram_sum         G = V^H V, t1 = V^H g (FP64 MFMA on row chunks, partials summed in order)
//   k_pT                       T (ZLARFT forward/columnwise) and t2 = T^H t1
//   k_pY                       Y = V T, g -= V t2 (rows of the panel)
//   k_hmm_b, k_hmm_sum         X = A22 Y (MFMA, full Hermitian storage, K slices)
//   k_gram, k_gram_sum         M = V^H X
//   k_pW                       W = X - 1/2 V (T^H M)
//   k_her2k_full               A22 -= V W^H + W V^H (MFMA, the tiles on and below the diagonal)
// COMPLEX*16 with b = 16 (band_panel_fits) has its own form of the same steps:
//   k_strip                    the panel's columns take the update of the panel before
//   k_qr_panel                 reflectors, T, Y = V T and the tracked vectors, in one launch
//   k_update_mul, k_um_sum     A22 takes the update of the panel before; X = A22 Y in that pass
//   k_qr_w                     W = X - 1/2 V (T^H (V^H X))
// The tracked vectors are carried conjugated (gc = conj(g)): Q^H gc = conj(Q^T g).
//
// Stage 2 (bulge chasing, FP64, band storage BD[c][d] = A(c + d, c), d <= 2b): sweep s
// annihilates column s below its subdiagonal; its tasks k = 0, 1, ... each apply one
// reflector (ZLARFG) two-sidedly to a diagonal block and the previous one from the right
// to the block below it (creating the bulge whose first column the next reflector
// annihilates).  One persistent kernel (k_chase) whose workgroups claim groups of sweeps in
// order from a counter; task k of sweep s waits until sweep s - 1 has finished its tasks
// 0..k+1 (its later tasks touch only rows below this task's), signalled through counters in
// LDS inside a group and through a progress counter in memory between groups (device-scope
// accesses, no cache maintenance).  Every wait is bounded, in memory and in LDS alike: past
// the limit the kernel sets an error flag that every waiting workgroup sees, all of them
// return, and what follows gets a zero tridiagonal and the status word.
#include "wtb_kernels.h"
#include <algorithm>
#include <atomic>

namespace wtb {

#define PR 256          // panel rows per workgroup (one per thread)
#define BMAX 32         // largest band width

// ---------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------
__device__ inline zc zdiv(zc a, zc b) {
  // a / b with the scaling of Smith's algorithm, both cases formed and one selected
  const bool re_big = fabs(b.re) >= fabs(b.im);
  const double p = re_big ? b.re : b.im, q = re_big ? b.im : b.re;
  const double r = q / p, den = p + q * r;
  const double xr = re_big ? a.re + a.im * r : a.re * r + a.im;
  const double xi = re_big ? a.im - a.re * r : a.im * r - a.re;
  return mkz(xr / den, xi / den);
}

// any NaN by its usual bits (the panels' exchange gives those of all ones a meaning)
__device__ inline zc clean_nan(zc v) {
  return mkz(v.re != v.re ? __builtin_nan("") : v.re, v.im != v.im ? __builtin_nan("") : v.im);
}

__device__ inline zc shfl_xor_z(zc v, int off) { return mkz(__shfl_xor(v.re, off), __shfl_xor(v.im, off)); }

// lane ^ 16 within 32 lanes, by a swizzle
__device__ inline double swz16_d(double x) {
  const long long v = __builtin_bit_cast(long long, x);
  const int lo = __builtin_amdgcn_ds_swizzle((int)v, 0x401F);
  const int hi = __builtin_amdgcn_ds_swizzle((int)(v >> 32), 0x401F);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (long long)(unsigned)lo);
}

// The value of the partner lane that differs from this one in lane bit OFF and agrees in
// the bits above it: ^1 and ^2 by quad permutations, i <-> 7 - i (row half mirror) for 4,
// a rotation by 8 in a row of 16 for 8, a swizzle for 16, a permute for 32.  Partners are
// mutual, so sums formed with them are the same in both lanes.
template <int OFF>
__device__ inline double xchg(double x) {
  if constexpr (OFF == 1) return dpp_d<0xB1>(x);
  else if constexpr (OFF == 2) return dpp_d<0x4E>(x);
  else if constexpr (OFF == 4) return dpp_d<0x141>(x);
  else if constexpr (OFF == 8) return dpp_d<0x128>(x);
  else if constexpr (OFF == 16) return swz16_d(x);
  else return __shfl_xor(x, 32);
}
template <int OFF>
__device__ inline zc xchg(zc v) { return mkz(xchg<OFF>(v.re), xchg<OFF>(v.im)); }

// Data handed between workgroups of one kernel (the panel's partial sums, the chase's band
// and tracked vectors) moves through device-scope (sc1) loads and stores, which the
// hardware keeps coherent across the XCDs' L2 caches; the writer's stores are complete
// (s_waitcnt) before its counter moves, so the hand-off needs no L2 write-back or
// invalidate.
__device__ inline zc ld_dev(const zc* p) {
  const double* q = reinterpret_cast<const double*>(p);
  return mkz(__hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
             __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ inline void st_dev(zc* p, zc v) {
  double* q = reinterpret_cast<double*>(p);
  __hip_atomic_store(q, v.re, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(q + 1, v.im, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// sum of p[b * stride] over b = b0, b0 + step, ... < b1 in that order, device-scope loads
// issued eight at a time
__device__ inline zc strided_sum_dev(const zc* p, size_t stride, int b0, int b1, int step) {
  zc acc = mkz(0, 0);
  for (int b = b0; b < b1; b += 8 * step) {
    zc v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int bu = b + u * step;
      v[u] = bu < b1 ? ld_dev(p + (size_t)bu * stride) : mkz(0, 0);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (b + u * step < b1) acc += v[u];
  }
  return acc;
}

// ZLARFG on (alpha, x) with |x|^2 = xn2: beta (real, returned as the new alpha), tau and
// the scale 1/(alpha - beta) of x.  tau = 0 (H = I) when x = 0 and alpha is real.
__device__ inline void larfg(zc alpha, double xn2, zc& beta, zc& tau, zc& scale) {
  const bool ident = xn2 == 0.0 && alpha.im == 0.0;
  const double nrm = sqrt(alpha.re * alpha.re + alpha.im * alpha.im + xn2);
  const double b = ident ? 1.0 : (alpha.re >= 0.0 ? -nrm : nrm);      // 1: any nonzero stand-in
  const zc t = mkz((b - alpha.re) / b, -alpha.im / b);
  const zc sc = zdiv(mkz(1, 0), mkz(alpha.re - b, alpha.im));
  beta = ident ? alpha : mkz(b, 0.0);
  tau = ident ? mkz(0, 0) : t;
  scale = ident ? mkz(0, 0) : sc;
}

// Sums over the 256 threads of a workgroup of one real value x0 and NB complex values
// v[0..NB) (NB a power of two <= 32).  Within a wave the NB sums are formed by a butterfly
// that halves the set each lane keeps (NB - 1 exchanges instead of 6 NB), after which lane
// l holds the wave's sum of value (l >> (6 - log2 NB)) & (NB - 1); the four waves are then
// added in index order.  Results: red[4 * (NB + 1) + q] (q = 0: x0, 1 + j: v[j]).
// one halving step of the butterfly: lanes with the OFF bit set keep values [n, 2n)
template <int OFF, int n, int NB>
__device__ inline void bf_step(zc (&v)[NB], int lane) {
  const bool up = (lane & OFF) != 0;
#pragma unroll
  for (int q = 0; q < n; ++q) {
    const zc recv = xchg<OFF>(up ? v[q] : v[q + n]);
    v[q] = (up ? v[q + n] : v[q]) + recv;
  }
}

template <int NB>
__device__ inline void block_sum_bf(double x0, zc (&v)[NB], zc* red /* [5][NB + 1] in LDS */) {
  static_assert(NB == 16 || NB == 32, "butterfly for 16 or 32 values");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  zc r;
  if constexpr (NB == 32) {
    bf_step<32, 16>(v, lane);
    bf_step<16, 8>(v, lane);
    bf_step<8, 4>(v, lane);
    bf_step<4, 2>(v, lane);
    bf_step<2, 1>(v, lane);
    r = v[0] + xchg<1>(v[0]);
  } else {
    bf_step<32, 8>(v, lane);
    bf_step<16, 4>(v, lane);
    bf_step<8, 2>(v, lane);
    bf_step<4, 1>(v, lane);
    r = v[0] + xchg<2>(v[0]);
    r += xchg<1>(r);
  }
  x0 += xchg<1>(x0);
  x0 += xchg<2>(x0);
  x0 += xchg<4>(x0);
  x0 += xchg<8>(x0);
  x0 += xchg<16>(x0);
  x0 += xchg<32>(x0);
  constexpr int SH = (NB == 32) ? 1 : 2;
  if ((lane & ((1 << SH) - 1)) == 0) red[wave * (NB + 1) + 1 + ((lane >> SH) & (NB - 1))] = r;
  if (lane == 0) red[wave * (NB + 1)] = mkz(x0, 0.0);
  __syncthreads();
  if ((int)threadIdx.x < NB + 1) {
    const int q = threadIdx.x;
    red[4 * (NB + 1) + q] = ((red[q] + red[(NB + 1) + q]) + red[2 * (NB + 1) + q]) + red[3 * (NB + 1) + q];
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// stage 1: panel QR, one launch per column
// ---------------------------------------------------------------------------
template <class T>
struct PanelArgs {
  T* A;            // the matrix (full storage), ld
  int ld, N, b;
  int c0, r0, m, k;     // panel columns c0..c0+b-1, rows r0..N-1 (m of them), k reflectors
  zc* Pw;          // panel working copy [b][N] (row i of the panel at Pw[i + N*j])
  zc* part;        // [2][nwg][BMAX + 1] partial sums (column c: slot c & 1)
  zc* rowc;        // [2][BMAX] row c of the panel before reflector c
  zc* tau;         // [BMAX]
  int nwg;
};

template <class T, int B>
__global__ __launch_bounds__(PR) void k_pqr_col(PanelArgs<T> a, int c) {
  __shared__ zc red[5 * (B + 1)];
  __shared__ zc sh[B + 4];
  __shared__ zc shs[256 / (B + 1)][B + 1];
  const int i = blockIdx.x * PR + threadIdx.x;       // panel row
  const bool live = i < a.m;
  const size_t N = a.N;
  zc row[B];
#pragma unroll
  for (int j = 0; j < B; ++j) row[j] = mkz(0, 0);
  if (live) {
    if (c == 0) {
#pragma unroll
      for (int j = 0; j < B; ++j)
        if (j < a.b) row[j] = ldz(a.A[(size_t)(a.r0 + i) + (size_t)a.ld * (a.c0 + j)]);
    } else {
#pragma unroll
      for (int j = 0; j < B; ++j)
        if (j >= c - 1 && j < a.b) row[j] = a.Pw[i + N * j];
    }
  }
  if (c > 0) {
    // finish reflector c - 1 from the partial sums of the previous launch
    const int cp = c - 1;
    const zc* pp = a.part + (size_t)(cp & 1) * a.nwg * (BMAX + 1);
    // sh[0].re = |x|^2 below the diagonal, sh[1 + j] = x^H P(:, j): the workgroups' partial
    // sums, NS threads per value each adding every NS-th partial (eight loads in flight),
    // then the NS sub-sums in order
    constexpr int NS = 256 / (B + 1);
    if ((int)threadIdx.x < NS * (B + 1)) {
      const int q = threadIdx.x % (B + 1), sub = threadIdx.x / (B + 1);
      shs[sub][q] = strided_sum(pp + q, BMAX + 1, sub, a.nwg, NS, mkz(0, 0));
    }
    __syncthreads();
    if ((int)threadIdx.x < B + 1) {
      zc t = shs[0][threadIdx.x];
      for (int u = 1; u < NS; ++u) t += shs[u][threadIdx.x];
      sh[threadIdx.x] = t;
    }
    __syncthreads();
    const zc* rc = a.rowc + (cp & 1) * BMAX;
    const zc alpha = rc[cp];
    zc beta, tau, scale;
    larfg(alpha, sh[0].re, beta, tau, scale);
    const zc ctau = conj(tau);
    // v_i = 1 (i == cp), x_i scale (i > cp), 0 above
    zc xcp = mkz(0, 0);                // row[cp] without a runtime index into the array
#pragma unroll
    for (int j = 0; j < B; ++j)
      if (j == cp) xcp = row[j];
    zc vi = mkz(0, 0);
    if (live && i == cp) vi = mkz(1, 0);
    if (live && i > cp) vi = xcp * scale;
    // w_j = v^H P(:, j) = P(cp, j) + conj(scale) (x^H P(:, j) - conj(alpha) P(cp, j))
    const zc cs = conj(scale);
#pragma unroll
    for (int j = 0; j < B; ++j) {
      if (j > cp && j < a.b) {
        const zc pj = rc[j];
        const zc wj = pj + cs * (sh[1 + j] - conj(alpha) * pj);
        if (live && i >= cp) row[j] -= (ctau * vi) * wj;
      }
    }
#pragma unroll
    for (int j = 0; j < B; ++j)
      if (j == cp && live && i >= cp) row[j] = (i == cp) ? beta : vi;
    if (blockIdx.x == 0 && threadIdx.x == 0) a.tau[cp] = tau;
    __syncthreads();
  }
  if (c < a.k) {
    // partial sums of column c over this workgroup's rows
    zc v[B];
    double x0 = 0.0;
#pragma unroll
    for (int q = 0; q < B; ++q) v[q] = mkz(0, 0);
    if (live && i >= c) {
      zc x = mkz(0, 0);
#pragma unroll
      for (int j = 0; j < B; ++j)
        if (j == c) x = row[j];
      if (i > c) x0 = norm2(x);
#pragma unroll
      for (int j = 0; j < B; ++j)
        if (j > c && j < a.b) v[j] = fma_conj(x, row[j], mkz(0, 0));
    }
    block_sum_bf<B>(x0, v, red);
    if ((int)threadIdx.x < B + 1) {
      zc* pp = a.part + (size_t)(c & 1) * a.nwg * (BMAX + 1) + (size_t)blockIdx.x * (BMAX + 1);
      pp[threadIdx.x] = red[4 * (B + 1) + threadIdx.x];
    }
    if (live && i == c) {
      zc* rc = a.rowc + (c & 1) * BMAX;
#pragma unroll
      for (int j = 0; j < B; ++j)
        if (j >= c && j < a.b) rc[j] = row[j];
    }
  }
  if (live) {
#pragma unroll
    for (int j = 0; j < B; ++j)
      if ((c == 0 || j >= c - 1) && j < a.b) a.Pw[i + N * j] = row[j];
  }
}

// explicit V (unit lower trapezoidal, zero above) and R = upper triangle of the panel back
// into the matrix
template <class T, int B>
__global__ __launch_bounds__(PR) void k_pfin(PanelArgs<T> a, zc* __restrict__ V) {
  const int i = blockIdx.x * PR + threadIdx.x;
  if (i >= a.m) return;
  const size_t N = a.N;
#pragma unroll
  for (int j = 0; j < B; ++j) {
    if (j >= a.b) continue;
    const zc p = a.Pw[i + N * j];
    if (i <= j) stz(a.A[(size_t)(a.r0 + i) + (size_t)a.ld * (a.c0 + j)], p);    // R
    zc x = mkz(0, 0);
    if (j < a.k) x = i == j ? mkz(1, 0) : (i > j ? p : mkz(0, 0));
    V[i + N * j] = x;
  }
}

// The panel in one launch: workgroup w keeps rows 256w .. 256w + 255 of the panel in
// registers through all of its k reflectors, and the workgroups meet once per column at a
// counter (bar[c]: the workgroups that have published their partial sums of column c),
// so the arithmetic is k_pqr_col's without the per-column launches and panel round trips.
// Every workgroup must be resident at once: the host launches it only with at most one
// workgroup per compute unit and no other kernel sharing the device, and every wait is
// bounded (err[0] set past the limit, after which every workgroup returns).  At the end
// the panel goes out as V (unit lower trapezoidal) and R (k_pfin's job).
template <class T, int B>
__global__ __launch_bounds__(PR) void k_panel(PanelArgs<T> a, zc* __restrict__ V, int* __restrict__ bar,
                                              int* __restrict__ err, long long spin_limit) {
  constexpr int NS = 256 / (B + 1);
  __shared__ zc red[5 * 17], red2[5 * 17];
  __shared__ zc sh[B + 4];
  __shared__ zc shs[NS][B + 1];
  __shared__ zc rcs[B];
  __shared__ int flag;
  const int i = blockIdx.x * PR + threadIdx.x;       // panel row
  const bool live = i < a.m;
  const size_t N = a.N;
  zc row[B];
#pragma unroll
  for (int j = 0; j < B; ++j)
    row[j] = (live && j < a.b) ? ldz(a.A[(size_t)(a.r0 + i) + (size_t)a.ld * (a.c0 + j)]) : mkz(0, 0);
  for (int c = 0; c <= a.k; ++c) {
    if (c > 0) {
      const int cp = c - 1;
      // every workgroup's partial sums of column cp are out
      if (threadIdx.x == 0) {
        long long n = 0;
        int bad = 0;
        while (__hip_atomic_load(bar + cp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < a.nwg) {
          if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 || ++n > spin_limit) {
            bad = 1;
            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
        flag = bad;
      }
      __syncthreads();
      if (flag) return;
      // sh[0].re = |x|^2 below the diagonal, sh[1 + j] = x^H P(:, j): NS threads per value
      // each adding every NS-th workgroup's partial, then the NS sub-sums in order
      const zc* pp = a.part + (size_t)(cp & 1) * a.nwg * (BMAX + 1);
      if ((int)threadIdx.x < NS * (B + 1)) {
        const int q = threadIdx.x % (B + 1), sub = threadIdx.x / (B + 1);
        shs[sub][q] = strided_sum_dev(pp + q, BMAX + 1, sub, a.nwg, NS);
      }
      if ((int)threadIdx.x < B) rcs[threadIdx.x] = ld_dev(a.rowc + (cp & 1) * BMAX + threadIdx.x);
      __syncthreads();
      if ((int)threadIdx.x < B + 1) {
        zc t = shs[0][threadIdx.x];
        for (int u = 1; u < NS; ++u) t += shs[u][threadIdx.x];
        sh[threadIdx.x] = t;
      }
      __syncthreads();
      const zc alpha = rcs[cp];
      zc beta, tau, scale;
      larfg(alpha, sh[0].re, beta, tau, scale);
      const zc ctau = conj(tau);
      // v_i = 1 (i == cp), x_i scale (i > cp), 0 above
      zc xcp = mkz(0, 0);
#pragma unroll
      for (int j = 0; j < B; ++j)
        if (j == cp) xcp = row[j];
      zc vi = mkz(0, 0);
      if (live && i == cp) vi = mkz(1, 0);
      if (live && i > cp) vi = xcp * scale;
      // w_j = v^H P(:, j) = P(cp, j) + conj(scale) (x^H P(:, j) - conj(alpha) P(cp, j))
      const zc cs = conj(scale);
#pragma unroll
      for (int j = 0; j < B; ++j) {
        if (j > cp && j < a.b) {
          const zc pj = rcs[j];
          const zc wj = pj + cs * (sh[1 + j] - conj(alpha) * pj);
          if (live && i >= cp) row[j] -= (ctau * vi) * wj;
        }
      }
#pragma unroll
      for (int j = 0; j < B; ++j)
        if (j == cp && live && i >= cp) row[j] = (i == cp) ? beta : vi;
      if (blockIdx.x == 0 && threadIdx.x == 0) a.tau[cp] = tau;
    }
    if (c < a.k) {
      // partial sums of column c over this workgroup's rows, 16 columns at a time (fewer
      // live registers), out with row c
      const bool on = live && i >= c;
      zc x = mkz(0, 0);
#pragma unroll
      for (int j = 0; j < B; ++j)
        if (j == c) x = row[j];
      const double x0 = (on && i > c) ? norm2(x) : 0.0;
#pragma unroll
      for (int h = 0; h < B / 16; ++h) {
        zc v[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const int j = 16 * h + q;
          v[q] = (on && j > c && j < a.b) ? fma_conj(x, row[j], mkz(0, 0)) : mkz(0, 0);
        }
        block_sum_bf<16>(h == 0 ? x0 : 0.0, v, h == 0 ? red : red2);
      }
      if ((int)threadIdx.x < B + 1) {
        const int q = threadIdx.x;
        const zc val = (q <= 16) ? red[4 * 17 + q] : red2[4 * 17 + q - 16];
        st_dev(a.part + (size_t)(c & 1) * a.nwg * (BMAX + 1) + (size_t)blockIdx.x * (BMAX + 1) + q, val);
      }
      if (live && i == c) {
#pragma unroll
        for (int j = 0; j < B; ++j)
          if (j >= c && j < a.b) st_dev(a.rowc + (c & 1) * BMAX + j, row[j]);
      }
      __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (threadIdx.x == 0) __hip_atomic_fetch_add(bar + c, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (!live) return;
#pragma unroll
  for (int j = 0; j < B; ++j) {
    if (j >= a.b) continue;
    if (i <= j) stz(a.A[(size_t)(a.r0 + i) + (size_t)a.ld * (a.c0 + j)], row[j]);    // R
    zc x = mkz(0, 0);
    if (j < a.k) x = i == j ? mkz(1, 0) : (i > j ? row[j] : mkz(0, 0));
    V[i + N * j] = x;
  }
}

// one workgroup: T (ZLARFT, forward, columnwise) from G = V^H V and tau, and t2 = T^H t1
// (t1 = V^H gc); G and t1 column-major with ld B, T stored [col][row].  T = (I + D U)^-1 D
// with D = diag(tau), U the strict upper triangle of G (the closed form of ZLARFT's
// recurrence T(0:c, c) = -tau_c T(0:c, 0:c) G(0:c, c), T(c, c) = tau_c, which also gives
// T(:, c) = 0 when tau_c = 0), so every column is an independent back substitution:
// column c by the eight lanes t = 8c .. 8c + 7, lane j holding T(q, c) for q = j (mod 8).
template <int B>
__global__ __launch_bounds__(256) void k_pT(int k, const zc* __restrict__ G, const zc* __restrict__ t1,
                                            const zc* __restrict__ tau, int nrhs, zc* __restrict__ Tm,
                                            zc* __restrict__ t2) {
  __shared__ zc Gs[B * B];
  __shared__ zc Ts[B * B];
  __shared__ zc taus[B];
  for (int q = threadIdx.x; q < B * B; q += 256) Gs[q] = G[q];   // G(r, c) at [c][r]
  if ((int)threadIdx.x < B) taus[threadIdx.x] = ((int)threadIdx.x < k) ? tau[threadIdx.x] : mkz(0, 0);
  __syncthreads();
  const int c = threadIdx.x >> 3, j = threadIdx.x & 7;
  constexpr int NU = B / 8;
  if (c < B) {
    zc tq[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) tq[u] = (j + 8 * u == c) ? taus[c] : mkz(0, 0);
    for (int r = c - 1; r >= 0; --r) {
      zc acc = mkz(0, 0);
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const int q = j + 8 * u;
        if (q > r && q <= c) acc = fma_z(Gs[q * B + r], tq[u], acc);
      }
#pragma unroll
      for (int off = 1; off < 8; off <<= 1) {
        acc.re += __shfl_xor(acc.re, off);
        acc.im += __shfl_xor(acc.im, off);
      }
      const zc val = mkz(0, 0) - taus[r] * acc;
#pragma unroll
      for (int u = 0; u < NU; ++u)
        if (j + 8 * u == r) tq[u] = val;
    }
#pragma unroll
    for (int u = 0; u < NU; ++u) Ts[c * B + j + 8 * u] = tq[u];
  }
  __syncthreads();
  for (int q = threadIdx.x; q < B * B; q += 256) Tm[q] = Ts[q];
  // t2(p, r) = sum_q conj(T(q, p)) t1(q, r), T(q, p) = Ts[p][q], q <= p
  for (int q = threadIdx.x; q < B * 6; q += 256) {
    const int p = q / 6, r = q % 6;
    zc sacc = mkz(0, 0);
    if (r < nrhs)
      for (int qq = 0; qq <= p; ++qq) sacc = fma_conj(Ts[p * B + qq], t1[(size_t)r * B + qq], sacc);
    t2[q] = sacc;
  }
}

// Y = V T (rows of the panel) and gc -= V t2
template <int B>
__global__ __launch_bounds__(PR) void k_pY(int m, int N, int r0, const zc* __restrict__ V, const zc* __restrict__ Tm,
                                           const zc* __restrict__ t2, int nrhs, zc* __restrict__ Y, zc* __restrict__ gc) {
  __shared__ zc Ts[B * B];
  __shared__ zc t2s[6 * B];
  for (int q = threadIdx.x; q < B * B; q += PR) Ts[q] = Tm[q];
  for (int q = threadIdx.x; q < 6 * B; q += PR) t2s[q] = t2[q];
  __syncthreads();
  const int i = blockIdx.x * PR + threadIdx.x;
  if (i >= m) return;
  zc v[B];
#pragma unroll
  for (int j = 0; j < B; ++j) v[j] = V[i + (size_t)N * j];
#pragma unroll
  for (int c = 0; c < B; ++c) {
    zc s = mkz(0, 0);
#pragma unroll
    for (int q = 0; q <= c; ++q) s = fma_z(v[q], Ts[c * B + q], s);
    Y[i + (size_t)N * c] = s;
  }
  for (int r = 0; r < nrhs; ++r) {
    zc s = mkz(0, 0);
#pragma unroll
    for (int q = 0; q < B; ++q) s = fma_z(v[q], t2s[q * 6 + r], s);
    gc[(size_t)r * N + r0 + i] -= s;
  }
}

// W = X - 1/2 V Z with Z = T^H M, M = V^H X (column-major, ld B)
template <int B>
__global__ __launch_bounds__(PR) void k_pW(int m, int N, const zc* __restrict__ V, const zc* __restrict__ Tm,
                                           const zc* __restrict__ M, zc* __restrict__ X) {
  __shared__ zc Zs[B * B];
  __shared__ zc Ts[B * B];
  __shared__ zc Ms[B * B];
  for (int q = threadIdx.x; q < B * B; q += PR) {
    Ts[q] = Tm[q];
    Ms[q] = M[q];
  }
  __syncthreads();
  for (int q = threadIdx.x; q < B * B; q += PR) {
    const int p = q / B, c = q % B;      // Z(p, c) = sum_r conj(T(r, p)) M(r, c), T(r, p) = Ts[p][r], r <= p
    zc sacc = mkz(0, 0);
    for (int r = 0; r <= p; ++r) sacc = fma_conj(Ts[p * B + r], Ms[c * B + r], sacc);
    Zs[q] = sacc;
  }
  __syncthreads();
  const int i = blockIdx.x * PR + threadIdx.x;
  if (i >= m) return;
  zc v[B];
#pragma unroll
  for (int j = 0; j < B; ++j) v[j] = V[i + (size_t)N * j];
#pragma unroll
  for (int c = 0; c < B; ++c) {
    zc sacc = mkz(0, 0);
#pragma unroll
    for (int p = 0; p < B; ++p) sacc = fma_z(v[p], Zs[p * B + c], sacc);
    X[i + (size_t)N * c] -= 0.5 * sacc;
  }
}

// Tall-skinny products out0 = A^H Y0 (B x B) and out1 = A^H Y1 (B x n1, n1 <= 16) over m
// rows (A, Y1 with ld N, Y0 with ld ldy0): FP64 MFMA on 64-row chunks staged through LDS,
// chunks c = blockIdx.x, + gridDim.x, ..., one partial per workgroup, summed in workgroup
// order by k_gram_sum.  Wave w accumulates the 16 x 16 output tiles w and w + 4.
#define GRAM_ROWS 64
#define GRAM_PMAX 64
template <int B>
__global__ __launch_bounds__(256) void k_gram(int m, int N, const zc* __restrict__ A, const zc* __restrict__ Y0,
                                              int ldy0, const zc* __restrict__ Y1, int n1, zc* __restrict__ part) {
  constexpr int NY = B + 16;                 // columns of [Y0 | Y1]
  constexpr int TI = B / 16;                 // output tile rows
  __shared__ zc As[GRAM_ROWS][B];
  __shared__ zc Ys[GRAM_ROWS][NY];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int ntile = TI * (TI + (n1 > 0 ? 1 : 0));
  d4 acc[2][2];                              // [tile slot][re, im]
  for (int x = 0; x < 2; ++x) acc[x][0] = acc[x][1] = d4{0, 0, 0, 0};
  const int nch = (m + GRAM_ROWS - 1) / GRAM_ROWS;
  for (int ch = blockIdx.x; ch < nch; ch += gridDim.x) {
    const int row0 = ch * GRAM_ROWS;
    __syncthreads();
    for (int e = t; e < GRAM_ROWS * B; e += 256) {
      const int rr = e % GRAM_ROWS, cc = e / GRAM_ROWS, row = row0 + rr;
      As[rr][cc] = row < m ? A[row + (size_t)N * cc] : mkz(0, 0);
      Ys[rr][cc] = row < m ? Y0[row + (size_t)ldy0 * cc] : mkz(0, 0);
    }
    for (int e = t; e < GRAM_ROWS * 16; e += 256) {
      const int rr = e % GRAM_ROWS, cc = e / GRAM_ROWS, row = row0 + rr;
      Ys[rr][B + cc] = (row < m && cc < n1) ? Y1[row + (size_t)N * cc] : mkz(0, 0);
    }
    __syncthreads();
    for (int x = 0; x < 2; ++x) {
      const int tile = wave + 4 * x;
      if (tile >= ntile) continue;
      const int ti = tile % TI, tj = tile / TI;
      const int i = ti * 16 + (lane & 15), j = tj * 16 + (lane & 15);
#pragma unroll 4
      for (int k0 = 0; k0 < GRAM_ROWS; k0 += 4) {
        const int kk = k0 + (lane >> 4);
        const zc av = As[kk][i], yv = Ys[kk][j];
        // conj(a) y = (ar yr + ai yi) + i (ar yi - ai yr)
        acc[x][0] = mfma16x16x4(av.re, yv.re, acc[x][0]);
        acc[x][0] = mfma16x16x4(av.im, yv.im, acc[x][0]);
        acc[x][1] = mfma16x16x4(av.re, yv.im, acc[x][1]);
        acc[x][1] = mfma16x16x4(-av.im, yv.re, acc[x][1]);
      }
    }
  }
  // partial: [blockIdx][B][NY] (row i of the output, column j of [Y0 | Y1])
  zc* pp = part + (size_t)blockIdx.x * B * NY;
  for (int x = 0; x < 2; ++x) {
    const int tile = wave + 4 * x;
    if (tile >= ntile) continue;
    const int ti = tile % TI, tj = tile / TI;
    for (int q = 0; q < 4; ++q) {
      const int i = ti * 16 + (lane >> 4) + 4 * q, j = tj * 16 + (lane & 15);
      pp[(size_t)i * NY + j] = mkz(acc[x][0][q], acc[x][1][q]);
    }
  }
}

// out0 (B x B, ld B) and out1 (B x n1, ld B) from the P partials, in workgroup order: four
// threads per output each add a quarter of the partials, then the quarters in order
template <int B>
__global__ __launch_bounds__(256) void k_gram_sum(int P, const zc* __restrict__ part, int n1, zc* __restrict__ out0,
                                                  zc* __restrict__ out1) {
  constexpr int NY = B + 16;
  const int o = blockIdx.x * 64 + (threadIdx.x >> 2), sub = threadIdx.x & 3;
  const int i = o / NY, j = o % NY;
  const bool live = i < B && (j < B || j - B < n1);
  const int per = (P + 3) / 4, w0 = sub * per, w1 = min(P, w0 + per);
  zc x = mkz(0, 0);
  if (live && w0 < w1) x = strided_sum(part + (size_t)i * NY + j, (size_t)B * NY, w0, w1, 1, mkz(0, 0));
  const zc x1 = shfl_xor_z(x, 1);
  const zc x2 = shfl_xor_z(x, 2), x3 = shfl_xor_z(x, 3);
  if (!live || sub != 0) return;
  const zc sum = ((x + x1) + x2) + x3;       // quarters 0, 1, 2, 3
  if (j < B) out0[i + (size_t)B * j] = sum;
  else out1[i + (size_t)B * (j - B)] = sum;
}

// X = A Y for the Hermitian trailing matrix A (m x m, lower triangle, ld) and the panel's
// Y (m x BC, ld ldy) on MFMA: FP32 operands and accumulation for the COMPLEX*8 matrix,
// FP64 for the COMPLEX*16 one.  A workgroup owns 128 rows and a K slice (blockIdx.y) and
// walks it in steps of 16 staged through LDS, the next step's loads in flight while the
// current one is multiplied; wave w computes rows 32w..32w+31 for all BC columns.  A step
// below the diagonal reads A(i, k) down the columns; a step above it reads conj(A(k, i))
// down the columns of the transposed block; a step across it reads element by element.
// With more than one slice the partials go to part[z][col][row] and k_hmm_sum adds them in
// slice order.
#define HB_R 128
#define HB_SMAX 16      // most K slices
template <class T, int BC>
__global__ __launch_bounds__(256) void k_hmm_b(int m, const T* __restrict__ A, int ld, const zc* __restrict__ Y,
                                               int ldy, int kc, zc* __restrict__ part, zc* __restrict__ X, int ldx) {
  constexpr bool F64 = sizeof(T) == sizeof(zc);
  typedef typename std::conditional<F64, double2, float2>::type ct;
  typedef typename std::conditional<F64, d4, f4>::type acc_t;
  constexpr int KS = F64 ? 16 : 32;                 // K per step (32 KB of the matrix in LDS)
  constexpr int NA = KS * HB_R / 256;               // matrix elements per thread and step
  constexpr int CT = BC / 16;                       // 16-column tiles
  constexpr int YP = KS * BC / 256;                 // Y elements per thread and step
  // rows padded by one element: the four k rows a wave reads at once (and the 16 rows the
  // transposed loads store at once) fall in different LDS banks
  __shared__ ct As[KS][HB_R + 1];
  __shared__ ct Ys[KS][BC + 1];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int i16 = lane & 15, kq = lane >> 4;
  const int R0 = blockIdx.x * HB_R;
  const int kbeg = blockIdx.y * kc, kend = min(m, kbeg + kc);
  // loaders: A(row R0 + (t & 127), k + (t >> 7) + 2u) below or across the diagonal,
  // conj(A(k + (t & 15) + 16 (u / 8), row R0 + (t >> 4) + 16 (u % 8))) above it (rows past m
  // read row m - 1, never stored); Y(k + (t % KS), t / KS + (256 / KS) u)
  const int arow = min(R0 + (t & 127), m - 1), ak = t >> 7;
  const int tk = t & 15, ti = t >> 4;
  const int yk = t % KS, ycol = t / KS;
  int lmode = 0;                                    // 0 below, 1 above, 2 across the diagonal
  acc_t cr[2][CT], ci[2][CT];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < CT; ++b) cr[a][b] = ci[a][b] = acc_t{0, 0, 0, 0};
  T ra[NA];
  zc ry[YP];
  auto gload = [&](int k0) {
    lmode = (k0 + KS - 1 <= R0) ? 0 : (k0 > R0 + HB_R - 1) ? 1 : 2;
    if (lmode == 1) {
#pragma unroll
      for (int u = 0; u < NA; ++u) {
        const int k = min(k0 + tk + 16 * (u / 8), m - 1);
        const int i = min(R0 + ti + 16 * (u % 8), m - 1);
        ra[u] = A[(size_t)k + (size_t)ld * i];
      }
    } else {
#pragma unroll
      for (int u = 0; u < NA; ++u) {
        const int k = min(k0 + ak + 2 * u, m - 1);  // past kend: Y is zero there
        ra[u] = (lmode == 0 || arow >= k) ? A[(size_t)arow + (size_t)ld * k] : A[(size_t)k + (size_t)ld * arow];
        if (lmode == 2 && arow < k) ra[u].im = -ra[u].im;
      }
    }
#pragma unroll
    for (int u = 0; u < YP; ++u) {
      const int k = k0 + yk;
      ry[u] = (k < kend) ? Y[(size_t)k + (size_t)ldy * (ycol + (256 / KS) * u)] : mkz(0, 0);
    }
  };
  gload(kbeg);
  for (int k0 = kbeg; k0 < kend; k0 += KS) {
    __syncthreads();                                  // the previous step is consumed
#pragma unroll
    for (int u = 0; u < NA; ++u) {
      ct v;
      v.x = ra[u].re;
      v.y = ra[u].im;
      if (lmode == 1) {
        v.y = -v.y;                                 // A(i, k) = conj(A(k, i))
        As[tk + 16 * (u / 8)][ti + 16 * (u % 8)] = v;
      } else {
        As[ak + 2 * u][t & 127] = v;
      }
    }
#pragma unroll
    for (int u = 0; u < YP; ++u) {
      ct v;
      v.x = ry[u].re;
      v.y = ry[u].im;
      Ys[yk][ycol + (256 / KS) * u] = v;
    }
    __syncthreads();
    if (k0 + KS < kend) gload(k0 + KS);
#pragma unroll
    for (int kk = 0; kk < KS / 4; ++kk) {
      const int k = 4 * kk + kq;
      ct av[2], yv[CT];
#pragma unroll
      for (int a = 0; a < 2; ++a) av[a] = As[k][32 * w + 16 * a + i16];
#pragma unroll
      for (int b = 0; b < CT; ++b) yv[b] = Ys[k][16 * b + i16];
      // (ar + i ai)(yr + i yi) = (ar yr - ai yi) + i (ar yi + ai yr).  Each accumulator
      // takes its two products in this order; the first products of all accumulators go
      // before the second ones, so that no MFMA waits on the one just issued
#pragma unroll
      for (int b = 0; b < CT; ++b)
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          if constexpr (F64) {
            cr[a][b] = mfma16x16x4(av[a].x, yv[b].x, cr[a][b]);
            ci[a][b] = mfma16x16x4(av[a].x, yv[b].y, ci[a][b]);
          } else {
            cr[a][b] = mfma16x16x4f32(av[a].x, yv[b].x, cr[a][b]);
            ci[a][b] = mfma16x16x4f32(av[a].x, yv[b].y, ci[a][b]);
          }
        }
#pragma unroll
      for (int b = 0; b < CT; ++b)
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          if constexpr (F64) {
            cr[a][b] = mfma16x16x4(-av[a].y, yv[b].y, cr[a][b]);
            ci[a][b] = mfma16x16x4(av[a].y, yv[b].x, ci[a][b]);
          } else {
            cr[a][b] = mfma16x16x4f32(-av[a].y, yv[b].y, cr[a][b]);
            ci[a][b] = mfma16x16x4f32(av[a].y, yv[b].x, ci[a][b]);
          }
        }
    }
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < CT; ++b) {
      const int col = 16 * b + i16;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        // f64 MFMA: register q holds row kq + 4q of the tile; f32 MFMA: row 4kq + q
        const int row = R0 + 32 * w + 16 * a + (F64 ? kq + 4 * q : 4 * kq + q);
        if (row >= m) continue;
        const zc v = mkz((double)cr[a][b][q], (double)ci[a][b][q]);
        if (part) part[(size_t)blockIdx.y * m * BC + (size_t)col * m + row] = v;
        else X[(size_t)row + (size_t)ldx * col] = v;
      }
    }
}

// X(row, col) = sum over the ns slices of part[z][col][row], in slice order
template <int BC>
__global__ __launch_bounds__(256) void k_hmm_sum(int m, int ns, const zc* __restrict__ part, zc* __restrict__ X,
                                                 int ldx) {
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= (size_t)m * BC) return;
  const int row = (int)(e % m), col = (int)(e / m);
  X[(size_t)row + (size_t)ldx * col] = strided_sum(part + e, (size_t)m * BC, 0, ns, 1, mkz(0, 0));
}

// A22 -= U, U = V W^H + W V^H, on the 64 x 64 tiles of the trailing matrix (rows and
// columns r0..N-1) on and below the diagonal, K = 2 b: FP64 MFMA on the COMPLEX*16 matrix, FP32 MFMA (FP32 operands
// and accumulation) on the COMPLEX*8 one.  The MFMA rows run over the tile's columns and
// its columns over the tile's rows, D(i, j) = U(c_i, r_j) = conj(U(r_j, c_i)) since U is
// Hermitian, so that a lane's result lands next to its neighbours' in the column-major
// matrix.
template <class T, int B>
__device__ __forceinline__ void her2k_tile(T* __restrict__ A, int ld, int m, int r0, int N, const zc* __restrict__ V,
                                           const zc* __restrict__ W, const int bx) {
  // one workgroup per tile on or below the diagonal: t -> tile row ti >= tile column tj
  const int t = bx;
  int ti = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
  while ((ti + 1) * (ti + 2) / 2 <= t) ++ti;
  while (ti * (ti + 1) / 2 > t) --ti;
  const int tj = t - ti * (ti + 1) / 2;
  constexpr bool F64 = sizeof(T) == sizeof(zc);
  constexpr int K = 2 * B;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ci0 = tj * 64 + (wave >> 1) * 32;           // tile columns (MFMA rows)
  const int rj0 = ti * 64 + (wave & 1) * 32;            // tile rows (MFMA columns)
  const int lr = lane & 15, lk = lane >> 4;
  typedef typename std::conditional<F64, d4, f4>::type acc_t;
  // COMPLEX*8: the tile's current values are loaded first, so that their latency overlaps
  // the products (at N = 36864 6.2 s against 6.5 s per matrix); the COMPLEX*16 tile would
  // cost the registers of two more waves per SIMD (8.5 % slower at N = 12000)
  constexpr int HV = F64 ? 1 : 16;
  T hv[HV];
  if constexpr (!F64) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int c = ci0 + x * 16 + 4 * lk + q, r = rj0 + y * 16 + lr;
          if (r < m && c < m) hv[(x * 2 + y) * 4 + q] = A[(size_t)(r0 + r) + (size_t)ld * (r0 + c)];
        }
  }
  acc_t cr[2][2], ci[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) cr[x][y] = ci[x][y] = acc_t{0, 0, 0, 0};
  if constexpr (!F64) {
    // COMPLEX*8: the tile's operands go through LDS once per workgroup, in FP32, half of K
    // at a time (a wave pair shares each operand); the products run in the order of k
    __shared__ zf As[B][65], Bs[B][65];     // padded rows: no bank conflicts between k rows
    const int cl0 = tj * 64, rl0 = ti * 64;
    const int ciw = (wave >> 1) * 32, rjw = (wave & 1) * 32;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // half 0: A = V(c, k), B = W(r, k); half 1: A = W(c, k), B = V(r, k)
      const zc* Asrc = h == 0 ? V : W;
      const zc* Bsrc = h == 0 ? W : V;
      if (h > 0) __syncthreads();
#pragma unroll 4
      for (int u = 0; u < B * 64 / 256; ++u) {
        const int e = threadIdx.x + 256 * u, kk = e >> 6, cc = e & 63;
        const int c = cl0 + cc, r = rl0 + cc;
        const zc a = (c < m) ? Asrc[(size_t)kk * N + c] : mkz(0, 0);
        const zc b = (r < m) ? Bsrc[(size_t)kk * N + r] : mkz(0, 0);
        As[kk][cc] = zf{(float)a.re, (float)a.im};
        Bs[kk][cc] = zf{(float)b.re, (float)b.im};
      }
      __syncthreads();
#pragma unroll
      for (int k0 = 0; k0 < B; k0 += 4) {
        const int kk = k0 + lk;
        zf af[2], bf[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          af[x] = As[kk][ciw + x * 16 + lr];
          bf[x] = Bs[kk][rjw + x * 16 + lr];
        }
        // first products of all accumulators, then the second ones (the order within
        // each accumulator is kept)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y) {
            cr[x][y] = mfma16x16x4f32(af[x].re, bf[y].re, cr[x][y]);
            ci[x][y] = mfma16x16x4f32(af[x].im, bf[y].re, ci[x][y]);
          }
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y) {
            cr[x][y] = mfma16x16x4f32(af[x].im, bf[y].im, cr[x][y]);
            ci[x][y] = mfma16x16x4f32(-af[x].re, bf[y].im, ci[x][y]);
          }
      }
    }
  } else {
  // A operand (i = column c, k): [V | W](c, k); B operand (k, j = row r): conj([W | V](r, k));
  // the operands of step k0 + 4 are loaded while step k0 is multiplied
  zc av[2], bv[2];
  auto oload = [&](int k0, zc (&pa)[2], zc (&pb)[2]) {
    const int k = k0 + lk;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int c = ci0 + x * 16 + lr, r = rj0 + x * 16 + lr;
      pa[x] = (c < m) ? ((k < B) ? V[(size_t)k * N + c] : W[(size_t)(k - B) * N + c]) : mkz(0, 0);
      pb[x] = (r < m) ? ((k < B) ? W[(size_t)k * N + r] : V[(size_t)(k - B) * N + r]) : mkz(0, 0);
    }
  };
  oload(0, av, bv);
#pragma unroll
  for (int k0 = 0; k0 < K; k0 += 4) {
    zc an[2], bn[2];
    if (k0 + 4 < K) oload(k0 + 4, an, bn);
    // a * conj(b): the first products of all accumulators, then the second ones (the order
    // within each accumulator is kept)
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        cr[x][y] = mfma16x16x4(av[x].re, bv[y].re, cr[x][y]);
        ci[x][y] = mfma16x16x4(av[x].im, bv[y].re, ci[x][y]);
      }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        cr[x][y] = mfma16x16x4(av[x].im, bv[y].im, cr[x][y]);
        ci[x][y] = mfma16x16x4(-av[x].re, bv[y].im, ci[x][y]);
      }
    if (k0 + 4 < K) {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        av[x] = an[x];
        bv[x] = bn[x];
      }
    }
  }
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        // f64 MFMA: register q holds D row lk + 4q; f32 MFMA: row 4 lk + q
        const int c = ci0 + x * 16 + (F64 ? lk + 4 * q : 4 * lk + q);
        const int r = rj0 + y * 16 + lr;
        if (r < m && c < m) {
          zc v;
          if constexpr (F64) v = ldz(A[(size_t)(r0 + r) + (size_t)ld * (r0 + c)]);
          else v = ldz(hv[(x * 2 + y) * 4 + q]);
          v.re -= cr[x][y][q];
          v.im += ci[x][y][q];       // - conj(D)
          stz(A[(size_t)(r0 + r) + (size_t)ld * (r0 + c)], v);
        }
      }
}
template <class T, int B>
__global__ __launch_bounds__(256, 4) void k_her2k_full(T* __restrict__ A, int ld, int m, int r0, int N,
                                                    const zc* __restrict__ V, const zc* __restrict__ W) {
  her2k_tile<T, B>(A, ld, m, r0, N, V, W, blockIdx.x);
}

// band of width b of the lower triangle into BD (FP64), zero for b < d <= 2b; gc = conj(g)
template <class T>
__device__ __forceinline__ void band_extract(const T* __restrict__ A, int ld, int N, int b, int LB,
                                             zc* __restrict__ BD, const int bx) {
  const int c = bx;
  for (int d = threadIdx.x; d < LB; d += blockDim.x) {
    zc v = mkz(0, 0);
    if (d <= b && c + d < N) v = ldz(A[(size_t)(c + d) + (size_t)ld * c]);
    if (d == 0) v.im = 0.0;
    BD[(size_t)c * LB + d] = v;
  }
}
template <class T>
__global__ void k_band_extract(const T* __restrict__ A, int ld, int N, int b, int LB, zc* __restrict__ BD) {
  band_extract(A, ld, N, b, LB, BD, blockIdx.x);
}

__global__ void k_conj_vec(int n, const zc* __restrict__ x, zc* __restrict__ y) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = clean_nan(conj(x[i]));
}

// sum over groups of SUB (8 or 16) consecutive lanes, the same bits in each: ^1, ^2, then
// i <-> 7 - i and i <-> 15 - i
template <int SUB>
__device__ inline zc sub_sum(zc x) {
  x += dpp_z<0xB1>(x);
  x += dpp_z<0x4E>(x);
  x += dpp_z<0x141>(x);
  if constexpr (SUB == 16) x += dpp_z<0x140>(x);
  return x;
}

__device__ inline zc fnma_z(zc a, zc b, zc c) {          // c - a b
  return mkz(fma(-a.re, b.re, fma(a.im, b.im, c.re)), fma(-a.re, b.im, fma(-a.im, b.re, c.im)));
}
__device__ inline zc fnma_zc(zc a, zc b, zc c) {         // c - a conj(b)
  return mkz(fma(-a.re, b.re, fma(-a.im, b.im, c.re)), fma(a.re, b.im, fma(-a.im, b.re, c.im)));
}

// ZLARFG as above for latency chains: beta from one reciprocal square root
// (two Newton steps, then a correction of the root), 1/(alpha - beta) from one reciprocal, each
// quotient corrected by its remainder to the rounding of a division; where squares near the
// range's ends would not do, as above
__device__ inline void larfg_fast(zc alpha, double xn2, zc& beta, zc& tau, zc& scale) {
  const bool ident = xn2 == 0.0 && alpha.im == 0.0;
  const double n2 = ident ? 1.0 : alpha.re * alpha.re + alpha.im * alpha.im + xn2;
  if (!(n2 > 1e-280 && n2 < 1e280)) {
    larfg(alpha, xn2, beta, tau, scale);
    return;
  }
  double y = __builtin_amdgcn_rsq(n2);
  const double hn = 0.5 * n2;
  y = fma(y, fma(-hn * y, y, 0.5), y);
  y = fma(y, fma(-hn * y, y, 0.5), y);
  double nrm = n2 * y;
  nrm = fma(fma(-nrm, nrm, n2), 0.5 * y, nrm);
  const double sg = alpha.re >= 0.0 ? -1.0 : 1.0;
  const double b = sg * nrm, rb = sg * y;
  const double dr = alpha.re - b;               // same signs: no cancellation
  const double den = fma(dr, dr, alpha.im * alpha.im);
  double rd = __builtin_amdgcn_rcp(den);
  rd = fma(rd, fma(-den, rd, 1.0), rd);
  rd = fma(rd, fma(-den, rd, 1.0), rd);
  auto quot = [](double x, double d, double r) {   // x / d with r about 1 / d
    const double q = x * r;
    return fma(fma(-d, q, x), r, q);
  };
  beta = ident ? alpha : mkz(b, 0.0);
  tau = ident ? mkz(0, 0) : mkz(quot(-dr, b, rb), quot(-alpha.im, b, rb));
  scale = ident ? mkz(0, 0) : mkz(quot(dr, den, rd), quot(-alpha.im, den, rd));
}

// One element by a buffer load or store that the caches of other XCDs see (sc1), 16 bytes at
// once; loads past the buffer's end give zero.  Aux bit 4 is sc1 on gfx94x and gfx950.
__device__ inline __amdgpu_buffer_rsrc_t dev_buffer(void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, (int)(bytes > 0xFFFFFFF0ull ? 0xFFFFFFF0ull : bytes), 0x00027000);
}
__device__ inline zc ld_buf(__amdgpu_buffer_rsrc_t rs, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(zc, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, 16));
}
__device__ inline void st_buf(__amdgpu_buffer_rsrc_t rs, unsigned voff, unsigned soff, zc v) {
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), rs, voff, soff, 16);
}

// ---------------------------------------------------------------------------
// stage 1, COMPLEX*16 matrix: the whole panel step up to Y in one launch
// ---------------------------------------------------------------------------
#define QP_WG 64          // most workgroups of the launch (panel rows up to 256 QP_WG)

// workgroup barrier for LDS traffic alone: global loads and stores stay in flight
__device__ inline void lds_barrier() { __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// a uniform lane's value, in scalar registers
__device__ inline double lane_value(double x, int l) {
  const unsigned long long v = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = __builtin_amdgcn_readlane((int)v, l), hi = __builtin_amdgcn_readlane((int)(v >> 32), l);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ inline zc lane_value(zc v, int l) { return mkz(lane_value(v.re, l), lane_value(v.im, l)); }

// Values handed from every workgroup to every workgroup: slot [round][workgroup][B], each
// slot written once per panel and filled with the bits ~0 before (a NaN; one of the input's
// could have them and keep them through arithmetic, so whatever the slots' sums are formed
// from is cleaned of such: the panel's columns, X and the tracked vectors), so that a reader
// polls the value itself: no counter, no fence, one store and one load apart.  Rounds 0 .. B - 1 are the panel's columns, B .. B + 5 the tracked vectors;
// entry nwg of a column's round is row c of the panel.
struct QrPanelArgs {
  zc* A;                 // the matrix, ld
  int ld, N;
  int c0, r0, m, k;      // panel columns c0 .. c0 + B - 1, rows r0 .. N - 1 (m), k reflectors
  zc *V, *Y;             // [B][N]
  zc* Tm;                // T(q, c) at [c][q]
  zc* gc;                // nrhs x N
  int nrhs;
  zc *ex, *ex_next;      // this panel's slots; the next panel's, filled here
  int exs;               // workgroups per round of the slots
  int nwg;
  int* err;
  int spin_limit;
  zc* tau;               // where column q's tau goes; V is kept below R then (null: neither)
};

__device__ inline bool is_empty(zc v) {
  return __builtin_bit_cast(unsigned long long, v.re) == ~0ull || __builtin_bit_cast(unsigned long long, v.im) == ~0ull;
}

// what a poll of slots starts with: the loads after it are not those of the poll before
__device__ inline void poll_again() { __asm__ volatile("" ::: "memory"); }

template <int B>
__host__ __device__ constexpr size_t qr_slots(int nwg_max) { return (size_t)(B + 6) * (nwg_max + 1) * B; }

// Householder QR of the panel (ZGEQRF's reflectors), V, R, T (ZLARFT), Y = V T and
// gc <- Q^H gc.  Workgroup w keeps rows 256 w .. of the panel in registers, one a thread.
// Per column one exchange: the sums d_j = sum over rows i > c of conj(x_i) row_j(i), for the
// columns j > c not yet reduced, j = c (|x|^2) and the finished reflectors j < c alike, and
// row c.  From these every workgroup forms the reflector, the update of its rows
// (v^H P_j = P(c, j) + conj(scale) d_j) and column c of T (v_j^H v_c = conj(V(c, j)) +
// scale conj(d_j)), the latter while the next column's sums are on their way; thread
// (i, j sub) holds T(i, j).
//
// Bound by latency: 54 us a panel of 16 columns (61 with more than 15 workgroups), about
// 6400 cycles a column, of which the exchange (store, first load that sees it) takes 2700 and the sums, the reflector and the
// update of the rows the rest; the launches that it replaces took about 10 us a column.  The
// launch needs every workgroup resident: band_panel_wg.
template <int B>
__device__ __forceinline__ void qr_panel(const QrPanelArgs& a, const int bx) {
  constexpr int SUB = 256 / B;                 // threads per exchanged value
  constexpr int NT = B / SUB;                  // T entries per thread
  __shared__ zc lp[4][4][B / 4][16];           // partial sums [wave][row quarter][column][lane]
  __shared__ zc dq[B], rq[B], rowc[B];         // totals and row c; row c on its way out
  __shared__ zc Ts[B][B + 1];
  __shared__ zc t1s[6][B], t2s[6][B];
  __shared__ int bad;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int i = bx * 256 + t;          // panel row
  const bool live = i < a.m;
  const int q = t / SUB, sub = t % SUB;        // exchanged value; T row and its columns sub + SUB u
  const size_t N = a.N;
  const unsigned RS = (unsigned)(a.exs * B) * (unsigned)sizeof(zc);   // bytes per round
  const __amdgpu_buffer_rsrc_t ex = dev_buffer(a.ex, (size_t)(B + 6) * RS);
  const unsigned mine = (unsigned)(bx * B) * (unsigned)sizeof(zc);
  if (t == 0) bad = 0;
  zc row[B];
  {
    const zc* ap = a.A + (size_t)(a.r0 + min(i, a.m - 1)) + (size_t)a.ld * a.c0;
#pragma unroll
    for (int j = 0; j < B; ++j) row[j] = ap[(size_t)a.ld * j];
    if (!live) {
#pragma unroll
      for (int j = 0; j < B; ++j) row[j] = mkz(0, 0);
    }
    if (a.c0 == 0) {                           // (the later panels' columns come from strip)
#pragma unroll
      for (int j = 0; j < B; ++j) row[j] = clean_nan(row[j]);
    }
  }
  // the next panel's slots
  const zc empty = __builtin_bit_cast(zc, make_uint4(~0u, ~0u, ~0u, ~0u));
  for (int e = t; e < (B + 6) * B; e += 256) a.ex_next[(size_t)(e / B) * a.exs * B + (size_t)bx * B + e % B] = empty;
  if (bx == 0)
    for (int e = t; e < B * B; e += 256) a.ex_next[(size_t)(e / B) * a.exs * B + (size_t)a.nwg * B + e % B] = empty;

  // sum over the workgroup of B values a thread: halved over the lane halves and the rows of
  // 16, the rest through LDS; threads (q, .) end with the sum of value q
  auto block_sums = [&](zc (&v)[B]) {
#pragma unroll
    for (int j = 0; j < B / 2; ++j) v[j] = mkz(add32(v[j].re, v[j + B / 2].re), add32(v[j].im, v[j + B / 2].im));
#pragma unroll
    for (int j = 0; j < B / 4; ++j) {
      v[j] = mkz(add16(v[j].re, v[j + B / 4].re), add16(v[j].im, v[j + B / 4].im));
      lp[wave][lane >> 4][j][lane & 15] = v[j];
    }
    lds_barrier();
    zc s = mkz(0, 0);
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int u = 0; u < 16; u += SUB) s += lp[w][q / (B / 4)][q % (B / 4)][sub + u];
    return sub_sum<SUB>(s);
  };
  // value q of rounds c .. c + nr - 1 summed over the workgroups, and entry nwg of round c
  // (row c); all loads of a pass at once, repeated until every value is there (bounded)
  auto gather_u = [&](auto nrc, auto uc, int n, int c, int nr, bool with_row, zc* tot, zc& rowv) {
    constexpr int NR = decltype(nrc)::value, U = decltype(uc)::value;
    zc s[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) s[r] = mkz(0, 0);
    for (int w0 = sub; w0 < n; w0 += U * SUB) {
      zc v[NR][U];
      for (int tries = 0;; ++tries) {
        bool ok = true;
        poll_again();
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if (r < nr)
#pragma unroll
            for (int u = 0; u < U; ++u)
              v[r][u] = ld_buf(ex, (unsigned)(min(w0 + u * SUB, n - 1) * B + q) * (unsigned)sizeof(zc), (c + r) * RS);
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if (r < nr)
#pragma unroll
            for (int u = 0; u < U; ++u) ok = ok && !is_empty(v[r][u]);
        if (ok) break;
        if (tries > a.spin_limit ||
            ((tries & 255) == 255 && __hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
          bad = 1;
          __hip_atomic_store(a.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int w = w0 + u * SUB;
        if (w < a.nwg) {
#pragma unroll
          for (int r = 0; r < NR; ++r)
            if (r < nr) s[r] += v[r][u];
        } else if (with_row && w == a.nwg) {
          rowv = v[0][u];
        }
      }
    }
#pragma unroll
    for (int r = 0; r < NR; ++r)
      if (r < nr) tot[r] = sub_sum<SUB>(s[r]);
  };
  // one slot a thread where that covers them (with four loads a poll throughout, a panel took
  // 60 us at N = 2116, with one 54)
  auto gather = [&](auto nrc, int c, int nr, bool with_row, zc* tot, zc& rowv) {
    const int n = a.nwg + (with_row ? 1 : 0);
    if (n <= SUB) gather_u(nrc, std::integral_constant<int, 1>{}, n, c, nr, with_row, tot, rowv);
    else gather_u(nrc, std::integral_constant<int, decltype(nrc)::value == 1 ? 4 : 2>{}, n, c, nr, with_row, tot, rowv);
  };

  zc T[NT], gcol[NT], taup = mkz(0, 0);
#pragma unroll
  for (int u = 0; u < NT; ++u) T[u] = mkz(0, 0);
  // column c of T: T(0:c, c) = -tau T(0:c, 0:c) (V^H v_c)(0:c), T(c, c) = tau
  auto t_column = [&](int c) {
    zc s = mkz(0, 0);
#pragma unroll
    for (int u = 0; u < NT; ++u)
      if (sub + SUB * u < c) s = fma_z(T[u], gcol[u], s);
    s = sub_sum<SUB>(s);
    const zc v = (q < c) ? mkz(0, 0) - taup * s : (q == c) ? taup : mkz(0, 0);
#pragma unroll
    for (int u = 0; u < NT; ++u)
      if (sub + SUB * u == c) T[u] = v;
  };
  // four columns at a time, then the registers turn by four: in block cb register p holds
  // column (p + 4 cb) % B, so that the column at work is register cc, a constant
  for (int cb = 0; cb < B / 4; ++cb) {
    const int base = 4 * cb;
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) {
      const int c = base + cc;
      if (c < a.k) {
        if (bx == 0 && i == c) {
#pragma unroll
          for (int p = 0; p < B; ++p) rowc[p] = row[p];
        }
        const zc x = row[cc];
        const zc xm = (i > c) ? x : mkz(0, 0);
        zc v[B];
#pragma unroll
        for (int p = 0; p < B; ++p) v[p] = fma_conj(xm, row[p], mkz(0, 0));
        const zc part = block_sums(v);
        if (sub == 0) st_buf(ex, mine + q * (unsigned)sizeof(zc), c * RS, part);
        if (bx == 0 && sub == 1) st_buf(ex, (unsigned)(a.nwg * B + q) * (unsigned)sizeof(zc), c * RS, rowc[q]);
        if (c > 0) t_column(c - 1);            // while the sums are on their way
        zc rowv = mkz(0, 0);
        zc tot;
        gather(std::integral_constant<int, 1>{}, c, 1, true, &tot, rowv);
        if (sub == 0) dq[q] = tot;
        if (sub == a.nwg % SUB) rq[q] = rowv;
        lds_barrier();
        if (bad) return;
        // lane l of every wave: register l % B of row c and its sum
        const zc dl = dq[lane % B], rl = rq[lane % B];
        zc beta, scale;
        larfg_fast(lane_value(rl, cc), lane_value(dl.re, cc), beta, taup, scale);
        // v^H P of the columns not yet reduced
        zc wl = fma_conj(scale, dl, rl);
        if (lane % B <= cc || lane % B >= B - base) wl = mkz(0, 0);
        const zc vi = (i > c) ? x * scale : (i == c ? mkz(1, 0) : mkz(0, 0));
        const zc cv = conj(taup) * vi;
#pragma unroll
        for (int p = cc + 1; p < B; ++p) row[p] = fnma_z(cv, lane_value(wl, p), row[p]);
        row[cc] = (i == c) ? beta : (i > c ? vi : x);
#pragma unroll
        for (int u = 0; u < NT; ++u) {
          const int p = (sub + SUB * u - base) & (B - 1);
          gcol[u] = fma_z(scale, conj(dq[p]), conj(rq[p]));
        }
      }
    }
    zc turn[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) turn[p] = row[p];
#pragma unroll
    for (int p = 0; p < B - 4; ++p) row[p] = row[p + 4];
#pragma unroll
    for (int p = 0; p < 4; ++p) row[B - 4 + p] = turn[p];
  }
  // R into the matrix, V explicit
#pragma unroll
  for (int j = 0; j < B; ++j) {
    const zc p = row[j];
    if (live && (i <= j || a.tau)) a.A[(size_t)(a.r0 + i) + (size_t)a.ld * (a.c0 + j)] = p;
    const zc x = (j < a.k) ? (i == j ? mkz(1, 0) : (i > j ? p : mkz(0, 0))) : mkz(0, 0);
    row[j] = x;
    if (live) a.V[i + N * j] = x;
  }
  // t1 = V^H gc
  zc g[6];
#pragma unroll
  for (int r = 0; r < 6; ++r) {
    if (r >= a.nrhs) break;
    g[r] = live ? a.gc[(size_t)r * N + a.r0 + i] : mkz(0, 0);
    zc v[B];
#pragma unroll
    for (int j = 0; j < B; ++j) v[j] = fma_conj(row[j], g[r], mkz(0, 0));
    if (r > 0) lds_barrier();                  // the partial sums of r - 1 are read
    const zc part = block_sums(v);
    if (sub == 0) st_buf(ex, mine + q * (unsigned)sizeof(zc), (B + r) * RS, part);
  }
  t_column(a.k - 1);
#pragma unroll
  for (int u = 0; u < NT; ++u) Ts[q][sub + SUB * u] = T[u];
  if (a.nrhs > 0) {
    zc tot[6], none;
    gather(std::integral_constant<int, 6>{}, B, a.nrhs, false, tot, none);
#pragma unroll
    for (int r = 0; r < 6; ++r)
      if (r < a.nrhs && sub == 0) t1s[r][q] = tot[r];
  }
  lds_barrier();
  if (bad) return;
  if (bx == 0) {
    for (int e = t; e < B * B; e += 256) a.Tm[e] = Ts[e % B][e / B];
    if (a.tau && t < a.k) a.tau[t] = Ts[t][t];
  }
  // t2 = T^H t1, gc -= V t2
#pragma unroll
  for (int r = 0; r < 6; ++r) {
    if (r >= a.nrhs) break;
    zc s = mkz(0, 0);
#pragma unroll
    for (int u = 0; u < NT; ++u) s = fma_conj(Ts[sub + SUB * u][q], t1s[r][sub + SUB * u], s);
    s = sub_sum<SUB>(s);
    if (sub == 0) t2s[r][q] = s;
  }
  lds_barrier();
#pragma unroll
  for (int r = 0; r < 6; ++r) {
    if (r >= a.nrhs) break;
    const zc tl = t2s[r][lane % B];
    zc s = g[r];
#pragma unroll
    for (int j = 0; j < B; ++j) s = fnma_z(row[j], lane_value(tl, j), s);
    if (live) a.gc[(size_t)r * N + a.r0 + i] = s;
  }
  // Y = V T, four columns at a time (T upper triangular)
  for (int cb = 0; cb < B / 4; ++cb) {
    zc tl[4], y[4];
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) {
      tl[cc] = Ts[lane % B][4 * cb + cc];
      y[cc] = mkz(0, 0);
    }
#pragma unroll
    for (int jb = 0; jb < B / 4; ++jb)
      if (jb <= cb) {
#pragma unroll
        for (int j = 4 * jb; j < 4 * jb + 4; ++j)
#pragma unroll
          for (int cc = 0; cc < 4; ++cc) y[cc] = fma_z(row[j], lane_value(tl[cc], j), y[cc]);
      }
    if (live) {
#pragma unroll
      for (int cc = 0; cc < 4; ++cc) a.Y[i + N * (4 * cb + cc)] = y[cc];
    }
  }
}
template <int B>
__global__ __launch_bounds__(256, 2) void k_qr_panel(QrPanelArgs a) {
  qr_panel<B>(a, blockIdx.x);
}

// W = X - 1/2 V (T^H (V^H X)) with X = A22 Y, in one launch: workgroup w takes rows 256 w ..,
// its part of M = V^H X on FP64 MFMA (operands straight from memory in the MFMA's layout),
// one exchange of the B x B parts as above (slots [workgroup][B B]), then Z = T^H M and its
// rows of W, whose V and X are loaded during the exchange (13.0 us without that, now 10.2
// at N = 2116).  Latency-bound; summing the parts of X here too, on the few workgroups of this
// launch, took 30 us against 17 + 5 with a launch of its own.
struct QrWArgs {
  int m, N;
  const zc *V, *Tm;
  zc* X;                 // in: X, out: W
  zc *ex, *ex_next;
  int nwg;
  int* err;
  int spin_limit;
};

template <int B>
__device__ __forceinline__ void qr_w(const QrWArgs& a, const int bx) {
  constexpr int TI = B / 16, NE = B * B / 256;
  __shared__ zc buf[4 * B * B];                // the waves' parts, then M, Z, T
  typedef zc Mat[B][B + 1];
  zc (*const red)[B * B] = reinterpret_cast<zc(*)[B * B]>(buf);
  Mat &Ms = *reinterpret_cast<Mat*>(buf), &Zs = *reinterpret_cast<Mat*>(buf + B * (B + 1)),
      &Ts = *reinterpret_cast<Mat*>(buf + 2 * B * (B + 1));
  __shared__ int bad;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const size_t N = a.N;
  const int row0 = bx * 256;
  const __amdgpu_buffer_rsrc_t ex = dev_buffer(a.ex, (size_t)a.nwg * B * B * sizeof(zc));
  if (t == 0) bad = 0;
  const zc empty = __builtin_bit_cast(zc, make_uint4(~0u, ~0u, ~0u, ~0u));
#pragma unroll
  for (int u = 0; u < NE; ++u) a.ex_next[(size_t)bx * B * B + t + 256 * u] = empty;
  zc tm[NE];
#pragma unroll
  for (int u = 0; u < NE; ++u) tm[u] = a.Tm[t + 256 * u];
  // this wave's 64 rows of M = V^H X
  d4 mr[TI][TI], mi[TI][TI];
#pragma unroll
  for (int x = 0; x < TI; ++x)
#pragma unroll
    for (int y = 0; y < TI; ++y) mr[x][y] = mi[x][y] = d4{0, 0, 0, 0};
  const int w0 = row0 + 64 * wave;
#pragma unroll
  for (int k0 = 0; k0 < 64; k0 += 4) {
    const int rr = w0 + k0 + lk;
    const bool on = rr < a.m;
    zc av[TI], xv[TI];
#pragma unroll
    for (int x = 0; x < TI; ++x) {
      av[x] = a.V[min(rr, a.m - 1) + N * (16 * x + lr)];
      xv[x] = a.X[min(rr, a.m - 1) + N * (16 * x + lr)];
      if (!on) av[x] = mkz(0, 0);
    }
    // conj(v) x = (vr xr + vi xi) + i (vr xi - vi xr)
#pragma unroll
    for (int x = 0; x < TI; ++x)
#pragma unroll
      for (int y = 0; y < TI; ++y) {
        mr[x][y] = mfma16x16x4(av[x].re, xv[y].re, mr[x][y]);
        mi[x][y] = mfma16x16x4(av[x].re, xv[y].im, mi[x][y]);
        mr[x][y] = mfma16x16x4(av[x].im, xv[y].im, mr[x][y]);
        mi[x][y] = mfma16x16x4(-av[x].im, xv[y].re, mi[x][y]);
      }
  }
#pragma unroll
  for (int x = 0; x < TI; ++x)
#pragma unroll
    for (int y = 0; y < TI; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[wave][(16 * x + lk + 4 * r) * B + 16 * y + lr] = mkz(mr[x][y][r], mi[x][y][r]);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NE; ++u) {
    const int e = t + 256 * u;
    const zc p = ((red[0][e] + red[1][e]) + red[2][e]) + red[3][e];
    st_buf(ex, (unsigned)((size_t)bx * B * B + e) * (unsigned)sizeof(zc), 0, p);
  }
  // while the sums are on their way: the rows of V and X that become W
  zc vv[4][B / 4], xx[4][TI][4];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) {
    const int rr = min(w0 + 16 * rt + lr, a.m - 1);
#pragma unroll
    for (int k = 0; k < B / 4; ++k) vv[rt][k] = a.V[rr + N * (4 * k + lk)];
#pragma unroll
    for (int x = 0; x < TI; ++x)
#pragma unroll
      for (int r = 0; r < 4; ++r) xx[rt][x][r] = a.X[rr + N * (16 * x + lk + 4 * r)];
  }
  lds_barrier();                               // red is read
#pragma unroll
  for (int u = 0; u < NE; ++u) Ts[(t + 256 * u) % B][(t + 256 * u) / B] = tm[u];
#pragma unroll
  for (int u = 0; u < NE; ++u) {
    const int e = t + 256 * u;
    zc s = mkz(0, 0);
    for (int wg0 = 0; wg0 < a.nwg; wg0 += 8) {
      zc v[8];
      for (int tries = 0;; ++tries) {
        bool ok = true;
        poll_again();
#pragma unroll
        for (int x = 0; x < 8; ++x)
          v[x] = ld_buf(ex, (unsigned)(min(wg0 + x, a.nwg - 1) * (B * B) + e) * (unsigned)sizeof(zc), 0);
#pragma unroll
        for (int x = 0; x < 8; ++x)
          ok = ok && !is_empty(v[x]);
        if (ok) break;
        if (tries > a.spin_limit ||
            ((tries & 255) == 255 && __hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
          bad = 1;
          __hip_atomic_store(a.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
      }
#pragma unroll
      for (int x = 0; x < 8; ++x)
        if (wg0 + x < a.nwg) s += v[x];
    }
    Ms[e / B][e % B] = s;
  }
  __syncthreads();
  if (bad) return;
  // Z = T^H M
#pragma unroll
  for (int u = 0; u < NE; ++u) {
    const int e = t + 256 * u, p = e / B, c = e % B;
    zc s = mkz(0, 0);
#pragma unroll 4
    for (int r = 0; r < B; ++r)
      if (r <= p) s = fma_conj(Ts[r][p], Ms[r][c], s);
    Zs[p][c] = s;
  }
  __syncthreads();
  // (V Z)^T by 16 x 16 tiles: MFMA rows over the columns of W, MFMA columns over its rows,
  // so that a lane's results lie next to its neighbours' in memory
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) {
    const int rr = w0 + 16 * rt + lr;
    d4 cr[TI], ci[TI];
#pragma unroll
    for (int x = 0; x < TI; ++x) cr[x] = ci[x] = d4{0, 0, 0, 0};
#pragma unroll
    for (int k0 = 0; k0 < B; k0 += 4) {
      const zc vk = vv[rt][k0 / 4];
#pragma unroll
      for (int x = 0; x < TI; ++x) {
        const zc zz = Zs[k0 + lk][16 * x + lr];
        cr[x] = mfma16x16x4(zz.re, vk.re, cr[x]);
        ci[x] = mfma16x16x4(zz.re, vk.im, ci[x]);
        cr[x] = mfma16x16x4(-zz.im, vk.im, cr[x]);
        ci[x] = mfma16x16x4(zz.im, vk.re, ci[x]);
      }
    }
    if (rr < a.m)
#pragma unroll
      for (int x = 0; x < TI; ++x)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const size_t at = rr + N * (16 * x + lk + 4 * r);
          const zc v = xx[rt][x][r];
          a.X[at] = mkz(v.re - 0.5 * cr[x][r], v.im - 0.5 * ci[x][r]);
        }
  }
}
template <int B>
__global__ __launch_bounds__(256, 2) void k_qr_w(QrWArgs a) {
  qr_w<B>(a, blockIdx.x);
}

// The 16 columns of the next panel, ahead of k_update_mul (5.4 us, latency-bound): A(:, 0:16) -= (V W^H + W V^H)(:, 0:16)
// on and below the diagonal, rows 0 .. m - 1 of the trailing matrix at A.  One 16 x 16 MFMA
// tile a wave, rows over the MFMA's columns as in k_her2k_full.
template <int B>
__device__ __forceinline__ void strip(zc* __restrict__ A, int ld, int m, int N, const zc* __restrict__ V,
                                      const zc* __restrict__ W, const int bx) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int r = bx * 64 + (threadIdx.x >> 6) * 16 + lr, rc = min(r, m - 1), c = min(lr, m - 1);
  zc av[B / 2], bv[B / 2], h[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) h[q] = A[(size_t)rc + (size_t)ld * min(lk + 4 * q, m - 1)];
#pragma unroll
  for (int s = 0; s < B / 2; ++s) {            // [V | W](c, k) and [W | V](r, k), k = 4 s + lk
    const int k = 4 * s + lk;
    av[s] = (k < B) ? V[(size_t)k * N + c] : W[(size_t)(k - B) * N + c];
    bv[s] = (k < B) ? W[(size_t)k * N + rc] : V[(size_t)(k - B) * N + rc];
  }
  d4 cr = {0, 0, 0, 0}, ci = {0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < B / 2; ++s) {
    cr = mfma16x16x4(av[s].re, bv[s].re, cr);
    ci = mfma16x16x4(av[s].im, bv[s].re, ci);
    cr = mfma16x16x4(av[s].im, bv[s].im, cr);
    ci = mfma16x16x4(-av[s].re, bv[s].im, ci);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int cc = lk + 4 * q;
    if (r < m && cc <= r) A[(size_t)r + (size_t)ld * cc] = clean_nan(mkz(h[q].re - cr[q], h[q].im + ci[q]));
  }
}
template <int B>
__global__ __launch_bounds__(256) void k_strip(zc* __restrict__ A, int ld, int m, int N, const zc* __restrict__ V,
                                               const zc* __restrict__ W) {
  strip<B>(A, ld, m, N, V, W, blockIdx.x);
}

// One pass over the trailing matrix A (m x m, lower triangle): the update of the panel before,
// A -= V W^H + W V^H (UPD), and the product of the updated values with this panel's Y, X = A Y.
// A workgroup takes 128 rows (block I) and 32 n columns of block J <= I, a wave 32 rows of
// them, and goes through the columns in steps of 32.  Every element is read and written once
// and serves both A(I, J) Y(J) -> X(I), accumulated over the steps, and A(I, J)^H Y(I) -> X(J),
// summed over the waves: the update, and with it the elements, is a 16 x 16 tile in the MFMA's
// result layout, which is its layout for an operand whose sum runs over the tile's
// columns, so the first product needs no data movement, and the second one transposes the
// tile through LDS.  The parts go to part[slot][col][row], the rows of block K in the slots
// 0 .. um_parts(K) - 1 (first the 4 (K + 1) / n column groups left of and in block K, then the
// row blocks from K on); k_um_sum adds them in order.
//
// 256 m^2 flops over 16 m^2 bytes and 2 m^2 of parts: at m = 14400 0.73 ms of the matrix cores
// and 0.73 ms of memory, and the kernel takes 1.15 ms (46 TFLOP/s, 3.7 TB/s with the operands
// that miss the L2; the matrix cores are busy 63 % of the time).  Two kernels, a product over
// 16 m^2 bytes and an update over 16 m^2, took 483 ms of a reduction at N = 14400 where this
// one and k_um_sum take 377, and 29 ms of one at N = 5184 (22 here).  Y ahead of the products
// that use it took 14 ms of that, their wave's priority 1 ms of a plan at N = 5184 (a higher
// priority for the loads instead cost 68 ms at 14400).  64 x 64 tiles, three waves per SIMD
// with spills, and an order of the tiles by XCD were no faster.
#define UM_R 128
__host__ __device__ inline int um_parts(int K, int n, int nt) { return 4 / n * (K + 1) + nt - K; }
template <int B, bool UPD>
__device__ __forceinline__ void update_mul(zc* __restrict__ A, int ld, int m, int N, const zc* __restrict__ V,
                                           const zc* __restrict__ W, const zc* __restrict__ Y, zc* __restrict__ part,
                                           int nt, int n, const int bx) {
  static_assert(B == 16, "one MFMA tile of Y columns");
  __shared__ zc tr[4][16 * 17];                // a wave's tile on its way through
  __shared__ zc red[4][2][4][64];              // the waves' parts of A^H Y
  const int ng = 4 / n, t = bx / ng;
  int ti = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
  while ((ti + 1) * (ti + 2) / 2 <= t) ++ti;
  while (ti * (ti + 1) / 2 > t) --ti;
  const int tj = t - ti * (ti + 1) / 2, g = tj * ng + bx % ng;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r0 = ti * UM_R + wave * 32;
  d4 ar[2], ai[2];                             // (A Y)^T of this wave's rows [y]
#pragma unroll
  for (int y = 0; y < 2; ++y) ar[y] = ai[y] = d4{0, 0, 0, 0};
#pragma unroll 1
  for (int u = 0; u < n; ++u) {
    const int c0 = (g * n + u) * 32;
    if (c0 >= m) break;
    int l = lane;
    __asm__ volatile("" : "+v"(l));            // no addresses kept from step to step
    const int lr = l & 15, lk = l >> 4;
    const unsigned lao = (unsigned)(lk * ld + lr);
    const bool on = r0 >= c0 && r0 < m;        // not above the diagonal or outside
    const bool diag = r0 == c0, edge = diag || r0 + 32 > m || c0 + 32 > m;
    zc* const Aw = A + (size_t)ld * c0 + r0;
    if (u > 0) lds_barrier();                  // the sums of the step before are taken
    if (on) {
      // h[x][y][2 e], [2 e + 1]: re and im of column c0 + 8 x + 4 e + lk, row r0 + 16 y + lr,
      // which are rows lk + 8 e and lk + 8 e + 4 of the MFMA's result: 16 bytes go to and come
      // from four registers next to each other.  The update is summed from zero and the
      // elements added to it, one rounding an element and panel instead of one a product.
      d4 h[4][2];
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) h[x][y] = d4{0, 0, 0, 0};
      zc ya[4][2], yb[2][4];                   // Y of the step's columns and of the rows
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int e = 0; e < 2; ++e) ya[x][e] = Y[(size_t)min(c0 + 8 * x + 4 * e + lk, m - 1) + (size_t)N * lr];
      if constexpr (UPD) {
        unsigned cc[4], rr[2];
#pragma unroll
        for (int x = 0; x < 4; ++x) cc[x] = (unsigned)(lk * N + min(c0 + 8 * x + (lr & 3) + 4 * (lr >> 3), m - 1));
#pragma unroll
        for (int y = 0; y < 2; ++y) rr[y] = (unsigned)(lk * N + min(r0 + 16 * y + lr, m - 1));
        const bool im = (lr & 4) != 0;
#pragma unroll
        for (int s = 0; s < B / 2; ++s) {      // h -= conj(a) b, a: [V | W](c, k), b: [W | V](r, k)
          const zc* pa = (s < B / 4) ? V + (size_t)(4 * s) * N : W + (size_t)(4 * s - B) * N;
          const zc* pb = (s < B / 4) ? W + (size_t)(4 * s) * N : V + (size_t)(4 * s - B) * N;
          double a1[4], a2[4];
          zc b[2];
#pragma unroll
          for (int y = 0; y < 2; ++y) b[y] = pb[rr[y]];
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const zc a = pa[cc[x]];
            a1[x] = im ? a.im : -a.re;
            a2[x] = im ? -a.re : -a.im;
          }
#pragma unroll
          for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) h[x][y] = mfma16x16x4(a1[x], b[y].re, h[x][y]);
#pragma unroll
          for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) h[x][y] = mfma16x16x4(a2[x], b[y].im, h[x][y]);
        }
      }
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const zc v = A[(size_t)min(r0 + 16 * y + lr, m - 1) + (size_t)ld * min(c0 + 8 * x + 4 * e + lk, m - 1)];
            h[x][y][2 * e] += v.re;
            h[x][y][2 * e + 1] += v.im;
          }
      if (edge) {                              // nothing above the diagonal or outside
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const int c = c0 + 8 * x + 4 * e + lk, r = r0 + 16 * y + lr;
              if (r >= m || c > r) h[x][y][2 * e] = h[x][y][2 * e + 1] = 0.0;
            }
      }
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int q = 0; q < 4; ++q) yb[y][q] = Y[(size_t)min(r0 + 16 * y + lk + 4 * q, m - 1) + (size_t)N * lr];
      // A Y: the sum runs over the columns.  The wave that has its operands goes before one
      // that still loads.
      __builtin_amdgcn_s_setprio(2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const zc* yv = ya[x];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
#pragma unroll
          for (int y = 0; y < 2; ++y) {
            ar[y] = mfma16x16x4(yv[e].re, h[x][y][2 * e], ar[y]);
            ai[y] = mfma16x16x4(yv[e].re, h[x][y][2 * e + 1], ai[y]);
          }
#pragma unroll
          for (int y = 0; y < 2; ++y) {
            ar[y] = mfma16x16x4(-yv[e].im, h[x][y][2 * e + 1], ar[y]);
            ai[y] = mfma16x16x4(yv[e].im, h[x][y][2 * e], ai[y]);
          }
        }
      }
      // A^H Y: the sum runs over the rows; the diagonal itself is in A Y already
      __builtin_amdgcn_sched_barrier(0);
      d4 br[2], bi[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) br[x] = bi[x] = d4{0, 0, 0, 0};
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        const zc* yv = yb[y];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            tr[wave][(lk + 4 * q) * 17 + lr] = mkz(h[2 * x + q / 2][y][2 * (q & 1)], h[2 * x + q / 2][y][2 * (q & 1) + 1]);
          if (diag && x == y && lane < 16) tr[wave][lane * 18] = mkz(0, 0);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const zc b = tr[wave][lr * 17 + lk + 4 * q];
            br[x] = mfma16x16x4(yv[q].re, b.re, br[x]);
            bi[x] = mfma16x16x4(yv[q].im, b.re, bi[x]);
            br[x] = mfma16x16x4(yv[q].im, b.im, br[x]);
            bi[x] = mfma16x16x4(-yv[q].re, b.im, bi[x]);
          }
        }
      }
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[wave][x][q][lane] = mkz(br[x][q], bi[x][q]);
      // the stores last: a later load's wait would wait for them too
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (UPD) {
        __asm__ volatile("" : "+v"(l));
        const int lr = l & 15, lk = l >> 4;
        const unsigned lao = (unsigned)(lk * ld + lr);
        auto put = [&](auto masked) {
#pragma unroll
          for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const int c = c0 + 8 * x + 4 * e + lk;
              zc* pc = Aw + (size_t)ld * (8 * x + 4 * e);
#pragma unroll
              for (int y = 0; y < 2; ++y)
                if (!decltype(masked)::value || (r0 + 16 * y + lr < m && c <= r0 + 16 * y + lr))
                  (pc + 16 * y)[lao] = mkz(h[x][y][2 * e], h[x][y][2 * e + 1]);
            }
        };
        if (edge) put(std::true_type{});
        else put(std::false_type{});
      }
    } else {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[wave][x][q][lane] = mkz(0, 0);
    }
    lds_barrier();
    const int row = c0 + 16 * (wave >> 1) + lr;
    zc* const pp = part + (size_t)(ng * (c0 / UM_R + 1) + ti - c0 / UM_R) * B * m + row;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int q = 2 * (wave & 1) + e;
      zc v = red[0][wave >> 1][q][lane];
#pragma unroll
      for (int o = 1; o < 4; ++o) v = v + red[o][wave >> 1][q][lane];
      if (row < m) pp[(size_t)(lk + 4 * q) * m] = v;
    }
  }
#pragma unroll
  for (int y = 0; y < 2; ++y) {
    const int row = r0 + 16 * y + (lane & 15);
    if (row < m)
#pragma unroll
      for (int q = 0; q < 4; ++q) part[((size_t)g * B + (lane >> 4) + 4 * q) * m + row] = mkz(ar[y][q], ai[y][q]);
  }
}
template <int B, bool UPD>
__global__ __launch_bounds__(256, 2) void k_update_mul(zc* __restrict__ A, int ld, int m, int N,
                                                       const zc* __restrict__ V, const zc* __restrict__ W,
                                                       const zc* __restrict__ Y, zc* __restrict__ part, int nt, int n) {
  update_mul<B, UPD>(A, ld, m, N, V, W, Y, part, nt, n, blockIdx.x);
}

// X(row, col) = the sum of the parts of k_update_mul, in slot order
template <int B>
__device__ __forceinline__ void um_sum(int m, int n, int nt, const zc* __restrict__ part, zc* __restrict__ X, int ldx,
                                       const int bx) {
  const size_t e = (size_t)bx * 256 + threadIdx.x;
  if (e >= (size_t)m * B) return;
  const int row = (int)(e % m), col = (int)(e / m);
  X[(size_t)row + (size_t)ldx * col] = clean_nan(strided_sum(part + e, (size_t)m * B, 0, um_parts(row / UM_R, n, nt), 1, mkz(0, 0)));
}
template <int B>
__global__ __launch_bounds__(256) void k_um_sum(int m, int n, int nt, const zc* __restrict__ part, zc* __restrict__ X,
                                                int ldx) {
  um_sum<B>(m, n, nt, part, X, ldx, blockIdx.x);
}

__global__ void k_fill_empty(zc* p, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = __builtin_bit_cast(zc, make_uint4(~0u, ~0u, ~0u, ~0u));
}

// ---------------------------------------------------------------------------
// stage 2: bulge chasing
// ---------------------------------------------------------------------------
template <int B>
struct ChaseDim {
  static constexpr int SW = (B == 16) ? 3 : 2;   // sweeps per workgroup, one wave each
  static constexpr int R = (B == 16) ? 4 : 2;    // LDS slots per boundary between sweeps
  static constexpr int NC = B * B / 64;          // columns per thread
  static constexpr int P = B + 1;                // column length of a slot
  static constexpr int G = 2 * B * P;            // offset of its tracked rows
  static constexpr int SLOT = G + 6 * P;
};

struct ChaseArgs {
  zc* BD;            // [N][2 B + 1]
  int N;
  zc* gc;            // nrhs x N (conjugated tracked vectors)
  int nrhs;
  int* prog;         // [group] tasks that the group's last sweep has finished
  int* ctl;          // [0] error flag, [32] next group to claim
  long long spin_limit;   // polls of a counter in memory
  int lds_limit;          // polls of a counter in LDS
  zc* Vc;            // the reflectors kept (VEC): row r of sweep s at (N - 1 - r) + ld (N - 1 - s)
  int ld;
  zc* tau;           // [sweep][task], kt tasks
  int kt;
};

__host__ __device__ inline int chase_ntasks(int N, int b, int s) { return 1 + (N - 2 - s) / b; }

// The chase keeps row r of a block in the lanes r (64 / B) + (column group), so that rows
// lie on the lane's high bits.  Sum over the rows (every lane ends with it): both halves,
// both rows of 16, rotations by 8 and 4 in a row of 16, and for B = 32 lane pairs ^2.
template <int B>
__device__ inline double row_group_sum(double x) {
  x = add32(x, x);
  x = add16(x, x);
  x += dpp_d<0x128>(x);                        // row_ror:8
  x += dpp_d<0x124>(x);                        // row_ror:4
  if constexpr (B == 32) x += dpp_d<0x4E>(x);  // quad_perm [2, 3, 0, 1]
  return x;
}
template <int B>
__device__ inline zc row_group_sum(zc x) {
  return mkz(row_group_sum<B>(x.re), row_group_sum<B>(x.im));
}

// Column sums of NC values: halved over the two highest row bits by the swaps (the lanes
// of row quarter u keep columns u NC / 4 ..), then summed over the row bits left
template <int B, int NC>
__device__ inline void col_sums(zc (&v)[NC]) {
#pragma unroll
  for (int q = 0; q < NC / 2; ++q) v[q] = mkz(add32(v[q].re, v[q + NC / 2].re), add32(v[q].im, v[q + NC / 2].im));
#pragma unroll
  for (int q = 0; q < NC / 4; ++q) {
    zc x = mkz(add16(v[q].re, v[q + NC / 4].re), add16(v[q].im, v[q + NC / 4].im));
    x += dpp_z<0x128>(x);
    x += dpp_z<0x124>(x);
    if constexpr (B == 32) x += dpp_z<0x4E>(x);
    v[q] = x;
  }
}

// sum over the column groups of a wave (the lane's low bits)
template <int B>
__device__ inline zc lane_group_sum(zc x) {
  x += dpp_z<0xB1>(x);
  if constexpr (B == 16) x += dpp_z<0x4E>(x);
  return x;
}

__device__ inline double first_lane(double x) {
  const unsigned long long v = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = __builtin_amdgcn_readfirstlane((int)v), hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ inline zc first_lane(zc v) { return mkz(first_lane(v.re), first_lane(v.im)); }

// a flag in LDS: LDS operations of a wave execute in order, so a wave's stores before
// lds_set are seen by a wave whose lds_get returned the value, and its loads are done
__device__ inline void lds_set(int* f, int v) {
  __asm__ volatile("" ::: "memory");
  __hip_atomic_store(f, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  __asm__ volatile("" ::: "memory");
}
__device__ inline int lds_get(int* f) {
  const int v = __builtin_amdgcn_readfirstlane(__hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
  __asm__ volatile("" ::: "memory");
  return v;
}

// Band -> tridiagonal.  A workgroup takes SW consecutive sweeps at a time (a group, claimed
// in order from a counter), one wave each, and one wave more that loads.  Task k of sweep s
// needs the tasks <= k + 1 of sweep s - 1 (the later ones touch only rows below).  The
// blocks move from sweep to sweep through rings of LDS slots with a counter of tasks
// written and one of tasks read, so that no wave waits at a barrier; only the group's ends
// meet global memory: the loader fetches what the sweep before the group left, the last
// sweep stores its blocks and publishes the count of a task one task later, when its stores
// are complete (device-scope accesses, no cache maintenance).  Every wait is bounded, and
// past the limit the error flag makes every workgroup return.
//
// An LDS slot holds the window [left block | diagonal block] of a task, element (r, c) at
// (c - 1) P + r, column 0 at (2B - 1) P + r; of the diagonal block the lower triangle counts
// (what lies above it is written and not read).  The tracked rows follow.  The next sweep
// reads its blocks one row and column on: rows 1 .. B - 1 of the slot, and for its last row
// row 0 of the slot of the next task (in the left block zero but for its last column: row B
// of every slot's first columns stays zero).
//
// What bounds it is the chain of 2 N dependent tasks, so a task is arranged for its latency,
// and that is its instruction count (a SIMD issues a wave's instructions four to five cycles
// apart, dependent or not) and its LDS traffic (about 70 cycles a round trip, 40 for every
// 16-byte access of a wave): lane (r, hg) keeps row r and NC columns of the two blocks in
// registers, exchanges go by swaps and DPP, and a row vector gets to the columns through LDS.
// Measured at N = 5184: 21.3 ms for band 16 (4.1 us a sweep, about 3600 cycles a task),
// 50.8 ms for band 32, whose wave holds four times the elements; a sweep per workgroup of
// four waves that met at barriers and moved every block through memory took 62 ms (band 32,
// 12 us a sweep).  With eight waves a sweep and barriers, band 16 took 28 ms.
template <int B, bool VEC>
__device__ __forceinline__ void chase(const ChaseArgs& a) {
  typedef ChaseDim<B> C;
  constexpr int SW = C::SW, R = C::R, NC = C::NC, P = C::P;
  constexpr int GPW = 64 / B;                  // column groups
  constexpr int NV = (6 + GPW - 1) / GPW;      // tracked vectors per column group: hg, hg + GPW, ..
  constexpr int LB = 2 * B + 1;
  constexpr unsigned CB = (LB - 1) * (unsigned)sizeof(zc);   // bytes from (r, c) to (r, c + 1) of the band
  __shared__ zc slot[SW][R][C::SLOT];          // boundary i: what sweep i of the group reads
  __shared__ zc xw[SW][B], zw[SW][B];          // a wave's own: v, then tau y, of every row; v^H O
  __shared__ int wrote[SW], read[SW];          // tasks written to and read from a boundary's slots
  __shared__ int group, bad;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int N = a.N, nrhs = a.nrhs;
  int* const err = a.ctl;
  const __amdgpu_buffer_rsrc_t bd = dev_buffer(a.BD, (size_t)N * LB * sizeof(zc));
  const __amdgpu_buffer_rsrc_t gb = dev_buffer(a.gc, (size_t)nrhs * N * sizeof(zc));
  for (int i = threadIdx.x; i < SW * R * C::SLOT; i += (SW + 1) * 64) (&slot[0][0][0])[i] = mkz(0, 0);
  if (threadIdx.x == 0) bad = 0;
  // past a limit: the flags for this workgroup's waves (there before this one leaves) and
  // for the other workgroups
  auto give_up = [&]() {
    lds_set(&bad, 1);
    __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  // wait for *f >= need; seen keeps the last count read
  auto wait_lds = [&](int* f, int need, int& seen) {
    for (int n = 0; seen < need; ++n) {
      seen = lds_get(f);
      if (seen >= need) break;
      if (lds_get(&bad)) return false;
      if (n > a.lds_limit) {
        give_up();
        return false;
      }
    }
    return true;
  };
  for (;;) {
    __syncthreads();
    // a wave that gave up has left (wave 0, which claims the groups, perhaps among them), so
    // the others do not start another group
    if (lds_get(&bad)) return;
    if (threadIdx.x == 0) group = atomicAdd(a.ctl + 32, 1);
    if ((int)threadIdx.x < SW) wrote[threadIdx.x] = read[threadIdx.x] = 0;
    __syncthreads();
    const int gidx = __builtin_amdgcn_readfirstlane(group);
    const int s0 = gidx * SW;
    if (s0 > N - 2) return;
    // each role takes its own opaque copy of the lane, so that the roles' addresses are not
    // kept in registers side by side
    int lane = threadIdx.x & 63;
    __asm__ volatile("" : "+v"(lane));
    if (wave == SW) {
      // ---- loader: the tasks of sweep s0 - 1 (s0 = 0: blocks of the band) ----------------
      const int r = lane / GPW, hg = lane % GPW, c0 = hg * NC;
      const unsigned bo = (unsigned)(c0 * (LB - 1) + r) * (unsigned)sizeof(zc);
      const int w0 = (hg == 0) ? (2 * B - 1) * P : (c0 - 1) * P;   // column c0 of the left block in a slot
      const int ntp = chase_ntasks(N, B, s0 - 1);
      int have = (gidx == 0) ? ntp : 0, seen = 0;
      for (int k = 0; k < ntp; ++k) {
        for (long long n = 0; have < k + 1; ++n) {
          have = __builtin_amdgcn_readfirstlane(
              __hip_atomic_load(a.prog + gidx - 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
          if (have >= k + 1) break;
          if (n > a.spin_limit ||
              ((n & 63) == 63 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
            give_up();
            return;
          }
        }
        // past the last row and above the diagonal something else is read and not used
        const int st = s0 + k * B;
        const unsigned sb = (unsigned)st * LB * (unsigned)sizeof(zc);
        zc o[NC], d[NC], g[NV];
#pragma unroll
        for (int q = 0; q < NC; ++q) o[q] = ld_buf(bd, bo + q * CB, k > 0 ? sb - B * CB : 0u);
#pragma unroll
        for (int q = 0; q < NC; ++q) d[q] = ld_buf(bd, bo + q * CB, sb);
#pragma unroll
        for (int u = 0; u < NV; ++u)
          if (u * GPW < nrhs)
            g[u] = ld_buf(gb, (unsigned)((hg + u * GPW) * N + r) * (unsigned)sizeof(zc), (unsigned)st * (unsigned)sizeof(zc));
        if (!wait_lds(&read[0], k + 1 - R, seen)) return;
        zc* const sl = slot[0][k & (R - 1)] + r;
#pragma unroll
        for (int q = 0; q < NC; ++q) sl[q == 0 ? w0 : (c0 + q - 1) * P] = o[q];
#pragma unroll
        for (int q = 0; q < NC; ++q) sl[(c0 + q + B - 1) * P] = d[q];
#pragma unroll
        for (int u = 0; u < NV; ++u)
          if (hg + u * GPW < nrhs) sl[C::G + (hg + u * GPW) * P] = g[u];
        lds_set(&wrote[0], k + 1);
      }
      continue;
    }
    // ---- sweep s ------------------------------------------------------------------------
    const int s = s0 + wave;
    if (s > N - 2) continue;
    const int r = lane / GPW, hg = lane % GPW, c0 = hg * NC;
    const unsigned bo = (unsigned)(c0 * (LB - 1) + r) * (unsigned)sizeof(zc);
    const bool last = wave == SW - 1 || s == N - 2;
    const int nt = chase_ntasks(N, B, s), ntp = chase_ntasks(N, B, s - 1);
    const int w0 = (hg == 0) ? (2 * B - 1) * P : (c0 - 1) * P;   // column c0 of the left block in a slot
    const bool lastrow = r == B - 1, corner = lastrow && hg == GPW - 1;
    int seen_w = 0, seen_r = 0;
    zc* const xv = xw[wave];
    zc taup = mkz(0, 0);
    zc vp[NC];                                 // previous reflector at this thread's columns
#pragma unroll
    for (int q = 0; q < NC; ++q) vp[q] = mkz(0, 0);
    auto publish = [&](int k) {                // the stores of task k - 1 are complete
      __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (lane == 0) __hip_atomic_store(a.prog + gidx, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    for (int k = 0; k < nt; ++k) {
      if (!wait_lds(&wrote[wave], min(k + 2, ntp), seen_w)) return;
      const int st = s + 1 + k * B;            // rows st .. st + len - 1
      const int len = min(B, N - st);
      const bool rin = r < len;
      const zc* const s1 = slot[wave][k & (R - 1)];
      const zc* const s2 = slot[wave][(k + 1) & (R - 1)];
      zc O[NC], D[NC], g[NV];
#pragma unroll
      for (int q = 0; q < NC; ++q)
        O[q] = *(q == NC - 1 && corner ? s2 + (2 * B - 1) * P : s1 + (c0 + q) * P + r + 1);
      const zc* const dr = lastrow ? s2 : s1 + B * P + r + 1;       // D(r, 0)
      const zc* const dc = s1 + (r + B) * P + 1;                    // D(0, r)
#pragma unroll
      for (int q = 0; q < NC; ++q) {           // above the diagonal: the conjugate of (c, r)
        const int c = c0 + q;
        D[q] = *(c <= r ? dr + c * P : (q == NC - 1 && hg == GPW - 1) ? s2 + r * P : dc + c);
      }
      // column 0 of the left block (k = 0: column s of the matrix; there is no left block
      // then, and nothing formed from O is used)
      zc x0 = *(k > 0 ? s1 + r + 1 : lastrow ? s2 + (2 * B - 1) * P : s1 + (B - 1) * P + r + 1);
#pragma unroll
      for (int u = 0; u < NV; ++u)
        if (u * GPW < nrhs) g[u] = (lastrow ? s2 : s1 + r + 1)[C::G + min(hg + u * GPW, 5) * P];
      lds_set(&read[wave], k + 1);
#pragma unroll
      for (int q = 0; q < NC; ++q)
        if (c0 + q > r) D[q].im = -D[q].im;
      if (len < B) {                           // the last task: nothing past row N - 1
        if (!rin) x0 = mkz(0, 0);
#pragma unroll
        for (int q = 0; q < NC; ++q) {
          if (!rin) O[q] = mkz(0, 0);
          if (!(rin && c0 + q < len)) D[q] = mkz(0, 0);
        }
#pragma unroll
        for (int u = 0; u < NV; ++u)
          if (!rin) g[u] = mkz(0, 0);
      }
      if (k > 0) {
        // (i) O -= tau' (O v') v'^H (v'(0) = 1)
        zc w = mkz(0, 0);
#pragma unroll
        for (int q = 0; q < NC; ++q) w = fma_z(O[q], vp[q], w);
        const zc tw = taup * lane_group_sum<B>(w);
#pragma unroll
        for (int q = 0; q < NC; ++q) O[q] = fnma_zc(tw, vp[q], O[q]);
        x0 -= tw;
        if (last) publish(k);
      }
      // (ii) the reflector of x0, at the columns too
      const double xn2 = row_group_sum<B>((r > 0) ? norm2(x0) : 0.0);
      zc beta, tau, scale;
      larfg_fast(first_lane(x0), xn2, beta, tau, scale);
      const zc vr = (r == 0) ? mkz(1, 0) : scale * x0;
      if (hg == 0) xv[r] = vr;
      if constexpr (VEC) {
        if (hg == 0 && rin) a.Vc[(size_t)(N - 1 - st - r) + (size_t)a.ld * (N - 1 - s)] = vr;
        if (lane == 0) a.tau[(size_t)s * a.kt + k] = tau;
      }
#pragma unroll
      for (int q = 0; q < NC; ++q) vp[q] = xv[c0 + q];
      // (iii) z = v^H O, row quarter u summing columns u NC / 4 ..
      zc tq[NC];
#pragma unroll
      for (int q = 0; q < NC; ++q) tq[q] = fma_conj(vr, O[q], mkz(0, 0));
      col_sums<B, NC>(tq);
      if (r % (B / 4) == 0) {
#pragma unroll
        for (int q = 0; q < NC / 4; ++q) zw[wave][c0 + (r / (B / 4)) * (NC / 4) + q] = tq[q];
      }
      // (iv) D <- H^H D H: y = D v, w = tau y - |tau|^2 (v^H y) / 2 v, D -= v w^H + w v^H
      zc y = mkz(0, 0);
#pragma unroll
      for (int q = 0; q < NC; ++q) y = fma_z(D[q], vp[q], y);
      y = lane_group_sum<B>(y);
      const zc ty = tau * y;
      if (hg == 0) xv[r] = ty;
      const double kap = 0.5 * norm2(tau) * row_group_sum<B>(fma(vr.re, y.re, vr.im * y.im));
      const zc wr = mkz(fma(-kap, vr.re, ty.re), fma(-kap, vr.im, ty.im));
      const zc ctv = conj(tau) * vr;
      // O(:, 1:) -= conj(tau) v z
#pragma unroll
      for (int q = 0; q < NC; ++q) O[q] = fnma_z(ctv, zw[wave][c0 + q], O[q]);
      if (hg == 0) O[0] = (r == 0) ? beta : mkz(0, 0);
#pragma unroll
      for (int q = 0; q < NC; ++q) {
        const zc tyc = xv[c0 + q];
        const zc wc = mkz(fma(-kap, vp[q].re, tyc.re), fma(-kap, vp[q].im, tyc.im));
        D[q] = fnma_zc(wr, vp[q], fnma_zc(vr, wc, D[q]));
      }
      // (v) tracked vectors: gc -= conj(tau) v (v^H gc)
#pragma unroll
      for (int q = 0; q < NV; ++q)
        if (q * GPW < nrhs) g[q] = fnma_z(ctv, row_group_sum<B>(fma_conj(vr, g[q], mkz(0, 0))), g[q]);
      if (k == 0 && r == 0) {
        // finished: the subdiagonal of column s, the diagonal and tracked rows of s + 1
        if (hg == 0) {
          st_dev(a.BD + (size_t)s * LB + 1, beta);
          st_dev(a.BD + (size_t)(s + 1) * LB, D[0]);
        }
#pragma unroll
        for (int q = 0; q < NV; ++q)
          if (hg + q * GPW < nrhs) st_dev(a.gc + (size_t)(hg + q * GPW) * N + s + 1, g[q]);
      }
      if (last) {
        if (rin) {
          const unsigned sb = (unsigned)st * LB * (unsigned)sizeof(zc);
#pragma unroll
          for (int q = 0; q < NC; ++q)
            if (c0 + q <= r) st_buf(bd, bo + q * CB, sb, D[q]);
          if (k > 0) {
#pragma unroll
            for (int q = 0; q < NC; ++q) st_buf(bd, bo + q * CB, sb - B * CB, O[q]);
          }
#pragma unroll
          for (int q = 0; q < NV; ++q)
            if (hg + q * GPW < nrhs)
              st_buf(gb, (unsigned)((hg + q * GPW) * N + r) * (unsigned)sizeof(zc), (unsigned)st * (unsigned)sizeof(zc), g[q]);
        }
      } else {
        const int nx = min(wave + 1, SW - 1);
        if (!wait_lds(&read[nx], k + 1 - R, seen_r)) return;
        zc* const so = slot[nx][k & (R - 1)] + r;
#pragma unroll
        for (int q = 0; q < NC; ++q) {
          so[q == 0 ? w0 : (c0 + q - 1) * P] = O[q];
          so[(c0 + q + B - 1) * P] = D[q];
        }
#pragma unroll
        for (int q = 0; q < NV; ++q)
          if (hg + q * GPW < nrhs) so[C::G + (hg + q * GPW) * P] = g[q];
        lds_set(&wrote[nx], k + 1);
      }
      taup = tau;
    }
    if (last) publish(nt);
  }
}
template <int B, bool VEC>
__global__ __launch_bounds__((ChaseDim<B>::SW + 1) * 64, 1) void k_chase(ChaseArgs a) {
  chase<B, VEC>(a);
}

// ---------------------------------------------------------------------------
// One matrix's arguments, and sets of matrices
// ---------------------------------------------------------------------------
// The arguments that do not change from panel to panel (COMPLEX*16, band 16); the launches of
// panel p take theirs from these, on the host for one matrix, on the device for a set
struct BandItem {
  zc* H;
  int ld, N, nrhs;
  zc *V, *X, *V2, *X2;   // of the even and of the odd panels
  zc *Y, *T, *gc, *part;
  zc* ex;                // exchange slots of the even, then of the odd panels
  size_t exn, wo;        // slots of one parity; where k_qr_w's begin
  int exw;               // workgroups that they hold
  int* err;
  int spin;
  zc* tau1;
  ChaseArgs chase;
};

// rows of the trailing matrix of panel p; a panel has at least two
__host__ __device__ inline int panel_rows(const BandItem& t, int p) { return t.N - 16 * (p + 1); }
__host__ __device__ inline int panel_wgs(const BandItem& t, int p) { return (panel_rows(t, p) + PR - 1) / PR; }
__host__ __device__ inline bool last_panel(const BandItem& t, int p) { return panel_rows(t, p + 1) < 2; }
__host__ __device__ inline zc* trailing(const BandItem& t, int p) { return t.H + (size_t)16 * (p + 1) * (t.ld + 1); }
__host__ __device__ inline zc* panel_v(const BandItem& t, int p) { return p & 1 ? t.V2 : t.V; }
__host__ __device__ inline zc* panel_x(const BandItem& t, int p) { return p & 1 ? t.X2 : t.X; }
__host__ __device__ inline QrPanelArgs qr_panel_args(const BandItem& t, int p) {
  const int m = panel_rows(t, p);
  return QrPanelArgs{t.H, t.ld, t.N, 16 * p, 16 * (p + 1), m, m > 16 ? 16 : m - 1, panel_v(t, p), t.Y, t.T, t.gc, t.nrhs,
                     t.ex + (p & 1) * t.exn, t.ex + ((p + 1) & 1) * t.exn, t.exw + 1, panel_wgs(t, p), t.err + 8, t.spin,
                     t.tau1 ? t.tau1 + 16 * p : nullptr};
}
__host__ __device__ inline QrWArgs qr_w_args(const BandItem& t, int p) {
  return QrWArgs{panel_rows(t, p), t.N, panel_v(t, p), t.T, panel_x(t, p), t.ex + (p & 1) * t.exn + t.wo,
                 t.ex + ((p + 1) & 1) * t.exn + t.wo, panel_wgs(t, p), t.err + 8, t.spin};
}
// steps of k_update_mul: fewer parts with more steps, more workgroups with fewer (at these
// sizes about 1200 workgroups either way, 512 run at once; lines at half and one and a half
// times these sizes measured within 1 %)
constexpr int UM_4 = 6144, UM_2 = 3072;
__host__ __device__ inline int um_steps(int m) { return m > UM_4 ? 4 : m > UM_2 ? 2 : 1; }
__host__ __device__ inline int um_blocks(int m) {
  const int nt = (m + UM_R - 1) / UM_R;
  return 4 / um_steps(m) * (nt * (nt + 1) / 2);
}

// One launch for a set: workgroup b belongs to the matrix whose range [pre[i], pre[i + 1])
// holds it and runs the one matrix's kernel body on that matrix's arguments with block index
// b - pre[i], so that every matrix goes through the arithmetic of its own reduction.  Bound by
// the chains of the largest member as long as the others fit beside it: eight matrices of
// N = 576 .. 2304 take 56 us a panel, 39 us an update and product and 9.3 ms the chase.
constexpr int kSetMax = 64;
struct BandSlots {
  const BandItem* items;       // of slot 0 on
  int n;
  int pre[kSetMax + 1];
};
__device__ inline int set_slot(const BandSlots& S, int b) {
  int lo = 0, hi = S.n;        // pre[lo] <= b < pre[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (S.pre[mid] <= b) lo = mid;
    else hi = mid;
  }
  return lo;
}
__global__ __launch_bounds__(256) void k_strip_s(BandSlots S, int p) {
  const int i = set_slot(S, blockIdx.x);
  const BandItem& t = S.items[i];
  strip<16>(trailing(t, p - 1), t.ld, panel_rows(t, p - 1), t.N, panel_v(t, p - 1), panel_x(t, p - 1), (int)blockIdx.x - S.pre[i]);
}
__global__ __launch_bounds__(256, 2) void k_qr_panel_s(BandSlots S, int p) {
  const int i = set_slot(S, blockIdx.x);
  qr_panel<16>(qr_panel_args(S.items[i], p), (int)blockIdx.x - S.pre[i]);
}
template <bool UPD>
__global__ __launch_bounds__(256, 2) void k_update_mul_s(BandSlots S, int p) {
  const int i = set_slot(S, blockIdx.x);
  const BandItem& t = S.items[i];
  const int m = panel_rows(t, p);
  update_mul<16, UPD>(trailing(t, p), t.ld, m, t.N, panel_v(t, p + 1) + 16, panel_x(t, p + 1) + 16, t.Y, t.part,
                      (m + UM_R - 1) / UM_R, um_steps(m), (int)blockIdx.x - S.pre[i]);
}
__global__ __launch_bounds__(256) void k_um_sum_s(BandSlots S, int p) {
  const int i = set_slot(S, blockIdx.x);
  const BandItem& t = S.items[i];
  const int m = panel_rows(t, p);
  um_sum<16>(m, um_steps(m), (m + UM_R - 1) / UM_R, t.part, panel_x(t, p), t.N, (int)blockIdx.x - S.pre[i]);
}
__global__ __launch_bounds__(256, 2) void k_qr_w_s(BandSlots S, int p) {
  const int i = set_slot(S, blockIdx.x);
  qr_w<16>(qr_w_args(S.items[i], p), (int)blockIdx.x - S.pre[i]);
}
__global__ __launch_bounds__(256, 4) void k_her2k_s(BandSlots S, int p) {
  const int i = set_slot(S, blockIdx.x);
  const BandItem& t = S.items[i];
  her2k_tile<zc, 16>(t.H, t.ld, panel_rows(t, p), 16 * (p + 1), t.N, panel_v(t, p), panel_x(t, p), (int)blockIdx.x - S.pre[i]);
}
__global__ void k_band_extract_s(BandSlots S) {
  const int i = set_slot(S, blockIdx.x);
  const BandItem& t = S.items[i];
  band_extract(t.H, t.ld, t.N, 16, 33, t.chase.BD, (int)blockIdx.x - S.pre[i]);
}
__global__ __launch_bounds__((ChaseDim<16>::SW + 1) * 64, 1) void k_chase_s(BandSlots S) {
  const ChaseArgs a = S.items[set_slot(S, blockIdx.x)].chase;
  chase<16, false>(a);
}

// d, e of the tridiagonal from the band; g = conj(gc).  After a stalled wait the band is
// unfinished and may hold anything: status is set and what follows works on zeros.
__global__ void k_band_finish(const zc* __restrict__ BD, int N, int LB, double* __restrict__ d, double* __restrict__ e,
                              const zc* __restrict__ gc, zc* __restrict__ g, int nrhs, const int* __restrict__ err,
                              int* __restrict__ status) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  const bool bad = err[0] || err[8];
  if (j == 0 && status && bad) status[0] |= 1 << WTB_ERR_EIG | kStalled;
  if (j >= N) return;
  d[j] = bad ? 0.0 : BD[(size_t)j * LB].re;
  e[j] = (!bad && j + 1 < N) ? BD[(size_t)j * LB + 1].re : 0.0;
  for (int r = 0; r < nrhs; ++r) g[(size_t)r * N + j] = bad ? mkz(0, 0) : conj(gc[(size_t)r * N + j]);
}

// X = Q2 Z: the chase's reflectors, sweeps last to first, onto columns kept in LDS.  Bound by
// the vector ALU: 8 N^2 flops a column as short dot products.  The wpc waves of a pair of
// columns take its 64-row pieces (four reflectors of B rows) in turn, lane = row; the four
// sums of a piece's two columns share their reduction over the 16 lanes (one column a wave
// took 3.3 ms where two take 2.5, N = 1290 with all vectors).  v and tau of a wave's next
// pieces are loaded while it works on the present ones, SB sweeps ahead where few pieces
// make a sweep short (288 vectors of N = 1000: 0.45 ms, 3.5 with one sweep ahead), and a
// barrier that leaves those loads in flight ends a sweep.
struct ChaseBackArgs {
  const zc* Vc;
  int ld;
  const zc* tau;
  int kt, N;
  const double* Z;       // N x ., columns c0 ..
  int c0, m;
  zc* X;
  int ldx, pairs, wpc;   // pairs of columns of a workgroup, waves of a pair
};
template <int B, int U, int SB>
__global__ __launch_bounds__(768) void k_chase_back(ChaseBackArgs a) {
  static_assert(B == 16, "a reflector on a row of 16 lanes");
  extern __shared__ zc xcol[];
  const int N = a.N, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int pair = wave / a.wpc, part = wave % a.wpc, c = 2 * (blockIdx.x * a.pairs + pair);
  const bool on = c < a.m, two = c + 1 < a.m;
  zc* const x0 = xcol + (size_t)2 * pair * N;
  zc* const x1 = x0 + N;
  for (int r = part * 64 + lane; r < N; r += a.wpc * 64) {
    x0[r] = mkz(on ? a.Z[(size_t)r + (size_t)N * (a.c0 + c)] : 0.0, 0.0);
    x1[r] = mkz(two ? a.Z[(size_t)r + (size_t)N * (a.c0 + c + 1)] : 0.0, 0.0);
  }
  const bool h8 = (lane & 8) != 0, h4 = (lane & 4) != 0;
  zc v[SB][U], t[SB][U], vn[SB][U], tn[SB][U];
  // pieces part + wpc (u0 .. u0 + U - 1) of sweeps s, s - 1, .. (SB of them)
  auto load = [&](int s, int u0, zc (&lv)[SB][U], zc (&lt)[SB][U]) {
#pragma unroll
    for (int h = 0; h < SB; ++h)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int o = 64 * (part + a.wpc * (u0 + u)) + lane, r = s - h + 1 + o;
        const bool ok = s >= h && r < N;
        lv[h][u] = ok ? a.Vc[(size_t)(N - 1 - r) + (size_t)a.ld * (N - 1 - s + h)] : mkz(0, 0);
        lt[h][u] = ok ? a.tau[(size_t)(s - h) * a.kt + o / B] : mkz(0, 0);
      }
  };
  load(N - 2, 0, v, t);
  lds_barrier();
  for (int s = N - 2; s >= 0; s -= SB) {
    for (int u0 = 0;; u0 += U) {
      const bool more = SB == 1 && part + a.wpc * (u0 + U) < (N - 1 - s + 63) / 64;
      if (more) load(s, u0 + U, vn, tn);
      else if (s >= SB) load(s - SB, 0, vn, tn);
#pragma unroll
      for (int h = 0; h < SB; ++h) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int rp = s - h + 1 + 64 * (part + a.wpc * (u0 + u)), r = rp + lane;
          if (s < h || rp >= N) break;
          const zc xa = x0[min(r, N - 1)], xb = x1[min(r, N - 1)];
          const zc da = fma_conj(v[h][u], xa, mkz(0, 0)), db = fma_conj(v[h][u], xb, mkz(0, 0));
          // the four sums over the 16 lanes: lanes with bit 8 keep xb's, with bit 4 the
          // imaginary part, two more steps, then a lane of each quarter gives its sum back
          const zc keep = h8 ? db : da;
          zc d = h8 ? da : db;
          d = keep + dpp_z<0x128>(d);            // row_ror:8
          double e = h4 ? d.im : d.re;
          const double f = h4 ? d.re : d.im;
          e += xchg<4>(f);
          e += dpp_d<0x4E>(e);                   // quad_perm ^2, ^1
          e += dpp_d<0xB1>(e);
          const zc sa = mkz(dpp_d<0x150>(e), dpp_d<0x154>(e));       // row_newbcast of lanes 0, 4, 8, 12
          const zc sb = mkz(dpp_d<0x158>(e), dpp_d<0x15C>(e));
          if (r < N) {
            x0[r] = fnma_z(t[h][u] * sa, v[h][u], xa);
            x1[r] = fnma_z(t[h][u] * sb, v[h][u], xb);
          }
        }
        if (h < SB - 1) lds_barrier();
      }
#pragma unroll
      for (int h = 0; h < SB; ++h)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          v[h][u] = vn[h][u];
          t[h][u] = tn[h][u];
        }
      if (!more) break;
    }
    lds_barrier();
  }
  for (int r = part * 64 + lane; r < N; r += a.wpc * 64) {
    if (on) a.X[(size_t)r + (size_t)a.ldx * c] = x0[r];
    if (two) a.X[(size_t)r + (size_t)a.ldx * (c + 1)] = x1[r];
  }
}

__global__ void k_zero_ints(int* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// the exchange slots of one panel parity: k_qr_panel's, then k_qr_w's
template <int B>
static size_t qr_ex_elems(int nwg_max) {
  return qr_slots<B>(nwg_max) + (size_t)nwg_max * B * B;
}

int band_panel_rows() { return QP_WG * PR + 16; }

// The panels' workgroups that the current device holds at once
static int band_resident() {
  static std::atomic<int> known[64];           // + 1; 0: not looked up yet
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (const int k = known[dev].load(std::memory_order_relaxed)) return k - 1;
  int cus = 0, n = 1 << 20;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  for (const void* k : {(const void*)k_qr_panel<16>, (const void*)k_qr_w<16>, (const void*)k_qr_panel_s, (const void*)k_qr_w_s}) {
    int per = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, 256, 0) != hipSuccess) return 0;
    n = std::min(n, per);
  }
  known[dev].store(cus * n + 1, std::memory_order_relaxed);
  return cus * n;
}

// Most workgroups of a panel's launch: an eighth of those, so that the launches of eight
// streams (a set's lanes, or several threads' plans; a process has four hardware queues by
// default) all get theirs, and at most QP_WG.  256 compute units hold two of these workgroups
// each: 64.  A chase beside them takes the LDS of one of the two from up to 176 units, but
// ends by itself.  More launches than that at once, or another process's, can keep each other
// waiting; then a wait ends at its limit and the caller solves by the one-stage form
// (kStalled).
static int band_panel_wg() { return std::min(QP_WG, band_resident() / 8); }

bool band_panel_fits(int N) { return N <= band_panel_rows() && (N - 16 + PR - 1) / PR <= band_panel_wg(); }

// whether one-launch panels may run, which keep the V and W of the panel before
static bool second_panel(int N, int b) { return b == 16 && N <= band_panel_rows(); }

// slots of the partial products for at most N rows: k_hmm_b's K slices, k_update_mul's parts
// (9 MB at N = 1024 beside a matrix of 17, 129 at 5184 beside 430, 420 at 14400 beside 3318)
static size_t hb_slots(int N, int b) {
  if (!second_panel(N, b)) return HB_SMAX;
  auto slots = [](int m) { const int nt = (m + UM_R - 1) / UM_R; return um_parts(nt - 1, um_steps(m), nt); };
  return std::max({(int)HB_SMAX, slots(N), slots(std::min(N, UM_4)), slots(std::min(N, UM_2))});
}

size_t band_work_bytes(int N, int b, int nrhs) {
  const size_t nwg = (N + PR - 1) / PR + 1;
  const size_t LB = 2 * (size_t)b + 1;
  size_t s = 0;
  auto add = [&](size_t bytes) { s += (bytes + 255) & ~size_t(255); };
  add(sizeof(zc) * (size_t)N * b);            // Pw
  add(sizeof(zc) * (size_t)N * b);            // V
  add(sizeof(zc) * (size_t)N * b);            // Y
  add(sizeof(zc) * (size_t)N * b);            // X / W
  add(sizeof(zc) * 2 * nwg * (BMAX + 1));     // part
  add(sizeof(zc) * 2 * BMAX);                 // rowc
  add(sizeof(zc) * BMAX);                     // tau
  add(sizeof(zc) * BMAX * BMAX);              // G
  add(sizeof(zc) * BMAX * 6);                 // t1
  add(sizeof(zc) * BMAX * BMAX);              // T
  add(sizeof(zc) * 6 * BMAX);                 // t2
  add(sizeof(zc) * BMAX * BMAX);              // M
  add(sizeof(zc) * nwg * BMAX * BMAX);        // K slices of the small products
  add(sizeof(zc) * GRAM_PMAX * BMAX * (BMAX + 16));   // partials of the tall-skinny products
  add(sizeof(zc) * hb_slots(N, b) * (size_t)N * b);    // partials of X = A22 Y
  if (second_panel(N, b)) add(sizeof(zc) * 2 * (size_t)N * b);   // V2, X2
  add(sizeof(zc) * (size_t)N * LB);           // band
  add(sizeof(zc) * (size_t)N * (nrhs > 0 ? nrhs : 1));   // gc
  add(sizeof(int) * ((size_t)N + 1));         // prog
  add(sizeof(int) * 64);                      // err
  add(sizeof(int) * ((size_t)N / b + 2) * (BMAX + 1));   // panel column counters
  add(sizeof(zc) * 2 * qr_ex_elems<BMAX>((int)std::min<size_t>(nwg, QP_WG)));   // exchange slots
  return s + 4096;
}

int band_bind(BandWork& w, void* base, int N, int b, int nrhs) {
  if (b != 16 && b != 32) {
    set_error("band reduction: band width must be 16 or 32");
    return WTB_ERR_ARG;
  }
  w.N = N;
  w.b = b;
  w.nrhs = nrhs;
  w.LB = 2 * b + 1;
  w.nwg_max = (N + PR - 1) / PR + 1;
  char* p = static_cast<char*>(base);
  auto take = [&](size_t bytes) {
    char* q = p;
    p += (bytes + 255) & ~size_t(255);
    return q;
  };
  const size_t nwg = w.nwg_max;
  w.Pw = (zc*)take(sizeof(zc) * (size_t)N * b);
  w.V = (zc*)take(sizeof(zc) * (size_t)N * b);
  w.Y = (zc*)take(sizeof(zc) * (size_t)N * b);
  w.X = (zc*)take(sizeof(zc) * (size_t)N * b);
  w.part = (zc*)take(sizeof(zc) * 2 * nwg * (BMAX + 1));
  w.rowc = (zc*)take(sizeof(zc) * 2 * BMAX);
  w.tau = (zc*)take(sizeof(zc) * BMAX);
  w.G = (zc*)take(sizeof(zc) * BMAX * BMAX);
  w.t1 = (zc*)take(sizeof(zc) * BMAX * 6);
  w.T = (zc*)take(sizeof(zc) * BMAX * BMAX);
  w.t2 = (zc*)take(sizeof(zc) * 6 * BMAX);
  w.M = (zc*)take(sizeof(zc) * BMAX * BMAX);
  w.gw = (zc*)take(sizeof(zc) * nwg * BMAX * BMAX);
  w.gw_elems = nwg * BMAX * BMAX;
  w.gp = (zc*)take(sizeof(zc) * GRAM_PMAX * BMAX * (BMAX + 16));
  w.hb = (zc*)take(sizeof(zc) * hb_slots(N, b) * (size_t)N * b);
  w.V2 = w.X2 = nullptr;
  if (second_panel(N, b)) {
    w.V2 = (zc*)take(sizeof(zc) * 2 * (size_t)N * b);
    w.X2 = w.V2 + (size_t)N * b;
  }
  w.BD = (zc*)take(sizeof(zc) * (size_t)N * w.LB);
  w.gc = (zc*)take(sizeof(zc) * (size_t)N * (nrhs > 0 ? nrhs : 1));
  w.prog = (int*)take(sizeof(int) * ((size_t)N + 1));
  w.err = (int*)take(sizeof(int) * 64);
  w.bar = (int*)take(sizeof(int) * ((size_t)N / b + 2) * (BMAX + 1));
  w.ex = (zc*)take(sizeof(zc) * 2 * qr_ex_elems<BMAX>((int)std::min<size_t>(nwg, QP_WG)));
  w.panel_wg = band_panel_wg();
  return WTB_OK;
}

// A22 -= V W^H + W V^H
template <class T, int B>
static void her2k_band(hipStream_t s, BandWork& w, T* H, int ld, int m, int r0, int k) {
  const int nt = (m + 63) / 64;
  const bool tev = w.kev && w.kev_used < w.kev_cap;
  if (tev) hipEventRecord(w.kev[2 * w.kev_used], s);
  hipLaunchKernelGGL((k_her2k_full<T, B>), dim3(nt * (nt + 1) / 2), dim3(256), 0, s, H, ld, m, r0, w.N, w.V, w.X);
  if (tev) {
    hipEventRecord(w.kev[2 * w.kev_used++ + 1], s);
    w.kev_flops += 8.0 * 0.5 * (double)m * (double)(m + 1) * (2.0 * k);   // lower triangle, 2k products each
  }
}

// X = A22 Y (m x B) with enough workgroups to fill the chip: K slices until the grid
// holds ~1024 workgroups (at most HB_SMAX slices), partials summed in slice order
template <class T, int B>
static void hmm_band(hipStream_t s, BandWork& w, int m, const T* A, int ld, const zc* Y, zc* X) {
  const int rb = (m + HB_R - 1) / HB_R;
  int ns = std::max(1, std::min(HB_SMAX, (1024 + rb - 1) / rb));
  const int kc = ((m + ns - 1) / ns + 31) / 32 * 32;   // a multiple of either K step
  ns = (m + kc - 1) / kc;
  hipLaunchKernelGGL((k_hmm_b<T, B>), dim3(rb, ns), dim3(256), 0, s, m, A, ld, Y, w.N, kc, ns > 1 ? w.hb : nullptr,
                     X, w.N);
  if (ns > 1) {
    const size_t tot = (size_t)m * B;
    hipLaunchKernelGGL(k_hmm_sum<B>, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, m, ns, w.hb, X, w.N);
  }
}

// out0 = A^H Y0 (B x B) and out1 = A^H Y1 (B x n1) over m rows, ld B
template <int B>
static void gram(hipStream_t s, BandWork& w, int m, const zc* A, const zc* Y0, int ldy0, const zc* Y1, int n1,
                 zc* out0, zc* out1) {
  const int nch = (m + GRAM_ROWS - 1) / GRAM_ROWS;
  const int P = min(nch, GRAM_PMAX);
  hipLaunchKernelGGL(k_gram<B>, dim3(P), dim3(256), 0, s, m, w.N, A, Y0, ldy0, Y1, n1, w.gp);
  const int nout = B * (B + 16);
  hipLaunchKernelGGL(k_gram_sum<B>, dim3((nout + 63) / 64), dim3(256), 0, s, P, w.gp, n1, out0, out1);
}

// whether the reduction of a COMPLEX*16 matrix takes one-launch panels
static bool qr_form(const BandWork& w) { return w.b == 16 && w.panel_wg >= (w.N - 16 + PR - 1) / PR; }
static int wait_polls(const BandWork& w) { return w.wait_limit > 0 ? w.wait_limit : 1 << 20; }
static int ex_wgs(const BandWork& w) { return min(w.nwg_max, QP_WG); }   // workgroups that the slots hold

static ChaseArgs chase_args(const BandWork& w, int nrhs) {
  ChaseArgs ca;
  ca.BD = w.BD;
  ca.N = w.N;
  ca.gc = w.gc;
  ca.nrhs = nrhs;
  ca.prog = w.prog;
  ca.ctl = w.err;
  // polls of about half a microsecond each: about a second; in LDS about two seconds
  ca.spin_limit = w.wait_limit > 0 ? w.wait_limit : 1 << 21;
  ca.lds_limit = w.wait_limit > 0 ? w.wait_limit : 1 << 25;
  ca.Vc = nullptr;
  ca.ld = 0;
  ca.tau = w.tau2;
  ca.kt = chase_ntasks(w.N, w.b, 0);
  return ca;
}

static BandItem band_item(const BandWork& w, zc* H, int ld, int nrhs) {
  return BandItem{H, ld, w.N, nrhs, w.V, w.X, w.V2, w.X2, w.Y, w.T, w.gc, w.hb, w.ex, qr_ex_elems<16>(ex_wgs(w)),
                  qr_slots<16>(ex_wgs(w)), ex_wgs(w), w.err, wait_polls(w), w.tau1, chase_args(w, nrhs)};
}

// workgroups of the chase: as many as groups of sweeps can be at work at once, each following
// the one before by more than two tasks a sweep
static int chase_wgs(int N, int b) {
  const int sw = (b == 16) ? ChaseDim<16>::SW : ChaseDim<32>::SW;
  return min((N - 1 + sw - 1) / sw, min(256, chase_ntasks(N, b, 0) / (2 * sw) + 4));
}

template <class T, int B>
static int stage1(hipStream_t s, BandWork& w, T* H, int ld, int nrhs) {
  const int N = w.N, b = B;
  // COMPLEX*16 panels of at most panel_wg workgroups: one launch for the panel and one for W
  // (5 launches a panel, one of them a pass over the trailing matrix that updates it for the
  // panel before and multiplies it with this one's Y).  The limit does not depend on how many
  // streams run, so that the results do not either.  The COMPLEX*8 form keeps the separate kernels, whose roundings
  // its stored matrix amplifies.
  const bool qr = std::is_same<T, zc>::value && qr_form(w);
  BandItem it{};
  if constexpr (std::is_same<T, zc>::value)
    if (qr) it = band_item(w, H, ld, nrhs);
  for (int p = 0;; ++p) {
    const int c0 = p * b, r0 = c0 + b;
    if (r0 >= N) break;
    const int m = N - r0;
    const int k = min(b, m - 1);
    if (k <= 0) break;
    PanelArgs<T> a;
    a.A = H;
    a.ld = ld;
    a.N = N;
    a.b = b;
    a.c0 = c0;
    a.r0 = r0;
    a.m = m;
    a.k = k;
    a.Pw = w.Pw;
    a.part = w.part;
    a.rowc = w.rowc;
    a.tau = w.tau;
    a.nwg = (m + PR - 1) / PR;
    const dim3 g(a.nwg), blk(PR);
    if constexpr (std::is_same<T, zc>::value && B == 16)
      if (qr) {
        zc *V = panel_v(it, p), *X = panel_x(it, p);                  // this panel's; the one's before:
        const zc *Vo = panel_v(it, p + 1), *Xo = panel_x(it, p + 1);
        if (p > 0)
          hipLaunchKernelGGL((k_strip<B>), dim3((m + B + 63) / 64), blk, 0, s, H + c0 + (size_t)ld * c0, ld, m + B, N, Vo, Xo);
        hipLaunchKernelGGL((k_qr_panel<B>), g, blk, 0, s, qr_panel_args(it, p));
        const int n = um_steps(m), nt = (m + UM_R - 1) / UM_R;
        auto um = p > 0 ? k_update_mul<B, true> : k_update_mul<B, false>;
        const bool tev = w.kev && w.kev_used < w.kev_cap;
        if (tev) hipEventRecord(w.kev[2 * w.kev_used], s);
        hipLaunchKernelGGL(um, dim3(um_blocks(m)), blk, 0, s, trailing(it, p), ld, m, N, Vo + B, Xo + B, w.Y, w.hb, nt, n);
        if (tev) {
          hipEventRecord(w.kev[2 * w.kev_used++ + 1], s);
          // the update's two products of B reflectors on the lower triangle, the product with Y
          w.kev_flops += (p > 0 ? 8.0 * 0.5 * (double)m * (double)(m + 1) * (2.0 * B) : 0.0) + 8.0 * (double)m * m * k;
        }
        const size_t tot = (size_t)m * B;
        hipLaunchKernelGGL(k_um_sum<B>, dim3((unsigned)((tot + 255) / 256)), blk, 0, s, m, n, nt, w.hb, X, N);
        hipLaunchKernelGGL((k_qr_w<B>), g, blk, 0, s, qr_w_args(it, p));
        // the last panel's update, which no further product waits for
        if (last_panel(it, p)) {
          const int nu = (m + 63) / 64;
          hipLaunchKernelGGL((k_her2k_full<T, B>), dim3(nu * (nu + 1) / 2), blk, 0, s, H, ld, m, r0, N, V, X);
        }
        continue;
      }
    if (w.panel_resident > 0 && a.nwg <= w.panel_resident) {
      hipLaunchKernelGGL((k_panel<T, B>), g, blk, 0, s, a, w.V, w.bar + (size_t)p * (BMAX + 1), w.err + 8,
                         (long long)wait_polls(w));
    } else {
      for (int c = 0; c <= k; ++c) hipLaunchKernelGGL((k_pqr_col<T, B>), g, blk, 0, s, a, c);
      hipLaunchKernelGGL((k_pfin<T, B>), g, blk, 0, s, a, w.V);
    }
    int rc;
    gram<B>(s, w, m, w.V, w.V, N, nrhs > 0 ? w.gc + r0 : nullptr, nrhs, w.G, w.t1);
    hipLaunchKernelGGL((k_pT<B>), dim3(1), dim3(256), 0, s, k, w.G, w.t1, w.tau, nrhs, w.T, w.t2);
    hipLaunchKernelGGL((k_pY<B>), g, blk, 0, s, m, N, r0, w.V, w.T, w.t2, nrhs, w.Y, w.gc);
    hmm_band<T, B>(s, w, m, H + r0 + (size_t)ld * r0, ld, w.Y, w.X);
    gram<B>(s, w, m, w.V, w.X, N, nullptr, 0, w.M, nullptr);
    hipLaunchKernelGGL((k_pW<B>), g, blk, 0, s, m, N, w.V, w.T, w.M, w.X);
    her2k_band<T, B>(s, w, H, ld, m, r0, k);
  }
  WTB_LAUNCH_CHECK();
  return WTB_OK;
}

// what the reduction finds before its first launch: flags, counters and slots cleared, the
// tracked vectors conjugated
static void band_begin(hipStream_t s, BandWork& w, const zc* g, int nrhs, bool qr) {
  const int N = w.N;
  if (nrhs > 0)
    hipLaunchKernelGGL(k_conj_vec, dim3((unsigned)(((size_t)nrhs * N + 255) / 256)), dim3(256), 0, s, nrhs * N, g,
                       w.gc);
  hipLaunchKernelGGL(k_zero_ints, dim3(1), dim3(64), 0, s, w.err, 64);
  hipLaunchKernelGGL(k_zero_ints, dim3((N + 64 + 255) / 256), dim3(256), 0, s, w.prog, N + 1);
  if (qr) {
    const size_t exn = 2 * qr_ex_elems<16>(ex_wgs(w));
    hipLaunchKernelGGL(k_fill_empty, dim3((unsigned)((exn + 255) / 256)), dim3(256), 0, s, w.ex, exn);
  } else {
    const int nb = (N / w.b + 2) * (BMAX + 1);
    hipLaunchKernelGGL(k_zero_ints, dim3((nb + 255) / 256), dim3(256), 0, s, w.bar, nb);
  }
}

static void band_finish(hipStream_t s, const BandWork& w, zc* g, double* d, double* e, int nrhs, int* status) {
  hipLaunchKernelGGL(k_band_finish, dim3((w.N + 255) / 256), dim3(256), 0, s, w.BD, w.N, w.LB, d, e, w.gc, g, nrhs,
                     w.err, status);
}

template <class T>
static int run_band_t(hipStream_t s, BandWork& w, T* H, int ld, zc* g, double* d, double* e, int* status) {
  const int N = w.N, b = w.b, nrhs = g ? w.nrhs : 0;
  if (N < 2) {
    set_error("band reduction: N < 2");
    return WTB_ERR_ARG;
  }
  if (nrhs > 6) return WTB_ERR_LIMIT;
  if (w.tau1) {
    // the kept reflectors are those of the one-launch panels of the COMPLEX*16 matrix
    if (!std::is_same<T, zc>::value || b != 16 || N > band_vec_rows() || !band_panel_fits(N)) return WTB_ERR_LIMIT;
    hipLaunchKernelGGL(k_zero_ints, dim3((4 * N + 255) / 256), dim3(256), 0, s, (int*)w.tau1, 4 * N);
  }
  w.kev_used = 0;
  w.kev_flops = 0.0;
  band_begin(s, w, g, nrhs, std::is_same<T, zc>::value && qr_form(w));
  int rc = (b == 16) ? stage1<T, 16>(s, w, H, ld, nrhs) : stage1<T, 32>(s, w, H, ld, nrhs);
  if (rc) return rc;
  hipLaunchKernelGGL(k_band_extract<T>, dim3(N), dim3(64), 0, s, H, ld, N, b, w.LB, w.BD);
  ChaseArgs ca = chase_args(w, nrhs);
  if constexpr (std::is_same<T, zc>::value)
    if (w.tau1) ca.Vc = H;
  ca.ld = ld;
  auto kern = b == 32 ? k_chase<32, false> : ca.Vc ? k_chase<16, true> : k_chase<16, false>;
  const int sw = (b == 16) ? ChaseDim<16>::SW : ChaseDim<32>::SW;
  hipLaunchKernelGGL(kern, dim3(chase_wgs(N, b)), dim3((sw + 1) * 64), 0, s, ca);
  band_finish(s, w, g, d, e, nrhs, status);
  WTB_LAUNCH_CHECK();
  return WTB_OK;
}

// ---- a set of reductions in shared launches -----------------------------------------------
// One launch per kernel and panel for every matrix that still has that panel, one launch of the
// chase for all.  A lane of its own per matrix instead keeps 4 to 20 compute units busy with
// one latency chain, at most four of them at once (a process's hardware queues): 64 models of
// N = 256 .. 1024 took 356 ms on one lane and 124 on four.
bool band_in_set(const BandWork& w) { return qr_form(w) && w.N >= 32 && !w.tau1; }

int band_panel_wgs(int N) { return (N - 16 + PR - 1) / PR; }

// A set's panel launch takes up to half of the workgroups that the device holds at once (its
// members' workgroups wait only for those of the same member), and leaves `beside` of them to
// panels that run at the same time.
int band_set_wg(int beside) { return std::min(band_resident() / 2, band_resident() - beside); }

int band_set_prepare(BandSet& S) {
  band_set_free(S);
  if (S.items.empty()) return WTB_OK;
  // largest first: the matrices that have panel p are the first ones
  std::stable_sort(S.items.begin(), S.items.end(), [](const BandSetItem& x, const BandSetItem& y) { return x.w->N > y.w->N; });
  std::vector<BandItem> h;
  for (const auto& x : S.items) h.push_back(band_item(*x.w, x.H, x.ld, x.g ? x.w->nrhs : 0));
  WTB_HIP(hipMalloc(&S.d_items, sizeof(BandItem) * h.size()));
  WTB_HIP(hipMemcpy(S.d_items, h.data(), sizeof(BandItem) * h.size(), hipMemcpyHostToDevice));
  return WTB_OK;
}

void band_set_free(BandSet& S) {
  if (S.d_items) (void)hipFree(S.d_items);
  S.d_items = nullptr;
}

void band_set_begin(hipStream_t s, const BandSetItem& x) { band_begin(s, *x.w, x.g, x.g ? x.w->nrhs : 0, true); }
void band_set_finish(hipStream_t s, const BandSetItem& x) {
  band_finish(s, *x.w, x.g, x.d, x.e, x.g ? x.w->nrhs : 0, x.status);
}

int run_band_set(hipStream_t s, const BandSet& S) {
  if (S.items.empty()) return WTB_OK;
  if (!S.d_items) return WTB_ERR_ARG;
  const BandItem* dev = static_cast<const BandItem*>(S.d_items);
  const int M = (int)S.items.size();
  auto rows = [&](int i, int p) { return S.items[i].w->N - 16 * (p + 1); };
  // items first .. last - 1, blocks(i) workgroups each, in launches of at most kSetMax members
  // and `most` workgroups
  auto launch = [&](auto kern, int first, int last, auto blocks, int most, int threads, auto... args) {
    for (int i = first; i < last;) {
      BandSlots L;
      L.items = dev + i;
      L.n = 0;
      L.pre[0] = 0;
      for (; i < last && L.n < kSetMax && (L.n == 0 || L.pre[L.n] + blocks(i) <= most); ++i, ++L.n)
        L.pre[L.n + 1] = L.pre[L.n] + blocks(i);
      hipLaunchKernelGGL(kern, dim3(L.pre[L.n]), dim3(threads), 0, s, L, args...);
    }
  };
  const int any = 1 << 30, set_wg = S.max_wg;
  for (int p = 0, n = M;; ++p) {
    while (n > 0 && rows(n - 1, p) < 2) --n;
    if (n == 0) break;
    auto wgs = [&](int i) { return (rows(i, p) + PR - 1) / PR; };
    if (p > 0) launch(k_strip_s, 0, n, [&](int i) { return (rows(i, p) + 16 + 63) / 64; }, any, 256, p);
    launch(k_qr_panel_s, 0, n, wgs, set_wg, 256, p);
    launch(p > 0 ? k_update_mul_s<true> : k_update_mul_s<false>, 0, n, [&](int i) { return um_blocks(rows(i, p)); }, any, 256, p);
    launch(k_um_sum_s, 0, n, [&](int i) { return (rows(i, p) * 16 + 255) / 256; }, any, 256, p);
    launch(k_qr_w_s, 0, n, wgs, set_wg, 256, p);
    int f = n;                                 // members whose last panel this is
    while (f > 0 && rows(f - 1, p + 1) < 2) --f;
    launch(k_her2k_s, f, n, [&](int i) { const int u = (rows(i, p) + 63) / 64; return u * (u + 1) / 2; }, any, 256, p);
  }
  launch(k_band_extract_s, 0, M, [&](int i) { return S.items[i].w->N; }, any, 64);
  launch(k_chase_s, 0, M, [&](int i) { return chase_wgs(S.items[i].w->N, 16); }, any, (ChaseDim<16>::SW + 1) * 64);
  WTB_LAUNCH_CHECK();
  return WTB_OK;
}

// two columns of X fit the LDS of a compute unit
int band_vec_rows() { return 160 * 1024 / (2 * (int)sizeof(zc)); }
// Whether a solve with m eigenvectors that are corrected afterwards (the iterative solver's
// small solves; its residuals are formed from the vectors) takes the two-stage reduction
// (COMPLEX*16).  It saves 8 to 16 us a column of the one-stage form and pays N^2 m for the
// chase's reflectors.  All vectors, two-stage / one-stage: N = 256 4.4 / 6.4 ms, 640 8.5 /
// 13.7, 1290 21 / 29, 2049 45 / 52, 2500 62 / 69, 3000 86 / 91: the line lies where N m is
// 3000^2.  wtb_zheev, whose vectors are the result, keeps the one-stage form's smaller error.
bool band_vec_two_stage(int N, int m) {
  return N >= 32 && N <= band_vec_rows() && (double)N * m <= 9e6 && band_panel_fits(N);
}
size_t band_tau_elems(int N) { return (size_t)N + (size_t)N * (N / 16 + 1); }

int run_band_backtr(hipStream_t s, const BandWork& w, const zc* H, int ld, const double* Z, int c0, int m, zc* X,
                    int ldx, int cus, void* work) {
  const int N = w.N;
  if (N < 2 || m < 1 || !w.tau1 || N > band_vec_rows()) return WTB_ERR_ARG;
  // every pair of columns at work at once where the LDS holds them, 12 waves a workgroup,
  // fewer where the pieces do not need them
  const int pieces = (N + 63) / 64, np = (m + 1) / 2;
  const int pairs = std::max(1, std::min({(np + std::max(cus, 1) - 1) / std::max(cus, 1), band_vec_rows() / N, 12}));
  const int wpc = std::max(1, std::min(12 / pairs, pieces));
  // pieces of a wave and sweeps ahead: few pieces need more sweeps to cover a load
  auto kern = pieces <= 2 * wpc ? k_chase_back<16, 2, 3> : k_chase_back<16, 4, 1>;
  WTB_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
  ChaseBackArgs a{H, ld, w.tau2, chase_ntasks(N, 16, 0), N, Z, c0, m, X, ldx, pairs, wpc};
  hipLaunchKernelGGL(kern, dim3((np + pairs - 1) / pairs), dim3(64 * pairs * wpc), 2 * pairs * N * (int)sizeof(zc), s, a);
  return run_backtr_band(s, H, ld, N, 16, w.tau1, m, X, ldx, work);
}

int run_band_tridiag(hipStream_t s, BandWork& w, zc* H, int ld, zc* g, double* d, double* e, int* status) {
  return run_band_t<zc>(s, w, H, ld, g, d, e, status);
}
int run_band_tridiag_f32(hipStream_t s, BandWork& w, zf* H, int ld, zc* g, double* d, double* e, int* status) {
  return run_band_t<zf>(s, w, H, ld, g, d, e, status);
}

}  // namespace wtb
