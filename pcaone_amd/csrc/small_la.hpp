// L x L steps in LDS by one workgroup of NT threads: inverse Cholesky factor,
// Householder column signs, 16 x 16 block products.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace pcaone {
namespace {

// f(B), ..., f(E - 1) with constant arguments: registers indexed by nested
// loops whose bounds depend on each other are not always unrolled, and are then
// moved through an index register.
template <int B, int E, class F>
__device__ __forceinline__ void static_for(const F& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

typedef double f64x4_t __attribute__((ext_vector_type(4)));

// Upper 16 x 16 blocks (i <= j) of an NB x NB block grid, numbered row by
// row: block t is (sym_block_i(t), sym_block_j(t)).
__host__ __device__ constexpr int sym_block_i(int t, int nb) {
  int i = 0;
  while (t >= nb - i) t -= nb - i, ++i;
  return i;
}
__host__ __device__ constexpr int sym_block_j(int t, int nb) {
  int i = 0;
  while (t >= nb - i) t -= nb - i, ++i;
  return i + t;
}
// LDS pitch of an L x L matrix (rows on 16-byte boundaries, off the bank period).
template <int NB>
constexpr int kLP = NB * 16 + 2;

// Lane I of every row of 16 lanes, to the whole row.
template <int I>
__device__ __forceinline__ double row_value(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)u, 0x150 + I, 0xF, 0xF, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), 0x150 + I, 0xF, 0xF, true);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// 1 / sqrt(d) and 1 / x of normal numbers to about one unit in the last place:
// v_rsq_f64 / v_rcp_f64 (2^-23) and one third-order step.  Half the dependent
// operations of a correctly rounded root or quotient, and no branch.
__device__ __forceinline__ double rsqrt_step(double d) {
  const double y = __builtin_amdgcn_rsq(d);
  const double e = fma(-(d * y), y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ double recip_step(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, y, 1.0);
  return fma(y * e, 1.0 + e, y);
}

// src (lp x lp in global memory) -> LDS, zero in rows and columns >= n, and
// below the diagonal blocks when `upper`.
template <int NB, int NT>
__device__ __forceinline__ void lds_load(double* M, const double* __restrict__ src, int n, bool upper) {
  constexpr int LP = NB * 16;
  for (int v = threadIdx.x; v < LP * LP; v += NT) {
    const int i = v / LP, k = v - i * LP;
    const bool in = i < n && k < n && (!upper || (i >> 4) <= (k >> 4));
    M[i * kLP<NB> + k] = in ? src[v] : 0.0;
  }
}

// acc += A[16 bi ..][k] B[k][16 bj ..] for k in [k0, k1), one 16 x 16 block per
// wave (accumulator register r: row q + 4 r, column r16).  TB: B is given as its
// transpose.
template <int NB, bool TB = false>
__device__ __forceinline__ f64x4_t block_product(f64x4_t acc, const double* A, const double* B, int bi, int bj, int k0,
                                                 int k1, int lane) {
  const int q = lane >> 4, r16 = lane & 15;
  for (int k = k0; k < k1; k += 4)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[(16 * bi + r16) * kLP<NB> + k + q],
                                               TB ? B[(16 * bj + r16) * kLP<NB> + k + q]
                                                  : B[(k + q) * kLP<NB> + 16 * bj + r16],
                                               acc, 0, 0, 0);
  return acc;
}

template <int NB>
__device__ __forceinline__ f64x4_t block_load(const double* M, int bi, int bj, int lane) {
  f64x4_t v;
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = M[(16 * bi + (lane >> 4) + 4 * r) * kLP<NB> + 16 * bj + (lane & 15)];
  return v;
}

template <int NB>
__device__ __forceinline__ void block_store(double* M, const f64x4_t& v, int bi, int bj, int lane) {
#pragma unroll
  for (int r = 0; r < 4; ++r) M[(16 * bi + (lane >> 4) + 4 * r) * kLP<NB> + 16 * bj + (lane & 15)] = v[r];
}

// In place: A (n x n, symmetric positive definite, upper blocks used, zero
// below the diagonal blocks and past n) -> R^-T in the blocks on and below the
// diagonal (zero above the diagonal within them), where A = R^T R; the blocks
// above keep R's.  Elimination of [A | 1]: the identity's columns take the rows
// below the diagonal blocks, which A does not use, and the same row operations,
// so that the inverse needs no serial steps of its own.  16 pivots at a time
// run inside a wave: lanes 0..15 hold the diagonal block's columns, the others
// 48 of the NB 16 columns left and right of it (registers = rows); the rows
// below follow by MFMA products.  Rows n .. of the last group of four pivots
// are left as the identity's.  Returns false (in every thread) on breakdown;
// *min_pivot (thread 0) receives the smallest pivot.
template <int NB, int NT>
__device__ bool lds_chol_inv(double* A, int n, double* min_pivot, int* flag) {
  constexpr int P = kLP<NB>, LP = NB * 16, NV = (LP + 63) / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nbn = (n + 15) / 16;
  double dmin = INFINITY;
  if (tid == 0) *flag = 0;
  __syncthreads();
  for (int b = 0; b < nbn; ++b) {
    const int r0 = 16 * b;
    const int v = 64 * wave + lane;
    const bool mine = wave < NV, in = v < LP;
    const bool unit = (v >> 4) == b;  // the identity's columns of this panel
    double g[16], a[16];
    if (mine) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        g[i] = A[(r0 + i) * P + r0 + (lane & 15)];
        a[i] = A[(r0 + i) * P + (in ? v : 0)];
        if (r0 + i >= n) g[i] = (lane & 15) == i ? 1.0 : 0.0;
        if (unit) a[i] = (lane & 15) == i ? 1.0 : 0.0;
      }
    }
    if constexpr (NV > 1) __syncthreads();  // the diagonal block is read by every wave and written by one
    if (mine) {
      bool bad = false;
      static_for<0, 4>([&](auto q) {
        if (r0 + 4 * q >= n) return;
        static_for<4 * q, 4 * q + 4>([&](auto j) {
          const double d = row_value<j>(g[j]);  // the same value in every lane
          dmin = r0 + j < n ? fmin(dmin, d) : dmin;
          bad |= !(d > 0.0 && d < INFINITY);
          const double inv = rsqrt_step(d);
          g[j] *= inv;
          a[j] *= inv;
          static_for<j + 1, 16>([&](auto i) {
            g[i] = fma(-row_value<i>(g[j]), g[j], g[i]);
            a[i] = fma(-row_value<i>(g[j]), a[j], a[i]);
          });
        });
      });
      if (bad && tid == 0) *flag = 1;
      if (in) {
#pragma unroll
        for (int i = 0; i < 16; ++i) A[(r0 + i) * P + v] = a[i];
      }
    }
    __syncthreads();
    if (*flag) return false;
    // rows below: A[bi][bj] -= R[b][bi]^T A[b][bj], bj <= b (the inverse) and bj >= bi
    const int w = b + 1;
    int x = wave;
    for (int bi = b + 1; bi < nbn; ++bi) {
      const int nt = w + nbn - bi;
      for (; x < nt; x += NT / 64) {
        const int bj = x < w ? x : bi + x - w;
        f64x4_t acc = block_load<NB>(A, bi, bj, lane);
#pragma unroll
        for (int k = 0; k < 16; k += 4) {
          const double* row = A + (r0 + k + (lane >> 4)) * P + (lane & 15);
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-row[16 * bi], row[16 * bj], acc, 0, 0, 0);
        }
        block_store<NB>(A, acc, bi, bj, lane);
      }
      x -= nt;
    }
    __syncthreads();
  }
  if (tid == 0) *min_pivot = dmin;
  return true;
}

// What lds_chol_inv leaves, as R^-1 (upper, zero past n): element (i, c).
template <int NB>
__device__ __forceinline__ double inv_upper_at(const double* A, int n, int i, int c) {
  return i <= c && c < n ? A[c * kLP<NB> + i] : 0.0;
}

// Householder diagonal signs of the thin QR whose Q has top block W (n x n in
// LDS, zero past n, destroyed): modified LU, s_i = -sign(u_ii) (Ballard et al.
// 2014).  sgn: NB 16 values.
template <int NB, int NT>
__device__ void lds_householder_signs(double* W, int n, double* sgn) {
  constexpr int P = kLP<NB>, LP = NB * 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nbn = (n + 15) / 16;
  for (int b = 0; b < nbn; ++b) {
    const int r0 = 16 * b;
    const bool more = b + 1 < nbn;  // at most 64 columns right and rows below: wave 0 and wave 1
    if (wave < (more ? 2 : 1)) {
      const int v = r0 + 16 + lane;
      const bool in = v < LP, rows = wave == 1;
      double g[16], a[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        g[i] = W[(r0 + i) * P + r0 + (lane & 15)];
        a[i] = rows ? W[(in ? v : r0) * P + r0 + i] : W[(r0 + i) * P + (in ? v : r0)];
      }
      double s = 0.0;
      const auto panel = [&](auto rows_tag) {
        static_for<0, 4>([&](auto q) {
          if (r0 + 4 * q >= n) return;  // rows past n are zero: nothing would change
          static_for<4 * q, 4 * q + 4>([&](auto i) {
            const double p = row_value<i>(g[i]);
            const double si = p >= 0.0 ? -1.0 : 1.0, inv = recip_step(p - si);
            const double t = g[i] * inv, ta = a[i] * inv;
            s = (lane & 15) == i ? si : s;
            static_for<i + 1, 16>([&](auto r) {
              const double f = -row_value<i>(g[r]);
              if constexpr (decltype(rows_tag)::value) a[r] = fma(-row_value<r>(g[i]), ta, a[r]);
              else a[r] = fma(f, ta, a[r]);
              g[r] = fma(f, t, g[r]);
            });
            if constexpr (decltype(rows_tag)::value) a[i] = ta;
          });
        });
      };
      if (rows) panel(std::true_type{});
      else panel(std::false_type{});
      if (!rows && lane < 16) sgn[r0 + lane] = s;
      if (in && more) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          if (rows) W[v * P + r0 + i] = a[i];
          else W[(r0 + i) * P + v] = a[i];
        }
      }
    }
    __syncthreads();
    const int t = nbn - b - 1;
    for (int x = wave; x < t * t; x += NT / 64) {
      const int bi = b + 1 + x / t, bj = b + 1 + x % t;
      f64x4_t acc = block_load<NB>(W, bi, bj, lane);
#pragma unroll
      for (int k = 0; k < 16; k += 4)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-W[(16 * bi + (lane & 15)) * P + r0 + k + (lane >> 4)],
                                                   W[(r0 + k + (lane >> 4)) * P + 16 * bj + (lane & 15)], acc, 0, 0, 0);
      block_store<NB>(W, acc, bi, bj, lane);
    }
    __syncthreads();
  }
}

}  // namespace
}  // namespace pcaone
