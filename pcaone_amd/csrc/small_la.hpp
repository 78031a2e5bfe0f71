// L x L steps in LDS by one workgroup of NT threads: Cholesky factor, triangular
// inverse, Householder column signs, 16 x 16 block products.
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

// The wave's index in the workgroup, as a scalar: branches on it take no lane masks.
__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }

// Lane I of every row of 16 lanes, to the whole row.
template <int I>
__device__ __forceinline__ double row_value(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)u, 0x150 + I, 0xF, 0xF, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), 0x150 + I, 0xF, 0xF, true);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// Lane S of every group of four lanes, to the whole group.
template <int S>
__device__ __forceinline__ double quad_value(double v) {
  constexpr int ctrl = S * 0x55;
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)u, ctrl, 0xF, 0xF, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), ctrl, 0xF, 0xF, true);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// r = sqrt(d) and inv = 1 / r, both rounded as the root and the quotient are, without
// their range checks, from y0 = 1 / sqrt(d) to 2^-23: one third-order step and
// Markstein's corrections of the root and of its reciprocal.  (The one significand
// that the latter does not cover, r of all ones, gives inv one unit low.)
__host__ __device__ __forceinline__ void refine_root(double d, double y0, double& r, double& inv) {
  const double e = fma(-(d * y0), y0, 1.0);
  const double y = fma(y0 * e, fma(0.375, e, 0.5), y0);
  const double g = d * y;
  r = fma(fma(-g, g, d), 0.5 * y, g);
  inv = fma(fma(-r, y, 1.0), y, y);
}
__device__ __forceinline__ void root_and_inverse(double d, double& r, double& inv) {
  refine_root(d, __builtin_amdgcn_rsq(d), r, inv);  // v_rsq_f64
}
// x / d with inv = 1 / d, rounded as the quotient is (Markstein's correction), for
// finite d and inv and a finite x that is 0 or at least 2^-960 in size (the residual
// x - q d is exact), without overflow.
__host__ __device__ __forceinline__ double quotient(double x, double d, double inv) {
  const double q = x * inv;
  return fma(fma(-q, d, x), inv, q);
}
// The same where x may be infinite or NaN or the quotient overflow: as the division.
__host__ __device__ __forceinline__ double quotient_any(double x, double d, double inv) {
  const double q = x * inv;
  return fabs(q) < INFINITY ? fma(fma(-q, d, x), inv, q) : q;
}
// Place of x[i stride] among the n values x[0], x[stride], ... in descending order,
// NaNs after the numbers and equal ones by index: a total order, so that the n
// places are a permutation whatever the values.
__host__ __device__ __forceinline__ int place_descending(const double* x, int stride, int n, int i) {
  const double v = x[i * stride];
  int place = 0;
  for (int j = 0; j < n; ++j) {
    const double y = x[j * stride];
    const bool ahead = v != v ? y == y || j < i : y > v || (y == v && j < i);
    place += ahead ? 1 : 0;
  }
  return place;
}
// 1 / x to about one unit in the last place.
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
// wave (accumulator register r: row q + 4 r, column r16).
template <int NB>
__device__ __forceinline__ f64x4_t block_product(f64x4_t acc, const double* A, const double* B, int bi, int bj, int k0,
                                                 int k1, int lane) {
  const int q = lane >> 4, r16 = lane & 15;
  for (int k = k0; k < k1; k += 4)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[(16 * bi + r16) * kLP<NB> + k + q],
                                               B[(k + q) * kLP<NB> + 16 * bj + r16], acc, 0, 0, 0);
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
// below the diagonal blocks and past n) -> upper R with A = R^T R, zero
// elsewhere.  Right-looking; DIV: rows divided by the pivot's root, else
// multiplied by its reciprocal.  16 pivots at a time run inside wave 0: g holds
// the diagonal block's columns in every 16 lanes, a the (at most 64) columns to
// the right, registers = rows, and a row's factor comes as a row broadcast of
// g; the rows below follow by MFMA products.  Returns false (in every thread) on
// breakdown; *min_pivot (thread 0) receives the smallest pivot.
template <int NB, int NT, bool DIV = false>
__device__ bool lds_chol_upper(double* A, int n, double* min_pivot, int* flag) {
  constexpr int P = kLP<NB>, LP = NB * 16;
  static_assert(NB <= 5, "one wave holds the columns right of a panel");
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index(), l16 = lane & 15;
  const int nbn = (n + 15) / 16;
  double dmin = INFINITY;
  if (tid == 0) *flag = 0;
  __syncthreads();
  for (int b = 0; b < nbn; ++b) {
    const int r0 = 16 * b;
    if (wave == 0) {
      const int v = r0 + 16 + lane;
      const bool in = v < LP;
      double g[16], a[16], piv = INFINITY, root = 0.0;  // lane j of 16: pivot j, its root
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        g[i] = A[(r0 + i) * P + r0 + l16];
        a[i] = A[(r0 + i) * P + (in ? v : r0)];
      }
      if (r0 + 16 > n) {
#pragma unroll
        for (int i = 0; i < 16; ++i)  // the rest of a group of four pivots: left as it is
          if (r0 + i >= n) g[i] = l16 == i ? 1.0 : 0.0;
      }
      static_for<0, 4>([&](auto q) {
        if (r0 + 4 * q >= n) return;
        static_for<4 * q, 4 * q + 4>([&](auto j) {
          const double d = row_value<j>(g[j]);  // the same value in every lane
          double rjj, inv;
          root_and_inverse(d, rjj, inv);
          piv = l16 == j ? d : piv;
          root = l16 == j ? rjj : root;
          g[j] = DIV ? quotient(g[j], rjj, inv) : g[j] * inv;
          a[j] = DIV ? quotient(a[j], rjj, inv) : a[j] * inv;
          static_for<j + 1, 16>([&](auto i) {
            const double f = -row_value<i>(g[j]);
            g[i] = fma(f, g[j], g[i]);
            a[i] = fma(f, a[j], a[i]);
          });
        });
      });
      const bool past = r0 + l16 >= n;
      if (__any(!past && !(piv > 0.0 && piv < INFINITY)) && lane == 0) *flag = 1;
      if (past) piv = INFINITY;
#pragma unroll
      for (int d = 1; d < 16; d <<= 1) piv = fmin(piv, __shfl_xor(piv, d));
      dmin = fmin(dmin, piv);
      if (lane < 16) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
          A[(r0 + i) * P + r0 + lane] = past || i > lane ? 0.0 : (i == lane ? root : g[i]);
      }
      if (in) {
#pragma unroll
        for (int i = 0; i < 16; ++i) A[(r0 + i) * P + v] = r0 + i < n ? a[i] : 0.0;
      }
    }
    __syncthreads();
    if (*flag) return false;
    // trailing blocks (bi <= bj): A -= R[panel]^T R[panel]
    const int t = nbn - b - 1, nt = t * (t + 1) / 2;
    for (int x = wave; x < nt; x += NT / 64) {
      int i = 0, y = x;
      while (y >= t - i) y -= t - i, ++i;
      const int bi = b + 1 + i, bj = bi + y;
      f64x4_t acc = block_load<NB>(A, bi, bj, lane);
#pragma unroll
      for (int k = 0; k < 16; k += 4) {
        const double* row = A + (r0 + k + (lane >> 4)) * P + (lane & 15);
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-row[16 * bi], row[16 * bj], acc, 0, 0, 0);
      }
      block_store<NB>(A, acc, bi, bj, lane);
    }
    __syncthreads();
  }
  if (tid == 0) *min_pivot = dmin;
  return true;
}

// X = R^-1 for the upper R in LDS (n x n, zero outside), by rows from the
// bottom: X[i][c] = (delta_ic - sum_{k > i} R[i][k] X[k][c]) / R[i][i], the sums
// taken in descending k.  Lane s of four holds the rows 4 m + s of one column
// c in x[m] (waves 0 .. NB - 1 take 16 columns each; a column's rows below the
// diagonal stay zero).  Four rows go without a branch between them, so that their
// factors are read ahead of the chain.  rt: scratch of NB 16 x kLP values, which
// may not overlap R; invd: NB 16 values.  The caller's barrier follows.
template <int NB, int NT>
__device__ __forceinline__ void lds_inv_upper(const double* R, double* rt, double* invd, int n, double (&x)[4 * NB]) {
  constexpr int LP = NB * 16, P = kLP<NB>, L4 = LP / 4;
  // rt[k][s L4 + m] = R[4 m + s][k]: a lane's factors of one k are contiguous
  for (int v = threadIdx.x; v < LP * LP; v += NT) {
    const int i = v / LP, k = v - i * LP;
    rt[k * P + (i & 3) * L4 + (i >> 2)] = R[i * P + k];
  }
  for (int i = threadIdx.x; i < LP; i += NT) invd[i] = i < n ? 1.0 / R[i * P + i] : 0.0;
#pragma unroll
  for (int m = 0; m < L4; ++m) x[m] = 0.0;
  __syncthreads();
  const int wave = wave_index(), c = threadIdx.x >> 2, s = threadIdx.x & 3;
  if (wave >= NB) return;
  const int kmax = 16 * wave + 16 < n ? 16 * wave + 16 : n;
  static_for<0, L4>([&](auto back) {
    constexpr int kk = L4 - 1 - decltype(back)::value;
    if (4 * kk >= kmax) return;  // the same in the whole wave; rows past n in the last four give zeros
    double f[4][kk + 1], id[4];
    static_for<0, 4>([&](auto S) {
#pragma unroll
      for (int m = 0; m <= kk; ++m) f[S][m] = rt[(4 * kk + S) * P + s * L4 + m];
      id[S] = invd[4 * kk + S];
    });
    static_for<0, 4>([&](auto rev) {
      constexpr int S = 3 - decltype(rev)::value, k = 4 * kk + S;
      double v = ((c == k ? 1.0 : 0.0) - x[kk]) * id[S];
      v = c >= k && c < n ? v : 0.0;
      const double xk = quad_value<S>(v);  // lane S holds row k
      x[kk] = s == S ? xk : (s < S ? fma(f[S][kk], xk, x[kk]) : x[kk]);
#pragma unroll
      for (int m = 0; m < kk; ++m) x[m] = fma(f[S][m], xk, x[m]);
    });
  });
}

// Householder diagonal signs of the thin QR whose Q has top block W (n x n in
// LDS, zero past n, destroyed): modified LU, s_i = -sign(u_ii) (Ballard et al.
// 2014).  sgn: NB 16 values.
template <int NB, int NT>
__device__ void lds_householder_signs(double* W, int n, double* sgn) {
  constexpr int P = kLP<NB>, LP = NB * 16;
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int nbn = (n + 15) / 16;
  for (int b = 0; b < nbn; ++b) {
    const int r0 = 16 * b;
    const bool more = b + 1 < nbn;  // at most 64 columns right and rows below: wave 0 and wave 1
    if (wave < (more ? 2 : 1)) {
      const int v = r0 + 16 + lane;
      const bool in = v < LP, rows = wave == 1;
      double g[16], a[16];
      const double* from = rows ? W + (in ? v : r0) * P + r0 : W + r0 * P + (in ? v : r0);
      const int step = rows ? 1 : P;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        g[i] = W[(r0 + i) * P + r0 + (lane & 15)];
        a[i] = from[i * step];
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
        double* to = rows ? W + v * P + r0 : W + r0 * P + v;
#pragma unroll
        for (int i = 0; i < 16; ++i) to[i * step] = a[i];
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
