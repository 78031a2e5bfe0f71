// L x L steps in LDS by one workgroup of NT threads: Cholesky factor, triangular
// inverse, Householder column signs, 16 x 16 block products.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace pcaone {
namespace {

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

__device__ __forceinline__ double lane_value(double v, int lane) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
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

// acc += sign * A[16 bi ..][k] B[k][16 bj ..] for k in [k0, k1), one 16 x 16
// block per wave (accumulator register r: row q + 4 r, column r16).
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
// multiplied by its reciprocal.  Returns false (in every thread) on breakdown;
// *min_pivot (thread 0) receives the smallest pivot.
template <int NB, int NT, bool DIV = false>
__device__ bool lds_chol_upper(double* A, int n, double* min_pivot, int* flag) {
  constexpr int P = kLP<NB>;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nbn = (n + 15) / 16;
  double dmin = INFINITY;
  if (tid == 0) *flag = 0;
  __syncthreads();
  for (int b = 0; b < nbn; ++b) {
    const int r0 = 16 * b, m = n - r0 - 16;  // m columns right of the panel's own
    // lanes 0..15: the diagonal block's columns; the others: 48 columns to the right
    const bool mine = wave < (m > 48 ? 2 : 1);
    const int col = lane < 16 ? r0 + lane : r0 + 48 * wave + lane;
    const bool in = mine && col < NB * 16;
    double a[16];
    if (mine) {
#pragma unroll
      for (int i = 0; i < 16; ++i) a[i] = A[(r0 + i) * P + (in ? col : r0)];
    }
    __syncthreads();  // wave 0 writes the diagonal block that both waves read
    if (mine) {
      bool ok = true;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        if (ok && r0 + j < n) {
          const double d = lane_value(a[j], j);
          if (!(d > 0.0) || !isfinite(d)) {  // the same value in every lane
            ok = false;
          } else {
            dmin = fmin(dmin, d);
            const double rjj = sqrt(d);
            double sj;
            if constexpr (DIV) {
              sj = a[j] / rjj;
            } else {
              const double inv = 1.0 / rjj;
              sj = a[j] * inv;
            }
            a[j] = lane == j ? rjj : sj;
#pragma unroll
            for (int i = j + 1; i < 16; ++i) a[i] = fma(-lane_value(sj, i), sj, a[i]);
          }
        }
      }
      if (!ok && tid == 0) *flag = 1;
      if (in && (lane >= 16 || wave == 0)) {
#pragma unroll
        for (int i = 0; i < 16; ++i) A[(r0 + i) * P + col] = (lane >= 16 || i <= lane) && r0 + i < n ? a[i] : 0.0;
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
// diagonal stay zero).  rt: scratch of NB 16 x kLP values, which may not
// overlap R; invd: NB 16 values.  The caller's barrier follows.
template <int NB, int NT>
__device__ __forceinline__ void lds_inv_upper(const double* R, double* rt, double* invd, int n, double (&x)[4 * NB]) {
  constexpr int LP = NB * 16, P = kLP<NB>, L4 = LP / 4;
  // rt[k][s L4 + m] = R[4 m + s][k]: a lane's factors of one k are contiguous
  for (int v = threadIdx.x; v < LP * LP; v += NT) {
    const int i = v / LP, k = v - i * LP;
    rt[k * P + (i & 3) * L4 + (i >> 2)] = R[i * P + k];
  }
  for (int i = threadIdx.x; i < n; i += NT) invd[i] = 1.0 / R[i * P + i];
#pragma unroll
  for (int m = 0; m < L4; ++m) x[m] = 0.0;
  __syncthreads();
  const int wave = threadIdx.x >> 6, c = threadIdx.x >> 2, s = threadIdx.x & 3;
  if (wave >= NB) return;
  const int kmax = 16 * wave + 16 < n ? 16 * wave + 16 : n;
#pragma unroll
  for (int kk = L4 - 1; kk >= 0; --kk) {
    auto row = [&]<int S>() {
      const int k = 4 * kk + S;
      if (k >= kmax) return;  // the same in the whole wave
      double v = ((c == k ? 1.0 : 0.0) - x[kk]) * invd[k];
      v = c >= k && c < n ? v : 0.0;
      const double xk = quad_value<S>(v);  // lane S holds row k
      const double* f = rt + k * P + s * L4;
#pragma unroll
      for (int m = 0; m < kk; ++m) x[m] = fma(f[m], xk, x[m]);
      x[kk] = s == S ? xk : (s < S ? fma(f[kk], xk, x[kk]) : x[kk]);
    };
    row.template operator()<3>();
    row.template operator()<2>();
    row.template operator()<1>();
    row.template operator()<0>();
  }
}

// Householder diagonal signs of the thin QR whose Q has top block W (n x n in
// LDS, zero past n, destroyed): modified LU, s_i = -sign(u_ii) (Ballard et al.
// 2014).
template <int NB, int NT>
__device__ void lds_householder_signs(double* W, int n, double* sgn) {
  constexpr int P = kLP<NB>, LP = NB * 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nbn = (n + 15) / 16;
  for (int b = 0; b < nbn; ++b) {
    const int r0 = 16 * b, m = n - r0 - 16;
    const int nr = m > 48 ? 2 : (m > 0 ? 1 : 0);  // waves for the rows below; the columns right take as many
    const int nu = nr > 1 ? nr : 1;
    double a[16];
    if (wave < nu) {  // lane = column, registers = the panel's rows
      const int col = lane < 16 ? r0 + lane : r0 + 48 * wave + lane;
      const bool in = col < LP;
#pragma unroll
      for (int i = 0; i < 16; ++i) a[i] = W[(r0 + i) * P + (in ? col : r0)];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if (r0 + i < n) {
          const double p = lane_value(a[i], i);
          const double si = p >= 0.0 ? -1.0 : 1.0, inv = 1.0 / (p - si);
          if (wave == 0 && lane == i) sgn[r0 + i] = si;
#pragma unroll
          for (int r = i + 1; r < 16; ++r) a[r] = fma(-(lane_value(a[r], i) * inv), a[i], a[r]);
        }
      }
      if (in && lane >= 16) {
#pragma unroll
        for (int i = 0; i < 16; ++i) W[(r0 + i) * P + col] = a[i];
      }
    } else if (wave < nu + nr) {  // lane = row, registers = the panel's columns
      const int row = lane < 16 ? r0 + lane : r0 + 48 * (wave - nu) + lane;
      const bool in = row < LP;
#pragma unroll
      for (int c = 0; c < 16; ++c) a[c] = W[(in ? row : r0) * P + r0 + c];
#pragma unroll
      for (int i = 0; i < 16; ++i) {  // the rows below exist: the panel is whole
        const double p = lane_value(a[i], i);
        const double inv = 1.0 / (p - (p >= 0.0 ? -1.0 : 1.0));
        const double l = a[i] * inv;
#pragma unroll
        for (int c = i + 1; c < 16; ++c) a[c] = fma(-l, lane_value(a[c], i), a[c]);
        a[i] = l;
      }
      if (in && lane >= 16) {
#pragma unroll
        for (int c = 0; c < 16; ++c) W[row * P + r0 + c] = a[c];
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
