// FP64 kernels around the genotype products: MFMA operand pieces, the affine
// epilogues of the two products, column sums, Gram reductions (CholeskyQR2,
// B*B^T, mev), small right-multiplications, flipOmg norms and the
// missing-entry (and EMU imputation) corrections.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "bf16.hpp"
#include "device.hpp"
#include "kernels.hpp"
#include "small_la.hpp"

namespace pcaone {
namespace {

inline unsigned grid_for(uint64_t n, unsigned block = 256, unsigned cap = 65535u * 8) {
  uint64_t g = (n + block - 1) / block;
  if (g > cap) g = cap;
  return (unsigned)(g ? g : 1);
}

#define GRID_STRIDE(t, n) \
  for (uint64_t t = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; t < (n); t += (uint64_t)gridDim.x * blockDim.x)


// Operand pieces of one form for each value y = X[r][l] colsign[l] rowscale[r]
// (F8 and I8: y / s, s the column scale), and the value they sum to (times s).
template <Form F>
struct Pieces;
template <>
struct Pieces<Form::FP64> {
  using w_t = double;
  static constexpr int P = 1;
  __device__ static double make(double y, double, w_t* pc) { return pc[0] = y; }
};
template <>
struct Pieces<Form::FP32> {
  using w_t = float;
  static constexpr int P = 1;
  __device__ static double make(double y, double, w_t* pc) { return (double)(pc[0] = (float)y); }
};
template <>
struct Pieces<Form::FP16> {
  using w_t = uint16_t;
  static constexpr int P = 1;
  __device__ static double make(double y, double, w_t* pc) {
    pc[0] = fp16_bits(y);
    return fp16_value(pc[0]);
  }
};
template <>
struct Pieces<Form::BF16X1> {
  using w_t = uint16_t;
  static constexpr int P = 1;
  __device__ static double make(double y, double, w_t* pc) {
    pc[0] = bf16_bits((float)y);
    return (double)bf16_value(pc[0]);
  }
};
template <>
struct Pieces<Form::BF16> {
  using w_t = uint16_t;
  static constexpr int P = 2;
  __device__ static double make(double y, double, w_t* pc) {
    pc[0] = bf16_bits((float)y);
    const double back = (double)bf16_value(pc[0]);
    pc[1] = bf16_bits((float)(y - back));
    return back + (double)bf16_value(pc[1]);
  }
};
template <>
struct Pieces<Form::F8> {
  using w_t = uint8_t;
  static constexpr int P = 3;
  // x1 = y / s (exact: s is a power of two, |y / s| <= 448) as three E4M3
  // pieces, each the nearest E4M3 to what the previous ones left
  __device__ static double make(double x1, double s, w_t* pc) {
    double v1, v2, v3;
    pc[0] = e4m3_bits(x1, &v1);
    pc[1] = e4m3_bits(x1 - v1, &v2);
    pc[2] = e4m3_bits(x1 - v1 - v2, &v3);
    return (v1 + v2 + v3) * s;
  }
};
template <>
struct Pieces<Form::I8> {
  using w_t = uint8_t;
  static constexpr int P = 2;
  // q = rint(y / s) within +-kI8Max; q = 256 q_hi + q_lo, q_lo in [-128, 127]
  __device__ static double make(double ys, double s, w_t* pc) {
    const int q = (int)fmin(fmax(rint(ys), -(double)kI8Max), (double)kI8Max);
    const int hi = (q + 128) >> 8, lo = q - 256 * hi;
    pc[0] = (uint8_t)(int8_t)hi;
    pc[1] = (uint8_t)(int8_t)lo;
    return (double)q * s;
  }
};

// Rows per workgroup of the row-tiled kernels below and the LDS row pitch of
// their transposed pieces (element size wsz bytes): padded so that the
// column groups of one store land in different banks.
constexpr int kEpiRows = 64;
constexpr int kEpiBatch = 4;  // rows a thread loads before it works on them
constexpr int epi_pitch(size_t wsz) { return kEpiRows + (wsz < 4 ? 4 / (int)wsz : 1); }

// The tile's transposed pieces, LDS -> wt[p][l][r0 + r] for r < nr, in stores of
// 8 bytes at aligned addresses (one element at a time at the tile's ends, where
// the window does not start or end on one), and the zeros of the `left` elements
// before row 0 and the `right` ones from row rows_end, each block a share of the
// rows.  wpitch and wpiece are multiples of 8 elements.
template <class w_t>
__device__ __forceinline__ void store_pieces(const w_t* pt, int np, int lp, w_t* wt, uint64_t wpitch, uint64_t wpiece,
                                             uint64_t r0, int nr, uint32_t left, uint64_t rows_end, uint32_t right) {
  constexpr int E = 8 / sizeof(w_t), PITCH = epi_pitch(sizeof(w_t));
  const auto row_of = [&](int pl) {
    const int p = (pl >= lp) + (pl >= 2 * lp);
    return wt + p * wpiece + (pl - p * lp) * wpitch;
  };
  if constexpr (E == 1) {
    for (int v = threadIdx.x; v < np * lp * kEpiRows; v += 256) {
      const int r = v % kEpiRows, pl = v / kEpiRows;
      if (r < nr) row_of(pl)[r0 + r] = pt[pl * PITCH + r];
    }
  } else {
    const int sh = (int)(reinterpret_cast<uintptr_t>(wt) / sizeof(w_t) % E);  // r0 is a multiple of E
    const auto run = [&](auto aligned) {
      constexpr bool kAligned = decltype(aligned)::value;
      constexpr int NG = kEpiRows / E + (kAligned ? 0 : 1);
      for (int v = threadIdx.x; v < np * lp * NG; v += 256) {
        const int pl = v / NG, r = (v - pl * NG) * E - (kAligned ? 0 : sh);
        w_t* d = row_of(pl) + r0;
        const w_t* s = pt + pl * PITCH + r;
        if (r >= 0 && r + E <= nr) {
          uint64_t u = 0;
          if constexpr (kAligned) {
            const uint32_t* s4 = reinterpret_cast<const uint32_t*>(s);
            u = (uint64_t)s4[1] << 32 | s4[0];
          } else {
#pragma unroll
            for (int e = 0; e < E; ++e) {
              using bits_t = typename std::conditional<
                  sizeof(w_t) == 4, uint32_t, typename std::conditional<sizeof(w_t) == 2, uint16_t, uint8_t>::type>::type;
              u |= (uint64_t)__builtin_bit_cast(bits_t, s[e]) << (8 * sizeof(w_t) * e);
            }
          }
          *reinterpret_cast<uint64_t*>(d + r) = u;
        } else {
          for (int e = 0; e < E; ++e)
            if (r + e >= 0 && r + e < nr) d[r + e] = s[e];
        }
      }
    };
    if (sh) run(std::false_type{});
    else run(std::true_type{});
  }
  if (left + right) {
    const uint32_t per = left + right;
    for (int pl = blockIdx.x; pl < np * lp; pl += gridDim.x) {
      w_t* d = row_of(pl);
      for (uint32_t c = threadIdx.x; c < per; c += 256) {
        if (c < left) (d - left)[c] = w_t(0);
        else d[rows_end + (c - left)] = w_t(0);
      }
    }
  }
}

// Operand pieces of X (rows x lp, row-major FP64), transposed to
// Wt[p][l][r], for a tile of 64 rows per workgroup.  Each thread owns 4
// adjacent columns of every RG-th row of the tile (16-byte loads along the
// row); the pieces go through LDS so that the transposed stores are coalesced
// along the rows.  Optional outputs: signed_out (X colsign), rounded (the
// pieces' sum / rowscale; in place over X allowed: every element is read and
// written by the same thread), and the per-tile column sums of
// w_r rounded[r][l] (w_r = bsc[r] (1/2 - bcf[r]), or 1 without bsc) in bpart.
// Bound by the conversions where the rows fill the chip (as FP8 about 150 VALU
// instructions a value: 1,000,000 x 80 take 469 us, 1.5 GB at 3.2 TB/s, two thirds of
// a copy's rate, against about 580 with a division per value, exponents taken apart
// by frexp and ldexp and one byte per store) and by a tile's own chain of loads
// where they do not (10,000 x 40 as BF16: 7.3 us against 10.0 with a row at a time).
template <Form F>
__global__ void __launch_bounds__(256) k_make_pieces(const double* X, uint64_t nreal, uint64_t rows_pad, int lp,
                                                     const double* __restrict__ rowscale,
                                                     const double* __restrict__ colsign, void* Wt, uint64_t wpitch,
                                                     uint64_t wpiece, double* rounded, double* __restrict__ signed_out,
                                                     const double* __restrict__ colscale,
                                                     const double* __restrict__ bsc, const double* __restrict__ bcf,
                                                     double* __restrict__ bpart, uint32_t left, uint32_t right) {
  using PF = Pieces<F>;
  using w_t = typename PF::w_t;
  constexpr int P = PF::P;
  constexpr int PITCH = epi_pitch(sizeof(w_t));
  extern __shared__ __align__(16) unsigned char sm[];
  w_t* pt = reinterpret_cast<w_t*>(sm);  // P x lp rows of PITCH
  double* bred = reinterpret_cast<double*>(sm + ((size_t)P * lp * PITCH * sizeof(w_t) + 15) / 16 * 16);
  const int CG = lp / 4, RG = 256 / CG;
  const int tid = threadIdx.x, cg = tid % CG, rg = tid / CG;
  const bool act = rg < RG;
  const uint64_t r0 = (uint64_t)blockIdx.x * kEpiRows;
  const int nr = (int)(rows_pad - r0 < (uint64_t)kEpiRows ? rows_pad - r0 : kEpiRows);
  double b4[4] = {0.0, 0.0, 0.0, 0.0};
  if (act) {
    // F8: sl = the column's scale 2^se.  I8: the scale is sl 2^se, is = 1 / sl.  The
    // exponents go through ldexp: the reciprocal of a whole scale may overflow.
    double cs[4] = {1.0, 1.0, 1.0, 1.0}, sl[4] = {1.0, 1.0, 1.0, 1.0}, is[4];
    int se[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (colsign) cs[q] = colsign[4 * cg + q];
      if constexpr (F == Form::F8) {
        sl[q] = colscale[4 * cg + q];
        (void)frexp(sl[q], &se[q]);
        --se[q];
      } else if constexpr (F == Form::I8) {
        sl[q] = frexp(colscale[4 * cg + q], &se[q]);
        is[q] = 1.0 / sl[q];
      }
    }
    for (int rb = rg; rb < nr; rb += kEpiBatch * RG) {
      double x[kEpiBatch][4], rs[kEpiBatch], w[kEpiBatch];
#pragma unroll
      for (int u = 0; u < kEpiBatch; ++u) {
        const uint64_t j = r0 + rb + u * RG;
        double2 v0{0.0, 0.0}, v1{0.0, 0.0};
        rs[u] = 1.0, w[u] = 0.0;
        if (rb + u * RG < nr) {
          if (j < nreal) {
            const double* xr = X + j * lp + 4 * cg;
            v0 = *reinterpret_cast<const double2*>(xr);
            v1 = *reinterpret_cast<const double2*>(xr + 2);
            w[u] = bsc ? bsc[j] * (0.5 - bcf[j]) : 1.0;
          }
          if (rowscale) rs[u] = rowscale[j];
        }
        x[u][0] = v0.x, x[u][1] = v0.y, x[u][2] = v1.x, x[u][3] = v1.y;
      }
#pragma unroll
      for (int u = 0; u < kEpiBatch; ++u) {
        const int r = rb + u * RG;
        if (r >= nr) break;
        const uint64_t j = r0 + r, t = j * lp + 4 * cg;
#pragma unroll
        for (int q = 0; q < 4; ++q) x[u][q] *= cs[q];
        if (signed_out) {
          *reinterpret_cast<double2*>(signed_out + t) = double2{x[u][0], x[u][1]};
          *reinterpret_cast<double2*>(signed_out + t + 2) = double2{x[u][2], x[u][3]};
        }
        const bool live = j < nreal && rs[u] != 0.0;
        const double irs = rowscale ? 1.0 / rs[u] : 1.0;
        double rd[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          double y = x[u][q] * rs[u];
          if constexpr (F == Form::F8) y = ldexp(y, -se[q]);
          if constexpr (F == Form::I8) y = quotient(ldexp(y, -se[q]), sl[q], is[q]);
          w_t pc[P];
          double back = PF::make(y, sl[q], pc);
          if constexpr (F == Form::I8) back = ldexp(back, se[q]);
          rd[q] = live ? (rowscale ? quotient_any(back, rs[u], irs) : back) : 0.0;
          b4[q] += w[u] * rd[q];
#pragma unroll
          for (int p = 0; p < P; ++p) pt[(p * lp + 4 * cg + q) * PITCH + r] = pc[p];
        }
        if (rounded) {
          *reinterpret_cast<double2*>(rounded + t) = double2{rd[0], rd[1]};
          *reinterpret_cast<double2*>(rounded + t + 2) = double2{rd[2], rd[3]};
        }
      }
    }
    if (bpart) {
#pragma unroll
      for (int q = 0; q < 4; ++q) bred[rg * lp + 4 * cg + q] = b4[q];
    }
  }
  __syncthreads();
  store_pieces(pt, P, lp, static_cast<w_t*>(Wt), wpitch, wpiece, r0, nr, left, rows_pad, right);
  if (bpart) {
    for (int l = threadIdx.x; l < lp; l += 256) {
      double sum = 0.0;
      for (int q = 0; q < RG; ++q) sum += bred[q * lp + l];
      bpart[(uint64_t)blockIdx.x * lp + l] = sum;
    }
  }
}

// colmul (nullable): per-column factor of the summed partials (the I8
// form's int32 partials are sum (v/2) q, so the factor is 2 s_l; the F8
// form's are sum v (w / s_l), so it is s_l).
template <class P>
__global__ void k_epi_g(const P* __restrict__ part, uint64_t nchunks, uint64_t stride, uint64_t nreal,
                        uint64_t rows_pad, int lp, const double* __restrict__ sc, const double* __restrict__ cf,
                        const double* __restrict__ colsum, double* __restrict__ out, const double* __restrict__ colmul) {
  const uint64_t n = rows_pad * (uint64_t)lp;
  GRID_STRIDE(t, n) {
    const uint64_t j = t / lp;
    const int l = (int)(t - j * lp);
    double v = 0.0;
    if (j < nreal) {
      double y = 0.0;
      for (uint64_t c = 0; c < nchunks; ++c) y += (double)part[c * stride + t];
      if (colmul) y *= colmul[l];
      const double s = sc[j];
      v = 0.25 * s * y + s * (0.5 - cf[j]) * colsum[l];
    }
    out[t] = v;
  }
}

// k_epi_g for 32-bit partials (FP32 or int32), 4 adjacent columns per thread
// (16-byte partial loads, 32-byte stores).
template <class PT>
__global__ void k_epi_g_v4(const PT* __restrict__ part, uint64_t nchunks, uint64_t stride, uint64_t nreal,
                           uint64_t rows_pad, int lp, const double* __restrict__ sc, const double* __restrict__ cf,
                           const double* __restrict__ colsum, double* __restrict__ out,
                           const double* __restrict__ colmul) {
  using v4 = typename std::conditional<std::is_same<PT, float>::value, float4, int4>::type;
  const uint64_t n4 = rows_pad * (uint64_t)lp / 4;
  GRID_STRIDE(t4, n4) {
    const uint64_t t = 4 * t4;
    const uint64_t j = t / lp;
    const int l = (int)(t - j * lp);
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    if (j < nreal) {
      double y[4] = {0.0, 0.0, 0.0, 0.0};
      for (uint64_t c = 0; c < nchunks; ++c) {
        const v4 a = *reinterpret_cast<const v4*>(part + c * stride + t);
        y[0] += (double)a.x, y[1] += (double)a.y, y[2] += (double)a.z, y[3] += (double)a.w;
      }
      const double s = sc[j], beta = s * (0.5 - cf[j]);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (colmul) y[q] *= colmul[l + q];
        v[q] = 0.25 * s * y[q] + beta * colsum[l + q];
      }
    }
    double2* o = reinterpret_cast<double2*>(out + t);
    o[0] = double2{v[0], v[1]};
    o[1] = double2{v[2], v[3]};
  }
}

// The largest of each column's RG values in red -> maxbits.  Every block's atomics
// go to the same lp words and are served one after another (164,000 of them from
// 2,048 blocks took 35 us), so that kernels with this at their end take at most
// kMaxBlocks blocks.
constexpr unsigned kMaxBlocks = 1024;
__device__ __forceinline__ void block_colmax(const double* red, int RG, int lp,
                                             unsigned long long* __restrict__ maxbits) {
  __syncthreads();
  if ((int)threadIdx.x < lp) {
    double mx = 0.0;
    for (int q = 0; q < RG; ++q) mx = fmax(mx, red[q * lp + threadIdx.x]);
    if (mx > 0.0) atomicMax(&maxbits[threadIdx.x], (unsigned long long)__double_as_longlong(mx));
  }
}

// k_epi_g_v4 for the column-scaled forms without missing entries, together with
// the column maxima of |sc_j out| (k_colmax with rowscale = sc): a thread keeps
// four columns of every (blocks x RG)-th row, so the maxima stay in registers and
// what was written is not read again.  Bound by memory (the chunks of partials
// and the FP64 rows).  1,000,000 x 80, 3 chunks: 311 us against 314 and 168 for the
// two kernels.
template <class PT>
__global__ void __launch_bounds__(256) k_epi_g_max(const PT* __restrict__ part, uint64_t nchunks, uint64_t stride,
                                                   uint64_t nrows, int lp, const double* __restrict__ sc,
                                                   const double* __restrict__ cf, const double* __restrict__ colsum,
                                                   double* __restrict__ out, const double* __restrict__ colmul,
                                                   unsigned long long* __restrict__ maxbits) {
  using v4 = typename std::conditional<std::is_same<PT, float>::value, float4, int4>::type;
  __shared__ double red[1024];  // RG lp values
  const int CG = lp / 4, RG = 256 / CG, cg = threadIdx.x % CG, rg = threadIdx.x / CG;
  if (rg < RG) {
    double cs[4], cm[4], mx[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 4; ++q) cs[q] = colsum[4 * cg + q], cm[q] = colmul[4 * cg + q];
    for (uint64_t j = (uint64_t)blockIdx.x * RG + rg; j < nrows; j += (uint64_t)gridDim.x * RG) {
      const uint64_t t = j * lp + 4 * cg;
      const double s = sc[j], beta = s * (0.5 - cf[j]);
      double y[4] = {0.0, 0.0, 0.0, 0.0};
      for (uint64_t c = 0; c < nchunks; c += 4) {  // four chunks in flight, added in order
        v4 a[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (c + u < nchunks) a[u] = *reinterpret_cast<const v4*>(part + (c + u) * stride + t);
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (c + u < nchunks)
            y[0] += (double)a[u].x, y[1] += (double)a[u].y, y[2] += (double)a[u].z, y[3] += (double)a[u].w;
      }
      double v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[q] = fma(0.25 * s, y[q] * cm[q], beta * cs[q]);
        mx[q] = fmax(mx[q], fabs(v[q] * s));
      }
      double2* o = reinterpret_cast<double2*>(out + t);
      o[0] = double2{v[0], v[1]};
      o[1] = double2{v[2], v[3]};
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) red[rg * lp + 4 * cg + q] = mx[q];
  }
  block_colmax(red, RG, lp, maxbits);
}

// Fused G epilogue for data without missing entries.  A workgroup takes 64
// SNP rows of the window: reduces the split-K partials, applies the affine
// correction (G_j = sc_j/4 y_j + sc_j (1/2 - cF_j) colsum), splits sc_j G_j
// into operand pieces, writes G~ = sum(pieces)/sc_j (FP64, row-major), the
// pieces transposed through LDS (coalesced along SNPs) and the per-block
// column sums of beta_j G~_j with beta_j = sc_j (1/2 - cF_j).  Each thread
// owns 4 adjacent columns (16-byte partial loads) of every RG-th row; its
// beta sums stay in registers and are combined across row groups in LDS.
// Bound by reading the partials (all split-K chunks) on long windows and by a
// tile's chain of loads on short ones, so 16 16-byte loads are in flight: 64
// windows of 500,000 SNPs, L = 40, 10 chunks each: 24 us on average against 36
// with a row and a chunk at a time.  The margins cost a kernel of their own (4 to
// 5 us) before.
template <Form F, class PT>
__global__ void __launch_bounds__(256) k_epi_g_fused(const PT* __restrict__ part, uint64_t nchunks, uint64_t stride,
                                                     uint64_t nwin, int lp, const double* __restrict__ sc,
                                                     const double* __restrict__ cf, const double* __restrict__ colsum,
                                                     double* __restrict__ gout, void* Wt, uint64_t wpitch,
                                                     uint64_t wpiece, double* __restrict__ bpart, uint32_t left,
                                                     uint32_t right) {
  using PF = Pieces<F>;
  using w_t = typename PF::w_t;
  constexpr int P = PF::P;
  extern __shared__ __align__(16) unsigned char sm[];
  constexpr int PITCH = epi_pitch(sizeof(w_t));
  w_t* pt = reinterpret_cast<w_t*>(sm);  // P x lp rows of PITCH (kEpiRows used)
  double* bred = reinterpret_cast<double*>(sm + ((size_t)P * lp * PITCH * sizeof(w_t) + 15) / 16 * 16);
  const int CG = lp / 4, RG = 256 / CG;  // column groups of 4, row groups
  const int tid = threadIdx.x, cg = tid % CG, rg = tid / CG;
  const bool act = rg < RG;
  const uint64_t r0 = (uint64_t)blockIdx.x * kEpiRows;
  const int nr = (int)(nwin - r0 < (uint64_t)kEpiRows ? nwin - r0 : kEpiRows);
  double b4[4] = {0.0, 0.0, 0.0, 0.0};
  if (act) {
    constexpr int B = 16 / sizeof(PT), NC = B;  // rows and chunks in flight
    double cs[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) cs[q] = colsum[4 * cg + q];
    for (int rb = rg; rb < nr; rb += B * RG) {
      double y[B][4], sj[B], cj[B];
#pragma unroll
      for (int u = 0; u < B; ++u) {
        const bool in = rb + u * RG < nr;
        sj[u] = in ? sc[r0 + rb + u * RG] : 0.0;
        cj[u] = in ? cf[r0 + rb + u * RG] : 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) y[u][q] = 0.0;
      }
      // the partials' chunks in order, NC of them in flight at a time
      const auto take = [&](auto nc_tag, uint64_t c) {
        constexpr int C = decltype(nc_tag)::value;
        PT v[C][B][4];
#pragma unroll
        for (int i = 0; i < C; ++i)
#pragma unroll
          for (int u = 0; u < B; ++u) {
            const bool in = rb + u * RG < nr;
            const PT* p = part + (c + i) * stride + (in ? r0 + rb + u * RG : r0) * lp + 4 * cg;
            if constexpr (sizeof(PT) == 4) {
              *reinterpret_cast<float4*>(v[i][u]) = *reinterpret_cast<const float4*>(p);
            } else {
              *reinterpret_cast<double2*>(v[i][u]) = *reinterpret_cast<const double2*>(p);
              *reinterpret_cast<double2*>(v[i][u] + 2) = *reinterpret_cast<const double2*>(p + 2);
            }
          }
#pragma unroll
        for (int i = 0; i < C; ++i)
#pragma unroll
          for (int u = 0; u < B; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) y[u][q] += (double)v[i][u][q];
      };
      uint64_t c = 0;
      for (; c + NC <= nchunks; c += NC) take(std::integral_constant<int, NC>{}, c);
      for (; c < nchunks; ++c) take(std::integral_constant<int, 1>{}, c);
#pragma unroll
      for (int u = 0; u < B; ++u) {
        const int r = rb + u * RG;
        if (r >= nr) break;
        const uint64_t t = (r0 + r) * lp + 4 * cg;
        const double s = sj[u], is = 1.0 / s;
        const double beta = s * (0.5 - cj[u]);
        double gr4[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double g = fma(0.25 * s, y[u][q], beta * cs[q]);
          w_t pc[P];
          const double back = PF::make(g * s, 1.0, pc);
          gr4[q] = s != 0.0 ? quotient_any(back, s, is) : 0.0;
          b4[q] += beta * gr4[q];
#pragma unroll
          for (int p = 0; p < P; ++p) pt[(p * lp + 4 * cg + q) * PITCH + r] = pc[p];
        }
        *reinterpret_cast<double2*>(gout + t) = double2{gr4[0], gr4[1]};
        *reinterpret_cast<double2*>(gout + t + 2) = double2{gr4[2], gr4[3]};
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) bred[rg * lp + 4 * cg + q] = b4[q];
  }
  __syncthreads();
  store_pieces(pt, P, lp, static_cast<w_t*>(Wt), wpitch, wpiece, r0, nr, left, nwin, right);
  for (int l = threadIdx.x; l < lp; l += 256) {
    double sum = 0.0;
    for (int q = 0; q < RG; ++q) sum += bred[q * lp + l];
    bpart[(uint64_t)blockIdx.x * lp + l] = sum;
  }
}

template <class P>
__global__ void k_epi_h(const P* __restrict__ part, uint64_t nchunks, uint64_t stride, uint64_t nreal,
                        uint64_t rows_pad, int lp, const double* __restrict__ b, double* __restrict__ out, int mode,
                        const double* __restrict__ colmul) {
  const uint64_t n = rows_pad * (uint64_t)lp;
  GRID_STRIDE(t, n) {
    const uint64_t i = t / lp;
    const int l = (int)(t - i * lp);
    if (i < nreal) {
      double y = 0.0;
      for (uint64_t c = 0; c < nchunks; ++c) y += (double)part[c * stride + t];
      if (colmul) y *= colmul[l];
      const double v = 0.25 * y + b[l];
      out[t] = mode ? out[t] + v : v;
    } else if (!mode) {
      out[t] = 0.0;
    }
  }
}

// The same for FP32 partials, 4 adjacent elements of one row per thread:
// 16-byte partial loads, four chunks loaded ahead of their additions, each
// element's chunks still added in chunk order.  Needs lp and the chunk
// stride to be multiples of 4 and 16-byte aligned partials.
__global__ void k_epi_h_f4(const float* __restrict__ part, uint64_t nchunks, uint64_t stride, uint64_t nreal,
                           uint64_t rows_pad, int lp, const double* __restrict__ b, double* __restrict__ out, int mode,
                           const double* __restrict__ colmul) {
  const uint64_t n4 = rows_pad * (uint64_t)lp / 4;
  GRID_STRIDE(t4, n4) {
    const uint64_t t = 4 * t4;
    const uint64_t i = t / lp;
    const int l = (int)(t - i * lp);
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    if (i < nreal) {
      double y[4] = {0.0, 0.0, 0.0, 0.0};
      const float* p = part + t;
      uint64_t c = 0;
      for (; c + 4 <= nchunks; c += 4) {
        float4 a[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) a[u] = *reinterpret_cast<const float4*>(p + (c + u) * stride);
#pragma unroll
        for (int u = 0; u < 4; ++u)
          y[0] += (double)a[u].x, y[1] += (double)a[u].y, y[2] += (double)a[u].z, y[3] += (double)a[u].w;
      }
      for (; c < nchunks; ++c) {
        const float4 a = *reinterpret_cast<const float4*>(p + c * stride);
        y[0] += (double)a.x, y[1] += (double)a.y, y[2] += (double)a.z, y[3] += (double)a.w;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (colmul) y[q] *= colmul[l + q];
        v[q] = 0.25 * y[q] + b[l + q];
      }
    } else if (mode) {
      continue;
    }
    double2* o = reinterpret_cast<double2*>(out + t);
    if (mode) {
      const double2 o0 = o[0], o1 = o[1];
      v[0] += o0.x, v[1] += o0.y, v[2] += o1.x, v[3] += o1.y;
    }
    o[0] = double2{v[0], v[1]};
    o[1] = double2{v[2], v[3]};
  }
}

// Column maxima of |X[r][l] rowscale[r]| over rows [0, nreal): each block
// reduces its rows in LDS and raises maxbits[l] (the bit pattern of a
// non-negative double orders like the value) with one atomic per column.  50,000 x
// 80: 15 us against 42 with a column per thread and 2,048 blocks.
__global__ void __launch_bounds__(256) k_colmax(const double* __restrict__ X, uint64_t nreal, int lp,
                                                const double* __restrict__ rowscale,
                                                unsigned long long* __restrict__ maxbits) {
  __shared__ double red[1024];  // RG lp values
  const int CG = lp / 4, RG = 256 / CG, cg = threadIdx.x % CG, rg = threadIdx.x / CG;
  if (rg < RG) {
    double mx[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (uint64_t r = (uint64_t)blockIdx.x * RG + rg; r < nreal; r += (uint64_t)gridDim.x * RG) {
      const double rs = rowscale ? rowscale[r] : 1.0;
      const double2 a = *reinterpret_cast<const double2*>(X + r * lp + 4 * cg);
      const double2 b = *reinterpret_cast<const double2*>(X + r * lp + 4 * cg + 2);
      mx[0] = fmax(mx[0], fabs(a.x * rs)), mx[1] = fmax(mx[1], fabs(a.y * rs));
      mx[2] = fmax(mx[2], fabs(b.x * rs)), mx[3] = fmax(mx[3], fabs(b.y * rs));
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) red[rg * lp + 4 * cg + q] = mx[q];
  }
  block_colmax(red, RG, lp, maxbits);
}

__global__ void k_zero_u64(unsigned long long* __restrict__ p, int n) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0ull;
}

// Column scales from the column maxima (1 for an all-zero column): I8
// s_l = max_l / kI8Max with epilogue factor 2 s_l; F8 s_l = 2^ceil(log2(max_l
// / 448)) (the column maximum lands in (224, 448]) with factor s_l.
__global__ void k_col_scales(const unsigned long long* __restrict__ maxbits, int lp, int f8, double* __restrict__ scale,
                             double* __restrict__ mul) {
  const int l = threadIdx.x;
  if (l >= lp) return;
  const double mx = __longlong_as_double((long long)maxbits[l]);
  double s = 1.0;
  if (mx > 0.0) {
    if (f8) {
      int e;
      const double f = frexp(mx / 448.0, &e);  // mx / 448 = f 2^e, f in [0.5, 1)
      s = ldexp(1.0, f == 0.5 ? e - 1 : e);    // smallest power of two >= mx / 448
    } else {
      s = mx / (double)kI8Max;
    }
  }
  scale[l] = s;
  mul[l] = f8 ? s : 2.0 * s;
}

// Stage 1 of a column reduction: block b sums rows [r0 + b*rpb, ...) for each column.
__global__ void k_colsum_partial(const double* __restrict__ X, uint64_t r0, uint64_t r1, int lp, uint64_t rpb,
                                 const double* __restrict__ sc, const double* __restrict__ cf,
                                 double* __restrict__ partial) {
  const uint64_t rb = r0 + (uint64_t)blockIdx.x * rpb;
  const uint64_t re = rb + rpb < r1 ? rb + rpb : r1;
  for (int l = threadIdx.x; l < lp; l += blockDim.x) {
    double s = 0.0;
    for (uint64_t r = rb; r < re; ++r) {
      const double w = sc ? sc[r] * (0.5 - cf[r]) : 1.0;
      s += w * X[r * lp + l];
    }
    partial[(uint64_t)blockIdx.x * lp + l] = s;
  }
}

// Sums of per-block partials, deterministic.  A workgroup owns 32
// consecutive outputs t of one slice of blocks: its 8 thread rows take every
// 8th block of the slice (coalesced 32-wide reads), combined in LDS in a
// fixed order.  Block b of the input sits at partial[b * bstride * width].
// With dst == partial (the first stage of a long reduction) the slice's sum
// replaces its first block; every workgroup reads its whole slice first.
__global__ void __launch_bounds__(256) k_sum_partials(double* partial, uint64_t nblocks, uint64_t width,
                                                      uint64_t bstride, uint64_t slice, double* dst) {
  __shared__ double red[8][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const uint64_t t = (uint64_t)blockIdx.x * 32 + tx;
  const uint64_t b0 = (uint64_t)blockIdx.y * slice;
  const uint64_t b1 = b0 + slice < nblocks ? b0 + slice : nblocks;
  const uint64_t step = bstride * width;
  double s0 = 0.0, s1 = 0.0;
  if (t < width) {
    uint64_t b = b0 + ty;
    for (; b + 8 < b1; b += 16) {
      s0 += partial[b * step + t];
      s1 += partial[(b + 8) * step + t];
    }
    if (b < b1) s0 += partial[b * step + t];
  }
  red[ty][tx] = s0 + s1;
  __syncthreads();
  if (ty == 0 && t < width) {
    double s = 0.0;
    for (int r = 0; r < 8; ++r) s += red[r][tx];
    if (dst == partial)
      partial[b0 * step + t] = s;
    else
      dst[t] = s;
  }
}

// out[t] = sum_b partial[b][t] for b < nblocks (partial is scratch: a long
// reduction first folds slices of 64 blocks in place).
inline void sum_partials(double* partial, uint64_t nblocks, uint64_t width, double* out, hipStream_t s) {
  const unsigned gx = (unsigned)((width + 31) / 32);
  constexpr uint64_t kSlice = 64;
  if (nblocks > 4 * kSlice) {
    const uint64_t ns = (nblocks + kSlice - 1) / kSlice;
    hipLaunchKernelGGL(k_sum_partials, dim3(gx, (unsigned)ns), dim3(256), 0, s, partial, nblocks, width, (uint64_t)1,
                       kSlice, partial);
    hipLaunchKernelGGL(k_sum_partials, dim3(gx, 1), dim3(256), 0, s, partial, ns, width, kSlice, ns, out);
    return;
  }
  hipLaunchKernelGGL(k_sum_partials, dim3(gx, 1), dim3(256), 0, s, partial, nblocks, width, (uint64_t)1, nblocks, out);
}

// What a Gram kernel multiplies: X^T X, X^T Y, (X + Y)^T (X + Y) with the sum
// written to Z, or (X T)^T (X T) for an LP x LP T.
enum GramMode : int { kGramSelf, kGramCross, kGramAdd, kGramApply };

// Rows staged per step, waves, and the LDS pitch (not a multiple of 32 values:
// the four rows of one MFMA operand lie in different banks).
constexpr int gram_tile_rows(int nb, int mode) {
  return nb <= 2 ? (mode == kGramCross ? 64 : 128) : (nb <= 5 ? (mode == kGramCross ? 32 : 64) : 32);
}
constexpr int gram_waves(int nb) { return nb <= 2 ? 4 : 8; }
constexpr int gram_pitch(int nb) { return 16 * nb + (nb % 2 ? 0 : 16); }
constexpr size_t gram_lds(int nb, int mode) {
  return ((size_t)gram_tile_rows(nb, mode) * gram_pitch(nb) * (mode == kGramCross ? 2 : 1) +
          (mode == kGramApply ? (size_t)256 * nb * nb : 0)) * sizeof(double);
}

// FP64-MFMA Gram partials: block b sums X[r]^T Y[r] over rows [b*rpb, ...).
// Cross products: the NB^2 16 x 16 output blocks are dealt round robin to the
// waves.  X^T X: only the NB (NB + 1) / 2 upper blocks, each also stored
// mirrored (the products are commutative, so the result is exactly symmetric).
// Row tiles of X (and Y) are staged in LDS, the next one loaded into
// registers meanwhile.  v_mfma_f64_16x16x4: A = X^T (lane l: X[k0 + l/16][16i +
// l%16]), B = Y (lane l: Y[k0 + l/16][16j + l%16]), accumulator lane group q,
// register r = output row q + 4r.
// At N of some thousands a block has one or a few tiles and is bound by the
// latencies in a row: the tiles are as high as LDS and registers allow (one
// wave per 16 columns with tiles of 32 rows took 11.5 us at 2,000 x 32 and 13.5
// us at 10,000 x 48, against 5.0 and 6.1 us).  kGramApply forms its tile of X T in
// LDS and never writes it (8.0 and 11.4 us, against 4.7 + 11.5 and 7.7 + 13.5 us
// for the product and its Gram); kGramAdd sums H1 + H2 on the way.
template <int NB, int MODE>
__global__ void __launch_bounds__(64 * gram_waves(NB)) k_gram(const double* __restrict__ X,
                                                              const double* __restrict__ Y, uint64_t nrows,
                                                              uint64_t rpb, double* __restrict__ partial,
                                                              double* __restrict__ Z) {
  constexpr int LP = NB * 16, P = gram_pitch(NB), TR = gram_tile_rows(NB, MODE), W = gram_waves(NB), NT = 64 * W;
  constexpr bool CROSS = MODE == kGramCross, APPLY = MODE == kGramApply;
  extern __shared__ __align__(16) double gm[];
  double *xs = gm, *ys = CROSS ? xs + TR * P : xs, *tl = xs + TR * P;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int q = lane >> 4, r16 = lane & 15;
  constexpr int NBLK = CROSS ? NB * NB : NB * (NB + 1) / 2, S = (NBLK + W - 1) / W;
  f64x4_t acc[S];
  int ci[S], cj[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    acc[s] = f64x4_t{0, 0, 0, 0};
    const int t = __builtin_amdgcn_readfirstlane(wave + W * s);
    ci[s] = t < NBLK ? 16 * (CROSS ? t / NB : sym_block_i(t, NB)) : 0;
    cj[s] = t < NBLK ? 16 * (CROSS ? t % NB : sym_block_j(t, NB)) : 0;
  }
  const uint64_t rb = (uint64_t)blockIdx.x * rpb;
  const uint64_t re = rb + rpb < nrows ? rb + rpb : nrows;
  // 16-byte pairs per thread and tile; rows past the block's end read as zero
  constexpr int PER = (TR * LP / 2 + NT - 1) / NT;
  constexpr bool EVEN = PER * NT * 2 == TR * LP;
  double2 px[APPLY ? 1 : PER], py[CROSS || MODE == kGramAdd ? PER : 1];
  auto fetch = [&](uint64_t r0) {
    const int nr = (int)(re - r0 < (uint64_t)TR ? re - r0 : TR);
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int v = 2 * (tid + e * NT);
      const bool in = v / LP < nr;  // nr <= TR: also past a tile that the threads cover unevenly
      px[e] = in ? *reinterpret_cast<const double2*>(X + r0 * LP + v) : double2{0.0, 0.0};
      if constexpr (CROSS || MODE == kGramAdd)
        py[e] = in ? *reinterpret_cast<const double2*>(Y + r0 * LP + v) : double2{0.0, 0.0};
    }
  };
  if constexpr (APPLY) {
    for (int v = tid; v < LP * LP; v += NT) tl[v] = Y[v];  // Y = T
  } else {
    if (rb < re) fetch(rb);
  }
  for (uint64_t r0 = rb; r0 < re; r0 += TR) {
    __syncthreads();
    if constexpr (APPLY) {
      // xs = X T for this tile: 16-row blocks dealt to the waves, k ascending
      for (int i = wave; i < TR / 16; i += W) {
        const uint64_t row = r0 + 16 * i + r16;
        const bool in = row < re;
        const double* x = X + row * LP;
        double av[LP / 4];
#pragma unroll
        for (int k = 0; k < LP / 4; ++k) av[k] = in ? x[4 * k + q] : 0.0;
        f64x4_t y[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) y[b] = f64x4_t{0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < LP / 4; ++k)
#pragma unroll
          for (int b = 0; b < NB; ++b)
            y[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[k], tl[(4 * k + q) * LP + 16 * b + r16], y[b], 0, 0, 0);
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) xs[(16 * i + q + 4 * r) * P + 16 * b + r16] = y[b][r];
      }
    } else {
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        const int v = 2 * (tid + e * NT), at = v / LP * P + v % LP;
        if (!EVEN && v >= TR * LP) continue;
        if constexpr (MODE == kGramAdd) {
          px[e].x += py[e].x, px[e].y += py[e].y;
          if (r0 + v / LP < re) *reinterpret_cast<double2*>(Z + r0 * LP + v) = px[e];
        }
        *reinterpret_cast<double2*>(xs + at) = px[e];
        if constexpr (CROSS) *reinterpret_cast<double2*>(ys + at) = py[e];
      }
    }
    __syncthreads();
    if constexpr (!APPLY) {
      if (r0 + TR < re) fetch(r0 + TR);
    }
#pragma unroll 8
    for (int k0 = 0; k0 < TR; k0 += 4) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        if (wave + W * s < NBLK)
          acc[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(xs[(k0 + q) * P + ci[s] + r16], ys[(k0 + q) * P + cj[s] + r16],
                                                        acc[s], 0, 0, 0);
      }
    }
  }
  double* o = partial + (uint64_t)blockIdx.x * LP * LP;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    if (wave + W * s < NBLK) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        o[(ci[s] + q + 4 * r) * LP + cj[s] + r16] = acc[s][r];
        if (!CROSS && ci[s] != cj[s]) o[(cj[s] + r16) * LP + ci[s] + q + 4 * r] = acc[s][r];  // the mirror block
      }
    }
  }
}

// FP64-MFMA right multiplication Y = X T for rows [0, nrows): one wave per 16
// rows computes all NB column blocks; A = X (lane l: X[16i + l%16][k0 + l/16]),
// B = T (lane l: T[k0 + l/16][16b + l%16]).  T is staged in LDS.
// FLIP: also this block's flipOmg norms of the Y it holds in registers,
// sum |O2 - Y| and sum |O2 + Y| per column, into partial[block][2 LP].  A pass
// of their own over O2 and Y, in blocks of 128 threads that walked their rows
// one after another, took 23-34 us and two reductions behind it per Omega
// update at N = 10,000-50,000; the norms add 3 us (L = 40, N = 10,000) to 12 us
// (L = 80, N = 50,000) to the product.
template <int NB, bool FLIP>
__global__ void __launch_bounds__(256) k_apply_mfma(const double* __restrict__ X, const double* __restrict__ T,
                                                    uint64_t nrows, double* __restrict__ Y,
                                                    const double* __restrict__ O2, double* __restrict__ partial) {
  constexpr int LP = NB * 16;
  extern __shared__ double tl[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int q = lane >> 4, r16 = lane & 15;
  for (int v = tid; v < LP * LP; v += 256) tl[v] = T[v];
  __syncthreads();
  double fa[FLIP ? NB : 1], fb[FLIP ? NB : 1];
  if constexpr (FLIP) {
#pragma unroll
    for (int b = 0; b < NB; ++b) fa[b] = fb[b] = 0.0;
  }
  const uint64_t nblk = (nrows + 15) / 16;
  for (uint64_t blk = (uint64_t)blockIdx.x * 4 + wave; blk < nblk; blk += (uint64_t)gridDim.x * 4) {
    const uint64_t row = blk * 16 + r16;
    const double* x = X + row * LP;
    const bool in = row < nrows;
    f64x4_t acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b] = f64x4_t{0, 0, 0, 0};
#pragma unroll 4
    for (int k0 = 0; k0 < LP; k0 += 4) {
      const double av = in ? x[k0 + q] : 0.0;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const double bv = tl[(k0 + q) * LP + 16 * b + r16];
        acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, acc[b], 0, 0, 0);
      }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint64_t orow = blk * 16 + q + 4 * r;
        if (orow < nrows) {
          Y[orow * LP + 16 * b + r16] = acc[b][r];
          if constexpr (FLIP) {
            const double o = O2[orow * LP + 16 * b + r16];
            fa[b] += fabs(o - acc[b][r]);
            fb[b] += fabs(o + acc[b][r]);
          }
        }
      }
  }
  if constexpr (FLIP) {
    __syncthreads();  // T has been read: its LDS takes the waves' sums, [wave][2 LP] (8 LP <= LP LP values)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      fa[b] += __shfl_xor(fa[b], 16);
      fa[b] += __shfl_xor(fa[b], 32);
      fb[b] += __shfl_xor(fb[b], 16);
      fb[b] += __shfl_xor(fb[b], 32);
      if (q == 0) {
        tl[wave * 2 * LP + 16 * b + r16] = fa[b];
        tl[wave * 2 * LP + LP + 16 * b + r16] = fb[b];
      }
    }
    __syncthreads();
    for (int t = tid; t < 2 * LP; t += 256) {
      double sum = 0.0;
#pragma unroll
      for (int w = 0; w < 4; ++w) sum += tl[w * 2 * LP + t];
      partial[(uint64_t)blockIdx.x * 2 * LP + t] = sum;
    }
  }
}

__global__ void k_flip_partial(const double* __restrict__ O2, const double* __restrict__ Q, uint64_t nrows, int lp,
                               uint64_t rpb, double* __restrict__ partial) {
  const uint64_t rb = (uint64_t)blockIdx.x * rpb;
  const uint64_t re = rb + rpb < nrows ? rb + rpb : nrows;
  for (int l = threadIdx.x; l < lp; l += blockDim.x) {
    double a = 0.0, b = 0.0;
    for (uint64_t r = rb; r < re; ++r) {
      const double o = O2[r * lp + l], q = Q[r * lp + l];
      a += fabs(o - q);
      b += fabs(o + q);
    }
    partial[(uint64_t)blockIdx.x * 2 * lp + l] = a;
    partial[(uint64_t)blockIdx.x * 2 * lp + lp + l] = b;
  }
}

// Column-major n x L (leading dimension n) -> row-major rows_pad x lp, zero
// outside the n x L block.
__global__ void k_colmajor_to_rows(const double* __restrict__ src, uint64_t n, int L, int lp, uint64_t rows_pad,
                                   double* __restrict__ dst) {
  GRID_STRIDE(t, rows_pad * (uint64_t)lp) {
    const uint64_t r = t / lp;
    const int l = (int)(t - r * lp);
    dst[t] = (r < n && l < L) ? src[(uint64_t)l * n + r] : 0.0;
  }
}

// Row-major n x lp -> k columns of col_len values (row r at place[r] when given,
// else at r), 32 rows per workgroup through LDS: whole rows read, 256-byte runs of
// each column written (one thread per output value would read 8 bytes of every row
// line it touched).  100,003 x 40 from lp = 48: 27 us, 2.6 TB/s read and written,
// half of a copy's rate: a workgroup reads, waits, and writes 12 KB once.
__global__ void __launch_bounds__(256) k_rows_to_colmajor(const double* __restrict__ src, uint64_t n, int lp, int k,
                                                          double* __restrict__ dst, uint64_t col_len,
                                                          const uint32_t* __restrict__ place) {
  extern __shared__ double tile[];  // 32 rows of lp + 1
  const uint64_t r0 = (uint64_t)blockIdx.x * 32;
  const int nr = (int)(n - r0 < 32 ? n - r0 : 32);
  for (int v = threadIdx.x; v < nr * lp; v += 256) {
    const int r = v / lp, l = v - r * lp;
    tile[r * (lp + 1) + l] = src[r0 * lp + v];
  }
  __syncthreads();
  for (int v = threadIdx.x; v < 32 * k; v += 256) {
    const int j = v >> 5, r = v & 31;
    if (r < nr) dst[(uint64_t)j * col_len + (place ? place[r0 + r] : r0 + r)] = tile[r * (lp + 1) + j];
  }
}

// flip_UV with V as the base (src/Utils.cpp:118-154): per column c < k of X
// (rows [0, n), pitch lp) the value at its first maximum of |x|.  Stage 1:
// block b takes rows [b rpb, ...), kAbsRows of them at a time, each thread
// one column of every kAbsRows-th row; stage 2 (one workgroup) the blocks.
// Candidates carry their row: the larger |x| wins, the smaller row on a tie,
// as Eigen's maxCoeff, whatever the order of the comparisons.  Bound by the
// latency of the loads: with one thread per column walking the blocks of 2,048
// stage 2 took 478 us; the two stages take 8.4 + 7.1 us at M = 60,000, k = 10.
struct AbsMax {
  double best, v;  // |x| (-1: none yet) and x
  uint64_t row;
  __device__ __forceinline__ void take(double b, double x, uint64_t r) {
    if (b > best || (b == best && r < row)) best = b, v = x, row = r;
  }
};

// Folds the groups' candidates of each column (threads g c-groups apart) into
// group 0's.
__device__ __forceinline__ void absmax_fold(AbsMax& m, AbsMax* red, int c, int g, int ng, int k) {
  if (g < ng) red[g * k + c] = m;
  __syncthreads();
  if (g == 0)
    for (int r = 1; r < ng; ++r) m.take(red[r * k + c].best, red[r * k + c].v, red[r * k + c].row);
}

__global__ void __launch_bounds__(256) k_col_absmax_partial(const double* __restrict__ X, uint64_t n, int lp, int k,
                                                            uint64_t rpb, double* __restrict__ pval,
                                                            uint64_t* __restrict__ prow) {
  __shared__ AbsMax red[256];
  const int ng = 256 / k, g = threadIdx.x / k, c = threadIdx.x - g * k;
  const uint64_t r0 = (uint64_t)blockIdx.x * rpb;
  const uint64_t r1 = r0 + rpb < n ? r0 + rpb : n;
  AbsMax m{-1.0, 0.0, 0};
  if (g < ng) {
#pragma unroll 4
    for (uint64_t r = r0 + g; r < r1; r += ng) {
      const double x = X[r * lp + c];
      m.take(fabs(x), x, r);
    }
  }
  absmax_fold(m, red, c, g, ng, k);
  if (g == 0) {
    pval[(uint64_t)blockIdx.x * k + c] = m.v;
    prow[(uint64_t)blockIdx.x * k + c] = m.row;
  }
}

__global__ void __launch_bounds__(256) k_col_absmax_sign(const double* __restrict__ pval,
                                                         const uint64_t* __restrict__ prow, uint64_t nb, int lp, int k,
                                                         double* __restrict__ sign) {
  __shared__ AbsMax red[256];
  const int ng = 256 / k, g = threadIdx.x / k, c = threadIdx.x - g * k;
  AbsMax m{-1.0, 0.0, 0};
  if (g < ng) {
#pragma unroll 4
    for (uint64_t b = g; b < nb; b += ng) {
      const double x = pval[b * k + c];
      m.take(fabs(x), x, prow[b * k + c]);
    }
  }
  absmax_fold(m, red, c, g, ng, k);
  if (g == 0) sign[c] = m.v < 0.0 ? -1.0 : 1.0;
  for (int l = k + threadIdx.x; l < lp; l += 256) sign[l] = 1.0;
}

__global__ void k_scale_cols(double* __restrict__ X, uint64_t n, int lp, const double* __restrict__ sign) {
  GRID_STRIDE(t, n * (uint64_t)lp) X[t] *= sign[t % lp];
}

// dst (rows x kp) = the first k columns of src (rows x lp), times scale[t]
// (null = 1), zero padded.
__global__ void k_impute_rows(const double* __restrict__ src, uint64_t rows, int lp, int k, int kp,
                              const double* __restrict__ scale, double* __restrict__ dst) {
  GRID_STRIDE(t, rows * (uint64_t)kp) {
    const uint64_t r = t / kp;
    const int c = (int)(t - r * kp);
    dst[t] = c < k ? src[r * lp + c] * (scale ? scale[c] : 1.0) : 0.0;
  }
}

// Per-SNP column state as read: cF = F and sc = 1 for j < m, zero padding to rows.
__global__ void k_pristine_cols(const double* __restrict__ F, uint64_t m, uint64_t rows, double* __restrict__ cf,
                                double* __restrict__ sc) {
  GRID_STRIDE(j, rows) {
    cf[j] = j < m ? F[j] : 0.0;
    sc[j] = j < m ? 1.0 : 0.0;
  }
}

// standardize_E's scale (src/Data.cpp:351-362): sc_j *= sqrt(ploidy) / sd_j with
// sd_j = sqrt(F_j (1 - F_j)) when sd_j > tol.
__global__ void k_standardize(const double* __restrict__ F, uint64_t m, double sqrt_ploidy, double tol,
                              double* __restrict__ sc) {
  GRID_STRIDE(j, m) {
    const double f = F[j];
    const double sd = sqrt(f * (1.0 - f));
    if (sd > tol) sc[j] *= sqrt_ploidy / sd;
  }
}

__global__ void k_gather_f64(const double* __restrict__ src, const uint32_t* __restrict__ idx, uint64_t n,
                             double* __restrict__ dst) {
  GRID_STRIDE(i, n) dst[i] = src[idx[i]];
}

__global__ void k_add(const double* __restrict__ X, const double* __restrict__ Z, double* __restrict__ Y, uint64_t n) {
  GRID_STRIDE(t, n) Y[t] = X[t] + Z[t];
}

// First list position in [lo, hi) whose index is >= key (lists are sorted).
__device__ __forceinline__ uint64_t lower_bound_ix(const uint32_t* ix, uint64_t lo, uint64_t hi, uint64_t key) {
  while (lo < hi) {
    const uint64_t mid = (lo + hi) / 2;
    if (ix[mid] < key) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// Entry range of row r restricted to indices [klo, khi).
__device__ __forceinline__ void entry_range(const uint64_t* rp, const uint32_t* ix, uint64_t r, uint64_t klo,
                                            uint64_t khi, uint64_t& e0, uint64_t& e1) {
  e0 = rp[r];
  e1 = rp[r + 1];
  if (klo > 0) e0 = lower_bound_ix(ix, e0, e1, klo);
  e1 = lower_bound_ix(ix, e0, e1, khi);
}

// Per-entry weights of the missing-entry corrections without imputation:
// w = -sc_c (1/2 - cF_c), which cancels the centering term the affine
// epilogue gave the entry.  One wave per row of the lists and index chunk
// (grid.y), lanes over the row's entries.
__global__ void k_missing_weights(MissWeightArgs a) {
  const uint64_t r = blockIdx.x * (uint64_t)(blockDim.x / 64) + threadIdx.x / 64;
  const int lane = threadIdx.x & 63;
  if (r >= a.nrows) return;
  const uint64_t klo = (uint64_t)blockIdx.y * a.kspan, khi = klo + a.kspan;
  uint64_t e0, e1;
  entry_range(a.rp, a.ix, r, klo, khi, e0, e1);
  for (uint64_t e = e0 + lane; e < e1; e += 64) {
    const uint64_t c = a.by_snp ? r : a.ix[e];  // SNP column
    a.w[e] = -a.sc[c] * (0.5 - a.cf[c]);
  }
}

// EMU weights (src/Data.cpp:318-348): w = -sc_c (1/2 - cF_c) + sc_c clamp(p, -F_c,
// 1 - F_c) with p = (U S)_i . V_c.  One wave per row of the lists (a SNP c for
// the by-SNP list, a sample i for the by-sample list) and index chunk
// (grid.y; chunks keep the gathered rows within L2).  The k-vectors are rows
// of pitch kp (whole 128-byte lines) read as 16-byte pairs, and a V row also
// carries its SNP's sc, cF and F, so an entry of the by-sample list touches
// one line.  The row's own vector sits in registers; the wave is split into
// 64 / LPE groups of LPE lanes (a power of two >= k / 2), each group taking
// one entry per step, reading the entry's vector as one contiguous access
// and reducing the dot product by butterfly shuffles.  The entries' indexes
// come 64 at a time (one coalesced load, the next batch's fetched during this
// one).
__global__ void __launch_bounds__(256) k_missing_weights_emu(MissWeightArgs a, int lpe) {
  const uint64_t r = blockIdx.x * 4ull + threadIdx.x / 64;
  const int lane = threadIdx.x & 63;
  if (r >= a.nrows) return;  // wave-uniform
  const uint64_t klo = (uint64_t)blockIdx.y * a.kspan, khi = klo + a.kspan;
  uint64_t e0, e1;
  entry_range(a.rp, a.ix, r, klo, khi, e0, e1);
  const int kk = a.kk, np = a.kp / 2;  // 16-byte pairs per row
  const int nk = (kk + 1) / 2;          // pairs holding loadings
  const int G = 64 / lpe, g = lane / lpe, cl = lane - g * lpe;
  const bool has = cl < nk;
  const double* ownrow = (a.by_snp ? a.V : a.US) + r * (uint64_t)a.kp;
  const double2* other = reinterpret_cast<const double2*>(a.by_snp ? a.US : a.V);
  // the row's own loadings (a zero past k in the last pair)
  double2 rv = double2{0.0, 0.0};
  if (has) {
    rv.x = ownrow[2 * cl];
    rv.y = 2 * cl + 1 < kk ? ownrow[2 * cl + 1] : 0.0;
  }
  double sc_r = 0.0, cf_r = 0.0, f_r = 0.0;  // the SNP's state for the by-SNP list
  if (a.by_snp) {
    sc_r = a.sc[r];
    cf_r = a.cf[r];
    f_r = a.Fclamp[r];
  }
  constexpr int U = 4;
  uint32_t nix = e0 + lane < e1 ? a.ix[e0 + lane] : 0u;
  for (uint64_t eb = e0; eb < e1; eb += 64) {
    const int nb = (int)min<uint64_t>(64, e1 - eb);
    const uint32_t myix = nix;
    nix = eb + 64 + lane < e1 ? a.ix[eb + 64 + lane] : 0u;
    const int steps = (nb + G - 1) / G;
    for (int st = 0; st < steps; st += U) {
      uint32_t kx[U];
      bool ok[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = (st + u) * G + g;
        kx[u] = __shfl(myix, j < 63 ? j : 63);
        ok[u] = j < nb;
      }
      double2 x[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        x[u] = has ? other[(ok[u] ? (uint64_t)kx[u] : 0) * np + cl] : double2{0.0, 0.0};
#pragma unroll
      for (int u = 0; u < U; ++u) {
        double p = rv.x * x[u].x + rv.y * x[u].y;
        for (int off = lpe / 2; off > 0; off >>= 1) p += __shfl_xor(p, off);
        const int j = (st + u) * G + g;
        if (cl == 0 && ok[u]) {
          double sc = sc_r, cf = cf_r, f = f_r;
          if (!a.by_snp) {  // the entry's SNP row carries its state after the loadings
            const double* vr = a.V + (uint64_t)kx[u] * a.kp + kk;
            sc = vr[0];
            cf = vr[1];
            f = vr[2];
          }
          double w = -sc * (0.5 - cf);
          w += sc * fmin(fmax(p, -f), 1.0 - f);
          a.w[eb + j] = w;
        }
      }
    }
  }
}

__global__ void k_pack_col_state(double* __restrict__ V, uint64_t m, int kp, int kk, const double* __restrict__ sc,
                                 const double* __restrict__ cf, const double* __restrict__ F) {
  GRID_STRIDE(j, m) {
    double* vr = V + j * (uint64_t)kp + kk;
    vr[0] = sc[j];
    vr[1] = cf[j];
    vr[2] = F[j];
  }
}

// out (rows x pitch, T) = the first L columns of src (rows x lp, FP64), zero padded.
template <class T>
__global__ void k_compact_rows(const double* __restrict__ src, uint64_t rows, int lp, int L, int pitch,
                               T* __restrict__ out) {
  GRID_STRIDE(t, rows * (uint64_t)pitch) {
    const uint64_t r = t / pitch;
    const int c = (int)(t - r * pitch);
    out[t] = c < L ? (T)src[r * lp + c] : (T)0;
  }
}

// Sparse correction out[r][c] (+)= sum_e w[e] src[ix[e] - src_k0][c], c < ncols,
// one wave per (target row, index chunk = grid.z).  The row's entries are
// taken 64 at a time (one coalesced load of their indexes and weights, the
// next batch's fetched during this one).  The wave is split into G groups of
// LPE = cp / VEC lanes, each lane holding VEC columns (16 bytes): per step
// every group takes one entry, receives its index and weight by lane permutes
// and reads the entry's compact source row as one contiguous access (16
// bytes per lane), accumulating in FP64.  The groups' sums are combined in a
// fixed order at the end.  With several index chunks each writes its own
// partial row (summed later in chunk order), else it adds to out.
template <class T>
__global__ void __launch_bounds__(256) k_missing_spmm(MissSpmmArgs a) {
  constexpr int VEC = 16 / sizeof(T);
  using V = typename std::conditional<sizeof(T) == 4, float4, double2>::type;
  const uint64_t r = blockIdx.x * 4ull + threadIdx.x / 64;
  const int lane = threadIdx.x & 63;
  if (r >= a.nrows) return;  // wave-uniform
  const int lpe = a.cp / VEC;  // lanes per entry (cp is a multiple of VEC)
  const int G = 64 / lpe;      // entries per step
  const uint64_t rpv = a.cpitch / VEC;  // 16-byte vectors per source row (whole cache lines)
  const int g = lane / lpe, cl = lane - g * lpe;
  const bool act = g < G;
  const uint64_t klo = a.k_lo + (uint64_t)blockIdx.z * a.kspan;
  const uint64_t khi = min(a.k_hi, klo + a.kspan);
  uint64_t e0, e1;
  entry_range(a.rp, a.ix, r, klo, khi, e0, e1);
  double acc[VEC];
#pragma unroll
  for (int q = 0; q < VEC; ++q) acc[q] = 0.0;
  const V* src = static_cast<const V*>(a.src);
  constexpr int U = 4;  // steps per pass: their gathers are issued together
  uint32_t nix = 0;
  double nw = 0.0;
  if (e0 + lane < e1) {
    nix = a.ix[e0 + lane];
    nw = a.w[e0 + lane];
  }
  for (uint64_t eb = e0; eb < e1; eb += 64) {
    const int nb = (int)min<uint64_t>(64, e1 - eb);
    const uint32_t myix = nix;
    const double myw = nw;
    if (eb + 64 + lane < e1) {
      nix = a.ix[eb + 64 + lane];
      nw = a.w[eb + 64 + lane];
    }
    const int steps = (nb + G - 1) / G;
    // an entry past the batch (or an idle lane) reads source row 0 and is
    // left out of the sum
    for (int st = 0; st < steps; st += U) {
      uint32_t kk[U];
      double ww[U];
      bool ok[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = (st + u) * G + g;
        const int jl = j < 63 ? j : 63;  // every lane takes part in the permutes
        kk[u] = __shfl(myix, jl);
        ww[u] = __shfl(myw, jl);
        ok[u] = act && j < nb;
      }
      V xv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) xv[u] = src[(ok[u] ? (uint64_t)kk[u] - a.src_k0 : 0) * rpv + cl];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const T* x = reinterpret_cast<const T*>(&xv[u]);
        if (ok[u]) {
#pragma unroll
          for (int q = 0; q < VEC; ++q) acc[q] += ww[u] * (double)x[q];
        }
      }
    }
  }
  // group 0 lane cl += the same lane of groups 1 .. G-1, in order
#pragma unroll
  for (int q = 0; q < VEC; ++q) {
    const double v = acc[q];
    double tot = v;
    for (int gg = 1; gg < G; ++gg) {
      const int sl = cl + gg * lpe;
      tot += __shfl(v, sl < 63 ? sl : 63);
    }
    acc[q] = tot;
  }
  if (g != 0) return;
  const bool partial = gridDim.z > 1;
  double* o = partial ? a.partial + ((uint64_t)blockIdx.z * a.nrows + r) * a.ncols : a.out + r * a.lp;
#pragma unroll
  for (int q = 0; q < VEC; ++q) {
    const int c = cl * VEC + q;
    if (c < a.ncols) o[c] = partial ? acc[q] : o[c] + acc[q];
  }
}

// ---- L x L steps of the thin-Q of H on the device (one workgroup each) ----
// Serial chains: n pivots of a Cholesky factorization, n rows of a triangular
// inverse, n pivots of a modified LU.  What bounds them is one wave's issue and
// the latency between one pivot and the next, so a panel of 16 pivots runs
// inside one wave with its registers indexed by constants only (lane = matrix
// column, registers = the panel's 16 rows, row broadcasts in place of LDS and
// barriers), a root and its reciprocal come from one approximation, the inverse
// gives each column of the result to four lanes of one wave and reads the
// factors of four rows ahead, and the 16-row updates between panels and the
// products are FP64 MFMAs.  v_mfma_f64_16x16x4 adds its four products to the
// accumulator one after another in ascending k as fused multiply-adds, so every
// element of T sees the operations of the unblocked elimination in the same order
// with the same roundings, and the results are the same bits (a rounding more or
// less here is a different FP32 Omega, and other signs of U's columns, in one run
// of six).
// One element per thread of a 16 x 16 grid and a barrier per pivot, then the
// panels with the later pivots' registers behind an index register, then this
// form, first + second kernel: L = 20 17 + 29 -> 13 + 19 -> 10 + 15 us, L = 40
// 48 + 79 -> 22 + 35 -> 17 + 30 us, L = 80 146 + 259 -> 43 + 77 -> 34 + 66 us.
constexpr int kThinqThreads = 512;
constexpr int kThinqMaxNB = 5;  // lp <= 80

template <int NB>
constexpr size_t thinq_lds() {
  return ((size_t)2 * NB * 16 * kLP<NB> + 3 * NB * 16 + 2) * sizeof(double);
}

// First pass: R1 = chol(G1), T1 = R1^-1 (lp x lp, zero padded; zero on
// breakdown).
template <int NB>
__global__ void __launch_bounds__(kThinqThreads) k_thinq_first(const double* __restrict__ G1, int n,
                                                               double* __restrict__ R1, double* __restrict__ T1,
                                                               int* __restrict__ status, double min_ratio) {
  constexpr int LP = NB * 16, P = kLP<NB>;
  extern __shared__ __align__(16) double lm[];
  double *A = lm, *rt = A + LP * P, *invd = rt + LP * P, *scal = invd + 3 * LP;
  int* flag = reinterpret_cast<int*>(scal + 1);
  const int tid = threadIdx.x;
  lds_load<NB, kThinqThreads>(A, G1, n, true);
  // largest diagonal entry of the Gram (before the factorization overwrites it)
  if (min_ratio > 0.0 && tid < 64) {
    double mx = 0.0;
    for (int i = tid; i < n; i += 64) mx = fmax(mx, G1[i * LP + i]);
    for (int d = 32; d > 0; d >>= 1) mx = fmax(mx, __shfl_xor(mx, d));
    if (tid == 0) scal[0] = mx;
  }
  __syncthreads();
  double dmin = 0.0;
  const bool ok = lds_chol_upper<NB, kThinqThreads>(A, n, &dmin, flag);
  if (!ok) {
    if (tid == 0) *status = 1;
    for (int v = tid; v < LP * LP; v += kThinqThreads) R1[v] = T1[v] = 0.0;
    return;
  }
  // the host's safety test of this Gram (smallest pivot / largest diagonal),
  // when the caller defers it to the device: a near rank-deficient H is marked
  if (min_ratio > 0.0 && tid == 0 && !(dmin > min_ratio * scal[0])) *status = 2;
  for (int v = tid; v < LP * LP; v += kThinqThreads) R1[v] = A[v / LP * P + v % LP];
  double x[4 * NB];
  lds_inv_upper<NB, kThinqThreads>(A, rt, invd, n, x);
  __syncthreads();  // R has been read: A takes X, so that its rows leave whole
  if (tid < 4 * LP) {
#pragma unroll
    for (int m = 0; m < 4 * NB; ++m) A[(4 * m + (tid & 3)) * P + (tid >> 2)] = x[m];
  }
  __syncthreads();
  for (int v = tid; v < LP * LP; v += kThinqThreads) T1[v] = A[v / LP * P + v % LP];
}

// Second pass: R2 = chol(G2), R^-1 = (R2 R1)^-1, the Householder signs s of
// Xtop R^-1 (Xtop = the first n rows of the thinned matrix) and
// T = R^-1 diag(s) (lp x lp, zero padded; zero on breakdown).
template <int NB>
__global__ void __launch_bounds__(kThinqThreads) k_thinq_second(const double* __restrict__ G2,
                                                                const double* __restrict__ R1,
                                                                const double* __restrict__ Xtop, int n,
                                                                double* __restrict__ T, int* __restrict__ status) {
  constexpr int LP = NB * 16, P = kLP<NB>, NW = kThinqThreads / 64;
  extern __shared__ __align__(16) double lm[];
  double *A = lm, *B = A + LP * P, *invd = B + LP * P, *sgn = invd + LP, *scal = invd + 3 * LP;
  int* flag = reinterpret_cast<int*>(scal + 1);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  lds_load<NB, kThinqThreads>(A, G2, n, true);
  lds_load<NB, kThinqThreads>(B, R1, n, true);
  __syncthreads();
  double dmin;
  if (!lds_chol_upper<NB, kThinqThreads>(A, n, &dmin, flag)) {  // R2
    if (tid == 0) *status = 1;
    for (int v = tid; v < LP * LP; v += kThinqThreads) T[v] = 0.0;
    return;
  }
  {  // A = R2 R1: the upper blocks
    constexpr int NT = NB * (NB + 1) / 2, S = (NT + NW - 1) / NW;
    f64x4_t c[S];
#pragma unroll
    for (int u = 0; u < S; ++u) {
      const int t = wave + NW * u;
      if (t < NT)
        c[u] = block_product<NB>(f64x4_t{0, 0, 0, 0}, A, B, sym_block_i(t, NB), sym_block_j(t, NB),
                                 16 * sym_block_i(t, NB), 16 * sym_block_j(t, NB) + 16, lane);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < S; ++u) {
      const int t = wave + NW * u;
      if (t < NT) block_store<NB>(A, c[u], sym_block_i(t, NB), sym_block_j(t, NB), lane);
    }
    __syncthreads();
  }
  double x[4 * NB];
  lds_inv_upper<NB, kThinqThreads>(A, B, invd, n, x);
  __syncthreads();
  if (tid < 4 * LP) {  // A = R^-1
#pragma unroll
    for (int m = 0; m < 4 * NB; ++m) A[(4 * m + (tid & 3)) * P + (tid >> 2)] = x[m];
  }
  lds_load<NB, kThinqThreads>(B, Xtop, n, false);
  __syncthreads();
  {  // B = Xtop R^-1 (R^-1 is upper: k up to the block's last column)
    constexpr int NT = NB * NB, S = (NT + NW - 1) / NW;
    f64x4_t c[S];
#pragma unroll
    for (int u = 0; u < S; ++u) {
      const int t = wave + NW * u;
      if (t < NT)
        c[u] = block_product<NB>(f64x4_t{0, 0, 0, 0}, B, A, t / NB, t % NB, 0, 16 * (t % NB) + 16, lane);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < S; ++u) {
      const int t = wave + NW * u;
      if (t < NT) block_store<NB>(B, c[u], t / NB, t % NB, lane);
    }
    __syncthreads();
  }
  lds_householder_signs<NB, kThinqThreads>(B, n, sgn);
  for (int v = tid; v < LP * LP; v += kThinqThreads) {
    const int c = v % LP;
    T[v] = c < n ? A[v / LP * P + c] * sgn[c] : 0.0;
  }
}

// flipOmg's decision (src/RSVD.hpp:80-89): column l flips when
// sum |Omg2 - Q| > 2 sum |Omg2 + Q|.  partial: nb blocks of the two norms
// (2 lp values each), summed here by one workgroup.
__global__ void __launch_bounds__(1024) k_flip_signs(const double* __restrict__ partial, int nb, int n, int lp,
                                                     double* __restrict__ sign) {
  __shared__ double red[1024];
  const int w = 2 * lp, G = 1024 / w;
  const int col = threadIdx.x % w, g = threadIdx.x / w;
  double s = 0.0;
  if (g < G) {
#pragma unroll 4
    for (int b = g; b < nb; b += G) s += partial[(uint64_t)b * w + col];
  }
  red[threadIdx.x] = s;
  __syncthreads();
  if (g == 0) {
    for (int r = 1; r < G; ++r) s += red[r * w + col];
    red[col] = s;
  }
  __syncthreads();
  const int l = threadIdx.x;
  if (l < lp) sign[l] = (l < n && red[l] > 2.0 * red[lp + l]) ? -1.0 : 1.0;
}

// out[r][l] += sum_z partial[z][r][l] (z in order), l < ncols.
__global__ void k_sum_chunks(const double* __restrict__ partial, uint64_t nz, uint64_t nrows, int ncols,
                             double* __restrict__ out, int lp) {
  GRID_STRIDE(t, nrows * (uint64_t)ncols) {
    const uint64_t r = t / ncols;
    const int l = (int)(t - r * ncols);
    double v = 0.0;
    for (uint64_t z = 0; z < nz; ++z) v += partial[z * nrows * ncols + t];
    out[r * lp + l] += v;
  }
}

}  // namespace

void launch_colmajor_to_rows(const double* src, uint64_t n, int L, int lp, uint64_t rows_pad, double* dst,
                             hipStream_t s) {
  hipLaunchKernelGGL(k_colmajor_to_rows, dim3(grid_for(rows_pad * lp)), dim3(256), 0, s, src, n, L, lp, rows_pad, dst);
  check_launch("colmajor_to_rows");
}

void launch_flip_cols_by_max(double* V, uint64_t m, double* U, uint64_t n, int lp, int k, double* partial,
                             double* sign, hipStream_t s) {
  require(k >= 1 && k <= lp && lp <= 128, kErrArgument, "flip_cols_by_max: bad column count");
  // about a block per CU, at least 64 rows each
  const uint64_t rpb = std::max<uint64_t>(64, (m + 255) / 256);
  const uint64_t nb = std::max<uint64_t>(1, (m + rpb - 1) / rpb);
  uint64_t* rows = reinterpret_cast<uint64_t*>(partial + 256 * 128);
  hipLaunchKernelGGL(k_col_absmax_partial, dim3((unsigned)nb), dim3(256), 0, s, V, m, lp, k, rpb, partial, rows);
  hipLaunchKernelGGL(k_col_absmax_sign, dim3(1), dim3(256), 0, s, partial, rows, nb, lp, k, sign);
  hipLaunchKernelGGL(k_scale_cols, dim3(grid_for(m * lp)), dim3(256), 0, s, V, m, lp, sign);
  hipLaunchKernelGGL(k_scale_cols, dim3(grid_for(n * lp)), dim3(256), 0, s, U, n, lp, sign);
  check_launch("flip_cols_by_max");
}

void launch_impute_rows(const double* src, uint64_t rows, int lp, int k, int kp, const double* scale, double* dst,
                        hipStream_t s) {
  if (!rows) return;
  hipLaunchKernelGGL(k_impute_rows, dim3(grid_for(rows * (uint64_t)kp)), dim3(256), 0, s, src, rows, lp, k, kp, scale,
                     dst);
  check_launch("impute_rows");
}

void launch_pristine_cols(const double* F, uint64_t m, uint64_t rows, double* cf, double* sc, hipStream_t s) {
  hipLaunchKernelGGL(k_pristine_cols, dim3(grid_for(rows)), dim3(256), 0, s, F, m, rows, cf, sc);
  check_launch("pristine_cols");
}

void launch_standardize(const double* F, uint64_t m, double sqrt_ploidy, double tol, double* sc, hipStream_t s) {
  hipLaunchKernelGGL(k_standardize, dim3(grid_for(m)), dim3(256), 0, s, F, m, sqrt_ploidy, tol, sc);
  check_launch("standardize");
}

void launch_gather_f64(const double* src, const uint32_t* idx, uint64_t n, double* dst, hipStream_t s) {
  hipLaunchKernelGGL(k_gather_f64, dim3(grid_for(n)), dim3(256), 0, s, src, idx, n, dst);
  check_launch("gather_f64");
}

void launch_rows_to_colmajor(const double* src, uint64_t n, int lp, int k, double* dst, uint64_t col_len,
                             hipStream_t s, const uint32_t* place) {
  if (!n || !k) return;
  require(lp >= 1 && lp <= 128 && k <= lp, kErrArgument, "rows_to_colmajor: bad column count");
  hipLaunchKernelGGL(k_rows_to_colmajor, dim3((unsigned)((n + 31) / 32)), dim3(256), 32 * (lp + 1) * sizeof(double), s,
                     src, n, lp, k, dst, col_len, place);
  check_launch("rows_to_colmajor");
}

template <Form F>
static void make_pieces_t(const double* X, uint64_t nreal, uint64_t rows_pad, int lp, const double* rowscale,
                          const double* colsign, void* Wt, uint64_t wpitch, uint64_t wpiece, double* rounded,
                          double* signed_out, const double* colscale, const double* bsc, const double* bcf,
                          double* bpart, uint32_t left, uint32_t right, hipStream_t s) {
  using w_t = typename Pieces<F>::w_t;
  constexpr int P = Pieces<F>::P;
  const auto lds_for = [](int l) {
    return ((size_t)epi_pitch(sizeof(w_t)) * l * P * sizeof(w_t) + 15) / 16 * 16 + (size_t)1024 * 8;
  };
  static bool attr = false;
  if (!attr) {
    PCAONE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_make_pieces<F>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_for(128)));
    attr = true;
  }
  const uint64_t nb = (rows_pad + kEpiRows - 1) / kEpiRows;
  hipLaunchKernelGGL(k_make_pieces<F>, dim3((unsigned)nb), dim3(256), lds_for(lp), s, X, nreal, rows_pad, lp, rowscale,
                     colsign, Wt, wpitch, wpiece, rounded, signed_out, colscale, bsc, bcf, bpart, left, right);
}

void launch_make_pieces(Form f, const double* X, uint64_t nreal, uint64_t rows_pad, int lp, const double* rowscale,
                        const double* colsign, void* Wt, uint64_t wpitch, uint64_t wpiece, double* rounded,
                        double* signed_out, hipStream_t s, const double* colscale, const double* bsc,
                        const double* bcf, double* bpart, uint64_t bpart_cap, double* bvec, uint32_t left,
                        uint32_t right) {
  require(!form_colscaled(f) || colscale, kErrInternal, "make_pieces: this form needs column scales");
  require(wpitch % 8 == 0 && wpiece % 8 == 0, kErrInternal, "make_pieces: bad pitch");
  require(lp >= 16 && lp <= 128 && lp % 4 == 0, kErrArgument, "make_pieces: bad lp");
  if (!rows_pad) return;
  const uint64_t nb = (rows_pad + kEpiRows - 1) / kEpiRows;
  // the column sums ride along when their per-tile partials fit the scratch
  const bool fuse = bvec && bpart && nb * (uint64_t)lp <= bpart_cap;
  double* bp = fuse ? bpart : nullptr;
  switch (f) {
    case Form::FP64: make_pieces_t<Form::FP64>(X, nreal, rows_pad, lp, rowscale, colsign, Wt, wpitch, wpiece, rounded, signed_out, colscale, bsc, bcf, bp, left, right, s); break;
    case Form::FP32: make_pieces_t<Form::FP32>(X, nreal, rows_pad, lp, rowscale, colsign, Wt, wpitch, wpiece, rounded, signed_out, colscale, bsc, bcf, bp, left, right, s); break;
    case Form::BF16: make_pieces_t<Form::BF16>(X, nreal, rows_pad, lp, rowscale, colsign, Wt, wpitch, wpiece, rounded, signed_out, colscale, bsc, bcf, bp, left, right, s); break;
    case Form::BF16X1: make_pieces_t<Form::BF16X1>(X, nreal, rows_pad, lp, rowscale, colsign, Wt, wpitch, wpiece, rounded, signed_out, colscale, bsc, bcf, bp, left, right, s); break;
    case Form::FP16: make_pieces_t<Form::FP16>(X, nreal, rows_pad, lp, rowscale, colsign, Wt, wpitch, wpiece, rounded, signed_out, colscale, bsc, bcf, bp, left, right, s); break;
    case Form::I8: make_pieces_t<Form::I8>(X, nreal, rows_pad, lp, rowscale, colsign, Wt, wpitch, wpiece, rounded, signed_out, colscale, bsc, bcf, bp, left, right, s); break;
    case Form::F8: make_pieces_t<Form::F8>(X, nreal, rows_pad, lp, rowscale, colsign, Wt, wpitch, wpiece, rounded, signed_out, colscale, bsc, bcf, bp, left, right, s); break;
  }
  check_launch("make_pieces");
  if (!bvec) return;
  if (fuse) {
    sum_partials(bpart, nb, (uint64_t)lp, bvec, s);
    check_launch("make_pieces_colsum");
  } else {
    require(rounded != nullptr && bpart != nullptr, kErrInternal, "make_pieces: column sums need rounded and scratch");
    launch_colsum(rounded, 0, nreal, lp, bsc, bcf, bpart, bvec, s);
  }
}

bool launch_epi_g(Form f, const void* P, uint64_t nchunks, uint64_t chunk_stride, uint64_t nreal, uint64_t rows_pad,
                  int lp, const double* sc, const double* cf, const double* colsum, double* out, hipStream_t s,
                  const double* colmul, unsigned long long* maxbits) {
  const unsigned g = grid_for(rows_pad * lp);
  require(!form_colscaled(f) || colmul, kErrInternal, "epi_g: this form needs column factors");
  if (maxbits && form_colscaled(f) && nreal == rows_pad && lp % 4 == 0 && lp <= 128 && chunk_stride % 4 == 0 &&
      reinterpret_cast<uintptr_t>(P) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0) {
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(128), 0, s, maxbits, lp);
    const unsigned gm = grid_for(nreal, 1024 / lp, kMaxBlocks);
    if (f == Form::I8)
      hipLaunchKernelGGL(k_epi_g_max<int32_t>, dim3(gm), dim3(256), 0, s, static_cast<const int32_t*>(P), nchunks,
                         chunk_stride, nreal, lp, sc, cf, colsum, out, colmul, maxbits);
    else
      hipLaunchKernelGGL(k_epi_g_max<float>, dim3(gm), dim3(256), 0, s, static_cast<const float*>(P), nchunks,
                         chunk_stride, nreal, lp, sc, cf, colsum, out, colmul, maxbits);
    check_launch("epi_g_max");
    return true;
  }
  if (f == Form::FP64)
    hipLaunchKernelGGL(k_epi_g<double>, dim3(g), dim3(256), 0, s, static_cast<const double*>(P), nchunks,
                       chunk_stride, nreal, rows_pad, lp, sc, cf, colsum, out, colmul);
  else if (lp % 4 == 0 && chunk_stride % 4 == 0 && reinterpret_cast<uintptr_t>(P) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(out) % 16 == 0) {
    const unsigned g4 = grid_for(rows_pad * lp / 4);
    if (f == Form::I8)
      hipLaunchKernelGGL(k_epi_g_v4<int32_t>, dim3(g4), dim3(256), 0, s, static_cast<const int32_t*>(P), nchunks,
                         chunk_stride, nreal, rows_pad, lp, sc, cf, colsum, out, colmul);
    else
      hipLaunchKernelGGL(k_epi_g_v4<float>, dim3(g4), dim3(256), 0, s, static_cast<const float*>(P), nchunks,
                         chunk_stride, nreal, rows_pad, lp, sc, cf, colsum, out, colmul);
  } else if (f == Form::I8)
    hipLaunchKernelGGL(k_epi_g<int32_t>, dim3(g), dim3(256), 0, s, static_cast<const int32_t*>(P), nchunks,
                       chunk_stride, nreal, rows_pad, lp, sc, cf, colsum, out, colmul);
  else
    hipLaunchKernelGGL(k_epi_g<float>, dim3(g), dim3(256), 0, s, static_cast<const float*>(P), nchunks, chunk_stride,
                       nreal, rows_pad, lp, sc, cf, colsum, out, colmul);
  check_launch("epi_g");
  return false;
}

void launch_col_scales(Form f, const double* X, uint64_t nreal, int lp, const double* rowscale,
                       unsigned long long* maxbits, double* scale, double* mul, hipStream_t s) {
  require(form_colscaled(f), kErrInternal, "col_scales: not a column-scaled form");
  if (X) {
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(128), 0, s, maxbits, lp);
    hipLaunchKernelGGL(k_colmax, dim3(grid_for(nreal, 8 * (1024 / lp), kMaxBlocks)), dim3(256), 0, s, X, nreal, lp, rowscale,
                       maxbits);
  }
  hipLaunchKernelGGL(k_col_scales, dim3(1), dim3(128), 0, s, maxbits, lp, f == Form::F8 ? 1 : 0, scale, mul);
  check_launch("col_scales");
}

uint64_t epi_g_fused_partial_elems(uint64_t nwin, int lp) { return (nwin + kEpiRows - 1) / kEpiRows * lp; }

template <Form F, class PT>
static void epi_fused_t(const void* P, uint64_t nchunks, uint64_t stride, uint64_t nwin, int lp, const double* sc,
                        const double* cf, const double* colsum, double* gout, void* Wt, uint64_t wpitch,
                        uint64_t wpiece, double* bpart, uint32_t left, uint32_t right, hipStream_t s) {
  constexpr int NP = Pieces<F>::P;
  constexpr size_t wsz = sizeof(typename Pieces<F>::w_t);
  // pieces (transposed) + the row groups' beta sums (256 / (lp / 4) groups x lp)
  const auto lds_for = [](int l) { return ((size_t)epi_pitch(wsz) * l * NP * wsz + 15) / 16 * 16 + (size_t)1024 * 8; };
  const size_t lds = lds_for(lp);
  static bool attr = false;
  if (!attr) {
    const size_t lds_max = lds_for(128);
    PCAONE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_epi_g_fused<F, PT>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_max));
    attr = true;
  }
  const uint64_t nb = (nwin + kEpiRows - 1) / kEpiRows;
  hipLaunchKernelGGL((k_epi_g_fused<F, PT>), dim3((unsigned)nb), dim3(256), lds, s, static_cast<const PT*>(P), nchunks,
                     stride, nwin, lp, sc, cf, colsum, gout, Wt, wpitch, wpiece, bpart, left, right);
}

void launch_epi_g_fused(Form f, const void* P, uint64_t nchunks, uint64_t stride, uint64_t nwin, int lp,
                        const double* sc, const double* cf, const double* colsum, double* gout, void* Wt,
                        uint64_t wpitch, uint64_t wpiece, double* bpart, double* bvec, uint32_t left, uint32_t right,
                        hipStream_t s) {
  if (!nwin) return;
  require(lp >= 16 && lp <= 128, kErrArgument, "epi_g_fused: bad lp");
  require(wpitch % 8 == 0 && wpiece % 8 == 0, kErrInternal, "epi_g_fused: bad pitch");
  switch (f) {
    case Form::FP64: epi_fused_t<Form::FP64, double>(P, nchunks, stride, nwin, lp, sc, cf, colsum, gout, Wt, wpitch, wpiece, bpart, left, right, s); break;
    case Form::FP32: epi_fused_t<Form::FP32, float>(P, nchunks, stride, nwin, lp, sc, cf, colsum, gout, Wt, wpitch, wpiece, bpart, left, right, s); break;
    case Form::BF16: epi_fused_t<Form::BF16, float>(P, nchunks, stride, nwin, lp, sc, cf, colsum, gout, Wt, wpitch, wpiece, bpart, left, right, s); break;
    case Form::BF16X1: epi_fused_t<Form::BF16X1, float>(P, nchunks, stride, nwin, lp, sc, cf, colsum, gout, Wt, wpitch, wpiece, bpart, left, right, s); break;
    case Form::FP16: epi_fused_t<Form::FP16, float>(P, nchunks, stride, nwin, lp, sc, cf, colsum, gout, Wt, wpitch, wpiece, bpart, left, right, s); break;
    case Form::I8:
    case Form::F8: fail(kErrInternal, "epi_g_fused: the column-scaled forms take the unfused epilogue");
  }
  check_launch("epi_g_fused");
  const uint64_t nb = (nwin + kEpiRows - 1) / kEpiRows;
  sum_partials(bpart, nb, (uint64_t)lp, bvec, s);
  check_launch("epi_g_fused_sum");
}

void launch_epi_h(Form f, const void* P, uint64_t nchunks, uint64_t chunk_stride, uint64_t nreal, uint64_t rows_pad,
                  int lp, const double* b, double* out, int mode, hipStream_t s, const double* colmul) {
  const unsigned g = grid_for(rows_pad * lp);
  require(!form_colscaled(f) || colmul, kErrInternal, "epi_h: this form needs column factors");
  if (f == Form::FP64)
    hipLaunchKernelGGL(k_epi_h<double>, dim3(g), dim3(256), 0, s, static_cast<const double*>(P), nchunks,
                       chunk_stride, nreal, rows_pad, lp, b, out, mode, colmul);
  else if (f == Form::I8)
    hipLaunchKernelGGL(k_epi_h<int32_t>, dim3(g), dim3(256), 0, s, static_cast<const int32_t*>(P), nchunks,
                       chunk_stride, nreal, rows_pad, lp, b, out, mode, colmul);
  else if (lp % 4 == 0 && chunk_stride % 4 == 0 && reinterpret_cast<uintptr_t>(P) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(out) % 16 == 0)
    hipLaunchKernelGGL(k_epi_h_f4, dim3(grid_for(rows_pad * lp / 4)), dim3(256), 0, s, static_cast<const float*>(P),
                       nchunks, chunk_stride, nreal, rows_pad, lp, b, out, mode, colmul);
  else
    hipLaunchKernelGGL(k_epi_h<float>, dim3(g), dim3(256), 0, s, static_cast<const float*>(P), nchunks, chunk_stride,
                       nreal, rows_pad, lp, b, out, mode, colmul);
  check_launch("epi_h");
}

static uint64_t colsum_rpb(uint64_t rows) {
  uint64_t rpb = (rows + 1023) / 1024;
  return rpb < 64 ? 64 : rpb;
}

void launch_colsum(const double* X, uint64_t r0, uint64_t r1, int lp, const double* w_sc, const double* w_cf,
                   double* partial, double* out, hipStream_t s) {
  if (r1 <= r0) {
    PCAONE_HIP(hipMemsetAsync(out, 0, lp * sizeof(double), s));
    return;
  }
  const uint64_t rpb = colsum_rpb(r1 - r0);
  const uint64_t nb = (r1 - r0 + rpb - 1) / rpb;
  hipLaunchKernelGGL(k_colsum_partial, dim3((unsigned)nb), dim3(128), 0, s, X, r0, r1, lp, rpb, w_sc, w_cf, partial);
  check_launch("colsum_partial");
  sum_partials(partial, nb, (uint64_t)lp, out, s);
  check_launch("colsum_sum");
}

// Rows per Gram partial: about 1,024 of them, a multiple of 32 and at least
// 128 rows each (the order of the sums is part of the result).
static uint64_t gram_rpb(uint64_t nrows) {
  uint64_t rpb = (nrows + 1023) / 1024;
  rpb = (rpb + 31) / 32 * 32;
  return rpb < 128 ? 128 : rpb;
}

uint64_t gram_partial_elems(uint64_t nrows, int lp) {
  const uint64_t rpb = gram_rpb(nrows ? nrows : 1);
  const uint64_t nb = (nrows + rpb - 1) / rpb;
  return (nb ? nb : 1) * (uint64_t)lp * lp;
}

template <int NB, int MODE>
static void gram_nb(const double* X, const double* Y, uint64_t nrows, uint64_t rpb, uint64_t nb, double* partial,
                    double* Z, hipStream_t s) {
  constexpr size_t lds = gram_lds(NB, MODE);
  static bool attr = false;
  if (!attr) {
    PCAONE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gram<NB, MODE>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr = true;
  }
  hipLaunchKernelGGL((k_gram<NB, MODE>), dim3((unsigned)nb), dim3(64 * gram_waves(NB)), lds, s, X, Y, nrows, rpb,
                     partial, Z);
}

template <int MODE>
static void gram_mode(const double* X, const double* Y, uint64_t nrows, int lp, double* partial, uint64_t partial_cap,
                      double* Z, double* out, hipStream_t s) {
  require(lp <= 128 && lp % 16 == 0 && lp >= 16, kErrArgument, "gram: bad lp");
  if (nrows == 0) {
    PCAONE_HIP(hipMemsetAsync(out, 0, (size_t)lp * lp * sizeof(double), s));
    return;
  }
  const uint64_t rpb = gram_rpb(nrows);
  const uint64_t nb = (nrows + rpb - 1) / rpb;
  require(nb * lp * lp <= partial_cap, kErrInternal, "gram: partial buffer too small");
  switch (lp / 16) {
    case 1: gram_nb<1, MODE>(X, Y, nrows, rpb, nb, partial, Z, s); break;
    case 2: gram_nb<2, MODE>(X, Y, nrows, rpb, nb, partial, Z, s); break;
    case 3: gram_nb<3, MODE>(X, Y, nrows, rpb, nb, partial, Z, s); break;
    case 4: gram_nb<4, MODE>(X, Y, nrows, rpb, nb, partial, Z, s); break;
    case 5: gram_nb<5, MODE>(X, Y, nrows, rpb, nb, partial, Z, s); break;
    default:
      if constexpr (MODE == kGramSelf || MODE == kGramCross) {
        if (lp == 96) gram_nb<6, MODE>(X, Y, nrows, rpb, nb, partial, Z, s);
        else if (lp == 112) gram_nb<7, MODE>(X, Y, nrows, rpb, nb, partial, Z, s);
        else gram_nb<8, MODE>(X, Y, nrows, rpb, nb, partial, Z, s);
      } else {  // T and the tile share LDS
        fail(kErrInternal, "gram: the fused forms take at most 80 columns");
      }
  }
  check_launch("gram");
  sum_partials(partial, nb, (uint64_t)lp * lp, out, s);
  check_launch("gram_sum");
}

void launch_gram(const double* X, const double* Y, uint64_t nrows, int lp, double* partial, uint64_t partial_cap,
                 double* out, hipStream_t s) {
  if (Y) gram_mode<kGramCross>(X, Y, nrows, lp, partial, partial_cap, nullptr, out, s);
  else gram_mode<kGramSelf>(X, nullptr, nrows, lp, partial, partial_cap, nullptr, out, s);
}

void launch_gram_add(const double* X, const double* Y, double* Z, uint64_t nrows, int lp, double* partial,
                     uint64_t partial_cap, double* out, hipStream_t s) {
  gram_mode<kGramAdd>(X, Y, nrows, lp, partial, partial_cap, Z, out, s);
}

void launch_gram_apply(const double* X, const double* T, uint64_t nrows, int lp, double* partial,
                       uint64_t partial_cap, double* out, hipStream_t s) {
  gram_mode<kGramApply>(X, T, nrows, lp, partial, partial_cap, nullptr, out, s);
}

// Blocks of the product with the flipOmg norms: their partials are summed by
// one workgroup, so no more of them than CUs.
constexpr uint64_t kFlipBlocks = 256;

template <int NB, bool FLIP>
static unsigned apply_nb(const double* X, const double* T, uint64_t nrows, double* Y, const double* O2,
                         double* partial, hipStream_t s) {
  constexpr size_t lds = (size_t)NB * 16 * NB * 16 * sizeof(double);
  static bool attr = false;
  if (!attr) {
    PCAONE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_apply_mfma<NB, FLIP>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr = true;
  }
  const uint64_t nblk = (nrows + 15) / 16;
  const unsigned g = (unsigned)std::min<uint64_t>((nblk + 3) / 4, FLIP ? kFlipBlocks : 4096);
  hipLaunchKernelGGL((k_apply_mfma<NB, FLIP>), dim3(g), dim3(256), lds, s, X, T, nrows, Y, O2, partial);
  return g;
}

template <bool FLIP>
static unsigned apply_lp(const double* X, const double* T, uint64_t nrows, int lp, double* Y, const double* O2,
                         double* partial, hipStream_t s) {
  require(lp <= 128 && lp % 16 == 0 && lp >= 16, kErrArgument, "apply: bad lp");
  unsigned g = 0;
  switch (lp / 16) {
    case 1: g = apply_nb<1, FLIP>(X, T, nrows, Y, O2, partial, s); break;
    case 2: g = apply_nb<2, FLIP>(X, T, nrows, Y, O2, partial, s); break;
    case 3: g = apply_nb<3, FLIP>(X, T, nrows, Y, O2, partial, s); break;
    case 4: g = apply_nb<4, FLIP>(X, T, nrows, Y, O2, partial, s); break;
    case 5: g = apply_nb<5, FLIP>(X, T, nrows, Y, O2, partial, s); break;
    case 6: g = apply_nb<6, FLIP>(X, T, nrows, Y, O2, partial, s); break;
    case 7: g = apply_nb<7, FLIP>(X, T, nrows, Y, O2, partial, s); break;
    case 8: g = apply_nb<8, FLIP>(X, T, nrows, Y, O2, partial, s); break;
  }
  check_launch("apply_mfma");
  return g;
}

void launch_apply(const double* X, const double* T, uint64_t nrows, int lp, double* Y, hipStream_t s) {
  if (nrows) apply_lp<false>(X, T, nrows, lp, Y, nullptr, nullptr, s);
}

void launch_apply_flip(const double* X, const double* T, uint64_t nrows, int n, int lp, double* Y, const double* O2,
                       double* partial, double* sign, hipStream_t s) {
  if (!nrows) return;
  const unsigned g = apply_lp<true>(X, T, nrows, lp, Y, O2, partial, s);
  launch_flip_signs(partial, (int)g, n, lp, sign, s);
}

void launch_flip_norms(const double* O2, const double* Q, uint64_t nrows, int lp, double* partial, double* out,
                       hipStream_t s) {
  const uint64_t rpb = colsum_rpb(nrows);
  const uint64_t nb = (nrows + rpb - 1) / rpb;
  hipLaunchKernelGGL(k_flip_partial, dim3((unsigned)nb), dim3(128), 0, s, O2, Q, nrows, lp, rpb, partial);
  check_launch("flip_partial");
  sum_partials(partial, nb, (uint64_t)2 * lp, out, s);
  check_launch("flip_sum");
}

void launch_add(const double* X, const double* Z, double* Y, uint64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_add, dim3(grid_for(n)), dim3(256), 0, s, X, Z, Y, n);
  check_launch("add");
}

void launch_missing_weights(const MissWeightArgs& a, hipStream_t s) {
  if (!a.nrows) return;
  require(a.kspan > 0, kErrArgument, "missing_weights: zero index span");
  const uint64_t nz = (a.kext + a.kspan - 1) / a.kspan;
  require(nz < 65536, kErrArgument, "missing_weights: too many index chunks");
  const dim3 grid((unsigned)((a.nrows + 3) / 4), (unsigned)std::max<uint64_t>(nz, 1));
  if (!a.Fclamp) {
    hipLaunchKernelGGL(k_missing_weights, grid, dim3(256), 0, s, a);
  } else {
    require(a.kk >= 1 && a.kk <= 128 && a.kp % 16 == 0 && a.kp >= a.kk + 3, kErrArgument,
            "missing_weights: imputation rank must be in [1, 128]");
    int lpe = 1;
    while (lpe < (a.kk + 1) / 2) lpe *= 2;
    hipLaunchKernelGGL(k_missing_weights_emu, grid, dim3(256), 0, s, a, lpe);
  }
  check_launch("missing_weights");
}

void launch_pack_col_state(double* V, uint64_t m, int kp, int kk, const double* sc, const double* cf, const double* F,
                           hipStream_t s) {
  if (!m) return;
  hipLaunchKernelGGL(k_pack_col_state, dim3(grid_for(m)), dim3(256), 0, s, V, m, kp, kk, sc, cf, F);
  check_launch("pack_col_state");
}

void launch_compact_rows(const double* src, uint64_t rows, int lp, int L, int pitch, bool f32, void* out,
                         hipStream_t s) {
  if (!rows) return;
  const unsigned g = grid_for(rows * (uint64_t)pitch);
  if (f32)
    hipLaunchKernelGGL(k_compact_rows<float>, dim3(g), dim3(256), 0, s, src, rows, lp, L, pitch,
                       static_cast<float*>(out));
  else
    hipLaunchKernelGGL(k_compact_rows<double>, dim3(g), dim3(256), 0, s, src, rows, lp, L, pitch,
                       static_cast<double*>(out));
  check_launch("compact_rows");
}

void launch_missing_spmm(const MissSpmmArgs& a, hipStream_t s) {
  if (!a.nrows || a.k_hi <= a.k_lo) return;
  const int vec = a.f32 ? 4 : 2;
  require(a.ncols >= 1 && a.ncols <= a.lp && a.cp >= a.ncols && a.cp % vec == 0 && a.cp <= 128 &&
              a.cpitch >= a.cp && a.cpitch % vec == 0,
          kErrArgument, "missing_spmm: bad column counts");
  const uint64_t span = a.k_hi - a.k_lo;
  const uint64_t nz = a.kspan ? (span + a.kspan - 1) / a.kspan : 1;
  require(nz < 65536 && (nz == 1 || (a.partial && nz * a.nrows * (uint64_t)a.ncols <= a.partial_cap)), kErrInternal,
          "missing_spmm: bad index chunking");
  const dim3 block(256);
  const unsigned gx = (unsigned)((a.nrows + 3) / 4), gz = (unsigned)nz;
  if (a.f32) hipLaunchKernelGGL((k_missing_spmm<float>), dim3(gx, 1, gz), block, 0, s, a);
  else hipLaunchKernelGGL((k_missing_spmm<double>), dim3(gx, 1, gz), block, 0, s, a);
  check_launch("missing_spmm");
  if (nz > 1) launch_sum_chunks(a.partial, nz, a.nrows, a.ncols, a.out, a.lp, s);
}

void launch_sum_chunks(const double* partial, uint64_t nz, uint64_t nrows, int ncols, double* out, int lp,
                       hipStream_t s) {
  if (!nrows || !ncols) return;
  hipLaunchKernelGGL(k_sum_chunks, dim3(grid_for(nrows * (uint64_t)ncols)), dim3(256), 0, s, partial, nz, nrows,
                     ncols, out, lp);
  check_launch("sum_chunks");
}

bool thinq_on_device(int lp) { return lp % 16 == 0 && lp <= 16 * kThinqMaxNB; }

template <int NB>
void thinq_first_nb(const double* G1, int n, double* R1, double* T1, int* status, double min_ratio, hipStream_t s) {
  static bool attr = false;
  if (!attr) {
    PCAONE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_thinq_first<NB>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)thinq_lds<NB>()));
    attr = true;
  }
  hipLaunchKernelGGL(k_thinq_first<NB>, dim3(1), dim3(kThinqThreads), thinq_lds<NB>(), s, G1, n, R1, T1, status,
                     min_ratio);
}

void launch_thinq_first(const double* G1, int n, int lp, double* R1, double* T1, int* status, hipStream_t s,
                        double min_ratio) {
  require(thinq_on_device(lp) && n <= lp, kErrInternal, "thinq: lp too large for the device path");
  switch (lp / 16) {
    case 1: thinq_first_nb<1>(G1, n, R1, T1, status, min_ratio, s); break;
    case 2: thinq_first_nb<2>(G1, n, R1, T1, status, min_ratio, s); break;
    case 3: thinq_first_nb<3>(G1, n, R1, T1, status, min_ratio, s); break;
    case 4: thinq_first_nb<4>(G1, n, R1, T1, status, min_ratio, s); break;
    default: thinq_first_nb<5>(G1, n, R1, T1, status, min_ratio, s); break;
  }
  check_launch("thinq_first");
}

template <int NB>
void thinq_second_nb(const double* G2, const double* R1, const double* Xtop, int n, double* T, int* status,
                     hipStream_t s) {
  static bool attr = false;
  if (!attr) {
    PCAONE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_thinq_second<NB>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)thinq_lds<NB>()));
    attr = true;
  }
  hipLaunchKernelGGL(k_thinq_second<NB>, dim3(1), dim3(kThinqThreads), thinq_lds<NB>(), s, G2, R1, Xtop, n, T, status);
}

void launch_thinq_second(const double* G2, const double* R1, const double* Xtop, int n, int lp, double* T,
                         int* status, hipStream_t s) {
  require(thinq_on_device(lp) && n <= lp, kErrInternal, "thinq: lp too large for the device path");
  switch (lp / 16) {
    case 1: thinq_second_nb<1>(G2, R1, Xtop, n, T, status, s); break;
    case 2: thinq_second_nb<2>(G2, R1, Xtop, n, T, status, s); break;
    case 3: thinq_second_nb<3>(G2, R1, Xtop, n, T, status, s); break;
    case 4: thinq_second_nb<4>(G2, R1, Xtop, n, T, status, s); break;
    default: thinq_second_nb<5>(G2, R1, Xtop, n, T, status, s); break;
  }
  check_launch("thinq_second");
}

void launch_flip_signs(const double* partial, int nb, int n, int lp, double* sign, hipStream_t s) {
  hipLaunchKernelGGL(k_flip_signs, dim3(1), dim3(1024), 0, s, partial, nb, n, lp, sign);
  check_launch("flip_signs");
}

}  // namespace pcaone
