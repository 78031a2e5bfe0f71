// FP32 form of the packed-genotype GEMM for column counts that leave a short
// last block of 16 (see gemm.hpp for the contract).
//
// The 16 x 16 x 4 MFMAs of k_packed_gemm multiply whole blocks of 16 columns:
// at L = 20 (k = 10 with the default oversampling) 12 of 32 are padding.  The
// FP32 product is bound by the matrix cores, so here only the full blocks go
// that way; the other columns go in groups of 4 through v_mfma_f32_4x4x1_16b,
// sixteen 4 x 4 blocks of 64 rows by the same 4 columns, at the same rate per
// multiply-add.  Both instructions add their products to the accumulator one by
// one as fused multiply-adds, in ascending k, so with the k slots fed in the
// order of the 16 x 16 x 4 form (code 64 q + 4 u + e: u, then e, then q) every
// output is the same bits.
//
// The FP32 MFMAs and the vector ALU take turns on a SIMD (35 cycles per 16 x 16 x 4
// MFMA, 4.3 per decode operation and 9 per change between the two, whichever
// wave issues them), so a u-step's decode stands together ahead of its MFMAs.
// Two workgroups of 4 waves share a CU, one computing where the other waits
// for its tile.  12,001 x 150,001, L = 20: 1,017 us per product with padded blocks,
// 708 us here (773 us with one workgroup of 8 waves, 937 us with the decode
// between the MFMAs); the MFMAs alone take 505 us.
//
// A wave owns 64 rows.  For the 16-column blocks lane (q, r) holds the codes of
// rows 16 rb + r, K quarter q; for the 4-column groups lane l holds row l, all
// four quarters: the decoded bytes of a u-step are transposed between the lane
// groups by four permlane swaps.  One group's column is read from LDS by 16
// lanes at once.  W tiles are double-buffered by direct global -> LDS loads,
// and the next u-step's B fragments are read while this one's MFMAs run.
#include <hip/hip_runtime.h>

#include "device.hpp"
#include "gemm.hpp"
#include "gemm_decode.hpp"

namespace pcaone {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

// m[i] of lane group j (16 lanes) <-> m[j] of lane group i.
__device__ __forceinline__ void transpose_groups(uint32_t (&m)[4]) {
  const auto a = __builtin_amdgcn_permlane32_swap(m[0], m[2], false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(m[1], m[3], false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  m[0] = c[0], m[1] = c[1], m[2] = d[0], m[3] = d[1];
}

constexpr int WAVES = 4;

template <int NCF, int NR>
__global__ void __launch_bounds__(64 * WAVES) k_packed_gemm_f32_r4(GemmArgs a) {
  constexpr int KS = 256, LP = 16 * (NCF + 1), LW = 16 * NCF + 4 * NR;
  constexpr int NVT = (LW + WAVES - 1) / WAVES;  // W rows (64 vectors of 16 bytes) per wave and tile
  extern __shared__ __align__(16) float wl[];    // two tiles of LW rows of KS
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int q = lane >> 4, r16 = lane & 15, c4 = lane & 3;
  const uint64_t rowbase = (uint64_t)blockIdx.x * (WAVES * 64) + (uint64_t)wave * 64;
  const uint64_t kb = a.k_begin + (uint64_t)blockIdx.y * a.kchunk;
  const uint64_t ke = kb + a.kchunk < a.k_end ? kb + a.kchunk : a.k_end;
  const float* wg = static_cast<const float*>(a.Wt);
  float* Y = static_cast<float*>(a.Y) + (uint64_t)blockIdx.y * a.ychunk;

  const uint32_t* xr[4];
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) xr[rb] = a.X + (rowbase + rb * 16 + r16) * a.xpitch + 4 * q;

  // vector v of W row `row` sits at slot v ^ (row & 15); the DMA writes a row's
  // 64 slots and fetches the vector that belongs in each
  auto tile_dma = [&](float* dst, uint64_t kk) {
#pragma unroll
    for (int i = 0; i < NVT; ++i) {
      const int row = wave + WAVES * i;
      if (row < LW) {
        const float* src = wg + row * a.wpitch + (lane ^ (row & 15)) * 4 + kk;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)(dst + row * KS), 16, 0, 0);
      }
    }
  };

  f32x4_t acc[4][NCF], acc4[NR];
#pragma unroll
  for (int rb = 0; rb < 4; ++rb)
#pragma unroll
    for (int cb = 0; cb < NCF; ++cb) acc[rb][cb] = f32x4_t{0, 0, 0, 0};
#pragma unroll
  for (int g = 0; g < NR; ++g) acc4[g] = f32x4_t{0, 0, 0, 0};

  struct BFrag {
    f32x4_t full[NCF], part[NR][4];
  };
  auto read_b = [&](const float* t, int u, BFrag& b) {
#pragma unroll
    for (int cb = 0; cb < NCF; ++cb)
      b.full[cb] = *reinterpret_cast<const f32x4_t*>(t + (cb * 16 + r16) * KS + ((16 * q + u) ^ r16) * 4);
#pragma unroll
    for (int g = 0; g < NR; ++g)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        b.part[g][k] = *reinterpret_cast<const f32x4_t*>(t + (16 * NCF + 4 * g + c4) * KS +
                                                         ((16 * k + u) ^ (4 * g + c4)) * 4);
  };

  if (kb < ke) {
    u32x4_t acur[4], anext[4];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) acur[rb] = *reinterpret_cast<const u32x4_t*>(xr[rb] + (kb >> 4));
    tile_dma(wl, kb);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int buf = 0;
    for (uint64_t k0 = kb; k0 < ke; k0 += KS) {
      const bool more = k0 + KS < ke;
      if (more) {
        tile_dma(wl + (buf ^ 1) * LW * KS, k0 + KS);
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) anext[rb] = *reinterpret_cast<const u32x4_t*>(xr[rb] + ((k0 + KS) >> 4));
      }
      const float* t = wl + buf * LW * KS;
      BFrag b[2];
      read_b(t, 0, b[0]);
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        if (u + 1 < 16) read_b(t, u + 1, b[(u + 1) & 1]);
        const BFrag& bc = b[u & 1];
        float av[4][4], a4[4][4];  // [e][row block], [e][K quarter]
        {
          uint32_t tb[4], tt[4];
#pragma unroll
          for (int rb = 0; rb < 4; ++rb) tt[rb] = tb[rb] = top_bytes(spread(acur[rb][u >> 2], u & 3));
          transpose_groups(tt);
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              av[e][i] = __uint_as_float(top_word(tb[i], e));
              a4[e][i] = __uint_as_float(top_word(tt[i], e));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int cb = 0; cb < NCF; ++cb)
              acc[i][cb] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[e][i], bc.full[cb][e], acc[i][cb], 0, 0, 0);
#pragma unroll
            for (int g = 0; g < NR; ++g)
              acc4[g] = __builtin_amdgcn_mfma_f32_4x4x1f32(a4[e][i], bc.part[g][i][e], acc4[g], 0, 0, 0);
            // a group's MFMAs depend on each other: each waits behind the full blocks' one before it
            __builtin_amdgcn_sched_barrier(0);
          }
      }
      if (more) {
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) acur[rb] = anext[rb];
      }
      __builtin_amdgcn_s_waitcnt(0);  // this wave's tile loads have landed
      __syncthreads();
      buf ^= 1;
    }
  }

#pragma unroll
  for (int rb = 0; rb < 4; ++rb)
#pragma unroll
    for (int cb = 0; cb < NCF; ++cb)
#pragma unroll
      for (int r = 0; r < 4; ++r) Y[(rowbase + rb * 16 + 4 * q + r) * LP + cb * 16 + r16] = acc[rb][cb][r];
#pragma unroll
  for (int g = 0; g < NR; ++g)
#pragma unroll
    for (int r = 0; r < 4; ++r) Y[(rowbase + 4 * (lane >> 2) + r) * LP + 16 * NCF + 4 * g + c4] = acc4[g][r];
#pragma unroll
  for (int c = LW; c < LP; c += 4)  // the padding columns read as zero
    *reinterpret_cast<f32x4_t*>(Y + (rowbase + lane) * LP + c) = f32x4_t{0, 0, 0, 0};
}

template <int NCF, int NR>
void launch_t(const GemmArgs& a, hipStream_t s) {
  constexpr size_t lds = (size_t)2 * (16 * NCF + 4 * NR) * 256 * sizeof(float);
  static bool attr = false;
  if (!attr) {
    PCAONE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_packed_gemm_f32_r4<NCF, NR>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr = true;
  }
  const uint64_t nchunks = (a.k_end - a.k_begin + a.kchunk - 1) / a.kchunk;
  hipLaunchKernelGGL((k_packed_gemm_f32_r4<NCF, NR>), dim3((unsigned)(a.rows / (WAVES * 64)), (unsigned)nchunks),
                     dim3(64 * WAVES), lds, s, a);
  check_launch("packed_gemm_f32_r4");
}

template <int NCF>
void launch_nr(int nr, const GemmArgs& a, hipStream_t s) {
  if (nr == 1) return launch_t<NCF, 1>(a, s);
  if (nr == 2) return launch_t<NCF, 2>(a, s);
  if constexpr (NCF == 1) launch_t<NCF, 3>(a, s);
}

}  // namespace

bool launch_packed_gemm_f32_r4(const GemmShape& g, const GemmArgs& a, hipStream_t s) {
  const int ncf = a.lp / 16 - 1, nr = (a.ncols - 16 * ncf + 3) / 4;
  if (g.wm != 4 || ncf < 1 || ncf > 2 || nr < 1 || nr > 4 - ncf) return false;
  // tiles of 8 waves split into two workgroups of 4
  ncf == 1 ? launch_nr<1>(nr, a, s) : launch_nr<2>(nr, a, s);
  return true;
}

}  // namespace pcaone
