// FP64 form of the packed-genotype GEMM for column counts that leave a short
// last block of 16 (see gemm.hpp for the contract; kernels_gemm_r4.hip is its
// FP32 counterpart).
//
// The full blocks of 16 columns go through v_mfma_f64_16x16x4, the columns past
// them in groups of 4 through v_mfma_f64_4x4x4_4b: four 4 x 4 blocks, i.e. 16
// rows by the same 4 columns by the same 4 k slots, at the same rate per
// multiply-add.  Its A operand has the lanes of the 16 x 16 x 4 one (row lane % 16,
// k slot lane / 16), so the decoded genotypes serve both, and both add their
// four products to the accumulator one by one in ascending k as fused
// multiply-adds: every output is the same bits as with a padded block.
//
// FP64 MFMAs and the vector ALU take turns on a SIMD, so the decode of a u-step
// stands together ahead of its MFMAs; the B fragments of the next step are read
// from LDS while they run.  3,001 x 50,021, L = 20: 184 us per product with a
// padded block, 117 us here (the MFMAs alone: 80 us).
#include <hip/hip_runtime.h>

#include "device.hpp"
#include "gemm.hpp"
#include "gemm_decode.hpp"

namespace pcaone {
namespace {

typedef double f64x4_t __attribute__((ext_vector_type(4)));
typedef double f64x2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

constexpr int WAVES = 4;  // a wave owns 16 rows

template <int NCF, int NR>
__global__ void __launch_bounds__(64 * WAVES) k_packed_gemm_f64_r4(GemmArgs a) {
  constexpr int KS = 128, LP = 16 * (NCF + 1), LW = 16 * NCF + 4 * NR;
  constexpr int NVT = (LW + WAVES - 1) / WAVES;  // W rows (64 vectors of 16 bytes) per wave and tile
  extern __shared__ __align__(16) double wl[];   // two tiles of LW rows of KS
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int q = lane >> 4, r16 = lane & 15, c4 = lane & 3;
  const uint64_t rowbase = (uint64_t)blockIdx.x * (WAVES * 16) + (uint64_t)wave * 16;
  const uint64_t kb = a.k_begin + (uint64_t)blockIdx.y * a.kchunk;
  const uint64_t ke = kb + a.kchunk < a.k_end ? kb + a.kchunk : a.k_end;
  const double* wg = static_cast<const double*>(a.Wt);
  double* Y = static_cast<double*>(a.Y) + (uint64_t)blockIdx.y * a.ychunk;
  const uint32_t* xr = a.X + (rowbase + r16) * a.xpitch + 2 * q;

  // vector v of W row `row` sits at slot v ^ (row & 15); the DMA writes a row's
  // 64 slots and fetches the vector that belongs in each
  auto tile_dma = [&](double* dst, uint64_t kk) {
#pragma unroll
    for (int i = 0; i < NVT; ++i) {
      const int row = wave + WAVES * i;
      if (row < LW) {
        const double* src = wg + row * a.wpitch + (lane ^ (row & 15)) * 2 + kk;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)(dst + row * KS), 16, 0, 0);
      }
    }
  };

  f64x4_t acc[NCF];
  double acc4[NR];
#pragma unroll
  for (int cb = 0; cb < NCF; ++cb) acc[cb] = f64x4_t{0, 0, 0, 0};
#pragma unroll
  for (int g = 0; g < NR; ++g) acc4[g] = 0.0;

  struct BFrag {
    f64x2_t full[NCF][2], part[NR][2];
  };
  auto read_b = [&](const double* t, int u, BFrag& b) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int cb = 0; cb < NCF; ++cb)
        b.full[cb][h] = *reinterpret_cast<const f64x2_t*>(t + (cb * 16 + r16) * KS + ((16 * q + 2 * u + h) ^ r16) * 2);
#pragma unroll
      for (int g = 0; g < NR; ++g)
        b.part[g][h] = *reinterpret_cast<const f64x2_t*>(t + (16 * NCF + 4 * g + c4) * KS +
                                                         ((16 * q + 2 * u + h) ^ (4 * g + c4)) * 2);
    }
  };

  if (kb < ke) {
    u32x2_t acur = *reinterpret_cast<const u32x2_t*>(xr + (kb >> 4)), anext;
    tile_dma(wl, kb);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int buf = 0;
    for (uint64_t k0 = kb; k0 < ke; k0 += KS) {
      const bool more = k0 + KS < ke;
      if (more) {
        tile_dma(wl + (buf ^ 1) * LW * KS, k0 + KS);
        anext = *reinterpret_cast<const u32x2_t*>(xr + ((k0 + KS) >> 4));
      }
      const double* t = wl + buf * LW * KS;
      BFrag b[2];
      read_b(t, 0, b[0]);
#pragma unroll
      for (int u = 0; u < KS / 16; ++u) {
        if (u + 1 < KS / 16) read_b(t, u + 1, b[(u + 1) & 1]);
        const BFrag& bc = b[u & 1];
        const uint32_t tb = top_bytes(spread(acur[u >> 2], u & 3));
        double av[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) av[e] = __hiloint2double((int)top_word(tb, e), 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int cb = 0; cb < NCF; ++cb)
            acc[cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[e], bc.full[cb][e >> 1][e & 1], acc[cb], 0, 0, 0);
#pragma unroll
          for (int g = 0; g < NR; ++g)
            acc4[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(av[e], bc.part[g][e >> 1][e & 1], acc4[g], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (more) acur = anext;
      __builtin_amdgcn_s_waitcnt(0);  // this wave's tile loads have landed
      __syncthreads();
      buf ^= 1;
    }
  }

#pragma unroll
  for (int cb = 0; cb < NCF; ++cb)
#pragma unroll
    for (int r = 0; r < 4; ++r) Y[(rowbase + q + 4 * r) * LP + cb * 16 + r16] = acc[cb][r];
#pragma unroll
  for (int g = 0; g < NR; ++g) Y[(rowbase + 4 * ((lane >> 2) & 3) + q) * LP + 16 * NCF + 4 * g + c4] = acc4[g];
#pragma unroll
  for (int c = LW; c < LP; c += 4)  // the padding columns read as zero
    Y[(rowbase + r16) * LP + c + q] = 0.0;
}

template <int NCF, int NR>
void launch_t(const GemmArgs& a, hipStream_t s) {
  constexpr size_t lds = (size_t)2 * (16 * NCF + 4 * NR) * 128 * sizeof(double);
  static bool attr = false;
  if (!attr) {
    PCAONE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_packed_gemm_f64_r4<NCF, NR>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr = true;
  }
  const uint64_t nchunks = (a.k_end - a.k_begin + a.kchunk - 1) / a.kchunk;
  hipLaunchKernelGGL((k_packed_gemm_f64_r4<NCF, NR>), dim3((unsigned)(a.rows / (WAVES * 16)), (unsigned)nchunks),
                     dim3(64 * WAVES), lds, s, a);
  check_launch("packed_gemm_f64_r4");
}

template <int NCF>
void launch_nr(int nr, const GemmArgs& a, hipStream_t s) {
  if (nr == 1) return launch_t<NCF, 1>(a, s);
  if (nr == 2) return launch_t<NCF, 2>(a, s);
  launch_t<NCF, 3>(a, s);
}

}  // namespace

bool launch_packed_gemm_f64_r4(const GemmArgs& a, hipStream_t s) {
  const int ncf = a.lp / 16 - 1, nr = (a.ncols - 16 * ncf + 3) / 4;
  if (ncf < 1 || ncf > 3 || nr < 1 || nr > 3) return false;
  ncf == 1 ? launch_nr<1>(nr, a, s) : (ncf == 2 ? launch_nr<2>(nr, a, s) : launch_nr<3>(nr, a, s));
  return true;
}

}  // namespace pcaone
