// f32 product with direct-to-LDS loads: C[M, N] (+)= A.B with the contract of gemm.hip (f32 operands and f32
// accumulation on v_mfma_f32_16x16x4_f32; reference: ojas-cpu/src/linalg.rs:69-210).
//
// Bound by the f32 matrix rate (64 operations a clock and SIMD): a 64 x 64 tile's 32-column step is 1024 clocks of matrix
// instructions over 16 KiB of operands. The register-staged kernel it replaces (128 x 128 tiles, one barrier between a
// step's loads and its products) ran at 60 % of that rate and, with a few hundred rows, had no tiles for half the chip or
// paid a second launch to add up a split reduction. Here the operands go straight into LDS, two to four stages deep, and
// several small workgroups share a compute unit, so that one's barriers and stores are under the others' products: 64 x 64
// tiles with two stages of 16 KiB come out ahead of 128 x 128 and 128 x 64 ones wherever there is a round of them (4096 x
// 3072 over 768: 155 us; 158 on 128 x 128, 218 before; 2048 x 8192 over 256: 88 -> 78). Smaller outputs take 64 x 32 tiles, or share K
// between two or four groups of waves of a workgroup, which meet in LDS (2048 x 256 over 1024: 19 -> 13 us).
//
// Sums. A chain of n roundings is off by sqrt(n / 2) units of the last place over random data. Every step of 32 sums into a
// register of its own that is added to the total when the step ends (16 vector additions per 32 matrix instructions, 3 to
// 8 % of the time): chains of 32 and of K / 32 instead of one of K. 2-norm error at K = 256, 512, 2048: 1.17e-7, 1.28e-7,
// 1.77e-7; one chain 2.9e-7, 4.1e-7, 8.1e-7; eight waves' chains (gemm_frag32.hip) 1.17e-7, 1.55e-7, 2.9e-7.
#include "gemm_dma32_impl.h"

namespace {

template <bool A_KM, bool B_KM, int WGM, int WGN, int TM, int TN, int NST, int KG, bool TAIL, int ACT>
__global__ __launch_bounds__(WGM* WGN* KG * 64, dma_waves_per_simd(WGM* WGN* KG, NST* KG*(WGM* TM + WGN * TN) * 16 * 128)) void
gemm_dma32_kernel(GemmArgs g) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  dma32_tile<A_KM, B_KM, WGM, WGN, TM, TN, NST, KG, TAIL, ACT>(g, blockIdx.x, smem);
}

template <bool A_KM, bool B_KM, int WGM, int WGN, int TM, int TN, int NST, int KG>
int32_t launch_dma32(omx_ctx* ctx, const GemmArgs& g) {
  constexpr int smem = NST * KG * (WGM * TM + WGN * TN) * 16 * 128;
  auto kernel = &gemm_dma32_kernel<A_KM, B_KM, WGM, WGN, TM, TN, NST, KG, false, 0>;
  if constexpr (A_KM && B_KM) {
    if (g.k_rows != g.K) kernel = &gemm_dma32_kernel<A_KM, B_KM, WGM, WGN, TM, TN, NST, KG, true, 0>;
  }
  if constexpr (!A_KM) {
    if (g.epi != OMX_EPI_NONE) kernel = g.epi_tanh ? &gemm_dma32_kernel<A_KM, B_KM, WGM, WGN, TM, TN, NST, KG, false, 2>
                                                   : &gemm_dma32_kernel<A_KM, B_KM, WGM, WGN, TM, TN, NST, KG, false, 1>;
  }
  if constexpr (smem > 64 * 1024)
    OMX_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
  omx_launch_timed(ctx, kernel, dim3(static_cast<unsigned>(g.tiles_m) * g.tiles_n * g.batches), dim3(WGM * WGN * KG * 64), smem,
                   ctx->timing_start, ctx->timing_stop, g);
  OMX_LAUNCH_CHECK(ctx, "gemm_dma32_kernel");
  return OMX_OK;
}
template <bool A_KM, bool B_KM>
int32_t launch_tile32(omx_ctx* ctx, const GemmArgs& g, int tile) {
  switch (tile) {
    case 0: return launch_dma32<A_KM, B_KM, 2, 2, 2, 2, 2, 1>(ctx, g);
    case 1: return launch_dma32<A_KM, B_KM, 2, 2, 2, 1, 4, 1>(ctx, g);
    case 2: return launch_dma32<A_KM, B_KM, 2, 2, 2, 1, 3, 2>(ctx, g);
    default: return launch_dma32<A_KM, B_KM, 2, 2, 1, 1, 3, 4>(ctx, g);
  }
}

}  // namespace

void omx_gemm_dma32_tile(int tile, int* bm, int* bn) {
  *bm = tile == 3 ? 32 : 64;
  *bn = tile == 0 ? 64 : 32;
}

// A k-contiguous operand's rows hold whole steps, a k-major one's whole pieces; both k-major, the reduction may end anywhere.
// From K = 256 on, where the sums of a step lose nothing against the other kernels' shorter chains (see above).
bool omx_gemm_dma32_eligible(const GemmArgs& g, bool a_km, bool b_km) {
  if (!g.a_vec || !g.b_vec || g.lda > 1l << 22 || g.ldb > 1l << 22 || g.K > 0x7fffffff - 32) return false;
  if (g.K < 256 || (g.K % 32 != 0 && !(a_km && b_km))) return false;
  return (!a_km || g.M % 4 == 0) && (!b_km || g.N % 4 == 0);
}

int32_t omx_gemm_dma32_launch(omx_ctx* ctx, const GemmArgs& g, bool a_km, bool b_km, int tile) {
  if (!a_km && !b_km) return launch_tile32<false, false>(ctx, g, tile);
  if (!a_km) return launch_tile32<false, true>(ctx, g, tile);
  if (!b_km) return launch_tile32<true, false>(ctx, g, tile);
  return launch_tile32<true, true>(ctx, g, tile);
}

// us, as for the tiles of gemm_frag32.hip: fitted together over 513 products of 32 .. 8192 rows and 256 .. 8192 columns over K
// = 256 .. 8192 in three layouts (rms 6 %); the tile they choose is 1.8 % behind the best one on average.
double omx_gemm_dma32_us(omx_ctx* ctx, const GemmArgs& g, int tile) {
  struct Cost {
    double first, step, more, more_step;
  };
  constexpr Cost COST[DMA32_TILES] = {{2.89, 0.651, 1.16, 0.442}, {2.93, 0.400, 0.93, 0.239}, {3.36, 0.300, 1.26, 0.242}, {3.72, 0.155, 2.46, 0.150}};
  int bm, bn;
  omx_gemm_dma32_tile(tile, &bm, &bn);
  const long units = ctx->cu_count > 0 ? ctx->cu_count : 256;
  const long groups = static_cast<long>((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn) * g.batches;
  if (groups > 0x7fffffffl) return -1.0;
  const double more = static_cast<double>((groups + units - 1) / units - 1), steps = (g.K + 31) / 32;
  return COST[tile].first + steps * COST[tile].step + more * (COST[tile].more + steps * COST[tile].more_step);
}
