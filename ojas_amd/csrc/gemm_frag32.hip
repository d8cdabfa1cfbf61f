// f32 product of a small output: C[M, N] (+)= A.B with the contract of gemm.hip (f32 operands and f32
// accumulation on v_mfma_f32_16x16x4_f32; reference: ojas-cpu/src/linalg.rs:69-210).
//
// A model a few hundred wide makes outputs of 64 Ki to a few Mi values: on 128 x 128 tiles that is 4 to 100
// workgroups for 256 compute units, so K was split into partials and added up by a second launch, and a
// tile's 64 matrix instructions per 32-column step ran as a chain of load, barrier, product (13 us and
// 4 us for the second launch, whatever the size). Here a workgroup owns 16 MB x 16 NB outputs and its waves
// share K, both operands go from memory straight into fragments and the waves' sums meet in LDS in wave
// order: one launch, no partials in memory, no barrier in the loop.
//
// Fragments. One 16-column step of K is four matrix instructions; instruction j takes the K values
// 4 g + j of the lanes' groups g = lane / 16, from both operands alike. A k-contiguous operand's lane then
// loads 16 bytes of its row. A k-major one loads, for each j, MB (NB) adjacent rows of K row 4 g + j in one
// piece: its blocks interleave, block m holding rows MB i + m, so one load serves every block.
#include <algorithm>

#include "gemm_tiles.h"

namespace {

typedef float floatx4_f __attribute__((ext_vector_type(4)));

// NBK blocks of 16 rows of one operand for a step: v[block][j] as above.
template <bool KM, int NBK>
struct Frag32 {
  const float* p[KM ? 1 : NBK];
  long ld;

  __device__ __forceinline__ void init(const float* base, long ld_, int row0, int rows, int lane) {
    const int i = lane & 15, g = lane >> 4;
    ld = ld_;
    if constexpr (KM) {
      // Whole pieces past the last row are read from it (rows is a multiple of NBK).
      p[0] = base + min(row0 + NBK * i, rows - NBK) + static_cast<long>(4 * g) * ld;
    } else {
#pragma unroll
      for (int b = 0; b < NBK; ++b) p[b] = base + static_cast<long>(min(row0 + 16 * b + i, rows - 1)) * ld + 4 * g;
    }
  }
  __device__ __forceinline__ void load(int k0, float (&v)[NBK][4]) const {
    if constexpr (KM) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float* q = p[0] + static_cast<long>(k0 + j) * ld;
        if constexpr (NBK == 4) {
          const float4 x = *reinterpret_cast<const float4*>(q);
          v[0][j] = x.x; v[1][j] = x.y; v[2][j] = x.z; v[3][j] = x.w;
        } else if constexpr (NBK == 2) {
          const float2 x = *reinterpret_cast<const float2*>(q);
          v[0][j] = x.x; v[1][j] = x.y;
        } else {
          v[0][j] = *q;
        }
      }
    } else {
#pragma unroll
      for (int b = 0; b < NBK; ++b) {
        const float4 x = *reinterpret_cast<const float4*>(p[b] + k0);
        v[b][0] = x.x; v[b][1] = x.y; v[b][2] = x.z; v[b][3] = x.w;
      }
    }
  }
  // The last step when K is no multiple of 16: values past K are zeros and are not read.
  __device__ __forceinline__ void load_tail(int k0, int K, int lane, float (&v)[NBK][4]) const {
    const int g = lane >> 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool in = k0 + 4 * g + j < K;
#pragma unroll
      for (int b = 0; b < NBK; ++b) {
        if constexpr (KM) v[b][j] = in ? p[0][static_cast<long>(k0 + j) * ld + b] : 0.0f;
        else v[b][j] = in ? p[b][k0 + j] : 0.0f;
      }
    }
  }
};

template <bool A_KM, bool B_KM, int MB, int NB, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void gemm_frag32_kernel(GemmArgs g) {
  constexpr int BM = 16 * MB, BN = 16 * NB, PITCH32 = BN + 4;  // the pad keeps 16-byte pieces and spreads banks
  extern __shared__ __attribute__((aligned(16))) float sums[];  // [WAVES][BM][PITCH32]
  gemm_select_batch(g, blockIdx.z);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row0 = blockIdx.y * BM, col0 = blockIdx.x * BN;
  Frag32<A_KM, MB> fa;
  Frag32<B_KM, NB> fb;
  fa.init(static_cast<const float*>(g.a), g.lda, row0, g.M, lane);
  fb.init(static_cast<const float*>(g.b), g.ldb, col0, g.N, lane);
  floatx4_f acc[MB][NB];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int n = 0; n < NB; ++n) acc[m][n] = floatx4_f{0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply = [&](const float (&a)[MB][4], const float (&b)[NB][4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int n = 0; n < NB; ++n)
          acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[n][j], a[m][j], acc[m][n], 0, 0, 0);
  };
  constexpr int CHUNK = MB + NB <= 4 ? 4 : 2;  // steps whose loads are in flight together
  const int whole = g.K / 16, steps = (g.K + 15) / 16;
  const int s_end = min(whole, steps * (wave + 1) / WAVES);
  for (int s0 = steps * wave / WAVES; s0 < s_end; s0 += CHUNK) {
    const int live = min(CHUNK, s_end - s0);  // uniform over the wave
    float a[CHUNK][MB][4], b[CHUNK][NB][4];
#pragma unroll
    for (int s = 0; s < CHUNK; ++s)
      if (s < live) {
        fa.load((s0 + s) * 16, a[s]);
        fb.load((s0 + s) * 16, b[s]);
      }
#pragma unroll
    for (int s = 0; s < CHUNK; ++s)
      if (s < live) multiply(a[s], b[s]);
  }
  if (whole < steps && wave == WAVES - 1) {
    float a[MB][4], b[NB][4];
    fa.load_tail(whole * 16, g.K, lane, a);
    fb.load_tail(whole * 16, g.K, lane, b);
    multiply(a, b);
  }
  // acc[m][n][v]: A's row i = lane % 16 of block m, B's row 4 (lane / 16) + v of block n, this wave's share of K.
  float* mine = sums + wave * (BM * PITCH32);
  const int i = lane & 15, kg = lane >> 4;
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    float* r = mine + (A_KM ? MB * i + m : 16 * m + i) * PITCH32;
    if constexpr (!B_KM) {
#pragma unroll
      for (int n = 0; n < NB; ++n) *reinterpret_cast<floatx4_f*>(r + 16 * n + 4 * kg) = acc[m][n];
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int n = 0; n < NB; ++n) r[NB * (4 * kg + v) + n] = acc[m][n][v];
    }
  }
  __syncthreads();
  bool bad = false;
  for (int c = threadIdx.x; c < BM * (BN / 4); c += WAVES * 64) {
    const int r = c / (BN / 4), cc = c % (BN / 4) * 4;
    float4 t = *reinterpret_cast<const float4*>(sums + r * PITCH32 + cc);
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
      const float4 u = *reinterpret_cast<const float4*>(sums + (w * BM + r) * PITCH32 + cc);
      t.x += u.x; t.y += u.y; t.z += u.z; t.w += u.w;
    }
    if (row0 + r < g.M && col0 + cc < g.N) bad |= gemm_store4(g, 0, row0 + r, col0 + cc, t.x, t.y, t.z, t.w);
  }
  if (bad) dev_raise_fault(g.fault, g.tag);
}

struct FragTile {
  int mb, nb, waves;
  double step, fixed;  // us per 16 columns of K and per workgroup besides
};
constexpr FragTile FRAG_TILES[] = {{1, 1, 8, 0.055, 0.1}, {1, 2, 8, 0.078, 0.1}, {2, 2, 8, 0.138, 0.2}, {4, 2, 8, 0.19, 0.5}, {4, 4, 4, 0.34, 1.4}};

// Whether an operand's pieces are whole and aligned for `blocks` blocks of 16 rows.
bool frag_fits(bool km, const void* p, long ld, int rows, int blocks, long batch_bytes) {
  const long piece = km ? blocks : 4;
  return ld % piece == 0 && (reinterpret_cast<uintptr_t>(p) & (piece * 4 - 1)) == 0 && batch_bytes % (piece * 4) == 0 &&
         (!km || (rows % blocks == 0 && rows >= blocks));
}

template <bool A_KM, bool B_KM, int T>
int32_t launch_frag(omx_ctx* ctx, const GemmArgs& g) {
  constexpr FragTile t = FRAG_TILES[T];
  constexpr int smem = t.waves * 16 * t.mb * (16 * t.nb + 4) * 4;
  auto kernel = &gemm_frag32_kernel<A_KM, B_KM, t.mb, t.nb, t.waves>;
  if constexpr (smem > 64 * 1024)
    OMX_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
  dim3 grid(static_cast<unsigned>((g.N + 16 * t.nb - 1) / (16 * t.nb)), static_cast<unsigned>((g.M + 16 * t.mb - 1) / (16 * t.mb)),
            static_cast<unsigned>(g.batches));
  omx_launch_timed(ctx, kernel, grid, dim3(t.waves * 64), smem, ctx->timing_start, ctx->timing_stop, g);
  OMX_LAUNCH_CHECK(ctx, "gemm_frag32_kernel");
  return OMX_OK;
}
template <bool A_KM, bool B_KM>
int32_t launch_frag_tile(omx_ctx* ctx, const GemmArgs& g, int tile) {
  switch (tile) {
    case 0: return launch_frag<A_KM, B_KM, 0>(ctx, g);
    case 1: return launch_frag<A_KM, B_KM, 1>(ctx, g);
    case 2: return launch_frag<A_KM, B_KM, 2>(ctx, g);
    case 3: return launch_frag<A_KM, B_KM, 3>(ctx, g);
    default: return launch_frag<A_KM, B_KM, 4>(ctx, g);
  }
}

}  // namespace

// The tile with the least estimated time, or -1 where the 128 x 128 kernel's is less still. Both estimates
// are rounds of workgroups on the compute units times what one costs, fitted over 37 shapes from 128 x 128
// over K = 64 to 4096 x 4096 over 1024 in three layouts: a small tile fills the chip but fetches more per
// product (1 x 1 blocks: 0.055 us per 16 columns of K, a sixth of what 4 x 4 take for a sixteenth of the outputs);
// the 128 x 128 tile is the cheapest per product (2.4 us per 32 columns) and pays some 8 us per launch, and as much
// again for partials and their second launch when its few tiles split K.
// Before and after, forward / input gradient / weight gradient layouts, us: 256 x 256 over 256: 14.3 / 14.5 / 15.6 ->
// 3.3 each; 2048 x 256 over 256: 18.4 / 18.8 / 19.8 -> 7.2 / 6.7 / 6.6; 1024 x 256 over 2048: 30.3 / 30.7 / 31.8 ->
// 23.3 / 21.7 / 19.1; 768 x 768 over 3072 stays (52 against 75).
int omx_gemm_frag32_tile(omx_ctx* ctx, const GemmArgs& g, bool a_km, bool b_km) {
  const long units = ctx->cu_count > 0 ? ctx->cu_count : 256;
  auto rounds = [&](long groups) { return static_cast<double>((groups + units - 1) / units); };
  const double steps = (g.K + 15) / 16;
  int best = -1;
  double best_us = 1e30;
  for (int t = 0; t < 5; ++t) {
    const FragTile& f = FRAG_TILES[t];
    if (!frag_fits(a_km, g.a, g.lda, g.M, f.mb, g.batch_a) || !frag_fits(b_km, g.b, g.ldb, g.N, f.nb, g.batch_b)) continue;
    const long m = (g.M + 16 * f.mb - 1) / (16 * f.mb), n = (g.N + 16 * f.nb - 1) / (16 * f.nb);
    if (m > 65535) continue;
    // Two k-contiguous operands of the larger tiles fetch up to 128 pieces of 64 bytes per step.
    const double step = t >= 3 && !a_km && !b_km ? 1.17 * f.step : f.step;
    const double us = 2.5 + rounds(m * n * g.batches) * (steps * step + f.fixed);
    if (us < best_us) {
      best = t;
      best_us = us;
    }
  }
  if (best < 0) return -1;
  // The 128 x 128 kernel with the splits that omx_gemm_impl gives it.
  const long tiles = static_cast<long>((g.M + 127) / 128) * ((g.N + 127) / 128) * g.batches, ksteps = (g.K + 31) / 32;
  long splits = 1;
  if (ksteps >= 8 && tiles < (g.batches == 1 ? 256 : 512))
    splits = std::max(1l, std::min(((g.batches == 1 ? 512 : 1024) + tiles - 1) / tiles, ksteps / 2));
  const long per_split = (ksteps + splits - 1) / splits;
  splits = (ksteps + per_split - 1) / per_split;
  const double old_us = (8.0 + (splits > 1 ? 8.0 : 0.0) + rounds(tiles * splits) * per_split * 2.4) * (b_km ? a_km ? 1.1 : 1.05 : 1.0);
  return best_us < old_us ? best : -1;
}

int32_t omx_gemm_frag32_launch(omx_ctx* ctx, const GemmArgs& g, bool a_km, bool b_km, int tile) {
  if (!a_km && !b_km) return launch_frag_tile<false, false>(ctx, g, tile);
  if (!a_km) return launch_frag_tile<false, true>(ctx, g, tile);
  if (!b_km) return launch_frag_tile<true, false>(ctx, g, tile);
  return launch_frag_tile<true, true>(ctx, g, tile);
}
