// bf16 product with few rows: C[M, N] = A.B with A [M, K] and B's columns [N, K] both k-contiguous (a decoder's
// linear layers on one token per sequence, or on a short prompt chunk). Same contract as gemm.hip
// (f32 accumulation; reference: ojas-cpu/src/linalg.rs:69-210).
//
// Such a product reads N x K of weights for 2 M operations per value: it is bound by reading the
// weights once, and with a few hundred KiB of them by one round of memory latency and the launch. The
// 128-row tiles of the other kernels leave all but N / 128 compute units idle and run their K loop as
// a serial chain of loads, barriers and products. Here a workgroup owns 16 NB columns and up to 64
// rows, and its waves share K between them: both operands go from memory straight into
// v_mfma_f32_16x16x32_bf16 fragments (a lane's eight k-consecutive values are one 16-byte load; no
// LDS, no barrier in the loop), CHUNK steps' loads are in flight together, and the waves'
// partial sums meet in LDS in wave order: one launch, no split-K pass.
#include "gemm_tiles.h"

namespace {

typedef __bf16 bf16x8_s __attribute__((ext_vector_type(8)));
typedef float floatx4_s __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_s __attribute__((ext_vector_type(4)));



// MB x NB blocks of 16 rows x 16 columns per workgroup.
// PLAIN: no activation in the store pass (whose code a call of a few rows would fetch for nothing: GELU is two thirds of
// the kernel).
template <int MB, int NB, int WAVES, int CHUNK, bool PLAIN>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_kernel(GemmArgs g) {
  extern __shared__ float skinny_red[];  // [WAVES][MB * NB][4][64]
  gemm_select_batch(g, blockIdx.z);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, kc = (lane >> 4) * 8;
  const int row0 = blockIdx.y * (16 * MB), col0 = blockIdx.x * (16 * NB);
  // Rows and columns past the end are read from the last one and never stored.
  const unsigned short* a[MB];
  const unsigned short* b[NB];
#pragma unroll
  for (int m = 0; m < MB; ++m)
    a[m] = static_cast<const unsigned short*>(g.a) + static_cast<long>(min(row0 + m * 16 + l16, g.M - 1)) * g.lda + kc;
#pragma unroll
  for (int n = 0; n < NB; ++n)
    b[n] = static_cast<const unsigned short*>(g.b) + static_cast<long>(min(col0 + n * 16 + l16, g.N - 1)) * g.ldb + kc;
  floatx4_s acc[MB][NB];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int n = 0; n < NB; ++n) acc[m][n] = floatx4_s{0.0f, 0.0f, 0.0f, 0.0f};

  const int steps = g.K / 32;
  const int s_end = steps * (wave + 1) / WAVES;
  for (int s0 = steps * wave / WAVES; s0 < s_end; s0 += CHUNK) {
    const int live = min(CHUNK, s_end - s0);  // uniform over the wave
    u32x4_s bf[CHUNK][NB], af[CHUNK][MB];
#pragma unroll
    for (int s = 0; s < CHUNK; ++s) {
      if (s < live) {
        const long k = static_cast<long>(s0 + s) * 32;
#pragma unroll
        for (int n = 0; n < NB; ++n) bf[s][n] = *reinterpret_cast<const u32x4_s*>(b[n] + k);
#pragma unroll
        for (int m = 0; m < MB; ++m) af[s][m] = *reinterpret_cast<const u32x4_s*>(a[m] + k);
      }
    }
#pragma unroll
    for (int s = 0; s < CHUNK; ++s)
      if (s < live)
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
          for (int m = 0; m < MB; ++m)
            acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_s, bf[s][n]),
                                                                __builtin_bit_cast(bf16x8_s, af[s][m]), acc[m][n], 0, 0, 0);
  }
  // acc[m][n][v] is row m * 16 + l16, column n * 16 + 4 * (lane / 16) + v of this wave's share of K.
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int v = 0; v < 4; ++v) skinny_red[((wave * (MB * NB) + m * NB + n) * 4 + v) * 64 + lane] = acc[m][n][v];
  __syncthreads();
  bool bad = false;
  for (int blk = wave; blk < MB * NB; blk += WAVES) {
    const int row = row0 + blk / NB * 16 + l16, col = col0 + blk % NB * 16 + (lane >> 4) * 4;
    // Neighbours first: the error of a sum of eight grows with three additions, not with seven.
    float x[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float part[WAVES];
#pragma unroll
      for (int w = 0; w < WAVES; ++w) part[w] = skinny_red[((w * (MB * NB) + blk) * 4 + v) * 64 + lane];
#pragma unroll
      for (int span = 1; span < WAVES; span *= 2)
#pragma unroll
        for (int w = 0; w < WAVES; w += 2 * span) part[w] += part[w + span];
      x[v] = part[0];
    }
    if (row < g.M && col < g.N)
      bad |= PLAIN ? gemm_store4(g, 0, row, col, x[0], x[1], x[2], x[3]) : gemm_store4_epi(g, 0, row, col, x[0], x[1], x[2], x[3]);
  }
  if (bad) dev_raise_fault(g.fault, g.tag);
}

// The same for up to four rows and few columns: four columns per workgroup, so that four times as many compute units read the
// weights. The 16 row and the 16 column places of a product are 4 rows or columns x 4 quarters of K; of its 256 sums the 64 whose two
// quarters agree are kept (lanes l16 / 4 == lane / 16), and a workgroup's 4 columns x K come in loads as wide as before. One row, 768
// columns, us in a decode step:
// K = 768 3.7 -> 3.0, K = 3072 6.2 -> 3.9 (16 columns there were 12 steps a wave, four at a time, and 98 KB a compute unit).
template <int WAVES, int CHUNK, bool PLAIN>
__global__ __launch_bounds__(WAVES * 64) void gemm_rows4_kernel(GemmArgs g) {
  __shared__ float red[WAVES * 64];  // [wave][quarter][row][column]
  gemm_select_batch(g, blockIdx.z);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, quarter = l16 >> 2, col0 = blockIdx.x * 4;
  const long k0 = static_cast<long>(quarter) * (g.K / 4) + (lane >> 4) * 8;
  // Rows and columns past the end are read from the last one and never stored.
  const unsigned short* a = static_cast<const unsigned short*>(g.a) + static_cast<long>(min(l16 & 3, g.M - 1)) * g.lda + k0;
  const unsigned short* b = static_cast<const unsigned short*>(g.b) + static_cast<long>(min(col0 + (l16 & 3), g.N - 1)) * g.ldb + k0;
  floatx4_s acc = {0.0f, 0.0f, 0.0f, 0.0f};
  const int steps = g.K / 128;
  const int s_end = steps * (wave + 1) / WAVES;
  for (int s0 = steps * wave / WAVES; s0 < s_end; s0 += CHUNK) {
    const int live = min(CHUNK, s_end - s0);  // uniform over the wave
    u32x4_s bf[CHUNK], af[CHUNK];
#pragma unroll
    for (int s = 0; s < CHUNK; ++s)
      if (s < live) {
        bf[s] = *reinterpret_cast<const u32x4_s*>(b + (s0 + s) * 32);
        af[s] = *reinterpret_cast<const u32x4_s*>(a + (s0 + s) * 32);
      }
#pragma unroll
    for (int s = 0; s < CHUNK; ++s)
      if (s < live)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_s, bf[s]), __builtin_bit_cast(bf16x8_s, af[s]), acc, 0, 0, 0);
  }
  // acc[v]: row place l16, column place 4 * (lane / 16) + v.
  if (quarter == lane >> 4) *reinterpret_cast<floatx4_s*>(red + wave * 64 + l16 * 4) = acc;
  __syncthreads();
  if (wave != 0) return;
  // Lane: row lane / 16, quarter lane / 4 % 4, column lane % 4. Neighbours first, then the quarters.
  float part[WAVES];
#pragma unroll
  for (int w = 0; w < WAVES; ++w) part[w] = red[w * 64 + (quarter * 4 + (lane >> 4)) * 4 + (lane & 3)];
#pragma unroll
  for (int span = 1; span < WAVES; span *= 2)
#pragma unroll
    for (int w = 0; w < WAVES; w += 2 * span) part[w] += part[w + span];
  float x = part[0];
  x += dev_dpp<0x128>(x);  // row_ror 8, 4: the quarter two away, then the other two
  x += dev_dpp<0x124>(x);
  const float x0 = dev_dpp<0x00>(x), x1 = dev_dpp<0x55>(x), x2 = dev_dpp<0xAA>(x), x3 = dev_dpp<0xFF>(x);  // quad_perm: one column to all
  const int row = lane >> 4;
  if (l16 == 0 && row < g.M) {
    const bool bad = PLAIN ? gemm_store4(g, 0, row, col0, x0, x1, x2, x3) : gemm_store4_epi(g, 0, row, col0, x0, x1, x2, x3);
    if (bad) dev_raise_fault(g.fault, g.tag);
  }
}

// The low-rank term of a workgroup's rows and columns, by one wave: operands straight from memory, 32 of the rank a step (16 past its end are
// zeros).
template <int MB>
__device__ __forceinline__ void skinny_low_rank(const GemmArgs& g, floatx4_s (&acc)[MB][4], int row0, int col0, int lane) {
  const int l16 = lane & 15, kg = lane >> 4;
#pragma unroll 1
  for (int p = kg * 8; p - kg * 8 < g.lr_rank; p += 32) {
    u32x4_s w[4], h[4][MB];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const long off = g.lr_block_cols > 0 ? static_cast<long>(min(col0 + n * 16, g.N - 1) / g.lr_block_cols) * g.lr_rank : 0;
      w[n] = u32x4_s{0u, 0u, 0u, 0u};
      if (p < g.lr_rank) w[n] = *reinterpret_cast<const u32x4_s*>(g.lr_w + min(col0 + n * 16 + l16, g.N - 1) * g.lr_w_pitch + p);
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        h[n][m] = u32x4_s{0u, 0u, 0u, 0u};
        if (p < g.lr_rank) h[n][m] = *reinterpret_cast<const u32x4_s*>(g.lr_h + min(row0 + m * 16 + l16, g.M - 1) * g.lr_pitch + off + p);
      }
    }
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int m = 0; m < MB; ++m)
        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_s, w[n]), __builtin_bit_cast(bf16x8_s, h[n][m]), acc[m][n], 0, 0, 0);
  }
}
// The waves' sums over 16 MB rows x 64 columns meet and go out: acc[m][n][v] is row m * 16 + lane % 16, column n * 16 + 4 * (lane / 16) + v.
template <int MB, int WAVES, bool PLAIN>
__device__ __forceinline__ void skinny_meet(const GemmArgs& g, const floatx4_s (&acc)[MB][4], float* red, int row0, int col0, int wave, int lane) {
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[((wave * (MB * 4) + m * 4 + n) * 4 + v) * 64 + lane] = acc[m][n][v];
  __syncthreads();
  bool bad = false;
  for (int blk = wave; blk < MB * 4; blk += WAVES) {
    const int row = row0 + blk / 4 * 16 + (lane & 15), col = col0 + blk % 4 * 16 + (lane >> 4) * 4;
    float x[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float part[WAVES];
#pragma unroll
      for (int w = 0; w < WAVES; ++w) part[w] = red[((w * (MB * 4) + blk) * 4 + v) * 64 + lane];
#pragma unroll
      for (int span = 1; span < WAVES; span *= 2)
#pragma unroll
        for (int w = 0; w < WAVES; w += 2 * span) part[w] += part[w + span];
      x[v] = part[0];
    }
    if (row < g.M && col < g.N)
      bad |= PLAIN ? gemm_store4(g, 0, row, col, x[0], x[1], x[2], x[3]) : gemm_store4_epi(g, 0, row, col, x[0], x[1], x[2], x[3]);
  }
  if (bad) dev_raise_fault(g.fault, g.tag);
}

// The same with B by rows of K (an input gradient's weights): 16 MB rows by 64 columns a workgroup, whose waves take runs of 32-row steps
// of K. B comes in pieces of a row and turns in LDS of the wave's own (144-byte rows: the four rows of a transposing read lie in
// different banks), SKINNY_KM_CHUNK steps in flight together, no barrier before the waves' sums meet.
typedef short short4_s __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_s __attribute__((ext_vector_type(2)));
constexpr int KM_PITCH = 144, KM_CHUNK = 2;
template <int MB, int WAVES>
constexpr int km_lds() {
  return WAVES * KM_CHUNK * 32 * KM_PITCH > WAVES * MB * 4096 ? WAVES * KM_CHUNK * 32 * KM_PITCH : WAVES * MB * 4096;
}
template <int MB, int WAVES, bool PLAIN>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny64_km_kernel(GemmArgs g) {
  extern __shared__ __attribute__((aligned(16))) char km_smem[];
  gemm_select_batch(g, blockIdx.z);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int l16 = lane & 15, kg = lane >> 4, piece = lane & 7, krow = lane >> 3;
  const int row0 = blockIdx.y * (16 * MB), col0 = blockIdx.x * 64;
  // Rows and columns past the end are read from the last ones and never stored.
  const unsigned short* a[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) a[m] = static_cast<const unsigned short*>(g.a) + static_cast<long>(min(row0 + m * 16 + l16, g.M - 1)) * g.lda + kg * 8;
  const unsigned short* const b = static_cast<const unsigned short*>(g.b) + min(col0 + piece * 8, g.N - 8) + static_cast<long>(krow) * g.ldb;
  char* const own = km_smem + wave * (KM_CHUNK * 32 * KM_PITCH);
  floatx4_s acc[MB][4];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[m][n] = floatx4_s{0.0f, 0.0f, 0.0f, 0.0f};
  const int steps = g.K / 32, s_end = steps * (wave + 1) / WAVES;
  u32x4_s bf[KM_CHUNK][4], af[KM_CHUNK][MB];
  auto fetch = [&](int s0) {
#pragma unroll
    for (int s = 0; s < KM_CHUNK; ++s)
      if (s0 + s < s_end) {  // uniform over the wave
        const long k = static_cast<long>(s0 + s) * 32;
#pragma unroll
        for (int i = 0; i < 4; ++i) bf[s][i] = *reinterpret_cast<const u32x4_s*>(b + (k + 8 * i) * g.ldb);
#pragma unroll
        for (int m = 0; m < MB; ++m) af[s][m] = *reinterpret_cast<const u32x4_s*>(a[m] + k);
      }
  };
  int s0 = steps * wave / WAVES;
  fetch(s0);
  for (; s0 < s_end; s0 += KM_CHUNK) {
    const int live = min(KM_CHUNK, s_end - s0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();  // the previous rows have been read
    u32x4_s am[KM_CHUNK][MB];
#pragma unroll
    for (int s = 0; s < KM_CHUNK; ++s)
      if (s < live) {
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4_s*>(own + (s * 32 + i * 8 + krow) * KM_PITCH + piece * 16) = bf[s][i];
#pragma unroll
        for (int m = 0; m < MB; ++m) am[s][m] = af[s][m];
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (s0 + KM_CHUNK < s_end) fetch(s0 + KM_CHUNK);
#pragma unroll
    for (int s = 0; s < KM_CHUNK; ++s)
      if (s < live) {
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          // Lane (column l16, kg) gets rows 8 kg .. 8 kg + 7 of column n * 16 + l16.
          typedef short4_s __attribute__((address_space(3))) * lds_ptr;
          const char* p = own + (s * 32 + kg * 8 + (l16 >> 2)) * KM_PITCH + n * 32 + (l16 & 3) * 8;
          const u32x2_s lo = __builtin_bit_cast(u32x2_s, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p)));
          const u32x2_s hi = __builtin_bit_cast(u32x2_s, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p + 4 * KM_PITCH)));
          const u32x4_s w = u32x4_s{lo.x, lo.y, hi.x, hi.y};
#pragma unroll
          for (int m = 0; m < MB; ++m)
            acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_s, w), __builtin_bit_cast(bf16x8_s, am[s][m]), acc[m][n], 0, 0, 0);
        }
      }
  }
  if (g.lr_rank > 0 && wave == 0) skinny_low_rank<MB>(g, acc, row0, col0, lane);  // (no wave has fewer steps)
  __syncthreads();  // the steps' LDS has been read
  skinny_meet<MB, WAVES, PLAIN>(g, acc, reinterpret_cast<float*>(km_smem), row0, col0, wave, lane);
}

// The same with B's columns by K, in steps of 64: a load takes whole 128-byte lines of 8 columns, where gemm_skinny_kernel's take half
// lines of 16, and half as many times as its 32 x 32 tiles do for their rows' share.
template <int MB, int WAVES>
constexpr int kc_lds() {
  return WAVES * 64 * KM_PITCH > WAVES * MB * 4096 ? WAVES * 64 * KM_PITCH : WAVES * MB * 4096;
}
template <int MB, int WAVES, bool PLAIN>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny64_kc_kernel(GemmArgs g) {
  extern __shared__ __attribute__((aligned(16))) char km_smem[];
  gemm_select_batch(g, blockIdx.z);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int l16 = lane & 15, kg = lane >> 4, piece = lane & 7, ncol = lane >> 3;
  const int row0 = blockIdx.y * (16 * MB), col0 = blockIdx.x * 64;
  const unsigned short* a[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) a[m] = static_cast<const unsigned short*>(g.a) + static_cast<long>(min(row0 + m * 16 + l16, g.M - 1)) * g.lda + kg * 8;
  const unsigned short* b[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) b[i] = static_cast<const unsigned short*>(g.b) + static_cast<long>(min(col0 + i * 8 + ncol, g.N - 1)) * g.ldb + piece * 8;
  char* const own = km_smem + wave * (64 * KM_PITCH);
  floatx4_s acc[MB][4];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[m][n] = floatx4_s{0.0f, 0.0f, 0.0f, 0.0f};
  const int steps = g.K / 64, s_end = steps * (wave + 1) / WAVES;
  u32x4_s bf[8], af[2][MB];
  auto fetch = [&](int s) {
    const long k = static_cast<long>(s) * 64;
#pragma unroll
    for (int i = 0; i < 8; ++i) bf[i] = *reinterpret_cast<const u32x4_s*>(b[i] + k);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int m = 0; m < MB; ++m) af[t][m] = *reinterpret_cast<const u32x4_s*>(a[m] + k + t * 32);
  };
  int s0 = steps * wave / WAVES;
  if (s0 < s_end) fetch(s0);
  for (; s0 < s_end; ++s0) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    u32x4_s am[2][MB];
#pragma unroll
    for (int i = 0; i < 8; ++i) *reinterpret_cast<u32x4_s*>(own + (i * 8 + ncol) * KM_PITCH + piece * 16) = bf[i];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int m = 0; m < MB; ++m) am[t][m] = af[t][m];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (s0 + 1 < s_end) fetch(s0 + 1);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const u32x4_s w = *reinterpret_cast<const u32x4_s*>(own + (n * 16 + l16) * KM_PITCH + t * 64 + kg * 16);
#pragma unroll
        for (int m = 0; m < MB; ++m)
          acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_s, w), __builtin_bit_cast(bf16x8_s, am[t][m]), acc[m][n], 0, 0, 0);
      }
  }
  if (g.lr_rank > 0 && wave == 0) skinny_low_rank<MB>(g, acc, row0, col0, lane);
  __syncthreads();
  skinny_meet<MB, WAVES, PLAIN>(g, acc, reinterpret_cast<float*>(km_smem), row0, col0, wave, lane);
}

struct SkinnyTile {
  int mb, nb;
};
constexpr SkinnyTile SKINNY_TILES[] = {{1, 1}, {1, 2}, {2, 2}, {4, 4}};
constexpr int SKINNY_CHUNK = 4;

// The smallest tile that makes at most one workgroup per compute unit: a workgroup's time is its own
// operand rows (2.5 us + about 1 ns per column of K and 16-row block: a CU fetches 64-byte row pieces at
// some 65 GB/s), so a bigger tile pays only when it saves a second round of workgroups. Beyond
// K (MB + NB) = 18000, some 20 us, splitting K over the chip and adding up in a second launch is as fast
// (768 columns over K = 3072: 13 against 19 us at 256 rows, 25 against 20 at 512). At most 32 rows of any
// width: the weights are nearly all there is to read, so the tile follows the rows and the columns run in as
// many rounds as they need (50304 columns over K = 768, one row: 14.4 us = 5.4 TB/s). -1: neither.
// One row, 768 x 768: 15.2 -> 3.2 us; 64 rows: 16.6 -> 3.8; 1024 rows: 19.3 -> 9.4 with their split pass.
int skinny_tile(const GemmArgs& g, long units) {
  const long m = (g.M + 15) / 16, n = (g.N + 15) / 16;
  for (int t = 0; t < 4; ++t) {
    const SkinnyTile tile = SKINNY_TILES[t];
    const long groups = ((m + tile.mb - 1) / tile.mb) * ((n + tile.nb - 1) / tile.nb);
    if (groups * g.batches <= units) return static_cast<long>(g.K) * (tile.mb + tile.nb) <= 18000 ? t : -1;
  }
  if (g.K > 4096) return -1;
  if (g.M <= 4) return 0;
  if (g.M <= 16) return 1;
  if (g.M <= 32) return 2;
  return -1;
}

template <int MB, int NB, int WAVES>
int32_t launch_skinny_waves(omx_ctx* ctx, const GemmArgs& g) {
  constexpr int smem = WAVES * MB * NB * 1024;
  auto kernel = g.epi == OMX_EPI_NONE ? &gemm_skinny_kernel<MB, NB, WAVES, SKINNY_CHUNK, true> : &gemm_skinny_kernel<MB, NB, WAVES, SKINNY_CHUNK, false>;
  if constexpr (smem > 64 * 1024)
    OMX_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
  dim3 grid(static_cast<unsigned>((g.N + 16 * NB - 1) / (16 * NB)), static_cast<unsigned>((g.M + 16 * MB - 1) / (16 * MB)),
            static_cast<unsigned>(g.batches));
  omx_launch_timed(ctx, kernel, grid, dim3(WAVES * 64), smem, ctx->timing_start, ctx->timing_stop, g);
  OMX_LAUNCH_CHECK(ctx, "gemm_skinny_kernel");
  return OMX_OK;
}
// Eight waves share K; up to 512 columns four do (two to four steps each), with half the sums to meet. (Sixteen over K = 3072, six
// steps in flight each: 64 rows by 768 columns 8.4 -> 8.9 us.)
template <int MB, int NB>
int32_t launch_skinny(omx_ctx* ctx, const GemmArgs& g) {
  return g.K <= 512 ? launch_skinny_waves<MB, NB, 4>(ctx, g) : launch_skinny_waves<MB, NB, 8>(ctx, g);
}

// Four rows at most, a workgroup per four columns at most one per compute unit, quarters of K whole steps.
bool rows4(const GemmArgs& g, long units) { return g.M <= 4 && g.K % 128 == 0 && (g.N + 3l) / 4 * g.batches <= units; }
int32_t launch_rows4(omx_ctx* ctx, const GemmArgs& g) {
  const bool plain = g.epi == OMX_EPI_NONE, few = g.K <= 1024;
  auto kernel = few ? (plain ? &gemm_rows4_kernel<4, 2, true> : &gemm_rows4_kernel<4, 2, false>)
                    : (plain ? &gemm_rows4_kernel<8, 4, true> : &gemm_rows4_kernel<8, 4, false>);
  dim3 grid(static_cast<unsigned>((g.N + 3) / 4), 1, static_cast<unsigned>(g.batches));
  omx_launch_timed(ctx, kernel, grid, dim3(few ? 256 : 512), 0, ctx->timing_start, ctx->timing_stop, g);
  OMX_LAUNCH_CHECK(ctx, "gemm_rows4_kernel");
  return OMX_OK;
}

template <int MB, bool B_KM>
int32_t launch_km(omx_ctx* ctx, const GemmArgs& g) {
  constexpr int WAVES = 8, smem = B_KM ? km_lds<MB, WAVES>() : kc_lds<MB, WAVES>();
  auto kernel = B_KM ? (g.epi == OMX_EPI_NONE ? &gemm_skinny64_km_kernel<MB, WAVES, true> : &gemm_skinny64_km_kernel<MB, WAVES, false>)
                     : (g.epi == OMX_EPI_NONE ? &gemm_skinny64_kc_kernel<MB, WAVES, true> : &gemm_skinny64_kc_kernel<MB, WAVES, false>);
  if constexpr (smem > 64 * 1024)
    OMX_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
  dim3 grid(static_cast<unsigned>((g.N + 63) / 64), static_cast<unsigned>((g.M + 16 * MB - 1) / (16 * MB)), static_cast<unsigned>(g.batches));
  omx_launch_timed(ctx, kernel, grid, dim3(WAVES * 64), smem, ctx->timing_start, ctx->timing_stop, g);
  OMX_LAUNCH_CHECK(ctx, "gemm_skinny64_km_kernel");
  return OMX_OK;
}

}  // namespace

// What the product takes here, in us; negative: not one for this kernel. Kernel times by tile (46 shapes of 48 to 1024 rows over 128 to 768; the
// last, whose sixteen blocks' sums meet, 700 to 2048 rows: 5.2 / 6.2 / 7.4 over 128 / 256 / 384, which 64 x 64 tiles take 4.0 / 4.5 /
// 4.9 for; with an activation a microsecond more: 2048 x 512 over 512 9.3, 5.5 there).
double omx_gemm_skinny_us(omx_ctx* ctx, const GemmArgs& g, bool a_km, bool b_km, bool activation) {
  if (a_km || b_km || g.K % 32 != 0 || !g.a_vec || !g.b_vec) return -1.0;
  const int t = skinny_tile(g, ctx->cu_count > 0 ? ctx->cu_count : 256);
  static constexpr double kBase[4] = {2.45, 2.85, 2.9, 4.2}, kColumn[4] = {1.9e-3, 2.7e-3, 3.8e-3, 8.1e-3};
  return t < 0 ? -1.0 : kBase[t] + kColumn[t] * g.K + (activation && t == 3 ? 1.0 : 0.0);
}

int32_t omx_gemm_skinny_launch(omx_ctx* ctx, const GemmArgs& g) {
  if (rows4(g, ctx->cu_count > 0 ? ctx->cu_count : 256)) return launch_rows4(ctx, g);
  switch (skinny_tile(g, ctx->cu_count > 0 ? ctx->cu_count : 256)) {
    case 0: return launch_skinny<1, 1>(ctx, g);
    case 1: return launch_skinny<1, 2>(ctx, g);
    case 2: return launch_skinny<2, 2>(ctx, g);
    default: return launch_skinny<4, 4>(ctx, g);
  }
}

// Row blocks of 16 that a workgroup of the 64-column kernels takes, and what the product takes there, in us; negative: not one for them. One
// block where that makes at most a workgroup per compute unit, else two where they do; a second round of workgroups is what
// the 64 x 64 tiles gain by (400 x 2048 over 768: 7.0 there, 8.4 to 10 here). us of a call. B by rows of K, 64 x 64 tiles / here:
// 282 x 640 and 768 over 768 6.3 / 4.7, over 1280 7.9 / 6.0, over 2048 10.3 / 7.5; 64 x 1024 over 768 6.1 / 4.8; 400 x 1024 over
// 1280 8.4 / 7.1 (two blocks); over 4096 and more the tiles' split reductions are ahead. B's columns by K, gemm_skinny_kernel's
// tiles of 16 x 32 and more / here: 200 x 640 over 2048 10.0 / 7.1, over 4096 17.1 / 10.9; 96 x 2048 over 3072 13.7 / 9.1; 512 x
// 384 over 2048 10.1 / 7.2; its 16 x 16 tiles stay ahead (64 x 768 over 1280 5.1 / 5.9). Sums of eight short chains, as there.
double omx_gemm_skinny64_us(omx_ctx* ctx, const GemmArgs& g, bool a_km, bool b_km, int* mb) {
  if (a_km || g.K % (b_km ? 32 : 64) != 0 || g.K > 4096 || (b_km && g.N % 8 != 0) || !g.a_vec || !g.b_vec || ctx->gemm_skinny64 == 0) return -1.0;
  const long units = ctx->cu_count > 0 ? ctx->cu_count : 256, cols = (g.N + 63l) / 64 * g.batches;
  if (ctx->gemm_skinny64 > 0) {  // forced (a grid's rows of workgroups are 16 bits)
    *mb = ctx->gemm_skinny64;
    return g.M <= 1 << 16 ? 0.0 : -1.0;
  }
  *mb = (g.M + 15l) / 16 * cols <= units ? 1 : 2;
  if (*mb == 2 && (g.M + 31l) / 32 * cols > units) return -1.0;
  // Kernel times. By rows of K a sixth less, for the 64 x 64 tiles take half a microsecond more there than their estimate says (512 x 256 over
  // 128 4.0, here 3.4).
  if (b_km) return 0.85 * (*mb == 1 ? 3.2 + 1.8e-3 * g.K : 3.4 + 2.5e-3 * g.K);
  return *mb == 1 ? 3.35 + 1.85e-3 * g.K : 3.7 + 2.75e-3 * g.K;
}

int32_t omx_gemm_skinny64_launch(omx_ctx* ctx, const GemmArgs& g, bool b_km, int mb) {
  if (!b_km) return mb == 1 ? launch_km<1, false>(ctx, g) : launch_km<2, false>(ctx, g);
  return mb == 1 ? launch_km<1, true>(ctx, g) : launch_km<2, true>(ctx, g);
}
