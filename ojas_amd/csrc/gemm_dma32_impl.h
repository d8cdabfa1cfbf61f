// One output tile of the f32 product with direct-to-LDS loads, for the kernels of gemm_dma32.hip (which says what bounds it) and
// the group of products in gemm_frag32.hip.
#pragma once
#include "gemm_tiles.h"

namespace {

typedef float floatx4_d __attribute__((ext_vector_type(4)));
typedef float floatx2_d __attribute__((ext_vector_type(2)));

// The fragments of T blocks of 16 rows (columns of B) over 16 K values, out of an LDS tile of ROWS rows: v[block][j] is K
// value 4 g + j of the lane's group g = lane / 16 (4 j + g where both operands are k-major, KIND 1: adjacent K rows, which
// a swizzle can part), so instruction j of four takes v[.][j] of both operands.
//   k-contiguous tile, [row][8 pieces of 16 bytes], piece p of row r in slot p ^ ((r >> 1) & 7): one 16-byte read a block.
//   k-major tile, [K row][ROWS / 4 pieces], piece p of K row r in slot p ^ km_swizzle(r): the blocks interleave (block m
//   holds rows T i + m), so one read of 4 T bytes serves all of them for one j.
template <bool KM, int ROWS, int T, int KIND>
struct Frag32Lds {
  int off[4];  // KM: per j; else per block
  __device__ __forceinline__ void init(int row0, int lane) {
    const int i = lane & 15, g = lane >> 4;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      if constexpr (KM) {
        const int kr = KIND == 1 ? 4 * x + g : 4 * g + x, col = row0 + T * i;
        off[x] = kr * (ROWS * 4) + (((col >> 2) ^ km_swizzle<2 * ROWS, KIND>(kr)) << 4) + (col & 3) * 4;
      } else {
        const int r = row0 + 16 * x + i;
        off[x] = r * 128 + ((g ^ ((r >> 1) & 7)) << 4);
      }
    }
  }
  // Half kk of a 32-deep step. (K rows 16 apart swizzle alike; piece 4 kk + g of a k-contiguous row is g with bit 2 flipped.)
  __device__ __forceinline__ void read(const char* tile, int kk, float (&v)[T][4]) const {
    if constexpr (KM) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const char* p = tile + off[j] + kk * (16 * ROWS * 4);
        if constexpr (T == 4) {
          const floatx4_d x = *reinterpret_cast<const floatx4_d*>(p);
          v[0][j] = x[0]; v[1][j] = x[1]; v[2][j] = x[2]; v[3][j] = x[3];
        } else if constexpr (T == 2) {
          const floatx2_d x = *reinterpret_cast<const floatx2_d*>(p);
          v[0][j] = x[0]; v[1][j] = x[1];
        } else {
          v[0][j] = *reinterpret_cast<const float*>(p);
        }
      }
    } else {
#pragma unroll
      for (int m = 0; m < T; ++m) {
        const floatx4_d x = *reinterpret_cast<const floatx4_d*>(tile + (off[m] ^ (kk << 6)));
        v[m][0] = x[0]; v[m][1] = x[1]; v[m][2] = x[2]; v[m][3] = x[3];
      }
    }
  }
};

// WGM x WGN waves of TM x TN blocks of 16 x 16, K steps of 32, NST stages. KG groups of such waves share the K steps (step
// s is group s % KG's) and meet in LDS at the end. TAIL: see StepBase (both operands k-major).
// ACT: GELU or its derivative in the store pass (A k-contiguous: an up-projection and the input gradient behind it); 1 erf, 2 tanh. Passes
// of their own took 5.5 and 6.0 us over 2048 x 1024, the step of four blocks 1248 us, 1224 with them here.
// Tile `index` of a product, or of a strided batch of them; smem: NST KG stages, 1024-byte aligned.
template <bool A_KM, bool B_KM, int WGM, int WGN, int TM, int TN, int NST, int KG, bool TAIL, int ACT>
__device__ __forceinline__ void dma32_tile(GemmArgs& g, int index, char* smem) {
  constexpr int BM = WGM * TM * 16, BN = WGN * TN * 16, BK = 32;
  constexpr int A_BYTES = BM * BK * 4, B_BYTES = BN * BK * 4, STAGE = A_BYTES + B_BYTES;
  constexpr int NW = WGM * WGN;           // waves per group
  constexpr int LPS = STAGE / 1024 / NW;  // loads per wave per step
  static_assert(A_BYTES % (1024 * NW) == 0 && B_BYTES % (1024 * NW) == 0, "the same number of loads in every wave");
  const int total = g.tiles_m * g.tiles_n;
  const int r = tile_of_eighth(index, total * g.batches), product = r / total, id = r - product * total;
  const int band = 4, band_id = id / (band * g.tiles_n), first_m = band_id * band;
  const int band_rows = min(band, g.tiles_m - first_m), in_band = id - band_id * (band * g.tiles_n);
  const int m0 = (first_m + in_band % band_rows) * BM, n0 = in_band / band_rows * BN;
  gemm_select_batch(g, product);
  const int lane = threadIdx.x & 63, wave_all = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int group = KG == 1 ? 0 : wave_all / NW, wave = KG == 1 ? wave_all : wave_all % NW;
  const int wm = wave / WGN, wn = wave % WGN;

  floatx4_d acc[TM][TN], sum[TM][TN];  // sum: of the step that runs
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) acc[m][n] = sum[m][n] = floatx4_d{0.0f, 0.0f, 0.0f, 0.0f};

  const int steps = g.K / BK;
  const int rounds = (steps + KG - 1) / KG;  // of every group
  const int mine = (steps - group + KG - 1) / KG;
  // (an f32 tile's pieces are those of a bf16 one with twice the columns)
  constexpr int KIND = A_KM && B_KM ? 1 : 2;
  TileLoadsOff<A_KM, A_KM ? 2 * BM : BM, A_KM ? BK : 2 * BK, NW, TAIL && A_KM, KIND> la;
  TileLoadsOff<B_KM, B_KM ? 2 * BN : BN, B_KM ? BK : 2 * BK, NW, TAIL && B_KM, KIND> lb;
  const int k0 = group * BK;
  la.init(static_cast<const unsigned short*>(g.a), 2 * g.lda, A_KM ? 2 * m0 : m0, A_KM ? 2 * g.M : g.M, A_KM ? k0 : 2 * k0, g.k_rows, wave, lane);
  lb.init(static_cast<const unsigned short*>(g.b), 2 * g.ldb, B_KM ? 2 * n0 : n0, B_KM ? 2 * g.N : g.N, B_KM ? k0 : 2 * k0, g.k_rows, wave, lane);
  Frag32Lds<A_KM, BM, TM, KIND> fa;
  Frag32Lds<B_KM, BN, TN, KIND> fb;
  fa.init(wm * TM * 16, lane);
  fb.init(wn * TN * 16, lane);
  char* const stages = smem + group * (NST * STAGE);
  const unsigned lds0 = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(reinterpret_cast<uintptr_t>(stages)));
  auto issue = [&](int stage) {
    la.issue(lds0 + stage * STAGE, wave);
    lb.issue(lds0 + stage * STAGE + A_BYTES, wave);
    if constexpr (KG > 1) {
#pragma unroll
      for (int skip = 1; skip < KG; ++skip) {
        la.base.advance();
        lb.base.advance();
      }
    }
  };
  static_assert((NST - 2) * LPS < 64, "vmcnt is six bits");
#pragma unroll
  for (int i = 0; i < NST - 1; ++i)
    if (i < mine) issue(i);
  wait_loads<NST - 2, LPS>(min(NST - 2, mine - 1));
  __syncthreads();
  float a[2][TM][4], b[2][TN][4];
  auto read = [&](const char* stage, int kk, int set) {
    fa.read(stage, kk, a[set]);
    fb.read(stage + A_BYTES, kk, b[set]);
  };
  auto multiply = [&](int set) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n) {
          const floatx4_d c = set == 0 && j == 0 ? floatx4_d{0.0f, 0.0f, 0.0f, 0.0f} : sum[m][n];
          sum[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[set][n][j], a[set][m][j], c, 0, 0, 0);
        }
  };
  auto fold = [&]() {
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n) acc[m][n] += sum[m][n];
  };
  if (mine > 0) read(stages, 0, 0);
  // As in gemm_dma_kernel (bf16): the second half's fragments are read before the first half is multiplied, the next step's first
  // ones right after the barrier that publishes its stage, before this step's second half is multiplied.
  for (int ks = 0; ks < rounds;) {
#pragma unroll
    for (int st = 0; st < NST; ++st) {
      const bool live = KG == 1 || ks < mine;
      if (ks + NST - 1 < mine) issue((st + NST - 1) % NST);
      if (live) {
        read(stages + st * STAGE, 1, 1);
        __builtin_amdgcn_sched_barrier(0);
        fold();
        multiply(0);
        __builtin_amdgcn_sched_barrier(0);
      }
      wait_loads<NST - 2, LPS>(max(0, min(NST - 2, mine - ks - 2)));
      __syncthreads();
      if (ks + 1 < mine) read(stages + (st + 1) % NST * STAGE, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (live) multiply(1);
      __builtin_amdgcn_sched_barrier(0);
      if (++ks >= rounds) break;
    }
  }
  fold();
  if constexpr (KG > 1) {
    // The other groups' sums, in group order (the last step's barrier has released the stages).
    floatx4_d* meet = reinterpret_cast<floatx4_d*>(smem);
    static_assert((KG - 1) * NW * TM * TN * 1024 <= NST * KG * STAGE, "the sums fit");
    if (group > 0)
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n) meet[((((group - 1) * NW + wave) * TM + m) * TN + n) * 64 + lane] = acc[m][n];
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int o = 0; o < KG - 1; ++o)
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n) acc[m][n] += meet[(((o * NW + wave) * TM + m) * TN + n) * 64 + lane];
  }
  // acc[m][n][v]: A's row i = lane % 16 of block m, B's row 4 (lane / 16) + v of block n.
  const int i = lane & 15, kg = lane >> 4;
  int bad = 0;
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int row = m0 + wm * TM * 16 + (A_KM ? TM * i + m : 16 * m + i);
    if (row < g.M) {
#pragma unroll
      for (int p = 0; p < TN; ++p) {  // four columns a piece
        const int col = n0 + wn * TN * 16 + (B_KM ? 4 * (TN * kg + p) : 16 * p + 4 * kg);
        float x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (B_KM) x[e] = acc[m][(4 * p + e) % TN][(4 * p + e) / TN];
          else x[e] = acc[m][p][e];
        }
        if (col < g.N) {
          if constexpr (ACT == 0) bad |= gemm_store4(g, 0, row, col, x[0], x[1], x[2], x[3]);
          else bad |= gemm_store4_act32<ACT == 2>(g, row, col, x[0], x[1], x[2], x[3]);
        }
      }
    }
  }
  if (bad & 1) dev_raise_fault(g.fault, g.tag);
  if (ACT != 0 && (bad & 2)) dev_raise_fault(g.fault, g.act_tag);
}

}  // namespace
