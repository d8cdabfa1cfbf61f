// f32 product of a small output: C[M, N] (+)= A.B with the contract of gemm.hip (f32 operands and f32
// accumulation on v_mfma_f32_16x16x4_f32; reference: ojas-cpu/src/linalg.rs:69-210).
//
// A model a few hundred wide makes outputs of 64 Ki to a few Mi values: on 128 x 128 tiles that is 4 to 100
// workgroups for 256 compute units, so K was split into partials and added up by a second launch, and a
// tile's 64 matrix instructions per 32-column step ran as a chain of load, barrier, product (13 us and
// 4 us for the second launch, whatever the size). gemm_dma32.hip's tiles fill the chip from some 256 x 512 outputs on; below,
// and where a k-contiguous operand's K is not whole steps of 32, this kernel stands. Here a workgroup owns 16 MB x 16 NB outputs and its waves
// share K, both operands go from memory straight into fragments and the waves' sums meet in LDS in wave
// order: one launch, no partials in memory, no barrier in the loop.
//
// Fragments. One 16-column step of K is four matrix instructions; instruction j takes the K values
// 4 g + j of the lanes' groups g = lane / 16, from both operands alike. A k-contiguous operand's lane then
// loads 16 bytes of its row. A k-major one loads, for each j, MB (NB) adjacent rows of K row 4 g + j in one
// piece: its blocks interleave, block m holding rows MB i + m, so one load serves every block.
#include "gemm_dma32_impl.h"

namespace {

typedef float floatx4_f __attribute__((ext_vector_type(4)));
typedef float floatx2_f __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(1))) char* GlobalBytes;
// A value of T at a scalar address plus the lane's offset (the empty assembly keeps the compiler from moving scalar
// parts of the address into vector registers).
template <typename T>
__device__ __forceinline__ T load_at(GlobalBytes at, unsigned off) {
  asm("" : "+s"(at));
  return *reinterpret_cast<const __attribute__((address_space(1))) T*>(at + off);
}

// NBK blocks of 16 rows of one operand for a step: v[block][j] as above. A step's address is a scalar, the lanes add
// 32-bit offsets that never change: with 64-bit addresses per lane and load, the multiplications of a step took a fifth
// of the issue slots that its matrix instructions need.
template <bool KM, int NBK>
struct Frag32 {
  GlobalBytes base;  // the tile's first row at K = 0
  long ld;           // bytes
  unsigned off[KM ? 1 : NBK];

  __device__ __forceinline__ void init(const float* first, long ld_, int row0, int rows, int lane) {
    const int i = lane & 15, g = lane >> 4;
    ld = ld_ * 4;
    const unsigned long long at = reinterpret_cast<unsigned long long>(first) + (KM ? row0 * 4l : row0 * ld);
    // (tile coordinates come out of vector divisions: back to scalars)
    const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(at));
    const unsigned hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(at >> 32));
    base = reinterpret_cast<GlobalBytes>((static_cast<unsigned long long>(hi) << 32) | lo);
    if constexpr (KM) {
      // Whole pieces past the last row are read from it (rows is a multiple of NBK).
      off[0] = static_cast<unsigned>(min(NBK * i, rows - NBK - row0)) * 4u + static_cast<unsigned>(4 * g) * static_cast<unsigned>(ld);
    } else {
#pragma unroll
      for (int b = 0; b < NBK; ++b)
        off[b] = static_cast<unsigned>(min(16 * b + i, rows - 1 - row0)) * static_cast<unsigned>(ld) + 16u * g;
    }
  }
  // Quarter `j` of a step's loads: K row 4 g + j of a k-major operand, a quarter of a k-contiguous one's blocks.
  __device__ __forceinline__ void load(int k0, int j, float (&v)[NBK][4]) const {
    if constexpr (KM) {
      GlobalBytes at = base + (k0 + j) * ld;
      if constexpr (NBK == 4) {
        const floatx4_f x = load_at<floatx4_f>(at, off[0]);
        v[0][j] = x[0]; v[1][j] = x[1]; v[2][j] = x[2]; v[3][j] = x[3];
      } else if constexpr (NBK == 2) {
        const floatx2_f x = load_at<floatx2_f>(at, off[0]);
        v[0][j] = x[0]; v[1][j] = x[1];
      } else {
        v[0][j] = load_at<float>(at, off[0]);
      }
    } else if (j * NBK % 4 == 0) {
      const int b = j * NBK / 4;
      const floatx4_f x = load_at<floatx4_f>(base + k0 * 4l, off[b]);
      v[b][0] = x[0]; v[b][1] = x[1]; v[b][2] = x[2]; v[b][3] = x[3];
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
        if constexpr (KM) v[b][j] = in ? load_at<float>(base + (k0 + j) * ld + 4 * b, off[0]) : 0.0f;
        else v[b][j] = in ? load_at<float>(base + (k0 + j) * 4l, off[b]) : 0.0f;
      }
    }
  }
};

// A wave's share of a tile's sums into its part of [WAVES][16 MB][16 NB + 4] in LDS. acc[m][n][v]: A's row i = lane % 16 of block
// m, B's row 4 (lane / 16) + v of block n.
template <bool A_KM, bool B_KM, int MB, int NB>
__device__ __forceinline__ void frag32_share(const floatx4_f (&acc)[MB][NB], int lane, int wave, float* sums) {
  constexpr int BM = 16 * MB, PITCH32 = 16 * NB + 4;
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
}

// The waves' shares of a tile. FOLD: every step of 16 K values sums into registers of its own that are added to the wave's total
// when the next one starts, chains of 16 and of K / (16 WAVES) instead of one of K / WAVES.
template <bool A_KM, bool B_KM, int MB, int NB, int WAVES, bool FOLD>
__device__ __forceinline__ void frag32_sums(const GemmArgs& g, int row0, int col0, float* sums) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  Frag32<A_KM, MB> fa;
  Frag32<B_KM, NB> fb;
  fa.init(static_cast<const float*>(g.a), g.lda, row0, g.M, lane);
  fb.init(static_cast<const float*>(g.b), g.ldb, col0, g.N, lane);
  floatx4_f acc[MB][NB], step_sum[MB][NB];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int n = 0; n < NB; ++n) acc[m][n] = step_sum[m][n] = floatx4_f{0.0f, 0.0f, 0.0f, 0.0f};
  auto fold = [&]() {
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int n = 0; n < NB; ++n) acc[m][n] += step_sum[m][n];
  };
  auto multiply = [&](const float (&a)[MB][4], const float (&b)[NB][4], int j) {
    if (FOLD && j == 0) fold();
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        if constexpr (FOLD) {
          const floatx4_f c = j == 0 ? floatx4_f{0.0f, 0.0f, 0.0f, 0.0f} : step_sum[m][n];
          step_sum[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[n][j], a[m][j], c, 0, 0, 0);
        } else {
          acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[n][j], a[m][j], acc[m][n], 0, 0, 0);
        }
      }
  };
  // Sets of fragments: one in use, two on their way. A quarter of a step's loads follows each quarter of its products: all
  // of them at once hold up the products behind them (loads between 64 and 128 products in a row: 97 and 133 us for 8192 x
  // 256 over 2048, 84 spread; four sets: 86). 2048 x 256 over 1024: 19.4 us with the loads of two steps waited for together, 15.9.
  constexpr int DEPTH = 3;
  const int whole = g.K / 16, steps = (g.K + 15) / 16;
  const int s_end = min(whole, steps * (wave + 1) / WAVES);
  int s0 = steps * wave / WAVES;
  float a[DEPTH][MB][4], b[DEPTH][NB][4];
  if (s0 < s_end) {
    // No load stands behind a branch: what is in flight is known at every wait, and a step waits for its own loads only.
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        fa.load(min(s0 + d, s_end - 1) * 16, j, a[d]);
        fb.load(min(s0 + d, s_end - 1) * 16, j, b[d]);
      }
#pragma unroll 1
    for (; s0 + DEPTH <= s_end; s0 += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        const int to = (d + DEPTH - 1) % DEPTH, k0 = min(s0 + d + DEPTH - 1, s_end - 1) * 16;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          multiply(a[d], b[d], j);
          fa.load(k0, j, a[to]);
          fb.load(k0, j, b[to]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
      if (s0 + d < s_end)
#pragma unroll
        for (int j = 0; j < 4; ++j) multiply(a[d], b[d], j);
  }
  if (whole < steps && wave == WAVES - 1) {
    fa.load_tail(whole * 16, g.K, lane, a[0]);
    fb.load_tail(whole * 16, g.K, lane, b[0]);
#pragma unroll
    for (int j = 0; j < 4; ++j) multiply(a[0], b[0], j);
  }
  if constexpr (FOLD) fold();
  frag32_share<A_KM, B_KM>(acc, lane, wave, sums);
}

// Output tile `index` (of one XCD's run each) of a product, or of a strided batch of them.
template <bool A_KM, bool B_KM, int MB, int NB, int WAVES, bool FOLD>
__device__ __forceinline__ void frag32_tile(GemmArgs& g, int index, float* sums) {
  constexpr int BM = 16 * MB, BN = 16 * NB, PITCH32 = BN + 4;  // the pad keeps 16-byte pieces and spreads banks
  const int total = g.tiles_m * g.tiles_n, r = tile_of_eighth(index, total * g.batches);
  const int product = r / total, id = r - product * total;
  // An XCD's run of tiles spans the output's shorter side.
  const int tile_m = g.tiles_m >= g.tiles_n ? id / g.tiles_n : id % g.tiles_m;
  const int tile_n = g.tiles_m >= g.tiles_n ? id % g.tiles_n : id / g.tiles_m;
  gemm_select_batch(g, product);
  const int row0 = tile_m * BM, col0 = tile_n * BN;
  frag32_sums<A_KM, B_KM, MB, NB, WAVES, FOLD>(g, row0, col0, sums);
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

template <bool A_KM, bool B_KM, int MB, int NB, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void gemm_frag32_kernel(GemmArgs g) {
  extern __shared__ __attribute__((aligned(16))) float sums[];  // [WAVES][16 MB][16 NB + 4]
  frag32_tile<A_KM, B_KM, MB, NB, WAVES, false>(g, blockIdx.x, sums);
}

// ---- a linear layer's two gradients in one launch ----
// A layer some hundred wide gives each of its two gradients less than a workgroup per compute unit or little more, and a call of the
// two a fixed part of some 3 us twice and two part-empty rounds: their tiles go out together. w: both operands k-major, usually the
// longer walk, so its workgroups come first; x: behind them, from workgroup `x_first` (a multiple of 8). x's sums are those of gemm_frag32_kernel's eight waves, whatever the tile: an
// input gradient's bits are the same from a call that asks for it alone. w's fold every 16 values (frag32_sums). Kernel time of a
// call of both: 1024 rows, 256 -> 256 10.6 -> 8.1 us, 256 -> 128 9.6 -> 6.9, 256 -> 12 9.4 -> 5.7 (9.2 and 7.8 for the first two inside a
// step, whose operands are further away); bound as gemm_frag32_kernel.
constexpr int PAIR_WAVES = 8;
template <int XM, int XN, int WM, int WN>
__global__ __launch_bounds__(PAIR_WAVES * 64) void gemm_frag32_pair_kernel(GemmArgs x, GemmArgs w, int x_first) {
  extern __shared__ __attribute__((aligned(16))) float sums[];
  const int index = blockIdx.x;
  if (index >= x_first) frag32_tile<false, true, XM, XN, PAIR_WAVES, false>(x, index - x_first, sums);
  else if (index < w.tiles_m * w.tiles_n) frag32_tile<true, true, WM, WN, PAIR_WAVES, true>(w, index, sums);
}

// The same where the input gradient alone would run on gemm_dma32_kernel with KG groups of waves: its sums, on eight waves. 1024 rows,
// 256 -> 704 17.2 -> 12.2 us, 704 -> 256 17.7 -> 13.8; 512 rows of 512 -> 512 12.7 -> 9.2.
template <int KG>
struct PairDma;  // waves of a group, blocks of a wave
template <> struct PairDma<1> { static constexpr int WGM = 4, WGN = 2, TM = 1, TN = 2; };
template <> struct PairDma<2> { static constexpr int WGM = 2, WGN = 2, TM = 2, TN = 1; };
template <> struct PairDma<4> { static constexpr int WGM = 1, WGN = 2, TM = 2, TN = 1; };
template <int KG>
__global__ __launch_bounds__(PAIR_WAVES * 64) void gemm_dma32_pair_kernel(GemmArgs x, GemmArgs w, int x_first) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  using D = PairDma<KG>;
  const int index = blockIdx.x;
  if (index >= x_first) dma32_tile<false, true, D::WGM, D::WGN, D::TM, D::TN, 2, KG, false, 0>(x, index - x_first, smem);
  else if (index < w.tiles_m * w.tiles_n) frag32_tile<true, true, 2, 2, PAIR_WAVES, true>(w, index, reinterpret_cast<float*>(smem));
}

// ---- several products in one launch ----
// Five shapes of a model's matrices are five chains of fifteen Newton-Schulz products, each a launch of 4 to 256 workgroups that takes
// 3 to 13 us and leaves most of the chip idle: the k-th products of all chains go out together. 32 x 32 tiles whose four waves share
// K. Four blocks of d = 256 (32 matrices): 33, 26 and 40 us for the first, second and third products of an iteration, 20, 13 and 28
// in one launch each; bound by the waits of short walks over K (a third of the f32 matrix rate). 64 x 32 tiles took 22, 16 and 30,
// steps of 32 K values with all of a step's loads together 28, 16 and 33. The third products, whose outputs are the matrices, go on
// gemm_dma32.hip's 64 x 64 tiles instead where those make half a workgroup per compute unit (28 -> 23 us: half the operand bytes a
// product; a step of the 32 matrices 337 -> 305 us, of 64 556 -> 502, 16 matrices 240 -> 231).
// `symmetric`: the output equals its transpose (X X^T, A A and their sums with a symmetric tensor): tiles below the diagonal are
// written from those above it, the same sums in the same order.
constexpr int GROUP_WAVES = 4, GROUP_TILE = 32, GROUP_DMA = 4, GROUP_DMA_TILE = 64;
constexpr int GROUP_LDS = 2 * 2 * GROUP_DMA_TILE * 128;  // two stages of two operands
static_assert(GROUP_LDS >= GROUP_WAVES * GROUP_TILE * (GROUP_TILE + 4) * 4, "the waves' sums fit");
struct FragProduct {
  const float *a, *b, *aux;
  float* c;
  long lda, ldb, ldc, batch;  // batch: BYTES between the products of a strided batch, in every operand
  int M, N, K, tiles_m, tiles_n, batches, layout, c_vec;  // layout: 2 A k-major + B k-major; GROUP_DMA: 64 x 64 tiles
};
struct FragGroup {
  FragProduct product[FRAG32_GROUP];
  int first[FRAG32_GROUP];  // a product's first workgroup, a multiple of 8
  int symmetric;
  float s1, s2;
  OmxFaultWord* fault;
  unsigned long long tag;
};
__global__ __launch_bounds__(GROUP_WAVES * 64) void gemm_frag32_group_kernel(FragGroup q) {
  __shared__ __attribute__((aligned(1024))) char smem[GROUP_LDS];
  float* const sums = reinterpret_cast<float*>(smem);  // [GROUP_WAVES][GROUP_TILE][GROUP_TILE + 4]
  constexpr int PITCH32 = GROUP_TILE + 4;
  int which = 0;  // (all of `first` in one load)
#pragma unroll
  for (int i = 1; i < FRAG32_GROUP; ++i) which += static_cast<int>(blockIdx.x) >= q.first[i];
  const FragProduct& p = q.product[which];
  const int total = p.tiles_m * p.tiles_n, index = blockIdx.x - q.first[which];
  if (index >= total * p.batches) return;
  GemmArgs g;
  g.a = p.a;
  g.b = p.b;
  g.c = p.c;
  g.aux_in = reinterpret_cast<const unsigned short*>(p.aux);
  g.aux_out = nullptr;
  g.lda = p.lda; g.ldb = p.ldb; g.ldc = p.ldc;
  g.M = p.M; g.N = p.N; g.K = g.k_rows = p.K;
  g.tiles_m = p.tiles_m; g.tiles_n = p.tiles_n;
  g.batches = p.batches;
  g.batch_a = g.batch_b = g.batch_c = p.batch;
  g.c_bf16 = 0;
  g.accumulate = p.aux ? 2 : 0;
  g.c_vec = p.c_vec;
  g.splits = 1;
  g.epi_s1 = q.s1; g.epi_s2 = q.s2;
  g.fault = q.fault;
  g.tag = g.act_tag = q.tag;
  if (p.layout == GROUP_DMA) {  // (uniform)
    dma32_tile<false, true, 2, 2, 2, 2, 2, 1, false, 0>(g, index, smem);
    return;
  }
  const int r = tile_of_eighth(index, total * p.batches), product = r / total, id = r - product * total;
  const int tile_m = id / p.tiles_n, tile_n = id - tile_m * p.tiles_n;
  if (q.symmetric && tile_m > tile_n) return;
  gemm_select_batch(g, product);
  const int row0 = tile_m * GROUP_TILE, col0 = tile_n * GROUP_TILE;
  switch (p.layout) {  // (uniform)
    case 0: frag32_sums<false, false, 2, 2, GROUP_WAVES, true>(g, row0, col0, sums); break;
    case 1: frag32_sums<false, true, 2, 2, GROUP_WAVES, true>(g, row0, col0, sums); break;
    case 2: frag32_sums<true, false, 2, 2, GROUP_WAVES, true>(g, row0, col0, sums); break;
    default: frag32_sums<true, true, 2, 2, GROUP_WAVES, true>(g, row0, col0, sums);
  }
  __syncthreads();
  // 256 threads, 256 pieces of four columns.
  const int row = threadIdx.x / (GROUP_TILE / 4), col = threadIdx.x % (GROUP_TILE / 4) * 4;
  auto meet = [&](int at, int step, float (&t)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] = sums[at + e * step];
#pragma unroll
    for (int w = 1; w < GROUP_WAVES; ++w)
#pragma unroll
      for (int e = 0; e < 4; ++e) t[e] += sums[w * (GROUP_TILE * PITCH32) + at + e * step];
  };
  bool bad = false;
  float t[4];
  meet(row * PITCH32 + col, 1, t);
  if (row0 + row < g.M && col0 + col < g.N) bad |= gemm_store4(g, 0, row0 + row, col0 + col, t[0], t[1], t[2], t[3]);
  if (q.symmetric && tile_m != tile_n) {
    meet(col * PITCH32 + row, PITCH32, t);
    if (col0 + row < g.M && row0 + col < g.N) bad |= gemm_store4(g, 0, col0 + row, row0 + col, t[0], t[1], t[2], t[3]);
  }
  if (bad) dev_raise_fault(q.fault, q.tag);
}

struct FragTile {
  int mb, nb, waves;
  // us: a call's first round of workgroups (fixed and per 16 columns of K), and each further round; both operands k-major.
  double first, step, more, more_step, km_first, km_step, km_more, km_more_step;
};
constexpr FragTile FRAG_TILES[] = {{1, 1, 8, 3.10, 0.0398, 0.12, 0.0460, 2.80, 0.0529, 0.54, 0.0352},
                                   {1, 2, 8, 3.17, 0.0613, 0.13, 0.0705, 3.16, 0.0544, 0.56, 0.0504},
                                   {2, 2, 8, 3.21, 0.0939, 0.44, 0.1021, 3.53, 0.0800, 0.76, 0.0806},
                                   {4, 2, 8, 3.22, 0.1761, 0.88, 0.1819, 3.55, 0.1496, 1.22, 0.1649},
                                   {4, 4, 4, 4.71, 0.2386, 1.72, 0.3680, 4.62, 0.2546, 1.66, 0.3086}};

// Whether an operand's pieces are whole and aligned for `blocks` blocks of 16 rows.
bool frag_fits(bool km, const void* p, long ld, int rows, int blocks, long batch_bytes) {
  const long piece = km ? blocks : 4;
  return ld % piece == 0 && ld <= 1l << 22 /* a tile's rows stay within 32 bits of bytes */ && (reinterpret_cast<uintptr_t>(p) & (piece * 4 - 1)) == 0 && batch_bytes % (piece * 4) == 0 &&
         (!km || (rows % blocks == 0 && rows >= blocks));
}

template <bool A_KM, bool B_KM, int T>
int32_t launch_frag(omx_ctx* ctx, const GemmArgs& g) {
  constexpr FragTile t = FRAG_TILES[T];
  constexpr int smem = t.waves * 16 * t.mb * (16 * t.nb + 4) * 4;
  auto kernel = &gemm_frag32_kernel<A_KM, B_KM, t.mb, t.nb, t.waves>;
  if constexpr (smem > 64 * 1024)
    OMX_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
  GemmArgs tiled = g;
  tiled.tiles_m = (g.M + 16 * t.mb - 1) / (16 * t.mb);
  tiled.tiles_n = (g.N + 16 * t.nb - 1) / (16 * t.nb);
  omx_launch_timed(ctx, kernel, dim3(static_cast<unsigned>(tiled.tiles_m) * tiled.tiles_n * g.batches), dim3(t.waves * 64), smem,
                   ctx->timing_start, ctx->timing_stop, tiled);
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

double omx_gemm_frag32_us(omx_ctx* ctx, const GemmArgs& g, bool a_km, bool b_km, int tile) {
  const FragTile& f = FRAG_TILES[tile];
  if (!frag_fits(a_km, g.a, g.lda, g.M, f.mb, g.batch_a) || !frag_fits(b_km, g.b, g.ldb, g.N, f.nb, g.batch_b)) return -1.0;
  const long units = ctx->cu_count > 0 ? ctx->cu_count : 256;
  const long m = (g.M + 16 * f.mb - 1) / (16 * f.mb), n = (g.N + 16 * f.nb - 1) / (16 * f.nb), groups = m * n * g.batches;
  if (groups > 0x7fffffffl) return -1.0;
  const double more = static_cast<double>((groups + units - 1) / units - 1), steps = (g.K + 15) / 16;
  return a_km && b_km ? f.km_first + steps * f.km_step + more * (f.km_more + steps * f.km_more_step)
                      : f.first + steps * f.step + more * (f.more + steps * f.more_step);
}

int32_t omx_gemm_frag32_launch(omx_ctx* ctx, const GemmArgs& g, bool a_km, bool b_km, int tile) {
  if (!a_km && !b_km) return launch_frag_tile<false, false>(ctx, g, tile);
  if (!a_km) return launch_frag_tile<false, true>(ctx, g, tile);
  if (!b_km) return launch_frag_tile<true, false>(ctx, g, tile);
  return launch_frag_tile<true, true>(ctx, g, tile);
}

namespace {
template <int XM, int XN, int WM, int WN>
int32_t launch_pair(omx_ctx* ctx, GemmArgs x, GemmArgs w) {
  constexpr int smem = PAIR_WAVES * 64 * std::max(XM * (16 * XN + 4), WM * (16 * WN + 4));
  auto kernel = &gemm_frag32_pair_kernel<XM, XN, WM, WN>;
  if constexpr (smem > 64 * 1024)
    OMX_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
  x.tiles_m = (x.M + 16 * XM - 1) / (16 * XM);
  x.tiles_n = (x.N + 16 * XN - 1) / (16 * XN);
  w.tiles_m = (w.M + 16 * WM - 1) / (16 * WM);
  w.tiles_n = (w.N + 16 * WN - 1) / (16 * WN);
  const int x_first = (w.tiles_m * w.tiles_n + 7) & ~7;
  omx_launch_timed(ctx, kernel, dim3(static_cast<unsigned>(x_first + x.tiles_m * x.tiles_n)), dim3(PAIR_WAVES * 64), smem, ctx->timing_start,
                   ctx->timing_stop, x, w, x_first);
  OMX_LAUNCH_CHECK(ctx, "gemm_frag32_pair_kernel");
  return OMX_OK;
}
template <int KG>
int32_t launch_dma_pair(omx_ctx* ctx, GemmArgs x, GemmArgs w) {
  using D = PairDma<KG>;
  constexpr int BM = D::WGM * D::TM * 16, BN = D::WGN * D::TN * 16;
  constexpr int smem = std::max(2 * KG * (BM + BN) * 128, PAIR_WAVES * 32 * 36 * 4);
  static_assert(smem <= 64 * 1024 && D::WGM * D::WGN * KG == PAIR_WAVES, "what a launch may ask for");
  x.tiles_m = (x.M + BM - 1) / BM;
  x.tiles_n = (x.N + BN - 1) / BN;
  w.tiles_m = (w.M + 31) / 32;
  w.tiles_n = (w.N + 31) / 32;
  const int x_first = (w.tiles_m * w.tiles_n + 7) & ~7;
  omx_launch_timed(ctx, gemm_dma32_pair_kernel<KG>, dim3(static_cast<unsigned>(x_first + x.tiles_m * x.tiles_n)), dim3(PAIR_WAVES * 64), smem,
                   ctx->timing_start, ctx->timing_stop, x, w, x_first);
  OMX_LAUNCH_CHECK(ctx, "gemm_dma32_pair_kernel");
  return OMX_OK;
}
// us: a fixed part, then what the tiles take side by side over the compute units and the longest walk of one, squares added. Fitted
// over 326 layers of 24 .. 6000 rows and 12 .. 1600 columns, each on all four pairs (rms 7 %); the tiles it chooses are 1.4 % behind
// the best of the four on average (32 x 32 for both 17 %).
constexpr double PAIR_US = 2.83;
struct PairTile {
  int xm, xn, wm, wn;
  double x_step, x_tile, w_step, w_tile;      // us per 16 columns of K and per tile, on one unit
  double x_walk, w_walk, x_alone, w_alone;  // per 16 columns and per tile, alone
};
constexpr PairTile PAIR_TILES[FRAG32_PAIRS] = {{1, 2, 2, 2, 0.0, 0.648, 0.1818, 1.805, 0.0544, 0.0825, 0.97, 1.54},
                                               {2, 2, 1, 1, 0.2329, 0.957, 0.0, 1.152, 0.0926, 0.0428, 1.44, 0.92},
                                               {2, 2, 2, 2, 0.0, 0.650, 0.1671, 1.895, 0.0869, 0.0842, 1.38, 1.48},
                                               {4, 2, 1, 2, 0.4083, 1.952, 0.0, 2.645, 0.1753, 0.0539, 1.70, 1.04}};
template <int T>
int32_t launch_pair_tile(omx_ctx* ctx, const GemmArgs& x, const GemmArgs& w) {
  constexpr PairTile t = PAIR_TILES[T];
  return launch_pair<t.xm, t.xn, t.wm, t.wn>(ctx, x, w);
}
}  // namespace

double omx_gemm_frag32_pair_us(omx_ctx* ctx, const GemmArgs& x, const GemmArgs& w, int tile) {
  const PairTile& t = PAIR_TILES[tile];
  if (!frag_fits(false, x.a, x.lda, x.M, t.xm, 0) || !frag_fits(true, x.b, x.ldb, x.N, t.xn, 0) || !frag_fits(true, w.a, w.lda, w.M, t.wm, 0) ||
      !frag_fits(true, w.b, w.ldb, w.N, t.wn, 0))
    return -1.0;
  auto tiles = [](const GemmArgs& g, int m, int n) { return ((g.M + 16l * m - 1) / (16 * m)) * ((g.N + 16l * n - 1) / (16 * n)); };
  const long x_tiles = tiles(x, t.xm, t.xn), w_tiles = tiles(w, t.wm, t.wn);
  if (x_tiles > 1l << 20 || w_tiles > 1l << 20) return -1.0;
  const double units = ctx->cu_count > 0 ? ctx->cu_count : 256, x_steps = (x.K + 15l) / 16, w_steps = (w.K + 15l) / 16;
  const double all = (x_tiles * (x_steps * t.x_step + t.x_tile) + w_tiles * (w_steps * t.w_step + t.w_tile)) / units;
  const double walk = std::max(x_steps * t.x_walk + t.x_alone, w_steps * t.w_walk + t.w_alone);
  return PAIR_US + sqrt(all * all + walk * walk);
}

int32_t omx_gemm_frag32_pair(omx_ctx* ctx, const GemmArgs& x, const GemmArgs& w, int tile) {
  switch (tile) {
    case 0: return launch_pair_tile<0>(ctx, x, w);
    case 1: return launch_pair_tile<1>(ctx, x, w);
    case 2: return launch_pair_tile<2>(ctx, x, w);
    default: return launch_pair_tile<3>(ctx, x, w);
  }
}
int32_t omx_gemm_dma32_pair(omx_ctx* ctx, const GemmArgs& x, const GemmArgs& w, int dma32) {
  if (dma32 < 2) return launch_dma_pair<1>(ctx, x, w);
  return dma32 == 2 ? launch_dma_pair<2>(ctx, x, w) : launch_dma_pair<4>(ctx, x, w);
}

// (The operands are the library's own scratch: what does not fit is a mistake of the caller's.)
static bool group_fits(const OmxGemmProduct& p) {
  const bool a_km = p.a_cs != 1, b_km = p.b_rs != 1;
  const long lda = static_cast<long>(a_km ? p.a_cs : p.a_rs), ldb = static_cast<long>(b_km ? p.b_rs : p.b_cs);
  const uint64_t most = 0x7fffffff, tiles = (p.m + GROUP_TILE - 1) / GROUP_TILE * ((p.n + GROUP_TILE - 1) / GROUP_TILE);
  return p.m <= most && p.n <= most && p.k <= most && p.batches > 0 && tiles <= most / FRAG32_GROUP / p.batches - 8 && p.stride % 4 == 0 &&
         (!a_km || p.a_rs == 1) && (!b_km || p.b_cs == 1) &&
         frag_fits(a_km, p.a, lda, static_cast<int>(p.m), 2, 0) && frag_fits(b_km, p.b, ldb, static_cast<int>(p.n), 2, 0);
}

// A k-contiguous, B k-major, whole steps of 32 and aligned pieces. From K = 192 on, where the 64 x 64 tile's sums (32 values a step)
// lose nothing against a launch for each shape: 2-norm error of 40 updates, together / apart, 128 x 128 7.2e-7 / 6.7e-7, 128 x 256
// 7.5e-7 / 7.3e-7, 160 x 160 7.0e-7 / 7.0e-7, 192 x 192 6.9e-7 / 7.1e-7, 256 x 256 6.7e-7 / 7.2e-7 (on 32 x 32 tiles 6.4e-7, 6.9e-7,
// 6.3e-7, 6.2e-7 and 6.1e-7).
constexpr uint64_t GROUP_DMA_K = 192;
static bool group_fits_dma(const OmxGemmProduct& p) {
  return p.k >= GROUP_DMA_K && p.a_cs == 1 && p.b_cs == 1 && p.b_rs != 1 && p.k % 32 == 0 && p.n % 4 == 0 && p.a_rs % 4 == 0 && p.b_rs % 4 == 0 && p.a_rs <= 1u << 22 &&
         p.b_rs <= 1u << 22 && ((reinterpret_cast<uintptr_t>(p.a) | reinterpret_cast<uintptr_t>(p.b)) & 15u) == 0;
}

int32_t omx_gemm_frag32_group(omx_ctx* ctx, const OmxGemmProduct* products, int count, bool symmetric, float s1, float s2, unsigned long long tag) {
  FragGroup q;
  q.symmetric = symmetric;
  q.s1 = s1;
  q.s2 = s2;
  q.fault = ctx->fault;
  q.tag = tag;
  uint64_t large_tiles = 0;
  double flops = 0.0;
  for (int i = 0; i < count; ++i) {
    const OmxGemmProduct& p = products[i];
    flops += 2.0 * static_cast<double>(p.m) * static_cast<double>(p.n) * static_cast<double>(p.k) * static_cast<double>(p.batches);
    if (!symmetric && group_fits_dma(p))
      large_tiles += ((p.m + GROUP_DMA_TILE - 1) / GROUP_DMA_TILE) * ((p.n + GROUP_DMA_TILE - 1) / GROUP_DMA_TILE) * p.batches;
  }
  const bool large = 2 * large_tiles >= static_cast<uint64_t>(ctx->cu_count > 0 ? ctx->cu_count : 256);
  int at = 0;
  for (int i = 0; i < count; ++i) {
    const OmxGemmProduct& p = products[i];
    if (!group_fits(p)) return omx_fail(ctx, OMX_UNSUPPORTED, "%s: products in one launch", omx_fault_name(tag & 0x7f));
    FragProduct& f = q.product[i];
    const bool a_km = p.a_cs != 1, b_km = p.b_rs != 1;
    f.a = p.a; f.b = p.b; f.aux = p.aux; f.c = p.c;
    f.lda = static_cast<long>(a_km ? p.a_cs : p.a_rs);
    f.ldb = static_cast<long>(b_km ? p.b_rs : p.b_cs);
    f.ldc = static_cast<long>(p.ldc);
    f.batch = static_cast<long>(p.stride) * 4;
    f.M = static_cast<int>(p.m); f.N = static_cast<int>(p.n); f.K = static_cast<int>(p.k);
    f.batches = static_cast<int>(p.batches);
    f.layout = large && !a_km && b_km && group_fits_dma(p) ? GROUP_DMA : 2 * a_km + b_km;
    const int tile = f.layout == GROUP_DMA ? GROUP_DMA_TILE : GROUP_TILE;
    f.tiles_m = (f.M + tile - 1) / tile;
    f.tiles_n = (f.N + tile - 1) / tile;
    f.c_vec = (reinterpret_cast<uintptr_t>(p.c) & 15u) == 0 && p.ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(p.aux) & 15u) == 0;
    q.first[i] = at;
    at += (f.tiles_m * f.tiles_n * f.batches + 7) & ~7;
  }
  for (int i = count; i < FRAG32_GROUP; ++i) {
    q.first[i] = 0x7fffffff;
    q.product[i] = FragProduct{};
  }
  omx_ctx::TimedLaunch timed{};
  int32_t rc = omx_timing_begin(ctx, flops, &timed);
  if (rc != OMX_OK) return rc;
  rc = [&]() -> int32_t {
    omx_launch_timed(ctx, gemm_frag32_group_kernel, dim3(static_cast<unsigned>(at)), dim3(GROUP_WAVES * 64), 0, ctx->timing_start, ctx->timing_stop, q);
    OMX_LAUNCH_CHECK(ctx, "gemm_frag32_group_kernel");
    return OMX_OK;
  }();
  omx_timing_end(ctx, rc == OMX_OK, timed);
  return rc;
}
