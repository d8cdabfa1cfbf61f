// The bf16 GEMM with one wave per SIMD: a 256 x 256 output tile per workgroup, one workgroup per
// compute unit, four waves of 128 x 128 each (16 accumulator blocks of 32 x 32: 256 of the wave's
// 512 registers); with TN = 3 the tile is 256 x 192 and a wave's part 128 x 96 (768 output columns
// are four such tiles: 16384 rows then make 256 tiles, one per compute unit, where 256 x 256 tiles
// make 192). A wave interleaves its own LDS reads and global -> LDS loads between its own
// matrix products, in an order fixed in the source: per product a wave reads two thirds of the
// fragment bytes that eight waves of 128 x 64 read, and no other wave on the SIMD takes issue
// slots from the products.
//
//   K steps of 64 columns, two LDS stages per operand (A0 A1 B0 B1, 32 KiB each). A step is 64
//   products per wave in two halves of 32, and a stage is refilled in two parts, each as soon as
//   every wave has read it:
//     A k-contiguous (a load covers 8 rows x 64 columns): half 0 is the wave's row blocks 0-1 over
//       the step's four K slabs against all of B, half 1 its row blocks 2-3 against the same B
//       fragments, which stay in registers. Part 0 = B and the A rows of half 0 (12 loads per
//       wave), part 1 = the A rows of half 1 (4 loads).
//     A and B k-major (a load covers 2 K rows x 256 rows): half h is K slabs 2h, 2h + 1 of every
//       block; part h = K rows 32h .. 32h + 31 of both operands (8 loads per wave).
//   During half 1 of step j the wave reads part 0 of step j + 1, during half 0 part 1 of step j.
//   Two barriers per step: B0, after the first 8 products of half 0, says that every wave has read
//   part 0 of this step, and publishes part 1; part 0 of step j + 2 is loaded behind it. B1,
//   between the halves, says that part 1 has been read and publishes part 0 of step j + 1; part 1
//   of step j + 2 is loaded behind it. Every load has more than a step to land.
//   The K loop holds one copy of the step per stage and nothing else: the last steps skip their
//   loads by scalar branches, and the step count is even (K a multiple of 128, an even number of
//   steps per split). With further copies of the step, or a branch around the second one, the
//   compiler permutes the 256 accumulator registers between the copies through scratch memory.
#pragma once
#include "gemm_tiles.h"

namespace {

constexpr int W4_BM = 256, W4_BK = 64;  // the tile is 256 rows by 64 TN columns (TN = 4, or 3: 192 columns)
constexpr int W4_OPERAND = W4_BM * W4_BK * 2;  // one stage of one operand
constexpr int W4_SMEM = 4 * W4_OPERAND;
constexpr int W4_B0 = 2 * W4_OPERAND;  // LDS byte offset of B's first stage

// The chunk swizzle of a k-major tile row (kr) of ROWS columns: 16-byte chunks moved by multiples of 64 bytes so that
// the four K rows a transposing read touches per clock fall into different banks (rows of 512 bytes all start in
// bank 0: four shifts; rows of 384 bytes alternate between banks 0 and 32: one shift for every second pair).
template <int ROWS>
__device__ __forceinline__ int w4_km_swizzle(int kr) {
  return ROWS == 256 ? (kr & 3) * 4 : ((kr >> 1) & 1) * 4;
}

// Loads of one operand (see StepBase for the base address and the end of the K rows).
template <bool KM, int ROWS, bool TAIL>
struct W4Loads {
  static constexpr int N = ROWS / 32;  // ROWS / 8 loads of 1 KiB per step, four waves
  unsigned off[N];
  StepBase<KM, TAIL> base;
  // Two row ranges, `half` apart, in one tile of 256: 64 rows of the first and the same of the second in turn. row0: of the first.
  __device__ __forceinline__ void init_pairs(const unsigned short* __restrict__ p, long ld, int row0, int half, int k0, int k_rows, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = (wave + 4 * i) * 8 + (lane >> 3), kc = (lane & 7) ^ ((r >> 1) & 7);
      const int unit = min(row0 + (r >> 7) * 64 + (r & 63), half - 1);
      off[i] = static_cast<unsigned>(unit - row0 + (r >> 6 & 1) * half) * static_cast<unsigned>(ld * 2) + kc * 16;
    }
    base.init(p, ld, row0, k0, k_rows, W4_BK);
  }
  __device__ __forceinline__ void init(const unsigned short* __restrict__ p, long ld, int row0, int rows, int k0,
                                       int k_rows, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int q = wave + 4 * i;
      if constexpr (!KM) {
        const int r = q * 8 + (lane >> 3);
        const int kc = (lane & 7) ^ ((r >> 1) & 7);
        int gr = row0 + r;
        gr = gr < rows ? gr : rows - 1;
        off[i] = static_cast<unsigned>(gr - row0) * static_cast<unsigned>(ld * 2) + kc * 16;
      } else {
        constexpr int CPR = ROWS / 8;  // 16-byte chunks per K row
        const int idx = q * 64 + lane;
        const int kr = idx / CPR, slot = idx % CPR;
        const int mc = slot ^ w4_km_swizzle<ROWS>(kr);
        int gm = mc * 8;
        gm = row0 + gm < rows ? gm : 0;
        off[i] = static_cast<unsigned>(kr) * static_cast<unsigned>(ld * 2) + gm * 2;
      }
    }
    base.init(p, ld, row0, k0, k_rows, W4_BK);
  }
  // Load I of this wave into LDS byte `lds_wave` + LDS_IMM.
  template <int I, int LDS_IMM>
  __device__ __forceinline__ void issue(unsigned lds_wave) const {
    base.template load<LDS_IMM>(off[I], lds_wave);
  }
};

// Fragment addresses of one operand tile of ROWS rows: four registers holding LDS byte addresses in stage 0; the
// block, the K slab and the stage are immediates of the read. `tile` is the tile's LDS address, `row_base` the first
// of the wave's rows in it.
template <bool KM, int ROWS>
struct W4Frags {
  unsigned b[4];
  __device__ __forceinline__ void init(unsigned tile, int row_base, int lane) {
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      if constexpr (!KM) {
        // [row][8 chunks of 16 bytes], chunk c of row r in slot c ^ ((r >> 1) & 7); x is the K slab.
        const int r = row_base + (lane & 31);
        const int kc = x * 2 + (lane >> 5);
        b[x] = tile + r * (W4_BK * 2) + ((kc ^ ((r >> 1) & 7)) << 4);
      } else {
        // [K row][ROWS / 8 chunks]; x is the 32-column block; the first of the two transposing reads.
        const int s16 = lane & 15, half = (lane >> 4) & 1, g = lane >> 5;
        const int kr = g * 8 + (s16 >> 2);
        const int col = row_base + x * 32 + half * 16 + (s16 & 3) * 4;
        b[x] = tile + kr * (ROWS * 2) + (((col >> 3) ^ w4_km_swizzle<ROWS>(kr)) << 4) + (col & 7) * 2;
      }
      // Held as it is: re-derived from its parts, a read would pay an addition for what the
      // instruction's offset field carries for nothing.
      asm volatile("" : "+v"(b[x]));
    }
  }
  template <int T, int KK, int STAGE>
  __device__ __forceinline__ u32x4 read() const {
    if constexpr (!KM) {
      typedef const u32x4 __attribute__((address_space(3))) * lds_ptr;
      return *reinterpret_cast<lds_ptr>(static_cast<uintptr_t>(b[KK] + (T * 32 * W4_BK * 2 + STAGE * W4_OPERAND)));
    } else {
      typedef short4v __attribute__((address_space(3))) * lds_ptr;
      const unsigned p = b[T] + (KK * 16 * ROWS * 2 + STAGE * W4_OPERAND);
      short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_ptr>(static_cast<uintptr_t>(p)));
      short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_ptr>(static_cast<uintptr_t>(p + 4 * ROWS * 2)));
      u32x2 x = __builtin_bit_cast(u32x2, lo), y = __builtin_bit_cast(u32x2, hi);
      return u32x4{x.x, x.y, y.x, y.y};
    }
  }
};

// LR: with a low-rank term.
// STORE: OMX_EPI_SWIGLU, OMX_EPI_ROPE and OMX_EPI_SWIGLU_BWD have a store pass of their own.
// PAIR: B's rows are gates and, N / 2 further, ups. A wave's 128 columns are 64 units' gates and ups, which meet in its store pass: C
// as it would be, in f32, and silu(gate) up beside it in bf16 (OMX_EPI_SWIGLU), where a pass of its own read C again. us, product and pass / so,
// inside a step: 8192 rows over 2048 -> 2 x 8192: 490 + 112 / 545; 16384 over 768 -> 2 x 2048: 130 + 59 / 154.
// ROPE: heads of 64 or 128 columns are turned in the store pass (OMX_EPI_ROPE), where the product went out in f32 and a pass read it: both halves of a
// head lie in a wave's 128 columns. us, product and pass / so, inside a step: 8192 rows over
// 2048 -> 48 heads of 128, two thirds of them turned: 213 + 51 / 204 (tables read row by row, after the staging: 241).
// DPAIR: the product is the gradient of silu(gate) up, and gates and ups (f32, 8 N bytes a row) are read, their gradients written, in the
// store pass (OMX_EPI_SWIGLU_BWD), where the product went out and a pass read it again. us, product and pass / so,
// inside a step: 8192 rows over 2048 -> 8192: 225 + 147 / 359; 16384 over 768 -> 2048: 60 + 72 / 116. The 4 N bytes a row that no longer go
// out and back are what it gives; the rest moves as before, and all workgroups reach their store passes together, so beside no product.
template <bool A_KM, bool B_KM, int TN, bool TAIL, bool LR = false, int STORE = OMX_EPI_NONE>
__global__ __launch_bounds__(256, 1) void gemm_w4_kernel(GemmArgs g) {
  static_assert(!A_KM || B_KM, "a k-major A goes with a k-major B");
  static_assert(TN == 4 || TN == 3, "256 x 256 or 256 x 192 tiles");
  constexpr bool PAIR = STORE == OMX_EPI_SWIGLU, ROPE = STORE == OMX_EPI_ROPE, DPAIR = STORE == OMX_EPI_SWIGLU_BWD;
  static_assert(!(PAIR || ROPE) || (!A_KM && !B_KM && TN == 4 && !TAIL && LR == ROPE), "one form of each");
  static_assert(!DPAIR || (!A_KM && B_KM && TN == 4 && !TAIL && !LR), "an input gradient");
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int TM = 4, NW = 4, W4_BN = TN * 64;
  // Tile order: as gemm_dma_kernel.
  const int total = g.tiles_m * g.tiles_n;
  int split = 0, id = blockIdx.x, product = blockIdx.y;
  if (g.batches > 1 && g.splits == 1 && ((total * g.batches) & 7) == 0) {
    const int linear = blockIdx.y * total + blockIdx.x;
    const int r = (linear & 7) * ((total * g.batches) >> 3) + (linear >> 3);
    product = r / total;
    id = r - product * total;
  } else if (g.splits > 1) {
    split = blockIdx.x % g.splits;
    id = blockIdx.x / g.splits;
  } else if (total % 8 == 0) {
    id = (id & 7) * (total >> 3) + (id >> 3);
  }
  const int band = 4;
  const int tiles_per_band = band * g.tiles_n;
  const int band_id = id / tiles_per_band;
  const int first_m = band_id * band;
  const int band_rows = min(band, g.tiles_m - first_m);
  const int in_band = id - band_id * tiles_per_band;
  const int tile_m = first_m + in_band % band_rows;
  const int tile_n = in_band / band_rows;
  // (the divisions above run on the vector unit: back to scalars, which the loads' bases need)
  const int m0 = __builtin_amdgcn_readfirstlane(tile_m * W4_BM), n0 = __builtin_amdgcn_readfirstlane(tile_n * W4_BN);
  product = __builtin_amdgcn_readfirstlane(product);
  split = __builtin_amdgcn_readfirstlane(split);
  gemm_select_batch(g, product);
  const unsigned short* __restrict__ A = static_cast<const unsigned short*>(g.a);
  const unsigned short* __restrict__ B = static_cast<const unsigned short*>(g.b);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;  // the wave's 128 rows and 32 TN columns of the tile
  const int l32 = lane & 31, lg = lane >> 5;

  floatx16 acc[TM][TN];
  // Cleared once the first loads are on their way (256 register writes).
  auto clear_acc = [&]() {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
    __builtin_amdgcn_sched_barrier(0);
  };

  const int ks_begin = split * g.ksteps_per_split;
  const int ks_end = min(g.K / W4_BK, ks_begin + g.ksteps_per_split);
  const int steps = ks_end - ks_begin;
  W4Loads<A_KM, W4_BM, TAIL> la;
  W4Loads<B_KM, W4_BN, TAIL> lb;
  la.init(A, g.lda, m0, g.M, ks_begin * W4_BK, g.k_rows, wave, lane);
  if constexpr (PAIR) lb.init_pairs(B, g.ldb, n0 / 2, g.N / 2, ks_begin * W4_BK, g.k_rows, wave, lane);
  else lb.init(B, g.ldb, n0, g.N, ks_begin * W4_BK, g.k_rows, wave, lane);
  const unsigned lds_wave =
      __builtin_amdgcn_readfirstlane(static_cast<unsigned>(reinterpret_cast<uintptr_t>(smem))) + wave * 1024;
  // Waits until at most YES (if `which`) or NO of this wave's loads, the most recently issued, are in flight.
  auto wait_loads = [&](bool which, auto yes_count, auto no_count) {
    if (which) __builtin_amdgcn_s_waitcnt(vmcnt_only(decltype(yes_count)::value));
    else __builtin_amdgcn_s_waitcnt(vmcnt_only(decltype(no_count)::value));
  };
  auto publish = [&](bool which, auto yes_count, auto no_count) {
    __builtin_amdgcn_sched_barrier(0);
    wait_loads(which, yes_count, no_count);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt == 0: this wave's fragment reads have returned
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  // The products are taken with the operands exchanged: a lane then holds, for ONE output row (block
  // row l32), four consecutive columns per register quad (8 (v / 4) + 4 lg + v % 4), which the
  // store pass packs and stages 8 or 16 bytes at a time.
  auto product_of = [&](floatx16& c, const u32x4& a, const u32x4& b) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, b), __builtin_bit_cast(bf16x8, a), c, 0, 0, 0);
  };
  const unsigned lds0 = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(reinterpret_cast<uintptr_t>(smem)));
  const std::integral_constant<int, 0> S0{};
  const std::integral_constant<int, 1> S1{};
  if constexpr (!A_KM) {
    W4Frags<false, W4_BM> ra;
    W4Frags<B_KM, W4_BN> rb;
    ra.init(lds0, wm * 128, lane);
    rb.init(lds0 + W4_B0, wn * TN * 32, lane);

    // Part 0 of a stage: all of B (2 TN loads per wave) and A's loads 0, 1, 4, 5 (rows 0-63 and 128-191 of the
    // tile); part 1: A's loads 2, 3, 6, 7. `n` counts the part's loads.
    constexpr int NB = 2 * TN, NP0 = NB + 4, NSTEP = NP0 + 4;
    constexpr int SL = 2 * TN, HL = 4 * SL;  // products per K slab of a half, per half
    typedef std::integral_constant<int, 0> C0;
    typedef std::integral_constant<int, 4> C4;
    typedef std::integral_constant<int, NSTEP> CSTEP;
    typedef std::integral_constant<int, 4 + NP0> C4P0;
    auto issue_p0 = [&](auto stage_index, auto n_index) {
      constexpr int stage = decltype(stage_index)::value, n = decltype(n_index)::value;
      if constexpr (n < NB) {
        lb.template issue<n, W4_B0 + stage * W4_OPERAND + NW * n * 1024>(lds_wave);
      } else {
        constexpr int i = n == NB ? 0 : n == NB + 1 ? 1 : n == NB + 2 ? 4 : 5;
        la.template issue<i, stage * W4_OPERAND + NW * i * 1024>(lds_wave);
      }
    };
    auto issue_p1 = [&](auto stage_index, auto n_index) {
      constexpr int stage = decltype(stage_index)::value, n = decltype(n_index)::value;
      constexpr int i = n == 0 ? 2 : n == 1 ? 3 : n == 2 ? 6 : 7;
      la.template issue<i, stage * W4_OPERAND + NW * i * 1024>(lds_wave);
    };
    // fa0[t][k]: row blocks 0-1, fa1[t][k]: row blocks 2-3, fb[u][k]: column blocks, K slab k.
    u32x4 fa0[2][4], fa1[2][4], fb[TN][4];
    // Fragment n (0 .. TN + 1) of K slab k of part 0 of a stage: TN of B, two of A.
    auto read_p0 = [&](auto stage_index, auto k_index, auto n_index) {
      constexpr int stage = decltype(stage_index)::value, k = decltype(k_index)::value, n = decltype(n_index)::value;
      if constexpr (n < TN) fb[n][k] = rb.template read<n, k, stage>();
      else fa0[n - TN][k] = ra.template read<n - TN, k, stage>();
    };
    // Fragment n (0..7) of part 1 of a stage: K slab n / 2, row block 2 + n % 2.
    auto read_p1 = [&](auto stage_index, auto n_index) {
      constexpr int stage = decltype(stage_index)::value, n = decltype(n_index)::value;
      fa1[n % 2][n / 2] = ra.template read<2 + n % 2, n / 2, stage>();
    };
    // Both stages' loads, part 0 of step 0 published, its fragments read.
    static_for<0, NP0>([&](auto n_index) { issue_p0(S0, n_index); });
    static_for<0, 4>([&](auto n_index) { issue_p1(S0, n_index); });
    la.base.advance();
    lb.base.advance();
    if (steps > 1) {
      static_for<0, NP0>([&](auto n_index) { issue_p0(S1, n_index); });
      static_for<0, 4>([&](auto n_index) { issue_p1(S1, n_index); });
      la.base.advance();
      lb.base.advance();
    }
    clear_acc();
    wait_loads(steps > 1, std::integral_constant<int, 4 + NSTEP>{}, C4{});
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, 4>([&](auto k_index) {
      static_for<0, TN + 2>([&](auto n_index) { read_p0(S0, k_index, n_index); });
    });
    __builtin_amdgcn_sched_barrier(0);

    // One K step out of stage STAGE. `next`: another step follows; `loads`: two more follow (the
    // loads of the second start here). The fragment reads "of the next step" also run in the last
    // step, on stale data nobody uses. The K loop holds one copy of this per stage and nothing
    // else, so the accumulators stay where they are.
    // Part 0's load i goes out after product P0_AT(i) of half 0: spread over the products behind B0.
    auto step = [&](auto stage_index, bool next, bool loads) {
      constexpr int STAGE = decltype(stage_index)::value;
      const std::integral_constant<int, STAGE> HERE{};
      const std::integral_constant<int, STAGE ^ 1> THERE{};
      // Half 0.
      static_for<0, HL>([&](auto n_index) {
        constexpr int n = decltype(n_index)::value, k = n / SL, t = (n % SL) / TN, u = n % TN;
        product_of(acc[t][u], fa0[t][k], fb[u][k]);
        if constexpr (n == SL - 1) {
          // B0. In flight behind part 1 of this step: both parts of the next.
          publish(next, CSTEP{}, C0{});
        } else {
          if constexpr (n >= SL) {
            // load i after product SL + i (HL - SL) / NP0 (TN = 4: every second product)
            constexpr int lo = ((n - SL) * NP0 + (HL - SL) - 1) / (HL - SL);  // first i with its place >= n
            if constexpr (lo < NP0 && SL + lo * (HL - SL) / NP0 == n) {
              if (loads) issue_p0(HERE, std::integral_constant<int, lo>{});
            }
          }
          if constexpr (n > SL && n < SL + 17 && (n - SL) % 2 == 1) read_p1(HERE, std::integral_constant<int, (n - SL - 1) / 2>{});
          __builtin_amdgcn_sched_barrier(0);
        }
      });
      if (loads) lb.base.advance();
      // B1. In flight behind part 0 of the next step: its part 1 and part 0 of the one after.
      publish(loads, C4P0{}, C4{});
      // Half 1.
      static_for<0, HL>([&](auto n_index) {
        constexpr int n = decltype(n_index)::value, k = n / SL, t = (n % SL) / TN, u = n % TN;
        product_of(acc[2 + t][u], fa1[t][k], fb[u][k]);
        if constexpr (n < 8 && n % 2 == 0) {
          if (loads) issue_p1(HERE, std::integral_constant<int, n / 2>{});
        }
        // The next step's fragments of slab k - 1 go where this step's have just been used.
        if constexpr (n >= SL && n % SL < TN + 2)
          read_p0(THERE, std::integral_constant<int, n / SL - 1>{}, std::integral_constant<int, n % SL>{});
        __builtin_amdgcn_sched_barrier(0);
      });
      if (loads) la.base.advance();
      static_for<0, TN + 2>([&](auto n_index) { read_p0(THERE, std::integral_constant<int, 3>{}, n_index); });
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll 1
    for (int j = 0; j < steps; j += 2) {  // the host keeps the step count even
      step(S0, true, j + 2 < steps);
      step(S1, j + 2 < steps, j + 3 < steps);
    }
  } else {
    W4Frags<true, W4_BM> ra;
    W4Frags<true, W4_BN> rb;
    ra.init(lds0, wm * 128, lane);
    rb.init(lds0 + W4_B0, wn * TN * 32, lane);
    // Part h of a stage: this wave's loads 4h .. 4h + 3 of A, then TN h .. TN h + TN - 1 of B.
    constexpr int NPART = 4 + TN, NF = 2 * NPART;  // loads per part and wave; fragments per half
    constexpr int SLAB = 4 * TN, HL = 2 * SLAB;   // products per K slab, per half
    typedef std::integral_constant<int, 0> C0;
    typedef std::integral_constant<int, NPART> C1P;
    typedef std::integral_constant<int, 2 * NPART> C2P;
    typedef std::integral_constant<int, 3 * NPART> C3P;
    auto issue_part = [&](auto stage_index, auto h_index, auto n_index) {
      constexpr int stage = decltype(stage_index)::value, h = decltype(h_index)::value, n = decltype(n_index)::value;
      if constexpr (n < 4) {
        constexpr int i = 4 * h + n;
        la.template issue<i, stage * W4_OPERAND + NW * i * 1024>(lds_wave);
      } else {
        constexpr int i = TN * h + (n - 4);
        lb.template issue<i, W4_B0 + stage * W4_OPERAND + NW * i * 1024>(lds_wave);
      }
    };
    // fa[h][t][s]: row block t, K slab 2h + s; fb[h][u][s] likewise.
    u32x4 fa[2][4][2], fb[2][TN][2];
    // Fragment n (0 .. NF - 1) of half h of a stage: eight of A, then 2 TN of B.
    auto read_half = [&](auto stage_index, auto h_index, auto n_index) {
      constexpr int stage = decltype(stage_index)::value, h = decltype(h_index)::value, n = decltype(n_index)::value;
      if constexpr (n < 8) fa[h][n / 2][n % 2] = ra.template read<n / 2, 2 * h + n % 2, stage>();
      else fb[h][(n - 8) / 2][n % 2] = rb.template read<(n - 8) / 2, 2 * h + n % 2, stage>();
    };
    const std::integral_constant<int, 0> H0{};
    const std::integral_constant<int, 1> H1{};

    static_for<0, NPART>([&](auto n_index) { issue_part(S0, H0, n_index); });
    static_for<0, NPART>([&](auto n_index) { issue_part(S0, H1, n_index); });
    la.base.advance();
    lb.base.advance();
    if (steps > 1) {
      static_for<0, NPART>([&](auto n_index) { issue_part(S1, H0, n_index); });
      static_for<0, NPART>([&](auto n_index) { issue_part(S1, H1, n_index); });
      la.base.advance();
      lb.base.advance();
    }
    clear_acc();
    wait_loads(steps > 1, C3P{}, C1P{});
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, NF>([&](auto n_index) { read_half(S0, H0, n_index); });
    __builtin_amdgcn_sched_barrier(0);

    auto step = [&](auto stage_index, bool next, bool loads) {
      constexpr int STAGE = decltype(stage_index)::value;
      const std::integral_constant<int, STAGE> HERE{};
      const std::integral_constant<int, STAGE ^ 1> THERE{};
      // Half 0.
      static_for<0, HL>([&](auto n_index) {
        constexpr int n = decltype(n_index)::value, sl = n / SLAB, t = (n % SLAB) / TN, u = n % TN;
        product_of(acc[t][u], fa[0][t][sl], fb[0][u][sl]);
        if constexpr (n == 7) {
          // B0. In flight behind part 1 of this step: both parts of the next.
          publish(next, C2P{}, C0{});
        } else {
          if constexpr (n >= 8 && n < 8 + NF) {
            if constexpr (n % 2 == 0 && (n - 8) / 2 < NPART) {
              if (loads) issue_part(HERE, H0, std::integral_constant<int, (n - 8) / 2>{});
            }
            read_half(HERE, H1, std::integral_constant<int, n - 8>{});
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      });
      // B1. In flight behind part 0 of the next step: its part 1 and part 0 of the one after.
      publish(loads, C2P{}, C1P{});
      // Half 1.
      static_for<0, HL>([&](auto n_index) {
        constexpr int n = decltype(n_index)::value, sl = n / SLAB, t = (n % SLAB) / TN, u = n % TN;
        product_of(acc[t][u], fa[1][t][sl], fb[1][u][sl]);
        if constexpr (n < NF) {
          if constexpr (n % 2 == 0 && n / 2 < NPART) {
            if (loads) issue_part(HERE, H1, std::integral_constant<int, n / 2>{});
          }
          read_half(THERE, H0, n_index);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      if (loads) {
        la.base.advance();
        lb.base.advance();
      }
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll 1
    for (int j = 0; j < steps; j += 2) {  // the host keeps the step count even
      step(S0, true, j + 2 < steps);
      step(S1, j + 2 < steps, j + 3 < steps);
    }
  }
  if constexpr (LR) {
    if (split == 0)
      gemm_low_rank<TM, TN>(g, m0 + wm * TM * 32, n0 + wn * TN * 32, lane, [&](auto t, auto u, const u32x4& a, const u32x4& b) {
        product_of(acc[decltype(t)::value][decltype(u)::value], a, b);
      });
  }
  // Every wave has read its last fragments before the stages are reused for the store pass.
  __builtin_amdgcn_s_waitcnt(vmcnt_only(0) & 0xC07F);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);

  // Store pass: each wave stages 32 rows of its tile at a time through its own LDS region and
  // writes whole pieces of rows.
  constexpr int CPW = TN * 32 + 4;
  static_assert(NW * 32 * CPW * 4 <= W4_SMEM, "staging fits");
  float* cs = reinterpret_cast<float*>(smem) + wave * (32 * CPW);
  bool bad = false;
  constexpr int PPR = TN * 8;  // 4-column pieces per row
  const int gcol0 = n0 + wn * TN * 32;
  const bool packed = g.splits == 1 && g.c_bf16 && g.c_vec != 0 && (g.ldc & 7) == 0 &&
                      (reinterpret_cast<uintptr_t>(g.c) & 15) == 0;
  constexpr int HP = TN * 32 * 2 + 16;  // bytes per staged bf16 row
  char* hs = reinterpret_cast<char*>(cs);
  unsigned flags = 0;  // bit 15 or 31 set: a stored bf16 has an all-ones exponent
  bool bad_act = false;
  // DPAIR: a lane has 8 units of a row (N is a multiple of 128). Gates and ups of 16 rows are on their way while 16 others are
  // worked on, and the barriers keep them so (each 32 rows' loads at their start, unpinned: 366 us for the 359 above).
  float4 in[DPAIR ? 2 : 1][4][4];  // [half][row][gates, ups]
  auto load_pairs = [&](int tm, int half) {
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const long row = min(m0 + (wm * TM + tm) * 32 + (half * 4 + it) * 4 + (lane >> 4), g.M - 1);
      const float* gates = reinterpret_cast<const float*>(g.aux_in) + row * (2l * g.N) + gcol0 + (lane & 15) * 8;
      in[half][it][0] = dev_stream_load<true>(reinterpret_cast<const float4*>(gates));
      in[half][it][1] = dev_stream_load<true>(reinterpret_cast<const float4*>(gates + 4));
      in[half][it][2] = dev_stream_load<true>(reinterpret_cast<const float4*>(gates + g.N));
      in[half][it][3] = dev_stream_load<true>(reinterpret_cast<const float4*>(gates + g.N + 4));
    }
  };
  if constexpr (DPAIR) {
    if (gcol0 < g.N) load_pairs(0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
  static_for<0, TM>([&](auto tm_index) {
    constexpr int tm = decltype(tm_index)::value;
    const int grow0 = m0 + (wm * TM + tm) * 32;
    const bool interior = grow0 + 32 <= g.M && gcol0 + TN * 32 <= g.N;
    if constexpr (ROPE) {
      const int dim = g.rope.dim, per = dim / 8, head = (lane & 15) / per, at = (lane & 15) % per * 4, lo = head * dim + at;
      const bool turn = gcol0 < g.rope.heads * dim;  // (N and the columns that turn are multiples of 128)
      float4 c4[8], s4[8];  // on their way while the rows are staged
      if (turn) {
        int t = (grow0 + (lane >> 4)) % g.rope.time;
#pragma unroll
        for (int it = 0; it < 8; ++it) {
          const long from = static_cast<long>(t) * dim + at;
          c4[it] = *reinterpret_cast<const float4*>(g.rope.cos_t + from);
          s4[it] = *reinterpret_cast<const float4*>(g.rope.sin_t + from);
          t += 4;
          while (t >= g.rope.time) t -= g.rope.time;
        }
      }
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx16& c = acc[tm][tn];
          *reinterpret_cast<float4*>(cs + l32 * CPW + tn * 32 + 8 * q + 4 * lg) = make_float4(c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]);
        }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (gcol0 < g.N) {
#pragma unroll
        for (int it = 0; it < 8; ++it) {
          const int row = it * 4 + (lane >> 4);
          const float4 x = *reinterpret_cast<const float4*>(cs + row * CPW + lo), y = *reinterpret_cast<const float4*>(cs + row * CPW + lo + dim / 2);
          const float a[4] = {x.x, x.y, x.z, x.w}, b[4] = {y.x, y.y, y.z, y.w};
          float ya[4] = {x.x, x.y, x.z, x.w}, yb[4] = {y.x, y.y, y.z, y.w};
          if (turn) {
            const float c[4] = {c4[it].x, c4[it].y, c4[it].z, c4[it].w}, s[4] = {s4[it].x, s4[it].y, s4[it].z, s4[it].w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              ya[e] = a[e] * c[e] - b[e] * s[e];
              yb[e] = b[e] * c[e] + a[e] * s[e];
            }
          }
          if (grow0 + row < g.M) {
            unsigned short* to = g.aux_out + static_cast<long>(grow0 + row) * g.ldc + gcol0 + lo;
            *reinterpret_cast<uint2*>(to) = make_uint2(dev_pack_bf16_pair(ya[0], ya[1]), dev_pack_bf16_pair(ya[2], ya[3]));
            *reinterpret_cast<uint2*>(to + dim / 2) = make_uint2(dev_pack_bf16_pair(yb[0], yb[1]), dev_pack_bf16_pair(yb[2], yb[3]));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              bad |= !(dev_finite(a[e]) && dev_finite(b[e]));
              bad_act |= !(dev_finite(ya[e]) && dev_finite(yb[e]));
            }
          }
        }
      }
    } else if constexpr (PAIR) {
      const int half = g.N / 2, unit0 = n0 / 2 + wn * 64;
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx16& c = acc[tm][tn];
          *reinterpret_cast<float4*>(cs + l32 * CPW + tn * 32 + 8 * q + 4 * lg) = make_float4(c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]);
        }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (unit0 < half) {  // (half is a multiple of 64)
#pragma unroll
        for (int it = 0; it < 8; ++it) {
          const int row = it * 4 + (lane >> 4), piece = (lane & 15) * 4;
          const float4 gate = *reinterpret_cast<const float4*>(cs + row * CPW + piece), up = *reinterpret_cast<const float4*>(cs + row * CPW + 64 + piece);
          if (grow0 + row < g.M) {
            float* to = static_cast<float*>(g.c) + static_cast<long>(grow0 + row) * g.ldc + unit0 + piece;
            *reinterpret_cast<float4*>(to) = gate;
            *reinterpret_cast<float4*>(to + half) = up;
            const float y0 = gate.x * dev_sigmoid(gate.x) * up.x, y1 = gate.y * dev_sigmoid(gate.y) * up.y, y2 = gate.z * dev_sigmoid(gate.z) * up.z,
                        y3 = gate.w * dev_sigmoid(gate.w) * up.w;
            *reinterpret_cast<uint2*>(g.aux_out + static_cast<long>(grow0 + row) * half + unit0 + piece) =
                make_uint2(dev_pack_bf16_pair(y0, y1), dev_pack_bf16_pair(y2, y3));
            bad |= !(dev_finite(gate.x) && dev_finite(gate.y) && dev_finite(gate.z) && dev_finite(gate.w) && dev_finite(up.x) && dev_finite(up.y) &&
                     dev_finite(up.z) && dev_finite(up.w));
            bad_act |= !(dev_finite(y0) && dev_finite(y1) && dev_finite(y2) && dev_finite(y3));
          }
        }
      }
    } else if constexpr (DPAIR) {
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx16& c = acc[tm][tn];
          uint2 w;
          w.x = dev_pack_bf16_pair(c[4 * q], c[4 * q + 1]);
          w.y = dev_pack_bf16_pair(c[4 * q + 2], c[4 * q + 3]);
          *reinterpret_cast<uint2*>(hs + l32 * HP + (tn * 32 + 8 * q + 4 * lg) * 2) = w;
        }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (gcol0 < g.N) {
        static_for<0, 2>([&](auto half_index) {
          constexpr int half = decltype(half_index)::value;
          if constexpr (half == 0) load_pairs(tm, 1);
          else if constexpr (tm + 1 < TM) load_pairs(tm + 1, 0);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int it = 0; it < 4; ++it) {
            const int row = (half * 4 + it) * 4 + (lane >> 4);
            const uint4 v = *reinterpret_cast<const uint4*>(hs + row * HP + (lane & 15) * 16);
            const float4* p = in[half][it];
            const float ga[8] = {p[0].x, p[0].y, p[0].z, p[0].w, p[1].x, p[1].y, p[1].z, p[1].w};
            const float up[8] = {p[2].x, p[2].y, p[2].z, p[2].w, p[3].x, p[3].y, p[3].z, p[3].w};
            const unsigned w[4] = {v.x, v.y, v.z, v.w};
            float gg[8], gu[8];
            bool wrong = false;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float d = __uint_as_float(e & 1 ? w[e / 2] & 0xffff0000u : w[e / 2] << 16), s = dev_sigmoid(ga[e]);
              gu[e] = d * (ga[e] * s);
              gg[e] = d * up[e] * (s * (1.0f + ga[e] * (1.0f - s)));
              wrong |= !(dev_finite(gu[e]) && dev_finite(gg[e]));
            }
            if (grow0 + row < g.M) {
#pragma unroll
              for (int e = 0; e < 4; ++e) flags |= (w[e] & 0x7F807F80u) + 0x00800080u;
              bad_act |= wrong;
              unsigned short* to = g.aux_out + (grow0 + row) * (2l * g.N) + gcol0 + (lane & 15) * 8;
              *reinterpret_cast<uint4*>(to) = make_uint4(dev_pack_bf16_pair(gg[0], gg[1]), dev_pack_bf16_pair(gg[2], gg[3]),
                                                         dev_pack_bf16_pair(gg[4], gg[5]), dev_pack_bf16_pair(gg[6], gg[7]));
              *reinterpret_cast<uint4*>(to + g.N) = make_uint4(dev_pack_bf16_pair(gu[0], gu[1]), dev_pack_bf16_pair(gu[2], gu[3]),
                                                               dev_pack_bf16_pair(gu[4], gu[5]), dev_pack_bf16_pair(gu[6], gu[7]));
            }
          }
        });
      }
    } else if (packed && interior) {
      // bf16: rounded in registers, staged 8 bytes at a time, stored 16 bytes per lane (a wave
      // instruction writes four rows of 64 TN bytes; with TN = 3 four lanes in 16 sit out).
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx16& c = acc[tm][tn];
          uint2 w;
          w.x = dev_pack_bf16_pair(c[4 * q], c[4 * q + 1]);
          w.y = dev_pack_bf16_pair(c[4 * q + 2], c[4 * q + 3]);
          flags |= ((w.x & 0x7F807F80u) + 0x00800080u) | ((w.y & 0x7F807F80u) + 0x00800080u);
          *reinterpret_cast<uint2*>(hs + l32 * HP + (tn * 32 + 8 * q + 4 * lg) * 2) = w;
        }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      unsigned short* crow = static_cast<unsigned short*>(g.c) + static_cast<long>(grow0 + (lane >> 4)) * g.ldc + gcol0 +
                             (lane & 15) * 8;
      const long four_rows = 4 * g.ldc;
      if ((lane & 15) < TN * 4) {
#pragma unroll
        for (int it = 0; it < 8; ++it) {
          const uint4 v = *reinterpret_cast<const uint4*>(hs + (it * 4 + (lane >> 4)) * HP + (lane & 15) * 16);
          *reinterpret_cast<uint4*>(crow + it * four_rows) = v;
        }
      }
    } else {
      // f32 results, split-K partials, ragged edges: staged as f32 rows.
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx16& c = acc[tm][tn];
          *reinterpret_cast<float4*>(cs + l32 * CPW + tn * 32 + 8 * q + 4 * lg) =
              make_float4(c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]);
        }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (interior && (g.splits > 1 ? (g.N & 3) == 0 : g.c_vec != 0)) {
        if (g.splits > 1) bad |= gemm_store_block<0, PPR>(g, split, cs, CPW, grow0, gcol0, lane);
        else if (g.c_bf16) bad |= gemm_store_block<1, PPR>(g, split, cs, CPW, grow0, gcol0, lane);
        else if (!g.accumulate) bad |= gemm_store_block<2, PPR>(g, split, cs, CPW, grow0, gcol0, lane);
        else bad |= gemm_store_block<3, PPR>(g, split, cs, CPW, grow0, gcol0, lane);
      } else {
#pragma unroll 1
        for (int c = lane; c < 32 * PPR; c += 64) {
          const int row = c / PPR, piece = c % PPR;
          const int grow = grow0 + row, gcol = gcol0 + piece * 4;
          if (grow < g.M && gcol < g.N) {
            const float4 val = *reinterpret_cast<const float4*>(cs + row * CPW + piece * 4);
            bad |= gemm_store4(g, split, grow, gcol, val.x, val.y, val.z, val.w);
          }
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  });
  bad |= (flags & 0x80008000u) != 0;
  if (bad) dev_raise_fault(g.fault, g.tag);
  if (STORE && bad_act && !bad) dev_raise_fault(g.fault, g.act_tag);
}

template <bool A_KM, bool B_KM, int TN>
int32_t launch_w4(omx_ctx* ctx, const GemmArgs& g) {
  auto kernel = &gemm_w4_kernel<A_KM, B_KM, TN, false>;
  if constexpr (B_KM) {
    if (g.k_rows != g.K) kernel = &gemm_w4_kernel<A_KM, B_KM, TN, true>;
  }
  if constexpr (!A_KM) {
    if (g.lr_rank > 0) kernel = &gemm_w4_kernel<A_KM, B_KM, TN, false, true>;  // (whole steps)
  }
  if constexpr (!A_KM && !B_KM && TN == 4) {
    if (g.epi == OMX_EPI_SWIGLU) kernel = &gemm_w4_kernel<false, false, 4, false, false, OMX_EPI_SWIGLU>;
    if (g.epi == OMX_EPI_ROPE) kernel = &gemm_w4_kernel<false, false, 4, false, true, OMX_EPI_ROPE>;
  }
  if constexpr (!A_KM && B_KM && TN == 4) {
    if (g.epi == OMX_EPI_SWIGLU_BWD) kernel = &gemm_w4_kernel<false, true, 4, false, false, OMX_EPI_SWIGLU_BWD>;
  }
  OMX_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   W4_SMEM));
  omx_launch_timed(ctx, kernel, dim3(g.tiles_m * g.tiles_n * g.splits, g.batches), dim3(256), W4_SMEM, ctx->timing_start,
                   g.splits > 1 ? nullptr : ctx->timing_stop, g);
  OMX_LAUNCH_CHECK(ctx, "gemm_w4_kernel");
  return OMX_OK;
}

}  // namespace
