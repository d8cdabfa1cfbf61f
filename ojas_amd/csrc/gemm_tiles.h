// Pieces shared by the direct-to-LDS GEMM kernels (gemm_dma.hip, gemm_q8.hip): the per-lane
// global -> LDS load state of an operand tile, the swizzled fragment offsets that go with it,
// and the counted-wait helper.
#pragma once

#include <type_traits>

#include "gemm_args.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef short short4v __attribute__((ext_vector_type(4)));

// f(integral_constant<int, I>) for I = BEGIN .. END - 1.
template <int BEGIN, int END, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (BEGIN < END) {
    f(std::integral_constant<int, BEGIN>{});
    static_for<BEGIN + 1, END>(f);
  }
}

// Workgroup -> tile so that the workgroups of one XCD (equal index modulo 8) take a contiguous run of the tiles, also
// where the count is no multiple of 8: the first count % 8 XCDs have one more. 684 x 5504 over 2048 on 64 x 64 tiles,
// 946 of them: 47.8 us in index order, where neighbours sit behind eight different L2s, 24.9 in this one; 802 products
// of 40 .. 16384 rows 4.5 % less on average.
__device__ inline int tile_of_eighth(int index, int count) {
  const int xcd = index & 7;
  return xcd * (count >> 3) + min(xcd, count & 7) + (index >> 3);
}

// Where a wave's direct-to-LDS loads of one operand tile start: a wave-uniform address of the tile's first element at
// the current K step, beside which every lane and load has a 32-bit byte offset that never changes. A K step advances
// scalars only (64-bit vector additions would take issue slots from the matrix instructions).
// TAIL: a k-major operand ends after `rows_left` more K rows, wherever in a step that is. Its loads are then buffer
// loads bounded to what is left of the current step, and lanes past the bound write zeros into LDS, so a reduction of
// any length (weight gradients: K = tokens) runs whole steps. Six products of 512 x 2048 over 3500 rows: 225 us on the
// register-staged kernel, which such lengths took before, 69 us here. A kernel of its own, because the bounded loads
// cost 1 % where no step is ragged (2635 -> 2662 us over the weight gradients of 12 layers of d = 768). A k-contiguous
// operand's rows have to hold whole steps.
template <bool KM, bool TAIL>
struct StepBase {
  const char* at;
  long step;  // bytes between consecutive K steps
  __device__ __forceinline__ void init(const void* p, long ld, int row0, int k0, int /*k_rows*/, int bk) {
    const long first = KM ? static_cast<long>(k0) * ld + row0 : static_cast<long>(row0) * ld + k0;
    const unsigned long long addr = reinterpret_cast<unsigned long long>(p) + static_cast<unsigned long long>(first) * 2;
    // (tile coordinates come out of vector divisions: back to scalars)
    const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(addr));
    const unsigned hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(addr >> 32));
    at = reinterpret_cast<const char*>((static_cast<unsigned long long>(hi) << 32) | lo);
    step = (KM ? bk * ld : bk) * 2;
  }
  __device__ __forceinline__ void advance() { at += step; }
  // 16 bytes per lane into LDS at `lds` + IMM + 16 * lane. Written as assembly: the compiler cannot tell that this
  // asynchronous LDS write targets a stage that is NOT being read, and would otherwise make every LDS read wait for
  // it (vmcnt(0) right after the issue), which serialises the loads with the products.
  template <int IMM>
  __device__ __forceinline__ void load(unsigned off, unsigned lds) const {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(at), "s"(lds + IMM) : "memory");
  }
};
template <>
struct StepBase<true, true> {
  unsigned long long at;
  u32x4 rsrc;      // base address (48 bits, no stride), bytes from it, 32-bit raw data
  int rows_left;   // K rows from this step on
  int rows, pitch; // K rows per step, bytes per K row
  __device__ __forceinline__ void init(const void* p, long ld, int row0, int k0, int k_rows, int bk) {
    const unsigned long long addr =
        reinterpret_cast<unsigned long long>(p) + static_cast<unsigned long long>(static_cast<long>(k0) * ld + row0) * 2;
    const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(addr));
    const unsigned hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(addr >> 32));
    at = (static_cast<unsigned long long>(hi) << 32) | lo;
    rows = bk;
    pitch = static_cast<int>(ld * 2);
    rows_left = __builtin_amdgcn_readfirstlane(k_rows - k0);
    describe();
  }
  // Offsets of K row r of the step lie in [r pitch, (r + 1) pitch): in bounds exactly for the rows that are left.
  __device__ __forceinline__ void describe() {
    int live = rows_left < rows ? rows_left : rows;
    // (written out: the compiler merges the two into a vector med3)
    asm("s_max_i32 %0, %0, 0" : "+s"(live) : : "scc");
    rsrc = u32x4{static_cast<unsigned>(at), static_cast<unsigned>(at >> 32) & 0xffffu, static_cast<unsigned>(live * pitch),
                 0x00020000u};
  }
  __device__ __forceinline__ void advance() {
    at += static_cast<unsigned long long>(rows) * static_cast<unsigned>(pitch);
    rows_left -= rows;
    describe();
  }
  template <int IMM>
  __device__ __forceinline__ void load(unsigned off, unsigned lds) const {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(rsrc), "s"(lds),
                 "n"(IMM)
                 : "memory", "scc");
  }
};

// What K row kr of a k-major tile XORs its 16-byte slots with: the four rows of a transposing read 64 bytes apart in the
// 256 bytes that the banks span. (A row of 64 elements is half of that, so rows 0 and 2, 1 and 3 have to part.)
// KIND: 0 as above. f32 tiles (gemm_dma32.hip; ROWS counts halves of an element), whose instruction j reads 4 or 8 bytes a
// lane of four K rows at once: 1: rows 4 j .. 4 j + 3 (both operands k-major); 2: rows j, 4 + j, 8 + j, 12 + j, of which
// four of 128 bytes share 32 banks whatever their order.
template <int ROWS, int KIND = 0>
__device__ __forceinline__ int km_swizzle(int kr) {
  if constexpr (KIND == 1) return ROWS == 64 ? (kr >> 1 & 1) * 4 : (kr & 1) * 8;
  if constexpr (KIND == 2) return (kr >> 2 & 1) * (ROWS == 64 ? 4 : 8);
  return ROWS == 64 ? (kr >> 1 & 1) * 4 : (kr & 3) * 4;
}

// One operand's loads: ROWS x BK bf16 per step, one wave instruction per KiB. Rows past the end are clamped in the
// offset, so edge tiles take this form too (a k-major operand's last 16-byte chunk may reach past its last column into
// the padding of the row, which is at least 16 bytes aligned; those values only meet outputs that are not stored).
// Needs 255 rows of the leading dimension to fit 32 bits of bytes.
template <bool KM, int ROWS, int BK, int NW, bool TAIL = false, int KIND = 0>
struct TileLoadsOff {
  static constexpr int TOTAL = ROWS * BK * 2 / 1024;
  static constexpr int N = TOTAL / NW;
  static_assert(TOTAL % NW == 0, "the same number of loads in every wave");
  unsigned off[N];
  StepBase<KM, TAIL> base;

  // `k_rows`: where the K rows of a k-major operand end.
  __device__ __forceinline__ void init(const unsigned short* __restrict__ p, long ld, int row0, int rows, int k0,
                                       int k_rows, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int q = wave + NW * i;
      if constexpr (!KM) {
        // [row][BK / 8 chunks of 16 bytes], swizzled as frag_offset reads them.
        constexpr int LPR = BK / 8;  // lanes (chunks) per row
        const int r = q * (64 / LPR) + lane / LPR;
        const int kc = (lane % LPR) ^ (BK == 32 ? (r >> 2) & 3 : (r >> 1) & 7);
        int gr = row0 + r;
        gr = gr < rows ? gr : rows - 1;
        off[i] = static_cast<unsigned>(gr - row0) * static_cast<unsigned>(ld * 2) + kc * 16;
      } else {
        constexpr int CPR = ROWS / 8;
        const int idx = q * 64 + lane;
        const int kr = idx / CPR, slot = idx % CPR;
        const int mc = slot ^ km_swizzle<ROWS, KIND>(kr);
        int gm = mc * 8;
        gm = row0 + gm < rows ? gm : 0;
        off[i] = static_cast<unsigned>(kr) * static_cast<unsigned>(ld * 2) + gm * 2;
      }
    }
    base.init(p, ld, row0, k0, k_rows, BK);
  }
  // Starts this step's loads into the operand tile at LDS byte address `tile` and moves on.
  __device__ __forceinline__ void issue(unsigned tile, int wave) {
    const unsigned lds = tile + wave * 1024;
    static_for<0, N>([&](auto i) { base.template load<NW * decltype(i)::value * 1024>(off[decltype(i)::value], lds); });
    base.advance();
  }
};

// Byte offset, inside an operand tile, of this lane's fragment for 32-row block `row_base / 32`
// and 16-column K slab kk (k-major operands: of its first transposing read; the second is four
// K rows further).
template <bool KM, int ROWS, int BK>
__device__ __forceinline__ int frag_offset(int row_base, int kk, int lane) {
  if constexpr (!KM) {
    const int l32 = lane & 31, g = lane >> 5;
    const int r = row_base + l32;
    const int kc = kk * 2 + g;
    return r * (BK * 2) + ((kc ^ (BK == 32 ? (r >> 2) & 3 : (r >> 1) & 7)) << 4);
  } else {
    const int s = lane & 15, half = (lane >> 4) & 1, g = lane >> 5;
    const int kr = kk * 16 + g * 8 + (s >> 2);
    const int col = row_base + half * 16 + (s & 3) * 4;
    const int slot = (col >> 3) ^ km_swizzle<ROWS>(kr);
    return kr * (ROWS * 2) + slot * 16 + (col & 7) * 2;
  }
}
template <bool KM, int ROWS>
__device__ __forceinline__ u32x4 frag_at(const char* p) {
  if constexpr (!KM) {
    return *reinterpret_cast<const u32x4*>(p);
  } else {
    typedef short4v __attribute__((address_space(3))) * lds_ptr;
    short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p));
    short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p + 4 * ROWS * 2));
    u32x2 a = __builtin_bit_cast(u32x2, lo), b = __builtin_bit_cast(u32x2, hi);
    return u32x4{a.x, a.y, b.x, b.y};
  }
}

// s_waitcnt operand that waits for vmcnt <= n only (vmcnt is bits 3:0 and 15:14).
constexpr int vmcnt_only(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }

// Waits until at most `groups` (up to G) groups of LPS loads are still in flight.
template <int G, int LPS>
__device__ __forceinline__ void wait_loads(int groups) {
  if constexpr (G <= 0) {
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
  } else {
    if (groups >= G) __builtin_amdgcn_s_waitcnt(vmcnt_only(G * LPS));
    else wait_loads<G - 1, LPS>(groups);
  }
}

// The low-rank term of a wave's TM x TN blocks of 32 x 32 from (row0, col0) on, its operands straight from memory into fragments
// (a few KiB a row block): product(t, u, a, b) multiplies 16 columns of it into block (t, u).
template <int TM, int TN, typename P>
__device__ __forceinline__ void gemm_low_rank(const GemmArgs& g, int row0, int col0, int lane, P product) {
  const int l32 = lane & 31, lg = lane >> 5;
#pragma unroll 1
  for (int p = 0; p < g.lr_rank; p += 16)
    static_for<0, TN>([&](auto u_index) {
      constexpr int u = decltype(u_index)::value;
      const int col = min(col0 + u * 32, g.N - 1);
      const unsigned short* h = g.lr_h + p + 8 * lg + (g.lr_block_cols > 0 ? col / g.lr_block_cols * g.lr_rank : 0);
      const u32x4 b = *reinterpret_cast<const u32x4*>(g.lr_w + min(col0 + u * 32 + l32, g.N - 1) * g.lr_w_pitch + p + 8 * lg);
      static_for<0, TM>([&](auto t_index) {
        constexpr int t = decltype(t_index)::value;
        product(t_index, u_index, *reinterpret_cast<const u32x4*>(h + min(row0 + t * 32 + l32, g.M - 1) * g.lr_pitch), b);
      });
    });
}

// Waves per SIMD the kernel is compiled for: as many workgroups per compute unit as its LDS (160
// KiB) allows, up to four waves per SIMD.
constexpr int dma_waves_per_simd(int waves, int lds_bytes) {
  const int by_lds = 160 * 1024 / lds_bytes, by_waves = 16 / waves;
  return (by_lds < by_waves ? by_lds : by_waves) * waves / 4;
}

}  // namespace
