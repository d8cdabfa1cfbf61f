// bf16 MFMA flash attention for head_dim 64 and 128: causal forward, and the backward
// as two passes (dK/dV per key block, dQ per query block) that recompute the
// probabilities from the saved log-sum-exp, so no T x T matrix exists and no
// atomics are needed (where several waves or workgroups share the tiles of one output, their sums are added in a fixed order).
//
// Reference semantics: ojas-cpu/src/attn.rs:176-227 (forward rows), :519-597
// (backward from saved output and lse); the blocked CPU kernel
// ojas-cpu/src/attn/flash.rs:1-41 is the Fast-tier precedent for this shape of
// algorithm (online softmax, delta = sum P dP).
//
// Mapping onto v_mfma_f32_32x32x16_bf16 (A: lane (i = l%32, g = l/32) holds
// A[i][8g..8g+7]; B: lane (j, g) holds B[8g..8g+7][j]; D: lane (j, g), register
// v holds D[8(v/4) + 4g + v%4][j]):
//   * scores are formed transposed, S^T = K . Q^T (forward, dQ pass), or plain,
//     S = Q . K^T (dK/dV pass), so that the index a softmax statistic belongs to
//     (the query in the first case, nothing per-lane in the second) is the
//     lane's column and every row reduction stays inside a lane plus one
//     exchange with lane l^32;
//   * an accumulator tile is reused directly as the B operand of the next
//     product (P^T for O^T = V^T P^T, P / dS for dV^T, dK^T, dS^T for dQ^T):
//     registers 8c..8c+7 of a lane are k-slab c, holding rows
//     16c + {4g..4g+3, 8+4g..8+4g+3}; the A operand stored transposed in LDS
//     keeps its k index in the matching order (bits 2 and 3 of the index
//     swapped), so one 16-byte LDS read fetches exactly those rows.
#include "omx_common.h"
#include <algorithm>
#include <cmath>
#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

namespace {

// Head dims 64 and 128 (template argument D of everything below).
constexpr int fpitch(int D) { return D * 2 + 16; }      // bytes per LDS row: D bf16 + 16 pad
constexpr int ftile(int D) { return 64 * fpitch(D); }   // a 64-row tile
constexpr int FT = 256;                                 // threads per block (4 waves of 32 rows)
constexpr float LOG2E = 1.4426950408889634f;
constexpr int flash_dkv_set(int D) { return 2 * 64 * D * 2 + 2 * 64 * 4; }  // bytes: query and gradient tile, two values a row
constexpr int FLASH_OWN_ROWS = 1024;                    // row terms that a key side's workgroup keeps for itself
constexpr int flash_dq_lds(int D, int groups) { return groups * 4 * ftile(D) + D * 4; }
constexpr int flash_dkv_waves(int D, int groups) { return D == 64 && groups <= 2 ? 2 : 1; }
constexpr bool flash_in_turn(int D, int groups) { return D > 64 || groups > 1; }  // (see flash_fwd_tile)
// Waves per SIMD the query-side passes are compiled for: what their LDS leaves room for.
constexpr int flash_waves(int D, int groups) { return groups == 1 ? (D == 64 ? 3 : 2) : groups == 2 && D == 64 ? 2 : 1; }

// Element strides of one tensor: between rows (time steps), heads and batches.
struct FlashStrides {
  long rs, hs, bs;
};
struct FlashShape {
  int batch, heads, kv_heads, time, window, rep;
  // One 128-row block per workgroup instead of a mirrored pair, heaviest blocks first (query side:
  // forward and dQ; key side: dK/dV). Chosen by the host when the pairs would leave workgroup
  // places empty (few planes) or, on the key side, need a half-empty second round.
  int q_single, kv_single;
  int direct;    // dK/dV: time where all rows of q, k, v and the output's gradient are 16-byte aligned (tiles go straight into LDS), else 0
  int kv_parts;  // dK/dV: workgroups that share a key block's query tiles
  float scale;
  FlashStrides q, kv, o;  // q and grad_q; k, v and their gradients; out and grad_out
};


// f(integral_constant<int, i>) for i = 0 .. N - 1.
template <int N, int I = 0, typename F>
__device__ __forceinline__ void for_sequence(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    for_sequence<N, I + 1>(f);
  }
}

__device__ __forceinline__ unsigned int pack2(float a, float b) {
  floatx2 f = {a, b};
  return __builtin_bit_cast(unsigned int, __builtin_convertvector(f, bf16x2));
}
__device__ __forceinline__ u32x4 pack8(const floatx16& acc, int c) {
  u32x4 r;
  r.x = pack2(acc[8 * c + 0], acc[8 * c + 1]);
  r.y = pack2(acc[8 * c + 2], acc[8 * c + 3]);
  r.z = pack2(acc[8 * c + 4], acc[8 * c + 5]);
  r.w = pack2(acc[8 * c + 6], acc[8 * c + 7]);
  return r;
}
// acc + both bf16 halves of w (v_dot2c_f32_bf16 against a pair of ones).
__device__ __forceinline__ float sum_pairs(unsigned int w, float acc) {
  typedef __bf16 bf16_pair __attribute__((ext_vector_type(2)));
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16_pair, w), __builtin_bit_cast(bf16_pair, 0x3F803F80u),
                                         acc, false);
}
// acc + the products of the two bf16 halves of a and b (v_dot2c_f32_bf16; a product of two bf16
// values is exact in f32).
__device__ __forceinline__ float dot_pairs(unsigned int a, unsigned int b, float acc) {
  typedef __bf16 bf16_pair __attribute__((ext_vector_type(2)));
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16_pair, a), __builtin_bit_cast(bf16_pair, b), acc, false);
}
__device__ __forceinline__ floatx16 mfma(const u32x4& a, const u32x4& b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}
// max(a, b, c) in one instruction. fmaxf first quiets each accumulator value (a v_max_f32 of the
// value with itself) because the compiler cannot know an MFMA result is canonical; this does not.
// NaNs are skipped, as by fmaxf.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ floatx16 zero16() {
  floatx16 z;
#pragma unroll
  for (int v = 0; v < 16; ++v) z[v] = 0.0f;
  return z;
}

// A 64-row x D-column bf16 tile starting at row `row0` of a [time, D] plane, moved by NT threads (a workgroup's, or a
// key group's): 8 D / NT 16-byte chunks per thread. Thread t moves chunk t % (D/8) of rows t / (D/8) + i * (8 NT / D); rows at
// or past `time` read as zeros.
template <int D, int NT>
__device__ __forceinline__ void tile_load(const unsigned short* __restrict__ plane, long rs, int row0, int time,
                                          u32x4 (&r)[8 * D / NT]) {
  constexpr int CPR = D / 8, RPP = NT / CPR;
  const int t = threadIdx.x % NT;
  const int row = row0 + t / CPR, kc = t % CPR;
#pragma unroll
  for (int i = 0; i < 8 * D / NT; ++i) {
    r[i] = u32x4{0u, 0u, 0u, 0u};
    if (row + i * RPP < time)
      r[i] = *reinterpret_cast<const u32x4*>(plane + static_cast<long>(row + i * RPP) * rs + kc * 8);
  }
}
// [row][d] form.
template <int D, int NT>
__device__ __forceinline__ void tile_store_rows(char* lds, const u32x4 (&r)[8 * D / NT]) {
  constexpr int CPR = D / 8, RPP = NT / CPR;
  const int t = threadIdx.x % NT;
  const int row = t / CPR, kc = t % CPR;
#pragma unroll
  for (int i = 0; i < 8 * D / NT; ++i) *reinterpret_cast<u32x4*>(lds + (row + i * RPP) * fpitch(D) + kc * 16) = r[i];
}
// The same loads with the per-thread part of the address formed once. A tile that ends inside the
// sequence is fetched from a wave-uniform base (plane + row0 rows) plus the thread's fixed 32-bit byte
// offset: no address arithmetic and no bounds test per load. Only the last, ragged tile takes the
// checked path. The host refuses row strides for which the offset would not fit.
template <int D, int NT>
struct TileFetch {
  static constexpr int CPR = D / 8, RPP = NT / CPR;
  unsigned off;  // bytes from a tile's first element to this thread's first chunk
  long rs;
  int time;
  __device__ __forceinline__ TileFetch(long row_stride, int t_end) : rs(row_stride), time(t_end) {
    const int t = threadIdx.x % NT;
    off = static_cast<unsigned>((t / CPR) * row_stride + (t % CPR) * 8) * 2u;
  }
  __device__ __forceinline__ void load(const unsigned short* __restrict__ plane, int row0, u32x4 (&r)[8 * D / NT]) const {
    if (row0 + 64 <= time) {
      const char* base = reinterpret_cast<const char*>(plane + static_cast<long>(row0) * rs);
#pragma unroll
      for (int i = 0; i < 8 * D / NT; ++i) r[i] = *reinterpret_cast<const u32x4*>(base + static_cast<long>(i * RPP) * rs * 2 + off);
    } else {
      tile_load<D, NT>(plane, rs, row0, time, r);
    }
  }
};
constexpr long FLASH_MAX_ROW_STRIDE = 1L << 24;  // elements: 63 rows of it, in bytes, and a row's pieces stay below 2^31

// The wave's index as a scalar, so that what depends on it (which tiles the wave takes, which of
// them the diagonal cuts) is decided by scalar branches.
__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)); }

// x combined with the value lane ^ 32 holds: v_permlane32_swap exchanges the upper half of one
// register with the lower half of another, so swapping x with a copy of itself leaves (x of the lower
// lane, x of the upper lane) in the register pair of both lanes. One VALU instruction, no LDS round trip.
__device__ __forceinline__ float halves_max(float x) {
  const unsigned int u = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  float m;
  asm("v_max_f32 %0, %1, %2" : "=v"(m) : "v"(__uint_as_float(r[0])), "v"(__uint_as_float(r[1])));
  return m;
}
__device__ __forceinline__ float halves_sum(float x) {
  const unsigned int u = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// A operand from a [row][d] tile: rows sub*32 + lane%32, d-slab kk.
template <int D>
__device__ __forceinline__ u32x4 frag_rows(const char* lds, int sub, int kk, int l32, int lg) {
  return *reinterpret_cast<const u32x4*>(lds + (sub * 32 + l32) * fpitch(D) + kk * 32 + lg * 16);
}
// A operand of a product whose K index is the tile's ROW (O^T = V^T P^T, dV^T = dO^T P,
// dK^T = Q^T dS, dQ^T = K^T dS^T), read straight from the [row][d] tile with the transposing LDS
// read: a 16-lane group fetches a 4-row x 16-column block (8 bytes per lane) and each lane gets
// one column's 4 rows. Lane (i = lane % 32, g = lane / 32) ends up with column d = mt*32 + i and
// rows sub*32 + 16c + {4g..4g+3, 8+4g..8+4g+3}: the order in which an accumulator tile, reused as
// the B operand, holds its rows.
typedef short short4v __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
template <int D>
__device__ __forceinline__ u32x4 frag_tr(const char* lds, int mt, int sub, int c, int lane) {
  constexpr int FPITCH = fpitch(D);
  const int s = lane & 15, half = (lane >> 4) & 1, g = lane >> 5;
  const char* p = lds + (sub * 32 + c * 16 + 4 * g + (s >> 2)) * FPITCH + (mt * 32 + half * 16 + (s & 3) * 4) * 2;
  typedef short4v __attribute__((address_space(3))) * lds_ptr;
  const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p));
  const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p + 8 * FPITCH));
  const u32x2 a = __builtin_bit_cast(u32x2, lo), b = __builtin_bit_cast(u32x2, hi);
  return u32x4{a.x, a.y, b.x, b.y};
}
// B operand held in registers: the lane's own row of a [time, D] plane (past its end the last one: what comes of it is masked or not stored).
template <int D>
__device__ __forceinline__ void row_frags(const unsigned short* __restrict__ plane, long rs, int row, int time, int lg,
                                          u32x4 (&f)[D / 16]) {
  const unsigned short* at = plane + static_cast<long>(min(row, time - 1)) * rs + lg * 8;
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) f[kk] = *reinterpret_cast<const u32x4*>(at + kk * 16);
}
// dO . O of the lane's row `row`, `g` its row of dO: each half-wave holds half of the row's values. (Without a residual the output is
// read twice, so that neither load waits for the other's products.)
template <int D>
__device__ __forceinline__ float flash_row_delta(const u32x4 (&g)[D / 16], const unsigned short* __restrict__ out, const unsigned short* __restrict__ resid,
                                                 long rs, int row, int time, int lg) {
  u32x4 o[D / 16], r[D / 16];
  row_frags<D>(out, rs, row, time, lg, o);
  row_frags<D>(resid ? resid : out, rs, row, time, lg, r);
  auto dot_rows = [&](const u32x4 (&x)[D / 16]) {
    float sum = 0.0f;
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk)
#pragma unroll
      for (int w = 0; w < 4; ++w) sum = dot_pairs(g[kk][w], x[kk][w], sum);
    return sum;
  };
  float del = dot_rows(o);
  if (resid) del += dot_rows(r);
  return halves_sum(del);
}
// Row index (within a 32-row sub-tile) that accumulator register v of this lane holds.
__device__ __forceinline__ int acc_row(int v, int lg) { return 8 * (v >> 2) + 4 * lg + (v & 3); }

// Stores transposed accumulators (d x rows) as rows of a [time, D] plane.
template <int D, typename TO>
__device__ __forceinline__ bool store_transposed_acc(TO* __restrict__ plane, long rs, int row, int time, int lg,
                                                     const floatx16 (&acc)[D / 32], float mul) {
  bool bad = false;
  if (row >= time) return false;
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int d = mt * 32 + 8 * q4 + 4 * lg;
      float x0 = acc[mt][4 * q4 + 0] * mul, x1 = acc[mt][4 * q4 + 1] * mul, x2 = acc[mt][4 * q4 + 2] * mul,
            x3 = acc[mt][4 * q4 + 3] * mul;
      bad |= !(dev_finite(x0) && dev_finite(x1) && dev_finite(x2) && dev_finite(x3));
      if constexpr (sizeof(TO) == 2) {
        uint2 w;
        w.x = pack2(x0, x1);
        w.y = pack2(x2, x3);
        *reinterpret_cast<uint2*>(plane + static_cast<long>(row) * rs + d) = w;
      } else {
        *reinterpret_cast<float4*>(plane + static_cast<long>(row) * rs + d) = make_float4(x0, x1, x2, x3);
      }
    }
  return bad;
}

// The bf16 store of the output together with what the rounding dropped: residual = x - bf16(x),
// itself rounded to bf16, so that bf16(x) + residual carries 16 bits of x's mantissa.
template <int D>
__device__ __forceinline__ bool store_transposed_acc_split(unsigned short* __restrict__ plane,
                                                           unsigned short* __restrict__ resid, long rs, int row,
                                                           int time, int lg, const floatx16 (&acc)[D / 32], float mul) {
  bool bad = false;
  if (row >= time) return false;
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int d = mt * 32 + 8 * q4 + 4 * lg;
      const float x0 = acc[mt][4 * q4 + 0] * mul, x1 = acc[mt][4 * q4 + 1] * mul, x2 = acc[mt][4 * q4 + 2] * mul,
                  x3 = acc[mt][4 * q4 + 3] * mul;
      bad |= !(dev_finite(x0) && dev_finite(x1) && dev_finite(x2) && dev_finite(x3));
      uint2 w, r;
      w.x = pack2(x0, x1);
      w.y = pack2(x2, x3);
      r.x = pack2(x0 - __uint_as_float(w.x << 16), x1 - __uint_as_float(w.x & 0xffff0000u));
      r.y = pack2(x2 - __uint_as_float(w.y << 16), x3 - __uint_as_float(w.y & 0xffff0000u));
      *reinterpret_cast<uint2*>(plane + static_cast<long>(row) * rs + d) = w;
      *reinterpret_cast<uint2*>(resid + static_cast<long>(row) * rs + d) = r;
    }
  return bad;
}

// Workgroup -> (pair of row blocks, plane). Workgroups go to the 8 XCDs round-robin by their
// linear index and every XCD has its own L2, so the `pairs` workgroups of one plane (one head's
// K and V, or Q and dO) are given indices that are equal modulo 8: they run on one XCD, side by
// side, and the plane's tiles are fetched into one L2 instead of into several.
__device__ __forceinline__ void flash_block_of(int pairs, int planes, int* pair, long* plane) {
  const int id = blockIdx.x;
  if ((planes & 7) == 0) {
    *plane = (id & 7) + 8 * (id / (8 * pairs));
    *pair = (id >> 3) % pairs;
  } else {
    *pair = id % pairs;
    *plane = id / pairs;
  }
}

// use(i, load(i)) for i = 0 .. N - 1, a load two uses ahead of its own. Left to itself the compiler reads an operand out of LDS right
// before the product that takes it (one set of registers, a full LDS latency a product), which few waves a SIMD do not hide.
// Forward and dQ pass of head_dim 128, 13 x 9 heads x 1177 rows: 107 -> 99 and 146 -> 138 us; 8 x 3 x 531: 19.1 -> 16.9 and 21.0 ->
// 19.1; one key tile, nothing else on the chip: 6.7 -> 6.5. Three and five ahead measure the same.
template <int N, typename Load, typename Use>
__device__ __forceinline__ void in_turn(Load&& load, Use&& use) {
  constexpr int AHEAD = 2 < N ? 2 : N;
  constexpr int VECTOR_SCALAR = 6;  // what may move across: vector and scalar arithmetic, neither reads nor products
  u32x4 f[AHEAD + 1];
  for_sequence<AHEAD>([&](auto i) { f[i.value] = load(i); });
  for_sequence<N>([&](auto i) {
    if constexpr (i.value + AHEAD < N) f[(i.value + AHEAD) % (AHEAD + 1)] = load(std::integral_constant<int, i.value + AHEAD>{});
    __builtin_amdgcn_sched_barrier(VECTOR_SCALAR);
    use(i, f[i.value % (AHEAD + 1)]);
    __builtin_amdgcn_sched_barrier(VECTOR_SCALAR);
  });
}

// ------------------------------------------------------------------ forward
// One 32-query x 64-key tile of one wave: scores, online softmax, weights times values.
//   NSUB      32-key halves of the tile that hold a visible key (the second half of a tile whose
//             first key is the wave's first query is hidden from all 32 rows and is left out);
//   MASK_SUB  the half the causal diagonal cuts (its keys start at the wave's first query), or -1;
//   GENERAL   the tile crosses the sequence end or a window edge: every element is tested.
//   IN_TURN   operands are read two products ahead (in_turn). Not at head_dim 64 with three waves a SIMD: the registers end (10
//             spilled, 46.2 against 46.3 us at 16 x 12 x 1024 and 37.2 against 36.6 at 12 x 12 x 999), and the waves fill in.
// `m` is the running maximum of the raw scores; the scale joins inside the fma. `lsum` sums the
// weights as computed, `wsum` their bf16 copies (this lane's half of the keys).
template <int D, int NSUB, int MASK_SUB, bool GENERAL, bool IN_TURN>
__device__ __forceinline__ void flash_fwd_tile(const char* k_rows, const char* v_rows, const u32x4 (&qf)[D / 16],
                                               floatx16 (&o)[D / 32], float& m, float& lsum, float& wsum,
                                               float scale_log2, int key0, int q_row, int T, int window, int lane) {
  constexpr int KK = D / 16, MT = D / 32;
  const int l32 = lane & 31, lg = lane >> 5;
  floatx16 sc[NSUB];
  // The SIMD serves its oldest wave first, and matrix and vector instructions of different waves
  // barely overlap (measured: three waves of 16 MFMAs + 160 FMAs take 0.88 of the sum of both alone).
  // A wave in its vector phase therefore holds up the others' products for the whole phase; raised
  // priority for the two short product phases keeps the matrix units fed (7 % on the forward pass).
  __builtin_amdgcn_s_setprio(2);
  if constexpr (IN_TURN) {
    in_turn<NSUB * KK>([&](auto i) { return frag_rows<D>(k_rows, i.value / KK, i.value % KK, l32, lg); },
                       [&](auto i, const u32x4& f) {
                         constexpr int sub = i.value / KK, kk = i.value % KK;
                         if constexpr (kk == 0) sc[sub] = zero16();
                         sc[sub] = mfma(f, qf[kk], sc[sub]);
                       });
  } else {
#pragma unroll
    for (int sub = 0; sub < NSUB; ++sub) {
      sc[sub] = zero16();
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) sc[sub] = mfma(frag_rows<D>(k_rows, sub, kk, l32, lg), qf[kk], sc[sub]);
    }
  }
  __builtin_amdgcn_s_setprio(0);
  if constexpr (GENERAL) {
#pragma unroll
    for (int sub = 0; sub < NSUB; ++sub)
#pragma unroll
      for (int vv = 0; vv < 16; ++vv) {
        const int key = key0 + sub * 32 + acc_row(vv, lg);
        const bool masked = key > q_row || key >= T || (window > 0 && key + window <= q_row);
        sc[sub][vv] = masked ? -INFINITY : sc[sub][vv];
      }
  } else if constexpr (MASK_SUB >= 0) {
    // Key 4 lg + acc_row(v, 0) of the half against query l32 of the wave: a constant against one
    // value that never changes (kept opaque: hoisted out of the tile loop, the sixteen compare
    // results would occupy 32 scalar registers for the whole kernel).
    int tri = l32 - 4 * lg;
    asm volatile("" : "+v"(tri));
#pragma unroll
    for (int vv = 0; vv < 16; ++vv) sc[MASK_SUB][vv] = acc_row(vv, 0) > tri ? -INFINITY : sc[MASK_SUB][vv];
  }
  // Two chains, so that neither waits on the other's result.
  float tmax, tmax2;
  if constexpr (NSUB == 2) {
    tmax = fmaxf(sc[0][0], sc[1][0]);
    tmax2 = fmaxf(sc[0][1], sc[1][1]);
#pragma unroll
    for (int vv = 2; vv < 16; vv += 2) {
      tmax = max3(tmax, sc[0][vv], sc[1][vv]);
      tmax2 = max3(tmax2, sc[0][vv + 1], sc[1][vv + 1]);
    }
  } else {
    tmax = fmaxf(sc[0][0], sc[0][1]);
    tmax2 = fmaxf(sc[0][2], sc[0][3]);
#pragma unroll
    for (int vv = 4; vv < 16; vv += 4) {
      tmax = max3(tmax, sc[0][vv], sc[0][vv + 1]);
      tmax2 = max3(tmax2, sc[0][vv + 2], sc[0][vv + 3]);
    }
  }
  tmax = halves_max(fmaxf(tmax, tmax2));
  // The reference point of the exponents moves only when a row's maximum grew by more than 8
  // binary orders (always on a row's first tile, where m is -inf): below that the weights of
  // this tile are at most 2^8, well inside f32 and bf16, and the accumulators need no rescaling.
  // The quotient at the end and the log-sum-exp use the same reference, so both stay exact.
  const bool grow = (tmax - m) * scale_log2 > 8.0f;
  const float new_m = grow ? tmax : m;
  const float m_safe = new_m == -INFINITY ? 0.0f : new_m;
  const float neg_m = -m_safe * scale_log2;
  float psum = 0.0f;
#pragma unroll
  for (int sub = 0; sub < NSUB; ++sub)
#pragma unroll
    for (int vv = 0; vv < 16; ++vv) {
      float p = __builtin_amdgcn_exp2f(fmaf(sc[sub][vv], scale_log2, neg_m));
      sc[sub][vv] = p;
      psum += p;
    }
  psum = halves_sum(psum);
  if (__any(grow)) {
    // Some row's reference moved: rescale what is accumulated so far (by exactly 1 in the
    // rows that keep theirs).
    const float alpha = __builtin_amdgcn_exp2f(fmaf(m, scale_log2, neg_m));
    lsum *= alpha;
    wsum *= alpha;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int vv = 0; vv < 16; ++vv) o[mt][vv] *= alpha;
  }
  lsum += psum;
  m = new_m;
  __builtin_amdgcn_s_setprio(2);
  u32x4 pb;
  auto weights = [&](auto sub, auto c) {
    pb = pack8(sc[sub], c);
    wsum = sum_pairs(pb.x, sum_pairs(pb.y, sum_pairs(pb.z, sum_pairs(pb.w, wsum))));
  };
  if constexpr (IN_TURN) {
    in_turn<NSUB * 2 * MT>([&](auto i) { return frag_tr<D>(v_rows, i.value % MT, i.value / (2 * MT), i.value / MT % 2, lane); },
                           [&](auto i, const u32x4& f) {
                             constexpr int mt = i.value % MT;
                             if constexpr (mt == 0) weights(i.value / (2 * MT), i.value / MT % 2);
                             o[mt] = mfma(f, pb, o[mt]);
                           });
  } else {
#pragma unroll
    for (int sub = 0; sub < NSUB; ++sub)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        weights(sub, c);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) o[mt] = mfma(frag_tr<D>(v_rows, mt, sub, c, lane), pb, o[mt]);
      }
  }
  __builtin_amdgcn_s_setprio(0);
}

// WIN: the sliding-window form (every tile tested element by element), compiled apart so that the
// plain causal kernel carries neither its code nor its registers.
// GROUPS > 1: the workgroup's waves form that many groups, which take the key tiles of 128 / GROUPS query rows in turn and
// meet in LDS at the end (flash_groups says when).
template <int D, typename TO, bool WIN, int GROUPS>
__global__ __launch_bounds__(FT, flash_waves(D, GROUPS)) void flash_fwd_kernel(const unsigned short* __restrict__ q,
                                                       const unsigned short* __restrict__ k,
                                                       const unsigned short* __restrict__ v, TO* __restrict__ out,
                                                       unsigned short* __restrict__ resid, float* __restrict__ lse,
                                                       FlashShape s, OmxFaultWord* fault, unsigned long long tag) {
  constexpr int NT = FT / GROUPS, ROW_WAVES = 4 / GROUPS, ROWS = 32 * ROW_WAVES;  // threads and waves of a group, rows of a block
  constexpr int KK = D / 16, MT = D / 32, NL = 8 * D / NT;  // d slabs, d blocks of the output, loads per thread and tile
  // Two key / value tile pairs (per group): the next tile is stored while this one is multiplied, so a tile
  // costs one barrier.
  __shared__ __attribute__((aligned(16))) char flash_lds[GROUPS * 4 * ftile(D)];
  const int lane = threadIdx.x & 63, l32 = lane & 31, lg = lane >> 5;
  const int group = GROUPS == 1 ? 0 : wave_index() / ROW_WAVES, wave = GROUPS == 1 ? wave_index() : wave_index() % ROW_WAVES;
  char* const smem = flash_lds + group * (4 * ftile(D));
  const int T = s.time;
  const TileFetch<D, NT> fetch(s.kv.rs, T);
  // Query block j sees j / 2 + 1 key tiles (causal): a workgroup takes a late block and then
  // its mirror image from the front, so every workgroup does the same amount of work and the
  // grid ends without a tail of half-empty compute units.
  const int q_blocks = (T + ROWS - 1) / ROWS;
  int pair;
  long plane;
  if (s.q_single) {  // block rank (0 = the last, heaviest block) in the high part of the index
    pair = static_cast<int>(blockIdx.x) / (s.batch * s.heads);
    plane = static_cast<int>(blockIdx.x) % (s.batch * s.heads);
  } else {
    flash_block_of((q_blocks + 1) / 2, s.batch * s.heads, &pair, &plane);
  }
  for (int pass = 0; pass < (s.q_single ? 1 : 2); ++pass) {
    const int qb = pass == 0 ? q_blocks - 1 - pair : pair;
    if (pass == 1 && qb >= q_blocks - 1 - pair) break;
    const int h = static_cast<int>(plane % s.heads), b = static_cast<int>(plane / s.heads);
    const int kvh = h / s.rep;
    const unsigned short* qp = q + b * s.q.bs + h * s.q.hs;
    const unsigned short* kp = k + b * s.kv.bs + kvh * s.kv.hs;
    const unsigned short* vp = v + b * s.kv.bs + kvh * s.kv.hs;
    const int wave_q0 = qb * ROWS + wave * 32;
    const int q_row = wave_q0 + l32;
    u32x4 qf[KK];
    row_frags<D>(qp, s.q.rs, q_row, T, lg, qf);
    floatx16 o[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) o[mt] = zero16();
    // `lsum` sums the weights as computed (the log-sum-exp, from which the backward pass rebuilds
    // them); `wsum` sums the bf16 copies the matrix units multiply into V (this lane's half of
    // the keys), and the output is divided by that: the output is then an exact weighted mean of
    // value rows, so a component shared by all of them passes through unchanged, and
    // dO . out cancels it against dP = dO . V in the backward pass. Divided by lsum it would
    // come through scaled by (sum of rounded weights) / (sum of weights).
    float m = -INFINITY, lsum = 0.0f, wsum = 0.0f;
    const float scale_log2 = s.scale * LOG2E;
    const int block_q0 = qb * ROWS, block_q1 = min(T - 1, qb * ROWS + ROWS - 1);
    const int kt_first = s.window > 0 ? max(0, block_q0 + 1 - s.window) / 64 : 0;
    const int kt_last = block_q1 / 64;
    // The tiles of this group: kt0, kt0 + GROUPS, ... (a group without one reads the first tile and leaves it).
    const int kt0 = kt_first + group;
    // The next tile's global loads are in flight while the current one is multiplied.
    u32x4 rk[NL], rv[NL];
    fetch.load(kp, min(kt0, kt_last) * 64, rk);
    fetch.load(vp, min(kt0, kt_last) * 64, rv);
    __syncthreads();  // the previous pass's reads of the first pair are done
    tile_store_rows<D, NT>(smem, rk);
    tile_store_rows<D, NT>(smem + ftile(D), rv);
    if (kt0 + GROUPS <= kt_last) {
      fetch.load(kp, (kt0 + GROUPS) * 64, rk);
      fetch.load(vp, (kt0 + GROUPS) * 64, rv);
    }
    // One step of the tile pipeline, taken by every wave for every tile of the block: wait for tile
    // kt's pair, store tile kt + 1 into the other pair, start the loads of tile kt + 2.
    const char* k_rows;
    const char* v_rows;
    auto advance = [&](int kt) {
      const int cur = GROUPS == 1 ? (kt - kt_first) & 1 : (kt - kt0) / GROUPS & 1;
      k_rows = smem + cur * 2 * ftile(D);
      v_rows = k_rows + ftile(D);
      __syncthreads();  // this pair is complete, and every wave is done with the other one
      if (kt + GROUPS <= kt_last) {
        char* next = smem + (cur ^ 1) * 2 * ftile(D);
        tile_store_rows<D, NT>(next, rk);
        tile_store_rows<D, NT>(next + ftile(D), rv);
        if (kt + 2 * GROUPS <= kt_last) {
          fetch.load(kp, (kt + 2 * GROUPS) * 64, rk);
          fetch.load(vp, (kt + 2 * GROUPS) * 64, rv);
        }
      }
    };
    int kt = kt0;
    const int kt_end = kt_last + group;  // every group takes as many steps as the first
    if constexpr (WIN) {
      for (; kt <= kt_end; kt += GROUPS) {
        advance(kt);
        const int key0 = kt * 64;
        if ((GROUPS == 1 || kt <= kt_last) && key0 <= wave_q0 + 31 && key0 + 63 + s.window > wave_q0)
          flash_fwd_tile<D, 2, -1, true, flash_in_turn(D, GROUPS)>(k_rows, v_rows, qf, o, m, lsum, wsum, scale_log2, key0, q_row, T, s.window, lane);
      }
    } else if (wave_q0 < T) {  // (a wave whose rows all lie past the sequence end only keeps the barriers)
      // The wave's first query is a multiple of 32 and a tile's first key a multiple of 64, so the
      // diagonal cuts exactly one 32 x 32 half of one tile, the wave's last: the first half of the tile
      // that starts at the wave's first query (whose second half no row sees), or the second half of
      // the tile that starts 32 keys earlier. The tiles before it need no mask, and their loop holds
      // nothing else: one body, so the accumulators stay in the registers the matrix units update.
      const int diag_kt = wave_q0 / 64;
      for (; kt < diag_kt; kt += GROUPS) {
        advance(kt);
        flash_fwd_tile<D, 2, -1, false, flash_in_turn(D, GROUPS)>(k_rows, v_rows, qf, o, m, lsum, wsum, scale_log2, kt * 64, q_row, T, 0, lane);
      }
      if (GROUPS == 1 || kt == diag_kt) {
        advance(kt);
        const int key0 = kt * 64;
        if (D > 64 || key0 + 63 >= T)  // (at head_dim 128 the two cut-tile forms cost registers the kernel does not have)
          flash_fwd_tile<D, 2, -1, true, flash_in_turn(D, GROUPS)>(k_rows, v_rows, qf, o, m, lsum, wsum, scale_log2, key0, q_row, T, 0, lane);
        else if (key0 == wave_q0)
          flash_fwd_tile<D, 1, 0, false, flash_in_turn(D, GROUPS)>(k_rows, v_rows, qf, o, m, lsum, wsum, scale_log2, key0, q_row, T, 0, lane);
        else
          flash_fwd_tile<D, 2, 1, false, flash_in_turn(D, GROUPS)>(k_rows, v_rows, qf, o, m, lsum, wsum, scale_log2, key0, q_row, T, 0, lane);
        kt += GROUPS;
      }
    }
    for (; kt <= kt_end; kt += GROUPS) advance(kt);  // tiles of the block's later waves (same barrier count for all)
    if constexpr (GROUPS > 1) {
      // The groups' weights and sums, moved to one reference point per row.
      constexpr int PART = (MT * 16 + 3) * 64;  // floats of a wave
      float* const meet = reinterpret_cast<float*>(flash_lds);
      __syncthreads();  // every wave is done with the tiles
      if (group > 0) {
        float* mine = meet + ((group - 1) * ROW_WAVES + wave) * PART + lane;
        mine[0] = m;
        mine[64] = lsum;
        mine[128] = wsum;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int vv = 0; vv < 16; ++vv) mine[(3 + mt * 16 + vv) * 64] = o[mt][vv];
      }
      __syncthreads();
      if (group > 0) return;
      const float* parts[GROUPS - 1];
      float top = m;
#pragma unroll
      for (int g = 0; g < GROUPS - 1; ++g) {
        parts[g] = meet + (g * ROW_WAVES + wave) * PART + lane;
        top = fmaxf(top, parts[g][0]);
      }
      const float neg_top = top == -INFINITY ? 0.0f : -top * scale_log2;
      const float own = __builtin_amdgcn_exp2f(fmaf(m, scale_log2, neg_top));
      lsum *= own;
      wsum *= own;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int vv = 0; vv < 16; ++vv) o[mt][vv] *= own;
#pragma unroll
      for (int g = 0; g < GROUPS - 1; ++g) {
        const float w = __builtin_amdgcn_exp2f(fmaf(parts[g][0], scale_log2, neg_top));
        lsum = fmaf(parts[g][64], w, lsum);
        wsum = fmaf(parts[g][128], w, wsum);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int vv = 0; vv < 16; ++vv) o[mt][vv] = fmaf(parts[g][(3 + mt * 16 + vv) * 64], w, o[mt][vv]);
      }
      m = top;
    }
    wsum = halves_sum(wsum);
    bool bad = false;
    if (q_row < T) {
      bad |= !(dev_finite(lsum) && lsum > 0.0f && wsum > 0.0f);
      if (lg == 0) lse[plane * T + q_row] = m * s.scale + logf(lsum);
    }
    const long o_off = b * s.o.bs + h * s.o.hs;
    if constexpr (sizeof(TO) == 2) {
      if (resid) bad |= store_transposed_acc_split<D>(out + o_off, resid + o_off, s.o.rs, q_row, T, lg, o, 1.0f / wsum);
      else bad |= store_transposed_acc<D, TO>(out + o_off, s.o.rs, q_row, T, lg, o, 1.0f / wsum);
    } else {
      bad |= store_transposed_acc<D, TO>(out + o_off, s.o.rs, q_row, T, lg, o, 1.0f / wsum);
    }
    if (bad) dev_raise_fault(fault, tag);
  }  // pass
}

// ------------------------------------------------------------------ backward: dK, dV
// ---- tiles that go from memory into LDS without passing through registers
// 64 rows of D bf16, unpadded: piece c (16 bytes) of row r in slot c ^ flash_slot(r). The four rows of a transposing read then lie in
// four different quarters of the banks, and a 16-byte read of 32 rows meets every slot as often as any other.
template <int D>
__device__ __forceinline__ constexpr unsigned flash_slot(unsigned r) {
  return D == 128 ? ((r & 3) << 2 | (r >> 2 & 3)) : ((r >> 1 & 1) << 2 | (r >> 2 & 3));
}
typedef __attribute__((address_space(3))) char* LdsBytes;
__device__ __forceinline__ unsigned lds_address(const void* p) { return static_cast<unsigned>(reinterpret_cast<uintptr_t>((LdsBytes)(p))); }
__device__ __forceinline__ u32x4 lds_read16(unsigned at) {
  typedef const u32x4 __attribute__((address_space(3))) * ptr;
  return *reinterpret_cast<ptr>(static_cast<uintptr_t>(at));
}
// A wave's share of a tile's loads: load I moves 1 KiB, WAVES waves take turns.
template <int D, int WAVES>
struct TileDma {
  static constexpr int CPR = D / 8, ROWS = 64 / CPR, LOADS = 64 / (ROWS * WAVES);  // pieces of a row, rows of a load, loads of a wave
  unsigned first, piece, step;  // bytes: the lane's row, its piece of the row, from load to load
  unsigned wave;
  __device__ __forceinline__ TileDma(long rs, int wave_, int lane) : wave(wave_) {
    const unsigned row = wave_ * ROWS + lane / CPR;
    first = row * static_cast<unsigned>(rs * 2);
    piece = (lane % CPR ^ flash_slot<D>(row)) * 16;
    step = WAVES * ROWS * static_cast<unsigned>(rs * 2);
  }
  // The tile that starts at `at`, `rows` of it: what lies past them reads as zeros.
  __device__ __forceinline__ static u32x4 describe(unsigned long long at, unsigned pitch, int rows) {
    const int live = min(64, rows);
    return u32x4{static_cast<unsigned>(at), static_cast<unsigned>(at >> 32) & 0xffffu, live > 0 ? (live - 1) * pitch + D * 2 : 0u, 0x00020000u};
  }
  // (Assembly: the compiler would make every LDS read wait for a load into LDS that it knows of.)
  template <int I>
  __device__ __forceinline__ void load(const u32x4& rsrc, unsigned tile) const {
    const unsigned off = first + I * step + (piece ^ flash_slot<D>(I * WAVES * ROWS) * 16);
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(rsrc),
                 "s"(tile + (I * WAVES + wave) * 1024)
                 : "memory");
  }
  // The same rows through registers, for planes that are not 16-byte aligned.
  __device__ __forceinline__ void copy(const unsigned short* first_row, long rs, int rows, char* tile, int lane) const {
#pragma unroll 1
    for (int i = 0; i < LOADS; ++i) {
      const int row = (i * WAVES + static_cast<int>(wave)) * ROWS + lane / CPR, c = lane % CPR;
      u32x4 x = u32x4{0u, 0u, 0u, 0u};
      if (row < rows) {
        const unsigned short* p = first_row + static_cast<long>(row) * rs + c * 8;
        for (int j = 0; j < 4; ++j) x[j] = p[2 * j] | static_cast<unsigned>(p[2 * j + 1]) << 16;
      }
      *reinterpret_cast<u32x4*>(tile + row * (D * 2) + (c ^ flash_slot<D>(row)) * 16) = x;
    }
  }
};
// Keeps the order of what is written before and after it.
__device__ __forceinline__ void pin() { __builtin_amdgcn_sched_barrier(4); }  // (but for scalar instructions)
// A lane's place in a tile: its row as an operand (frag_rows), and its part of the transposing reads (frag_tr).
template <int D>
struct TilePlace {
  unsigned rows, tr;
  __device__ __forceinline__ explicit TilePlace(int lane) {
    const unsigned l32 = lane & 31, g = lane >> 5, s = lane & 15, half = lane >> 4 & 1, r = 4 * g + (s >> 2);
    rows = l32 * (D * 2) + (g ^ flash_slot<D>(l32)) * 16;
    tr = r * (D * 2) + ((half * 2 + ((s & 3) >> 1)) ^ flash_slot<D>(r)) * 16 + (s & 1) * 8;
  }
  __device__ __forceinline__ u32x4 row(unsigned tile, int sub, int kk) const { return lds_read16(((tile + rows) ^ kk * 32) + sub * 64 * D); }
  __device__ __forceinline__ u32x4 column(unsigned tile, int mt, int sub, int c) const {
    typedef short4v __attribute__((address_space(3))) * ptr;
    const unsigned at = tile + tr, imm = (sub * 32 + c * 16) * D * 2;
    const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<ptr>(static_cast<uintptr_t>((at ^ mt * 64) + imm)));
    const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<ptr>(static_cast<uintptr_t>((at ^ mt * 64 ^ 32) + (imm + 8 * D * 2))));
    const u32x2 a = __builtin_bit_cast(u32x2, lo), b = __builtin_bit_cast(u32x2, hi);
    return u32x4{a.x, a.y, b.x, b.y};
  }
};

// Transposed accumulators of a wave's 32 rows as rows of a [time, D] plane, by way of 32 rows of LDS of the wave's own: whole lines
// leave the wave where lanes of their own rows would store 8 bytes each.
template <int D, typename TO>
__device__ __forceinline__ bool store_acc_rows(TO* __restrict__ plane, long rs, int row0, int time, int lane, const floatx16 (&acc)[D / 32],
                                               float mul, char* stage) {
  constexpr int PITCH = D * sizeof(TO), CPR = PITCH / 16, RPI = 64 / CPR;
  const int l32 = lane & 31, lg = lane >> 5;
  const unsigned slot = flash_slot<128>(l32);
  bool bad = false;
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const float x0 = acc[mt][4 * q4 + 0] * mul, x1 = acc[mt][4 * q4 + 1] * mul, x2 = acc[mt][4 * q4 + 2] * mul,
                  x3 = acc[mt][4 * q4 + 3] * mul;
      bad |= !(dev_finite(x0) && dev_finite(x1) && dev_finite(x2) && dev_finite(x3));
      if constexpr (sizeof(TO) == 2) {
        *reinterpret_cast<uint2*>(stage + l32 * PITCH + ((mt * 4 + q4) ^ (slot & (CPR - 1))) * 16 + lg * 8) = make_uint2(pack2(x0, x1), pack2(x2, x3));
      } else {
        *reinterpret_cast<float4*>(stage + l32 * PITCH + ((mt * 8 + q4 * 2 + lg) ^ slot) * 16) = make_float4(x0, x1, x2, x3);
      }
    }
  bad &= row0 + l32 < time;
#pragma unroll
  for (int i = 0; i < 32 / RPI; ++i) {
    const int r = i * RPI + lane / CPR, c = lane % CPR;
    const u32x4 x = *reinterpret_cast<const u32x4*>(stage + r * PITCH + (c ^ (flash_slot<128>(r) & (CPR - 1))) * 16);
    if (row0 + r < time) *reinterpret_cast<u32x4*>(reinterpret_cast<char*>(plane + static_cast<long>(row0 + r) * rs) + c * 16) = x;
  }
  return bad;
}

// The dK/dV pass of one wave over 32 queries x its 32 keys, in three phases whose order the compiler keeps: scores and dP, the
// transposed operands of the third phase on their way from LDS; P and dS; dV and dK, the next 32 queries on their way.
// The rows' values, log-sum-exp (times log2 e) and delta, are read by every lane for its accumulator's rows: at head_dim 128 with the
// next rows, at 64, where two waves share a SIMD, with the transposed operands.
template <int D>
struct DkvHalf {
  static constexpr int KK = D / 16, MT = D / 32, TILE = 64 * D * 2;
  static constexpr bool EARLY = D == 128;
  u32x4 q[KK], g[KK];  // rows
  u32x4 gt[2][MT], qt[2][MT];
  float4 lse[4], del[4];
  floatx16 sc, dp;
  u32x4 pb[2], dsb[2];
  // Rows `sub` of the set at `set`, piece kk.
  __device__ __forceinline__ void fetch_q(const TilePlace<D>& place, unsigned set, int sub, int kk, int lg) {
    q[kk] = place.row(set, sub, kk);
    if (EARLY && kk < 4) lse[kk] = values(set, sub, kk, lg);
  }
  __device__ __forceinline__ void fetch_g(const TilePlace<D>& place, unsigned set, int sub, int kk, int lg) {
    g[kk] = place.row(set + TILE, sub, kk);
    if (EARLY && kk < 4) del[kk] = values(set + 256, sub, kk, lg);
  }
  __device__ __forceinline__ static float4 values(unsigned set, int sub, int q4, int lg) {
    return __builtin_bit_cast(float4, lds_read16(set + lg * 16 + (2 * TILE + (sub * 32 + 8 * q4) * 4)));
  }
  __device__ __forceinline__ void fetch(const TilePlace<D>& place, unsigned set, int sub, int lg) {
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      fetch_q(place, set, sub, kk, lg);
      fetch_g(place, set, sub, kk, lg);
    }
  }
  __device__ __forceinline__ void scores(const u32x4 (&kf)[KK], const u32x4 (&vf)[KK], const TilePlace<D>& place, unsigned set, int sub, int lg) {
    sc = zero16();
    dp = zero16();
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      sc = mfma(q[kk], kf[kk], sc);
      gt[kk / MT][kk % MT] = place.column(set + TILE, kk % MT, sub, kk / MT);
      if (!EARLY) lse[kk] = values(set, sub, kk, lg);
      pin();
      dp = mfma(g[kk], vf[kk], dp);
      qt[kk / MT][kk % MT] = place.column(set, kk % MT, sub, kk / MT);
      if (!EARLY) del[kk] = values(set + 256, sub, kk, lg);
      pin();
    }
  }
  __device__ __forceinline__ void weights(bool cut, float scale_log2, int q0, int key_row, int T, int window, int lg) {
    if (__builtin_expect(cut, 0)) {
      asm volatile("");  // (a branch: as selects, the test would go with every tile)
#pragma unroll
      for (int vv = 0; vv < 16; ++vv) {
        const int qi = q0 + acc_row(vv, lg);
        const bool masked = key_row > qi || qi >= T || key_row >= T || (window > 0 && key_row + window <= qi);
        sc[vv] = masked ? -INFINITY : sc[vv];
      }
    }
    // P = 2^(s * scale * log2e - lse * log2e); dS / scale = P (dP - delta): the scale joins dK at the end.
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const float lv[4] = {lse[q4].x, lse[q4].y, lse[q4].z, lse[q4].w}, dl[4] = {del[q4].x, del[q4].y, del[q4].z, del[q4].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int vv = 4 * q4 + j;
        const float p = __builtin_amdgcn_exp2f(fmaf(sc[vv], scale_log2, -lv[j]));
        dp[vv] = p * (dp[vv] - dl[j]);
        sc[vv] = p;
      }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      pb[c] = pack8(sc, c);
      dsb[c] = pack8(dp, c);
    }
    pin();
  }
  // `between(i)`, i of KK, after each pair of products.
  template <typename F>
  __device__ __forceinline__ void sums(floatx16 (&dk)[MT], floatx16 (&dv)[MT], const TilePlace<D>& place, unsigned next, int next_sub, int lg,
                                       F between) {
    for_sequence<KK>([&](auto i) {
      constexpr int kk = decltype(i)::value, c = kk / MT, mt = kk % MT;
      dv[mt] = mfma(gt[c][mt], pb[c], dv[mt]);
      fetch_q(place, next, next_sub, kk, lg);
      pin();
      dk[mt] = mfma(qt[c][mt], dsb[c], dk[mt]);
      fetch_g(place, next, next_sub, kk, lg);
      between(i);
      pin();
    });
  }
};

// One key block of one KV head: the loop over the query tiles that see it, accumulating dK and dV for the wave's 32 keys, then their
// stores. head_dim 64: two waves per SIMD; at 128 the two sums (128 registers), keys and values (64) and the operands on their way
// take more than 256 registers, so one wave has its SIMD to itself, and everything it waits for has to be on its way: tiles go straight
// into LDS a tile ahead, operands come from LDS a phase ahead (DkvHalf), rows go out whole lines at a time.
// What bounds it: products and vector work, which do not overlap, about 0.6 of the time; then the first tile and the last rows (5 us a
// workgroup at 128). us, through registers (two walks at 128, scores formed twice) / now: 4 x 16 x 2048 x 128: 221 / 168; 8 x 16 x 1024 x
// 128: 141 / 110; 16 x 12 x 1024 x 64: 83 / 74; 8 x 12 x 1024 x 64: 46 / 42. Waiting for a tile, storing it and asking for the next were
// 1500 of 5900 clocks a tile, the waits for operands 1000. Scores and dP from accumulators that start at the rows' values would save a
// subtraction each (159 and 70 us), in other roundings.
// GROUPS > 1: groups of the waves take the query tiles of 128 / GROUPS keys in turn, as in the forward.
// SPLIT: the tiles of s.kv_parts workgroups are consecutive shares of the sequence over the heads, this one's is `part`, and its sums go
// out as rows of gk and gv, each [part][b, KV head][time][D].
// OWN: delta is formed here, for the rows that see the block, in `own` (FLASH_OWN_ROWS values of LDS).
template <int D, typename TO, int GROUPS, bool SPLIT, bool OWN = false>
__device__ __forceinline__ bool flash_dkv_block(const unsigned short* __restrict__ q,
                                                const unsigned short* __restrict__ k,
                                                const unsigned short* __restrict__ v, const float* __restrict__ lse,
                                                const float* __restrict__ delta, const unsigned short* __restrict__ gy,
                                                TO* __restrict__ gk, TO* __restrict__ gv, const FlashShape& s, char* lds,
                                                int kb, int b, int gidx, int part, const unsigned short* __restrict__ out = nullptr,
                                                const unsigned short* __restrict__ resid = nullptr, float* own = nullptr) {
  constexpr int ROW_WAVES = 4 / GROUPS, ROWS = 32 * ROW_WAVES;
  constexpr int KK = D / 16, MT = D / 32, TILE = 64 * D * 2, SET = flash_dkv_set(D);
  typedef TileDma<D, ROW_WAVES> Dma;
  const int lane = threadIdx.x & 63, l32 = lane & 31, lg = lane >> 5;
  const int group = GROUPS == 1 ? 0 : wave_index() / ROW_WAVES, wave = GROUPS == 1 ? wave_index() : wave_index() % ROW_WAVES;
  char* const smem = lds + group * (2 * SET);
  const unsigned sets = lds_address(smem);
  const int T = s.time;
  const Dma dma_q(s.q.rs, wave, lane), dma_g(s.o.rs, wave, lane);
  const TilePlace<D> place(lane);
  const long kv_off = b * s.kv.bs + gidx * s.kv.hs;
  const int wave_k0 = kb * ROWS + wave * 32;
  const int key_row = wave_k0 + l32;
  const int block_k0 = kb * ROWS, block_k1 = min(T - 1, kb * ROWS + ROWS - 1);
  const int qt_first = block_k0 / 64;
  const int qt_last = (s.window > 0 ? min(T - 1, block_k1 + s.window - 1) : T - 1) / 64;
  // One flat sequence of (query head of the group, query tile), ascending, so that the next tiles can be on their way.
  const int nq = qt_last - qt_first + 1;
  // The workgroup's tiles (none of a late key block's may be left for a late part: its sums are zeros then).
  const int share_at = SPLIT ? static_cast<int>(static_cast<long>(s.rep) * nq * part / s.kv_parts) : 0;
  const int share = (SPLIT ? static_cast<int>(static_cast<long>(s.rep) * nq * (part + 1) / s.kv_parts) : s.rep * nq) - share_at;
  const int r_first = SPLIT ? share_at / nq : 0, qt_start = SPLIT ? qt_first + share_at % nq : qt_first;
  const int steps = (share - group + GROUPS - 1) / GROUPS;  // this group's: GROUPS tiles apart
  // The tile that is loaded next: its head of the group, what is left of that, and where it lies.
  const unsigned pitch_q = static_cast<unsigned>(s.q.rs * 2), pitch_g = static_cast<unsigned>(s.o.rs * 2);
  int next_r = r_first, next_qt = qt_start;
  const unsigned short *next_q, *next_g;
  long next_row;
  auto head = [&]() {
    const long h = static_cast<long>(gidx) * s.rep + min(next_r, s.rep - 1);  // (past the last tile nothing is loaded)
    next_q = q + b * s.q.bs + h * s.q.hs + static_cast<long>(next_qt) * 64 * s.q.rs;
    next_g = gy + b * s.o.bs + h * s.o.hs + static_cast<long>(next_qt) * 64 * s.o.rs;
    next_row = (static_cast<long>(b) * s.heads + h) * T + next_qt * 64;
  };
  auto skip = [&]() {
    next_q += 64 * s.q.rs;
    next_g += 64 * s.o.rs;
    next_row += 64;
    if (++next_qt > qt_last) {
      next_qt = qt_first;
      ++next_r;
      head();
    }
  };
  head();
  for (int i = 0; i < group; ++i) skip();
  // The tile on its way: a lane's row value, two loads a wave where it is the group's only one.
  constexpr int VALUES = ROW_WAVES > 1 ? 1 : 2;
  const int value_of = wave & 1;  // 0: lse, 1: delta (other waves repeat them)
  const unsigned short *coming_q = next_q, *coming_g = next_g;
  int coming_q0 = 0, coming_own = 0;
  float value[VALUES];
  u32x4 rsrc_q, rsrc_g;
  auto aim = [&](bool more) {  // (past the last tile, and of rows that are not 16-byte aligned, which arrive() copies: zeros, nothing is read)
    coming_q = next_q;
    coming_g = next_g;
    coming_q0 = next_qt * 64;
    const int live = more ? s.direct - coming_q0 : 0;
    rsrc_q = Dma::describe(reinterpret_cast<unsigned long long>(next_q), pitch_q, live);
    rsrc_g = Dma::describe(reinterpret_cast<unsigned long long>(next_g), pitch_g, live);
    const long row = next_row + min(lane, T - 1 - coming_q0);  // (what a row past the end carries is masked)
#pragma unroll
    for (int j = 0; j < VALUES; ++j) value[j] = !OWN && (VALUES == 2 ? j : value_of) ? delta[row] : lse[row];
    if constexpr (OWN) coming_own = min(next_r, s.rep - 1) * (T - qt_first * 64) + coming_q0 - qt_first * 64 + min(lane, T - 1 - coming_q0);
    for (int i = 0; i < GROUPS; ++i) skip();
  };
  auto load = [&](auto i, unsigned set) {
    constexpr int I = decltype(i)::value;
    if constexpr (I < Dma::LOADS) dma_q.template load<I>(rsrc_q, set);
    else dma_g.template load<I - Dma::LOADS>(rsrc_g, set + TILE);
  };
  auto load_all = [&](unsigned set) {
    for_sequence<2 * Dma::LOADS>([&](auto i) { load(i, set); });
  };
  // The set that was on its way is complete for this wave, its rows' values with it.
  auto arrive = [&](int set) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (__builtin_expect(s.direct == 0, 0)) {
      dma_q.copy(coming_q, s.q.rs, T - coming_q0, smem + set * SET, lane);
      dma_g.copy(coming_g, s.o.rs, T - coming_q0, smem + set * SET + TILE, lane);
    }
#pragma unroll
    for (int j = 0; j < VALUES; ++j) {
      const int which = VALUES == 2 ? j : value_of;
      if constexpr (OWN)
        if (which) value[j] = own[coming_own];
      *reinterpret_cast<float*>(smem + set * SET + 2 * TILE + which * 256 + lane * 4) = value[j] * (which ? 1.0f : LOG2E);
    }
  };
  auto meet = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    pin();
  };
  __syncthreads();  // an earlier block's reads of LDS are done
  aim(true);
  load_all(sets);
  u32x4 kf[KK], vf[KK];
  row_frags<D>(k + kv_off, s.kv.rs, key_row, T, lg, kf);
  row_frags<D>(v + kv_off, s.kv.rs, key_row, T, lg, vf);
  floatx16 dk[MT], dv[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    dk[mt] = zero16();
    dv[mt] = zero16();
  }
  const float scale_log2 = s.scale * LOG2E;
  if constexpr (OWN) {
    // The rows of tiles qt_first .. qt_last of every head of the group, 32 a wave at a time.
    const int from = qt_first * 64, each = (min(T, qt_last * 64 + 64) - from + 31) / 32;
    for (int n = wave_index(); n < s.rep * each; n += 4) {
      const int r = n / each, row = from + (n - r * each) * 32 + l32;
      const long off = b * s.o.bs + (static_cast<long>(gidx) * s.rep + r) * s.o.hs;
      u32x4 gf[KK];
      row_frags<D>(gy + off, s.o.rs, row, T, lg, gf);
      const float del = flash_row_delta<D>(gf, out + off, resid ? resid + off : nullptr, s.o.rs, row, T, lg);
      if (lg == 0 && row < T) own[r * (T - from) + row - from] = del;
    }
    __syncthreads();
  }
  arrive(0);
  meet();
  aim(steps > 1);
  load_all(sets + SET);
  // A tile of every wave, one barrier each, between its last weights and its last sums: the next tile is complete by then, and this wave
  // has read all it needs of this one, whose set the tile after the next goes into.
  int qt = qt_start;
  auto turn = [&]() {
    if (++qt > qt_last) qt = qt_first;
  };
  for (int i = 0; i < group; ++i) turn();
  const int rounds = (share + GROUPS - 1) / GROUPS;
  DkvHalf<D> half;
  half.fetch(place, sets, 0, lg);
#pragma unroll 1
  for (int i = 0; i < rounds; ++i) {
    const unsigned set = sets + (i & 1) * SET, other = sets + ((i & 1) ^ 1) * SET;
    const int q0 = qt * 64;
    const bool none = GROUPS > 1 && i * GROUPS + group >= share;  // (this group is through: all of it is masked)
    const bool cut = none || q0 < wave_k0 + 32 || q0 + 64 > T || wave_k0 + 31 >= T || (s.window > 0 && q0 + 63 >= wave_k0 + s.window);
    const int from = none ? T : key_row;
    half.scores(kf, vf, place, set, 0, lg);
    half.weights(cut, scale_log2, q0, from, T, s.window, lg);
    half.sums(dk, dv, place, set, 1, lg, [](auto) {});
    half.scores(kf, vf, place, set, 1, lg);
    half.weights(cut, scale_log2, q0 + 32, from, T, s.window, lg);
    arrive((i & 1) ^ 1);
    meet();
    aim(i + 2 < steps);
    pin();
    half.sums(dk, dv, place, other, 0, lg, [&](auto kk) {
      constexpr int EACH = 2 * Dma::LOADS / KK;
      for_sequence<EACH>([&](auto j) { load(std::integral_constant<int, decltype(kk)::value * EACH + decltype(j)::value>{}, set); });
    });
    for (int j = 0; j < GROUPS; ++j) turn();
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();  // every wave is done with the tiles, the last loads into LDS with them
  bool bad = false;
  if constexpr (GROUPS > 1) {
    constexpr int PART = 2 * MT * 16 * 64;  // floats of a wave
    float* const meet = reinterpret_cast<float*>(lds);
    if (group > 0) {
      float* mine = meet + ((group - 1) * ROW_WAVES + wave) * PART + lane;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int vv = 0; vv < 16; ++vv) {
          mine[(mt * 16 + vv) * 64] = dk[mt][vv];
          mine[(MT * 16 + mt * 16 + vv) * 64] = dv[mt][vv];
        }
    }
    __syncthreads();
    if (group > 0) return bad;
#pragma unroll
    for (int g = 0; g < GROUPS - 1; ++g) {
      const float* part = meet + (g * ROW_WAVES + wave) * PART + lane;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int vv = 0; vv < 16; ++vv) {
          dk[mt][vv] += part[(mt * 16 + vv) * 64];
          dv[mt][vv] += part[(MT * 16 + mt * 16 + vv) * 64];
        }
    }
  }
  const long out_off = SPLIT ? ((static_cast<long>(part) * s.batch + b) * s.kv_heads + gidx) * T * D : kv_off, out_rs = SPLIT ? D : s.kv.rs;
  if constexpr (GROUPS > 1) {  // (whole lines, by way of LDS, would wait for it once more and cost 0.5 to 1 us here)
    bad |= store_transposed_acc<D, TO>(gk + out_off, out_rs, key_row, T, lg, dk, s.scale);
    bad |= store_transposed_acc<D, TO>(gv + out_off, out_rs, key_row, T, lg, dv, 1.0f);
  } else {
    char* const stage = lds + wave * (32 * D * static_cast<int>(sizeof(TO)));
    bad |= store_acc_rows<D, TO>(gk + out_off, out_rs, wave_k0, T, lane, dk, s.scale, stage);
    bad |= store_acc_rows<D, TO>(gv + out_off, out_rs, wave_k0, T, lane, dv, 1.0f, stage);
  }
  return bad;
}

template <int D, typename TO, int GROUPS, bool SPLIT>
__global__ __launch_bounds__(FT, flash_dkv_waves(D, GROUPS)) void flash_bwd_dkv_kernel(
    const unsigned short* __restrict__ q, const unsigned short* __restrict__ k, const unsigned short* __restrict__ v,
    const float* __restrict__ lse, const float* __restrict__ delta, const unsigned short* __restrict__ gy,
    TO* __restrict__ gk, TO* __restrict__ gv, FlashShape s, OmxFaultWord* fault, unsigned long long tag) {
  // Two sets of (query tile, gradient tile, 64 log-sum-exp values, 64 row terms): the next set comes
  // while this one is multiplied, so a tile costs one barrier.
  __shared__ __attribute__((aligned(256))) char smem[GROUPS * 2 * flash_dkv_set(D)];
  // Early key blocks are seen by the most queries: a workgroup takes one of them and then its
  // mirror image from the back (see the forward kernel).
  const int k_blocks = (s.time + 128 / GROUPS - 1) / (128 / GROUPS);
  int pair, part = 0;
  long kv_plane;
  if constexpr (SPLIT) {  // (one block per workgroup)
    const int planes = s.batch * s.kv_heads, rest = static_cast<int>(blockIdx.x) % (planes * s.kv_parts);
    pair = static_cast<int>(blockIdx.x) / (planes * s.kv_parts);
    part = rest / planes;
    kv_plane = rest % planes;
  } else if (s.kv_single) {  // block index (0 = the first, heaviest block) in the high part of the index
    pair = static_cast<int>(blockIdx.x) / (s.batch * s.kv_heads);
    kv_plane = static_cast<int>(blockIdx.x) % (s.batch * s.kv_heads);
  } else {
    flash_block_of((k_blocks + 1) / 2, s.batch * s.kv_heads, &pair, &kv_plane);
  }
  const int b = static_cast<int>(kv_plane) / s.kv_heads, gidx = static_cast<int>(kv_plane) - b * s.kv_heads;
  bool bad = false;
  for (int pass = 0; pass < (SPLIT || s.kv_single ? 1 : 2); ++pass) {
    const int kb = pass == 0 ? pair : k_blocks - 1 - pair;
    if (pass == 1 && kb <= pair) break;
    bad |= flash_dkv_block<D, TO, GROUPS, SPLIT>(q, k, v, lse, delta, gy, gk, gv, s, smem, kb, b, gidx, part);
  }
  if (bad) dev_raise_fault(fault, tag);
}

// Adds up the parts of a split dK/dV pass, first tiles first: 8 values of a row a thread. blockIdx.y: 0 dK, 1 dV.
template <int D, typename TO>
__global__ __launch_bounds__(256) void flash_parts_kernel(const float* __restrict__ parts, TO* __restrict__ gk, TO* __restrict__ gv,
                                                          FlashShape s, OmxFaultWord* fault, unsigned long long tag) {
  const long total = static_cast<long>(s.batch) * s.kv_heads * s.time * D, at = (static_cast<long>(blockIdx.x) * 256 + threadIdx.x) * 8;
  if (at >= total) return;
  const float* src = parts + static_cast<long>(blockIdx.y) * s.kv_parts * total + at;
  float4 lo = *reinterpret_cast<const float4*>(src), hi = *reinterpret_cast<const float4*>(src + 4);
#pragma unroll 4
  for (int z = 1; z < s.kv_parts; ++z) {
    const float4 l = *reinterpret_cast<const float4*>(src + z * total), h = *reinterpret_cast<const float4*>(src + z * total + 4);
    lo.x += l.x; lo.y += l.y; lo.z += l.z; lo.w += l.w;
    hi.x += h.x; hi.y += h.y; hi.z += h.z; hi.w += h.w;
  }
  const long row = at / D, plane = row / s.time, b = plane / s.kv_heads;
  TO* dst = (blockIdx.y ? gv : gk) + b * s.kv.bs + (plane - b * s.kv_heads) * s.kv.hs + (row - plane * s.time) * s.kv.rs + (at - row * D);
  if constexpr (sizeof(TO) == 2) {
    *reinterpret_cast<uint2*>(dst) = make_uint2(pack2(lo.x, lo.y), pack2(lo.z, lo.w));
    *reinterpret_cast<uint2*>(dst + 4) = make_uint2(pack2(hi.x, hi.y), pack2(hi.z, hi.w));
  } else {
    *reinterpret_cast<float4*>(dst) = lo;
    *reinterpret_cast<float4*>(dst + 4) = hi;
  }
  if (!(dev_finite(lo.x) && dev_finite(lo.y) && dev_finite(lo.z) && dev_finite(lo.w) && dev_finite(hi.x) && dev_finite(hi.y) &&
        dev_finite(hi.z) && dev_finite(hi.w)))
    dev_raise_fault(fault, tag);
}

// ------------------------------------------------------------------ backward: dQ
// This thread's share of the sum of up to 64 of a head's key rows, evenly spaced in time: part[row group][D]. The dQ pass
// needs a vector close to what the key rows share, not their exact mean (what it does with it is exact for any vector), so
// a sample is enough; every workgroup takes its own (8 KiB out of L2 beside its tiles; a launch of its own before the
// pass cost 2 to 5 us). A thread reads 8 values of a row, 256 / (D / 8) rows go round at once.
template <int D>
__device__ __forceinline__ void key_sample_sum(const unsigned short* __restrict__ kp, long rs, int time, float* part) {
  constexpr int LPR = D / 8, ROWS = FT / LPR;
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // (the sample's addresses, formed ahead of the blocks' loop, would cost the loop registers)
  const int col = (tid % LPR) * 8, first = tid / LPR;
  const int samples = min(time, 64);
  float sum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int n = 0; n < 64 / ROWS; ++n) {
    const int i = first + n * ROWS;
    if (i < samples) {
      const long row = static_cast<long>(i) * time / samples;
      const u32x4 w = *reinterpret_cast<const u32x4*>(kp + row * rs + col);
      const unsigned int ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sum[2 * j] += __uint_as_float(ww[j] << 16);
        sum[2 * j + 1] += __uint_as_float(ww[j] & 0xffff0000u);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) part[first * D + col + i] = sum[i];
}

// One 32-query x 64-key tile of one wave in the dQ pass. GENERAL: the tile crosses the diagonal,
// the sequence end or a window edge and every element is tested (the forward's cheaper forms of
// the cut tile cost registers this kernel does not have: with them it spills, and runs 11 % slower).
// dS / scale = P (dP - delta) goes into dQ^T through the matrix units, and `ds_sum` collects this
// lane's share of the row sum of its bf16 copy.
// IN_TURN as in the forward. At head_dim 64 with one group, in turn / left to the compiler: 8 x 12 x 1024 42.2 / 41.2 us, 16 x 12 x 1024
// 66.9 / 65.8, 8 x 12 x 640 22.0 / 21.6, but 12 x 12 over 3 x 999 53.2 / 55.3: left.
template <int D, bool GENERAL, bool IN_TURN>
__device__ __forceinline__ void flash_dq_tile(const char* k_rows, const char* v_rows, const u32x4 (&qf)[D / 16],
                                              const u32x4 (&gf)[D / 16], floatx16 (&dq)[D / 32], float& ds_sum,
                                              float scale_log2, float neg_lse, float row_del, int key0, int q_row, int T,
                                              int window, int lane) {
  constexpr int KK = D / 16, MT = D / 32;
  const int l32 = lane & 31, lg = lane >> 5;
#pragma unroll
  for (int sub = 0; sub < 2; ++sub) {
    floatx16 sc = zero16(), dp = zero16();
    if constexpr (IN_TURN) {
      in_turn<2 * KK>([&](auto i) { return frag_rows<D>(i.value % 2 ? v_rows : k_rows, sub, i.value / 2, l32, lg); },
                      [&](auto i, const u32x4& f) {
                        if constexpr (i.value % 2 == 0) sc = mfma(f, qf[i.value / 2], sc);
                        else dp = mfma(f, gf[i.value / 2], dp);
                      });
    } else {
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        sc = mfma(frag_rows<D>(k_rows, sub, kk, l32, lg), qf[kk], sc);
        dp = mfma(frag_rows<D>(v_rows, sub, kk, l32, lg), gf[kk], dp);
      }
    }
    if constexpr (GENERAL) {
#pragma unroll
      for (int vv = 0; vv < 16; ++vv) {
        const int key = key0 + sub * 32 + acc_row(vv, lg);
        const bool masked = key > q_row || key >= T || q_row >= T || (window > 0 && key + window <= q_row);
        sc[vv] = masked ? -INFINITY : sc[vv];
      }
    }
#pragma unroll
    for (int vv = 0; vv < 16; ++vv) {
      const float p = __builtin_amdgcn_exp2f(fmaf(sc[vv], scale_log2, neg_lse));
      dp[vv] = p * (dp[vv] - row_del);  // dS / scale: the scale joins dQ at the end
    }
    if constexpr (IN_TURN) {
      u32x4 dsb;
      in_turn<2 * MT>([&](auto i) { return frag_tr<D>(k_rows, i.value % MT, sub, i.value / MT, lane); },
                      [&](auto i, const u32x4& f) {
                        if constexpr (i.value % MT == 0) {
                          dsb = pack8(dp, i.value / MT);
                          ds_sum = sum_pairs(dsb.x, sum_pairs(dsb.y, sum_pairs(dsb.z, sum_pairs(dsb.w, ds_sum))));
                        }
                        dq[i.value % MT] = mfma(f, dsb, dq[i.value % MT]);
                      });
    } else {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const u32x4 dsb = pack8(dp, c);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) dq[mt] = mfma(frag_tr<D>(k_rows, mt, sub, c, lane), dsb, dq[mt]);
        ds_sum = sum_pairs(dsb.x, sum_pairs(dsb.y, sum_pairs(dsb.z, sum_pairs(dsb.w, ds_sum))));
      }
    }
  }
}

// A workgroup's blocks of the dQ pass: a late query block, then its mirror image from the front (see the forward kernel). `lds` holds
// flash_dq_lds bytes; the mean key behind the tiles.
template <int D, typename TO, bool WIN, int GROUPS>
__device__ __forceinline__ void flash_dq_blocks(
    const unsigned short* __restrict__ q, const unsigned short* __restrict__ k, const unsigned short* __restrict__ v,
    const unsigned short* __restrict__ out, const unsigned short* __restrict__ resid, const float* __restrict__ lse,
    float* __restrict__ delta, const unsigned short* __restrict__ gy, TO* __restrict__ gq, const FlashShape& s, char* flash_lds, int pair, long plane,
    OmxFaultWord* fault, unsigned long long tag) {
  constexpr int NT = FT / GROUPS, ROW_WAVES = 4 / GROUPS, ROWS = 32 * ROW_WAVES;
  constexpr int KK = D / 16, MT = D / 32, NL = 8 * D / NT;
  const int lane = threadIdx.x & 63, l32 = lane & 31, lg = lane >> 5;
  const int group = GROUPS == 1 ? 0 : wave_index() / ROW_WAVES, wave = GROUPS == 1 ? wave_index() : wave_index() % ROW_WAVES;
  // Two key / value tile pairs (per group), as in the forward: one barrier per tile.
  char* const smem = flash_lds + group * (4 * ftile(D));
  float* const mean_key = reinterpret_cast<float*>(flash_lds + GROUPS * 4 * ftile(D));
  const int T = s.time;
  const TileFetch<D, NT> fetch(s.kv.rs, T);
  const int q_blocks = (T + ROWS - 1) / ROWS;
  for (int pass = 0; pass < (s.q_single ? 1 : 2); ++pass) {
    const int qb = pass == 0 ? q_blocks - 1 - pair : pair;
    if (pass == 1 && qb >= q_blocks - 1 - pair) break;
    const int h = static_cast<int>(plane % s.heads), b = static_cast<int>(plane / s.heads);
    const int kvh = h / s.rep;
    const unsigned short* kp = k + b * s.kv.bs + kvh * s.kv.hs;
    const unsigned short* vp = v + b * s.kv.bs + kvh * s.kv.hs;
    const int wave_q0 = qb * ROWS + wave * 32;
    const int q_row = wave_q0 + l32;
    u32x4 qf[KK], gf[KK];
    row_frags<D>(q + b * s.q.bs + h * s.q.hs, s.q.rs, q_row, T, lg, qf);
    row_frags<D>(gy + b * s.o.bs + h * s.o.hs, s.o.rs, q_row, T, lg, gf);
    // delta = dO . O of this lane's row: each half-wave holds half of the row's values. The
    // dK/dV pass, launched after this one, reads it back from `delta`. dS = P (dP - delta) sums to
    // zero along a row only as far as delta matches sum_j P dP: taken from the bf16 output alone it
    // is off by 2^-9 of |dO| |O|, which a component shared by all value rows (and by all key rows,
    // in dQ = dS K) turns into a multiple of the gradient itself. With the saved rounding residual
    // of the output the mismatch drops to 2^-17.
    const long o_off = b * s.o.bs + h * s.o.hs;
    const float row_del = flash_row_delta<D>(gf, out + o_off, resid ? resid + o_off : nullptr, s.o.rs, q_row, T, lg);
    float row_lse = 0.0f;
    bool bad = false;
    if (q_row < T) {
      row_lse = lse[plane * T + q_row];
      if (delta && lg == 0 && group == 0) delta[plane * T + q_row] = row_del;
      bad |= !(dev_finite(row_lse) && dev_finite(row_del));
    }
    const float neg_lse = -row_lse * LOG2E;
    floatx16 dq[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) dq[mt] = zero16();
    // A row of dS sums to zero, so dQ = dS K does not see a vector added to every key row. The
    // bf16 copy of dS that the matrix units read sums to its rounding error instead, and that
    // error times a component shared by all key rows (a residual stream grows one) lands in dQ at
    // 2^-9 of the component, however small the part of K that varies. `ds_sum` collects this
    // lane's share of the row sum of the rounded dS; the end takes (row sum) x (mean key) off.
    float ds_sum = 0.0f;
    const float scale_log2 = s.scale * LOG2E;
    const int block_q0 = qb * ROWS, block_q1 = min(T - 1, qb * ROWS + ROWS - 1);
    const int kt_first = s.window > 0 ? max(0, block_q0 + 1 - s.window) / 64 : 0;
    const int kt_last = block_q1 / 64;
    const int kt0 = kt_first + group, kt_end = kt_last + group;  // the group's tiles, as in the forward
    u32x4 rk[NL], rv[NL];
    fetch.load(kp, min(kt0, kt_last) * 64, rk);
    fetch.load(vp, min(kt0, kt_last) * 64, rv);
    if (pass == 0) {  // (both blocks of a workgroup lie in one plane)
      float* const part = reinterpret_cast<float*>(flash_lds + 2 * ftile(D));  // the first group's second pair, still unused
      static_assert(FT / (D / 8) * D * 4 <= 2 * ftile(D), "the sample's partial sums fit");
      key_sample_sum<D>(kp, s.kv.rs, T, part);
      __syncthreads();
      if (threadIdx.x < D) {
        float total = 0.0f;
#pragma unroll
        for (int r = 0; r < FT / (D / 8); ++r) total += part[r * D + threadIdx.x];
        mean_key[threadIdx.x] = total / static_cast<float>(min(T, 64));
      }
    }
    __syncthreads();  // the previous pass's reads of the first pair are done
    tile_store_rows<D, NT>(smem, rk);
    tile_store_rows<D, NT>(smem + ftile(D), rv);
    if (kt0 + GROUPS <= kt_last) {
      fetch.load(kp, (kt0 + GROUPS) * 64, rk);
      fetch.load(vp, (kt0 + GROUPS) * 64, rv);
    }
    // The tile pipeline and the split into unmasked tiles, the wave's diagonal tile and the other
    // waves' tiles are the forward kernel's.
    const char* k_rows;
    const char* v_rows;
    auto advance = [&](int kt) {
      const int cur = GROUPS == 1 ? (kt - kt_first) & 1 : (kt - kt0) / GROUPS & 1;
      k_rows = smem + cur * 2 * ftile(D);
      v_rows = k_rows + ftile(D);
      __syncthreads();  // this pair is complete, and every wave is done with the other one
      if (kt + GROUPS <= kt_last) {
        char* next = smem + (cur ^ 1) * 2 * ftile(D);
        tile_store_rows<D, NT>(next, rk);
        tile_store_rows<D, NT>(next + ftile(D), rv);
        if (kt + 2 * GROUPS <= kt_last) {
          fetch.load(kp, (kt + 2 * GROUPS) * 64, rk);
          fetch.load(vp, (kt + 2 * GROUPS) * 64, rv);
        }
      }
    };
    int kt = kt0;
    if constexpr (WIN) {
      for (; kt <= kt_end; kt += GROUPS) {
        advance(kt);
        const int key0 = kt * 64;
        if ((GROUPS == 1 || kt <= kt_last) && key0 <= wave_q0 + 31 && key0 + 63 + s.window > wave_q0)
          flash_dq_tile<D, true, flash_in_turn(D, GROUPS)>(k_rows, v_rows, qf, gf, dq, ds_sum, scale_log2, neg_lse, row_del, key0, q_row, T, s.window,
                                 lane);
      }
    } else if (wave_q0 < T) {
      const int diag_kt = wave_q0 / 64;
      for (; kt < diag_kt; kt += GROUPS) {
        advance(kt);
        flash_dq_tile<D, false, flash_in_turn(D, GROUPS)>(k_rows, v_rows, qf, gf, dq, ds_sum, scale_log2, neg_lse, row_del, kt * 64, q_row, T, 0, lane);
      }
      if (GROUPS == 1 || kt == diag_kt) {
        advance(kt);
        flash_dq_tile<D, true, flash_in_turn(D, GROUPS)>(k_rows, v_rows, qf, gf, dq, ds_sum, scale_log2, neg_lse, row_del, kt * 64, q_row, T, 0, lane);
        kt += GROUPS;
      }
    }
    for (; kt <= kt_end; kt += GROUPS) advance(kt);  // tiles of the block's later waves (same barrier count for all)
    if constexpr (GROUPS > 1) {
      constexpr int PART = (MT * 16 + 1) * 64;
      float* const meet = reinterpret_cast<float*>(flash_lds);
      __syncthreads();  // every wave is done with the tiles
      if (group > 0) {
        float* mine = meet + ((group - 1) * ROW_WAVES + wave) * PART + lane;
        mine[0] = ds_sum;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int vv = 0; vv < 16; ++vv) mine[(1 + mt * 16 + vv) * 64] = dq[mt][vv];
      }
      __syncthreads();
      if (group > 0) return;
#pragma unroll
      for (int g = 0; g < GROUPS - 1; ++g) {
        const float* part = meet + (g * ROW_WAVES + wave) * PART + lane;
        ds_sum += part[0];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int vv = 0; vv < 16; ++vv) dq[mt][vv] += part[(1 + mt * 16 + vv) * 64];
      }
    }
    {
      const float row_sum = halves_sum(ds_sum);  // the two half-waves hold half the keys each
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const float4 m = *reinterpret_cast<const float4*>(mean_key + mt * 32 + 8 * q4 + 4 * lg);
          dq[mt][4 * q4 + 0] = fmaf(-row_sum, m.x, dq[mt][4 * q4 + 0]);
          dq[mt][4 * q4 + 1] = fmaf(-row_sum, m.y, dq[mt][4 * q4 + 1]);
          dq[mt][4 * q4 + 2] = fmaf(-row_sum, m.z, dq[mt][4 * q4 + 2]);
          dq[mt][4 * q4 + 3] = fmaf(-row_sum, m.w, dq[mt][4 * q4 + 3]);
        }
    }
    bad |= store_transposed_acc<D, TO>(gq + b * s.q.bs + h * s.q.hs, s.q.rs, q_row, T, lg, dq, s.scale);
    if (bad) dev_raise_fault(fault, tag);
  }  // pass
}

template <int D, typename TO, bool WIN, int GROUPS>
__global__ __launch_bounds__(FT, flash_waves(D, GROUPS)) void flash_bwd_dq_kernel(
    const unsigned short* __restrict__ q, const unsigned short* __restrict__ k, const unsigned short* __restrict__ v,
    const unsigned short* __restrict__ out, const unsigned short* __restrict__ resid, const float* __restrict__ lse,
    float* __restrict__ delta, const unsigned short* __restrict__ gy, TO* __restrict__ gq, FlashShape s, OmxFaultWord* fault, unsigned long long tag) {
  __shared__ __attribute__((aligned(16))) char flash_lds[flash_dq_lds(D, GROUPS)];
  int pair;
  long plane;
  if (s.q_single) {  // block rank (0 = the last, heaviest block) in the high part of the index
    pair = static_cast<int>(blockIdx.x) / (s.batch * s.heads);
    plane = static_cast<int>(blockIdx.x) % (s.batch * s.heads);
  } else {
    flash_block_of((s.time + 256 / GROUPS - 1) / (256 / GROUPS), s.batch * s.heads, &pair, &plane);
  }
  flash_dq_blocks<D, TO, WIN, GROUPS>(q, k, v, out, resid, lse, delta, gy, gq, s, flash_lds, pair, plane, fault, tag);
}

// Both passes in one launch (flash_together says when): the key side's workgroups, which form delta themselves, then the dQ pass's. Every
// block is a workgroup's of its own (s.q_single, s.kv_single). The dQ pass's windowed form also serves calls without a window.
template <int D, typename TO, int GROUPS>
__global__ __launch_bounds__(FT, flash_dkv_waves(D, GROUPS)) void flash_bwd_kernel(
    const unsigned short* __restrict__ q, const unsigned short* __restrict__ k, const unsigned short* __restrict__ v,
    const unsigned short* __restrict__ out, const unsigned short* __restrict__ resid, const float* __restrict__ lse,
    const unsigned short* __restrict__ gy, TO* __restrict__ gq, TO* __restrict__ gk, TO* __restrict__ gv, FlashShape s, OmxFaultWord* fault,
    unsigned long long tag) {
  constexpr int KEY_LDS = GROUPS * 2 * flash_dkv_set(D) + FLASH_OWN_ROWS * 4;
  __shared__ __attribute__((aligned(256))) char lds[KEY_LDS > flash_dq_lds(D, GROUPS) ? KEY_LDS : flash_dq_lds(D, GROUPS)];
  const int blocks = (s.time + 128 / GROUPS - 1) / (128 / GROUPS), kv_planes = s.batch * s.kv_heads, q_planes = s.batch * s.heads;
  const int index = static_cast<int>(blockIdx.x);
  if (index < blocks * kv_planes) {
    const int kb = index / kv_planes, plane = index - kb * kv_planes, b = plane / s.kv_heads;
    const bool bad = flash_dkv_block<D, TO, GROUPS, false, true>(q, k, v, lse, nullptr, gy, gk, gv, s, lds, kb, b, plane - b * s.kv_heads, 0, out, resid,
                                                                 reinterpret_cast<float*>(lds + GROUPS * 2 * flash_dkv_set(D)));
    if (bad) dev_raise_fault(fault, tag);
  } else {
    const int n = index - blocks * kv_planes, pair = n / q_planes;
    flash_dq_blocks<D, TO, true, GROUPS>(q, k, v, out, resid, lse, nullptr, gy, gq, s, lds, pair, n - pair * q_planes, fault, tag);
  }
}

// `strides`: nine element strides (row, head, batch of q; of k / v; of out), or null for
// contiguous [batch, heads, time, dim] tensors.
FlashShape make_shape(uint64_t batch, uint64_t heads, uint64_t kv_heads, uint64_t time, uint64_t dim, uint64_t window,
                      float scale, const long* strides) {
  FlashShape s;
  const long T = static_cast<long>(time), FD = static_cast<long>(dim);
  s.q = {FD, T * FD, static_cast<long>(heads) * T * FD};
  s.kv = {FD, T * FD, static_cast<long>(kv_heads) * T * FD};
  s.o = s.q;
  if (strides) {
    s.q = {strides[0], strides[1], strides[2]};
    s.kv = {strides[3], strides[4], strides[5]};
    s.o = {strides[6], strides[7], strides[8]};
  }
  s.batch = static_cast<int>(batch);
  s.heads = static_cast<int>(heads);
  s.kv_heads = static_cast<int>(kv_heads);
  s.time = static_cast<int>(time);
  s.window = static_cast<int>(window);
  s.rep = static_cast<int>(heads / kv_heads);
  s.q_single = s.kv_single = 0;
  s.kv_parts = 1;
  s.direct = 0;
  s.scale = scale;
  return s;
}

// Whether a pass takes one block per workgroup: when the mirrored pairs are no more than the chip's
// workgroup places (`per_cu` per compute unit), twice as many workgroups fill them, and where the
// pairs fill the places exactly the lighter blocks still help: a compute unit serves its oldest
// workgroup first, so equal workgroups that start together end one after another (30, 38 and 45 us
// measured for the three of a unit), and the light blocks of the second half fill that tail
// (forward 43.2 -> 42.1 us at 768 pairs). Over a few rounds of places pairs end with a round that runs part empty, where single blocks
// go out heaviest first: up to `rounds` of them. Beyond, a plane's blocks, which single ones spread over the whole grid, find its
// tiles in an L2 no longer. us of pairs and of single blocks, forward / dQ, by how often the pairs fill the places: head_dim 128, 96 planes
// x 1500 (1.12) 117, 93 / 157, 139; 117 x 1177 (1.14) 98, 80 / 125, 110; 256 x 700 (1.5) 72, 71 / 96, 102; 200 x 900 (1.56) 92, 85 / 137,
// 121; 144 x 1500 (1.69) 125, 119 / 186, 167; 117 x 2048 (1.83) 181, 187 / 256, 254; 256 x 900 (2) 97, 113 / 146, 153; head_dim 64, 200 x
// 900 (1.04) 58, 45 / 78, 65; 384 x 531 (1.5) 43, 38 / 63, 54; 512 x 700 (2) 70, 69 / 106, 108; 200 x 2048 (2.08) 167, 152 / 229, 218; 256 x
// 2048 (2.67) 199, 215 / 311, 300.
// dK/dV (two places a unit) of pairs and of single blocks: head_dim 128, 200 x 2048 (3.1) 590, 599; 256 x 2048 (4) 738, 765; 512 x 1177
// (5) 624, 668; under four blocks, whose pairs are uneven, 1024 x 260 228, 195; head_dim 64 the same everywhere (512 x 1500 437, 435), and
// 100, 86 at 1024 x 260.
int flash_single(omx_ctx* ctx, unsigned pair_groups, int per_cu, double rounds) {
  if (ctx->flash_schedule != 0) return ctx->flash_schedule == 2 ? 0 : 1;  // forced (tests cover both)
  return pair_groups <= (ctx->cu_count > 0 ? ctx->cu_count : 256) * per_cu * rounds ? 1 : 0;
}

// f(integral_constant) of a group count the kernels of head dim D are compiled for.
template <int D, typename F>
void for_groups(int groups, F&& f) {
  if (groups == 1) return f(std::integral_constant<int, 1>{});
  if constexpr (D == 64) {
    if (groups == 4) return f(std::integral_constant<int, 4>{});
  }
  f(std::integral_constant<int, 2>{});
}

// How many groups of waves share the 64-row tiles that a row block walks (`tiles`: the most of them; `planes` of `time` rows).
// A block's tiles are a chain, 0.9 us each where a wave has its SIMD to itself, and a causal block's neighbours are done
// before the heaviest one. Two groups of 64 rows a workgroup halve the chain and double the workgroups, four of 32 rows do
// so again, while the chip has places for them: the groups' tiles take 72 and 144 KiB of LDS (two and one workgroups per
// compute unit, at head_dim 128 one), and a tile serves 64 or 32 rows instead of 128, so a full chip loses by them (batch 16
// of 12 heads x 1024: 47 -> 62 us). Where the places are taken once over, the chains' skew still pays for a round or so more.
// us with 1 / 2 / 4 groups, forward: 12 heads x 2048: 33 / 24 / 33; 8 x 1024: 18.5 / 13.2 / 11.2; 7 x 8 x 500: 12.2 / 10.5 / 23;
// 96 x 360: 11.8 / 13.6 / 33; backward of 8 heads over 2 key heads x 777, batch 2: 114 / 72 / 63. Over 187 shapes (558 passes) the rule
// is 0.5 % behind the best count on average, 12 % ahead of one group.
int flash_groups(omx_ctx* ctx, unsigned planes, int time, int tiles, bool window, int dim) {
  const int most = dim == 64 ? 4 : 2;
  if (ctx->flash_schedule >= 3) return std::min(most, ctx->flash_schedule == 3 ? 2 : 4);  // forced
  if (ctx->flash_schedule != 0 || tiles < 2) return 1;
  const long units = ctx->cu_count > 0 ? ctx->cu_count : 256;
  const long two = static_cast<long>(planes) * ((time + 63) / 64), four = static_cast<long>(planes) * ((time + 31) / 32);
  const int skew = window ? 0 : tiles;
  if (dim == 128) return two <= units || (two <= 2 * units && skew >= 12) ? 2 : 1;
  if ((four <= units && tiles >= 4) || (four <= 2 * units && skew >= 24)) return 4;
  return two <= 2 * units || (two <= 3 * units && skew >= 12) || (two <= 4 * units && skew >= 32) ? 2 : 1;
}

// The most 64-row tiles that a 128-row block walks.
int flash_tiles(const FlashShape& s) {
  return ((s.window > 0 && s.window < s.time - 127 ? s.window + 127 : s.time) + 63) / 64;
}

template <int D>
void launch_forward(omx_ctx* ctx, const unsigned short* q, const unsigned short* k, const unsigned short* v, void* out,
                    int32_t out_dtype, void* out_residual, float* lse, const FlashShape& shape, unsigned long long tag) {
  FlashShape s = shape;
  // Two 128-row query blocks per workgroup (see the kernel), or one when the pairs would not fill
  // the chip's workgroup places.
  const unsigned q_blocks = static_cast<unsigned>((s.time + 127) / 128), planes = static_cast<unsigned>(s.batch * s.heads);
  const int tiles = flash_tiles(s);
  // Head dim 128: from 12 tiles on (16 heads x 1024: 32 -> 23 us). A group rounds its probabilities against its own running maximum and not
  // the row's, which is another rounding of the same width: gradients of adapters against 64 bits keep their error normwise (1.00 of
  // one group's, 0.99 to 1.01, over 54 models of 512 to 2048 columns and 512 to 2048 positions), while which element is the worst is
  // chance (two groups / one: 0.81 to 1.28). At 2048 columns it is 0.99 on average from 768 positions on, but 1.03 to 1.10 on each of four
  // models over 512, so there, where groups gain 0.4 to 4 us (16 heads x 128 / 512: 8.4 -> 8.0, 18.8 -> 14.6), one group stays.
  const int groups = D == 128 && tiles < 12 && ctx->flash_schedule == 0 ? 1 : flash_groups(ctx, planes, s.time, tiles, s.window > 0, D);
  s.q_single = groups > 1 || flash_single(ctx, (q_blocks + 1) / 2 * planes, D == 64 ? 3 : 2, D == 64 ? 2.25 : 1.75);
  const unsigned rows = 128 / groups;
  dim3 grid((s.q_single ? (s.time + rows - 1) / rows : (q_blocks + 1) / 2) * planes), block(FT);
  // Causal-counted work: half of the 4 B H T^2 D of the two full products.
  OmxKernelTimer timer(ctx, OMX_K_FLASH_FWD, 2.0 * s.batch * s.heads * static_cast<double>(s.time) * s.time * D);
  auto go = [&](auto kernel, auto* out_ptr, unsigned short* resid_ptr) {
    omx_launch_timed(ctx, kernel, grid, block, 0, timer.start(), timer.stop(), q, k, v, out_ptr, resid_ptr, lse, s,
                     ctx->fault, tag);
  };
  unsigned short* resid = static_cast<unsigned short*>(out_residual);
  auto with_groups = [&](auto count) {
    constexpr int G = decltype(count)::value;
    if (out_dtype == OMX_BF16) {
      if (s.window > 0) go(flash_fwd_kernel<D, unsigned short, true, G>, static_cast<unsigned short*>(out), resid);
      else go(flash_fwd_kernel<D, unsigned short, false, G>, static_cast<unsigned short*>(out), resid);
    } else {
      if (s.window > 0) go(flash_fwd_kernel<D, float, true, G>, static_cast<float*>(out), static_cast<unsigned short*>(nullptr));
      else go(flash_fwd_kernel<D, float, false, G>, static_cast<float*>(out), static_cast<unsigned short*>(nullptr));
    }
  };
  for_groups<D>(groups, with_groups);
}

// How the key side's pass is cut: groups of waves that take a key block's query tiles in turn (flash_groups), and parts, consecutive shares of
// those tiles on workgroups of their own, whose f32 sums go through scratch to a second launch that adds them in order. The pass has a
// workgroup per key block and KV head, so few KV heads leave units idle however many query heads there are, and a workgroup walks the
// tiles of all of them, 1.3 to 1.9 us apiece. Parts are taken where an estimate says that they gain a tenth: the root of the squares of the
// longest walk and of the chip's work, per key block of 128, 64 or 32 keys, fitted to 32 shapes x 3 group counts x 8 part counts (rms 9
// to 12 %); the second launch takes 4.5 us or 2 us and 0.14 us a megabyte. Over those shapes the choice takes 1.5 % more than the
// best of all counts on average, 13 % at most. us of the pass, one group and part / by the rule: 10 x 13 heads over one x 670: 207 /
// 45; 2 x 8 over 2 x 1024 x 128: 125 / 38; 8 over 2 x 291 x 128: 54 / 29; 12 x 2048: 43 / 31; 8 x 1024: 25 / 15; many planes (8 x 12
// x 1024: 44) stay whole.
struct FlashKeyPlan {
  int groups, parts, whole_groups;  // whole_groups: without parts
};
FlashKeyPlan flash_key_plan(omx_ctx* ctx, const FlashShape& s, int dim) {
  const long units = ctx->cu_count > 0 ? ctx->cu_count : 256, planes = static_cast<long>(s.batch) * s.kv_heads;
  if (ctx->flash_schedule != 0) {  // forced (tests)
    const int groups = ctx->flash_schedule < 3 ? 1 : std::min(dim == 64 ? 4 : 2, ctx->flash_schedule == 3 ? 2 : 4);
    return {groups, std::max(1, ctx->flash_kv_parts), groups};
  }
  const int whole_groups = flash_groups(ctx, static_cast<unsigned>(planes), s.time, static_cast<int>(std::min<long>(static_cast<long>(flash_tiles(s)) * s.rep, 1 << 20)),
                                        s.window > 0, dim);
  if (ctx->flash_kv_parts || planes * ((s.time + 127) / 128) >= 2 * units) return {whole_groups, std::max(1, ctx->flash_kv_parts), whole_groups};
  struct Fit {
    double first, step, work, each;  // us: of a workgroup, of a tile on its way; of a unit's tiles, of a unit's workgroups
  };
  const Fit fits[2][3] = {{{9.5, 1.33, 0.60, 4.2}, {9.4, 1.42, 0.83, 4.0}, {8.7, 1.81, 1.55, 7.55}}, {{13.2, 1.82, 1.85, 9.6}, {13.6, 1.90, 1.92, 10.0}, {}}};
  const double megabytes = 8e-6 * static_cast<double>(planes) * s.time * dim;
  double whole = 1e30, least = 1e30;
  FlashKeyPlan plan = {whole_groups, 1, whole_groups};
  for (int shift = 0; shift < (dim == 64 ? 3 : 2); ++shift) {
    const int g = 1 << shift, rows = 128 / g, blocks = (s.time + rows - 1) / rows;
    const Fit& f = fits[dim == 128][shift];
    long all = 0, most = 0;
    for (int kb = 0; kb < blocks; ++kb) {
      const int last = s.window > 0 ? std::min<long>(s.time - 1, std::min(s.time - 1, kb * rows + rows - 1) + static_cast<long>(s.window) - 1) : s.time - 1;
      const long tiles = static_cast<long>(s.rep) * (last / 64 - kb * rows / 64 + 1);
      all += tiles;
      most = std::max(most, tiles);
    }
    for (const int p : {1, 2, 3, 4, 6, 8, 12, 16, 24}) {
      if (p > 1 && (p > most || p * megabytes > 256.0)) break;
      const double groups_of_units = static_cast<double>(blocks * planes * p) / static_cast<double>(units);
      const double walk = f.first + f.step * static_cast<double>((most + p * g - 1) / (p * g));
      const double work = f.work * (static_cast<double>(all * planes) / static_cast<double>(g * units) + (p * g > 1 ? 0.5 * groups_of_units : 0.0)) + f.each * groups_of_units;
      const double us = std::sqrt(walk * walk + work * work) + (p > 1 ? std::max(4.5, 2.0 + 0.14 * megabytes * p) : 0.0);
      if (p == 1) whole = std::min(whole, us);
      if (p > 1 && us < least) {
        least = us;
        plan.groups = g;
        plan.parts = p;
      }
    }
  }
  if (least >= 0.9 * whole) plan = {whole_groups, 1, whole_groups};
  return plan;
}

// Whether the two passes of the backward share a launch, and then how many groups of waves take a block's tiles (0: two launches). Each
// pass alone is a chain: a launch, loads, tiles of 0.9 us and more, a store; over few tiles, with places for the workgroups of both, the
// chains run side by side. us of a backward, two launches / one: 8 x 12 heads x 64: 14.7 / 8.1, 96 planes x 128 18.4 / 11.3, x 256 25.2 / 21.0;
// 2 x 8 x 512 22.9 / 16.9; 10 x 3 x 320 23.1 / 16.3; head_dim 128: 4 x 8 x 64 20.8 / 12.0, x 256 30.8 / 20.2, x 640 59 / 43. Groups by an
// estimate of the form of flash_key_plan's, fitted to 412 timings (rms 6 to 9 %); over 126 shapes the choice among one launch and two
// takes 0.7 % more than the best of all, 22 % less than two launches. Left to two: many workgroups, where the dQ pass alone has three
// per compute unit (16 x 16 x 256: 32.6 / 36.3; head_dim 128, 13 x 12 x 256: 53 / 54, x 512 101 / 131), and many query heads over a KV
// head, whose tiles one workgroup walks (6 x 12 over 3 x 256: 29.1 / 29.7; the parts of flash_key_plan take those).
// Under a window of at most 129 keys no workgroup walks far, however long the sequence, and one launch stays ahead with more of them: 8 x 12
// heads, window 100, x 640 41 / 36; window 64, x 1000 49 / 46; 16 x 16, window 128, x 260 44 / 42; head_dim 128, 8 x 12, window 100, x 256
// 42 / 36; x 320 (2.25 blocks a unit) 44 / 44.
// Gradients over what the other pass still reads take two launches too, as they always could.
int flash_together(omx_ctx* ctx, const FlashShape& s, int dim, const void* q, const void* k, const void* v, const void* out, const void* resid,
                   const void* gy, const void* gq, const void* gk, const void* gv) {
  if (ctx->attention_together == 0 || static_cast<long>(s.rep) * s.time > FLASH_OWN_ROWS) return 0;
  const long units = ctx->cu_count > 0 ? ctx->cu_count : 256, planes = static_cast<long>(s.batch) * (s.kv_heads + s.heads);
  if (planes * ((s.time + 31) / 32) > 0x7fffffffl) return 0;
  const int tiles = flash_tiles(s);
  if (ctx->attention_together < 0) {
    if (ctx->flash_schedule != 0) return 0;  // (a forced cut is that of two launches)
    const long ones = (s.time + 127) / 128 * planes, fours = (s.time + 31) / 32 * planes;
    const bool few = dim == 64 ? (tiles <= 13 && 8 * ones <= 25 * units && (s.rep == 1 || s.rep * tiles <= 16)) || (s.rep == 1 && fours <= units)
                               : (ones <= units || (tiles >= 5 && 8 * ones <= 15 * units)) && (s.rep == 1 || s.rep * tiles <= 12);
    const bool narrow = s.window > 0 && tiles <= 4 && s.rep == 1 && 2 * ones <= (dim == 64 ? 12 : 3) * units;
    if (!few && !narrow) return 0;
  }
  struct Range {
    const char *first, *end;
  };
  auto range = [&](const void* p, const FlashStrides& t, long n) {
    const char* first = static_cast<const char*>(p);
    return Range{first, first + 2 * ((s.batch - 1) * t.bs + (n - 1) * t.hs + (s.time - 1) * t.rs + dim)};
  };
  const Range read[] = {range(q, s.q, s.heads), range(k, s.kv, s.kv_heads), range(v, s.kv, s.kv_heads), range(out, s.o, s.heads),
                        range(gy, s.o, s.heads), range(resid ? resid : out, s.o, s.heads)};
  const Range written[] = {range(gq, s.q, s.heads), range(gk, s.kv, s.kv_heads), range(gv, s.kv, s.kv_heads)};
  for (const Range& r : read)
    for (const Range& w : written)
      if (r.first < w.end && w.first < r.end) return 0;
  const int most = dim == 64 ? 4 : 2;
  if (ctx->flash_schedule != 0) return ctx->flash_schedule < 3 ? 1 : std::min(most, ctx->flash_schedule == 3 ? 2 : 4);
  struct Fit {
    double first, step, work, each;  // us: of a workgroup, of a tile on its way; of a unit's tiles, of a unit's workgroups
  };
  const Fit fits[2][3] = {{{6.1, 2.1, 1.26, 4.0}, {7.1, 2.4, 1.15, 4.8}, {7.7, 3.0, 3.25, 4.5}}, {{9.2, 3.15, 2.9, 10.0}, {9.6, 4.3, 2.7, 11.0}, {}}};
  int best = 1;
  double least = 1e30;
  for (int g = 1, shift = 0; g <= most; g *= 2, ++shift) {
    const int rows = 128 / g, blocks = (s.time + rows - 1) / rows;
    const Fit& f = fits[dim == 128][shift];
    long walk = 0, all = 0;
    for (int n = 0; n < blocks; ++n) {
      const int first = n * rows, last = std::min(s.time - 1, first + rows - 1);
      const int until = s.window > 0 ? std::min(s.time - 1l, last + s.window - 1l) : s.time - 1, from = s.window > 0 ? std::max(0, first + 1 - s.window) : 0;
      const long keys = (static_cast<long>(s.rep) * (until / 64 - first / 64 + 1) + g - 1) / g, queries = (last / 64 - from / 64 + g) / g;
      all += s.batch * (s.kv_heads * keys + s.heads * queries);
      walk = std::max(walk, keys);
    }
    const double one = f.first + f.step * static_cast<double>(walk);
    const double work = (f.work * static_cast<double>(all) + f.each * static_cast<double>(blocks * planes)) / static_cast<double>(units);
    const double us = one * one + work * work;
    if (us < least) {
      least = us;
      best = g;
    }
  }
  return best;
}

template <int D>
void launch_backward(omx_ctx* ctx, const unsigned short* q, const unsigned short* k, const unsigned short* v,
                     const unsigned short* out, const unsigned short* resid, const float* lse, float* delta,
                     const unsigned short* gy, void* gq, void* gk, void* gv, int32_t grad_dtype,
                     const FlashShape& shape, unsigned long long tag) {
  FlashShape s = shape;
  // Five causal-counted products (S and dP twice each way, dV, dQ, dK) of B H T^2 D each.
  OmxKernelTimer timer(ctx, OMX_K_FLASH_BWD, 5.0 * s.batch * s.heads * static_cast<double>(s.time) * s.time * D);
  // dQ first: it also leaves delta = dO . O per row for the dK/dV pass.
  dim3 block(FT);
  const unsigned pairs = static_cast<unsigned>((s.time + 127) / 128 + 1) / 2;  // two 128-row blocks per workgroup
  const unsigned kv_planes = static_cast<unsigned>(s.batch * s.kv_heads), q_planes = static_cast<unsigned>(s.batch * s.heads);
  const int together = grad_dtype == OMX_BF16 ? flash_together(ctx, s, D, q, k, v, out, resid, gy, gq, gk, gv) : 0;
  if (together) {
    const unsigned rows = 128 / together, blocks = (static_cast<unsigned>(s.time) + rows - 1) / rows;
    s.q_single = s.kv_single = 1;
    if (s.window == 0) s.window = s.time;  // (the same pairs)
    for_groups<D>(together, [&](auto count) {
      omx_launch_timed(ctx, flash_bwd_kernel<D, unsigned short, decltype(count)::value>, dim3(blocks * (kv_planes + q_planes)), block, 0, timer.start(),
                       timer.stop(), q, k, v, out, resid, lse, gy, static_cast<unsigned short*>(gq), static_cast<unsigned short*>(gk),
                       static_cast<unsigned short*>(gv), s, ctx->fault, tag);
    });
    return;
  }
  const int tiles = flash_tiles(s);
  const int q_groups = flash_groups(ctx, q_planes, s.time, tiles, s.window > 0, D);
  const FlashKeyPlan plan = flash_key_plan(ctx, s, D);
  // Split where that takes less and there is room for all parts' sums: a shape's gradients are summed in one of two orders, not in one for
  // each number of parts that a budget might hold.
  const long kv_total = static_cast<long>(kv_planes) * s.time * D;
  float* const parts = plan.parts > 1 ? static_cast<float*>(omx_workspace_if_room(ctx, static_cast<uint64_t>(plan.parts) * kv_total * 8, kExtraSlot)) : nullptr;
  s.kv_parts = parts ? plan.parts : 1;
  const int kv_groups = s.kv_parts > 1 ? plan.groups : plan.whole_groups;
  const unsigned q_rows = 128 / q_groups, kv_rows = 128 / kv_groups;
  s.q_single = q_groups > 1 || flash_single(ctx, pairs * q_planes, D == 64 ? 3 : 2, 1.75);
  s.kv_single = kv_groups > 1 || flash_single(ctx, pairs * kv_planes, 2, D == 64 || s.time <= 384 ? 1e9 : 3.5);
  if (s.kv_parts > 1) s.kv_single = 1;
  dim3 kv_grid((s.kv_single ? (s.time + kv_rows - 1) / kv_rows : pairs) * kv_planes * s.kv_parts);
  dim3 q_grid((s.q_single ? (s.time + q_rows - 1) / q_rows : pairs) * q_planes);
  auto go_dq = [&](auto kernel, auto* gq_ptr) {
    omx_launch_timed(ctx, kernel, q_grid, block, 0, timer.start(), nullptr, q, k, v, out, resid, lse, delta, gy, gq_ptr, s, ctx->fault, tag);
  };
  auto go_dkv = [&](auto kernel, auto* gk_ptr, auto* gv_ptr) {
    omx_launch_timed(ctx, kernel, kv_grid, block, 0, nullptr, s.kv_parts > 1 ? nullptr : timer.stop(), q, k, v, lse, delta, gy, gk_ptr,
                     gv_ptr, s, ctx->fault, tag);
  };
  auto both = [&](auto* gq_ptr, auto* gk_ptr, auto* gv_ptr) {
    typedef std::remove_pointer_t<decltype(gq_ptr)> T;
    for_groups<D>(q_groups, [&](auto count) {
      constexpr int G = decltype(count)::value;
      if (s.window > 0) go_dq(flash_bwd_dq_kernel<D, T, true, G>, gq_ptr);
      else go_dq(flash_bwd_dq_kernel<D, T, false, G>, gq_ptr);
    });
    for_groups<D>(kv_groups, [&](auto count) {
      constexpr int G = decltype(count)::value;
      float* const part_v = parts + s.kv_parts * kv_total;
      if (s.kv_parts > 1) go_dkv(flash_bwd_dkv_kernel<D, float, G, true>, parts, part_v);
      else go_dkv(flash_bwd_dkv_kernel<D, T, G, false>, gk_ptr, gv_ptr);
    });
    if (s.kv_parts > 1)
      omx_launch_timed(ctx, flash_parts_kernel<D, T>, dim3(static_cast<unsigned>((kv_total / 8 + 255) / 256), 2), dim3(256), 0, nullptr,
                       timer.stop(), static_cast<const float*>(parts), gk_ptr, gv_ptr, s, ctx->fault, tag);
  };
  if (grad_dtype == OMX_BF16)
    both(static_cast<unsigned short*>(gq), static_cast<unsigned short*>(gk), static_cast<unsigned short*>(gv));
  else
    both(static_cast<float*>(gq), static_cast<float*>(gk), static_cast<float*>(gv));
}

// The tile loads add a thread's rows as a 32-bit byte offset to a scalar base.
int32_t check_row_strides(omx_ctx* ctx, const FlashShape& s) {
  for (long rs : {s.q.rs, s.kv.rs, s.o.rs})
    if (rs < 1 || rs > FLASH_MAX_ROW_STRIDE)
      return omx_fail(ctx, OMX_SHAPE, "flash attention: row stride %ld outside 1..%ld elements", rs, FLASH_MAX_ROW_STRIDE);
  return OMX_OK;
}

}  // namespace

bool omx_flash_sdpa_supports(uint64_t dim, int32_t operand_dtype) {
  return (dim == 64 || dim == 128) && operand_dtype == OMX_BF16;
}

int32_t omx_flash_sdpa_forward(omx_ctx* ctx, const void* q, const void* k, const void* v, void* out, int32_t out_dtype,
                               void* out_residual, float* lse, uint64_t batch, uint64_t heads, uint64_t kv_heads,
                               uint64_t time, uint64_t dim, uint64_t window, float scale, unsigned long long tag,
                               const long* strides) {
  if (dim != 64 && dim != 128)
    return omx_fail(ctx, OMX_UNSUPPORTED_HEAD_DIM, "head_dim %llu: the MFMA kernels take 64 and 128",
                    (unsigned long long)dim);
  FlashShape s = make_shape(batch, heads, kv_heads, time, dim, window, scale, strides);
  if (int32_t rc = check_row_strides(ctx, s); rc != OMX_OK) return rc;
  const unsigned short* qs = static_cast<const unsigned short*>(q);
  const unsigned short* ks = static_cast<const unsigned short*>(k);
  const unsigned short* vs = static_cast<const unsigned short*>(v);
  if (dim == 64) launch_forward<64>(ctx, qs, ks, vs, out, out_dtype, out_residual, lse, s, tag);
  else launch_forward<128>(ctx, qs, ks, vs, out, out_dtype, out_residual, lse, s, tag);
  OMX_LAUNCH_CHECK(ctx, "flash_fwd_kernel");
  return OMX_OK;
}

int32_t omx_flash_sdpa_backward(omx_ctx* ctx, const void* q, const void* k, const void* v, const void* out,
                                const void* out_residual, const float* lse, const void* gy, void* gq, void* gk,
                                void* gv, int32_t grad_dtype,
                                uint64_t batch, uint64_t heads, uint64_t kv_heads, uint64_t time, uint64_t dim,
                                uint64_t window, float scale, unsigned long long tag, const long* strides) {
  if (dim != 64 && dim != 128)
    return omx_fail(ctx, OMX_UNSUPPORTED_HEAD_DIM, "head_dim %llu: the MFMA kernels take 64 and 128",
                    (unsigned long long)dim);
  FlashShape s = make_shape(batch, heads, kv_heads, time, dim, window, scale, strides);
  if (int32_t rc = check_row_strides(ctx, s); rc != OMX_OK) return rc;
  const bool aligned = ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(gy)) & 15u) == 0 &&
              ((s.q.rs | s.q.hs | s.q.bs | s.kv.rs | s.kv.hs | s.kv.bs | s.o.rs | s.o.hs | s.o.bs) & 7) == 0;
  s.direct = aligned ? s.time : 0;
  const long rows = static_cast<long>(batch * heads * time);
  void* ws = nullptr;
  int32_t rc = omx_workspace(ctx, rows * sizeof(float), &ws);
  if (rc != OMX_OK) return rc;
  float* delta = static_cast<float*>(ws);
  const unsigned short* qs = static_cast<const unsigned short*>(q);
  const unsigned short* ks = static_cast<const unsigned short*>(k);
  const unsigned short* vs = static_cast<const unsigned short*>(v);
  const unsigned short* os = static_cast<const unsigned short*>(out);
  const unsigned short* rs = static_cast<const unsigned short*>(out_residual);
  const unsigned short* gs = static_cast<const unsigned short*>(gy);
  if (dim == 64) launch_backward<64>(ctx, qs, ks, vs, os, rs, lse, delta, gs, gq, gk, gv, grad_dtype, s, tag);
  else launch_backward<128>(ctx, qs, ks, vs, os, rs, lse, delta, gs, gq, gk, gv, grad_dtype, s, tag);
  OMX_LAUNCH_CHECK(ctx, "flash backward kernels");
  return OMX_OK;
}
