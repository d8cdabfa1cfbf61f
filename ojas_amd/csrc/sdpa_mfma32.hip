// f32 attention on the f32 matrix instructions (v_mfma_f32_16x16x4_f32), head dims 16 / 32 / 64 / 128: causal SDPA
// forward and backward of the f32 tier and the attention of a prompt chunk over a KV cache (over bf16 caches of head dim
// 64 and 128 on the bf16 ones, sdpa_prompt_kernel).
//
// Reference: ojas-cpu/src/attn.rs (causal_sdpa_*; trait ojas-core/src/backend.rs:1729-1792) and
// ojas-cpu/src/kv.rs (cached_attention_forward, backend.rs:2526-2555). Same formulas as sdpa.hip's row
// kernels: p = e^(s - max), out = sum p v / sum p, lse = max + ln(sum); backward p = e^(s - lse),
// dS = scale p (dP - dO . O).
//
// What bounds it: the matrix units have the vector units' f32 rate (157 TFLOP/s) but take their operands from a
// quarter of the LDS traffic. On vector instructions 64 x 64 tiles ran at 5 to 12 % of that rate, bound by LDS reads,
// and the key / value pass of a grouped model had a workgroup per 64 keys of a KV head: 52 for 256 units.
//
// Rows are packed: row r of a KV head is query r / rep of its head r % rep, so grouped heads share every key
// and value tile. Score tiles are formed with the rows that softmax runs over in the accumulator's registers (lane
// l: row l % 16, values 4 (l / 16) + v), which is exactly the operand layout of the product that follows (its
// instruction j takes K values 4 (l / 16) + j): probabilities and dS go from accumulator to operand without
// moving. The other operand of that product is read from LDS along its fast index: one 16-byte read serves four
// interleaved blocks of result columns (block c VW + e holds columns 16 VW c + VW i + e).
//
// 64-row tiles are fetched into registers while the previous one is multiplied. Where there are few rows, or the other
// side is long (at_narrow), the four waves of a workgroup split the keys (KW = 4) instead of the rows and meet in LDS: no wave
// reads another's blocks then, so they come from memory straight into operands, a block ahead, with no barrier in the
// loop. A block that is read in both forms (keys in the dQ pass, rows in the key / value pass) goes through 16 rows of LDS of the
// wave's own for the second: fetched twice, the passes were bound by their loads' latency (2 x 8 heads over 2 x 777, backward:
// 131 us through shared tiles, 118 with two fetches, 104). The key / value pass splits
// its rows over the grid when keys alone do not fill the chip, and a second launch adds the parts in order.
// No atomics; every sum has a fixed order.
//
// A step whose rows see every one of its keys (all but the diagonal's and a window's ends) is told by scalar compares and takes
// no mask; rows are rescaled only where one of the wave's has a new maximum; a lane's address is 32 bits beside a scalar. With a mask
// on every score and 64-bit addresses: forward / backward 68 / 222 us -> 64 / 198 at 2 x 12 x 1024 x 64, 26 / 103 -> 25 / 96 at 2 x 8
// over 2 x 777, 154 / 557 -> 147 / 494 at 4 x 8 x 1024 x 128. With a plane's blocks on few L2s (at_place) from there: 48 / 154,
// 23 / 88, 107 / 366.
//
// On vector instructions, through shared tiles and now, us, forward / backward (batch x heads over KV heads x time x head
// dim): 8 x 4/4 x 256 x 64: 38 / 109, 13 / 34, 11 / 30; 2 x 8/2 x 777 x 64 in a window of 256: 47 / 370, 20 / 66, 19 / 55; 16 x 12/12
// x 512 x 64 (shared tiles still): 272 / 1337, 132 / 439 (48 and 37 TFLOP/s, causal-counted); 16 x 4096 x 64: 587 / 1868 through shared
// tiles, 325 / 1120; 1 x 2/1 x 3000 x 128: 696 / 3334, 151 / 409, 86 / 216.
#include <algorithm>
#include <cmath>

#include "sdpa_mfma32.h"

namespace {

typedef float floatx4_a __attribute__((ext_vector_type(4)));
constexpr int AT_THREADS = 256, AT_ROWS = 64;  // rows per LDS tile
constexpr float AT_LOG2E = 1.4426950408889634f, AT_LN2 = 0.6931471805599453f;

__device__ __forceinline__ floatx4_a at_mfma(float a, float b, floatx4_a c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ floatx4_a at_zero() { return floatx4_a{0.0f, 0.0f, 0.0f, 0.0f}; }
// Over the four lanes that hold one row.
template <typename F>
__device__ __forceinline__ float at_row(float v, F f) {
  return dev_meet_32(dev_meet_16(v, f), f);
}
__device__ __forceinline__ float at_row_max(float v) { return at_row(v, [](float x, float y) { return fmaxf(x, y); }); }
__device__ __forceinline__ float at_row_sum(float v) { return at_row(v, [](float x, float y) { return x + y; }); }

template <int D>
struct AtDim {
  static constexpr int S = D / 16;             // 16-column steps of a product over the head dim; column blocks of a result
  static constexpr int VW = S < 4 ? S : 4;     // interleaved column blocks per LDS read
  static constexpr int NC = S / VW;
  static constexpr int P = D + 4;              // LDS row pitch: 16 rows' 16-byte pieces fall in distinct banks
  static constexpr int PIECES = AT_ROWS * D / 4 / AT_THREADS;  // 16-byte pieces of a tile per thread (at least 1)
};

// A tile on its way: PIECES pieces per thread, in memory's type until they are stored.
template <int D, typename T>
struct AtTile {
  using Raw = std::conditional_t<sizeof(T) == 4, float4, uint2>;
  Raw raw[AtDim<D>::PIECES];
  // `row_at(r)`: pointer to tile row r, or null for a row of zeros.
  template <typename F>
  __device__ __forceinline__ void fetch(F row_at) {
#pragma unroll
    for (int i = 0; i < AtDim<D>::PIECES; ++i) {
      const int idx = threadIdx.x + i * AT_THREADS, r = idx / (D / 4), c = idx % (D / 4);
      const T* p = row_at(r);
      if (p) raw[i] = *reinterpret_cast<const Raw*>(p + 4 * c);
      else raw[i] = Raw{};
    }
  }
  __device__ __forceinline__ void store(float* lds) const {
#pragma unroll
    for (int i = 0; i < AtDim<D>::PIECES; ++i) {
      const int idx = threadIdx.x + i * AT_THREADS, r = idx / (D / 4), c = idx % (D / 4);
      float4 v;
      if constexpr (sizeof(T) == 4) {
        v = raw[i];
      } else {
        v = make_float4(__uint_as_float(raw[i].x << 16), __uint_as_float(raw[i].x & 0xffff0000u), __uint_as_float(raw[i].y << 16),
                        __uint_as_float(raw[i].y & 0xffff0000u));
      }
      *reinterpret_cast<float4*>(lds + r * AtDim<D>::P + 4 * c) = v;
    }
  }
};

// ---- without LDS: a wave that shares its 16-row blocks with no other reads them straight into operands
// Rows are addressed as a scalar plus a 32-bit lane offset, so that a block whose rows lie in order needs no vector arithmetic
// for its addresses (64-bit ones took half as many issue slots as the products). The empty assembly keeps the compiler
// from moving the scalar part into vector registers.
typedef const __attribute__((address_space(1))) char* AtBytes;
__device__ __forceinline__ AtBytes at_bytes(const void* p) { return (AtBytes)(p); }
template <typename V>
__device__ __forceinline__ V at_load(AtBytes at, unsigned off) {
  asm("" : "+s"(at));
  return *reinterpret_cast<const __attribute__((address_space(1))) V*>(at + off);
}
template <typename T, int N>
using AtVec = T __attribute__((ext_vector_type(N)));
__device__ __forceinline__ float4 at_widen(const AtVec<float, 4>& v) { return make_float4(v[0], v[1], v[2], v[3]); }
__device__ __forceinline__ float4 at_widen(const AtVec<unsigned short, 4>& v) {
  return make_float4(dev_bf16_bits_to_f32(v[0]), dev_bf16_bits_to_f32(v[1]), dev_bf16_bits_to_f32(v[2]), dev_bf16_bits_to_f32(v[3]));
}
__device__ __forceinline__ float at_value(float v) { return v; }
__device__ __forceinline__ float at_value(unsigned short v) { return dev_bf16_bits_to_f32(v); }
// One block for at_dot: lane i's row, pieces 4 g of each 16 columns. `off`: bytes from `at` to the row's element 4 g.
template <int D, typename T>
struct AtDotBlock {
  AtVec<T, 4> raw[AtDim<D>::S];
  __device__ __forceinline__ void fetch(AtBytes at, unsigned off) {
#pragma unroll
    for (int s = 0; s < AtDim<D>::S; ++s) raw[s] = at_load<AtVec<T, 4>>(at + 16 * s * sizeof(T), off);
  }
  __device__ __forceinline__ floatx4_a dot(const float4 (&own)[AtDim<D>::S]) const {
    floatx4_a acc = at_zero();
#pragma unroll
    for (int s = 0; s < AtDim<D>::S; ++s) {
      const float4 t = at_widen(raw[s]);
      acc = at_mfma(t.x, own[s].x, acc);
      acc = at_mfma(t.y, own[s].y, acc);
      acc = at_mfma(t.z, own[s].z, acc);
      acc = at_mfma(t.w, own[s].w, acc);
    }
    return acc;
  }
};
// The block as at_accumulate reads it, in LDS of this wave's own (16 rows of pitch P).
template <int D>
__device__ __forceinline__ void at_stage(const AtDotBlock<D, float>& block, float* tile16, int i, int g) {
#pragma unroll
  for (int s = 0; s < AtDim<D>::S; ++s) *reinterpret_cast<AtVec<float, 4>*>(tile16 + i * AtDim<D>::P + 16 * s + 4 * g) = block.raw[s];
}
// One block for at_accumulate: rows 4 g + j, columns VW i .. of each 64 (of 32, of 16). `off`: bytes to row 4 g + j's element VW i.
template <int D, typename T>
struct AtSumBlock {
  using X = AtDim<D>;
  AtVec<T, X::VW> raw[4][X::NC];
  __device__ __forceinline__ void fetch(AtBytes at, const unsigned (&off)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int c = 0; c < X::NC; ++c) raw[j][c] = at_load<AtVec<T, X::VW>>(at + 64 * c * sizeof(T), off[j]);
  }
  __device__ __forceinline__ void accumulate(const floatx4_a& weight, floatx4_a (&out)[X::S]) const {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int c = 0; c < X::NC; ++c)
#pragma unroll
        for (int e = 0; e < X::VW; ++e) out[c * X::VW + e] = at_mfma(at_value(raw[j][c][e]), weight[j], out[c * X::VW + e]);
  }
};

// acc (values 4 g + v of 16 tile rows, this lane's own row) = tile rows . own row over the head dim.
template <int D>
__device__ __forceinline__ floatx4_a at_dot(const float* tile16, const float4 (&own)[AtDim<D>::S], int i, int g) {
  floatx4_a acc = at_zero();
  const float* p = tile16 + i * AtDim<D>::P + 4 * g;
#pragma unroll
  for (int s = 0; s < AtDim<D>::S; ++s) {
    const float4 t = *reinterpret_cast<const float4*>(p + 16 * s);
    acc = at_mfma(t.x, own[s].x, acc);
    acc = at_mfma(t.y, own[s].y, acc);
    acc = at_mfma(t.z, own[s].z, acc);
    acc = at_mfma(t.w, own[s].w, acc);
  }
  return acc;
}
// out[block] += sum over 16 tile rows of weight[row] * tile row, weights in at_dot's layout.
template <int D>
__device__ __forceinline__ void at_accumulate(const float* tile16, const floatx4_a& weight, floatx4_a (&out)[AtDim<D>::S], int i, int g) {
  using X = AtDim<D>;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float* row = tile16 + (4 * g + j) * X::P + X::VW * i;
#pragma unroll
    for (int c = 0; c < X::NC; ++c) {
      float t[X::VW];
      if constexpr (X::VW == 4) {
        const float4 x = *reinterpret_cast<const float4*>(row + 64 * c);
        t[0] = x.x; t[1] = x.y; t[2] = x.z; t[3] = x.w;
      } else if constexpr (X::VW == 2) {
        const float2 x = *reinterpret_cast<const float2*>(row);
        t[0] = x.x; t[1] = x.y;
      } else {
        t[0] = *row;
      }
#pragma unroll
      for (int e = 0; e < X::VW; ++e) out[c * X::VW + e] = at_mfma(t[e], weight[j], out[c * X::VW + e]);
    }
  }
}
// A row's result columns held by this lane, times `f`, for accumulator registers v0 .. v0 + NV - 1.
template <int D, int NV>
__device__ __forceinline__ bool at_store(float* row, const floatx4_a (&out)[AtDim<D>::S], float f, int g, int v0) {
  using X = AtDim<D>;
  bool bad = false;
#pragma unroll
  for (int c = 0; c < X::NC; ++c)
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      float* p = row + c * 16 * X::VW + X::VW * (4 * g + v0 + u);
#pragma unroll
      for (int e = 0; e < X::VW; ++e) {
        float x = 0.0f;
#pragma unroll
        for (int v = 0; v < 4; ++v) x = v == v0 + u ? out[c * X::VW + e][v] : x;  // a register index known only when NV < 4
        x *= f;
        bad |= !dev_finite(x);
        p[e] = x;
      }
    }
  return bad;
}

// This workgroup's block of rows (or keys) and its (batch, KV head) plane. Workgroups go round-robin over the 8 XCDs by their linear
// index, and each XCD has its own L2: planes are dealt so that one is read through as few of them as their number allows (one
// where it is a multiple of 8, all eight where it is odd), its blocks in turn over those. With a plane's blocks over all eight, 12
// heads x 64 of 4 sequences, 256 new positions of 700: 72 MB came from beyond the L2s for 9 of keys and values.
struct AtPlace {
  int block, plane;
};
__device__ __forceinline__ AtPlace at_place(unsigned index, unsigned blocks, unsigned planes) {
  const unsigned share = min(8u, planes & (0u - planes));
  const unsigned n = index / share, run = n / blocks;
  return {static_cast<int>(n - run * blocks), static_cast<int>(index % share + share * run)};
}
__device__ __forceinline__ AtPlace at_place() { return at_place(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x, gridDim.y); }
// Where part blockIdx.z of a row's result goes (Sdpa32Args::partial).
__device__ __forceinline__ float* at_partial(const Sdpa32Args& a, int dim, int b, int kvh, int query, int head) {
  const long row = (static_cast<long>(b) * a.tq + query) * a.kv_heads * a.rep + static_cast<long>(kvh) * a.rep + head;
  return a.partial + (row * a.nparts + blockIdx.z) * (dim + 2);
}
// This workgroup's share of the tiles first .. last: all of them, or part blockIdx.z (which may be empty).
__device__ __forceinline__ void at_key_part(const Sdpa32Args& a, int* first, int* last) {
  if (a.nparts > 1) {
    const int each = (*last - *first + a.nparts) / a.nparts;
    *first += static_cast<int>(blockIdx.z) * each;
    *last = min(*last, *first + each - 1);
  }
}

struct AtRow {
  int query, head;  // head within the group
};
__device__ __forceinline__ AtRow at_unpack(int r, int rep) {
  AtRow x;
  if (rep == 1) {
    x.query = r;
    x.head = 0;
  } else {
    x.query = r / rep;
    x.head = r - x.query * rep;
  }
  return x;
}
// at_unpack in a loop: a multiplication for the division (exact while r * rep < 2^32: with m = ceil(2^32 / rep), r m / 2^32 is
// above r / rep by less than r / 2^32).
struct AtUnpack {
  int rep;
  unsigned magic;
  __device__ __forceinline__ explicit AtUnpack(int rep_) : rep(rep_), magic(rep_ == 1 ? 0u : 0xffffffffu / static_cast<unsigned>(rep_) + 1u) {}
  __device__ __forceinline__ AtRow operator()(int r) const {
    AtRow x;
    x.query = rep == 1 ? r : static_cast<int>(__umulhi(static_cast<unsigned>(r), magic));
    x.head = r - x.query * rep;
    return x;
  }
};
// Own row `r` of a [.., row, D] tensor as a product operand.
template <int D>
__device__ __forceinline__ void at_own(const float* row, float4 (&own)[AtDim<D>::S], int g) {
#pragma unroll
  for (int s = 0; s < AtDim<D>::S; ++s) own[s] = *reinterpret_cast<const float4*>(row + 16 * s + 4 * g);
}

// ---------------------------------------------------------------- forward
template <int D, int KW, typename TK>
__global__ __launch_bounds__(AT_THREADS) void sdpa32_fwd_kernel(Sdpa32Args a) {
  using X = AtDim<D>;
  // KW = 4: nothing but the waves' sums goes through LDS; a wave takes 16 keys of each 64, BLOCKS times 64 a step.
  constexpr int QW = 4 / KW, BQ = 16 * QW, BLOCKS = KW == 1 ? 4 : D <= 64 ? 2 : 1, NEXT = KW == 1 ? 16 : 64;  // from block to block
  __shared__ __align__(16) float lds[KW == 1 ? 2 * AT_ROWS * X::P : 128 + 4 * X::S * 256];
  float* kt = lds;
  float* vt = lds + AT_ROWS * X::P;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)), i = lane & 15, g = lane >> 4;
  const int qw = wave % QW, kw = wave / QW;
  const AtPlace place = at_place();
  const int b = place.plane / a.kv_heads, kvh = place.plane - b * a.kv_heads;
  const int rows = a.tq * a.rep;
  const int r0 = (gridDim.x - 1 - place.block) * BQ;  // the rows that see the most keys first
  const int r = r0 + qw * 16 + i;
  const AtRow at = at_unpack(min(r, rows - 1), a.rep);
  const long q_at = b * a.q_b + (static_cast<long>(kvh) * a.rep + at.head) * a.q_h + static_cast<long>(at.query) * a.q_t;
  float4 q[X::S];
  at_own<D>(a.q + q_at, q, g);
  const int pos = r < rows ? a.q_pos0 + at.query : -1;
  const int low = a.window > 0 ? max(0, pos + 1 - a.window) : 0;
  const int first_pos = a.q_pos0 + at_unpack(r0, a.rep).query;
  const int last_pos = a.q_pos0 + at_unpack(min(r0 + BQ, rows) - 1, a.rep).query;
  int t_first = (a.window > 0 ? max(0, first_pos + 1 - a.window) : 0) / AT_ROWS, t_last = last_pos / AT_ROWS;
  at_key_part(a, &t_first, &t_last);
  const TK* kb = static_cast<const TK*>(a.k) + b * a.k_b + kvh * a.k_h;
  const TK* vb = static_cast<const TK*>(a.v) + b * a.k_b + kvh * a.k_h;
  auto slot_at = [&](int key) {
    // A ring wraps at most once over the keys that are read (slot0 + key can pass 2^31).
    const unsigned int slot = static_cast<unsigned int>(a.slot0) + key, capacity = a.capacity;
    return static_cast<long>(slot >= capacity ? slot - capacity : slot) * a.k_t;
  };
  const float scale2 = a.scale * AT_LOG2E;
  floatx4_a o[X::S];
#pragma unroll
  for (int m = 0; m < X::S; ++m) o[m] = at_zero();
  float mx = -INFINITY, sum = 0.0f;  // in the exp2 domain; `sum` over this lane's keys only
  bool bad = false;
  // Scores to weights for `key0` and the keys after it: masks where a row or its window ends among them, the running maximum,
  // the rescaling that it asks for where one of the wave's rows has a new one.
  const int end_pos = min(last_pos, t_last * AT_ROWS + AT_ROWS - 1);  // (a part of the keys ends with tile t_last)
  const int whole_to = r0 + BQ <= rows ? min(first_pos, end_pos) : -1, whole_from = a.window > 0 ? max(0, last_pos + 1 - a.window) : 0;
  const int high = min(pos, end_pos);
  float check = 0.0f;  // NaN once a score that counts was not finite
  auto weights = [&](floatx4_a (&s)[BLOCKS], int key0) {
    float top = -INFINITY;
    if (key0 + (BLOCKS - 1) * NEXT + 15 <= whole_to && key0 >= whole_from) {  // (uniform)
#pragma unroll
      for (int n = 0; n < BLOCKS; ++n)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          s[n][v] *= scale2;
          check = fmaf(s[n][v], 0.0f, check);
          top = fmaxf(top, s[n][v]);
        }
    } else {
#pragma unroll
      for (int n = 0; n < BLOCKS; ++n)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int key = key0 + n * NEXT + 4 * g + v;
          const bool seen = key <= high && key >= low;
          const float x = s[n][v] * scale2;
          bad |= seen && !dev_finite(x);
          s[n][v] = seen ? x : -INFINITY;
          top = fmaxf(top, s[n][v]);
        }
    }
    top = at_row_max(top);
    if (__any(top > mx)) {
      const float mx_new = fmaxf(mx, top);
      const float rescale = mx_new == mx ? 1.0f : __builtin_amdgcn_exp2f(mx - mx_new);  // 0 on the first keys
      mx = mx_new;
      sum *= rescale;
#pragma unroll
      for (int m = 0; m < X::S; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v) o[m][v] *= rescale;
    }
    const float base = mx == -INFINITY ? 0.0f : mx;
#pragma unroll
    for (int n = 0; n < BLOCKS; ++n)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        s[n][v] = __builtin_amdgcn_exp2f(s[n][v] - base);
        sum += s[n][v];
      }
  };
  if constexpr (KW == 1) {
    AtTile<D, TK> kn, vn;
    auto fetch = [&](int t) {
      auto row_of = [&](const TK* base, int row) {
        const int key = t * AT_ROWS + row;
        return key < a.tk ? base + slot_at(key) : nullptr;
      };
      kn.fetch([&](int row) { return row_of(kb, row); });
      vn.fetch([&](int row) { return row_of(vb, row); });
    };
    if (t_first <= t_last) fetch(t_first);
    for (int t = t_first; t <= t_last; ++t) {
      __syncthreads();  // the previous tile has been read
      kn.store(kt);
      vn.store(vt);
      __syncthreads();
      if (t < t_last) fetch(t + 1);
      floatx4_a s[BLOCKS];
#pragma unroll
      for (int n = 0; n < BLOCKS; ++n) s[n] = at_dot<D>(kt + n * 16 * X::P, q, i, g);
      weights(s, t * AT_ROWS);
#pragma unroll
      for (int n = 0; n < BLOCKS; ++n) at_accumulate<D>(vt + n * 16 * X::P, s[n], o, i, g);
    }
  } else {
    // Values are on their way while the scores are formed, the next keys during softmax and the second product. (Keys past
    // the last one are read from it; their weights are 0.)
    AtDotBlock<D, TK> keys[BLOCKS];
    AtSumBlock<D, TK> values[BLOCKS];
    // Up to `straight` the keys lie in order and whole (beyond: the ring's end, or the last key).
    const int straight = min(a.tk, a.capacity - a.slot0);
    const unsigned pitch = static_cast<unsigned>(a.k_t) * sizeof(TK);
    unsigned k_off = i * pitch + 4 * g * sizeof(TK), v_off[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v_off[j] = (4 * g + j) * pitch + X::VW * i * sizeof(TK);
    // A block's first row, and row `r` of it from there.
    auto block_at = [&](const TK* base, int key0) { return at_bytes(base + (key0 + 16 <= straight ? (a.slot0 + key0) * a.k_t : 0l)); };
    auto row_off = [&](int key0, int r) {
      const unsigned int slot = static_cast<unsigned int>(a.slot0) + min(key0 + r, a.tk - 1), capacity = a.capacity;
      return (slot >= capacity ? slot - capacity : slot) * pitch;
    };
    // This wave's block of tile `t`, and whether a row of the workgroup sees any of it.
    const int from_pos = a.window > 0 ? max(0, first_pos + 1 - a.window) : 0;
    auto block_of = [&](int t) { return t * AT_ROWS + kw * 16; };
    auto counts = [&](int key0) { return key0 <= end_pos && key0 + 15 >= from_pos; };
    auto fetch = [&](int t) {
#pragma unroll
      for (int n = 0; n < BLOCKS; ++n) {
        const int key0 = min(block_of(t + n), end_pos & ~15);  // (one that does not count reads the last that does)
        unsigned off = k_off;
        if (key0 + 16 > straight) off = row_off(key0, i) + 4 * g * sizeof(TK);
        keys[n].fetch(block_at(kb, key0), off);
      }
    };
    if (t_first <= t_last) fetch(t_first);
    for (int t = t_first; t <= t_last; t += BLOCKS) {
#pragma unroll
      for (int n = 0; n < BLOCKS; ++n) {
        const int key0 = min(block_of(t + n), end_pos & ~15);
        unsigned off[4] = {v_off[0], v_off[1], v_off[2], v_off[3]};
        if (key0 + 16 > straight) {
#pragma unroll
          for (int j = 0; j < 4; ++j) off[j] = row_off(key0, 4 * g + j) + X::VW * i * sizeof(TK);
        }
        values[n].fetch(block_at(vb, key0), off);
      }
      floatx4_a s[BLOCKS];
#pragma unroll
      for (int n = 0; n < BLOCKS; ++n) {
        s[n] = at_zero();
        if (counts(block_of(t + n))) s[n] = keys[n].dot(q);
      }
      fetch(min(t + BLOCKS, t_last));
      weights(s, block_of(t));
#pragma unroll
      for (int n = 0; n < BLOCKS; ++n)
        if (counts(block_of(t + n))) values[n].accumulate(s[n], o);
    }
  }
  bad |= check != 0.0f;
  sum = at_row_sum(sum);
  float* out = a.out + b * a.o_b + (static_cast<long>(kvh) * a.rep + at.head) * a.o_h + static_cast<long>(at.query) * a.o_t;
  float* lse = a.lse ? a.lse + (static_cast<long>(b) * a.kv_heads * a.rep + static_cast<long>(kvh) * a.rep + at.head) * a.tq + at.query : nullptr;
  // A part's maximum and sum, by one lane of the row.
  auto store_part = [&](float top, float total, float* row) {
    row[D] = top * AT_LN2;  // (minus infinity where the row saw none of the part's keys)
    row[D + 1] = total;
  };
  if constexpr (KW == 1) {
    if (r < rows) {
      if (a.nparts > 1) {
        float* row = at_partial(a, D, b, kvh, at.query, at.head);
        bad |= at_store<D, 4>(row, o, 1.0f, g, 0);
        if (g == 0) store_part(mx, sum, row);
      } else {
        bad |= !(dev_finite(sum) && sum > 0.0f);
        bad |= at_store<D, 4>(out, o, 1.0f / sum, g, 0);
        if (lse && g == 0) *lse = mx * AT_LN2 + logf(sum);
      }
    }
  } else {
    // The four waves' shares of the same rows: every wave adds up one register of each block.
    __syncthreads();
    float* stat = lds;                   // [4][2][16]
    float* part = lds + 128;             // [4][S * 4][64]
    if (g == 0) {
      stat[kw * 32 + i] = mx;
      stat[kw * 32 + 16 + i] = sum;
    }
#pragma unroll
    for (int m = 0; m < X::S; ++m)
#pragma unroll
      for (int v = 0; v < 4; ++v) part[((kw * X::S + m) * 4 + v) * 64 + lane] = o[m][v];
    __syncthreads();
    float all = -INFINITY, weight[4], total = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) all = fmaxf(all, stat[w * 32 + i]);
    const float base = all == -INFINITY ? 0.0f : all;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      weight[w] = __builtin_amdgcn_exp2f(stat[w * 32 + i] - base);
      total = fmaf(weight[w], stat[w * 32 + 16 + i], total);
    }
#pragma unroll
    for (int m = 0; m < X::S; ++m) {
      float x = 0.0f;
#pragma unroll
      for (int w = 0; w < 4; ++w) x = fmaf(weight[w], part[((w * X::S + m) * 4 + kw) * 64 + lane], x);
      o[m] = floatx4_a{x, x, x, x};
    }
    if (r < rows) {
      if (a.nparts > 1) {
        float* row = at_partial(a, D, b, kvh, at.query, at.head);
        bad |= at_store<D, 1>(row, o, 1.0f, g, kw);
        if (g == 0 && kw == 0) store_part(all, total, row);
      } else {
        bad |= !(dev_finite(total) && total > 0.0f);
        bad |= at_store<D, 1>(out, o, 1.0f / total, g, kw);
        if (lse && g == 0 && kw == 0) *lse = all * AT_LN2 + logf(total);
      }
    }
  }
  if (bad) dev_raise_fault(a.fault, a.tag);
}

// ---------------------------------------------------------------- forward over bf16 caches
// Keys and values are bf16 there, so the bf16 matrix instructions (sixteen times the f32 rate) multiply them exactly;
// the f32 operand beside them, a query or a probability, is cut into three bf16 parts that hold all of its 24 bits
// (each cut is exact), and the three products are added up in f32, smallest first. Every product is exact, as on the
// f32 instructions, and a row's sums have half as many roundings; three sixteenths of the matrix time.
//
// A workgroup takes 16 MB rows and its four waves share the keys, AtPrompt::KEYS at a time. No wave reads another's
// keys, so keys go from memory straight into fragments and only values pass through LDS, a region per wave, where
// the transposing reads form the other operand: no barrier before the waves meet. The next keys and values are on
// their way during softmax and the second product. A step that every row sees whole takes no mask, rows are rescaled only where a
// maximum moves, addresses are a scalar and 32 bits (half of the vector instructions went there). Bound by the way from the L2s
// (13 TB/s of keys and values; without the loads three quarters of the time) and by vector instructions: softmax and the cuts.
// us on f32 instructions, on bf16 ones, with neither masks nor planes over all L2s (relative error against 64 bits): 4 x 12 heads x
// 64, 256 new positions of 700: 38.6, 20.5, 17.5 (2.5e-7, 1.5e-7, the same); 8 x 16 over 4 KV heads x 64, 512 of 1024: 173, 85, 67
// (5.2e-7, 1.6e-7); 2 x 8 over 2 x 128, 100 of 800: 41, 16, 13.7 (2.9e-7, 1.5e-7); 16 x 12 x 64, 256 of 1000: 77, 58 from there.
typedef __bf16 bf16x8_a __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4_a __attribute__((ext_vector_type(4)));
typedef short short4_a __attribute__((ext_vector_type(4)));

struct AtParts {
  u32x4_a part[3];  // largest first
  __device__ __forceinline__ void cut(const float (&x)[8]) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      float a = x[2 * p], b = x[2 * p + 1];
#pragma unroll
      for (int n = 0; n < 3; ++n) {
        const unsigned int wa = __float_as_uint(a), wb = __float_as_uint(b);
        part[n][p] = __builtin_amdgcn_perm(wb, wa, 0x07060302u);  // the upper halves, a's below b's
        a -= __uint_as_float(wa & 0xffff0000u);
        b -= __uint_as_float(wb & 0xffff0000u);
      }
    }
  }
};
// acc += A . B, lane values 8 g + j of both. A sum takes an operand's parts smallest first.
__device__ __forceinline__ floatx4_a at_mfma16(u32x4_a a, u32x4_a b, floatx4_a acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_a, a), __builtin_bit_cast(bf16x8_a, b), acc, 0, 0, 0);
}

template <int D>
struct AtPrompt {
  static constexpr int KEYS = 4096 / D;      // per wave and step
  static constexpr int NB = KEYS / 16;       // blocks of 16 keys
  static constexpr int KS = D / 32, DB = D / 16;
  static constexpr int PITCH = 2 * D + 32;   // bytes of a value row in LDS: eight rows' 32-byte pieces in distinct banks
  static constexpr int PIECES = KEYS * D / 8 / 64;
};

// (three workgroups per compute unit with one block of rows: 168 registers, none to spare for the parts of split keys)
template <int D, int MB, bool SPLIT>
__global__ __launch_bounds__(AT_THREADS, D == 64 && MB == 1 ? 3 : 2) void sdpa_prompt_kernel(Sdpa32Args a) {
  using X = AtPrompt<D>;
  __shared__ __align__(16) char lds[4 * X::KEYS * X::PITCH];
  static_assert(512 + 4 * X::DB * 1024 <= 4 * X::KEYS * X::PITCH, "the waves' sums fit");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)), i = lane & 15, g = lane >> 4;
  const AtPlace place = at_place();
  const int b = place.plane / a.kv_heads, kvh = place.plane - b * a.kv_heads;
  const int rows = a.tq * a.rep;
  const int r0 = (gridDim.x - 1 - place.block) * (16 * MB);  // the rows that see the most keys first
  AtRow at[MB];
  AtParts q[MB][X::KS];
  int pos[MB], low[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int r = r0 + m * 16 + i;
    at[m] = at_unpack(min(r, rows - 1), a.rep);
    const float* row = a.q + b * a.q_b + (static_cast<long>(kvh) * a.rep + at[m].head) * a.q_h + static_cast<long>(at[m].query) * a.q_t;
#pragma unroll
    for (int s = 0; s < X::KS; ++s) {
      const float4 x = *reinterpret_cast<const float4*>(row + 32 * s + 8 * g), y = *reinterpret_cast<const float4*>(row + 32 * s + 8 * g + 4);
      const float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
      q[m][s].cut(v);
    }
    pos[m] = r < rows ? a.q_pos0 + at[m].query : -1;
    low[m] = a.window > 0 ? max(0, pos[m] + 1 - a.window) : 0;
  }
  const int first_pos = a.q_pos0 + at_unpack(r0, a.rep).query;
  const int last_pos = a.q_pos0 + at_unpack(min(r0 + 16 * MB, rows) - 1, a.rep).query;
  int t_first = (a.window > 0 ? max(0, first_pos + 1 - a.window) : 0) / X::KEYS, t_last = last_pos / X::KEYS;
  if constexpr (SPLIT) at_key_part(a, &t_first, &t_last);
  const int last_low = a.window > 0 ? max(0, last_pos + 1 - a.window) : 0;
  const unsigned short* kb = static_cast<const unsigned short*>(a.k) + b * a.k_b + kvh * a.k_h;
  const unsigned short* vb = static_cast<const unsigned short*>(a.v) + b * a.k_b + kvh * a.k_h;
  char* region = lds + wave * (X::KEYS * X::PITCH);

  u32x4_a kn[X::NB][X::KS], vn[X::PIECES];
  // Rows by 32-bit lane offsets from the tile's first row, or, past the ring's end, from the ring's first (at_prompt). Keys past
  // the last one are read from it; their weights are 0.
  const int straight = min(a.tk, a.capacity - a.slot0);  // up to here the keys lie in order
  const unsigned pitch = 2u * static_cast<unsigned>(a.k_t);
  const unsigned k_off = i * pitch + 16 * g, v_off = lane / (D / 8) * pitch + lane % (D / 8) * 16;
  auto fetch = [&](int t) {
    const int key0 = t * X::KEYS;
    const bool plain = key0 + X::KEYS <= straight;                          // (uniform)
    const unsigned row0 = plain || straight == a.tk ? a.slot0 + key0 : 0u;  // the first row
    unsigned k_at[X::NB], v_at[X::PIECES];
    if (plain) {
      unsigned step = pitch;
      asm("" : "+s"(step));  // (twelve sums rather than twelve registers across the loop)
#pragma unroll
      for (int n = 0; n < X::NB; ++n) k_at[n] = k_off + n * 16 * step;
#pragma unroll
      for (int p = 0; p < X::PIECES; ++p) v_at[p] = v_off + p * (512 / D) * step;
    } else {
      auto row_off = [&](int row) {
        const unsigned slot = static_cast<unsigned>(a.slot0) + min(key0 + row, a.tk - 1), capacity = a.capacity;
        return ((slot >= capacity ? slot - capacity : slot) - row0) * pitch;
      };
#pragma unroll
      for (int n = 0; n < X::NB; ++n) k_at[n] = row_off(n * 16 + i) + 16 * g;
#pragma unroll
      for (int p = 0; p < X::PIECES; ++p) v_at[p] = row_off(lane / (D / 8) + p * (512 / D)) + lane % (D / 8) * 16;
    }
    const AtBytes ka = at_bytes(kb + row0 * a.k_t), va = at_bytes(vb + row0 * a.k_t);
#pragma unroll
    for (int n = 0; n < X::NB; ++n)
#pragma unroll
      for (int s = 0; s < X::KS; ++s) kn[n][s] = at_load<u32x4_a>(ka + 64 * s, k_at[n]);
#pragma unroll
    for (int p = 0; p < X::PIECES; ++p) vn[p] = at_load<u32x4_a>(va, v_at[p]);
  };

  const float scale2 = a.scale * AT_LOG2E;
  floatx4_a o[MB][X::DB];
  float mx[MB], sum[MB];  // in the exp2 domain; `sum` over this lane's keys only
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    mx[m] = -INFINITY;
    sum[m] = 0.0f;
#pragma unroll
    for (int d = 0; d < X::DB; ++d) o[m][d] = at_zero();
  }
  float least = 0.0f;  // of the scores that no mask looked at: minus infinity where one is; NaN and infinity show in the sums
  bool bad = false;
  if (t_first + wave <= t_last) fetch(t_first + wave);
  for (int t = t_first + wave; t <= t_last; t += 4) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();  // the previous values have been read
#pragma unroll
    for (int p = 0; p < X::PIECES; ++p) {
      const int idx = lane + 64 * p;
      *reinterpret_cast<u32x4_a*>(region + idx / (D / 8) * X::PITCH + idx % (D / 8) * 16) = vn[p];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    floatx4_a s[MB][X::NB];
#pragma unroll
    for (int n = 0; n < X::NB; ++n)
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        s[m][n] = at_zero();
#pragma unroll
        for (int ks = 0; ks < X::KS; ++ks)
#pragma unroll
          for (int part = 2; part >= 0; --part) s[m][n] = at_mfma16(kn[n][ks], q[m][ks].part[part], s[m][n]);
      }
    if (t + 4 <= t_last) fetch(t + 4);
    const bool whole = t * X::KEYS + X::KEYS - 1 <= first_pos && t * X::KEYS >= last_low;  // (uniform)
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      float top = -INFINITY;
      if (whole) {
#pragma unroll
        for (int n = 0; n < X::NB; ++n)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            s[m][n][v] *= scale2;
            top = fmaxf(top, s[m][n][v]);
            least = fminf(least, s[m][n][v]);
          }
      } else {
#pragma unroll
        for (int n = 0; n < X::NB; ++n)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int key = t * X::KEYS + n * 16 + 4 * g + v;
            const bool seen = key <= pos[m] && key >= low[m];
            const float x = s[m][n][v] * scale2;
            bad |= seen && !dev_finite(x);
            s[m][n][v] = seen ? x : -INFINITY;
            top = fmaxf(top, s[m][n][v]);
          }
      }
      top = at_row_max(top);
      if (__any(top > mx[m])) {
        const float mx_new = fmaxf(mx[m], top);
        const float rescale = mx_new == mx[m] ? 1.0f : __builtin_amdgcn_exp2f(mx[m] - mx_new);  // 0 on the first keys
        mx[m] = mx_new;
        sum[m] *= rescale;
#pragma unroll
        for (int d = 0; d < X::DB; ++d)
#pragma unroll
          for (int v = 0; v < 4; ++v) o[m][d][v] *= rescale;
      }
      const float base = mx[m] == -INFINITY ? 0.0f : mx[m];
#pragma unroll
      for (int n = 0; n < X::NB; ++n)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          s[m][n][v] = __builtin_amdgcn_exp2f(s[m][n][v] - base);
          sum[m] += s[m][n][v];
        }
    }
    // 32 keys at a time: a lane's eight are 4 g + v of two blocks, and so are the transposed values'.
#pragma unroll
    for (int h = 0; h < X::NB / 2; ++h) {
      AtParts p[MB];
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const float x[8] = {s[m][2 * h][0], s[m][2 * h][1], s[m][2 * h][2], s[m][2 * h][3],
                            s[m][2 * h + 1][0], s[m][2 * h + 1][1], s[m][2 * h + 1][2], s[m][2 * h + 1][3]};
        p[m].cut(x);
      }
      u32x4_a value[X::DB];
#pragma unroll
      for (int d = 0; d < X::DB; ++d) {
        typedef short4_a __attribute__((address_space(3))) * lds_ptr;
        char* at_v = region + (32 * h + 4 * g + (i >> 2)) * X::PITCH + 32 * d + (i & 3) * 8;
        const short4_a lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(at_v));
        const short4_a hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(at_v + 16 * X::PITCH));
        const uint2 l = __builtin_bit_cast(uint2, lo), u = __builtin_bit_cast(uint2, hi);
        value[d] = u32x4_a{l.x, l.y, u.x, u.y};
      }
#pragma unroll
      for (int n = 2; n >= 0; --n)  // over all sums between two products of one: these wait for each other (17.8 -> 17.5 us at 4 x 12, 256 of 700)
#pragma unroll
        for (int d = 0; d < X::DB; ++d)
#pragma unroll
          for (int m = 0; m < MB; ++m)
            o[m][d] = at_mfma16(value[d], p[m].part[n], o[m][d]);
    }
  }
  bad |= least == -INFINITY;
#pragma unroll
  for (int m = 0; m < MB; ++m) bad |= !dev_finite(sum[m]);
  // The four waves' shares of the same rows: wave w adds up the column blocks w, w + 4, ...
  float* stat = reinterpret_cast<float*>(lds);                // [4][2][16]
  float4* part = reinterpret_cast<float4*>(lds + 512);        // [4][DB][64]
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const float all_keys = at_row_sum(sum[m]);
    __syncthreads();
    if (g == 0) {
      stat[wave * 32 + i] = mx[m];
      stat[wave * 32 + 16 + i] = all_keys;
    }
#pragma unroll
    for (int d = 0; d < X::DB; ++d) part[(wave * X::DB + d) * 64 + lane] = make_float4(o[m][d][0], o[m][d][1], o[m][d][2], o[m][d][3]);
    __syncthreads();
    float all = -INFINITY, weight[4], total = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) all = fmaxf(all, stat[w * 32 + i]);
    const float base = all == -INFINITY ? 0.0f : all;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      weight[w] = __builtin_amdgcn_exp2f(stat[w * 32 + i] - base);
      total = fmaf(weight[w], stat[w * 32 + 16 + i], total);
    }
    if (r0 + m * 16 + i < rows) {
      if constexpr (SPLIT) {
        if (wave == 0 && g == 0) {
          float* row = at_partial(a, D, b, kvh, at[m].query, at[m].head);
          row[D] = all * AT_LN2;
          row[D + 1] = total;
        }
      } else {
        bad |= !(dev_finite(total) && total > 0.0f);
      }
      const float f = SPLIT ? 1.0f : 1.0f / total;
      float* out = SPLIT ? at_partial(a, D, b, kvh, at[m].query, at[m].head) : a.out + b * a.o_b + (static_cast<long>(kvh) * a.rep + at[m].head) * a.o_h + static_cast<long>(at[m].query) * a.o_t;
#pragma unroll
      for (int d0 = 0; d0 < X::DB; d0 += 4) {
        float x[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const float4 y = part[(w * X::DB + d0 + wave) * 64 + lane];
          x[0] = fmaf(weight[w], y.x, x[0]);
          x[1] = fmaf(weight[w], y.y, x[1]);
          x[2] = fmaf(weight[w], y.z, x[2]);
          x[3] = fmaf(weight[w], y.w, x[3]);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          x[v] *= f;
          bad |= !dev_finite(x[v]);
        }
        float* to = out + (d0 + wave) * 16 + 4 * g;
        if constexpr (SPLIT) {  // (a part's rows are 8-byte aligned)
#pragma unroll
          for (int v = 0; v < 4; ++v) to[v] = x[v];
        } else {
          *reinterpret_cast<float4*>(to) = make_float4(x[0], x[1], x[2], x[3]);
        }
      }
    }
  }
  if (bad) dev_raise_fault(a.fault, a.tag);
}

// ---------------------------------------------------------------- backward
// p and dS of one lane's four scores, from the score and dP accumulators.
struct AtGrad {
  float scale, scale2;
  __device__ __forceinline__ void operator()(bool seen, float score, float dp, float lse2, float delta, float* p, float* ds,
                                             bool* bad) const {
    const float x = score * scale2;
    const float pr = seen ? __builtin_amdgcn_exp2f(x - lse2) : 0.0f;
    *bad |= seen && !(dev_finite(x) && dev_finite(pr));
    *p = pr;
    *ds = seen ? scale * (pr * (dp - delta)) : 0.0f;
  }
  // The same for a score that is seen; `check` turns NaN where the other form says bad.
  __device__ __forceinline__ void whole(float score, float dp, float lse2, float delta, float* p, float* ds, float* check) const {
    const float x = score * scale2;
    *p = __builtin_amdgcn_exp2f(x - lse2);
    *check = fmaf(x, 0.0f, fmaf(*p, 0.0f, *check));
    *ds = scale * (*p * (dp - delta));
  }
};

// dQ, and the row term delta = dO . O when `out` is given (it is read from `delta` otherwise).
// Three workgroups per compute unit at D = 64, KW = 4: left to itself the compiler takes 172
// registers, which is two, and 780 workgroups (2 x 8 heads, 777 rows, window 256) leave most of the
// second of their two rounds idle. At 152, without spills, they fit one: backward 58.8 -> 54.9 us
// (360 rows, 32 planes 53.3 -> 49.7). At D = 128 a bound of two spills and costs 8-28 %: none there.
template <int D, int KW>
constexpr int at_dq_lds() { return KW == 1 ? 2 * AT_ROWS * AtDim<D>::P : 4 * 16 * AtDim<D>::P; }
template <int D, int KW>
__device__ __forceinline__ void at_dq(const Sdpa32Args& a, AtPlace place, int blocks, float* lds) {
  using X = AtDim<D>;
  constexpr int QW = 4 / KW, BQ = 16 * QW, BLOCKS = KW == 1 ? 4 : 1, KEYS = 16 * BLOCKS;
  static_assert(16 * X::P >= X::S * 256, "the waves' sums fit");
  float* kt = lds;
  float* vt = lds + AT_ROWS * X::P;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)), i = lane & 15, g = lane >> 4;
  const int qw = wave % QW, kw = wave / QW;
  const int b = place.plane / a.kv_heads, kvh = place.plane - b * a.kv_heads;
  const int rows = a.tq * a.rep;
  const int r0 = (blocks - 1 - place.block) * BQ;
  const int r = r0 + qw * 16 + i;
  const AtRow at = at_unpack(min(r, rows - 1), a.rep);
  const long head = static_cast<long>(kvh) * a.rep + at.head;
  const long q_at = b * a.q_b + head * a.q_h + static_cast<long>(at.query) * a.q_t;
  const long o_at = b * a.o_b + head * a.o_h + static_cast<long>(at.query) * a.o_t;
  float4 q[X::S], dout[X::S];
  at_own<D>(a.q + q_at, q, g);
  at_own<D>(a.gy + o_at, dout, g);
  const long stat = (static_cast<long>(b) * a.kv_heads * a.rep + head) * a.tq + at.query;
  float delta;
  if (a.out) {
    float4 saved[X::S];
    at_own<D>(a.out + o_at, saved, g);
    delta = 0.0f;
#pragma unroll
    for (int s = 0; s < X::S; ++s)
      delta += dout[s].x * saved[s].x + dout[s].y * saved[s].y + dout[s].z * saved[s].z + dout[s].w * saved[s].w;
    delta = at_row_sum(delta);
    if (g == 0 && kw == 0 && r < rows) a.delta[stat] = delta;
  } else {
    delta = a.delta[stat];
  }
  const float lse2 = a.lse[stat] * AT_LOG2E;
  const int pos = r < rows ? at.query : -1;
  const int low = a.window > 0 ? max(0, pos + 1 - a.window) : 0;
  const int first_pos = at_unpack(r0, a.rep).query, last_pos = at_unpack(min(r0 + BQ, rows) - 1, a.rep).query;
  const int t_first = (a.window > 0 ? max(0, first_pos + 1 - a.window) : 0) / KEYS, t_last = last_pos / KEYS;
  const float* kb = static_cast<const float*>(a.k) + b * a.k_b + kvh * a.k_h;
  const float* vb = static_cast<const float*>(a.v) + b * a.k_b + kvh * a.k_h;
  const AtGrad grad{a.scale, a.scale * AT_LOG2E};
  floatx4_a dq[X::S];
#pragma unroll
  for (int m = 0; m < X::S; ++m) dq[m] = at_zero();
  bool bad = false;
  // dS of keys key0 + 4 g + v, from the scores and dP; without masks where every row sees them all.
  const int whole_to = r0 + BQ <= rows ? first_pos : -1, whole_from = a.window > 0 ? max(0, last_pos + 1 - a.window) : 0;
  float check = 0.0f;
  auto slopes = [&](const floatx4_a& s, const floatx4_a& dp, int key0) {
    floatx4_a ds;
    const bool whole = key0 + 15 <= whole_to && key0 >= whole_from;  // (uniform)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int key = key0 + 4 * g + v;
      float p, d;
      if (whole) grad.whole(s[v], dp[v], lse2, delta, &p, &d, &check);
      else grad(key <= pos && key >= low, s[v], dp[v], lse2, delta, &p, &d, &bad);
      ds[v] = d;
    }
    return ds;
  };
  if constexpr (KW == 1) {
    AtTile<D, float> kn, vn;
    auto fetch = [&](int t) {
      kn.fetch([&](int row) { const int key = t * AT_ROWS + row; return key < a.tk ? kb + static_cast<long>(key) * a.k_t : nullptr; });
      vn.fetch([&](int row) { const int key = t * AT_ROWS + row; return key < a.tk ? vb + static_cast<long>(key) * a.k_t : nullptr; });
    };
    fetch(t_first);
    for (int t = t_first; t <= t_last; ++t) {
      __syncthreads();
      kn.store(kt);
      vn.store(vt);
      __syncthreads();
      if (t < t_last) fetch(t + 1);
#pragma unroll
      for (int n = 0; n < BLOCKS; ++n) {
        const int row = n * 16;
        const floatx4_a s = at_dot<D>(kt + row * X::P, q, i, g);
        const floatx4_a dp = at_dot<D>(vt + row * X::P, dout, i, g);
        at_accumulate<D>(kt + row * X::P, slopes(s, dp, t * AT_ROWS + row), dq, i, g);
      }
    }
  } else {
    // Keys and values come straight into the first two products' operands, a whole block ahead; the keys' other form goes through
    // LDS of the wave's own. (Keys past the last one are read from it; their dS is 0.)
    AtDotBlock<D, float> keys[2], values[2];
    float* const own = lds + kw * (16 * X::P);
    const unsigned pitch = static_cast<unsigned>(a.k_t) * 4u, off0 = i * pitch + 16u * g;
    auto fetch = [&](int set, int t) {
      const int key0 = t * KEYS;
      unsigned off = off0;
      if (key0 + KEYS > a.tk) off = min(i, a.tk - 1 - key0) * pitch + 16u * g;
      keys[set].fetch(at_bytes(kb + key0 * a.k_t), off);
      values[set].fetch(at_bytes(vb + key0 * a.k_t), off);
    };
    auto step = [&](int set, int t) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();  // the previous block has been read
      at_stage<D>(keys[set], own, i, g);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      fetch(set ^ 1, min(t + KW, t_last));
      const floatx4_a s = keys[set].dot(q), dp = values[set].dot(dout);
      at_accumulate<D>(own, slopes(s, dp, t * KEYS), dq, i, g);
    };
    int t = t_first + kw;
    if (t <= t_last) fetch(0, t);
    for (; t <= t_last; t += 2 * KW) {
      step(0, t);
      if (t + KW > t_last) break;
      step(1, t + KW);
    }
  }
  bad |= check != 0.0f;
  float* out = a.gq + q_at;
  if constexpr (KW == 1) {
    if (r < rows) bad |= at_store<D, 4>(out, dq, 1.0f, g, 0);
  } else {
    __syncthreads();
    float* part = lds;  // [4][S * 4][64]
#pragma unroll
    for (int m = 0; m < X::S; ++m)
#pragma unroll
      for (int v = 0; v < 4; ++v) part[((kw * X::S + m) * 4 + v) * 64 + lane] = dq[m][v];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < X::S; ++m) {
      float x = 0.0f;
#pragma unroll
      for (int w = 0; w < 4; ++w) x += part[((w * X::S + m) * 4 + kw) * 64 + lane];
      dq[m] = floatx4_a{x, x, x, x};
    }
    if (r < rows) bad |= at_store<D, 1>(out, dq, 1.0f, g, kw);
  }
  if (bad) dev_raise_fault(a.fault, a.tag);
}
template <int D, int KW>
__global__ __launch_bounds__(AT_THREADS, D == 64 && KW == 4 ? 3 : 1) void sdpa32_dq_kernel(Sdpa32Args a) {
  __shared__ __align__(16) float lds[at_dq_lds<D, KW>()];
  at_dq<D, KW>(a, at_place(), static_cast<int>(gridDim.x), lds);
}

// dK and dV of 16 KG keys, over a share (blockIdx.z of gridDim.z) of the row tiles that see them.
// Two workgroups per compute unit at D = 128, RW = 1 (LDS allows two; without the bound registers
// allow one): 512 rows of 64 planes, backward 308 -> 278 us; 12 bytes of a lane go to scratch.
// OWN: each row's delta is formed here, from `out`, and not read from what the dQ pass left (RW = 4).
template <int D, int RW>
constexpr int at_dkv_lds() { return RW == 1 ? 2 * AT_ROWS * AtDim<D>::P + 2 * AT_ROWS : 4 * 2 * 16 * AtDim<D>::P; }
template <int D, int RW, bool OWN>  // RW waves share a tile's rows, 4 / RW take 16 keys each
__device__ __forceinline__ void at_dkv(const Sdpa32Args& a, AtPlace place, int part, int parts, int planes, float* lds) {
  using X = AtDim<D>;
  // RW = 4: nothing but the waves' sums goes through LDS; row tiles are blocks of 16 rows.
  constexpr int KG = 4 / RW, BK = 16 * KG, NB = AT_ROWS / 16, ROWS = RW == 1 ? AT_ROWS : 16;
  float* qt = lds;
  float* gt = lds + AT_ROWS * X::P;
  float* lse_t = gt + AT_ROWS * X::P;
  float* delta_t = lse_t + AT_ROWS;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)), i = lane & 15, g = lane >> 4;
  const int kg = wave % KG, rw = wave / KG;
  const int b = place.plane / a.kv_heads, kvh = place.plane - b * a.kv_heads;
  const int rows = a.tq * a.rep;
  const int j0 = place.block * BK, key = j0 + kg * 16 + i;
  const long k_at = b * a.k_b + kvh * a.k_h + static_cast<long>(min(key, a.tk - 1)) * a.k_t;
  float4 k[X::S], v4[X::S];
  at_own<D>(static_cast<const float*>(a.k) + k_at, k, g);
  at_own<D>(static_cast<const float*>(a.v) + k_at, v4, g);
  // Queries that see key j: j .. min(T - 1, j + window - 1). Row tiles from the first key's to the last key's.
  const int key_last = min(j0 + BK, a.tk) - 1;
  const int q_last = a.window > 0 ? min(a.tk - 1, key_last + a.window - 1) : a.tk - 1;
  const int u_first = j0 * a.rep / ROWS, u_end = ((q_last + 1) * a.rep + ROWS - 1) / ROWS;
  const int share = (u_end - u_first + parts - 1) / parts;
  const int u0 = u_first + part * share, u1 = min(u_end, u0 + share);
  const long stat_b = (static_cast<long>(b) * a.kv_heads + kvh) * a.rep;
  const float* qb = a.q + b * a.q_b + static_cast<long>(kvh) * a.rep * a.q_h;
  const float* gb = a.gy + b * a.o_b + static_cast<long>(kvh) * a.rep * a.o_h;
  const AtGrad grad{a.scale, a.scale * AT_LOG2E};
  floatx4_a dk[X::S], dv[X::S];
#pragma unroll
  for (int m = 0; m < X::S; ++m) dk[m] = dv[m] = at_zero();
  bool bad = false;
  if constexpr (RW == 1) {
    AtTile<D, float> qn, gn;
    float lse_n = 0.0f, delta_n = 0.0f;
    auto fetch = [&](int u) {
      auto row_of = [&](int row, long h_stride, long t_stride) {
        const AtRow x = at_unpack(u * AT_ROWS + row, a.rep);
        return x.head * h_stride + static_cast<long>(x.query) * t_stride;
      };
      qn.fetch([&](int row) { return u * AT_ROWS + row < rows ? qb + row_of(row, a.q_h, a.q_t) : nullptr; });
      gn.fetch([&](int row) { return u * AT_ROWS + row < rows ? gb + row_of(row, a.o_h, a.o_t) : nullptr; });
      if (threadIdx.x < AT_ROWS && u * AT_ROWS + static_cast<int>(threadIdx.x) < rows) {
        const AtRow x = at_unpack(u * AT_ROWS + threadIdx.x, a.rep);
        const long at = (stat_b + x.head) * a.tq + x.query;
        lse_n = a.lse[at] * AT_LOG2E;
        delta_n = a.delta[at];
      }
    };
    if (u0 < u1) fetch(u0);
    for (int u = u0; u < u1; ++u) {
      __syncthreads();
      qn.store(qt);
      gn.store(gt);
      if (threadIdx.x < AT_ROWS) {
        lse_t[threadIdx.x] = lse_n;
        delta_t[threadIdx.x] = delta_n;
      }
      __syncthreads();
      if (u + 1 < u1) fetch(u + 1);
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        const int row = n * 16;
        const floatx4_a s = at_dot<D>(qt + row * X::P, k, i, g);
        const floatx4_a dp = at_dot<D>(gt + row * X::P, v4, i, g);
        const float4 l4 = *reinterpret_cast<const float4*>(lse_t + row + 4 * g);
        const float4 d4 = *reinterpret_cast<const float4*>(delta_t + row + 4 * g);
        const float lv[4] = {l4.x, l4.y, l4.z, l4.w}, dl[4] = {d4.x, d4.y, d4.z, d4.w};
        floatx4_a p, ds;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int packed = u * AT_ROWS + row + 4 * g + v, query = at_unpack(packed, a.rep).query;
          const bool seen = packed < rows && key < a.tk && key <= query && (a.window == 0 || query < key + a.window);
          float pv, dsv;
          grad(seen, s[v], dp[v], lv[v], dl[v], &pv, &dsv, &bad);
          p[v] = pv;
          ds[v] = dsv;
        }
        at_accumulate<D>(gt + row * X::P, p, dv, i, g);
        at_accumulate<D>(qt + row * X::P, ds, dk, i, g);
      }
    }
  } else {
    // Rows past the last one are read from it; their weights are 0.
    const AtUnpack unpack(a.rep);
    const unsigned q_pitch = static_cast<unsigned>(a.q_t) * 4u, o_pitch = static_cast<unsigned>(a.o_t) * 4u;
    const unsigned q_head = static_cast<unsigned>(a.q_h) * 4u, o_head = static_cast<unsigned>(a.o_h) * 4u;
    // A block comes straight into the first two products' operands, a block ahead (a whole one where there are registers for
    // two); the other form goes through LDS of the wave's own.
    constexpr int SETS = D <= 64 ? 2 : 1;
    AtDotBlock<D, float> qn[SETS], gn[SETS], on[OWN ? SETS : 1];
    const float* ob = OWN ? a.out + b * a.o_b + static_cast<long>(kvh) * a.rep * a.o_h : nullptr;
    float lse_n[SETS][4], delta_n[SETS][4];
    float* const own_q = lds + rw * (2 * 16 * X::P);
    float* const own_g = own_q + 16 * X::P;
    int u = u0 + rw;
    float check = 0.0f;
    // Where 16 rows are whole queries of the group (1, 2, 4, 8 or 16 heads) a block's offsets from its first row never change.
    const bool even = 16 % a.rep == 0;
    const AtRow own0 = unpack(i);
    const unsigned q_off0 = own0.head * q_head + own0.query * q_pitch + 16u * g, g_off0 = own0.head * o_head + own0.query * o_pitch + 16u * g;
    unsigned stat0[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const AtRow y = unpack(4 * g + j);
      stat0[j] = (static_cast<unsigned>(y.head) * a.tq + y.query) * 4u;
    }
    auto fetch = [&](int set, int u_next) {
      const int first = 16 * u_next;
      const bool in_order = even && first + 16 <= rows;
      const long query0 = in_order ? unpack(first).query : 0;
      unsigned q_off = q_off0, g_off = g_off0, stat[4] = {stat0[0], stat0[1], stat0[2], stat0[3]};
      if (!in_order) {
        const AtRow x = unpack(min(first + i, rows - 1));
        q_off = x.head * q_head + x.query * q_pitch + 16u * g;
        g_off = x.head * o_head + x.query * o_pitch + 16u * g;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const AtRow y = unpack(min(first + 4 * g + j, rows - 1));
          stat[j] = (static_cast<unsigned>(y.head) * a.tq + y.query) * 4u;
        }
      }
      qn[set].fetch(at_bytes(qb + query0 * a.q_t), q_off);
      gn[set].fetch(at_bytes(gb + query0 * a.o_t), g_off);
      if constexpr (OWN) on[set].fetch(at_bytes(ob + query0 * a.o_t), g_off);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        lse_n[set][j] = at_load<float>(at_bytes(a.lse + stat_b * a.tq + query0), stat[j]);
        if constexpr (!OWN) delta_n[set][j] = at_load<float>(at_bytes(a.delta + stat_b * a.tq + query0), stat[j]);
      }
    };
    auto step = [&](int set, int u_now) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();  // the previous block has been read
      at_stage<D>(qn[set], own_q, i, g);
      at_stage<D>(gn[set], own_g, i, g);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if constexpr (SETS == 2) fetch(set ^ 1, min(u_now + RW, u1 - 1));
      const floatx4_a s = qn[set].dot(k), dp = gn[set].dot(v4);
      float lv[4], dl[4];
      float row = 0.0f;  // delta of row i, as the dQ pass sums it
      if constexpr (OWN) {
#pragma unroll
        for (int n = 0; n < X::S; ++n)
          row += gn[set].raw[n][0] * on[set].raw[n][0] + gn[set].raw[n][1] * on[set].raw[n][1] + gn[set].raw[n][2] * on[set].raw[n][2] + gn[set].raw[n][3] * on[set].raw[n][3];
        row = at_row_sum(row);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        lv[j] = lse_n[set][j] * AT_LOG2E;
        dl[j] = OWN ? __shfl(row, 4 * g + j) : delta_n[set][j];
      }
      if constexpr (SETS == 1) fetch(set, min(u_now + RW, u1 - 1));
      // Without masks where the block's first and last queries see every key (uniform).
      const int from = unpack(16 * u_now).query, to = unpack(16 * u_now + 15).query;
      const bool whole = from >= j0 + BK - 1 && 16 * u_now + 16 <= rows && j0 + BK <= a.tk && (a.window == 0 || to < j0 + a.window);
      floatx4_a p, ds;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float pv, dsv;
        if (whole) {
          grad.whole(s[v], dp[v], lv[v], dl[v], &pv, &dsv, &check);
        } else {
          const int packed = 16 * u_now + 4 * g + v, query = unpack(packed).query;
          const bool seen = packed < rows && key < a.tk && key <= query && (a.window == 0 || query < key + a.window);
          grad(seen, s[v], dp[v], lv[v], dl[v], &pv, &dsv, &bad);
        }
        p[v] = pv;
        ds[v] = dsv;
      }
      at_accumulate<D>(own_g, p, dv, i, g);
      at_accumulate<D>(own_q, ds, dk, i, g);
    };
    if (u < u1) fetch(0, u);
    for (; u < u1; u += RW * SETS) {
      step(0, u);
      if constexpr (SETS == 2) {
        if (u + RW >= u1) break;
        step(1, u + RW);
      }
    }
    bad |= check != 0.0f;
  }
  const bool split = parts > 1;
  const long plane = static_cast<long>(a.tk) * D;  // parts: [z][b, kv head][tk][D], dK's then dV's
  const long part_at = ((static_cast<long>(part) * planes + place.plane) * a.tk + min(key, a.tk - 1)) * D;
  float* ok = split ? a.parts + part_at : a.gk + k_at;
  float* ov = split ? a.parts + static_cast<long>(parts) * planes * plane + part_at : a.gv + k_at;
  if constexpr (RW == 1) {
    if (key < a.tk) {
      bad |= at_store<D, 4>(ok, dk, 1.0f, g, 0);
      bad |= at_store<D, 4>(ov, dv, 1.0f, g, 0);
    }
  } else {
    auto meet = [&](floatx4_a (&x)[X::S]) {
      __syncthreads();
#pragma unroll
      for (int m = 0; m < X::S; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v) lds[((rw * X::S + m) * 4 + v) * 64 + lane] = x[m][v];
      __syncthreads();
#pragma unroll
      for (int m = 0; m < X::S; ++m) {
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) sum += lds[((w * X::S + m) * 4 + rw) * 64 + lane];
        x[m] = floatx4_a{sum, sum, sum, sum};
      }
    };
    meet(dk);
    meet(dv);
    if (key < a.tk) {
      bad |= at_store<D, 1>(ok, dk, 1.0f, g, rw);
      bad |= at_store<D, 1>(ov, dv, 1.0f, g, rw);
    }
  }
  if (bad) dev_raise_fault(a.fault, a.tag);
}
template <int D, int RW>
__global__ __launch_bounds__(AT_THREADS, D == 128 && RW == 1 ? 2 : 1) void sdpa32_dkv_kernel(Sdpa32Args a) {
  __shared__ __align__(16) float lds[at_dkv_lds<D, RW>()];
  at_dkv<D, RW, false>(a, at_place(), static_cast<int>(blockIdx.z), static_cast<int>(gridDim.z), static_cast<int>(gridDim.y), lds);
}

// Both passes in one launch (at_bwd_together says when): the key side's workgroups, a part after the other, then the dQ pass's. The grid has
// planes along y as those of the two passes have, so that what their launches hold this one holds (an axis takes 2^32 threads, and 16384
// planes of 8192 positions come to 2^24 workgroups); a plane's are below 2^23, its rows of 16 values and more staying below 2^30 (at_narrow).
template <int D>
__global__ __launch_bounds__(AT_THREADS, 2) void sdpa32_bwd_kernel(Sdpa32Args a, unsigned planes, unsigned row_blocks, unsigned key_blocks, unsigned parts) {
  __shared__ __align__(16) float lds[at_dkv_lds<D, 4>() > at_dq_lds<D, 4>() ? at_dkv_lds<D, 4>() : at_dq_lds<D, 4>()];
  const unsigned index = blockIdx.y * gridDim.x + blockIdx.x, each = key_blocks * planes, keys = each * parts;
  if (index < keys) {
    const unsigned part = index / each;
    at_dkv<D, 4, true>(a, at_place(index - part * each, key_blocks, planes), static_cast<int>(part), static_cast<int>(parts), static_cast<int>(planes), lds);
  } else {
    at_dq<D, 4>(a, at_place(index - keys, row_blocks, planes), static_cast<int>(row_blocks), lds);
  }
}

// Adds up the parts of a split key / value pass, lowest rows first. blockIdx.y: 0 dK, 1 dV.
__global__ __launch_bounds__(AT_THREADS) void sdpa32_parts_kernel(Sdpa32Args a, int parts, int dim, long total) {
  const long n = static_cast<long>(blockIdx.x) * AT_THREADS + threadIdx.x;  // a 16-byte piece
  if (n * 4 >= total) return;
  const float* src = a.parts + static_cast<long>(blockIdx.y) * parts * total + n * 4;
  float4 t = *reinterpret_cast<const float4*>(src);
  for (int z = 1; z < parts; ++z) {
    const float4 u = *reinterpret_cast<const float4*>(src + z * total);
    t.x += u.x; t.y += u.y; t.z += u.z; t.w += u.w;
  }
  const long row = n * 4 / dim, plane = row / a.tk;
  const long b = plane / a.kv_heads, kvh = plane - b * a.kv_heads;
  float* dst = (blockIdx.y ? a.gv : a.gk) + b * a.k_b + kvh * a.k_h + (row - plane * a.tk) * a.k_t + (n * 4 - row * dim);
  *reinterpret_cast<float4*>(dst) = t;
  if (!(dev_finite(t.x) && dev_finite(t.y) && dev_finite(t.z) && dev_finite(t.w))) dev_raise_fault(a.fault, a.tag);
}

// Rows (keys) per workgroup: 64 that share every tile of the other side in LDS, or 16 whose waves take that side's blocks in
// turn, straight into operands, with no barrier before they meet. The second is ahead where 64 would leave compute units without a
// workgroup, and over a long other side (`span`) at any size: nothing waits for a tile there (16 heads x 4096: forward 587 ->
// 382 us, backward 1868 -> 1290; 2 x 12 x 1024: 92 -> 64, 290 -> 198; 8 x 12 x 512: 71 -> 78, 217 -> 266; planes over all L2s); over a short one its
// first loads and the meeting weigh more (16 x 12 x 64: 7.3 -> 8.7, 21 -> 26).
bool at_narrow(omx_ctx* ctx, const Sdpa32Args& a, long planes, long rows, long span) {
  // The second form's lane offsets are 32 bits of bytes over a plane, its row numbers 32 bits times the group's heads.
  const long limit = 1l << 30, heads = a.rep - 1l;
  if (a.capacity * a.k_t >= limit || a.tk * a.k_t >= limit || a.tq * a.q_t + heads * a.q_h >= limit || a.tq * a.o_t + heads * a.o_h >= limit ||
      (static_cast<long>(a.tq) * a.rep + 64) * a.rep >= 4 * limit)
    return false;
  const long blocks = planes * ((rows + 63) / 64), units = ctx->cu_count > 0 ? ctx->cu_count : 256;
  return span >= 1024 || blocks < (span >= 512 ? 2 * units : span > 128 ? units : units / 2);
}
// What one row's, or key's, other side comes to.
long at_span(const Sdpa32Args& a) { return a.window > 0 ? std::min<long>(a.tk, a.window + 15l) : a.tk; }

// Whether the two passes of the backward share a launch (16-row and 16-key workgroups of head_dim up to 64, the output at hand). The key side
// then forms delta itself, from the output's rows beside the gradient's, and nothing waits for the dQ pass: its workgroups
// fill in where the longer ones of the key side, which go out first, leave room. Every bit is the same. us of a backward, two launches / one (head
// dim 64): 2 x 8 over 2 x 777 in a window of 256: 54 / 44; the same without: 74 / 66; 1 x 4 x 128: 13.6 / 8.2; 8 x 4 x 256: 30 / 27;
// 4 over 1 x 1500: 79 / 65; 2 x 12 x 1024: 152 / 150; 2 x 2048: 78 / 83; 16 x 4096: 1125 / 1238; 2 x 8 x 500 x 16: 20 / 15.
// Gradients over what the other pass still reads (keys and values, or the output) take two launches, as they always could.
bool at_bwd_together(omx_ctx* ctx, const Sdpa32Args& a, int planes, int dim) {
  if (!a.out || (ctx->attention_together >= 0 ? ctx->attention_together == 0 : at_span(a) > 1536)) return false;
  struct Range {
    const char *first, *end;
  };
  const long batches = planes / a.kv_heads, heads = static_cast<long>(a.kv_heads) * a.rep;
  auto range = [&](const void* p, long b, long h, long t, long n, long rows) {
    const char* first = static_cast<const char*>(p);
    return Range{first, first + 4 * ((batches - 1) * b + (n - 1) * h + (rows - 1) * t + dim)};
  };
  const Range read[] = {range(a.q, a.q_b, a.q_h, a.q_t, heads, a.tq), range(a.k, a.k_b, a.k_h, a.k_t, a.kv_heads, a.tk),
                        range(a.v, a.k_b, a.k_h, a.k_t, a.kv_heads, a.tk), range(a.out, a.o_b, a.o_h, a.o_t, heads, a.tq),
                        range(a.gy, a.o_b, a.o_h, a.o_t, heads, a.tq)};
  const Range written[] = {range(a.gq, a.q_b, a.q_h, a.q_t, heads, a.tq), range(a.gk, a.k_b, a.k_h, a.k_t, a.kv_heads, a.tk),
                           range(a.gv, a.k_b, a.k_h, a.k_t, a.kv_heads, a.tk)};
  for (const Range& r : read)
    for (const Range& w : written)
      if (r.first < w.end && w.first < r.end) return false;
  return true;
}

// sdpa_prompt_kernel: bf16 caches of wider heads, unless a ring's rows lie past 32 bits of lane offset from its first (4 GiB and
// more of one batch entry's keys) and the keys that are read run past its end.
bool at_prompt(const Sdpa32Args& a, int dim, bool bf16_cache) {
  const bool wraps = static_cast<long>(a.slot0) + a.tk > a.capacity;
  return dim >= 64 && bf16_cache && a.k_t < 1l << 24 && !(wraps && a.capacity * a.k_t >= 1l << 31);
}

// Rows per workgroup of the forward.
long forward_rows(omx_ctx* ctx, const Sdpa32Args& a, int dim, long planes, long rows, bool bf16_cache) {
  if (at_prompt(a, dim, bf16_cache)) {
    // Twice the rows on a key's way where the chip has a workgroup of them for every unit and the fullest unit has less to do: one
    // takes 1.6 to 1.9 times as long as one of 16 rows. Workgroups of 16 rows, us with 16 / 32 rows: 512 17.0 / 13.9, 768 17.3 / 18.6,
    // 1024 17.8 / 15.2, 1152 24.4 / 24.2, 1536 35.2 / 32.8.
    const long units = ctx->cu_count > 0 ? ctx->cu_count : 256, few = (rows + 31) / 32 * planes, many = (rows + 15) / 16 * planes;
    return dim == 64 && few >= units && 7 * ((few + units - 1) / units) < 4 * ((many + units - 1) / units) ? 32 : 16;
  }
  return at_narrow(ctx, a, planes, rows, at_span(a)) ? 16 : 64;
}

template <int D>
int32_t forward(omx_ctx* ctx, const Sdpa32Args& a, int planes, bool bf16_cache) {
  const long rows = static_cast<long>(a.tq) * a.rep, per = forward_rows(ctx, a, D, planes, rows, bf16_cache);
  const dim3 grid(static_cast<unsigned>((rows + per - 1) / per), planes, static_cast<unsigned>(std::max(1, a.nparts)));
  if constexpr (D >= 64) {
    if (at_prompt(a, D, bf16_cache)) {  // (attention over a cache has no lse)
      const bool two = per == 32, split = a.nparts > 1;  // (two: a workgroup per compute unit and more, never split)
      if constexpr (D == 64) {
        if (two) omx_launch(ctx, (sdpa_prompt_kernel<D, 2, false>), grid, dim3(AT_THREADS), 0, a);
      }
      if (!two) omx_launch(ctx, (split ? &sdpa_prompt_kernel<D, 1, true> : &sdpa_prompt_kernel<D, 1, false>), grid, dim3(AT_THREADS), 0, a);
      OMX_LAUNCH_CHECK(ctx, "sdpa_prompt_kernel");
      return OMX_OK;
    }
  }
  const bool narrow = per == 16;
  if (!bf16_cache) omx_launch(ctx, (narrow ? &sdpa32_fwd_kernel<D, 4, float> : &sdpa32_fwd_kernel<D, 1, float>), grid, dim3(AT_THREADS), 0, a);
  else if (!narrow) omx_launch(ctx, (sdpa32_fwd_kernel<D, 1, unsigned short>), grid, dim3(AT_THREADS), 0, a);
  else if constexpr (D < 64) omx_launch(ctx, (sdpa32_fwd_kernel<D, 4, unsigned short>), grid, dim3(AT_THREADS), 0, a);
  else return omx_fail(ctx, OMX_UNSUPPORTED, "cached attention: no narrow form over bf16 caches of head_dim %d", D);  // (prompt or wide)
  OMX_LAUNCH_CHECK(ctx, "sdpa32_fwd_kernel");
  return OMX_OK;
}

template <int D>
int32_t backward(omx_ctx* ctx, Sdpa32Args a, int planes) {
  const long rows = static_cast<long>(a.tq) * a.rep;
  const bool row_narrow = at_narrow(ctx, a, planes, rows, at_span(a));
  const long bq = row_narrow ? 16 : 64, row_blocks = (rows + bq - 1) / bq;
  const bool narrow = at_narrow(ctx, a, planes, a.tk, at_span(a) * a.rep);
  const long bk = narrow ? 16 : 64, blocks = (a.tk + bk - 1) / bk;
  // Into how many parts the rows are split: two workgroups per compute unit or more, as long as a share keeps two tiles of 64. Under the
  // causal mask, where the first keys' workgroups are the longest, more where that is less of: their steps, 0.8 us each at head_dim 64,
  // 0.45 times for each workgroup of a compute unit (the longest go out first, the shorter ones fill in), and for parts a second launch
  // with their write and read. (In a window all are as long: 57 us with two parts, 61 with four over 777 in 256. One is 54, but a
  // part's sum is a chain, and one chain's error against 64 bits was 13 % larger.) Backward, us, without the second rule / now:
  // 8 heads over 2 x 777, batch 2: 89 / 74; 8 over 4 x 777 x 128: 152 / 130; 4 over 1 x 2048: 132 / 121; 2 over 1 x 3000 x 128: 270 / 216.
  const long seen = a.window > 0 ? std::min<long>(a.tk, a.window + bk) : a.tk;
  const long tiles = std::max<long>(1, seen * a.rep / AT_ROWS), units = ctx->cu_count > 0 ? ctx->cu_count : 256;
  auto cost = [&](long p) {
    const double shared = std::max(1.0, 0.45 * static_cast<double>(planes * blocks * p) / static_cast<double>(units));
    return 0.0125 * D * static_cast<double>((tiles + p - 1) / p) * shared + (p > 1 ? 3.0 + 0.5 * static_cast<double>(p) : 0.0);
  };
  long parts = std::max<long>(1, std::min<long>(2l * units / (planes * blocks), tiles / 2));
  if (a.window <= 0 || a.window >= a.tk)
    for (long p = parts + 1; p <= std::min(tiles / 2, 64l); ++p)
      if (cost(p) < cost(parts)) parts = p;
  const long total = static_cast<long>(planes) * a.tk * D;
  while (parts > 1 && parts * total * 8 > (256l << 20)) --parts;
  // (as many as there is room for, down to one workgroup's walk over all rows)
  for (; parts > 1; --parts)
    if ((a.parts = static_cast<float*>(omx_workspace_if_room(ctx, static_cast<uint64_t>(parts) * total * 8, 1)))) break;
  // In one launch where the other side is short enough for the ends of two to weigh more than the third workgroup per compute unit that the
  // dQ pass has alone (at_bwd_together).
  if (D <= 64 && narrow && row_narrow && at_bwd_together(ctx, a, planes, D)) {
    if constexpr (D <= 64)
      omx_launch(ctx, sdpa32_bwd_kernel<D>, dim3(static_cast<unsigned>(row_blocks + blocks * parts), planes), dim3(AT_THREADS), 0, a,
                 static_cast<unsigned>(planes), static_cast<unsigned>(row_blocks), static_cast<unsigned>(blocks), static_cast<unsigned>(parts));
    OMX_LAUNCH_CHECK(ctx, "sdpa32_bwd_kernel");
  } else {
    const dim3 row_grid(static_cast<unsigned>(row_blocks), planes), grid(static_cast<unsigned>(blocks), planes, static_cast<unsigned>(parts));
    if (row_narrow) omx_launch(ctx, (sdpa32_dq_kernel<D, 4>), row_grid, dim3(AT_THREADS), 0, a);
    else omx_launch(ctx, (sdpa32_dq_kernel<D, 1>), row_grid, dim3(AT_THREADS), 0, a);
    OMX_LAUNCH_CHECK(ctx, "sdpa32_dq_kernel");
    if (narrow) omx_launch(ctx, (sdpa32_dkv_kernel<D, 4>), grid, dim3(AT_THREADS), 0, a);
    else omx_launch(ctx, (sdpa32_dkv_kernel<D, 1>), grid, dim3(AT_THREADS), 0, a);
    OMX_LAUNCH_CHECK(ctx, "sdpa32_dkv_kernel");
  }
  if (parts > 1) {
    omx_launch(ctx, sdpa32_parts_kernel, dim3(static_cast<unsigned>((total / 4 + AT_THREADS - 1) / AT_THREADS), 2), dim3(AT_THREADS), 0, a, static_cast<int>(parts), D, total);
    OMX_LAUNCH_CHECK(ctx, "sdpa32_parts_kernel");
  }
  return OMX_OK;
}

}  // namespace

bool omx_sdpa32_supports(uint64_t dim, uint64_t planes, std::initializer_list<const void*> ptrs, std::initializer_list<long> strides) {
  if ((dim != 16 && dim != 32 && dim != 64 && dim != 128) || planes > 65535) return false;
  for (const void* p : ptrs)
    if (reinterpret_cast<uintptr_t>(p) & 15u) return false;
  for (long s : strides)
    if (s % 4 != 0) return false;
  return true;
}

// A workgroup's chain of steps (each one set of keys for all of its rows) in us, slower by what shares its compute unit (the
// bf16 form is bound by vector instructions, two workgroups of the f32 one take 1.36 times as long as one), against a second
// launch that adds the parts up, 0.55 us for each. 16 heads over one KV head x 64, one new token, 8192 positions, one
// workgroup without parts: 68 -> 20 us over a bf16 cache, 204 -> 28 over an f32 one; 12 heads x 16 new tokens 70 -> 20 and
// 206 -> 30; 1024 positions 12.5 -> 11 and 28 -> 14. (The kernels for few rows: 85, 85; 82, 88; 24, 24.)
int omx_sdpa32_key_parts(omx_ctx* ctx, const Sdpa32Args& a, int batch, int dim, bool bf16_cache) {
  const long rows = static_cast<long>(a.tq) * a.rep, planes = static_cast<long>(batch) * a.kv_heads;
  const long per = forward_rows(ctx, a, dim, planes, rows, bf16_cache), blocks = (rows + per - 1) / per * planes;
  const bool prompt = at_prompt(a, dim, bf16_cache);
  const long keys = prompt ? 4 * (4096 / dim) : AT_ROWS;
  const double step = prompt ? (dim == 64 ? 2.0 : 1.45) : 0.5 + 0.0175 * dim;
  const long steps = (a.tk + keys - 1) / keys, cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
  const long most = per == 32 ? 1 : std::min(std::min(2 * cus / blocks, steps), 64l);  // (32 rows: no form for parts)
  long best = 1;
  double least = 0.0;
  for (long p = 1; p <= std::max(1l, most); ++p) {
    const long shared = (blocks * p + cus - 1) / cus;  // on the fullest compute unit
    const double slower = shared == 1 ? 1.0 : prompt ? static_cast<double>(shared) : 0.68 * static_cast<double>(shared);
    const double us = static_cast<double>((steps + p - 1) / p) * step * slower + (p > 1 ? 3.0 + 0.55 * static_cast<double>(p) : 0.0);
    if (p == 1 || us < least) {
      best = p;
      least = us;
    }
  }
  return static_cast<int>(best);
}

int32_t omx_sdpa32_forward(omx_ctx* ctx, const Sdpa32Args& a, int batch, int dim, bool bf16_cache) {
  const int planes = batch * a.kv_heads;
  if (dim == 16) return forward<16>(ctx, a, planes, bf16_cache);
  if (dim == 32) return forward<32>(ctx, a, planes, bf16_cache);
  if (dim == 64) return forward<64>(ctx, a, planes, bf16_cache);
  return forward<128>(ctx, a, planes, bf16_cache);
}

int32_t omx_sdpa32_backward(omx_ctx* ctx, const Sdpa32Args& a, int batch, int dim) {
  const int planes = batch * a.kv_heads;
  if (dim == 16) return backward<16>(ctx, a, planes);
  if (dim == 32) return backward<32>(ctx, a, planes);
  if (dim == 64) return backward<64>(ctx, a, planes);
  return backward<128>(ctx, a, planes);
}
