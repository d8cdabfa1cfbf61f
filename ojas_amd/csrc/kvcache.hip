// KV-cache attention for decode (and prefill onto a non-empty cache) and the cache write.
//
// Reference: BackendModule::cached_attention_forward / kv_cache_write
// (ojas-core/src/backend.rs:2526-2565; validators ojas-core/src/shapes.rs:2758-2879; CPU
// ojas-cpu/src/kv.rs). Caches are time-major rings [B, Tcap, Hkv, D]: position j lives in slot
// j % Tcap. Query i of Tq sits at position p = kv_len - Tq + i and attends to positions
// first..=p (first = 0, or p + 1 - window); head h reads KV head h / (H / Hkv).
//
// The op is bound by reading the cache once. One wave per block walks a run of 64-key tiles for up
// to 8 query rows that share a KV head (the heads of a group and/or consecutive queries), so the
// keys and values of a group are read once for all of its query heads:
//   * the K and V tiles are loaded with 16-byte coalesced reads into LDS;
//   * scores: lane j owns key j and reads its row from LDS (row pitch dim + 4 floats, so the 16
//     lanes a clock serves hit 64 distinct banks); the query rows are LDS broadcasts;
//   * softmax statistics are kept online per row (running max and sum), exact rescaling;
//   * values: lane d owns output column d (+ 64, 128, 192), the key's weight comes from its lane
//     with a readlane.
// Each block writes one partial (unnormalised output, max, sum) per row; a second kernel merges a
// row's partials in ascending order, so the result does not depend on scheduling.
// Values read from the cache or the queries that are NaN or infinite, and scores that overflow,
// raise the deferred fault; slots no query reads are never touched.
#include <algorithm>

#include "omx_common.h"
#include "sdpa_mfma32.h"

namespace {

constexpr int KV_TILE = 64;  // keys per tile
constexpr int KV_ROWS = 8;   // query rows per block

struct KvArgs {
  const float* q;
  const void* k_cache;
  const void* v_cache;
  float* partial;  // [rows_total][nparts][dim + 2]
  float* out;
  int batch, tq, heads, kv_heads, dim, capacity, group;
  long kv_len, window, read_lo;
  int tiles_per_block, nparts;
  unsigned int read_slot;  // the ring's slot of position read_lo
  float scale;
  OmxFaultWord* fault;
  unsigned long long tag;
};

// Copies tile rows [pos0, pos0 + 64) of one KV head of both caches into LDS, widened to f32; rows
// at or past kv_len become zeros. A lane's 16-byte pieces are chunk indices lane, lane + 64, ...
// of the tile's 64 * dim / 4; (key0, piece0) locates chunk `lane`. Loads are issued eight keys'
// worth at a time for each cache before any is used, so their latencies overlap.
// Returns whether a value read was not finite.
constexpr int KV_BATCH = 8;
template <typename T>
__device__ __forceinline__ bool load_tiles(const T* __restrict__ kc, const T* __restrict__ vc, float* __restrict__ kt,
                                           float* __restrict__ vt, const KvArgs& a, long base_b, int kvh, long pos0,
                                           int key0, int piece0) {
  bool bad = false;
  const int dim = a.dim, pieces = dim >> 2, kpitch = dim + 4;
  const int step_keys = 64 / pieces, step_pieces = 64 - step_keys * pieces;  // chunk index + 64
  const int slot0 = static_cast<int>(pos0 % a.capacity);
  const int live = static_cast<int>(min(static_cast<long>(KV_TILE), a.kv_len - pos0));
  int key = key0, piece = piece0;
  for (int done = 0; done < pieces; done += KV_BATCH) {  // a lane has `pieces` chunks per tile
    float kv[KV_BATCH][4], vv[KV_BATCH][4];
    int at_key[KV_BATCH], at_d[KV_BATCH];
#pragma unroll
    for (int i = 0; i < KV_BATCH; ++i) {
      at_key[i] = key;
      at_d[i] = piece << 2;
#pragma unroll
      for (int e = 0; e < 4; ++e) kv[i][e] = vv[i][e] = 0.0f;
      if (done + i < pieces && key < live) {
        int slot = slot0 + key;  // the positions of a tile wrap the ring at most once
        slot = slot >= a.capacity ? slot - a.capacity : slot;
        const size_t off = static_cast<size_t>(((base_b + slot) * a.kv_heads + kvh) * dim + at_d[i]);
        dev_load4(kc, off, kv[i]);
        dev_load4(vc, off, vv[i]);
      }
      key += step_keys;
      piece += step_pieces;
      if (piece >= pieces) {
        piece -= pieces;
        ++key;
      }
    }
#pragma unroll
    for (int i = 0; i < KV_BATCH; ++i) {
      if (done + i < pieces) {
        bad |= !(dev_finite(kv[i][0]) && dev_finite(kv[i][1]) && dev_finite(kv[i][2]) && dev_finite(kv[i][3]) &&
                 dev_finite(vv[i][0]) && dev_finite(vv[i][1]) && dev_finite(vv[i][2]) && dev_finite(vv[i][3]));
        *reinterpret_cast<float4*>(kt + at_key[i] * kpitch + at_d[i]) = float4{kv[i][0], kv[i][1], kv[i][2], kv[i][3]};
        *reinterpret_cast<float4*>(vt + at_key[i] * dim + at_d[i]) = float4{vv[i][0], vv[i][1], vv[i][2], vv[i][3]};
      }
    }
  }
  return bad;
}

template <typename T, int NPL>  // NPL: output columns per lane (dim <= 64 * NPL)
__global__ __launch_bounds__(64) void cached_attention_partial_kernel(KvArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int lane = threadIdx.x;
  const int part = blockIdx.x, chunk = blockIdx.y;
  const int b = blockIdx.z / a.kv_heads, kvh = blockIdx.z - b * a.kv_heads;
  const int dim = a.dim, kpitch = dim + 4;
  float* kt = lds;                        // [64][dim + 4]
  float* vt = kt + KV_TILE * kpitch;      // [64][dim]
  float* qs = vt + KV_TILE * dim;         // [KV_ROWS][dim]
  const int rows_all = a.tq * a.group;
  const int row0 = chunk * KV_ROWS;
  const int rows = min(KV_ROWS, rows_all - row0);
  bool bad = false;

  // Row r of this block: query i = (row0 + r) / group, head kvh * group + (row0 + r) % group.
  long p_of[KV_ROWS], first_of[KV_ROWS];
  long out_row[KV_ROWS];
#pragma unroll
  for (int r = 0; r < KV_ROWS; ++r) {
    const int rr = min(row0 + r, rows_all - 1);
    const int i = rr / a.group, h = kvh * a.group + (rr - i * a.group);
    p_of[r] = a.kv_len - a.tq + i;
    first_of[r] = a.window > 0 ? max(0l, p_of[r] + 1 - a.window) : 0l;
    out_row[r] = (static_cast<long>(b) * a.tq + i) * a.heads + h;
  }
  for (int c = lane; c < rows * dim; c += 64) {
    const int r = c / dim, d = c - r * dim;
    const float v = a.q[out_row[r] * dim + d];
    bad |= !dev_finite(v);
    qs[r * dim + d] = v;
  }

  float m[KV_ROWS], l[KV_ROWS], acc[KV_ROWS][NPL];
#pragma unroll
  for (int r = 0; r < KV_ROWS; ++r) {
    m[r] = -INFINITY;
    l[r] = 0.0f;
#pragma unroll
    for (int n = 0; n < NPL; ++n) acc[r][n] = 0.0f;
  }

  const long base_b = static_cast<long>(b) * a.capacity;
  const int key0 = lane / (dim >> 2), piece0 = lane - key0 * (dim >> 2);
  const T* kc = static_cast<const T*>(a.k_cache);
  const T* vc = static_cast<const T*>(a.v_cache);
  for (int t = 0; t < a.tiles_per_block; ++t) {
    const long pos0 = a.read_lo + (static_cast<long>(part) * a.tiles_per_block + t) * KV_TILE;
    if (pos0 >= a.kv_len) break;
    __syncthreads();  // the previous tile has been consumed
    bad |= load_tiles<T>(kc, vc, kt, vt, a, base_b, kvh, pos0, key0, piece0);
    __syncthreads();

    // Scores of key `lane` against every row.
    float s[KV_ROWS];
#pragma unroll
    for (int r = 0; r < KV_ROWS; ++r) s[r] = 0.0f;
    const float* krow = kt + lane * kpitch;
    for (int d = 0; d < dim; d += 4) {
      const float4 kv = *reinterpret_cast<const float4*>(krow + d);
#pragma unroll
      for (int r = 0; r < KV_ROWS; ++r) {
        if (r < rows) {
          const float4 qv = *reinterpret_cast<const float4*>(qs + r * dim + d);
          s[r] = fmaf(qv.x, kv.x, s[r]);
          s[r] = fmaf(qv.y, kv.y, s[r]);
          s[r] = fmaf(qv.z, kv.z, s[r]);
          s[r] = fmaf(qv.w, kv.w, s[r]);
        }
      }
    }
    const long pos = pos0 + lane;
    float p[KV_ROWS];
#pragma unroll
    for (int r = 0; r < KV_ROWS; ++r) {
      p[r] = 0.0f;
      if (r < rows) {
        const bool seen = pos <= p_of[r] && pos >= first_of[r];
        const float sc = s[r] * a.scale;
        bad |= seen && !dev_finite(sc);
        const float masked = seen ? sc : -INFINITY;
        const float tile_max = wave_max(masked);
        const float m_new = fmaxf(m[r], tile_max);
        if (m_new > -INFINITY) {  // uniform across the wave
          const float corr = expf(m[r] - m_new);  // 0 when this is the row's first visible tile
          p[r] = expf(masked - m_new);            // 0 for a hidden key
          l[r] = l[r] * corr + wave_sum(p[r]);
#pragma unroll
          for (int n = 0; n < NPL; ++n) acc[r][n] *= corr;
          m[r] = m_new;
        }
      }
    }
    // Values: out[r][d] += p[r][key] * V[key][d].
    const int keys = static_cast<int>(min(static_cast<long>(KV_TILE), a.kv_len - pos0));
    for (int j = 0; j < keys; ++j) {
      float v[NPL];
#pragma unroll
      for (int n = 0; n < NPL; ++n) v[n] = (lane + 64 * n < dim) ? vt[j * dim + lane + 64 * n] : 0.0f;
#pragma unroll
      for (int r = 0; r < KV_ROWS; ++r) {
        if (r < rows) {
          const float w = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p[r]), j));
#pragma unroll
          for (int n = 0; n < NPL; ++n) acc[r][n] = fmaf(w, v[n], acc[r][n]);
        }
      }
    }
  }

  const int width = dim + 2;
#pragma unroll
  for (int r = 0; r < KV_ROWS; ++r) {
    if (r < rows) {
      float* dst = a.partial + (out_row[r] * a.nparts + part) * width;
#pragma unroll
      for (int n = 0; n < NPL; ++n)
        if (lane + 64 * n < dim) dst[lane + 64 * n] = acc[r][n];
      if (lane == 0) {
        dst[dim] = m[r];
        dst[dim + 1] = l[r];
      }
    }
  }
  if (bad) dev_raise_fault(a.fault, a.tag);
}

// ---- the fast path: head_dim a power of two ----
// A key's row is read by LPK = dim / 4 adjacent lanes, 16 bytes each, so one load instruction
// covers 64 / LPK keys with whole cache lines and needs no LDS. A tile is 16 such rounds; all 32
// loads of a tile (K and V) are issued before the first is used. Scores are reduced across the LPK
// lanes with DPP adds (bpermutes above 16 lanes); each lane group keeps the output columns of its
// own keys and the groups are summed once, at the end of the block.
constexpr int KG_ROUNDS = 16;
constexpr int KG_ROWS = 4;  // query rows per block
// Waves of a block with one row where blocks are few: sixteen of eight rounds (half the registers) over bf16 caches, eight
// of sixteen over f32 ones, whose pieces would not fit the 128 registers a sixteen-wave block leaves each lane.
template <typename T>
constexpr int KG_FEW_WAVES = sizeof(T) == 2 ? 16 : 8;

// Sum over the LPK adjacent lanes that hold one key; every one of them receives the total.
template <int LPK>
__device__ __forceinline__ float group_sum(float v) {
  const auto add = [](float x, float y) { return x + y; };
  if constexpr (LPK >= 2) v += dev_dpp<0xB1>(v);   // quad_perm [1,0,3,2]
  if constexpr (LPK >= 4) v += dev_dpp<0x4E>(v);   // quad_perm [2,3,0,1]
  if constexpr (LPK >= 8) v += dev_dpp<0x141>(v);  // row_half_mirror
  if constexpr (LPK >= 16) v += dev_dpp<0x140>(v); // row_mirror
  if constexpr (LPK >= 32) v = dev_meet_16(v, add);
  if constexpr (LPK >= 64) v = dev_meet_32(v, add);
  return v;
}
// Combines the 64 / LPK lane groups (lanes that differ in the bits at and above LPK).
template <int LPK, typename F>
__device__ __forceinline__ float across_groups(float v, F f) {
  if constexpr (LPK <= 1) v = f(v, dev_dpp<0xB1>(v));
  if constexpr (LPK <= 2) v = f(v, dev_dpp<0x4E>(v));
  if constexpr (LPK <= 4) v = f(v, __shfl_xor(v, 4));
  if constexpr (LPK <= 8) v = f(v, dev_dpp<0x128>(v));  // row_ror 8
  if constexpr (LPK <= 16) v = dev_meet_16(v, f);
  if constexpr (LPK <= 32) v = dev_meet_32(v, f);
  return v;
}

// Four elements of a cache row as they sit in memory. `get<true>` is a point that no use of them moves ahead of.
template <typename T>
struct KvPiece {
  float4 q;
  template <bool STREAM>
  __device__ __forceinline__ void load(const T* p) { q = dev_stream_load<STREAM>(reinterpret_cast<const float4*>(p)); }
  template <bool HOLD>
  __device__ __forceinline__ void get(float (&v)[4]) {
    if constexpr (HOLD) asm volatile("" : "+v"(q.x), "+v"(q.y), "+v"(q.z), "+v"(q.w));
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
  }
};
template <>
struct KvPiece<unsigned short> {
  uint2 q;
  template <bool STREAM>
  __device__ __forceinline__ void load(const unsigned short* p) { q = dev_stream_load<STREAM>(reinterpret_cast<const uint2*>(p)); }
  template <bool HOLD>
  __device__ __forceinline__ void get(float (&v)[4]) {
    if constexpr (HOLD) asm volatile("" : "+v"(q.x), "+v"(q.y));
    v[0] = __uint_as_float(q.x << 16); v[1] = __uint_as_float(q.x & 0xffff0000u);
    v[2] = __uint_as_float(q.y << 16); v[3] = __uint_as_float(q.y & 0xffff0000u);
  }
};

// ROWS query rows per block: KG_ROWS, or one where a KV head has a single row (ungrouped heads, one new
// token), which is a quarter of the code and half the registers. A call of few blocks runs every instruction about
// once, so it is bound by fetching its own code and by one chain of memory latencies: positions are 32-bit offsets from
// the tile, non-finite values are collected with one multiply-add each (x * 0 is NaN for them), and a single row
// takes more waves of fewer rounds (KG_FEW_WAVES): 15.0 -> 5.3 KiB, 12 heads x 301 positions 12.1 -> 6.5 us.
// WAVES waves share a block's keys (a contiguous run each) and add up in LDS in wave order. When one block
// covers a row's whole span (nparts == 1) it writes the output itself: no partials in memory, no second launch.
template <typename T, int LPK, int WAVES, int ROWS, int ROUNDS, bool STREAM = false>
__global__ __launch_bounds__(WAVES * 64) void cached_attention_group_kernel(KvArgs a) {
  __shared__ float meet[WAVES][ROWS][LPK * 4 + 2];
  constexpr int G = 64 / LPK;               // keys per round
  constexpr int TILE = ROUNDS * G;       // keys per tile
  constexpr float LOG2E = 1.4426950408889634f;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int part = blockIdx.x, chunk = blockIdx.y;
  const int b = blockIdx.z / a.kv_heads, kvh = blockIdx.z - b * a.kv_heads;
  const int g = lane / LPK, d0 = (lane % LPK) * 4;
  constexpr int dim = LPK * 4;
  const int rows_all = a.tq * a.group;
  const int row0 = chunk * ROWS;
  const int rows = ROWS == 1 ? 1 : min(ROWS, rows_all - row0);
  bool bad = false;
  float check[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // NaN once a value row that was read is not finite

  long p_of[ROWS], first_of[ROWS], out_row[ROWS];
  float q[ROWS][4];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    if constexpr (ROWS == 1) {  // the only row: the last position, which sees every key that is read
      p_of[r] = a.kv_len - 1;
      first_of[r] = a.read_lo;
      out_row[r] = static_cast<long>(b) * a.heads + kvh;
    } else {
      const int rr = min(row0 + r, rows_all - 1);
      const int i = rr / a.group, h = kvh * a.group + (rr - i * a.group);
      p_of[r] = a.kv_len - a.tq + i;
      first_of[r] = a.window > 0 ? max(0l, p_of[r] + 1 - a.window) : 0l;
      out_row[r] = (static_cast<long>(b) * a.tq + i) * a.heads + h;
    }
    const float4 qv = *reinterpret_cast<const float4*>(a.q + out_row[r] * dim + d0);
    q[r][0] = qv.x; q[r][1] = qv.y; q[r][2] = qv.z; q[r][3] = qv.w;
    bad |= !(dev_finite(qv.x) && dev_finite(qv.y) && dev_finite(qv.z) && dev_finite(qv.w));
  }
  // Scores are kept in the exp2 domain: s * scale * log2(e).
  const float scale2 = a.scale * LOG2E;
  float m[ROWS], l[ROWS], acc[ROWS][4];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    m[r] = -INFINITY;
    l[r] = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[r][e] = 0.0f;
  }

  const long base_b = static_cast<long>(b) * a.capacity;
  const T* kc = static_cast<const T*>(a.k_cache);
  const T* vc = static_cast<const T*>(a.v_cache);
  const long span_keys = static_cast<long>(a.tiles_per_block) * KV_TILE;  // the host counts 64-key tiles
  const long block_lo = a.read_lo + part * span_keys;
  const long block_hi = min(a.kv_len, block_lo + span_keys);
  const long wave_keys = ((block_hi - block_lo + WAVES - 1) / WAVES + G - 1) / G * G;
  const long part_lo = block_lo + wave * wave_keys;
  const long part_hi = min(block_hi, part_lo + wave_keys);
  for (long pos0 = part_lo; pos0 < part_hi; pos0 += TILE) {
    const int left = static_cast<int>(min(static_cast<long>(TILE), part_hi - pos0));
    // The span is within the capacity: a position wraps the ring at most once.
    const unsigned int ahead = a.read_slot + static_cast<unsigned int>(pos0 - a.read_lo), capacity = a.capacity;
    const unsigned int slot0 = ahead >= capacity ? ahead - capacity : ahead;
    KvPiece<T> kr[ROUNDS], vr[ROUNDS];
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
      // Every lane loads, with no branch around the load, so that the compiler issues all 32
      // before it waits for the first: a key past the end of the part re-reads the tile's first
      // key (a slot this block reads anyway), and its weight below is exactly zero.
      const int key = i * G + g < left ? i * G + g : 0;
      unsigned int slot = slot0 + key;  // a tile wraps the ring at most once
      slot = slot >= capacity ? slot - capacity : slot;
      const size_t off = static_cast<size_t>(((base_b + slot) * a.kv_heads + kvh) * dim + d0);
      kr[i].template load<STREAM>(kc + off);
      vr[i].template load<STREAM>(vc + off);
    }
    // Every load goes out before the first product (the compiler otherwise moves products up between them, each with
    // its wait: 64 sequences of 1024 positions, 103 us instead of 73). Four rows have no registers to hold them all.
    if constexpr (ROWS == 1) asm volatile("" ::: "memory");
    float kv[ROUNDS][4], vv[ROUNDS][4];
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
      kr[i].template get<ROWS == 1>(kv[i]);
      vr[i].template get<ROWS == 1>(vv[i]);
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      if (r < rows) {  // uniform
        float s[ROUNDS];
        float tile_max = -INFINITY;
        // The keys of this tile that the row sees: low <= offset <= high.
        const int low = ROWS == 1 ? 0 : static_cast<int>(min(static_cast<long>(TILE), max(0l, first_of[r] - pos0)));
        const int high = ROWS == 1 ? left - 1 : static_cast<int>(max(-1l, min(static_cast<long>(left - 1), p_of[r] - pos0)));
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i) {
          float dot = q[r][0] * kv[i][0];
          dot = fmaf(q[r][1], kv[i][1], dot);
          dot = fmaf(q[r][2], kv[i][2], dot);
          dot = fmaf(q[r][3], kv[i][3], dot);
          dot = group_sum<LPK>(dot);
          const bool seen = i * G + g <= high && i * G + g >= low;
          const float sc = dot * scale2;
          bad |= seen && !dev_finite(sc);
          s[i] = seen ? sc : -INFINITY;
          tile_max = fmaxf(tile_max, s[i]);
        }
        tile_max = across_groups<LPK>(tile_max, [](float x, float y) { return fmaxf(x, y); });
        const float m_new = fmaxf(m[r], tile_max);
        if (m_new > -INFINITY) {  // uniform: the row sees a key in this tile or saw one before
          const float corr = __builtin_amdgcn_exp2f(m[r] - m_new);
          float sum = 0.0f;
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[r][e] *= corr;
#pragma unroll
          for (int i = 0; i < ROUNDS; ++i) {
            const float p = __builtin_amdgcn_exp2f(s[i] - m_new);  // 0 for a hidden key
            sum += p;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              acc[r][e] = fmaf(p, vv[i][e], acc[r][e]);
              if constexpr (ROWS == 1) check[e] = fmaf(vv[i][e], 0.0f, check[e]);
            }
          }
          l[r] = l[r] * corr + sum;  // this lane group's keys only
          m[r] = m_new;
        }
      }
    }
    // (a single row sees every key that is read: one that is not finite shows in its score)
    if constexpr (ROWS > 1) {
#pragma unroll
      for (int i = 0; i < ROUNDS; ++i)
        bad |= !(dev_finite(kv[i][0]) && dev_finite(kv[i][1]) && dev_finite(kv[i][2]) && dev_finite(kv[i][3]) &&
                 dev_finite(vv[i][0]) && dev_finite(vv[i][1]) && dev_finite(vv[i][2]) && dev_finite(vv[i][3]));
    }
  }
  if constexpr (ROWS == 1) bad |= !(check[0] == 0.0f && check[1] == 0.0f && check[2] == 0.0f && check[3] == 0.0f);

#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    if (r < rows) {
      const float total = across_groups<LPK>(l[r], [](float x, float y) { return x + y; });
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float sum = across_groups<LPK>(acc[r][e], [](float x, float y) { return x + y; });
        if (g == 0) meet[wave][r][d0 + e] = sum;
      }
      if (lane == 0) {
        meet[wave][r][dim] = m[r];
        meet[wave][r][dim + 1] = total;
      }
    }
  }
  __syncthreads();
  // A thread per (row, column): the waves' shares, lowest keys first.
  for (int c = threadIdx.x; c < rows * dim; c += WAVES * 64) {
    const int r = c / dim, d = c - r * dim;
    float top = -INFINITY;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) top = fmaxf(top, meet[w][r][dim]);
    float total = 0.0f, sum = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float weight = meet[w][r][dim] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(meet[w][r][dim] - top);
      total = fmaf(meet[w][r][dim + 1], weight, total);
      sum = fmaf(meet[w][r][d], weight, sum);
    }
    long out_at = out_row[0];
    if constexpr (ROWS > 1) {
      const int rr = row0 + r, i = rr / a.group;
      out_at = (static_cast<long>(b) * a.tq + i) * a.heads + kvh * a.group + (rr - i * a.group);
    }
    if (a.nparts == 1) {
      bad |= !(dev_finite(total) && total > 0.0f);
      a.out[out_at * dim + d] = sum * (1.0f / total);
    } else {
      constexpr float LN2 = 0.6931471805599453f;
      float* dst = a.partial + (out_at * a.nparts + part) * (dim + 2);
      dst[d] = sum;
      if (d == 0) {
        dst[dim] = top * LN2;  // the merge works in the natural-log domain
        dst[dim + 1] = total;
      }
    }
  }
  if (bad) dev_raise_fault(a.fault, a.tag);
}

// One wave per output row: merges the row's partials, lowest part first.
template <int NPL>
__global__ __launch_bounds__(64) void cached_attention_merge_kernel(KvArgs a, long rows_total) {
  const long row = blockIdx.x;
  if (row >= rows_total) return;
  const int lane = threadIdx.x, dim = a.dim, width = dim + 2;
  const float* src = a.partial + row * a.nparts * width;
  float top = -INFINITY;
  for (int s = 0; s < a.nparts; ++s) top = fmaxf(top, src[s * width + dim]);
  float total = 0.0f, acc[NPL];
#pragma unroll
  for (int n = 0; n < NPL; ++n) acc[n] = 0.0f;
  for (int s = 0; s < a.nparts; ++s) {
    const float ms = src[s * width + dim];
    if (ms == -INFINITY) continue;  // a part in which this row saw no key
    const float w = expf(ms - top);
    total = fmaf(src[s * width + dim + 1], w, total);
#pragma unroll
    for (int n = 0; n < NPL; ++n)
      if (lane + 64 * n < dim) acc[n] = fmaf(src[s * width + lane + 64 * n], w, acc[n]);
  }
  const bool ok = dev_finite(total) && total > 0.0f;
  const float inv = 1.0f / total;
#pragma unroll
  for (int n = 0; n < NPL; ++n)
    if (lane + 64 * n < dim) a.out[row * dim + lane + 64 * n] = acc[n] * inv;
  if (!ok) dev_raise_fault(a.fault, a.tag);
}

// ---- the cache write: all or nothing ----
struct KvWrite {
  void* cache;
  const float* src;
  unsigned int* refused;  // of the two-launch form: 64 bits with the tag of a scan that refused, then how many workgroups saw it
  size_t n;               // elements of src
  unsigned int capacity, step, tn, at;  // at: already modulo the capacity
  OmxFaultWord* fault;
  unsigned long long tag;
};
// VEC consecutive elements of src (n, step and every address a multiple of VEC elements).
template <int VEC>
__device__ __forceinline__ bool kv_finite(const float* p) {
  if constexpr (VEC == 4) {
    const float4 v = *reinterpret_cast<const float4*>(p);
    return dev_finite(v.x) && dev_finite(v.y) && dev_finite(v.z) && dev_finite(v.w);
  } else {
    return dev_finite(*p);
  }
}
// Where element i of src goes.
template <typename T, typename Index>
__device__ __forceinline__ T* kv_place(const KvWrite& w, Index i) {
  const Index row = i / w.step, b = row / w.tn;
  const unsigned int e = static_cast<unsigned int>(i - row * w.step);
  const unsigned int j = static_cast<unsigned int>(row - b * w.tn);
  const unsigned int slot = w.at + j < w.capacity ? w.at + j : w.at + j - w.capacity;  // at < capacity, tn <= capacity
  return static_cast<T*>(w.cache) + (static_cast<size_t>(b) * w.capacity + slot) * w.step + e;
}
template <typename T, int VEC>
__device__ __forceinline__ void kv_put(const KvWrite& w, size_t i) {
  // (32-bit divisions where they do)
  T* dst = w.n <= 0xffffffffull ? kv_place<T>(w, static_cast<unsigned int>(i)) : kv_place<T>(w, i);
  if constexpr (VEC == 4) {
    float v[4];
    dev_load4(w.src, i, v);
    dev_store4(dst, 0, v);
  } else {
    dev_store(dst, 0, w.src[i]);
  }
}
// A short src (one token per sequence): every workgroup scans all of it, which is cheaper than a second
// launch, and writes its own share: one launch instead of a fill, a scan and a write (6.3 -> 2.7 us for one
// token of 768 values). All workgroups walk the same addresses together, so they wait for the same memory
// channels: at 49152 values the scan alone is 10 us, and two launches are ahead from some 16384 on.
constexpr size_t KV_ONE_LAUNCH = 1u << 14;
constexpr int KV_SCAN_THREADS = 1024;
// A thread writes at most one piece, which it loads first: one workgroup (4096 values) has scanned everything with that.
template <typename T, int VEC>
__global__ __launch_bounds__(KV_SCAN_THREADS) void kv_scan_write_kernel(KvWrite w) {
  constexpr unsigned int STRIDE = KV_SCAN_THREADS * VEC;
  const unsigned int n = static_cast<unsigned int>(w.n), own = (blockIdx.x * KV_SCAN_THREADS + threadIdx.x) * VEC;
  float v[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) v[e] = 0.0f;
  T* dst = nullptr;
  if (own < n) {
    if constexpr (VEC == 4) dev_load4(w.src, own, v);
    else v[0] = w.src[own];
    dst = kv_place<T>(w, own);
  }
  bool bad = false;
#pragma unroll
  for (int e = 0; e < VEC; ++e) bad |= !dev_finite(v[e]);
  if (gridDim.x > 1) {
#pragma unroll 4
    for (unsigned int i = threadIdx.x * VEC; i < n; i += STRIDE) bad |= !kv_finite<VEC>(w.src + i);
  }
  if (__syncthreads_or(bad)) {
    if (bad) dev_raise_fault(w.fault, w.tag);
    return;
  }
  if (own < n) {
    if constexpr (VEC == 4) dev_store4(dst, 0, v);
    else dev_store(dst, 0, v[0]);
  }
}
// A longer one: the first launch scans, the second copies unless the scan refused. The word between them
// holds the tag of a refused scan; the second launch's last workgroup takes it back, for a replay of the two out of a
// captured graph comes with the same tag (nothing is cleared where nothing was refused).
template <int VEC>
__global__ __launch_bounds__(256) void kv_scan_kernel(KvWrite w) {
  bool bad = false;
  for (size_t i = (static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x) * VEC; i < w.n; i += static_cast<size_t>(gridDim.x) * 256 * VEC)
    bad |= !kv_finite<VEC>(w.src + i);
  if (bad) {
    atomicExch(reinterpret_cast<unsigned long long*>(w.refused), w.tag);
    dev_raise_fault(w.fault, w.tag);
  }
}
template <typename T, int VEC>
__global__ __launch_bounds__(256) void kv_write_kernel(KvWrite w) {
  if (*reinterpret_cast<const volatile unsigned long long*>(w.refused) == w.tag) {
    __syncthreads();  // the whole workgroup has read it
    if (threadIdx.x == 0 && atomicAdd(w.refused + 2, 1u) == gridDim.x - 1) {
      w.refused[2] = 0u;
      atomicExch(reinterpret_cast<unsigned long long*>(w.refused), 0ull);
    }
    return;
  }
  for (size_t i = (static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x) * VEC; i < w.n; i += static_cast<size_t>(gridDim.x) * 256 * VEC)
    kv_put<T, VEC>(w, i);
}
template <typename T, int VEC>
int32_t launch_kv_write(omx_ctx* ctx, const KvWrite& w) {
  const unsigned blocks = static_cast<unsigned>(std::min<size_t>((w.n / VEC + 255) / 256, 8192));
  if (w.n <= KV_ONE_LAUNCH) {
    omx_launch(ctx, (kv_scan_write_kernel<T, VEC>), dim3((blocks + 3) / 4), dim3(KV_SCAN_THREADS), 0, w);
    OMX_LAUNCH_CHECK(ctx, "kv_scan_write_kernel");
    return OMX_OK;
  }
  omx_launch(ctx, (kv_scan_kernel<VEC>), dim3(blocks), dim3(256), 0, w);
  OMX_LAUNCH_CHECK(ctx, "kv_scan_kernel");
  omx_launch(ctx, (kv_write_kernel<T, VEC>), dim3(blocks), dim3(256), 0, w);
  OMX_LAUNCH_CHECK(ctx, "kv_write_kernel");
  return OMX_OK;
}

// Bytes of keys and values from which a call reads them past the caches: half of the memory-side cache, of which a model, with its
// weights, leaves nothing for the next token. Whole steps of d = 768 over 1024 positions, us without and with the hint: twelve layers of
// 126 MiB (f32) 2107, 2108; 138 MiB 2159, 2132; 150 2183, 2142; of 129 MiB (bf16) 2222, 2200; two layers of 126 MiB 448, 444; 138 462, 450;
// one layer of 144 MiB 278, 282; 180 285, 284 (three runs of each, within 2 % at two layers and fewer). The call alone, in turn over twelve
// caches: 144 MiB 37.9, 35.7; 384 (64 sequences) 75.0, 68.1; bf16 129 MiB 39.3, 37.1; 192 48.2, 45.3. Left: one cache over and over with
// nothing else read in between, which stays up to its size: f32 144 MiB 30.5, 33.2; 240 42.7, 46.6; 318 62.3, 58.7; two in turn, bf16 129
// MiB 35.1, 36.7; 144 38.1, 37.3.
constexpr uint64_t KV_STREAM = 128ull << 20;
template <typename T, int LPK, int NPL>
int32_t launch_group(omx_ctx* ctx, const KvArgs& a, dim3 grid, long rows_total, int waves) {
  auto go = [&](auto most, auto four, auto one) {
    omx_launch(ctx, (waves >= 8 ? most : waves == 4 ? four : one), grid, dim3(waves * 64), 0, a);
  };
  const uint64_t span = std::min<uint64_t>(a.kv_len - a.read_lo, a.capacity);
  if (a.tq * a.group == 1 && waves <= 4 && 2 * sizeof(T) * a.batch * span * a.kv_heads * a.dim >= KV_STREAM)
    omx_launch(ctx, (waves == 4 ? &cached_attention_group_kernel<T, LPK, 4, 1, KG_ROUNDS, true> : &cached_attention_group_kernel<T, LPK, 1, 1, KG_ROUNDS, true>),
               grid, dim3(waves * 64), 0, a);
  else if (a.tq * a.group == 1)
    go(&cached_attention_group_kernel<T, LPK, KG_FEW_WAVES<T>, 1, 8 * KG_ROUNDS / KG_FEW_WAVES<T>>, &cached_attention_group_kernel<T, LPK, 4, 1, KG_ROUNDS>,
       &cached_attention_group_kernel<T, LPK, 1, 1, KG_ROUNDS>);
  else
    go(&cached_attention_group_kernel<T, LPK, 8, KG_ROWS, KG_ROUNDS / 2>, &cached_attention_group_kernel<T, LPK, 4, KG_ROWS, KG_ROUNDS>,
       &cached_attention_group_kernel<T, LPK, 1, KG_ROWS, KG_ROUNDS>);
  OMX_LAUNCH_CHECK(ctx, "cached_attention_group_kernel");
  if (a.nparts == 1) return OMX_OK;
  omx_launch(ctx, (cached_attention_merge_kernel<NPL>), dim3(static_cast<unsigned>(rows_total)), dim3(64), 0, a, rows_total);
  OMX_LAUNCH_CHECK(ctx, "cached_attention_merge_kernel");
  return OMX_OK;
}

template <typename T>
int32_t launch_attention(omx_ctx* ctx, const KvArgs& a, dim3 grid, size_t lds_bytes, long rows_total) {
  auto run = [&](auto kernel, auto merge) -> int32_t {
    if (lds_bytes > 64 * 1024)  // beyond the default limit: ask for it (cheap, and idempotent)
      OMX_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes)));
    omx_launch(ctx, kernel, grid, dim3(64), lds_bytes, a);
    OMX_LAUNCH_CHECK(ctx, "cached_attention_partial_kernel");
    omx_launch(ctx, merge, dim3(static_cast<unsigned>(rows_total)), dim3(64), 0, a, rows_total);
    OMX_LAUNCH_CHECK(ctx, "cached_attention_merge_kernel");
    return OMX_OK;
  };
  if (a.dim <= 64) return run(&cached_attention_partial_kernel<T, 1>, &cached_attention_merge_kernel<1>);
  if (a.dim <= 128) return run(&cached_attention_partial_kernel<T, 2>, &cached_attention_merge_kernel<2>);
  return run(&cached_attention_partial_kernel<T, 4>, &cached_attention_merge_kernel<4>);
}

}  // namespace

extern "C" {

int32_t omx_cached_attention_forward(omx_ctx* ctx, const void* q, const void* k_cache, const void* v_cache,
                                     int32_t cache_dtype, void* out, uint64_t batch, uint64_t tq, uint64_t heads,
                                     uint64_t kv_heads, uint64_t head_dim, uint64_t capacity, uint64_t kv_len,
                                     uint64_t window) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "cached_attention_forward";
  if (!q || !k_cache || !v_cache || !out) return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  if (cache_dtype != OMX_F32 && cache_dtype != OMX_BF16) return omx_fail(ctx, OMX_DTYPE, "%s: cache dtype", op);
  if (batch == 0 || tq == 0 || heads == 0 || head_dim == 0 || capacity == 0 || kv_heads == 0)
    return omx_fail(ctx, OMX_SHAPE, "%s: zero dimension in q or cache", op);
  if (heads % kv_heads != 0)
    return omx_fail(ctx, OMX_SHAPE, "%s: %llu query heads over %llu kv heads", op, (unsigned long long)heads,
                    (unsigned long long)kv_heads);
  if (kv_len < tq)
    return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: kv_len %llu is below the %llu new positions", op,
                    (unsigned long long)kv_len, (unsigned long long)tq);
  if (window >= kv_len) window = 0;  // a window that covers every position is no window
  uint64_t span = kv_len;
  if (window != 0 && tq + (window - 1) < kv_len) span = tq + (window - 1);
  if (span > capacity)
    return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: the %llu positions read up to kv_len %llu exceed cache capacity %llu",
                    op, (unsigned long long)span, (unsigned long long)kv_len, (unsigned long long)capacity);
  if (head_dim % 4 != 0 || head_dim > 256)
    return omx_fail(ctx, OMX_UNSUPPORTED_HEAD_DIM, "%s: head_dim %llu (a multiple of 4 up to 256)", op,
                    (unsigned long long)head_dim);
  const uint64_t rows_total = batch * tq * heads;
  if (batch * kv_heads > 65535 || rows_total > 0x7fffffffull || capacity > 0x7fffffffull || kv_len > (1ull << 40))
    return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: extent too large", op);

  // A prompt chunk: from 16 rows per KV head on, every tile of keys serves 16 rows and more, and the products go to
  // the matrix units (the kernels below read a key's row once per 4 or 8 query rows and take the sums on vector
  // instructions). 4 x 12 heads, 256 new positions of 700: 186 -> 38 us per call. Where those rows make few workgroups over
  // a long cache, the keys are split over more of them and the merge kernel adds the parts up.
  const bool bf16 = cache_dtype == OMX_BF16;
  const long step = static_cast<long>(kv_heads * head_dim);
  if (tq * (heads / kv_heads) >= 16 && tq * (heads / kv_heads) <= 0x7fffffffull && ctx->kv_attention_mode == 0 &&
      omx_sdpa32_supports(head_dim, batch * kv_heads, {q, k_cache, v_cache, out}, {})) {
    Sdpa32Args m{};
    m.q = static_cast<const float*>(q);
    m.k = k_cache;
    m.v = v_cache;
    m.out = static_cast<float*>(out);
    m.q_h = m.o_h = m.k_h = static_cast<long>(head_dim);
    m.q_t = m.o_t = static_cast<long>(heads * head_dim);
    m.q_b = m.o_b = static_cast<long>(tq * heads * head_dim);
    m.k_t = step;
    m.k_b = static_cast<long>(capacity) * step;
    m.kv_heads = static_cast<int>(kv_heads);
    m.rep = static_cast<int>(heads / kv_heads);
    m.tq = static_cast<int>(tq);
    m.tk = static_cast<int>(span);
    m.q_pos0 = static_cast<int>(span - tq);
    m.slot0 = static_cast<int>((kv_len - span) % capacity);
    m.capacity = static_cast<int>(capacity);
    m.window = window < span ? static_cast<int>(window) : 0;
    m.scale = 1.0f / std::sqrt(static_cast<float>(head_dim));
    m.fault = ctx->fault;
    m.tag = omx_tag(ctx, F_CACHED_ATTENTION);
    // Few rows over a long cache: their keys are split over workgroups (without the scratch for it, one walks them all).
    m.nparts = omx_sdpa32_key_parts(ctx, m, static_cast<int>(batch), static_cast<int>(head_dim), bf16);
    const uint64_t bytes = rows_total * m.nparts * (head_dim + 2) * sizeof(float);
    m.partial = m.nparts > 1 ? static_cast<float*>(omx_workspace_if_room(ctx, bytes)) : nullptr;
    if (!m.partial) m.nparts = 1;
    const int32_t rc = omx_sdpa32_forward(ctx, m, static_cast<int>(batch), static_cast<int>(head_dim), bf16);
    if (rc != OMX_OK || m.nparts == 1) return rc;
    KvArgs merge{};
    merge.partial = m.partial;
    merge.nparts = m.nparts;
    merge.out = m.out;
    merge.dim = static_cast<int>(head_dim);
    merge.fault = m.fault;
    merge.tag = m.tag;
    const long rows = static_cast<long>(rows_total);
    omx_launch(ctx, (head_dim <= 64 ? &cached_attention_merge_kernel<1> : &cached_attention_merge_kernel<2>),
               dim3(static_cast<unsigned>(rows)), dim3(64), 0, merge, rows);
    OMX_LAUNCH_CHECK(ctx, "cached_attention_merge_kernel");
    return OMX_OK;
  }

  KvArgs a;
  a.q = static_cast<const float*>(q);
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.out = static_cast<float*>(out);
  a.batch = static_cast<int>(batch);
  a.tq = static_cast<int>(tq);
  a.heads = static_cast<int>(heads);
  a.kv_heads = static_cast<int>(kv_heads);
  a.dim = static_cast<int>(head_dim);
  a.capacity = static_cast<int>(capacity);
  a.group = static_cast<int>(heads / kv_heads);
  a.kv_len = static_cast<long>(kv_len);
  a.window = static_cast<long>(window);
  a.read_lo = static_cast<long>(kv_len - span);
  a.read_slot = static_cast<unsigned int>((kv_len - span) % capacity);
  a.scale = 1.0f / std::sqrt(static_cast<float>(head_dim));
  a.fault = ctx->fault;
  a.tag = omx_tag(ctx, F_CACHED_ATTENTION);

  // Power-of-two head dims take the lane-group kernel; others the LDS-tiled one. The option
  // "kv_attention" = 1 forces the LDS-tiled kernel (for tests and measurements).
  const bool grouped = (head_dim & (head_dim - 1)) == 0 && ctx->kv_attention_mode != 1;
  const uint64_t block_rows = grouped ? KG_ROWS : KV_ROWS;
  const uint64_t rows_per_group = tq * (heads / kv_heads);
  const uint64_t chunks = (rows_per_group + block_rows - 1) / block_rows;
  if (chunks > 65535) return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: too many query rows per KV head", op);
  const uint64_t tiles = (span + KV_TILE - 1) / KV_TILE;
  const uint64_t groups = batch * kv_heads * chunks;
  uint64_t waves = 1, parts;
  if (grouped) {
    // Few blocks take eight or sixteen waves each (they share the keys and meet in LDS), a few thousand fill the chip
    // with one. A row's keys are split over blocks, with partials in memory and a merge launch, only
    // when there are not waves enough and every wave still has a tile of 64 keys.
    waves = groups <= static_cast<uint64_t>(ctx->cu_count) ? (rows_per_group > 1 ? 8 : bf16 ? KG_FEW_WAVES<unsigned short> : KG_FEW_WAVES<float>) : groups <= 4ull * ctx->cu_count ? 4 : 1;
    parts = std::min<uint64_t>((8ull * ctx->cu_count + groups * waves - 1) / (groups * waves), (tiles + waves - 1) / waves);
  } else {
    // Enough blocks to fill the chip several times over, but no more parts than tiles.
    parts = std::min<uint64_t>((8ull * ctx->cu_count + groups - 1) / groups, tiles);
  }
  parts = std::max<uint64_t>(1, parts);
  a.tiles_per_block = static_cast<int>((tiles + parts - 1) / parts);
  a.nparts = static_cast<int>((tiles + a.tiles_per_block - 1) / a.tiles_per_block);

  a.partial = nullptr;
  if (!grouped || a.nparts > 1) {
    void* ws = nullptr;
    int32_t rc = omx_workspace(ctx, rows_total * a.nparts * (head_dim + 2) * sizeof(float), &ws);
    if (rc != OMX_OK) return rc;
    a.partial = static_cast<float*>(ws);
  }
  const size_t lds_bytes = (KV_TILE * (head_dim + 4) + KV_TILE * head_dim + KV_ROWS * head_dim) * sizeof(float);
  dim3 grid(static_cast<unsigned>(a.nparts), static_cast<unsigned>(chunks), static_cast<unsigned>(batch * kv_heads));
  const long nrows = static_cast<long>(rows_total);
  if (grouped) {
    const bool f32 = cache_dtype == OMX_F32;
    switch (head_dim) {
#define OMX_KV_CASE(DIM, NPL)                                                                     \
  case DIM:                                                                                       \
    return f32 ? launch_group<float, DIM / 4, NPL>(ctx, a, grid, nrows, static_cast<int>(waves))                           \
               : launch_group<unsigned short, DIM / 4, NPL>(ctx, a, grid, nrows, static_cast<int>(waves));
      OMX_KV_CASE(4, 1)
      OMX_KV_CASE(8, 1)
      OMX_KV_CASE(16, 1)
      OMX_KV_CASE(32, 1)
      OMX_KV_CASE(64, 1)
      OMX_KV_CASE(128, 2)
      OMX_KV_CASE(256, 4)
#undef OMX_KV_CASE
      default:
        break;
    }
  }
  if (cache_dtype == OMX_F32) return launch_attention<float>(ctx, a, grid, lds_bytes, nrows);
  return launch_attention<unsigned short>(ctx, a, grid, lds_bytes, nrows);
}

int32_t omx_kv_cache_write(omx_ctx* ctx, void* cache, int32_t cache_dtype, const void* src, uint64_t batch,
                           uint64_t capacity, uint64_t kv_heads, uint64_t head_dim, uint64_t tn, uint64_t at) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "kv_cache_write";
  if (!cache || !src) return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  if (cache_dtype != OMX_F32 && cache_dtype != OMX_BF16) return omx_fail(ctx, OMX_DTYPE, "%s: cache dtype", op);
  if (batch == 0 || capacity == 0 || kv_heads == 0 || head_dim == 0 || tn == 0)
    return omx_fail(ctx, OMX_SHAPE, "%s: zero dimension in cache or src", op);
  if (at + tn < at)
    return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: at %llu + %llu overflows", op, (unsigned long long)at,
                    (unsigned long long)tn);
  if (tn > capacity)
    return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: %llu positions exceed capacity %llu", op, (unsigned long long)tn,
                    (unsigned long long)capacity);
  if (capacity > 0x7fffffffull || kv_heads > 0x7fffffffull || head_dim > 0x7fffffffull || kv_heads * head_dim > 0x7fffffffull)
    return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: extent too large", op);
  KvWrite w;
  w.cache = cache;
  w.src = static_cast<const float*>(src);
  w.refused = ctx->kv_refused;
  w.capacity = static_cast<unsigned int>(capacity);
  w.step = static_cast<unsigned int>(kv_heads * head_dim);
  w.tn = static_cast<unsigned int>(tn);
  w.at = static_cast<unsigned int>(at % capacity);
  w.n = batch * tn * w.step;
  w.fault = ctx->fault;
  w.tag = omx_tag(ctx, F_KV_CACHE_WRITE);
  const bool f32 = cache_dtype == OMX_F32;
  const bool vec = w.step % 4 == 0 && (reinterpret_cast<uintptr_t>(src) & 15u) == 0 &&
                   (reinterpret_cast<uintptr_t>(cache) & (f32 ? 15u : 7u)) == 0;
  if (vec) return f32 ? launch_kv_write<float, 4>(ctx, w) : launch_kv_write<unsigned short, 4>(ctx, w);
  return f32 ? launch_kv_write<float, 1>(ctx, w) : launch_kv_write<unsigned short, 1>(ctx, w);
}

}  // extern "C"
