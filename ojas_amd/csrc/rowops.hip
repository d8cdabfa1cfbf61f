// Row-wise bandwidth-bound kernels: RMSNorm forward/backward, embedding
// gather / scatter-add, argmax and top-k. One wave (64 lanes) owns one row;
// reductions are wavefront shuffles; every tensor is read from HBM once.
//
// Reference semantics:
//   rms_norm_*   ojas-cpu/src/norm.rs:24-204   (trait backend.rs:1658-1672)
//   embedding_*  ojas-cpu/src/pointwise.rs:77-215 (trait backend.rs:1610-1626)
//   argmax/topk  ojas-core/src/backend.rs:184-195,1514-1606
#include <utility>

#include "omx_common.h"

namespace {

constexpr int ROW_THREADS = 256;  // 4 waves per block, one row per wave at a time

// ---------------------------------------------------------------- RMSNorm
// PER = ceil(dim / 64): lane l owns columns l, l + 64, ... so a wave's loads
// are contiguous 64-element runs and the row stays in registers between the
// sum-of-squares pass and the scaling pass.
// One tensor, or two (queries and keys) side by side in the grid's second axis: apart they are two launches of 3 to 4 us, and two more
// for their column sums, whatever their size.
struct RmsRows {
  const void *x, *gy;
  const float* w;
  void* y;         // the normed rows, or gx
  float* partial;  // backward: [blocks][dim]
  size_t rows;
  int rows_per_block;
  unsigned long long tag;
};
struct RmsTensors {
  RmsRows of[2];
};
template <typename TX, typename TY, int PER>
__global__ __launch_bounds__(ROW_THREADS) void rms_fwd_kernel(RmsTensors tensors, int dim, float eps, OmxFaultWord* fault) {
  const RmsRows& t = tensors.of[blockIdx.y];
  const TX* __restrict__ x = static_cast<const TX*>(t.x);
  const float* __restrict__ w = t.w;
  TY* __restrict__ y = static_cast<TY*>(t.y);
  const int lane = threadIdx.x & 63;
  const size_t row = static_cast<size_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= t.rows) return;
  const TX* xr = x + row * dim;
  float xv[PER];
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    int c = j * 64 + lane;
    xv[j] = c < dim ? dev_load<TX>(xr, c) : 0.0f;
    ss += xv[j] * xv[j];
  }
  ss = wave_sum(ss);
  float denom = ss / static_cast<float>(dim) + eps;
  float rstd = 1.0f / sqrtf(denom);
  bool bad = !(dev_finite(denom) && denom > 0.0f && dev_finite(rstd));
  TY* yr = y + row * dim;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    int c = j * 64 + lane;
    if (c < dim) {
      float v = xv[j] * rstd * w[c];
      bad |= !dev_finite(v);
      dev_store<TY>(yr, c, v);
    }
  }
  if (bad) dev_raise_fault(fault, t.tag);
}

// Backward: gx per row, and per-block partial column sums of g * xhat that a
// second kernel adds in ascending block order (no atomics, deterministic).
template <typename TX, typename TG, typename TO, int PER>
__global__ __launch_bounds__(ROW_THREADS) void rms_bwd_kernel(RmsTensors tensors, int dim, float eps, OmxFaultWord* fault) {
  extern __shared__ float lds[];  // [4][dim]
  const RmsRows& t = tensors.of[blockIdx.y];
  const TX* __restrict__ x = static_cast<const TX*>(t.x);
  const float* __restrict__ w = t.w;
  const TG* __restrict__ gy = static_cast<const TG*>(t.gy);
  TO* __restrict__ gx = static_cast<TO*>(t.y);
  float* __restrict__ partial = t.partial;
  const size_t rows = t.rows;
  const int rows_per_block = t.rows_per_block;
  if (static_cast<size_t>(blockIdx.x) * rows_per_block >= rows) return;  // (the whole workgroup)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float inv_dim = 1.0f / static_cast<float>(dim);
  float wv[PER], accw[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    int c = j * 64 + lane;
    wv[j] = c < dim ? w[c] : 0.0f;
    accw[j] = 0.0f;
  }
  bool bad = false;
  // Short rows: a wave's next few at once, or each waits for its loads and two reductions behind the one before (4096 rows of 64:
  // 9.4 us with 8 rows in turn on 128 blocks, 5.2 with 4 at once on 256).
  constexpr int AT_ONCE = PER <= 2 ? 4 : 1;
  const size_t first = static_cast<size_t>(blockIdx.x) * rows_per_block;
  const size_t last = min(rows, first + rows_per_block);
  for (size_t row0 = first + wave; row0 < last; row0 += 4 * AT_ONCE) {
    float xv[AT_ONCE][PER], gv[AT_ONCE][PER], ss[AT_ONCE], rstd[AT_ONCE], dot[AT_ONCE];
#pragma unroll
    for (int r = 0; r < AT_ONCE; ++r) {
      const size_t row = min(row0 + 4 * r, last - 1);  // (one past the last is read and left out)
      const TX* xr = x + row * dim;
      const TG* gr = gy + row * dim;
      ss[r] = 0.0f;
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        int c = j * 64 + lane;
        xv[r][j] = c < dim ? dev_load<TX>(xr, c) : 0.0f;
        gv[r][j] = c < dim ? dev_load<TG>(gr, c) : 0.0f;
        ss[r] += xv[r][j] * xv[r][j];
      }
    }
#pragma unroll
    for (int r = 0; r < AT_ONCE; ++r) ss[r] = wave_sum(ss[r]);
#pragma unroll
    for (int r = 0; r < AT_ONCE; ++r) {
      float denom = ss[r] * inv_dim + eps;
      rstd[r] = 1.0f / sqrtf(denom);
      bad |= row0 + 4 * r < last && !(dev_finite(denom) && denom > 0.0f && dev_finite(rstd[r]));
      dot[r] = 0.0f;
#pragma unroll
      for (int j = 0; j < PER; ++j) dot[r] += (gv[r][j] * wv[j]) * (xv[r][j] * rstd[r]);
    }
#pragma unroll
    for (int r = 0; r < AT_ONCE; ++r) dot[r] = wave_sum(dot[r]);
#pragma unroll
    for (int r = 0; r < AT_ONCE; ++r) {
      if (row0 + 4 * r >= last) break;
      float mean = dot[r] * inv_dim;
      TO* gxr = gx + (row0 + 4 * r) * dim;
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        int c = j * 64 + lane;
        float xhat = xv[r][j] * rstd[r];
        float v = (gv[r][j] * wv[j] - xhat * mean) * rstd[r];
        accw[j] += gv[r][j] * xhat;
        if (c < dim) {
          bad |= !dev_finite(v);
          dev_store<TO>(gxr, c, v);
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    int c = j * 64 + lane;
    if (c < dim) lds[wave * dim + c] = accw[j];
  }
  __syncthreads();
  for (int c = threadIdx.x; c < dim; c += ROW_THREADS) {
    float s = ((lds[c] + lds[dim + c]) + lds[2 * dim + c]) + lds[3 * dim + c];
    partial[static_cast<size_t>(blockIdx.x) * dim + c] = s;
  }
  if (bad) dev_raise_fault(fault, t.tag);
}

// out[c] = sum over blocks of partial[b][c]: 64 columns per workgroup, four
// row groups that each add their strided share, then a fixed four-way sum.
__global__ __launch_bounds__(256) void column_sum_kernel(const float* __restrict__ partial, float* __restrict__ out,
                                                         int blocks, int dim, OmxFaultWord* fault,
                                                         unsigned long long tag) {
  __shared__ float red[4][64];
  const int lane = threadIdx.x & 63, group = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  float s = 0.0f;
  if (c < dim)
    for (int b = group; b < blocks; b += 4) s += partial[static_cast<size_t>(b) * dim + c];
  red[group][lane] = s;
  __syncthreads();
  if (group == 0 && c < dim) {
    float total = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
    out[c] = total;
    if (!dev_finite(total)) dev_raise_fault(fault, tag);
  }
}

// The same for tens to a few hundred rows in one launch: 16 row groups of 64 columns (1024 threads), four
// loads in flight per thread, the groups added in a fixed order.
__device__ __forceinline__ void column_sum_wide(const float* __restrict__ partial, float* __restrict__ out, int blocks, int dim,
                                                OmxFaultWord* fault, unsigned long long tag) {
  __shared__ float red[16][64];
  const int lane = threadIdx.x & 63, group = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
  if (c < dim) {
    const float* col = partial + c;
    int b = group;
    for (; b + 48 < blocks; b += 64) {
      s0 += col[static_cast<size_t>(b) * dim];
      s1 += col[static_cast<size_t>(b + 16) * dim];
      s2 += col[static_cast<size_t>(b + 32) * dim];
      s3 += col[static_cast<size_t>(b + 48) * dim];
    }
    for (; b < blocks; b += 16) s0 += col[static_cast<size_t>(b) * dim];
  }
  red[group][lane] = (s0 + s1) + (s2 + s3);
  __syncthreads();
  if (group == 0 && c < dim) {
    float total = 0.0f;
#pragma unroll
    for (int g = 0; g < 16; ++g) total += red[g][lane];
    out[c] = total;
    if (!dev_finite(total)) dev_raise_fault(fault, tag);
  }
}
__global__ __launch_bounds__(1024) void column_sum_wide_kernel(const float* __restrict__ partial,
                                                               float* __restrict__ out, int blocks, int dim,
                                                               OmxFaultWord* fault, unsigned long long tag) {
  column_sum_wide(partial, out, blocks, dim, fault, tag);
}

// One column whose sum is a value blend's: 256 threads in order, then a tree.
__device__ __forceinline__ void column_sum_blend(const OmxColumnSum& s, OmxFaultWord* fault) {
  __shared__ float red[256];
  if (threadIdx.x < 256) {
    float acc = 0.0f;
    for (int b = threadIdx.x; b < s.blocks; b += 256) acc += s.partial[b];
    red[threadIdx.x] = acc;
  }
  __syncthreads();
  for (int step = 128; step >= 1; step >>= 1) {
    if (threadIdx.x < step) red[threadIdx.x] += red[threadIdx.x + step];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    float sig, rest;
    dev_sigmoid_both(*s.blend, &sig, &rest);
    const float v = red[0] * sig * rest;
    if (!dev_finite(v)) dev_raise_fault(fault, s.tag);
    *s.out = v;
  }
}

// Many of them in one launch. One is 4 to 18 workgroups that wait for memory, 4 to 5 us whatever its size; the norms' of a
// backward together take about as long as one (a step with nine norms over 2048 x 256: 1233 -> 1212 us; with thirteen over 3500 x 512:
// 2373 -> 2346).
constexpr int SUM_LIST = 64;
struct ColumnSumList {
  OmxColumnSum of[SUM_LIST];  // (2.5 KiB of kernel arguments)
};
__global__ __launch_bounds__(1024) void column_sum_list_kernel(ColumnSumList list, OmxFaultWord* fault) {
  const OmxColumnSum& s = list.of[blockIdx.y];
  if (static_cast<int>(blockIdx.x) * 64 >= s.dim) return;
  if (s.blend) column_sum_blend(s, fault);
  else column_sum_wide(s.partial, s.out, s.blocks, s.dim, fault, s.tag);
}

// Stage 1 of a tall column sum: block (x, g) adds rows [g * per_group, (g + 1) * per_group) of its
// 64 columns, four row groups in parallel, then a fixed four-way sum.
__global__ __launch_bounds__(256) void column_sum_groups_kernel(const float* __restrict__ partial,
                                                                float* __restrict__ scratch, int blocks, int dim,
                                                                int per_group) {
  __shared__ float red[4][64];
  const int lane = threadIdx.x & 63, group = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  const int first = blockIdx.y * per_group, last = min(blocks, first + per_group);
  float s = 0.0f;
  if (c < dim)
    for (int b = first + group; b < last; b += 4) s += partial[static_cast<size_t>(b) * dim + c];
  red[group][lane] = s;
  __syncthreads();
  if (group == 0 && c < dim)
    scratch[static_cast<size_t>(blockIdx.y) * dim + c] = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
}

// ---------------------------------------------------------------- embedding
template <typename TT, typename TO>
__global__ void embedding_fwd_kernel(const TT* __restrict__ table, const unsigned int* __restrict__ ids,
                                     TO* __restrict__ out, size_t tokens, size_t vocab, int dim, OmxFaultWord* fault,
                                     unsigned long long tag) {
  const int lane = threadIdx.x & 63;
  const size_t n = static_cast<size_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (n >= tokens) return;
  size_t id = ids[n];
  TO* dst = out + n * dim;
  if (id >= vocab) {
    // Refused id: the row is zero-filled and the call reports OutOfRange.
    for (int c = lane; c < dim; c += 64) dev_store<TO>(dst, c, 0.0f);
    if (lane == 0) dev_raise_range(fault, tag);
    return;
  }
  const TT* src = table + id * dim;
  if constexpr (sizeof(TT) == sizeof(TO)) {
    // Same storage: a bit copy (NaN payloads and -0 survive).
    for (int c = lane; c < dim; c += 64) dst[c] = src[c];
  } else {
    for (int c = lane; c < dim; c += 64) dev_store<TO>(dst, c, dev_load<TT>(src, c));
  }
}

__global__ void count_ids_kernel(const unsigned int* __restrict__ ids, unsigned int* __restrict__ counts,
                                 size_t tokens, size_t vocab, OmxFaultWord* fault, unsigned long long tag) {
  size_t n = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (n >= tokens) return;
  unsigned int id = ids[n];
  if (id >= vocab) {
    dev_raise_range(fault, tag);
    return;
  }
  atomicAdd(&counts[id], 1u);
}

// Exclusive scan of counts[vocab] into offsets[vocab + 1] and a copy into
// cursor[vocab]; one 1024-thread block walks the array in 1024-wide strips.
__global__ __launch_bounds__(1024) void scan_counts_kernel(const unsigned int* __restrict__ counts,
                                                           unsigned int* __restrict__ offsets,
                                                           unsigned int* __restrict__ cursor, size_t vocab) {
  __shared__ unsigned int wave_tot[16];
  __shared__ unsigned int carry;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (size_t base = 0; base < vocab; base += 1024) {
    size_t i = base + threadIdx.x;
    unsigned int v = i < vocab ? counts[i] : 0u;
    unsigned int incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      unsigned int t = __shfl_up(incl, off, 64);
      if (lane >= off) incl += t;
    }
    if (lane == 63) wave_tot[wave] = incl;
    __syncthreads();
    unsigned int before = carry;
    for (int wv = 0; wv < wave; ++wv) before += wave_tot[wv];
    unsigned int excl = before + incl - v;
    if (i < vocab) {
      offsets[i] = excl;
      cursor[i] = excl;
    }
    __syncthreads();
    if (threadIdx.x == 1023) carry = excl + v;
    __syncthreads();
  }
  if (threadIdx.x == 0) offsets[vocab] = carry;
}

// The same scan over many blocks, for tables of more than a few thousand rows (one block walks
// 50304 counts in 55 us): every block of 1024 counts leaves its total, then every block adds up the
// totals before it (at most SCAN_MAX_BLOCKS of them) and scans its own counts behind that.
constexpr int SCAN_MAX_BLOCKS = 1024;
__device__ __forceinline__ unsigned int scan_block_1024(unsigned int v, unsigned int* wave_tot, unsigned int* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned int incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    unsigned int t = __shfl_up(incl, off, 64);
    if (lane >= off) incl += t;
  }
  if (lane == 63) wave_tot[wave] = incl;
  __syncthreads();
  unsigned int before = 0, all = 0;
  for (int wv = 0; wv < 16; ++wv) {
    if (wv < wave) before += wave_tot[wv];
    all += wave_tot[wv];
  }
  *total = all;
  return before + incl - v;  // exclusive, within the block
}
__global__ __launch_bounds__(1024) void scan_totals_kernel(const unsigned int* __restrict__ counts,
                                                           unsigned int* __restrict__ totals, size_t vocab) {
  __shared__ unsigned int wave_tot[16];
  const size_t i = static_cast<size_t>(blockIdx.x) * 1024 + threadIdx.x;
  unsigned int total;
  scan_block_1024(i < vocab ? counts[i] : 0u, wave_tot, &total);
  if (threadIdx.x == 0) totals[blockIdx.x] = total;
}
__global__ __launch_bounds__(1024) void scan_blocks_kernel(const unsigned int* __restrict__ counts,
                                                           const unsigned int* __restrict__ totals,
                                                           unsigned int* __restrict__ offsets,
                                                           unsigned int* __restrict__ cursor, size_t vocab) {
  __shared__ unsigned int wave_tot[16];
  __shared__ unsigned int lead_tot[16];
  // The totals of the blocks before this one: thread t takes block t's.
  unsigned int mine = threadIdx.x < blockIdx.x ? totals[threadIdx.x] : 0u;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mine += __shfl_xor(mine, off, 64);
  if ((threadIdx.x & 63) == 0) lead_tot[threadIdx.x >> 6] = mine;
  __syncthreads();
  unsigned int lead = 0;
  for (int wv = 0; wv < 16; ++wv) lead += lead_tot[wv];
  const size_t i = static_cast<size_t>(blockIdx.x) * 1024 + threadIdx.x;
  const unsigned int v = i < vocab ? counts[i] : 0u;
  unsigned int total;
  const unsigned int excl = lead + scan_block_1024(v, wave_tot, &total);
  if (i < vocab) {
    offsets[i] = excl;
    cursor[i] = excl;
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) offsets[vocab] = lead + total;
}

__global__ void fill_positions_kernel(const unsigned int* __restrict__ ids, unsigned int* __restrict__ cursor,
                                      unsigned int* __restrict__ positions, size_t tokens, size_t vocab) {
  size_t n = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (n >= tokens) return;
  unsigned int id = ids[n];
  if (id >= vocab) return;
  unsigned int slot = atomicAdd(&cursor[id], 1u);
  positions[slot] = static_cast<unsigned int>(n);
}

// The three in one for a batch and a table that one workgroup's LDS holds the counts of: counts, offsets and positions (2048 tokens
// in a table of 8192: 5.3 us against five launches of 2.5 to 4.7 each).
constexpr uint64_t INDEX_TOKENS = 16384, INDEX_VOCAB = 34816;
__device__ __host__ inline unsigned int index_at(unsigned int i) { return i + (i >> 5); }  // a thread's run of 32 counts: distinct banks
__global__ __launch_bounds__(1024) void index_ids_kernel(const unsigned int* __restrict__ ids, unsigned int* __restrict__ offsets,
                                                         unsigned int* __restrict__ positions, unsigned int tokens,
                                                         unsigned int vocab, OmxFaultWord* fault, unsigned long long tag) {
  extern __shared__ unsigned int index_counts[];  // [index_at(vocab)]: counts, then where a row's next position goes
  __shared__ unsigned int wave_tot[16];
  constexpr int EACH = INDEX_TOKENS / 1024;
  const unsigned int tid = threadIdx.x;
  unsigned int id[EACH];  // all in flight at once, and kept for the second pass
#pragma unroll
  for (int i = 0; i < EACH; ++i)
    if (i * 1024u < tokens) id[i] = ids[min(tid + i * 1024u, tokens - 1)];
  for (unsigned int i = tid; i < vocab; i += 1024) index_counts[index_at(i)] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < EACH; ++i)
    if (tid + i * 1024u < tokens) {
      if (id[i] >= vocab) dev_raise_range(fault, tag);
      else atomicAdd(&index_counts[index_at(id[i])], 1u);
    }
  __syncthreads();
  const unsigned int each = (vocab + 1023) / 1024, first = min(vocab, tid * each), last = min(vocab, first + each);
  unsigned int mine = 0;
  for (unsigned int i = first; i < last; ++i) mine += index_counts[index_at(i)];
  unsigned int total;
  unsigned int at = scan_block_1024(mine, wave_tot, &total);
  for (unsigned int i = first; i < last; ++i) {
    const unsigned int c = index_counts[index_at(i)];
    index_counts[index_at(i)] = at;
    at += c;
  }
  __syncthreads();
  for (unsigned int i = tid; i < vocab; i += 1024) offsets[i] = index_counts[index_at(i)];
  if (tid == 0) offsets[vocab] = total;
  __syncthreads();  // (read before the positions move them)
#pragma unroll
  for (int i = 0; i < EACH; ++i)
    if (tid + i * 1024u < tokens && id[i] < vocab) positions[atomicAdd(&index_counts[index_at(id[i])], 1u)] = tid + i * 1024u;
}

// One wave per table row and columns blockIdx.y, + gridDim.y, ... of 64 x 4 (x 8 of single ones): zero them, or add the row's tokens'
// gradients in ascending token order, so the f32 sums carry the CPU scatter's bits (pointwise.rs:196-207). `positions` hold a row's
// tokens in arrival order. Up to 64 are sorted by a bitonic network over the lanes; more, by the whole workgroup, whose waves then take
// the row's columns in turn: a bitmap of 32768 tokens at a time, its set bits listed 2048 tokens at a time. Bound by the latency of
// the gradient rows, so eight are in flight (one at a time, 16 tokens each of 1024 rows of 768: 38.7 us, now 12.3 on three times the
// waves; a bitmap per wave had the empty rows of a large table wait for LDS: 16384 tokens of 50304 rows 54 us, now 36).
// V = 4: a lane owns four consecutive columns (16-byte accesses; dim a multiple of 4, aligned rows).
// ADD: the row's sum, complete, is added to what `table_grad` holds (the bits of the scatter
// followed by accumulate_grad), and rows no token names are left alone.
template <typename TG, int V, bool ADD>
__global__ __launch_bounds__(ROW_THREADS) void embedding_bwd_kernel(const unsigned int* __restrict__ offsets,
                                                                    const unsigned int* __restrict__ positions,
                                                                    const TG* __restrict__ grad,
                                                                    float* __restrict__ table_grad, size_t vocab,
                                                                    int dim, size_t tokens, OmxFaultWord* fault,
                                                                    unsigned long long tag) {
  constexpr int WINDOW = 32768, GROUP = 2048;  // tokens; a group is a word per lane
  constexpr unsigned int SHORT = 64;
  __shared__ unsigned int bitmap[WINDOW / 32];
  __shared__ unsigned short list[GROUP];
  __shared__ unsigned int listed;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const size_t v0 = static_cast<size_t>(blockIdx.x) * 4;
  unsigned int at[5];  // where the four rows' positions start
#pragma unroll
  for (int r = 0; r < 5; ++r) at[r] = offsets[min(v0 + r, vocab)];
  constexpr int CHUNKS = V == 4 ? 1 : 8, COLUMNS = 64 * V * CHUNKS;
  bool bad = false;
  float acc[CHUNKS][V];
  auto clear = [&] {
#pragma unroll
    for (int j = 0; j < CHUNKS; ++j)
#pragma unroll
      for (int e = 0; e < V; ++e) acc[j][e] = 0.0f;
  };
  // The gradients of tokens p of lanes s .. s + AHEAD - 1, and of lanes 0 .. n - 1, in that order.
  auto add_some = [&](int c0, unsigned int p, unsigned int s, auto ahead) {
    constexpr int AHEAD = decltype(ahead)::value;
    float g[AHEAD][CHUNKS][V];
#pragma unroll
    for (int r = 0; r < AHEAD; ++r) {
      const TG* src = grad + static_cast<size_t>(static_cast<unsigned int>(__builtin_amdgcn_readlane(p, s + r))) * dim;
#pragma unroll
      for (int j = 0; j < CHUNKS; ++j) {
        const int c = c0 + (j * 64 + lane) * V;
        if constexpr (V == 4) dev_load4<TG>(src, min(c, dim - 4), g[r][j]);
        else g[r][j][0] = dev_load<TG>(src, min(c, dim - 1));
      }
    }
#pragma unroll
    for (int r = 0; r < AHEAD; ++r)
#pragma unroll
      for (int j = 0; j < CHUNKS; ++j)
#pragma unroll
        for (int e = 0; e < V; ++e) acc[j][e] = acc[j][e] + g[r][j][e];
  };
  auto add_rows = [&](int c0, unsigned int p, unsigned int n) {
    unsigned int s = 0;
    if constexpr (V == 4)
      for (; s + 8 <= n; s += 8) add_some(c0, p, s, std::integral_constant<int, 8>());
    for (; s + 2 <= n; s += 2) add_some(c0, p, s, std::integral_constant<int, 2>());
    if (s < n) add_some(c0, p, s, std::integral_constant<int, 1>());
  };
  auto store = [&](float* dst, int c0, bool add) {
#pragma unroll
    for (int j = 0; j < CHUNKS; ++j) {
      const int c = c0 + (j * 64 + lane) * V;
      if (c < dim) {
#pragma unroll
        for (int e = 0; e < V; ++e) bad |= !dev_finite(acc[j][e]);
        if (add) {
          if constexpr (V == 4) {
            const float4 old = *reinterpret_cast<const float4*>(dst + c);
            acc[j][0] = old.x + acc[j][0];
            acc[j][1] = old.y + acc[j][1];
            acc[j][2] = old.z + acc[j][2];
            acc[j][3] = old.w + acc[j][3];
          } else {
            acc[j][0] = dst[c] + acc[j][0];
          }
        }
        if constexpr (V == 4) *reinterpret_cast<float4*>(dst + c) = make_float4(acc[j][0], acc[j][1], acc[j][2], acc[j][3]);
        else dst[c] = acc[j][0];
      }
    }
  };
  const size_t v = v0 + wave;
  const unsigned int begin = wave == 0 ? at[0] : wave == 1 ? at[1] : wave == 2 ? at[2] : at[3];
  const unsigned int len = (wave == 0 ? at[1] : wave == 1 ? at[2] : wave == 2 ? at[3] : at[4]) - begin;
  if (v < vocab && len <= SHORT && !(ADD && len == 0)) {
    unsigned int few = 0xffffffffu;
    if (static_cast<unsigned int>(lane) < len) few = positions[begin + lane];
    for (unsigned int k = 2; k >> 1 < len; k <<= 1)
      for (unsigned int j = k >> 1; j > 0; j >>= 1) {
        const unsigned int other = __shfl_xor(few, j, 64);
        const bool ascending = (lane & k) == 0, keep_min = ((lane & j) == 0) == ascending;
        few = keep_min ? min(few, other) : max(few, other);
      }
    for (int c0 = blockIdx.y * COLUMNS; c0 < dim; c0 += gridDim.y * COLUMNS) {
      clear();
      add_rows(c0, few, len);
      store(table_grad + v * dim, c0, ADD);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (at[r + 1] - at[r] <= SHORT) continue;  // (the workgroup's: so are the barriers below)
    for (int pass0 = blockIdx.y * COLUMNS; pass0 < dim; pass0 += 4 * gridDim.y * COLUMNS) {
      const int c0 = pass0 + wave * gridDim.y * COLUMNS;
      clear();
      unsigned int left = at[r + 1] - at[r];
      for (size_t base = 0; base < tokens && left > 0; base += WINDOW) {
        __syncthreads();
        for (int i = threadIdx.x; i < WINDOW / 32; i += ROW_THREADS) bitmap[i] = 0;
        __syncthreads();
        for (unsigned int s = at[r] + threadIdx.x; s < at[r + 1]; s += ROW_THREADS) {
          const size_t rel = static_cast<size_t>(positions[s]) - base;  // wraps far above the window when below it
          if (rel < WINDOW) atomicOr(&bitmap[rel >> 5], 1u << (rel & 31));
        }
        for (int group = 0; group < WINDOW / GROUP && left > 0; ++group) {
          __syncthreads();  // the bitmap is whole, the previous list has been read
          if (wave == 0) {
            unsigned int w = bitmap[group * 64 + lane], incl = __popc(w);
            const unsigned int count = incl;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
              const unsigned int t = __shfl_up(incl, off, 64);
              if (lane >= off) incl += t;
            }
            if (lane == 63) listed = incl;
            for (unsigned int to = incl - count; w; w &= w - 1) list[to++] = static_cast<unsigned short>(lane * 32 + __ffs(w) - 1);
          }
          __syncthreads();
          const unsigned int total = __builtin_amdgcn_readfirstlane(listed);
          if (c0 < dim)
            for (unsigned int s = 0; s < total; s += 64)
              add_rows(c0, static_cast<unsigned int>(base) + group * GROUP + list[min(s + lane, total - 1)], min(64u, total - s));
          left -= total;
        }
      }
      if (c0 < dim) store(table_grad + (v0 + r) * dim, c0, ADD);
    }
  }
  if (bad) dev_raise_fault(fault, tag);
}

// ---------------------------------------------------------------- argmax / top-k
// Order of rank_logits (backend.rs:184-195): value descending with +0 == -0,
// then column ascending. `before(a, b)`: a ranks ahead of b.
__device__ __forceinline__ float rank_key(float v) { return v == 0.0f ? 0.0f : v; }
__device__ __forceinline__ bool ranks_before(float va, unsigned int ia, float vb, unsigned int ib) {
  float ka = rank_key(va), kb = rank_key(vb);
  return ka > kb || (ka == kb && ia < ib);
}

// One workgroup per row. The row is read once, in 16-byte pieces between its first and last aligned element;
// what bounds it is latency, so a long row takes 1024 threads with eight pieces in flight each (one wave per row
// walked 50304 columns in 786 dependent loads: 209 us for one row, now 10). Ties go to the lowest
// column: every comparison prefers it, so the order in which threads meet does not matter.
// SLICES > 1 (few long rows): that many workgroups per row, each leaving its best in `parts` for argmax_meet_kernel: one row of 50304
// columns 11.6 us on one compute unit, 7.9 in both launches.
constexpr int ARGMAX_SLICES = 16;
template <int THREADS, int SLICES>
__global__ __launch_bounds__(THREADS) void argmax_rows_kernel(const float* __restrict__ x, unsigned int cols,
                                                              unsigned int* __restrict__ out, uint2* __restrict__ parts,
                                                              OmxFaultWord* fault, unsigned long long tag) {
  __shared__ float wave_best[THREADS / 64];
  __shared__ unsigned int wave_idx[THREADS / 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const size_t row = blockIdx.x;
  const float* r = x + row * cols;
  float best = -INFINITY;
  unsigned int idx = 0xffffffffu;
  bool bad = false;
  auto take = [&](float v, unsigned int c) {
    bad |= !dev_finite(v);
    if (idx == 0xffffffffu || v > best || (v == best && c < idx)) {
      best = v;
      idx = c;
    }
  };
  const unsigned int lead = min(cols, static_cast<unsigned int>((16 - (reinterpret_cast<uintptr_t>(r) & 15)) & 15) / 4);
  const unsigned int pieces = (cols - lead) / 4;
  if (blockIdx.y == 0 && tid < static_cast<int>(lead)) take(r[tid], tid);
  const float4* body = reinterpret_cast<const float4*>(r + lead);
  const unsigned int each = SLICES == 1 ? pieces : (pieces + SLICES - 1) / SLICES;
  const unsigned int from = min(pieces, each * blockIdx.y), to = min(pieces, from + each);
  for (unsigned int p0 = from + tid; p0 < to; p0 += 8 * THREADS) {
    float4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = body[min(p0 + i * THREADS, to - 1)];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const unsigned int c = lead + min(p0 + i * THREADS, to - 1) * 4;  // a repeated piece changes nothing
      take(v[i].x, c);
      take(v[i].y, c + 1);
      take(v[i].z, c + 2);
      take(v[i].w, c + 3);
    }
  }
  if (blockIdx.y == gridDim.y - 1)
    for (unsigned int c = lead + pieces * 4 + tid; c < cols; c += THREADS) take(r[c], c);
  auto meet = [&](float ov, unsigned int oi) {
    if (oi != 0xffffffffu && (idx == 0xffffffffu || ov > best || (ov == best && oi < idx))) {
      best = ov;
      idx = oi;
    }
  };
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float ov = __shfl_xor(best, off, 64);
    const unsigned int oi = __shfl_xor(idx, off, 64);
    meet(ov, oi);
  }
  if (lane == 0) {
    wave_best[tid >> 6] = best;
    wave_idx[tid >> 6] = idx;
  }
  bad = __syncthreads_or(bad);
  if (tid == 0) {
    for (int w = 1; w < THREADS / 64; ++w) meet(wave_best[w], wave_idx[w]);
    if constexpr (SLICES == 1) out[row] = idx;
    else parts[row * SLICES + blockIdx.y] = make_uint2(__float_as_uint(best), idx);
    if (bad) dev_raise_fault(fault, tag);
  }
}
__global__ __launch_bounds__(64) void argmax_meet_kernel(const uint2* __restrict__ parts, unsigned int* __restrict__ out) {
  const uint2 part = parts[blockIdx.x * ARGMAX_SLICES + threadIdx.x % ARGMAX_SLICES];
  float best = __uint_as_float(part.x);
  unsigned int idx = part.y;
#pragma unroll
  for (int off = ARGMAX_SLICES / 2; off > 0; off >>= 1) {
    const float ov = __shfl_xor(best, off, 64);
    const unsigned int oi = __shfl_xor(idx, off, 64);
    if (oi != 0xffffffffu && (idx == 0xffffffffu || ov > best || (ov == best && oi < idx))) {
      best = ov;
      idx = oi;
    }
  }
  if (threadIdx.x == 0) out[blockIdx.x] = idx;
}

// k passes over the row; pass j picks the best element ranked after pass
// j-1's pick. NaN and +inf are refused, -inf sorts last.
__global__ void topk_rows_kernel(const float* __restrict__ x, size_t rows, unsigned int cols, unsigned int k,
                                 float* __restrict__ values, unsigned int* __restrict__ ids, OmxFaultWord* fault,
                                 unsigned long long tag) {
  const int lane = threadIdx.x & 63;
  const size_t row = static_cast<size_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float* r = x + row * cols;
  bool bad = false;
  float prev_v = 0.0f;
  unsigned int prev_i = 0;
  for (unsigned int j = 0; j < k; ++j) {
    float best = 0.0f;
    unsigned int idx = 0xffffffffu;
    for (unsigned int c = lane; c < cols; c += 64) {
      float v = r[c];
      if (j == 0) bad |= (v != v) || v == INFINITY;
      if (j > 0 && !ranks_before(prev_v, prev_i, v, c)) continue;
      if (idx == 0xffffffffu || ranks_before(v, c, best, idx)) {
        best = v;
        idx = c;
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      float ov = __shfl_xor(best, off, 64);
      unsigned int oi = __shfl_xor(idx, off, 64);
      if (oi != 0xffffffffu && (idx == 0xffffffffu || ranks_before(ov, oi, best, idx))) {
        best = ov;
        idx = oi;
      }
    }
    prev_v = best;
    prev_i = idx;
    if (lane == 0) {
      values[row * k + j] = best;
      ids[row * k + j] = idx;
    }
  }
  bad = __any(bad);
  if (lane == 0 && bad) dev_raise_fault(fault, tag);
}

inline int per_for_dim(uint64_t dim) {
  const int options[] = {1, 2, 4, 8, 12, 16, 32, 64, 128};
  for (int p : options)
    if (static_cast<uint64_t>(p) * 64 >= dim) return p;
  return 0;
}

template <typename TX, typename TY>
int32_t launch_rms_fwd(omx_ctx* ctx, const RmsTensors& t, int count, uint64_t dim, float eps) {
  const dim3 grid(static_cast<unsigned>((std::max(t.of[0].rows, t.of[1].rows) + 3) / 4), count), block(ROW_THREADS);
#define RMS_FWD(P)                                                                                                   \
  case P:                                                                                                            \
    omx_launch(ctx, (rms_fwd_kernel<TX, TY, P>), grid, block, 0, t, static_cast<int>(dim), eps, ctx->fault);         \
    break;
  switch (per_for_dim(dim)) {
    RMS_FWD(1) RMS_FWD(2) RMS_FWD(4) RMS_FWD(8) RMS_FWD(12) RMS_FWD(16) RMS_FWD(32) RMS_FWD(64) RMS_FWD(128)
    default:
      return omx_fail(ctx, OMX_UNSUPPORTED, "rms_norm_forward: dim %llu above 8192", (unsigned long long)dim);
  }
#undef RMS_FWD
  OMX_LAUNCH_CHECK(ctx, "rms_fwd_kernel");
  return OMX_OK;
}
int32_t launch_rms_fwd(omx_ctx* ctx, const RmsTensors& t, int count, int32_t x_dtype, int32_t y_dtype, uint64_t dim, float eps) {
  if (x_dtype == OMX_F32 && y_dtype == OMX_F32) return launch_rms_fwd<float, float>(ctx, t, count, dim, eps);
  if (x_dtype == OMX_F32) return launch_rms_fwd<float, unsigned short>(ctx, t, count, dim, eps);
  if (y_dtype == OMX_F32) return launch_rms_fwd<unsigned short, float>(ctx, t, count, dim, eps);
  return launch_rms_fwd<unsigned short, unsigned short>(ctx, t, count, dim, eps);
}

// 32 rows per block, 16 where those are under a block per compute unit and there is room for as many partial rows, more when that
// would leave over 2048 partial rows to add.
uint64_t rms_partial_bytes(uint64_t blocks, uint64_t dim) { return (blocks + OMX_COLUMN_SUM_GROUPS) * dim * sizeof(float); }
int rms_rows_per_block(omx_ctx* ctx, uint64_t rows, uint64_t dim) {
  int rows_per_block = rows < 32ull * 256 && omx_workspace_fits(ctx, rms_partial_bytes((rows + 15) / 16, dim)) ? 16 : 32;
  while ((rows + rows_per_block - 1) / rows_per_block > 2048 && rows_per_block < (1 << 20)) rows_per_block *= 2;
  return rows_per_block;
}
uint64_t rms_blocks(const RmsRows& t) { return (t.rows + t.rows_per_block - 1) / t.rows_per_block; }

template <typename TX, typename TG, typename TO>
int32_t launch_rms_bwd(omx_ctx* ctx, const RmsTensors& t, int count, uint64_t dim, float eps) {
  const uint64_t blocks = count == 1 ? rms_blocks(t.of[0]) : std::max(rms_blocks(t.of[0]), rms_blocks(t.of[1]));
  dim3 grid(static_cast<unsigned>(blocks), count), block(ROW_THREADS);
  size_t smem = 4 * dim * sizeof(float);
#define RMS_BWD(P)                                                                                                   \
  case P:                                                                                                            \
    omx_launch(ctx, (rms_bwd_kernel<TX, TG, TO, P>), grid, block, smem, t, static_cast<int>(dim), eps, ctx->fault);  \
    break;
  switch (per_for_dim(dim)) {
    RMS_BWD(1) RMS_BWD(2) RMS_BWD(4) RMS_BWD(8) RMS_BWD(12) RMS_BWD(16) RMS_BWD(32) RMS_BWD(64)
    default:
      return omx_fail(ctx, OMX_UNSUPPORTED, "rms_norm_backward: dim %llu above 4096", (unsigned long long)dim);
  }
#undef RMS_BWD
  OMX_LAUNCH_CHECK(ctx, "rms_bwd_kernel");
  return OMX_OK;
}
int32_t launch_rms_bwd(omx_ctx* ctx, const RmsTensors& t, int count, int32_t x_dtype, int32_t gy_dtype, int32_t gx_dtype, uint64_t dim,
                       float eps) {
  typedef unsigned short h16;
  switch ((x_dtype == OMX_BF16 ? 4 : 0) | (gy_dtype == OMX_BF16 ? 2 : 0) | (gx_dtype == OMX_BF16 ? 1 : 0)) {
    case 0: return launch_rms_bwd<float, float, float>(ctx, t, count, dim, eps);
    case 1: return launch_rms_bwd<float, float, h16>(ctx, t, count, dim, eps);
    case 2: return launch_rms_bwd<float, h16, float>(ctx, t, count, dim, eps);
    case 3: return launch_rms_bwd<float, h16, h16>(ctx, t, count, dim, eps);
    case 4: return launch_rms_bwd<h16, float, float>(ctx, t, count, dim, eps);
    case 5: return launch_rms_bwd<h16, float, h16>(ctx, t, count, dim, eps);
    case 6: return launch_rms_bwd<h16, h16, float>(ctx, t, count, dim, eps);
    default: return launch_rms_bwd<h16, h16, h16>(ctx, t, count, dim, eps);
  }
}

// Whether two ranges share no byte.
bool no_overlap(const void* a, uint64_t a_bytes, const void* b, uint64_t b_bytes) {
  const uintptr_t pa = reinterpret_cast<uintptr_t>(a), pb = reinterpret_cast<uintptr_t>(b);
  return pa + a_bytes <= pb || pb + b_bytes <= pa;
}
uint64_t float_bytes(int32_t dtype) { return dtype == OMX_BF16 ? 2 : 4; }

int32_t rms_forward_impl(omx_ctx* ctx, const char* op, uint32_t fault_op, const void* x, int32_t x_dtype,
                         const void* w, void* y, int32_t y_dtype, uint64_t rows, uint64_t dim, float eps) {
  unsigned long long tag = omx_tag(ctx, fault_op);
  (void)op;
  const float* wf = static_cast<const float*>(w);
  if (omx_rms_vec_eligible(dim, {x, w, y}))
    return omx_rms_forward_vec(ctx, x, x_dtype, nullptr, OMX_F32, wf, nullptr, y, y_dtype, rows, dim, eps, tag);
  RmsTensors t{};
  t.of[0] = {x, nullptr, wf, y, nullptr, rows, 0, tag};
  return launch_rms_fwd(ctx, t, 1, x_dtype, y_dtype, dim, eps);
}

int32_t rms_backward_impl(omx_ctx* ctx, uint32_t fault_op, const void* x, int32_t x_dtype, const void* w,
                          const void* gy, int32_t gy_dtype, void* gx, int32_t gx_dtype, void* gw, uint64_t rows,
                          uint64_t dim, float eps) {
  unsigned long long tag = omx_tag(ctx, fault_op);
  const float* wf = static_cast<const float*>(w);
  float* gwf = static_cast<float*>(gw);
  if (omx_rms_vec_eligible(dim, {x, w, gy, gx, gw}))
    return omx_rms_backward_vec(ctx, x, x_dtype, wf, gy, gy_dtype, nullptr, gx, gx_dtype, nullptr, gwf, rows, dim, eps,
                                tag);
  RmsTensors t{};
  t.of[0] = {x, gy, wf, gx, nullptr, rows, rms_rows_per_block(ctx, rows, dim), tag};
  const uint64_t blocks = rms_blocks(t.of[0]);
  void* partial = nullptr;
  int32_t rc = omx_workspace(ctx, rms_partial_bytes(blocks, dim), &partial);
  if (rc != OMX_OK) return rc;
  t.of[0].partial = static_cast<float*>(partial);
  rc = launch_rms_bwd(ctx, t, 1, x_dtype, gy_dtype, gx_dtype, dim, eps);
  if (rc != OMX_OK) return rc;
  // A narrow row leaves the column sum one or two workgroups: it then adds its rows in two stages.
  return omx_column_sum(ctx, t.of[0].partial, gwf, blocks, dim, tag, t.of[0].partial + blocks * dim);
}

bool finite_host(float v) { return v == v && v != INFINITY && v != -INFINITY; }

}  // namespace

int32_t omx_column_sum(omx_ctx* ctx, const float* partial, float* out, uint64_t blocks, uint64_t dim,
                       unsigned long long tag, float* scratch, hipEvent_t stop, bool wait) {
  if (wait) {
    ctx->sums.push_back({partial, out, tag, static_cast<int>(blocks), static_cast<int>(dim)});
    return OMX_OK;
  }
  const unsigned col_blocks = static_cast<unsigned>((dim + 63) / 64);
  // Sixteen rows at once from 17 rows on (four at a time, each waiting for the one before, 128 rows of 256 columns took
  // 9.2 us, now 2.9).
  if (blocks > 16 && blocks <= OMX_COLUMN_SUM_WIDE_ROWS) {
    omx_launch_timed(ctx, column_sum_wide_kernel, dim3(col_blocks), dim3(1024), 0, nullptr, stop, partial, out,
                     static_cast<int>(blocks), static_cast<int>(dim), ctx->fault, tag);
    OMX_LAUNCH_CHECK(ctx, "column_sum_wide_kernel");
    return OMX_OK;
  }
  if (scratch && blocks > 4 * OMX_COLUMN_SUM_GROUPS) {
    // Stage 1: group g adds its contiguous share of the rows into scratch[g]; stage 2 adds the groups.
    const int per_group = static_cast<int>((blocks + OMX_COLUMN_SUM_GROUPS - 1) / OMX_COLUMN_SUM_GROUPS);
    omx_launch(ctx, column_sum_groups_kernel, dim3(col_blocks, OMX_COLUMN_SUM_GROUPS), dim3(256), 0,
                       partial, scratch, static_cast<int>(blocks), static_cast<int>(dim), per_group);
    OMX_LAUNCH_CHECK(ctx, "column_sum_groups_kernel");
    partial = scratch;
    blocks = OMX_COLUMN_SUM_GROUPS;
  }
  omx_launch_timed(ctx, column_sum_kernel, dim3(col_blocks), dim3(256), 0, nullptr, stop, partial, out,
                   static_cast<int>(blocks), static_cast<int>(dim), ctx->fault, tag);
  OMX_LAUNCH_CHECK(ctx, "column_sum_kernel");
  return OMX_OK;
}

int32_t omx_column_sums(omx_ctx* ctx, const OmxColumnSum* sums, int count, bool wait) {
  if (wait) {
    ctx->sums.insert(ctx->sums.end(), sums, sums + count);
    return OMX_OK;
  }
  for (int first = 0; first < count; first += SUM_LIST) {
    ColumnSumList list{};
    const int n = std::min(SUM_LIST, count - first);
    int dim = 0;
    for (int i = 0; i < n; ++i) {
      list.of[i] = sums[first + i];
      dim = std::max(dim, list.of[i].dim);
    }
    OmxKernelTimer timer(ctx, OMX_K_RMS_BWD, 0.0);  // (the norms' own launches count the bytes)
    omx_launch_timed(ctx, column_sum_list_kernel, dim3((dim + 63) / 64, static_cast<unsigned>(n)), dim3(1024), 0, timer.start(), timer.stop(),
                     list, ctx->fault);
    OMX_LAUNCH_CHECK(ctx, "column_sum_list_kernel");
  }
  return OMX_OK;
}

// In the kernel's order of rows; the partial rows' memory is free again behind it. Nothing waits any more if a launch fails.
int32_t omx_form_sums(omx_ctx* ctx) {
  const std::vector<OmxColumnSum> sums = std::exchange(ctx->sums, {});
  ctx->sums_used = 0;
  return omx_column_sums(ctx, sums.data(), static_cast<int>(sums.size()), false);
}

// The rows are those of the wide kernel, whose order the list keeps. Full memory is formed and used again. (Rows of more than 1 MiB
// too: 16384 rows of 768 leave 1.5 MiB a norm, and the step that makes 25 of them takes 18.03 ms, 18.11 with a launch for each; with
// 8192 rows 11.44 and 11.51, with gates 26.06 and 26.19. Three runs of each, in turn; those of one side are within 0.06.)
float* omx_partial_rows(omx_ctx* ctx, uint64_t blocks, uint64_t dim) {
  if (!ctx->sums_wait || blocks <= 16 || blocks > OMX_COLUMN_SUM_WIDE_ROWS) return nullptr;
  constexpr uint64_t kMost = 64ull << 20;
  const uint64_t bytes = (blocks * dim * sizeof(float) + 255) / 256 * 256;
  if (ctx->sums_used + bytes > ctx->workspace_bytes[kSumsSlot] && omx_form_sums(ctx) != OMX_OK) return nullptr;
  const uint64_t held = ctx->workspace_bytes[kSumsSlot];
  uint64_t want = held >= ctx->sums_used + bytes ? held : std::max(bytes, std::min(kMost, bytes * ctx->sums_expected));
  while (want >= 8 * bytes && !omx_workspace_fits(ctx, want, kSumsSlot)) want /= 2;
  void* arena = omx_workspace_if_room(ctx, want, kSumsSlot);
  if (!arena) return nullptr;
  float* at = reinterpret_cast<float*>(static_cast<char*>(arena) + ctx->sums_used);
  ctx->sums_used += bytes;
  return at;
}

extern "C" {

int32_t omx_defer_weight_sums(omx_ctx* ctx, uint32_t expected) {
  OMX_REQUIRE_CTX(ctx);
  const int32_t rc = omx_form_sums(ctx);
  if (rc != OMX_OK) return rc;
  ctx->sums_expected = expected;
  ctx->sums_wait = true;
  ctx->prepare_sums_wait = false;
  return OMX_OK;
}

int32_t omx_defer_prepare_sums(omx_ctx* ctx) {
  OMX_REQUIRE_CTX(ctx);
  ctx->prepare_sums_wait = ctx->sums_wait;
  return OMX_OK;
}

int32_t omx_form_weight_sums(omx_ctx* ctx, int32_t form) {
  OMX_REQUIRE_CTX(ctx);
  ctx->sums_wait = ctx->prepare_sums_wait = false;
  if (form) return omx_form_sums(ctx);
  ctx->sums.clear();
  ctx->sums_used = 0;
  return OMX_OK;
}

int32_t omx_rms_norm_forward(omx_ctx* ctx, const void* x, int32_t x_dtype, const void* w, void* y, int32_t y_dtype,
                             uint64_t rows, uint64_t dim, float eps) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "rms_norm_forward";
  if (!x || !w || !y) return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  if (!omx_valid_float_dtype(x_dtype) || !omx_valid_float_dtype(y_dtype))
    return omx_fail(ctx, OMX_DTYPE, "%s: dtype must be f32 or bf16", op);
  if (rows == 0 || dim == 0) return omx_fail(ctx, OMX_SHAPE, "%s: zero-sized axis", op);
  if (!(eps == eps) || eps == INFINITY || eps == -INFINITY) return omx_fail(ctx, OMX_NON_FINITE, "%s", op);
  return rms_forward_impl(ctx, op, F_RMS_FORWARD, x, x_dtype, w, y, y_dtype, rows, dim, eps);
}

int32_t omx_rms_norm_backward(omx_ctx* ctx, const void* x, int32_t x_dtype, const void* w, const void* gy,
                              int32_t gy_dtype, void* gx, int32_t gx_dtype, void* gw, uint64_t rows, uint64_t dim,
                              float eps) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "rms_norm_backward";
  if (!x || !w || !gy || !gx || !gw) return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  if (!omx_valid_float_dtype(x_dtype) || !omx_valid_float_dtype(gy_dtype) || !omx_valid_float_dtype(gx_dtype))
    return omx_fail(ctx, OMX_DTYPE, "%s: dtype must be f32 or bf16", op);
  if (rows == 0 || dim == 0) return omx_fail(ctx, OMX_SHAPE, "%s: zero-sized axis", op);
  if (!(eps == eps) || eps == INFINITY || eps == -INFINITY) return omx_fail(ctx, OMX_NON_FINITE, "%s", op);
  return rms_backward_impl(ctx, F_RMS_BACKWARD, x, x_dtype, w, gy, gy_dtype, gx, gx_dtype, gw, rows, dim, eps);
}

int32_t omx_rms_qk_norm_forward(omx_ctx* ctx, const void* q, const void* k, int32_t x_dtype, const void* q_weight,
                                const void* k_weight, void* q_out, void* k_out, int32_t y_dtype, uint64_t q_rows,
                                uint64_t k_rows, uint64_t dim, float eps) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "rms_qk_norm_forward";
  if (!q || !k || !q_weight || !k_weight || !q_out || !k_out)
    return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  if (!omx_valid_float_dtype(x_dtype) || !omx_valid_float_dtype(y_dtype))
    return omx_fail(ctx, OMX_DTYPE, "%s: dtype must be f32 or bf16", op);
  if (q_rows == 0 || k_rows == 0 || dim == 0) return omx_fail(ctx, OMX_SHAPE, "%s: zero-sized axis", op);
  if (!finite_host(eps)) return omx_fail(ctx, OMX_NON_FINITE, "%s", op);
  const uint64_t in = float_bytes(x_dtype) * dim, out = float_bytes(y_dtype) * dim;
  if (!omx_rms_vec_eligible(dim, {q, q_weight, q_out}) && !omx_rms_vec_eligible(dim, {k, k_weight, k_out}) &&
      no_overlap(q_out, q_rows * out, k, k_rows * in) && no_overlap(q_out, q_rows * out, k_weight, dim * 4) &&
      no_overlap(k_out, k_rows * out, q, q_rows * in) && no_overlap(k_out, k_rows * out, q_weight, dim * 4) &&
      no_overlap(q_out, q_rows * out, k_out, k_rows * out)) {
    RmsTensors t{};
    t.of[0] = {q, nullptr, static_cast<const float*>(q_weight), q_out, nullptr, q_rows, 0, omx_tag(ctx, F_RMS_QK_FORWARD)};
    t.of[1] = {k, nullptr, static_cast<const float*>(k_weight), k_out, nullptr, k_rows, 0, omx_tag(ctx, F_RMS_QK_FORWARD)};
    return launch_rms_fwd(ctx, t, 2, x_dtype, y_dtype, dim, eps);
  }
  int32_t rc = rms_forward_impl(ctx, op, F_RMS_QK_FORWARD, q, x_dtype, q_weight, q_out, y_dtype, q_rows, dim, eps);
  if (rc != OMX_OK) return rc;
  return rms_forward_impl(ctx, op, F_RMS_QK_FORWARD, k, x_dtype, k_weight, k_out, y_dtype, k_rows, dim, eps);
}

int32_t omx_rms_qk_norm_backward(omx_ctx* ctx, const void* q, const void* k, int32_t x_dtype, const void* q_weight,
                                 const void* k_weight, const void* grad_q, const void* grad_k, int32_t gy_dtype,
                                 void* gq, void* gk, int32_t gx_dtype, void* gq_weight, void* gk_weight,
                                 uint64_t q_rows, uint64_t k_rows, uint64_t dim, float eps) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "rms_qk_norm_backward";
  if (!q || !k || !q_weight || !k_weight || !grad_q || !grad_k || !gq || !gk || !gq_weight || !gk_weight)
    return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  if (!omx_valid_float_dtype(x_dtype) || !omx_valid_float_dtype(gy_dtype) || !omx_valid_float_dtype(gx_dtype))
    return omx_fail(ctx, OMX_DTYPE, "%s: dtype must be f32 or bf16", op);
  if (q_rows == 0 || k_rows == 0 || dim == 0) return omx_fail(ctx, OMX_SHAPE, "%s: zero-sized axis", op);
  if (!finite_host(eps)) return omx_fail(ctx, OMX_NON_FINITE, "%s", op);
  const uint64_t in = float_bytes(x_dtype) * dim, grad = float_bytes(gy_dtype) * dim, out = float_bytes(gx_dtype) * dim;
  bool together = !omx_rms_vec_eligible(dim, {q, q_weight, grad_q, gq, gq_weight}) && !omx_rms_vec_eligible(dim, {k, k_weight, grad_k, gk, gk_weight}) &&
                  no_overlap(gq, q_rows * out, gk, k_rows * out);
  struct Range {
    const void* at;
    uint64_t bytes;
  };
  const Range of_q[] = {{q, q_rows * in}, {q_weight, dim * 4}, {grad_q, q_rows * grad}, {gq_weight, dim * 4}};
  const Range of_k[] = {{k, k_rows * in}, {k_weight, dim * 4}, {grad_k, k_rows * grad}, {gk_weight, dim * 4}};
  for (const Range& r : of_k) together = together && no_overlap(gq, q_rows * out, r.at, r.bytes) && no_overlap(gq_weight, dim * 4, r.at, r.bytes);
  for (const Range& r : of_q) together = together && no_overlap(gk, k_rows * out, r.at, r.bytes) && no_overlap(gk_weight, dim * 4, r.at, r.bytes);
  if (together) {
    RmsTensors t{};
    t.of[0] = {q, grad_q, static_cast<const float*>(q_weight), gq, nullptr, q_rows, rms_rows_per_block(ctx, q_rows, dim), 0};
    t.of[1] = {k, grad_k, static_cast<const float*>(k_weight), gk, nullptr, k_rows, rms_rows_per_block(ctx, k_rows, dim), 0};
    const uint64_t blocks[2] = {rms_blocks(t.of[0]), rms_blocks(t.of[1])};
    const uint64_t q_bytes = (rms_partial_bytes(blocks[0], dim) + 255) / 256 * 256, bytes = q_bytes + rms_partial_bytes(blocks[1], dim);
    void* partial = omx_workspace_if_room(ctx, bytes);
    if (partial) {
      float* const weights[2] = {static_cast<float*>(gq_weight), static_cast<float*>(gk_weight)};
      bool wide = true;
      for (int i = 0; i < 2; ++i) {
        t.of[i].partial = reinterpret_cast<float*>(static_cast<char*>(partial) + i * q_bytes);
        t.of[i].tag = omx_tag(ctx, F_RMS_QK_BACKWARD);
        wide = wide && blocks[i] > 16 && blocks[i] <= OMX_COLUMN_SUM_WIDE_ROWS;
      }
      int32_t rc = launch_rms_bwd(ctx, t, 2, x_dtype, gy_dtype, gx_dtype, dim, eps);
      if (rc != OMX_OK) return rc;
      if (wide) {
        ColumnSumList list{};
        for (int i = 0; i < 2; ++i) list.of[i] = {t.of[i].partial, weights[i], t.of[i].tag, static_cast<int>(blocks[i]), static_cast<int>(dim)};
        omx_launch(ctx, column_sum_list_kernel, dim3(static_cast<unsigned>((dim + 63) / 64), 2), dim3(1024), 0, list, ctx->fault);
        OMX_LAUNCH_CHECK(ctx, "column_sum_list_kernel");
        return OMX_OK;
      }
      for (int i = 0; i < 2 && rc == OMX_OK; ++i)
        rc = omx_column_sum(ctx, t.of[i].partial, weights[i], blocks[i], dim, t.of[i].tag, t.of[i].partial + blocks[i] * dim);
      return rc;
    }
  }
  int32_t rc = rms_backward_impl(ctx, F_RMS_QK_BACKWARD, q, x_dtype, q_weight, grad_q, gy_dtype, gq, gx_dtype,
                                 gq_weight, q_rows, dim, eps);
  if (rc != OMX_OK) return rc;
  return rms_backward_impl(ctx, F_RMS_QK_BACKWARD, k, x_dtype, k_weight, grad_k, gy_dtype, gk, gx_dtype, gk_weight,
                           k_rows, dim, eps);
}

int32_t omx_embedding_forward(omx_ctx* ctx, const void* table, int32_t table_dtype, const void* ids, void* out,
                              int32_t out_dtype, uint64_t tokens, uint64_t vocab, uint64_t dim) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "embedding_forward";
  if (!table || !ids || !out) return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  if (!omx_valid_float_dtype(table_dtype) || !omx_valid_float_dtype(out_dtype))
    return omx_fail(ctx, OMX_DTYPE, "%s: dtype must be f32 or bf16", op);
  if (tokens == 0 || vocab == 0 || dim == 0) return omx_fail(ctx, OMX_SHAPE, "%s: zero-sized axis", op);
  if (dim > 0x7fffffffull) return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: dim does not fit in i32", op);
  unsigned long long tag = omx_tag(ctx, F_EMBEDDING_FORWARD);
  dim3 grid(static_cast<unsigned>((tokens + 3) / 4)), block(ROW_THREADS);
  const unsigned int* idp = static_cast<const unsigned int*>(ids);
#define EMB_FWD(TT, TO)                                                                                      \
  omx_launch(ctx, (embedding_fwd_kernel<TT, TO>), grid, block, 0, static_cast<const TT*>(table), \
                     idp, static_cast<TO*>(out), tokens, vocab, static_cast<int>(dim), ctx->fault, tag)
  if (table_dtype == OMX_F32 && out_dtype == OMX_F32) EMB_FWD(float, float);
  else if (table_dtype == OMX_F32) EMB_FWD(float, unsigned short);
  else if (out_dtype == OMX_F32) EMB_FWD(unsigned short, float);
  else EMB_FWD(unsigned short, unsigned short);
#undef EMB_FWD
  OMX_LAUNCH_CHECK(ctx, "embedding_fwd_kernel");
  return OMX_OK;
}

static int32_t embedding_backward_impl(omx_ctx* ctx, const void* ids, const void* grad, int32_t grad_dtype,
                                       void* table_grad, uint64_t tokens, uint64_t vocab, uint64_t dim, bool add) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = add ? "embedding_backward_accumulate" : "embedding_backward";
  if (!ids || !grad || !table_grad) return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  if (!omx_valid_float_dtype(grad_dtype)) return omx_fail(ctx, OMX_DTYPE, "%s: dtype must be f32 or bf16", op);
  if (tokens == 0 || vocab == 0 || dim == 0) return omx_fail(ctx, OMX_SHAPE, "%s: zero-sized axis", op);
  if (tokens > 0xfffffffeull || vocab > 0xfffffffeull || dim > 0x7fffffffull)
    return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: axis does not fit in u32", op);
  // Workspace: offsets[V+1], positions[N]; where one workgroup's LDS does not hold the counts also counts[V], cursor[V] and the
  // scan's totals.
  const bool small = tokens <= INDEX_TOKENS && vocab <= INDEX_VOCAB;
  const uint64_t scan_blocks = (vocab + 1023) / 1024;
  const uint64_t words = vocab + 1 + tokens + (small ? 0 : 2 * vocab + scan_blocks);
  void* ws = nullptr;
  int32_t rc = omx_workspace(ctx, words * 4, &ws);
  if (rc != OMX_OK) return rc;
  unsigned int* offsets = static_cast<unsigned int*>(ws);
  unsigned int* positions = offsets + vocab + 1;
  unsigned long long tag = omx_tag(ctx, F_EMBEDDING_BACKWARD);
  const unsigned int* idp = static_cast<const unsigned int*>(ids);
  // Bytes: every gradient row read once, every table row written once (rows no token names get
  // zeros); the adding form reads and writes at most one table row per token.
  const double table_rows = add ? 2.0 * static_cast<double>(tokens < vocab ? tokens : vocab) : static_cast<double>(vocab);
  OmxKernelTimer timer(ctx, OMX_K_EMBED_BWD,
                       static_cast<double>(dim) * (static_cast<double>(tokens) * (grad_dtype == OMX_BF16 ? 2.0 : 4.0) +
                                                   table_rows * 4.0));
  if (small) {
    const int lds = static_cast<int>((index_at(static_cast<unsigned int>(vocab)) + 1) * 4);
    if (lds > 64 * 1024)
      OMX_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(&index_ids_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    omx_launch_timed(ctx, index_ids_kernel, dim3(1), dim3(1024), lds, timer.start(), nullptr, idp, offsets, positions,
                     static_cast<unsigned int>(tokens), static_cast<unsigned int>(vocab), ctx->fault, tag);
    OMX_LAUNCH_CHECK(ctx, "index_ids_kernel");
  } else {
    unsigned int* counts = positions + tokens;
    unsigned int* cursor = counts + vocab;
    unsigned int* scan_totals = cursor + vocab;
    rc = omx_fill_zero(ctx, counts, vocab * 4);
    if (rc != OMX_OK) return rc;
    dim3 tgrid(static_cast<unsigned>((tokens + 255) / 256));
    omx_launch_timed(ctx, count_ids_kernel, tgrid, dim3(256), 0, timer.start(), nullptr, idp, counts, tokens, vocab,
                     ctx->fault, tag);
    OMX_LAUNCH_CHECK(ctx, "count_ids_kernel");
    if (scan_blocks > 4 && scan_blocks <= SCAN_MAX_BLOCKS) {
      const dim3 sgrid(static_cast<unsigned>(scan_blocks));
      omx_launch(ctx, scan_totals_kernel, sgrid, dim3(1024), 0, counts, scan_totals, vocab);
      OMX_LAUNCH_CHECK(ctx, "scan_totals_kernel");
      omx_launch(ctx, scan_blocks_kernel, sgrid, dim3(1024), 0, counts, scan_totals, offsets, cursor, vocab);
      OMX_LAUNCH_CHECK(ctx, "scan_blocks_kernel");
    } else {
      omx_launch(ctx, scan_counts_kernel, dim3(1), dim3(1024), 0, counts, offsets, cursor, vocab);
      OMX_LAUNCH_CHECK(ctx, "scan_counts_kernel");
    }
    omx_launch(ctx, fill_positions_kernel, tgrid, dim3(256), 0, idp, cursor, positions, tokens, vocab);
    OMX_LAUNCH_CHECK(ctx, "fill_positions_kernel");
  }
  const bool vec4 = dim % 4 == 0 && (reinterpret_cast<uintptr_t>(grad) & 15u) == 0 &&
                    (reinterpret_cast<uintptr_t>(table_grad) & 15u) == 0 && (grad_dtype == OMX_F32 || dim % 8 == 0);
  // A wave per row; where rows are few, per row and 256 columns.
  const uint64_t columns = vec4 ? 256 : 512;
  dim3 vgrid(static_cast<unsigned>((vocab + 3) / 4), vocab <= 4096 ? static_cast<unsigned>(std::min<uint64_t>((dim + columns - 1) / columns, 64)) : 1u);
#define EMB_BWD(TG_, V_)                                                                                         \
  do {                                                                                                          \
    if (add)                                                                                                    \
      omx_launch_timed(ctx, embedding_bwd_kernel<TG_, V_, true>, vgrid, dim3(ROW_THREADS), 0, nullptr,          \
                       timer.stop(), offsets, positions, static_cast<const TG_*>(grad),                            \
                       static_cast<float*>(table_grad), vocab, static_cast<int>(dim), tokens, ctx->fault, tag); \
    else                                                                                                        \
      omx_launch_timed(ctx, embedding_bwd_kernel<TG_, V_, false>, vgrid, dim3(ROW_THREADS), 0, nullptr,         \
                       timer.stop(), offsets, positions, static_cast<const TG_*>(grad),                            \
                       static_cast<float*>(table_grad), vocab, static_cast<int>(dim), tokens, ctx->fault, tag); \
  } while (0)
  if (grad_dtype == OMX_F32) {
    if (vec4) EMB_BWD(float, 4);
    else EMB_BWD(float, 1);
  } else {
    if (vec4) EMB_BWD(unsigned short, 4);
    else EMB_BWD(unsigned short, 1);
  }
#undef EMB_BWD
  OMX_LAUNCH_CHECK(ctx, "embedding_bwd_kernel");
  return OMX_OK;
}

int32_t omx_embedding_backward(omx_ctx* ctx, const void* ids, const void* grad, int32_t grad_dtype, void* table_grad,
                               uint64_t tokens, uint64_t vocab, uint64_t dim) {
  return embedding_backward_impl(ctx, ids, grad, grad_dtype, table_grad, tokens, vocab, dim, false);
}

int32_t omx_embedding_backward_accumulate(omx_ctx* ctx, const void* ids, const void* grad, int32_t grad_dtype,
                                          void* table_grad, uint64_t tokens, uint64_t vocab, uint64_t dim) {
  return embedding_backward_impl(ctx, ids, grad, grad_dtype, table_grad, tokens, vocab, dim, true);
}

int32_t omx_argmax_rows(omx_ctx* ctx, const void* x, uint64_t rows, uint64_t cols, void* out) {
  OMX_REQUIRE_CTX(ctx);
  if (!x || !out) return omx_fail(ctx, OMX_PLACEMENT, "argmax_rows: null device pointer");
  if (rows == 0 || cols == 0) return omx_fail(ctx, OMX_SHAPE, "argmax_rows: zero-sized axis");
  if (cols > 0xfffffffeull) return omx_fail(ctx, OMX_OUT_OF_RANGE, "argmax_rows: cols does not fit in u32");
  if (rows > 0x7fffffffull) return omx_fail(ctx, OMX_OUT_OF_RANGE, "argmax_rows: rows does not fit in i32");
  uint2* parts = nullptr;
  auto launch = [&](auto kernel, int threads, int slices) {
    omx_launch(ctx, kernel, dim3(static_cast<unsigned>(rows), slices), dim3(threads), 0, static_cast<const float*>(x),
                       static_cast<unsigned int>(cols), static_cast<unsigned int*>(out), parts, ctx->fault, omx_tag(ctx, F_ARGMAX));
  };
  // A quarter of a thousand columns feeds a wave; from four thousand on a row has work for sixteen, from sixteen thousand on, where
  // rows leave compute units empty, for as many workgroups (without the scratch for their results, one workgroup a row).
  if (cols >= 16384 && rows * ARGMAX_SLICES <= 256)
    parts = static_cast<uint2*>(omx_workspace_if_room(ctx, rows * ARGMAX_SLICES * sizeof(uint2)));
  if (parts) {
    launch(&argmax_rows_kernel<256, ARGMAX_SLICES>, 256, ARGMAX_SLICES);
    OMX_LAUNCH_CHECK(ctx, "argmax_rows_kernel");
    omx_launch(ctx, argmax_meet_kernel, dim3(static_cast<unsigned>(rows)), dim3(64), 0, static_cast<const uint2*>(parts),
               static_cast<unsigned int*>(out));
    OMX_LAUNCH_CHECK(ctx, "argmax_meet_kernel");
    return OMX_OK;
  }
  if (cols <= 256) launch(&argmax_rows_kernel<64, 1>, 64, 1);
  else if (cols <= 4096) launch(&argmax_rows_kernel<256, 1>, 256, 1);
  else launch(&argmax_rows_kernel<1024, 1>, 1024, 1);
  OMX_LAUNCH_CHECK(ctx, "argmax_rows_kernel");
  return OMX_OK;
}

int32_t omx_topk_rows(omx_ctx* ctx, const void* x, uint64_t rows, uint64_t cols, uint64_t k, void* values,
                      void* ids) {
  OMX_REQUIRE_CTX(ctx);
  if (!x || !values || !ids) return omx_fail(ctx, OMX_PLACEMENT, "topk_rows: null device pointer");
  if (rows == 0 || cols == 0) return omx_fail(ctx, OMX_SHAPE, "topk_rows: zero-sized axis");
  if (k == 0 || k > cols) return omx_fail(ctx, OMX_SHAPE, "topk_rows: k %llu outside 1..=%llu", (unsigned long long)k,
                                          (unsigned long long)cols);
  if (cols > 0xfffffffeull) return omx_fail(ctx, OMX_OUT_OF_RANGE, "topk_rows: cols does not fit in u32");
  omx_launch(ctx, topk_rows_kernel, dim3(static_cast<unsigned>((rows + 3) / 4)), dim3(ROW_THREADS), 0,
                     static_cast<const float*>(x), rows, static_cast<unsigned int>(cols), static_cast<unsigned int>(k),
                     static_cast<float*>(values), static_cast<unsigned int*>(ids), ctx->fault, omx_tag(ctx, F_TOPK));
  OMX_LAUNCH_CHECK(ctx, "topk_rows_kernel");
  return OMX_OK;
}

}  // extern "C"
