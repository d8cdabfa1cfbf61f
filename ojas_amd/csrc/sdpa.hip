// Causal scaled-dot-product attention, forward and backward.
//
// Reference semantics: ojas-cpu/src/attn.rs:47-124,176-227 (forward),
// :437-597 (backward from the saved output and log-sum-exp); trait
// ojas-core/src/backend.rs:1729-1792. Layout [B, H, T, D]; query t sees keys
// max(0, t + 1 - window) ..= t; query head h reads KV head h / (H / Hkv);
// scale = 1 / sqrt(D) formed in f32 (backend.rs:159). lse = max + ln(sum).
// Backward: P = e^(S - lse), Dr = dO . O, dS = scale * P * (dP - Dr);
// dQ = dS K, dK = dS^T Q, dV = P^T dO, with the query heads of one KV head
// summed in ascending head order.
//
// Three families of kernels:
//   * row kernels (this file): one wavefront per query row (or per key row in
//     the dK/dV pass), any head_dim up to 256, f32 arithmetic. They serve every
//     head_dim and mix of storage types the other two do not cover.
//   * f32 matrix kernels (sdpa_mfma32.hip): f32 tensors at head_dim 16 / 32 / 64 / 128.
//   * flash kernels (flash_sdpa.hip): bf16 MFMA tiles for head_dim 64 / 128.
// None forms a T x T matrix; no atomics are used, so results do not depend
// on scheduling.
#include <algorithm>

#include "omx_common.h"
#include "sdpa_mfma32.h"

int32_t omx_flash_sdpa_forward(omx_ctx* ctx, const void* q, const void* k, const void* v, void* out,
                               int32_t out_dtype, void* out_residual, float* lse, uint64_t batch, uint64_t heads,
                               uint64_t kv_heads, uint64_t time, uint64_t dim, uint64_t window, float scale,
                               unsigned long long tag, const long* strides);
int32_t omx_flash_sdpa_backward(omx_ctx* ctx, const void* q, const void* k, const void* v, const void* out,
                                const void* out_residual, const float* lse, const void* gy, void* gq, void* gk,
                                void* gv, int32_t grad_dtype,
                                uint64_t batch, uint64_t heads, uint64_t kv_heads, uint64_t time, uint64_t dim,
                                uint64_t window, float scale, unsigned long long tag, const long* strides);
bool omx_flash_sdpa_supports(uint64_t dim, int32_t operand_dtype);

namespace {

constexpr int SD_THREADS = 256;  // 4 waves: 4 rows per block
constexpr int MAXD = 256;

struct SdpaShape {
  int batch, heads, kv_heads, time, dim, window, rep;
  float scale;
  // Element strides of a batch, a head and a row: q (and gq), k and v (and gk, gv), out (and gy). lse is [batch, heads, time].
  long q_b, q_h, q_t, k_b, k_h, k_t, o_b, o_h, o_t;
};

__device__ __forceinline__ int first_key(const SdpaShape& s, int t) {
  return s.window > 0 ? max(0, t + 1 - s.window) : 0;
}
__device__ __forceinline__ int last_query(const SdpaShape& s, int j) {
  // Queries that see key j: j ..= min(T-1, j + window - 1).
  return s.window > 0 ? min(s.time - 1, j + s.window - 1) : s.time - 1;
}

// One wave per query row. Lane l scores keys j0 + l of each 64-key block
// (dot over D from LDS-broadcast q), the block is folded into the running
// softmax, and lanes then switch to owning output dims for the P.V update.
template <typename TI, typename TO>
__global__ __launch_bounds__(SD_THREADS) void sdpa_fwd_rows_kernel(const TI* __restrict__ q, const TI* __restrict__ k,
                                                                   const TI* __restrict__ v, TO* __restrict__ out,
                                                                   float* __restrict__ lse, SdpaShape s,
                                                                   OmxFaultWord* fault, unsigned long long tag) {
  __shared__ float q_lds[4][MAXD];
  __shared__ float p_lds[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long row = static_cast<long>(blockIdx.x) * 4 + wave;  // (b*H + h)*T + t
  const long total = static_cast<long>(s.batch) * s.heads * s.time;
  if (row >= total) return;
  const int t = static_cast<int>(row % s.time);
  const long plane = row / s.time;
  const int h = static_cast<int>(plane % s.heads), b = static_cast<int>(plane / s.heads);
  const long kv_plane = b * s.k_b + h / s.rep * s.k_h;
  const TI* qr = q + b * s.q_b + h * s.q_h + t * s.q_t;
  const TI* kh = k + kv_plane;
  const TI* vh = v + kv_plane;
  const int D = s.dim;
  for (int d = lane; d < D; d += 64) q_lds[wave][d] = dev_load<TI>(qr, d);
  constexpr int ND = MAXD / 64;
  float acc[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i) acc[i] = 0.0f;
  float run_max = -INFINITY, run_sum = 0.0f;
  bool bad = false;
  const int j_begin = first_key(s, t), j_end = t + 1;
  for (int j0 = j_begin; j0 < j_end; j0 += 64) {
    const int j = j0 + lane;
    float sc = -INFINITY;
    if (j < j_end) {
      const TI* kr = kh + j * s.k_t;
      float dot = 0.0f;
      for (int d = 0; d < D; ++d) dot += q_lds[wave][d] * dev_load<TI>(kr, d);
      sc = dot * s.scale;
      bad |= !dev_finite(sc);
    }
    float blk_max = wave_max(sc);
    float new_max = fmaxf(run_max, blk_max);
    float p = j < j_end ? expf(sc - new_max) : 0.0f;
    float blk_sum = wave_sum(p);
    float rescale = expf(run_max - new_max);  // 0 on the first block (run_max = -inf)
    run_sum = run_sum * rescale + blk_sum;
    run_max = new_max;
    p_lds[wave][lane] = p;
    // Same-wave LDS traffic: the wave executes in lockstep, a fence orders it.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int nk = min(64, j_end - j0);
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      const int d = i * 64 + lane;
      if (d < D) {
        float a = acc[i] * rescale;
        for (int jj = 0; jj < nk; ++jj) a += p_lds[wave][jj] * dev_load<TI>(vh, (j0 + jj) * s.k_t + d);
        acc[i] = a;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  bad |= !(dev_finite(run_sum) && run_sum > 0.0f);
  const float inv = 1.0f / run_sum;
  TO* orow = out + b * s.o_b + h * s.o_h + t * s.o_t;
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    const int d = i * 64 + lane;
    if (d < D) {
      float o = acc[i] * inv;
      bad |= !dev_finite(o);
      dev_store<TO>(orow, d, o);
    }
  }
  if (lane == 0) lse[row] = run_max + logf(run_sum);
  if (bad) dev_raise_fault(fault, tag);
}

// Dr[row] = dO[row] . O[row] (f32), one wave per row.
template <typename TOUT, typename TGY>
__global__ __launch_bounds__(SD_THREADS) void sdpa_delta_kernel(const TOUT* __restrict__ out,
                                                                const TGY* __restrict__ gy,
                                                                float* __restrict__ delta, SdpaShape s) {
  const int lane = threadIdx.x & 63;
  const long row = static_cast<long>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= static_cast<long>(s.batch) * s.heads * s.time) return;
  const long plane = row / s.time;
  const long at = plane / s.heads * s.o_b + plane % s.heads * s.o_h + row % s.time * s.o_t;
  float acc = 0.0f;
  for (int d = lane; d < s.dim; d += 64) acc += dev_load<TGY>(gy, at + d) * dev_load<TOUT>(out, at + d);
  acc = wave_sum(acc);
  if (lane == 0) delta[row] = acc;
}

// An f32 attention output as the pair the bf16 MFMA backward reads: hi = bf16(x) and
// residual = bf16(x - hi), so hi + residual carries x to 2^-17.
__global__ void sdpa_split_output_kernel(const float* __restrict__ x, unsigned short* __restrict__ hi,
                                         unsigned short* __restrict__ residual, long n) {
  for (long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<long>(gridDim.x) * blockDim.x) {
    const float v = x[i];
    const unsigned short h = dev_f32_to_bf16_bits(v);
    hi[i] = h;
    residual[i] = dev_f32_to_bf16_bits(v - dev_bf16_bits_to_f32(h));
  }
}

// dQ: one wave per query row, the forward's structure with dS in place of P.
template <typename TI, typename TO>
__global__ __launch_bounds__(SD_THREADS) void sdpa_bwd_dq_rows_kernel(
    const TI* __restrict__ q, const TI* __restrict__ k, const TI* __restrict__ v, const float* __restrict__ lse,
    const float* __restrict__ delta, const TI* __restrict__ gy, TO* __restrict__ gq, SdpaShape s, OmxFaultWord* fault,
    unsigned long long tag) {
  __shared__ float q_lds[4][MAXD];
  __shared__ float g_lds[4][MAXD];
  __shared__ float c_lds[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long row = static_cast<long>(blockIdx.x) * 4 + wave;
  const long total = static_cast<long>(s.batch) * s.heads * s.time;
  if (row >= total) return;
  const int t = static_cast<int>(row % s.time);
  const long plane = row / s.time;
  const int h = static_cast<int>(plane % s.heads), b = static_cast<int>(plane / s.heads);
  const long kv_plane = b * s.k_b + h / s.rep * s.k_h, q_row = b * s.q_b + h * s.q_h + t * s.q_t;
  const long o_row = b * s.o_b + h * s.o_h + t * s.o_t;
  const TI* kh = k + kv_plane;
  const TI* vh = v + kv_plane;
  const int D = s.dim;
  for (int d = lane; d < D; d += 64) {
    q_lds[wave][d] = dev_load<TI>(q, q_row + d);
    g_lds[wave][d] = dev_load<TI>(gy, o_row + d);
  }
  const float row_lse = lse[row], dr = delta[row];
  bool bad = !(dev_finite(row_lse) && dev_finite(dr));
  constexpr int ND = MAXD / 64;
  float acc[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i) acc[i] = 0.0f;
  const int j_begin = first_key(s, t), j_end = t + 1;
  for (int j0 = j_begin; j0 < j_end; j0 += 64) {
    const int j = j0 + lane;
    float coef = 0.0f;
    if (j < j_end) {
      const TI* kr = kh + j * s.k_t;
      const TI* vr = vh + j * s.k_t;
      float dot = 0.0f, dp = 0.0f;
      for (int d = 0; d < D; ++d) {
        dot += q_lds[wave][d] * dev_load<TI>(kr, d);
        dp += g_lds[wave][d] * dev_load<TI>(vr, d);
      }
      float sc = dot * s.scale;
      float p = expf(sc - row_lse);
      bad |= !(dev_finite(sc) && dev_finite(p));
      coef = s.scale * (p * (dp - dr));
    }
    c_lds[wave][lane] = coef;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int nk = min(64, j_end - j0);
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      const int d = i * 64 + lane;
      if (d < D) {
        float a = acc[i];
        for (int jj = 0; jj < nk; ++jj) a += c_lds[wave][jj] * dev_load<TI>(kh, (j0 + jj) * s.k_t + d);
        acc[i] = a;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    const int d = i * 64 + lane;
    if (d < D) {
      bad |= !dev_finite(acc[i]);
      dev_store<TO>(gq, q_row + d, acc[i]);
    }
  }
  if (bad) dev_raise_fault(fault, tag);
}

// dK, dV: one wave per key row of a KV head; walks the query heads of the
// group in ascending order and, within a head, queries in ascending order.
template <typename TI, typename TO>
__global__ __launch_bounds__(SD_THREADS) void sdpa_bwd_dkv_rows_kernel(
    const TI* __restrict__ q, const TI* __restrict__ k, const TI* __restrict__ v, const float* __restrict__ lse,
    const float* __restrict__ delta, const TI* __restrict__ gy, TO* __restrict__ gk, TO* __restrict__ gv, SdpaShape s,
    OmxFaultWord* fault, unsigned long long tag) {
  __shared__ float k_lds[4][MAXD];
  __shared__ float v_lds[4][MAXD];
  __shared__ float c_lds[4][64];
  __shared__ float p_lds[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long row = static_cast<long>(blockIdx.x) * 4 + wave;  // (b*Hkv + g)*T + j
  const long total = static_cast<long>(s.batch) * s.kv_heads * s.time;
  if (row >= total) return;
  const int j = static_cast<int>(row % s.time);
  const long kv_plane = row / s.time;
  const int g = static_cast<int>(kv_plane % s.kv_heads), b = static_cast<int>(kv_plane / s.kv_heads);
  const int D = s.dim;
  const long k_row = b * s.k_b + g * s.k_h + j * s.k_t;
  for (int d = lane; d < D; d += 64) {
    k_lds[wave][d] = dev_load<TI>(k, k_row + d);
    v_lds[wave][d] = dev_load<TI>(v, k_row + d);
  }
  constexpr int ND = MAXD / 64;
  float acck[ND], accv[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i) acck[i] = accv[i] = 0.0f;
  bool bad = false;
  const int t_end = last_query(s, j) + 1;
  for (int r = 0; r < s.rep; ++r) {
    const long head = static_cast<long>(g) * s.rep + r, q_plane = static_cast<long>(b) * s.heads + head;
    const TI* qh = q + b * s.q_b + head * s.q_h;
    const TI* gh = gy + b * s.o_b + head * s.o_h;
    const float* lse_h = lse + q_plane * s.time;
    const float* del_h = delta + q_plane * s.time;
    for (int t0 = j; t0 < t_end; t0 += 64) {
      const int t = t0 + lane;
      float coef = 0.0f, p = 0.0f;
      if (t < t_end) {
        const TI* qr = qh + t * s.q_t;
        const TI* gr = gh + t * s.o_t;
        float dot = 0.0f, dp = 0.0f;
        for (int d = 0; d < D; ++d) {
          dot += dev_load<TI>(qr, d) * k_lds[wave][d];
          dp += dev_load<TI>(gr, d) * v_lds[wave][d];
        }
        float sc = dot * s.scale;
        p = expf(sc - lse_h[t]);
        bad |= !(dev_finite(sc) && dev_finite(p));
        coef = s.scale * (p * (dp - del_h[t]));
      }
      c_lds[wave][lane] = coef;
      p_lds[wave][lane] = p;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const int nq = min(64, t_end - t0);
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        const int d = i * 64 + lane;
        if (d < D) {
          float ak = acck[i], av = accv[i];
          for (int tt = 0; tt < nq; ++tt) {
            ak += c_lds[wave][tt] * dev_load<TI>(qh, (t0 + tt) * s.q_t + d);
            av += p_lds[wave][tt] * dev_load<TI>(gh, (t0 + tt) * s.o_t + d);
          }
          acck[i] = ak;
          accv[i] = av;
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    const int d = i * 64 + lane;
    if (d < D) {
      bad |= !(dev_finite(acck[i]) && dev_finite(accv[i]));
      dev_store<TO>(gk, k_row + d, acck[i]);
      dev_store<TO>(gv, k_row + d, accv[i]);
    }
  }
  if (bad) dev_raise_fault(fault, tag);
}

int32_t check_shape(omx_ctx* ctx, const char* op, uint64_t batch, uint64_t heads, uint64_t kv_heads, uint64_t time,
                    uint64_t dim, uint64_t window, SdpaShape* s) {
  if (batch == 0 || heads == 0 || kv_heads == 0 || time == 0 || dim == 0)
    return omx_fail(ctx, OMX_SHAPE, "%s: zero-sized axis", op);
  if (kv_heads > heads || heads % kv_heads != 0)
    return omx_fail(ctx, OMX_SHAPE, "%s: heads %llu is not a multiple of kv heads %llu", op,
                    (unsigned long long)heads, (unsigned long long)kv_heads);
  if (dim > MAXD) return omx_fail(ctx, OMX_UNSUPPORTED_HEAD_DIM, "head_dim %llu limit %d", (unsigned long long)dim, MAXD);
  if (batch * heads * time > 0x7fffffffull || time > 0x3fffffffull)
    return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: B*H*T does not fit in i32", op);
  s->batch = static_cast<int>(batch);
  s->heads = static_cast<int>(heads);
  s->kv_heads = static_cast<int>(kv_heads);
  s->time = static_cast<int>(time);
  s->dim = static_cast<int>(dim);
  // A window of at least T is every earlier key (attn.rs:745).
  s->window = (window == 0 || window >= time) ? 0 : static_cast<int>(window);
  s->rep = static_cast<int>(heads / kv_heads);
  s->scale = 1.0f / sqrtf(static_cast<float>(static_cast<uint32_t>(dim)));
  const long plane = static_cast<long>(time) * s->dim;  // contiguous [B, H, T, D]
  s->q_t = s->k_t = s->o_t = s->dim;
  s->q_h = s->k_h = s->o_h = plane;
  s->q_b = s->o_b = plane * s->heads;
  s->k_b = plane * s->kv_heads;
  return OMX_OK;
}

// The f32 matrix kernels' arguments.
Sdpa32Args sdpa32_args(omx_ctx* ctx, const void* q, const void* k, const void* v, const SdpaShape& s, unsigned long long tag) {
  Sdpa32Args a{};
  a.q = static_cast<const float*>(q);
  a.k = k;
  a.v = v;
  a.q_b = s.q_b; a.q_h = s.q_h; a.q_t = s.q_t;
  a.k_b = s.k_b; a.k_h = s.k_h; a.k_t = s.k_t;
  a.o_b = s.o_b; a.o_h = s.o_h; a.o_t = s.o_t;
  a.kv_heads = s.kv_heads;
  a.rep = s.rep;
  a.tq = a.tk = a.capacity = s.time;
  a.window = s.window;
  a.scale = s.scale;
  a.fault = ctx->fault;
  a.tag = tag;
  return a;
}

// A wave per row: any head dim up to 256 and any number of planes.
template <typename TI, typename TO>
int32_t rows_forward(omx_ctx* ctx, const void* q, const void* k, const void* v, void* out, void* lse, const SdpaShape& s,
                     unsigned long long tag) {
  const long rows = static_cast<long>(s.batch) * s.heads * s.time;
  omx_launch(ctx, (sdpa_fwd_rows_kernel<TI, TO>), dim3(static_cast<unsigned>((rows + 3) / 4)), dim3(SD_THREADS), 0,
             static_cast<const TI*>(q), static_cast<const TI*>(k), static_cast<const TI*>(v), static_cast<TO*>(out),
             static_cast<float*>(lse), s, ctx->fault, tag);
  OMX_LAUNCH_CHECK(ctx, "sdpa_fwd_rows_kernel");
  return OMX_OK;
}
template <typename TOUT, typename TGY>
int32_t rows_delta(omx_ctx* ctx, const void* out, const void* gy, float* delta, const SdpaShape& s) {
  const long rows = static_cast<long>(s.batch) * s.heads * s.time;
  omx_launch(ctx, (sdpa_delta_kernel<TOUT, TGY>), dim3(static_cast<unsigned>((rows + 3) / 4)), dim3(SD_THREADS), 0,
             static_cast<const TOUT*>(out), static_cast<const TGY*>(gy), delta, s);
  OMX_LAUNCH_CHECK(ctx, "sdpa_delta_kernel");
  return OMX_OK;
}
template <typename TI, typename TO>
int32_t rows_backward(omx_ctx* ctx, const void* q, const void* k, const void* v, const float* lse, const float* delta, const void* gy,
                      void* gq, void* gk, void* gv, const SdpaShape& s, unsigned long long tag) {
  const long rows = static_cast<long>(s.batch) * s.heads * s.time, kv_rows = static_cast<long>(s.batch) * s.kv_heads * s.time;
  const TI *tq = static_cast<const TI*>(q), *tk = static_cast<const TI*>(k), *tv = static_cast<const TI*>(v);
  const TI* tg = static_cast<const TI*>(gy);
  omx_launch(ctx, (sdpa_bwd_dq_rows_kernel<TI, TO>), dim3(static_cast<unsigned>((rows + 3) / 4)), dim3(SD_THREADS), 0, tq, tk, tv, lse,
             delta, tg, static_cast<TO*>(gq), s, ctx->fault, tag);
  omx_launch(ctx, (sdpa_bwd_dkv_rows_kernel<TI, TO>), dim3(static_cast<unsigned>((kv_rows + 3) / 4)), dim3(SD_THREADS), 0, tq, tk, tv,
             lse, delta, tg, static_cast<TO*>(gk), static_cast<TO*>(gv), s, ctx->fault, tag);
  OMX_LAUNCH_CHECK(ctx, "sdpa backward row kernels");
  return OMX_OK;
}

}  // namespace

extern "C" {

int32_t omx_causal_sdpa_forward(omx_ctx* ctx, const void* q, const void* k, const void* v, int32_t operand_dtype,
                                void* out, int32_t out_dtype, void* lse, uint64_t batch, uint64_t heads,
                                uint64_t kv_heads, uint64_t time, uint64_t head_dim, uint64_t window) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "causal_sdpa_forward";
  if (!q || !k || !v || !out || !lse) return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  if (!omx_valid_float_dtype(operand_dtype) || !omx_valid_float_dtype(out_dtype))
    return omx_fail(ctx, OMX_DTYPE, "%s: dtype must be f32 or bf16", op);
  SdpaShape s;
  int32_t rc = check_shape(ctx, op, batch, heads, kv_heads, time, head_dim, window, &s);
  if (rc != OMX_OK) return rc;
  unsigned long long tag = omx_tag(ctx, F_SDPA_FORWARD);
  if (omx_flash_sdpa_supports(head_dim, operand_dtype))
    return omx_flash_sdpa_forward(ctx, q, k, v, out, out_dtype, nullptr, static_cast<float*>(lse), batch, heads,
                                  kv_heads, time, head_dim, s.window, s.scale, tag, nullptr);
  if (ctx->sdpa_tiled && operand_dtype == OMX_F32 && out_dtype == OMX_F32 &&
      omx_sdpa32_supports(head_dim, batch * kv_heads, {q, k, v, out}, {})) {
    Sdpa32Args a = sdpa32_args(ctx, q, k, v, s, tag);
    a.out = static_cast<float*>(out);
    a.lse = static_cast<float*>(lse);
    return omx_sdpa32_forward(ctx, a, s.batch, s.dim, false);
  }
  const auto rows = operand_dtype == OMX_F32 ? (out_dtype == OMX_F32 ? &rows_forward<float, float> : &rows_forward<float, unsigned short>)
                    : out_dtype == OMX_F32   ? &rows_forward<unsigned short, float>
                                             : &rows_forward<unsigned short, unsigned short>;
  return rows(ctx, q, k, v, out, lse, s, tag);
}

int32_t omx_causal_sdpa_backward(omx_ctx* ctx, const void* q, const void* k, const void* v, const void* out,
                                 const void* lse, const void* gy, int32_t operand_dtype, int32_t out_dtype,
                                 int32_t gy_dtype, void* gq, void* gk, void* gv, int32_t grad_dtype, uint64_t batch,
                                 uint64_t heads, uint64_t kv_heads, uint64_t time, uint64_t head_dim,
                                 uint64_t window) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "causal_sdpa_backward";
  if (!q || !k || !v || !out || !lse || !gy || !gq || !gk || !gv)
    return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  if (!omx_valid_float_dtype(operand_dtype) || !omx_valid_float_dtype(grad_dtype) ||
      !omx_valid_float_dtype(out_dtype) || !omx_valid_float_dtype(gy_dtype))
    return omx_fail(ctx, OMX_DTYPE, "%s: dtype must be f32 or bf16", op);
  SdpaShape s;
  int32_t rc = check_shape(ctx, op, batch, heads, kv_heads, time, head_dim, window, &s);
  if (rc != OMX_OK) return rc;
  unsigned long long tag = omx_tag(ctx, F_SDPA_BACKWARD);
  const long rows = static_cast<long>(batch) * heads * time;
  const uint64_t n = static_cast<uint64_t>(rows) * head_dim;
  if (omx_flash_sdpa_supports(head_dim, operand_dtype)) {
    // The MFMA kernels read bf16: an f32 output goes in as bf16 + rounding residual (nothing of it
    // is lost to the row term dO . O), an f32 grad_output rounded to bf16.
    const void* out16 = out;
    const void* residual = nullptr;
    const void* gy16 = gy;
    if (out_dtype == OMX_F32 || gy_dtype == OMX_F32) {
      void* ws = nullptr;
      rc = omx_workspace(ctx, 3 * n * 2, &ws, 1);
      if (rc != OMX_OK) return rc;
      unsigned short* base = static_cast<unsigned short*>(ws);
      if (out_dtype == OMX_F32) {
        const unsigned blocks = static_cast<unsigned>(std::min<uint64_t>((n + 255) / 256, 65536));
        omx_launch(ctx, sdpa_split_output_kernel, dim3(blocks), dim3(256), 0,
                           static_cast<const float*>(out), base, base + n, static_cast<long>(n));
        OMX_LAUNCH_CHECK(ctx, "sdpa_split_output_kernel");
        out16 = base;
        residual = base + n;
      }
      if (gy_dtype == OMX_F32) {
        rc = omx_convert(ctx, gy, OMX_F32, base + 2 * n, OMX_BF16, n);
        if (rc != OMX_OK) return rc;
        gy16 = base + 2 * n;
      }
    }
    return omx_flash_sdpa_backward(ctx, q, k, v, out16, residual, static_cast<const float*>(lse), gy16, gq, gk, gv,
                                   grad_dtype, batch, heads, kv_heads, time, head_dim, s.window, s.scale, tag, nullptr);
  }
  void* ws = nullptr;
  rc = omx_workspace(ctx, rows * sizeof(float), &ws);
  if (rc != OMX_OK) return rc;
  float* delta = static_cast<float*>(ws);
  const float* lsef = static_cast<const float*>(lse);
  const bool matrix = ctx->sdpa_tiled && operand_dtype == OMX_F32 && grad_dtype == OMX_F32 && gy_dtype == OMX_F32 &&
                      out_dtype == OMX_F32 && omx_sdpa32_supports(head_dim, batch * kv_heads, {q, k, v, out, gy, gq, gk, gv}, {});
  if (matrix) {
    Sdpa32Args a = sdpa32_args(ctx, q, k, v, s, tag);
    a.out = const_cast<float*>(static_cast<const float*>(out));  // read only: the dQ pass takes the row term from it
    a.lse = const_cast<float*>(lsef);
    a.gy = static_cast<const float*>(gy);
    a.gq = static_cast<float*>(gq);
    a.gk = static_cast<float*>(gk);
    a.gv = static_cast<float*>(gv);
    a.delta = delta;
    return omx_sdpa32_backward(ctx, a, s.batch, s.dim);
  }
  // The row term reads out and grad_output as they are stored; the two passes read grad_output in
  // the operands' storage type.
  const auto row_term = out_dtype == OMX_F32 ? (gy_dtype == OMX_F32 ? &rows_delta<float, float> : &rows_delta<float, unsigned short>)
                        : gy_dtype == OMX_F32 ? &rows_delta<unsigned short, float>
                                              : &rows_delta<unsigned short, unsigned short>;
  rc = row_term(ctx, out, gy, delta, s);
  if (rc != OMX_OK) return rc;
  if (gy_dtype != operand_dtype) {
    void* conv = nullptr;
    rc = omx_workspace(ctx, n * omx_dtype_size(operand_dtype), &conv, 1);
    if (rc != OMX_OK) return rc;
    rc = omx_convert(ctx, gy, gy_dtype, conv, operand_dtype, n);
    if (rc != OMX_OK) return rc;
    gy = conv;
  }
  const auto passes = operand_dtype == OMX_F32 ? (grad_dtype == OMX_F32 ? &rows_backward<float, float> : &rows_backward<float, unsigned short>)
                      : grad_dtype == OMX_F32  ? &rows_backward<unsigned short, float>
                                               : &rows_backward<unsigned short, unsigned short>;
  return passes(ctx, q, k, v, lsef, delta, gy, gq, gk, gv, s, tag);
}

int32_t omx_causal_sdpa_backward_recompute(omx_ctx* ctx, const void* q, const void* k, const void* v, const void* gy,
                                           int32_t operand_dtype, int32_t gy_dtype, void* gq, void* gk, void* gv,
                                           int32_t grad_dtype, uint64_t batch, uint64_t heads, uint64_t kv_heads,
                                           uint64_t time, uint64_t head_dim, uint64_t window) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "causal_sdpa_backward_recompute";
  // The gradient's arguments are checked before the forward runs (backend.rs:1781-1792).
  if (!q || !k || !v || !gy || !gq || !gk || !gv) return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  if (!omx_valid_float_dtype(operand_dtype) || !omx_valid_float_dtype(grad_dtype) || !omx_valid_float_dtype(gy_dtype))
    return omx_fail(ctx, OMX_DTYPE, "%s: dtype must be f32 or bf16", op);
  SdpaShape s;
  int32_t rc = check_shape(ctx, op, batch, heads, kv_heads, time, head_dim, window, &s);
  if (rc != OMX_OK) return rc;
  // The forward's output stays f32 (the unrounded O the row term needs) in the library's own scratch.
  const uint64_t rows = batch * heads * time;
  const uint64_t out_bytes = (rows * head_dim * 4 + 255) & ~255ull;
  void* ws = nullptr;
  rc = omx_workspace(ctx, out_bytes + rows * 4, &ws, 2);
  if (rc != OMX_OK) return rc;
  void* out = ws;
  void* lse = static_cast<char*>(ws) + out_bytes;
  rc = omx_causal_sdpa_forward(ctx, q, k, v, operand_dtype, out, OMX_F32, lse, batch, heads, kv_heads, time, head_dim,
                               window);
  if (rc != OMX_OK) return rc;
  return omx_causal_sdpa_backward(ctx, q, k, v, out, lse, gy, operand_dtype, OMX_F32, gy_dtype, gq, gk, gv, grad_dtype,
                                  batch, heads, kv_heads, time, head_dim, window);
}

// Time-major attention: the permute -> causal_sdpa -> permute of
// ojas-model/src/block.rs:186-199 (causal_attention) in one pass over [B, T, heads, D] tensors.
static int32_t check_attention(omx_ctx* ctx, const char* op, int32_t operand_dtype, uint64_t head_dim, uint64_t heads,
                               uint64_t kv_heads, uint64_t q_pitch, uint64_t kv_pitch, uint64_t out_pitch,
                               std::initializer_list<const void*> ptrs) {
  for (const void* p : ptrs) {
    if (!p) return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
    if (reinterpret_cast<uintptr_t>(p) & 15u) return omx_fail(ctx, OMX_SHAPE, "%s: tensor not 16-byte aligned", op);
  }
  if (!omx_flash_sdpa_supports(head_dim, operand_dtype))
    return omx_fail(ctx, OMX_UNSUPPORTED, "%s: only bf16 operands with head_dim 64 (compose permute and causal_sdpa)",
                    op);
  if (q_pitch < heads * head_dim || out_pitch < heads * head_dim || kv_pitch < kv_heads * head_dim ||
      (q_pitch | kv_pitch | out_pitch) % 8 != 0)
    return omx_fail(ctx, OMX_SHAPE, "%s: row pitch below heads * head_dim or not a multiple of 8", op);
  return OMX_OK;
}

static int32_t attention_forward(omx_ctx* ctx, const char* op, const void* q, uint64_t q_pitch, const void* k,
                                 const void* v, uint64_t kv_pitch, int32_t operand_dtype, void* out,
                                 void* out_residual, uint64_t out_pitch, int32_t out_dtype, void* lse, uint64_t batch,
                                 uint64_t time, uint64_t heads, uint64_t kv_heads, uint64_t head_dim, uint64_t window) {
  OMX_REQUIRE_CTX(ctx);
  if (out_dtype != OMX_BF16) return omx_fail(ctx, OMX_DTYPE, "%s: output must be bf16", op);
  SdpaShape s;
  int32_t rc = check_shape(ctx, op, batch, heads, kv_heads, time, head_dim, window, &s);
  if (rc != OMX_OK) return rc;
  rc = check_attention(ctx, op, operand_dtype, head_dim, heads, kv_heads, q_pitch, kv_pitch, out_pitch,
                       {q, k, v, out, lse});
  if (rc != OMX_OK) return rc;
  if (reinterpret_cast<uintptr_t>(out_residual) & 15u)
    return omx_fail(ctx, OMX_SHAPE, "%s: tensor not 16-byte aligned", op);
  const long D = static_cast<long>(head_dim), T = static_cast<long>(time);
  const long strides[9] = {static_cast<long>(q_pitch),   D, T * static_cast<long>(q_pitch),
                           static_cast<long>(kv_pitch),  D, T * static_cast<long>(kv_pitch),
                           static_cast<long>(out_pitch), D, T * static_cast<long>(out_pitch)};
  return omx_flash_sdpa_forward(ctx, q, k, v, out, out_dtype, out_residual, static_cast<float*>(lse), batch, heads,
                                kv_heads, time, head_dim, s.window, s.scale, omx_tag(ctx, F_SDPA_FORWARD), strides);
}

static int32_t attention_backward(omx_ctx* ctx, const char* op, const void* q, uint64_t q_pitch, const void* k,
                                  const void* v, uint64_t kv_pitch, const void* out, const void* out_residual,
                                  const void* gy, uint64_t out_pitch, const void* lse, int32_t operand_dtype, void* gq,
                                  void* gk, void* gv, int32_t grad_dtype, uint64_t batch, uint64_t time, uint64_t heads,
                                  uint64_t kv_heads, uint64_t head_dim, uint64_t window) {
  OMX_REQUIRE_CTX(ctx);
  if (grad_dtype != OMX_BF16) return omx_fail(ctx, OMX_DTYPE, "%s: gradients must be bf16", op);
  SdpaShape s;
  int32_t rc = check_shape(ctx, op, batch, heads, kv_heads, time, head_dim, window, &s);
  if (rc != OMX_OK) return rc;
  rc = check_attention(ctx, op, operand_dtype, head_dim, heads, kv_heads, q_pitch, kv_pitch, out_pitch,
                       {q, k, v, out, gy, lse, gq, gk, gv});
  if (rc != OMX_OK) return rc;
  if (reinterpret_cast<uintptr_t>(out_residual) & 15u)
    return omx_fail(ctx, OMX_SHAPE, "%s: tensor not 16-byte aligned", op);
  const long D = static_cast<long>(head_dim), T = static_cast<long>(time);
  const long strides[9] = {static_cast<long>(q_pitch),   D, T * static_cast<long>(q_pitch),
                           static_cast<long>(kv_pitch),  D, T * static_cast<long>(kv_pitch),
                           static_cast<long>(out_pitch), D, T * static_cast<long>(out_pitch)};
  return omx_flash_sdpa_backward(ctx, q, k, v, out, out_residual, static_cast<const float*>(lse), gy, gq, gk, gv,
                                 grad_dtype, batch, heads, kv_heads, time, head_dim, s.window, s.scale,
                                 omx_tag(ctx, F_SDPA_BACKWARD), strides);
}

int32_t omx_causal_attention_forward(omx_ctx* ctx, const void* q, uint64_t q_pitch, const void* k, const void* v,
                                     uint64_t kv_pitch, int32_t operand_dtype, void* out, uint64_t out_pitch,
                                     int32_t out_dtype, void* lse, uint64_t batch, uint64_t time, uint64_t heads,
                                     uint64_t kv_heads, uint64_t head_dim, uint64_t window) {
  return attention_forward(ctx, "causal_attention_forward", q, q_pitch, k, v, kv_pitch, operand_dtype, out, nullptr,
                           out_pitch, out_dtype, lse, batch, time, heads, kv_heads, head_dim, window);
}

int32_t omx_causal_attention_backward(omx_ctx* ctx, const void* q, uint64_t q_pitch, const void* k, const void* v,
                                      uint64_t kv_pitch, const void* out, const void* gy, uint64_t out_pitch,
                                      const void* lse, int32_t operand_dtype, void* gq, void* gk, void* gv,
                                      int32_t grad_dtype, uint64_t batch, uint64_t time, uint64_t heads,
                                      uint64_t kv_heads, uint64_t head_dim, uint64_t window) {
  return attention_backward(ctx, "causal_attention_backward", q, q_pitch, k, v, kv_pitch, out, nullptr, gy, out_pitch,
                            lse, operand_dtype, gq, gk, gv, grad_dtype, batch, time, heads, kv_heads, head_dim, window);
}

int32_t omx_causal_attention_forward_saving(omx_ctx* ctx, const void* q, uint64_t q_pitch, const void* k,
                                            const void* v, uint64_t kv_pitch, int32_t operand_dtype, void* out,
                                            void* out_residual, uint64_t out_pitch, int32_t out_dtype, void* lse,
                                            uint64_t batch, uint64_t time, uint64_t heads, uint64_t kv_heads,
                                            uint64_t head_dim, uint64_t window) {
  const char* op = "causal_attention_forward_saving";
  if (ctx && !out_residual) return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  return attention_forward(ctx, op, q, q_pitch, k, v, kv_pitch, operand_dtype, out, out_residual, out_pitch, out_dtype,
                           lse, batch, time, heads, kv_heads, head_dim, window);
}

int32_t omx_causal_attention_backward_saved(omx_ctx* ctx, const void* q, uint64_t q_pitch, const void* k,
                                            const void* v, uint64_t kv_pitch, const void* out,
                                            const void* out_residual, const void* gy, uint64_t out_pitch,
                                            const void* lse, int32_t operand_dtype, void* gq, void* gk, void* gv,
                                            int32_t grad_dtype, uint64_t batch, uint64_t time, uint64_t heads,
                                            uint64_t kv_heads, uint64_t head_dim, uint64_t window) {
  const char* op = "causal_attention_backward_saved";
  if (ctx && !out_residual) return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  return attention_backward(ctx, op, q, q_pitch, k, v, kv_pitch, out, out_residual, gy, out_pitch, lse, operand_dtype,
                            gq, gk, gv, grad_dtype, batch, time, heads, kv_heads, head_dim, window);
}

// The shape with the time-major tensors' strides, or why there is none. `rows`: on the kernels of a wave per row (the option
// "sdpa_tiled" 0, or more planes than a grid of the matrix kernels has).
static int32_t attention_f32(omx_ctx* ctx, const char* op, uint64_t q_pitch, uint64_t kv_pitch, uint64_t out_pitch, uint64_t batch,
                             uint64_t time, uint64_t heads, uint64_t kv_heads, uint64_t head_dim, uint64_t window,
                             std::initializer_list<const void*> ptrs, SdpaShape* s, bool* rows) {
  for (const void* p : ptrs)
    if (!p) return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
  int32_t rc = check_shape(ctx, op, batch, heads, kv_heads, time, head_dim, window, s);
  if (rc != OMX_OK) return rc;
  if (q_pitch < heads * head_dim || out_pitch < heads * head_dim || kv_pitch < kv_heads * head_dim)
    return omx_fail(ctx, OMX_SHAPE, "%s: row pitch below heads * head_dim", op);
  const long qp = static_cast<long>(q_pitch), kp = static_cast<long>(kv_pitch), op_ = static_cast<long>(out_pitch);
  if (!omx_sdpa32_supports(head_dim, 1, ptrs, {qp, kp, op_}))
    return omx_fail(ctx, OMX_UNSUPPORTED, "%s: head_dim %llu (16, 32, 64 or 128), 16-byte aligned tensors and pitches", op,
                    (unsigned long long)head_dim);
  *rows = !ctx->sdpa_tiled || !omx_sdpa32_supports(head_dim, batch * kv_heads, ptrs, {qp, kp, op_});
  s->q_h = s->k_h = s->o_h = s->dim;
  s->q_t = qp;
  s->k_t = kp;
  s->o_t = op_;
  s->q_b = qp * s->time;
  s->k_b = kp * s->time;
  s->o_b = op_ * s->time;
  return OMX_OK;
}

int32_t omx_causal_attention_f32_forward(omx_ctx* ctx, const void* q, uint64_t q_pitch, const void* k, const void* v, uint64_t kv_pitch,
                                         void* out, uint64_t out_pitch, void* lse, uint64_t batch, uint64_t time, uint64_t heads,
                                         uint64_t kv_heads, uint64_t head_dim, uint64_t window) {
  OMX_REQUIRE_CTX(ctx);
  SdpaShape s;
  bool rows;
  int32_t rc = attention_f32(ctx, "causal_attention_f32_forward", q_pitch, kv_pitch, out_pitch, batch, time, heads, kv_heads, head_dim,
                             window, {q, k, v, out, lse}, &s, &rows);
  if (rc != OMX_OK) return rc;
  const unsigned long long tag = omx_tag(ctx, F_SDPA_FORWARD);
  if (rows) return rows_forward<float, float>(ctx, q, k, v, out, lse, s, tag);
  Sdpa32Args a = sdpa32_args(ctx, q, k, v, s, tag);
  a.out = static_cast<float*>(out);
  a.lse = static_cast<float*>(lse);
  return omx_sdpa32_forward(ctx, a, static_cast<int>(batch), static_cast<int>(head_dim), false);
}

int32_t omx_causal_attention_f32_backward(omx_ctx* ctx, const void* q, uint64_t q_pitch, const void* k, const void* v, uint64_t kv_pitch,
                                          const void* out, const void* gy, uint64_t out_pitch, const void* lse, void* gq, void* gk, void* gv,
                                          uint64_t batch, uint64_t time, uint64_t heads, uint64_t kv_heads, uint64_t head_dim,
                                          uint64_t window) {
  OMX_REQUIRE_CTX(ctx);
  SdpaShape s;
  bool rows;
  int32_t rc = attention_f32(ctx, "causal_attention_f32_backward", q_pitch, kv_pitch, out_pitch, batch, time, heads, kv_heads, head_dim,
                             window, {q, k, v, out, gy, lse, gq, gk, gv}, &s, &rows);
  if (rc != OMX_OK) return rc;
  void* ws = nullptr;
  rc = omx_workspace(ctx, batch * heads * time * sizeof(float), &ws);
  if (rc != OMX_OK) return rc;
  const unsigned long long tag = omx_tag(ctx, F_SDPA_BACKWARD);
  if (rows) {
    rc = rows_delta<float, float>(ctx, out, gy, static_cast<float*>(ws), s);
    if (rc != OMX_OK) return rc;
    return rows_backward<float, float>(ctx, q, k, v, static_cast<const float*>(lse), static_cast<const float*>(ws), gy, gq, gk, gv, s, tag);
  }
  Sdpa32Args a = sdpa32_args(ctx, q, k, v, s, tag);
  a.out = const_cast<float*>(static_cast<const float*>(out));  // read only
  a.lse = const_cast<float*>(static_cast<const float*>(lse));
  a.gy = static_cast<const float*>(gy);
  a.gq = static_cast<float*>(gq);
  a.gk = static_cast<float*>(gk);
  a.gv = static_cast<float*>(gv);
  a.delta = static_cast<float*>(ws);
  return omx_sdpa32_backward(ctx, a, static_cast<int>(batch), static_cast<int>(head_dim));
}

}  // extern "C"
