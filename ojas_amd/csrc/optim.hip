// Optimizer kernels: AdamW, Muon NS5 and gradient clipping.
//
// Reference semantics:
//   adamw_step       ojas-cpu/src/optim.rs:302-395 (Fast f32 element math), two-pass
//                    all-or-nothing :513-621; scalars ojas-core/src/backend.rs:312-477
//   muon_ns5_step    ojas-cpu/src/optim.rs:684-743 (momentum, Nesterov, scale, decay),
//                    :841-985 (Newton-Schulz, f32 and bf16)
//   clip_grad_norm   ojas-cpu/src/backend.rs:770-795, optim.rs:61-160, clip_scale backend.rs:277-303
//
// Each element pass reads and writes every word once with 16-byte accesses.
// An optimizer step is all-or-nothing: a check pass decides on the device,
// and the apply pass writes nothing when any value of the call is non-finite.
#include <algorithm>
#include <cmath>

#include "omx_common.h"

namespace {

constexpr int OPT_THREADS = 256;
// Bytes of parameters, gradients and moments from which AdamW reads and writes them past the caches, which a step between two
// updates has long filled with other things: 124.4 M parameters inside their step 696 -> 649 us (5.7 TB/s), 35.5 M 186 -> 158. Alone,
// behind 1 GiB of other reads and writes, us without and with the hint: 192 MiB 109, 109; 256 146, 142; 384 213, 206; 1024 556, 514; one
// update straight after another, whose tensors partly stay, 256 MiB 118, 123; 320 170, 157; 512 291, 247.
constexpr uint64_t OPT_STREAM = 256ull << 20;

struct AdamWords {
  float decay, one_minus_b1, lerp_high, beta2, one_minus_b2, step_size, bc2_sqrt, eps;
  int decays, lerp_low;
};

// ojas-core/src/backend.rs:244-257
double pow_u64(double base, uint64_t exp) {
  double result = 1.0, b = base;
  while (exp > 0) {
    if (exp & 1) result *= b;
    exp >>= 1;
    if (exp > 0) b *= b;
  }
  return result;
}

__device__ __forceinline__ void adam_elem(const AdamWords& a, float p, float g, float m, float v, float* np,
                                          float* nm, float* nv, bool* ok) {
  // torch lerp: below weight 0.5 `m + w (g - m)`, else `g - (g - m)(1 - w)`.
  float m1 = a.lerp_low ? m + a.one_minus_b1 * (g - m) : g - (g - m) * a.lerp_high;
  float v1 = a.beta2 * v + a.one_minus_b2 * g * g;
  float denom = sqrtf(v1) / a.bc2_sqrt + a.eps;
  float delta = (-a.step_size) * m1 / denom;
  float q = p;
  if (a.decays) q *= a.decay;
  q += delta;
  // Without decay a zero step keeps the stored bits (-0.0 + 0.0 would flip a negative zero).
  float new_p = (!a.decays && delta == 0.0f) ? p : q;
  *ok = dev_finite(m1) && dev_finite(v1) && dev_finite(denom) && dev_finite(delta) && dev_finite(new_p);
  *np = new_p;
  *nm = m1;
  *nv = v1;
}

// What `omx_adamw_step_bounded` tracks: every stored value below 2^60 in magnitude (false for NaN).
constexpr float ADAM_BOUND = 1152921504606846976.0f;  // 2^60
__device__ __forceinline__ bool within_bound(float p, float m, float v) {
  return fabsf(p) < ADAM_BOUND && fabsf(m) < ADAM_BOUND && fabsf(v) < ADAM_BOUND;
}

__global__ __launch_bounds__(OPT_THREADS) void adamw_check_kernel(const float* __restrict__ p,
                                                                  const float* __restrict__ g,
                                                                  const float* __restrict__ m,
                                                                  const float* __restrict__ v, size_t n, AdamWords a,
                                                                  unsigned int* __restrict__ refuse,
                                                                  unsigned int* __restrict__ unbounded,
                                                                  OmxFaultWord* fault, unsigned long long tag) {
  bool bad = false, big = false;
  size_t stride = static_cast<size_t>(gridDim.x) * OPT_THREADS;
  for (size_t i = static_cast<size_t>(blockIdx.x) * OPT_THREADS + threadIdx.x; i < n; i += stride) {
    float np, nm, nv;
    bool ok;
    const float pi = p[i], mi = m[i], vi = v[i];
    adam_elem(a, pi, g[i], mi, vi, &np, &nm, &nv, &ok);
    bad |= !ok;
    big |= !within_bound(pi, mi, vi);
  }
  if (bad) {
    atomicOr(refuse, 1u);
    dev_raise_fault(fault, tag);
  }
  if (big && unbounded) atomicOr(unbounded, 1u);
}

__global__ __launch_bounds__(OPT_THREADS) void adamw_apply_kernel(float* __restrict__ p, const float* __restrict__ g,
                                                                  float* __restrict__ m, float* __restrict__ v,
                                                                  size_t n, AdamWords a,
                                                                  const unsigned int* __restrict__ refuse,
                                                                  unsigned int* __restrict__ unbounded,
                                                                  unsigned short* __restrict__ p_bf16) {
  if (refuse && *refuse) return;
  bool big = false;
  size_t stride = static_cast<size_t>(gridDim.x) * OPT_THREADS;
  for (size_t i = static_cast<size_t>(blockIdx.x) * OPT_THREADS + threadIdx.x; i < n; i += stride) {
    float np, nm, nv;
    bool ok;
    adam_elem(a, p[i], g[i], m[i], v[i], &np, &nm, &nv, &ok);
    p[i] = np;
    m[i] = nm;
    v[i] = nv;
    if (p_bf16) p_bf16[i] = dev_f32_to_bf16_bits(np);
    big |= !within_bound(np, nm, nv);
  }
  if (big && unbounded) atomicOr(unbounded, 1u);
}

// The same update on four consecutive elements per thread (16-byte accesses); every pointer
// 16-byte aligned (the bf16 copy 8-byte). The last n % 4 elements are thread 0's.
// SCALED: the gradient is scaled on its way through and written back, 4 bytes an element where a pass of its own takes 8 and its launch
// (124 million elements: 144 + 620 us, 649 together; 35 million 41 + 156, 170).
template <bool STREAM, bool SCALED>
__global__ __launch_bounds__(OPT_THREADS) void adamw_apply_vec_kernel(float* __restrict__ p,
                                                                      float* __restrict__ g,
                                                                      float* __restrict__ m, float* __restrict__ v,
                                                                      size_t n, AdamWords a,
                                                                      const unsigned int* __restrict__ refuse,
                                                                      unsigned int* __restrict__ unbounded,
                                                                      unsigned short* __restrict__ p_bf16, float scale) {
  if (refuse && *refuse) return;
  bool big = false;
  const size_t quads = n / 4;
  const size_t stride = static_cast<size_t>(gridDim.x) * OPT_THREADS;
  float4* p4 = reinterpret_cast<float4*>(p);
  float4* g4 = reinterpret_cast<float4*>(g);
  float4* m4 = reinterpret_cast<float4*>(m);
  float4* v4 = reinterpret_cast<float4*>(v);
  for (size_t i = static_cast<size_t>(blockIdx.x) * OPT_THREADS + threadIdx.x; i < quads; i += stride) {
    const float4 pq = dev_stream_load<STREAM>(p4 + i);
    float4 gq = dev_stream_load<STREAM>(g4 + i);
    const float4 mq = dev_stream_load<STREAM>(m4 + i), vq = dev_stream_load<STREAM>(v4 + i);
    if constexpr (SCALED) {
      gq = make_float4(gq.x * scale, gq.y * scale, gq.z * scale, gq.w * scale);
      dev_stream_store<STREAM>(g4 + i, gq);
    }
    const float pi[4] = {pq.x, pq.y, pq.z, pq.w}, gi[4] = {gq.x, gq.y, gq.z, gq.w};
    const float mi[4] = {mq.x, mq.y, mq.z, mq.w}, vi[4] = {vq.x, vq.y, vq.z, vq.w};
    float np[4], nm[4], nv[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      bool ok;
      adam_elem(a, pi[e], gi[e], mi[e], vi[e], &np[e], &nm[e], &nv[e], &ok);
      big |= !within_bound(np[e], nm[e], nv[e]);
    }
    dev_stream_store<STREAM>(p4 + i, make_float4(np[0], np[1], np[2], np[3]));
    dev_stream_store<STREAM>(m4 + i, make_float4(nm[0], nm[1], nm[2], nm[3]));
    dev_stream_store<STREAM>(v4 + i, make_float4(nv[0], nv[1], nv[2], nv[3]));
    if (p_bf16) {
      uint2 q;
      q.x = dev_pack_bf16_pair(np[0], np[1]);
      q.y = dev_pack_bf16_pair(np[2], np[3]);
      reinterpret_cast<uint2*>(p_bf16)[i] = q;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    for (size_t i = quads * 4; i < n; ++i) {
      float np, nm, nv;
      bool ok;
      if constexpr (SCALED) g[i] *= scale;
      adam_elem(a, p[i], g[i], m[i], v[i], &np, &nm, &nv, &ok);
      p[i] = np;
      m[i] = nm;
      v[i] = nv;
      if (p_bf16) p_bf16[i] = dev_f32_to_bf16_bits(np);
      big |= !within_bound(np, nm, nv);
    }
  }
  if (big && unbounded) atomicOr(unbounded, 1u);
}

// Sum of squares in f64, one partial per 16Ki-element block, summed inside a
// block in a fixed order (lane-strided, then a tree), so the norm does not
// depend on scheduling.
constexpr size_t NORM_BLOCK = 1 << 14;
__device__ __forceinline__ double sumsq4(const float4& u) {
  const double a = u.x, b = u.y, c = u.z, d = u.w;
  return (a * a + b * b) + (c * c + d * d);
}
// Block `block` of x; `red` is the workgroup's.
__device__ __forceinline__ void sumsq_block(const float* __restrict__ x, size_t n, unsigned block, double* red,
                                            double* __restrict__ out) {
  size_t begin = static_cast<size_t>(block) * NORM_BLOCK;
  size_t end = min(n, begin + NORM_BLOCK);
  double acc = 0.0;
  if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) {
    // 16-byte loads, four of them in flight per thread; the tail of the last block one by one.
    const float4* x4 = reinterpret_cast<const float4*>(x);
    const size_t q_begin = begin / 4, q_end = end / 4;  // NORM_BLOCK is a multiple of 4
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    size_t i = q_begin + threadIdx.x;
    for (; i + 3 * OPT_THREADS < q_end; i += 4 * OPT_THREADS) {
      const float4 u0 = x4[i], u1 = x4[i + OPT_THREADS], u2 = x4[i + 2 * OPT_THREADS], u3 = x4[i + 3 * OPT_THREADS];
      a0 += sumsq4(u0);
      a1 += sumsq4(u1);
      a2 += sumsq4(u2);
      a3 += sumsq4(u3);
    }
    for (; i < q_end; i += OPT_THREADS) a0 += sumsq4(x4[i]);
    acc = (a0 + a1) + (a2 + a3);
    for (size_t j = q_end * 4 + threadIdx.x; j < end; j += OPT_THREADS) {
      const double v = static_cast<double>(x[j]);
      acc += v * v;
    }
  } else {
    for (size_t i = begin + threadIdx.x; i < end; i += OPT_THREADS) {
      double v = static_cast<double>(x[i]);
      acc += v * v;
    }
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = OPT_THREADS / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}
__global__ __launch_bounds__(1024) void sumsq_final_kernel(const double* __restrict__ partial, size_t count,
                                                           double* __restrict__ out) {
  __shared__ double red[1024];
  double acc = 0.0;
  for (size_t i = threadIdx.x; i < count; i += 1024) acc += partial[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}
// Several tensors per launch, their pointers in the kernel's arguments: a model has tens of small vectors, and a launch
// for each is most of what clipping and stepping them costs (27 gradients of a small model: 54 launches to clip, 3.5 us
// each, now 3). Block b works on the tensor whose blocks start last at or before b.
constexpr int LIST_MAX = 48;
struct TensorSpans {
  uint64_t n[LIST_MAX];
  unsigned first[LIST_MAX + 1];  // first block of each tensor; first[count] ends the last one
  int count;
};
__device__ __forceinline__ int span_of(const TensorSpans& s, unsigned block) {
  int lo = 0, hi = s.count - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (s.first[mid] <= block) lo = mid;
    else hi = mid - 1;
  }
  return __builtin_amdgcn_readfirstlane(lo);
}

struct NormList {
  TensorSpans spans;
  const float* x[LIST_MAX];
};
__global__ __launch_bounds__(OPT_THREADS) void sumsq_list_kernel(NormList list, double* __restrict__ partial) {
  __shared__ double red[OPT_THREADS];
  const int t = span_of(list.spans, blockIdx.x);
  sumsq_block(list.x[t], list.spans.n[t], blockIdx.x - list.spans.first[t], red, partial + blockIdx.x);
}

struct ScaleList {
  TensorSpans spans;
  float* x[LIST_MAX];
};
// Four elements per thread, as 16 bytes where the tensor's alignment allows.
__global__ __launch_bounds__(OPT_THREADS) void scale_list_kernel(ScaleList list, float s) {
  const int t = span_of(list.spans, blockIdx.x);
  float* x = list.x[t];
  const size_t n = list.spans.n[t], base = static_cast<size_t>(blockIdx.x - list.spans.first[t]) * (OPT_THREADS * 4);
  const size_t i = base + threadIdx.x * 4;
  if ((reinterpret_cast<uintptr_t>(x) & 15) == 0 && i + 4 <= n) {
    float4 v = *reinterpret_cast<float4*>(x + i);
    v.x *= s;
    v.y *= s;
    v.z *= s;
    v.w *= s;
    *reinterpret_cast<float4*>(x + i) = v;
  } else {
    for (size_t j = i; j < i + 4 && j < n; ++j) x[j] *= s;
  }
}

// acc += grad over a list (accumulate_grad on each).
struct AccumulateList {
  TensorSpans spans;
  float* acc[LIST_MAX];
  const float* grad[LIST_MAX];
};
__global__ __launch_bounds__(OPT_THREADS) void accumulate_list_kernel(AccumulateList list, OmxFaultWord* fault,
                                                                      unsigned long long tag) {
  const int t = span_of(list.spans, blockIdx.x);
  float* acc = list.acc[t];
  const float* g = list.grad[t];
  const size_t n = list.spans.n[t], i = static_cast<size_t>(blockIdx.x - list.spans.first[t]) * (OPT_THREADS * 4) + threadIdx.x * 4;
  bool bad = false;
  if (((reinterpret_cast<uintptr_t>(acc) | reinterpret_cast<uintptr_t>(g)) & 15) == 0 && i + 4 <= n) {
    float4 v = *reinterpret_cast<float4*>(acc + i);
    const float4 w = *reinterpret_cast<const float4*>(g + i);
    v.x += w.x;
    v.y += w.y;
    v.z += w.z;
    v.w += w.w;
    bad = !(dev_finite(v.x) && dev_finite(v.y) && dev_finite(v.z) && dev_finite(v.w));
    *reinterpret_cast<float4*>(acc + i) = v;
  } else {
    for (size_t j = i; j < i + 4 && j < n; ++j) {
      acc[j] += g[j];
      bad |= !dev_finite(acc[j]);
    }
  }
  if (bad) dev_raise_fault(fault, tag);
}

// AdamW over a list: the check of every tensor in one launch, the update in another; each tensor has its own refusal
// word, so each is all-or-nothing by itself as with a call of its own.
struct AdamList {
  TensorSpans spans;
  float* p[LIST_MAX];
  const float* g[LIST_MAX];
  float* m[LIST_MAX];
  float* v[LIST_MAX];
};
template <bool APPLY>
__global__ __launch_bounds__(OPT_THREADS) void adamw_list_kernel(AdamList list, AdamWords a, unsigned int* __restrict__ refuse,
                                                                 OmxFaultWord* fault, unsigned long long tag) {
  const int t = span_of(list.spans, blockIdx.x);
  if (APPLY && refuse[t]) return;
  float* p = list.p[t];
  const float* g = list.g[t];
  float* m = list.m[t];
  float* v = list.v[t];
  const size_t n = list.spans.n[t], i = static_cast<size_t>(blockIdx.x - list.spans.first[t]) * (OPT_THREADS * 4) + threadIdx.x * 4;
  bool bad = false;
  const uintptr_t bits = reinterpret_cast<uintptr_t>(p) | reinterpret_cast<uintptr_t>(g) | reinterpret_cast<uintptr_t>(m) |
                         reinterpret_cast<uintptr_t>(v);
  if ((bits & 15) == 0 && i + 4 <= n) {
    const float4 pq = *reinterpret_cast<const float4*>(p + i), gq = *reinterpret_cast<const float4*>(g + i);
    const float4 mq = *reinterpret_cast<const float4*>(m + i), vq = *reinterpret_cast<const float4*>(v + i);
    const float pi[4] = {pq.x, pq.y, pq.z, pq.w}, gi[4] = {gq.x, gq.y, gq.z, gq.w};
    const float mi[4] = {mq.x, mq.y, mq.z, mq.w}, vi[4] = {vq.x, vq.y, vq.z, vq.w};
    float np[4], nm[4], nv[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      bool ok;
      adam_elem(a, pi[e], gi[e], mi[e], vi[e], &np[e], &nm[e], &nv[e], &ok);
      bad |= !ok;
    }
    if (APPLY) {
      *reinterpret_cast<float4*>(p + i) = make_float4(np[0], np[1], np[2], np[3]);
      *reinterpret_cast<float4*>(m + i) = make_float4(nm[0], nm[1], nm[2], nm[3]);
      *reinterpret_cast<float4*>(v + i) = make_float4(nv[0], nv[1], nv[2], nv[3]);
    }
  } else {
    for (size_t j = i; j < i + 4 && j < n; ++j) {
      float np, nm, nv;
      bool ok;
      adam_elem(a, p[j], g[j], m[j], v[j], &np, &nm, &nv, &ok);
      bad |= !ok;
      if (APPLY) {
        p[j] = np;
        m[j] = nm;
        v[j] = nv;
      }
    }
  }
  if (!APPLY && bad) {
    atomicOr(refuse + t, 1u);
    dev_raise_fault(fault, tag);
  }
}

// Fills a list's spans from lens[0 .. count) in blocks of `per_block` elements, up to LIST_MAX tensors or 2^30 blocks;
// returns how many tensors it took.
inline uint64_t fill_spans(TensorSpans& s, const uint64_t* lens, uint64_t count, uint64_t per_block) {
  uint64_t at = 0, t = 0;
  for (; t < count && t < LIST_MAX; ++t) {
    const uint64_t nb = (lens[t] + per_block - 1) / per_block;
    if (t > 0 && at + nb > (1ull << 30)) break;
    s.n[t] = lens[t];
    s.first[t] = static_cast<unsigned>(at);
    at += nb;
  }
  s.first[t] = static_cast<unsigned>(at);
  s.count = static_cast<int>(t);
  return t;
}

// A list's tensors step side by side, so one that overlaps another's result has to wait for the next launch, as it would
// for the next call. What the entries of a list read and write:
struct Touched {
  struct Span {
    uintptr_t begin, end;
    uint64_t entry;
    bool write;
  } spans[4 * LIST_MAX];
  int count = 0;
  void add(const void* p, uint64_t floats, uint64_t entry, bool write) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(p);
    spans[count++] = Span{at, at + floats * sizeof(float), entry, write};
  }
  // How many of the first `took` entries can step side by side (one at least).
  uint64_t apart(uint64_t took) {
    std::sort(spans, spans + count, [](const Span& a, const Span& b) { return a.begin < b.begin; });
    for (int i = 0; i < count; ++i)
      for (int j = i + 1; j < count && spans[j].begin < spans[i].end; ++j)
        if (spans[i].entry != spans[j].entry && (spans[i].write || spans[j].write))
          took = std::min(took, std::max(spans[i].entry, spans[j].entry));
    return took;
  }
};

inline unsigned grid_for(uint64_t n, int cu_count) {
  uint64_t blocks = (n + OPT_THREADS * 4 - 1) / (OPT_THREADS * 4);
  uint64_t cap = static_cast<uint64_t>(cu_count > 0 ? cu_count : 256) * 16;
  if (blocks > cap) blocks = cap;
  return static_cast<unsigned>(blocks ? blocks : 1);
}

}  // namespace

// The step's scalars from its configuration, or why there are none.
static int32_t adam_words(omx_ctx* ctx, const char* op, const omx_adamw_config* c, uint64_t step, AdamWords* out) {
  // check_adamw, ojas-core/src/backend.rs:312-352.
  const double scalars[5] = {c->lr, c->beta1, c->beta2, c->eps, c->weight_decay};
  for (double s : scalars)
    if (!std::isfinite(s)) return omx_fail(ctx, OMX_NON_FINITE, "%s", op);
  if (!(c->beta1 >= 0.0 && c->beta1 < 1.0 && c->beta2 >= 0.0 && c->beta2 < 1.0))
    return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: adamw beta must be in [0, 1)", op);
  if (c->eps <= 0.0) return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: adamw eps must be > 0", op);
  if (c->lr < 0.0) return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: lr %g is negative", op, c->lr);
  if (c->weight_decay < 0.0)
    return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: weight_decay %g is negative", op, c->weight_decay);
  if (step == UINT64_MAX) return omx_fail(ctx, OMX_OUT_OF_RANGE, "next_step: step counter is u64::MAX");
  const uint64_t next = step + 1;
  const double bc1 = 1.0 - pow_u64(c->beta1, next), bc2 = 1.0 - pow_u64(c->beta2, next);
  if (!(std::isfinite(bc1) && std::isfinite(bc2) && bc1 > 0.0 && bc2 > 0.0))
    return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: adamw bias correction is not a positive finite value", op);
  // AdamWScalars::from_bias_corrections + f32_words, backend.rs:387-477.
  const double one_minus_b1 = 1.0 - c->beta1;
  AdamWords& a = *out;
  a.decay = static_cast<float>(1.0 - c->lr * c->weight_decay);
  a.one_minus_b1 = static_cast<float>(one_minus_b1);
  a.lerp_high = 1.0f - a.one_minus_b1;
  a.beta2 = static_cast<float>(c->beta2);
  a.one_minus_b2 = static_cast<float>(1.0 - c->beta2);
  a.step_size = static_cast<float>(c->lr / bc1);
  a.bc2_sqrt = static_cast<float>(std::sqrt(bc2));
  a.eps = static_cast<float>(c->eps);
  a.decays = c->weight_decay != 0.0;
  a.lerp_low = a.one_minus_b1 < 0.5f;
  const float words[7] = {a.decay, a.one_minus_b1, a.beta2, a.one_minus_b2, a.step_size, a.bc2_sqrt, a.eps};
  for (float wd : words)
    if (!std::isfinite(wd)) return omx_fail(ctx, OMX_NON_FINITE, "%s", op);
  return OMX_OK;
}

// With every input below 2^60 in magnitude no result can be non-finite, provided the scalars
// are moderate: |m1| < 2^61, v1 < 2^121, denom >= eps, |delta| = step_size |m1| / denom
// < 2^20 2^61 2^40 = 2^121, |new p| <= 2 |p| + |delta|. The checking pass has nothing to find then.
static bool adam_moderate(const AdamWords& a) {
  return a.step_size <= 0x1p20f && fabsf(a.decay) <= 2.0f && a.eps >= 0x1p-40f && a.bc2_sqrt >= 0x1p-30f;
}
static bool adam_quads(const void* param, const void* grad, const void* moment1, const void* moment2, const void* param_bf16, uint64_t n) {
  const uintptr_t bits = reinterpret_cast<uintptr_t>(param) | reinterpret_cast<uintptr_t>(grad) |
                         reinterpret_cast<uintptr_t>(moment1) | reinterpret_cast<uintptr_t>(moment2) |
                         (reinterpret_cast<uintptr_t>(param_bf16) << 1);
  return (bits & 15) == 0 && n >= 4;
}

// `unbounded` (device u32 or null) collects whether any stored parameter or moment reaches 2^60;
// `inputs_bounded` is the caller's word that none of the four inputs does. `scale` other than 1 (an unchecked update of quads):
// the gradient is scaled by it in place.
static int32_t adamw_impl(omx_ctx* ctx, const char* op, void* param, const void* grad, void* moment1, void* moment2,
                   uint64_t n, uint64_t step, const omx_adamw_config* c, void* param_bf16, bool inputs_bounded,
                   unsigned int* unbounded, float scale = 1.0f) {
  OMX_REQUIRE_CTX(ctx);
  if (!param || !grad || !moment1 || !moment2 || !c) return omx_fail(ctx, OMX_PLACEMENT, "%s: null pointer", op);
  if (n == 0) return omx_fail(ctx, OMX_SHAPE, "%s: zero-sized axis", op);
  AdamWords a;
  const int32_t words_rc = adam_words(ctx, op, c, step, &a);
  if (words_rc != OMX_OK) return words_rc;

  const bool skip_check = inputs_bounded && adam_moderate(a);
  dim3 grid(grid_for(n, ctx->cu_count)), block(OPT_THREADS);
  unsigned int* refuse = nullptr;
  // Parameter, gradient and both moments read, parameter and moments written: 28 bytes per
  // element, and 2 more with the bf16 copy of the parameter, 4 with the gradient written back.
  OmxKernelTimer timer(ctx, OMX_K_ADAMW, (28.0 + (param_bf16 ? 2.0 : 0.0) + (scale != 1.0f ? 4.0 : 0.0)) * static_cast<double>(n));
  if (!skip_check) {
    void* ws = nullptr;
    int32_t rc = omx_workspace(ctx, 256, &ws);
    if (rc != OMX_OK) return rc;
    refuse = static_cast<unsigned int*>(ws);
    rc = omx_fill_zero(ctx, refuse, 4);
    if (rc != OMX_OK) return rc;
    omx_launch_timed(ctx, adamw_check_kernel, grid, block, 0, timer.start(), nullptr, static_cast<const float*>(param),
                     static_cast<const float*>(grad), static_cast<const float*>(moment1),
                     static_cast<const float*>(moment2), n, a, refuse, unbounded, ctx->fault, omx_tag(ctx, F_ADAMW));
    OMX_LAUNCH_CHECK(ctx, "adamw_check_kernel");
  }
  if (adam_quads(param, grad, moment1, moment2, param_bf16, n)) {
    dim3 vec_grid(static_cast<unsigned>((n / 4 + OPT_THREADS - 1) / OPT_THREADS));
    const bool stream = n * 16 >= OPT_STREAM;
    auto kernel = scale != 1.0f ? (stream ? &adamw_apply_vec_kernel<true, true> : &adamw_apply_vec_kernel<false, true>)
                                : (stream ? &adamw_apply_vec_kernel<true, false> : &adamw_apply_vec_kernel<false, false>);
    omx_launch_timed(ctx, kernel, vec_grid, block, 0, skip_check ? timer.start() : nullptr,
                     timer.stop(), static_cast<float*>(param), static_cast<float*>(const_cast<void*>(grad)),
                     static_cast<float*>(moment1), static_cast<float*>(moment2), n, a, refuse, unbounded,
                     static_cast<unsigned short*>(param_bf16), scale);
  } else {
    omx_launch_timed(ctx, adamw_apply_kernel, grid, block, 0, skip_check ? timer.start() : nullptr, timer.stop(),
                     static_cast<float*>(param), static_cast<const float*>(grad), static_cast<float*>(moment1),
                     static_cast<float*>(moment2), n, a, refuse, unbounded, static_cast<unsigned short*>(param_bf16));
  }
  OMX_LAUNCH_CHECK(ctx, "adamw_apply_kernel");
  return OMX_OK;
}

extern "C" {

int32_t omx_adamw_step(omx_ctx* ctx, void* param, const void* grad, void* moment1, void* moment2, uint64_t n,
                       uint64_t step, const omx_adamw_config* c, void* param_bf16) {
  return adamw_impl(ctx, "adamw_step", param, grad, moment1, moment2, n, step, c, param_bf16, false, nullptr);
}

int32_t omx_adamw_step_bounded(omx_ctx* ctx, void* param, const void* grad, void* moment1, void* moment2, uint64_t n,
                               uint64_t step, const omx_adamw_config* c, void* param_bf16, int32_t inputs_bounded,
                               void* unbounded_flag) {
  OMX_REQUIRE_CTX(ctx);
  if (!unbounded_flag) return omx_fail(ctx, OMX_PLACEMENT, "adamw_step_bounded: null pointer");
  return adamw_impl(ctx, "adamw_step_bounded", param, grad, moment1, moment2, n, step, c, param_bf16,
                    inputs_bounded != 0 && ctx->adamw_trust != 0, static_cast<unsigned int*>(unbounded_flag));
}

int32_t omx_adamw_step_batched(omx_ctx* ctx, void* const* params, const void* const* grads, void* const* moments1,
                               void* const* moments2, const uint64_t* lens, uint64_t count, uint64_t step,
                               const omx_adamw_config* c) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "adamw_step";
  if (!params || !grads || !moments1 || !moments2 || !lens || !c) return omx_fail(ctx, OMX_PLACEMENT, "%s: null pointer", op);
  if (count == 0) return omx_fail(ctx, OMX_SHAPE, "%s: no tensors", op);
  for (uint64_t t = 0; t < count; ++t) {
    if (!params[t] || !grads[t] || !moments1[t] || !moments2[t]) return omx_fail(ctx, OMX_PLACEMENT, "%s: null pointer", op);
    if (lens[t] == 0) return omx_fail(ctx, OMX_SHAPE, "%s: zero-sized axis", op);
  }
  AdamWords a;
  int32_t rc = adam_words(ctx, op, c, step, &a);
  if (rc != OMX_OK) return rc;
  void* ws = nullptr;
  rc = omx_workspace(ctx, count * sizeof(unsigned int), &ws);
  if (rc != OMX_OK) return rc;
  rc = omx_fill_zero(ctx, ws, count * sizeof(unsigned int));
  if (rc != OMX_OK) return rc;
  for (uint64_t t = 0; t < count;) {
    AdamList list;
    uint64_t took = fill_spans(list.spans, lens + t, count - t, OPT_THREADS * 4);
    Touched touched;
    for (uint64_t i = 0; i < took; ++i) {
      for (const void* p : {params[t + i], moments1[t + i], moments2[t + i]}) touched.add(p, lens[t + i], i, true);
      touched.add(grads[t + i], lens[t + i], i, false);
    }
    list.spans.count = static_cast<int>(took = touched.apart(took));
    for (uint64_t i = 0; i < took; ++i) {
      list.p[i] = static_cast<float*>(params[t + i]);
      list.g[i] = static_cast<const float*>(grads[t + i]);
      list.m[i] = static_cast<float*>(moments1[t + i]);
      list.v[i] = static_cast<float*>(moments2[t + i]);
    }
    unsigned int* refuse = static_cast<unsigned int*>(ws) + t;
    const dim3 grid(list.spans.first[took]), block(OPT_THREADS);
    omx_launch(ctx, adamw_list_kernel<false>, grid, block, 0, list, a, refuse, ctx->fault, omx_tag(ctx, F_ADAMW));
    omx_launch(ctx, adamw_list_kernel<true>, grid, block, 0, list, a, refuse, ctx->fault, omx_tag(ctx, F_ADAMW));
    OMX_LAUNCH_CHECK(ctx, "adamw_list_kernel");
    t += took;
  }
  return OMX_OK;
}

int32_t omx_accumulate_grads(omx_ctx* ctx, void* const* accs, const void* const* grads, const uint64_t* lens, uint64_t count) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "accumulate_grad";
  if (!accs || !grads || !lens) return omx_fail(ctx, OMX_PLACEMENT, "%s: null pointer", op);
  if (count == 0) return omx_fail(ctx, OMX_SHAPE, "%s: no tensors", op);
  for (uint64_t t = 0; t < count; ++t) {
    if (!accs[t] || !grads[t]) return omx_fail(ctx, OMX_PLACEMENT, "%s: null device pointer", op);
    if (lens[t] == 0) return omx_fail(ctx, OMX_SHAPE, "%s: zero-sized axis", op);
  }
  for (uint64_t t = 0; t < count;) {
    AccumulateList list;
    uint64_t took = fill_spans(list.spans, lens + t, count - t, OPT_THREADS * 4);
    Touched touched;
    for (uint64_t i = 0; i < took; ++i) {
      touched.add(accs[t + i], lens[t + i], i, true);
      touched.add(grads[t + i], lens[t + i], i, false);
    }
    list.spans.count = static_cast<int>(took = touched.apart(took));
    for (uint64_t i = 0; i < took; ++i) {
      list.acc[i] = static_cast<float*>(accs[t + i]);
      list.grad[i] = static_cast<const float*>(grads[t + i]);
    }
    omx_launch(ctx, accumulate_list_kernel, dim3(list.spans.first[took]), dim3(OPT_THREADS), 0, list, ctx->fault,
                       omx_tag(ctx, F_ACCUMULATE));
    OMX_LAUNCH_CHECK(ctx, "accumulate_list_kernel");
    t += took;
  }
  return OMX_OK;
}

}  // extern "C"

static int32_t clip_coefficient(omx_ctx* ctx, const void* const* grads, const uint64_t* lens, uint64_t count, float max_norm,
                                float* norm_out, float* scale_out) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "clip_grad_norm";
  if (!grads || !lens || !norm_out || !scale_out) return omx_fail(ctx, OMX_PLACEMENT, "%s: null pointer", op);
  if (count == 0) return omx_fail(ctx, OMX_SHAPE, "%s: no gradients", op);
  uint64_t blocks = 0;
  for (uint64_t t = 0; t < count; ++t) {
    if (!grads[t]) return omx_fail(ctx, OMX_PLACEMENT, "%s: gradient %llu is null", op, (unsigned long long)t);
    if (lens[t] == 0) return omx_fail(ctx, OMX_SHAPE, "%s: gradient %llu is empty", op, (unsigned long long)t);
    blocks += (lens[t] + NORM_BLOCK - 1) / NORM_BLOCK;
  }
  void* ws = nullptr;
  int32_t rc = omx_workspace(ctx, (blocks + 1) * sizeof(double), &ws);
  if (rc != OMX_OK) return rc;
  double* partial = static_cast<double*>(ws);
  double* total = partial + blocks;
  uint64_t at = 0;
  for (uint64_t t = 0; t < count;) {
    NormList list;
    const uint64_t took = fill_spans(list.spans, lens + t, count - t, NORM_BLOCK);
    for (uint64_t i = 0; i < took; ++i) list.x[i] = static_cast<const float*>(grads[t + i]);
    omx_launch(ctx, sumsq_list_kernel, dim3(list.spans.first[took]), dim3(OPT_THREADS), 0, list, partial + at);
    OMX_LAUNCH_CHECK(ctx, "sumsq_list_kernel");
    at += list.spans.first[took];
    t += took;
  }
  omx_launch(ctx, sumsq_final_kernel, dim3(1), dim3(1024), 0, partial, blocks, total);
  OMX_LAUNCH_CHECK(ctx, "sumsq_final_kernel");
  // The norm is a host value: this is the step's first sync point, and it
  // also reports any fault raised by the ops that produced the gradients.
  double sum_sq = 0.0;
  rc = omx_download(ctx, &sum_sq, total, 0, sizeof(double));
  if (rc != OMX_OK) return rc;
  float norm = static_cast<float>(std::sqrt(sum_sq));
  if (!std::isfinite(norm)) return omx_fail(ctx, OMX_NON_FINITE, "%s", op);
  // clip_scale, ojas-core/src/backend.rs:277-303.
  if (std::isnan(max_norm) || max_norm == -INFINITY) return omx_fail(ctx, OMX_NON_FINITE, "%s", op);
  if (max_norm < 0.0f) return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: max_norm %g is negative", op, max_norm);
  float coef = max_norm / (norm + 1e-6f);
  if (std::isnan(coef)) return omx_fail(ctx, OMX_NON_FINITE, "%s", op);
  if (coef > 1.0f) coef = 1.0f;
  *norm_out = norm;
  *scale_out = coef;
  return OMX_OK;
}

// grads *= scale, once for each time a tensor is listed.
static int32_t scale_gradients(omx_ctx* ctx, void* const* grads, const uint64_t* lens, uint64_t count, float scale) {
  for (uint64_t t = 0; t < count;) {
    ScaleList list;
    uint64_t took = fill_spans(list.spans, lens + t, count - t, OPT_THREADS * 4);
    Touched touched;
    for (uint64_t i = 0; i < took; ++i) touched.add(grads[t + i], lens[t + i], i, true);
    list.spans.count = static_cast<int>(took = touched.apart(took));
    for (uint64_t i = 0; i < took; ++i) list.x[i] = static_cast<float*>(grads[t + i]);
    omx_launch(ctx, scale_list_kernel, dim3(list.spans.first[took]), dim3(OPT_THREADS), 0, list, scale);
    OMX_LAUNCH_CHECK(ctx, "scale_list_kernel");
    t += took;
  }
  return OMX_OK;
}

extern "C" {

int32_t omx_clip_grad_norm(omx_ctx* ctx, void* const* grads, const uint64_t* lens, uint64_t count, float max_norm,
                           float* norm_out) {
  float norm = 0.0f, scale = 1.0f;
  int32_t rc = clip_coefficient(ctx, grads, lens, count, max_norm, norm_out ? &norm : nullptr, &scale);
  if (rc == OMX_OK && scale < 1.0f) rc = scale_gradients(ctx, grads, lens, count, scale);
  if (rc == OMX_OK) *norm_out = norm;
  return rc;
}

int32_t omx_clip_scale(omx_ctx* ctx, const void* const* grads, const uint64_t* lens, uint64_t count, float max_norm, float* norm_out,
                       float* scale_out) {
  return clip_coefficient(ctx, grads, lens, count, max_norm, norm_out, scale_out);
}

int32_t omx_adamw_step_scaled(omx_ctx* ctx, void* param, void* grad, void* moment1, void* moment2, uint64_t n, uint64_t step,
                              const omx_adamw_config* c, void* param_bf16, int32_t inputs_bounded, void* unbounded_flag, float scale) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "adamw_step_bounded";
  if (!(scale >= 0.0f && scale <= 1.0f)) return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: scale %g is outside [0, 1]", op, scale);
  if (!param || !grad || !moment1 || !moment2 || !c || !unbounded_flag) return omx_fail(ctx, OMX_PLACEMENT, "%s: null pointer", op);
  if (n == 0) return omx_fail(ctx, OMX_SHAPE, "%s: zero-sized axis", op);
  const bool bounded = inputs_bounded != 0 && ctx->adamw_trust != 0;
  AdamWords a;
  if (scale < 1.0f && !(bounded && adam_quads(param, grad, moment1, moment2, param_bf16, n) && adam_words(ctx, op, c, step, &a) == OMX_OK && adam_moderate(a))) {
    const int32_t rc = scale_gradients(ctx, &grad, &n, 1, scale);  // (an update that is checked, and may be refused, finds it scaled)
    if (rc != OMX_OK) return rc;
    scale = 1.0f;
  }
  return adamw_impl(ctx, op, param, grad, moment1, moment2, n, step, c, param_bf16, bounded, static_cast<unsigned int*>(unbounded_flag), scale);
}

}  // extern "C"
