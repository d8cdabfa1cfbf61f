// Muon NS5 step: BackendModule::muon_ns5_step (ojas-core/src/backend.rs:2480-2491,
// config :548-570). CPU reference: ojas-cpu/src/optim.rs:684-743 (momentum,
// Nesterov blend, scale, decay, update) and :841-985 (Newton-Schulz).
//
//   buf = mom * m + g;  u = nesterov ? fma(mom, buf, g) : buf
//   X = u / (||u||_F + 1e-7)        (norm from an f64 sum of squares; read as the
//                                    short-side-first matrix, a stride choice here)
//   5 x { A = X X^T;  B = b A + c A A;  X = a X + B X }   (a,b,c) = (3.4445, -4.7750, 2.0315)
//   p = fma(-lr * sqrt(max(1, rows/cols)), X, p * (1 - lr * wd));  m = buf
//
// In bf16 mode X, the norm, the sum with the epsilon, the quotient, every GEMM
// output and every scalar multiple and sum are rounded to bf16 (optim.rs:947-971);
// the iterate then lives in bf16 storage and the three products run on the
// bf16 MFMA lane, whose bf16 output store is exactly that rounding.
//
// The step is all-or-nothing, for the batch or (the list form) for each matrix: a refuse flag raised by any non-finite
// intermediate keeps the final pass from writing the parameter or the momentum.
#include <algorithm>
#include <cmath>
#include <vector>

#include "gemm_args.h"
#include "packs.h"

namespace {

constexpr int MU_THREADS = 256;
constexpr int MU_ITERATIONS = 5;
constexpr size_t MU_BLOCK = 1 << 11;  // elements per sum-of-squares partial (8 per thread: a 768 x 768 matrix fills the chip)

struct MuonScalars {
  float mom, decay, a, b, c;
  int nesterov, decays, bf16;
};

inline unsigned mu_grid(uint64_t n) {
  uint64_t blocks = (n + MU_THREADS * 4 - 1) / (MU_THREADS * 4);
  if (blocks > 4096) blocks = 4096;
  return static_cast<unsigned>(blocks ? blocks : 1);
}

// One launch serves up to MU_MAX_BATCH matrices: block (x, y) works on matrix y. The tensors the caller owns come as pointer
// tables in the kernel arguments; the intermediates of matrix y start `at` x 256 bytes into the workspace, at the offsets of
// its MuonLayout.
constexpr int MU_MAX_BATCH = 64;
struct MuonLayout {
  uint64_t buf, u, x, xn, a, a2, partial, scalars, total;
};
__host__ __device__ inline MuonLayout muon_layout(uint64_t rows, uint64_t cols) {
  auto up = [](uint64_t v) { return (v + 255) & ~255ull; };
  const uint64_t len = rows * cols, r = rows < cols ? rows : cols;
  MuonLayout L;
  uint64_t at = 0;
  L.buf = at;
  at += up(len * 4);
  L.u = at;
  at += up(len * 4);
  L.x = at;
  at += up(len * 4);
  L.xn = at;
  at += up(len * 4);
  L.a = at;
  at += up(r * r * 4);
  L.a2 = at;
  at += up(r * r * 4);
  L.partial = at;
  at += up(((len + MU_BLOCK - 1) / MU_BLOCK) * 8);
  L.scalars = at;
  at += 256;
  L.total = at;
  return L;
}
struct MuonTensors {
  float* p[MU_MAX_BATCH];
  const float* g[MU_MAX_BATCH];
  float* m[MU_MAX_BATCH];
  unsigned short* p16[MU_MAX_BATCH];  // entries may be null
  unsigned int at[MU_MAX_BATCH], rows[MU_MAX_BATCH], cols[MU_MAX_BATCH];
  float alpha[MU_MAX_BATCH];
};
struct MuonWork {
  char* ws;
  int each;  // the flag that keeps the final pass from writing: one for the launch (matrix 0's), or one for each matrix
};
// Matrix blockIdx.y of a launch.
struct MuonMatrix {
  char* ws;
  unsigned int* refuse;
  MuonLayout L;
  size_t n;
  __device__ __forceinline__ MuonMatrix(const MuonTensors& t, const MuonWork& w) {
    const unsigned y = blockIdx.y, f = w.each ? y : 0;
    ws = w.ws + static_cast<uint64_t>(t.at[y]) * 256;
    L = muon_layout(t.rows[y], t.cols[y]);
    n = static_cast<size_t>(t.rows[y]) * t.cols[y];
    refuse = reinterpret_cast<unsigned int*>(w.ws + static_cast<uint64_t>(t.at[f]) * 256 + muon_layout(t.rows[f], t.cols[f]).scalars);
  }
  template <typename T>
  __device__ __forceinline__ T* at(uint64_t offset) const {
    return reinterpret_cast<T*>(ws + offset);
  }
  // The iterate after `steps` iterations, which take turns in two buffers.
  __device__ __forceinline__ uint64_t iterate(int steps) const { return steps & 1 ? L.xn : L.x; }
};

template <bool STREAM>
__device__ __forceinline__ float mu_load(const float* p) { return STREAM ? __builtin_nontemporal_load(p) : *p; }

// f(integral_constant V, pack) for the packs of n elements that are this thread's: of four where every pointer allows (`quads`), the
// last ones, or all, of one. 24 matrices of 768 x 3072 and 48 of 768 x 768, bf16, an element a lane and now: apply 318 -> 255 us
// (6.7 TB/s), check 130 -> 106, normalize (with u in 16 bits) 123 -> 76, momentum 222 -> 208.
template <typename F>
__device__ __forceinline__ void mu_over(size_t n, bool quads, F&& f) {
  const size_t first = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x, stride = static_cast<size_t>(gridDim.x) * blockDim.x;
  const size_t packs = quads ? n / 4 : 0;
  for (size_t i = first; i < packs; i += stride) f(std::integral_constant<int, 4>{}, i);
  for (size_t i = packs * 4 + first; i < n; i += stride) f(std::integral_constant<int, 1>{}, i);
}
__device__ __forceinline__ bool mu_quads(const float* a, const float* b = nullptr, const unsigned short* c = nullptr) {
  return ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(c) << 1) & 15) == 0;
}

// buf, the update u (kept as TX: in the bf16 tier it is rounded to that), and per-block f64 sums of u^2.
template <bool STREAM, typename TX>
__global__ __launch_bounds__(MU_THREADS) void muon_momentum_kernel(MuonTensors t, MuonWork work, MuonScalars s, OmxFaultWord* fault,
                                                                   unsigned long long tag) {
  __shared__ double red[MU_THREADS];
  const MuonMatrix w(t, work);
  const size_t n = w.n;
  const float* __restrict__ g = t.g[blockIdx.y];
  const float* __restrict__ m = t.m[blockIdx.y];
  float* __restrict__ buf = w.at<float>(w.L.buf);
  TX* __restrict__ u = w.at<TX>(w.L.u);
  double* __restrict__ partial = w.at<double>(w.L.partial);
  const size_t begin = static_cast<size_t>(blockIdx.x) * MU_BLOCK, end = min(n, begin + MU_BLOCK);
  if (begin >= n) return;
  double acc = 0.0;
  bool bad = false;
  for (size_t i = begin + threadIdx.x; i < end; i += MU_THREADS) {
    const float gi = mu_load<STREAM>(g + i), b = s.mom * mu_load<STREAM>(m + i) + gi;
    bad |= !(dev_finite(b) && dev_finite(gi));
    float upd = s.nesterov ? fmaf(s.mom, b, gi) : b;
    if (s.bf16) upd = dev_round_bf16(upd);
    buf[i] = b;
    dev_store<TX>(u, i, upd);
    acc += static_cast<double>(upd) * static_cast<double>(upd);
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int st = MU_THREADS / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
  if (bad) {
    atomicOr(w.refuse, 1u);
    dev_raise_fault(fault, tag);
  }
}

__global__ void muon_clear_flags_kernel(MuonTensors t, MuonWork work) {
  const MuonMatrix w(t, work);
  if (threadIdx.x == 0) *w.refuse = 0u;
}

// One block per matrix (blockIdx.y): the norm and the quotient's denominator.
__global__ __launch_bounds__(1024) void muon_norm_kernel(MuonTensors t, MuonWork work, int bf16, OmxFaultWord* fault,
                                                         unsigned long long tag) {
  __shared__ double red[1024];
  const MuonMatrix w(t, work);
  const size_t count = (w.n + MU_BLOCK - 1) / MU_BLOCK;
  const double* __restrict__ partial = w.at<double>(w.L.partial);
  double acc = 0.0;
  for (size_t i = threadIdx.x; i < count; i += 1024) acc += partial[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int st = 512; st > 0; st >>= 1) {
    if (threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    float norm = static_cast<float>(sqrt(red[0]));
    const float eps = 1e-7f;
    float denom = bf16 ? dev_round_bf16(dev_round_bf16(norm) + eps) : norm + eps;
    *w.at<float>(w.L.scalars + 16) = denom;
    if (!(dev_finite(denom) && denom != 0.0f)) {
      atomicOr(w.refuse, 1u);
      dev_raise_fault(fault, tag);
    }
  }
}

template <typename TX>
__global__ void muon_normalize_kernel(MuonTensors t, MuonWork work) {
  const MuonMatrix w(t, work);
  const size_t n = w.n;
  const TX* __restrict__ u = w.at<TX>(w.L.u);
  TX* __restrict__ x = w.at<TX>(w.iterate(0));
  const float d = *w.at<float>(w.L.scalars + 16);
  mu_over(n, true, [&](auto size, size_t i) {
    constexpr int V = size.value;
    float v[V];
    load_pack<TX, V>(u, i, v);
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] /= d;
    store_pack<TX, V>(x, i, v);  // bf16 storage rounds the quotient
  });
}

// B = b A + c A2 (in place over A2), with the bf16 roundings of optim.rs:913-921.
template <typename TX>
__global__ void muon_combine_b_kernel(MuonTensors t, MuonWork work, MuonScalars s) {
  const MuonMatrix w(t, work);
  const size_t side = min(t.rows[blockIdx.y], t.cols[blockIdx.y]), n = side * side;
  const TX* __restrict__ am = w.at<TX>(w.L.a);
  TX* __restrict__ a2 = w.at<TX>(w.L.a2);
  for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<size_t>(gridDim.x) * blockDim.x) {
    float av = dev_load<TX>(am, i), a2v = dev_load<TX>(a2, i);
    float r;
    if (s.bf16) r = dev_round_bf16(s.b * av) + dev_round_bf16(s.c * a2v);
    else r = s.b * av + s.c * a2v;
    dev_store<TX>(a2, i, r);
  }
}

// X_next = a X + BX (in place over BX), finite-checked (optim.rs:950-962).
template <typename TX>
__global__ void muon_combine_x_kernel(MuonTensors t, MuonWork work, int steps, MuonScalars s, OmxFaultWord* fault,
                                      unsigned long long tag) {
  const MuonMatrix w(t, work);
  const size_t n = w.n;
  const TX* __restrict__ x = w.at<TX>(w.iterate(steps));
  TX* __restrict__ bx = w.at<TX>(w.iterate(steps + 1));
  bool bad = false;
  for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<size_t>(gridDim.x) * blockDim.x) {
    float xv = dev_load<TX>(x, i), bxv = dev_load<TX>(bx, i);
    float r = s.bf16 ? dev_round_bf16(s.a * xv) + bxv : s.a * xv + bxv;
    if (s.bf16) r = dev_round_bf16(r);
    bad |= !dev_finite(r);
    dev_store<TX>(bx, i, r);
  }
  if (bad) {
    atomicOr(w.refuse, 1u);
    dev_raise_fault(fault, tag);
  }
}

template <typename TX>
__global__ void muon_check_update_kernel(MuonTensors t, MuonWork work, MuonScalars s, OmxFaultWord* fault,
                                         unsigned long long tag) {
  const MuonMatrix w(t, work);
  const size_t n = w.n;
  const float alpha = t.alpha[blockIdx.y];
  const float* __restrict__ p = t.p[blockIdx.y];
  const TX* __restrict__ x = w.at<TX>(w.iterate(MU_ITERATIONS));
  bool bad = false;
  mu_over(n, mu_quads(p), [&](auto size, size_t i) {
    constexpr int V = size.value;
    float v[V], xv[V];
    load_pack<float, V>(p, i, v);
    load_pack<TX, V>(x, i, xv);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const float base = s.decays ? v[e] * s.decay : v[e];
      bad |= !dev_finite(fmaf(alpha, xv[e], base));
    }
  });
  if (bad) {
    atomicOr(w.refuse, 1u);
    dev_raise_fault(fault, tag);
  }
}

template <typename TX>
__global__ void muon_apply_kernel(MuonTensors t, MuonWork work, MuonScalars s) {
  const MuonMatrix w(t, work);
  if (*w.refuse) return;
  const size_t n = w.n;
  const float alpha = t.alpha[blockIdx.y];
  float* __restrict__ p = t.p[blockIdx.y];
  float* __restrict__ m = t.m[blockIdx.y];
  unsigned short* __restrict__ p_bf16 = t.p16[blockIdx.y];
  const float* __restrict__ buf = w.at<float>(w.L.buf);
  const TX* __restrict__ x = w.at<TX>(w.iterate(MU_ITERATIONS));
  mu_over(n, mu_quads(p, m, p_bf16), [&](auto size, size_t i) {
    constexpr int V = size.value;
    float v[V], xv[V], bv[V];
    load_pack<float, V>(p, i, v);
    load_pack<TX, V>(x, i, xv);
    load_pack<float, V>(buf, i, bv);
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = fmaf(alpha, xv[e], s.decays ? v[e] * s.decay : v[e]);
    store_pack<float, V>(p, i, v);
    store_pack<float, V>(m, i, bv);
    if (p_bf16) store_pack<unsigned short, V>(p_bf16, i, v);
  });
}

// Bytes of parameters, gradients, momenta and scratch from which gradients and momenta are read past the caches (48 matrices of 768 x
// 768: 98 -> 79 us; the update and the momentum just written stay there for the next passes).
constexpr uint64_t MU_STREAM = 256ull << 20;

// Matrices of one shape that lie one after another in a launch's tables.
struct MuonRun {
  unsigned first, count;
  uint64_t rows, cols;
};

// The Newton-Schulz iterations of one run, its products as strided batches.
template <typename TX>
int32_t iterate_run(omx_ctx* ctx, const MuonTensors& t, const MuonWork& w, const MuonRun& run, MuonScalars s, unsigned long long tag) {
  const uint64_t rows = run.rows, cols = run.cols;
  const MuonLayout L = muon_layout(rows, cols);
  const int32_t XD = sizeof(TX) == 2 ? OMX_BF16 : OMX_F32;
  char* ws = w.ws + static_cast<uint64_t>(t.at[run.first]) * 256;
  const bool tall = rows > cols;
  const uint64_t r = tall ? cols : rows, c = tall ? rows : cols;
  const uint64_t es = L.total / sizeof(TX);  // elements between consecutive matrices' buffers
  const OmxGemmBatch batch{run.count, es, es, es};
  const OmxGemmBatch* bp = run.count > 1 ? &batch : nullptr;
  // X X^T and the sum with its square equal their transposes.
  OmxGemmBatch half = batch;
  half.symmetric = ctx->muon_symmetric;
  const OmxGemmBatch* hp = bp ? &half : nullptr;
  TX* am = reinterpret_cast<TX*>(ws + L.a);
  TX* a2 = reinterpret_cast<TX*>(ws + L.a2);
  // The two-term sums after the second and third product ride in those products' store passes (the same roundings in the same
  // order as the combine kernels below; a non-finite value raises the fault there and reaches the final check through the remaining
  // products). bf16 tier: strided batches only, since a single product may split its reduction, which its store-pass sum cannot
  // follow. f32: the sums were 46 launches of 3 to 5 us in a step over five shapes.
  const bool fused = ctx->muon_fused_sums && (sizeof(TX) == 2 ? s.bf16 && run.count > 1 : !s.bf16);
  for (int it = 0; it < MU_ITERATIONS; ++it) {
    TX* x = reinterpret_cast<TX*>(ws + (it & 1 ? L.xn : L.x));
    TX* xn = reinterpret_cast<TX*>(ws + (it & 1 ? L.x : L.xn));
    int32_t rc;
    // A = X' X'^T with X' the short-side-first reading of X.
    if (!tall) rc = omx_gemm_impl(ctx, F_MUON, x, cols, 1, x, 1, cols, XD, am, XD, r, r, c, r, 0, nullptr, hp);
    else rc = omx_gemm_impl(ctx, F_MUON, x, 1, cols, x, cols, 1, XD, am, XD, r, r, c, r, 0, nullptr, hp);
    if (rc != OMX_OK) return rc;
    // B = b A + c A^2
    const OmxGemmEpilogue sum_b{OMX_EPI_AXPBY, 0, am, nullptr, s.b, s.c};
    // (A is its own transpose: read along its rows it is B's operand too)
    rc = omx_gemm_impl(ctx, F_MUON, am, r, 1, am, 1, r, XD, a2, XD, r, r, r, r, 0, fused ? &sum_b : nullptr, hp);
    if (rc != OMX_OK) return rc;
    if (!fused)
      omx_launch(ctx, (muon_combine_b_kernel<TX>), dim3(mu_grid(r * r), run.count), dim3(MU_THREADS), 0, t, w, s);
    // X_next = a X + B X, with BX in X's own physical layout: B X' when wide, X B^T when tall.
    const OmxGemmEpilogue sum_x{OMX_EPI_AXPBY, 0, x, nullptr, s.a, 1.0f};
    const OmxGemmEpilogue* ex = fused ? &sum_x : nullptr;
    if (!tall) rc = omx_gemm_impl(ctx, F_MUON, a2, r, 1, x, cols, 1, XD, xn, XD, cols, r, r, c, 0, ex, bp);
    else rc = omx_gemm_impl(ctx, F_MUON, x, cols, 1, a2, 1, r, XD, xn, XD, cols, rows, cols, cols, 0, ex, bp);
    if (rc != OMX_OK) return rc;
    if (!fused)
      omx_launch(ctx, (muon_combine_x_kernel<TX>), dim3(mu_grid(rows * cols), run.count), dim3(MU_THREADS), 0, t, w, it, s, ctx->fault, tag);
    OMX_LAUNCH_CHECK(ctx, "muon newton-schulz step");
  }
  return OMX_OK;
}

// The k-th products of several f32 runs in one launch, with the sums in their store passes.
int32_t iterate_together(omx_ctx* ctx, const MuonTensors& t, const MuonWork& w, const MuonRun* runs, int count, MuonScalars s) {
  for (int it = 0; it < MU_ITERATIONS; ++it)
    for (int stage = 0; stage < 3; ++stage) {
      OmxGemmProduct products[FRAG32_GROUP];
      for (int i = 0; i < count; ++i) {
        const MuonRun& run = runs[i];
        const MuonLayout L = muon_layout(run.rows, run.cols);
        char* ws = w.ws + static_cast<uint64_t>(t.at[run.first]) * 256;
        const float* x = reinterpret_cast<const float*>(ws + (it & 1 ? L.xn : L.x));
        float* xn = reinterpret_cast<float*>(ws + (it & 1 ? L.x : L.xn));
        float *am = reinterpret_cast<float*>(ws + L.a), *a2 = reinterpret_cast<float*>(ws + L.a2);
        const bool tall = run.rows > run.cols;
        const uint64_t r = tall ? run.cols : run.rows, c = tall ? run.rows : run.cols, cols = run.cols, es = L.total / 4;
        if (stage == 0) products[i] = tall ? OmxGemmProduct{x, 1, cols, x, cols, 1, am, r, r, c, r, nullptr, run.count, es}
                                           : OmxGemmProduct{x, cols, 1, x, 1, cols, am, r, r, c, r, nullptr, run.count, es};
        else if (stage == 1) products[i] = OmxGemmProduct{am, r, 1, am, r, 1, a2, r, r, r, r, am, run.count, es};
        else products[i] = tall ? OmxGemmProduct{x, cols, 1, a2, r, 1, xn, cols, run.rows, cols, cols, x, run.count, es}
                                : OmxGemmProduct{a2, r, 1, x, cols, 1, xn, cols, r, r, c, x, run.count, es};
      }
      const int32_t rc = omx_gemm_frag32_group(ctx, products, count, stage < 2, stage == 1 ? s.b : s.a, stage == 1 ? s.c : 1.0f, omx_tag(ctx, F_MUON));
      if (rc != OMX_OK) return rc;
    }
  return OMX_OK;
}
// The matrices of `runs` (at most MU_MAX_BATCH in all), their workspace blocks where t.at says, a run's one after another. More than
// one run: f32, and every run's products go out with the others'.
template <typename TX>
int32_t run_muon(omx_ctx* ctx, const MuonTensors& t, const std::vector<MuonRun>& runs, MuonScalars s, char* ws, bool each, unsigned long long tag) {
  unsigned count = 0;
  uint64_t most = 0, total = 0;
  for (const MuonRun& run : runs) {
    count += run.count;
    total += run.count * run.rows * run.cols;
    most = std::max(most, run.rows * run.cols);
  }
  const MuonWork w{ws, each};
  omx_launch(ctx, muon_clear_flags_kernel, dim3(1, each ? count : 1), dim3(64), 0, t, w);
  OMX_LAUNCH_CHECK(ctx, "muon_clear_flags_kernel");
  const dim3 block(MU_THREADS), over_len(mu_grid(most), count);
  const bool stream = total * 16 >= MU_STREAM;
  omx_launch(ctx, stream ? &muon_momentum_kernel<true, TX> : &muon_momentum_kernel<false, TX>, dim3(static_cast<unsigned>((most + MU_BLOCK - 1) / MU_BLOCK), count), block, 0, t, w, s, ctx->fault, tag);
  omx_launch(ctx, muon_norm_kernel, dim3(1, count), dim3(1024), 0, t, w, s.bf16, ctx->fault, tag);
  omx_launch(ctx, (muon_normalize_kernel<TX>), over_len, block, 0, t, w);
  OMX_LAUNCH_CHECK(ctx, "muon prologue");
  if (runs.size() == 1) {
    const int32_t rc = iterate_run<TX>(ctx, t, w, runs[0], s, tag);
    if (rc != OMX_OK) return rc;
  } else {
    for (size_t i = 0; i < runs.size(); i += FRAG32_GROUP) {
      const int32_t rc = iterate_together(ctx, t, w, runs.data() + i, static_cast<int>(std::min<size_t>(FRAG32_GROUP, runs.size() - i)), s);
      if (rc != OMX_OK) return rc;
    }
  }
  omx_launch(ctx, (muon_check_update_kernel<TX>), over_len, block, 0, t, w, s, ctx->fault, tag);
  omx_launch(ctx, (muon_apply_kernel<TX>), over_len, block, 0, t, w, s);
  OMX_LAUNCH_CHECK(ctx, "muon apply");
  return OMX_OK;
}

// check_muon (ojas-cpu/src/optim.rs:664-681) and the step's scalars.
int32_t muon_scalars(omx_ctx* ctx, const char* op, const omx_muon_config* c, uint64_t rows, uint64_t cols,
                     MuonScalars* out) {
  if (rows == 0 || cols == 0) return omx_fail(ctx, OMX_SHAPE, "%s: empty tensor", op);
  if (rows > 0x7fffffffull || cols > 0x7fffffffull) return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: axis too large", op);
  if (!std::isfinite(c->lr) || !std::isfinite(c->momentum) || !std::isfinite(c->weight_decay))
    return omx_fail(ctx, OMX_NON_FINITE, "%s", op);
  if (c->lr < 0.0) return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: lr %g is negative", op, c->lr);
  if (c->momentum < 0.0) return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: momentum %g is negative", op, c->momentum);
  if (c->weight_decay < 0.0)
    return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: weight_decay %g is negative", op, c->weight_decay);
  MuonScalars s;
  s.mom = static_cast<float>(c->momentum);
  s.decay = static_cast<float>(1.0 - c->lr * c->weight_decay);
  s.a = static_cast<float>(3.4445);
  s.b = static_cast<float>(-4.7750);
  s.c = static_cast<float>(2.0315);
  s.nesterov = c->nesterov != 0;
  s.decays = c->weight_decay != 0.0;
  s.bf16 = c->ns5_bf16 != 0;
  *out = s;
  return OMX_OK;
}

// The step length of one shape.
float muon_alpha(const omx_muon_config* c, uint64_t rows, uint64_t cols) {
  const double ratio = static_cast<double>(rows) / static_cast<double>(cols);
  return static_cast<float>(-c->lr * std::sqrt(ratio > 1.0 ? ratio : 1.0));
}

// `list`: each tensor all-or-nothing by itself, and as many at a time as MU_SCRATCH holds and the budget has room for, one
// at least.
constexpr uint64_t MU_SCRATCH = 256ull << 20;
int32_t muon_batch(omx_ctx* ctx, const char* op, void* const* params, const void* const* grads, void* const* momenta,
                   void* const* params_bf16, uint64_t count, uint64_t rows, uint64_t cols, const omx_muon_config* c,
                   bool list) {
  MuonScalars s;
  int32_t rc = muon_scalars(ctx, op, c, rows, cols, &s);
  if (rc != OMX_OK) return rc;
  for (uint64_t i = 0; i < count; ++i)
    if (!params[i] || !grads[i] || !momenta[i]) return omx_fail(ctx, OMX_PLACEMENT, "%s: null pointer", op);
  const MuonLayout L = muon_layout(rows, cols);
  uint64_t most = MU_MAX_BATCH;
  if (list) {
    most = std::max<uint64_t>(1, std::min<uint64_t>(most, MU_SCRATCH / L.total));
    most = std::min(most, count);
    while (most > 1 && !omx_workspace_fits(ctx, L.total * most)) --most;
  }
  for (uint64_t first = 0; first < count;) {
    unsigned n = static_cast<unsigned>(std::min<uint64_t>(most, count - first));
    void* ws = nullptr;
    rc = omx_workspace(ctx, L.total * n, &ws);
    if (rc == OMX_CAPACITY_EXCEEDED && list && n > 1) {  // (no memory left on the device)
      most = (n + 1) / 2;
      continue;
    }
    if (rc != OMX_OK) return rc;
    MuonTensors t{};
    for (unsigned i = 0; i < n; ++i) {
      t.p[i] = static_cast<float*>(params[first + i]);
      t.g[i] = static_cast<const float*>(grads[first + i]);
      t.m[i] = static_cast<float*>(momenta[first + i]);
      t.p16[i] = params_bf16 ? static_cast<unsigned short*>(params_bf16[first + i]) : nullptr;
      t.at[i] = static_cast<unsigned>(i * (L.total / 256));
      t.rows[i] = static_cast<unsigned>(rows);
      t.cols[i] = static_cast<unsigned>(cols);
      t.alpha[i] = muon_alpha(c, rows, cols);
    }
    const unsigned long long tag = omx_tag(ctx, F_MUON);
    const std::vector<MuonRun> runs{{0, n, rows, cols}};
    rc = s.bf16 ? run_muon<unsigned short>(ctx, t, runs, s, static_cast<char*>(ws), list, tag)
                : run_muon<float>(ctx, t, runs, s, static_cast<char*>(ws), list, tag);
    if (rc != OMX_OK) return rc;
    first += n;
  }
  return OMX_OK;
}

// Whether a shape's products go out with other shapes': f32 with the sums in the store passes, operands whose rows the group's tiles can
// read (widths in multiples of four), and at most MU_TOGETHER multiplications a product, its batch in all: there a launch's fixed time
// is worth more than the larger tiles that a launch of its own would take. A model's step, us, a set of launches for each shape / one
// for those that go together (with half the limit): 4 blocks of d = 128 413 / 134, of 256 586 / 305, 8 of 256 767 / 502 (588), 4 of 384
// 1190 / 891 (1004), of 512 1686 / 1565 (1631).
constexpr uint64_t MU_TOGETHER = 1ull << 30;
bool goes_together(omx_ctx* ctx, uint64_t rows, uint64_t cols, uint64_t count, bool bf16) {
  if (bf16 || !ctx->muon_fused_sums || ctx->gemm_dma_mode != 1 || ctx->gemm_f32_tile >= 0 /* a forced kernel or tile */ || rows % 4 != 0 || cols % 4 != 0 || rows > 1u << 15 || cols > 1u << 15) return false;
  return std::min(rows, cols) * rows * cols <= MU_TOGETHER / count;
}

// Tensors of several shapes, each all-or-nothing by itself: the shapes that go together in one set of launches (as many tensors at
// a time as a launch, MU_SCRATCH and the budget take), every other shape in one of its own.
int32_t muon_shapes(omx_ctx* ctx, const char* op, void* const* params, const void* const* grads, void* const* momenta, void* const* params_bf16,
                    const uint64_t* rows, const uint64_t* cols, uint64_t count, const omx_muon_config* c) {
  MuonScalars s;
  std::vector<std::vector<uint64_t>> shapes;  // the tensors of each, in the order of the first
  for (uint64_t i = 0; i < count; ++i) {
    const int32_t rc = muon_scalars(ctx, op, c, rows[i], cols[i], &s);
    if (rc != OMX_OK) return rc;
    if (!params[i] || !grads[i] || !momenta[i]) return omx_fail(ctx, OMX_PLACEMENT, "%s: null pointer", op);
    size_t k = 0;
    while (k < shapes.size() && (rows[shapes[k][0]] != rows[i] || cols[shapes[k][0]] != cols[i])) ++k;
    if (k == shapes.size()) shapes.emplace_back();
    shapes[k].push_back(i);
  }
  // The longest walks over K first: what starts last should be short.
  std::stable_sort(shapes.begin(), shapes.end(), [&](const std::vector<uint64_t>& x, const std::vector<uint64_t>& y) {
    return std::max(rows[x[0]], cols[x[0]]) > std::max(rows[y[0]], cols[y[0]]);
  });
  auto joins = [&](const std::vector<uint64_t>& shape) { return goes_together(ctx, rows[shape[0]], cols[shape[0]], shape.size(), s.bf16 != 0); };
  const bool several = std::count_if(shapes.begin(), shapes.end(), joins) > 1;
  std::vector<uint64_t> order;
  for (const auto& shape : shapes) {
    if (several && joins(shape)) {
      order.insert(order.end(), shape.begin(), shape.end());
      continue;
    }
    std::vector<void*> p, m, p16;
    std::vector<const void*> g;
    for (uint64_t i : shape) {
      p.push_back(params[i]);
      g.push_back(grads[i]);
      m.push_back(momenta[i]);
      p16.push_back(params_bf16 ? params_bf16[i] : nullptr);
    }
    const int32_t rc = muon_batch(ctx, op, p.data(), g.data(), m.data(), p16.data(), shape.size(), rows[shape[0]], cols[shape[0]], c, true);
    if (rc != OMX_OK) return rc;
  }
  uint64_t most = MU_MAX_BATCH;
  for (size_t first = 0; first < order.size();) {
    MuonTensors t{};
    std::vector<MuonRun> runs;
    uint64_t bytes = 0;
    unsigned n = 0;
    for (; n < most && first + n < order.size(); ++n) {
      const uint64_t i = order[first + n], need = muon_layout(rows[i], cols[i]).total;
      if (n > 0 && (bytes + need > MU_SCRATCH || !omx_workspace_fits(ctx, bytes + need))) break;
      if (runs.empty() || runs.back().rows != rows[i] || runs.back().cols != cols[i]) runs.push_back({n, 0, rows[i], cols[i]});
      ++runs.back().count;
      t.p[n] = static_cast<float*>(params[i]);
      t.g[n] = static_cast<const float*>(grads[i]);
      t.m[n] = static_cast<float*>(momenta[i]);
      t.p16[n] = params_bf16 ? static_cast<unsigned short*>(params_bf16[i]) : nullptr;
      t.at[n] = static_cast<unsigned>(bytes / 256);
      t.rows[n] = static_cast<unsigned>(rows[i]);
      t.cols[n] = static_cast<unsigned>(cols[i]);
      t.alpha[n] = muon_alpha(c, rows[i], cols[i]);
      bytes += need;
    }
    void* ws = nullptr;
    int32_t rc = omx_workspace(ctx, bytes, &ws);
    if (rc == OMX_CAPACITY_EXCEEDED && n > 1) {  // (no memory left on the device)
      most = (n + 1) / 2;
      continue;
    }
    if (rc != OMX_OK) return rc;
    rc = run_muon<float>(ctx, t, runs, s, static_cast<char*>(ws), true, omx_tag(ctx, F_MUON));
    if (rc != OMX_OK) return rc;
    first += n;
  }
  return OMX_OK;
}

}  // namespace

extern "C" {

uint64_t omx_muon_scratch_bytes(uint64_t rows, uint64_t cols) {
  if (rows == 0 || cols == 0) return 0;
  return muon_layout(rows, cols).total;
}

int32_t omx_muon_ns5_step(omx_ctx* ctx, void* param, const void* grad, void* momentum, uint64_t rows, uint64_t cols,
                          const omx_muon_config* c, void* param_bf16) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "muon_ns5_step";
  if (!param || !grad || !momentum || !c) return omx_fail(ctx, OMX_PLACEMENT, "%s: null pointer", op);
  void* mirrors[1] = {param_bf16};
  const void* grads[1] = {grad};
  return muon_batch(ctx, op, &param, grads, &momentum, param_bf16 ? mirrors : nullptr, 1, rows, cols, c, false);
}

int32_t omx_muon_ns5_step_batched(omx_ctx* ctx, void* const* params, const void* const* grads, void* const* momenta,
                                  void* const* params_bf16, uint64_t count, uint64_t rows, uint64_t cols,
                                  const omx_muon_config* c) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "muon_ns5_step";
  if (!params || !grads || !momenta || !c) return omx_fail(ctx, OMX_PLACEMENT, "%s: null pointer", op);
  if (count == 0) return omx_fail(ctx, OMX_SHAPE, "%s: no tensors", op);
  return muon_batch(ctx, op, params, grads, momenta, params_bf16, count, rows, cols, c, false);
}

int32_t omx_muon_ns5_step_list(omx_ctx* ctx, void* const* params, const void* const* grads, void* const* momenta,
                               void* const* params_bf16, uint64_t count, uint64_t rows, uint64_t cols,
                               const omx_muon_config* c) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "muon_ns5_step";
  if (!params || !grads || !momenta || !c) return omx_fail(ctx, OMX_PLACEMENT, "%s: null pointer", op);
  if (count == 0) return omx_fail(ctx, OMX_SHAPE, "%s: no tensors", op);
  return muon_batch(ctx, op, params, grads, momenta, params_bf16, count, rows, cols, c, true);
}

int32_t omx_muon_ns5_step_shapes(omx_ctx* ctx, void* const* params, const void* const* grads, void* const* momenta,
                                 void* const* params_bf16, const uint64_t* rows, const uint64_t* cols, uint64_t count,
                                 const omx_muon_config* c) {
  OMX_REQUIRE_CTX(ctx);
  const char* op = "muon_ns5_step";
  if (!params || !grads || !momenta || !rows || !cols || !c) return omx_fail(ctx, OMX_PLACEMENT, "%s: null pointer", op);
  if (count == 0) return omx_fail(ctx, OMX_SHAPE, "%s: no tensors", op);
  return muon_shapes(ctx, op, params, grads, momenta, params_bf16, rows, cols, count, c);
}

}  // extern "C"
