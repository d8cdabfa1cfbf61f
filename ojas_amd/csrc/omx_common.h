// Internal declarations shared by the kernel files of libojas_mi355x.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <hip/hip_bf16.h>

#include <cstdarg>
#include <cstdint>
#include <tuple>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <map>
#include <set>
#include <string>
#include <unordered_map>
#include <vector>

#include "ojas_mi355x.h"

// Ops that can raise a deferred non-finite fault, in the order their bits sit
// in the fault word. The name is what OjasError::NonFinite { op } carries.
enum OmxFaultOp : uint32_t {
  F_LINEAR_FORWARD = 0,
  F_LINEAR_BACKWARD,
  F_GEMM,
  F_SDPA_FORWARD,
  F_SDPA_BACKWARD,
  F_RMS_FORWARD,
  F_RMS_BACKWARD,
  F_CE_FORWARD,
  F_CE_BACKWARD,
  F_LINEAR_CE,
  F_EMBEDDING_FORWARD,
  F_EMBEDDING_BACKWARD,
  F_ADAMW,
  F_MUON,
  F_CLIP,
  F_RESIDUAL_ADD,
  F_ACCUMULATE,
  F_SCALE_GRAD,
  F_GELU_FORWARD,
  F_GELU_BACKWARD,
  F_ARGMAX,
  F_TOPK,
  F_SILU_FORWARD,
  F_SILU_BACKWARD,
  F_MUL_FORWARD,
  F_MUL_BACKWARD,
  F_ROPE_FORWARD,
  F_ROPE_BACKWARD,
  F_RMS_QK_FORWARD,
  F_RMS_QK_BACKWARD,
  F_GATE_FORWARD,
  F_GATE_BACKWARD,
  F_VRES_FORWARD,
  F_VRES_BACKWARD,
  F_CACHED_ATTENTION,
  F_KV_CACHE_WRITE,
  F_COUNT
};
const char* omx_fault_name(uint32_t op);

// Device-side fault record: a bit mask plus the launch sequence number of the
// first op that faulted (lowest sequence wins), so the error can name it.
struct OmxFaultWord {
  unsigned long long mask;
  unsigned long long first;  // (sequence << 8) | op, ~0 when clear
};

// out[c] = sum over b < blocks of partial[b * dim + c].
struct OmxColumnSum {
  const float* partial;
  float* out;
  unsigned long long tag;
  int blocks, dim;
  const float* blend = nullptr;  // dim 1: out = s (1 - s) x the sum, s = sigmoid(*blend) (the gradient of a value blend's lambda)
};

// Freed blocks of one size, kept for the next request of it; the numbers of the last two requests (omx_ctx::requests).
struct OmxParked {
  std::vector<std::map<void*, uint64_t>::node_type> blocks;
  uint64_t last = 0, before = 0;
};

struct OmxI8Copy {
  uint64_t offset = 0, total = 0, formed = 0;
};
struct omx_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  uint64_t budget_limit = 0, budget_live = 0, budget_peak = 0;
  std::map<void*, uint64_t> allocations;
  // Freed blocks kept for reuse by size (see omx_free); not charged to the budget.
  std::unordered_map<uint64_t, OmxParked> pool;
  uint64_t pooled_bytes = 0, requests = 0;
  // Blocks freed while the stream was captured, which a graph may still write: they stay with the context, and while no one holds them they
  // are in for_graphs, by size, for allocations inside captures only.
  std::set<void*> freed_in_capture;
  std::multimap<uint64_t, std::map<void*, uint64_t>::node_type> for_graphs;
  OmxFaultWord* fault = nullptr;  // device
  OmxFaultWord* fault_host = nullptr;  // pinned, with kReadback bytes for what a small download brings behind it
  // Pinned memory that small uploads pass through (omx_upload_staged), taken by the first; up to `staged` the stream may still read it.
  char* stage = nullptr;
  uint64_t staged = 0;
  unsigned int* kv_refused = nullptr;  // device, behind the fault word: KvWrite::refused, zero between calls
  uint64_t sequence = 0;
  std::string last_error;
  std::string arch;
  // Scratch the library owns (charged to the budget); grown on demand.
  // Slot 0: per-op scratch. Slot 1: split-K partials of the GEMM (which an op
  // may call while it holds slot 0) and operands converted for an op that holds slot 0.
  // Slot 2: tensors an op keeps across calls into other ops (a recomputed attention output).
  void* workspace[6] = {};
  uint64_t workspace_bytes[6] = {};
  int slot_in_use = -1;  // kExtraSlot or kCopiesSlot, by the op that runs
  // The copy that the next int8 product keeps (omx_i8_copy_next), and what its copy, or the last one's, is known by.
  OmxI8Copy copy_next;
  uint64_t copy_formed = 0, copies_generation = 0;  // (the second: blocks that were workspace kCopiesSlot so far)
  bool copies_dropped = false;                      // an allocation needed their memory: no more of them
  // Column sums that wait (omx_defer_weight_sums), their partial rows in workspace kSumsSlot up to sums_used.
  bool sums_wait = false, prepare_sums_wait = false;
  uint32_t sums_expected = 0;
  uint64_t sums_used = 0;
  std::vector<OmxColumnSum> sums;
  bool workspace_captured[6] = {};  // handed out while the stream was captured
  int cu_count = 0;
  // This device's copy of the static scratch of omx_cross_entropy_mean_forward_static, looked up
  // when the context is opened (the lookup is not stream work and may load the code object).
  void* ce_static_scratch = nullptr;
  // Optional per-launch timing of the GEMM kernel (benchmark only).
  // 0: 128x128 register-staged kernel only; 1: choose by shape; others force a direct-to-LDS tiling (omx_set_option).
  int gemm_dma_mode = 1;
  int q8_widen = -1;         // int8 products over a widened copy of the weight: -1 by rule, 0 never, 1 wherever they can
  int gemm_f32_tile = -1;    // f32 products: -1: choose by estimate; 0..4, 5..8: a tile of gemm_frag32.hip, gemm_dma32.hip; 9: the register-staged kernel
  int gemm_f32_pair = -1;    // both f32 gradients of a linear layer in one launch: -1: by estimate; 0: never; 1..4: on these tiles
  int gemm_row_split = 1;    // 0: a product whose last round of 256 x 256 tiles is mostly empty is not cut by rows
  bool gemm_in_row_split = false;  // set while omx_gemm_impl runs the two halves of a cut product
  int gemm_forced_tiling = -1;     // the tiling the first half keeps, whatever its own tile count says
  int gemm_thin = 1;         // outputs of at most 64 columns over many rows take gemm_thin_kernel
  int flash_schedule = 0;     // 0: by the chip's workgroup places; 1: one 128-row block per workgroup; 2: mirrored pairs
  int flash_kv_parts = 0;     // workgroups that share a key block's query tiles: 0: by estimate; 1..64: always that many
  int attention_together = -1;  // attention backward in one launch: -1: by rule; 0: never; 1: wherever it can
  int kv_attention_mode = 0;  // 1: cached attention always takes the LDS-tiled kernel
  int adamw_trust = 1;        // 0: omx_adamw_step_bounded always runs its checking pass
  int ce_fused = 1;           // 0: linear-CE always takes the separate statistics and gradient kernels
  int sdpa_tiled = 1;         // 0: f32 attention always takes the one-wave-per-row kernels
  int gemm_skinny64 = -1;    // few rows on 64 columns a workgroup: -1: by rule; 0: never; 1, 2: wherever it fits, that many 16-row blocks a workgroup
  int muon_symmetric = 1;     // 0: bf16 Newton-Schulz forms both halves of X X^T and b A + c A^2
  int muon_fused_sums = 1;    // 0: Newton-Schulz forms b A + c A^2 and a X + B X in kernels of their own
  bool profile_gemm = false;
  uint32_t profile_classes = 0;  // bit per OmxKernelClass other than the products (omx_profile_kernels)
  // The events of the product being launched (null when not timing): the first kernel of the
  // product takes `timing_start`, its last one `timing_stop`.
  hipEvent_t timing_start = nullptr, timing_stop = nullptr;
  struct TimedLaunch {
    hipEvent_t start, stop;
    double flops;  // the launch's algorithmic work: FLOPs for the matrix-unit classes, bytes for the others
    int cls = 0;
  };
  std::vector<TimedLaunch> timed;
  std::vector<hipEvent_t> event_pool;
  bool launch_too_large = false;  // since the last OMX_LAUNCH_CHECK
};

// A kernel launch on the context's stream, the arguments converted to the kernel's parameter types. Straight through
// hipLaunchKernel: the <<<>>> form pushes the launch's shape onto a stack and pops it again in a stub of the kernel's,
// 0.25 us more of host time (3.1 -> 2.8 us), which is what bounds a chain of small kernels.
// A launch has at most 2^32 threads along an axis. The runtime multiplies in 32 bits and runs what is left of a larger one.
inline bool omx_launchable(omx_ctx* ctx, dim3 grid, dim3 block) {
  const bool fits = static_cast<uint64_t>(grid.x) * block.x <= 0xffffffffull && static_cast<uint64_t>(grid.y) * block.y <= 0xffffffffull;
  ctx->launch_too_large |= !fits;
  return fits;
}
template <typename... P, typename... Args>
inline void omx_launch(omx_ctx* ctx, void (*kernel)(P...), dim3 grid, dim3 block, unsigned smem, Args... args) {
  static_assert(sizeof...(P) == sizeof...(Args), "one argument for each parameter");
  if (!omx_launchable(ctx, grid, block)) return;
  std::tuple<P...> packed(static_cast<P>(args)...);
  void* at[sizeof...(P) ? sizeof...(P) : 1];
  std::apply([&](auto&... a) {
    size_t i = 0;
    ((at[i++] = const_cast<void*>(static_cast<const volatile void*>(&a))), ...);
  }, packed);
  (void)hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, at, smem, ctx->stream);
}
// The same; with events, the dispatch itself carries them (its own
// begin and end timestamps, no extra packets in the queue).
template <typename F, typename... Args>
inline void omx_launch_timed(omx_ctx* ctx, F kernel, dim3 grid, dim3 block, unsigned smem, hipEvent_t start,
                             hipEvent_t stop, Args... args) {
  if ((start || stop) && !omx_launchable(ctx, grid, block)) return;
  if (start || stop) hipExtLaunchKernelGGL(kernel, grid, block, smem, ctx->stream, start, stop, 0, args...);
  else omx_launch(ctx, kernel, grid, block, smem, args...);
}

int32_t omx_fail(omx_ctx* ctx, omx_status code, const char* fmt, ...);
void omx_release_pool(omx_ctx* ctx);
// The device address of the static cross-entropy scratch on the current device (loss.hip), or null.
void* omx_ce_static_scratch_address();
// Per-product timing for callers outside gemm.hip: takes a pair of events for the product about
// to be launched (when omx_profile_gemm is on) and files them with its FLOP count afterwards.
int32_t omx_timing_begin(omx_ctx* ctx, double flops, omx_ctx::TimedLaunch* timed);
void omx_timing_end(omx_ctx* ctx, bool launched, const omx_ctx::TimedLaunch& timed);

// Kernel classes that can be timed per launch (benchmark only); the values are those of
// omx_profile_kernels in the public header.
enum OmxKernelClass {
  OMX_K_GEMM = 0, OMX_K_FLASH_FWD = 1, OMX_K_FLASH_BWD = 2, OMX_K_CE = 3, OMX_K_ADAMW = 4, OMX_K_RMS_FWD = 5,
  OMX_K_RMS_BWD = 6, OMX_K_EMBED_BWD = 7, OMX_K_CLASSES = 8
};
// Events for one launch (or one run of launches) of a timed class: the first kernel is launched
// with start(), the last with stop() (both null while the class is off, which makes
// omx_launch_timed an ordinary launch); the destructor files the pair with `work`.
struct OmxKernelTimer {
  omx_ctx* ctx;
  omx_ctx::TimedLaunch t{};
  bool on = false;
  OmxKernelTimer(omx_ctx* ctx, int cls, double work);
  ~OmxKernelTimer();
  OmxKernelTimer(const OmxKernelTimer&) = delete;
  OmxKernelTimer& operator=(const OmxKernelTimer&) = delete;
  hipEvent_t start() const { return on ? t.start : nullptr; }
  hipEvent_t stop() const { return on ? t.stop : nullptr; }
};

int32_t omx_hip_fail(omx_ctx* ctx, hipError_t err, const char* what);
// Workspaces kExtraSlot, kSumsSlot and kCopiesSlot are for what an op can do without: any allocation that would be refused takes them back
// first.
constexpr int kExtraSlot = 3, kSumsSlot = 4, kCopiesSlot = 5;
constexpr bool can_do_without(int slot) { return slot >= kExtraSlot; }
// Grows workspace `slot` to at least `bytes` (budget-charged).
int32_t omx_workspace(omx_ctx* ctx, uint64_t bytes, void** out, int slot = 0);
// Whether the budget has room for workspace `slot` at that size (for an op that can do with less), counting what those three
// would give back.
bool omx_workspace_fits(const omx_ctx* ctx, uint64_t bytes, int slot = 0);
// Workspace `slot` for an op that can do without: null where the budget or the device lacks the room, and where a capture would have to
// allocate it.
void* omx_workspace_if_room(omx_ctx* ctx, uint64_t bytes, int slot = 0);
// Next launch tag for fault attribution: (sequence << 8) | op.
inline unsigned long long omx_tag(omx_ctx* ctx, uint32_t op) {
  return (static_cast<unsigned long long>(++ctx->sequence) << 8) | op;
}

// C[m,n] (+)= A.B with element strides; `ldc` is C's row pitch in elements.
// Optional elementwise work in the GEMM's store pass (bf16 outputs, or f32 throughout; `aux` has C's type and row pitch):
//   OMX_EPI_GELU_FWD: C = u (rounded to bf16) and aux_out = gelu(u). f32: nothing is rounded between, and shapes without a store pass
//     for it take a pass of its own;
//   OMX_EPI_GELU_BWD: C = round_bf16(A.B) * gelu'(aux_in). f32: as above;
//   OMX_EPI_AXPBY: C = round_bf16(s1 aux_in) + round_bf16(s2 round_bf16(A.B)): the product stored as
//     bf16, then the two-term sum a separate pass over it would form, in one store. f32 operands and output: C = s1 aux_in +
//     s2 A.B, each term rounded as a pass of its own would.
//   OMX_EPI_SWIGLU: C (f32, its first half of columns gates, the second ups) = A.B and aux_out [m, n / 2] (bf16) = silu(gate) up, every
//     bit as omx_swiglu_forward over C would have it; shapes without that store pass take the pass.
//   OMX_EPI_ROPE: aux_out [m, n] (bf16) = what omx_rope_half_split_pitched makes of A.B in f32, its bits; C (f32, [m, n]) is scratch for shapes
//     that take the pass, and is left alone otherwise.
//   OMX_EPI_SWIGLU_BWD: aux_out [m, 2 n] (bf16) = what omx_swiglu_backward makes of aux_in [m, 2 n] (f32, gates and ups) and A.B rounded
//     to bf16, its bits; C (bf16, [m, n]) is scratch for shapes that take the pass, and is left alone otherwise.
// aux tensors have C's layout (pitch, and batch stride in a strided batch).
enum { OMX_EPI_NONE = 0, OMX_EPI_GELU_FWD = 1, OMX_EPI_GELU_BWD = 2, OMX_EPI_AXPBY = 3, OMX_EPI_SWIGLU = 4, OMX_EPI_ROPE = 5, OMX_EPI_SWIGLU_BWD = 6 };
// The rotation of OMX_EPI_ROPE: tables [time, dim], rows are tokens of sequences of `time`, the first `heads` heads turn, `plain` follow.
struct OmxRope {
  const float *cos_t, *sin_t;
  int time, heads, plain, dim;
};
// A term of small rank beside a bf16 product, added in its accumulators (GemmArgs: lr_*).
struct OmxLowRank {
  const void *h, *w;
  uint64_t h_pitch, w_pitch, rank, block_cols;
};
struct OmxGemmEpilogue {
  int mode;
  int tanh_form;
  const void* aux_in;
  void* aux_out;
  float s1 = 0.0f, s2 = 0.0f;  // OMX_EPI_AXPBY
  OmxRope rope = {};           // OMX_EPI_ROPE
};
// `count` products of one shape whose operands lie `stride_*` ELEMENTS apart (16-byte multiples), one launch.
struct OmxGemmBatch {
  uint64_t count, stride_a, stride_b, stride_c;
  bool symmetric = false;  // every C equals its transpose, and aux_in too: kernels may form one half and store it twice
};
// `a_k`: columns of a k-contiguous A's rows that may be read, k of them and zeros after (0: just k).
int32_t omx_gemm_impl(omx_ctx* ctx, uint32_t fault_op, const void* a, uint64_t a_rs, uint64_t a_cs, const void* b,
                      uint64_t b_rs, uint64_t b_cs, int32_t operand_dtype, void* c, int32_t c_dtype, uint64_t ldc,
                      uint64_t m, uint64_t k, uint64_t n, int32_t accumulate, const OmxGemmEpilogue* epi = nullptr,
                      const OmxGemmBatch* batch = nullptr, uint64_t a_k = 0, const OmxLowRank* low_rank = nullptr);
bool omx_linear_backward_pair(omx_ctx* ctx, const float* x, const float* w, const float* gy, float* gx, float* gw, uint64_t rows, uint64_t in,
                              uint64_t out, bool onto, int32_t* rc);
double omx_gemm_bf16_us(const omx_ctx* ctx, uint64_t m, uint64_t k, uint64_t n);
// Whether omx_gemm_impl takes a bf16 product k-contiguous in A with a low-rank term (on the direct-to-LDS kernels).
bool omx_gemm_takes_low_rank(const omx_ctx* ctx, const void* a, uint64_t lda, const void* b, uint64_t ldb, uint64_t k);
// out[c] = sum over b < blocks of partial[b * dim + c], added in a fixed order.
// `scratch` (OMX_COLUMN_SUM_GROUPS * dim floats, may be null) lets a tall `partial` be added in two stages.
constexpr int OMX_COLUMN_SUM_GROUPS = 32;
// Up to this many rows a tall sum is one launch of 1024-thread workgroups.
constexpr int OMX_COLUMN_SUM_WIDE_ROWS = 1024;
// Sums wait in a list (`wait`) where omx_partial_rows has said so.
int32_t omx_column_sum(omx_ctx* ctx, const float* partial, float* out, uint64_t blocks, uint64_t dim, unsigned long long tag,
                       float* scratch = nullptr, hipEvent_t stop = nullptr, bool wait = false);
// Sums of 17 to OMX_COLUMN_SUM_WIDE_ROWS rows (with `blend`: of any number) in one launch, or in the list where `wait`.
int32_t omx_column_sums(omx_ctx* ctx, const OmxColumnSum* sums, int count, bool wait);
// Where sums wait and there is room, memory for their partial rows; else null.
float* omx_partial_rows(omx_ctx* ctx, uint64_t blocks, uint64_t dim);
// Forms every sum that waits.
int32_t omx_form_sums(omx_ctx* ctx);
// RMSNorm with 16-byte accesses for row widths 256..2048 (rmsvec.hip). `add` (forward) and
// `add_in` / `gx16` (backward) are optional fused operands.
bool omx_rms_vec_eligible(uint64_t dim, std::initializer_list<const void*> ptrs);
int32_t omx_rms_forward_vec(omx_ctx* ctx, const void* x, int32_t x_dtype, const void* add, int32_t add_dtype,
                            const float* w, float* sum_out, void* y, int32_t y_dtype, uint64_t rows, uint64_t dim,
                            float eps, unsigned long long tag);
int32_t omx_rms_backward_vec(omx_ctx* ctx, const void* x, int32_t x_dtype, const float* w, const void* gy,
                             int32_t gy_dtype, const float* add_in, void* gx, int32_t gx_dtype, void* gx16, float* gw,
                             uint64_t rows, uint64_t dim, float eps, unsigned long long tag);
// Elementwise conversions on the context's stream (no fault reporting).
int32_t omx_convert(omx_ctx* ctx, const void* src, int32_t src_dtype, void* dst, int32_t dst_dtype, uint64_t n);

#define OMX_HIP(ctx, expr)                                   \
  do {                                                       \
    hipError_t e_ = (expr);                                  \
    if (e_ != hipSuccess) return omx_hip_fail(ctx, e_, #expr); \
  } while (0)

#define OMX_LAUNCH_CHECK(ctx, what)                               \
  do {                                                            \
    hipError_t e_ = hipGetLastError();                            \
    if (e_ != hipSuccess) return omx_hip_fail(ctx, e_, what);     \
    if ((ctx)->launch_too_large) {                                \
      (ctx)->launch_too_large = false;                            \
      return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: more threads than a launch may have", what); \
    }                                                             \
  } while (0)

#define OMX_REQUIRE_CTX(ctx) \
  do {                       \
    if (!(ctx)) return OMX_BACKEND; \
  } while (0)

// ---- device helpers ----
typedef __hip_bfloat16 bf16_t;

// sigmoid(u) and 1 - sigmoid(u), both without cancellation.
__device__ __forceinline__ void dev_sigmoid_both(float u, float* s, float* rest) {
  const float e = __expf(-fabsf(u));
  const float inv = 1.0f / (1.0f + e);
  *s = u >= 0.0f ? inv : e * inv;
  *rest = u >= 0.0f ? e * inv : inv;
}
__device__ __forceinline__ float dev_sigmoid(float x) { return 1.0f / (1.0f + __expf(-x)); }
__device__ __forceinline__ bool dev_finite(float x) {
  return (__float_as_uint(x) & 0x7fffffffu) < 0x7f800000u;
}

// Round to nearest even on the dropped 16 bits; NaN keeps sign and payload and
// sets the quiet bit (ojas-core/src/autocast.rs:70-96). The integer form of the rule:
__device__ __forceinline__ unsigned short dev_f32_to_bf16_bits_integer_rule(float v) {
  unsigned int b = __float_as_uint(v);
  if (v != v) return static_cast<unsigned short>((b >> 16) | 0x0040u);
  unsigned int round = 0x7fffu + ((b >> 16) & 1u);
  return static_cast<unsigned short>((b + round) >> 16);
}
// The conversion instruction (v_cvt_pk_bf16_f32) gives the bits of that rule on every one of the
// 2^32 f32 patterns, NaN payloads and denormals included (checked exhaustively on the device;
// tests/test_gpu_parity_ops.py holds the casts to the rule over every exponent and the special
// values), at one instruction per pair instead of seven per value.
__device__ __forceinline__ unsigned int dev_pack_bf16_pair(float lo, float hi) {
  typedef __bf16 omx_bf16x2 __attribute__((ext_vector_type(2)));
  typedef float omx_floatx2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned int, __builtin_convertvector(omx_floatx2{lo, hi}, omx_bf16x2));
}
__device__ __forceinline__ unsigned short dev_f32_to_bf16_bits(float v) {
  return static_cast<unsigned short>(dev_pack_bf16_pair(v, 0.0f) & 0xffffu);
}
__device__ __forceinline__ float dev_bf16_bits_to_f32(unsigned short b) {
  return __uint_as_float(static_cast<unsigned int>(b) << 16);
}
__device__ __forceinline__ float dev_round_bf16(float v) {
  return dev_bf16_bits_to_f32(dev_f32_to_bf16_bits(v));
}

// The low byte of a tag is the op (bits 0-6) and the fault kind (bit 7:
// 0 = non-finite value, 1 = index out of range).
__device__ __forceinline__ void dev_raise_fault(OmxFaultWord* fault, unsigned long long tag) {
  atomicOr(&fault->mask, 1ull << (tag & 0x3full));
  atomicMin(&fault->first, tag);
}
__device__ __forceinline__ void dev_raise_range(OmxFaultWord* fault, unsigned long long tag) {
  atomicOr(&fault->mask, 1ull << (tag & 0x3full));
  atomicMin(&fault->first, tag | 0x80ull);
}

// Loads element i of a tensor stored as f32 or bf16, widened exactly.
template <typename T>
__device__ __forceinline__ float dev_load(const T* p, size_t i);
template <>
__device__ __forceinline__ float dev_load<float>(const float* p, size_t i) {
  return p[i];
}
template <>
__device__ __forceinline__ float dev_load<unsigned short>(const unsigned short* p, size_t i) {
  return dev_bf16_bits_to_f32(p[i]);
}
template <typename T>
__device__ __forceinline__ void dev_store(T* p, size_t i, float v);
template <>
__device__ __forceinline__ void dev_store<float>(float* p, size_t i, float v) {
  p[i] = v;
}
template <>
__device__ __forceinline__ void dev_store<unsigned short>(unsigned short* p, size_t i, float v) {
  p[i] = dev_f32_to_bf16_bits(v);
}

// 16 or 8 bytes that nothing reads again before the caches have forgotten them (STREAM), or as any other load or store. Reading 400 MB
// out of a set that the 256 MiB memory-side cache does not hold: 6.0 TB/s, 6.6 to 6.9 with the hint.
template <bool STREAM>
__device__ __forceinline__ float4 dev_stream_load(const float4* p) {
  if constexpr (!STREAM) return *p;
  typedef float f4 __attribute__((ext_vector_type(4)));
  const f4 v = __builtin_nontemporal_load(reinterpret_cast<const f4*>(p));
  return make_float4(v[0], v[1], v[2], v[3]);
}
template <bool STREAM>
__device__ __forceinline__ uint2 dev_stream_load(const uint2* p) {
  if constexpr (!STREAM) return *p;
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  const u2 v = __builtin_nontemporal_load(reinterpret_cast<const u2*>(p));
  return make_uint2(v[0], v[1]);
}
template <bool STREAM>
__device__ __forceinline__ uint4 dev_stream_load(const uint4* p) {
  if constexpr (!STREAM) return *p;
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  const u4 v = __builtin_nontemporal_load(reinterpret_cast<const u4*>(p));
  return make_uint4(v[0], v[1], v[2], v[3]);
}
template <bool STREAM>
__device__ __forceinline__ void dev_stream_store(float4* p, const float4& x) {
  if constexpr (STREAM) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    __builtin_nontemporal_store(f4{x.x, x.y, x.z, x.w}, reinterpret_cast<f4*>(p));
  } else {
    *p = x;
  }
}

template <bool STREAM>
__device__ __forceinline__ void dev_stream_store(uint4* p, const uint4& x) {
  if constexpr (STREAM) {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    __builtin_nontemporal_store(u4{x.x, x.y, x.z, x.w}, reinterpret_cast<u4*>(p));
  } else {
    *p = x;
  }
}

// Four consecutive elements starting at element index i (a multiple of 4; the
// address must be 16-byte aligned for f32 and 8-byte aligned for bf16).
template <typename T>
__device__ __forceinline__ void dev_load4(const T* p, size_t i, float (&v)[4]) {
  if constexpr (sizeof(T) == 4) {
    const float4 q = *reinterpret_cast<const float4*>(p + i);
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
  } else {
    const uint2 q = *reinterpret_cast<const uint2*>(p + i);
    v[0] = __uint_as_float(q.x << 16); v[1] = __uint_as_float(q.x & 0xffff0000u);
    v[2] = __uint_as_float(q.y << 16); v[3] = __uint_as_float(q.y & 0xffff0000u);
  }
}
template <typename T>
__device__ __forceinline__ void dev_store4(T* p, size_t i, const float (&v)[4]) {
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<float4*>(p + i) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    uint2 q;
    q.x = dev_pack_bf16_pair(v[0], v[1]);
    q.y = dev_pack_bf16_pair(v[2], v[3]);
    *reinterpret_cast<uint2*>(p + i) = q;
  }
}

// The wave's sum or maximum in every lane (all 64 active), halves first, by lane swaps and row rotations: once lanes 8 apart agree a
// rotation by 4 meets what an exchange with lane ^ 4 would. Exchanges through LDS wait some 60 clocks each, six
// times: norm backward over 4096 rows of 64 5.2 -> 4.2 us, over 3500 of 512 7.5 -> 7.1.
template <int CTRL>
__device__ __forceinline__ float dev_dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <typename F>
__device__ __forceinline__ float dev_meet_16(float v, F f) {  // lanes 16 apart
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <typename F>
__device__ __forceinline__ float dev_meet_32(float v, F f) {  // lanes 32 apart
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <typename F>
__device__ __forceinline__ float dev_wave_fold(float v, F f) {
  v = dev_meet_16(dev_meet_32(v, f), f);
  v = f(v, dev_dpp<0x128>(v));  // row_ror 8, 4, 2, 1
  v = f(v, dev_dpp<0x124>(v));
  v = f(v, dev_dpp<0x122>(v));
  return f(v, dev_dpp<0x121>(v));
}
__device__ __forceinline__ float wave_sum(float v) {
  return dev_wave_fold(v, [](float x, float y) { return x + y; });
}
__device__ __forceinline__ float wave_max(float v) {
  return dev_wave_fold(v, [](float x, float y) { return fmaxf(x, y); });
}

// GELU in f32. The erf form is 0.5 x (1 + erf(x / sqrt 2)); the tanh form is
// x * sigmoid(2 sqrt(2/pi) (x + 0.044715 x^3)), which has no cancellation in
// the negative tail (ojas-core/src/gelu_tanh.rs:8-15).
__device__ __forceinline__ float dev_gelu_erf(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float dev_gelu_erf_grad(float x) {
  float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
  float pdf = 0.3989422804014327f * __expf(-0.5f * x * x);
  return cdf + x * pdf;
}
__device__ __forceinline__ void dev_sigmoid_pair(float u, float* s, float* slope) {
  float e = __expf(-fabsf(u));
  float denom = 1.0f + e;
  *s = u >= 0.0f ? 1.0f / denom : e / denom;
  *slope = e / (denom * denom);
}
__device__ __forceinline__ float dev_gelu_tanh(float x) {
  float u = 2.0f * 0.7978845608028654f * (x + 0.044715f * x * x * x);
  float s, slope;
  dev_sigmoid_pair(u, &s, &slope);
  return x * s;
}
__device__ __forceinline__ float dev_gelu_tanh_grad(float x) {
  float u = 2.0f * 0.7978845608028654f * (x + 0.044715f * x * x * x);
  float s, slope;
  dev_sigmoid_pair(u, &s, &slope);
  float du = 2.0f * 0.7978845608028654f * (1.0f + 3.0f * 0.044715f * x * x);
  return s + x * slope * du;
}

// The same four functions for values stored in bf16 (8 bits of mantissa): the exact forms above cost
// 40 to 60 instructions per element (erff, IEEE divisions) and made the products that apply them in
// their store pass half as long again. These take one hardware exp2, one hardware reciprocal
// (1 ulp) and a few fmas. erf: Abramowitz & Stegun 7.1.26, |error| <= 1.5e-7, evaluated as erfc so
// the negative tail x * Phi(x) has no cancellation; exp(-z^2) doubles as the density in the
// derivative.
// tail = Phi(-|x|) and e = exp(-x^2 / 2). With w = |x| sqrt(log2(e) / 2): e = exp2(-w^2), and the
// series' argument |x| / sqrt 2 is w / sqrt(log2 e), so its constant folds into the fma that feeds
// the reciprocal; the 1/2 of erfc / 2 is folded into the coefficients.
__device__ __forceinline__ void dev_normal_tail_fast(float x, float* tail, float* e) {
  const float w = fabsf(x) * 0.84932180028801904f;
  const float t = __builtin_amdgcn_rcpf(fmaf(0.27273748087922250f, w, 1.0f));
  *e = __builtin_amdgcn_exp2f(-(w * w));
  float poly = fmaf(t, 0.5307027145f, -0.7265760135f);
  poly = fmaf(t, poly, 0.7107068705f);
  poly = fmaf(t, poly, -0.142248368f);
  poly = fmaf(t, poly, 0.127414796f);
  *tail = (poly * t) * *e;
}
// x Phi(x) = max(x, 0) - |x| Phi(-|x|): no branch on the sign and no 1 - tail.
__device__ __forceinline__ float dev_gelu_erf_fast(float x) {
  float tail, e;
  dev_normal_tail_fast(x, &tail, &e);
  return fmaf(-fabsf(x), tail, fmaxf(x, 0.0f));
}
__device__ __forceinline__ float dev_gelu_erf_grad_fast(float x) {
  float tail, e;
  dev_normal_tail_fast(x, &tail, &e);
  const float cdf = x >= 0.0f ? 1.0f - tail : tail;
  return fmaf(x, 0.3989422804014327f * e, cdf);
}
__device__ __forceinline__ void dev_sigmoid_pair_fast(float u, float* s, float* slope) {
  const float e = __builtin_amdgcn_exp2f(fabsf(u) * -1.4426950408889634f);
  const float r = __builtin_amdgcn_rcpf(1.0f + e);
  *s = u >= 0.0f ? r : e * r;
  *slope = e * r * r;
}
// 2 sqrt(2/pi) (x + 0.044715 x^3) as x (c0 + c1 x^2).
__device__ __forceinline__ float dev_gelu_tanh_arg_fast(float x) {
  return x * fmaf(0.07135481627260025f, x * x, 1.5957691216057308f);
}
__device__ __forceinline__ float dev_gelu_tanh_fast(float x) {
  const float u = dev_gelu_tanh_arg_fast(x);
  float s, slope;
  dev_sigmoid_pair_fast(u, &s, &slope);
  return x * s;
}
__device__ __forceinline__ float dev_gelu_tanh_grad_fast(float x) {
  const float u = dev_gelu_tanh_arg_fast(x);
  float s, slope;
  dev_sigmoid_pair_fast(u, &s, &slope);
  const float du = fmaf(0.21406444881780074f, x * x, 1.5957691216057308f);
  return fmaf(x * slope, du, s);
}
// GELU of a value whose storage type is T: exact for f32, the fast forms for bf16.
template <typename T, bool TANH>
__device__ __forceinline__ float dev_gelu_of(float x) {
  if constexpr (sizeof(T) == 2) return TANH ? dev_gelu_tanh_fast(x) : dev_gelu_erf_fast(x);
  else return TANH ? dev_gelu_tanh(x) : dev_gelu_erf(x);
}
template <typename T, bool TANH>
__device__ __forceinline__ float dev_gelu_grad_of(float x) {
  if constexpr (sizeof(T) == 2) return TANH ? dev_gelu_tanh_grad_fast(x) : dev_gelu_erf_grad_fast(x);
  else return TANH ? dev_gelu_tanh_grad(x) : dev_gelu_erf_grad(x);
}

inline bool omx_valid_float_dtype(int32_t d) { return d == OMX_F32 || d == OMX_BF16; }
inline size_t omx_dtype_size(int32_t d) { return d == OMX_BF16 ? 2 : 4; }
