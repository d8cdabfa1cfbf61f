// Context, budget, residency and deferred-fault plumbing of libojas_mi355x.
//
// Mirrors what a device backend owns below ojas_core::Backend: placement
// (upload/download, backend.rs:908-973), budget charging that refuses rather
// than clamps (ojas-core/src/budget.rs:257-316), and the deferred non-finite
// contract of a device backend (ojas-wgpu/src/backend.rs:35-73).
#include <algorithm>
#include <functional>

#include "omx_common.h"

static const char* kFaultNames[F_COUNT] = {
    "linear_forward",
    "linear_backward",
    "gemm",
    "causal_sdpa_forward",
    "causal_sdpa_backward",
    "rms_norm_forward",
    "rms_norm_backward",
    "cross_entropy_mean_forward",
    "cross_entropy_mean_backward",
    "linear_cross_entropy_mean",
    "embedding_forward",
    "embedding_backward",
    "adamw_step",
    "muon_ns5_step",
    "clip_grad_norm",
    "residual_add_forward",
    "accumulate_grad",
    "scale_grad",
    "gelu_forward",
    "gelu_backward",
    "argmax_rows",
    "topk_rows",
    "silu_forward",
    "silu_backward",
    "mul_forward",
    "mul_backward",
    "rope_half_split_forward",
    "rope_half_split_backward",
    "rms_qk_norm_forward",
    "rms_qk_norm_backward",
    "per_head_sigmoid_gate_forward",
    "per_head_sigmoid_gate_backward",
    "value_residual_blend_forward",
    "value_residual_blend_backward",
    "cached_attention_forward",
    "kv_cache_write",
};

const char* omx_fault_name(uint32_t op) { return op < F_COUNT ? kFaultNames[op] : "unknown"; }

int32_t omx_fail(omx_ctx* ctx, omx_status code, const char* fmt, ...) {
  if (ctx) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    ctx->last_error = buf;
  }
  return code;
}

// HIP status mapping follows ojas-hip/src/lib.rs:106-122: 2 is out of memory,
// 3/4/35/100/101 mean no usable device, anything else is a launch failure.
int32_t omx_hip_fail(omx_ctx* ctx, hipError_t err, const char* what) {
  (void)hipGetLastError();  // it is reported here: the check after the next launch would find it again
  int code = static_cast<int>(err);
  omx_status st = OMX_BACKEND;
  if (code == 2) st = OMX_CAPACITY_EXCEEDED;
  else if (code == 3 || code == 4 || code == 35 || code == 100 || code == 101) st = OMX_DEVICE_LOST;
  return omx_fail(ctx, st, "hip: %s failed: %s (%d)", what, hipGetErrorString(err), code);
}

namespace {
constexpr uint64_t kReadback = 4096, kStage = 1ull << 20, kStageMost = 256ull << 10;
char* readback(omx_ctx* ctx) { return reinterpret_cast<char*>(ctx->fault_host) + 64; }

// The fault word and `n` bytes of `src` into pinned host memory.
__global__ __launch_bounds__(256) void read_back_kernel(const OmxFaultWord* fault, OmxFaultWord* fault_host, const char* src, char* dst, int n) {
  if (threadIdx.x == 0) *fault_host = *fault;
  for (int i = threadIdx.x; i < n; i += 256) dst[i] = src[i];
}
// Out of pinned host memory, 16 bytes a thread (both 16-byte aligned) and what is left of them.
__global__ __launch_bounds__(256) void stage_kernel(const char* src, char* dst, int n) {
  const int at = (blockIdx.x * 256 + threadIdx.x) * 16;
  if (at + 16 <= n) *reinterpret_cast<uint4*>(dst + at) = *reinterpret_cast<const uint4*>(src + at);
  else
    for (int i = at; i < n; ++i) dst[i] = src[i];
}

// Whether these bytes lie in one of the context's own blocks. What else a caller names (a range past its block, another device's
// memory, a host pointer) keeps the runtime's copy and its checks.
bool own_range(const omx_ctx* ctx, const void* at, uint64_t n) {
  auto block = ctx->allocations.upper_bound(const_cast<void*>(at));
  if (block == ctx->allocations.begin()) return false;
  --block;
  const uint64_t from = static_cast<uint64_t>(static_cast<const char*>(at) - static_cast<const char*>(block->first));
  return from <= block->second && n <= block->second - from;
}

int32_t wait(omx_ctx* ctx) {
  OMX_HIP(ctx, hipStreamSynchronize(ctx->stream));
  ctx->staged = 0;
  return OMX_OK;
}
}  // namespace

static int32_t reset_fault(omx_ctx* ctx) {
  ctx->fault_host->mask = 0;
  ctx->fault_host->first = ~0ull;
  OMX_HIP(ctx, hipMemcpyAsync(ctx->fault, ctx->fault_host, sizeof(OmxFaultWord), hipMemcpyHostToDevice,
                              ctx->stream));
  OMX_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return OMX_OK;
}

extern "C" {

int32_t omx_open(int32_t device, uint64_t budget_bytes, omx_ctx** out) {
  if (!out) return OMX_BACKEND;
  *out = nullptr;
  int count = 0;
  hipError_t err = hipGetDeviceCount(&count);
  if (err != hipSuccess || count <= 0 || device < 0 || device >= count) return OMX_DEVICE_LOST;
  omx_ctx* ctx = new omx_ctx();
  ctx->device = device;
  ctx->budget_limit = budget_bytes;
  if (hipSetDevice(device) != hipSuccess) {
    delete ctx;
    return OMX_DEVICE_LOST;
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) != hipSuccess) {
    delete ctx;
    return OMX_DEVICE_LOST;
  }
  ctx->arch = prop.gcnArchName;
  ctx->cu_count = prop.multiProcessorCount;
  if (ctx->arch.rfind("gfx950", 0) != 0) {
    // The kernels are built for gfx950 only; any other device cannot run them.
    delete ctx;
    return OMX_UNSUPPORTED;
  }
  if (hipStreamCreate(&ctx->stream) != hipSuccess || hipMalloc(&ctx->fault, 256) != hipSuccess ||
      hipHostMalloc(&ctx->fault_host, 64 + kReadback) != hipSuccess) {
    delete ctx;
    return OMX_BACKEND;
  }
  if (reset_fault(ctx) != OMX_OK) {
    delete ctx;
    return OMX_BACKEND;
  }
  static_assert(sizeof(OmxFaultWord) <= 64, "the refused-write word lies behind the fault word");
  ctx->kv_refused = reinterpret_cast<unsigned int*>(reinterpret_cast<char*>(ctx->fault) + 64);
  if (omx_fill_zero(ctx, ctx->kv_refused, 64) != OMX_OK || hipStreamSynchronize(ctx->stream) != hipSuccess) {
    delete ctx;
    return OMX_BACKEND;
  }
  ctx->ce_static_scratch = omx_ce_static_scratch_address();
  *out = ctx;
  return OMX_OK;
}

void omx_close(omx_ctx* ctx) {
  if (!ctx) return;
  (void)hipSetDevice(ctx->device);
  (void)hipStreamSynchronize(ctx->stream);
  for (auto& kv : ctx->allocations) (void)hipFree(kv.first);
  for (auto& parked : ctx->pool)
    for (auto& block : parked.second.blocks) (void)hipFree(block.key());
  for (auto& kept : ctx->for_graphs) (void)hipFree(kept.second.key());
  if (ctx->fault) (void)hipFree(ctx->fault);
  if (ctx->fault_host) (void)hipHostFree(ctx->fault_host);
  if (ctx->stage) (void)hipHostFree(ctx->stage);
  if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
  delete ctx;
}

size_t omx_last_error(omx_ctx* ctx, char* buf, size_t cap) {
  if (!ctx) return 0;
  if (buf && cap) {
    size_t n = ctx->last_error.size() < cap - 1 ? ctx->last_error.size() : cap - 1;
    memcpy(buf, ctx->last_error.data(), n);
    buf[n] = 0;
  }
  return ctx->last_error.size();
}

size_t omx_device_name(omx_ctx* ctx, char* buf, size_t cap) {
  if (!ctx) return 0;
  if (buf && cap) {
    size_t n = ctx->arch.size() < cap - 1 ? ctx->arch.size() : cap - 1;
    memcpy(buf, ctx->arch.data(), n);
    buf[n] = 0;
  }
  return ctx->arch.size();
}

}  // extern "C"

// Returns every parked block to the device (waits for the stream first).
void omx_release_pool(omx_ctx* ctx) {
  if (ctx->pooled_bytes == 0) return;
  (void)hipStreamSynchronize(ctx->stream);
  for (auto& parked : ctx->pool)
    for (auto& block : parked.second.blocks) (void)hipFree(block.key());
  ctx->pool.clear();
  ctx->pooled_bytes = 0;
}

namespace {
constexpr uint64_t kMaxBlock = 256ull << 20, kMaxPool = 4ull << 30;  // parked: a block at most, all of them together
constexpr size_t kMaxSizes = 4096;  // sizes remembered

bool capturing(const omx_ctx* ctx) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(ctx->stream, &status) == hipSuccess && status != hipStreamCaptureStatusNone;
}

// Whether drop_extra gives workspace `slot` (one that ops can do without) back: not while the op that runs uses it, a graph holds its
// address or a capture is on.
bool droppable(const omx_ctx* ctx, int slot) {
  return ctx->workspace[slot] && slot != ctx->slot_in_use && !ctx->workspace_captured[slot] && !capturing(ctx);
}

// Gives workspaces kExtraSlot, kSumsSlot and kCopiesSlot back, with the sums that wait there formed. Whether there was one. (No op allocates
// between omx_partial_rows and its omx_column_sum.)
bool drop_extra(omx_ctx* ctx) {
  bool dropped = false;
  for (int slot : {kExtraSlot, kSumsSlot, kCopiesSlot}) {
    void*& held = ctx->workspace[slot];
    if (!droppable(ctx, slot) || (slot == kSumsSlot && omx_form_sums(ctx) != OMX_OK)) continue;
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) return dropped;
    ctx->budget_live -= ctx->allocations[held];
    ctx->allocations.erase(held);
    (void)hipFree(held);
    held = nullptr;
    ctx->workspace_bytes[slot] = 0;
    ctx->copies_dropped |= slot == kCopiesSlot;
    dropped = true;
  }
  return dropped;
}

// Room in a full pool for a block of `bytes`: out go blocks of sizes that were last asked for before number `since`, longest ago first, and
// an eighth of the pool at once, for every time is a wait. `since` is the request for `bytes` before its last one. So a size that comes
// back takes the place of sizes that did not come back meanwhile, and a program that goes round through more than the pool holds keeps
// what it has, each of its sizes having been asked for since. Without this the blocks of two closed trainers held the pool for good:
// a decode step of 64 sequences, 12.9 MB of logits allocated and freed in each, 1.93 ms after them and 1.47 in a process of its own.
void make_room(omx_ctx* ctx, uint64_t bytes, uint64_t since) {
  std::vector<std::pair<uint64_t, uint64_t>> old;  // last asked for, size
  for (const auto& parked : ctx->pool)
    if (!parked.second.blocks.empty() && parked.second.last < since) old.emplace_back(parked.second.last, parked.first);
  if (old.empty() || hipStreamSynchronize(ctx->stream) != hipSuccess) return;
  std::sort(old.begin(), old.end());
  for (const auto& [last, size] : old) {
    auto& blocks = ctx->pool[size].blocks;
    for (size_t i = blocks.size(); i-- > 0;) {
      if (ctx->pooled_bytes + bytes <= kMaxPool - kMaxPool / 8) return;
      (void)hipFree(blocks[i].key());
      blocks.erase(blocks.begin() + static_cast<std::ptrdiff_t>(i));
      ctx->pooled_bytes -= size;
    }
  }
}
}  // namespace

extern "C" {

int32_t omx_alloc(omx_ctx* ctx, uint64_t bytes, void** out) {
  OMX_REQUIRE_CTX(ctx);
  if (!out) return omx_fail(ctx, OMX_BACKEND, "omx_alloc: null out");
  *out = nullptr;
  if (bytes == 0) return omx_fail(ctx, OMX_SHAPE, "omx_alloc: zero bytes");
  // Charge before allocating; refuse, never clamp (budget.rs:257-316).
  if (ctx->budget_limit && bytes <= ctx->budget_limit && ctx->budget_live > ctx->budget_limit - bytes) drop_extra(ctx);
  if (ctx->budget_limit && (bytes > ctx->budget_limit || ctx->budget_live > ctx->budget_limit - bytes))
    return omx_fail(ctx, OMX_CAPACITY_EXCEEDED, "requested %llu cap %llu live %llu", (unsigned long long)bytes,
                    (unsigned long long)ctx->budget_limit, (unsigned long long)ctx->budget_live);
  if (ctx->pool.size() >= kMaxSizes && ctx->pool.find(bytes) == ctx->pool.end())
    for (auto at = ctx->pool.begin(); at != ctx->pool.end();) at = at->second.blocks.empty() ? ctx->pool.erase(at) : std::next(at);
  OmxParked& parked = ctx->pool[bytes];
  parked.before = parked.last;
  parked.last = ++ctx->requests;
  void* p = nullptr;
  auto kept = ctx->for_graphs.find(bytes);
  if (kept != ctx->for_graphs.end() && capturing(ctx)) {
    p = kept->second.key();
    ctx->allocations.insert(std::move(kept->second));
    ctx->for_graphs.erase(kept);
  } else if (!parked.blocks.empty()) {
    // A block of this size freed earlier: every use of it is on this context's stream, so work
    // launched from here on is ordered after whatever still reads it.
    p = parked.blocks.back().key();
    ctx->allocations.insert(std::move(parked.blocks.back()));
    parked.blocks.pop_back();
    ctx->pooled_bytes -= bytes;
  } else {
    hipError_t err = hipMalloc(&p, bytes);
    if (err != hipSuccess && ctx->pooled_bytes) {
      // Out of device memory with blocks parked in the pool: give them back and try once more.
      (void)hipGetLastError();
      omx_release_pool(ctx);
      err = hipMalloc(&p, bytes);
    }
    if (err != hipSuccess && drop_extra(ctx)) {
      (void)hipGetLastError();
      err = hipMalloc(&p, bytes);
    }
    if (err != hipSuccess) return omx_hip_fail(ctx, err, "hipMalloc");
    ctx->allocations[p] = bytes;
  }
  ctx->budget_live += bytes;
  if (ctx->budget_live > ctx->budget_peak) ctx->budget_peak = ctx->budget_live;
  *out = p;
  return OMX_OK;
}

int32_t omx_free(omx_ctx* ctx, void* ptr) {
  OMX_REQUIRE_CTX(ctx);
  if (!ptr) return OMX_OK;
  auto it = ctx->allocations.find(ptr);
  if (it == ctx->allocations.end()) return omx_fail(ctx, OMX_PLACEMENT, "omx_free: pointer not from this context");
  const uint64_t bytes = it->second;
  // A sum that waits would be written over whatever gets this block next.
  const char* const from = static_cast<const char*>(ptr);
  const std::less<const char*> before;
  for (const OmxColumnSum& s : ctx->sums) {
    auto inside = [&](const void* p) { return p && !before(static_cast<const char*>(p), from) && before(static_cast<const char*>(p), from + bytes); };
    if (!inside(s.out) && !inside(s.blend)) continue;
    const int32_t rc = omx_form_sums(ctx);
    if (rc != OMX_OK) return rc;
    break;
  }
  ctx->budget_live -= bytes;
  // Freeing for real would wait for the stream (work that still reads the buffer is on it) and for
  // the whole device (hipFree). Blocks of moderate size are parked instead and handed out again by
  // omx_alloc to a request of the same size; reuse is safe without a wait because the next user's
  // work goes onto the same stream. The pool is not charged to the budget: the budget counts what
  // callers hold.
  if (capturing(ctx)) ctx->freed_in_capture.insert(ptr);
  if (ctx->freed_in_capture.count(ptr)) {
    // The graph writes this block whenever it is replayed, and nothing tells the context when that is over: never eager memory again,
    // and not the device's either. Captures after this one take it, so that recording a graph anew needs no more.
    ctx->for_graphs.emplace(bytes, ctx->allocations.extract(it));
    return OMX_OK;
  }
  if (bytes <= kMaxBlock) {
    OmxParked& parked = ctx->pool[bytes];
    if (ctx->pooled_bytes + bytes > kMaxPool) make_room(ctx, bytes, parked.before);
    if (ctx->pooled_bytes + bytes <= kMaxPool) {
      parked.blocks.push_back(ctx->allocations.extract(it));
      ctx->pooled_bytes += bytes;
      return OMX_OK;
    }
  }
  ctx->allocations.erase(it);
  OMX_HIP(ctx, hipStreamSynchronize(ctx->stream));
  OMX_HIP(ctx, hipFree(ptr));
  return OMX_OK;
}

uint64_t omx_budget_live(omx_ctx* ctx) { return ctx ? ctx->budget_live : 0; }
uint64_t omx_budget_peak(omx_ctx* ctx) { return ctx ? ctx->budget_peak : 0; }
uint64_t omx_budget_limit(omx_ctx* ctx) { return ctx ? ctx->budget_limit : 0; }
uint64_t omx_budget_pooled(omx_ctx* ctx) { return ctx ? ctx->pooled_bytes : 0; }
void omx_budget_reset_peak(omx_ctx* ctx) {
  if (ctx) ctx->budget_peak = ctx->budget_live;
}

int32_t omx_upload(omx_ctx* ctx, void* dst, uint64_t dst_offset, const void* host_src, uint64_t bytes) {
  OMX_REQUIRE_CTX(ctx);
  if (!dst || !host_src) return omx_fail(ctx, OMX_PLACEMENT, "upload: null pointer");
  if (bytes == 0) return OMX_OK;
  // Pageable source: the copy is staged, so the call returns once the source
  // has been read and the caller may reuse it.
  OMX_HIP(ctx, hipMemcpyAsync(static_cast<char*>(dst) + dst_offset, host_src, bytes, hipMemcpyHostToDevice,
                              ctx->stream));
  OMX_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return OMX_OK;
}

// For inputs that only work on this stream reads (a step's tokens): no wait. An upload and its wait were some 12 us in which a small
// model's step had not begun.
int32_t omx_upload_staged(omx_ctx* ctx, void* dst, uint64_t dst_offset, const void* host_src, uint64_t bytes) {
  OMX_REQUIRE_CTX(ctx);
  char* to = static_cast<char*>(dst) + dst_offset;
  if (!dst || !host_src || bytes == 0 || bytes > kStageMost || (reinterpret_cast<uintptr_t>(to) & 15u) || capturing(ctx) ||
      !own_range(ctx, to, bytes))
    return omx_upload(ctx, dst, dst_offset, host_src, bytes);
  if (!ctx->stage && hipHostMalloc(&ctx->stage, kStage) != hipSuccess) {
    (void)hipGetLastError();
    ctx->stage = nullptr;
    return omx_upload(ctx, dst, dst_offset, host_src, bytes);
  }
  if (ctx->staged + bytes > kStage) {
    const int32_t rc = wait(ctx);
    if (rc != OMX_OK) return rc;
  }
  char* from = ctx->stage + ctx->staged;
  memcpy(from, host_src, bytes);
  omx_launch(ctx, stage_kernel, dim3(static_cast<unsigned>((bytes + 4095) / 4096)), dim3(256), 0, from, to, static_cast<int>(bytes));
  OMX_LAUNCH_CHECK(ctx, "stage_kernel");
  ctx->staged += (bytes + 255) & ~255ull;
  return OMX_OK;
}

}  // extern "C"

namespace {
// Waits for submitted work and reports a deferred fault; with the fault word come `n` (at most kReadback) bytes of `src`, to readback().
// One launch and one wait: a copy of the fault word, a wait, a copy of the value and a wait were some 25 us between two halves of a step.
int32_t sync_with(omx_ctx* ctx, const void* src, uint64_t n) {
  const int32_t formed = omx_form_sums(ctx);
  if (formed != OMX_OK) return formed;
  omx_launch(ctx, read_back_kernel, dim3(1), dim3(256), 0, ctx->fault, ctx->fault_host, static_cast<const char*>(src), readback(ctx), static_cast<int>(n));
  OMX_LAUNCH_CHECK(ctx, "read_back_kernel");
  const int32_t waited = wait(ctx);
  if (waited != OMX_OK) return waited;
  if (ctx->fault_host->mask != 0) {
    uint32_t op = static_cast<uint32_t>(ctx->fault_host->first & 0x7full);
    bool range = (ctx->fault_host->first & 0x80ull) != 0;
    int32_t rc = reset_fault(ctx);
    if (rc != OMX_OK) return rc;
    if (range) return omx_fail(ctx, OMX_OUT_OF_RANGE, "%s: index outside its table", omx_fault_name(op));
    return omx_fail(ctx, OMX_NON_FINITE, "%s", omx_fault_name(op));
  }
  return OMX_OK;
}
}  // namespace

extern "C" {

int32_t omx_sync(omx_ctx* ctx) {
  OMX_REQUIRE_CTX(ctx);
  return sync_with(ctx, nullptr, 0);
}

int32_t omx_download(omx_ctx* ctx, void* host_dst, const void* src, uint64_t src_offset, uint64_t bytes) {
  OMX_REQUIRE_CTX(ctx);
  if (!host_dst || !src) return omx_fail(ctx, OMX_PLACEMENT, "download: null pointer");
  const char* from = static_cast<const char*>(src) + src_offset;
  const bool small = bytes <= kReadback && own_range(ctx, from, bytes);
  const int32_t rc = sync_with(ctx, from, small ? bytes : 0);
  if (rc != OMX_OK || bytes == 0) return rc;
  if (small) {
    memcpy(host_dst, readback(ctx), bytes);
    return OMX_OK;
  }
  OMX_HIP(ctx, hipMemcpyAsync(host_dst, from, bytes, hipMemcpyDeviceToHost, ctx->stream));
  OMX_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return OMX_OK;
}

int32_t omx_copy(omx_ctx* ctx, void* dst, const void* src, uint64_t bytes) {
  OMX_REQUIRE_CTX(ctx);
  if (bytes == 0) return OMX_OK;
  OMX_HIP(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, ctx->stream));
  return OMX_OK;
}

int32_t omx_read_scalar_f32(omx_ctx* ctx, const void* src, float* out) {
  return omx_download(ctx, out, src, 0, sizeof(float));
}

void* omx_stream(omx_ctx* ctx) { return ctx ? static_cast<void*>(ctx->stream) : nullptr; }

int32_t omx_unsupported(omx_ctx* ctx, const char* op) {
  return omx_fail(ctx, OMX_UNSUPPORTED, "%s", op ? op : "unknown op");
}

}  // extern "C"

namespace {
uint64_t workspace_size(uint64_t bytes) { return (bytes + (1ull << 20) - 1) & ~((1ull << 20) - 1); }
}  // namespace

bool omx_workspace_fits(const omx_ctx* ctx, uint64_t bytes, int slot) {
  const uint64_t held = ctx->workspace_bytes[slot];
  if (bytes <= held || ctx->budget_limit == 0) return true;
  uint64_t back = ctx->workspace_captured[slot] || capturing(ctx) ? 0 : held;  // what growing it gives back
  // An op's plan does not depend on what others can do without: omx_alloc takes that back for it.
  if (!can_do_without(slot))
    for (int extra : {kExtraSlot, kSumsSlot, kCopiesSlot})
      if (droppable(ctx, extra)) back += ctx->workspace_bytes[extra];
  return ctx->budget_live - back + workspace_size(bytes) <= ctx->budget_limit;
}

int32_t omx_workspace(omx_ctx* ctx, uint64_t bytes, void** out, int slot) {
  const bool in_graph = capturing(ctx);
  if (bytes <= ctx->workspace_bytes[slot]) {
    ctx->workspace_captured[slot] |= in_graph;
    *out = ctx->workspace[slot];
    return OMX_OK;
  }
  if (in_graph || ctx->workspace_captured[slot]) {
    // A captured graph holds the block's address for as long as it is replayed, which nothing tells the context: the block stays,
    // charged, until the context closes. (In a capture nothing can be waited for, so nothing is freed there either.)
    ctx->workspace[slot] = nullptr;
    ctx->workspace_bytes[slot] = 0;
  } else if (ctx->workspace[slot]) {
    // An outgrown workspace goes back to the driver, not into the pool: its size (a multiple of
    // 1 MiB that only this slot ever asked for) would match no later request and stay parked.
    auto it = ctx->allocations.find(ctx->workspace[slot]);
    if (it != ctx->allocations.end()) {
      ctx->budget_live -= it->second;
      ctx->allocations.erase(it);
    }
    OMX_HIP(ctx, hipStreamSynchronize(ctx->stream));
    OMX_HIP(ctx, hipFree(ctx->workspace[slot]));
    ctx->workspace[slot] = nullptr;
    ctx->workspace_bytes[slot] = 0;
  }
  const uint64_t rounded = workspace_size(bytes);
  int32_t rc = omx_alloc(ctx, rounded, &ctx->workspace[slot]);
  if (rc != OMX_OK) return rc;
  ctx->workspace_bytes[slot] = rounded;
  ctx->workspace_captured[slot] = in_graph;
  if (slot == kCopiesSlot) ++ctx->copies_generation;
  *out = ctx->workspace[slot];
  return OMX_OK;
}

void* omx_workspace_if_room(omx_ctx* ctx, uint64_t bytes, int slot) {
  if (bytes > ctx->workspace_bytes[slot] && (capturing(ctx) || !omx_workspace_fits(ctx, bytes, slot))) return nullptr;
  void* ws = nullptr;
  return omx_workspace(ctx, bytes, &ws, slot) == OMX_OK ? ws : nullptr;
}
