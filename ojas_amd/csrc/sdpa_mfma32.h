// f32 attention kernels on the f32 matrix instructions (sdpa_mfma32.hip), shared by causal SDPA and the KV-cache
// attention.
#pragma once

#include "omx_common.h"

// Tensors by element strides: batch, head and row (a row's dim values are adjacent). Forward: queries 0 .. tq - 1
// sit at key index q_pos0 + i of the tk keys that are read; key j is row (slot0 + j) mod capacity of k and v.
// Backward: self-attention (tq == tk, q_pos0 == slot0 == 0).
struct Sdpa32Args {
  const float* q;
  const void *k, *v;  // f32, or bf16 in the forward's cache form
  float* out;         // forward: written; dQ pass: read for the row term (null: read from `delta`)
  float* lse;         // [batch, heads, tq]; may be null in the forward
  const float* gy;    // strides of out
  float *gq, *gk, *gv;
  float* delta;       // [batch, heads, tq]
  float* parts;       // set by the backward itself
  // Forward over a cache with the keys split over workgroups: [batch, tq, heads][nparts][dim + 2], a part's unnormalised
  // output, its maximum (natural logarithm) and its sum; null: the output itself.
  float* partial;
  int nparts;
  long q_b, q_h, q_t, k_b, k_h, k_t, o_b, o_h, o_t;
  int kv_heads, rep, tq, tk, q_pos0, slot0, capacity, window;
  float scale;
  OmxFaultWord* fault;
  unsigned long long tag;
};

// Head dims 16 / 32 / 64 / 128, 16-byte aligned tensors and strides, at most 65535 (batch, KV head) planes.
bool omx_sdpa32_supports(uint64_t dim, uint64_t planes, std::initializer_list<const void*> ptrs, std::initializer_list<long> strides);
// Into how many parts the forward over a cache had better split each row's keys (1: none).
int omx_sdpa32_key_parts(omx_ctx* ctx, const Sdpa32Args& a, int batch, int dim, bool bf16_cache);
int32_t omx_sdpa32_forward(omx_ctx* ctx, const Sdpa32Args& a, int batch, int dim, bool bf16_cache);
int32_t omx_sdpa32_backward(omx_ctx* ctx, const Sdpa32Args& a, int batch, int dim);
