// Launch arguments shared by the GEMM kernels (gemm.hip, gemm_dma.hip).
#pragma once

#include "omx_common.h"

struct GemmArgs {
  const void* a;
  const void* b;
  void* c;
  long lda, ldb, ldc;
  int M, N, K;
  int k_rows;  // direct-to-LDS kernels: K is rounded up to whole steps, k-major operands end after k_rows rows
  int a_k;     // columns of a k-contiguous A's rows that may be read (zeros past K); K itself otherwise
  int c_bf16, accumulate;  // accumulate 2 (f32 output): C = epi_s1 * aux_in (as f32) + epi_s2 * A.B
  int a_vec, b_vec;  // 16-byte loads allowed (alignment of base and leading dimension)
  int c_vec;         // 4-column stores allowed (alignment of C and its row pitch)
  int tiles_m, tiles_n;
  int splits, ksteps_per_split;  // split-K: each split writes an f32 partial
  float* partial;                // [splits][M][N] when splits > 1
  int epi, epi_tanh;             // OMX_EPI_* (no split)
  const unsigned short* aux_in;  // of the output's type: f32 in disguise where that is
  unsigned short* aux_out;
  float epi_s1, epi_s2;  // OMX_EPI_AXPBY
  OmxFaultWord* fault;
  unsigned long long tag, act_tag;  // act_tag: of the f32 store pass's activation
  // bf16, A k-contiguous: C[m, n] += sum_p lr_h[m][off + p] lr_w[n][p] in the accumulators, p < lr_rank (a multiple of 16; 0:
  // none), off = n / lr_block_cols * lr_rank where lr_block_cols (a multiple of 32) is not 0. Pitches in elements.
  const unsigned short *lr_h, *lr_w;
  long lr_pitch, lr_w_pitch;
  int lr_rank, lr_block_cols;
  OmxRope rope;  // OMX_EPI_ROPE
  // Strided batch: block (x, y) works on product y, whose operands start batch_* BYTES after
  // product y - 1's. batches == 1 for a single product.
  int batches;
  int symmetric;  // C (bf16, square) equals its transpose: tiles below the diagonal are not formed but stored with those above
  long batch_a, batch_b, batch_c;
};

// Tiles of a symmetric output of `m` rows that are formed: those not wholly below the diagonal.
inline long omx_symmetric_tiles(long m, int bm, int bn) {
  long kept = 0;
  const long tiles_n = (m + bn - 1) / bn;
  for (long i = 0; i * bm < m; ++i) kept += tiles_n - i * bm / bn;
  return kept;
}
// Workgroups of a product of a batch.
inline long omx_gemm_tiles(const GemmArgs& g, int bm, int bn) {
  return g.symmetric ? omx_symmetric_tiles(g.M, bm, bn) : static_cast<long>(g.tiles_m) * g.tiles_n;
}

// The arguments of product `product` of a strided batch.
__device__ __forceinline__ void gemm_select_batch(GemmArgs& g, int product) {
  if (g.batches > 1) {
    const long y = product;
    g.a = static_cast<const char*>(g.a) + y * g.batch_a;
    g.b = static_cast<const char*>(g.b) + y * g.batch_b;
    g.c = static_cast<char*>(g.c) + y * g.batch_c;
    // A split product of a batch keeps its partial sums behind the earlier products'.
    if (g.splits > 1) g.partial += y * g.splits * static_cast<long>(g.M) * g.N;
    // aux tensors have the output's type and layout (f32 with a two-term sum, bf16 with the rest): the same byte stride.
    if (g.aux_in) g.aux_in = reinterpret_cast<const unsigned short*>(reinterpret_cast<const char*>(g.aux_in) + y * g.batch_c);
    if (g.aux_out) g.aux_out = reinterpret_cast<unsigned short*>(reinterpret_cast<char*>(g.aux_out) + y * g.batch_c);
  }
}

// What an accumulating f32 product stores: `old` is C's value, or aux_in's (accumulate 2).
__device__ __forceinline__ float gemm_add32(const GemmArgs& g, float old, float acc) {
  return g.accumulate == 2 ? g.epi_s1 * old + g.epi_s2 * acc : acc + old;
}

// Stores four consecutive columns of one output row (row `grow`, columns
// gcol..gcol+3, clipped to N): a split-K partial, a bf16 result, or an f32
// result with optional accumulation. Returns true when a stored value is
// non-finite (partials are checked by the reduce kernel instead).
__device__ __forceinline__ bool gemm_store4(const GemmArgs& g, int split, int grow, int gcol, float x0, float x1,
                                            float x2, float x3) {
  float x[4] = {x0, x1, x2, x3};
  bool bad = false;
  if (g.splits > 1) {
    float* part = g.partial + static_cast<long>(split) * g.M * g.N + static_cast<long>(grow) * g.N + gcol;
    if ((g.N & 3) == 0 && gcol + 4 <= g.N) {
      *reinterpret_cast<float4*>(part) = make_float4(x0, x1, x2, x3);
    } else {
      for (int e = 0; e < 4 && gcol + e < g.N; ++e) part[e] = x[e];
    }
    return false;
  }
  const long off = static_cast<long>(grow) * g.ldc + gcol;
  const bool whole = g.c_vec != 0 && gcol + 4 <= g.N;
  if (g.c_bf16) {
    unsigned short* cp = static_cast<unsigned short*>(g.c) + off;
    if (whole) {
      uint2 w;
      w.x = dev_pack_bf16_pair(x0, x1);
      w.y = dev_pack_bf16_pair(x2, x3);
      *reinterpret_cast<uint2*>(cp) = w;
      bad = !(dev_finite(x0) && dev_finite(x1) && dev_finite(x2) && dev_finite(x3));
    } else {
      for (int e = 0; e < 4 && gcol + e < g.N; ++e) {
        cp[e] = dev_f32_to_bf16_bits(x[e]);
        bad |= !dev_finite(x[e]);
      }
    }
  } else {
    float* cp = static_cast<float*>(g.c) + off;
    const float* ap = g.accumulate == 2 ? reinterpret_cast<const float*>(g.aux_in) + off : cp;
    if (whole) {
      if (g.accumulate) {
        const float4 old = *reinterpret_cast<const float4*>(ap);
        x[0] = gemm_add32(g, old.x, x[0]);
        x[1] = gemm_add32(g, old.y, x[1]);
        x[2] = gemm_add32(g, old.z, x[2]);
        x[3] = gemm_add32(g, old.w, x[3]);
      }
      *reinterpret_cast<float4*>(cp) = make_float4(x[0], x[1], x[2], x[3]);
      bad = !(dev_finite(x[0]) && dev_finite(x[1]) && dev_finite(x[2]) && dev_finite(x[3]));
    } else {
      for (int e = 0; e < 4 && gcol + e < g.N; ++e) {
        float y = g.accumulate ? gemm_add32(g, ap[e], x[e]) : x[e];
        cp[e] = y;
        bad |= !dev_finite(y);
      }
    }
  }
  return bad;
}

// The f32 product with its activation: C = the value and aux_out = GELU of it, or C = the value times GELU' of aux_in (f32 all, C's
// layout), as a pass of its own over the stored product would form them. Returns which is not finite: 1 the product, 2 the activation.
template <bool TANH>
__device__ __forceinline__ int gemm_store4_act32(const GemmArgs& g, int grow, int gcol, float x0, float x1, float x2, float x3) {
  const long off = static_cast<long>(grow) * g.ldc + gcol;
  float x[4] = {x0, x1, x2, x3};
  const int n = min(4, g.N - gcol);
  const bool whole = g.c_vec != 0 && n == 4;
  int bad = 0;
  if (g.epi == OMX_EPI_GELU_FWD) {
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[e] = dev_gelu_of<float, TANH>(x[e]);
      if (e < n && !dev_finite(y[e])) bad |= 2;
    }
    float* to = reinterpret_cast<float*>(g.aux_out) + off;
    if (whole) *reinterpret_cast<float4*>(to) = make_float4(y[0], y[1], y[2], y[3]);
    else
      for (int e = 0; e < n; ++e) to[e] = y[e];
    if (gemm_store4(g, 0, grow, gcol, x[0], x[1], x[2], x[3])) bad |= 1;
  } else {
    const float* u = reinterpret_cast<const float*>(g.aux_in) + off;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (whole) dev_load4<float>(u, 0, v);
    else
      for (int e = 0; e < n; ++e) v[e] = u[e];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (e < n && !dev_finite(x[e])) bad |= 1;
      x[e] = x[e] * dev_gelu_grad_of<float, TANH>(v[e]);
    }
    if (gemm_store4(g, 0, grow, gcol, x[0], x[1], x[2], x[3])) bad |= 2;
  }
  return bad;
}

// gemm_store4 with the optional activation of OmxGemmEpilogue applied first (bf16 outputs, no
// split). Kept apart from the plain store so the plain epilogue loops stay small enough to unroll.
// OMX_EPI_AXPBY on one element: `aux` as stored, `acc` the product's f32 accumulator.
__device__ __forceinline__ float gemm_axpby(const GemmArgs& g, float aux, float acc) {
  return dev_round_bf16(g.epi_s1 * aux) + dev_round_bf16(g.epi_s2 * dev_round_bf16(acc));
}

__device__ __forceinline__ bool gemm_store4_epi(const GemmArgs& g, int split, int grow, int gcol, float x0, float x1,
                                                float x2, float x3) {
  bool bad = false;
  const long off = static_cast<long>(grow) * g.ldc + gcol;
  const bool whole = g.c_vec != 0 && gcol + 4 <= g.N;
  {
    if (g.epi == OMX_EPI_GELU_FWD) {
      // The activation is taken of the value the pre-activation is stored as.
      const float u0 = dev_round_bf16(x0), u1 = dev_round_bf16(x1), u2 = dev_round_bf16(x2), u3 = dev_round_bf16(x3);
      const float a0 = g.epi_tanh ? dev_gelu_tanh_fast(u0) : dev_gelu_erf_fast(u0);
      const float a1 = g.epi_tanh ? dev_gelu_tanh_fast(u1) : dev_gelu_erf_fast(u1);
      const float a2 = g.epi_tanh ? dev_gelu_tanh_fast(u2) : dev_gelu_erf_fast(u2);
      const float a3 = g.epi_tanh ? dev_gelu_tanh_fast(u3) : dev_gelu_erf_fast(u3);
      unsigned short* ap = g.aux_out + off;
      if (whole) {
        uint2 w;
        w.x = dev_pack_bf16_pair(a0, a1);
        w.y = dev_pack_bf16_pair(a2, a3);
        *reinterpret_cast<uint2*>(ap) = w;
        bad = !(dev_finite(a0) && dev_finite(a1) && dev_finite(a2) && dev_finite(a3));
      } else {
        if (gcol + 0 < g.N) { ap[0] = dev_f32_to_bf16_bits(a0); bad |= !dev_finite(a0); }
        if (gcol + 1 < g.N) { ap[1] = dev_f32_to_bf16_bits(a1); bad |= !dev_finite(a1); }
        if (gcol + 2 < g.N) { ap[2] = dev_f32_to_bf16_bits(a2); bad |= !dev_finite(a2); }
        if (gcol + 3 < g.N) { ap[3] = dev_f32_to_bf16_bits(a3); bad |= !dev_finite(a3); }
      }
    } else if (g.epi == OMX_EPI_GELU_BWD || g.epi == OMX_EPI_AXPBY) {
      const unsigned short* ap = g.aux_in + off;
      float u0 = 0.0f, u1 = 0.0f, u2 = 0.0f, u3 = 0.0f;
      if (whole) {
        const uint2 w = *reinterpret_cast<const uint2*>(ap);
        u0 = __uint_as_float(w.x << 16);
        u1 = __uint_as_float(w.x & 0xffff0000u);
        u2 = __uint_as_float(w.y << 16);
        u3 = __uint_as_float(w.y & 0xffff0000u);
      } else {
        if (gcol + 0 < g.N) u0 = dev_bf16_bits_to_f32(ap[0]);
        if (gcol + 1 < g.N) u1 = dev_bf16_bits_to_f32(ap[1]);
        if (gcol + 2 < g.N) u2 = dev_bf16_bits_to_f32(ap[2]);
        if (gcol + 3 < g.N) u3 = dev_bf16_bits_to_f32(ap[3]);
      }
      if (g.epi == OMX_EPI_AXPBY) {
        x0 = gemm_axpby(g, u0, x0);
        x1 = gemm_axpby(g, u1, x1);
        x2 = gemm_axpby(g, u2, x2);
        x3 = gemm_axpby(g, u3, x3);
      } else {
        x0 = dev_round_bf16(x0) * (g.epi_tanh ? dev_gelu_tanh_grad_fast(u0) : dev_gelu_erf_grad_fast(u0));
        x1 = dev_round_bf16(x1) * (g.epi_tanh ? dev_gelu_tanh_grad_fast(u1) : dev_gelu_erf_grad_fast(u1));
        x2 = dev_round_bf16(x2) * (g.epi_tanh ? dev_gelu_tanh_grad_fast(u2) : dev_gelu_erf_grad_fast(u2));
        x3 = dev_round_bf16(x3) * (g.epi_tanh ? dev_gelu_tanh_grad_fast(u3) : dev_gelu_erf_grad_fast(u3));
      }
    }
  }
  return gemm_store4(g, split, grow, gcol, x0, x1, x2, x3) || bad;
}

// The activation epilogue for a 32-row block of a wave's tile that lies wholly inside the output
// (16-byte stores allowed): `staged` holds the block's f32 values, `pitch` floats per row,
// PPR 4-column pieces per row. One straight-line body per piece (the form of the activation is
// a template argument, the bounds are known), all of the backward's pre-activation loads issued
// ahead of the arithmetic. Returns true when a stored value is non-finite.
template <int EPI, bool TANH, int PPR>
__device__ __forceinline__ bool gemm_epilogue_block(const GemmArgs& g, const float* staged, int pitch, int grow0,
                                                    int gcol0, int lane) {
  constexpr int ITERS = 32 * PPR / 64;
  unsigned short* cbase = static_cast<unsigned short*>(g.c);
  // Non-finite values are found in the packed words that get stored: a bf16 is infinite or NaN
  // when its eight exponent bits are all set, and adding one at the exponent's lowest bit then
  // carries into the half's top bit. (GELU of a finite value is finite, so the forward tests the
  // pre-activation words only.)
  unsigned int flags = 0;
  auto note = [&](unsigned int w) { flags |= (w & 0x7F807F80u) + 0x00800080u; };
  long off[ITERS];
  uint2 aux[ITERS];
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = lane + it * 64, row = c / PPR, piece = c % PPR;
    off[it] = static_cast<long>(grow0 + row) * g.ldc + gcol0 + piece * 4;
    if constexpr (EPI != OMX_EPI_GELU_FWD) aux[it] = *reinterpret_cast<const uint2*>(g.aux_in + off[it]);
  }
  auto pack = [](float a, float b) {
    return dev_pack_bf16_pair(a, b);
  };
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = lane + it * 64, row = c / PPR, piece = c % PPR;
    const float4 val = *reinterpret_cast<const float4*>(staged + row * pitch + piece * 4);
    float x[4] = {val.x, val.y, val.z, val.w};
    if constexpr (EPI == OMX_EPI_GELU_FWD) {
      // The activation is taken of the value the pre-activation is stored as: one conversion per
      // pair gives both the stored word and, widened again, the activation's argument.
      const unsigned int w01 = pack(x[0], x[1]), w23 = pack(x[2], x[3]);
      const float u[4] = {__uint_as_float(w01 << 16), __uint_as_float(w01 & 0xffff0000u), __uint_as_float(w23 << 16),
                          __uint_as_float(w23 & 0xffff0000u)};
      float a[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = TANH ? dev_gelu_tanh_fast(u[e]) : dev_gelu_erf_fast(u[e]);
      note(w01);
      note(w23);
      *reinterpret_cast<uint2*>(cbase + off[it]) = make_uint2(w01, w23);
      *reinterpret_cast<uint2*>(g.aux_out + off[it]) = make_uint2(pack(a[0], a[1]), pack(a[2], a[3]));
    } else {
      const float u[4] = {__uint_as_float(aux[it].x << 16), __uint_as_float(aux[it].x & 0xffff0000u),
                          __uint_as_float(aux[it].y << 16), __uint_as_float(aux[it].y & 0xffff0000u)};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (EPI == OMX_EPI_AXPBY) x[e] = gemm_axpby(g, u[e], x[e]);
        else x[e] = dev_round_bf16(x[e]) * (TANH ? dev_gelu_tanh_grad_fast(u[e]) : dev_gelu_erf_grad_fast(u[e]));
      }
      const unsigned int w01 = pack(x[0], x[1]), w23 = pack(x[2], x[3]);
      note(w01);
      note(w23);
      *reinterpret_cast<uint2*>(cbase + off[it]) = make_uint2(w01, w23);
    }
  }
  return (flags & 0x80008000u) != 0;
}

// The transpose of a 32-row block of a symmetric output, COLS columns wide (bf16; plain or OMX_EPI_AXPBY, whose aux_in is
// symmetric too): row gcol0 + i takes the staged column i, 64 contiguous bytes. The bits of the block itself, whose
// non-finite values its own store has found.
template <int EPI, int COLS>
__device__ __forceinline__ void gemm_store_mirrored(const GemmArgs& g, const float* staged, int pitch, int grow0, int gcol0, int lane) {
  constexpr int ITERS = COLS * 8 / 64;
  unsigned short* cbase = static_cast<unsigned short*>(g.c);
  const bool interior = grow0 + 32 <= g.M && gcol0 + COLS <= g.N && g.c_vec != 0;
  if (interior) {
    long off[ITERS];
    uint2 aux[ITERS];
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int c = lane + it * 64, row = c >> 3, piece = c & 7;
      off[it] = static_cast<long>(gcol0 + row) * g.ldc + grow0 + piece * 4;
      if constexpr (EPI == OMX_EPI_AXPBY) aux[it] = *reinterpret_cast<const uint2*>(g.aux_in + off[it]);
    }
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int c = lane + it * 64, row = c >> 3, piece = c & 7;
      float x[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = staged[(piece * 4 + e) * pitch + row];
      if constexpr (EPI == OMX_EPI_AXPBY) {
        x[0] = gemm_axpby(g, __uint_as_float(aux[it].x << 16), x[0]);
        x[1] = gemm_axpby(g, __uint_as_float(aux[it].x & 0xffff0000u), x[1]);
        x[2] = gemm_axpby(g, __uint_as_float(aux[it].y << 16), x[2]);
        x[3] = gemm_axpby(g, __uint_as_float(aux[it].y & 0xffff0000u), x[3]);
      }
      *reinterpret_cast<uint2*>(cbase + off[it]) = make_uint2(dev_pack_bf16_pair(x[0], x[1]), dev_pack_bf16_pair(x[2], x[3]));
    }
    return;
  }
#pragma unroll 1
  for (int c = lane; c < COLS * 8; c += 64) {
    const int row = c >> 3, piece = c & 7, grow = gcol0 + row, gcol = grow0 + piece * 4;
    if (grow >= g.M || gcol >= g.N) continue;
    const float* x = staged + piece * 4 * pitch + row;
    if constexpr (EPI == OMX_EPI_AXPBY) gemm_store4_epi(g, 0, grow, gcol, x[0], x[pitch], x[2 * pitch], x[3 * pitch]);
    else gemm_store4(g, 0, grow, gcol, x[0], x[pitch], x[2 * pitch], x[3 * pitch]);
  }
}

// The plain store of a 32-row block that lies wholly inside the output, in the same straight-line
// form. KIND 0: f32 split-K partial; 1: bf16 result; 2: f32 result; 3: f32 result added to the
// stored one.
template <int KIND, int PPR>
__device__ __forceinline__ bool gemm_store_block(const GemmArgs& g, int split, const float* staged, int pitch,
                                                 int grow0, int gcol0, int lane) {
  constexpr int ITERS = 32 * PPR / 64;
  bool bad = false;
  const long ld = KIND == 0 ? g.N : g.ldc;
  float* fbase = KIND == 0 ? g.partial + static_cast<long>(split) * g.M * g.N : static_cast<float*>(g.c);
  unsigned short* hbase = static_cast<unsigned short*>(g.c);
  float4 old[ITERS];
  if constexpr (KIND == 3) {
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int c = lane + it * 64, row = c / PPR, piece = c % PPR;
      old[it] = *reinterpret_cast<const float4*>(fbase + static_cast<long>(grow0 + row) * ld + gcol0 + piece * 4);
    }
  }
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = lane + it * 64, row = c / PPR, piece = c % PPR;
    const long off = static_cast<long>(grow0 + row) * ld + gcol0 + piece * 4;
    float4 val = *reinterpret_cast<const float4*>(staged + row * pitch + piece * 4);
    if constexpr (KIND == 3) {
      val.x += old[it].x;
      val.y += old[it].y;
      val.z += old[it].z;
      val.w += old[it].w;
    }
    if constexpr (KIND == 1) {
      uint2 w;
      w.x = dev_pack_bf16_pair(val.x, val.y);
      w.y = dev_pack_bf16_pair(val.z, val.w);
      *reinterpret_cast<uint2*>(hbase + off) = w;
    } else {
      *reinterpret_cast<float4*>(fbase + off) = val;
    }
    // Partials are checked by the reduce kernel.
    if constexpr (KIND != 0) bad |= !(dev_finite(val.x) && dev_finite(val.y) && dev_finite(val.z) && dev_finite(val.w));
  }
  return bad;
}

// bf16 kernels with direct-to-LDS loads and a 256 x 256 (variant 9), 256 x 128 (variant 3) or
// 128 x 128 (variant 6) workgroup tile. Needs 16-byte aligned operands, and whole K steps in the
// rows of k-contiguous ones.
bool omx_gemm_dma_eligible(const GemmArgs& g, bool a_km, bool b_km, bool plain);
bool omx_gemm_w4_eligible(const GemmArgs& g, bool a_km, bool b_km, bool plain);
void omx_gemm_dma_tile(int variant, int* bm, int* bn);
int32_t omx_gemm_dma_launch(omx_ctx* ctx, const GemmArgs& g, bool a_km, bool b_km, int variant);

// bf16 kernel for outputs of at most 64 columns over at least 1024 rows of a k-contiguous A
// (K a multiple of 128, no accumulation): one pass over A, no split-K reduce.
bool omx_gemm_thin_eligible(const GemmArgs& g, bool a_km, bool b_km);
int32_t omx_gemm_thin_launch(omx_ctx* ctx, const GemmArgs& g, bool b_km);

// bf16 kernel for outputs of at most 16 rows from two k-major operands, A's pitch any (no accumulation).
bool omx_gemm_heads_eligible(const GemmArgs& g, bool a_km, bool b_km);
int omx_gemm_heads_splits(const GemmArgs& g);
int32_t omx_gemm_heads_launch(omx_ctx* ctx, const GemmArgs& g);

// bf16 kernel for products of few rows or few outputs, both operands k-contiguous, K a multiple of 32.
double omx_gemm_skinny_us(omx_ctx* ctx, const GemmArgs& g, bool a_km, bool b_km, bool activation);
int32_t omx_gemm_skinny_launch(omx_ctx* ctx, const GemmArgs& g);
// The same on 64 columns a workgroup, B in either layout (k-major: N a multiple of 8; else K of 64); `mb`: 16-row blocks of a workgroup.
double omx_gemm_skinny64_us(omx_ctx* ctx, const GemmArgs& g, bool a_km, bool b_km, int* mb);
int32_t omx_gemm_skinny64_launch(omx_ctx* ctx, const GemmArgs& g, bool b_km, int mb);

// f32 kernels: small outputs (gemm_frag32.hip) and direct-to-LDS loads (gemm_dma32.hip; g.K counts whole 32-column steps).
// `_us`: what a tile is estimated to take; negative: not one for it.
constexpr int FRAG32_TILES = 5, DMA32_TILES = 4;
constexpr int FRAG32_EIGHT_WAVES = 4;  // tiles below this one share K between eight waves: the same sums in all
// x: A k-contiguous, B k-major; w: both k-major. Estimate of a call of both (< 0: the tile does not fit), launch.
constexpr int FRAG32_PAIRS = 4;
double omx_gemm_frag32_pair_us(omx_ctx* ctx, const GemmArgs& x, const GemmArgs& w, int tile);
int32_t omx_gemm_frag32_pair(omx_ctx* ctx, const GemmArgs& x, const GemmArgs& w, int tile);
int32_t omx_gemm_dma32_pair(omx_ctx* ctx, const GemmArgs& x, const GemmArgs& w, int dma32);
double omx_gemm_frag32_us(omx_ctx* ctx, const GemmArgs& g, bool a_km, bool b_km, int tile);
int32_t omx_gemm_frag32_launch(omx_ctx* ctx, const GemmArgs& g, bool a_km, bool b_km, int tile);
// Independent f32 products C = A.B, or s1 aux + s2 A.B where `aux` is set (C's layout), in one launch; strides in elements, as
// omx_gemm_impl's; `stride`: between the `batches` products of a strided batch, of every operand. `symmetric`: every C equals its
// transpose.
struct OmxGemmProduct {
  const float* a;
  uint64_t a_rs, a_cs;
  const float* b;
  uint64_t b_rs, b_cs;
  float* c;
  uint64_t ldc, m, k, n;
  const float* aux;
  uint64_t batches, stride;
};
constexpr int FRAG32_GROUP = 8;
int32_t omx_gemm_frag32_group(omx_ctx* ctx, const OmxGemmProduct* products, int count, bool symmetric, float s1, float s2, unsigned long long tag);
bool omx_gemm_dma32_eligible(const GemmArgs& g, bool a_km, bool b_km);
double omx_gemm_dma32_us(omx_ctx* ctx, const GemmArgs& g, int tile);
void omx_gemm_dma32_tile(int tile, int* bm, int* bn);
int32_t omx_gemm_dma32_launch(omx_ctx* ctx, const GemmArgs& g, bool a_km, bool b_km, int tile);
