// Device helpers shared by the GEMM kernels' epilogues: SwiGLU with the
// staged exp2 table, the destination of an int8 head row (dense rows or a
// paged K/V slot), and a compile-time loop.
#pragma once

#include <type_traits>
#include <utility>

#include "q3_device.h"
#include "q3_kernels.h"

namespace q3 {

// ref_qwen3.py:194-200: e = exp(-g); e = e + 1; e = 1/e; out = (g * e) * u
// (exp table staged in LDS by stage_exp2_table).
__device__ __forceinline__ float swiglu_tab(float g, float u, const uint64_t *tab) {
  float e = __fmul_rn(g, -1.0f);
  e = exp_f32_tab(e, tab);
  e = __fadd_rn(e, 1.0f);
  e = __fdiv_rn(1.0f, e);
  return __fmul_rn(__fmul_rn(g, e), u);
}

// swiglu_tab of N (gate, up) pairs with exp2f_fast and the Newton reciprocal:
// the same values with two thirds of the instructions.  A wave that holds
// exp(-g) + 1 >= 2^126 (or a NaN) divides.
template <int N>
__device__ __forceinline__ void swiglu_n(const float (&g)[N], const float (&u)[N], float (&out)[N],
                                         const uint64_t *tab) {
  float e[N], top = 0.0f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    float x2 = __fmul_rn(__fmul_rn(g[i], -1.0f), bits_f32(0x3FB8AA3Bu));
    x2 = __builtin_elementwise_minimum(__builtin_elementwise_maximum(x2, -151.0f), 200.0f);
    e[i] = __fadd_rn(exp2f_fast(x2, tab), 1.0f);
    top = __builtin_elementwise_maximum(top, e[i]);
  }
  if (__builtin_amdgcn_ballot_w64(!(top < 0x1p+126f)) == 0) {
#pragma unroll
    for (int i = 0; i < N; ++i) out[i] = __fmul_rn(__fmul_rn(g[i], rcp_ge1(e[i])), u[i]);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) out[i] = __fmul_rn(__fmul_rn(g[i], __fdiv_rn(1.0f, e[i])), u[i]);
  }
}

// ---- row epilogues over four rows per wave -------------------------------
// A row of the f32 tile in LDS is held by 16 lanes, lane q of them with
// columns 4 q + 64 i .. + 3, so that a row's scalar work (norm factor, f64
// reciprocal of the scale, reductions) is done once per four rows and wave
// instead of once per row and wave, 16-byte LDS reads hit every bank once,
// and the int8 results leave as words.

__device__ __forceinline__ float row16_max(float m) {
  m = fmaxf(m, lane_xor<1>(m));
  m = fmaxf(m, lane_xor<2>(m));
  m = fmaxf(m, lane_xor<4>(m));
  return fmaxf(m, lane_xor<8>(m));
}

// int8 of 4 values with y = rcp64(scale), packed
__device__ __forceinline__ uint32_t quant4(const float *v, double y) {
  const uint32_t b0 = static_cast<uint32_t>(quant_rcp(v[0], y)), b1 = static_cast<uint32_t>(quant_rcp(v[1], y));
  const uint32_t b2 = static_cast<uint32_t>(quant_rcp(v[2], y)), b3 = static_cast<uint32_t>(quant_rcp(v[3], y));
  return __builtin_amdgcn_perm(__builtin_amdgcn_perm(b3, b2, 0x0c0c0400u), __builtin_amdgcn_perm(b1, b0, 0x0c0c0400u),
                               0x05040100u);
}

// 4 packed bytes to p (a destination row may have any alignment)
__device__ __forceinline__ void store4(int8_t *p, uint32_t w) {
  if ((reinterpret_cast<uintptr_t>(p) & 3) == 0) {
    *reinterpret_cast<uint32_t *>(p) = w;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = static_cast<int8_t>(w >> (8 * i));
  }
}

// The 4 floats p[0], p[st], p[2 st], p[3 st]; one load when vec (dense and
// 16-byte aligned)
__device__ __forceinline__ void load4(const float *p, int64_t st, bool vec, float *v) {
  if (vec) {
    const float4 x = *reinterpret_cast<const float4 *>(p);
    v[0] = x.x;
    v[1] = x.y;
    v[2] = x.z;
    v[3] = x.w;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = p[i * st];
  }
}

// Operands of a 128-column head row's lane q: gains of its 8 columns, RoPE
// factors of columns 4 q .. 4 q + 3 (shared by both halves).
struct HeadOps {
  float w[8], c[4], s[4];
};

// The head epilogue (group_gemm.h:173-193 / norm_rope_quant.h:17-86) of the
// row whose columns 4 q .. and 64 + 4 q .. the lane holds in t[0..3], t[4..7]
// (16 lanes a row): norm + RoPE (norm), then int8.
__device__ __forceinline__ void head_row16(float (&t)[8], bool norm, const HeadOps &o, float inv_hd, float *scale,
                                           uint32_t (&q8)[2]) {
  if (norm) {
    float b[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // 32-column blocks: 8 lanes, adjacent pairs first
      const float *x = t + 4 * h;
      float p = __fadd_rn(__fadd_rn(__fmul_rn(x[0], x[0]), __fmul_rn(x[1], x[1])),
                          __fadd_rn(__fmul_rn(x[2], x[2]), __fmul_rn(x[3], x[3])));
      p = __fadd_rn(p, lane_xor<1>(p));
      p = __fadd_rn(p, lane_xor<2>(p));
      b[h] = __fadd_rn(p, lane_xor<4>(p));
    }
    float ss = __fadd_rn(0.0f, row_bcast<0>(b[0]));
    ss = __fadd_rn(ss, row_bcast<8>(b[0]));
    ss = __fadd_rn(ss, row_bcast<0>(b[1]));
    ss = __fadd_rn(ss, row_bcast<8>(b[1]));
    const float rinv = rms_factor(ss, inv_hd);
#pragma unroll
    for (int i = 0; i < 8; ++i) t[i] = __fmul_rn(__fmul_rn(t[i], rinv), o.w[i]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float y0 = t[i], y1 = t[4 + i];
      t[i] = __fsub_rn(__fmul_rn(y0, o.c[i]), __fmul_rn(y1, o.s[i]));
      t[4 + i] = __fadd_rn(__fmul_rn(y0, o.s[i]), __fmul_rn(y1, o.c[i]));
    }
  }
  float m = fabsf(t[0]);
#pragma unroll
  for (int i = 1; i < 8; ++i) m = fmaxf(m, fabsf(t[i]));
  *scale = __fmul_rn(row16_max(m), inv127());
  const double y = rcp64(*scale);
  q8[0] = quant4(t, y);
  q8[1] = quant4(t + 4, y);
}

// swiglu_quant.h:195-231: per-256-column absmax * (1/127) and int8 of the
// tile row at src (16 lanes a row) into dst / *scale.
__device__ __forceinline__ void quant256_row16(const float *src, int q, bool store, int8_t *dst, float *scale) {
  float v[4][4], m = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    load4(src + 64 * i + 4 * q, 1, true, v[i]);
#pragma unroll
    for (int e = 0; e < 4; ++e) m = fmaxf(m, fabsf(v[i][e]));
  }
  const float sc = __fmul_rn(row16_max(m), inv127());
  const double y = rcp64(sc);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = quant4(v[i], y);
    if (store) store4(dst + 64 * i + 4 * q, w);
  }
  if (store && q == 0) *scale = sc;
}

// Slot pointers of token position t in page `page` of a paged K/V pool,
// head `head`.
__device__ __forceinline__ void qdest_slot(const QDest &d, uint32_t page, uint32_t t, int head, int8_t **row8,
                                           float **scale) {
  const uint32_t slot = t % d.page_tokens;
  *row8 = d.q8 + page * d.page_bytes + slot * d.row_bytes + head * 128;
  *scale = reinterpret_cast<float *>(reinterpret_cast<int8_t *>(d.qs) + page * d.scale_page_bytes +
                                     slot * d.scale_row_bytes) + head;
}

// Row destination of the int8 head output of row m, head `head`: a dense
// [rows][heads * 128] view, or the page slot of token pos0 + m (or
// row_pos[m] through that row's own table) of a paged K/V pool.
__device__ __forceinline__ void qdest_row(const QDest &d, int m, int head, int8_t **row8, float **scale) {
  if (d.table || d.row_pos) {
    uint32_t t = d.pos0 + static_cast<uint32_t>(m);
    if (d.pos_dev) t += static_cast<uint32_t>(*d.pos_dev);
    const uint16_t *table = d.table;
    if (d.row_pos) {
      t = static_cast<uint32_t>(d.row_pos[m]);
      table = d.row_tables + m * d.ld_table;
    }
    qdest_slot(d, table[t / d.page_tokens], t, head, row8, scale);
  } else {
    *row8 = d.q8 + static_cast<int64_t>(m) * d.ldq8 + head * 128;
    *scale = d.qs + static_cast<int64_t>(m) * d.ldqs + head * d.qs_col;
  }
}

// f(std::integral_constant<int, 0>{}), ..., f(std::integral_constant<int, N - 1>{})
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

}  // namespace q3
