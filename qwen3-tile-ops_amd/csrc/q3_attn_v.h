// P8.V of a 32-key block on the matrix cores, shared by the decode attention
// kernels (k_attn_decode.hip, k_attn_split.hip).
//
// A block's V rows go from memory straight into an LDS stage, [32 keys][8 x
// 16 B] with 16-byte chunk c of key r at position c ^ vswz(r), so that the
// 8 keys a transposing read gathers fall on 8 different chunks.
#pragma once

#include "q3_device.h"

namespace q3 {
namespace {

constexpr int HD = 128;

typedef int v4i_d __attribute__((ext_vector_type(4)));
typedef int v2i_d __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) v2i_d *lds_v2i_ptr_d;
__device__ __forceinline__ int vswz(int key) { return (key & 3) | ((key >> 2) & 4); }

// 16 bytes per lane global -> LDS (lane l writes lds + 16 l), as inline
// assembly: the compiler does not count it among the loads in flight, so
// its waits for later loads only become stricter (loads complete in
// order), while its own global_load_lds would make it wait for every load
// before the next use of any.  A copy is issued in front of loads whose
// wait then covers it.
// (NT: a non-temporal read, for rows read once that no prefetch brought in)
template <bool NT = false>
__device__ __forceinline__ void lds_copy16(const void *src, const void *lds) {
  const uint32_t m0v =
      __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(to_lds(lds))));
  if constexpr (NT)
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" ::"v"(src), "s"(m0v)
                 : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(m0v)
                 : "memory", "m0");
}

// Byte position of key c's P8 in a block's 32-byte P8 row, so that lane L's
// 8 bytes at 8 (L / 16) are the keys 16 (j / 4) + 4 (L / 16) + j % 4,
// j = 0..7: the keys ds_read_b64_tr_b8 hands lane L of the V operand (in
// each 16-lane group, result lane i byte j is byte i % 8 of the 8 bytes
// addressed by source lane 2 j + i / 8).
__device__ __forceinline__ int p8_pos(int c) { return 8 * ((c & 15) >> 2) + (((c >> 4) << 2) | (c & 3)); }

__device__ __forceinline__ int sdot4(int a, int b, int c) {
  return __builtin_amdgcn_sdot4(a, b, c, false);
}

}  // namespace
}  // namespace q3
