// What the backward kernels for head dims above 128 share (bwd_wide.hip, bwd_wide_pair.hip): the layout of a staged
// tile, its loads and its reads.
#pragma once

#include <utility>

#include "bwd_mfma.h"

namespace mi355 {

constexpr int DW = 256;           // the width the kernels are built for
constexpr int BT = 32;            // rows of a staged tile
constexpr int TILE_ELEMS = BT * DW;

typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 tr_read(const uint16_t* ptr) {
  const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(ptr));
  return __builtin_bit_cast(u32x2, v);
}

// raw buffer resource, in scalar registers
__device__ __forceinline__ u32x4 wide_descriptor(const void* base, int64_t bytes) {
  const uint64_t a = (uint64_t)base;
  return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
               (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu)),
               (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}
// (m0 holds the LDS address of such a load, one wait state after it is written)
__device__ __forceinline__ void wide_tile_load(const u32x4& rsrc, uint32_t voffset, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :: "s"(__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(voffset), "s"(rsrc) : "memory", "m0");
}
// byte offset of this lane's chunk of load `ld` inside a tile whose first row is the buffer's base
__device__ __forceinline__ uint32_t wide_chunk_off(int ld, int lane, int row_stride, int width) {
  const int pos = ld * 64 + lane, r = pos / (DW / 8), ch = (pos % (DW / 8)) ^ tile_swz<DW>(r);
  return ch * 8 < width ? (uint32_t)((r * row_stride + ch * 8) * 2) : 0xfffffff0u;
}

// compile-time loop: f(std::integral_constant<int, 0>{}) ... f(std::integral_constant<int, N - 1>{})
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// dK / dV at the full width without a bias or dropout (bwd_wide_pair.hip)
int launch_bwd_wide_pair(const BwdM& g, int dtype, hipStream_t s);

}  // namespace mi355
