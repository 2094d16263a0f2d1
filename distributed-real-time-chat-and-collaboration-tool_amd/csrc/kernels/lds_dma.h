// Loads from memory straight into LDS, with waits that count them (gfx950).  A wave's loads land in the
// order in which it issued them; stores in between only make a wait longer.
#pragma once
#include "common.h"

namespace drtc {

typedef __attribute__((address_space(3))) void* lds_ptr;
constexpr unsigned kNoRow = 0x80000000u;  // an offset past every descriptor's range: zeros, no memory access

DRTC_DEVICE __amdgpu_buffer_rsrc_t dma_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, 0x7FFFFFFF, 0x00020000);
}
// At most N of the wave's loads and stores are still under way.
template <int N>
DRTC_DEVICE void wait_vm() {
  constexpr int imm = (N & 0xF) | (0x7 << 4) | (0xF << 8) | ((N >> 4) << 14);
  __builtin_amdgcn_s_waitcnt(imm);
}
// All but the ``younger`` last groups of D loads have landed; younger <= Y.
template <int D, int Y>
DRTC_DEVICE void wait_groups(int younger) {
  if constexpr (Y == 0) {
    wait_vm<0>();
  } else {
    if (younger >= Y) wait_vm<Y * D>();
    else wait_groups<D, Y - 1>(younger);
  }
}
// 16 bytes a lane from base + voff + soff to dst + 16 lane; NT: non-temporal, for what is read once.
template <bool NT>
DRTC_DEVICE void dma16(unsigned dst, unsigned voff, __amdgpu_buffer_rsrc_t rsrc, unsigned soff) {
  unsigned keep;
  if constexpr (NT)
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\t"
        "buffer_load_dwordx4 %2, %3, %4 offen nt lds\n\ts_mov_b32 m0, %0"
        : "=&s"(keep)
        : "s"(dst), "v"(voff), "s"(rsrc), "s"(soff)
        : "memory");
  else
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\t"
        "buffer_load_dwordx4 %2, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
        : "=&s"(keep)
        : "s"(dst), "v"(voff), "s"(rsrc), "s"(soff)
        : "memory");
}

}  // namespace drtc
