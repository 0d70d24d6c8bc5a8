// K/V tile primitives shared by the prefill and decode kernels that stage
// tiles in LDS: raw buffer resources, the LDS DMA, the swizzled tile layout with
// its transposing V read, and the row max of an S^T accumulator.
#pragma once

#include "fa_common.h"

namespace fa {

namespace {

constexpr uint32_t kRsrcWord3 = 0x00020000u;  // raw buffer, dword data format (gfx9)
constexpr float kRescaleLog2 = 8.f;

// v_max3_f32 without the canonicalising moves fmaxf adds for inputs the
// compiler cannot prove canonical (MFMA results): the hardware max already
// treats a quiet NaN input as missing, and no input here is a signalling NaN.
__device__ __forceinline__ float vmax3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// Max of 16 values as a depth-3 tree of max3 (six independent max3, then two,
// then one), instead of a dependent chain of eight.
__device__ __forceinline__ float max16(const floatx16& s) {
  const float a0 = vmax3(s[0], s[1], s[2]), a1 = vmax3(s[3], s[4], s[5]);
  const float a2 = vmax3(s[6], s[7], s[8]), a3 = vmax3(s[9], s[10], s[11]);
  const float a4 = vmax3(s[12], s[13], s[14]);
  const float b0 = vmax3(a0, a1, a2), b1 = vmax3(a3, a4, s[15]);
  return vmax3(b0, b1, b1);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes,
                                           (int)kRsrcWord3);
}

// One 16-byte-per-lane LDS DMA: M0 holds the wave's LDS destination, the
// lanes' rows land one after another from there. Issued as inline asm so the
// compiler does not track it: it puts an `s_waitcnt vmcnt(0)` in front of
// every ds_read_b64_tr_b16 that follows a DMA it knows of, which would make
// each wave wait for its next tile's DMA before reading V of the current one.
// Ordering is explicit instead: every DMA is waited for (vmcnt) before the
// barrier that precedes the reads of its stage. The `s_nop 0` is the wait
// state an LDS DMA needs after an SALU write of M0. NT sets the non-temporal
// cache policy, for K/V that no other workgroup reads.
template <bool NT>
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t r, void* lds, uint32_t voffset) {
  const uint32_t m0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  if constexpr (NT)
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen nt lds"
                 :: "v"(voffset), "s"(r), "{m0}"(m0) : "memory");
  else
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
                 :: "v"(voffset), "s"(r), "{m0}"(m0) : "memory");
}

// N LDS DMAs of one slab through one resource, each 1 KB further on in LDS. The
// resource may come from a register restore (v_readlane), and a VMEM
// instruction that reads an SGPR needs five wait states after a VALU write
// of it, which the compiler does not add for inline assembly: the leading
// s_nop has them.
template <int N>
__device__ __forceinline__ void lds_dma_slab(__amdgpu_buffer_rsrc_t r, void* lds, const uint32_t* v) {
  static_assert(N == 1 || N == 2 || N == 4, "slab sizes in use");
  uint32_t m0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  if constexpr (N == 1)
    asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds"
                 : "+{m0}"(m0) : "v"(v[0]), "s"(r) : "memory");
  else if constexpr (N == 2)
    asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %1, %3, 0 offen nt lds\n\t"
                 "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %2, %3, 0 offen nt lds"
                 : "+{m0}"(m0) : "v"(v[0]), "v"(v[1]), "s"(r) : "memory", "scc");
  else
    asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %1, %5, 0 offen nt lds\n\t"
                 "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %2, %5, 0 offen nt lds\n\t"
                 "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %3, %5, 0 offen nt lds\n\t"
                 "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %4, %5, 0 offen nt lds"
                 : "+{m0}"(m0) : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "s"(r) : "memory", "scc");
}

template <int D>
struct DmaCfg {
  static constexpr int ROWB = 2 * D;             // bytes per key row
  static constexpr int CH = D / 8;               // 16-byte chunks per row
  static constexpr int RPI = 1024 / ROWB;        // rows per wave-wide 16-byte load
  __device__ static int swz_k(int row) { return row % CH; }
  __device__ static int swz_v(int row) { return (4 * row) % CH; }
};

// V^T operand (8 keys of one d per lane) of PV step s, d block i, via two
// transposing reads; voff holds the lane's byte offset from `buf`.
template <int D>
__device__ __forceinline__ half8 ld_vt(const char* buf, const int* voff, int s, int i) {
  using C = DmaCfg<D>;
  const char* va = buf + voff[i] + 16 * s * C::ROWB;
  const half4 lo = __builtin_bit_cast(
      half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v*)(va)));
  const half4 hi = __builtin_bit_cast(
      half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                 (__attribute__((address_space(3))) short4v*)(va + 8 * C::ROWB)));
  return half8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

}  // namespace

}  // namespace fa
