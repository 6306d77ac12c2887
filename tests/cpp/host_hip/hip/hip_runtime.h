// A stand-in for the HIP headers that lets dma_order.cpp run one lane of one wave of a kernel on the host, with its
// loads in flight as late as its waits allow. A wave's vector-memory operations retire in issue order: a direct
// global -> LDS load makes its bytes poison when it is issued and lands when a counted wait (or a younger operation's)
// covers it; a load to registers only takes its place in the order, and not even that where nothing reads what it loads (the
// compiler may drop it): past a segment's last whole turn of the register sets.
#pragma once
#include <math.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <deque>

#define __global__
#define __device__
#define __host__
#define __shared__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))
using std::max;
using std::min;

struct Idx {
  unsigned x = 0, y = 0, z = 0;
};
inline Idx threadIdx, blockIdx, gridDim;
typedef void* hipStream_t;
struct alignas(16) float4 {
  float x, y, z, w;
};
inline float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }
inline float __uint_as_float(uint32_t u) { return __builtin_bit_cast(float, u); }
inline uint32_t __float_as_uint(float f) { return __builtin_bit_cast(uint32_t, f); }
inline float __int_as_float(int u) { return __builtin_bit_cast(float, u); }
inline int __float_as_int(float f) { return __builtin_bit_cast(int, f); }
template <class T>
T __shfl_xor(T v, int, int) {
  return v;
}
inline void __syncthreads() {}

namespace emu {
constexpr uint32_t kPoison = 0xFFFFFFFFu, kTag = 0xA5000000u;  // bytes in flight; an activation group's bytes
struct Op {
  uint8_t* lds;  // null: a load to registers
  int bytes;
  uint32_t value;
};
inline std::deque<Op> queue;
inline const void* act = nullptr;  // the activations' address: their DMAs land as kTag | 64-group
inline long mfma = 0, bad = 0;
inline int per_unit = 1, units = 1, first = 0, step = 1;  // MFMAs of a unit, units of a segment, their 64-groups
inline int unread = 1;                                    // the first unit whose register loads nothing reads
inline void land() {
  const Op op = queue.front();
  queue.pop_front();
  for (int i = 0; op.lds && i < op.bytes; i += 4) memcpy(op.lds + i, &op.value, 4);
}
inline void wait(int n) {
  while ((int)queue.size() > n) land();
}
inline void dma(const void* base, uint8_t* lds, int bytes, uint32_t soff) {
  for (int i = 0; i < bytes; i += 4) memcpy(lds + i, &kPoison, 4);
  queue.push_back({lds, bytes, base == act ? kTag | soff / 128 : 0u});
}
inline int unit() { return (int)(mfma / per_unit % units); }
inline void reg_load() {
  if (unit() < unread) queue.push_back({});
}
inline void operand(const void* v) {
  uint32_t w[4];
  memcpy(w, v, 16);
  for (uint32_t x : w) {
    const bool nan = (x & 0x7F80u) == 0x7F80u || (x & 0x7F800000u) == 0x7F800000u;
    if (nan || (x >> 24 == kTag >> 24 && (x & 0xFFFFFFu) != (uint32_t)(first + step * unit()))) bad++;
  }
}
}  // namespace emu

struct __amdgpu_buffer_rsrc_t {
  const void* base;
};
typedef __attribute__((ext_vector_type(4))) uint32_t emu_u4;
typedef __attribute__((ext_vector_type(8))) __bf16 emu_bf8;
typedef __attribute__((ext_vector_type(16))) float emu_f16;
typedef __attribute__((ext_vector_type(4))) int32_t emu_i4;
typedef __attribute__((ext_vector_type(16))) int32_t emu_i16;
inline __amdgpu_buffer_rsrc_t __builtin_amdgcn_make_buffer_rsrc(void* p, int, int, int) { return {p}; }
inline void __builtin_amdgcn_raw_ptr_buffer_load_lds(__amdgpu_buffer_rsrc_t r, __attribute__((address_space(3))) void* l,
                                                     int size, int, int soff, int, int) {
  emu::dma(r.base, (uint8_t*)l, 64 * size, (uint32_t)soff);
}
inline void __builtin_amdgcn_global_load_lds(const void* g, __attribute__((address_space(3))) void* l, int size, int, int) {
  emu::dma(g, (uint8_t*)l, 64 * size, 0);
}
inline emu_u4 __builtin_amdgcn_raw_buffer_load_b128(__amdgpu_buffer_rsrc_t, int, int, int) {
  emu::reg_load();
  return emu_u4{0, 0, 0, 0};
}
inline uint32_t __builtin_amdgcn_raw_buffer_load_b32(__amdgpu_buffer_rsrc_t, int, int, int) {
  emu::reg_load();
  return 0;
}
inline emu_f16 __builtin_amdgcn_mfma_f32_32x32x16_bf16(emu_bf8 a, emu_bf8 b, emu_f16 c, int, int, int) {
  emu::operand(&a), emu::operand(&b), emu::mfma++;
  return c;
}
inline emu_i16 __builtin_amdgcn_mfma_i32_32x32x32_i8(emu_i4, emu_i4, emu_i16 c, int, int, int) { return c; }
template <class T>
T __builtin_amdgcn_readfirstlane(T v) {
  return v;
}
inline int __builtin_amdgcn_readlane(int v, int) { return v; }
inline int __builtin_amdgcn_update_dpp(int, int v, int, int, int, bool) { return v; }
inline uint32_t __builtin_amdgcn_perm(uint32_t, uint32_t b, uint32_t) { return b; }
inline emu_u4 __builtin_amdgcn_permlane32_swap(uint32_t a, uint32_t b, bool, bool) { return emu_u4{a, b, 0, 0}; }
inline void __builtin_amdgcn_sched_barrier(int) {}
inline void __builtin_amdgcn_sched_group_barrier(int, int, int) {}
