// What the expert kernels share.
#pragma once

#include "common.h"

typedef int i32x4v __attribute__((ext_vector_type(4)));
typedef int i32x8v __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2n __attribute__((ext_vector_type(2)));

namespace {

DEVINL uint32_t pack_bf16(float a, float b) {
  bf16x2n p;
  p[0] = (__bf16)a;
  p[1] = (__bf16)b;
  return __builtin_bit_cast(uint32_t, p);
}

// 16 bytes a lane from memory to LDS, at + 16 lane. In assembly, without a register
// of its own: of the builtin the compiler knows that it writes LDS, and where the
// places rotate it waits for every copy in flight once a loop's turn before it reads.
DEVINL void copy16(const void* src, uint32_t at) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :: "v"(src), "s"(at) : "m0", "memory");
}
// The same from a uniform base: no address arithmetic a lane.
DEVINL void copy16(const uint8_t* base, uint32_t off, uint32_t at) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(off), "s"(base), "s"(at) : "m0", "memory");
}

DEVINL uint32_t lds_address(const void* p) {
  return __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p);
}

// the gated activation of four features, one uniform branch for them
DEVINL void activate(float limit, int gelu, f32x4v g, f32x4v u, float (&v)[4]) {
  if (limit > 0.f) {  // gpt-oss clamped act
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float a = fminf(g[s], limit);
      const float b = fminf(fmaxf(u[s], -limit), limit);
      v[s] = (b + 1.f) * (a / (1.f + __expf(-a * 1.702f)));
    }
  } else if (gelu) {
    const float c = 0.7978845608028654f;
#pragma unroll
    for (int s = 0; s < 4; ++s)
      v[s] = 0.5f * g[s] *
             (1.f + tanhf(c * (g[s] + 0.044715f * g[s] * g[s] * g[s]))) * u[s];
  } else {
#pragma unroll
    for (int s = 0; s < 4; ++s) v[s] = g[s] / (1.f + __expf(-g[s])) * u[s];
  }
}

}  // namespace
