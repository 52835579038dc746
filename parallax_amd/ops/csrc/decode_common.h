// What the decode attention kernels share.
#pragma once

#include "common.h"

typedef __bf16 bf16x2n __attribute__((ext_vector_type(2)));

namespace {

DEVINL uint32_t pack_bf16(float a, float b) {
  bf16x2n p;
  p[0] = (__bf16)a;
  p[1] = (__bf16)b;
  return __builtin_bit_cast(uint32_t, p);
}

// over the four lanes that hold one query head (l, l + 16, l + 32, l + 48)
template <class F>
DEVINL float over_head(float v, F f) {
  const auto a = __builtin_amdgcn_permlane16_swap(
      __float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

}  // namespace
