// Device helpers shared by the attention kernels.
#pragma once
#include "yr_common.h"

namespace yr {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLazy = 8.f;  // running-max slack (log2 units)

// 4 consecutive 16-bit elements from LDS, transposed across each 16-lane group
// (an address-space cast, not a trip through an integer: the compiler keeps
// track of the LDS object and does not wait for direct loads into others)
__device__ __forceinline__ uint2 lds_tr4(const uint16_t* p) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)p));
}

// max over lanes l and l ^ 16 (l ^ 32): a permlane swap of the value with
// itself hands each 16-lane row its partner row, in registers (no LDS trip)
__device__ __forceinline__ float max_xor16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float max_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// 16 bytes per lane from global memory straight into LDS: lane l's data
// lands at lds_base + 16 l (lds_base wave-uniform)
__device__ __forceinline__ void lds_load16(const uint16_t* g, uint16_t* lds_base) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(g),
                                   reinterpret_cast<__attribute__((address_space(3))) void*>(
                                       reinterpret_cast<__attribute__((address_space(3))) char*>(
                                           reinterpret_cast<uintptr_t>(lds_base))),
                                   16, 0, 0);
}

}  // namespace yr
