// Shared pieces of the quantizer kernels: 16-byte element loads and a division by a shared scale.
#pragma once

#include "sqx_common.h"

namespace sqx {

// Eight consecutive elements (fp32 / bf16 / fp16) from a 16-byte aligned element index as fp32.
__device__ inline void load8_f32(const void* p, int dtype, int64_t e0, float (&v)[8]) {
  if (dtype == SQX_DTYPE_F32) {
    const u32x4_t* q = reinterpret_cast<const u32x4_t*>(static_cast<const float*>(p) + e0);
    const u32x4_t a = q[0], b = q[1];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t x = a[j], y = b[j];  // through scalars: hipcc's bit_cast of a vector element reads element 0
      v[j] = __builtin_bit_cast(float, x);
      v[4 + j] = __builtin_bit_cast(float, y);
    }
  } else {
    const u32x4_t a = *reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(p) + e0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t x = a[j];
      v[2 * j] = dtype == SQX_DTYPE_BF16 ? bf16_lo(x) : f16_bits_to_f32(static_cast<uint16_t>(x));
      v[2 * j + 1] = dtype == SQX_DTYPE_BF16 ? bf16_hi(x) : f16_bits_to_f32(static_cast<uint16_t>(x >> 16));
    }
  }
}

// v / s correctly rounded, for many v and one s, in three operations instead of the dozen of an IEEE fp32
// division: with r = RN(1/s), q = RN(v r) is within an ulp of v / s, the residual fma(-q, s, v) is exact, and
// RN(q + residual r) is the correctly rounded quotient (Markstein, "Computation of elementary functions on the
// IBM RISC System/6000 processor", 1990; compared with the division on the CPU for every 16-bit mantissa of v against
// every s, and on 1.2e10 fp32 pairs). The scale's range keeps q and the residual of every quotient of
// magnitude 2**-20 .. 2**100 away from underflow and overflow; smaller quotients may be off in their last place
// (and a zero loses its sign), which no code of these quantizers sees. Outside it, and for v that are not
// finite or huge, the division itself.
struct SharedDiv {
  float s, r;
  bool ok;
};
__device__ inline SharedDiv shared_div(float s) {
  return SharedDiv{s, __fdiv_rn(1.0f, s), s >= 0x1p-60f && s <= 0x1p60f};
}
__device__ inline bool fast_div(const SharedDiv& d, float v) { return d.ok && fabsf(v) <= 0x1p60f; }
__device__ inline float quick_div(const SharedDiv& d, float v) {  // where fast_div
  const float q = v * d.r;
  return fmaf(fmaf(-q, d.s, v), d.r, q);
}
__device__ inline float div_by(const SharedDiv& d, float v) {
  return fast_div(d, v) ? quick_div(d, v) : __fdiv_rn(v, d.s);
}

}  // namespace sqx
