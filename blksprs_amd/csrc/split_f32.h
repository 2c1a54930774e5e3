// fp32 products on the bf16 matrix instructions.
#pragma once
#include "attn_mfma_common.h"

namespace bsa {
namespace split {

using namespace mfma;

__device__ static inline float as_float(uint32_t v) { return __builtin_bit_cast(float, v); }

// fp32 values as three bf16 parts: the value rounded to 8 bits, what is left of it rounded to 8 bits, and the rest, which fits.
// A product of two such values is six products of parts (what the other three are worth lies below 2^-26 of the product), each
// exact, added up in fp32 by matrix instructions of 16 times the fp32 instruction's rate: 2.7 times the products per second,
// with one rounding per 16 (32) contracted values and part where the fp32 instruction rounds every 2 (4).  Sums of 64 / 512 / 2048
// random products are 1.09e-7 / 3.4e-7 / 7.1e-7 from 64 bits, the fp32 instruction's 1.45e-7 / 4.1e-7 / 8.1e-7.
// An infinite or NaN value (or one that rounds to infinity) has NaN among its parts, so it makes NaN of every sum it enters;
// parts below bf16's range are lost.  in_doubt() finds both in the sums, which are then formed with the fp32 instruction.
struct Parts {
  u32x4 high, mid, low;
  __device__ inline Parts() {}
  __device__ inline Parts(u32x4 a, u32x4 b) {  // eight values
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float x = as_float(i < 2 ? a[2 * i] : b[2 * i - 4]), y = as_float(i < 2 ? a[2 * i + 1] : b[2 * i - 3]);
      uint32_t packed = MBf16::pack2(x, y);
      asm("" : "+v"(packed));  // or each value is converted once more by itself for the subtraction
      high[i] = packed;
      x -= as_float(packed << 16), y -= as_float(packed & 0xffff0000u);
      packed = MBf16::pack2(x, y);
      asm("" : "+v"(packed));
      mid[i] = packed;
      x -= as_float(packed << 16), y -= as_float(packed & 0xffff0000u);
      low[i] = MBf16::pack2(x, y);
    }
  }
};

// acc += a x b, the small products first
__device__ static inline void multiply_part(f32x16 &acc, u32x4 a, u32x4 b) { acc = MBf16::mfma(a, b, acc); }
__device__ static inline void multiply_part(f32x4 &acc, u32x4 a, u32x4 b) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
}
// kExchanged: in the order of the exchanged operands, so that a x b and b x a are the same bits in two kernels
template <bool kExchanged = false, typename Acc>
__device__ static inline void multiply_parts(Acc &acc, const Parts &a, const Parts &b) {
  multiply_part(acc, kExchanged ? a.high : a.low, kExchanged ? b.low : b.high);
  multiply_part(acc, kExchanged ? a.low : a.high, kExchanged ? b.high : b.low);
  multiply_part(acc, a.mid, b.mid);
  multiply_part(acc, kExchanged ? a.high : a.mid, kExchanged ? b.mid : b.high);
  multiply_part(acc, kExchanged ? a.mid : a.high, kExchanged ? b.high : b.mid);
  multiply_part(acc, a.high, b.high);
}

// Whether sums of a wave formed from parts are to be formed again: one is infinite or NaN, or all are so small that parts of
// what they were formed from may have been lost (a value below 2^-102 has less than 24 bits in its parts).
template <int NS, int kRegs, typename Acc>
__device__ static inline bool in_doubt(const Acc (&acc)[NS], float also = 0.f) {
  float nan = also * 0.f, largest = 0.f;
#pragma unroll
  for (int h = 0; h < NS; ++h)
#pragma unroll
    for (int r = 0; r < kRegs; ++r) {
      nan = fmaf(acc[h][r], 0.f, nan);
      largest = fmaxf(largest, fabsf(acc[h][r]));
    }
  return __any(nan != 0.f) || (!__any(largest >= 0x1p-80f) && __any(largest > 0.f));
}

}  // namespace split
}  // namespace bsa
