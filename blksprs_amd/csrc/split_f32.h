// fp32 products on the bf16 matrix instructions.
#pragma once
#include "attn_mfma_common.h"

namespace bsa {
namespace split {

using namespace mfma;

__device__ static inline float as_float(uint32_t v) { return __builtin_bit_cast(float, v); }

// fp32 values as three bf16 parts: the value rounded to 8 bits, what is left of it rounded to 8 bits, and the rest, which fits
// (G. Henry, P. T. P. Tang and A. Heinecke, Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations, 2019).  A product of two such values is six products of parts, each exact, added up in fp32 by matrix instructions
// of 16 times the fp32 instruction's rate: 2.7 times the products per second.  The other three are worth up to 2^-24 of the
// product (the second part is up to 2^-8 of a value, the third 2^-17), 0.1 of that in the mean square.  The sums come
// with one rounding per 16 (32) contracted values and part where the fp32 instruction rounds every 2 (4).  Sums of 64 / 512 / 2048
// random products are 1.09e-7 / 3.4e-7 / 7.1e-7 from 64 bits, the fp32 instruction's 1.45e-7 / 4.1e-7 / 8.1e-7.
//
// Range: bf16 has fp32's exponents, but the parts of a value below 2^-102 reach below its smallest normal number, and lose bits
// there.  So a value is multiplied by kUp before it is split: every fp32 value below 2^104, subnormal ones included, is the sum of
// its parts, and a sum of products is kUp^2 times what it should be (x = 2^-118 z, y = 2^60 z': without kUp 1e-5 from 64 bits).
// What does not fit, an infinite or NaN value or one from 2^104 on, or a sum from 2^80 on, leaves a sum that is not finite:
// not_finite() finds it, and the sums are formed again with the fp32 instruction.  Scores, which are told from one another
// by their differences and may be masked afterwards, are formed without kUp (scores_in_doubt).
constexpr float kUp = 0x1p24f, kDown = 0x1p-24f;

struct Parts {
  u32x4 high, mid, low;
  __device__ inline Parts() {}
  // of eight values, times `up` (kUp or 1).  kDot: what is left of a value in one instruction, exact since it is a difference of
  // fewer bits than either, instead of 1.5.  Fewer instructions and registers, but not faster ones: attention at head
  // dimension 64, where two waves share a SIMD, is 3 to 7 % slower with it (dK / dV 82 -> 88 us), at 128 with one wave 2 to 15 %
  // faster (forward 112 -> 110, dQ 153 -> 148, dK / dV 244 -> 208), products of blocks of 64 1 % (8 x 2048 queries, half of the blocks).
  template <bool kDot>
  __device__ static inline Parts of(u32x4 a, u32x4 b, float up) {
    Parts p;
    // held in registers: written into the instruction, 0x0000bf80 becomes the inline constant -1.0, and that is 0xbf800000
    uint32_t minus_first = 0x0000bf80u, minus_second = 0xbf800000u;
    if constexpr (kDot) asm("" : "+s"(minus_first), "+s"(minus_second));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float x = as_float(i < 2 ? a[2 * i] : b[2 * i - 4]) * up, y = as_float(i < 2 ? a[2 * i + 1] : b[2 * i - 3]) * up;
      auto part = [&]() __attribute__((always_inline)) {
        uint32_t packed = MBf16::pack2(x, y);
        if constexpr (kDot) {
          x = MBf16::dot2(packed, minus_first, x), y = MBf16::dot2(packed, minus_second, y);
        } else {
          asm("" : "+v"(packed));  // or each value is converted once more by itself for the subtraction
          x -= as_float(packed << 16), y -= as_float(packed & 0xffff0000u);
        }
        return packed;
      };
      p.high[i] = part();
      p.mid[i] = part();
      p.low[i] = MBf16::pack2(x, y);
    }
    return p;
  }
};

// acc += a x b, the small products first
// kExchanged: in the order of the exchanged operands, so that a x b and b x a are the same bits in two kernels
template <bool kExchanged = false>
__device__ static inline void multiply_parts(f32x16 &acc, const Parts &a, const Parts &b) {
  acc = MBf16::mfma(kExchanged ? a.high : a.low, kExchanged ? b.low : b.high, acc);
  acc = MBf16::mfma(kExchanged ? a.low : a.high, kExchanged ? b.high : b.low, acc);
  acc = MBf16::mfma(a.mid, b.mid, acc);
  acc = MBf16::mfma(kExchanged ? a.high : a.mid, kExchanged ? b.mid : b.high, acc);
  acc = MBf16::mfma(kExchanged ? a.mid : a.high, kExchanged ? b.high : b.mid, acc);
  acc = MBf16::mfma(a.high, b.high, acc);
}

// Whether one of a wave's sums is infinite or NaN
template <int NS, int kRegs, typename Acc>
__device__ static inline bool not_finite(const Acc (&acc)[NS], float also = 0.f) {
  float nan = also * 0.f;
#pragma unroll
  for (int h = 0; h < NS; ++h)
#pragma unroll
    for (int r = 0; r < kRegs; ++r) nan = fmaf(acc[h][r], 0.f, nan);
  return __any(nan != 0.f);
}

}  // namespace split

// matmul_split.hip: fp32, sbs 64 and above
int matmul_split_f32(const void *x, const void *y, void *out, const int32_t *pair_offsets, const int32_t *pairs,
                     const int32_t *block_order, int64_t nnz_o, int64_t nnz_x, int64_t nnz_y, int sbs, int trans_x, int trans_y,
                     hipStream_t s);
}  // namespace bsa
