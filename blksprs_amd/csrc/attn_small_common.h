// Pieces shared by the attention kernels for blocks of 16 and 32, and for fp32 blocks of 64 as halves of 32
// (attn_small_fwd.hip, attn_small_bwd.hip, attn_shares.hip): LDS layout of a block slice, operand fragments, asynchronous
// copies of block slices, waits, the walk over a list of partner blocks, the order of the rows.
//
// A block slice (SBS x SBS elements, 512 bytes to 4 KiB, contiguous in memory) lies row-major in LDS, the 16-byte chunks
// of a row exchanged by a function of the row.  It is read both ways: rows as they lie (contraction over the head
// dimension: one 128-bit read per fragment) and columns (contraction over the sequence: the transposing LDS read for
// 16-bit elements, 32-bit reads for fp32).  Products: 32x32x16 (blocks of 32) and 16x16x32 (blocks of 16, where the 32
// contracted values of a score product are two head slices and those of a value product two partner blocks) for 16-bit
// elements; for fp32 32x32x16 of bf16 parts (blocks of 32) and 16x16x4 (blocks of 16; 32x32x2 where the parts do not hold the
// values or slices are missing), whose contracted values are taken in an order that suits the 128-bit reads.
#pragma once
#include <type_traits>

#include "attn_mfma_common.h"
#include "split_f32.h"

namespace bsa {
namespace small {

using namespace mfma;
using namespace split;

struct SBf16 : MBf16 {
  static constexpr int kElem = 2;
  // acc += fragment x fragment: 32 rows each, or 16
  __device__ static void rows(f32x16 &acc, u32x4 a, u32x4 b) { acc = mfma(a, b, acc); }
  __device__ static void rows(f32x4 &acc, u32x4 a, u32x4 b) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
  }
  __device__ static float dot(u32x4 a, u32x4 b, float c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = dot2(a[i], b[i], c);
    return c;
  }
};
struct SF16 : MF16 {
  static constexpr int kElem = 2;
  __device__ static void rows(f32x16 &acc, u32x4 a, u32x4 b) { acc = mfma(a, b, acc); }
  __device__ static void rows(f32x4 &acc, u32x4 a, u32x4 b) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), acc, 0, 0, 0);
  }
  __device__ static float dot(u32x4 a, u32x4 b, float c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = dot2(a[i], b[i], c);
    return c;
  }
};
struct SF32 {
  static constexpr int kElem = 4;
  __device__ static float as_float(uint32_t v) { return __builtin_bit_cast(float, v); }
  __device__ static f32x16 one(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
  __device__ static f32x4 one(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  template <typename Acc>
  __device__ static void rows(Acc &acc, u32x4 a, u32x4 b) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = one(as_float(a[j]), as_float(b[j]), acc);
  }
  __device__ static float dot(u32x4 a, u32x4 b, float c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = fmaf(as_float(a[i]), as_float(b[i]), c);
    return c;
  }
};

// fp32 products from bf16 parts: of blocks of 32 (and halves of blocks of 64) all of whose slices are there.  Blocks of 16, whose
// fp32 products take half as long for the same values to split, are no faster with it (6 x 1040 queries, causal, head dimension
// 32: forward 16.1 -> 16.6 us, dK / dV 20.0 -> 21.9).  Blocks of 32, fp32 instruction -> parts, us (8 x 2048, half of the blocks):
//     head dimension     32             64             96             128
//     forward       32.4 -> 29.8   55.2 -> 46.5   96.5 -> 83.7   122 -> 105
//     dQ            42.8 -> 38.4   76.7 -> 63.2    128 -> 110    166 -> 140
//     dK / dV       54.1 -> 47.8   97.6 -> 81.0    170 -> 152    219 -> 198
// causal and BigBird layouts 4 to 24 % less (dK / dV of BigBird at 128: 138 -> 132), blocks of 64 at 128 2 to 12 %.
struct SSplit : SF32 {};
template <int NS>
constexpr bool kDotParts = NS > 2;  // Parts::of
// What the partner's and the own values of a product other than the scores are multiplied by
template <typename Ar>
constexpr float up_of() {
  return std::is_same_v<Ar, SSplit> ? kUp : 1.f;
}
template <typename Tr, int SBS, bool kSome>
constexpr bool in_parts() {
  return Tr::kElem == 4 && SBS == 32 && !kSome;
}

// Waits until at most N vector memory operations of the wave are outstanding.  The clobber keeps LDS reads behind it.
template <int N>
__device__ static inline void wait_vmem() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// LDS reads issued so far have returned: their buffer may be copied over
__device__ static inline void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// XOR on the 16-byte chunk index of row r of a block slice.  Eight consecutive rows read at one chunk index must fall on
// different chunks of a 128-byte bank period.  16-bit rows of 64 bytes (SBS 32): sixteen rows also spread over 256 bytes,
// and the four rows r .. r + 3 (r a multiple of 4) of a transposing read use different halves of their rows.  16-bit rows
// of 32 bytes: a transposing read of four rows covers 128 consecutive bytes anyway.  fp32 rows of 64 bytes (SBS 16) are
// stored at row_place(r) so that the four rows r, r + 4, r + 8, r + 12 of a column read are neighbours.
template <int ES, int SBS>
__device__ static inline int chunk_swizzle(int r) {
  if constexpr (ES == 4 && SBS == 32) return r & 7;
  else if constexpr (ES == 4) return r & 3;
  else if constexpr (SBS == 32) return ((((r >> 1) ^ (r >> 3)) & 1) << 1) | ((r >> 2) & 1);
  else return ((r >> 2) ^ (r >> 3)) & 1;
}
template <int ES, int SBS>
__device__ static inline int row_place(int r) {
  if constexpr (ES == 4 && SBS == 16) return 4 * (r & 3) + (r >> 2);
  else return r;
}

// transposing LDS read of 8 bytes per lane
__device__ static inline u32x2 read_tr(const char *p) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4 *)p));
}

// The kernel's own argument block, read again where it is used.  Its fields are loop invariants, and the compiler would
// load all of them in front of the loop and spill what the scalar registers do not hold into lanes of vector registers,
// in the loop; the empty assembly keeps it from moving the loads of rarely taken paths and of the epilogue.
typedef const __attribute__((address_space(4))) bsa_attn_args *late_args_t;
__device__ static inline late_args_t late_args() {
  late_args_t p = (late_args_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}

// Asynchronous copies of N consecutive KiB (1 to 4), global -> LDS, lane l supplying the bytes at position 16 l of each
template <int N>
__device__ static inline void copy_kib_to_lds(const char *base, uint32_t off, char *dst) {
  const uint32_t lds_addr = (uint32_t)(uintptr_t)(lds_ptr_t)dst;
  if constexpr (N == 1)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(lds_addr) : "memory");
  else if constexpr (N == 2)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024"
                 : : "v"(off), "s"(base), "s"(lds_addr) : "memory");
  else if constexpr (N == 3)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024\n\t"
                 "global_load_lds_dwordx4 %0, %1 offset:2048"
                 : : "v"(off), "s"(base), "s"(lds_addr) : "memory");
  else
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024\n\t"
                 "global_load_lds_dwordx4 %0, %1 offset:2048\n\tglobal_load_lds_dwordx4 %0, %1 offset:3072"
                 : : "v"(off), "s"(base), "s"(lds_addr) : "memory");
}

// N KiB of LDS (2 or 4) from every second KiB of memory: half of the columns of blocks twice as wide.  The offset field
// moves both addresses, the other KiB comes from the lane's offset.
template <int N>
__device__ static inline void copy_every_second_kib_to_lds(const char *base, uint32_t off, char *dst) {
  const uint32_t lds_addr = (uint32_t)(uintptr_t)(lds_ptr_t)dst;
  static_assert(N == 2 || N == 4, "KiB of a slice");
  if constexpr (N == 2)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %3, %1 offset:1024"
                 : : "v"(off), "s"(base), "s"(lds_addr), "v"(off + 1024) : "memory");
  else
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %3, %1 offset:1024\n\t"
                 "global_load_lds_dwordx4 %4, %1 offset:2048\n\tglobal_load_lds_dwordx4 %5, %1 offset:3072"
                 : : "v"(off), "s"(base), "s"(lds_addr), "v"(off + 1024), "v"(off + 2048), "v"(off + 3072) : "memory");
}

// Where the blocks of the kernels lie in memory.  kHalves 1: a block is a block of the layout.  kHalves 2: a block of the
// layout (64 x 64) is four of theirs, its head slice two of theirs: block i of a row is half i % 2 of the rows of the layout's
// block i / 2, slice h the columns from SBS (h % 2) of the layout's slice h / 2.  A wave has the
// accumulators that it has for blocks of 32, and a layout twice as many rows to spread over the chip.
template <int ES, int SBS, int kHalves>
struct Place {
  static constexpr int kPitch = kHalves * SBS * ES;             // bytes from row to row
  static constexpr int64_t kBlockBytes = (int64_t)kHalves * SBS * kPitch;  // of a slice of a block of the layout
  // byte offset of (row r, slice h) of block `own`, whose slice h / kHalves has packed index idx
  __device__ static inline int64_t row(int64_t idx, int own, int r, int h) {
    return idx * kBlockBytes + (int64_t)(own % kHalves * SBS + r) * kPitch + h % kHalves * (SBS * ES);
  }
};

// Geometry of one wave's tile: NB partner blocks of NS head slices each, slice h of block t at piece t * NS + h.
template <int ES, int SBS, int NS, int NB, int kHalves = 1>
struct Tile {
  static constexpr int kPiece = SBS * SBS * ES;
  static constexpr int kRowBytes = SBS * ES;
  static constexpr int kBlock = NS * kPiece;     // one partner block
  static constexpr int kBytes = NB * kBlock;
  static constexpr int kBlockCopies = (kBlock + 1023) / 1024;
  static constexpr int kCopies = NB * kBlockCopies;  // asynchronous copies per tile

  // This lane's source offset for a copy that fills LDS linearly.  All KiB of a block share it: a KiB holds eight rows
  // of 128 bytes or sixteen of 64, or two slices of sixteen rows of 32 bytes.
  __device__ static inline uint32_t source_offset(int lane) {
    constexpr int kChunks = kRowBytes / 16;
    const int place = lane / kChunks % SBS;  // row_place is its own inverse
    const int r = row_place<ES, SBS>(place);
    return (uint32_t)((lane * 16 / kPiece) * kPiece + r * (kHalves * kRowBytes) + (((lane % kChunks) ^ chunk_swizzle<ES, SBS>(r)) << 4));
  }

  // Requests block t of the tile, all of whose slices are there and lie one behind the other from packed index idx (kHalves
  // times the packed index, plus the half): kBlockCopies asynchronous copies.
  __device__ static inline void copy_block(const char *tensor, int idx, char *dst, uint32_t offset, int lane) {
    if constexpr (kHalves == 2) {
      static_assert(SBS == 32 && NS % 2 == 0, "halves of blocks of 64");
      const char *src = tensor + (uint64_t)(uint32_t)idx * (2 * kPiece);
#pragma unroll
      for (int h = 0; h < NS; ++h)
        copy_every_second_kib_to_lds<kPiece / 1024>(src + h / 2 * (4 * kPiece) + h % 2 * kRowBytes, offset, dst + h * kPiece);
      return;
    }
    const char *src = tensor + (uint64_t)(uint32_t)idx * kPiece;
    constexpr int kKib = kBlock / 1024;
#pragma unroll
    for (int i = 0; i + 4 <= kKib; i += 4) copy_kib_to_lds<4>(src + 1024 * i, offset, dst + 1024 * i);
    constexpr int kDone = kKib / 4 * 4;
    if constexpr (kKib % 4 != 0) copy_kib_to_lds<kKib % 4>(src + 1024 * kDone, offset, dst + 1024 * kDone);
    if constexpr (kBlock % 1024 != 0) {  // an odd number of slices of 512 bytes: the last one by half of the lanes
      if (lane < 32) copy_kib_to_lds<1>(src + 1024 * kKib, offset, dst + 1024 * kKib);
    }
  }

  // The same for one slice of a block, packed index idx
  __device__ static inline void copy_piece(const char *tensor, int idx, char *dst, uint32_t offset, int lane) {
    const char *src = tensor + (uint64_t)(uint32_t)idx * kPiece;
    if constexpr (kPiece >= 1024) copy_kib_to_lds<kPiece / 1024>(src, offset, dst);
    else if (lane < 32) copy_kib_to_lds<1>(src, offset, dst);
  }

  // zeros for a whole block, written by the wave itself
  __device__ static inline void clear_block(char *dst, int lane) {
#pragma unroll
    for (int i = 0; i < kBlock; i += 1024)
      if (kBlock - i >= 1024 || lane < 32) *reinterpret_cast<u32x4 *>(dst + i + lane * 16) = u32x4{0u, 0u, 0u, 0u};
  }

  // ---- row fragments (contraction over the head dimension): 16 bytes of a row per lane
  // 16-bit, SBS 32: fragment f of a block = values 16 f .. + 15 (2 per slice), this lane row lane % 32, values
  // 8 (lane / 32) .. + 7.  SBS 16: fragment f = slices 2 f, 2 f + 1, this lane row lane % 16, 8 values of slice
  // 2 f + lane / 32 from 8 (lane / 16 % 2); behind the last slice of an odd count the upper half of the lanes hold zeros.
  // (The product of 16 values for that slice is not used: its sum, fed by a product of 32 values right in front of it,
  // came out without it.)
  // fp32: fragment f = values 8 f .. + 7 (SBS 32) or 16 f .. + 15 (SBS 16), this lane row lane % SBS, the four values
  // from 4 (lane / SBS); product j of the fragment contracts element j of every lane.
  static constexpr int kFrags = ES == 4 ? NS * kRowBytes / 16 / (64 / SBS) : SBS == 32 ? 2 * NS : (NS + 1) / 2;
  static constexpr int kSliceFrags = ES == 4 ? kFrags / NS : 2;  // of SBS 32 and fp32
  static constexpr bool kHalfLast = ES == 2 && SBS == 16 && (NS & 1);

  struct RowReader {
    static constexpr int kBases = ES == 2 && SBS == 16 ? 1 : kSliceFrags;
    const char *base[kBases];
    bool beyond;  // 16-bit, SBS 16: this lane's half of the last fragment of an odd slice count is beyond the block
    __device__ RowReader(const char *lds, int lane) : beyond(lane >= 32) {
      const int r = lane % SBS, g = lane / SBS, place = row_place<ES, SBS>(r) * kRowBytes, x = chunk_swizzle<ES, SBS>(r);
      if constexpr (ES == 2 && SBS == 16) {
        base[0] = lds + (g >> 1) * kPiece + place + (((g & 1) ^ x) << 4);
      } else {
#pragma unroll
        for (int i = 0; i < kBases; ++i) base[i] = lds + place + (((64 / SBS * i + g) ^ x) << 4);
      }
    }
    __device__ void shift(int bytes) {
#pragma unroll
      for (int i = 0; i < kBases; ++i) base[i] += bytes;
    }
    __device__ u32x4 frag(int t, int f) const {
      if constexpr (ES == 4 || SBS == 32)
        return *reinterpret_cast<const u32x4 *>(base[f % kBases] + (t * NS + f / kBases) * kPiece);
      u32x4 v = *reinterpret_cast<const u32x4 *>(base[0] + (t * NS + 2 * f) * kPiece);
      if (kHalfLast && f == kFrags - 1 && beyond) v = u32x4{0u, 0u, 0u, 0u};
      return v;
    }
  };

  // ---- column fragments (contraction over the rows of the partner blocks)
  // 16-bit, SBS 32: fragment m of block t, slice h: column lane % 32, rows 16 m + 4 kg .. + 3 and 16 m + 8 + 4 kg .. + 3
  // (kg = lane / 32): the rows whose values a lane holds in accumulator registers 8 m .. 8 m + 7.  SBS 16: fragment of
  // blocks t and t + 1, slice h: column lane % 16, rows 4 (lane / 16) .. + 3 of either block: the rows of accumulator
  // registers 0 .. 3 of the two blocks.
  // fp32: element (row of accumulator register r, column lane % SBS) of block t, slice h.
  struct ColReader {
    static constexpr int kBases = ES == 4 ? 4 : SBS == 32 ? 2 : 1;
    const char *base[kBases];
    __device__ ColReader(const char *lds, int lane) {
      if constexpr (ES == 4) {
        const int c = lane % SBS, g = lane / SBS;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = 4 * g + j;
          base[j] = lds + row_place<ES, SBS>(r) * kRowBytes + (((c >> 2) ^ chunk_swizzle<ES, SBS>(r)) << 4) + (c & 3) * 4;
        }
      } else {
        const int s = lane & 15, half = SBS == 32 ? (lane >> 4) & 1 : 0;
#pragma unroll
        for (int i = 0; i < kBases; ++i) {
          const int r = 8 * i + 4 * (lane / SBS) + (s >> 2), c = 2 * half + ((s & 3) >> 1);
          base[i] = lds + r * kRowBytes + ((c ^ chunk_swizzle<ES, SBS>(r)) << 4) + ((s & 1) << 3);
        }
      }
    }
    __device__ void shift(int bytes) {
#pragma unroll
      for (int i = 0; i < kBases; ++i) base[i] += bytes;
    }
    __device__ u32x4 frag(int t, int m, int h) const {
      u32x2 lo, hi;
      if constexpr (SBS == 32) {
        lo = read_tr(base[0] + (t * NS + h) * kPiece + m * 1024);
        hi = read_tr(base[kBases - 1] + (t * NS + h) * kPiece + m * 1024);
      } else {
        lo = read_tr(base[0] + ((t + 2 * m) * NS + h) * kPiece);
        hi = read_tr(base[0] + ((t + 2 * m + 1) * NS + h) * kPiece);
      }
      return u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
    __device__ float value(int t, int h, int r) const {
      return *reinterpret_cast<const float *>(base[r % 4] + (t * NS + h) * kPiece + (r / 4) * 8 * kRowBytes);
    }
  };
};

// One block's own rows as the other operand of the score products, in registers for the whole walk (the same values
// per lane as RowReader's fragments).
template <int ES, int SBS, int NS, int kHalves>
struct OwnRows {
  using T = Tile<ES, SBS, NS, 2, kHalves>;
  u32x4 fr[T::kFrags];
  uint32_t there;  // bit h: the block has slice h of the layout (wave uniform)

  // pidx: packed indices of the slices of block `own` in the layout, n_slices of them are there
  __device__ inline void load(const void *tensor, const int64_t *pidx, int n_slices, int64_t n_blocks, int own, int lane) {
    const int r = lane % SBS, g = lane / SBS;
    const int64_t mine = lane < n_slices ? pidx[lane] : -1;
    there = (uint32_t)__ballot(mine >= 0 && mine < n_blocks);
#pragma unroll
    for (int f = 0; f < T::kFrags; ++f) {
      int h, chunk;
      if constexpr (ES == 2 && SBS == 16) h = 2 * f + (g >> 1), chunk = g & 1;
      else h = f / T::kSliceFrags, chunk = 64 / SBS * (f % T::kSliceFrags) + g;
      const int64_t idx = h / kHalves < n_slices ? pidx[h / kHalves] : -1;
      fr[f] = u32x4{0u, 0u, 0u, 0u};
      if (idx >= 0 && idx < n_blocks)
        fr[f] = *reinterpret_cast<const u32x4 *>(static_cast<const char *>(tensor) + Place<ES, SBS, kHalves>::row(idx, own, r, h) +
                                                 chunk * 16);
    }
  }
};

// The own rows as the products of arithmetic Ar take them; kSecond: of the second tensor (Walk), otherwise for scores
template <typename Ar, int SBS, int NS, int kHalves, bool kSecond>
struct OwnOperand {
  const OwnRows<Ar::kElem, SBS, NS, kHalves> &rows;
  __device__ inline explicit OwnOperand(const OwnRows<Ar::kElem, SBS, NS, kHalves> &own) : rows(own) {}
};
// in parts: fragments 2 p and 2 p + 1 in one
template <int SBS, int NS, int kHalves, bool kSecond>
struct OwnOperand<SSplit, SBS, NS, kHalves, kSecond> {
  static constexpr int kFrags = OwnRows<4, SBS, NS, kHalves>::T::kFrags, kParts = kFrags / 2;
  static_assert(kFrags % 2 == 0, "whole pairs of fragments");
  Parts parts[kParts];
  __device__ inline explicit OwnOperand(const OwnRows<4, SBS, NS, kHalves> &own) {
#pragma unroll
    for (int p = 0; p < kParts; ++p)
      parts[p] = Parts::of<kDotParts<NS>>(own.fr[2 * p], own.fr[2 * p + 1], kSecond ? kUp : 1.f);
  }
};

// Makes the compiler wait for the loads of the own rows here: left to their first use, the wait sits inside the loop and
// is for every load in flight, each time round.
template <int ES, int SBS, int NS, int kHalves>
__device__ static inline void settle(OwnRows<ES, SBS, NS, kHalves> &own) {
#pragma unroll
  for (int f = 0; f < OwnRows<ES, SBS, NS, kHalves>::T::kFrags; ++f) asm volatile("" : "+v"(own.fr[f]));
}

// Whether scores from parts, formed without kUp, could be off by more than 2^-30.  The own values are exact in their parts if they
// are 0 or at least 2^-102; those of the partners are off by 2^-125 at most, and a score by 128 times that, the largest own value
// and the scale.  (A score that overflows is as good as infinite, or leaves NaN in the sums.)
template <int ES, int SBS, int NS, int kHalves>
__device__ static inline bool scores_in_doubt(const OwnRows<ES, SBS, NS, kHalves> &own, float scale) {
  constexpr int kFrags = OwnRows<ES, SBS, NS, kHalves>::T::kFrags;
  float least = INFINITY, most = 0.f;
#pragma unroll
  for (int f = 0; f < kFrags; ++f)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v = fabsf(as_float(own.fr[f][i]));
      least = fminf(least, v), most = fmaxf(most, v);
    }
  bool small = __any(least < 0x1p-102f);
  if (small) {  // or zero
    least = INFINITY;
#pragma unroll
    for (int f = 0; f < kFrags; ++f)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = fabsf(as_float(own.fr[f][i]));
        least = fminf(least, v > 0.f ? v : INFINITY);
      }
    small = __any(least < 0x1p-102f);
  }
  return small || __any(most > 0x1p70f) || scale > 0x1p17f;
}

// acc (per partner block t) = partner rows x own rows over all head slices: acc[t] belongs to this lane's own row
// (lane % SBS) and partner rows 8 (r / 4) + 4 (lane / 32) + r % 4 (SBS 32) or 4 (lane / 16) + r (SBS 16).
// kOwnIsQuery, kSecond: as in Walk; a score from parts is the same bits wherever it is formed, but forward and backward kernels
// look at blocks of their own before they form one from parts (scores_in_doubt) and may differ there by its rounding; of the second tensor acc is
// up_of^2 times the product
template <typename Tr, int SBS, int NS, int NB, int kHalves, bool kOwnIsQuery, bool kSecond, typename Acc>
__device__ static inline void product_rows(Acc (&acc)[NB], const typename Tile<Tr::kElem, SBS, NS, NB, kHalves>::RowReader &rows,
                                           const OwnOperand<Tr, SBS, NS, kHalves, kSecond> &own) {
  constexpr int kFrags = Tile<Tr::kElem, SBS, NS, NB>::kFrags;
#pragma unroll
  for (int t = 0; t < NB; ++t)
#pragma unroll
    for (int r = 0; r < (SBS == 32 ? 16 : 4); ++r) acc[t][r] = 0.f;
  if constexpr (std::is_same_v<Tr, SSplit>) {
#pragma unroll
    for (int p = 0; p < OwnOperand<Tr, SBS, NS, kHalves, kSecond>::kParts; ++p)
#pragma unroll
      for (int t = 0; t < NB; ++t)
        multiply_parts<!kOwnIsQuery>(acc[t], Parts::of<kDotParts<NS>>(rows.frag(t, 2 * p), rows.frag(t, 2 * p + 1), kSecond ? kUp : 1.f),
                                     own.parts[p]);
  } else {
#pragma unroll
    for (int f = 0; f < kFrags; ++f)
#pragma unroll
      for (int t = 0; t < NB; ++t) Tr::rows(acc[t], rows.frag(t, f), own.rows.fr[f]);
  }
}

// The same over the slices in have[t] only: a slice that one of the two blocks does not have adds nothing, where its zeros
// would turn an infinite or NaN value of the other into NaN
template <typename Tr, int SBS, int NS, int NB, typename Acc>
__device__ static inline void product_some_rows(Acc (&acc)[NB], const typename Tile<Tr::kElem, SBS, NS, NB>::RowReader &rows,
                                                const OwnRows<Tr::kElem, SBS, NS, 1> &own, const uint32_t (&have)[NB], int lane) {
  using T = Tile<Tr::kElem, SBS, NS, NB>;
#pragma unroll
  for (int t = 0; t < NB; ++t)
#pragma unroll
    for (int r = 0; r < (SBS == 32 ? 16 : 4); ++r) acc[t][r] = 0.f;
#pragma unroll
  for (int t = 0; t < NB; ++t)
#pragma unroll
    for (int f = 0; f < T::kFrags; ++f) {
      if constexpr (Tr::kElem == 2 && SBS == 16) {  // lanes below 32 hold slice 2 f, the others 2 f + 1
        const bool on = (have[t] >> (2 * f + (lane >> 5))) & 1;
        const u32x4 none{0u, 0u, 0u, 0u}, theirs = rows.frag(t, f);
        Tr::rows(acc[t], on ? theirs : none, on ? own.fr[f] : none);
      } else {
        if ((have[t] >> (f / T::kSliceFrags)) & 1) Tr::rows(acc[t], rows.frag(t, f), own.fr[f]);
      }
    }
}

// Probabilities (or dS) of a step, as the accumulators of its NB blocks hold them one after the other, made the second
// operand of product_cols: rounded to the operand type and packed.
template <typename Tr, int kScores>
struct Weights {
  u32x4 w[kScores / 8];
  __device__ inline explicit Weights(const float *v) {
#pragma unroll
    for (int m = 0; m < kScores / 8; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) w[m][i] = Tr::pack2(v[8 * m + 2 * i], v[8 * m + 2 * i + 1]);
  }
};
template <int kScores>
struct Weights<SF32, kScores> {
  float w[kScores];
  __device__ inline explicit Weights(const float *v) {
#pragma unroll
    for (int x = 0; x < kScores; ++x) w[x] = v[x];
  }
};

template <int kScores>
struct Weights<SSplit, kScores> : Weights<SF32, kScores> {
  using Weights<SF32, kScores>::Weights;
};

// out[h] += partner columns^T x weights, times up_of: weights that are up_of times theirs leave up_of^2 times the product
template <typename Tr, int SBS, int NS, int NB, int kHalves, int kScores, typename Acc>
__device__ static inline void product_cols(Acc (&out)[NS], const typename Tile<Tr::kElem, SBS, NS, NB, kHalves>::ColReader &cols,
                                           const Weights<Tr, kScores> &w) {
  if constexpr (std::is_same_v<Tr, SSplit>) {
    constexpr int kRegs = kScores / NB;
#pragma unroll
    for (int x = 0; x < kScores; x += 8) {
      u32x4 v[2];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i / 4][i % 4] = __builtin_bit_cast(uint32_t, w.w[x + i]);
      const Parts weights = Parts::of<kDotParts<NS>>(v[0], v[1], 1.f);
#pragma unroll
      for (int h = 0; h < NS; ++h) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i / 4][i % 4] = __builtin_bit_cast(uint32_t, cols.value((x + i) / kRegs, h, (x + i) % kRegs));
        multiply_parts(out[h], Parts::of<kDotParts<NS>>(v[0], v[1], kUp), weights);
      }
    }
  } else if constexpr (Tr::kElem == 4) {
    constexpr int kRegs = kScores / NB;
#pragma unroll
    for (int x = 0; x < kScores; ++x)
#pragma unroll
      for (int h = 0; h < NS; ++h) out[h] = Tr::one(cols.value(x / kRegs, h, x % kRegs), w.w[x], out[h]);
  } else {
#pragma unroll
    for (int h = 0; h < NS; ++h)
#pragma unroll
      for (int m = 0; m < kScores / 8; ++m)
        Tr::rows(out[h], SBS == 32 ? cols.frag(m >> 1, m & 1, h) : cols.frag(0, m, h), w.w[m]);
  }
}

// the same over the slices in have[t]
template <typename Tr, int SBS, int NS, int NB, int kScores, typename Acc>
__device__ static inline void product_some_cols(Acc (&out)[NS], const typename Tile<Tr::kElem, SBS, NS, NB>::ColReader &cols,
                                                const Weights<Tr, kScores> &w, const uint32_t (&have)[NB]) {
  if constexpr (Tr::kElem == 4) {
    constexpr int kRegs = kScores / NB;
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
      for (int h = 0; h < NS; ++h)
        if ((have[t] >> h) & 1) {
#pragma unroll
          for (int r = 0; r < kRegs; ++r) out[h] = Tr::one(cols.value(t, h, r), w.w[kRegs * t + r], out[h]);
        }
  } else if constexpr (SBS == 32) {
#pragma unroll
    for (int h = 0; h < NS; ++h)
      if ((have[0] >> h) & 1) {
#pragma unroll
        for (int m = 0; m < 2; ++m) Tr::rows(out[h], cols.frag(0, m, h), w.w[m]);
      }
  } else {  // one product of two blocks: registers 0 and 1 of either operand the first, 2 and 3 the second
#pragma unroll
    for (int h = 0; h < NS; ++h) {
      const bool on0 = (have[0] >> h) & 1, on1 = (have[NB - 1] >> h) & 1;
      if (!on0 && !on1) continue;
      const u32x4 f = cols.frag(0, 0, h), v = w.w[0];
      Tr::rows(out[h], u32x4{on0 ? f[0] : 0u, on0 ? f[1] : 0u, on1 ? f[2] : 0u, on1 ? f[3] : 0u},
               u32x4{on0 ? v[0] : 0u, on0 ? v[1] : 0u, on1 ? v[2] : 0u, on1 ? v[3] : 0u});
    }
  }
}

// The factor cc of the scores, inside the exponential.  16-bit: fused with the subtraction of the maximum or lse.  fp32: a
// multiplication of its own in front, since the maximum and lse come from products that were rounded: the score they come
// from must differ from them by exactly zero (a probability of exactly 1: the output of a query that sees one key is that
// key's value), where a fused product leaves the rounding of the first (dV of short causal rows 6 % further from 64 bits).
template <typename Tr, int kScores>
__device__ static inline void apply_factor(float *sv, float cc) {
  if constexpr (Tr::kElem == 4) {
#pragma unroll
    for (int x = 0; x < kScores; ++x) {
      sv[x] *= cc;
      asm("" : "+v"(sv[x]));  // not to be fused after all
    }
  }
}
template <typename Tr>
__device__ static inline float late_factor(float cc) {
  return Tr::kElem == 4 ? 1.f : cc;
}

// four consecutive values of an output row
template <typename Tr>
__device__ static inline void store4(char *p, float a, float b, float c, float d) {
  if constexpr (Tr::kElem == 4) *reinterpret_cast<f32x4 *>(p) = f32x4{a, b, c, d};
  else *reinterpret_cast<u32x2 *>(p) = u32x2{Tr::pack2(a, b), Tr::pack2(c, d)};
}

// The lane's number, of which the compiler knows nothing.  The loads of the own rows in front of a second walk over a list are
// those in front of the first; with one lane number in both, their addresses stay in registers through the first walk, for the
// second that is hardly ever made: the forward kernel of fp32 at head dimension 64 then needs 172 registers (with this 164,
// which is a wave per SIMD more), dK / dV 12 more than the 256 there are.
__device__ static inline int fresh_lane() {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));
  return lane;
}

// Sums of products from parts (up_of) at their own size
template <typename Ar, int NS, int kRegs, typename Acc>
__device__ static inline void scale_down(Acc (&acc)[NS]) {
  constexpr float kFactor = 1.f / (up_of<Ar>() * up_of<Ar>());
#pragma unroll
  for (int h = 0; h < NS; ++h)
#pragma unroll
    for (int r = 0; r < kRegs; ++r) acc[h][r] *= kFactor;
}

// Maximum / sum over the lanes that hold the same own row (lanes l, l + SBS, ...)
template <int SBS>
__device__ static inline float row_max(float v) {
  if constexpr (SBS == 16) {
    float lower = v, upper = v;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(lower), "+v"(upper));
    v = fmaxf(lower, upper);
  }
  return max_across32(v);
}
template <int SBS>
__device__ static inline float row_sum(float v) {
  if constexpr (SBS == 16) {
    float lower = v, upper = v;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(lower), "+v"(upper));
    v = lower + upper;
  }
  return sum_across32(v);
}

// One wave's walk over the list of partner blocks of one block of its own: key blocks of a query block, or (kOwnIsQuery
// false) query blocks of a key block.
//
// The list is read 64 entries at a time, one per lane: the partner block, the packed indices of its first slices (of K
// and V, or of Q and dO), its mask and bias block.  Entries the causal predicate rules out as a whole are left out of
// `live`; `special` marks those whose scores need more than the scale.
//
// kSome: head slices may be missing on either side, or q / k and v / o have different numbers of them (NS is the larger
// one); only slices that are there are copied, and only those that both blocks of a pair have are multiplied.  `apart` marks
// entries of whose slices some are missing or do not lie one behind the other.  The two are kernels of their own: with
// both kinds of products in one loop the compiler needs 5 to 30 registers more, which costs a wave per SIMD or spills.
// 16 x 2048 queries, a quarter of the blocks, head dimension 64, 9 of 10 slices there, forward / forward and backward: bf16,
// sbs 16: 45 / 165 us (61 / 189 with every block of a window of 64 gathered as soon as one had a gap), fp32: 96 / 352
// (131 / 453); full layouts 27 / 164 and 67 / 256.
// kHalves 2 (blocks of 64): blocks, slices and places are those of the kernels (Place), so an entry of the list is two.
template <int ES, int SBS, int NS, int NB, bool kOwnIsQuery, bool kSome, int kHalves>
struct Walk {
  static_assert(kHalves == 1 || !kSome, "missing slices of blocks of 64 take another kernel");
  using T = Tile<ES, SBS, NS, NB, kHalves>;
  int64_t b, own;          // batch entry, own block
  int list, first, step;   // start of the list; the wave's places in it: first, first + step, ...
  int end, base, seq_len;  // their number, the first one of the window; valid length of a causal sequence
  int other, first_a, first_b, mask, bias;  // of this lane's entry
  uint64_t live, special, apart;

  // a step: how many entries it takes and their places in the window, and, if special, their facts (the window may be
  // another one by the time the scores are formed)
  struct Step {
    int count, slot[NB], other[NB], mask[NB], bias[NB];
    bool special;
    uint32_t have[NB];  // kSome: slices of each block that are there, bits 0 .. 7 of the first tensor, 8 .. 15 of the second; set by copy()
  };

  // part of parts: this wave walks every parts-th entry of the list.  The sums of the parts then have about the same size: with
  // contiguous parts the first query rows of a causal layout, whose probabilities are the largest, all go into one of them,
  // and dV of fp32 is 3 to 10 % further from 64 bits.
  __device__ inline void start(const bsa_attn_args &a, int64_t b_, int64_t own_, bool there, int part, int parts) {
    b = b_, own = own_;
    seq_len = 0x7fffffff;
    if (a.causal_lengths) {
      const int64_t len = a.causal_lengths[b];
      seq_len = len < 0 ? 0 : (len > 0x7fffffffLL ? 0x7fffffff : (int)len);
    }
    const int32_t *offsets = (kOwnIsQuery ? a.key_offsets : a.query_offsets) + b * (kOwnIsQuery ? a.nq : a.nk) + own / kHalves;
    list = first_lane(offsets[0]);
    first = part;
    step = parts;
    const int left = kHalves * (first_lane(offsets[1]) - list) - part;
    end = left > 0 ? (int)(((unsigned)left + parts - 1) / parts) : 0;
    if (!there || (int)own * SBS >= seq_len) end = 0;
    base = -64;
    other = first_a = first_b = 0;
    mask = bias = -1;
    live = special = apart = 0;
  }

  // the first of n packed indices; far if they are not one behind the other or do not all exist
  __device__ static inline int in_a_row(const int64_t *pidx, int n, int64_t n_blocks, bool &far) {
    const int64_t first = n > 0 ? pidx[0] : 0;
    far = far || first < 0 || first + n > n_blocks;
    for (int h = 1; h < n; ++h) far = far || pidx[h] != first + h;
    return (int)first;
  }

  __device__ inline void refill(int lane) {
    const late_args_t p = late_args();
    base += 64;
    bool in = base + lane < end;
    const int at = first + step * (base + lane);
    other = in ? kHalves * (kOwnIsQuery ? p->key_indices : p->query_indices)[list + at / kHalves] + at % kHalves : 0;
    const bool causal = p->causal_lengths != nullptr;
    in = in && !(causal && ((kOwnIsQuery ? other > (int)own : other < (int)own) || other * SBS >= seq_len));
    const int64_t place = b * (kOwnIsQuery ? p->nk : p->nq) + other / kHalves;
    const int64_t *pa = kOwnIsQuery ? p->pidx_k : p->pidx_q, *pb = kOwnIsQuery ? p->pidx_v : p->pidx_o;
    const int64_t end_a = kOwnIsQuery ? p->n_k_blocks : p->n_q_blocks, end_b = kOwnIsQuery ? p->n_v_blocks : p->n_o_blocks;
    if constexpr (kSome) {
      bool far = false;
      if (in) {
        first_a = in_a_row(pa + place * p->nh, (int)p->nh, end_a, far);
        first_b = in_a_row(pb + place * p->nhv, (int)p->nhv, end_b, far);
      }
      apart = __ballot(in && far);
    } else if (in) {  // every slice of every partner block is there: the others follow the first
      constexpr int kSlices = NS / kHalves;  // of the layout
      const int64_t a0 = pa[place * kSlices], b0 = pb[place * kSlices];
      first_a = kHalves * (int)a0 + other % kHalves;
      first_b = kHalves * (int)b0 + other % kHalves;
      // a wrong index must not turn into a wild read
      in = a0 >= 0 && b0 >= 0 && a0 + kSlices <= end_a && b0 + kSlices <= end_b;
    }
    bool extra = causal && (other == (int)own || ((int)own + 1) * SBS > seq_len || (other + 1) * SBS > seq_len);
    const int64_t mine = own / kHalves, theirs = other / kHalves;
    const int64_t pair = kOwnIsQuery ? (b * p->nq + mine) * p->nk + theirs : (b * p->nq + theirs) * p->nk + mine;
    if (p->mask) {
      const int64_t m = in ? p->pidx_mask[pair] : -1;
      mask = m < p->n_mask_blocks ? (int)m : -1;
      extra = extra || mask >= 0;
    }
    if (p->bias) {
      const int64_t m = in ? p->pidx_bias[pair] : -1;
      bias = m < p->n_bias_blocks ? (int)m : -1;
      extra = true;
    }
    live = __ballot(in);
    special = __ballot(in && extra);
  }

  __device__ inline void take(Step &s, int lane) {
    while (live == 0 && base + 64 < end) refill(lane);
    s.count = 0;
    uint64_t taken = 0;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const uint64_t lowest = live & -live;
      s.slot[t] = lowest ? __builtin_ctzll(lowest) : 0;
      if constexpr (kSome) s.have[t] = 0;
      s.count += lowest ? 1 : 0;
      live ^= lowest;
      taken |= lowest;
    }
    s.special = (taken & special) != 0 || (NB > 1 && s.count < NB);
    if (s.special) {
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        s.other[t] = __builtin_amdgcn_readlane(other, s.slot[t]);
        s.mask[t] = t < s.count ? __builtin_amdgcn_readlane(mask, s.slot[t]) : -1;
        s.bias[t] = t < s.count ? __builtin_amdgcn_readlane(bias, s.slot[t]) : -1;
      }
    }
  }

  // Requests the step's blocks of the first (K or Q) or second (V or dO) tensor; returns whether exactly T::kCopies
  // asynchronous copies are on their way.  To be called before the next take().
  template <bool kSecond>
  __device__ inline bool copy(Step &s, const char *tensor, char *dst, uint32_t offset, int lane) const {
    if constexpr (kSome) {
      copy_some<kSecond>(s, tensor, dst, offset, lane);
      return false;
    }
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      char *const to = dst + t * T::kBlock;
      if (NB == 1 || t < s.count)
        T::copy_block(tensor, __builtin_amdgcn_readlane(kSecond ? first_b : first_a, s.slot[t]), to, offset, lane);
      else T::clear_block(to, lane);  // the last step of a list
    }
    return NB == 1 || s.count == NB;
  }
  template <bool kSecond>
  __device__ inline void copy_some(Step &s, const char *tensor, char *dst, uint32_t offset, int lane) const {
    const late_args_t p = late_args();
    const int n = kSecond ? (int)p->nhv : (int)p->nh;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      uint32_t on = 0;
      if (t < s.count) {
        int mine = __builtin_amdgcn_readlane(kSecond ? first_b : first_a, s.slot[t]) + lane;  // lane h: packed index of slice h
        on = (1u << n) - 1;
        if ((apart >> s.slot[t]) & 1) {
          const int64_t place = b * (kOwnIsQuery ? p->nk : p->nq) + __builtin_amdgcn_readlane(other, s.slot[t]);
          const int64_t *pidx = kSecond ? (kOwnIsQuery ? p->pidx_v : p->pidx_o) : (kOwnIsQuery ? p->pidx_k : p->pidx_q);
          const int64_t count = kSecond ? (kOwnIsQuery ? p->n_v_blocks : p->n_o_blocks) : (kOwnIsQuery ? p->n_k_blocks : p->n_q_blocks);
          const int64_t at = lane < n ? pidx[place * n + lane] : -1;
          on = (uint32_t)__ballot(at >= 0 && at < count);
          mine = (int)at;
        }
        for (uint32_t left = on; left != 0; left &= left - 1) {
          const int h = __builtin_ctz(left);
          T::copy_piece(tensor, __builtin_amdgcn_readlane(mine, h), dst + t * T::kBlock + h * T::kPiece, offset, lane);
        }
      }
      if constexpr (kSecond) s.have[t] = (s.have[t] & 0xffu) | on << 8;
      else s.have[t] = (s.have[t] & 0xff00u) | on;
    }
  }

  // acc = rows of the step's blocks of the first (second) tensor x own rows, and out += their columns^T x weights
  template <typename Tr, bool kSecond, typename Acc>
  __device__ static inline void multiply_rows(Acc (&acc)[NB], const Step &s, const typename T::RowReader &rows,
                                              const OwnOperand<Tr, SBS, NS, kHalves, kSecond> &own, int lane) {
    if constexpr (kSome) {
      uint32_t have[NB];
#pragma unroll
      for (int t = 0; t < NB; ++t) have[t] = (kSecond ? s.have[t] >> 8 : s.have[t]) & own.rows.there;
      product_some_rows<Tr, SBS, NS, NB>(acc, rows, own.rows, have, lane);
    } else {
      product_rows<Tr, SBS, NS, NB, kHalves, kOwnIsQuery, kSecond>(acc, rows, own);
    }
  }
  template <typename Tr, bool kSecond, int kScores, typename Acc>
  __device__ static inline void multiply_cols(Acc (&out)[NS], const Step &s, const typename T::ColReader &cols,
                                              const Weights<Tr, kScores> &w) {
    if constexpr (kSome) {
      uint32_t have[NB];
#pragma unroll
      for (int t = 0; t < NB; ++t) have[t] = kSecond ? s.have[t] >> 8 : s.have[t];
      product_some_cols<Tr, SBS, NS, NB>(out, cols, w, have);
    } else {
      product_cols<Tr, SBS, NS, NB, kHalves>(out, cols, w);
    }
  }

  // Bias, mask, causal predicate and missing blocks of a special step, in this order (blksprs/ops/flash_attention.py
  // :1110-1150).  sv: the step's scores up to the factor cc of the exponential, block after block; with a bias they leave
  // multiplied by qk_scale and complete, and cc is 1.  me: this lane's own row; group: lane / SBS.
  template <typename Tr>
  __device__ inline void finish_scores(const Step &s, float *sv, float qk_scale, int me, int group) const {
    // fp32 up to head dimension 64: what the lane's addresses in a mask or bias block have in common is formed here and not in front
    // of the walk, where it takes registers that dK / dV does not have (BigBird: 53.4 -> 51.9 us; dK / dV at 128, which spills
    // others then, 134 -> 140)
    if constexpr (ES == 4 && NS <= 2) asm volatile("" : "+v"(me), "+v"(group));
    constexpr int kRegs = SBS == 32 ? 16 : 4;
    constexpr int kSide = kHalves * SBS;  // of a block of the layout, for mask and bias
    const late_args_t p = late_args();
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      float *v = sv + kRegs * t;
      // first row and column of this block's part of the layout's mask and bias blocks
      const int mine0 = (int)own % kHalves * SBS, theirs0 = s.other[t] % kHalves * SBS;
      const int corner = kOwnIsQuery ? mine0 * kSide + theirs0 : theirs0 * kSide + mine0;
      // registers 4 w .. 4 w + 3 belong to partner rows 8 w + 4 group .. + 3
      if (p->bias) {
        const char *blk = static_cast<const char *>(p->bias) + ((int64_t)s.bias[t] * (kSide * kSide) + corner) * ES;
#pragma unroll
        for (int w = 0; w < kRegs / 4; ++w)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int theirs = 8 * w + 4 * group + i;
            const int at = kOwnIsQuery ? me * kSide + theirs : theirs * kSide + me;
            float bias_value = 0.f;
            if (s.bias[t] >= 0) {
              if constexpr (ES == 4) bias_value = reinterpret_cast<const float *>(blk)[at];
              else bias_value = Tr::widen(reinterpret_cast<const uint16_t *>(blk)[at]);
            }
            v[4 * w + i] = v[4 * w + i] * qk_scale + bias_value * kLog2e;
          }
      }
      if (s.mask[t] >= 0) {
        const uint8_t *blk = static_cast<const uint8_t *>(p->mask) + (int64_t)s.mask[t] * (kSide * kSide) + corner;
        uint32_t mw[kRegs / 4];
#pragma unroll
        for (int w = 0; w < kRegs / 4; ++w) {
          if constexpr (kOwnIsQuery) {
            mw[w] = *reinterpret_cast<const uint32_t *>(blk + me * kSide + 8 * w + 4 * group);
          } else {
            const uint8_t *col = blk + (8 * w + 4 * group) * kSide + me;
            mw[w] = col[0] | (uint32_t)col[kSide] << 8 | (uint32_t)col[2 * kSide] << 16 | (uint32_t)col[3 * kSide] << 24;
          }
        }
#pragma unroll
        for (int r = 0; r < kRegs; ++r)
          if ((mw[r / 4] >> (8 * (r % 4))) & 0xffu) v[r] = -INFINITY;
      }
      if (p->causal_lengths) {
        const int mine = (int)own * SBS + me;
#pragma unroll
        for (int r = 0; r < kRegs; ++r) {
          const int theirs = s.other[t] * SBS + 8 * (r / 4) + 4 * group + r % 4;
          if ((kOwnIsQuery ? theirs > mine : theirs < mine) || mine >= seq_len || theirs >= seq_len) v[r] = -INFINITY;
        }
      }
      if (t >= s.count) {
#pragma unroll
        for (int r = 0; r < kRegs; ++r) v[r] = -INFINITY;
      }
    }
  }
};

// Whether all blocks of all rows have all their head slices, as many of q / k as of v / o: the block counts say so.  Of the output
// only the backward kernels read, and query blocks that attend to nothing may go without.
inline bool all_slices(const bsa_attn_args &a, bool backward) {
  if (a.nh != a.nhv || a.n_q_blocks != a.B * a.nq * a.nh || a.n_k_blocks != a.B * a.nk * a.nh || a.n_v_blocks != a.B * a.nk * a.nhv)
    return false;
  return !backward || a.n_o_blocks == a.B * a.nq * a.nhv || a.o_rows_whole != 0;
}

// Whether the kernels for blocks of 16 and 32 take these arguments (up to the head slices they are built for).  Blocks of 64
// are for them only in fp32 (16-bit operands: attn_mfma.hip, attn_bwd_mfma.hip) and with all slices there.
inline bool small_applies(const bsa_attn_args &a, bool backward) {
  if (a.sbs != 16 && a.sbs != 32 && !(a.sbs == 64 && a.dtype == BSA_F32 && all_slices(a, backward))) return false;
  // the forward kernel takes the row maximum before the scale is applied
  if (!(a.scale > 0.f) || a.scale > 3.0e38f) return false;
  const int64_t most = a.sbs == 64 ? 0x3fffffffLL : 0x7fffffffLL;  // indices (of halves) and positions are 32-bit numbers
  if (a.n_q_blocks > most || a.n_k_blocks > most || a.n_v_blocks > most || a.n_o_blocks > most ||
      a.n_mask_blocks > most || a.n_bias_blocks > most || a.nq * a.sbs > most || a.nk * a.sbs > most)
    return false;
  // slices are copied into LDS and stored 16 bytes at a time, mask rows are read 4 bytes at a time: a tensor that starts in
  // the middle of such a piece (a view into a larger buffer) takes the kernels that load through registers
  const uintptr_t starts = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.k) |
                           reinterpret_cast<uintptr_t>(a.v) | reinterpret_cast<uintptr_t>(a.o) |
                           reinterpret_cast<uintptr_t>(a.d_o) | reinterpret_cast<uintptr_t>(a.dq) |
                           reinterpret_cast<uintptr_t>(a.dk) | reinterpret_cast<uintptr_t>(a.dv) |
                           reinterpret_cast<uintptr_t>(a.dbias);
  if ((starts & 15) != 0 || (reinterpret_cast<uintptr_t>(a.mask) & 3) != 0) return false;
  const int64_t slices = a.nh > a.nhv ? a.nh : a.nhv;
  return slices >= 1 && slices <= 128 / a.sbs;
}

// Waves that share one row of a launch of `rows` rows, each walking every second or fourth entry of its list.  A launch
// lasts as long as the serial walk of its longest lists, and the last round of a launch of few rounds is mostly empty:
// shorter shares help until their prologue (four dependent loads) costs more than the walk.  bf16 forward, one / two /
// four waves, us (sbs 32, head dimension 64; every block of a half, causal, windows of 9 blocks, BigBird):
//     512 rows of 32 blocks:   18.3 / 12.2 / 10.1   31.2 / 18.6 / 12.4   13.1 / 9.5 / 8.6      34.8 / 20.5 / 14.5
//    1024 rows of 32 blocks:   19.6 / 14.8 / 14.6   32.4 / 19.9 / 13.8   13.7 / 10.6 / 10.7    35.8 / 23.5 / 19.2
//    4096 rows of 64 blocks:   66.1 / 64.1 / 69.1   67.3 / 45.8 / 51.4   26.1 / 26.8 / 35.3    96.3 / 73.6 / 72.9
//    8192 rows of 64 blocks:    138 / 129 / 139     81.8 / 86.7 / 98.6   42.6 / 47.3 / 65.4     131 / 117 / 127
//   16384 rows of 64 blocks:    333 / 261 / 280      152 / 166 / 195     76.5 / 89.8 / 126      233 / 249 / 251
// Up to 512 rows four are best throughout; at 1024 they are for half of the layouts, and at head dimension 128 two are (22.9
// against 27.7 for every block of a half).  From 8192 rows it depends on the layout, which the rule does not look at:
// short and causal lists want one wave, long lists of about equal length two.  Uneven lists: attn_shares.hip.
// fp32: always four, for four partial sums: with two and one, O is 14 and 38 % further from 64 bits, dK and dV of a
// causal layout 26 and 50 % (1024 keys, sbs 16).  Never more waves than a list of all partners has steps.
template <int ES>
inline int waves_per_row(int64_t rows, int64_t partners, int blocks_per_step) {
  const int64_t steps = cdiv(partners, (int64_t)blocks_per_step);
  const int most = steps >= 3 ? 4 : steps == 2 ? 2 : 1;
  const int wanted = ES == 4 || rows <= 512 ? 4 : rows <= 8192 ? 2 : 1;
  return wanted < most ? wanted : most;
}

// The row of a wave.  Workgroup g runs on XCD g % 8, each with its own L2.  Of B batch entries an XCD takes B / 8 whole
// ones, whose partner blocks no other XCD reads, and every eighth row of the B % 8 that are left.  It walks the rows of all
// its entries together, eight neighbours (whose lists overlap) of one entry, then eight of the next, in the order in which
// a causal layout's lists get shorter (the last query blocks, the first key blocks first): a launch lasts as long as its
// longest lists, and there none starts late.  Entry by entry, the long lists of an XCD's last entry start behind the short ones
// of the others, 6144 rows (sbs 32, windows of 33 blocks, a quarter of the rows beyond the sequences): 79 / 95 us
// (forward / dQ) against 70 / 89; 4128 rows (sbs 16, causal): 57.5 against 48.5; 8192 rows (sbs 32, causal): 172 / 212
// against 156 / 198; two long columns among short ones in 13 entries (dK / dV, where XCDs also differed in work): 97 against
// 67; lists of equal lengths: the same.  Rows of one entry on several XCDs where whole entries would do: 5 to 14 % slower
// (their partner blocks pass several L2s).  List lengths are not looked at: where the first query blocks have the longest lists
// (global rows of a BigBird layout) these start last, unless the launch has shares (attn_shares.hip).
// Entries of fewer than eight rows are taken as they are: with eight places each, most of them empty, an entry of one row
// (64 key blocks, 4096 entries, head dimension 64, sbs 32, fp32, forward) took 3.17 ms, now 0.77; bf16 0.72, now 0.38.
// Item `item` of XCD `xcd` in that order; whether the row is there.
__host__ __device__ inline bool row_of_item(uint32_t xcd, uint32_t item, int64_t batches, int64_t rows_per_batch, bool last_first,
                                            int64_t &b, int64_t &own) {
  // up to eight rows of every entry: as many items for each of an XCD's own entries, one for each shared one (the last of all)
  const uint32_t near = rows_per_batch < 8 ? (uint32_t)rows_per_batch : 8, entries = (uint32_t)(batches >> 3);
  const uint32_t own_items = entries * near, items = own_items + ((uint32_t)batches & 7);
  const uint32_t eight = item / items, rest = item - eight * items;
  if (rest < own_items) {
    const uint32_t entry = near == 8 ? rest >> 3 : rest / near;
    b = (int64_t)xcd * entries + entry;
    own = (int64_t)eight * 8 + (rest - entry * near);
  } else {
    b = (int64_t)entries * 8 + (rest - own_items);
    own = (int64_t)eight * 8 + ((xcd + rest + eight) & 7);
  }
  const bool there = own < rows_per_batch;
  if (!there) b = own = 0;
  if (last_first) own = rows_per_batch - 1 - own;
  return there;
}

// Items of each XCD
inline int64_t row_items(int64_t batches, int64_t rows_per_batch) {
  return cdiv(rows_per_batch, (int64_t)8) * ((batches >> 3) * (rows_per_batch < 8 ? rows_per_batch : 8) + (batches & 7));
}

// What a launch knows of the shares of its rows (bsa_attn_shares); groups NULL: `split` waves for every row
struct Shares {
  const int32_t *groups;
  float *partials;  // one per slot (and half, where blocks are halves of the layout's)
};

struct RowOfWave {
  int64_t b, own;
  int part, parts;   // this wave walks every parts-th entry of the row's list, from entry `part` on
  int place, waves;  // among the waves of this workgroup that share the row
  int slot;          // the workgroup's sum is one of several: where it goes; -1: it is the row's
  bool there;
  __device__ inline RowOfWave(const Shares &shares, int halves, int64_t batches, int64_t rows_per_batch, bool last_first, int wave,
                              int waves_of_group, int split) {
    if (shares.groups) {
      // groups of an XCD are eight (XCDs) apart, also with two halves each
      const uint32_t xcd = blockIdx.x & 7, turn = blockIdx.x >> 3;
      const int32_t *g = shares.groups + (int64_t)((turn / halves) * 8 + xcd) * BSA_SHARE_INTS;
      own = first_lane(g[wave]);
      b = first_lane(g[4 + wave]);
      there = own >= 0 && own < rows_per_batch / halves && b >= 0 && b < batches;
      if (!there) b = own = 0;
      own = own * halves + turn % halves;
      parts = first_lane(g[9]);
      waves = parts < waves_of_group ? parts : waves_of_group;
      place = wave % waves;
      part = first_lane(g[8]) + place;
      const int s = first_lane(g[10]);
      slot = s < 0 ? -1 : s * halves + (int)(turn % halves);
    } else {
      part = place = wave % split;
      parts = waves = split;
      slot = -1;
      there = row_of_item(blockIdx.x & 7, (blockIdx.x >> 3) * (waves_of_group / split) + wave / split, batches, rows_per_batch,
                          last_first, b, own);
    }
  }
};

// Sums of a row that several workgroups share: accumulators as they lie, 16 bytes per lane
template <int NS, int kRegs, typename Acc, typename Float>
__device__ static inline void leave_partial(const Acc (&acc)[NS], Float *mine, int lane) {
#pragma unroll
  for (int h = 0; h < NS; ++h)
#pragma unroll
    for (int r = 0; r < kRegs; r += 4)
      *reinterpret_cast<f32x4 *>(mine + ((h * kRegs + r) / 4 * 64 + lane) * 4) =
          f32x4{acc[h][r], acc[h][r + 1], acc[h][r + 2], acc[h][r + 3]};
}
template <int NS, int kRegs, typename Acc>
__device__ static inline void add_partial(Acc (&acc)[NS], const float *other, int lane) {
#pragma unroll
  for (int h = 0; h < NS; ++h)
#pragma unroll
    for (int r = 0; r < kRegs; r += 4) {
      const f32x4 v = *reinterpret_cast<const f32x4 *>(other + ((h * kRegs + r) / 4 * 64 + lane) * 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[h][r + i] += v[i];
    }
}

inline int64_t row_groups(int64_t batches, int64_t rows_per_batch, int waves, int split) {
  return cdiv(row_items(batches, rows_per_batch), (int64_t)(waves / split)) * 8;
}
// a launch has fewer than 2^32 threads; what is more goes to the kernels that give a workgroup a row
inline bool fits_launch(int64_t groups, int waves) { return groups * waves * 64 < ((int64_t)1 << 32); }

}  // namespace small
}  // namespace bsa
