// Pieces shared by the 16-bit attention kernels for blocks of 16 and 32 (attn_small_fwd.hip, attn_small_bwd.hip):
// LDS layout of a block slice, operand fragments, asynchronous copies of block slices, waits.
//
// A block slice (SBS x SBS 16-bit elements, 512 or 2048 contiguous bytes in memory) lies row-major in LDS, the
// 16-byte chunks of a row exchanged by chunk_swizzle(row).  It is read both ways: rows as they lie (contraction over
// the head dimension: one 128-bit read per fragment) and columns through the transposing LDS read (contraction over
// the sequence).  Products use v_mfma_f32_32x32x16 for blocks of 32 and v_mfma_f32_16x16x32 for blocks of 16, where
// the 32 contracted values of a score product are two head slices and those of a value product two partner blocks.
#pragma once
#include "attn_mfma_common.h"

namespace bsa {
namespace small {

using namespace mfma;

struct SBf16 : MBf16 {
  __device__ static f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
struct SF16 : MF16 {
  __device__ static f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

// Waits until at most N vector memory operations of the wave are outstanding.  The clobber keeps LDS reads behind it.
template <int N>
__device__ static inline void wait_vmem() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// LDS reads issued so far have returned: their buffer may be copied over
__device__ static inline void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// XOR on the 16-byte chunk index of row r of a block slice.  Rows of 64 bytes (SBS 32): eight consecutive rows read at
// one chunk index fall on different chunks of a 128-byte bank period and sixteen of a 256-byte one, and the four rows
// r .. r + 3 (r a multiple of 4) of a transposing read use different halves of their rows.  Rows of 32 bytes (SBS 16):
// the same for the row reads; a transposing read of four rows covers 128 consecutive bytes anyway.  Depends on
// r % 16 only.
template <int SBS>
__device__ static inline int chunk_swizzle(int r) {
  if constexpr (SBS == 32) return ((((r >> 1) ^ (r >> 3)) & 1) << 1) | ((r >> 2) & 1);
  else return ((r >> 2) ^ (r >> 3)) & 1;
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

// Geometry of one wave's tile: NB partner blocks of NS head slices each, slice h of block t at piece t * NS + h.
template <int SBS, int NS, int NB>
struct Tile {
  static constexpr int kPiece = SBS * SBS * 2;
  static constexpr int kBlock = NS * kPiece;     // one partner block
  static constexpr int kBytes = NB * kBlock;
  static constexpr int kBlockCopies = (kBlock + 1023) / 1024;
  static constexpr int kCopies = NB * kBlockCopies;  // asynchronous copies per tile

  // this lane's source offset for a copy that fills LDS linearly (all KiB of a block share it: the swizzle depends on
  // row % 16 only, and a KiB holds 16 rows of 64 bytes or two slices of 16 rows of 32 bytes)
  __device__ static inline uint32_t source_offset(int lane) {
    if constexpr (SBS == 32) {
      const int r = lane >> 2;
      return (uint32_t)(r * 64 + (((lane & 3) ^ chunk_swizzle<32>(r)) << 4));
    } else {
      const int r = (lane & 31) >> 1;
      return (uint32_t)((lane >> 5) * 512 + r * 32 + (((lane & 1) ^ chunk_swizzle<16>(r)) << 4));
    }
  }

  // Requests block t of the tile, all of whose slices are there and lie one behind the other from packed index idx:
  // kBlockCopies asynchronous copies.
  __device__ static inline void copy_block(const char *tensor, int idx, char *dst, uint32_t offset, int lane) {
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

  // The same for a block whose slices are missing (zeros) or lie apart: synchronous, slice by slice.  pidx: the packed
  // indices of the block's n_slices slices (wave uniform).
  __device__ static inline void gather_block(const char *tensor, const int64_t *pidx, int n_slices, int64_t n_blocks,
                                             char *dst, uint32_t offset, int lane) {
    for (int h = 0; h < NS; ++h) {
      const int64_t idx = h < n_slices ? pidx[h] : -1;
      const bool on = idx >= 0 && idx < n_blocks;
#pragma unroll
      for (int i = 0; i < kPiece; i += 1024) {
        u32x4 v{0u, 0u, 0u, 0u};
        if (SBS == 32 || lane < 32) {
          if (on) v = *reinterpret_cast<const u32x4 *>(tensor + idx * kPiece + i + offset);
          *reinterpret_cast<u32x4 *>(dst + h * kPiece + i + lane * 16) = v;
        }
      }
    }
  }

  // ---- row fragments (contraction over the head dimension) ----
  // SBS 32: fragment f of a block = values 16 f .. + 15 (2 per slice), this lane row lane % 32, values 8 (lane / 32) .. + 7.
  // SBS 16: fragment f = slices 2 f, 2 f + 1, this lane row lane % 16, 8 values of slice 2 f + lane / 32 from
  // 8 (lane / 16 % 2); behind the last slice of an odd count the upper half of the lanes hold zeros.  (The product of 16
  // values for that slice is not used: its sum, fed by a product of 32 values right in front of it, came out without it.)
  static constexpr int kFrags = SBS == 32 ? 2 * NS : (NS + 1) / 2;
  static constexpr bool kHalfLast = SBS == 16 && (NS & 1);

  struct RowReader {
    const char *base0, *base1;  // SBS 32: even and odd fragments
    bool beyond;                // SBS 16: this lane's half of the last fragment of an odd slice count is beyond the block
    __device__ RowReader(const char *lds, int lane) : beyond(lane >= 32) {
      if constexpr (SBS == 32) {
        const int r = lane & 31, c = (lane >> 5) ^ chunk_swizzle<32>(r);
        base0 = lds + r * 64 + (c << 4);
        base1 = lds + r * 64 + ((c ^ 2) << 4);
      } else {
        const int r = lane & 15, g = lane >> 4;
        base0 = base1 = lds + (g >> 1) * kPiece + r * 32 + (((g & 1) ^ chunk_swizzle<16>(r)) << 4);
      }
    }
    __device__ u32x4 frag(int t, int f) const {
      if constexpr (SBS == 32) return *reinterpret_cast<const u32x4 *>(((f & 1) ? base1 : base0) + (t * NS + (f >> 1)) * kPiece);
      u32x4 v = *reinterpret_cast<const u32x4 *>(base0 + (t * NS + 2 * f) * kPiece);
      if (kHalfLast && f == kFrags - 1 && beyond) v = u32x4{0u, 0u, 0u, 0u};
      return v;
    }
  };

  // ---- column fragments (contraction over the rows of the partner blocks) ----
  // SBS 32: fragment m of block t, slice h: column lane % 32, rows 16 m + 4 kg .. + 3 and 16 m + 8 + 4 kg .. + 3
  // (kg = lane / 32): the rows whose values a lane holds in accumulator registers 8 m .. 8 m + 7.
  // SBS 16: fragment of blocks t and t + 1 (zeros for t + 1 == NB), slice h: column lane % 16, rows
  // 4 (lane / 16) .. + 3 of either block: the rows of accumulator registers 0 .. 3 of the two blocks.
  struct ColReader {
    const char *base0, *base1;  // SBS 32: first and second four rows of a fragment
    __device__ ColReader(const char *lds, int lane) {
      const int s = lane & 15;
      if constexpr (SBS == 32) {
        const int r = 4 * (lane >> 5) + (s >> 2), c = 2 * ((lane >> 4) & 1) + ((s & 3) >> 1);
        base0 = lds + r * 64 + ((c ^ chunk_swizzle<32>(r)) << 4) + ((s & 1) << 3);
        base1 = lds + (r + 8) * 64 + ((c ^ chunk_swizzle<32>(r + 8)) << 4) + ((s & 1) << 3);
      } else {
        const int r = 4 * (lane >> 4) + (s >> 2), c = (s & 3) >> 1;
        base0 = base1 = lds + r * 32 + ((c ^ chunk_swizzle<16>(r)) << 4) + ((s & 1) << 3);
      }
    }
    __device__ u32x4 frag(int t, int m, int h) const {
      u32x2 lo, hi;
      if constexpr (SBS == 32) {
        lo = read_tr(base0 + (t * NS + h) * kPiece + m * 1024);
        hi = read_tr(base1 + (t * NS + h) * kPiece + m * 1024);
      } else {
        lo = read_tr(base0 + ((t + 2 * m) * NS + h) * kPiece);
        hi = read_tr(base0 + ((t + 2 * m + 1) * NS + h) * kPiece);
      }
      return u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  };
};

// One block's own rows as the other operand of the score products, in registers for the whole walk (the same values
// per lane as RowReader's fragments).
template <int SBS, int NS>
struct OwnRows {
  using T = Tile<SBS, NS, SBS == 32 ? 1 : 2>;
  u32x4 fr[T::kFrags];

  // pidx: packed indices of the block's slices, n_slices of them are there
  __device__ inline void load(const void *tensor, const int64_t *pidx, int n_slices, int64_t n_blocks, int lane) {
    const char *p = static_cast<const char *>(tensor);
    if constexpr (SBS == 32) {
#pragma unroll
      for (int h = 0; h < NS; ++h) {
        const int64_t idx = h < n_slices ? pidx[h] : -1;
        const bool on = idx >= 0 && idx < n_blocks;
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          fr[2 * h + m] = u32x4{0u, 0u, 0u, 0u};
          if (on) fr[2 * h + m] = *reinterpret_cast<const u32x4 *>(p + idx * T::kPiece + (lane & 31) * 64 + (2 * m + (lane >> 5)) * 16);
        }
      }
    } else {
      const int g = lane >> 4;
#pragma unroll
      for (int f = 0; f < T::kFrags; ++f) {
        const int h = 2 * f + (g >> 1);
        const int64_t idx = h < n_slices ? pidx[h] : -1;
        fr[f] = u32x4{0u, 0u, 0u, 0u};
        if (idx >= 0 && idx < n_blocks)
          fr[f] = *reinterpret_cast<const u32x4 *>(p + idx * T::kPiece + (lane & 15) * 32 + (g & 1) * 16);
      }
    }
  }
};

// Makes the compiler wait for the loads of the own rows here: left to their first use, the wait sits inside the loop and
// is for every load in flight, each time round.
template <int SBS, int NS>
__device__ static inline void settle(OwnRows<SBS, NS> &own) {
#pragma unroll
  for (int f = 0; f < OwnRows<SBS, NS>::T::kFrags; ++f) asm volatile("" : "+v"(own.fr[f]));
}

// acc (per partner block t) = partner rows x own rows over all head slices: acc[t] belongs to this lane's own row
// (lane % SBS) and partner rows 8 (r / 4) + 4 (lane / 32) + r % 4 (SBS 32) or 4 (lane / 16) + r (SBS 16).
template <typename Tr, int SBS, int NS, int NB, typename Acc>
__device__ static inline void product_rows(Acc (&acc)[NB], const typename Tile<SBS, NS, NB>::RowReader &rows,
                                           const OwnRows<SBS, NS> &own) {
  using T = Tile<SBS, NS, NB>;
#pragma unroll
  for (int t = 0; t < NB; ++t) {
#pragma unroll
    for (int r = 0; r < (SBS == 32 ? 16 : 4); ++r) acc[t][r] = 0.f;
#pragma unroll
    for (int f = 0; f < T::kFrags; ++f) {
      if constexpr (SBS == 32) acc[t] = Tr::mfma(rows.frag(t, f), own.fr[f], acc[t]);
      else acc[t] = Tr::mfma16(rows.frag(t, f), own.fr[f], acc[t]);
    }
  }
}

// out[h] += partner columns^T x weights, weights packed from accumulator registers: w[m] holds registers 8 m .. 8 m + 7
// of the NB blocks' accumulators, one after the other
template <typename Tr, int SBS, int NS, int NB, typename Acc>
__device__ static inline void product_cols(Acc (&out)[NS], const typename Tile<SBS, NS, NB>::ColReader &cols,
                                           const u32x4 (&w)[SBS == 32 ? 2 * NB : NB / 2]) {
#pragma unroll
  for (int h = 0; h < NS; ++h)
#pragma unroll
    for (int m = 0; m < (SBS == 32 ? 2 * NB : NB / 2); ++m) {
      if constexpr (SBS == 32) out[h] = Tr::mfma(cols.frag(m >> 1, m & 1, h), w[m], out[h]);
      else out[h] = Tr::mfma16(cols.frag(0, m, h), w[m], out[h]);
    }
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

}  // namespace small
}  // namespace bsa
