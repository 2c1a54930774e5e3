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

// One wave's walk over the list of partner blocks of one block of its own: key blocks of a query block, or (kOwnIsQuery
// false) query blocks of a key block.
//
// The list is read 64 entries at a time, one per lane: the partner block, the packed indices of its first slices (of K
// and V, or of Q and dO), its mask and bias block.  Entries the causal predicate rules out as a whole are left out of
// `live`; `special` marks those whose scores need more than the scale; `apart` says that some block's slices are
// missing or do not lie one behind the other.
template <int SBS, int NS, int NB, bool kOwnIsQuery>
struct Walk {
  using T = Tile<SBS, NS, NB>;
  int64_t b, own;          // batch entry, own block
  int end, base, seq_len;  // end of the list, first entry of the window; valid length of a causal sequence
  int other, first_a, first_b, mask, bias;  // of this lane's entry
  uint64_t live, special;
  bool apart;

  // a step: how many entries it takes and their places in the window, and, if special, their facts (the window may be
  // another one by the time the scores are formed)
  struct Step {
    int count, slot[NB], other[NB], mask[NB], bias[NB];
    bool special, apart;
  };

  // part of parts: the contiguous share of the list that this wave walks
  __device__ inline void start(const bsa_attn_args &a, int64_t b_, int64_t own_, bool there, int part, int parts) {
    b = b_, own = own_;
    seq_len = 0x7fffffff;
    if (a.causal_lengths) {
      const int64_t len = a.causal_lengths[b];
      seq_len = len < 0 ? 0 : (len > 0x7fffffffLL ? 0x7fffffff : (int)len);
    }
    const int32_t *offsets = (kOwnIsQuery ? a.key_offsets : a.query_offsets) + b * (kOwnIsQuery ? a.nq : a.nk) + own;
    int begin = first_lane(offsets[0]);
    end = first_lane(offsets[1]);
    if (parts > 1) {
      const int64_t n = end - begin;
      end = begin + (int)(n * (part + 1) / parts);
      begin += (int)(n * part / parts);
    }
    if (!there || (int)own * SBS >= seq_len) end = begin;
    base = begin - 64;
    other = first_a = first_b = 0;
    mask = bias = -1;
    live = special = 0;
    apart = false;
  }

  __device__ inline void refill(int lane) {
    const late_args_t p = late_args();
    base += 64;
    const int e = base + lane;
    bool in = e < end;
    other = in ? (kOwnIsQuery ? p->key_indices : p->query_indices)[e] : 0;
    const bool causal = p->causal_lengths != nullptr;
    in = in && !(causal && ((kOwnIsQuery ? other > (int)own : other < (int)own) || other * SBS >= seq_len));
    const int64_t place = b * (kOwnIsQuery ? p->nk : p->nq) + other;
    bool far = p->nh != NS || p->nhv != NS;
    if (in && !far) {
      const int64_t *pa = (kOwnIsQuery ? p->pidx_k : p->pidx_q) + place * NS;
      const int64_t *pb = (kOwnIsQuery ? p->pidx_v : p->pidx_o) + place * NS;
      const int64_t a0 = pa[0], b0 = pb[0];
      far = a0 < 0 || b0 < 0 || a0 + NS > (kOwnIsQuery ? p->n_k_blocks : p->n_q_blocks) ||
            b0 + NS > (kOwnIsQuery ? p->n_v_blocks : p->n_o_blocks);
#pragma unroll
      for (int h = 1; h < NS; ++h) far = far || pa[h] != a0 + h || pb[h] != b0 + h;
      first_a = (int)a0;
      first_b = (int)b0;
    }
    apart = __any(in && far);
    bool extra = causal && (other == (int)own || ((int)own + 1) * SBS > seq_len || (other + 1) * SBS > seq_len);
    const int64_t pair = kOwnIsQuery ? (b * p->nq + own) * p->nk + other : (b * p->nq + other) * p->nk + own;
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
      s.count += lowest ? 1 : 0;
      live ^= lowest;
      taken |= lowest;
    }
    s.apart = apart;
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
  // asynchronous copies are on their way.  To be called before the next take().  Blocks that are not there (the last
  // step of a list) become zeros.
  template <bool kSecond>
  __device__ inline bool copy(const Step &s, const char *tensor, char *dst, uint32_t offset, int lane) const {
    if (!s.apart) {
#pragma unroll
      for (int t = 0; t < NB; ++t)
        if (NB == 1 || t < s.count)
          T::copy_block(tensor, __builtin_amdgcn_readlane(kSecond ? first_b : first_a, s.slot[t]), dst + t * T::kBlock, offset, lane);
      if (NB == 1 || s.count == NB) return true;
    }
    const late_args_t p = late_args();
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      if (!s.apart && t < s.count) continue;
      const int n = t < s.count ? (int)(kSecond ? p->nhv : p->nh) : 0;
      const int64_t place = b * (kOwnIsQuery ? p->nk : p->nq) + __builtin_amdgcn_readlane(other, s.slot[t]);
      const int64_t *pidx = kSecond ? (kOwnIsQuery ? p->pidx_v : p->pidx_o) : (kOwnIsQuery ? p->pidx_k : p->pidx_q);
      const int64_t count = kSecond ? (kOwnIsQuery ? p->n_v_blocks : p->n_o_blocks) : (kOwnIsQuery ? p->n_k_blocks : p->n_q_blocks);
      T::gather_block(tensor, pidx + place * n, n, count, dst + t * T::kBlock, offset, lane);
    }
    return false;
  }

  // Bias, mask, causal predicate and missing blocks of a special step, in this order (blksprs/ops/flash_attention.py
  // :1110-1150).  sv: the step's scores up to the factor cc of the exponential, block after block; with a bias they leave
  // multiplied by qk_scale and complete, and cc is 1.  me: this lane's own row; group: lane / SBS.
  template <typename Tr>
  __device__ inline void finish_scores(const Step &s, float *sv, float qk_scale, int me, int group) const {
    constexpr int kRegs = SBS == 32 ? 16 : 4;
    const late_args_t p = late_args();
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      float *v = sv + kRegs * t;
      // registers 4 w .. 4 w + 3 belong to partner rows 8 w + 4 group .. + 3
      if (p->bias) {
        const char *blk = static_cast<const char *>(p->bias) + (int64_t)s.bias[t] * T::kPiece;
#pragma unroll
        for (int w = 0; w < kRegs / 4; ++w) {
          u32x2 bw{0u, 0u};
          if (s.bias[t] >= 0) {
            if constexpr (kOwnIsQuery) {
              bw = *reinterpret_cast<const u32x2 *>(blk + me * (2 * SBS) + 16 * w + 8 * group);
            } else {
              const uint16_t *col = reinterpret_cast<const uint16_t *>(blk) + (8 * w + 4 * group) * SBS + me;
              bw = u32x2{col[0] | (uint32_t)col[SBS] << 16, col[2 * SBS] | (uint32_t)col[3 * SBS] << 16};
            }
          }
#pragma unroll
          for (int i = 0; i < 4; ++i)
            v[4 * w + i] = v[4 * w + i] * qk_scale + Tr::widen((uint16_t)(bw[i / 2] >> (16 * (i % 2)))) * kLog2e;
        }
      }
      if (s.mask[t] >= 0) {
        const uint8_t *blk = static_cast<const uint8_t *>(p->mask) + (int64_t)s.mask[t] * (SBS * SBS);
        uint32_t mw[kRegs / 4];
#pragma unroll
        for (int w = 0; w < kRegs / 4; ++w) {
          if constexpr (kOwnIsQuery) {
            mw[w] = *reinterpret_cast<const uint32_t *>(blk + me * SBS + 8 * w + 4 * group);
          } else {
            const uint8_t *col = blk + (8 * w + 4 * group) * SBS + me;
            mw[w] = col[0] | (uint32_t)col[SBS] << 8 | (uint32_t)col[2 * SBS] << 16 | (uint32_t)col[3 * SBS] << 24;
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

// Whether the kernels for blocks of 16 and 32 take these arguments (up to the head slices they are built for)
inline bool small_applies(const bsa_attn_args &a) {
  if (a.sbs != 16 && a.sbs != 32) return false;
  if (a.dtype != BSA_BF16 && a.dtype != BSA_F16) return false;
  // the forward kernel takes the row maximum before the scale is applied
  if (!(a.scale > 0.f) || a.scale > 3.0e38f) return false;
  const int64_t most = 0x7fffffffLL;  // indices and positions are 32-bit numbers
  if (a.n_q_blocks > most || a.n_k_blocks > most || a.n_v_blocks > most || a.n_o_blocks > most ||
      a.n_mask_blocks > most || a.n_bias_blocks > most || a.nq * a.sbs > most || a.nk * a.sbs > most)
    return false;
  const int64_t slices = a.nh > a.nhv ? a.nh : a.nhv;
  return slices >= 1 && slices <= 128 / a.sbs;
}

// Waves that share one row of a launch of `rows` rows, each walking a contiguous part of its list.  A launch lasts as
// long as the serial walk of its longest lists, and the last round of a launch of few rounds is mostly empty: shorter
// shares help until their prologue (four dependent loads) costs more than the walk.  Forward, 64 rows (8 key blocks
// each, sbs 32): 9.6 us with two waves per row, 8.1 with four; 4128 rows (sbs 16, causal, up to 65 steps): 80 / 60 / 61 us
// with one, two, four; 6144 rows (sbs 32, 33 steps): 83 / 75 / 82.
inline int waves_per_row(int64_t rows) { return rows <= 512 ? 4 : rows <= 8192 ? 2 : 1; }

// The row of a wave.  XCD c (workgroup g runs on XCD g % 8) takes a contiguous eighth of the rows, so that the waves in
// flight on one L2 share few batch entries' partner blocks; inside a batch entry the long rows of a causal layout (the
// last query blocks, the first key blocks) come first.
struct RowOfWave {
  int64_t b, own;
  int part;
  bool there;
  __device__ inline RowOfWave(int64_t batches, int64_t rows_per_batch, bool last_first, int wave, int waves, int split) {
    const int64_t group = (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const int64_t item = group * (waves / split) + wave / split;
    part = wave % split;
    there = item < batches * rows_per_batch;
    b = there ? item / rows_per_batch : 0;
    own = there ? item % rows_per_batch : 0;
    if (last_first) own = rows_per_batch - 1 - own;
  }
};
inline unsigned row_groups(int64_t rows, int waves, int split) {
  return (unsigned)(cdiv(cdiv(rows, (int64_t)(waves / split)), (int64_t)8) * 8);
}

}  // namespace small
}  // namespace bsa
