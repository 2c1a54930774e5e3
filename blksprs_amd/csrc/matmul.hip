// Block-sparse GEMM: out[n] = sum over the contraction list of block n of x[px] @ y[py].
//
// Block sizes 16 and 32: a wave owns a run of consecutive output blocks and walks their pairs (matmul_small16_kernel,
// matmul_small16_f32_kernel, matmul_runs32_kernel); larger blocks: a workgroup owns a 64 x 64 tile (matmul_quad_kernel, and
// matmul_split.hip for fp32).  Every kernel walks a block's pairs in ascending k, so only non-zero K-blocks are touched and the
// fp32 accumulation order is fixed.
//
// An operand whose k index is contiguous in memory (x, or y read transposed) is read from LDS as it lies; one whose k index
// is strided (y, or x read transposed) through the transposing LDS read for 16-bit types, and by 32-bit reads for fp32.
//
// The product is formed transposed (y fragments as the A operand, x fragments as B), which leaves 4 consecutive output
// columns of one row in each lane.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <type_traits>

#include "attn_mfma_common.h"
#include "split_f32.h"

namespace {

// native vectors (not HIP's uint4 struct): arrays of them are always promoted to registers
using bsa::mfma::bf16x8;
using bsa::mfma::f16x8;
using bsa::mfma::f32x16;
using bsa::mfma::f32x4;
using bsa::mfma::i16x4;
using bsa::mfma::u32x2;
using bsa::mfma::u32x4;

struct Bf16Traits {
  static constexpr int kElem = 2;
  using store_t = uint16_t;
  __device__ static f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
  }
  // round to nearest even, NaN kept quiet (the hardware conversion of gfx950)
  __device__ static uint16_t round(float v) { return __builtin_bit_cast(uint16_t, (__bf16)v); }
  __device__ static float widen(uint16_t h) { return __builtin_bit_cast(float, (uint32_t)h << 16); }
};

struct F16Traits {
  static constexpr int kElem = 2;
  using store_t = uint16_t;
  __device__ static f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
  }
  __device__ static uint16_t round(float v) { return __builtin_bit_cast(uint16_t, (_Float16)v); }
  __device__ static float widen(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }
};

struct F32Traits {
  static constexpr int kElem = 4;
  using store_t = float;
  // by-value helper: __builtin_bit_cast applied directly to a vector component reads component 0
  __device__ static float as_float(uint32_t v) { return __builtin_bit_cast(float, v); }
  // one fragment = 4 floats = 4 rank-2 updates
  __device__ static f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(as_float(a[0]), as_float(b[0]), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(as_float(a[1]), as_float(b[1]), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(as_float(a[2]), as_float(b[2]), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(as_float(a[3]), as_float(b[3]), c, 0, 0, 0);
    return c;
  }
  __device__ static float round(float v) { return v; }
  __device__ static float widen(float v) { return v; }
};

// ---- blocks of 32 x 32 in LDS: rows of 64 bytes (16-bit) or 128 (fp32), the 16-byte chunks of row r exchanged by an XOR
template <typename Tr>
struct Block32 {
  static constexpr int ES = Tr::kElem;
  static constexpr int kRow = 32 * ES, kBytes = 32 * kRow, kChunks = kRow / 16;
  static constexpr int kCopies = kBytes / 1024;  // asynchronous copies per block
  // along the contraction; fragment s: values 16 s + 8 (lane / 32) .. + 7 (fp32: 8 s + 4 (lane / 32) .. + 3)
  static constexpr int kFrags = ES == 2 ? 2 : 4;

  // eight consecutive rows read at one chunk fall on different chunks of 128 bytes; 16-bit rows r and r + 2 also put the 32
  // bytes of a transposing read into different halves
  __device__ static int swizzle(int r) { return ES == 4 ? r & 7 : ((((r >> 1) ^ (r >> 3)) & 1) << 1) | ((r >> 2) & 1); }

  // lane l supplies the 16 bytes at position 16 l of every KiB (the swizzle is the same for all of them)
  __device__ static uint32_t source_offset(int lane) {
    const int r = lane / kChunks;
    return (uint32_t)(r * kRow + (((lane % kChunks) ^ swizzle(r)) << 4));
  }
  __device__ static void request(const char *base, uint32_t off, char *dst) {
#pragma unroll
    for (int i = 0; i < kBytes; i += 2048) bsa::mfma::copy_2k_to_lds(base + i, off, dst + i);
  }

  // fragments of an operand whose contraction runs along the rows (row lane % 32), or down the columns (column lane % 32)
  template <bool kDown>
  struct Reader {
    static constexpr int kBases = !kDown ? 1 : ES == 2 ? 2 : 4;
    uint32_t at[kBases];
    __device__ explicit Reader(int lane) {
      const int li = lane & 31, kg = lane >> 5;
      if constexpr (!kDown) {
        at[0] = li * kRow + ((kg ^ swizzle(li)) << 4);
      } else if constexpr (ES == 2) {
        // lane s of a group of 16 points at row s / 4 of four, values 4 (s % 4) .. + 3 of the group's 16 columns
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int r = 8 * kg + 4 * i + ((lane & 15) >> 2), c = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
          at[i] = r * kRow + ((c ^ swizzle(r)) << 4) + ((lane & 1) << 3);
        }
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) at[t] = (4 * kg + t) * kRow + (((li >> 2) ^ swizzle(4 * kg + t)) << 4) + ((li & 3) << 2);
      }
    }
    __device__ u32x4 frag(const char *lds, int s) const {
      u32x4 v;
      if constexpr (!kDown) {
        v = *reinterpret_cast<const u32x4 *>(lds + (at[0] ^ (32 * s)));
      } else if constexpr (ES == 2) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const auto t = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4 *)(lds + at[i] + 1024 * s));
          const u32x2 w = __builtin_bit_cast(u32x2, t);
          v[2 * i] = w[0], v[2 * i + 1] = w[1];
        }
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = *reinterpret_cast<const uint32_t *>(lds + at[t] + 1024 * s);
      }
      return v;
    }
  };
};



// sbs 32.  A wave owns a run of consecutive output blocks, whose pairs are one contiguous range of the pair list, and walks
// the pairs with the operand blocks of the next ones on their way into its own LDS (asynchronous copies, no barriers): a
// pair is copied over as soon as its fragments are in registers, so one pair in LDS (fp32, where a pair's products last
// longer than its copies) or two (16-bit) keep the loads going, and 20 waves share a compute unit.  A finished block is
// rounded and stored in between.  The products of a block are added in list order.
//
// With a block order (the caller has one for long lists) a wave owns a single block, and the blocks in flight on an L2 lie
// in one super-tile of the output, whose operands it then holds: bf16, 4 x 4096^3, 128 / 32 / 16 pairs per block, storage
// order in runs 2184 / 566 / 258 us, in the order 1312 / 365 / 190.
//
// What bounds it for 16-bit operands: the operand bytes behind the L2 (4 KiB per pair of 65 kFLOP; of the 8.6 GB of 16
// x 4096^3 at 25 % 3.0 pass it in storage order), then the instructions of a pair's control; fp32: the matrix cores,
// half busy.  Against a kernel that staged operands through registers and gave a wave one block: that size, bf16, out /
// dX / dY: 0.096 / 0.100 / 0.107 -> 0.094 / 0.093 / 0.098 ms, 16 x 4096^3 0.553 / 0.684 / 0.591 -> 0.490 / 0.545 /
// 0.566; fp32 0.366 / 0.324 / 0.308 -> 0.276 / 0.298 / 0.277 ms.  Two pairs in LDS for fp32 leave 10 waves: 0.316 /
// 0.328 / 0.323.
template <typename Tr, bool XT, bool YT>
__global__ __launch_bounds__(256, 5) void matmul_runs32_kernel(
    const char *__restrict__ x, const char *__restrict__ y, char *__restrict__ out, const int32_t *__restrict__ pair_offsets,
    const int32_t *__restrict__ pairs, const int32_t *__restrict__ block_order, int64_t nnz_o, int64_t nnz_x, int64_t nnz_y,
    int run) {
  using B = Block32<Tr>;
  constexpr int ES = B::ES, kPair = 2 * B::kBytes, kStores = B::kBytes / 1024, kWaves = 4;
  constexpr int kDepth = ES == 2 ? 2 : 1;  // pairs in LDS or on their way
  __shared__ __attribute__((aligned(1024))) char smem[kWaves * kDepth * kPair];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // every XCD takes a contiguous eighth of the runs (workgroup g runs on XCD g % 8)
  const int64_t group = (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  int64_t n0 = (group * kWaves + wave) * run;
  if (n0 >= nnz_o) return;
  const int count = (int)(nnz_o - n0 < run ? nnz_o - n0 : run);
  if (block_order) n0 = __builtin_amdgcn_readfirstlane(block_order[n0]);  // with an order, runs are single blocks
  const int off_win = pair_offsets[n0 + (lane <= count ? lane : count)];
  const int p_first = __builtin_amdgcn_readlane(off_win, 0), p_last = __builtin_amdgcn_readlane(off_win, count);
  char *const ring = smem + wave * kDepth * kPair;
  const uint32_t source = B::source_offset(lane);
  const typename B::template Reader<XT> rx(lane);
  const typename B::template Reader<!YT> ry(lane);

  // 64 entries of the pair list at a time, one per lane; a corrupt list must not turn into a wild read
  int next = p_first, base = p_first - 64;  // the next pair to request
  uint32_t win_x = 0, win_y = 0;
  auto request = [&](char *slot) {
    if (next - base >= 64) {
      base += 64;
      u32x2 v{0u, 0u};
      if (base + lane < p_last) v = *reinterpret_cast<const u32x2 *>(pairs + 2 * (int64_t)(base + lane));
      win_x = v[0] < (uint32_t)nnz_x ? v[0] : 0u;
      win_y = v[1] < (uint32_t)nnz_y ? v[1] : 0u;
    }
    const uint32_t px = __builtin_amdgcn_readlane((int)win_x, next - base), py = __builtin_amdgcn_readlane((int)win_y, next - base);
    B::request(x + (uint64_t)px * B::kBytes, source, slot);
    B::request(y + (uint64_t)py * B::kBytes, source, slot + B::kBytes);
    ++next;
  };

  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  int done = 0, block_end = __builtin_amdgcn_readlane(off_win, 1);  // the block in work, the end of its pairs
  const int li = lane & 31, kg = lane >> 5;
  // acc[r] = O[lane % 32][8 (r / 4) + 4 (lane / 32) + r % 4]: through LDS into whole rows, stored past the caches
  auto flush = [&](char *stage) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int at = (8 * q + 4 * kg) * ES;  // byte of the row
      char *dst = stage + li * B::kRow + ((((at >> 4) ^ li) & (B::kChunks - 1)) << 4) + (at & 15);
      if constexpr (ES == 2)
        *reinterpret_cast<uint2 *>(dst) = uint2{(uint32_t)Tr::round(acc[4 * q]) | ((uint32_t)Tr::round(acc[4 * q + 1]) << 16),
                                                (uint32_t)Tr::round(acc[4 * q + 2]) | ((uint32_t)Tr::round(acc[4 * q + 3]) << 16)};
      else
        *reinterpret_cast<f32x4 *>(dst) = f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    char *ob = out + (n0 + done) * B::kBytes + lane * 16;
#pragma unroll
    for (int t = 0; t < kStores; ++t) {
      const int row = (t * 64 + lane) / B::kChunks, chunk = lane & (B::kChunks - 1);
      const u32x4 v = *reinterpret_cast<const u32x4 *>(stage + row * B::kRow + (((chunk ^ row) & (B::kChunks - 1)) << 4));
      __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(ob + t * 1024));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  };
  auto advance = [&]() {
    ++done;
    block_end = __builtin_amdgcn_readlane(off_win, done + 1 <= count ? done + 1 : count);
  };
  // blocks without a pair in front of pair p
  auto zeros_until = [&](int p) {
    while (done < count && block_end <= p) {
      char *ob = out + (n0 + done) * B::kBytes + lane * 16;
#pragma unroll
      for (int t = 0; t < kStores; ++t) __builtin_nontemporal_store(u32x4{0u, 0u, 0u, 0u}, reinterpret_cast<u32x4 *>(ob + t * 1024));
      advance();
    }
  };

  if (p_first < p_last) request(ring);
  if (kDepth > 1 && p_first + 1 < p_last) request(ring + kPair);
  zeros_until(p_first);
  int place = 0;
  bool stored = false;  // exactly kStores stores were issued between the requests of the next two pairs
  for (int p = p_first; p < p_last; ++p) {
    // this pair's copies have landed; what may be on its way is what was issued behind them
    if (kDepth == 1 || p + 1 >= p_last) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (stored) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * B::kCopies + kStores) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * B::kCopies) : "memory");
    stored = false;
    char *const slot = ring + place;
    if (kDepth > 1) place ^= kPair;
    u32x4 fx[B::kFrags], fy[B::kFrags];
#pragma unroll
    for (int s = 0; s < B::kFrags; ++s) fx[s] = rx.frag(slot, s), fy[s] = ry.frag(slot + B::kBytes, s);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the next blocks are copied over them
    // the products at one place: with a copy of them behind each test the sums travelled from registers to registers, 32 moves
    // a pair that wait for the products (8 x 2976 x 4064 x 2080 at 25 %: bf16 280 -> 274 us for the three, fp32 855 -> 827)
    const bool last = p + 1 >= block_end;
    if (!last && next < p_last) request(slot);
#pragma unroll
    for (int s = 0; s < B::kFrags; ++s) acc = Tr::mfma(fy[s], fx[s], acc);
    if (last) {
      flush(slot);
      advance();
      stored = done == count || block_end > p + 1;
      zeros_until(p + 1);
      if (next < p_last) request(slot);
    }
  }
}

// ---- LDS chunks of the kernel whose workgroup shares a tile: 64 rows of 128 bytes (k contiguous, or k rows)

// chunk index XOR of a 128-byte row, by row % 8: row reads of eight consecutive rows fall on eight chunks, and the four
// rows of a transposing read on different halves of their rows
__device__ inline int quad_swizzle(int r) { return bsa::mfma::t_swizzle(r & 7); }
// 16 bytes of k of one row
__device__ inline u32x4 quad_rows(const char *lds, int row, int chunk) {
  return *reinterpret_cast<const u32x4 *>(lds + row * 128 + ((chunk ^ quad_swizzle(row)) << 4));
}
// the same values of k (step s: 16 s + 8 (lane / 32) .. + 7) of column col0 + lane % 32, from k rows
__device__ inline u32x4 quad_cols(const char *lds, int col0, int s, int lane) {
  const int kg = lane >> 5, chunk = (col0 >> 3) + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
  u32x4 v;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 16 * s + 8 * kg + 4 * i + ((lane & 15) >> 2);
    const char *p = lds + r * 128 + ((chunk ^ quad_swizzle(r)) << 4) + ((lane & 1) << 3);
    const auto t = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4 *)p);
    const u32x2 w = __builtin_bit_cast(u32x2, t);
    v[2 * i] = w[0];
    v[2 * i + 1] = w[1];
  }
  return v;
}

// 16-bit elements at sbs 128 and above, or at 64 where neither the row nor the line kernel applies (fp32: matmul_split.hip).
// A workgroup of four waves owns one 64 x 64 tile of an output block, each wave a 32 x 32 quadrant, and walks
// the block's pair list in chunks of 128 bytes of k; the chunk of x and the chunk of y lie in LDS for all four waves,
// double buffered, copied asynchronously while the chunk before is multiplied, with one barrier per chunk.
//
// What this split is for: lists differ in length (a few pairs, Poisson-like), and a wave that owns a whole 64 x 64 tile
// takes the whole difference: 2080 tiles of 4 to 16 pairs on 2048 places of a wave (two per SIMD, by registers and LDS) run
// as long as the SIMD with the two longest, and a workgroup of four such tiles holds its LDS until the longest is done.
// Here the four waves of a workgroup are equal, five workgroups share a compute unit, and tiles are handed out as places
// become free.  bf16, sbs 128, 8 x 2944 x 3968 x 2048 at 25 %: 0.064 -> 0.059, 0.061 -> 0.055, 0.064 -> 0.052 ms.  What is left is the
// chain in front of a tile's first chunk (order, offsets, pairs, operands) and the last tiles of a launch.
template <typename Tr, bool XT, bool YT>
__global__ __launch_bounds__(256, 5) void matmul_quad_kernel(const char *__restrict__ x, const char *__restrict__ y,
                                                             char *__restrict__ out,
                                                             const int32_t *__restrict__ pair_offsets,
                                                             const int32_t *__restrict__ pairs,
                                                             const int32_t *__restrict__ block_order, int64_t first,
                                                             int64_t end, int sbs, int side_log2, int64_t nnz_x,
                                                             int64_t nnz_y) {
  constexpr int ES = 2, KC = 128 / ES;  // k per chunk
  constexpr int kOperand = 64 * 128, kBuffer = 2 * kOperand;
  __shared__ __attribute__((aligned(1024))) char smem[2 * kBuffer];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wi = wave >> 1, wj = wave & 1;  // the wave's quadrant
  // XCD c takes the c-th contiguous eighth of the launch's part of the ordered work list (workgroup g runs on XCD g % 8)
  const int64_t item = first + (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (item >= end) return;
  const int64_t per_block = (int64_t)1 << (2 * side_log2);
  const int64_t n = block_order ? (int64_t)__builtin_amdgcn_readfirstlane(block_order[item >> (2 * side_log2)])
                                : item >> (2 * side_log2);
  const int tile = (int)(item & (per_block - 1));
  const int ti = tile >> side_log2, tj = tile & ((1 << side_log2) - 1);
  const int64_t block_bytes = (int64_t)sbs * sbs * ES;
  const uint32_t ld = (uint32_t)sbs * ES;
  const int n_chunks = sbs / KC;  // per pair

  const int p_begin = __builtin_amdgcn_readfirstlane(pair_offsets[n]);
  const int p_end = __builtin_amdgcn_readfirstlane(pair_offsets[n + 1]);

  // Copies: one instruction moves 1 KiB, lane l supplying the 16 bytes at position l; wave w takes KiB 2 w and 2 w + 1 of
  // either chunk: 64 rows (of k, unless k is contiguous) of 128 bytes, eight to a KiB, chunk index swizzled by the row.
  const int row8 = lane >> 3;
  const uint32_t off128 = (uint32_t)row8 * ld + (uint32_t)(((lane & 7) ^ quad_swizzle(row8)) << 4);
  auto copy_operand = [&](const char *base, char *dst) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      bsa::mfma::copy_1k_to_lds(base + (int64_t)((2 * wave + i) * 8) * ld, off128, dst + (2 * wave + i) * 1024);
  };
  // 64 entries of the pair list at a time, one per lane
  int win_base = p_begin, win_x = 0, win_y = 0;
  auto load_window = [&]() {
    const int t = win_base + lane;
    win_x = win_y = 0;
    if (t < p_end) {
      const int2 v = *reinterpret_cast<const int2 *>(pairs + 2 * (int64_t)t);
      win_x = v.x;
      win_y = v.y;
    }
  };
  int p = p_begin, kc = 0;  // next chunk to request
  auto request = [&](char *buf) {
    if (p - win_base >= 64) {
      win_base += 64;
      load_window();
    }
    const int sel = p - win_base;
    int64_t px = __builtin_amdgcn_readlane(win_x, sel), py = __builtin_amdgcn_readlane(win_y, sel);
    // a corrupt list must not turn into a wild read
    px = (px < 0 || px >= nnz_x) ? 0 : px;
    py = (py < 0 || py >= nnz_y) ? 0 : py;
    // x: rows i from 64 ti, k from kc KC; y: k likewise, columns j from 64 tj; a transposed operand is stored the other way
    const int64_t k_along = (int64_t)kc * 128, k_down = (int64_t)kc * KC * ld;
    const int64_t i_down = (int64_t)ti * 64 * ld, i_along = (int64_t)ti * 64 * ES;
    const int64_t j_down = (int64_t)tj * 64 * ld, j_along = (int64_t)tj * 64 * ES;
    copy_operand(x + px * block_bytes + (XT ? k_down + i_along : i_down + k_along), buf);
    copy_operand(y + py * block_bytes + (YT ? j_down + k_along : k_down + j_along), buf + kOperand);
    if (++kc == n_chunks) kc = 0, ++p;
  };

  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  const int n_iter = (p_end - p_begin) * n_chunks;
  const int li = lane & 31, kg = lane >> 5;
  if (n_iter > 0) {
    load_window();
    request(smem);
  }
  for (int it = 0; it < n_iter; ++it) {
    // the copies of this chunk have landed and, behind the barrier, those of the other waves too; nobody reads the other
    // buffer any more
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    if (it + 1 < n_iter) request(smem + ((it + 1) & 1) * kBuffer);
    const char *bx = smem + (it & 1) * kBuffer, *by = bx + kOperand;
    u32x4 fx[4], fy[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      fx[s] = XT ? quad_cols(bx, 32 * wi, s, lane) : quad_rows(bx, 32 * wi + li, 2 * s + kg);
      fy[s] = YT ? quad_rows(by, 32 * wj + li, 2 * s + kg) : quad_cols(by, 32 * wj, s, lane);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = Tr::mfma(fy[s], fx[s], acc);
  }

  // acc[r] = O[i = 32 wi + lane % 32][j = 32 wj + 8 (r / 4) + 4 (lane / 32) + r % 4]: through LDS (the wave's own 4 KiB,
  // when nobody reads the tiles any more) into whole rows of the quadrant, stored past the caches
  __syncthreads();
  constexpr int kRow = 32 * ES, kChunks = kRow / 16;
  char *stage = smem + wave * 4096;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int at = (8 * q + 4 * kg) * ES;  // byte of the row
    char *dst = stage + li * kRow + ((((at >> 4) ^ li) & (kChunks - 1)) << 4) + (at & 15);
    *reinterpret_cast<uint2 *>(dst) = uint2{(uint32_t)Tr::round(acc[4 * q]) | ((uint32_t)Tr::round(acc[4 * q + 1]) << 16),
                                            (uint32_t)Tr::round(acc[4 * q + 2]) | ((uint32_t)Tr::round(acc[4 * q + 3]) << 16)};
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  char *ob = out + n * block_bytes + (int64_t)(64 * ti + 32 * wi) * ld + (64 * tj + 32 * wj) * ES;
#pragma unroll
  for (int t = 0; t < 32 * kChunks / 64; ++t) {
    const int row = (t * 64 + lane) / kChunks, chunk = lane & (kChunks - 1);
    const u32x4 v = *reinterpret_cast<const u32x4 *>(stage + row * kRow + (((chunk ^ row) & (kChunks - 1)) << 4));
    __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(ob + row * ld + chunk * 16));
  }
}

// sbs == 16, 16-bit elements: one 16 x 16 x 16 matrix-core product per pair.  A block is 512 bytes and an output
// block has one or two pairs, so a wave that handled a single block would be a chain of dependent loads
// (offsets -> pairs -> operands -> store) and nothing else.  Here a wave owns a run of consecutive output blocks,
// whose pairs are one contiguous range of the pair list: it reads that range and the run's offsets once (one
// entry per lane), then walks the pairs with the operand loads of the next two pairs in flight.
// The product is formed transposed (A = y fragment, B = x fragment), which leaves four consecutive output columns
// of one row in each lane: the wave's 8-byte stores cover the whole output block.  One 16-byte load per lane
// fetches both operand blocks of a pair (lanes 0-31 the x block, lanes 32-63 the y block: one memory instruction
// per pair instead of two, which is what the kernel's time follows); both pass through 1 KiB of LDS, from which
// an operand whose contraction index is contiguous in memory (x, or y when it is used transposed) is read as it
// lies and the other one through the transposing read.
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

struct Bf16Small {
  __device__ static f32x4 mfma(u32x2 a, u32x2 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(i16x4, a), __builtin_bit_cast(i16x4, b), c, 0, 0, 0);
  }
  __device__ static uint32_t pack2(float lo, float hi) {
    return (uint32_t)Bf16Traits::round(lo) | ((uint32_t)Bf16Traits::round(hi) << 16);
  }
};
struct F16Small {
  __device__ static f32x4 mfma(u32x2 a, u32x2 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
  }
  __device__ static uint32_t pack2(float lo, float hi) {
    return (uint32_t)F16Traits::round(lo) | ((uint32_t)F16Traits::round(hi) << 16);
  }
};

constexpr int kSmallDepth = 2;    // pairs whose operand loads are in flight
constexpr int kSmallRunMax = 63;  // output blocks per wave: their offsets (one more) fit one entry per lane

// The output of a run as a buffer resource: the block's byte offset travels in a scalar register (`soffset`) and
// the lane's offset inside a block is a constant, so a store needs no per-lane address arithmetic.
__device__ inline __amdgpu_buffer_rsrc_t small_resource(const char *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(base), 0, (int)bytes, 0x00020000);
}

template <typename Ts, bool XT, bool YT>
__global__ __launch_bounds__(256) void matmul_small16_kernel(const char *__restrict__ x, const char *__restrict__ y,
                                                             char *__restrict__ out,
                                                             const int32_t *__restrict__ pair_offsets,
                                                             const int32_t *__restrict__ pairs, int64_t nnz_o,
                                                             int64_t nnz_x, int64_t nnz_y, int run) {
  __shared__ __attribute__((aligned(16))) char stage[4][1024];  // per wave: the x block, then the y block
  const int lane = threadIdx.x & 63;
  // everything that steers the loops below is built from values the compiler knows to be the same in all lanes
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // workgroup g runs on XCD g % 8: every XCD takes a contiguous eighth of the runs, so that the operand blocks in
  // flight on one L2 belong to few batch entries
  const int64_t group = (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int64_t n0 = (group * 4 + wave) * run;
  if (n0 >= nnz_o) return;
  const int count = (int)(nnz_o - n0 < run ? nnz_o - n0 : run);
  // fragment of a k-contiguous operand: row lane % 16, values 4 (lane / 16) .. + 3
  const int direct_off = (lane & 15) * 32 + (lane >> 4) * 8;
  // the other operand is read transposed: inside a group of 16 lanes, lane s points at row
  // 4 (lane / 16) + s / 4, values 4 (s % 4) .. + 3
  const int turned_off = (4 * (lane >> 4) + ((lane & 15) >> 2)) * 32 + (lane & 3) * 8;
  char *slot = stage[wave];
  const uint32_t nx = (uint32_t)nnz_x, ny = (uint32_t)nnz_y;  // the pair list holds 32-bit indices
  const __amdgpu_buffer_rsrc_t ro = small_resource(out + n0 * 512, (uint32_t)count * 512u);

  // offsets of the run (count + 1 of them), one per lane
  const int off_win = pair_offsets[n0 + (lane <= count ? lane : count)];
  const int p_first = __builtin_amdgcn_readlane(off_win, 0);
  const int p_last = __builtin_amdgcn_readlane(off_win, count);

  f32x4 acc{0.f, 0.f, 0.f, 0.f};
  int done = 0;                                           // output blocks of the run already stored
  int block_end = __builtin_amdgcn_readlane(off_win, 1);  // end of the pairs of block `done`
  auto flush_until = [&](int p) {
    // store every block whose pairs end at or before p (blocks without pairs become zeros)
    while (done < count && block_end <= p) {
      u32x2 w;
      w[0] = Ts::pack2(acc[0], acc[1]);
      w[1] = Ts::pack2(acc[2], acc[3]);
      // written once, not read back by this kernel: past the caches
      __builtin_amdgcn_raw_buffer_store_b64(w, ro, direct_off, done * 512, 2);
      acc = f32x4{0.f, 0.f, 0.f, 0.f};
      ++done;
      block_end = __builtin_amdgcn_readlane(off_win, done + 1 <= count ? done + 1 : count);
    }
  };

  // the pairs of the run, 64 at a time: one entry per lane, handed out with readlane
  for (int base = p_first; base < p_last; base += 64) {
    const int n = p_last - base < 64 ? p_last - base : 64;
    u32x2 win{0u, 0u};
    if (lane < n) win = *reinterpret_cast<const u32x2 *>(pairs + 2 * (int64_t)(base + lane));
    auto issue = [&](int i, u32x4 &xy) {
      // past the end: the last pair again (a cache hit), so that every step issues the same loads and the
      // compiler can count the loads in flight instead of waiting for all of them in front of every use
      const int at = i < n ? i : n - 1;
      const uint32_t px = (uint32_t)__builtin_amdgcn_readlane((int)win[0], at);
      const uint32_t py = (uint32_t)__builtin_amdgcn_readlane((int)win[1], at);
      // a corrupt list must not turn into a wild read: such a pair reads block 0
      const char *xb = x + (int64_t)(px < nx ? px : 0) * 512;
      const char *yb = y + (int64_t)(py < ny ? py : 0) * 512;
      const char *mine = (lane < 32 ? xb : yb) + (lane & 31) * 16;
      xy = *reinterpret_cast<const u32x4 *>(mine);
    };
    u32x4 xys[kSmallDepth];
#pragma unroll
    for (int d = 0; d < kSmallDepth; ++d) issue(d, xys[d]);
    for (int i = 0; i < n; i += kSmallDepth) {
#pragma unroll
      for (int d = 0; d < kSmallDepth; ++d) {
        if (i + d < n) {
          flush_until(base + i + d);
          *reinterpret_cast<u32x4 *>(slot + lane * 16) = xys[d];
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          u32x2 fx, fy;
          if (XT) fx = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4 *)(slot + turned_off)));
          else fx = *reinterpret_cast<const u32x2 *>(slot + direct_off);
          if (YT) fy = *reinterpret_cast<const u32x2 *>(slot + 512 + direct_off);
          else fy = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4 *)(slot + 512 + turned_off)));
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          acc = Ts::mfma(fy, fx, acc);
        }
        issue(i + d + kSmallDepth, xys[d]);
      }
    }
  }
  flush_until(p_last);
}

// sbs == 16, fp32: the same walk.  A block is 1 KiB, 16 bytes per lane.  An operand whose contraction index is contiguous is
// a matrix operand as it is loaded (lane: row lane % 16, values 4 (lane / 16) .. + 3, one per 16 x 16 x 4 product); the other
// one passes through LDS, its rows placed so that the four rows of a read (r, r + 4, r + 8, r + 12) are neighbours.  The product
// is formed transposed: a lane ends with 16 consecutive bytes of an output row, a store covers the block.
// It is bound like the 16-bit kernel by its memory instructions and the latency of a wave's chain.  Against one wave per
// block and FMAs from LDS: out / dX / dY of 64 x 2048^3 at 5 %: 0.238 / 0.207 / 0.203 -> 0.070 / 0.093 / 0.088 ms; 8 x 2976 x 4064 x 2080
// at 12.5 %: 0.404 / 0.393 / 0.387 -> 0.122 / 0.123 / 0.117.
template <bool XT, bool YT>
__global__ __launch_bounds__(256) void matmul_small16_f32_kernel(const char *__restrict__ x, const char *__restrict__ y,
                                                                 char *__restrict__ out,
                                                                 const int32_t *__restrict__ pair_offsets,
                                                                 const int32_t *__restrict__ pairs, int64_t nnz_o,
                                                                 int64_t nnz_x, int64_t nnz_y, int run) {
  __shared__ __attribute__((aligned(16))) char stage[4][2048];  // per wave: the x block, the y block
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t group = (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int64_t n0 = (group * 4 + wave) * run;
  if (n0 >= nnz_o) return;
  const int count = (int)(nnz_o - n0 < run ? nnz_o - n0 : run);
  const int li = lane & 15, kg = lane >> 4;
  // a direct operand: row li, chunk kg; one that goes through LDS: as it lies, lane l the 16 bytes at 16 l
  const int direct_off = li * 64 + kg * 16, linear_off = lane * 16;
  const int x_off = XT ? linear_off : direct_off, y_off = YT ? direct_off : linear_off;
  const int row = lane >> 2, write_off = (4 * (row & 3) + (row >> 2)) * 64 + (lane & 3) * 16;
  const int read_off = kg * 64 + li * 4;  // + 256 j: row 4 kg + j, column li
  char *slot = stage[wave];
  const uint32_t nx = (uint32_t)nnz_x, ny = (uint32_t)nnz_y;
  const __amdgpu_buffer_rsrc_t ro = small_resource(out + n0 * 1024, (uint32_t)count * 1024u);

  const int off_win = pair_offsets[n0 + (lane <= count ? lane : count)];
  const int p_first = __builtin_amdgcn_readlane(off_win, 0);
  const int p_last = __builtin_amdgcn_readlane(off_win, count);
  f32x4 acc{0.f, 0.f, 0.f, 0.f};
  int done = 0;
  int block_end = __builtin_amdgcn_readlane(off_win, 1);
  auto flush_until = [&](int p) {
    while (done < count && block_end <= p) {
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc), ro, direct_off, done * 1024, 2);
      acc = f32x4{0.f, 0.f, 0.f, 0.f};
      ++done;
      block_end = __builtin_amdgcn_readlane(off_win, done + 1 <= count ? done + 1 : count);
    }
  };
  for (int base = p_first; base < p_last; base += 64) {
    const int n = p_last - base < 64 ? p_last - base : 64;
    u32x2 win{0u, 0u};
    if (lane < n) win = *reinterpret_cast<const u32x2 *>(pairs + 2 * (int64_t)(base + lane));
    auto issue = [&](int i, u32x4 &xr, u32x4 &yr) {
      const int at = i < n ? i : n - 1;  // past the end: the last pair again, so that every step issues the same loads
      const uint32_t px = (uint32_t)__builtin_amdgcn_readlane((int)win[0], at);
      const uint32_t py = (uint32_t)__builtin_amdgcn_readlane((int)win[1], at);
      // a corrupt list must not turn into a wild read: such a pair reads block 0
      xr = *reinterpret_cast<const u32x4 *>(x + (int64_t)(px < nx ? px : 0) * 1024 + x_off);
      yr = *reinterpret_cast<const u32x4 *>(y + (int64_t)(py < ny ? py : 0) * 1024 + y_off);
    };
    u32x4 xs[kSmallDepth], ys[kSmallDepth];
#pragma unroll
    for (int d = 0; d < kSmallDepth; ++d) issue(d, xs[d], ys[d]);
    for (int i = 0; i < n; i += kSmallDepth) {
#pragma unroll
      for (int d = 0; d < kSmallDepth; ++d) {
        if (i + d < n) {
          flush_until(base + i + d);
          if (XT) *reinterpret_cast<u32x4 *>(slot + write_off) = xs[d];
          if (!YT) *reinterpret_cast<u32x4 *>(slot + 1024 + write_off) = ys[d];
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          f32x4 fx = __builtin_bit_cast(f32x4, xs[d]), fy = __builtin_bit_cast(f32x4, ys[d]);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (XT) fx[j] = *reinterpret_cast<const float *>(slot + read_off + 256 * j);
            if (!YT) fy[j] = *reinterpret_cast<const float *>(slot + 1024 + read_off + 256 * j);
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
          for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fy[j], fx[j], acc, 0, 0, 0);
        }
        issue(i + d + kSmallDepth, xs[d], ys[d]);
      }
    }
  }
  flush_until(p_last);
}

// Workgroups of 256 in one launch.  A launch has fewer than 2^32 threads; one that asks for more is not refused, the
// workgroups beyond are missing from it.
constexpr int64_t kMostWorkgroups = (int64_t)1 << 23;

template <typename Tr>
int launch_runs32(const void *x, const void *y, void *out, const int32_t *pair_offsets, const int32_t *pairs,
                  const int32_t *block_order, int64_t nnz_o, int64_t nnz_x, int64_t nnz_y, int trans_x, int trans_y,
                  hipStream_t s) {
  constexpr int kWaves = 4;
  // Where a forward product's lists are short and its output dense, a run of up to three blocks spreads a wave's first loads
  // (offsets, pairs, operands: three latencies) over more pairs, as long as there are enough waves (bf16, 16 x 4096^3, run
  // 1 / 2 / 3 / 4: 521 / 487 / 490 / 488 us; 36259 blocks of 1.2 pairs: 28.9 / 26.6 / 24.9 / 25.2).  The gradients' lists are
  // long, and longer runs only scatter what is in flight on an L2 (dX of the first: 545 / 764 / 875 / 927).
  int64_t run = trans_x || trans_y || block_order ? 1 : nnz_o / 12288;
  run = run < 1 ? 1 : (run > 3 ? 3 : run);
  // a launch has fewer than 2^32 threads: longer runs where these would be more workgroups
  const int64_t least = bsa::cdiv(nnz_o, kWaves * kMostWorkgroups);
  run = run < least ? least : run;
  const int32_t *const order = run == 1 ? block_order : nullptr;  // longer runs lie in storage order
  if (run > kSmallRunMax) return bsa::fail(BSA_ELIMIT, "bsa_matmul: too many output blocks");
  const int64_t blocks = bsa::cdiv(bsa::cdiv(bsa::cdiv(nnz_o, run), (int64_t)kWaves), (int64_t)8) * 8;
  const char *xc = static_cast<const char *>(x);
  const char *yc = static_cast<const char *>(y);
  char *oc = static_cast<char *>(out);
#define BSA_MM_LAUNCH(XT, YT)                                                                                        \
  matmul_runs32_kernel<Tr, XT, YT><<<(unsigned)blocks, 64 * kWaves, 0, s>>>(xc, yc, oc, pair_offsets, pairs, order, \
                                                                            nnz_o, nnz_x, nnz_y, (int)run)
  if (!trans_x && !trans_y) BSA_MM_LAUNCH(false, false);
  else if (!trans_x && trans_y) BSA_MM_LAUNCH(false, true);
  else if (trans_x && !trans_y) BSA_MM_LAUNCH(true, false);
  else BSA_MM_LAUNCH(true, true);
#undef BSA_MM_LAUNCH
  return bsa::check_launch("matmul_runs32_kernel");
}

template <typename Tr>
int launch_quad(const void *x, const void *y, void *out, const int32_t *pair_offsets, const int32_t *pairs,
                const int32_t *block_order, int64_t nnz_o, int64_t nnz_x, int64_t nnz_y, int sbs, int trans_x,
                int trans_y, hipStream_t s) {
  int side_log2 = 0;
  while ((64 << side_log2) < sbs) ++side_log2;
  const int64_t n_tiles = nnz_o << (2 * side_log2);
  const char *xc = static_cast<const char *>(x);
  const char *yc = static_cast<const char *>(y);
  char *oc = static_cast<char *>(out);
#define BSA_MM_LAUNCH(XT, YT)                                                                                        \
  matmul_quad_kernel<Tr, XT, YT><<<(unsigned)(bsa::cdiv(tiles, 8) * 8), 256, 0, s>>>(                                \
      xc, yc, oc, pair_offsets, pairs, block_order, first, first + tiles, sbs, side_log2, nnz_x, nnz_y)
  for (int64_t first = 0; first < n_tiles; first += kMostWorkgroups) {
    const int64_t tiles = n_tiles - first < kMostWorkgroups ? n_tiles - first : kMostWorkgroups;
    if (!trans_x && !trans_y) BSA_MM_LAUNCH(false, false);
    else if (!trans_x && trans_y) BSA_MM_LAUNCH(false, true);
    else if (trans_x && !trans_y) BSA_MM_LAUNCH(true, false);
    else BSA_MM_LAUNCH(true, true);
    if (int rc = bsa::check_launch("matmul_quad_kernel")) return rc;
  }
#undef BSA_MM_LAUNCH
  return BSA_OK;
}

// Output blocks per wave of the kernels for blocks of 16: as many as leave 32768 waves, four times what the chip holds at
// once.  Output blocks come with one or two pairs (forward) or with ten (gradients, of which there are fewer): waves must
// stay many rather than their runs long.  16-bit, dX and dY of 64 x 2048^3 at 5 % (52611 blocks, 6.4 pairs each), runs of 1 /
// 2 / 4 / 8 blocks: 41 / 41 / 46 / 55 and 39 / 40 / 49 / 60 us; forward (289445 blocks, 1.2 pairs each), 2 / 4 / 8: 55 / 44 / 40 us.
int64_t small_run(int64_t nnz_o) {
  const int64_t run = nnz_o / (256 * 32 * 4);
  return run < 1 ? 1 : (run > kSmallRunMax ? kSmallRunMax : run);
}

template <typename Tr>
int launch_any(const void *x, const void *y, void *out, const int32_t *pair_offsets, const int32_t *pairs,
               const int32_t *block_order, int64_t nnz_o, int64_t nnz_x, int64_t nnz_y, int sbs, int trans_x,
               int trans_y, hipStream_t s) {
  if (sbs == 16 && Tr::kElem == 2) {
    using Ts = std::conditional_t<std::is_same_v<Tr, Bf16Traits>, Bf16Small, F16Small>;
    const int64_t run = small_run(nnz_o);
    const int64_t blocks = bsa::cdiv(bsa::cdiv(bsa::cdiv(nnz_o, run), 4), 8) * 8;
    if (blocks > 0x7fffffffLL) return bsa::fail(BSA_ELIMIT, "bsa_matmul: too many output blocks");
    const char *xc = static_cast<const char *>(x);
    const char *yc = static_cast<const char *>(y);
    char *oc = static_cast<char *>(out);
#define BSA_MM_SMALL(XT, YT)                                                                                        \
  matmul_small16_kernel<Ts, XT, YT><<<(unsigned)blocks, 256, 0, s>>>(xc, yc, oc, pair_offsets, pairs, nnz_o, nnz_x, \
                                                                     nnz_y, (int)run)
    if (!trans_x && !trans_y) BSA_MM_SMALL(false, false);
    else if (!trans_x && trans_y) BSA_MM_SMALL(false, true);
    else if (trans_x && !trans_y) BSA_MM_SMALL(true, false);
    else BSA_MM_SMALL(true, true);
#undef BSA_MM_SMALL
    return bsa::check_launch("matmul_small16_kernel");
  }
  if (sbs == 16) {
    const int64_t run = small_run(nnz_o);
    const int64_t blocks = bsa::cdiv(bsa::cdiv(bsa::cdiv(nnz_o, run), 4), 8) * 8;
    if (blocks > 0x7fffffffLL) return bsa::fail(BSA_ELIMIT, "bsa_matmul: too many output blocks");
    const char *xc = static_cast<const char *>(x);
    const char *yc = static_cast<const char *>(y);
    char *oc = static_cast<char *>(out);
#define BSA_MM_SMALL(XT, YT)                                                                                          \
  matmul_small16_f32_kernel<XT, YT><<<(unsigned)blocks, 256, 0, s>>>(xc, yc, oc, pair_offsets, pairs, nnz_o, nnz_x, nnz_y, \
                                                                     (int)run)
    if (!trans_x && !trans_y) BSA_MM_SMALL(false, false);
    else if (!trans_x && trans_y) BSA_MM_SMALL(false, true);
    else if (trans_x && !trans_y) BSA_MM_SMALL(true, false);
    else BSA_MM_SMALL(true, true);
#undef BSA_MM_SMALL
    return bsa::check_launch("matmul_small16_f32_kernel");
  }
  if (sbs == 32)
    return launch_runs32<Tr>(x, y, out, pair_offsets, pairs, block_order, nnz_o, nnz_x, nnz_y, trans_x, trans_y, s);
  if constexpr (std::is_same_v<Tr, F32Traits>)
    return bsa::matmul_split_f32(x, y, out, pair_offsets, pairs, block_order, nnz_o, nnz_x, nnz_y, sbs, trans_x, trans_y, s);
  else
    return launch_quad<Tr>(x, y, out, pair_offsets, pairs, block_order, nnz_o, nnz_x, nnz_y, sbs, trans_x, trans_y, s);
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

extern "C" int bsa_matmul(const void *x, const void *y, void *out, const int32_t *pair_offsets, const int32_t *pairs,
                          const int32_t *block_order, int64_t nnz_o, int64_t nnz_x, int64_t nnz_y, int sbs, int dtype, int trans_x, int trans_y,
                          bsa_stream_t stream) {
  BSA_REQUIRE(sbs >= 16 && bsa::is_pow2(sbs), "bsa_matmul: sbs must be a power of two >= 16 (got %d)", sbs);
  BSA_REQUIRE(nnz_o >= 0 && nnz_x >= 0 && nnz_y >= 0, "bsa_matmul: negative size");
  BSA_REQUIRE(dtype == BSA_F32 || dtype == BSA_F16 || dtype == BSA_BF16, "bsa_matmul: unknown dtype %d", dtype);
  if (nnz_o == 0) return BSA_OK;
  BSA_REQUIRE(out && pair_offsets, "bsa_matmul: NULL pointer");
  BSA_REQUIRE(aligned16(x) && aligned16(y) && aligned16(out), "bsa_matmul: buffers must be 16-byte aligned");
  hipStream_t s = bsa::as_stream(stream);
  switch (dtype) {
    case BSA_BF16:
      return launch_any<Bf16Traits>(x, y, out, pair_offsets, pairs, block_order, nnz_o, nnz_x, nnz_y, sbs, trans_x, trans_y, s);
    case BSA_F16:
      return launch_any<F16Traits>(x, y, out, pair_offsets, pairs, block_order, nnz_o, nnz_x, nnz_y, sbs, trans_x, trans_y, s);
    default:
      return launch_any<F32Traits>(x, y, out, pair_offsets, pairs, block_order, nnz_o, nnz_x, nnz_y, sbs, trans_x, trans_y, s);
  }
}
