// Block-sparse GEMM, fp32 blocks of 64 and above: out[n] = sum over the contraction list of block n of x[px] @ y[py], on the
// bf16 matrix instructions (split_f32.h).
//
// A workgroup of four waves owns one 64 x 64 tile of an output block, each wave a 32 x 32 quadrant, and walks the block's pair
// list in ascending k, 32 values at a time.  Every value is split into its three parts once per workgroup: a lane loads eight
// consecutive k of one row of x (of one column of y) into registers, one chunk ahead, splits them when the chunk is due and
// leaves them in LDS, a plane of 64 rows of 32 k for each part, where the waves of both quadrants that need them read them as
// operands.  The chunk of 24 KiB is not double buffered: six workgroups share a compute unit, and one splits or waits while
// another multiplies.
//
// What bounds it: per chunk and wave 12 products of 32 cycles and 114 vector instructions of 4, 72 of them for the split (the two
// overlap by half, measured alone), on a card that lowers its clock for bf16 products of random values (1600 TFLOP/s of 2500
// without anything beside them, where fp32 products run at 137 of 157); then tiles in the order in which places become free, the
// last of which run alone.  Waves that multiply go first (s_setprio: dX 77 -> 71 us).  Two buffers with one barrier and the split
// in the shadow of the wave's own products, which leaves three workgroups: 93 / 78 / 82 us where this takes 80 / 71 / 81 (8 x
// 2048^3 at 25 %, sbs 64, forward / dX / dY; 1 % more since the values are multiplied by kUp).  The kernel before it, on the fp32 instruction, five workgroups of asynchronous
// copies: 103 / 99 / 99; 3 x 1920 x 2944 x 1664 at 30 %, sbs 128, all three: 199 -> 173.
#include "split_f32.h"

namespace bsa {
namespace {

using namespace split;

constexpr int64_t kMostWorkgroups = (int64_t)1 << 23;  // of a launch, which has fewer than 2^32 threads
constexpr int kChunk = 32;                    // values of k
constexpr int kPlane = 64 * kChunk * 2;       // one part of a chunk of one operand
constexpr int kOperand = 3 * kPlane;

// 16 bytes (eight k) number c of row r of a plane: at one number, eight consecutive rows fall on different 16 bytes of 128 and
// sixteen on different ones of 256
__device__ inline int plane_at(int r, int c) { return r * 64 + ((c ^ ((((r >> 1) ^ (r >> 3)) & 1) << 1 | ((r >> 2) & 1))) << 4); }

// Eight values of one operand: consecutive in memory, or one of each of eight rows
template <bool kStrided>
struct Eight {
  u32x4 a, b;
  __device__ inline void load(const char *p, uint32_t ld) {
    if constexpr (kStrided) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = *reinterpret_cast<const uint32_t *>(p + i * ld);
        b[i] = *reinterpret_cast<const uint32_t *>(p + (4 + i) * ld);
      }
    } else {
      a = *reinterpret_cast<const u32x4 *>(p);
      b = *reinterpret_cast<const u32x4 *>(p + 16);
    }
  }
};

// Four values of an operand for the fp32 instruction
template <bool kStrided>
__device__ inline u32x4 load_four(const char *p, uint32_t ld) {
  if constexpr (!kStrided) return *reinterpret_cast<const u32x4 *>(p);
  u32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const uint32_t *>(p + i * ld);
  return v;
}

template <bool XT, bool YT>
__global__ __launch_bounds__(256, 5) void matmul_split_kernel(const char *__restrict__ x, const char *__restrict__ y,
                                                              char *__restrict__ out, const int32_t *__restrict__ pair_offsets,
                                                              const int32_t *__restrict__ pairs, const int32_t *__restrict__ block_order,
                                                              int64_t first, int64_t end, int sbs, int side_log2, int64_t nnz_x,
                                                              int64_t nnz_y) {
  __shared__ __attribute__((aligned(1024))) char smem[2 * kOperand];
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
  const int64_t block_bytes = (int64_t)sbs * sbs * 4;
  const uint32_t ld = (uint32_t)sbs * 4;
  const int n_chunks = sbs / kChunk;  // per pair

  const int p_begin = __builtin_amdgcn_readfirstlane(pair_offsets[n]);
  const int p_end = __builtin_amdgcn_readfirstlane(pair_offsets[n + 1]);

  // byte offset of (row or column r of the tile, k) in a block of x (of y): a transposed x and a y as it lies have k down
  auto at = [&](bool k_down, int64_t r, int64_t k) { return k_down ? k * ld + r * 4 : r * ld + k * 4; };
  const int64_t x_tile = at(XT, 64 * ti, 0), y_tile = at(!YT, 64 * tj, 0);
  // 64 entries of the pair list at a time, one per lane; a corrupt list must not turn into a wild read
  int win_base = p_begin, win_x = 0, win_y = 0;
  auto load_window = [&]() {
    const int t = win_base + lane;
    win_x = win_y = 0;
    if (t < p_end) {
      const int2 v = *reinterpret_cast<const int2 *>(pairs + 2 * (int64_t)t);
      win_x = v.x < 0 || v.x >= nnz_x ? 0 : v.x;
      win_y = v.y < 0 || v.y >= nnz_y ? 0 : v.y;
    }
  };

  // The lane's share of a chunk: k down, a wave loads eight rows of 64 values; k along, 16 rows of 32, four lanes to a row.
  const int along_r = 16 * wave + (lane >> 2), along_c = lane & 3;
  const int xr = XT ? lane : along_r, xc = XT ? wave : along_c, yr = YT ? along_r : lane, yc = YT ? along_c : wave;
  const uint32_t x_mine = (uint32_t)at(XT, xr, 8 * xc), y_mine = (uint32_t)at(!YT, yr, 8 * yc);
  const int64_t x_step = at(XT, 0, kChunk), y_step = at(!YT, 0, kChunk);
  char *const x_put = smem + plane_at(xr, xc), *const y_put = smem + kOperand + plane_at(yr, yc);
  Eight<XT> ex;
  Eight<!YT> ey;
  int p = p_begin, kc = 0;  // next chunk to load
  auto load = [&]() {
    if (p - win_base >= 64) {
      win_base += 64;
      load_window();
    }
    const int sel = p - win_base;
    const int64_t px = __builtin_amdgcn_readlane(win_x, sel), py = __builtin_amdgcn_readlane(win_y, sel);
    ex.load(x + (px * block_bytes + x_tile + kc * x_step) + x_mine, ld);
    ey.load(y + (py * block_bytes + y_tile + kc * y_step) + y_mine, ld);
    if (++kc == n_chunks) kc = 0, ++p;
  };

  f32x16 acc[1];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[0][r] = 0.f;
  const int n_iter = (p_end - p_begin) * n_chunks;
  const int li = lane & 31, kg = lane >> 5;
  if (n_iter > 0) {
    load_window();
    load();
  }
  for (int it = 0; it < n_iter; ++it) {
    const Parts px = Parts::of<true>(ex.a, ex.b, kUp), py = Parts::of<true>(ey.a, ey.b, kUp);
    __syncthreads();  // nobody reads the chunk before any more
    *reinterpret_cast<u32x4 *>(x_put) = px.high;
    *reinterpret_cast<u32x4 *>(x_put + kPlane) = px.mid;
    *reinterpret_cast<u32x4 *>(x_put + 2 * kPlane) = px.low;
    *reinterpret_cast<u32x4 *>(y_put) = py.high;
    *reinterpret_cast<u32x4 *>(y_put + kPlane) = py.mid;
    *reinterpret_cast<u32x4 *>(y_put + 2 * kPlane) = py.low;
    if (it + 1 < n_iter) load();
    // the writes have to be there, the loads just issued not: no wait for vector memory at this barrier
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < kChunk / 16; ++s) {
      const char *bx = smem + plane_at(32 * wi + li, 2 * s + kg), *by = smem + kOperand + plane_at(32 * wj + li, 2 * s + kg);
      Parts fx, fy;
      fx.high = *reinterpret_cast<const u32x4 *>(bx);
      fy.high = *reinterpret_cast<const u32x4 *>(by);
      fx.mid = *reinterpret_cast<const u32x4 *>(bx + kPlane);
      fy.mid = *reinterpret_cast<const u32x4 *>(by + kPlane);
      fx.low = *reinterpret_cast<const u32x4 *>(bx + 2 * kPlane);
      fy.low = *reinterpret_cast<const u32x4 *>(by + 2 * kPlane);
      multiply_parts(acc[0], fy, fx);
    }
    __builtin_amdgcn_s_setprio(0);
  }

  const bool again = not_finite<1, 16>(acc);
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[0][r] = again ? 0.f : acc[0][r] * (kDown * kDown);
  if (again) {  // with the fp32 instruction, from memory
    for (int q = p_begin; q < p_end; ++q) {
      const int2 v = *reinterpret_cast<const int2 *>(pairs + 2 * (int64_t)q);
      const int64_t bx = v.x < 0 || v.x >= nnz_x ? 0 : v.x, by = v.y < 0 || v.y >= nnz_y ? 0 : v.y;
      for (int k = 4 * kg; k < sbs; k += 8) {
        const u32x4 fx = load_four<XT>(x + bx * block_bytes + x_tile + at(XT, 32 * wi + li, k), ld);
        const u32x4 fy = load_four<!YT>(y + by * block_bytes + y_tile + at(!YT, 32 * wj + li, k), ld);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(as_float(fy[i]), as_float(fx[i]), acc[0], 0, 0, 0);
      }
    }
  }

  // acc[r] = O[i = 32 wi + lane % 32][j = 32 wj + 8 (r / 4) + 4 (lane / 32) + r % 4]: through LDS (the wave's own 4 KiB,
  // when nobody reads the tiles any more) into whole rows of the quadrant, stored past the caches
  __syncthreads();
  char *stage = smem + wave * 4096;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *reinterpret_cast<f32x4 *>(stage + li * 128 + (((2 * q + kg) ^ (li & 7)) << 4)) =
        f32x4{acc[0][4 * q], acc[0][4 * q + 1], acc[0][4 * q + 2], acc[0][4 * q + 3]};
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  char *ob = out + n * block_bytes + (int64_t)(64 * ti + 32 * wi) * ld + (64 * tj + 32 * wj) * 4;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int row = 8 * t + (lane >> 3), chunk = lane & 7;
    const u32x4 v = *reinterpret_cast<const u32x4 *>(stage + row * 128 + ((chunk ^ (row & 7)) << 4));
    __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(ob + row * ld + chunk * 16));
  }
}

}  // namespace

int matmul_split_f32(const void *x, const void *y, void *out, const int32_t *pair_offsets, const int32_t *pairs,
                     const int32_t *block_order, int64_t nnz_o, int64_t nnz_x, int64_t nnz_y, int sbs, int trans_x, int trans_y,
                     hipStream_t s) {
  int side_log2 = 0;
  while ((64 << side_log2) < sbs) ++side_log2;
  const int64_t n_tiles = nnz_o << (2 * side_log2);
  auto *kernel = trans_x ? (trans_y ? &matmul_split_kernel<true, true> : &matmul_split_kernel<true, false>)
                         : (trans_y ? &matmul_split_kernel<false, true> : &matmul_split_kernel<false, false>);
  for (int64_t first = 0; first < n_tiles; first += kMostWorkgroups) {
    const int64_t tiles = n_tiles - first < kMostWorkgroups ? n_tiles - first : kMostWorkgroups;
    kernel<<<(unsigned)(cdiv(tiles, (int64_t)8) * 8), 256, 0, s>>>(static_cast<const char *>(x), static_cast<const char *>(y),
                                                                  static_cast<char *>(out), pair_offsets, pairs, block_order, first,
                                                                  first + tiles, sbs, side_log2, nnz_x, nnz_y);
    if (int rc = check_launch("matmul_split_kernel")) return rc;
  }
  return BSA_OK;
}

}  // namespace bsa
