// Row-wise softmax over the active blocks of a block row (fp32), forward and backward.
//
// The blocks of one block row are consecutive in the compressed tensor (row-major
// block order), so a row is `count` whole blocks starting at row_offsets[r].  One
// wavefront owns a group of element rows of one block row and reads them with one
// float4 per lane.  sbs/4 lanes cover an element row of one block; where rows are long,
// 2, 4 or 8 such groups of lanes share it, each taking every second, fourth or eighth
// block (make_geom), so that it fits their registers: rows of up to 16 float4 units per
// lane (32 in the forward pass where no row is shared, and of sbs >= 128) stay there between the reduction and the
// write (one HBM read + one write), longer rows make two read passes.  The reductions stay inside the lanes of a row.
//
// Bound by HBM.  Block-causal rows of n = 2048 elements and 10 % more blocks, us forward +
// backward, a row on sbs/4 lanes (32 units in registers) -> shared: sbs 16, 16 matrices
// 87 + 165 -> 62 + 83; sbs 32 77 + 125 -> 57 + 82; sbs 64, 32 matrices 114 + 165 -> 106 + 153
// (5.7 and 5.9 TB/s); three matrices of 37 blocks of 32 a side 13.3 + 16.0 -> 6.6 + 7.9.
// Which rows are shared follows from the mean, so a few long rows among short ones are not: the kernels without kShared keep 32
// units forward and have nothing to do with lanes that leave a unit out.  128 matrices of 32 blocks a side, a diagonal and the
// one beside it with two whole rows, forward + backward with (16 units) -> without: sbs 64 95 + 145 -> 76 + 144, sbs 32
// 36.6 + 35.8 -> 26.4 + 35.1, sbs 16 (256 matrices) 19.3 + 19.9 -> 16.2 + 18.3; 24 blocks of 64, windows of four, where no row is
// long: 53.3 + 98.5 -> 54.8 + 96.1.
#include "common.h"

namespace {

constexpr int kBwdUnits = 16;  // float4 units per lane in registers, of either tensor
constexpr int kWaves = 4;  // waves (tasks) per workgroup

struct RowGeom {
  int sbs_log2;
  int lpr;          // lanes on one block of an element row = min(64, sbs/4)
  int nq_log2;      // float4 units per lane per block = max(1, sbs/256), as log2
  int split_log2;   // lane groups that share an element row, each taking every 2^split_log2-th block of it
  int lanes;        // lanes of an element row = lpr << split_log2
  int groups_log2;  // wave tasks per block row = sbs * lanes / 64, as log2
};

// The reductions over the lanes of an element row, without a trip through LDS (a shuffle computes a lane
// address, goes through LDS and waits for it).  Steps 1 and 2 exchange inside a group of four lanes (DPP quad_perm);
// after them the four lanes of a group agree, so mirroring a half row (lane i <-> 7 - i) pairs every group with its
// neighbour and mirroring a row (i <-> 15 - i) pairs the two halves of 16 lanes: partners other than those of an
// xor exchange, holding the same values.  Steps 16 and 32 trade register halves (v_permlane16_swap /
// v_permlane32_swap with the same value in both operands: one result holds the even groups' values twice, the other
// the odd groups').  Every step combines a value with its partner's by a commutative operation, so all lanes of a
// row end with the same bits, as with xor shuffles.
template <int CTRL>
__device__ inline float dpp_partner(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
template <typename Op>
__device__ inline float lanes_reduce(float v, int lpr, Op op) {
  if (lpr > 1) v = op(v, dpp_partner<0xB1>(v));   // quad_perm [1, 0, 3, 2]
  if (lpr > 2) v = op(v, dpp_partner<0x4E>(v));   // quad_perm [2, 3, 0, 1]
  if (lpr > 4) v = op(v, dpp_partner<0x141>(v));  // row_half_mirror
  if (lpr > 8) v = op(v, dpp_partner<0x140>(v));  // row_mirror
  if (lpr > 16) {
    float lower = v, upper = v;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(lower), "+v"(upper));
    v = op(lower, upper);
  }
  if (lpr > 32) {
    float lower = v, upper = v;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(lower), "+v"(upper));
    v = op(lower, upper);
  }
  return v;
}
__device__ inline float lanes_max(float v, int lpr) {
  return lanes_reduce(v, lpr, [](float a, float b) { return fmaxf(a, b); });
}
__device__ inline float lanes_sum(float v, int lpr) {
  return lanes_reduce(v, lpr, [](float a, float b) { return a + b; });
}

// float offset of unit u, relative to the first block of the row and to the lane's own offset (the same for every
// lane: the compiler keeps it in scalar registers)
template <bool kShared>
__device__ inline int64_t unit_offset(int u, const RowGeom &g) {
  const int t = kShared ? (u >> g.nq_log2) << g.split_log2 : u >> g.nq_log2;
  const int q = u & ((1 << g.nq_log2) - 1);
  return ((int64_t)t << (2 * g.sbs_log2)) + q * 256;
}

// What this wave works on: `first` (float offset of the row's first block) and `units` (rounds of float4 units per lane)
// are the same for all lanes and are computed from values the compiler knows to be wave-uniform, so the loops over units
// branch on scalar registers instead of masking lanes.  A lane group whose part of the row has no unit in the last round
// (in_last) reads the first group's there (its tail_base), which changes no maximum, and leaves it out of sums and results.
struct RowTask {
  int64_t first;
  int units, lane_base, tail_base;
  bool in_last;
};
template <bool kShared>
__device__ inline bool wave_task(const RowGeom &g, const int32_t *row_offsets, int64_t n_tasks, RowTask &task) {
  // Workgroup b runs on XCD b % 8: each XCD takes a contiguous eighth of the tasks, so the waves that read
  // neighbouring KiB of the same blocks (the tasks of one block row) share one L2.
  const int64_t n_groups = (n_tasks + kWaves - 1) / kWaves, per_xcd = (n_groups + 7) >> 3;
  const int64_t group = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  const int64_t wave = group * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (group >= n_groups || wave >= n_tasks) return false;
  const int lane = threadIdx.x & 63;
  const int64_t r = wave >> g.groups_log2;
  const int grp = (int)(wave & ((1 << g.groups_log2) - 1));
  const int start = row_offsets[r];
  const int count = row_offsets[r + 1] - start;
  if (count <= 0) return false;
  task.first = (int64_t)start << (2 * g.sbs_log2);
  if constexpr (!kShared) {
    task.units = count << g.nq_log2;
    task.lane_base = task.tail_base = ((grp * (64 / g.lpr) + lane / g.lpr) << g.sbs_log2) + (lane % g.lpr) * 4;
    task.in_last = true;
    return true;
  }
  const int split = 1 << g.split_log2, rounds = (count + split - 1) >> g.split_log2;
  task.units = rounds << g.nq_log2;
  const int part = lane / g.lpr & (split - 1);
  const int row_in_block = grp * (64 / g.lanes) + lane / g.lanes;
  task.tail_base = (row_in_block << g.sbs_log2) + (lane % g.lpr) * 4;
  task.lane_base = task.tail_base + (part << (2 * g.sbs_log2));
  task.in_last = part < count - ((rounds - 1) << g.split_log2);
  if (task.in_last) task.tail_base = task.lane_base;
  return true;
}

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// the result is written once and not read back by the kernel: the store bypasses the caches
__device__ inline void store_streaming(float *p, float4 o) {
  __builtin_nontemporal_store(f32x4_t{o.x, o.y, o.z, o.w}, reinterpret_cast<f32x4_t *>(p));
}

// e^(v - m) through the hardware's 2^x as 2^(v * log2(e) - m2) with m2 = m * log2(e): one fused multiply-add and
// one transcendental instruction per element.  The rounding of m2 is a factor common to every element of the
// row and cancels against the row sum; what is left is the rounding of the exponent's argument, a relative
// error of about |v - m| * 1e-7, far inside the 1e-5 the operation is held to.  (The library's expf costs ten
// times the instructions, which made the kernel compute-bound.)
constexpr float kLog2e = 1.44269504088896341f;
__device__ inline float exp_rel(float v, float m2) { return __builtin_amdgcn_exp2f(__builtin_fmaf(v, kLog2e, -m2)); }
__device__ inline float exp2_of(float d) { return __builtin_amdgcn_exp2f(d); }

// max(m, v.x, v.y, v.z, v.w) in two instructions.  fmaxf first quiets signalling NaNs (one more instruction per
// operand); here a NaN may come out either way: it reaches every output of the row through the exponentials.
__device__ inline float max_with(float m, float4 v) {
  float t;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(t) : "v"(v.x), "v"(v.y), "v"(v.z));
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(t) : "v"(t), "v"(v.w), "v"(m));
  return t;
}

// This lane's part of a row of a tensor.  kShared: several groups of lanes share the row
template <bool kShared>
struct RowPart {
  const float *row, *tail;  // where its units are read from, in all rounds and in the last
  int last;                 // the last round
  __device__ inline RowPart(const float *tensor, const RowTask &task)
      : row(tensor + task.first + task.lane_base), tail(tensor + task.first + task.tail_base), last(task.units - 1) {}
  __device__ inline float4 unit(int u, const RowGeom &g) const {
    return *reinterpret_cast<const float4 *>((kShared && u == last ? tail : row) + unit_offset<kShared>(u, g));
  }
};

// Loads units [0, units) of a row into v, four at a time: within a group of four the index is clamped to the last
// unit (a repeated load of a line just fetched) so that the group has no branch, and no load is followed by its
// use: all loads of the row are in flight together.  Entries at and beyond `units` hold copies of the last unit.
template <int N, bool kShared>
__device__ inline void load_row(float4 (&v)[N], const RowPart<kShared> &part, const RowGeom &g) {
#pragma unroll
  for (int c = 0; c < N; c += 4) {
    if (c <= part.last) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[c + j] = part.unit(c + j < part.last ? c + j : part.last, g);
    }
  }
}

// Units [u0, u0 + count) of a row, count <= N: the index is clamped to the last of them, so the loads have no
// branch between them; entries at and beyond `count` hold copies of the last unit.
constexpr int kChunk = 8;
template <int N, bool kShared>
__device__ inline void load_chunk(float4 (&v)[N], const RowPart<kShared> &part, int u0, int count, const RowGeom &g) {
#pragma unroll
  for (int j = 0; j < N; ++j) v[j] = part.unit(u0 + (j < count ? j : count - 1), g);
}

// use(j) for the units [u0, u0 + count) of a chunk that are this lane's (mine).  A whole chunk in front of the last unit is used
// without tests: with them alone the compiler moves loads behind them, each with a wait of its own (backward, 64 matrices of 128
// blocks of 16 a side, a window of 3 blocks and one whole row: 65 us, 37 so).
template <typename Mine, typename Use>
__device__ inline void each_of_chunk(int u0, int count, int units, Mine mine, Use use) {
  if (u0 + kChunk < units) {
#pragma unroll
    for (int j = 0; j < kChunk; ++j) use(j);
  } else {
#pragma unroll
    for (int j = 0; j < kChunk; ++j)
      if (j < count && mine(u0 + j)) use(j);
  }
}

// kUnits: float4 units per lane in registers
template <int kUnits, bool kShared>
__global__ __launch_bounds__(64 * kWaves) void softmax_fwd_kernel(const float *__restrict__ x, float *__restrict__ out,
                                                          const int32_t *__restrict__ row_offsets, int64_t n_tasks,
                                                          RowGeom g) {
  RowTask task;
  if (!wave_task<kShared>(g, row_offsets, n_tasks, task)) return;
  const int units = task.units;
  const RowPart<kShared> xr(x, task);
  float *orow = out + task.first + task.lane_base;
  auto mine = [&](int u) { return !kShared || u < units - 1 || task.in_last; };  // of u < units

  if (units <= kUnits) {
    float4 v[kUnits];
    load_row(v, xr, g);
    float m = -INFINITY;
#pragma unroll
    for (int c = 0; c < kUnits; c += 4) {
      if (c < units) {  // the copies of the last unit change no maximum
#pragma unroll
        for (int j = 0; j < 4; ++j) m = max_with(m, v[c + j]);
      }
    }
    const float m2 = lanes_max(m, g.lanes) * kLog2e;
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
      if (u < units && mine(u)) {
        v[u].x = exp_rel(v[u].x, m2);
        v[u].y = exp_rel(v[u].y, m2);
        v[u].z = exp_rel(v[u].z, m2);
        v[u].w = exp_rel(v[u].w, m2);
        s += (v[u].x + v[u].y) + (v[u].z + v[u].w);
      }
    }
    s = lanes_sum(s, g.lanes);
    const float inv = 1.f / s;  // one division per row, then products
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
      if (u < units && mine(u)) {
        float4 o;
        o.x = v[u].x * inv;
        o.y = v[u].y * inv;
        o.z = v[u].z * inv;
        o.w = v[u].w * inv;
        store_streaming(orow + unit_offset<kShared>(u, g), o);
      }
    }
    return;
  }

  // long rows: max pass and sum pass folded into one online pass, then the write pass; both in chunks of
  // kChunk units whose loads are all issued before the first one is used
  // m2: what the exponentials in s were taken against.  A sum is brought to a larger one by the difference of the two, nothing
  // where the maximum stays.  (Formed from m again it is off by the rounding of m2, once more with every chunk: a row of 300
  // blocks of 64, maximum 13.3, 1.8e-5 off 64 bits, 88.8 1.5e-4; so 8e-8.)
  float m = -INFINITY, m2 = -INFINITY, s = 0.f;
  for (int u0 = 0; u0 < units; u0 += kChunk) {
    const int count = units - u0 < kChunk ? units - u0 : kChunk;
    float4 v[kChunk];
    load_chunk(v, xr, u0, count, g);
    float mn = m;
#pragma unroll
    for (int j = 0; j < kChunk; ++j) mn = max_with(mn, v[j]);  // the copies of the last unit change no maximum
    if (mn != -INFINITY) {
      const float mn2 = mn * kLog2e;
      float add = 0.f;
      each_of_chunk(u0, count, units, mine, [&](int j) {
        add += (exp_rel(v[j].x, mn2) + exp_rel(v[j].y, mn2)) + (exp_rel(v[j].z, mn2) + exp_rel(v[j].w, mn2));
      });
      s = s * exp2_of(m2 - mn2) + add;
      m2 = mn2;
    } else {
      bool any_nan = false;  // a maximum that dropped a NaN: keep it visible in the sum
#pragma unroll
      for (int j = 0; j < kChunk; ++j)
        any_nan |= v[j].x != v[j].x || v[j].y != v[j].y || v[j].z != v[j].z || v[j].w != v[j].w;
      if (any_nan) s = NAN;
    }
    m = mn;
  }
  const float mall = lanes_max(m, g.lanes);
  const float mall2 = mall * kLog2e;
  float part = (m == -INFINITY) ? ((s != s) ? s : 0.f) : s * exp2_of(m2 - mall2);
  const float sall = lanes_sum(part, g.lanes);
  const float inv_all = 1.f / sall;
  for (int u0 = 0; u0 < units; u0 += kChunk) {
    const int count = units - u0 < kChunk ? units - u0 : kChunk;
    float4 v[kChunk];
    load_chunk(v, xr, u0, count, g);
    each_of_chunk(u0, count, units, mine, [&](int j) {
      float4 o;
      o.x = exp_rel(v[j].x, mall2) * inv_all;
      o.y = exp_rel(v[j].y, mall2) * inv_all;
      o.z = exp_rel(v[j].z, mall2) * inv_all;
      o.w = exp_rel(v[j].w, mall2) * inv_all;
      store_streaming(orow + unit_offset<kShared>(u0 + j, g), o);
    });
  }
}

template <bool kShared>
__global__ __launch_bounds__(64 * kWaves) void softmax_bwd_kernel(const float *__restrict__ grad_out,
                                                          const float *__restrict__ y, float *__restrict__ grad_in,
                                                          const int32_t *__restrict__ row_offsets, int64_t n_tasks,
                                                          RowGeom g) {
  RowTask task;
  if (!wave_task<kShared>(g, row_offsets, n_tasks, task)) return;
  const int units = task.units;
  const RowPart<kShared> gr(grad_out, task), yr(y, task);
  float *dr = grad_in + task.first + task.lane_base;
  auto mine = [&](int u) { return !kShared || u < units - 1 || task.in_last; };  // of u < units

  if (units <= kBwdUnits) {
    float4 yv[kBwdUnits], gv[kBwdUnits];
    load_row(yv, yr, g);
    load_row(gv, gr, g);
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < kBwdUnits; ++u) {
      if (u < units && mine(u)) s += (yv[u].x * gv[u].x + yv[u].y * gv[u].y) + (yv[u].z * gv[u].z + yv[u].w * gv[u].w);
    }
    s = lanes_sum(s, g.lanes);
#pragma unroll
    for (int u = 0; u < kBwdUnits; ++u) {
      if (u < units && mine(u)) {
        float4 o;
        o.x = yv[u].x * (gv[u].x - s);
        o.y = yv[u].y * (gv[u].y - s);
        o.z = yv[u].z * (gv[u].z - s);
        o.w = yv[u].w * (gv[u].w - s);
        store_streaming(dr + unit_offset<kShared>(u, g), o);
      }
    }
    return;
  }

  if (units <= 2 * kBwdUnits) {
    // middle rows: y stays in registers, the gradient passes twice in chunks (once for the row's sum, once for the
    // result): 1.5 instead of 2 reads of the row's 2 x 16 bytes per element
    float4 yv[2 * kBwdUnits];
    load_row(yv, yr, g);
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < 2 * kBwdUnits; c += kChunk) {
      if (c < units) {
        const int count = units - c < kChunk ? units - c : kChunk;
        float4 gv[kChunk];
        load_chunk(gv, gr, c, count, g);
        each_of_chunk(c, count, units, mine, [&](int j) {
          s += (yv[c + j].x * gv[j].x + yv[c + j].y * gv[j].y) + (yv[c + j].z * gv[j].z + yv[c + j].w * gv[j].w);
        });
      }
    }
    s = lanes_sum(s, g.lanes);
#pragma unroll
    for (int c = 0; c < 2 * kBwdUnits; c += kChunk) {
      if (c < units) {
        const int count = units - c < kChunk ? units - c : kChunk;
        float4 gv[kChunk];
        load_chunk(gv, gr, c, count, g);
        each_of_chunk(c, count, units, mine, [&](int j) {
          float4 o;
          o.x = yv[c + j].x * (gv[j].x - s);
          o.y = yv[c + j].y * (gv[j].y - s);
          o.z = yv[c + j].z * (gv[j].z - s);
          o.w = yv[c + j].w * (gv[j].w - s);
          store_streaming(dr + unit_offset<kShared>(c + j, g), o);
        });
      }
    }
    return;
  }

  // long rows: two passes in chunks whose loads are all issued before the first one is used
  float s = 0.f;
  for (int u0 = 0; u0 < units; u0 += kChunk) {
    const int count = units - u0 < kChunk ? units - u0 : kChunk;
    float4 yv[kChunk], gv[kChunk];
    load_chunk(yv, yr, u0, count, g);
    load_chunk(gv, gr, u0, count, g);
    each_of_chunk(u0, count, units, mine, [&](int j) {
      s += (yv[j].x * gv[j].x + yv[j].y * gv[j].y) + (yv[j].z * gv[j].z + yv[j].w * gv[j].w);
    });
  }
  s = lanes_sum(s, g.lanes);
  for (int u0 = 0; u0 < units; u0 += kChunk) {
    const int count = units - u0 < kChunk ? units - u0 : kChunk;
    float4 yv[kChunk], gv[kChunk];
    load_chunk(yv, yr, u0, count, g);
    load_chunk(gv, gr, u0, count, g);
    each_of_chunk(u0, count, units, mine, [&](int j) {
      float4 o;
      o.x = yv[j].x * (gv[j].x - s);
      o.y = yv[j].y * (gv[j].y - s);
      o.z = yv[j].z * (gv[j].z - s);
      o.w = yv[j].w * (gv[j].w - s);
      store_streaming(dr + unit_offset<kShared>(u0 + j, g), o);
    });
  }
}

int make_geom(const char *who, int sbs, int64_t n_rows, int64_t nnz, int units, RowGeom &g) {
  BSA_REQUIRE(sbs >= 16 && bsa::is_pow2(sbs), "%s: sbs must be a power of two >= 16 (got %d)", who, sbs);
  int l = 0;
  while ((1 << l) < sbs) ++l;
  g.sbs_log2 = l;
  g.lpr = sbs / 4 < 64 ? sbs / 4 : 64;
  int nq = sbs / 256 > 1 ? sbs / 256 : 1;
  g.nq_log2 = 0;
  while ((1 << g.nq_log2) < nq) ++g.nq_log2;
  // As many groups of lanes on a row as bring one 5/3 times as long as the mean (a block-causal layout's longest is twice the
  // mean) down to `units` rounds.  Blocks of 16 keep two rows per wave, whole lines of 128 bytes (forward, sbs 16, above: 62
  // us so, 74 with a row per wave).  The launch stays below 2^31 threads.
  const int most = sbs == 16 ? 32 : 64;
  g.split_log2 = 0, g.lanes = g.lpr;
  while (2 * g.lanes <= most && 5 * (nnz >> g.split_log2) > 3 * units * n_rows && n_rows * sbs * 2 * g.lanes < ((int64_t)1 << 31))
    ++g.split_log2, g.lanes *= 2;
  g.groups_log2 = 0;
  while ((1 << g.groups_log2) < sbs * g.lanes / 64) ++g.groups_log2;
  return BSA_OK;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

// Forward, shared rows of eight units per lane leave seven waves per SIMD: sbs 64, above, 106 us, 114 with 16 to 32 units.  Rows
// of wider blocks stay whole up to 32 units: sbs 128 110 us so, 119 with 16 units in registers, 113 with two groups of lanes on a row.
// Backward, 16 units of both tensors: 153 us either way, but fewer, longer rounds at sbs 16 (83 against 92).
extern "C" int bsa_softmax_fwd(const float *x, float *out, const int32_t *row_offsets, int64_t n_rows, int64_t nnz,
                               int sbs, bsa_stream_t stream) {
  RowGeom g;
  if (int rc = make_geom("bsa_softmax_fwd", sbs, n_rows, nnz, sbs < 128 ? 8 : 32, g)) return rc;
  BSA_REQUIRE(n_rows >= 0 && nnz >= 0, "bsa_softmax_fwd: negative size");
  if (n_rows == 0 || nnz == 0) return BSA_OK;
  BSA_REQUIRE(x && out && row_offsets, "bsa_softmax_fwd: NULL pointer");
  BSA_REQUIRE(aligned16(x) && aligned16(out), "bsa_softmax_fwd: buffers must be 16-byte aligned");
  if (nnz > 0x7fffffffLL) return bsa::fail(BSA_ELIMIT, "bsa_softmax_fwd: more than 2^31-1 blocks");
  const int64_t n_tasks = n_rows << g.groups_log2;
  const int64_t blocks = bsa::cdiv(bsa::cdiv(n_tasks, kWaves), 8) * 8;  // a whole number of workgroups per XCD
  if (blocks > 0x7fffffffLL) return bsa::fail(BSA_ELIMIT, "bsa_softmax_fwd: too many rows");
  auto kernel = g.split_log2 == 0 ? &softmax_fwd_kernel<32, false> : sbs < 128 ? &softmax_fwd_kernel<16, true> : &softmax_fwd_kernel<32, true>;
  kernel<<<(unsigned)blocks, 64 * kWaves, 0, bsa::as_stream(stream)>>>(x, out, row_offsets, n_tasks, g);
  return bsa::check_launch("softmax_fwd_kernel");
}

extern "C" int bsa_softmax_bwd(const float *grad_out, const float *y, float *grad_in, const int32_t *row_offsets,
                               int64_t n_rows, int64_t nnz, int sbs, bsa_stream_t stream) {
  RowGeom g;
  if (int rc = make_geom("bsa_softmax_bwd", sbs, n_rows, nnz, kBwdUnits, g)) return rc;
  BSA_REQUIRE(n_rows >= 0 && nnz >= 0, "bsa_softmax_bwd: negative size");
  if (n_rows == 0 || nnz == 0) return BSA_OK;
  BSA_REQUIRE(grad_out && y && grad_in && row_offsets, "bsa_softmax_bwd: NULL pointer");
  BSA_REQUIRE(aligned16(grad_out) && aligned16(y) && aligned16(grad_in),
              "bsa_softmax_bwd: buffers must be 16-byte aligned");
  if (nnz > 0x7fffffffLL) return bsa::fail(BSA_ELIMIT, "bsa_softmax_bwd: more than 2^31-1 blocks");
  const int64_t n_tasks = n_rows << g.groups_log2;
  const int64_t blocks = bsa::cdiv(bsa::cdiv(n_tasks, kWaves), 8) * 8;  // a whole number of workgroups per XCD
  if (blocks > 0x7fffffffLL) return bsa::fail(BSA_ELIMIT, "bsa_softmax_bwd: too many rows");
  auto kernel = g.split_log2 == 0 ? &softmax_bwd_kernel<false> : &softmax_bwd_kernel<true>;
  kernel<<<(unsigned)blocks, 64 * kWaves, 0, bsa::as_stream(stream)>>>(grad_out, y, grad_in, row_offsets, n_tasks, g);
  return bsa::check_launch("softmax_bwd_kernel");
}
