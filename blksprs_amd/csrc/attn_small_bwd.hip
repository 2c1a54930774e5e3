// Block-sparse flash attention backward for blocks of 16 and 32 and head dimensions up to 128, fp16, bf16 and fp32 (the
// forward kernel: attn_small_fwd.hip; tiles, fragments and the walk over a list: attn_small_common.h).
//
// Two launches, no atomics, fixed summation order.  The first gives a wave a query block: delta = rowsum(o * dO) from the
// fragments of o and dO it holds anyway, then dQ (and dBias) over the block's key list.  The second gives a wave a key
// block: dK and dV over its query list.  Both form scores, probabilities and dP of every pair themselves, so no
// intermediate of the size of the attention layout exists; a wave walks alone, without barriers.  A lane owns one
// row of the own block in every product, so P and dS pass from the accumulators of one product into the operands of
// the next without leaving registers:
//
//   dQ kernel, lane owns a query i, registers run over keys j:
//     dP^T = V dO^T, S^T = K Q^T    rows of V, K from LDS, dO and Q in registers
//     dQ^T += K^T dS^T              columns of K from LDS
//   dK / dV kernel, lane owns a key j, registers run over queries i:
//     S = Q K^T, dP = dO V^T        rows of Q, dO from LDS, K and V in registers
//     dV^T += dO^T P, dK^T += Q^T dS columns of dO, Q from LDS
//
// What bounds it: the chain of a step (tiles awaited, products, exponentials, products) with one (dK / dV at head dimension 128)
// to seven waves per SIMD to overlap it, two or three for blocks of 32 at 64.  Against the fp32 matrix-core kernels that ran these shapes before (48 x 4096 queries, sbs 32, head
// dimension 64, fp16, 33 key blocks per query block): delta + zero fill 0.071 -> 0, dK / dV 1.89 -> 0.125 ms (530 TFLOP/s),
// dQ 1.24 -> 0.090 ms (delta included); fp32, sbs 32, products from bf16 parts (split_f32.h), 8 x 2048 queries, half of the
// blocks, head dimension 64: dK / dV 94.5 -> 73.1, dQ 74.8 -> 55.8 us (118 and 115 TFLOP/s) against the fp32 instruction.  fp32
// blocks of 64, whose halves walk alone like blocks of 32: 20 x 960, causal, head dimension 64: delta + zero fill 19 -> 0, dK /
// dV 129 (eight waves to a tile) -> 44, dQ 128 -> 37 us.
//
// Scores as in the forward kernel; p = exp2(s - lse), 0 where lse = -inf; P and dS are rounded to the operand type
// before they enter a product (blksprs/ops/flash_attention.py:1452, :1468, :1692).
#include <type_traits>

#include "attn_small_common.h"

namespace bsa {
namespace {

using namespace small;

constexpr int kWaves = 4;

template <int ES, int SBS, int NS, int kHalves>
struct BwdShape {
  static constexpr int NB = SBS == 32 ? 1 : 2;  // partner blocks per step
  using T = Tile<ES, SBS, NS, NB, kHalves>;
  static constexpr int kRegs = SBS == 32 ? 16 : 4;
  static constexpr int kScores = kRegs * NB;
  static constexpr int kPartial = SBS * SBS * NS * 4;
  static constexpr int kSlot = SBS * SBS * NS;  // floats of a slot of the scratch, twice for dK and dV
  static constexpr int kStats = 256;  // lse and delta of the 32 queries of a step
  // the last row fragment of an odd number of slices of 16 reads (and drops) a slice beyond its tile
  static constexpr int kPad = T::kHalfLast ? T::kPiece : 0;
  // dK / dV kernel of 16-bit blocks of 32: tiles of two steps, so that a step's copies go out a step ahead.  Up to head dimension 64 a
  // wave has LDS for both tiles twice, which its own dK and dV need anyway once it is done.  Beyond, that (twice the tiles of a step)
  // left a SIMD one wave: there the sums go through the tiles of all waves of a row, P is used up before dP is formed, and only Q,
  // which is read first and last in a step, has a second tile: two waves at 96, one and shorter waits at 128.  Forward + backward of
  // bf16: 24 x 4096, windows of 1024, head dimension 96: 243 -> 213 us; causal, 128: 530 -> 512.  The same at 64, with one tile of
  // each and three waves (five registers spilled), is faster where three are there to be run and lists are even, 24 x 2048, 30 %
  // of the blocks, 84 -> 81, and slower elsewhere: 12 x 3008, causal, 108 -> 118, 24 x 1536 65 -> 70, 4 x 1024 34.3 -> 36.3;
  // at 32 (four waves for three) backward of 24 x 2048, 30 %, 39.0 -> 40.9, of 8 x 1024 15.1 -> 16.1.
  static constexpr bool kTwoQ = ES == 2 && SBS == 32, kTwoG = kTwoQ && NS <= 2;
  static constexpr int kTiles = kTwoG ? 4 : kTwoQ ? 3 : 2;
  static constexpr int kKvLds = kPad + kTiles * T::kBytes + (kTwoQ ? 2 : 1) * kStats;
  static constexpr int kQLds = kPad + (2 * T::kBytes > kPartial ? 2 * T::kBytes : kPartial);
  static constexpr int kQMinWaves = ES == 4 ? (NS * SBS <= 64 ? 2 : 1) : SBS == 32 ? (NS <= 2 ? 3 : 2) : (NS <= 4 ? 4 : 2);
  static constexpr int kKvMinWaves = ES == 4 ? (NS * SBS <= 64 ? 2 : 1) : SBS == 32 ? (NS <= 3 ? 2 : 1) : (NS <= 4 ? 3 : 2);
};

// 4 bytes per lane, global -> LDS: lane l's value lands at dst + 4 l
__device__ inline void copy_words_to_lds(const float *addr, char *dst) {
  const uint32_t lds_addr = (uint32_t)(uintptr_t)(lds_ptr_t)dst;
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(addr), "s"(lds_addr) : "memory");
}

// NS gradient blocks of the own row, from slice `first` on, columns 2 r + 4 group .. + 3 of a row per lane
template <typename Tr, int SBS, int NS, int kHalves, typename Acc>
__device__ inline void store_gradient(const Acc (&acc)[NS], float scale, void *out, const int64_t *pidx, int n_slices,
                                      int64_t n_blocks, int own, int first, int me, int group) {
  constexpr int kRegs = SBS == 32 ? 16 : 4;
#pragma unroll
  for (int h = 0; h < NS; ++h) {
    const int slice = first + h;
    if (slice / kHalves >= n_slices) break;
    const int64_t p = pidx[slice / kHalves];
    if (p < 0 || p >= n_blocks) continue;
    char *blk = static_cast<char *>(out) + Place<Tr::kElem, SBS, kHalves>::row(p, own, me, slice) + 4 * group * Tr::kElem;
#pragma unroll
    for (int r = 0; r < kRegs; r += 4)
      store4<Tr>(blk + 2 * r * Tr::kElem, acc[h][r] * scale, acc[h][r + 1] * scale, acc[h][r + 2] * scale, acc[h][r + 3] * scale);
  }
}

// kHalves 2: blocks of 64, whose halves are the blocks of 32 spoken of here (Place)
template <typename Tr, int SBS, int NS, bool kSome, int kHalves>
__global__ __launch_bounds__(64 * kWaves, (BwdShape<Tr::kElem, SBS, NS, kHalves>::kQMinWaves)) void attn_small_dq_kernel(bsa_attn_args a, int split, Shares shares) {
  using Shape = BwdShape<Tr::kElem, SBS, NS, kHalves>;
  using T = typename Shape::T;
  using W = Walk<Tr::kElem, SBS, NS, Shape::NB, true, kSome, kHalves>;
  constexpr int NB = Shape::NB, kScores = Shape::kScores, kRegs = Shape::kRegs;
  using acc_t = std::conditional_t<SBS == 32, f32x16, f32x4>;
  extern __shared__ __attribute__((aligned(1024))) char small_smem[];
  const int lane = threadIdx.x & 63;
  const int wave = first_lane(threadIdx.x >> 6);
  char *lds_k = small_smem + wave * Shape::kQLds, *lds_v = lds_k + T::kBytes;

  const RowOfWave me(shares, kHalves, a.B, kHalves * a.nq, true, wave, kWaves, split);
  const int64_t row = me.b * a.nq + me.own / kHalves;  // of the layout
  const int64_t stats = (row * kHalves + me.own % kHalves) * SBS;  // of lse and delta
  const int qi = lane % SBS, kq = lane / SBS;
  W walk;
  walk.start(a, me.b, me.own, me.there, me.part, me.parts);

  OwnRows<Tr::kElem, SBS, NS, kHalves> qf, gf;
  acc_t dq[NS];
  auto start_row = [&](int lane) __attribute__((always_inline)) {
    qf.load(a.q, a.pidx_q + row * a.nh, (int)a.nh, a.n_q_blocks, (int)me.own, lane);
    gf.load(a.d_o, a.pidx_o + row * a.nhv, (int)a.nhv, a.n_o_blocks, (int)me.own, lane);
#pragma unroll
    for (int h = 0; h < NS; ++h)
#pragma unroll
      for (int r = 0; r < kRegs; ++r) dq[h][r] = 0.f;
  };
  start_row(lane);
  float delta = 0.f, neg_lse = -a.lse[stats + qi];
  if (neg_lse == INFINITY) neg_lse = -INFINITY;  // a query that sees nothing: p = 0
  {
    OwnRows<Tr::kElem, SBS, NS, kHalves> of;
    of.load(a.o, a.pidx_o + row * a.nhv, (int)a.nhv, a.n_o_blocks, (int)me.own, lane);
#pragma unroll
    for (int f = 0; f < T::kFrags; ++f) delta = Tr::dot(of.fr[f], gf.fr[f], delta);
    delta = row_sum<SBS>(delta);
    if (me.there && me.part == 0 && kq == 0) a.delta[stats + qi] = delta;
  }
  const float qk_scale = a.scale * kLog2e;
  const float cc = a.bias ? 1.f : qk_scale;
  const uint32_t source = T::source_offset(lane);
  const char *const tensor_k = static_cast<const char *>(a.k), *const tensor_v = static_cast<const char *>(a.v);
  const typename T::RowReader k_rows(lds_k, lane), v_rows(lds_v, lane);
  const typename T::ColReader k_cols(lds_k, lane);
  // whether the sums are what they should be (from parts they may not be)
  auto walk_list = [&](auto arithmetic) __attribute__((always_inline)) -> bool {
    using Ar = decltype(arithmetic);
    typename W::Step now, next;
    walk.take(now, lane);
    settle(qf);
    settle(gf);
    if constexpr (std::is_same_v<Ar, SSplit>) {
      if (scores_in_doubt(qf, a.scale)) return false;
    }
    const OwnOperand<Ar, SBS, NS, kHalves, false> q_operand(qf);
    const OwnOperand<Ar, SBS, NS, kHalves, true> g_operand(gf);
    constexpr float kTimes = up_of<Ar>();
    const float delta_up = delta * kTimes;
    bool counted = false;  // exactly kCopies copies were issued after the tile that is needed next
    if (now.count) {
      walk.template copy<true>(now, tensor_v, lds_v, source, lane);
      counted = walk.template copy<false>(now, tensor_k, lds_k, source, lane);
    }
    while (now.count) {
      // ---- dP^T = V dO^T.  In flight at most: V and K of this step, in that order.
      if (counted) wait_vmem<T::kCopies>();
      else wait_vmem<0>();
      acc_t dp[NB], sacc[NB];
      W::template multiply_rows<Ar, true>(dp, now, v_rows, g_operand, lane);
      wait_lds();
      walk.take(next, lane);
      counted = false;
      if (next.count) counted = walk.template copy<true>(next, tensor_v, lds_v, source, lane);

      // ---- S^T = K Q^T.  In flight at most: K of this step, V of the next.
      if (counted) wait_vmem<T::kCopies>();
      else wait_vmem<0>();
      W::template multiply_rows<Ar, false>(sacc, now, k_rows, q_operand, lane);
      float sv[kScores];
#pragma unroll
      for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int r = 0; r < kRegs; ++r) sv[kRegs * t + r] = sacc[t][r];
      if (now.special) walk.template finish_scores<Tr>(now, sv, qk_scale, qi, kq);
      apply_factor<Tr, kScores>(sv, cc);

      // ---- dS = P (dP - delta), times up_of as a second operand (dP: up_of^2)
#pragma unroll
      for (int x = 0; x < kScores; ++x)
        sv[x] = __builtin_amdgcn_exp2f(fmaf(sv[x], late_factor<Tr>(cc), neg_lse)) * fmaf(dp[x / kRegs][x % kRegs], 1.f / kTimes, -delta_up);
      if (now.special) {
        const late_args_t p = late_args();
        if (p->dbias) {  // every pair is visited once: plain stores
#pragma unroll
          for (int t = 0; t < NB; ++t)
            if (now.bias[t] >= 0) {
              constexpr int kSide = kHalves * SBS;
              float *out = p->dbias + ((int64_t)now.bias[t] * kSide + (int)me.own % kHalves * SBS + qi) * kSide +
                           now.other[t] % kHalves * SBS + 4 * kq;
#pragma unroll
              for (int r = 0; r < kRegs; r += 4) {
                const float *v = sv + kRegs * t + r;
                *reinterpret_cast<f32x4 *>(out + 2 * r) = f32x4{v[0], v[1], v[2], v[3]} * (1.f / kTimes);
              }
            }
        }
      }
      // ---- dQ^T += K^T dS^T
      W::template multiply_cols<Ar, false, kScores>(dq, now, k_cols, Weights<Ar, kScores>(sv));
      wait_lds();
      counted = false;
      if (next.count) counted = walk.template copy<false>(next, tensor_k, lds_k, source, lane);
      now = next;
    }
    if constexpr (!std::is_same_v<Ar, SSplit>) return true;
    scale_down<Ar, NS, kRegs>(dq);
    return !not_finite<NS, kRegs>(dq);
  };
  if constexpr (in_parts<Tr, SBS, kSome>()) {
    if (!walk_list(SSplit{})) {  // once more with the fp32 instruction
      walk.start(a, me.b, me.own, me.there, me.part, me.parts);
      start_row(fresh_lane());
      walk_list(Tr{});
    }
  } else {
    walk_list(Tr{});
  }
  if (me.waves > 1) {
    float *mine = reinterpret_cast<float *>(lds_k);
    if (me.place != 0) leave_partial<NS, kRegs>(dq, mine, lane);
    __syncthreads();
    if (me.place != 0) return;
    for (int p = 1; p < me.waves; ++p) add_partial<NS, kRegs>(dq, mine + p * (Shape::kQLds / 4), lane);
  }
  if (!me.there) return;
  if (me.slot >= 0) {  // other workgroups have the rest of the row: attn_small_bwd_merge_kernel adds them up
    leave_partial<NS, kRegs>(dq, shares.partials + (int64_t)me.slot * Shape::kSlot, lane);
    return;
  }
  const late_args_t p = late_args();
  store_gradient<Tr, SBS, NS, kHalves>(dq, p->scale, p->dq, p->pidx_q + row * p->nh, (int)p->nh, p->n_q_blocks, (int)me.own, 0, qi, kq);
}

template <typename Tr, int SBS, int NS, bool kSome, int kHalves>
__global__ __launch_bounds__(64 * kWaves, (BwdShape<Tr::kElem, SBS, NS, kHalves>::kKvMinWaves)) void attn_small_dkv_kernel(bsa_attn_args a, int split, Shares shares) {
  using Shape = BwdShape<Tr::kElem, SBS, NS, kHalves>;
  using T = typename Shape::T;
  using W = Walk<Tr::kElem, SBS, NS, Shape::NB, false, kSome, kHalves>;
  constexpr int NB = Shape::NB, kScores = Shape::kScores, kRegs = Shape::kRegs;
  constexpr bool kTwoQ = Shape::kTwoQ, kTwoG = Shape::kTwoG;
  using acc_t = std::conditional_t<SBS == 32, f32x16, f32x4>;
  extern __shared__ __attribute__((aligned(1024))) char small_smem[];
  const int lane = threadIdx.x & 63;
  const int wave = first_lane(threadIdx.x >> 6);
  char *lds = small_smem + wave * Shape::kKvLds;  // a Q and a dO tile, the second ones, lse and delta of one or two steps

  const RowOfWave me(shares, kHalves, a.B, kHalves * a.nk, false, wave, kWaves, split);
  const int64_t row = me.b * a.nk + me.own / kHalves;  // of the layout
  const int kj = lane % SBS, kq = lane / SBS;  // key row; which queries of a block this lane's registers hold
  W walk;
  walk.start(a, me.b, me.own, me.there, me.part, me.parts);

  OwnRows<Tr::kElem, SBS, NS, kHalves> kf, vf;
  acc_t dk[NS], dv[NS];
  auto start_row = [&](int lane) __attribute__((always_inline)) {
    kf.load(a.k, a.pidx_k + row * a.nh, (int)a.nh, a.n_k_blocks, (int)me.own, lane);
    vf.load(a.v, a.pidx_v + row * a.nhv, (int)a.nhv, a.n_v_blocks, (int)me.own, lane);
#pragma unroll
    for (int h = 0; h < NS; ++h)
#pragma unroll
      for (int r = 0; r < kRegs; ++r) dk[h][r] = dv[h][r] = 0.f;
  };
  start_row(lane);

  const float qk_scale = a.scale * kLog2e;
  const float cc = a.bias ? 1.f : qk_scale;
  const uint32_t source = T::source_offset(lane);
  const char *const tensor_q = static_cast<const char *>(a.q), *const tensor_g = static_cast<const char *>(a.d_o);
  // this lane's share of the statistics copy: lanes 0 .. 31 lse, 32 .. 63 delta of the step's 32 queries
  const int64_t queries = me.b * a.nq * (kHalves * SBS);
  const float *const stats = (lane < 32 ? a.lse : a.delta) + queries + lane % SBS;
  const int stats_block = SBS == 16 ? (lane >> 4) & 1 : 0;
  // 16-bit blocks of 32 beyond head dimension 64: addresses are formed where they are used, since registers are what limits the waves
  constexpr bool kLateAddresses = kTwoQ && !kTwoG;
  auto copy_stats = [&](const typename W::Step &s, char *dst) {
    int other = __builtin_amdgcn_readlane(walk.other, s.slot[0]);
    if constexpr (kLateAddresses) {
      const late_args_t p = late_args();
      const int l = fresh_lane();
      const float *lse = p->lse + queries, *delta = p->delta + queries;
      lse += (int64_t)other * SBS, delta += (int64_t)other * SBS;
      copy_words_to_lds((l < 32 ? lse : delta) + l % SBS, dst);
      return;
    }
    if constexpr (NB > 1) {
      const int second = s.count > 1 ? __builtin_amdgcn_readlane(walk.other, s.slot[1]) : other;
      other = stats_block ? second : other;
    }
    copy_words_to_lds(stats + (int64_t)other * SBS, dst);
  };
  constexpr int kStatsAt = Shape::kTiles * T::kBytes;
  const typename T::RowReader q_rows0(lds, lane), g_rows0(lds + T::kBytes, lane);
  const typename T::ColReader q_cols0(lds, lane), g_cols0(lds + T::kBytes, lane);
  auto walk_list = [&](auto arithmetic) __attribute__((always_inline)) -> bool {  // as in the dQ kernel
    using Ar = decltype(arithmetic);
    typename W::Step now, next;
    walk.take(now, lane);
    settle(kf);
    settle(vf);
    if constexpr (std::is_same_v<Ar, SSplit>) {
      if (scores_in_doubt(kf, a.scale)) return false;
    }
    const OwnOperand<Ar, SBS, NS, kHalves, false> k_operand(kf);
    const OwnOperand<Ar, SBS, NS, kHalves, true> v_operand(vf);
    constexpr float kTimes = up_of<Ar>();  // of P and dS as second operands; dP: the square
    // kTwoQ: Q and the statistics of a step are requested a step ahead; dO as well (kTwoG), or as soon as this step has used its own
    int at = 0;  // 0 or 1: which of two tiles and statistics
    bool g_counted = kTwoG;  // dO of this step: exactly kCopies copies (kTwoG: in place with Q)
    typename T::RowReader q_rows = q_rows0, g_rows = g_rows0;
    typename T::ColReader q_cols = q_cols0, g_cols = g_cols0;
    const float *lse = reinterpret_cast<const float *>(lds + kStatsAt);
    if (now.count) {
      walk.template copy<false>(now, tensor_q, lds, source, lane);
      copy_stats(now, lds + kStatsAt);
      const bool counted = walk.template copy<true>(now, tensor_g, lds + T::kBytes, source, lane);
      if constexpr (!kTwoG) g_counted = counted;
    }
    while (now.count) {
      bool counted = false;  // what is requested here for the next step: exactly kCopies + 1 copies (kTwoG: 2 kCopies + 1)
      if constexpr (kTwoQ) {
        // the copies of slices that may be missing are not counted: this step's are awaited before the next step's go out (behind
        // them the wait is for both: backward of 24 x 2048, 30 % of the blocks, a tenth of the slices missing, 64 84.7 -> 82.8 us,
        // 96 121 -> 118, 128 184 -> 179)
        if constexpr (kSome) wait_vmem<0>();
        walk.take(next, lane);
        if (next.count) {
          char *const to = lds + (at ^ 1) * 2 * T::kBytes;
          counted = walk.template copy<false>(next, tensor_q, to, source, lane);
          if constexpr (kTwoG) counted = walk.template copy<true>(next, tensor_g, to + T::kBytes, source, lane) && counted;
          copy_stats(next, lds + kStatsAt + (at ^ 1) * Shape::kStats);
        }
        if constexpr (!kSome) {
          if (counted && g_counted) wait_vmem<2 * T::kCopies + 1>();
          else wait_vmem<0>();
        }
      } else {
        wait_vmem<0>();
      }
      const float *const delta = lse + 32;

      // ---- S = Q K^T, P = exp2(S - lse)
      acc_t sacc[NB], dp[NB];
      W::template multiply_rows<Ar, false>(sacc, now, q_rows, k_operand, lane);
      float sv[kScores], ls[kScores];
#pragma unroll
      for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int r = 0; r < kRegs; ++r) sv[kRegs * t + r] = sacc[t][r];
      if (now.special) walk.template finish_scores<Tr>(now, sv, qk_scale, kj, kq);
      apply_factor<Tr, kScores>(sv, cc);
#pragma unroll
      for (int x = 0; x < kScores; x += 4) {
        const f32x4 l4 = *reinterpret_cast<const f32x4 *>(lse + (x / kRegs) * SBS + 2 * (x % kRegs) + 4 * kq);
#pragma unroll
        for (int i = 0; i < 4; ++i) ls[x + i] = l4[i];
      }
      // in parts, and where only Q has two tiles, P is used up before dP is formed, for want of registers
      constexpr bool kLateDp = std::is_same_v<Ar, SSplit> || (kTwoQ && !kTwoG);
      if constexpr (!kLateDp) W::template multiply_rows<Ar, true>(dp, now, g_rows, v_operand, lane);
      float lowest = ls[0];
#pragma unroll
      for (int x = 1; x < kScores; ++x) lowest = fminf(lowest, ls[x]);
      if (__any(lowest == -INFINITY)) {  // a query that sees nothing: p = 0
#pragma unroll
        for (int x = 0; x < kScores; ++x)
          if (ls[x] == -INFINITY) ls[x] = INFINITY;
      }
#pragma unroll
      for (int x = 0; x < kScores; ++x) sv[x] = __builtin_amdgcn_exp2f(fmaf(sv[x], late_factor<Tr>(cc), -ls[x])) * kTimes;
      const Weights<Ar, kScores> pw(sv);
      if constexpr (kTwoQ && !kTwoG && !kSome) {
        if (counted) wait_vmem<T::kCopies + 1>();
        else wait_vmem<0>();
      }
      if constexpr (kLateDp) {
        W::template multiply_cols<Ar, true, kScores>(dv, now, g_cols, pw);
        W::template multiply_rows<Ar, true>(dp, now, g_rows, v_operand, lane);
      }

      // ---- dS = P (dP - delta)
#pragma unroll
      for (int x = 0; x < kScores; x += 4) {
        const f32x4 d4 = *reinterpret_cast<const f32x4 *>(delta + (x / kRegs) * SBS + 2 * (x % kRegs) + 4 * kq);
#pragma unroll
        for (int i = 0; i < 4; ++i) sv[x + i] *= fmaf(dp[x / kRegs][x % kRegs + i], 1.f / (kTimes * kTimes), -d4[i]);
      }
      // ---- dV^T += dO^T P
      if constexpr (!kLateDp) W::template multiply_cols<Ar, true, kScores>(dv, now, g_cols, pw);
      if constexpr (!kTwoG) {
        wait_lds();
        if constexpr (!kTwoQ) walk.take(next, lane);
        if (next.count) {
          g_counted = walk.template copy<true>(next, tensor_g, lds + T::kBytes, source, lane);
          if constexpr (!kTwoQ) copy_stats(next, lds + kStatsAt);
        }
      }
      // ---- dK^T += Q^T dS
      W::template multiply_cols<Ar, false, kScores>(dk, now, q_cols, Weights<Ar, kScores>(sv));
      wait_lds();
      if constexpr (kTwoQ) {
        const int turn = at ? -1 : 1;
        q_rows.shift(turn * 2 * T::kBytes), q_cols.shift(turn * 2 * T::kBytes);
        if constexpr (kTwoG) g_rows.shift(turn * 2 * T::kBytes), g_cols.shift(turn * 2 * T::kBytes);
        lse += turn * (Shape::kStats / 4);
        at ^= 1;
      } else if (next.count) {
        walk.template copy<false>(next, tensor_q, lds, source, lane);
      }
      now = next;
    }
    if constexpr (!std::is_same_v<Ar, SSplit>) return true;
    scale_down<Ar, NS, kRegs>(dk);
    scale_down<Ar, NS, kRegs>(dv);
    return !not_finite<NS, kRegs>(dk) && !not_finite<NS, kRegs>(dv);
  };
  if constexpr (in_parts<Tr, SBS, kSome>()) {
    if (!walk_list(SSplit{})) {  // once more with the fp32 instruction
      walk.start(a, me.b, me.own, me.there, me.part, me.parts);
      start_row(fresh_lane());
      walk_list(Tr{});
    }
  } else {
    walk_list(Tr{});
  }
  if (me.waves > 1) {
    if constexpr (Shape::kKvLds >= 2 * Shape::kPartial) {
      float *mine = reinterpret_cast<float *>(lds);
      if (me.place != 0) {
        leave_partial<NS, kRegs>(dk, mine, lane);
        leave_partial<NS, kRegs>(dv, mine + Shape::kPartial / 4, lane);
      }
      __syncthreads();
      if (me.place != 0) return;
      for (int p = 1; p < me.waves; ++p) {
        add_partial<NS, kRegs>(dk, mine + p * (Shape::kKvLds / 4), lane);
        add_partial<NS, kRegs>(dv, mine + p * (Shape::kKvLds / 4) + Shape::kPartial / 4, lane);
      }
    } else {
      // sums that are larger than a wave's tiles (16-bit blocks of 32 beyond head dimension 64): the tiles of all waves of the row
      // take in as many sums at a time as they hold, once the walks are over
      static_assert(Shape::kKvLds >= Shape::kPartial, "the sums of a wave in the tiles of two");
      float *const sums = reinterpret_cast<float *>(lds - me.place * Shape::kKvLds);
      const int fit = me.waves * Shape::kKvLds / (2 * Shape::kPartial);
      for (int first = 1; first < me.waves; first += fit) {
        __syncthreads();
        if (me.place >= first && me.place < first + fit) {
          float *mine = sums + (me.place - first) * (Shape::kPartial / 2);
          leave_partial<NS, kRegs>(dk, mine, lane);
          leave_partial<NS, kRegs>(dv, mine + Shape::kPartial / 4, lane);
        }
        __syncthreads();
        if (me.place != 0) continue;
        for (int p = first; p < me.waves && p < first + fit; ++p) {
          const float *other = sums + (p - first) * (Shape::kPartial / 2);
          add_partial<NS, kRegs>(dk, other, lane);
          add_partial<NS, kRegs>(dv, other + Shape::kPartial / 4, lane);
        }
      }
      if (me.place != 0) return;
    }
  }
  if (!me.there) return;
  if (me.slot >= 0) {
    float *out = shares.partials + (int64_t)me.slot * (2 * Shape::kSlot);
    leave_partial<NS, kRegs>(dk, out, lane);
    leave_partial<NS, kRegs>(dv, out + Shape::kSlot, lane);
    return;
  }
  const late_args_t p = late_args();
  store_gradient<Tr, SBS, NS, kHalves>(dk, p->scale, p->dk, p->pidx_k + row * p->nh, (int)p->nh, p->n_k_blocks, (int)me.own, 0, kj, kq);
  store_gradient<Tr, SBS, NS, kHalves>(dv, 1.f, p->dv, p->pidx_v + row * p->nhv, (int)p->nhv, p->n_v_blocks, (int)me.own, 0, kj, kq);
}

// The gradients of rows that several workgroups share, a wave for each head slice (blockIdx.y): dQ of the first n_q merges
// (times the halves), then dK and dV (blockIdx.z) of the others.  A merge is (batch entry, row of the layout, first slot, slots).
template <typename Tr, int SBS, int NS, int kHalves>
__global__ __launch_bounds__(64) void attn_small_bwd_merge_kernel(bsa_attn_args a, const int32_t *merges_q, const float *partials_q,
                                                                  int64_t n_q, const int32_t *merges_kv, const float *partials_kv) {
  using Shape = BwdShape<Tr::kElem, SBS, NS, kHalves>;
  constexpr int kRegs = Shape::kRegs;
  using acc_t = std::conditional_t<SBS == 32, f32x16, f32x4>;
  const int lane = threadIdx.x, me = lane % SBS, group = lane / SBS, half = blockIdx.x % kHalves, h = blockIdx.y;
  const int64_t m = blockIdx.x / kHalves;
  const bool is_q = m < n_q, is_v = blockIdx.z == 1;
  if (is_q && is_v) return;
  const int32_t *merge = is_q ? merges_q + m * 4 : merges_kv + (m - n_q) * 4;
  const int64_t row = (int64_t)merge[0] * (is_q ? a.nq : a.nk) + merge[1];
  const int own = merge[1] * kHalves + half, n = merge[3];
  const int64_t slot = is_q ? Shape::kSlot : 2 * Shape::kSlot, step = kHalves * slot;
  const float *part = (is_q ? partials_q : partials_kv) + ((int64_t)merge[2] * kHalves + half) * slot + (is_v ? Shape::kSlot : 0) +
                      h * kRegs * 64;
  acc_t acc[1];
#pragma unroll
  for (int r = 0; r < kRegs; ++r) acc[0][r] = 0.f;
#pragma unroll 4
  for (int s = 0; s < n; ++s) add_partial<1, kRegs>(acc, part + s * step, lane);
  if (is_v) store_gradient<Tr, SBS, 1, kHalves>(acc, 1.f, a.dv, a.pidx_v + row * a.nhv, (int)a.nhv, a.n_v_blocks, own, h, me, group);
  else if (is_q) store_gradient<Tr, SBS, 1, kHalves>(acc, a.scale, a.dq, a.pidx_q + row * a.nh, (int)a.nh, a.n_q_blocks, own, h, me, group);
  else store_gradient<Tr, SBS, 1, kHalves>(acc, a.scale, a.dk, a.pidx_k + row * a.nh, (int)a.nh, a.n_k_blocks, own, h, me, group);
}

// bias blocks outside the attention layout, and pairs the causal predicate rules out, have no wave that writes them
__global__ void small_zero_kernel(f32x4 *out, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) out[i] = f32x4{0.f, 0.f, 0.f, 0.f};
}

template <typename Tr, int SBS, int NS, bool kSome, int kHalves>
int launch_kind(const bsa_attn_args &a, const bsa_attn_shares *sh_q, const bsa_attn_shares *sh_kv, hipStream_t s) {
  using Shape = BwdShape<Tr::kElem, SBS, NS, kHalves>;
  constexpr int q_lds = Shape::kQLds * kWaves, kv_lds = Shape::kKvLds * kWaves;
  static_assert(q_lds <= 160 * 1024 && kv_lds <= 160 * 1024, "LDS");
  static LdsLimit limit_q, limit_kv;
  if (int rc = allow_lds(limit_q, &attn_small_dq_kernel<Tr, SBS, NS, kSome, kHalves>, q_lds)) return rc;
  if (int rc = allow_lds(limit_kv, &attn_small_dkv_kernel<Tr, SBS, NS, kSome, kHalves>, kv_lds)) return rc;
  const int64_t q_rows = kHalves * a.nq, k_rows = kHalves * a.nk;  // of a batch entry
  const int q_split = waves_per_row<Tr::kElem>(a.B * q_rows, k_rows, Shape::NB);
  const int kv_split = waves_per_row<Tr::kElem>(a.B * k_rows, q_rows, Shape::NB);
  const int64_t q_groups = sh_q ? kHalves * sh_q->n_groups : row_groups(a.B, q_rows, kWaves, q_split);
  const int64_t kv_groups = sh_kv ? kHalves * sh_kv->n_groups : row_groups(a.B, k_rows, kWaves, kv_split);
  if (!fits_launch(q_groups, kWaves) || !fits_launch(kv_groups, kWaves)) return 1;
  Shares shares_q{nullptr, nullptr}, shares_kv{nullptr, nullptr};
  for (const bsa_attn_shares *sh : {sh_q, sh_kv}) {
    if (!sh) continue;
    const int64_t need = sh->n_slots * kHalves * Shape::kSlot * 4 * (sh == sh_kv ? 2 : 1);
    BSA_REQUIRE(need <= sh->scratch_bytes, "bsa_attn_bwd_shares: scratch holds %lld bytes, %lld are needed",
                (long long)sh->scratch_bytes, (long long)need);
    (sh == sh_q ? shares_q : shares_kv) = Shares{sh->groups, static_cast<float *>(sh->scratch)};
  }
  if (a.dbias && a.n_bias_blocks > 0) {
    const int64_t n = a.n_bias_blocks * a.sbs * a.sbs / 4, blocks = cdiv(n, (int64_t)256);
    small_zero_kernel<<<(unsigned)(blocks < 65536 ? blocks : 65536), 256, 0, s>>>(reinterpret_cast<f32x4 *>(a.dbias), n);
    if (int rc = check_launch("small_zero_kernel")) return rc;
  }
  if (a.B * a.nq) {
    attn_small_dq_kernel<Tr, SBS, NS, kSome, kHalves><<<(unsigned)q_groups, 64 * kWaves, q_lds, s>>>(a, q_split, shares_q);
    if (int rc = check_launch("attn_small_dq_kernel")) return rc;
  }
  if (a.B * a.nk) {
    attn_small_dkv_kernel<Tr, SBS, NS, kSome, kHalves><<<(unsigned)kv_groups, 64 * kWaves, kv_lds, s>>>(a, kv_split, shares_kv);
    if (int rc = check_launch("attn_small_dkv_kernel")) return rc;
  }
  const int64_t q_merges = sh_q ? sh_q->n_merges : 0, kv_merges = sh_kv ? sh_kv->n_merges : 0;
  if (q_merges + kv_merges > 0) {
    attn_small_bwd_merge_kernel<Tr, SBS, NS, kHalves><<<dim3((unsigned)((q_merges + kv_merges) * kHalves), NS, kv_merges ? 2 : 1), 64, 0, s>>>(
        a, sh_q ? sh_q->merges : nullptr, shares_q.partials, q_merges, sh_kv ? sh_kv->merges : nullptr, shares_kv.partials);
    if (int rc = check_launch("attn_small_bwd_merge_kernel")) return rc;
  }
  return BSA_OK;
}

template <typename Tr, int SBS, int NS>
int launch(const bsa_attn_args &a, const bsa_attn_shares *sh_q, const bsa_attn_shares *sh_kv, hipStream_t s) {
  return all_slices(a, true) ? launch_kind<Tr, SBS, NS, false, 1>(a, sh_q, sh_kv, s) : launch_kind<Tr, SBS, NS, true, 1>(a, sh_q, sh_kv, s);
}

template <typename Tr>
int dispatch(const bsa_attn_args &a, const bsa_attn_shares *sh_q, const bsa_attn_shares *sh_kv, hipStream_t s) {
  const int64_t slices = a.nh > a.nhv ? a.nh : a.nhv;
  if constexpr (Tr::kElem == 4) {
    if (a.sbs == 64) return slices == 1 ? launch_kind<Tr, 32, 2, false, 2>(a, sh_q, sh_kv, s) : launch_kind<Tr, 32, 4, false, 2>(a, sh_q, sh_kv, s);
  }
  if (a.sbs == 32) {
    switch (slices) {
      case 1: return launch<Tr, 32, 1>(a, sh_q, sh_kv, s);
      case 2: return launch<Tr, 32, 2>(a, sh_q, sh_kv, s);
      case 3: return launch<Tr, 32, 3>(a, sh_q, sh_kv, s);
      case 4: return launch<Tr, 32, 4>(a, sh_q, sh_kv, s);
    }
    return 1;
  }
  switch (slices) {
    case 1: return launch<Tr, 16, 1>(a, sh_q, sh_kv, s);
    case 2: return launch<Tr, 16, 2>(a, sh_q, sh_kv, s);
    case 3: return launch<Tr, 16, 3>(a, sh_q, sh_kv, s);
    case 4: return launch<Tr, 16, 4>(a, sh_q, sh_kv, s);
    case 5: return launch<Tr, 16, 5>(a, sh_q, sh_kv, s);
    case 6: return launch<Tr, 16, 6>(a, sh_q, sh_kv, s);
    case 7: return launch<Tr, 16, 7>(a, sh_q, sh_kv, s);
    case 8: return launch<Tr, 16, 8>(a, sh_q, sh_kv, s);
  }
  return 1;
}

}  // namespace

// 1: not covered
int attn_bwd_small(const bsa_attn_args &a, const bsa_attn_shares *sh_q, const bsa_attn_shares *sh_kv, hipStream_t s) {
  if (!small_applies(a, true)) return 1;
  return a.dtype == BSA_BF16 ? dispatch<SBf16>(a, sh_q, sh_kv, s) : a.dtype == BSA_F16 ? dispatch<SF16>(a, sh_q, sh_kv, s) : dispatch<SF32>(a, sh_q, sh_kv, s);
}

}  // namespace bsa
