// Block-sparse flash attention forward for blocks of 16 and 32 and head dimensions up to 128, fp16, bf16 and fp32, on the
// matrix cores of the operand type, or bf16's for fp32 blocks of 32 (in_parts).
//
// A wave owns one query block (or a share of its key list, below) and walks the list alone: no barrier, no tile
// shared between waves, so waves of a compute unit drift apart and fill each other's waits.  A step takes one key
// block of 32 or two of 16.  The products are formed transposed (S^T = K Q^T, O^T = V^T P^T): a lane owns one
// query row, the statistics of the softmax are in-lane reductions plus one or two lane swaps, and the probabilities
// are, as they sit in the accumulators of the score product, the second operand of the value product.
//
// Data: Q stays in registers.  K and V of a step lie in one LDS tile each (private to the wave), copied
// asynchronously: K of the next step is requested as soon as the scores of this one are formed, V of the next step
// when this one's value product is done, so each copy has the other half of a step (and the steps of the other waves
// of the SIMD) to arrive.  A single tile of each kind per wave, instead of two, is what lets 8 to 16 waves share a
// compute unit's LDS.  The list's entries and the packed indices they lead to are read 64 at a time, one per lane, and
// handed out with v_readlane.  Entries the causal predicate rules out as a whole are taken out of the list there.
//
// What bounds it: a wave's chain per step (copies awaited, scores, softmax, value product) and the instructions of one
// wave at a time.  Against the fp32 matrix-core kernel that ran these shapes before: 48 x 4096 queries, sbs 32, head
// dimension 64, fp16, 33 key blocks per query block: 0.65 -> 0.072 ms (460 TFLOP/s, 18 % of the matrix cores' peak); 32
// prompts of 1032 to 2064 tokens, sbs 16, bf16, causal: 0.54 -> 0.044 ms.  fp32, sbs 32, products from bf16 parts (split_f32.h):
// 8 x 2048 queries, half of the blocks, head dimension 64: 51.1 -> 41.0 us (105 TFLOP/s) against the fp32 instruction; the 490
// vector instructions of a step that split its values cost more than its 48 products, and 512 lists of 32 +- 4 blocks cut in
// four fill the chip once, so the launch waits for the longest.  fp32 blocks of 64, whose halves walk alone like blocks of 32:
// 20 x 960, causal, head dimension 64: 97.8 (eight waves to a tile) -> 27.4 us.
//
// Score pipeline (log2 domain), in the reference's order (blksprs/ops/flash_attention.py:1058-1224): scale * q k^T,
// + bias, native causal predicate, explicit mask; probabilities are rounded to the operand type before they multiply
// V, the row sum uses the unrounded values; a row that sees nothing gives zeros and lse = -inf.
#include <type_traits>

#include "attn_small_common.h"

namespace bsa {
namespace {

using namespace small;

constexpr int kWaves = 4;

template <int ES, int SBS, int NS, int kHalves>
struct FwdShape {
  // Key blocks per step.  Two blocks of 32 leave registers for three waves per SIMD instead of four (97 against 84 us,
  // 6144 rows of 33 blocks, head dimension 64); four blocks of 16 take twice the LDS, which leaves half the waves (76
  // against 60 us, 4128 rows, causal, head dimension 64).
  static constexpr int NB = SBS == 32 ? 1 : 2;
  using T = Tile<ES, SBS, NS, NB, kHalves>;
  static constexpr int kScores = SBS == 32 ? 16 * NB : 4 * NB;  // per lane and step
  static constexpr int kRegs = SBS == 32 ? 16 : 4;              // accumulator registers per block
  // K tile, V tile; at the end the partial output of a wave that shares a query block with others
  static constexpr int kPartial = SBS * SBS * NS * 4;
  static constexpr int kSlot = SBS * SBS * NS + 2 * SBS;  // floats of a slot of the scratch: O, then (m, l) of every query
  static constexpr int kLds = (2 * T::kBytes > kPartial ? 2 * T::kBytes : kPartial) + 512;
  static constexpr int kMinWaves = ES == 4 ? (NS * SBS <= 64 ? 2 : 1) : SBS == 32 ? (NS <= 2 ? 4 : 2) : (NS <= 4 ? 4 : 3);
};

// (m_i, l_i, oacc) of a row and those of another part of its list, scaled to the common maximum and added up
template <int NS, int kRegs, typename Acc>
__device__ inline void merge_partial(Acc (&oacc)[NS], float &m_i, float &l_i, const float *other, float m_o, float l_o, int lane) {
  const float m_new = fmaxf(m_i, m_o);
  const bool nothing = m_new == -INFINITY;
  const float s_i = nothing ? 1.f : __builtin_amdgcn_exp2f(m_i - m_new);
  const float s_o = nothing ? 1.f : __builtin_amdgcn_exp2f(m_o - m_new);
  l_i = l_i * s_i + l_o * s_o;
  m_i = m_new;
#pragma unroll
  for (int h = 0; h < NS; ++h)
#pragma unroll
    for (int r = 0; r < kRegs; r += 4) {
      const f32x4 o4 = *reinterpret_cast<const f32x4 *>(other + ((h * kRegs + r) / 4 * 64 + lane) * 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) oacc[h][r + i] = oacc[h][r + i] * s_i + o4[i] * s_o;
    }
}

// NS slices of the output, from slice `first` on, and lse of query block `own`, which belongs to `row` of the layout
template <typename Tr, int SBS, int NS, int kHalves, typename Acc>
__device__ inline void store_output(const Acc (&oacc)[NS], float m_i, float l_i, int64_t row, int own, int first, int qi, int kq) {
  constexpr int kRegs = SBS == 32 ? 16 : 4;
  const late_args_t p = late_args();
  const int nhv = (int)p->nhv;
  const float inv_l = (l_i != 0.f) ? 1.f / l_i : 0.f;
#pragma unroll
  for (int h = 0; h < NS; ++h) {
    const int slice = first + h;
    if (slice / kHalves >= nhv) break;
    const int64_t po = p->pidx_o[row * nhv + slice / kHalves];
    if (po < 0 || po >= p->n_o_blocks) continue;
    char *out = static_cast<char *>(p->o) + Place<Tr::kElem, SBS, kHalves>::row(po, own, qi, slice);
#pragma unroll
    for (int r = 0; r < kRegs; r += 4)  // columns 2 r + 4 kq .. + 3 of a row per lane
      store4<Tr>(out + (2 * r + 4 * kq) * Tr::kElem, oacc[h][r] * inv_l, oacc[h][r + 1] * inv_l, oacc[h][r + 2] * inv_l,
                 oacc[h][r + 3] * inv_l);
  }
  if (kq == 0 && first == 0) p->lse[(row * kHalves + own % kHalves) * SBS + qi] = (l_i != 0.f) ? m_i + log2f(l_i) : -INFINITY;
}

// split: 1, 2 or 4 waves share one query block, each walking every split-th entry of its key list, unless `shares` says how
// many do, of how many workgroups
// kHalves 2: blocks of 64, whose halves are the blocks of 32 spoken of here (Place)
template <typename Tr, int SBS, int NS, bool kSome, int kHalves>
__global__ __launch_bounds__(64 * kWaves, (FwdShape<Tr::kElem, SBS, NS, kHalves>::kMinWaves)) void attn_small_fwd_kernel(bsa_attn_args a, int split, Shares shares) {
  using Shape = FwdShape<Tr::kElem, SBS, NS, kHalves>;
  using T = typename Shape::T;
  using W = Walk<Tr::kElem, SBS, NS, Shape::NB, true, kSome, kHalves>;
  constexpr int NB = Shape::NB, kScores = Shape::kScores, kRegs = Shape::kRegs;
  using acc_t = std::conditional_t<SBS == 32, f32x16, f32x4>;
  extern __shared__ __attribute__((aligned(1024))) char small_smem[];
  const int lane = threadIdx.x & 63;
  const int wave = first_lane(threadIdx.x >> 6);
  char *lds_k = small_smem + wave * Shape::kLds, *lds_v = lds_k + T::kBytes;

  const RowOfWave me(shares, kHalves, a.B, kHalves * a.nq, true, wave, kWaves, split);
  const int64_t row = me.b * a.nq + me.own / kHalves;  // of the layout
  const int qi = lane % SBS, kq = lane / SBS;  // query row; which keys of a block this lane's registers hold
  W walk;
  walk.start(a, me.b, me.own, me.there, me.part, me.parts);

  OwnRows<Tr::kElem, SBS, NS, kHalves> qf;
  acc_t oacc[NS];
  float m_i, l_i;
  auto start_row = [&](int lane) __attribute__((always_inline)) {
    qf.load(a.q, a.pidx_q + row * a.nh, (int)a.nh, a.n_q_blocks, (int)me.own, lane);
#pragma unroll
    for (int h = 0; h < NS; ++h)
#pragma unroll
      for (int r = 0; r < kRegs; ++r) oacc[h][r] = 0.f;
    m_i = -INFINITY, l_i = 0.f;
  };
  start_row(lane);

  const float qk_scale = a.scale * kLog2e;
  const float cc = a.bias ? 1.f : qk_scale;
  const uint32_t source = T::source_offset(lane);
  const char *const tensor_k = static_cast<const char *>(a.k), *const tensor_v = static_cast<const char *>(a.v);

  const typename T::RowReader k_rows(lds_k, lane);
  const typename T::ColReader v_cols(lds_v, lane);
  // whether the sums are what they should be (from parts they may not be)
  auto walk_list = [&](auto arithmetic) __attribute__((always_inline)) -> bool {
    using Ar = decltype(arithmetic);
    typename W::Step now, next;
    walk.take(now, lane);
    settle(qf);
    if constexpr (std::is_same_v<Ar, SSplit>) {
      if (scores_in_doubt(qf, a.scale)) return false;
    }
    const OwnOperand<Ar, SBS, NS, kHalves, false> q_operand(qf);
    bool counted = false;  // exactly kCopies copies (the V tile's) were issued after the K tile's
    if (now.count) {
      walk.template copy<false>(now, tensor_k, lds_k, source, lane);
      counted = walk.template copy<true>(now, tensor_v, lds_v, source, lane);
    }
    while (now.count) {
      // ---- S^T = K Q^T.  In flight at most: K and V of this step, in that order.
      if (counted) wait_vmem<T::kCopies>();
      else wait_vmem<0>();
      acc_t sacc[NB];
      W::template multiply_rows<Ar, false>(sacc, now, k_rows, q_operand, lane);

      // ---- K of the next step
      wait_lds();
      walk.take(next, lane);
      counted = false;
      if (next.count) counted = walk.template copy<false>(next, tensor_k, lds_k, source, lane);

      // ---- scores: sv holds them up to the positive factor cc, applied inside the exponential (16-bit)
      float sv[kScores];
#pragma unroll
      for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int r = 0; r < kRegs; ++r) sv[kRegs * t + r] = sacc[t][r];
      if (now.special) walk.template finish_scores<Tr>(now, sv, qk_scale, qi, kq);
      apply_factor<Tr, kScores>(sv, cc);

      // ---- online softmax of the row.  The reference is the exact running maximum: the largest probabilities then lie at
      // and just below 1, where rounding to 16 bits costs least.  A maximum that follows in steps of up to 2^8 (as in
      // attn_mfma.hip) saves most of the rescaling and lets them fall anywhere between two powers of two: errors of the output
      // against 64 bits of 2.27e-3 instead of 2.09e-3 (bf16, 1024 keys, half of the blocks).
      float m_blk = sv[0];
#pragma unroll
      for (int x = 1; x < kScores; ++x) m_blk = fmaxf(m_blk, sv[x]);
      m_blk = row_max<SBS>(m_blk) * late_factor<Tr>(cc);
      const float m_cand = fmaxf(m_i, m_blk);
      if (__any(m_cand > m_i)) {
        const float alpha = m_cand > m_i ? __builtin_amdgcn_exp2f(m_i - m_cand) : 1.f;
        m_i = m_cand;
        l_i *= alpha;
#pragma unroll
        for (int h = 0; h < NS; ++h)
#pragma unroll
          for (int r = 0; r < kRegs; ++r) oacc[h][r] *= alpha;
      }
      const float m_sub = (m_i == -INFINITY) ? 0.f : m_i;
      float sum = 0.f;
#pragma unroll
      for (int x = 0; x < kScores; ++x) {
        sv[x] = __builtin_amdgcn_exp2f(fmaf(sv[x], late_factor<Tr>(cc), -m_sub));
        sum += sv[x];
      }
      l_i += sum;
      if constexpr (up_of<Ar>() != 1.f) {
#pragma unroll
        for (int x = 0; x < kScores; ++x) sv[x] *= up_of<Ar>();
      }
      const Weights<Ar, kScores> pf(sv);

      // ---- O^T += V^T P^T.  In flight at most: V of this step, K of the next.
      if (counted) wait_vmem<T::kCopies>();
      else wait_vmem<0>();
      W::template multiply_cols<Ar, true, kScores>(oacc, now, v_cols, pf);
      wait_lds();
      counted = false;
      if (next.count) counted = walk.template copy<true>(next, tensor_v, lds_v, source, lane);
      now = next;
    }
    if constexpr (!std::is_same_v<Ar, SSplit>) return true;
    scale_down<Ar, NS, kRegs>(oacc);
    return !not_finite<NS, kRegs>(oacc, l_i);
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

  // ---- epilogue
  l_i = row_sum<SBS>(l_i);
  if (me.waves > 1) {
    // every wave leaves (m, l, O) of its part; the first wave of a query block scales them to the common maximum and
    // adds them up, in order
    float *mine = reinterpret_cast<float *>(lds_k);
    constexpr int kStats = Shape::kLds / 4 - 128;
    if (me.place != 0) {
      leave_partial<NS, kRegs>(oacc, mine, lane);
      if (kq == 0) mine[kStats + 2 * qi] = m_i, mine[kStats + 2 * qi + 1] = l_i;
    }
    __syncthreads();
    if (me.place != 0) return;
    for (int p = 1; p < me.waves; ++p) {
      const float *other = mine + p * (Shape::kLds / 4);
      merge_partial<NS, kRegs>(oacc, m_i, l_i, other, other[kStats + 2 * qi], other[kStats + 2 * qi + 1], lane);
    }
  }
  if (!me.there) return;
  if (me.slot >= 0) {  // other workgroups have the rest of the row: attn_small_fwd_merge_kernel adds them up
    float *out = shares.partials + (int64_t)me.slot * Shape::kSlot;
    leave_partial<NS, kRegs>(oacc, out, lane);
    if (kq == 0) out[Shape::kSlot - 2 * SBS + 2 * qi] = m_i, out[Shape::kSlot - 2 * SBS + 2 * qi + 1] = l_i;
    return;
  }
  store_output<Tr, SBS, NS, kHalves>(oacc, m_i, l_i, row, (int)me.own, 0, qi, kq);
}

// The sums of query blocks that several workgroups share, a wave for each head slice (blockIdx.y): merges[m] is (batch entry,
// query block of the layout, first slot, slots).  All slots' sums are read independently of one another: with one wave per
// query block that scaled slot by slot, 8 blocks of 128 entries at head dimension 128 took 29 us, now 4.5.
template <typename Tr, int SBS, int NS, int kHalves>
__global__ __launch_bounds__(64) void attn_small_fwd_merge_kernel(bsa_attn_args a, const int32_t *merges, const float *partials) {
  using Shape = FwdShape<Tr::kElem, SBS, NS, kHalves>;
  constexpr int kRegs = Shape::kRegs;
  constexpr int64_t kStep = kHalves * Shape::kSlot;
  using acc_t = std::conditional_t<SBS == 32, f32x16, f32x4>;
  const int lane = threadIdx.x, qi = lane % SBS, kq = lane / SBS, half = blockIdx.x % kHalves, h = blockIdx.y;
  const int32_t *merge = merges + (int64_t)(blockIdx.x / kHalves) * 4;
  const int64_t row = (int64_t)merge[0] * a.nq + merge[1];
  const float *part = partials + ((int64_t)merge[2] * kHalves + half) * Shape::kSlot;
  const float *stats = part + (Shape::kSlot - 2 * SBS) + 2 * qi;
  const int n = merge[3];
  float m_i = -INFINITY, l_i = 0.f;
#pragma unroll 4
  for (int s = 0; s < n; ++s) m_i = fmaxf(m_i, stats[s * kStep]);
  const float m_sub = m_i == -INFINITY ? 0.f : m_i;
  acc_t oacc[1];
#pragma unroll
  for (int r = 0; r < kRegs; ++r) oacc[0][r] = 0.f;
  part += h * kRegs * 64;
#pragma unroll 4
  for (int s = 0; s < n; ++s) {
    const float scale = __builtin_amdgcn_exp2f(stats[s * kStep] - m_sub);
    l_i = fmaf(stats[s * kStep + 1], scale, l_i);
#pragma unroll
    for (int r = 0; r < kRegs; r += 4) {
      const f32x4 o4 = *reinterpret_cast<const f32x4 *>(part + s * kStep + (r / 4 * 64 + lane) * 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) oacc[0][r + i] = fmaf(o4[i], scale, oacc[0][r + i]);
    }
  }
  store_output<Tr, SBS, 1, kHalves>(oacc, m_i, l_i, row, merge[1] * kHalves + half, h, qi, kq);
}

template <typename Tr, int SBS, int NS, bool kSome, int kHalves>
int launch_kind(const bsa_attn_args &a, const bsa_attn_shares *sh, hipStream_t s) {
  using Shape = FwdShape<Tr::kElem, SBS, NS, kHalves>;
  const int64_t rows = kHalves * a.nq;  // of a batch entry
  const int split = waves_per_row<Tr::kElem>(a.B * rows, kHalves * a.nk, Shape::NB);
  const int64_t groups = sh ? kHalves * sh->n_groups : row_groups(a.B, rows, kWaves, split);
  if (!fits_launch(groups, kWaves)) return 1;
  constexpr int lds = Shape::kLds * kWaves;
  static_assert(lds <= 160 * 1024, "LDS");
  static LdsLimit limit;
  if (int rc = allow_lds(limit, &attn_small_fwd_kernel<Tr, SBS, NS, kSome, kHalves>, lds)) return rc;
  Shares shares{nullptr, nullptr};
  if (sh) {
    const int64_t need = sh->n_slots * kHalves * Shape::kSlot * 4;
    BSA_REQUIRE(need <= sh->scratch_bytes, "bsa_attn_fwd_shares: scratch holds %lld bytes, %lld are needed",
                (long long)sh->scratch_bytes, (long long)need);
    shares = Shares{sh->groups, static_cast<float *>(sh->scratch)};
  }
  attn_small_fwd_kernel<Tr, SBS, NS, kSome, kHalves><<<(unsigned)groups, 64 * kWaves, lds, s>>>(a, split, shares);
  if (int rc = check_launch("attn_small_fwd_kernel")) return rc;
  if (!sh || sh->n_merges == 0) return BSA_OK;
  attn_small_fwd_merge_kernel<Tr, SBS, NS, kHalves><<<dim3((unsigned)(sh->n_merges * kHalves), NS), 64, 0, s>>>(a, sh->merges, shares.partials);
  return check_launch("attn_small_fwd_merge_kernel");
}

template <typename Tr, int SBS, int NS>
int launch(const bsa_attn_args &a, const bsa_attn_shares *sh, hipStream_t s) {
  return all_slices(a, false) ? launch_kind<Tr, SBS, NS, false, 1>(a, sh, s) : launch_kind<Tr, SBS, NS, true, 1>(a, sh, s);
}

template <typename Tr>
int dispatch(const bsa_attn_args &a, const bsa_attn_shares *sh, hipStream_t s) {
  const int64_t slices = a.nh > a.nhv ? a.nh : a.nhv;
  if constexpr (Tr::kElem == 4) {
    if (a.sbs == 64) return slices == 1 ? launch_kind<Tr, 32, 2, false, 2>(a, sh, s) : launch_kind<Tr, 32, 4, false, 2>(a, sh, s);
  }
  if (a.sbs == 32) {
    switch (slices) {
      case 1: return launch<Tr, 32, 1>(a, sh, s);
      case 2: return launch<Tr, 32, 2>(a, sh, s);
      case 3: return launch<Tr, 32, 3>(a, sh, s);
      case 4: return launch<Tr, 32, 4>(a, sh, s);
    }
    return 1;
  }
  switch (slices) {
    case 1: return launch<Tr, 16, 1>(a, sh, s);
    case 2: return launch<Tr, 16, 2>(a, sh, s);
    case 3: return launch<Tr, 16, 3>(a, sh, s);
    case 4: return launch<Tr, 16, 4>(a, sh, s);
    case 5: return launch<Tr, 16, 5>(a, sh, s);
    case 6: return launch<Tr, 16, 6>(a, sh, s);
    case 7: return launch<Tr, 16, 7>(a, sh, s);
    case 8: return launch<Tr, 16, 8>(a, sh, s);
  }
  return 1;
}

}  // namespace

// 1: not covered
int attn_fwd_small(const bsa_attn_args &a, const bsa_attn_shares *sh, hipStream_t s) {
  if (!small_applies(a, false)) return 1;
  if (a.B * a.nq == 0) return BSA_OK;
  return a.dtype == BSA_BF16 ? dispatch<SBf16>(a, sh, s) : a.dtype == BSA_F16 ? dispatch<SF16>(a, sh, s) : dispatch<SF32>(a, sh, s);
}

}  // namespace bsa
