// Block-sparse flash attention forward for 16-bit operands in blocks of 16 and 32, on the 16-bit matrix cores.
//
// A wave owns one query block (or a share of its key list, below) and walks the list alone: no barrier, no tile
// shared between waves, so waves of a compute unit drift apart and fill each other's waits.  A step takes one key
// block of 32 or up to four of 16.  The products are formed transposed (S^T = K Q^T, O^T = V^T P^T): a lane owns one
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
// wave at a time; matrix cores 16 % busy, 113 vector and 63 scalar instructions per step of 32 x 32 at head dimension 64.
// Against the fp32 matrix-core kernel that ran these shapes before: 48 x 4096 queries, sbs 32, head dimension 64, fp16,
// 33 key blocks per query block: 0.65 -> 0.075 ms (443 TFLOP/s); 32 prompts of 1032 to 2064 tokens, sbs 16, bf16, causal:
// 0.54 -> 0.076 ms.
//
// Score pipeline (log2 domain), in the reference's order (blksprs/ops/flash_attention.py:1058-1224): scale * q k^T,
// + bias, native causal predicate, explicit mask; probabilities are rounded to the operand type before they multiply
// V, the row sum uses the unrounded values; a row that sees nothing gives zeros and lse = -inf.
#include <type_traits>

#include "attn_small_common.h"

namespace bsa {
namespace {

using namespace small;

constexpr float kRescaleStep = 8.f;  // log2 units, see attn_mfma.hip
constexpr int kWaves = 4;

template <int SBS, int NS>
struct FwdShape {
  // Key blocks per step.  Two blocks of 32 leave registers for three waves per SIMD instead of four (97 against 84 us,
  // 6144 rows of 33 blocks, head dimension 64); two blocks of 16 instead of four make no difference.
  static constexpr int NB = SBS == 32 ? 1 : (NS <= 4 ? 4 : 2);
  using T = Tile<SBS, NS, NB>;
  static constexpr int kScores = SBS == 32 ? 16 * NB : 4 * NB;  // per lane and step
  static constexpr int kRegs = SBS == 32 ? 16 : 4;              // accumulator registers per block
  // K tile, V tile; at the end the partial output of a wave that shares a query block with others
  static constexpr int kPartial = SBS * SBS * NS * 4;
  static constexpr int kLds = (2 * T::kBytes > kPartial ? 2 * T::kBytes : kPartial) + 512;
  static constexpr int kMinWaves = SBS == 32 ? (NS <= 2 ? 4 : 2) : (NS <= 2 ? 4 : 2);
};

// split: 1, 2 or 4 waves share one query block, each walking a contiguous part of its key list
template <typename Tr, int SBS, int NS>
__global__ __launch_bounds__(64 * kWaves, (FwdShape<SBS, NS>::kMinWaves)) void attn_small_fwd_kernel(bsa_attn_args a, int split) {
  using Shape = FwdShape<SBS, NS>;
  using T = typename Shape::T;
  constexpr int NB = Shape::NB, kScores = Shape::kScores, kRegs = Shape::kRegs, kPiece = T::kPiece;
  using acc_t = std::conditional_t<SBS == 32, f32x16, f32x4>;
  extern __shared__ __attribute__((aligned(1024))) char small_smem[];
  const int lane = threadIdx.x & 63;
  const int wave = first_lane(threadIdx.x >> 6);
  char *lds_k = small_smem + wave * Shape::kLds, *lds_v = lds_k + T::kBytes;

  // XCD c (workgroup g runs on XCD g % 8) takes a contiguous eighth of the query blocks, so that the waves in flight
  // on one L2 share few batch entries' K and V; inside a batch entry the last query blocks, which are the long ones
  // under a causal layout, come first.
  const int per_group = kWaves / split;
  const int64_t group = (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int64_t item = group * per_group + wave / split;
  const int part = wave % split;
  const bool has_row = item < a.B * a.nq;
  const int64_t b = has_row ? item / a.nq : 0, qb = has_row ? a.nq - 1 - item % a.nq : 0;
  const int64_t row = b * a.nq + qb;
  const int qi = lane % SBS, kq = lane / SBS;  // query row; which keys of a block this lane's registers hold

  OwnRows<SBS, NS> qf;
  qf.load(a.q, a.pidx_q + row * a.nh, (int)a.nh, a.n_q_blocks, lane);
  acc_t oacc[NS];
#pragma unroll
  for (int h = 0; h < NS; ++h)
#pragma unroll
    for (int r = 0; r < kRegs; ++r) oacc[h][r] = 0.f;
  float m_i = -INFINITY, l_i = 0.f;

  const float qk_scale = a.scale * kLog2e;
  const float cc = a.bias ? 1.f : qk_scale;
  int seq_len = 0x7fffffff;
  if (a.causal_lengths) {
    const int64_t len = a.causal_lengths[b];
    seq_len = len < 0 ? 0 : (len > 0x7fffffffLL ? 0x7fffffff : (int)len);
  }
  int e_begin = first_lane(a.key_offsets[row]), e_end = first_lane(a.key_offsets[row + 1]);
  if (split > 1) {
    const int n = e_end - e_begin;
    e_end = e_begin + (int)((int64_t)n * (part + 1) / split);
    e_begin = e_begin + (int)((int64_t)n * part / split);
  }
  if (!has_row || (int)qb * SBS >= seq_len) e_end = e_begin;

  // ---- The list, 64 entries at a time, one per lane: key block, packed index of the first K and V slice, mask and bias
  // block.  Entries the causal predicate rules out are not in w_live; w_special marks those whose scores need more
  // than the scale.  w_apart: some block's slices are missing or not one behind the other.
  int w_base = e_begin - 64, w_kb = 0, w_pk = 0, w_pv = 0, w_pm = -1, w_pb = -1;
  uint64_t w_live = 0, w_special = 0;
  bool w_apart = false;
  auto refill = [&]() {
    const late_args_t p = late_args();
    w_base += 64;
    const int e = w_base + lane;
    bool in = e < e_end;
    w_kb = in ? p->key_indices[e] : 0;
    const bool causal = p->causal_lengths != nullptr;
    in = in && !(causal && (w_kb > (int)qb || w_kb * SBS >= seq_len));
    const int64_t kv = b * p->nk + w_kb;
    const int nh = (int)p->nh, nhv = (int)p->nhv;
    bool apart = nh != NS || nhv != NS;
    if (in && !apart) {
      const int64_t *pk = p->pidx_k + kv * NS, *pv = p->pidx_v + kv * NS;
      const int64_t k0 = pk[0], v0 = pv[0];
      apart = k0 < 0 || v0 < 0 || k0 + NS > p->n_k_blocks || v0 + NS > p->n_v_blocks;
#pragma unroll
      for (int h = 1; h < NS; ++h) apart = apart || pk[h] != k0 + h || pv[h] != v0 + h;
      w_pk = (int)k0;
      w_pv = (int)v0;
    }
    w_apart = __any(in && apart);
    bool special = causal && (w_kb == (int)qb || ((int)qb + 1) * SBS > seq_len || (w_kb + 1) * SBS > seq_len);
    if (p->mask) {
      const int64_t pm = in ? p->pidx_mask[row * p->nk + w_kb] : -1;
      w_pm = pm < p->n_mask_blocks ? (int)pm : -1;
      special = special || w_pm >= 0;
    }
    if (p->bias) {
      const int64_t pb = in ? p->pidx_bias[row * p->nk + w_kb] : -1;
      w_pb = pb < p->n_bias_blocks ? (int)pb : -1;
      special = true;
    }
    w_live = __ballot(in);
    w_special = __ballot(in && special);
  };
  // a step: how many entries it takes, their places in the window and whether their slices lie apart, and, if special,
  // their facts (the window may be another one by the time the scores are formed)
  struct Step {
    int count, slot[NB], kb[NB], pm[NB], pb[NB];
    bool special, apart;
  };
  auto take = [&](Step &s) {
    while (w_live == 0 && w_base + 64 < e_end) refill();
    s.count = 0;
    uint64_t taken = 0;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const uint64_t lowest = w_live & -w_live;
      s.slot[t] = lowest ? __builtin_ctzll(lowest) : 0;
      s.count += lowest ? 1 : 0;
      w_live ^= lowest;
      taken |= lowest;
    }
    s.apart = w_apart;
    s.special = (taken & w_special) != 0 || (NB > 1 && s.count < NB);
    if (s.special) {
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        s.kb[t] = __builtin_amdgcn_readlane(w_kb, s.slot[t]);
        s.pm[t] = t < s.count ? __builtin_amdgcn_readlane(w_pm, s.slot[t]) : -1;
        s.pb[t] = t < s.count ? __builtin_amdgcn_readlane(w_pb, s.slot[t]) : -1;
      }
    }
  };
  const uint32_t source = T::source_offset(lane);
  const char *const tensor_k = static_cast<const char *>(a.k), *const tensor_v = static_cast<const char *>(a.v);
  // requests the step's K (V) blocks; returns whether exactly kCopies asynchronous copies are on their way
  auto copy = [&](const Step &s, bool is_k) {
    const char *tensor = is_k ? tensor_k : tensor_v;
    char *dst = is_k ? lds_k : lds_v;
    if (!s.apart) {
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        // a block that is not there: the copy of the one in front of it once more, its scores become -inf and its V zeros
        if (NB == 1 || t < s.count)
          T::copy_block(tensor, __builtin_amdgcn_readlane(is_k ? w_pk : w_pv, s.slot[t]), dst + t * T::kBlock, source, lane);
      }
      if (NB == 1 || s.count == NB) return true;
    }
    const late_args_t p = late_args();
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      if (!s.apart && t < s.count) continue;
      const int n = t < s.count ? (int)(is_k ? p->nh : p->nhv) : 0;
      const int64_t kv = b * p->nk + __builtin_amdgcn_readlane(w_kb, s.slot[t]);
      T::gather_block(tensor, (is_k ? p->pidx_k : p->pidx_v) + kv * n, n, is_k ? p->n_k_blocks : p->n_v_blocks,
                      dst + t * T::kBlock, source, lane);
    }
    return false;
  };

  const typename T::RowReader k_rows(lds_k, lane);
  const typename T::ColReader v_cols(lds_v, lane);
  Step now, next;
  take(now);
  settle(qf);
  bool counted = false;  // exactly kCopies copies (the V tile's) were issued after the K tile's
  if (now.count) {
    copy(now, true);
    counted = copy(now, false);
  }
  while (now.count) {
    // ---- S^T = K Q^T.  In flight at most: K and V of this step, in that order.
    if (counted) wait_vmem<T::kCopies>();
    else wait_vmem<0>();
    acc_t sacc[NB];
    product_rows<Tr, SBS, NS, NB>(sacc, k_rows, qf);

    // ---- K of the next step
    wait_lds();
    take(next);
    counted = false;
    if (next.count) counted = copy(next, true);

    // ---- scores: sv holds them up to the positive factor cc, applied inside the exponential
    float sv[kScores];
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
      for (int r = 0; r < kRegs; ++r) sv[kRegs * t + r] = sacc[t][r];
    if (now.special) {
      const late_args_t p = late_args();
      const int qpos = (int)qb * SBS + qi;
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        float *s = sv + kRegs * t;
        if (p->bias) {  // finished scores; the factor inside the exponential is 1 then
          u32x2 bw[kRegs / 4];
#pragma unroll
          for (int w = 0; w < kRegs / 4; ++w) {
            bw[w] = u32x2{0u, 0u};
            if (now.pb[t] >= 0)
              bw[w] = *reinterpret_cast<const u32x2 *>(static_cast<const char *>(p->bias) + (int64_t)now.pb[t] * kPiece +
                                                       qi * (2 * SBS) + 16 * w + 8 * kq);
          }
#pragma unroll
          for (int r = 0; r < kRegs; ++r)
            s[r] = s[r] * qk_scale + Tr::widen((uint16_t)(bw[r / 4][(r % 4) / 2] >> (16 * (r % 2)))) * kLog2e;
        }
        if (now.pm[t] >= 0) {
          const char *words = static_cast<const char *>(p->mask) + (int64_t)now.pm[t] * (SBS * SBS) + qi * SBS + 4 * kq;
          uint32_t mw[kRegs / 4];
#pragma unroll
          for (int w = 0; w < kRegs / 4; ++w) mw[w] = *reinterpret_cast<const uint32_t *>(words + 8 * w);
#pragma unroll
          for (int r = 0; r < kRegs; ++r)
            if ((mw[r / 4] >> (8 * (r % 4))) & 0xffu) s[r] = -INFINITY;
        }
        if (p->causal_lengths) {
#pragma unroll
          for (int r = 0; r < kRegs; ++r) {
            const int kpos = now.kb[t] * SBS + 8 * (r / 4) + 4 * kq + r % 4;
            if (kpos > qpos || qpos >= seq_len || kpos >= seq_len) s[r] = -INFINITY;
          }
        }
        if (t >= now.count) {
#pragma unroll
          for (int r = 0; r < kRegs; ++r) s[r] = -INFINITY;
        }
      }
    }

    // ---- online softmax of the row, the reference maximum following lazily (attn_mfma.hip)
    float m_blk = sv[0];
#pragma unroll
    for (int x = 1; x < kScores; ++x) m_blk = fmaxf(m_blk, sv[x]);
    m_blk = row_max<SBS>(m_blk) * cc;
    const float m_cand = fmaxf(m_i, m_blk);
    if (__any((m_cand - m_i) > kRescaleStep)) {
      const bool both_ninf = (m_i == -INFINITY) && (m_cand == -INFINITY);
      const float alpha = both_ninf ? 1.f : __builtin_amdgcn_exp2f(m_i - m_cand);
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
      sv[x] = __builtin_amdgcn_exp2f(fmaf(sv[x], cc, -m_sub));
      sum += sv[x];
    }
    l_i += sum;
    u32x4 pf[kScores / 8];
#pragma unroll
    for (int m = 0; m < kScores / 8; ++m)
#pragma unroll
      for (int w = 0; w < 4; ++w) pf[m][w] = Tr::pack2(sv[8 * m + 2 * w], sv[8 * m + 2 * w + 1]);

    // ---- O^T += V^T P^T.  In flight at most: V of this step, K of the next.
    if (counted) wait_vmem<T::kCopies>();
    else wait_vmem<0>();
    product_cols<Tr, SBS, NS, NB>(oacc, v_cols, pf);
    wait_lds();
    counted = false;
    if (next.count) counted = copy(next, false);
    now = next;
  }

  // ---- epilogue
  l_i = row_sum<SBS>(l_i);
  if (split > 1) {
    // every wave leaves (m, l, O) of its part; the first wave of a query block scales them to the common maximum and
    // adds them up, in order
    float *mine = reinterpret_cast<float *>(lds_k);
    if (part != 0) {
#pragma unroll
      for (int h = 0; h < NS; ++h)
#pragma unroll
        for (int r = 0; r < kRegs; r += 4)
          *reinterpret_cast<f32x4 *>(mine + ((h * kRegs + r) / 4 * 64 + lane) * 4) =
              f32x4{oacc[h][r], oacc[h][r + 1], oacc[h][r + 2], oacc[h][r + 3]};
      if (kq == 0) {
        mine[Shape::kLds / 4 - 128 + 2 * qi] = m_i;
        mine[Shape::kLds / 4 - 128 + 2 * qi + 1] = l_i;
      }
    }
    __syncthreads();
    if (part != 0) return;
    for (int p = 1; p < split; ++p) {
      const float *other = mine + p * (Shape::kLds / 4);
      const float m_o = other[Shape::kLds / 4 - 128 + 2 * qi], l_o = other[Shape::kLds / 4 - 128 + 2 * qi + 1];
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
  }
  if (!has_row) return;
  const late_args_t p = late_args();
  const int nhv = (int)p->nhv;
  const float inv_l = (l_i != 0.f) ? 1.f / l_i : 0.f;
#pragma unroll
  for (int h = 0; h < NS; ++h) {
    if (h >= nhv) break;
    const int64_t po = p->pidx_o[row * nhv + h];
    if (po < 0 || po >= p->n_o_blocks) continue;
    char *out = static_cast<char *>(p->o) + po * kPiece;
#pragma unroll
    for (int r = 0; r < kRegs; r += 4) {  // eight bytes of a row per lane: columns 2 r + 4 kq .. + 3
      u32x2 w;
      w[0] = Tr::pack2(oacc[h][r] * inv_l, oacc[h][r + 1] * inv_l);
      w[1] = Tr::pack2(oacc[h][r + 2] * inv_l, oacc[h][r + 3] * inv_l);
      *reinterpret_cast<u32x2 *>(out + qi * (2 * SBS) + 4 * r + 8 * kq) = w;
    }
  }
  if (kq == 0) p->lse[row * SBS + qi] = (l_i != 0.f) ? m_i + log2f(l_i) : -INFINITY;
}

template <typename Tr, int SBS, int NS>
int launch(const bsa_attn_args &a, hipStream_t s) {
  using Shape = FwdShape<SBS, NS>;
  const int64_t rows = a.B * a.nq;
  // A launch lasts as long as the serial walk of its longest lists, and the last round of a launch of few rounds is
  // mostly empty: shorter shares of a list help until their prologue (four dependent loads) costs more than the walk.
  // 64 rows (8 key blocks each, sbs 32): 9.6 us with two waves per row, 8.1 with four; 4128 rows (sbs 16, causal, up to
  // 33 steps): 79 / 76 / 94 us with one, two, four; 6144 rows (sbs 32, 33 steps): 83 / 75 / 82.
  const int split = rows <= 512 ? 4 : rows <= 8192 ? 2 : 1;
  const int64_t groups = cdiv(cdiv(rows, (int64_t)(kWaves / split)), (int64_t)8) * 8;
  constexpr int lds = Shape::kLds * kWaves;
  static_assert(lds <= 160 * 1024, "LDS");
  if (lds > 64 * 1024) {
    static const hipError_t raised = hipFuncSetAttribute(
        reinterpret_cast<const void *>(&attn_small_fwd_kernel<Tr, SBS, NS>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    BSA_HIP(raised);
  }
  attn_small_fwd_kernel<Tr, SBS, NS><<<(unsigned)groups, 64 * kWaves, lds, s>>>(a, split);
  return check_launch("attn_small_fwd_kernel");
}

template <typename Tr>
int dispatch(const bsa_attn_args &a, hipStream_t s) {
  const int64_t slices = a.nh > a.nhv ? a.nh : a.nhv;
  if (a.sbs == 32) {
    switch (slices) {
      case 1: return launch<Tr, 32, 1>(a, s);
      case 2: return launch<Tr, 32, 2>(a, s);
      case 3: return launch<Tr, 32, 3>(a, s);
      case 4: return launch<Tr, 32, 4>(a, s);
    }
    return 1;
  }
  switch (slices) {
    case 1: return launch<Tr, 16, 1>(a, s);
    case 2: return launch<Tr, 16, 2>(a, s);
    case 3: return launch<Tr, 16, 3>(a, s);
    case 4: return launch<Tr, 16, 4>(a, s);
    case 5: return launch<Tr, 16, 5>(a, s);
    case 6: return launch<Tr, 16, 6>(a, s);
    case 7: return launch<Tr, 16, 7>(a, s);
    case 8: return launch<Tr, 16, 8>(a, s);
  }
  return 1;
}

}  // namespace

// 1: not covered
int attn_fwd_small(const bsa_attn_args &a, hipStream_t s) {
  if (a.sbs != 16 && a.sbs != 32) return 1;
  if (a.dtype != BSA_BF16 && a.dtype != BSA_F16) return 1;
  // the row maximum is taken before the scale is applied
  if (!(a.scale > 0.f) || a.scale > 3.0e38f) return 1;
  if (a.n_k_blocks > 0x7fffffffLL || a.n_v_blocks > 0x7fffffffLL || a.n_mask_blocks > 0x7fffffffLL ||
      a.n_bias_blocks > 0x7fffffffLL)
    return 1;
  // positions are 32-bit numbers
  if (a.nq * a.sbs > 0x7fffffffLL || a.nk * a.sbs > 0x7fffffffLL) return 1;
  if (a.B * a.nq == 0) return BSA_OK;
  return a.dtype == BSA_BF16 ? dispatch<SBf16>(a, s) : dispatch<SF16>(a, s);
}

}  // namespace bsa
