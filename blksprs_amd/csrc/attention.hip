// C ABI of block-sparse flash attention: argument checks and the choice of kernels: 16-bit operands in 64 x 64 blocks
// with at most two head slices (attn_mfma.hip, attn_bwd_mfma.hip), blocks of 16 and 32 and fp32 blocks of 64 with head
// dimensions up to 128 (attn_small_fwd.hip, attn_small_bwd.hip), the rest on the fp32 matrix-core instruction
// (attn_f32mma.hip: fp32 blocks of 64 with missing slices, longer head dimensions, scales that are not positive, tensors that
// do not start on 16 bytes), and the generic
// kernels for more head slices than fit LDS.
#include "attn_common.h"

namespace {

int check_args(const char *who, const bsa_attn_args *a, bool backward) {
  BSA_REQUIRE(a != nullptr, "%s: NULL argument block", who);
  BSA_REQUIRE(a->sbs == 16 || a->sbs == 32 || a->sbs == 64, "%s: sbs must be 16, 32 or 64 (got %d)", who, a->sbs);
  BSA_REQUIRE(a->dtype == BSA_F32 || a->dtype == BSA_F16 || a->dtype == BSA_BF16, "%s: unknown dtype %d", who,
              a->dtype);
  BSA_REQUIRE(a->B >= 0 && a->nq >= 0 && a->nk >= 0 && a->nh >= 0 && a->nhv >= 0, "%s: negative layout size", who);
  BSA_REQUIRE(a->n_q_blocks >= 0 && a->n_k_blocks >= 0 && a->n_v_blocks >= 0 && a->n_o_blocks >= 0 &&
                  a->n_mask_blocks >= 0 && a->n_bias_blocks >= 0,
              "%s: negative block count", who);
  BSA_REQUIRE(a->mask_kind == 0 || a->mask_kind == 1, "%s: mask_kind must be 0 or 1", who);
  BSA_REQUIRE((a->mask != nullptr) == (a->mask_kind == 1), "%s: mask pointer and mask_kind disagree", who);
  if (a->B * a->nq == 0 && a->B * a->nk == 0) return BSA_OK;
  BSA_REQUIRE(a->key_offsets != nullptr, "%s: key_offsets is NULL", who);
  BSA_REQUIRE(a->lse != nullptr || a->B * a->nq == 0, "%s: lse is NULL", who);
  BSA_REQUIRE(a->nh == 0 || (a->pidx_q && a->pidx_k), "%s: pidx_q / pidx_k is NULL", who);
  BSA_REQUIRE(a->nhv == 0 || (a->pidx_v && a->pidx_o), "%s: pidx_v / pidx_o is NULL", who);
  BSA_REQUIRE(!a->mask || a->pidx_mask, "%s: mask without pidx_mask", who);
  BSA_REQUIRE(!a->bias || a->pidx_bias, "%s: bias without pidx_bias", who);
  BSA_REQUIRE(a->B * a->nq < 0x7fffffffLL && a->B * a->nk < 0x7fffffffLL, "%s: too many sequence blocks", who);
  BSA_REQUIRE(a->nh < 65536 && a->nhv < 65536, "%s: too many head slices", who);
  BSA_REQUIRE(a->group_size >= 0 && a->group_size <= 2, "%s: group_size must be 0, 1 or 2", who);
  BSA_REQUIRE(a->group_size == 0 || a->group_offsets, "%s: group_size without group_offsets", who);
  if (backward) {
    BSA_REQUIRE(a->query_offsets != nullptr, "%s: query_offsets is NULL", who);
    BSA_REQUIRE(a->delta != nullptr || a->B * a->nq == 0, "%s: delta is NULL", who);
    BSA_REQUIRE(a->n_o_blocks == 0 || (a->o && a->d_o), "%s: o / d_o is NULL", who);
    BSA_REQUIRE(a->n_q_blocks == 0 || a->dq, "%s: dq is NULL", who);
    BSA_REQUIRE(a->n_k_blocks == 0 || a->dk, "%s: dk is NULL", who);
    BSA_REQUIRE(a->n_v_blocks == 0 || a->dv, "%s: dv is NULL", who);
    BSA_REQUIRE(!a->dbias || a->bias, "%s: dbias without bias", who);
  } else {
    BSA_REQUIRE(a->n_o_blocks == 0 || a->o, "%s: o is NULL", who);
  }
  return BSA_OK;
}

int check_shares(const char *who, const bsa_attn_shares *s) {
  if (s == nullptr) return BSA_OK;
  BSA_REQUIRE(s->n_groups >= 0 && s->n_merges >= 0 && s->n_slots >= 0 && s->scratch_bytes >= 0, "%s: negative number in the shares", who);
  BSA_REQUIRE(s->n_groups < 0x7fffffffLL && s->n_merges < 0x3fffffffLL && s->n_slots < 0x3fffffffLL, "%s: too many shares", who);
  BSA_REQUIRE(s->groups != nullptr && s->n_groups > 0 && s->n_groups % 8 == 0, "%s: shares without groups, or not as many for each XCD", who);
  BSA_REQUIRE(s->n_merges == 0 || (s->merges != nullptr && s->scratch != nullptr), "%s: shares without merges or scratch", who);
  BSA_REQUIRE((reinterpret_cast<uintptr_t>(s->scratch) & 15) == 0, "%s: scratch of the shares must be 16-byte aligned", who);
  return BSA_OK;
}

int check_plan(const char *who, const bsa_attn_args *a, int key_rows) {
  BSA_REQUIRE(a != nullptr, "%s: NULL argument block", who);
  BSA_REQUIRE(key_rows == 0 || key_rows == 1, "%s: key_rows must be 0 or 1 (got %d)", who, key_rows);
  BSA_REQUIRE(a->B >= 0 && a->nq >= 0 && a->nk >= 0 && a->nh >= 0 && a->nhv >= 0, "%s: negative layout size", who);
  BSA_REQUIRE(a->B * a->nq < 0x7fffffffLL && a->B * a->nk < 0x7fffffffLL, "%s: too many sequence blocks", who);
  return BSA_OK;
}

}  // namespace

extern "C" int bsa_attn_fwd(const bsa_attn_args *args, bsa_stream_t stream) { return bsa_attn_fwd_shares(args, nullptr, stream); }

extern "C" int bsa_attn_shares_piece(const bsa_attn_args *a, int key_rows, int64_t n_entries, int64_t longest, int64_t *piece,
                                     int64_t *max_groups, int64_t *max_merges) {
  const char *who = "bsa_attn_shares_piece";
  const bool for_one_call = (key_rows & BSA_SHARES_FOR_ONE_CALL) != 0;
  key_rows &= ~BSA_SHARES_FOR_ONE_CALL;
  if (int rc = check_plan(who, a, key_rows)) return rc;
  BSA_REQUIRE(piece && max_groups && max_merges, "%s: NULL argument", who);
  *piece = bsa::attn_shares_piece(*a, key_rows != 0, for_one_call, n_entries, longest);
  *max_groups = *max_merges = 0;
  if (*piece > 0) bsa::attn_shares_limits(*a, key_rows != 0, n_entries, *piece, max_groups, max_merges);
  return BSA_OK;
}

extern "C" int bsa_attn_shares_build(const bsa_attn_args *a, int key_rows, int64_t piece, int64_t max_groups, int64_t max_merges,
                                     int32_t *groups, int32_t *merges, int64_t *stats, bsa_stream_t stream) {
  const char *who = "bsa_attn_shares_build";
  if (int rc = check_plan(who, a, key_rows)) return rc;
  BSA_REQUIRE(piece > 0, "%s: piece must be positive", who);
  BSA_REQUIRE(max_groups > 0 && max_groups % 8 == 0 && max_merges > 0, "%s: bad limits", who);
  BSA_REQUIRE((key_rows ? a->query_offsets : a->key_offsets) != nullptr && groups && merges && stats, "%s: NULL argument", who);
  BSA_REQUIRE(a->B > 0 && (key_rows ? a->nk : a->nq) > 0 && a->B * (key_rows ? a->nk : a->nq) <= 65536, "%s: 1 to 65536 rows", who);
  return bsa::attn_shares_build(*a, key_rows != 0, piece, max_groups, max_merges, groups, merges, stats, bsa::as_stream(stream));
}

extern "C" size_t bsa_attn_shares_scratch_bytes(const bsa_attn_args *a, int what, int64_t n_slots) {
  if (a == nullptr || what < 0 || what > 2 || n_slots <= 0) return 0;
  return (size_t)(n_slots * bsa::attn_shares_slot_bytes(*a, what));
}

extern "C" int bsa_attn_fwd_shares(const bsa_attn_args *args, const bsa_attn_shares *shares, bsa_stream_t stream) {
  if (int rc = check_args("bsa_attn_fwd", args, false)) return rc;
  if (int rc = check_shares("bsa_attn_fwd_shares", shares)) return rc;
  hipStream_t s = bsa::as_stream(stream);
  int rc = bsa::attn_fwd_mfma(*args, s);          // 16-bit operands, 64 x 64 blocks
  if (rc == 1) rc = bsa::attn_fwd_small(*args, shares, s);  // blocks of 16 and 32, fp32 blocks of 64
  if (rc == 1) rc = bsa::attn_fwd_f32mma(*args, s);         // everything else, on the fp32 matrix-core instruction
  if (rc == 1) rc = bsa::attn_fwd_generic(*args, s);
  return rc;
}

extern "C" int bsa_attn_fwd_records(const bsa_attn_args *a, const int32_t *group_entries, int32_t *records,
                                    bsa_stream_t stream) {
  const char *who = "bsa_attn_fwd_records";
  BSA_REQUIRE(a != nullptr, "%s: NULL argument block", who);
  BSA_REQUIRE(a->group_size == 1 || a->group_size == 2, "%s: group_size must be 1 or 2 (got %d)", who, a->group_size);
  BSA_REQUIRE(a->B >= 0 && a->nq >= 0 && a->nk >= 0, "%s: negative layout size", who);
  BSA_REQUIRE(a->nh >= 0 && a->nh <= 2 && a->nhv >= 0 && a->nhv <= 2, "%s: at most two head slices", who);
  BSA_REQUIRE(a->nk < (1 << 28), "%s: too many key blocks for a list entry", who);
  if (a->B * a->nq == 0) return BSA_OK;
  BSA_REQUIRE(a->group_offsets != nullptr, "%s: group_offsets is NULL", who);
  BSA_REQUIRE(a->nh == 0 || a->pidx_k, "%s: pidx_k is NULL", who);
  BSA_REQUIRE(a->nhv == 0 || a->pidx_v, "%s: pidx_v is NULL", who);
  BSA_REQUIRE(a->B * ((a->nq + a->group_size - 1) / a->group_size) < 0x7fffffffLL, "%s: too many groups", who);
  if (group_entries == nullptr || records == nullptr) return BSA_OK;  // no entries
  return bsa::attn_fwd_records(*a, group_entries, records, bsa::as_stream(stream));
}

namespace {

// One workgroup: a caller's sequences are few, and the launch in front of the attention kernels takes its 3 us anyway.  Written
// by the kernel itself: a copy to the host passes a copy engine, and what follows in the stream waits for that.  range[2]: the
// other two are there.
__global__ __launch_bounds__(256) void causal_lengths_range_kernel(const int64_t *__restrict__ lengths, int64_t n, int64_t *range) {
  __shared__ int64_t low[256], high[256];
  int64_t lo = lengths[0], hi = lo;
  for (int64_t i = threadIdx.x; i < n; i += 256) {
    const int64_t v = lengths[i];
    lo = v < lo ? v : lo;
    hi = v > hi ? v : hi;
  }
  low[threadIdx.x] = lo;
  high[threadIdx.x] = hi;
  for (int step = 128; step > 0; step >>= 1) {
    __syncthreads();
    if (threadIdx.x < step) {
      const int64_t l = low[threadIdx.x + step], h = high[threadIdx.x + step];
      if (l < low[threadIdx.x]) low[threadIdx.x] = l;
      if (h > high[threadIdx.x]) high[threadIdx.x] = h;
    }
  }
  if (threadIdx.x == 0) {
    __hip_atomic_store(range, low[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(range + 1, high[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(range + 2, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

}  // namespace

extern "C" int bsa_causal_lengths_range(const int64_t *lengths, int64_t n, int64_t *range, bsa_stream_t stream) {
  const char *who = "bsa_causal_lengths_range";
  BSA_REQUIRE(n >= 1, "%s: no lengths", who);
  BSA_REQUIRE(lengths != nullptr && range != nullptr, "%s: NULL argument", who);
  __atomic_store_n(range + 2, (int64_t)0, __ATOMIC_RELEASE);
  causal_lengths_range_kernel<<<1, 256, 0, bsa::as_stream(stream)>>>(lengths, n, range);
  return bsa::check_launch(who);
}

extern "C" int bsa_causal_lengths_wait(const int64_t *range, int64_t longest, bsa_stream_t stream) {
  const char *who = "bsa_causal_lengths_wait";
  BSA_REQUIRE(range != nullptr, "%s: NULL argument", who);
  if (!bsa::wait_for_word(who, range + 2, 0, stream)) return BSA_ELAUNCH;
  return range[0] < 0 || range[1] > longest ? 1 : BSA_OK;
}

extern "C" int bsa_attn_mask_dead(const void *mask, int64_t n_mask_blocks, int32_t sbs, uint8_t *dead,
                                  bsa_stream_t stream) {
  const char *who = "bsa_attn_mask_dead";
  BSA_REQUIRE(sbs == 64, "%s: only 64 x 64 blocks (got %d)", who, sbs);
  BSA_REQUIRE(n_mask_blocks >= 0 && n_mask_blocks < 0x7fffffffLL, "%s: bad number of mask blocks", who);
  if (n_mask_blocks == 0) return BSA_OK;
  BSA_REQUIRE(mask != nullptr && dead != nullptr, "%s: NULL argument", who);
  BSA_REQUIRE((reinterpret_cast<uintptr_t>(mask) & 15) == 0, "%s: mask must be 16-byte aligned", who);
  return bsa::attn_mask_dead(mask, n_mask_blocks, dead, bsa::as_stream(stream));
}

extern "C" size_t bsa_attn_bwd_scratch_bytes(int64_t B, int64_t nq, int64_t nk, int64_t n_layout_blocks,
                                             int64_t n_mask_blocks) {
  if (B < 0 || nq < 0 || nk < 0 || n_layout_blocks < 0 || n_mask_blocks < 0) return 0;
  return bsa::attn_bwd_scratch_bytes(B, nq, nk, n_layout_blocks, n_mask_blocks);
}

extern "C" size_t bsa_attn_bwd_ds_bytes(int64_t n_layout_blocks, int32_t sbs) {
  if (n_layout_blocks < 0 || sbs != 64) return 0;
  return bsa::attn_bwd_ds_bytes(n_layout_blocks);
}

extern "C" int bsa_attn_bwd(const bsa_attn_args *args, bsa_stream_t stream) {
  return bsa_attn_bwd_shares(args, nullptr, nullptr, stream);
}

extern "C" int bsa_attn_bwd_shares(const bsa_attn_args *args, const bsa_attn_shares *query_shares, const bsa_attn_shares *key_shares,
                                   bsa_stream_t stream) {
  if (int rc = check_args("bsa_attn_bwd", args, true)) return rc;
  if (int rc = check_shares("bsa_attn_bwd_shares", query_shares)) return rc;
  if (int rc = check_shares("bsa_attn_bwd_shares", key_shares)) return rc;
  BSA_REQUIRE(args->bwd_scratch == nullptr || args->n_layout_blocks >= 0, "bsa_attn_bwd: negative n_layout_blocks");
  BSA_REQUIRE(args->bwd_scratch_bytes >= 0, "bsa_attn_bwd: negative bwd_scratch_bytes");
  BSA_REQUIRE((reinterpret_cast<uintptr_t>(args->bwd_scratch) & 15) == 0, "bsa_attn_bwd: bwd_scratch must be 16-byte aligned");
  BSA_REQUIRE(args->bwd_ds_bytes >= 0, "bsa_attn_bwd: negative bwd_ds_bytes");
  BSA_REQUIRE((reinterpret_cast<uintptr_t>(args->bwd_ds) & 15) == 0, "bsa_attn_bwd: bwd_ds must be 16-byte aligned");
  if (args->bwd_scratch != nullptr && args->bwd_scratch_bytes > 0) {
    const size_t need = bsa::attn_bwd_scratch_bytes(args->B, args->nq, args->nk, args->n_layout_blocks, args->n_mask_blocks);
    BSA_REQUIRE((size_t)args->bwd_scratch_bytes >= need, "bsa_attn_bwd: bwd_scratch holds %lld bytes, %zu are needed",
                (long long)args->bwd_scratch_bytes, need);
  }
  hipStream_t s = bsa::as_stream(stream);
  int rc = bsa::attn_bwd_mfma(*args, s);
  if (rc == 1) rc = bsa::attn_bwd_small(*args, query_shares, key_shares, s);
  if (rc == 1) rc = bsa::attn_bwd_f32mma(*args, s);
  if (rc == 1) rc = bsa::attn_bwd_generic(*args, s);
  return rc;
}
