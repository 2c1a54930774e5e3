// Shares of the rows of an attention layout for the kernels of attn_small_fwd.hip and attn_small_bwd.hip, where its lists are
// uneven: which rows a workgroup of four waves takes, and how many waves, of how many workgroups, share a row.
//
// Without them every row of a launch gets the same number of waves (waves_per_row), and the launch lasts as long as the walk
// of its longest list: the global rows and columns of a BigBird layout have ten times the blocks of the others, the last
// rows of one long causal sequence twice the mean of a launch that leaves half of the chip idle.  Here a row gets waves by its
// own length, so that none walks much more than `piece` entries: the mean of a wave of a full chip, or the least that is worth a
// wave's start.  None gets fewer than waves_per_row gives it: every part of a list rounds its probabilities against a maximum of
// its own, and with one part instead of four the short rows of 16-bit operands were 1 to 4 % further from 64 bits.  Rows of more
// than four waves are several workgroups', whose sums a small launch adds up, in order.  Long rows come first, then the others
// by the waves they get, each kind in the order of RowOfWave.
//
// 7 sequences of 3328, sbs 32, head dimension 96, BigBird, bf16, forward: 27 us with, 76 without; 14 of 1056, sbs 32, head
// dimension 128, BigBird, fp32, forward and backward: 248 with, 340 without; one of 6080, sbs 64, head dimension 64, causal,
// fp32, the same: 279 with, 429 without.
#include "attn_small_common.h"

namespace bsa {
namespace {

using namespace small;

constexpr int kThreads = 1024, kClasses = 5;  // several workgroups, four waves of a long list, four, two, one
constexpr int kXcds = 8;

// How long rows are cut: pieces of about `piece` entries, by more than four waves (whose sums take a scratch and a launch more)
// above `most` entries, by at least min_parts
struct Cut {
  int halves, min_parts;
  int64_t piece, most;
};

struct Item {
  int64_t b, own, parts;
  int kind;  // its class, -1: no row
};
__device__ inline Item item_of(const int32_t *offsets, uint32_t item, int64_t items, int64_t batches, int64_t rows,
                               bool last_first, const Cut &cut) {
  Item it;
  it.kind = -1, it.parts = 0;
  if (item < items && row_of_item(blockIdx.x, item, batches, rows, last_first, it.b, it.own)) {
    const int64_t row = it.b * rows + it.own, n = (int64_t)cut.halves * (offsets[row + 1] - offsets[row]);
    const int64_t parts = 2 * n <= 3 * cut.piece ? 1
                          : n <= 3 * cut.piece   ? 2
                          : n <= cut.most        ? 4
                                                 : 4 * ((n + 4 * cut.piece - 1) / (4 * cut.piece));
    it.parts = parts < cut.min_parts ? cut.min_parts : parts;
    it.kind = parts > 4 ? 0 : parts > 2 ? 1 : it.parts == 4 ? 2 : it.parts == 2 ? 3 : 4;
  }
  return it;
}

// Exclusive sums over the threads of the block, and the totals, of one small number per class
__device__ inline void scan_classes(int (&v)[kClasses], int (&total)[kClasses], int (*lds)[kThreads / 64]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int c = 0; c < kClasses; ++c) {
    int sum = v[c];
    for (int d = 1; d < 64; d <<= 1) {
      const int below = __shfl_up(sum, d);
      if (lane >= d) sum += below;
    }
    if (lane == 63) lds[c][wave] = sum;
    v[c] = sum - v[c];
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < kClasses; ++c) {
    total[c] = 0;
    for (int w = 0; w < kThreads / 64; ++w) {
      if (w == wave) v[c] += total[c];
      total[c] += lds[c][w];
    }
  }
  __syncthreads();
}

// One workgroup per XCD: counts its rows by class, then hands out its groups.  stats: most groups of an XCD, merges, slots.
__global__ __launch_bounds__(kThreads) void attn_shares_kernel(const int32_t *__restrict__ offsets, int64_t items, int64_t batches,
                                                               int64_t rows, bool last_first, Cut cut, int64_t max_groups,
                                                               int64_t max_merges, int32_t *__restrict__ groups,
                                                               int32_t *__restrict__ merges, unsigned long long *__restrict__ stats) {
  __shared__ int sums[kClasses][kThreads / 64];
  const int xcd = blockIdx.x;
  int mine[kClasses] = {}, all[kClasses];
  for (int64_t base = 0; base < items; base += kThreads) {
    const Item it = item_of(offsets, (uint32_t)(base + threadIdx.x), items, batches, rows, last_first, cut);
#pragma unroll
    for (int c = 0; c < kClasses; ++c) mine[c] += it.kind != c ? 0 : c == 0 ? (int)(it.parts / 4) : 1;
  }
  scan_classes(mine, all, sums);
  // first group of every class
  const int64_t whole = (int64_t)all[0] + all[1] + all[2];
  const int64_t first[kClasses] = {0, all[0], (int64_t)all[0] + all[1], whole, whole + (all[3] + 1) / 2};
  const int64_t n_groups = first[4] + (all[4] + 3) / 4;

  int done[kClasses] = {};
  for (int64_t base = 0; base < items; base += kThreads) {
    const Item it = item_of(offsets, (uint32_t)(base + threadIdx.x), items, batches, rows, last_first, cut);
    int before[kClasses], chunk[kClasses];
#pragma unroll
    for (int c = 0; c < kClasses; ++c) before[c] = it.kind != c ? 0 : c == 0 ? (int)(it.parts / 4) : 1;
    scan_classes(before, chunk, sums);
    int rank = 0, last = 0;
    int64_t from = 0;
#pragma unroll
    for (int c = 0; c < kClasses; ++c) {
      if (it.kind == c) rank = done[c] + before[c], last = all[c] - 1, from = first[c];
      done[c] += chunk[c];
    }
    if (it.kind < 0) continue;
    const int per_group = it.kind <= 2 ? 1 : it.kind == 3 ? 2 : 4;  // rows
    const int waves = 4 / per_group, n = it.kind == 0 ? (int)(it.parts / 4) : 1;
    int slot = -1;
    if (it.kind == 0) {
      slot = (int)atomicAdd(&stats[2], (unsigned long long)n);
      const int64_t m = (int64_t)atomicAdd(&stats[1], 1ull);
      if (m < max_merges) {
        int32_t *merge = merges + 4 * m;
        merge[0] = (int)it.b, merge[1] = (int)it.own, merge[2] = slot, merge[3] = n;
      }
    }
    for (int i = 0; i < n; ++i) {
      const int64_t at = from + (rank + i) / per_group;
      if (at >= max_groups) break;
      int32_t *g = groups + (at * kXcds + xcd) * BSA_SHARE_INTS;
      const int w0 = (rank + i) % per_group * waves;
      for (int w = w0; w < w0 + waves; ++w) g[w] = (int)it.own, g[4 + w] = (int)it.b;
      if (w0 == 0) g[8] = 4 * i, g[9] = (int)it.parts, g[10] = slot < 0 ? -1 : slot + i, g[11] = 0;
      if (rank == last)  // the last group of its kind may have room left
        for (int w = w0 + waves; w < 4; ++w) g[w] = -1, g[4 + w] = 0;
    }
  }
  for (int64_t at = n_groups + threadIdx.x; at < max_groups; at += kThreads) {
    int32_t *g = groups + (at * kXcds + xcd) * BSA_SHARE_INTS;
    for (int w = 0; w < 4; ++w) g[w] = -1, g[4 + w] = 0;
    g[8] = 0, g[9] = 1, g[10] = -1, g[11] = 0;
  }
  if (threadIdx.x == 0) atomicMax(&stats[0], (unsigned long long)n_groups);
}

int halves_of(const bsa_attn_args &a) { return a.sbs == 64 ? 2 : 1; }
int64_t slices_of(const bsa_attn_args &a) { return a.nh > a.nhv ? a.nh : a.nhv; }

}  // namespace

static int least_parts(const bsa_attn_args &a, bool key_rows) {
  const int64_t halves = halves_of(a), rows = halves * a.B * (key_rows ? a.nk : a.nq), partners = halves * (key_rows ? a.nq : a.nk);
  const int per_step = a.sbs == 16 ? 2 : 1;
  return a.dtype == BSA_F32 ? waves_per_row<4>(rows, partners, per_step) : waves_per_row<2>(rows, partners, per_step);
}

// Entries from which a row is several workgroups'.  The scratch, the launch that adds the sums and its host work cost some
// 15 us: as long as these many steps (head dimensions up to 64, beyond) by which a quarter of the list has to be longer than
// a piece.
static int64_t steps_of_a_scratch(const bsa_attn_args &a) {
  const bool small_head = slices_of(a) * a.sbs <= 64;
  return (a.dtype == BSA_F32 ? (small_head ? 6 : 3) : (small_head ? 24 : 16)) * (a.sbs == 16 ? 2 : 1);
}
static int64_t most_of_a_group(const bsa_attn_args &a, int64_t piece) {
  const int64_t most = 4 * (piece + steps_of_a_scratch(a));
  return most > 6 * piece ? most : 6 * piece;
}

// The longest share a wave should walk, in blocks of the kernels, or 0: the rows are even enough for waves_per_row, or not for
// the kernels that read shares.
//
// waves: what the chip holds of these kernels at a time (their registers and LDS).  least: entries of a wave's walk that cost
// about as much as its start and end, six steps (16-bit; four of fp32, whose products take longer).  Shares have to be long enough
// for the host work of a call (7 us, 22 with a scratch) and the 70 us that a new layout's first call pays: eight steps (fp32: four)
// and half a mean above the mean, and they have to change something.  Times are GPU times of forward + backward, without ->
// with shares, us:
//   cut    The longest rows become several workgroups'.  Where lengths fall off evenly (causal) those just below
//          most_of_a_group stay, and the launch gets shorter by the difference only: fp32 causal, head dimension 64, sbs 32, 8 x 2048
//          (64 blocks, cut from 61 on) 180 -> 197, 4 x 2048 (from 45 on) 162 -> 146, 2 x 4096 (128, from 61 on) 292 -> 206; bf16, 2 x
//          4096 (128, from 121 on) 76 -> 84.  A few long ones among short ones: 2 x 4096 BigBird, fp32 331 -> 104, bf16 107 -> 49.
//          6 x 1664 BigBird, fp32, sbs 64, head dimension 128 (52 halves, cut from 49 on) 382 -> 330.
//   waves  The longest rows get more waves than waves_per_row gives them.  Longest share of 3.4 pieces (24 x 1536 causal, bf16, sbs
//          32) 80 -> 63, 3.8 (8 x 2048, fp16, sbs 16) 95 -> 70; 1.7 (24 x 1536, bf16 at head dimension 128; fp16, sbs 16) 134 -> 137, 85 -> 87.
//   order  A launch of more than one round would start its longest lists, more than twice the mean, anywhere: 24 x 1536 BigBird, fp32,
//          sbs 32, head dimension 64 (share 12, piece 8) 275 -> 215; at 128 (piece 15, so no share is long) 630 -> 642.  The
//          walk of one takes 22 steps (14 at head dimensions above 64, fp32 8) or more.
// for_one_call: without a layout cache the tables and the wait for their size, some 50 us each, are this call's alone: only a
// share that gets shorter by four times what pays for a scratch is worth them (fp32: one sequence of 6080, sbs 64, causal, forward
// and backward, a call 600 without, 554 us with; 8 x 2048 causal 395 and 495, 14 x 1056 BigBird at 128 479 and 484; 16-bit: 7 x 3328
// BigBird forward 237 and 265, 5 x 3152 causal 373 and 460).
int64_t attn_shares_piece(const bsa_attn_args &a, bool key_rows, bool for_one_call, int64_t n_entries, int64_t longest) {
  const int halves = halves_of(a);
  const bool wide = a.dtype == BSA_F32;
  if ((a.sbs != 16 && a.sbs != 32 && !(a.sbs == 64 && wide)) || n_entries <= 0 || longest <= 0) return 0;
  const int64_t slices = slices_of(a), rows = halves * a.B * (key_rows ? a.nk : a.nq);
  if (slices < 1 || slices > 128 / a.sbs || rows > 65536) return 0;
  const bool small_head = slices * a.sbs <= 64;
  const int per_step = a.sbs == 16 ? 2 : 1;
  const int64_t waves = wide ? (small_head ? 2048 : 1024) : (small_head && !key_rows ? 4096 : 2048);
  const int64_t least = (wide ? 4 : 6) * per_step, entries = (int64_t)halves * halves * n_entries;
  const int64_t mean = cdiv(entries, waves), piece = mean > least ? mean : least;
  const int split = least_parts(a, key_rows);
  const int64_t most = most_of_a_group(a, piece), n = halves * longest, share = n / split, worth = (wide ? 4 : 8) * per_step;
  const bool long_shares = 2 * share > 3 * piece && share >= piece + worth;
  const bool cut = long_shares && n > most && (n * rows > 3 * entries || n - most > (wide ? 1 : 2) * steps_of_a_scratch(a));
  const bool more_waves = long_shares && split < 4 && share >= 2 * piece;
  const bool order = rows * split > waves && n * rows > 2 * entries && share >= piece &&
                     share >= least + (wide || !small_head ? worth : 2 * worth);
  if (for_one_call && share < piece + 4 * steps_of_a_scratch(a)) return 0;
  return cut || more_waves || order ? piece : 0;
}

int attn_shares_build(const bsa_attn_args &a, bool key_rows, int64_t piece, int64_t max_groups, int64_t max_merges, int32_t *groups,
                      int32_t *merges, int64_t *stats, hipStream_t s) {
  const int64_t rows = key_rows ? a.nk : a.nq;
  const Cut cut{halves_of(a), least_parts(a, key_rows), piece, most_of_a_group(a, piece)};
  attn_shares_kernel<<<kXcds, kThreads, 0, s>>>(key_rows ? a.query_offsets : a.key_offsets, row_items(a.B, rows), a.B, rows,
                                                !key_rows, cut, max_groups / kXcds, max_merges, groups, merges,
                                                reinterpret_cast<unsigned long long *>(stats));
  return check_launch("attn_shares_kernel");
}

void attn_shares_limits(const bsa_attn_args &a, bool key_rows, int64_t n_entries, int64_t piece, int64_t *max_groups, int64_t *max_merges) {
  // a row of n entries takes at most one workgroup and n / (4 piece) more, and is merged if n > 6 piece
  const int64_t entries = halves_of(a) * n_entries;
  *max_groups = kXcds * (row_items(a.B, key_rows ? a.nk : a.nq) + entries / (4 * piece) + 1);
  *max_merges = entries / (6 * piece) + 1;
}

int64_t attn_shares_slot_bytes(const bsa_attn_args &a, int what) {
  const int64_t block = a.sbs == 16 ? 256 : 1024, side = a.sbs == 16 ? 16 : 32;  // of the kernels
  const int64_t sums = slices_of(a) * halves_of(a) * block;
  return halves_of(a) * 4 * (what == 0 ? sums + 2 * side : what == 1 ? sums : 2 * sums);
}

}  // namespace bsa
