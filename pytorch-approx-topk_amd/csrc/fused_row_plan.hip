// Host-side planning and dispatch of the fused one-workgroup-per-row kernel.
#include <cmath>

#include "fused_row.h"

namespace atk {
namespace fused {

namespace {
// Rows below which one workgroup per row leaves most of the 256 CUs idle: taken
// then only for rows one workgroup reads in a few microseconds, where saving
// the second launch is what counts (1-96 rows in a HIP graph, bf16 up to 128K
// elements: 16-31 % faster; rows of 512 KiB: even to 13 % slower; of 1 MiB: 20-60 %
// slower).
constexpr int64_t kMinRows = 128;
constexpr size_t kSoloRow = 256 * 1024;
// Dynamic LDS a workgroup may use (candidates + hand-over); the select's own
// block adds about 9 KiB.
constexpr size_t kLdsBudget = 64 * 1024;
// The candidates may take twice that, one workgroup of sixteen waves per CU
// then: the alternative parks them in HBM and selects with one workgroup per
// row as well.  Measured against the two-kernel path: fp16 [256, 65536]
// k0=32768 71 -> 38 us, [1024, 65536] 312 -> 142 us, [512, 262144] 184 -> 113 us,
// [128, 2^20] 90 -> 85 us, fp32 [256, 65536] k0=16384 52 -> 35 us, [2048, 131072]
// 375 -> 336 us.  (With eight waves the larger budget lost for rows beyond
// 256 KiB: [128, 2^20] 87 -> 115 us.)
constexpr size_t kLdsBudgetLarge = 128 * 1024;
// Most waves per workgroup.  Measured over shapes from [4096, 4096] to
// [256, 65536]: 8 beats 16 (more workgroups per CU, in different phases, and
// cheaper barriers) and is never far behind 4.
constexpr uint32_t kMaxWaves = 8;
// Corners in which the two-kernel path may be the faster one (see make_plan).
constexpr int64_t kManyRows = 1024, kAllCus = 256;
// Longest contiguous bucket (bytes) the register kernel takes.
constexpr int64_t kShortBucket = 256;
constexpr size_t kShortRow = 128 * 1024, kLongRow = 512 * 1024;

// Whether rows that do not all start on 16 bytes (8 for one-byte elements) are faster in one kernel.  256 calls of such rows timed against the
// two kernels (with the width of loads that the planner takes there): what decides is how many sub-rows a wave
// goes through (`run`, over all its tiles), for which the two kernels have any number of workgroups.
//   Fewer rows than kMinRows: runs of up to 40 sub-rows with queues of one or two entries, of up to 20 with more, and
//   sub-rows of 256 bytes (fp16 [75, 42783] b=952 j=2, run 22, 15.6 -> 11.0 us, [16, 45917] b=1276, run 36, 10.9 -> 8.1, but
//   [5, 104575] b=392 j=2, run 67, 10.2 -> 15.7, bf16 [4, 118981] b=1072 j=3, run 111, 13.5 -> 19.9, [7, 2193] b=16 j=4
//   9.0 -> 11.8); longer queues with sub-rows of 2.5 KB and more, runs of up to 64 (i16 [46, 72589] b=1428 j=4, run 50,
//   17.3 -> 14.0; f32 [14, 51519] b=344 j=4, run 37, 13.5 -> 16.8); of eight-byte elements they lose throughout (fp64
//   [14, 3303] b=32 j=4 13.6 -> 25.2).
//   Fewer rows than CUs: runs of up to 256 (fp32 [193, 82525] b=680 j=3, run 60, 29.1 -> 23.0; fp16 [183, 340470] b=304
//   j=4, run 280, 49.7 -> 59, i16 [152, 394615] b=1140 j=4, run 346, 49.9 -> 60.3).
//   More rows: all (fp16 [742, 9559] b=264 15.4 -> 11.0, bf16 [552, 6915] b=132 j=4 17.4 -> 12.4, i16 [759, 57865]
//   b=448 j=4 48.4 -> 42.1).
//   One-byte elements, whose packed queues this kernel lacks: batches with queues of one or two entries (uint8 [1354, 66483]
//   j=1 67.0 -> 50.5, [374, 23585] j=2 23.4 -> 19.2, but [1538, 37707] j=4 74 -> 214, [11, 10433] j=4 10.6 -> 40.7), and those of more
//   rows than the second stage's workgroups of up to 1024 threads have launches for (threads are counted in 32 bits).
bool loose_rows_gain(int64_t rows, int64_t sub_row_bytes, int64_t run, int j, int es) {
  if (es == 1) return (rows >= kMinRows && j <= 2) || rows > 0xffffffffll / 1024;
  if (rows >= kMinRows) return rows >= kAllCus || run <= 256;
  return run <= (j <= 2 ? 40 : es == 8 ? 0 : sub_row_bytes >= 2560 ? 64 : 20) && sub_row_bytes >= 256;
}
}  // namespace

// Staged results leave in non-temporal stores when the launch is one round of workgroups
// (no more rows than the GPU holds at once) and a row's results are an eighth of its bytes
// or more.  What a kernel has written sits in the L2 of its XCD until the kernel ends and
// is written back then, with nothing left to hide it behind: first workgroup's start to
// last store 22.8 us of fp16 [1024, 32768] k=2048 j=4 k_mult=4's 27.1 us per call.  Sent
// past the cache the results travel while other workgroups still work: 27.6 -> 25.4 us
// there, fp16 [256, 131072] k=4096 j=4 k_mult=2 22.2 -> 20.1 us, fp32 [512, 32768] k=2048
// j=4 k_mult=4 24.4 -> 23.1 us.  With several rounds the write-back hides behind the
// later rounds by itself and the stores past the cache cost more than they save ([4096,
// 8192] k=512 35.6 -> 36.9 us, [2048, 32768] 46.3 -> 47.3 us), as they do with little
// output ([1024, 65536] k=512 44.0 -> 45.1 us).
static bool stores_past_cache(int64_t rows, int64_t n, int64_t k, int64_t es) {
  return rows <= kManyRows && k * (es + 8) * 8 >= n * es;
}

// Contiguous buckets, all of one length of 16 to kShortBucket bytes, elements of
// two or four bytes: a lane of the register kernel loads its four buckets whole.  The
// alternative is a stage-1 kernel that copies spans of buckets through LDS and
// parks the candidates in HBM for a stand-alone select: fp16 [1024, 32768]
// k=2048 j=4 k_mult=4 (buckets of 32 bytes) 68.6 us that way against 35; buckets of
// 128 bytes fp16 [256, 131072] k0=8192 39.2 against 33.3 us, fp32 [64, 32768] k0=2048
// 17.4 against 12.7 us; of 256 bytes fp16 [256, 262144] k0=8192 57.6 against 49.4 us,
// [1024, 131072] 109.9 against 110.3 us.
static Plan plan_short_buckets(int64_t rows, int64_t n, int64_t k0, int j, int64_t k, int dtype) {
  Plan pl{};
  pl.ok = false;
  if (rows > 0x7fffffffll) return pl;
  if (k0 <= 0 || k <= 0 || k >= k0 || j < 1 || j > 4 || k0 % j) return pl;
  const int es = elem_bytes(dtype);
  if (es != 2 && es != 4) return pl;
  // fewer rows than CUs: only rows one workgroup reads in a few microseconds (fp32 [130, 131072]
  // with 2048 buckets of 256 bytes: 38.4 us here against 32.4 through two kernels, whose stage 1
  // has sixteen workgroups per row)
  if (rows < kAllCus && (size_t)n * es > kSoloRow) return pl;
  const int64_t b = k0 / j;
  if (n % b) return pl;
  const int64_t m = n / b;
  if ((m * es) % 16 || m * es > kShortBucket || m < j) return pl;
  pl.full_rows = (uint32_t)m;
  pl.pos16 = true;
  pl.packed = es == 2;
  pl.vec = 4;
  // whole tiles only: a lane's buckets lie a wave's width apart
  if (b % (stream::kWave * pl.vec)) return pl;
  pl.tiles = (uint32_t)(b / (stream::kWave * pl.vec));
  if (pl.tiles > kMaxWaves) return pl;
  pl.index_bits = 1;
  while (pl.index_bits < 63 && (1ll << pl.index_bits) < n) ++pl.index_bits;
  pl.split = 1;
  pl.waves = pl.tiles;
  pl.contig = pl.in_registers = true;
  const size_t cand_bytes = (((size_t)k0 * es + 15) & ~(size_t)15) + (((size_t)k0 * 2 + 15) & ~(size_t)15);
  pl.lds_bytes = cand_bytes > regs::kLdsBytes ? cand_bytes : regs::kLdsBytes;
  pl.staged = (size_t)k * 8 <= kLdsBudget;
  if (pl.staged && pl.lds_bytes < (size_t)k * 8) pl.lds_bytes = (size_t)k * 8;
  pl.past_cache = pl.staged && stores_past_cache(rows, n, k, es);
  pl.ok = true;
  return pl;
}

// Interleaved buckets, loads of `vec` elements.  `by_size`: only where the rules of size below call this path the faster one
// (they were measured with loads of the usual width); else wherever the kernels take the call.
static Plan plan_interleaved(int64_t rows, int64_t n, int64_t k0, int j, int64_t k, int dtype, bool aligned, int vec,
                             bool by_size) {
  Plan pl{};
  pl.ok = false;
  if (rows > 0x7fffffffll) return pl;
  if (k0 <= 0 || k <= 0 || k >= k0 || j < 1 || j > 4 || k0 % j) return pl;
  const int es = elem_bytes(dtype);
  if (!es) return pl;
  if (by_size && rows < kMinRows && (size_t)n * es > kSoloRow) return pl;
  const int64_t b = k0 / j;
  const int64_t full = n / b;
  if (full < j || full > 0x7fffffffll) return pl;
  pl.full_rows = (uint32_t)full;
  pl.rem = (uint32_t)(n - full * b);
  pl.pad_tail = 0;
  pl.pos16 = full + 1 <= 0xffff;
  pl.packed = (dtype == ATK_F16 || dtype == ATK_BF16 || dtype == ATK_I16) && full <= stream::kPackedMaxSubRow;
  pl.vec = vec;
  // packed queues at half the load width need about 50 VGPRs instead of 127:
  // twice the workgroups per CU, which is worth more here than 16-byte loads
  if (pl.packed && pl.vec == stream::full_vec(es)) pl.vec /= 2;
  if (b % pl.vec) return pl;
  const int64_t bound = (full + 1) * b;  // indices are < this
  pl.index_bits = 1;
  while (pl.index_bits < 63 && (1ll << pl.index_bits) < bound) ++pl.index_bits;

  const int64_t tile_cols = (int64_t)stream::kWave * pl.vec;
  pl.tiles = (uint32_t)((b + tile_cols - 1) / tile_cols);
  // Few buckets: a sub-row of b elements is all a wave loads at a time here
  // (this kernel does not fold sub-rows side by side as the streaming kernel
  // does), so with narrow sub-rows most lanes idle and the few that work walk
  // the whole row.  Measured against the two-kernel path (fp16 and fp32, 8-256
  // buckets, k_mult = 2): fp16 [256, 2^22] with 8 buckets 10.2 ms against
  // 0.36 ms, [2048, 8192] with 32 buckets 29 against 14 us, while rows of a few
  // KiB still gain from the saved launch (5.5 against 7.7 us).  The sub-row a
  // call needs grows with the row and with the number of rows.  Batches of up to
  // 1 MiB in all are bound by launches, not by bytes: there this kernel takes
  // 5 us + 11 ns per sub-row of the row ([4, 32768] with 4 buckets: 94-118 us)
  // against 8-15 us for the two kernels whatever the shape, and narrow sub-rows
  // are taken while the row has fewer than 256 of them.
  {
    const size_t sub_row_bytes = (size_t)b * es, row_bytes_ = (size_t)n * es;
    size_t least = 128;
    if (row_bytes_ > 16 * 1024) least = 256;
    if (row_bytes_ > 32 * 1024 || rows >= 2048) least = 512;
    const bool small_batch = (size_t)rows * row_bytes_ <= (1u << 20);
    if (by_size && sub_row_bytes < least && (!small_batch || full >= 256)) return pl;
  }
  // One launch instead of two, and no candidates parked in HBM: measured over
  // 128-4096 rows of 8192-262144 elements with 256-4096 candidates, this kernel
  // is 5-40 % faster than the two-kernel path for the packed 16-bit types
  // throughout and for wider types except in two corners: many short rows
  // (>= 1024 rows of < 128 KiB: +5-35 %; the stand-alone select runs more rows
  // per CU) and fewer rows than CUs with j >= 3 and rows of >= 512 KiB (+10-30 %;
  // the two-kernel path cuts such rows into slabs).  There, and for 1-byte
  // types (whose packed queues only the streaming kernel has), it is taken only
  // when parking the candidates would cost a good part of what reading the row
  // costs: written and re-read k0*(es+8) bytes against n*es.
  const size_t row_bytes = (size_t)n * es;
  const bool corner = es == 1 || (!pl.packed && ((rows >= kManyRows && row_bytes < kShortRow) ||
                                                 (rows < kAllCus && j >= 3 && row_bytes >= kLongRow)));
  if (by_size && corner && (size_t)k0 * (es + 8) * 4 < row_bytes) return pl;
  const int skey = (dtype == ATK_U8 || dtype == ATK_I8) ? 2 : es;  // stored key width
  const size_t cand_bytes = (((size_t)k0 * skey + 15) & ~(size_t)15) +
                            (((size_t)k0 * (pl.pos16 ? 2 : 4) + 15) & ~(size_t)15);
  const size_t lds_budget = kLdsBudgetLarge;
  if (cand_bytes > lds_budget) return pl;

  // With more than the usual LDS budget taken, or with no more rows than CUs, one
  // workgroup has the CU to itself: sixteen waves then, when eight would go through
  // the tiles in several rounds (the scan and the selection both gain: fp16
  // [256, 65536] k0=16384 32.8 -> 25.8 us, [200, 32768] k0=16384 30.3 -> 22.7 us; with
  // 300-512 rows eight waves stay ahead, 43 against 49 us at [512, 65536]).
  const uint32_t max_waves =
      (cand_bytes > kLdsBudget || (rows <= kAllCus && pl.tiles > kMaxWaves)) ? 2 * kMaxWaves : kMaxWaves;
  // Waves sharing a tile: as many as keep each share at least max(j, 8)
  // sub-rows long, the workgroup within its wave limit and LDS within budget.
  // When all tiles are in flight at once the hand-over area may lie on top of
  // the candidates.
  const int cmp_size = es > 4 ? 8 : 4;
  const int64_t min_run = j > 8 ? j : 8;
  auto hand_bytes = [&](uint32_t split) {
    const uint32_t waves = pl.tiles * split <= max_waves ? pl.tiles * split : max_waves;
    return (size_t)(waves - waves / split) * pl.vec * j * stream::kWave * (cmp_size + 4);
  };
  auto lds_need = [&](uint32_t split) {
    const bool one_round = pl.tiles * split <= max_waves;
    const size_t hand = hand_bytes(split);
    return one_round ? (hand > cand_bytes ? hand : cand_bytes) : cand_bytes + hand;
  };
  uint32_t split = 1;
  if (pl.tiles < max_waves) {
    for (uint32_t cand = 2; cand * pl.tiles <= max_waves; cand *= 2) {
      if (full / cand < min_run || lds_need(cand) > lds_budget) break;
      split = cand;
    }
  }
  pl.split = split;
  pl.waves = pl.tiles * split <= max_waves ? pl.tiles * split : max_waves;
  const int64_t turns = ((int64_t)pl.tiles * split + pl.waves - 1) / pl.waves;
  if (by_size && !aligned && !loose_rows_gain(rows, b * es, full / split * turns, j, es)) return pl;
  const bool one_round = pl.tiles * split <= max_waves;
  pl.hand_off = (split > 1 && !one_round) ? (uint32_t)cand_bytes : 0u;
  pl.lds_bytes = lds_need(split);
  // every tile has its waves: stage 2 runs on the candidates where they are, in
  // registers, and needs the histogram's room in LDS
  pl.in_registers = one_round && pl.waves <= kMaxWaves;  // (the register kernel is built for eight waves)
  if (pl.in_registers) {
    // the hand-over area lies behind the first digits' histogram, which is counted while it is in use
    pl.hand_off = split > 1 ? (uint32_t)(regs::kHistWords * sizeof(uint32_t)) : 0u;
    const size_t hand = pl.hand_off + (size_t)(pl.waves - pl.waves / split) * pl.vec * j * stream::kWave *
                                          (pl.packed ? 4 : cmp_size + 4);
    pl.lds_bytes = hand > cand_bytes ? hand : cand_bytes;
    if (pl.lds_bytes < regs::kLdsBytes) pl.lds_bytes = regs::kLdsBytes;
  }
  // survivors staged in LDS, eight bytes each (element, 32-bit index), when that fits
  pl.staged = pl.in_registers && pl.pos16 && es <= 4 && (size_t)k * 8 <= kLdsBudget;
  if (pl.staged && pl.lds_bytes < (size_t)k * 8) pl.lds_bytes = (size_t)k * 8;
  pl.past_cache = pl.staged && stores_past_cache(rows, n, k, es);
  pl.ok = true;
  return pl;
}

// Whether the rules of size alone, which the figure of atk_topk_workspace_bytes_at follows, choose one kernel.
bool taken_by_size(int64_t rows, int64_t n, int64_t k0, int j, int64_t k, int layout, int dtype, bool aligned) {
  if (layout == ATK_BALANCED) return plan_short_buckets(rows, n, k0, j, k, dtype).ok;
  const int es = elem_bytes(dtype);
  return layout == ATK_INTERLEAVED && es != 0 &&
         plan_interleaved(rows, n, k0, j, k, dtype, aligned, stream::full_vec(es), true).ok;
}

namespace {
// Rows and candidates up to which the estimates below were fitted.
constexpr int64_t kEstimatedRow = 1 << 20, kEstimatedCandidates = 8192;
// A call that the rules of size leave to two kernels takes one where its estimate is this share of theirs.  On 1500 calls that
// both take and neither estimate was fitted to, the choice (the rules of size included) is 1.2 % slower than the better of the
// two, one kernel throughout 33 %, two 20 %; the share could be 1.0, but for rows whose cut falls among ties, which cost one
// kernel more (of 43 such shapes four were over 10 % slower at 0.85).
constexpr double kOneKernelShare = 0.9;

// Estimated microseconds of the register kernel under a plan of elements of two or four bytes: the scan (memory, instructions
// and the round trips of a wave's loads, which overlap: the root of the sum of their squares), and what every
// round of workgroups that the GPU holds at once goes through behind it, the fold of the waves that share a tile and the
// selection, by the candidates of a lane and the waves that wait for one another.
// The constants are a least-squares fit to 1415 launches of 620 calls (fp32 and fp16, 1-8192 rows of 2048-2^18 elements,
// half of them of no round length, 32-8192 candidates, j 1, 2, 4, k_mult 2-8, up to 160 MiB; every width of load): off by
// 10 % in the root mean square.  Among those calls, the choice by these estimates was 2.2 % slower than the best of two kernels
// and one with each width; the rules of size with the usual width, which stood before, are 16 %.  (float32 [859, 2048]
// k=64 j=4 k_mult=2 29.1 us by the rules, 10.1 with one column a lane; [1053, 19352] k=152 j=1 k_mult=2 35.5 in two kernels, 21.4
// in one; fp16 [2048, 8192] k=100 j=2 k_mult=4 37.5 in two kernels, 17.3 in one.)
double estimate(const Plan& pl, int64_t rows, int64_t n, int j, int es) {
  constexpr double kBytes = 5.2e6;                                      // per us
  constexpr double kLaunch = 1.45, kTrip = 0.14, kShare = 0.51;         // us; kShare: a SIMD's wave beside others
  constexpr double kLoad = 0.0225, kPush = 0.0128, kPushEntry = 0.0056; // us per sub-row, column, entry: 4-byte elements
  constexpr double kLoad2 = 0.0206, kPush2 = 0.0142, kPushEntry2 = 0.003;  // ... 2-byte elements
  constexpr double kChain = 2.32, kChainWave = 0.081, kChainEntry = 0.298, kFoldEntry = 0.002;
  const int entries = pl.vec * j;  // of a lane
  const double run = (double)pl.full_rows / pl.split;
  const int loads = es == 2 ? (entries <= 8 ? 8 : 4) : (j <= 2 ? 8 : 4);  // in flight
  const double sub_row = es == 2 ? kLoad2 + pl.vec * (kPush2 + kPushEntry2 * j) : kLoad + pl.vec * (kPush + kPushEntry * j);
  // workgroups a CU holds: by registers (waves per SIMD) and by LDS, the kernel's own 5.6 KB included
  const int waves_per_simd = es == 4 && pl.vec == 4 ? (j == 1 ? 5 : 4) : 8;
  const int by_waves = waves_per_simd * 4 / (int)pl.waves, by_lds = (int)(160 * 1024 / (pl.lds_bytes + 5600));
  const double held = by_waves < by_lds ? by_waves : by_lds;
  const double rounds = (double)rows > 256 * held ? (double)rows / (256 * held) : 1.0;
  const double on_cu = std::ceil((double)rows / 256);
  const double on_simd = pl.waves * (on_cu < held ? on_cu : held) / 4;
  const double share = on_simd > 1 ? on_simd * kShare : kShare;
  const double memory = (double)rows * (double)n * es / kBytes;
  const double issue = run * sub_row * (share > 1 ? share : 1.0) * rounds;
  const double trips = kTrip * (run > loads ? run / loads : 1.0) * rounds;
  return kLaunch + std::sqrt(memory * memory + issue * issue + trips * trips) +
         rounds * (kChain + kChainWave * pl.waves + kChainEntry * entries + kFoldEntry * (pl.split - 1) * entries);
}
}  // namespace

Plan make_plan(int64_t rows, int64_t n, int64_t k0, int j, int64_t k, int layout, int dtype, bool aligned) {
  if (layout == ATK_BALANCED) return plan_short_buckets(rows, n, k0, j, k, dtype);
  Plan pl{};
  pl.ok = false;
  const int es = elem_bytes(dtype);
  // (a padded row is never reduced further: its callers keep every bucket)
  if (layout != ATK_INTERLEAVED || es == 0) return pl;
  pl = plan_interleaved(rows, n, k0, j, k, dtype, aligned, stream::full_vec(es), true);
  if ((es != 2 && es != 4) || n * es > kEstimatedRow || k0 > kEstimatedCandidates || (pl.ok && !pl.in_registers)) return pl;
  // the register kernel with every width of load that it takes here
  Plan best = pl;
  double least = pl.ok ? estimate(pl, rows, n, j, es)
                       : kOneKernelShare * stream::estimate_two_kernels(rows, n, k0, j, dtype);
  for (int vec = stream::full_vec(es) / (es == 2 ? 2 : 1); vec >= 4 / es; vec /= 2) {
    if (pl.ok && vec == pl.vec) continue;
    const Plan other = plan_interleaved(rows, n, k0, j, k, dtype, aligned, vec, false);
    if (!other.ok || !other.in_registers || !other.pos16 || other.packed != (es == 2)) continue;
    // Few rows off 16 bytes whose sub-rows leave more than half of a wave's lanes idle stay with two kernels: short ones
    // would gain (fp32 [22, 3603] b=24 j=4 9.0 -> 5.6 us), long ones lose many times over, and of 40 such calls the
    // estimate is off most (fp16 [14, 15031] b=40 j=2 7.7 -> 8.9).
    if (!pl.ok && !aligned && rows < kMinRows && k0 / j * 2 < (int64_t)stream::kWave * vec) continue;
    if (rows > 0xffffffffll / (64 * (int64_t)other.waves)) continue;  // (a launch's threads are counted in 32 bits)
    const double us = estimate(other, rows, n, j, es);
    if (us < least) { best = other; least = us; }
  }
  return best;
}

}  // namespace fused

bool rows_on_load_width(const void* x, int64_t row_stride, int dtype) {
  const int es = elem_bytes(dtype);
  return es && (uintptr_t)x % 16 == 0 && row_stride % stream::full_vec(es) == 0;
}

namespace {
// Rows may start at any element (rows of odd length do, and views): the 16-byte loads take such addresses.
// The plans of a thread's last shapes are kept: every call asks for its plan, and a program repeats few shapes.
fused::Plan plan_for(const void* x, int64_t rows, int64_t n, int64_t row_stride, int64_t k0, int j, int64_t k,
                     int layout, int dtype) {
  struct Made {
    int64_t rows, n, k0, k;  // rows == 0: nothing made yet (such calls have no plan)
    int j, layout, dtype, aligned;
    fused::Plan plan;
  };
  constexpr uint64_t kMade = 16;
  static thread_local Made made[kMade];
  const int aligned = rows_on_load_width(x, row_stride, dtype) ? 1 : 0;
  const uint64_t h = ((uint64_t)rows * 31 + (uint64_t)n) * 31 + (uint64_t)k0 * 7 + (uint64_t)k;
  Made& m = made[(h ^ (h >> 17)) % kMade];
  if (rows <= 0 || m.rows != rows || m.n != n || m.k0 != k0 || m.k != k || m.j != j || m.layout != layout ||
      m.dtype != dtype || m.aligned != aligned)
    m = Made{rows, n, k0, k, j, layout, dtype, aligned, fused::make_plan(rows, n, k0, j, k, layout, dtype, aligned != 0)};
  return m.plan;
}
}  // namespace

bool fused_row_taken_by_size(const void* x, int64_t rows, int64_t n, int64_t row_stride, int64_t k0, int j, int64_t k,
                             int layout, int dtype) {
  return fused::taken_by_size(rows, n, k0, j, k, layout, dtype, rows_on_load_width(x, row_stride, dtype));
}

bool fused_row_takes(const void* x, int64_t rows, int64_t n, int64_t row_stride, int64_t k0, int j, int64_t k,
                     int layout, int dtype) {
  return plan_for(x, rows, n, row_stride, k0, j, k, layout, dtype).ok;
}

bool describe_fused_row(const void* x, int64_t rows, int64_t n, int64_t row_stride, int64_t k0, int j, int64_t k,
                        int layout, int dtype, std::string& out) {
  const fused::Plan pl = plan_for(x, rows, n, row_stride, k0, j, k, layout, dtype);
  if (!pl.ok) return false;
  out += std::string(pl.in_registers ? "fused_regs_kernel<" : "fused_row_kernel<") + dtype_name(dtype) + ", J=" +
         std::to_string(j) + ", V=" + std::to_string(pl.vec) + ", pos" + (pl.pos16 ? "16" : "32") +
         ", PACKED=" + (pl.packed ? "1" : "0") + "> grid=" + std::to_string(rows) + " block=" +
         std::to_string(64 * pl.waves) + " tiles=" + std::to_string(pl.tiles) + " split=" + std::to_string(pl.split) +
         " lds=" + std::to_string(pl.lds_bytes) + (pl.in_registers && pl.staged ? (pl.past_cache ? " staged past-cache" : " staged") : "") +
         (pl.contig ? " short contiguous buckets" : "");
  return true;
}

int launch_fused_row(const void* x, int64_t rows, int64_t n, int64_t row_stride, int64_t k0, int j,
                     int64_t k, int layout, int dtype, void* values, IndexOut indices, hipStream_t stream,
                     bool* handled) {
  const fused::Plan pl = plan_for(x, rows, n, row_stride, k0, j, k, layout, dtype);
  *handled = pl.ok;
  if (!pl.ok) return ATK_OK;
  int rc = ATK_ERR_DTYPE;
  ATK_DTYPE_SWITCH(dtype, E, rc = ATK_ERR_DTYPE,
                   rc = fused::launch_typed<E>(pl, x, rows, row_stride, k0, j, k, values, indices, stream));
  return rc;
}

}  // namespace atk
