// Host-side planning and dispatch of the streaming stage-1 kernels.
#include <cmath>

#include "stage1_stream.h"

namespace atk {
namespace stream {

namespace {
inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Waves wanted in the grid before a row is cut into slabs: one per SIMD of the
// 256 CUs x 4 SIMDs (each keeps 8 KiB of loads in flight).
constexpr int64_t kTargetWaves = 1024;
constexpr int64_t kCus = 256;
// Fewest bytes a wave reads, and most bytes of partial queues, of slabs that are cut to have a workgroup on every CU.
constexpr int64_t kWaveBytes = 8 << 10, kRaisedBytes = 2 << 20;
// Most partial queues of a row whose merge selects, with slabs that are cut to have a workgroup on every CU.
constexpr int64_t kRaisedSelectQueues = 4096;
// Workgroups from which calls of up to kRaisedEnoughBytes are left as they are with 16-byte loads (see plan_with).
constexpr int64_t kRaisedEnough = 96, kRaisedEnoughBytes = 32 << 20;
// Bytes of which a slab that is cut must not be nearly a multiple (4-byte elements, one-element loads).
constexpr int64_t kStep = 128 << 10;
// Partial queues of a row above which slabs of one-element loads are not cut to have the merge select.
constexpr int64_t kCutSelectQueues = 8192;
// How much longer a slab may get to have no more workgroups than CUs.
constexpr double kLonger = 1.34, kLongerOneByte = 1.17;
// Sub-rows worth giving to one wave before a row is also cut into slabs.
constexpr int64_t kSlabRun = 16;
// Fewest workgroups of a launch whose results take the trip through LDS.
constexpr int64_t kTransposeGroups = 2048;
// Sub-rows a wave keeps when a row is cut only to put a second wave on every SIMD.
constexpr int64_t kLongRun = 64;
// Fewest sub-rows a wave scans when several share a tile: with runs of 2 the
// hand-over costs more than the scan (measured at 16 sub-rows: 4 waves x 4 beat
// 8 x 2 by 25-45 %).
constexpr int64_t kMinRun = 4;
// Fewest sub-rows per wave for which a workgroup may take more LDS than kMergeLdsLimit.
constexpr int64_t kLongWaveRun = 16;
// Buckets at least this long are folded when they do not fill a column tile
// (measured down to 8: fp32 [32768, 1024] with 16 buckets 104 -> 22 us, bf16
// 193 -> 32 us; [65536, 256] with 16 buckets 70 -> 31 us).
constexpr int64_t kFoldMinLength = 8;
// Candidates, and entries of all their partial queues, up to which the merge of a row takes the second
// stage along.  One workgroup reads these entries: up to 16384 it saves 1-5 us in rows of 2^20 to 2^24, beyond
// that it wins and loses (fp32 [1, 2^22] k=64 j=4 k_mult=2, 32768 entries, 27.4 -> 24.1 us; k=500 j=2 k_mult=4,
// 64000 entries, 19.9 -> 26.5; k=256 j=4 k_mult=4, 262144, 30.7 -> 58.0).
constexpr int64_t kMergeSelectMax = 2048, kMergeSelectEntries = 16384;
// Calls of more bytes than this (kLargeEight: of eight-byte elements) take one-element loads only where their estimate
// is that share of the other (see estimate): what counts there is memory, of which the estimate sees little.
// 150 calls of 128 to 640 MiB: 1.4 % slower than the better one in the mean, 16-byte loads throughout 3.4 %,
// one-element loads 27 % (fp16 [136579, 2311] b=4 j=4 679 us wide, 425 narrow, fp32 [17703, 2921] b=66 j=4 112 and 82).
constexpr int64_t kLargeBytes = 128 << 20, kLargeEight = 48 << 20;
constexpr double kLargeShare = 0.95;
// Buckets from this length on are folded whatever the fold.
constexpr int64_t kFoldAnyLength = 128;

// The plan with 16-byte loads (`wide`) or with one-element loads.  `second_stage`: behind the candidates (without
// one, rows are cut into as many slabs or more: the bound of the workspace).
Plan plan_with(int64_t rows, int64_t n, int64_t k0, int j, int layout, int dtype, bool wide, bool second_stage) {
  Plan pl{};
  pl.ok = false;
  if (layout != ATK_INTERLEAVED && layout != ATK_INTERLEAVED_PADDED) return pl;
  if (rows <= 0 || k0 <= 0 || j < 1 || j > 4 || k0 % j) return pl;
  const int es = elem_bytes(dtype);
  if (!es) return pl;
  const int64_t b = k0 / j;
  const int64_t length = n / b;  // elements every bucket has
  if (length < j || length > 0xfffffffell || b > 0x7fffffffll) return pl;
  const int vf = full_vec(es);

  // Few buckets: scan `fold` sub-rows side by side so that the lanes of a wave
  // are all busy (the largest fold that fits one column tile, keeps 16-byte
  // loads possible and leaves every scanned column j elements); the scanning
  // workgroup puts each bucket back together.
  int64_t fold = 1;
  if (length >= kFoldMinLength) {
    const int v = wide ? vf : 1;
    int64_t f = (int64_t)kWave * v / b;
    while (f > 1 && n / (b * f) < j) --f;
    // whole vectors when that costs at most a quarter of the lanes
    int64_t whole = f;
    while (whole > 1 && (b * whole) % v != 0) --whole;
    if (whole > 1 && whole * 4 >= f * 3) f = whole;
    // short buckets: only when at least three lanes in four would idle (a fold of
    // two costs more in the merge than it gains: [128, 4096] with 128 buckets, j = 4, +23 %)
    if (f > 1 && (length >= kFoldAnyLength || f >= 4)) fold = f;
  }
  pl.fold = (uint32_t)fold;
  const int64_t width = b * fold;
  pl.width = width;
  const int64_t full = n / width;
  pl.full_rows = (uint32_t)full;
  pl.rem = (uint32_t)(n - full * width);
  pl.pad_tail = layout == ATK_INTERLEAVED_PADDED ? 1u : 0u;
  pl.vec = wide && width >= vf ? vf : 1;
  pl.packed = ((dtype == ATK_F16 || dtype == ATK_BF16 || dtype == ATK_I16) && full <= kPackedMaxSubRow) ||
              ((dtype == ATK_U8 || dtype == ATK_I8) && full <= kByteMaxSubRow);

  const int64_t tile_cols = (int64_t)kWave * pl.vec;
  pl.col_tiles = (uint32_t)((width + tile_cols - 1) / tile_cols);

  // Waves per workgroup.  Wave 0's serial work per column is its own run,
  // full/w pushes, plus (w-1)*j pushes to fold the other waves' queues.  Take
  // the largest w within 30 % of the cheapest (short-lived waves keep more of
  // the HBM bandwidth: measured, 8 waves x 4 sub-rows beats 4 x 8 at the
  // headline shape), with every run at least max(j, 4) long and the LDS
  // hand-over within its budget.
  const int entry_bytes = pl.packed ? 4 : (es > 4 ? 8 : 4) + 4;
  int64_t cost[4] = {full, 0, 0, 0};
  int cands = 1;
  for (int cand = 2; cand <= 8; cand *= 2, ++cands) {
    const size_t hand = merge_lds_bytes(pl.vec, j, cand, entry_bytes);
    if (full / cand < (j > kMinRun ? j : kMinRun) || hand > merge_lds_limit(entry_bytes)) break;
    // Beyond the usual budget (packed queues of four entries, eight waves: 56 KiB, two workgroups
    // per CU) only for long runs.  Measured, fp16 [256, 2^20], j = 4: columns of 256 sub-rows
    // 125 -> 117 us, [1, 2^26] k = 16384 k_mult = 2 63 -> 47 us, but columns of 64 (runs of 8) 150 -> 162 us.
    if (hand > kMergeLdsLimit && full / cand < kLongWaveRun) break;
    cost[cands] = full / cand + (int64_t)(cand - 1) * j;
  }
  int64_t best = cost[0];
  for (int i = 1; i < cands; ++i) best = cost[i] < best ? cost[i] : best;
  int w = 1;
  for (int i = 0; i < cands; ++i)
    if (cost[i] * 10 <= best * 13) w = 1 << i;
  pl.waves = w;

  // Slabs: only when the grid would still be small and the runs are long.
  // Once a row is cut at all (the merge launch is then paid for anyway), short
  // queues (j <= 2, whose merge is cheap) are cut for twice as many waves:
  // measured 41 -> 28 us on fp32 [2, 2^24] with 4096 buckets, 57 -> 52 us on
  // [1, 2^26] with 16384 buckets at j = 2; j = 4 loses a little.
  pl.slabs = 1;
  const int64_t waves = rows * pl.col_tiles * w;
  const int64_t most = full / (w * kSlabRun);
  if (waves < kTargetWaves && most > 1) {
    const int64_t target = j <= 2 ? 2 * kTargetWaves : kTargetWaves;
    int64_t slabs = (target + waves - 1) / waves;
    if (slabs > most) slabs = most;
    pl.slabs = (uint32_t)slabs;
  }
  // Elements of one or two bytes cost twice or more the instructions per byte
  // loaded; a second wave per SIMD hides them, while every wave still has a
  // long run (measured on fp16 [128, 2^20] with 16 to 256 buckets: 87 -> 56 us
  // at j = 1, 120 -> 89 us at j = 4; with shorter runs the merge eats the gain).
  if (es <= 2) {
    int64_t slabs = (2 * kTargetWaves + waves - 1) / waves;
    const int64_t longest = full / (w * kLongRun);
    if (slabs > longest) slabs = longest;
    if (slabs > (int64_t)pl.slabs) pl.slabs = (uint32_t)slabs;
  }
  // A launch of more workgroups than CUs gives some CUs twice the work, with the others waiting: down to no more
  // workgroups than CUs, in fewer and longer slabs.  How much longer they may get lies with how well a CU's second
  // workgroup hides behind the first.  Time cut over time as asked, 960 launches (all types, 1-200 rows of 2^13 to 2^26):
  //   eight waves with 16-byte loads, or of eight-byte elements, each a CU's worth of instructions: 236 launches 0.80, of
  //     them slabs a third to a half longer (three slabs to two: 172 to 200 workgroups) 51 launches 0.87, none over
  //     1.03 (fp32 [42, 632917] k=484 j=2 294 -> 252 workgroups 30.1 -> 24.6 us, bf16 [89, 266666] k=23 267 -> 178 18.8 -> 15.8);
  //   four waves: up to a third longer 59 launches 0.90 (one over 1.05); beyond, of 2-byte elements with three and four of
  //     a bucket 66 launches 0.95, with two 35 launches 1.06 (fp16 [2, 45395679] b=75 j=2, 512 -> 256 workgroups, 51.0 ->
  //     59.1 us) and of 4-byte ones 30 launches 1.26: those keep two workgroups a CU, but no more (513 -> 510, 20 launches 0.79);
  //   one-element loads, of the calls that are not faster with wider ones: 2- and 4-byte elements up to a third longer 95
  //     launches 0.93, beyond 28 launches 0.99 and up to 1.18; one byte up to a sixth longer 19 launches 0.94, beyond 20
  //     launches 1.02 and up to 1.11.  Of 4-byte elements not where a slab would get up to a twentieth longer and 1 to 4 KiB
  //     off a multiple of 128 KiB, as slabs of a 255th of 2^k elements are (read in step from the same parts of memory, it
  //     seems): 109 launches 1.15, 104 of them over 1.03, against 599 launches 0.98 with four over 1.03 at other lengths
  //     (int32 [3, 2^23] k=64 j=2, 258 -> 255 workgroups, 25.6 -> 27.2 us).
  // (With one slab left, and no merge, some lose a third.)  One-element loads keep their slabs where fewer of them would
  // have the merge select, of a row with more than kCutSelectQueues: 15 launches 1.10 (bf16 [1, 3212725] k=24 k_mult=8, 258 ->
  // 255 workgroups and 16320 queues in one of them, 12.7 -> 15.9 us; with fewer queues, or 16-byte loads, 18 launches 0.90).
  const int64_t per_slab = rows * pl.col_tiles;  // workgroups
  const uint32_t slabs_asked = pl.slabs;
  const int64_t in_one_turn = kCus / per_slab;  // slabs
  const bool may_select = second_stage && es <= 4 && k0 <= kMergeSelectMax;
  const bool long_select = pl.vec == 1 && may_select && k0 * (int64_t)pl.slabs > kMergeSelectEntries &&
                           k0 * in_one_turn <= kMergeSelectEntries && b * in_one_turn > kCutSelectQueues;
  const int64_t off_step = in_one_turn > 0 ? full / in_one_turn * width * es % kStep : 0;
  const bool in_step = es == 4 && pl.vec == 1 && 20 * (int64_t)pl.slabs <= 21 * in_one_turn &&
                       ((off_step >= 1024 && off_step <= 4096) ||
                        (kStep - off_step >= 1024 && kStep - off_step <= 4096));
  if (in_one_turn > 1 && (int64_t)pl.slabs > in_one_turn && !long_select && !in_step) {
    const double longer = (double)pl.slabs / (double)in_one_turn;
    const bool whole_cu = es == 8 || (pl.vec > 1 && w == 8), long_queues = w < 8 && es <= 2 && j >= 3;
    if (whole_cu || long_queues || longer <= (es == 1 ? kLongerOneByte : kLonger))
      pl.slabs = (uint32_t)in_one_turn;
    else if (w < 8 && (int64_t)pl.slabs > 2 * kCus / per_slab)
      pl.slabs = (uint32_t)(2 * kCus / per_slab);
  }
  // CUs left idle while every wave has a long way to go: up to a workgroup each, with what a wave reads at kWaveBytes or
  // more, and the second stage left in the merge where it is (132 -> 252 workgroups fp16 [7, 2^22] k=32 j=4 k_mult=2 28.8 ->
  // 24.0 us, 144 -> 252 bf16 [9, 2^22] k=512 j=4 32.9 -> 24.7, fp32 [2, 2^23] k=1024 j=4 k_mult=4 128 -> 256 37.2 -> 29.3; with 2-4 KB
  // a wave, f16 [3, 346950] k=324 j=2, 7.7 -> 8.3).  Small partial queues only: the workspace stays within what the call
  // that cannot allocate has taken.  One workgroup a row reads them all where the merge selects: up to
  // kRaisedSelectQueues (107 launches up to there 0.92, of one to three elements a bucket and more queues 29 launches
  // 1.03: bf16 [1, 11732747] k=16 k_mult=2, 179 -> 256 slabs, 14.4 -> 17.1 us).
  // Not with 16-byte loads from kRaisedEnough workgroups on in calls of up to kRaisedEnoughBytes, which have the memory
  // busy for a few microseconds as they are: of 4-byte elements 310 launches 1.01 (83 over 1.03: fp32 [1, 3091105] k=24 j=4
  // 191 -> 256 workgroups 14.5 -> 20.4 us, [8, 2^20] k=72 j=3 k_mult=2 128 -> 256 19.1 -> 22.0), of 1- and 2-byte ones raised by less
  // than half 242 launches 1.00 (by more 547 launches 0.96); all others 2647 launches 0.94.
  if (pl.slabs > 1 && pl.slabs * per_slab < kCus && rows * k0 * (es + 8) <= kRaisedBytes) {
    int64_t slabs = in_one_turn;
    const int64_t by_wave = full * kWave * pl.vec * es / (w * kWaveBytes), by_queues = kRaisedBytes / (rows * k0 * (es + 4));
    if (slabs > by_wave) slabs = by_wave;
    if (slabs > by_queues) slabs = by_queues;
    if (k0 <= kMergeSelectMax && k0 * (int64_t)pl.slabs <= kMergeSelectEntries) {
      const int64_t most_queues = second_stage && es <= 4 ? kRaisedSelectQueues : kMergeSelectEntries / j;
      if (slabs > most_queues / b) slabs = most_queues / b;
    }
    const bool enough = pl.vec > 1 && pl.slabs * per_slab >= kRaisedEnough && rows * n * es <= kRaisedEnoughBytes &&
                        (es == 4 || (es <= 2 && 2 * slabs < 3 * (int64_t)pl.slabs));
    if (slabs > (int64_t)pl.slabs && !enough) pl.slabs = (uint32_t)slabs;
  }
  pl.slab_len = (uint32_t)(full / pl.slabs);
  // every wave scans exactly 4 or 8 sub-rows: straight-line kernels exist for that
  pl.run = 0;
  if (pl.vec > 1 && pl.slabs == 1 && full % pl.waves == 0) {
    const int64_t run = full / pl.waves;
    if ((run == 4 || run == 8) && run >= j) pl.run = (int)run;
  }
  // the slabs' queues (one per bucket: a workgroup merges the folded columns of
  // its slab itself) go to the workspace and the merge kernel follows
  pl.merge = pl.slabs > 1;
  if (pl.merge) {
    // (sized for the slabs as first asked for where they are more: the figure callers size their buffers by stays)
    const size_t entries = (size_t)rows * (pl.slabs > slabs_asked ? pl.slabs : slabs_asked) * (size_t)b * (size_t)j;
    pl.part_values_off = 0;
    pl.part_pos_off = align_up(entries * es, 256);
    pl.ws_bytes = pl.part_pos_off + align_up(entries * sizeof(uint32_t), 256);
  }
  // Results through LDS in whole-wave stores (emit_transposed): when a lane's stretch of
  // the output is long (its indices 128 bytes or more) or its elements short, the launch
  // has workgroups by the thousand, and a workgroup writes at least an eighth of what it reads
  // (at a twelfth, fp16 [256, 2^20] k=16384: j=2 112.6 -> 115.1 us, j=4 118.2 -> 115.2 us, j=1 104.9 -> 102.5 us).
  pl.wave_stores = false;
  if (pl.vec > 1 && width % pl.vec == 0 && es <= 4 && !pl.merge && pl.fold == 1) {
    const int64_t entries = (int64_t)pl.vec * j;  // of a lane
    const bool whole_pieces = entries % 4 == 0 && entries % (16 / es) == 0 && j != 3;  // (Transposed::available)
    const int64_t groups = rows * (int64_t)pl.col_tiles;
    const int64_t in_bytes = full * kWave * pl.vec * es, out_bytes = kWave * entries * (es + 8);
    pl.wave_stores = whole_pieces && (entries * 8 >= 128 || es < 4) && groups >= kTransposeGroups &&
                     out_bytes * 8 >= in_bytes;
  }
  pl.ok = true;
  return pl;
}
}  // namespace

namespace {
// Estimated microseconds of a call, for the choice between 16-byte and one-element loads where both are possible, and
// for that between these kernels and the one-kernel path.  With one-element loads a lane owns one column instead of two to
// eight: more workgroups, in rows cut into slabs fewer partial queues, and a shorter end of every workgroup, against fewer
// bytes in flight, a load for every element and more waves to launch.  What a plan takes is
//   the scan: memory, instructions, the launch of the waves and the round trips of a wave's loads, which overlap
//     (the root of the sum of their squares);
//   a workgroup's end: the other waves' queues folded into the leading wave's, folded columns put together, and a
//     lane's entries written, by one wave, next to the ends and scans of the workgroups that the CU holds with it;
//   the launches behind it: the merge of the slabs, with or without the second stage, or a select of its own.
// The scan's and the end's constants are a least-squares fit to 2070 calls timed both ways (all nine types, 1-20000 rows
// of 37 to 2^24 elements, up to 128 MiB, j 1-4, k_mult 1-8, half of them few rows, most of them off 16 bytes); those of the
// launches behind them to 18500 launches of 8900 calls with the merge and the selects as they are (four partial queues
// a thread; up to 512 MiB): off by 16 % in the root mean square.  On 3000 other calls the choice is 1.1 % slower than the better
// one of the two in the geometric mean (10 % and more in one call of 26), 16-byte loads throughout 11 %, one-element loads
// throughout 11 %: fp32 [3, 2^21] b=128 j=4 k_mult=8 30.2 us wide, 17.9 narrow, int8
// [1, 172601] b=1310 j=4 8.3 and 4.0, uint8 [39, 152696] b=201 j=4 14.5 and 8.7, fp64 [2, 310384] b=799 j=4 12.3 and
// 10.8, fp16 [168, 298475] b=544 j=4 67.9 and 42.1, but int8 [51, 507136] b=2391 j=3 11.2 and 16.9, fp16 [21, 1426304]
// b=8338 j=2 16.8 and 23.5.
double estimate(const Plan& pl, int64_t rows, int64_t n, int64_t k0, int j, int dtype, int64_t select_bound) {
  constexpr double kBytes = 5.1e6, kSlowFolds = 1.2, kWaveLaunch = 3.6e-4;  // per us; us
  constexpr double kTrip = 0.34, kLoad = 0.0087;          // us: a batch of loads, issuing one (a wave per SIMD)
  constexpr double kHandOver = 0.008, kEntry = 0.067;     // us an entry of a lane: handed over, written
  constexpr double kFold = 0.4, kFoldStep = 0.039;
  constexpr double kLaunch = 2.42, kMerge = 2.49, kMergeStep = 0.107, kMergeSelect = 4.3, kMergeSelectEntry = 3.6e-4;
  constexpr double kRank = 3.22, kRankEntry = 3.76e-3, kOneLaunch = 5.96, kOneLaunchEntry = 2.7e-4, kSelect = 6.49,
                   kSelectEntry = 1.24e-3;
  constexpr double kLastTurn = 0.37;
  struct Push { double column, entry; };                  // us per sub-row (a wave per SIMD): a column, and per entry kept
  const int es = elem_bytes(dtype);
  const Push push = es == 1 ? Push{0.0067, 0.001} : es == 8 ? Push{0.0026, 0.029} : es == 4 ? Push{0.021, 0.0036}
                    : pl.packed ? Push{0.019, 0.0} : Push{0.011, 0.0068};
  const int loads = deep_loads_for_short_columns(dtype, j, pl.vec, pl.packed, pl.run, pl.full_rows)
                        ? 8
                        : loads_in_flight(dtype, j, pl.vec, pl.packed);
  const double b = (double)(k0 / j), groups = (double)rows * pl.slabs * pl.col_tiles, waves = groups * pl.waves;
  const double run = (double)pl.full_rows / pl.slabs / pl.waves;  // sub-rows a wave scans
  const double bytes = (double)rows * (double)n * es + (double)rows * pl.slabs * (double)k0 * (es + 8);
  // folded sub-rows of four-byte elements in rows cut into slabs: short queues wait for memory longer with 16-byte loads
  // (20 such calls of 12 MiB and more: 9 % slower than one-element loads, where this estimate saw 2 % the other way)
  const bool slow_folds = es == 4 && j <= 2 && pl.vec > 1 && pl.fold > 1 && pl.slabs > 1;
  const double memory = bytes / kBytes * (slow_folds ? kSlowFolds : 1.0), launch = waves * kWaveLaunch;
  const double trips = kTrip * (1 + (run > loads ? run / loads : 1.0));
  // (slabs that were left with a few workgroups more than CUs: the CUs with one more take part of a turn longer)
  double turns = groups / kCus;
  if (pl.merge && pl.vec == 1 && es < 8 && turns > 1 && turns <= 4) turns += kLastTurn * (std::ceil(turns) - turns);
  const double on_simd = turns * pl.waves / 4;
  const double pushes = run * (kLoad + pl.vec * (push.column + j * push.entry)) * (on_simd > 1 ? on_simd : 1.0);
  double us = kLaunch + std::sqrt(memory * memory + launch * launch + trips * trips + pushes * pushes);
  double end = (kHandOver * (pl.waves - 1) + kEntry) * j * pl.vec;
  if (pl.fold > 1) {
    uint32_t at_once = kWave;  // buckets (see fold_columns)
    while (at_once > 1 && at_once / 2 >= b) at_once /= 2;
    const double shares = (double)kWave / at_once;
    end += kFold + kFoldStep * j * std::ceil(pl.fold / shares) * std::ceil(b / at_once);
  }
  // workgroups that a CU holds: by their LDS, and sixteen waves with 16-byte loads, twice as many with one-element loads
  const int entry_bytes = pl.packed ? 4 : (es > 4 ? 8 : 4) + 4;
  const double hand = (double)merge_lds_bytes(pl.vec, j, pl.waves, entry_bytes);
  const double words = (double)kWave * pl.vec * j * (es == 8 ? 16 : 8);
  const double by_lds = 160 * 1024 / (hand > words ? hand : words), by_waves = (pl.vec > 1 ? 16.0 : 32.0) / pl.waves;
  const double held = by_lds < by_waves ? (by_lds > 1 ? by_lds : 1.0) : by_waves;
  us += end * (groups > 256 * held ? groups / (256 * held) : 1.0);
  const bool selects = select_bound > 0 && selects_in_merge(pl, k0, select_bound, dtype);
  if (selects) {
    us += kMergeSelect + kMergeSelectEntry * (double)pl.slabs * (double)k0;
  } else if (pl.merge) {
    uint32_t at_once = kWave;  // buckets (as the launch chooses them)
    while (at_once > 1 && (at_once / 2 >= b || (int64_t)pl.slabs * at_once > kMergeQueues * kMergeThreads)) at_once /= 2;
    us += kMerge + kMergeStep * j * std::ceil((double)pl.slabs * at_once / kMergeThreads);
  }
  if (select_bound > 0 && !selects) {
    const double many = rows > kCus ? (double)rows / kCus : 1.0;
    if (rank_select_takes(rows, k0, select_bound, dtype)) us += kRank + kRankEntry * (double)k0 * many;
    else if (one_launch_select_takes(rows, k0, select_bound, dtype)) us += kOneLaunch + kOneLaunchEntry * (double)k0;
    else us += kSelect + kSelectEntry * (double)k0 * many;
  }
  return us;
}
}  // namespace

Plan make_plan(int64_t rows, int64_t n, int64_t k0, int j, int layout, int dtype, int64_t select_bound) {
  const Plan w = plan_with(rows, n, k0, j, layout, dtype, true, select_bound > 0);
  if (!w.ok || w.vec == 1) return w;
  // whole-wave stores spare the lanes' entries most of what the estimate takes for them; with half of the lanes at work
  // they stay ahead (i8 [4475, 6579] b=320 j=2 42.8 us, 56.5 with one-element loads; bf16 [10470, 6399] b=136 j=4 163 and 114)
  if (w.wave_stores && 2 * w.width >= (int64_t)w.col_tiles * kWave * w.vec) return w;
  const Plan v = plan_with(rows, n, k0, j, layout, dtype, false, select_bound > 0);
  // (a launch's threads are counted in 32 bits)
  if (!v.ok || rows * (int64_t)v.slabs * v.col_tiles > 0xffffffffll / (kWave * v.waves)) return w;
  auto us = [&](const Plan& pl) { return estimate(pl, rows, n, k0, j, dtype, select_bound); };
  const int es = elem_bytes(dtype);
  const bool large = rows * n * es > (es == 8 ? kLargeEight : kLargeBytes);
  return us(v) < us(w) * (large ? kLargeShare : 1.0) ? v : w;
}

double estimate_two_kernels(int64_t rows, int64_t n, int64_t k0, int j, int dtype) {
  const Plan pl = make_plan(rows, n, k0, j, ATK_INTERLEAVED, dtype, n);
  if (!pl.ok) return INFINITY;
  return estimate(pl, rows, n, k0, j, dtype, n);
}

bool selects_in_merge(const Plan& pl, int64_t k0, int64_t index_bound, int dtype) {
  return pl.ok && pl.merge && elem_bytes(dtype) <= 4 && index_bound <= 0xffffffffll && k0 <= kMergeSelectMax &&
         k0 * (int64_t)pl.slabs <= kMergeSelectEntries;
}

}  // namespace stream

size_t stage1_stream_workspace_bytes(int64_t rows, int64_t n, int64_t k0, int j, int layout, int dtype) {
  // (make_plan picks one of these)
  const stream::Plan a = stream::plan_with(rows, n, k0, j, layout, dtype, true, false);
  const stream::Plan u = stream::plan_with(rows, n, k0, j, layout, dtype, false, false);
  size_t need = 0;
  if (a.ok && a.ws_bytes > need) need = a.ws_bytes;
  if (u.ok && u.ws_bytes > need) need = u.ws_bytes;
  return need;
}

bool describe_stage1_stream(int64_t rows, int64_t n, int64_t k0, int j, int64_t k, int layout,
                            int dtype, int64_t index_bound, bool* selected, std::string& out) {
  *selected = false;
  const stream::Plan pl = stream::make_plan(rows, n, k0, j, layout, dtype, k < k0 ? index_bound : 0);
  if (!pl.ok) return false;
  const int loads = stream::deep_loads_for_short_columns(dtype, j, pl.vec, pl.packed, pl.run, pl.full_rows)
                        ? 8
                        : stream::loads_in_flight(dtype, j, pl.vec, pl.packed);
  out += "stream_kernel<" + std::string(dtype_name(dtype)) + ", J=" + std::to_string(j) +
         ", V=" + std::to_string(pl.vec) + ", W=" + std::to_string(pl.waves) + ", U=" + std::to_string(loads) +
         ", RUN=" + std::to_string(pl.run) + ", PACKED=" + (pl.packed ? "1" : "0") + "> grid=" +
         std::to_string(rows * (int64_t)pl.slabs * pl.col_tiles) + " block=" + std::to_string(64 * pl.waves) +
         " fold=" + std::to_string(pl.fold) + " slabs=" + std::to_string(pl.slabs) +
         (pl.wave_stores ? " wave-stores" : "");
  if (pl.merge) {
    *selected = k < k0 && stream::selects_in_merge(pl, k0, index_bound, dtype);
    out += std::string(" + stream_merge_") + (*selected ? "select_" : "") + "kernel<" + dtype_name(dtype) + ", J=" +
           std::to_string(j) + ">";
  }
  return true;
}

int launch_stage1_stream(const void* x, int64_t rows, int64_t n, int64_t row_stride, int64_t k0, int j,
                         int layout, int dtype, void* values, IndexOut indices, void* ws,
                         size_t ws_bytes, hipStream_t stream, bool* handled, KeyRangeOut* ranges, SelectOut* last) {
  const stream::Plan pl = stream::make_plan(rows, n, k0, j, layout, dtype, last != nullptr ? last->index_bound : 0);
  *handled = pl.ok;
  if (!pl.ok) return ATK_OK;
  if (pl.ws_bytes && (!ws || ws_bytes < pl.ws_bytes || (uintptr_t)ws % 16 != 0)) return ATK_ERR_WORKSPACE;
  if (last != nullptr) last->wanted = stream::selects_in_merge(pl, k0, last->index_bound, dtype);
  if (last != nullptr && last->wanted) ranges = nullptr;  // (no chained select follows)
  int rc = ATK_ERR_DTYPE;
  ATK_DTYPE_SWITCH(dtype, E, rc = ATK_ERR_DTYPE,
                   rc = stream::launch_typed<E>(pl, x, rows, row_stride, j, values, indices, ws,
                                                stream, ranges, last));
  return rc;
}

}  // namespace atk
