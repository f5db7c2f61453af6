// Host-side planning and dispatch of the contiguous-layout stage-1 kernel.
#include "stage1_contig.h"

namespace atk {
namespace contig {

namespace {
// Workgroups wanted in the grid before long buckets are left whole.
constexpr int64_t kTargetGroups = 1024;
// split_bucket_kernel: buckets of a launch from which on a wave may take more than kFewTurns turns
// at its bucket, and from which on buckets shorter than one piece go there.
constexpr int64_t kManyWaves = 512, kFewTurns = 8, kManyBuckets = 16384;
// The same for queues of three or four entries of four bytes, from kFewTurns turns on.
constexpr int64_t kManyLong = 1024;
// Workgroups whose threads a launch can count (in 32 bits); contig_kernel gives a short bucket fewer lanes.
constexpr int64_t kMostGroups = 0xffffffffll / kThreads;
}  // namespace

Plan make_plan(int64_t rows, int64_t n, int64_t k0, int j, int layout, int dtype, bool aligned) {
  Plan pl{};
  pl.ok = false;
  if (layout != ATK_BALANCED && layout != ATK_CEIL_CHUNK) return pl;
  if (rows <= 0 || n <= 0 || k0 <= 0 || j < 1 || j > 4 || k0 % j) return pl;
  const int es = elem_bytes(dtype);
  if (!es) return pl;
  const int64_t b = k0 / j;
  const int64_t m = layout == ATK_BALANCED ? n / b : (n + b - 1) / b;
  const int64_t r = layout == ATK_BALANCED ? n - m * b : 0;
  // every bucket holds at least j elements; positions fit 32 bits
  if (m < j || b > 0x7fffffffll || (double)b * (double)m + (double)r > 4294967294.0) return pl;
  const int64_t longest = m + (r > 0 ? 1 : 0);
  const int64_t piece = max_piece(es);

  Geom& g = pl.geom;
  g.n = n;
  g.b = (uint32_t)b;
  g.m = (uint32_t)m;
  g.r = (uint32_t)r;
  uint32_t lg = 0;
  while (lg < 8 && ((longest + (1ll << lg) - 1) >> lg) > piece) ++lg;
  // Few buckets: more threads per bucket (shorter pieces, more merge rounds)
  // as long as one workgroup still covers all of them and a piece keeps at
  // least four elements, so that the threads of the workgroup all scan.
  while (lg < 8 && (int64_t)(kThreads >> (lg + 1)) >= b && (m >> (lg + 1)) >= (j > 4 ? j : 4)) ++lg;
  g.pieces_log2 = lg;
  const int64_t per_thread = (longest + (1ll << lg) - 1) >> lg;
  if (per_thread > piece) {  // lg == 8: a workgroup per bucket, in chunks of 256 pieces
    g.chunks = (uint32_t)((longest + kThreads * piece - 1) / (kThreads * piece));
    g.trip = (uint32_t)piece;
  } else {
    g.chunks = 1;
    g.trip = (uint32_t)per_thread;
    g.sure = (uint32_t)(m >> lg);
  }
  const int64_t per_group = kThreads >> lg;
  g.groups = (uint32_t)((b + per_group - 1) / per_group);
  // Few rows of few very long buckets: share a bucket's chunks out over
  // workgroups (at least two chunks each, so that every workgroup starts on a
  // full chunk) until the grid has about kTargetGroups of them.
  g.slabs = 1;
  g.slab_chunks = g.chunks;
  if (g.chunks >= 4 && rows * b < kTargetGroups / 2) {
    int64_t slabs = (kTargetGroups + rows * b - 1) / (rows * b);
    if (slabs > g.chunks / 2) slabs = g.chunks / 2;
    if (slabs > 256) slabs = 256;
    g.slabs = (uint32_t)slabs;
    g.slab_chunks = g.chunks / g.slabs;
    g.groups = (uint32_t)(b * slabs);
    pl.ws_bytes = (size_t)rows * (size_t)b * (size_t)slabs * 4 * (es == 8 ? 16 : 8);
  }
  if (rows * (int64_t)g.groups > 0x7fffffffll) return pl;

  // 16-byte loads in rows off 16 bytes: they pay for elements of four bytes and more (fp32 [16, 2000003] with
  // buckets of 40 KB 51.6 -> 48.0 us; fp16 41.2 -> 43.3, and [512, 100003] k=50000 j=4 115 -> 155, where
  // the eight elements of a load are parked in LDS a word at a time)
  pl.vec = aligned || es >= 4 ? stream::full_vec(es) : 1;
  // LDS: the longest span (whole packs, one element of slack) with its padding, or the queues
  const int64_t span = (g.chunks > 1 ? kThreads * piece : per_group * longest) + 2 * pl.vec + 2;
  const size_t data_bytes = (size_t)(span + ((span >> 5) + 1) * pad_elems(es)) * es;
  const size_t list_bytes = (size_t)4 * kThreads * (es == 8 ? 16 : 8);
  pl.lds_bytes = ((data_bytes > list_bytes ? data_bytes : list_bytes) + 15) / 16 * 16;
  // scan_even: buckets of one length, whole in the span, pieces of whole 16-byte packs, sub-row
  // numbers that fit the packed entries
  const int64_t per_pack = pl.vec;  // elements of a pack
  g.fast = 0;
  if (pl.vec > 1 && es <= 4 && r == 0 && g.chunks == 1 && (m >> lg) << lg == m && (m >> lg) % per_pack == 0 &&
      (m >> lg) >= per_pack && per_pack >= j && (es != 2 || m <= (int64_t)stream::kPackedMaxSubRow)) {
    const size_t packs = (size_t)(per_group * m) / per_pack;
    const size_t even_bytes = even_offset((uint32_t)packs, (uint32_t)(per_pack * es)) + 16;
    if (even_bytes <= 64 * 1024) {
      g.fast = 1;
      if (pl.lds_bytes < even_bytes) pl.lds_bytes = (even_bytes + 15) / 16 * 16;
    }
  }
  // whole_bucket_kernel: a lane per bucket, no LDS
  g.whole = 0;
  if (pl.vec > 1 && (es == 2 || es == 4) && r == 0 && (int64_t)b * m == n && (m * es) % 16 == 0 &&
      m * es <= (int64_t)kWholeBucket) {
    g.whole = 1;
    g.slabs = 1;
    pl.ws_bytes = 0;
    pl.lds_bytes = 0;
  }
  // split_bucket_kernel: adjacent lanes share a bucket, no LDS.  (A padded row's last bucket may
  // reach past the row: not here.)  contig_kernel keeps:
  //   the even shapes, whose packs it copies and scans whole (fp32 [128, 2^20] with buckets of 256 bytes
  //   99 against 111 us, fp16 of 512 bytes 84 against 90);
  //   buckets of which more than a quarter is kept, three or four elements each (fp32 [256, 100003] k=50000 j=4
  //   68.6 against 76.2 us; with j=2 and buckets of 16 bytes 64.4 against 46.5);
  //   few buckets that a wave would need many turns for (200 of 40 KB in one row 11.9 against 13.4 us, but 800 in
  //   four rows 17.3 against 13.9), and with queues of three or four four-byte entries up to twice as many (128 of 28 KB,
  //   j=4 7.5 against 10.4 us, 512 of 50 KB 16.0 against 20.8; 1024 of 63 KB 25.1 against 25.4, 2048 of 28 KB 23.9 against 17.2);
  //   small launches of short buckets, which take the same either way (fp32 [64, 8200] k=1024 j=2 11.7 against 11.5).
  g.split = 0;
  if ((es == 2 || es == 4) && !g.whole && !g.fast && (layout == ATK_BALANCED || b * m == n) &&
      longest * es <= (int64_t)kSplitBucket && (j <= 2 || m >= 4 * j) &&
      (m * es >= (int64_t)kSplitBytes || rows * b >= kManyBuckets)) {
    uint32_t pieces_log2 = 0;
    while (((longest + (1ll << pieces_log2) - 1) >> pieces_log2) * es > (int64_t)kSplitBytes) ++pieces_log2;
    g.split_log2 = pieces_log2;
    const int64_t turns = (1ll << pieces_log2) / stream::kWave;
    const bool long_queues = es == 4 && j >= 3 && turns >= kFewTurns;
    if ((m >> pieces_log2) * es >= 16 && (turns <= kFewTurns || rows * b >= kManyWaves) &&
        (!long_queues || rows * b >= kManyLong) && bucket_groups(g, rows) <= kMostGroups) {
      g.split = 1;
      g.split_trip = (uint32_t)((longest + (1ll << pieces_log2) - 1) >> pieces_log2);
      g.slabs = 1;
      pl.ws_bytes = 0;
      pl.lds_bytes = 0;
    }
  }
  if (pl.lds_bytes > 64 * 1024) return pl;
  pl.ok = true;
  return pl;
}

}  // namespace contig

namespace {
contig::Plan plan_for(const void* x, int64_t rows, int64_t n, int64_t row_stride, int64_t k0, int j, int layout,
                      int dtype) {
  return contig::make_plan(rows, n, k0, j, layout, dtype, rows_on_load_width(x, row_stride, dtype));
}
}  // namespace

size_t stage1_contig_workspace_bytes(int64_t rows, int64_t n, int64_t k0, int j, int layout, int dtype) {
  const contig::Plan a = contig::make_plan(rows, n, k0, j, layout, dtype, true);
  const contig::Plan u = contig::make_plan(rows, n, k0, j, layout, dtype, false);
  size_t need = 0;
  if (a.ok && a.ws_bytes > need) need = a.ws_bytes;
  if (u.ok && u.ws_bytes > need) need = u.ws_bytes;
  return need;
}

bool describe_stage1_contig(const void* x, int64_t rows, int64_t n, int64_t row_stride, int64_t k0, int j,
                            int layout, int dtype, std::string& out) {
  const contig::Plan pl = plan_for(x, rows, n, row_stride, k0, j, layout, dtype);
  if (!pl.ok) return false;
  if (pl.geom.whole) {
    out += "whole_bucket_kernel<" + std::string(dtype_name(dtype)) + ", J=" + std::to_string(j) + "> grid=" +
           std::to_string(contig::bucket_groups(pl.geom, rows)) + " block=256";
    return true;
  }
  if (pl.geom.split) {
    out += "split_bucket_kernel<" + std::string(dtype_name(dtype)) + ", J=" + std::to_string(j) + "> grid=" +
           std::to_string(contig::bucket_groups(pl.geom, rows)) + " block=256 pieces=" +
           std::to_string(1 << pl.geom.split_log2);
    return true;
  }
  out += "contig_kernel<" + std::string(dtype_name(dtype)) + ", J=" + std::to_string(j) + ", V=" +
         std::to_string(pl.vec) + "> grid=" + std::to_string(rows * (int64_t)pl.geom.groups) + " block=256 chunks=" +
         std::to_string(pl.geom.chunks) + " slabs=" + std::to_string(pl.geom.slabs) +
         (pl.geom.fast ? " even" : "");
  if (pl.geom.slabs > 1) out += " + contig_merge_kernel<" + std::string(dtype_name(dtype)) + ", J=" + std::to_string(j) + ">";
  return true;
}

int launch_stage1_contig(const void* x, int64_t rows, int64_t n, int64_t row_stride, int64_t k0, int j,
                         int layout, int dtype, void* values, IndexOut indices, void* ws, size_t ws_bytes,
                         hipStream_t stream, bool* handled) {
  const contig::Plan pl = plan_for(x, rows, n, row_stride, k0, j, layout, dtype);
  *handled = pl.ok;
  if (!pl.ok) return ATK_OK;
  if (pl.ws_bytes && (!ws || ws_bytes < pl.ws_bytes || (uintptr_t)ws % 16 != 0)) return ATK_ERR_WORKSPACE;
  int rc = ATK_ERR_DTYPE;
  ATK_DTYPE_SWITCH(dtype, E, rc = ATK_ERR_DTYPE,
                   rc = contig::launch_typed<E>(pl, x, rows, row_stride, j, values, indices, ws, stream));
  return rc;
}

}  // namespace atk
