// The gradient of the selected values with respect to the input: every row of the result is
// zero but for the k positions a forward call selected, which hold the gradients of its values.
//
// Bound: HBM writes, n * sizeof(T) per row, plus k * (sizeof(T) + 8) read.  Filling the row with
// zeros and scattering into it afterwards writes it twice and more: single elements spread over
// the row make the memory read and write back whole lines.  Here a workgroup owns a tile of the
// row in LDS, zeroes it, puts its entries in and writes it out once, in 16-byte stores.
//
// Which entries a tile has.  A forward call returns its results bucket by bucket, so the entries
// of a range of buckets are adjacent.  An interleaved row is the matrix [sub-rows][b], bucket c its
// column c: a tile is a block of columns over a run of sub-rows, and its entries lie between two
// positions, c * j when every bucket kept j (one stage), else found by a 64-way search over the
// entries' buckets (three rounds for 2^18 entries).  With few entries a tile is a run of whole
// sub-rows instead and looks at all of them.  A contiguous row's tile is a run of positions.
// Rows that a tile holds whole are put into it one after the other, with all their entries.
#include <hip/hip_runtime.h>

#include "atk_device.h"
#include "atk_launch.h"
#include "stage1_stream.h"

namespace atk {
namespace {

constexpr uint32_t kThreads = 512, kWave = 64;
// LDS of a tile: two workgroups of eight waves per CU.  (Half the tile, or workgroups of 256 or 1024
// threads: within 5 % either way at fp32 [64, 2^20] k=65536, [8, 2^23] k=4096 and the shape above.)
constexpr uint32_t kTileBytes = 64 * 1024;
// Entries (12 bytes each or less) every tile may look at: a quarter of what it writes.
constexpr int64_t kFewEntries = 1024;
// Bytes of a sub-row a column tile has at least: whole lines of the memory.
constexpr uint32_t kMinSegment = 512;
// Tiles of a launch before one holds several rows: two rounds of two workgroups per CU.
constexpr int64_t kManyTiles = 1024;

struct Grad {
  int64_t k;            // entries per row
  int64_t rows;
  uint32_t n, b, j;
  uint32_t base, longer;  // contiguous buckets: elements of a bucket, buckets with one more
  uint32_t tile_cols;   // columns of a tile (a power of two), or 0: tiles are runs of positions
  uint32_t vecs_shift;  // log2 of a tile's 16-byte pieces per sub-row
  uint32_t tile_len;    // sub-rows of a tile, or positions
  uint32_t tile_rows;   // rows of a tile: more than one only when it holds whole rows
  uint32_t col_tiles, run_tiles;
  int contiguous;       // bucket layout
  int full;             // every bucket kept j entries
  int all;              // a tile looks at all entries of its row
};

__device__ __forceinline__ uint32_t bucket_of(const Grad& g, uint32_t index) {
  if (!g.contiguous) return index % g.b;
  const uint32_t head = g.longer * (g.base + 1);
  return index < head ? index / (g.base + 1) : g.longer + (index - head) / g.base;
}

// One wave: how many of the row's entries belong to buckets below `bucket`.
__device__ __forceinline__ uint32_t entries_below(const Grad& g, const int64_t* __restrict__ indices, uint32_t bucket,
                                                  uint32_t lane) {
  uint32_t a = 0, z = (uint32_t)g.k;  // the answer lies in [a, z]
  while (a < z) {
    const uint32_t step = (z - a + kWave - 1) / kWave;
    const uint32_t e = a + lane * step;
    const bool below = e < z && bucket_of(g, (uint32_t)indices[e]) < bucket;
    const uint32_t count = (uint32_t)__popcll(__ballot(below));  // the lanes below come first
    if (count == 0) break;
    const uint32_t last = a + (count - 1) * step;
    z = last + step < z ? last + step : z;
    a = last + 1;
  }
  return a;
}

template <typename raw_t>
__global__ __launch_bounds__(kThreads) void topk_grad_kernel(const raw_t* __restrict__ grad,
                                                             const int64_t* __restrict__ indices,
                                                             raw_t* __restrict__ out, const Grad g) {
  constexpr uint32_t V = 16 / sizeof(raw_t);
  extern __shared__ __align__(16) unsigned char dyn_lds[];
  raw_t* tile = reinterpret_cast<raw_t*>(dyn_lds);
  __shared__ uint32_t bounds[2];
  const uint32_t tid = threadIdx.x, lane = tid % kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  uint32_t blk = blockIdx.x;
  const uint32_t col_tile = __builtin_amdgcn_readfirstlane(blk % g.col_tiles);
  blk /= g.col_tiles;
  const uint32_t run = __builtin_amdgcn_readfirstlane(blk % g.run_tiles);
  const int64_t row = (int64_t)__builtin_amdgcn_readfirstlane(blk / g.run_tiles) * g.tile_rows;
  const uint32_t held = g.rows - row < g.tile_rows ? (uint32_t)(g.rows - row) : g.tile_rows;  // rows of this tile
  const uint32_t k = (uint32_t)g.k;
  grad += row * g.k;
  indices += row * g.k;
  out += row * (int64_t)g.n;

  const uint32_t c0 = col_tile * g.tile_cols;
  const uint32_t c1 = c0 + g.tile_cols < g.b ? c0 + g.tile_cols : g.b;
  const uint32_t first = run * g.tile_len;  // sub-row or position
  const uint32_t elements = g.tile_cols != 0 ? g.tile_cols * g.tile_len : g.tile_len;
  const uint32_t cols_shift = g.vecs_shift + __builtin_ctz(V);

  uint32_t lo = 0, hi = held * k;  // (at most a tile's elements when it holds several rows)
  if (!g.all) {
    uint32_t below0 = c0, below1 = c1;  // buckets of this tile: [below0, below1)
    if (g.tile_cols == 0) {
      const uint32_t end = g.n - first < g.tile_len ? g.n : first + g.tile_len;
      below0 = bucket_of(g, first);
      below1 = bucket_of(g, end - 1) + 1;
    }
    if (g.full) {
      lo = below0 * g.j;
      hi = below1 * g.j;
    } else {
      if (wave < 2) {
        const uint32_t found = entries_below(g, indices, wave == 0 ? below0 : below1, lane);
        if (lane == 0) bounds[wave] = found;
      }
      __syncthreads();
      lo = bounds[0];
      hi = bounds[1];
    }
  }
  // the first entries are on their way while the tile is zeroed
  constexpr uint32_t kAhead = 2;
  uint32_t index[kAhead];
  raw_t value[kAhead];
  auto fetch = [&](uint32_t e0) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t u = 0; u < kAhead; ++u) {
      const uint32_t e = e0 + u * kThreads;
      index[u] = e < hi ? (uint32_t)indices[e] : ~0u;
      value[u] = e < hi ? grad[e] : (raw_t)0;
    }
  };
  fetch(lo + tid);
  for (uint32_t i = tid * V; i < elements; i += kThreads * V)
    *reinterpret_cast<uint4*>(&tile[i]) = make_uint4(0, 0, 0, 0);
  __syncthreads();
  for (uint32_t e0 = lo + tid;;) {
#pragma unroll
    for (uint32_t u = 0; u < kAhead; ++u) {
      if (g.tile_rows > 1) {
        if (index[u] < g.n) tile[(e0 + u * kThreads) / k * g.n + index[u]] = value[u];
      } else if (g.tile_cols == 0) {
        if (index[u] - first < g.tile_len) tile[index[u] - first] = value[u];
      } else {
        const uint32_t p = index[u] / g.b, c = index[u] - p * g.b;
        if (index[u] < g.n && p - first < g.tile_len && c - c0 < g.tile_cols)
          tile[((p - first) << cols_shift) + (c - c0)] = value[u];
      }
    }
    e0 += kAhead * kThreads;
    if (e0 - tid >= hi) break;  // (the same trips for every thread)
    fetch(e0);
  }
  __syncthreads();

  using stream::Pack;
  using stream::store_pack;
  if (g.tile_cols == 0) {
    const uint32_t left = held * g.n - first, len = left < g.tile_len ? left : g.tile_len;
    const uint32_t whole = len / V * V;
    for (uint32_t i = tid * V; i < whole; i += kThreads * V)
      store_pack<raw_t, V>(out + first + i, *reinterpret_cast<const Pack<raw_t, V>*>(&tile[i]));
    if (tid < len - whole) out[first + whole + tid] = tile[whole + tid];
  } else {
    const uint32_t sub_rows = (g.n + g.b - 1) / g.b;
    const uint32_t end = sub_rows - first < g.tile_len ? sub_rows - first : g.tile_len;
    for (uint32_t i = tid; i < end << g.vecs_shift; i += kThreads) {
      const uint32_t p = i >> g.vecs_shift, c = (i - (p << g.vecs_shift)) * V;
      if (c0 + c >= c1) continue;
      const int64_t at = (int64_t)(first + p) * g.b + c0 + c;
      const int64_t left = (int64_t)g.n - at;  // (the last sub-row may be a part of one)
      const uint32_t width = c1 - c0 - c < V ? c1 - c0 - c : V;
      const raw_t* from = &tile[i * V];
      if (width == V && left >= (int64_t)V) {
        store_pack<raw_t, V>(out + at, *reinterpret_cast<const Pack<raw_t, V>*>(from));
      } else {
        for (uint32_t v = 0; v < width && (int64_t)v < left; ++v) out[at + v] = from[v];
      }
    }
  }
}

Grad plan_grad(int64_t rows, int64_t n, int64_t k0, int j, int64_t k, int layout, uint32_t es) {
  Grad g{};
  g.k = k;
  g.rows = rows;
  g.n = (uint32_t)n;
  g.b = (uint32_t)(k0 / j);
  g.j = (uint32_t)j;
  g.base = g.n / g.b;
  g.longer = g.n % g.b;
  g.contiguous = layout == ATK_BALANCED;
  g.full = k == k0;
  const uint32_t room = kTileBytes / es;
  g.all = n <= room || k <= kFewEntries;
  g.col_tiles = 1;
  g.tile_rows = 1;
  if (n <= room) {
    // Short rows, as many to a tile as it holds while that leaves kManyTiles: results are dense, so the rows of a
    // tile are one run of memory.  A workgroup to every row costs 1.5 ns a row whatever it writes: fp32 [10^6, 64]
    // k=4 1480 us against 244 us of zeros and a scatter, 52 us this way; [10^5, 256] k=16 152, 56 and 18.5 us,
    // [10^4, 1000] k=62 19.6, 29.2 and 8.2 us; fp16 [10^6, 16] k=4 1471, 30 and 12 us.
    const int64_t most = room / n, wanted = (rows + kManyTiles - 1) / kManyTiles;
    g.tile_rows = (uint32_t)(wanted < most ? wanted : most);
    g.tile_len = g.tile_rows * g.n;
    g.run_tiles = 1;
    return g;
  }
  if (g.all || g.contiguous) {
    g.tile_len = room;
    g.run_tiles = (g.n + g.tile_len - 1) / g.tile_len;
    return g;
  }
  // Columns: as many as let a tile hold every sub-row, within whole lines and what LDS holds.
  const uint32_t sub_rows = (g.n + g.b - 1) / g.b;
  uint32_t cols = kMinSegment / es;
  while (cols < g.b && (uint64_t)cols * 2 * sub_rows <= room) cols *= 2;
  g.tile_cols = cols;
  g.vecs_shift = (uint32_t)__builtin_ctz(cols * es / 16);
  g.tile_len = room / cols < sub_rows ? room / cols : sub_rows;
  g.col_tiles = (g.b + cols - 1) / cols;
  g.run_tiles = (sub_rows + g.tile_len - 1) / g.tile_len;
  return g;
}

}  // namespace

int launch_topk_grad(const void* grad_values, const int64_t* indices, int64_t rows, int64_t n, int64_t k0, int j,
                     int64_t k, int layout, int dtype, void* grad_x, hipStream_t stream) {
  const uint32_t es = (uint32_t)elem_bytes(dtype);
  const Grad g = plan_grad(rows, n, k0, j, k, layout, es);
  const int64_t groups = (rows + g.tile_rows - 1) / g.tile_rows * (int64_t)g.col_tiles * g.run_tiles;
  if (groups > 0xffffffffll / kThreads) return ATK_ERR_TOO_LARGE;  // (a launch's threads are counted in 32 bits)
  const uint32_t elements = g.tile_cols != 0 ? g.tile_cols * g.tile_len : g.tile_len;
  const size_t lds = ((size_t)elements * es + 15) & ~(size_t)15;
  auto go = [&](auto zero) {
    using raw_t = decltype(zero);
    auto kern = topk_grad_kernel<raw_t>;
    if (lds > 48 * 1024 &&
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds) != hipSuccess)
      return (int)ATK_ERR_LAUNCH;
    hipLaunchKernelGGL(kern, dim3((unsigned)groups), dim3(kThreads), lds, stream,
                       static_cast<const raw_t*>(grad_values), indices, static_cast<raw_t*>(grad_x), g);
    return (int)(hipGetLastError() == hipSuccess ? ATK_OK : ATK_ERR_LAUNCH);
  };
  switch (es) {
    case 1: return go(uint8_t{});
    case 2: return go(uint16_t{});
    case 4: return go(uint32_t{});
    case 8: return go(uint64_t{});
  }
  return ATK_ERR_DTYPE;
}

}  // namespace atk
