// Fill, strided gather and batched pad/crop copies (bit copies of raw words).
#include "common.h"

namespace {

// 16-byte stores of a replicated pattern, then the sub-16-byte tail.
template <typename T>
__global__ void fill_kernel(T* __restrict__ dst, int64_t count, T value, uint4 pattern) {
  const int64_t total_bytes = count * int64_t(sizeof(T));
  const int64_t n16 = total_bytes / 16;
  uint4* d16 = reinterpret_cast<uint4*>(dst);
  const int64_t stride = int64_t(gridDim.x) * blockDim.x;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n16; i += stride) d16[i] = pattern;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    for (int64_t e = n16 * 16 / int64_t(sizeof(T)); e < count; ++e) dst[e] = value;
  }
}

// Strided gathers. dst is C-ordered; src element i sits at
// offset + sum_d coord_d(i) * strides[d]. Both kernels are bound by HBM and by
// how whole the 128-byte lines are that they touch; neither divides by a
// runtime extent (Divider) while the element count fits 31 bits.

// Division by a fixed extent d of n < 2^31: n / d = (mulhi(n, mul) + n) >> shift
// with shift = ceil(log2 d) and mul = floor(2^32 (2^shift - d) / d) + 1
// (Granlund and Montgomery, "Division by invariant integers using
// multiplication", 1994, the round-up form). A 64-bit division costs dozens of
// instructions per element and axis, more than the copy itself.
struct Divider {
  uint32_t extent, mul, shift;
};

Divider make_divider(int64_t extent) {
  Divider d{uint32_t(extent), 0, 0};
  while ((uint64_t(1) << d.shift) < uint64_t(extent)) ++d.shift;
  d.mul = uint32_t((((uint64_t(1) << d.shift) - uint64_t(extent)) << 32) / uint64_t(extent) + 1);
  return d;
}

struct Strided {
  int64_t shape[8];
  int64_t strides[8];
  Divider div[8];  // set when every index fits 31 bits
};

// Quotient and remainder of `rest` by axis d's extent.
template <typename I>
__device__ __forceinline__ I split(I rest, const Strided& layout, int d, I& coord) {
  I q;
  if constexpr (sizeof(I) == 4) {
    const Divider& by = layout.div[d];
    q = (__umulhi(rest, by.mul) + rest) >> by.shift;
    coord = rest - q * by.extent;
  } else {
    const I extent = I(layout.shape[d]);
    q = rest / extent;
    coord = rest - q * extent;
  }
  return q;
}

// Source element of axes [0, axes) at C-order index `rest` over them.
template <typename I>
__device__ __forceinline__ int64_t source_at(I rest, int axes, const Strided& layout) {
  int64_t at = 0;
  for (int d = axes - 1; d >= 0; --d) {
    I coord;
    rest = split<I>(rest, layout, d, coord);
    at += int64_t(coord) * layout.strides[d];
  }
  return at;
}

// V elements as one access that needs element alignment only (gfx950 takes
// global vector accesses at any dword, and bytes at any byte).
template <typename T, int V>
struct Packed {
  typedef T type __attribute__((ext_vector_type(V), aligned(sizeof(T))));
};

// Elements in order of dst: a thread moves G runs of V consecutive dst elements
// (16 bytes for 4- and 8-byte words), all loads before the first store. A run
// inside one innermost row takes one index computation, and one vector load
// when the row is contiguous in src (UNIT); a run that crosses a row end takes
// an index computation per element. Either way it is one vector store: runs
// are contiguous in dst. Strided rows (UNIT = 0) load V words and rely on the
// caches for the parts of lines that neighbours use. (Runs that crossed went
// element by element, each load behind the store before it, and every wave of
// an odd row length has such runs: columns 1 to 9 of 3000000 x 11 float32
// 68.6 us, every seventh column 55.5, a 3 x 1080 x 1920 image to channels last
// in float64 22.5; now 37.7, 25.9 and 17.)
template <typename T, int V, bool UNIT, typename I, int G>
__global__ __launch_bounds__(256) void gather_rows_kernel(const T* __restrict__ src, T* __restrict__ dst, I count,
                                                          int rank, Strided layout) {
  using Vec = typename Packed<T, V>::type;
  const I length = I(layout.shape[rank - 1]);
  const int64_t step = UNIT ? 1 : layout.strides[rank - 1];
  Vec v[G];
  I at[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const I i = ((I(blockIdx.x) * G + g) * 256 + threadIdx.x) * V;
    at[g] = i;
    if (i >= count) continue;
    I col;
    const I row = split<I>(i, layout, rank - 1, col);
    if (col + V > length) {
#pragma unroll
      for (int j = 0; j < V; ++j) v[g][j] = i + j < count ? src[source_at<I>(i + j, rank, layout)] : T(0);
      continue;
    }
    const T* p = src + source_at<I>(row, rank - 1, layout) + int64_t(col) * step;
    if constexpr (UNIT) {
      v[g] = *reinterpret_cast<const Vec*>(p);
    } else {
#pragma unroll
      for (int j = 0; j < V; ++j) v[g][j] = p[j * step];
    }
  }
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const I i = at[g];
    if (i + V <= count) {
      *reinterpret_cast<Vec*>(dst + i) = v[g];
    } else {
#pragma unroll
      for (int j = 0; j < V; ++j)
        if (i + j < count) dst[i + j] = v[g][j];
    }
  }
}

// Transposing gathers: the fastest axis of src (`lane`, stride `lane_step`) is
// not the innermost axis of dst, so rows of one side are columns of the other.
// A 256-thread workgroup moves a kTile x kTile block of those two axes through
// LDS: it reads runs of V elements along `lane` and writes runs of V along
// dst's innermost axis, whole lines on both sides but for the block's edges.
// Without it every wave reads 64 lines for 256 bytes. Blocks are numbered with
// dst's innermost axis fastest and renumbered so that an XCD (ids i % 8) owns
// consecutive ones: neighbours' partial lines of dst then meet in one L2.
// LDS rows are kTile + 1 words long: both the writes (4 lane elements apart)
// and the reads (V apart along a row) of a wave then spread over all banks.
// Measured (float32, 32 x 1031 x 4096): transposing the last two axes and
// cropping to every other column, 1.62 GB together, 826 us with one element
// per thread and 64-bit divisions, 391 us like this (4.1 TB/s; a plain copy of
// the size reaches 4.7 TB/s).
constexpr int kTile = 64;

struct Transposed {
  Strided outer;  // the other axes of dst, in order (rank `axes`)
  int64_t outer_dst[8];
  int axes;
  int64_t lane_extent, lane_step, lane_dst;  // axis that is fastest in src: strides in src and dst
  int64_t row_extent, row_step;              // dst's innermost axis: stride in src
  uint32_t lane_tiles, row_tiles;
};

template <typename T, int V, bool UNIT>
__global__ __launch_bounds__(256) void gather_tiles_kernel(const T* __restrict__ src, T* __restrict__ dst,
                                                           Transposed t) {
  using Vec = typename Packed<T, V>::type;
  constexpr int kRuns = kTile / V;           // runs across the tile
  constexpr int kStep = 256 / kRuns;         // tile rows per pass of the workgroup
  __shared__ T tile[kTile][kTile + 1];       // [lane][row]
  const uint32_t full = gridDim.x / 8 * 8;
  const uint32_t id = blockIdx.x < full ? (blockIdx.x % 8) * (full / 8) + blockIdx.x / 8 : blockIdx.x;
  const uint32_t per_lane = id / t.row_tiles;
  const int64_t row0 = int64_t(id - per_lane * t.row_tiles) * kTile;
  uint32_t rest = per_lane / t.lane_tiles;
  const int64_t lane0 = int64_t(per_lane - rest * t.lane_tiles) * kTile;
  for (int d = t.axes - 1; d >= 0; --d) {
    const uint32_t extent = uint32_t(t.outer.shape[d]);
    const uint32_t q = rest / extent;
    src += int64_t(rest - q * extent) * t.outer.strides[d];
    dst += int64_t(rest - q * extent) * t.outer_dst[d];
    rest = q;
  }
  src += lane0 * t.lane_step + row0 * t.row_step;
  dst += lane0 * t.lane_dst + row0;
  const int lanes = int(t.lane_extent - lane0 < kTile ? t.lane_extent - lane0 : kTile);
  const int rows = int(t.row_extent - row0 < kTile ? t.row_extent - row0 : kTile);
  const int run = (threadIdx.x % kRuns) * V, first = threadIdx.x / kRuns;
  Vec v[kTile / kStep];
#pragma unroll
  for (int s = 0; s < kTile / kStep; ++s) {
    const int r = first + s * kStep;
    const T* p = src + int64_t(r) * t.row_step + int64_t(run) * t.lane_step;
    if (UNIT && r < rows && run + V <= lanes) {
      v[s] = *reinterpret_cast<const Vec*>(p);
    } else {
#pragma unroll
      for (int j = 0; j < V; ++j) v[s][j] = r < rows && run + j < lanes ? p[j * t.lane_step] : T(0);
    }
  }
#pragma unroll
  for (int s = 0; s < kTile / kStep; ++s)
#pragma unroll
    for (int j = 0; j < V; ++j) tile[run + j][first + s * kStep] = v[s][j];
  __syncthreads();
#pragma unroll
  for (int s = 0; s < kTile / kStep; ++s) {
    const int l = first + s * kStep;
    Vec w;
#pragma unroll
    for (int j = 0; j < V; ++j) w[j] = tile[l][run + j];
    T* p = dst + int64_t(l) * t.lane_dst + run;
    if (l < lanes && run + V <= rows) {
      *reinterpret_cast<Vec*>(p) = w;
    } else if (l < lanes) {
#pragma unroll
      for (int j = 0; j < V; ++j)
        if (run + j < rows) p[j] = w[j];
    }
  }
}

// One workgroup per destination row (grid-stride over rows); lanes walk
// columns. Each lane issues kPadUnroll loads before its stores, so a row of a
// few thousand elements is one or two rounds of independent loads rather than
// a chain of load-store pairs. Rows of padded operands are rarely 16-byte
// aligned on both sides, so accesses stay element-wide (coalesced per wave).
constexpr int kPadUnroll = 8;

template <typename T>
__global__ void pad_kernel(const T* __restrict__ src, T* __restrict__ dst, int64_t rows_total, int64_t src_rows,
                           int64_t src_cols, int64_t dst_rows, int64_t dst_cols) {
  for (int64_t row = blockIdx.x; row < rows_total; row += gridDim.x) {
    const int64_t b = row / dst_rows;
    const int64_t r = row - b * dst_rows;
    T* out = dst + row * dst_cols;
    const bool from_src = r < src_rows;
    const T* in = src + (from_src ? (b * src_rows + r) * src_cols : 0);
    const int64_t copy_cols = from_src ? (src_cols < dst_cols ? src_cols : dst_cols) : 0;
    const int64_t step = int64_t(blockDim.x) * kPadUnroll;
    for (int64_t base = threadIdx.x; base < dst_cols; base += step) {
      T v[kPadUnroll];
#pragma unroll
      for (int j = 0; j < kPadUnroll; ++j) {
        const int64_t c = base + int64_t(j) * blockDim.x;
        v[j] = c < copy_cols ? in[c] : T(0);
      }
#pragma unroll
      for (int j = 0; j < kPadUnroll; ++j) {
        const int64_t c = base + int64_t(j) * blockDim.x;
        if (c < dst_cols) out[c] = v[j];
      }
    }
  }
}

int64_t grid_for(int64_t work, int64_t per_block) {
  int64_t g = hp::ceil_div(work, per_block);
  if (g < 1) g = 1;
  return g > 65536 * 16 ? 65536 * 16 : g;
}

// The axis whose src stride makes a transposing gather worth its LDS tile, or
// -1. It is the axis of the smallest stride (<= 16 bytes: neighbours share
// lines) and not the innermost one, whose steps are lines apart or nearly
// (kApart). A tile costs what a whole one costs however much of it is used, so
// the share of its kTile x kTile elements decides, against rows that read each
// line anew unless the caches keep it: they do for blocks of up to some hundred
// lines (`rows`, the innermost extent), hardly for a thousand. Measured, us in
// rows / tiles, 64 MB each: float32 blocks of 32 x 32 (a quarter used) 22 / 32,
// 48 x 32 23 / 24, 48 x 64 34 / 20; 16 lanes (a quarter) x 256 36 / 31, x 4096
// 78 / 30, x 500000 149 / 31; 12 lanes (0.19) x 256 36 / 39, x 1024 46 / 39;
// float64 16 x 16 (0.06; 205 MB) 72 / 257, 16 lanes x 256 34 / 27, 12 lanes x 256
// 30 / 33, x 1024 84 / 33. Runs that cross row ends cost rows a little: 33 x 33
// (0.27; 20000 float64) 85 / 73. A last tile of a few rows writes parts of lines:
// 65 x 65 (0.26; 20000 float64) 327 / 519, 80 x 80 (0.39) 509 / 550.
int transposed_axis(int rank, const int64_t* shape, const int64_t* strides, int elem_bytes) {
  const int64_t kApart = elem_bytes >= 4 ? 48 : 128;
  const auto bytes = [&](int d) { return (strides[d] < 0 ? -strides[d] : strides[d]) * elem_bytes; };
  if (rank < 2 || bytes(rank - 1) < kApart) return -1;
  int best = -1;
  for (int d = 0; d < rank - 1; ++d)
    if (shape[d] > 1 && bytes(d) > 0 && bytes(d) <= 16 && (best < 0 || bytes(d) < bytes(best))) best = d;
  if (best < 0) return -1;
  const int64_t lanes = shape[best], rows = shape[rank - 1];
  const auto share = [](int64_t n) { return double(n) / double(hp::ceil_div(n, kTile) * kTile); };
  const bool sliver = rows > kTile && rows < 256 && (rows - 1) % kTile < 16;
  const bool crossing = elem_bytes >= 4 && rows % (16 / elem_bytes) != 0;
  const double least = sliver ? 0.45 : rows < 64 ? (crossing ? 0.25 : 1.0 / 3) : rows < 1024 ? 0.23 : 0.18;
  return share(lanes) * share(rows) >= least ? best : -1;
}

template <typename T, int V, int G>
void run_gather_rows(hp_ctx* ctx, const T* src, T* dst, int64_t count, int rank, Strided& layout) {
  const int64_t grid = hp::ceil_div(count, 256 * V * G);
  hp::require(grid <= hp::kMaxGrid, "gather too large for one launch");
  const bool unit = layout.strides[rank - 1] == 1 || layout.shape[rank - 1] == 1;
  // 31-bit indices, the overhang of the last workgroup included.
  if (grid * 256 * V * G <= INT32_MAX) {
    for (int d = 0; d < rank; ++d) layout.div[d] = make_divider(layout.shape[d]);
    if (unit) gather_rows_kernel<T, V, true, uint32_t, G><<<grid, 256, 0, ctx->stream>>>(src, dst, uint32_t(count), rank, layout);
    else gather_rows_kernel<T, V, false, uint32_t, G><<<grid, 256, 0, ctx->stream>>>(src, dst, uint32_t(count), rank, layout);
  } else {
    if (unit) gather_rows_kernel<T, V, true, int64_t, G><<<grid, 256, 0, ctx->stream>>>(src, dst, count, rank, layout);
    else gather_rows_kernel<T, V, false, int64_t, G><<<grid, 256, 0, ctx->stream>>>(src, dst, count, rank, layout);
  }
}

template <typename T, int V>
void run_gather(hp_ctx* ctx, const void* src_, void* dst_, int64_t count, int64_t offset, int rank, Strided layout) {
  const T* src = static_cast<const T*>(src_) + offset;
  T* dst = static_cast<T*>(dst_);
  const int lane = transposed_axis(rank, layout.shape, layout.strides, sizeof(T));
  if (lane >= 0) {
    Transposed t{};
    int64_t dst_step = 1, batches = 1;
    int64_t steps[8];
    for (int d = rank - 1; d >= 0; --d) {
      steps[d] = dst_step;
      dst_step *= layout.shape[d];
    }
    for (int d = 0; d < rank - 1; ++d) {
      if (d == lane) continue;
      t.outer.shape[t.axes] = layout.shape[d];
      t.outer.strides[t.axes] = layout.strides[d];
      t.outer_dst[t.axes++] = steps[d];
      batches *= layout.shape[d];
    }
    t.lane_extent = layout.shape[lane];
    t.lane_step = layout.strides[lane];
    t.lane_dst = steps[lane];
    t.row_extent = layout.shape[rank - 1];
    t.row_step = layout.strides[rank - 1];
    const int64_t lane_tiles = hp::ceil_div(t.lane_extent, kTile), row_tiles = hp::ceil_div(t.row_extent, kTile);
    if (batches <= hp::kMaxGrid / (lane_tiles * row_tiles)) {
      t.lane_tiles = uint32_t(lane_tiles);
      t.row_tiles = uint32_t(row_tiles);
      const int64_t grid = batches * lane_tiles * row_tiles;
      if (t.lane_step == 1) gather_tiles_kernel<T, V, true><<<grid, 256, 0, ctx->stream>>>(src, dst, t);
      else gather_tiles_kernel<T, V, false><<<grid, 256, 0, ctx->stream>>>(src, dst, t);
      return;
    }
  }
  if (rank == 0) {
    layout.shape[0] = 1;
    layout.strides[0] = 1;
    rank = 1;
  }
  // Runs per thread: one where every run crosses (every seventh column of
  // 3000000 x 11 float32: 25.9 us, 27.7 with two), four where 8-byte words
  // of a run are 32 bytes apart or more (300000 x 15 float64, transposed: 72 us
  // against 80 with two; 1000000 x 4 20.5 against 22.4), else two (columns 1 to 9 of 3000000 x 11 float64: 88.7
  // us against 92 with four).
  const int64_t step = layout.strides[rank - 1] < 0 ? -layout.strides[rank - 1] : layout.strides[rank - 1];
  if (layout.shape[rank - 1] < V) run_gather_rows<T, V, 1>(ctx, src, dst, count, rank, layout);
  else if (sizeof(T) == 8 && step >= 4) run_gather_rows<T, V, 4>(ctx, src, dst, count, rank, layout);
  else run_gather_rows<T, V, 2>(ctx, src, dst, count, rank, layout);
}

uint4 replicate(uint64_t bits, int elem_bytes) {
  uint64_t word = 0;
  switch (elem_bytes) {
    case 1: word = (bits & 0xFF) * 0x0101010101010101ull; break;
    case 2: word = (bits & 0xFFFF) * 0x0001000100010001ull; break;
    case 4: word = (bits & 0xFFFFFFFFull) * 0x0000000100000001ull; break;
    default: word = bits; break;
  }
  uint4 p;
  p.x = uint32_t(word);
  p.y = uint32_t(word >> 32);
  p.z = p.x;
  p.w = p.y;
  return p;
}

}  // namespace

using hp::guarded;
using hp::require;

extern "C" {

int hp_fill(hp_ctx* ctx, void* dst, int64_t count, int elem_bytes, uint64_t bits) {
  return guarded([&] {
    hp::enter(ctx);
    require(count >= 0, "negative count");
    require(elem_bytes == 1 || elem_bytes == 2 || elem_bytes == 4 || elem_bytes == 8,
            "elem_bytes must be 1, 2, 4 or 8");
    if (count == 0) return;
    require(dst != nullptr, "null destination");
    require(reinterpret_cast<uintptr_t>(dst) % 16 == 0, "fill destination must be 16-byte aligned");
    const uint4 pattern = replicate(bits, elem_bytes);
    const int64_t grid = grid_for(count * elem_bytes / 16 + 1, 256 * 4);
    switch (elem_bytes) {
      case 1: fill_kernel<uint8_t><<<grid, 256, 0, ctx->stream>>>((uint8_t*)dst, count, uint8_t(bits), pattern); break;
      case 2: fill_kernel<uint16_t><<<grid, 256, 0, ctx->stream>>>((uint16_t*)dst, count, uint16_t(bits), pattern); break;
      case 4: fill_kernel<uint32_t><<<grid, 256, 0, ctx->stream>>>((uint32_t*)dst, count, uint32_t(bits), pattern); break;
      default: fill_kernel<uint64_t><<<grid, 256, 0, ctx->stream>>>((uint64_t*)dst, count, uint64_t(bits), pattern); break;
    }
    hp::check_launch("fill");
  });
}

int hp_gather(hp_ctx* ctx, int elem_bytes, const void* src, void* dst, int64_t offset, int rank,
              const int64_t* shape, const int64_t* strides) {
  return guarded([&] {
    hp::enter(ctx);
    require(rank >= 0 && rank <= 8, "gather rank must be <= 8");
    require(elem_bytes == 1 || elem_bytes == 2 || elem_bytes == 4 || elem_bytes == 8,
            "elem_bytes must be 1, 2, 4 or 8");
    Strided layout{};
    int64_t count = 1;
    for (int d = 0; d < rank; ++d) {
      require(shape[d] >= 0, "negative extent");
      layout.shape[d] = shape[d];
      layout.strides[d] = strides[d];
      count *= shape[d];
    }
    if (count == 0) return;
    require(src != nullptr && dst != nullptr, "null pointer");
    for (int d = 0; d < rank; ++d) require(layout.shape[d] > 0, "empty extent");
    switch (elem_bytes) {
      case 1: run_gather<uint8_t, 4>(ctx, src, dst, count, offset, rank, layout); break;
      case 2: run_gather<uint16_t, 4>(ctx, src, dst, count, offset, rank, layout); break;
      case 4: run_gather<uint32_t, 4>(ctx, src, dst, count, offset, rank, layout); break;
      default: run_gather<uint64_t, 2>(ctx, src, dst, count, offset, rank, layout); break;
    }
    hp::check_launch("gather");
  });
}

int hp_pad_copy(hp_ctx* ctx, int elem_bytes, const void* src, void* dst, int64_t batch, int64_t src_rows,
                int64_t src_cols, int64_t dst_rows, int64_t dst_cols) {
  return guarded([&] {
    hp::enter(ctx);
    require(elem_bytes == 4 || elem_bytes == 8, "pad copies move 4- or 8-byte words");
    require(batch >= 0 && src_rows >= 0 && src_cols >= 0 && dst_rows >= 0 && dst_cols >= 0,
            "negative extent");
    const int64_t rows_total = batch * dst_rows;
    if (rows_total == 0 || dst_cols == 0) return;
    require(dst != nullptr, "null destination");
    require(src != nullptr || src_rows == 0 || src_cols == 0, "null source");
    // A source with no rows or no columns contributes only zeros.
    int64_t sr = src_rows, sc = src_cols;
    if (sr == 0 || sc == 0) sr = 0;
    const int64_t grid = rows_total < 65536 * 4 ? rows_total : 65536 * 4;
    const int block = dst_cols >= 256 ? 256 : 64;
    if (elem_bytes == 4) {
      pad_kernel<uint32_t><<<grid, block, 0, ctx->stream>>>((const uint32_t*)src, (uint32_t*)dst, rows_total, sr,
                                                           sc, dst_rows, dst_cols);
    } else {
      pad_kernel<uint64_t><<<grid, block, 0, ctx->stream>>>((const uint64_t*)src, (uint64_t*)dst, rows_total, sr,
                                                           sc, dst_rows, dst_cols);
    }
    hp::check_launch("pad_copy");
  });
}

}  // extern "C"
