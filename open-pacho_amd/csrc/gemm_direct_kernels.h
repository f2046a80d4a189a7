// Kernels and launches of the direct products (see gemm_direct.h); included by
// gemm_direct_f32.hip and gemm_direct_f64.hip only.
#pragma once

#include "gemm_direct.h"

namespace {

using hpgemm::BatchDesc;
using hpgemm::DirectPlan;

constexpr int kWaves = 4;  // per tile, each taking every fourth slice
// Slices after which a wave's accumulators join its sums (DEPTH where that is
// more): the chain of a sum is 4 MFMAs per slice of a run, then the runs of a
// wave, so that its error stays below that of the staged kernels' cut tiles
// (160 shapes, K up to 8192: 0.65 of theirs in the mean in fp32, 0.69 in fp64;
// with one chain per wave it was up to 2.1 times theirs). Runs of 4 cost 3% of
// the MFMA time; the 64 x 64 tile, whose registers are full, takes 8.
template <int FI, int FJ>
constexpr int run_slices() {
  return FI * FJ == 16 ? 8 : 4;
}
constexpr int kGroupM = 4;  // tile rows per group: neighbours share operand panels in an XCD's L2

template <typename T, int N>
struct Pack {
  typedef T type __attribute__((ext_vector_type(N), aligned(sizeof(T))));
};

template <typename T>
struct Mfma;
template <>
struct Mfma<float> {
  typedef float Acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ Acc apply(float a, float b, Acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  // Row of accumulator element r: columns are lane % 16.
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};
template <>
struct Mfma<double> {
  typedef double Acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ Acc apply(double a, double b, Acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * r + (lane >> 4); }
};

// One operand of a tile: rows r0 .. r0 + 16 F - 1 of op(A), or columns of op(B).
// KC: element (row, k) at base[row * ld + k], else at base[k * ld + row]. Tiles
// lie inside the operand (tile_origin) unless F == 1, where every kind reads
// clamped rows.
template <typename T, int F, bool KC>
struct Operand {
  using Four = typename Pack<T, 4>::type;
  using Rows = typename Pack<T, F>::type;
  const T* p[KC ? F : 1];
  int64_t ld;

  __device__ __forceinline__ void init(const T* base, int64_t r0, int64_t rows, int64_t ld_, int lane) {
    ld = ld_;
    const int k_lane = 4 * (lane >> 4);
    const int64_t first = r0 + (KC ? 1 : F) * (lane & 15);
    if constexpr (KC) {
#pragma unroll
      for (int f = 0; f < F; ++f) p[f] = base + (F > 1 || first < rows ? first + 16 * f : rows - 1) * ld + k_lane;
    } else {
      p[0] = base + k_lane * ld + (F > 1 || first < rows ? first : rows - 1);
    }
  }

  // v[f][q]: row of fragment f at k = k0 + k_lane + q.
  __device__ __forceinline__ void load(int64_t k0, T (&v)[F][4]) const {
    if constexpr (KC) {
#pragma unroll
      for (int f = 0; f < F; ++f) {
        const Four x = *reinterpret_cast<const Four*>(p[f] + k0);
#pragma unroll
        for (int q = 0; q < 4; ++q) v[f][q] = x[q];
      }
    } else {
      const T* at = p[0] + k0 * ld;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const Rows x = *reinterpret_cast<const Rows*>(at + q * ld);
#pragma unroll
        for (int f = 0; f < F; ++f) v[f][q] = x[f];
      }
    }
  }

  // The same of the slice that holds the end of K: `left` k values from this
  // lane's first (may be negative) exist, the others read as +0.
  __device__ __forceinline__ void load_end(int64_t k0, int64_t left, T (&v)[F][4]) const {
#pragma unroll
    for (int f = 0; f < F; ++f)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if constexpr (KC) v[f][q] = q < left ? p[f][k0 + q] : T(0);
        else v[f][q] = q < left ? p[0][(k0 + q) * ld + f] : T(0);
      }
  }

  // Row of the tile behind fragment f's row x.
  static __device__ __forceinline__ int row(int f, int x) { return KC ? 16 * f + x : F * x + f; }
};

// Origin of the tile that owns [t0, t0 + tile) of an axis: the last one moves
// back inside; what it then shares with its neighbour, the neighbour stores.
__device__ __forceinline__ int64_t tile_origin(int64_t t0, int64_t extent, int tile) {
  const int64_t last = extent > tile ? extent - tile : 0;
  return t0 < last ? t0 : last;
}

struct Tiles {
  int64_t tiles_m, tiles_n, per_batch, total;  // total over the batch
  int64_t slices, per_split;
  int64_t lda, ldb;
  int64_t first;  // tile of this launch's first workgroup
};

template <typename T, int FI, int FJ, int DEPTH, bool TA, bool TB>
__global__ __launch_bounds__(64 * kWaves, sizeof(T) == 4 ? 2 : 1) void direct_kernel(
    const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ out, int64_t M, int64_t N, int64_t K,
    BatchDesc bd, Tiles t) {
  using Acc = typename Mfma<T>::Acc;
  using OA = Operand<T, FI, !TA>;
  using OB = Operand<T, FJ, TB>;
  constexpr int kCols = 16 * FJ, kPitch = kCols + 4;
  __shared__ T stage[kWaves][16 * kPitch];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // Consecutive ids of one XCD (id % 8) take neighbouring tiles, in groups of
  // kGroupM tile rows.
  const uint32_t full = gridDim.x / 8 * 8;
  const uint32_t at = blockIdx.x < full ? (blockIdx.x % 8) * (full / 8) + blockIdx.x / 8 : blockIdx.x;
  const int64_t id = t.first + at;
  const int64_t split = id / t.total;
  int64_t rest = id - split * t.total;
  const int64_t batch = rest / t.per_batch;
  rest -= batch * t.per_batch;
  const int64_t group = rest / (kGroupM * t.tiles_n), first = group * kGroupM;
  const int64_t high = t.tiles_m - first < kGroupM ? t.tiles_m - first : kGroupM;
  const int64_t in_group = rest - group * kGroupM * t.tiles_n;
  const int64_t m_own = (first + in_group % high) * (16 * FI), n_own = in_group / high * kCols;
  const int64_t m0 = tile_origin(m_own, M, 16 * FI), n0 = tile_origin(n_own, N, kCols);

  int64_t a_off, b_off;
  hpgemm::batch_offsets(batch, bd, a_off, b_off);
  OA oa;
  OB ob;
  oa.init(A + a_off, m0, M, t.lda, lane);
  ob.init(B + b_off, n0, N, t.ldb, lane);

  Acc acc[FI][FJ], sums[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j) acc[i][j] = sums[i][j] = Acc{T(0), T(0), T(0), T(0)};
  auto flush = [&] {
#pragma unroll
    for (int i = 0; i < FI; ++i)
#pragma unroll
      for (int j = 0; j < FJ; ++j) {
        sums[i][j] += acc[i][j];
        acc[i][j] = Acc{T(0), T(0), T(0), T(0)};
      }
  };

  // This wave's slices: begin + wave, + kWaves, ...
  const int64_t begin = split * t.per_split;
  const int64_t end = begin + t.per_split < t.slices ? begin + t.per_split : t.slices;
  const int64_t whole = K / 16 < end ? K / 16 : end;  // the slice with the end of K comes last
  const int64_t count = whole - begin > wave ? (whole - begin - wave + kWaves - 1) / kWaves : 0;
  T a[DEPTH][FI][4], b[DEPTH][FJ][4];
  auto load = [&](int64_t s, T(&va)[FI][4], T(&vb)[FJ][4]) {
    const int64_t k0 = (begin + wave + s * kWaves) * 16;
    oa.load(k0, va);
    ob.load(k0, vb);
  };
  auto fold = [&](const T(&va)[FI][4], const T(&vb)[FJ][4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < FI; ++i)
#pragma unroll
        for (int j = 0; j < FJ; ++j) acc[i][j] = Mfma<T>::apply(va[i][q], vb[j][q], acc[i][j]);
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (d < count) load(d, a[d], b[d]);
  int64_t s = 0;
  int run = 0;
  for (; s + 2 * DEPTH <= count; s += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      fold(a[d], b[d]);
      load(s + DEPTH + d, a[d], b[d]);
    }
    if (++run == (run_slices<FI, FJ>() + DEPTH - 1) / DEPTH) {
      flush();
      run = 0;
    }
  }
  for (; s < count; s += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (s + d < count) fold(a[d], b[d]);
      if (s + DEPTH + d < count) load(s + DEPTH + d, a[d], b[d]);
    }
    if constexpr (sizeof(T) == 4 && FI * FJ < 16) flush();
  }

  if (whole < end && (whole - begin) % kWaves == wave) {
    const int64_t left = K - whole * 16 - 4 * (lane >> 4);
    oa.load_end(whole * 16, left, a[0]);
    ob.load_end(whole * 16, left, b[0]);
    fold(a[0], b[0]);
  }
  flush();

  // Rows 16 at a time (those of accumulator blocks i): the waves' tiles meet in
  // LDS, are added in wave order and stored four columns per thread.
  T* C = out + (split * (t.total / t.per_batch) + batch) * M * N;
  constexpr int kThreads = 16 * FJ * 4;  // threads with columns to store
#pragma unroll
  for (int i = 0; i < FI; ++i) {
    if (i > 0) __syncthreads();
#pragma unroll
    for (int j = 0; j < FJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) stage[wave][Mfma<T>::row(lane, r) * kPitch + OB::row(j, lane & 15)] = sums[i][j][r];
    __syncthreads();
    if (threadIdx.x < kThreads) {
      const int x = threadIdx.x / (4 * FJ), y = threadIdx.x % (4 * FJ) * 4;
      const int64_t row = m0 + OA::row(i, x), col = n0 + y;
      typename Pack<T, 4>::type sum;
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] = stage[0][x * kPitch + y + e];
#pragma unroll
      for (int w = 1; w < kWaves; ++w)
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] += stage[w][x * kPitch + y + e];
      if (row >= m_own && row < M) {
        if (col >= n_own && col + 4 <= N) {
          *reinterpret_cast<typename Pack<T, 4>::type*>(C + row * N + col) = sum;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (col + e >= n_own && col + e < N) C[row * N + col + e] = sum[e];
        }
      }
    }
  }
}

// c[i] = the splits' partial sums of element i, in split order.
template <typename T>
__global__ __launch_bounds__(256) void add_splits_kernel(const T* __restrict__ partial, T* __restrict__ c,
                                                         int64_t count, int64_t splits) {
  using Four = typename Pack<T, 4>::type;
  const int64_t i = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i + 4 <= count) {
    Four sum = *reinterpret_cast<const Four*>(partial + i);
#pragma unroll 8
    for (int64_t s = 1; s < splits; ++s) sum += *reinterpret_cast<const Four*>(partial + s * count + i);
    *reinterpret_cast<Four*>(c + i) = sum;
  } else {
    for (int64_t e = i; e < count; ++e) {
      T sum = partial[e];
      for (int64_t s = 1; s < splits; ++s) sum += partial[s * count + e];
      c[e] = sum;
    }
  }
}

template <typename T, int FI, int FJ, int DEPTH>
void launch(hp_ctx* ctx, const DirectPlan& plan, bool ta, bool tb, const T* a, const T* b, T* c, int64_t m, int64_t n,
            int64_t k, const BatchDesc& bd, int64_t batch) {
  Tiles t{plan.tiles_m, plan.tiles_n, plan.tiles_m * plan.tiles_n, plan.tiles, plan.slices, plan.per_split,
          ta ? m : k, tb ? k : n, 0};
  const int64_t workgroups = plan.tiles * plan.splits, count = m * n * batch;
  T* target = plan.splits > 1 ? static_cast<T*>(hp::scratch_alloc(ctx, size_t(plan.splits) * count * sizeof(T))) : c;
  // Batches of many small matrices pass what one launch takes.
  for (; t.first < workgroups; t.first += hp::kMaxGrid) {
    const int64_t grid = workgroups - t.first < hp::kMaxGrid ? workgroups - t.first : hp::kMaxGrid;
#define PACHO_DIRECT(TA, TB) \
  direct_kernel<T, FI, FJ, DEPTH, TA, TB><<<grid, 64 * kWaves, 0, ctx->stream>>>(a, b, target, m, n, k, bd, t)
    if (ta && tb) PACHO_DIRECT(true, true);
    else if (ta) PACHO_DIRECT(true, false);
    else if (tb) PACHO_DIRECT(false, true);
    else PACHO_DIRECT(false, false);
#undef PACHO_DIRECT
    hp::check_launch("gemm_direct");
  }
  if (plan.splits == 1) return;
  add_splits_kernel<T><<<hp::ceil_div(count, 1024), 256, 0, ctx->stream>>>(target, c, count, plan.splits);
  hp::check_launch("gemm_add_splits");
  hp::scratch_free(ctx, target);
}

// The tiles that direct_plan chooses among; DEPTH keeps the loads of a slice
// about 2000 cycles of MFMA ahead.
template <typename T>
void run_direct(hp_ctx* ctx, const DirectPlan& plan, bool ta, bool tb, const void* a_, const void* b_, void* c_,
                int64_t m, int64_t n, int64_t k, const BatchDesc& bd, int64_t batch) {
  const T* a = static_cast<const T*>(a_);
  const T* b = static_cast<const T*>(b_);
  T* c = static_cast<T*>(c_);
  constexpr int kDeep = sizeof(T) == 4 ? 3 : 2;
  const int shape = plan.fi * 10 + plan.fj;
  if constexpr (sizeof(T) == 4) {  // in fp64 its accumulators, sums and fragments exceed the registers
    if (shape == 44) return launch<T, 4, 4, 2>(ctx, plan, ta, tb, a, b, c, m, n, k, bd, batch);
  }
  if (shape == 42) launch<T, 4, 2, kDeep>(ctx, plan, ta, tb, a, b, c, m, n, k, bd, batch);
  else if (shape == 24) launch<T, 2, 4, kDeep>(ctx, plan, ta, tb, a, b, c, m, n, k, bd, batch);
  else if (shape == 22) launch<T, 2, 2, 4>(ctx, plan, ta, tb, a, b, c, m, n, k, bd, batch);
  else if (shape == 41) launch<T, 4, 1, 4>(ctx, plan, ta, tb, a, b, c, m, n, k, bd, batch);
  else if (shape == 14) launch<T, 1, 4, 4>(ctx, plan, ta, tb, a, b, c, m, n, k, bd, batch);
  else if (shape == 11) launch<T, 1, 1, 4>(ctx, plan, ta, tb, a, b, c, m, n, k, bd, batch);
  else hp::fail(HP_E_HIP, "internal: no such direct tile");
}

}  // namespace
