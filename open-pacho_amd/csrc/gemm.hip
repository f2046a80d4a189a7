// GEMM entry points: C[b] = A[b'] @ B[b''] (hp_gemm) and the 2-D products
// with transposed operands (hp_gemm_layout). The kernels are described in
// gemm_kernels.h. Reference semantics: _gemm.py:24-137 (per-batch broadcast
// offsets _offset :13-21, never reads C), _cuda.py:493-518 and :619-636;
// transposed operands: _matmul_layout.py:9-48 (TransposedGemm.run).
#include <algorithm>

#include "gemm.h"
#include "gemm_direct.h"

namespace {

template <typename T>
__global__ __launch_bounds__(256) void zero_kernel(T* __restrict__ out, int64_t count) {
  for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < count; i += int64_t(gridDim.x) * 256) out[i] = T(0);
}

// Products of every layout: C[b] = op(A[b']) @ op(B[b'']).
void run(hp_ctx* ctx, int dtype, bool ta, bool tb, const void* a, const void* b, void* c, int64_t m, int64_t n,
         int64_t k, const hpgemm::BatchDesc& bd, int64_t batch) {
  const hpgemm::DirectPlan direct = hpgemm::direct_plan(ctx->compute_units, dtype, m, n, k, batch);
  if (direct.fi > 0 && !ctx->staged_products) {
    (dtype == HP_F32 ? hpgemm::direct_f32 : hpgemm::direct_f64)(ctx, direct, ta, tb, a, b, c, m, n, k, bd, batch);
    return;
  }
  static const hpgemm::Run table[2][4] = {
      {hpgemm::f32_nn, hpgemm::f32_tn, hpgemm::f32_nt, hpgemm::f32_tt},
      {hpgemm::f64_nn, hpgemm::f64_tn, hpgemm::f64_nt, hpgemm::f64_tt},
  };
  table[dtype == HP_F32 ? 0 : 1][(ta ? 1 : 0) + (tb ? 2 : 0)](ctx, a, b, c, m, n, k, bd, batch);
}

// Zero-fills C for k == 0 (no product launch).
void zero_output(hp_ctx* ctx, int dtype, void* c, int64_t outputs) {
  const int64_t grid = std::min<int64_t>(hp::ceil_div(outputs, 256), 65536);
  switch (dtype) {
    case HP_F32: zero_kernel<float><<<grid, 256, 0, ctx->stream>>>(static_cast<float*>(c), outputs); break;
    case HP_F64: zero_kernel<double><<<grid, 256, 0, ctx->stream>>>(static_cast<double*>(c), outputs); break;
    case HP_BOOL: zero_kernel<uint8_t><<<grid, 256, 0, ctx->stream>>>(static_cast<uint8_t*>(c), outputs); break;
    case HP_I32:
    case HP_U32: zero_kernel<uint32_t><<<grid, 256, 0, ctx->stream>>>(static_cast<uint32_t*>(c), outputs); break;
    default: zero_kernel<uint64_t><<<grid, 256, 0, ctx->stream>>>(static_cast<uint64_t*>(c), outputs); break;
  }
  hp::check_launch("gemm_zero");
}

// Integer and bool products, as NumPy computes them: sums of products in the
// operand type, wrapping modulo 2^bits (signed types are multiplied and added
// as unsigned words, whose two's-complement result is the same), and for bool
// the logical or of ands. Both are exact in any order, so this simple kernel
// is bit-identical to any other summation order (reference: the OpenCL
// backend's generic product, _opencl.py:386-420). One 256-thread workgroup
// per 16 x 16 output tile, 16-deep K slices staged in LDS.
template <typename W>
struct IntOps {
  static __device__ __forceinline__ W fma(W acc, W a, W b) { return acc + a * b; }
};
template <>
struct IntOps<uint8_t> {  // bool
  static __device__ __forceinline__ uint8_t fma(uint8_t acc, uint8_t a, uint8_t b) {
    return uint8_t(acc | ((a != 0) & (b != 0)));
  }
};

template <typename W>
__global__ __launch_bounds__(256) void int_gemm_kernel(const W* __restrict__ A, const W* __restrict__ B,
                                                       W* __restrict__ C, int64_t M, int64_t N, int64_t K,
                                                       hpgemm::BatchDesc bd, int64_t tiles_m, int64_t tiles_n) {
  __shared__ W As[16][17], Bs[16][17];
  const int64_t tile = blockIdx.x;
  const int64_t batch = tile / (tiles_m * tiles_n);
  const int64_t rest = tile - batch * tiles_m * tiles_n;
  const int64_t row = (rest / tiles_n) * 16 + (threadIdx.x >> 4);
  const int64_t col = (rest % tiles_n) * 16 + (threadIdx.x & 15);
  const int ty = threadIdx.x >> 4, tx = threadIdx.x & 15;
  int64_t a_off, b_off;
  hpgemm::batch_offsets(batch, bd, a_off, b_off);
  const W* a = A + a_off;
  const W* b = B + b_off;
  W acc = 0;
  for (int64_t k0 = 0; k0 < K; k0 += 16) {
    As[ty][tx] = row < M && k0 + tx < K ? a[row * K + k0 + tx] : W(0);
    Bs[ty][tx] = k0 + ty < K && col < N ? b[(k0 + ty) * N + col] : W(0);
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) acc = IntOps<W>::fma(acc, As[ty][kk], Bs[kk][tx]);
    __syncthreads();
  }
  if (row < M && col < N) C[batch * M * N + row * N + col] = acc;
}

void run_int(hp_ctx* ctx, int dtype, const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k,
             const hpgemm::BatchDesc& bd, int64_t batch) {
  const int64_t tiles_m = hp::ceil_div(m, 16), tiles_n = hp::ceil_div(n, 16);
  const int64_t grid = batch * tiles_m * tiles_n;
  hp::require(grid <= hp::kMaxGrid, "integer product has too many tiles for one launch");
#define PACHO_INT_GEMM(W)                                                                                   \
  int_gemm_kernel<W><<<grid, 256, 0, ctx->stream>>>(static_cast<const W*>(a), static_cast<const W*>(b),    \
                                                    static_cast<W*>(c), m, n, k, bd, tiles_m, tiles_n)
  switch (dtype) {
    case HP_BOOL: PACHO_INT_GEMM(uint8_t); break;
    case HP_I32:
    case HP_U32: PACHO_INT_GEMM(uint32_t); break;
    default: PACHO_INT_GEMM(uint64_t); break;
  }
#undef PACHO_INT_GEMM
  hp::check_launch("int_gemm");
}

}  // namespace

namespace {

// Whether the direct kernels take a product: where the LDS-staged tiles of
// gemm_kernels.h are mostly padding or too few for the chip. The direct kernels
// reach 55-65% of the MFMA rate whatever the shape; the staged ones 80-95% of
// it on large whole tiles, little where tiles are cut, and the fp64 ones need
// 256 x 128 outputs per workgroup. Lines between measurements on one MI355X, us
// staged / direct:
//   fp32, padding of the staged tiles (128 x 128, or 256 x 256 for more than
//   256 slices) over 40%: 16 x 8192 x 8192 (m, n, k) 273 / 47, 128 x 8192 x 8192
//   274 / 157, 202 x (29 x 18 x 936) 71 / 17; over 15%: 700 x 700 x 3000 49 / 34,
//   56 x (592 x 429 x 173) 100 / 99, 400 x 4000 x 2000 (3.2e9) 78 / 86; up to one
//   and a half 64 x 64 tiles per compute unit: 1000^3 33 / 25, 512 x 512 x 8192
//   70 / 54, 1200 x 1200 x 2000 (2.9e9) 64 / 64; else 1000 x 3000 x 333 35 / 39,
//   2500 x 2500 x 100 23 / 35. Products of the narrow kernel's extents stay
//   there (1024^3 21 / 24, 8 x 512^3 21 / 30).
//   fp64: 560 x 453 x 688 56 / 17, 1024^3 60 / 44, 128 x 8192 x 8192 577 / 303;
//   whole staged tiles on half of the chip 2048 x 2048 x 256 62 / 66; large
//   products 1200 x 1200 x 2000 125 / 133, 2048^3 277 / 299; the staged kernel
//   for any K (no multiple of 16) 1500^3 166 / 130, 2000 x 600 x 3000 178 / 134;
//   few slices in many tiles 3025 x 2024 x 75 33 / 55.
bool direct_serves(int64_t cus, int dtype, int64_t m, int64_t n, int64_t k, int64_t batch) {
  const double work = double(m) * double(n) * double(k) * double(batch);
  const int64_t slices = hp::ceil_div(k, 16);
  const double tiles64 = double(hp::ceil_div(m, 64)) * double(hp::ceil_div(n, 64)) * double(batch);
  const auto fill = [&](int64_t bm, int64_t bn) {
    return double(m) * double(n) / (double(hp::ceil_div(m, bm) * bm) * double(hp::ceil_div(n, bn) * bn));
  };
  if (dtype == HP_F64) {
    if (slices <= 8 && tiles64 > 2.0 * cus) return false;
    if (k % 16 == 0 && m % 256 == 0 && n % 128 == 0 && double(m / 256) * double(n / 128) * batch * 2 >= cus) return false;
    return fill(256, 128) < 0.6 || work <= 2.4e9 || (k % 16 != 0 && slices >= 64 && work <= 8e9);
  }
  const bool narrow = m % 64 == 0 && n % 64 == 0 && k % 16 == 0 && tiles64 >= cus && tiles64 <= 4.0 * cus &&
                      work <= double(cus) * double(1 << 23);
  if (narrow) return false;
  const double filled = slices > 256 ? fill(256, 256) : fill(128, 128);
  if (filled < 0.6) return work <= 9e9;
  if (filled < 0.85) return work <= 2.6e9;
  return tiles64 <= 1.5 * cus && work <= 2.2e9;
}

// Whether the staged kernels take a product of few K slices in less time than
// `p`. A direct tile costs a start, a merge of four waves' accumulators and a
// store, whatever K is: with one or two slices to a wave that is most of its
// time, while a staged tile starts its stores after a slice or two. Times, us,
// of rounds of one tile per compute unit: staged 128 x 128 in fp32 2.2 + 1.1 per
// slice, 3.5 + 2.3 where one extent is shorter than the tile and 6 + 4 where
// both are (4-byte loads); 256 x 128 in fp64 6 + 3.5 per slice, 4.3 with a K
// edge. Direct 64 x 64 in fp32 1.4 + 1.4 per slice of a wave, an eighth more with
// a K edge, smaller tiles 0.22 of it and the rest by area; 32 x 64 in fp64 2.6 +
// 1.5, 0.1 and the rest by area. Fitted to 25 shapes in both types with K from 4
// to 300 (staged | direct): 288 x (130 x 667 x 20) 61 | 107, 600 x (80 x 450 x 16)
// 51 | 92, x 64 112 | 105, 2000 x (100 x 100 x 8) 80 | 94, x 32 116 | 94, 5606 x 426
// x 25 10.4 | 12.7; fp64 290 x 3952 x 13 12 | 15, x 20 17 | 15, 288 x (130 x 667 x
// 200) 429 | 537, x 300 643 | 612.
bool staged_serves_few_slices(int64_t cus, int dtype, int64_t m, int64_t n, int64_t k, int64_t batch,
                              const hpgemm::DirectPlan& p) {
  const bool single = dtype == HP_F32;
  if (p.splits > 1 || p.tiles <= cus || p.slices > (single ? 16 : 24)) return false;
  const auto rounds = [&](int64_t tiles) { return double(hp::ceil_div(tiles, cus)); };
  const double slices = double(p.slices), steps = double(hp::ceil_div(p.slices, 4));
  const bool edge = k % 16 != 0;
  double staged, direct;
  if (single) {
    const int cut = (m < 128) + (n < 128);
    staged = cut == 0 ? 2.2 + 1.1 * slices : cut == 1 ? 3.5 + 2.3 * slices : 6 + 4 * slices;
    // Three of its workgroups share a compute unit, so that part of a round takes part of its time.
    staged *= 1.15 * std::max(1.0, double(hp::ceil_div(m, 128) * hp::ceil_div(n, 128) * batch) / double(cus));
    direct = 1.4 * (1 + steps) * (edge ? 1.125 : 1.0) * (0.22 + 0.78 * p.fi * p.fj / 16.0);
  } else {
    staged = 1.05 * (6 + (edge ? 4.3 : 3.5) * slices) * rounds(hp::ceil_div(m, 256) * hp::ceil_div(n, 128) * batch);
    direct = (2.6 + 1.5 * steps) * (0.1 + 0.9 * p.fi * p.fj / 8.0);
  }
  return staged < direct * rounds(p.tiles);
}

}  // namespace

// Tile and K split by the time they would take: a compute unit works off its
// workgroups' tiles one after the other, each wave a quarter of the slices, so
// a candidate costs (workgroups per compute unit, rounded up) x (MFMA blocks of
// the tile) x (slices per wave), over the share of the MFMA rate its loads let
// it reach, and a split the second kernel. `rate` and the overheads are fitted
// to sweeps of every tile and split over 24 shapes in both types; the choice
// was the fastest or within 6% of it on all but two.
hpgemm::DirectPlan hpgemm::direct_plan(int compute_units, int dtype, int64_t m, int64_t n, int64_t k, int64_t batch) {
  struct Candidate {
    int fi, fj;
    double rate;
  };
  static constexpr Candidate kCandidates[] = {{4, 4, 1.0},  {2, 4, 0.95}, {4, 2, 0.95}, {2, 2, 0.9},
                                              {1, 4, 0.75}, {4, 1, 0.75}, {1, 1, 0.5}};
  constexpr double kTile = 0.3, kSplit = 4.0;  // us: a workgroup's start and store; the second kernel
  DirectPlan best;
  if (!direct_serves(compute_units, dtype, m, n, k, batch)) return best;
  double least = 0;
  const int64_t slices = hp::ceil_div(k, 16);
  const double unit = dtype == HP_F32 ? 0.053 : 0.107;  // us: one block over one slice
  for (const Candidate& c : kCandidates) {
    if (c.fi * c.fj == 16 && dtype == HP_F64) continue;  // does not fit the registers
    // Tiles move inside the operands, which only one-block extents may undercut.
    if ((c.fi > 1 && m < 16 * c.fi) || (c.fj > 1 && n < 16 * c.fj)) continue;
    DirectPlan p;
    p.fi = c.fi;
    p.fj = c.fj;
    p.tiles_m = hp::ceil_div(m, 16 * c.fi);
    p.tiles_n = hp::ceil_div(n, 16 * c.fj);
    p.tiles = p.tiles_m * p.tiles_n * batch;
    p.slices = slices;
    for (int64_t splits = 1; splits <= 32; splits *= 2) {
      if (splits > 1 && (slices < 16 * splits || p.tiles * splits > 4 * int64_t(compute_units))) break;
      p.per_split = hp::ceil_div(slices, splits);
      p.splits = hp::ceil_div(slices, p.per_split);
      const double rounds = double(hp::ceil_div(p.tiles * p.splits, compute_units));
      const double cost = rounds * (c.fi * c.fj * unit / c.rate * double(hp::ceil_div(p.per_split, 4)) + kTile) +
                          (p.splits > 1 ? kSplit : 0.0);
      if (best.fi == 0 || cost < least) {
        best = p;
        least = cost;
      }
    }
  }
  return staged_serves_few_slices(compute_units, dtype, m, n, k, batch, best) ? DirectPlan{} : best;
}

using hp::guarded;
using hp::require;

extern "C" {

int hp_gemm(hp_ctx* ctx, int dtype, const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k,
            int batch_rank, const int64_t* batch_shape, const int64_t* a_batch_strides,
            const int64_t* b_batch_strides) {
  return guarded([&] {
    hp::enter(ctx);
    require(dtype >= HP_BOOL && dtype <= HP_F64, "unknown dtype code");
    require(m >= 0 && n >= 0 && k >= 0, "negative extent");
    require(batch_rank >= 0 && batch_rank <= 6, "batch rank must be <= 6");
    hpgemm::BatchDesc bd{};
    bd.rank = batch_rank;
    int64_t batch = 1;
    for (int d = 0; d < batch_rank; ++d) {
      require(batch_shape[d] >= 0, "negative batch extent");
      bd.shape[d] = batch_shape[d];
      bd.a_stride[d] = a_batch_strides[d];
      bd.b_stride[d] = b_batch_strides[d];
      batch *= batch_shape[d];
    }
    const int64_t outputs = batch * m * n;
    if (outputs == 0) return;
    require(c != nullptr, "null output");
    if (k == 0) {
      zero_output(ctx, dtype, c, outputs);
      return;
    }
    require(a != nullptr && b != nullptr, "null input");
    if (dtype == HP_F32 || dtype == HP_F64) {
      run(ctx, dtype, false, false, a, b, c, m, n, k, bd, batch);
    } else {
      run_int(ctx, dtype, a, b, c, m, n, k, bd, batch);
    }
  });
}

int hp_gemm_layout(hp_ctx* ctx, int dtype, const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k,
                   int transpose_a, int transpose_b) {
  return guarded([&] {
    hp::enter(ctx);
    require(dtype == HP_F32 || dtype == HP_F64, "gemm supports float32 and float64");
    require(m >= 0 && n >= 0 && k >= 0, "negative extent");
    if (m == 0 || n == 0) return;
    require(c != nullptr, "null output");
    if (k == 0) {
      zero_output(ctx, dtype, c, m * n);
      return;
    }
    require(a != nullptr && b != nullptr, "null input");
    hpgemm::BatchDesc bd{};
    run(ctx, dtype, transpose_a != 0, transpose_b != 0, a, b, c, m, n, k, bd, 1);
  });
}

int hp_debug_staged_products(hp_ctx* ctx, int on) {
  return guarded([&] {
    hp::enter(ctx);
    ctx->staged_products = on != 0;
  });
}

int hp_debug_direct_plan(int compute_units, int dtype, int64_t m, int64_t n, int64_t k, int64_t batch,
                         int64_t* plan) {
  return guarded([&] {
    require(dtype == HP_F32 || dtype == HP_F64, "gemm supports float32 and float64");
    require(compute_units > 0 && m > 0 && n > 0 && k > 0 && batch > 0 && plan != nullptr, "not a product");
    const hpgemm::DirectPlan p = hpgemm::direct_plan(compute_units, dtype, m, n, k, batch);
    plan[0] = 16 * p.fi;
    plan[1] = 16 * p.fj;
    plan[2] = p.splits;
  });
}

}  // extern "C"
