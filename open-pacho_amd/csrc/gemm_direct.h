// Direct MFMA products: operands go from global memory straight into the MFMA
// fragments, without LDS, for products too small, too narrow or too ragged to
// fill the chip with the LDS-staged tiles of gemm_kernels.h.
//
// A 256-thread workgroup owns a (16 FI) x (16 FJ) tile of C; each of its four
// waves computes the whole tile over every fourth 16-deep K slice, so waves
// share no operand and the K loop has no barrier and no LDS traffic. The four
// accumulator tiles are added in wave order through LDS at the end. Where the
// tiles alone would leave compute units idle, K is also cut into `splits` runs
// of slices, one workgroup each, whose tiles a second kernel adds in order. All
// orders are fixed by (m, n, k, batch) alone: repeated products, and products
// of stored and of transposed operands, agree bit for bit.
//
// A wave's slice is 16 bytes (two times 16 in fp64) per lane and fragment at
// element alignment, whatever the layout:
//   k-contiguous operand: lane l reads k = 4 (l / 16) .. + 3 of row 16 f + l % 16
//     of fragment f: one vector of the row;
//   row-contiguous operand: lane l reads rows F (l % 16) .. + F - 1 at each of
//     those four k: a vector of F rows, whose elements are fragments 0 .. F - 1.
// MFMA number q then contracts k = {q, 4 + q, 8 + q, 12 + q} for both kinds.
// Rows past the end read clamped addresses and feed outputs that are not
// stored; k past the end reads as +0 for both operands (one guarded slice).
//
// Bound by: MFMA issue in the 64 x 64 tile (fp32; 64 MFMAs per 8 KB of loads;
// DEPTH slices of registers keep the next loads in flight behind them), by the
// reads of the wide operand in the 16- and 32-row tiles.
#pragma once

#include "gemm.h"

namespace hpgemm {

// Tile and split chosen for a product; fi == 0: the product is not for these
// kernels.
struct DirectPlan {
  int fi = 0, fj = 0;
  int64_t tiles_m = 0, tiles_n = 0, tiles = 0, splits = 1, slices = 0, per_split = 0;
};

// By the product's extents alone.
DirectPlan direct_plan(int compute_units, int dtype, int64_t m, int64_t n, int64_t k, int64_t batch);

void direct_f32(hp_ctx* ctx, const DirectPlan& plan, bool ta, bool tb, const void* a, const void* b, void* c,
                int64_t m, int64_t n, int64_t k, const BatchDesc& bd, int64_t batch);
void direct_f64(hp_ctx* ctx, const DirectPlan& plan, bool ta, bool tb, const void* a, const void* b, void* c,
                int64_t m, int64_t n, int64_t k, const BatchDesc& bd, int64_t batch);

}  // namespace hpgemm
