// Products of matrices of many rows (tile_gemm.hip).
#pragma once

#include "common.h"

// How a product's tiles are spread: the first `whole` by a workgroup each,
// each of the others by `split` workgroups that share the inner dimension.
struct TilePlan {
  int rows;                       // of a tile: a multiple of 32, 128 to 256
  int tiles_m, tiles_n, whole, split;
  __host__ __device__ int rest() const { return tiles_m * tiles_n - whole; }
  // floats of the shares
  long shares() const {
    return split > 1 ? (long)rest() * split * rows * 256 : 0;
  }
  double us;                      // what it is to take
};

// out [m, n] = a b^T + bias, all bf16 and sums in 32 bits. An operand has its
// rows of the inner dimension k contiguous, ld apart; or, if flipped, is
// stored the other way, with rows of m (or n) contiguous, ld apart.
struct TileGemm {
  bf16_t* out;
  const bf16_t *a, *b, *bias;
  int m, n, k;
  long a_ld, b_ld;
  bool a_flipped, b_flipped;
  // the first n / 2 columns gate the others: out [m, n / 2] = silu(gate) * up
  bool gated;
  // out is the gelu of the rounded columns; of operands that are not flipped
  bool gelu;
};

bool tile_gemm_takes(long m, long n, long k, long a_ld, long b_ld,
                     bool a_flipped, bool b_flipped, bool gated);
TilePlan tile_gemm_plan(long m, long n, long k, bool a_flipped,
                        bool b_flipped);
bool tile_gemm_pays(long m, long n, long k, bool a_flipped, bool b_flipped,
                    bool gated);
void launch_tile_gemm(const TileGemm& g, const TilePlan& plan, float* shares,
                      hipStream_t stream);
