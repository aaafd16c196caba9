// Products of 17 to 256 rows with a weight matrix (mid_gemm.hip).
#pragma once

#include "rows_gemm.h"

// y [m, n] = x w^T + bias
struct MidGemm {
  bf16_t* y;
  const bf16_t *x, *w, *bias;
  int m, n, k;
  long x_ld, y_ld;
  // set by launch_mid_gemm: blocks of rows; y's columns come in aligned fours
  int blocks;
  bool quads;
};

// A workgroup's rows (32, 64, 96 or 128) and tiles of 16 columns (4 or 8), and
// the workgroups that share the inner dimension.
struct MidPlan {
  int rows, tiles, splits;
  double us;                      // what it is to take
  long shares(long m, long n) const {     // floats
    return splits > 1 ? splits * m * ((n + 15) / 16 * 16) : 0;
  }
};

// What follows the sums of shares, where each row's are one workgroup's: total = h +
// the product's row, y the RMSNorm of that.
struct MidNorm {
  const bf16_t *h, *weight;
  bf16_t* total;
  float eps;
};

bool mid_gemm_takes(long m, long n, long k, bool paired);
MidPlan mid_gemm_plan(long m, long n, long k);
bool mid_gemm_pays(long m, long n, long k, bool paired, bool normed = false);
bool mid_norm_takes(long m, long n, long k);
void launch_mid_gemm(const MidGemm& a, const MidPlan& plan, const Heads* heads,
                     bool gated, bool gelu, const MidNorm* norm, float* part,
                     hipStream_t stream);
