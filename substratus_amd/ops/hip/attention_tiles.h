// What the attention kernels of prompts and of training share: workgroups of four
// waves with 32 rows each, rows of the other side on their way through LDS, and
// operands of 32x32x16 products from there and from accumulators.
//
// Accumulators hold row (r & 3) + 8 (r >> 2) + 4 (lane >> 5) in register r, column
// lane & 31; a first operand has row lane & 31 and a second column lane & 31, both
// the inner places 8 (lane >> 5) on.
#pragma once

#include "common.h"

typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) short short4v;
typedef __attribute__((ext_vector_type(16))) float float16v;

namespace {

constexpr int WAVES = 4;
constexpr int ROWS = 32 * WAVES;      // keys, or queries, of a workgroup
constexpr int THREADS = WAVES * WAVE;
constexpr float LOG2E = 1.44269504088896340736f;
constexpr int BUFFER_FLAGS = 0x00020000;   // untyped, offset-checked

DEV_INLINE unsigned cvt_pk_bf16(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  typedef __attribute__((ext_vector_type(2))) float floatx2;
  return __builtin_bit_cast(
      unsigned, __builtin_convertvector((floatx2){lo, hi}, bf16x2));
}

DEV_INLINE float16v mma(short8 a, short8 b, float16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Place of 16 bytes of a row in LDS; rows by themselves would share banks.
template <int D>
DEV_INLINE int place(int row, int piece) {
  return row * (D / 8) + (piece ^ (D == 64 ? row & 7 : 2 * (row & 7)));
}

// 16 rows of a tile from `row` on as the inner dimension of a first operand whose
// rows are the 32 columns from 32 c on.
template <int D>
DEV_INLINE short8 turned(const uint4v* tile, int row, int c, int lane) {
  short4v part[2];
  #pragma unroll
  for (int sel = 0; sel < 2; ++sel) {
    const int r = row + (lane >> 5) * 8 + sel * 4 + (lane >> 2 & 3);
    const int piece = c * 4 + (lane >> 4 & 1) * 2 + (lane >> 1 & 1);
    const short* p = reinterpret_cast<const short*>(tile + place<D>(r, piece)) +
                     (lane & 1) * 4;
    part[sel] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) short4v*)p);
  }
  short8 f;
  #pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[i] = part[0][i];
    f[4 + i] = part[1][i];
  }
  return f;
}

// STEP rows of D numbers on their way from memory to LDS.
template <int D, int STEP>
struct Rows {
  static constexpr int ROW = D / 8, LOADS = STEP * ROW / THREADS;
  uint4v u[LOADS];

  // As a bounded buffer: rows from the `rows`th on are zero.
  DEV_INLINE void load(const bf16_t* p, int rows, int row_bytes, int tid) {
    const auto from = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(p), 0,
        (min(STEP, rows) - 1) * row_bytes + D * 2, BUFFER_FLAGS);
    #pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int at = i * THREADS + tid;
      u[i] = __builtin_amdgcn_raw_buffer_load_b128(
          from, at / ROW * row_bytes + at % ROW * 16, 0, 0);
    }
  }
  DEV_INLINE void store(uint4v* tile, int tid) const {
    #pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int at = i * THREADS + tid;
      tile[place<D>(at / ROW, at % ROW)] = u[i];
    }
  }
};

// Eight rows of an accumulator, two in a word, as half of a second operand's inner
// dimension of 16: the other half of the wave has the rows between.
DEV_INLINE short8 operand(const unsigned* w) {
  const auto a = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
  return __builtin_bit_cast(short8, (uint4v){a[0], b[0], a[1], b[1]});
}

// One wave per row and head.
template <int D>
__global__ void attn_bwd_delta_kernel(float* __restrict__ delta,
                                      const bf16_t* __restrict__ dout,
                                      const bf16_t* __restrict__ out,
                                      long rows) {
  const long wid = ((long)blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  const int lane = threadIdx.x % WAVE;
  const long nw = ((long)gridDim.x * blockDim.x) / WAVE;
  constexpr int DU = D / 2;           // uints (2 bf16) per row
  for (long r = wid; r < rows; r += nw) {
    const unsigned* dp = reinterpret_cast<const unsigned*>(dout + r * D);
    const unsigned* op = reinterpret_cast<const unsigned*>(out + r * D);
    float acc = 0.f;
    #pragma unroll
    for (int i = lane; i < DU; i += WAVE) {
      const float2 dv = unpack_bf16x2(dp[i]);
      const float2 ov = unpack_bf16x2(op[i]);
      acc += dv.x * ov.x + dv.y * ov.y;
    }
    acc = wave_sum(acc);
    if (lane == 0) delta[r] = acc;
  }
}

}  // namespace
