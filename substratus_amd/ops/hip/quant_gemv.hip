// Fused block-dequant GEMV + dequant kernels for GGUF-quantized weights
// (SURVEY.md §2.5 ledger item 8: "block-dequant fused into GEMV for
// single-token decode" — the first-party replacement for the reference's
// llama.cpp serving path).
//
// Weight storage (repacked at load from GGUF for aligned GPU access):
//   scales: fp16 [N, K/32]
//   qs:     q4_0 -> uint8 [N, K/2] (nibble i of byte b packs weights b and
//           b+16 of the 32-block: llama.cpp layout), q8_0 -> int8 [N, K]
//
// quant_gemv: one wave per output element row of one row of x, for what
// rows_quant.hip does not take (k no multiple of 64) and q8_0 with a single
// row of x, where that kernel's workgroups of 16 weight rows leave the chip
// unevenly filled (N=5120: 9.4 us here, 11.1 there); each lane owns blocks
// lane, lane+64, ... (scale 2 B + 16 B nibbles via uint4); x read through L2;
// wave-reduced fp32 accumulation.
//
// dequant (prefill / large M): block-parallel expansion to bf16, then the
// caller runs hipBLASLt.
#include "common.h"

typedef _Float16 f16_t;

template <bool Q8>
__global__ __launch_bounds__(256)
void quant_gemv_kernel(bf16_t* __restrict__ y,         // [M, N]
                       const bf16_t* __restrict__ x,   // [M, K]
                       const f16_t* __restrict__ scales,  // [N, K/32]
                       const unsigned char* __restrict__ qs,
                       int n, int k) {
  const int row = blockIdx.x * 4 + threadIdx.x / WAVE;  // 4 waves = 4 rows
  if (row >= n) return;
  x += (long)blockIdx.y * k;
  const int lane = threadIdx.x % WAVE;
  const int nblocks = k / 32;
  const f16_t* srow = scales + (long)row * nblocks;
  float acc = 0.f;

  if (!Q8) {
    const uint4* qrow = reinterpret_cast<const uint4*>(qs + (long)row * k / 2);
    for (int b = lane; b < nblocks; b += WAVE) {
      const uint4 nib = qrow[b];
      const unsigned int w[4] = {nib.x, nib.y, nib.z, nib.w};
      const uint4* xb = reinterpret_cast<const uint4*>(x + b * 32);
      uint4 xv[4];
      #pragma unroll
      for (int c = 0; c < 4; ++c) xv[c] = xb[c];
      float partial = 0.f;
      #pragma unroll
      for (int c = 0; c < 4; ++c) {   // 4 bytes -> weights i..i+3, i+16..19
        const uint4 lo4 = xv[c / 2], hi4 = xv[2 + c / 2];
        const unsigned int xlo[2] = {c % 2 == 0 ? lo4.x : lo4.z,
                                     c % 2 == 0 ? lo4.y : lo4.w};
        const unsigned int xhi[2] = {c % 2 == 0 ? hi4.x : hi4.z,
                                     c % 2 == 0 ? hi4.y : hi4.w};
        #pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float lo = (float)((w[c] >> (8 * j)) & 0xF) - 8.f;
          const float hi = (float)((w[c] >> (8 * j + 4)) & 0xF) - 8.f;
          const float2 xl = unpack_bf16x2(xlo[j / 2]);
          const float2 xh = unpack_bf16x2(xhi[j / 2]);
          partial += lo * (j % 2 == 0 ? xl.x : xl.y) +
                     hi * (j % 2 == 0 ? xh.x : xh.y);
        }
      }
      acc += partial * (float)srow[b];
    }
  } else {
    const uint4* qrow = reinterpret_cast<const uint4*>(qs + (long)row * k);
    for (int b = lane; b < nblocks; b += WAVE) {
      const float s = (float)srow[b];
      // 32 int8 = 2 x uint4
      const uint4 q0 = qrow[b * 2], q1 = qrow[b * 2 + 1];
      const unsigned int w[8] = {q0.x, q0.y, q0.z, q0.w,
                                 q1.x, q1.y, q1.z, q1.w};
      const uint4* xb = reinterpret_cast<const uint4*>(x + b * 32);
      uint4 xv[4];
      #pragma unroll
      for (int c = 0; c < 4; ++c) xv[c] = xb[c];
      float partial = 0.f;
      #pragma unroll
      for (int c = 0; c < 4; ++c) {
        const unsigned int xs[4] = {xv[c].x, xv[c].y, xv[c].z, xv[c].w};
        #pragma unroll
        for (int j = 0; j < 2; ++j) {  // 2 words of 4 int8 per uint4-pair
          const unsigned int word = w[c * 2 + j];
          #pragma unroll
          for (int t = 0; t < 4; ++t) {
            const float qv = (float)(signed char)((word >> (8 * t)) & 0xFF);
            const float2 xp = unpack_bf16x2(xs[j * 2 + t / 2]);
            partial += qv * ((t % 2 == 0) ? xp.x : xp.y);
          }
        }
      }
      acc += partial * s;
    }
  }
  const float v = wave_sum(acc);
  if (lane == 0) y[(long)blockIdx.y * n + row] = f2bf(v);
}

// expand quantized rows to bf16 (prefill path feeds hipBLASLt)
template <bool Q8>
__global__ void dequant_kernel(bf16_t* __restrict__ out,   // [N, K]
                               const f16_t* __restrict__ scales,
                               const unsigned char* __restrict__ qs,
                               long nblocks_total, int k) {
  // one 32-weight block per thread
  const long blk = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (blk >= nblocks_total) return;
  const int nb_per_row = k / 32;
  const long row = blk / nb_per_row;
  const int brow = (int)(blk % nb_per_row);
  const float s = (float)scales[blk];
  bf16_t* o = out + row * k + brow * 32;
  if (!Q8) {
    const unsigned char* q = qs + row * (long)(k / 2) + brow * 16;
    #pragma unroll
    for (int i = 0; i < 16; ++i) {
      const unsigned char byte = q[i];
      o[i] = f2bf(((float)(byte & 0xF) - 8.f) * s);
      o[i + 16] = f2bf(((float)(byte >> 4) - 8.f) * s);
    }
  } else {
    const signed char* q =
        reinterpret_cast<const signed char*>(qs) + row * (long)k + brow * 32;
    #pragma unroll
    for (int i = 0; i < 32; ++i) o[i] = f2bf((float)q[i] * s);
  }
}

void launch_quant_gemv(bf16_t* y, const bf16_t* x, const void* scales,
                       const unsigned char* qs, int m, int n, int k,
                       bool q8, hipStream_t stream) {
  dim3 grid((n + 3) / 4, m);
  dim3 block(256);
  const f16_t* sc = reinterpret_cast<const f16_t*>(scales);
  if (q8) {
    quant_gemv_kernel<true><<<grid, block, 0, stream>>>(y, x, sc, qs, n, k);
  } else {
    quant_gemv_kernel<false><<<grid, block, 0, stream>>>(y, x, sc, qs, n, k);
  }
}

void launch_dequant(bf16_t* out, const void* scales, const unsigned char* qs,
                    long n, int k, bool q8, hipStream_t stream) {
  const long nblocks = n * (long)(k / 32);
  const int bsz = 256;
  const long grid = (nblocks + bsz - 1) / bsz;
  const f16_t* sc = reinterpret_cast<const f16_t*>(scales);
  if (q8)
    dequant_kernel<true><<<dim3((unsigned)grid), dim3(bsz), 0, stream>>>(
        out, sc, qs, nblocks, k);
  else
    dequant_kernel<false><<<dim3((unsigned)grid), dim3(bsz), 0, stream>>>(
        out, sc, qs, nblocks, k);
}
