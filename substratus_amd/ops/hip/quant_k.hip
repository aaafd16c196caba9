// K-quant (GGUF Q4_K / Q6_K) dequantization — the super-block formats real
// ecosystem *.Q4_K_M.gguf files use (the reference served them through
// llama.cpp; models/gguf.py has the codec spec and the torch reference this
// is parity-tested against). Products of few rows: rows_quant.hip.
//
// Storage (repacked at load by models/quant.py repack_k for aligned GPU
// access; llama.cpp's packed blocks are 144/210 bytes — 210 is not even
// 4-aligned):
//   q4_K: scales fp16 [N, 2*SB] (d, dmin interleaved per super-block);
//         qs uint8 [N, SB*8 (6-bit sc) | SB*8 (6-bit mn) | K/2 nibbles]
//   q6_K: scales fp16 [N, SB] (d); qs uint8 [N, K/2 ql | K/4 qh | K/16 sc]
//   SB = K/256 super-blocks per row.
#include "common.h"

typedef _Float16 f16_t;

namespace quantk {

// ---- dequant (prefill / large-M path: expand to bf16, hipBLASLt after)
template <bool Q6>
__global__ void dequant_k_kernel(bf16_t* __restrict__ out,  // [N, K]
                                 const f16_t* __restrict__ scales,
                                 const unsigned char* __restrict__ qs,
                                 int n, int k) {
  const int sb = k / 256;
  const long total = (long)n * (Q6 ? k / 128 : k / 64);
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < total;
       t += (long)gridDim.x * blockDim.x) {
    if (!Q6) {
      const int row = (int)(t / (k / 64));
      const int c = (int)(t % (k / 64));
      const int s = c >> 2, qt = c & 3;
      const long row_q = (long)row * (sb * 16 + k / 2);
      const unsigned char* scb = qs + row_q;
      const unsigned char* mnb = scb + sb * 8;
      const unsigned char* nib = mnb + sb * 8 + c * 32;
      const f16_t* sr = scales + (long)row * 2 * sb;
      const float d = (float)sr[2 * s], dm = (float)sr[2 * s + 1];
      const float sc0 = d * scb[s * 8 + 2 * qt];
      const float sc1 = d * scb[s * 8 + 2 * qt + 1];
      const float m0 = dm * mnb[s * 8 + 2 * qt];
      const float m1 = dm * mnb[s * 8 + 2 * qt + 1];
      bf16_t* op = out + (long)row * k + c * 64;
      for (int l = 0; l < 32; ++l) {
        const unsigned b = nib[l];
        op[l] = f2bf(sc0 * (float)(b & 0xF) - m0);
        op[l + 32] = f2bf(sc1 * (float)(b >> 4) - m1);
      }
    } else {
      const int row = (int)(t / (k / 128));
      const int c = (int)(t % (k / 128));
      const int s = c >> 1, hf = c & 1;
      const long row_q = (long)row * (k / 2 + k / 4 + k / 16);
      const unsigned char* qlb = qs + row_q + s * 128 + hf * 64;
      const unsigned char* qhb = qs + row_q + k / 2 + s * 64 + hf * 32;
      const signed char* scl = reinterpret_cast<const signed char*>(
          qs + row_q + k / 2 + k / 4) + s * 16 + hf * 8;
      const float d = (float)scales[(long)row * sb + s];
      bf16_t* op = out + (long)row * k + s * 256 + hf * 128;
      for (int l = 0; l < 32; ++l) {
        const unsigned lo1 = qlb[l], lo2 = qlb[l + 32], h = qhb[l];
        const int e0 = (int)((lo1 & 0xF) | ((h & 3) << 4)) - 32;
        const int e1 = (int)((lo2 & 0xF) | (((h >> 2) & 3) << 4)) - 32;
        const int e2 = (int)((lo1 >> 4) | (((h >> 4) & 3) << 4)) - 32;
        const int e3 = (int)((lo2 >> 4) | (((h >> 6) & 3) << 4)) - 32;
        op[l] = f2bf(d * (float)scl[0 + (l >> 4)] * e0);
        op[l + 32] = f2bf(d * (float)scl[2 + (l >> 4)] * e1);
        op[l + 64] = f2bf(d * (float)scl[4 + (l >> 4)] * e2);
        op[l + 96] = f2bf(d * (float)scl[6 + (l >> 4)] * e3);
      }
    }
  }
}

}  // namespace quantk

void launch_dequant_k(bf16_t* out, const void* scales,
                      const unsigned char* qs, int n, int k, bool q6,
                      hipStream_t stream) {
  const long chunks = (long)n * (q6 ? k / 128 : k / 64);
  const int blocks = (int)min((chunks + 255) / 256, (long)4096);
  if (q6)
    quantk::dequant_k_kernel<true><<<blocks, 256, 0, stream>>>(
        out, (const f16_t*)scales, qs, n, k);
  else
    quantk::dequant_k_kernel<false><<<blocks, 256, 0, stream>>>(
        out, (const f16_t*)scales, qs, n, k);
}
