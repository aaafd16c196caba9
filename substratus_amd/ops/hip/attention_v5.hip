// Causal attention of packed prompts, and training's forward with log-sums; heads
// of a group share keys and values.
//
// A wave has 32 queries: Q in registers as the second operand of S^T = K Q^T, so a
// lane's scores are of one query and the softmax stays in its registers, with one
// exchange between the halves of a wave; weights become the second operand of
// O^T = V^T P the same way. Keys come by 64, one step of the running softmax each,
// in two places of LDS; the next are under way in registers. The maximum moves only
// where some query's has grown by more than 2^8 (the weights' sum is in 32 bits,
// the weights' largest is 2^8 then).
//
// Bound by vector arithmetic on scores: positions are compared on the diagonal
// only, scale and maximum are one operation, the longest rows begin first.
// Workgroups are of four waves, two or three on a CU, so that one's matrix products
// go beside another's arithmetic.
// us on a MI355X, before (eight waves, one workgroup a CU, a turned copy of V in
// LDS) and now, sequences x length:
//   71 heads on one of 64   1 x 1024 41 -> 33      2 x 2048 158 -> 120
//   of 128   16 on 16   3 x 777 41 -> 35           32 on 8   1 x 2000 83 -> 69
//            32 on 32   24 of 370 and less 95 -> 62
//                       5 of 1333 and less 135 -> 111   4 x 2048 202 -> 186
// (Of one tile per head, 1 x 128, either takes 15 to 19 with its launch.)
#include <type_traits>

#include "attention_tiles.h"

// ---- 32x32x16 fragment-map probe (GPU test: test_mfma32_fragment_layout)
__global__ void mfma32_probe_kernel(float* __restrict__ dout,  // [32, 32]
                                    const bf16_t* __restrict__ a,  // [32,16]
                                    const bf16_t* __restrict__ b) {  // [16,32]
  const int lane = threadIdx.x % WAVE;
  const int lo5 = lane & 31, hi = lane >> 5;
  short8 af, bf;
  #pragma unroll
  for (int j = 0; j < 8; ++j) {
    af[j] = *reinterpret_cast<const short*>(&a[lo5 * 16 + hi * 8 + j]);
    bf[j] = *reinterpret_cast<const short*>(&b[(hi * 8 + j) * 32 + lo5]);
  }
  float16v acc = {};
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, bf, acc, 0, 0, 0);
  #pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = (r & 3) + 8 * (r >> 2) + 4 * hi;
    dout[row * 32 + lo5] = acc[r];
  }
}

void launch_mfma32_probe(float* dout, const bf16_t* a, const bf16_t* b,
                         hipStream_t stream) {
  mfma32_probe_kernel<<<1, 64, 0, stream>>>(dout, a, b);
}

namespace {

template <int D>
__global__ __launch_bounds__(THREADS, D == 64 ? 3 : 2)
void attn_v5_kernel(bf16_t* __restrict__ out,      // [T, HQ, D]
                    const bf16_t* __restrict__ q,  // [T, HQ, D]
                    const bf16_t* __restrict__ k,  // [T, HKV, D]
                    const bf16_t* __restrict__ v,  // [T, HKV, D]
                    const int* __restrict__ seq_start,  // [S + 1]
                    int hq, int hkv, float scale,
                    float* __restrict__ lse) {     // [T, HQ] or null
  constexpr int KK = D / 16, DC = D / 32;
  constexpr int STEP = 64;                     // keys
  constexpr int PIECES = STEP * D / 8;
  __shared__ uint4v lds[4 * PIECES];           // two places of K and V
  auto tile = [&](int b, int of) { return lds + (2 * b + of) * PIECES; };

  const int s = blockIdx.x, head = blockIdx.y, kvh = head / (hq / hkv);
  const int base = seq_start[s];
  const int n = seq_start[s + 1] - base;
  // the last rows have the most keys: they begin first
  const int tile0 = (gridDim.z - 1 - blockIdx.z) * ROWS;
  if (tile0 >= n) return;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int lane = tid % WAVE, lo5 = lane & 31, hi = lane >> 5;
  const int q0 = tile0 + wave * 32;
  const int qpos = q0 + lo5;                   // the lane's query
  const int steps = (min(tile0 + ROWS, n) + STEP - 1) / STEP;

  short8 qreg[KK];
  const long row = (long)(base + min(qpos, n - 1)) * hq + head;
  #pragma unroll
  for (int c = 0; c < KK; ++c)
    qreg[c] = *reinterpret_cast<const short8*>(q + row * D + c * 16 + hi * 8);
  if (scale < 0.f) {             // the largest product has the largest score
    #pragma unroll
    for (int c = 0; c < KK; ++c) qreg[c] ^= (short)0x8000;
    scale = -scale;
  }
  const float scale2 = scale * LOG2E;

  float m = -INFINITY, l = 0.f;
  float16v o_t[DC];                            // [32 columns][the lane's query]
  #pragma unroll
  for (int c = 0; c < DC; ++c) o_t[c] = float16v{};

  Rows<D, STEP> next[2];
  auto fetch = [&](int kbase) {
    const long at = ((long)(base + kbase) * hkv + kvh) * D;
    next[0].load(k + at, n - kbase, hkv * D * 2, tid);
    next[1].load(v + at, n - kbase, hkv * D * 2, tid);
  };
  auto put = [&](int b) {
    next[0].store(tile(b, 0), tid);
    next[1].store(tile(b, 1), tid);
  };

  fetch(0);
  put(0);
  for (int i = 0; i < steps; ++i) {
    __syncthreads();
    const int b = i & 1, kbase = i * STEP;
    if (i + 1 < steps) fetch(kbase + STEP);
    if (q0 < n && kbase <= q0 + 31) {          // uniform
      float16v sacc[STEP / 32];
      #pragma unroll
      for (int sc = 0; sc < STEP / 32; ++sc) {
        sacc[sc] = float16v{};
        #pragma unroll
        for (int kk = 0; kk < KK; ++kk)
          sacc[sc] = mma(
              __builtin_bit_cast(
                  short8, tile(b, 0)[place<D>(sc * 32 + lo5, kk * 2 + hi)]),
              qreg[kk], sacc[sc]);
      }
      const bool edge = kbase + STEP - 1 > q0;           // uniform
      float mraw = -INFINITY;
      if (edge) {
        #pragma unroll
        for (int sc = 0; sc < STEP / 32; ++sc)
          #pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int kpos = kbase + sc * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi;
            if (kpos > qpos || kpos >= n) sacc[sc][r] = -INFINITY;
            mraw = fmaxf(mraw, sacc[sc][r]);
          }
      } else {
        #pragma unroll
        for (int sc = 0; sc < STEP / 32; ++sc)
          #pragma unroll
          for (int r = 0; r < 16; ++r) mraw = fmaxf(mraw, sacc[sc][r]);
      }
      mraw = across<32>(mraw, Larger{});
      const float mloc = mraw == -INFINITY ? mraw : mraw * scale2;
      constexpr float MOST = 8.f;
      float alpha = 1.f;
      // branches of whole waves: matrix instructions take all lanes
      if (!__all(mloc == -INFINITY || mloc - m <= MOST)) {
        const float mn = fmaxf(m, mloc);
        alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
        m = mn;
        #pragma unroll
        for (int c = 0; c < DC; ++c)
          #pragma unroll
          for (int r = 0; r < 16; ++r) o_t[c][r] *= alpha;
      }
      float rowsum = 0.f;
      unsigned w[STEP / 32][8];
      auto weigh = [&](auto holes) {
        #pragma unroll
        for (int sc = 0; sc < STEP / 32; ++sc)
          #pragma unroll
          for (int j = 0; j < 8; ++j) {
            float p[2];
            #pragma unroll
            for (int t = 0; t < 2; ++t) {
              const float x = sacc[sc][2 * j + t];
              p[t] = decltype(holes)::value && x == -INFINITY
                  ? 0.f : __builtin_amdgcn_exp2f(fmaf(x, scale2, -m));
            }
            rowsum += p[0] + p[1];
            w[sc][j] = cvt_pk_bf16(p[0], p[1]);
          }
      };
      if (edge || !__all(mloc != -INFINITY)) weigh(std::true_type{});
      else weigh(std::false_type{});
      rowsum = across<32>(rowsum, Plus{});
      l = l * alpha + rowsum;
      #pragma unroll
      for (int sc = 0; sc < STEP / 32; ++sc)
        #pragma unroll
        for (int g = 0; g < 2; ++g) {
          const short8 pb = operand(w[sc] + 4 * g);
          #pragma unroll
          for (int c = 0; c < DC; ++c)
            o_t[c] = mma(turned<D>(tile(b, 1), sc * 32 + g * 16, c, lane), pb,
                         o_t[c]);
        }
    }
    if (i + 1 < steps) put(b ^ 1);
  }

  if (qpos >= n) return;
  const float invl = l > 0.f ? 1.f / l : 0.f;
  bf16_t* to = out + row * D + 4 * hi;
  #pragma unroll
  for (int c = 0; c < DC; ++c)
    #pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<uint2*>(to + c * 32 + 2 * r) = make_uint2(
          cvt_pk_bf16(o_t[c][r] * invl, o_t[c][r + 1] * invl),
          cvt_pk_bf16(o_t[c][r + 2] * invl, o_t[c][r + 3] * invl));
  if (lse != nullptr && hi == 0) lse[row] = m + __builtin_amdgcn_logf(l);
}

}  // namespace

void launch_attn_v5(bf16_t* out, const bf16_t* q, const bf16_t* k,
                    const bf16_t* v, const int* seq_start, int num_seqs,
                    int max_len, int hq, int hkv, int d, float scale,
                    hipStream_t stream, float* lse) {
  const dim3 grid(num_seqs, hq, (max_len + ROWS - 1) / ROWS);
  auto kernel = d == 128 ? attn_v5_kernel<128> : attn_v5_kernel<64>;
  kernel<<<grid, dim3(THREADS), 0, stream>>>(out, q, k, v, seq_start, hq, hkv,
                                             scale, lse);
}

bool attn_v5_supported(int d) { return d == 128 || d == 64; }
