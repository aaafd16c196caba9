// Backward of causal attention in training, of packed sequences; heads of a
// group share keys and values, which are not repeated.
//
//   Delta = sum over columns of dO O
//   S  = Q K^T             P  = exp2(S scale log2(e) - L)
//   dP = dO V^T            dS = P (dP - Delta)
//   dQ = dS K scale        dK = dS^T Q scale        dV = P^T dO
//
// L: the forward's log-sums, in powers of two.
//
// Keys and values: a wave has 32 keys, K and V in registers as second operands,
// dK^T and dV^T in accumulators. Queries come by 64, of some heads of a group one
// after the other. The scores' accumulators hold a key per lane and queries in
// registers, so P and dS become operands of dV^T = dO^T P and dK^T = Q^T dS by
// exchanges between the halves of a wave, with no way through memory. Queries:
// the same with their parts exchanged, dQ^T = K^T dS^T.
//
// Bound by LDS and by vector arithmetic on scores beside the matrix cores. Hence
// 32 keys for every operand that is read (16 read each twice as often), and one
// copy of Q and dO, which transposing reads turn where that is needed. The next
// rows are on their way, in registers, while these are taken, and go to the other
// of two places, so a step has one barrier. Workgroups are of four waves, so that
// one's matrix products go beside another's vector arithmetic: two or three of
// them share a CU but in the keys' kernel of 128 columns, whose accumulators take
// the registers of two (with V in LDS and half as many queries at a time, two
// took half as long again: registers spilled).
//
// us of the backward on a MI355X, before (16 keys of a wave, or 32 of eight
// waves; two copies of each tile, waited for) and now; sequences x length, heads:
//   71 on one of 64    1 x 1024 128 -> 98      2 x 2048 554 -> 359
//                      1 x 128 31 -> 27        2 x 8192 6046 -> 4741
//   of 128     16 on 16   3 x 777 111 -> 84    1 x 128 32 -> 31
//              32 on 32   4 x 2048 929 -> 700
//              32 on 8    8 x 2048 1602 -> 1224      1 x 8192 2950 -> 2149
#include <algorithm>
#include <type_traits>

#include "attention_tiles.h"

namespace {

template <int D>
__global__ __launch_bounds__(THREADS, D == 64 ? 2 : 1)
void attn_bwd_dkv_kernel(float* __restrict__ dk,          // [T, HKV, D]
                         float* __restrict__ dv,
                         const bf16_t* __restrict__ q,    // [T, HQ, D]
                         const bf16_t* __restrict__ k,    // [T, HKV, D]
                         const bf16_t* __restrict__ v,
                         const bf16_t* __restrict__ dout,
                         const float* __restrict__ lse,   // [T, HQ]
                         const float* __restrict__ delta,
                         const int* __restrict__ seq_start, int hq, int hkv,
                         int most, float scale) {
  constexpr int KK = D / 16, DC = D / 32;
  constexpr int STEP = 64;
  constexpr int PIECES = STEP * D / 8;         // of a tile, 16 bytes each
  constexpr int OUT = D + 4;                   // floats of a key on the way out
  // two places of Q and dO; the results on their way out
  __shared__ uint4v lds[4 * PIECES];
  __shared__ alignas(16) float stats[2][2][STEP];
  static_assert(sizeof(lds) >= WAVES * 16 * OUT * sizeof(float));
  auto tile = [&](int b, int of) { return lds + (2 * b + of) * PIECES; };

  const int s = blockIdx.x;
  const int grp = hq / hkv;
  const int per = (grp + most - 1) / most;     // workgroups of a group
  const int kvh = blockIdx.y / per;
  const int head0 = kvh * grp + blockIdx.y % per * most;
  const int heads = min(most, (kvh + 1) * grp - head0);
  const int base = seq_start[s];
  const int n = seq_start[s + 1] - base;
  const int tile0 = blockIdx.z * ROWS;
  if (tile0 >= n) return;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int lane = tid % WAVE, lo5 = lane & 31, hi = lane >> 5;
  const int kv0 = tile0 + wave * 32;
  const int kpos = kv0 + lo5;                  // the lane's key
  const int first = tile0 / STEP;              // no query before it sees a key
  const int steps = (n + STEP - 1) / STEP - first;

  short8 kreg[KK], vreg[KK];
  {
    const long at = ((long)(base + min(kpos, n - 1)) * hkv + kvh) * D + hi * 8;
    #pragma unroll
    for (int c = 0; c < KK; ++c) {
      kreg[c] = *reinterpret_cast<const short8*>(k + at + c * 16);
      vreg[c] = *reinterpret_cast<const short8*>(v + at + c * 16);
    }
  }
  float16v dk_t[DC], dv_t[DC];                 // [32 columns][the lane's key]
  #pragma unroll
  for (int c = 0; c < DC; ++c) dk_t[c] = dv_t[c] = float16v{};
  const float scale2 = scale * LOG2E;

  Rows<D, STEP> next[2];
  float stat;
  auto fetch = [&](int head, int qbase) {
    const long at = ((long)(base + qbase) * hq + head) * D;
    next[0].load(q + at, n - qbase, hq * D * 2, tid);
    next[1].load(dout + at, n - qbase, hq * D * 2, tid);
    const float* of = tid & STEP ? delta : lse;
    stat = of[(long)(base + min(qbase + tid % STEP, n - 1)) * hq + head];
  };
  auto put = [&](int b) {
    next[0].store(tile(b, 0), tid);
    next[1].store(tile(b, 1), tid);
    if (tid < 2 * STEP) stats[b][tid / STEP][tid % STEP] = stat;
  };

  fetch(head0, first * STEP);
  put(0);
  int head = head0, qc = first;
  const int all_steps = heads * steps;
  for (int i = 0; i < all_steps; ++i) {
    __syncthreads();
    const int b = i & 1, qbase = qc * STEP;
    if (++qc == first + steps) {
      qc = first;
      ++head;
    }
    if (i + 1 < all_steps) fetch(head, qc * STEP);
    #pragma unroll
    for (int sc = 0; sc < STEP / 32; ++sc) {
      const int q0 = qbase + sc * 32;
      if (q0 + 31 < kv0 || q0 >= n) continue;            // uniform
      float16v sacc = {}, dpacc = {};
      #pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        const int at = place<D>(sc * 32 + lo5, kk * 2 + hi);
        sacc = mma(__builtin_bit_cast(short8, tile(b, 0)[at]), kreg[kk], sacc);
        dpacc = mma(__builtin_bit_cast(short8, tile(b, 1)[at]), vreg[kk],
                    dpacc);
      }
      unsigned wp[8], wd[8];
      auto scores = [&](auto inside) {
        #pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int at = sc * 32 + 8 * g + 4 * hi;
          const float4 l = *reinterpret_cast<const float4*>(&stats[b][0][at]);
          const float4 d = *reinterpret_cast<const float4*>(&stats[b][1][at]);
          const float lq[4] = {l.x, l.y, l.z, l.w};
          const float dq[4] = {d.x, d.y, d.z, d.w};
          float p[4], ds[4];
          #pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int qpos = qbase + at + t;
            p[t] = decltype(inside)::value ||
                           (qpos >= kpos && qpos < n && kpos < n)
                ? __builtin_amdgcn_exp2f(
                      fmaf(sacc[4 * g + t], scale2, -lq[t]))
                : 0.f;
            ds[t] = p[t] * (dpacc[4 * g + t] - dq[t]);
          }
          #pragma unroll
          for (int t = 0; t < 2; ++t) {
            wp[2 * g + t] = cvt_pk_bf16(p[2 * t], p[2 * t + 1]);
            wd[2 * g + t] = cvt_pk_bf16(ds[2 * t], ds[2 * t + 1]);
          }
        }
      };
      // positions are compared at the edges only
      if (q0 >= kv0 + 31 && q0 + 31 < n) scores(std::true_type{});
      else scores(std::false_type{});
      #pragma unroll
      for (int g = 0; g < 2; ++g) {
        const short8 pb = operand(wp + 4 * g), db = operand(wd + 4 * g);
        #pragma unroll
        for (int c = 0; c < DC; ++c) {
          const int row = sc * 32 + g * 16;
          dv_t[c] = mma(turned<D>(tile(b, 1), row, c, lane), pb, dv_t[c]);
          dk_t[c] = mma(turned<D>(tile(b, 0), row, c, lane), db, dk_t[c]);
        }
      }
    }
    if (i + 1 < all_steps) put(b ^ 1);
  }

  // A group's only workgroup stores four numbers of a key at a time.
  if (per == 1) {
    if (kpos >= n) return;
    const long at = ((long)(base + kpos) * hkv + kvh) * D + 4 * hi;
    #pragma unroll
    for (int c = 0; c < DC; ++c)
      #pragma unroll
      for (int r = 0; r < 16; r += 4) {
        const int d = c * 32 + 2 * r;
        *reinterpret_cast<float4*>(dk + at + d) =
            make_float4(dk_t[c][r] * scale, dk_t[c][r + 1] * scale,
                        dk_t[c][r + 2] * scale, dk_t[c][r + 3] * scale);
        *reinterpret_cast<float4*>(dv + at + d) =
            make_float4(dv_t[c][r], dv_t[c][r + 1], dv_t[c][r + 2],
                        dv_t[c][r + 3]);
      }
    return;
  }
  // Others go through LDS, 16 keys at a time, so that a wave's additions to
  // memory go to consecutive numbers.
  __syncthreads();
  float* out = reinterpret_cast<float*>(lds) + wave * 16 * OUT;
  auto leave = [&](float* to, const float16v* acc, float by) {
    #pragma unroll
    for (int h = 0; h < 2; ++h) {
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      if ((lo5 >> 4) == h) {
        #pragma unroll
        for (int c = 0; c < DC; ++c)
          #pragma unroll
          for (int r = 0; r < 16; ++r)
            out[(lo5 & 15) * OUT + c * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi] =
                acc[c][r] * by;
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      float f[16][D / WAVE];
      #pragma unroll
      for (int i = 0; i < 16; ++i)
        #pragma unroll
        for (int j = 0; j < D / WAVE; ++j)
          f[i][j] = out[i * OUT + j * WAVE + lane];
      #pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = kv0 + h * 16 + i;
        if (key >= n) break;
        float* at = to + ((long)(base + key) * hkv + kvh) * D + lane;
        #pragma unroll
        for (int j = 0; j < D / WAVE; ++j)
          unsafeAtomicAdd(at + j * WAVE, f[i][j]);
      }
    }
  };
  leave(dk, dk_t, scale);
  leave(dv, dv_t, 1.f);
}

// Gradients of queries, the same way about: a wave has 32 queries, Q and dO in
// registers, and dQ^T = K^T dS^T in accumulators; keys come by 64.
template <int D>
__global__ __launch_bounds__(THREADS, D == 64 ? 3 : 2)
void attn_bwd_dq_kernel(bf16_t* __restrict__ dq,          // [T, HQ, D]
                        const bf16_t* __restrict__ q,     // [T, HQ, D]
                        const bf16_t* __restrict__ k,     // [T, HKV, D]
                        const bf16_t* __restrict__ v,
                        const bf16_t* __restrict__ dout,
                        const float* __restrict__ lse,    // [T, HQ]
                        const float* __restrict__ delta,
                        const int* __restrict__ seq_start, int hq, int hkv,
                        float scale) {
  constexpr int KK = D / 16, DC = D / 32;
  constexpr int STEP = D == 64 ? 64 : 32;
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

  short8 qreg[KK], doreg[KK];
  const long row = (long)(base + min(qpos, n - 1)) * hq + head;
  #pragma unroll
  for (int c = 0; c < KK; ++c) {
    qreg[c] = *reinterpret_cast<const short8*>(q + row * D + c * 16 + hi * 8);
    doreg[c] =
        *reinterpret_cast<const short8*>(dout + row * D + c * 16 + hi * 8);
  }
  const float lq = lse[row], dlt = delta[row];
  float16v dq_t[DC];                           // [32 columns][the lane's query]
  #pragma unroll
  for (int c = 0; c < DC; ++c) dq_t[c] = float16v{};
  const float scale2 = scale * LOG2E;

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
    #pragma unroll
    for (int sc = 0; sc < STEP / 32; ++sc) {
      const int k0 = kbase + sc * 32;
      if (k0 > q0 + 31 || q0 >= n) continue;   // uniform
      float16v sacc = {}, dpacc = {};
      #pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        const int at = place<D>(sc * 32 + lo5, kk * 2 + hi);
        sacc = mma(__builtin_bit_cast(short8, tile(b, 0)[at]), qreg[kk], sacc);
        dpacc = mma(__builtin_bit_cast(short8, tile(b, 1)[at]), doreg[kk],
                    dpacc);
      }
      unsigned w[8];
      auto scores = [&](auto inside) {
        #pragma unroll
        for (int i = 0; i < 8; ++i) {
          float ds[2];
          #pragma unroll
          for (int t = 0; t < 2; ++t) {
            const int r = 2 * i + t;
            const int kpos = k0 + (r & 3) + 8 * (r >> 2) + 4 * hi;
            const float p = decltype(inside)::value || kpos <= qpos
                ? __builtin_amdgcn_exp2f(fmaf(sacc[r], scale2, -lq)) : 0.f;
            ds[t] = p * (dpacc[r] - dlt);
          }
          w[i] = cvt_pk_bf16(ds[0], ds[1]);
        }
      };
      // positions are compared on the diagonal only
      if (k0 + 31 <= q0) scores(std::true_type{});
      else scores(std::false_type{});
      #pragma unroll
      for (int g = 0; g < 2; ++g) {
        const short8 db = operand(w + 4 * g);
        #pragma unroll
        for (int c = 0; c < DC; ++c)
          dq_t[c] = mma(turned<D>(tile(b, 0), sc * 32 + g * 16, c, lane), db,
                        dq_t[c]);
      }
    }
    if (i + 1 < steps) put(b ^ 1);
  }
  if (qpos >= n) return;
  bf16_t* to = dq + row * D + 4 * hi;
  #pragma unroll
  for (int c = 0; c < DC; ++c)
    #pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<uint2*>(to + c * 32 + 2 * r) = make_uint2(
          cvt_pk_bf16(dq_t[c][r] * scale, dq_t[c][r + 1] * scale),
          cvt_pk_bf16(dq_t[c][r + 2] * scale, dq_t[c][r + 3] * scale));
}

}  // namespace

void launch_attn_bwd_delta(float* delta, const bf16_t* dout,
                           const bf16_t* out, long rows, int d,
                           hipStream_t stream) {
  const int threads = 256;
  const long waves = (rows + 3) / 4;
  const int blocks = (int)min(waves, (long)2048);
  if (d == 128)
    attn_bwd_delta_kernel<128><<<blocks, threads, 0, stream>>>(
        delta, dout, out, rows);
  else
    attn_bwd_delta_kernel<64><<<blocks, threads, 0, stream>>>(
        delta, dout, out, rows);
}

// Query heads of a group whose shares of dK and dV a workgroup adds up in
// registers before its atomic additions. More of them leave too few workgroups.
// us of the backward on a MI355X with 1, 2, 4 heads (sequences x length):
//   71 on 1 of 64   1 x 1024  105  113  166      2 x 2048  518  425  459
//                   8 x 2048 1803 1662 1581     16 x 512   514  416  367
//   32 on 8 of 128  2 x 512    83   98  140      2 x 2048  405  355  473
//                   8 x 2048 1589 1444 1359      8 x 512   232  181  176
int attn_bwd_heads(int num_seqs, int max_len, int hq, int hkv) {
  const long all = (long)num_seqs * hq * ((max_len + ROWS - 1) / ROWS);
  return std::min(all >= 4096 ? 4 : all >= 640 ? 2 : 1, hq / hkv);
}

bool attn_bwd_supported(int d) { return d == 128 || d == 64; }

void launch_attn_bwd_dq(bf16_t* dq, const bf16_t* q, const bf16_t* k,
                        const bf16_t* v, const bf16_t* dout, const float* lse,
                        const float* delta, const int* seq_start, int num_seqs,
                        int max_len, int hq, int hkv, int d, float scale,
                        hipStream_t stream) {
  const dim3 grid(num_seqs, hq, (max_len + ROWS - 1) / ROWS);
  auto kernel = d == 128 ? attn_bwd_dq_kernel<128> : attn_bwd_dq_kernel<64>;
  kernel<<<grid, dim3(THREADS), 0, stream>>>(dq, q, k, v, dout, lse, delta,
                                             seq_start, hq, hkv, scale);
}

void launch_attn_bwd_dkv(float* dk, float* dv, const bf16_t* q,
                         const bf16_t* k, const bf16_t* v, const bf16_t* dout,
                         const float* lse, const float* delta,
                         const int* seq_start, int num_seqs, int max_len,
                         int hq, int hkv, int d, float scale,
                         hipStream_t stream) {
  const int most = attn_bwd_heads(num_seqs, max_len, hq, hkv);
  const dim3 grid(num_seqs, hkv * ((hq / hkv + most - 1) / most),
                  (max_len + ROWS - 1) / ROWS);
  auto kernel = d == 128 ? attn_bwd_dkv_kernel<128> : attn_bwd_dkv_kernel<64>;
  kernel<<<grid, dim3(THREADS), 0, stream>>>(dk, dv, q, k, v, dout, lse, delta,
                                             seq_start, hq, hkv, most, scale);
}
