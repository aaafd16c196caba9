// Fused sampling kernel: temperature / top-k /
// top-p + inverse-CDF draw, one workgroup per logits row.
//
// A row is read once, 16 bytes per load, and stays in registers as
// exp(x/T - max): a thread has 8 consecutive logits of every 8192. Thresholds
// are searched over the logits' own ordered bit patterns, so that 16 steps
// (32-bit logits: 32) end on an exact logit: top-k counts what is not below
// (one comparison per logit, a wave's count out of its mask), top-p adds it
// up. A step costs one barrier.
//
// Bound by the chain of steps; one row occupies a CU. On a MI355X, 192 rows
// of 32000, a quarter each greedy and top-k, half top-p: 32 us (292 us with
// the row in LDS, 256 threads and 24 halvings of the value range per
// threshold). 256 rows of 65024: 27 us greedy, 89 without thresholds, 123
// with them as above (87, 133, 594); registers spill from 32768 logits on.
#include "common.h"

#define SBLOCK 1024
#define SNW (SBLOCK / WAVE)
#define SVEC 8                    // consecutive logits of a thread per round
#define SROUND (SBLOCK * SVEC)
#define RUNS 256                  // runs of tokens that a draw's edges are of

namespace {

DEV_INLINE float val(const bf16_t& v) { return bf2f(v); }
DEV_INLINE float val(const float& v) { return v; }

// Ordered bit patterns: a <= b as floats just if key(a) <= key(b).
template <class T> struct Key;
template <> struct Key<bf16_t> {
  static constexpr unsigned TOP = 0x8000u, ALL = 0xffffu;
  DEV_INLINE static unsigned bits(float f) { return __float_as_uint(f) >> 16; }
  DEV_INLINE static float number(unsigned b) { return __uint_as_float(b << 16); }
};
template <> struct Key<float> {
  static constexpr unsigned TOP = 0x80000000u, ALL = 0xffffffffu;
  DEV_INLINE static unsigned bits(float f) { return __float_as_uint(f); }
  DEV_INLINE static float number(unsigned b) { return __uint_as_float(b); }
};
template <class T> DEV_INLINE unsigned key_of(float f) {
  const unsigned b = Key<T>::bits(f);
  return b & Key<T>::TOP ? Key<T>::ALL ^ b : b | Key<T>::TOP;
}
template <class T> DEV_INLINE float of_key(unsigned k) {
  return Key<T>::number(k & Key<T>::TOP ? k ^ Key<T>::TOP : Key<T>::ALL ^ k);
}

// VEC: the row is whole 16-byte pieces, of which each is there or not.
template <class T, bool VEC>
DEV_INLINE void load8(const T* row, int at, int vocab, float v[SVEC]) {
  constexpr int PER = 16 / sizeof(T);
  #pragma unroll
  for (int p = 0; p < SVEC; p += PER) {
    if constexpr (VEC) {
      const int from = at + p < vocab ? at + p : 0;
      const uint4v u = *reinterpret_cast<const uint4v*>(row + from);
      #pragma unroll
      for (int j = 0; j < PER; ++j)
        v[p + j] = at + p >= vocab ? -INFINITY
            : sizeof(T) == 4 ? __uint_as_float(u[j % 4])
            : __uint_as_float(j & 1 ? u[j / 2] & 0xffff0000u : u[j / 2] << 16);
    } else {
      #pragma unroll
      for (int j = 0; j < PER; ++j)
        v[p + j] = at + p + j < vocab ? val(row[at + p + j]) : -INFINITY;
    }
  }
}

// The sum over the workgroup, in all threads: one barrier, and the next call
// takes the other half of the scratch.
struct Totals {
  float (*s)[SNW];
  int turn = 0;
  DEV_INLINE float add(float wave_total) {
    float* t = s[turn ^= 1];
    if ((threadIdx.x & (WAVE - 1)) == 0) t[threadIdx.x / WAVE] = wave_total;
    __syncthreads();
    float v = 0.f;
    #pragma unroll
    for (int i = 0; i < SNW; ++i) v += t[i];
    return v;
  }
  DEV_INLINE float most(float wave_most) {
    float* t = s[turn ^= 1];
    if ((threadIdx.x & (WAVE - 1)) == 0) t[threadIdx.x / WAVE] = wave_most;
    __syncthreads();
    float v = t[0];
    #pragma unroll
    for (int i = 1; i < SNW; ++i) v = fmaxf(v, t[i]);
    return v;
  }
};

// NR: rounds of 8192 logits that cover the row
template <class T, int NR, bool VEC>
__global__ __launch_bounds__(SBLOCK)
void softmax_sample_kernel(long* __restrict__ out,          // [B]
                           const T* __restrict__ logits,  // [B, V]
                           const float* __restrict__ temperature,
                           const int* __restrict__ top_k,
                           const float* __restrict__ top_p,
                           const float* __restrict__ uniform, int vocab) {
  __shared__ float s_tot[2][SNW];
  __shared__ int s_idx[SNW];
  __shared__ int s_tok;
  Totals totals{s_tot};
  const int b = blockIdx.x, tid = threadIdx.x;
  const int wave = tid / WAVE, lane = tid % WAVE;
  const T* row = logits + (long)b * vocab;
  const float temp = temperature[b];

  // the largest logit; the smallest index of several. NaN is passed over.
  float e[NR][SVEC];
  float best = -INFINITY;
  int besti = 0x7fffffff;
  #pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int at = r * SROUND + tid * SVEC;
    load8<T, VEC>(row, at, vocab, e[r]);
    #pragma unroll
    for (int j = 0; j < SVEC; ++j)
      if (e[r][j] > best) { best = e[r][j]; besti = at + j; }
  }

  // ---- greedy ---------------------------------------------------------
  if (temp <= 0.f) {
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float ov = __shfl_xor(best, off, WAVE);
      const int oi = __shfl_xor(besti, off, WAVE);
      if (ov > best || (ov == best && oi < besti)) { best = ov; besti = oi; }
    }
    if (lane == 0) { s_tot[0][wave] = best; s_idx[wave] = besti; }
    __syncthreads();
    if (tid == 0) {
      for (int w = 1; w < SNW; ++w)
        if (s_tot[0][w] > best || (s_tot[0][w] == best && s_idx[w] < besti)) {
          best = s_tot[0][w];
          besti = s_idx[w];
        }
      out[b] = besti < vocab ? besti : 0;
    }
    return;
  }

  // temperature is applied in fp32, to the logits as they came
  const float inv_t = 1.f / temp;
  const float top = totals.most(wave_max(best));
  const float m = top * inv_t;
  // NaN, and what went past the largest number beside the largest logit: 0. A
  // logit below the largest may be equal to it once scaled (of neighbours in 32
  // bits about a tenth are), and weighs as much then.
  const float past = m == -INFINITY ? m : INFINITY;
  auto weight = [&](float v) {
    const float x = v * inv_t, below = __expf(x - m);
    return v == top ? 1.f : x < past ? below : 0.f;
  };
  #pragma unroll
  for (int r = 0; r < NR; ++r)
    #pragma unroll
    for (int j = 0; j < SVEC; ++j) {
      const int at = r * SROUND + tid * SVEC + j;
      e[r][j] = at < vocab ? weight(e[r][j]) : -1.f;    // -1: not a token
      // one after the other, or their parts take the registers of the row
      __builtin_amdgcn_sched_barrier(0);
    }
  const unsigned first = key_of<T>(-INFINITY), last = key_of<T>(top);
  // the largest key whose logits and all above them satisfy enough(their
  // weight's threshold)
  auto search = [&](auto enough) {
    unsigned lo = first, hi = last + 1;     // holds at lo, not at hi
    while (hi - lo > 1) {
      const unsigned mid = lo + (hi - lo) / 2;
      if (enough(weight(of_key<T>(mid)))) lo = mid; else hi = mid;
    }
    return lo;
  };
  auto sum_from = [&](float t) {
    float s = 0.f;
    #pragma unroll
    for (int r = 0; r < NR; ++r) {
      #pragma unroll
      for (int j = 0; j < SVEC; ++j) s += e[r][j] >= t ? e[r][j] : 0.f;
      __builtin_amdgcn_sched_barrier(0);
    }
    return totals.add(wave_sum(s));
  };

  // ---- top-k: as many largest as are no more than k with all their equals,
  // ---- the largest and its equals in any case
  float thresh = 0.f;
  const int k = top_k[b];
  if (k > 0 && k < vocab) {
    const unsigned more = search([&](float t) {
      int n = 0;
      #pragma unroll
      for (int r = 0; r < NR; ++r) {
        #pragma unroll
        for (int j = 0; j < SVEC; ++j)
          n += __popcll(__ballot(e[r][j] >= t));
        __builtin_amdgcn_sched_barrier(0);
      }
      return totals.add((float)n) > (float)k;
    });
    thresh = weight(of_key<T>(min(more + 1, last)));
  }

  // ---- top-p: the fewest largest weights with that share ----------------
  const float p_target = top_p[b];
  if (p_target > 0.f && p_target < 1.f) {
    const float goal = p_target * sum_from(thresh);
    const float low = thresh;
    thresh = fmaxf(low, weight(of_key<T>(search([&](float t) {
      return t < low || sum_from(t) >= goal;
    }))));
  }

  // ---- inverse-CDF draw, in token order ---------------------------------
  // Which token a number falls to depends on how sums are rounded: about every
  // two-hundredth draw from thousands of tokens lies that close to an edge. So
  // that a row and a number keep their token, the sum is that of 256 threads
  // over every 256th token, the edges those of 256 runs of tokens, added up
  // from left to right, as they always were (2 us of the 32 above).
  constexpr bool KEPT = NR <= 4;      // weights fit LDS; else made again, out
  constexpr int RAW = KEPT || sizeof(T) == 4    // of logits where those do
      ? 1 : NR * SROUND < 77824 ? NR * SROUND : 77824;
  __shared__ float s_w[KEPT ? NR * SROUND : 1];
  __shared__ T s_raw[RAW];
  __shared__ float s_run[RUNS];
  if constexpr (KEPT) {
    #pragma unroll
    for (int r = 0; r < NR; ++r) {
      float4 w[2];
      float* f = reinterpret_cast<float*>(w);
      #pragma unroll
      for (int j = 0; j < SVEC; ++j) f[j] = e[r][j] >= thresh ? e[r][j] : 0.f;
      float4* to = reinterpret_cast<float4*>(s_w + r * SROUND + tid * SVEC);
      to[0] = w[0];
      to[1] = w[1];
    }
  } else if constexpr (RAW > 1) {
    #pragma unroll 8
    for (int i = tid; i < min(vocab, RAW); i += SBLOCK) s_raw[i] = row[i];
  }
  if (tid == 0) s_tok = -1;
  __syncthreads();
  auto kept_weight = [&](int i) {
    if constexpr (KEPT) {
      return s_w[i];
    } else {
      const float w =
          weight(val(RAW > 1 && i < RAW ? s_raw[i] : row[i]));
      return w >= thresh ? w : 0.f;
    }
  };
  const int run = (vocab + RUNS - 1) / RUNS;
  if (tid < RUNS) {
    float sum = 0.f;
    #pragma unroll 16
    for (int i = tid; i < vocab; i += RUNS) sum += kept_weight(i);
    sum = wave_sum(sum);
    if (lane == 0) s_tot[0][wave] = sum;
  } else if (tid < 2 * RUNS) {
    const int from = (tid - RUNS) * run, end = min(from + run, vocab);
    float sum = 0.f;
    #pragma unroll 16
    for (int i = from; i < end; ++i) sum += kept_weight(i);
    s_run[tid - RUNS] = sum;
  }
  __syncthreads();
  if (wave == 0) {
    float z = 0.f;
    #pragma unroll
    for (int q = 0; q < RUNS / WAVE; ++q) z += s_tot[0][q];
    const float goal = uniform[b] * z;
    constexpr int EACH = RUNS / WAVE;
    float mine[EACH], edge[EACH], before = 0.f, upto = 0.f;
    #pragma unroll
    for (int q = 0; q < EACH; ++q) mine[q] = s_run[lane * EACH + q];
    for (int l = 0; l < WAVE; ++l) {
      if (lane == l) before = upto;
      #pragma unroll
      for (int q = 0; q < EACH; ++q) {
        upto += __uint_as_float(
            __builtin_amdgcn_readlane(__float_as_uint(mine[q]), l));
        if (lane == l) edge[q] = upto;
      }
    }
    #pragma unroll
    for (int q = 0; q < EACH; ++q) {
      if (goal >= before && goal < edge[q]) {
        const int from = (lane * EACH + q) * run;
        const int end = min(from + run, vocab);
        float acc = before;
        int sel = -1;
        for (int i = from; i < end && sel < 0; i += 8) {
          float w[8];
          #pragma unroll
          for (int j = 0; j < 8; ++j)
            w[j] = i + j < end ? kept_weight(i + j) : 0.f;
          #pragma unroll
          for (int j = 0; j < 8; ++j) {
            acc += w[j];
            if (sel < 0 && w[j] > 0.f && acc > goal) sel = i + j;
          }
        }
        if (sel >= 0) s_tok = sel;
      }
      before = edge[q];
    }
  }
  __syncthreads();
  if (s_tok >= 0) {
    if (tid == 0) out[b] = s_tok;
    return;
  }
  // rounding at the very end (goal ~ z): the last token that may be drawn
  int kept = -1;
  #pragma unroll
  for (int r = 0; r < NR; ++r)
    #pragma unroll
    for (int j = 0; j < SVEC; ++j)
      if (e[r][j] >= thresh) kept = r * SROUND + tid * SVEC + j;
  #pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    kept = max(kept, __shfl_xor(kept, off, WAVE));
  if (lane == 0) s_idx[wave] = kept;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < SNW; ++w) kept = max(kept, s_idx[w]);
    out[b] = max(kept, 0);
  }
}

template <class T>
void launch(long* out, const T* logits, const float* temperature,
            const int* top_k, const float* top_p, const float* uniform,
            int bsz, int vocab, hipStream_t stream) {
  const bool vec = vocab * sizeof(T) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(logits) % 16 == 0;
  auto go = [&](auto nr) {
    constexpr int NR = decltype(nr)::value;
    if (vec) {
      softmax_sample_kernel<T, NR, true>
          <<<dim3(bsz), dim3(SBLOCK), 0, stream>>>(
              out, logits, temperature, top_k, top_p, uniform, vocab);
    } else {
      softmax_sample_kernel<T, NR, false>
          <<<dim3(bsz), dim3(SBLOCK), 0, stream>>>(
              out, logits, temperature, top_k, top_p, uniform, vocab);
    }
  };
  if (vocab <= SROUND) go(std::integral_constant<int, 1>{});
  else if (vocab <= 4 * SROUND) go(std::integral_constant<int, 4>{});
  else if (vocab <= 7 * SROUND) go(std::integral_constant<int, 7>{});
  else go(std::integral_constant<int, 10>{});
}

}  // namespace

void launch_softmax_sample(long* out, const bf16_t* logits,
                           const float* temperature, const int* top_k,
                           const float* top_p, const float* uniform, int bsz,
                           int vocab, hipStream_t stream) {
  launch(out, logits, temperature, top_k, top_p, uniform, bsz, vocab, stream);
}

void launch_softmax_sample(long* out, const float* logits,
                           const float* temperature, const int* top_k,
                           const float* top_p, const float* uniform, int bsz,
                           int vocab, hipStream_t stream) {
  launch(out, logits, temperature, top_k, top_p, uniform, bsz, vocab, stream);
}
