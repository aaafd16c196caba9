// The row work of a training step between its products: residual additions
// with the norm that follows, forward and backward; the split of a fused
// projection with its rotation, forward and backward; the gated activation's
// backward.
//
// All of it is bound by memory. As single tensor operations the same work was
// 32-bit copies of every operand, a pass for each addition, product and
// concatenation, and launches of 5 us. In a step of four layers on a MI355X
// (rows x width, launches of everything, us of everything but products,
// attention and update):
//   4096 x 4544, 71 heads on 1 of 64, LayerNorm   502 -> 238, 6950 -> 3900
//   2331 x 2048, 16 heads of 128, RMS, gated       496 -> 194, 3350 -> 1190
// At 4096 x 4544 the norm of two additions takes 33 us (5.6 TB/s), its
// backward 38 and 9 for the sum of shares, split and join 14 and 16.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace {

constexpr int BLOCK = 256;
constexpr int NWAVES = BLOCK / WAVE;

DEV_INLINE void unpack8(uint4 u, float* f) {
  const unsigned int w[4] = {u.x, u.y, u.z, u.w};
  #pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float2 p = unpack_bf16x2(w[j]);
    f[2 * j] = p.x;
    f[2 * j + 1] = p.y;
  }
}

DEV_INLINE uint4 pack8(const float* f) {
  return make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]),
                    pack_bf16x2(f[4], f[5]), pack_bf16x2(f[6], f[7]));
}

// One workgroup per row, the row in registers. h + d1 + d2 is rounded after
// each addition, as the separate additions round it; sums are in 32 bits, the
// variance about the mean. stats: mean (0 for RMS) and 1/deviation per row.
template <int CAP, bool RMS>
__global__ __launch_bounds__(BLOCK) void add_norm_fwd_kernel(
    bf16_t* __restrict__ y, bf16_t* __restrict__ sum,
    float2* __restrict__ stats, const bf16_t* __restrict__ h,
    const bf16_t* __restrict__ d1, const bf16_t* __restrict__ d2,
    const bf16_t* __restrict__ weight, const bf16_t* __restrict__ bias,
    int hidden, float eps) {
  __shared__ float scratch[2 * NWAVES];
  const long row = blockIdx.x;
  const int nvec = hidden / 8;
  const uint4* hv = reinterpret_cast<const uint4*>(h + row * hidden);
  const uint4* v1 = reinterpret_cast<const uint4*>(d1 + row * hidden);
  const uint4* v2 = reinterpret_cast<const uint4*>(d2 + row * hidden);
  uint4* sv = reinterpret_cast<uint4*>(sum + row * hidden);
  float f[CAP][8];
  float s = 0.f;
  #pragma unroll
  for (int c = 0; c < CAP; ++c) {
    const int i = threadIdx.x + c * BLOCK;
    #pragma unroll
    for (int j = 0; j < 8; ++j) f[c][j] = 0.f;
    if (i < nvec) {
      uint4 u = hv[i];
      unpack8(u, f[c]);
      #pragma unroll
      for (int n = 0; n < 2; ++n) {
        if ((n ? d2 : d1) == nullptr) continue;
        float a[8];
        unpack8((n ? v2 : v1)[i], a);
        #pragma unroll
        for (int j = 0; j < 8; ++j) a[j] += f[c][j];
        u = pack8(a);
        unpack8(u, f[c]);
      }
      if (d1) sv[i] = u;
    }
    #pragma unroll
    for (int j = 0; j < 8; ++j) s += RMS ? f[c][j] * f[c][j] : f[c][j];
  }
  const float first = block_sum<NWAVES>(s, scratch) / (float)hidden;
  const float mean = RMS ? 0.f : first;
  float var = first;
  if (!RMS) {
    s = 0.f;
    #pragma unroll
    for (int c = 0; c < CAP; ++c)
      if ((int)threadIdx.x + c * BLOCK < nvec) {
        #pragma unroll
        for (int j = 0; j < 8; ++j)
          s += (f[c][j] - mean) * (f[c][j] - mean);
      }
    var = block_sum<NWAVES>(s, scratch + NWAVES) / (float)hidden;
  }
  const float inv = rsqrtf(var + eps);
  if (threadIdx.x == 0) stats[row] = make_float2(mean, inv);
  const uint4* wv = reinterpret_cast<const uint4*>(weight);
  const uint4* bv = reinterpret_cast<const uint4*>(bias);
  uint4* yv = reinterpret_cast<uint4*>(y + row * hidden);
  #pragma unroll
  for (int c = 0; c < CAP; ++c) {
    const int i = threadIdx.x + c * BLOCK;
    if (i >= nvec) break;
    float w[8], b[8];
    unpack8(wv[i], w);
    if (!RMS) unpack8(bv[i], b);
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      w[j] *= (f[c][j] - mean) * inv;
      if (!RMS) w[j] += b[j];
    }
    yv[i] = pack8(w);
  }
}

// dh = dres + inv * (w dy - mean(w dy) - x^ mean(w dy x^)), x^ the normed row
// (the first mean only where the norm takes a mean off). A workgroup takes
// rows a grid apart and loads the next one while it sums the last; its share
// of the weights' gradients stays in registers until its last row.
template <int CAP, bool RMS>
__global__ __launch_bounds__(BLOCK) void add_norm_bwd_kernel(
    bf16_t* __restrict__ dh, float* __restrict__ dw, float* __restrict__ db,
    const bf16_t* __restrict__ dy, const bf16_t* __restrict__ dres,
    const bf16_t* __restrict__ x, const float2* __restrict__ stats,
    const bf16_t* __restrict__ weight, long rows, int hidden) {
  __shared__ float scratch[2][2 * NWAVES];
  const int nvec = hidden / 8;
  const int tid = threadIdx.x;
  float aw[CAP][8], ab[CAP][8];
  #pragma unroll
  for (int c = 0; c < CAP; ++c)
    #pragma unroll
    for (int j = 0; j < 8; ++j) aw[c][j] = ab[c][j] = 0.f;
  const uint4* wv = reinterpret_cast<const uint4*>(weight);
  const uint4 none = make_uint4(0, 0, 0, 0);
  uint4 gy[CAP], gx[CAP], gr[CAP];
  auto load = [&](long row) {
    const uint4* yv = reinterpret_cast<const uint4*>(dy + row * hidden);
    const uint4* xv = reinterpret_cast<const uint4*>(x + row * hidden);
    const uint4* rv = reinterpret_cast<const uint4*>(dres + row * hidden);
    #pragma unroll
    for (int c = 0; c < CAP; ++c) {
      const int i = tid + c * BLOCK;
      gy[c] = gx[c] = gr[c] = none;
      if (i < nvec) {
        gy[c] = yv[i];
        gx[c] = xv[i];
        if (dres) gr[c] = rv[i];
      }
    }
  };
  long row = blockIdx.x;
  if (row < rows) load(row);
  for (int turn = 0; row < rows; row += gridDim.x, turn ^= 1) {
    const float2 st = stats[row];
    float s1 = 0.f, s2 = 0.f;
    uint4 ry[CAP], rx[CAP], rr[CAP];
    #pragma unroll
    for (int c = 0; c < CAP; ++c) {
      const int i = tid + c * BLOCK;
      ry[c] = gy[c]; rx[c] = gx[c]; rr[c] = gr[c];
      float g[8], v[8], w[8];
      unpack8(ry[c], g);
      unpack8(rx[c], v);
      unpack8(i < nvec ? wv[i] : none, w);
      #pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float n = (v[j] - st.x) * st.y;
        aw[c][j] += g[j] * n;
        if (!RMS) ab[c][j] += g[j];
        s1 += g[j] * w[j];
        s2 += g[j] * w[j] * n;
      }
    }
    if (row + gridDim.x < rows) load(row + gridDim.x);
    // the other half of the scratch is read until the next turn's barrier
    float* sc = scratch[turn];
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
    if (tid % WAVE == 0) {
      sc[tid / WAVE] = s1;
      sc[NWAVES + tid / WAVE] = s2;
    }
    __syncthreads();
    s1 = s2 = 0.f;
    #pragma unroll
    for (int n = 0; n < NWAVES; ++n) {
      s1 += sc[n];
      s2 += sc[NWAVES + n];
    }
    s1 = RMS ? 0.f : s1 / (float)hidden;
    s2 /= (float)hidden;
    uint4* ov = reinterpret_cast<uint4*>(dh + row * hidden);
    #pragma unroll
    for (int c = 0; c < CAP; ++c) {
      const int i = tid + c * BLOCK;
      if (i >= nvec) break;
      float g[8], v[8], w[8], r[8];
      unpack8(ry[c], g);
      unpack8(rx[c], v);
      unpack8(wv[i], w);
      unpack8(rr[c], r);
      #pragma unroll
      for (int j = 0; j < 8; ++j)
        r[j] += st.y * (g[j] * w[j] - s1 - (v[j] - st.x) * st.y * s2);
      ov[i] = pack8(r);
    }
  }
  float4* ow = reinterpret_cast<float4*>(dw + blockIdx.x * (long)hidden);
  float4* ob = reinterpret_cast<float4*>(db + blockIdx.x * (long)hidden);
  #pragma unroll
  for (int c = 0; c < CAP; ++c) {
    const int i = tid + c * BLOCK;
    if (i >= nvec) break;
    #pragma unroll
    for (int k = 0; k < 2; ++k) {
      ow[2 * i + k] = make_float4(aw[c][4 * k], aw[c][4 * k + 1],
                                  aw[c][4 * k + 2], aw[c][4 * k + 3]);
      if (!RMS)
        ob[2 * i + k] = make_float4(ab[c][4 * k], ab[c][4 * k + 1],
                                    ab[c][4 * k + 2], ab[c][4 * k + 3]);
    }
  }
}

// Sums of the workgroups' shares, 64 columns a workgroup.
__global__ __launch_bounds__(BLOCK) void shares_sum_kernel(
    bf16_t* __restrict__ dw, bf16_t* __restrict__ db,
    const float* __restrict__ pw, const float* __restrict__ pb, int shares,
    int hidden) {
  __shared__ float part[NWAVES][WAVE];
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  const int col = blockIdx.x * WAVE + lane;
  const float* p = blockIdx.y ? pb : pw;
  float s = 0.f;
  if (col < hidden) {
    #pragma unroll 8
    for (int n = wave; n < shares; n += NWAVES) s += p[n * (long)hidden + col];
  }
  part[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && col < hidden)
    (blockIdx.y ? db : dw)[col] =
        f2bf((part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]));
}

// One workgroup per token; a thread keeps its 8 angles for all heads it
// takes (BLOCK is a multiple of the d / 16 threads a head needs).
__global__ __launch_bounds__(BLOCK) void rope_split_kernel(
    bf16_t* __restrict__ q, bf16_t* __restrict__ k, bf16_t* __restrict__ v,
    const bf16_t* __restrict__ qkv, const float* __restrict__ cosine,
    const float* __restrict__ sine, int length, int hq, int hkv, int d) {
  const long row = blockIdx.x;
  const int per = d / 16, j = threadIdx.x % per;
  float c[8], s[8];
  if (cosine) {
    const long at = (row % length) * (d / 2) + j * 8;
    #pragma unroll
    for (int e = 0; e < 8; ++e) {
      c[e] = cosine[at + e];
      s[e] = sine[at + e];
    }
  }
  const int heads = hq + 2 * hkv;
  const uint4* in = reinterpret_cast<const uint4*>(qkv + row * heads * d);
  for (int head = threadIdx.x / per; head < heads; head += BLOCK / per) {
    uint4 lo = in[head * 2 * per + j], hi = in[head * 2 * per + per + j];
    bf16_t* out = head < hq ? q + (row * hq + head) * d
                  : head < hq + hkv ? k + (row * hkv + head - hq) * d
                                    : v + (row * hkv + head - hq - hkv) * d;
    if (cosine && head < hq + hkv) {
      float a[8], b[8], na[8], nb[8];
      unpack8(lo, a);
      unpack8(hi, b);
      #pragma unroll
      for (int e = 0; e < 8; ++e) {
        na[e] = a[e] * c[e] - b[e] * s[e];
        nb[e] = b[e] * c[e] + a[e] * s[e];
      }
      lo = pack8(na);
      hi = pack8(nb);
    }
    uint4* ov = reinterpret_cast<uint4*>(out);
    ov[j] = lo;
    ov[per + j] = hi;
  }
}

DEV_INLINE void load8(const float* p, float* f) {
  const float4 a = reinterpret_cast<const float4*>(p)[0];
  const float4 b = reinterpret_cast<const float4*>(p)[1];
  f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
  f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
}

// The gradients of q, k and v back into one row, turned the other way. Those
// of k and v come as the 32-bit sums of the attention's backward.
__global__ __launch_bounds__(BLOCK) void rope_join_kernel(
    bf16_t* __restrict__ dqkv, const bf16_t* __restrict__ dq,
    const float* __restrict__ dk, const float* __restrict__ dv,
    const float* __restrict__ cosine, const float* __restrict__ sine,
    int length, int hq, int hkv, int d) {
  const long row = blockIdx.x;
  const int per = d / 16, j = threadIdx.x % per;
  float c[8], s[8];
  if (cosine) {
    const long at = (row % length) * (d / 2) + j * 8;
    #pragma unroll
    for (int e = 0; e < 8; ++e) {
      c[e] = cosine[at + e];
      s[e] = sine[at + e];
    }
  }
  const int heads = hq + 2 * hkv;
  uint4* out = reinterpret_cast<uint4*>(dqkv + row * heads * d);
  for (int head = threadIdx.x / per; head < heads; head += BLOCK / per) {
    float a[8], b[8];
    if (head < hq) {
      const uint4* in =
          reinterpret_cast<const uint4*>(dq + (row * hq + head) * d);
      unpack8(in[j], a);
      unpack8(in[per + j], b);
    } else {
      const float* in = head < hq + hkv
                            ? dk + (row * hkv + head - hq) * d
                            : dv + (row * hkv + head - hq - hkv) * d;
      load8(in + j * 8, a);
      load8(in + (per + j) * 8, b);
    }
    if (cosine && head < hq + hkv) {
      #pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float na = a[e] * c[e] + b[e] * s[e];
        b[e] = b[e] * c[e] - a[e] * s[e];
        a[e] = na;
      }
    }
    out[head * 2 * per + j] = pack8(a);
    out[head * 2 * per + per + j] = pack8(b);
  }
}

// x: [rows, 2F] (gate, up), dy: [rows, F], dx like x.
__global__ __launch_bounds__(BLOCK) void silu_mul_bwd_kernel(
    bf16_t* __restrict__ dx, const bf16_t* __restrict__ dy,
    const bf16_t* __restrict__ x, int f) {
  const long row = blockIdx.x;
  const int nvec = f / 8;
  const uint4* gv = reinterpret_cast<const uint4*>(x + row * 2 * f);
  const uint4* yv = reinterpret_cast<const uint4*>(dy + row * f);
  uint4* ov = reinterpret_cast<uint4*>(dx + row * 2 * f);
  for (int i = blockIdx.y * BLOCK + threadIdx.x; i < nvec;
       i += gridDim.y * BLOCK) {
    float g[8], u[8], t[8];
    unpack8(gv[i], g);
    unpack8(gv[nvec + i], u);
    unpack8(yv[i], t);
    #pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float sig = 1.f / (1.f + __expf(-g[e]));
      const float act = g[e] * sig;
      const float slope = sig + act * (1.f - sig);
      g[e] = t[e] * u[e] * slope;
      u[e] = t[e] * act;
    }
    ov[i] = pack8(g);
    ov[nvec + i] = pack8(u);
  }
}

// Gradient of a lookup, whose rows are zero already. A workgroup per token: the
// first one of a number adds up the rows of all of them, in their order, unless
// there are more than OFTEN, which it leaves to the kernel after this one: a row
// after the other takes 0.3 us. It looks through all tokens for them, which is
// less than sorting them up to some thousands.
// us on a MI355X, torch's kernels (without the zeros), the first one of these
// alone, both; 2331 tokens of 32000 x 2048, 4096 of 65024 x 4544, 8192 of 32000 x
// 2048:
//   every number about as often           179   11  14   184   26  30   179   53   58
//   the k-th most frequent 1/k as often   177   71  30   155  157  62   156  231   87
//   half of them one number               193  339  34   177  956  89   235 1236  122
//   one number only                       251  692  41   211 1767  72   329 2440  134
constexpr int OFTEN = 32;

template <int CAP>
__global__ __launch_bounds__(BLOCK) void lookup_bwd_kernel(
    bf16_t* __restrict__ dw, unsigned char* __restrict__ often,
    const bf16_t* __restrict__ dy, const long* __restrict__ tokens, int n,
    long rows, int hidden) {
  __shared__ unsigned long long same[NWAVES];
  const int i = blockIdx.x, tid = threadIdx.x;
  if (tid == 0) often[i] = 0;
  const long t = tokens[i];
  if (t < 0 || t >= rows) return;
  bool before = false;
  for (int j = tid; j < i; j += BLOCK) before |= tokens[j] == t;
  if (__syncthreads_or(before)) return;
  const int nvec = hidden / 8;
  float sum[CAP][8];
  #pragma unroll
  for (int c = 0; c < CAP; ++c)
    #pragma unroll
    for (int e = 0; e < 8; ++e) sum[c][e] = 0.f;
  int count = 0;
  for (int j0 = i; j0 < n; j0 += BLOCK) {
    const int j = j0 + tid;
    const unsigned long long mine =
        __ballot(j < n && tokens[min(j, n - 1)] == t);
    if (tid % WAVE == 0) same[tid / WAVE] = mine;
    __syncthreads();
    #pragma unroll
    for (int w = 0; w < NWAVES; ++w) count += __popcll(same[w]);
    if (count > OFTEN) {
      if (tid == 0) often[i] = 1;
      return;
    }
    for (int w = 0; w < NWAVES; ++w)
      for (unsigned long long m = same[w]; m; m &= m - 1) {
        const long row = j0 + w * WAVE + __builtin_ctzll(m);
        const uint4* v = reinterpret_cast<const uint4*>(dy + row * hidden);
        #pragma unroll
        for (int c = 0; c < CAP; ++c) {
          const int at = tid + c * BLOCK;
          if (at >= nvec) break;
          float f[8];
          unpack8(v[at], f);
          #pragma unroll
          for (int e = 0; e < 8; ++e) sum[c][e] += f[e];
        }
      }
    __syncthreads();
  }
  uint4* out = reinterpret_cast<uint4*>(dw + t * hidden);
  #pragma unroll
  for (int c = 0; c < CAP; ++c) {
    const int at = tid + c * BLOCK;
    if (at < nvec) out[at] = pack8(sum[c]);
  }
}

// The numbers that come often: a workgroup for 64 columns of those whose first
// tokens are a grid apart, eight threads a row, 32 rows at once.
constexpr int SLICE = 64;

__global__ __launch_bounds__(BLOCK) void lookup_bwd_often_kernel(
    bf16_t* __restrict__ dw, const unsigned char* __restrict__ often,
    const bf16_t* __restrict__ dy, const long* __restrict__ tokens, int n,
    int hidden) {
  constexpr int SLOTS = BLOCK / 8;
  __shared__ unsigned long long mask[2][NWAVES];
  __shared__ int list[BLOCK];
  __shared__ float part[SLOTS][SLICE];
  const int tid = threadIdx.x, wave = tid / WAVE, slot = tid / 8;
  const int lane8 = tid % 8 * 8, col = blockIdx.y * SLICE + lane8;
  const int grid = gridDim.x;
  for (int i0 = blockIdx.x; i0 < n; i0 += grid * BLOCK) {
    const long mine = i0 + (long)tid * grid;
    const unsigned long long b = __ballot(mine < n && often[mine]);
    if (tid % WAVE == 0) mask[0][wave] = b;
    __syncthreads();
    for (int w = 0; w < NWAVES; ++w)
      for (unsigned long long m = mask[0][w]; m; m &= m - 1) {
        const int i = i0 + (w * WAVE + __builtin_ctzll(m)) * grid;
        const long t = tokens[i];
        float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int j0 = i; j0 < n; j0 += BLOCK) {
          const int j = j0 + tid;
          const bool same = j < n && tokens[min(j, n - 1)] == t;
          const unsigned long long all = __ballot(same);
          if (tid % WAVE == 0) mask[1][wave] = all;
          __syncthreads();
          int before = 0, count = 0;
          #pragma unroll
          for (int q = 0; q < NWAVES; ++q) {
            const int some = __popcll(mask[1][q]);
            before += q < wave ? some : 0;
            count += some;
          }
          if (same)
            list[before + __popcll(all & ((1ull << (tid % WAVE)) - 1))] = j;
          __syncthreads();
          if (col < hidden) {
            #pragma unroll 4
            for (int r = slot; r < count; r += SLOTS) {
              float f[8];
              unpack8(*reinterpret_cast<const uint4*>(
                          dy + (long)list[r] * hidden + col), f);
              #pragma unroll
              for (int e = 0; e < 8; ++e) sum[e] += f[e];
            }
          }
          __syncthreads();
        }
        #pragma unroll
        for (int e = 0; e < 8; ++e) part[slot][lane8 + e] = sum[e];
        __syncthreads();
        const int at = blockIdx.y * SLICE + tid;
        if (tid < SLICE && at < hidden) {
          float s = 0.f;
          #pragma unroll
          for (int q = 0; q < SLOTS; ++q) s += part[q][tid];
          dw[t * hidden + at] = f2bf(s);
        }
        __syncthreads();
      }
    __syncthreads();
  }
}

template <class F>
void by_width(int hidden, F go) {
  const int cap = (hidden / 8 + BLOCK - 1) / BLOCK;
  if (cap <= 1) go(std::integral_constant<int, 1>());
  else if (cap <= 2) go(std::integral_constant<int, 2>());
  else if (cap <= 3) go(std::integral_constant<int, 3>());
  else go(std::integral_constant<int, 4>());
}

}  // namespace

// Rows wider than 4 vectors a thread do not stay in registers beside the
// weights' gradients.
bool train_norm_takes(int hidden) {
  return hidden % 8 == 0 && hidden > 0 && hidden <= 4 * BLOCK * 8;
}

void launch_add_norm_fwd(bf16_t* y, bf16_t* sum, float* stats,
                         const bf16_t* h, const bf16_t* d1, const bf16_t* d2,
                         const bf16_t* w, const bf16_t* b, long rows,
                         int hidden, float eps, bool rms, hipStream_t stream) {
  by_width(hidden, [&](auto cap) {
    constexpr int C = decltype(cap)::value;
    auto kernel = rms ? add_norm_fwd_kernel<C, true>
                      : add_norm_fwd_kernel<C, false>;
    kernel<<<dim3(rows), dim3(BLOCK), 0, stream>>>(
        y, sum, reinterpret_cast<float2*>(stats), h, d1, d2, w, b, hidden,
        eps);
  });
}

// Two workgroups a CU hide each other's sums; more of them only write more
// shares of the weights' gradients.
int train_norm_shares(long rows) { return (int)std::min(rows, (long)512); }

void launch_add_norm_bwd(bf16_t* dh, bf16_t* dw, bf16_t* db, float* shares,
                         const bf16_t* dy, const bf16_t* dres,
                         const bf16_t* x, const float* stats, const bf16_t* w,
                         long rows, int hidden, bool rms, hipStream_t stream) {
  const int n = train_norm_shares(rows);
  float* second = shares + (rms ? 0 : n * (long)hidden);
  by_width(hidden, [&](auto cap) {
    constexpr int C = decltype(cap)::value;
    auto kernel = rms ? add_norm_bwd_kernel<C, true>
                      : add_norm_bwd_kernel<C, false>;
    kernel<<<dim3(n), dim3(BLOCK), 0, stream>>>(
        dh, shares, second, dy, dres, x,
        reinterpret_cast<const float2*>(stats), w, rows, hidden);
  });
  shares_sum_kernel<<<dim3((hidden + WAVE - 1) / WAVE, rms ? 1 : 2),
                      dim3(BLOCK), 0, stream>>>(dw, db, shares, second, n,
                                                hidden);
}

void launch_rope_split(bf16_t* q, bf16_t* k, bf16_t* v, const bf16_t* qkv,
                       const float* cosine, const float* sine, long rows,
                       int length, int hq, int hkv, int d,
                       hipStream_t stream) {
  rope_split_kernel<<<dim3(rows), dim3(BLOCK), 0, stream>>>(
      q, k, v, qkv, cosine, sine, length, hq, hkv, d);
}

void launch_rope_join(bf16_t* dqkv, const bf16_t* dq, const float* dk,
                      const float* dv, const float* cosine, const float* sine,
                      long rows, int length, int hq, int hkv, int d,
                      hipStream_t stream) {
  rope_join_kernel<<<dim3(rows), dim3(BLOCK), 0, stream>>>(
      dqkv, dq, dk, dv, cosine, sine, length, hq, hkv, d);
}

void launch_silu_mul_bwd(bf16_t* dx, const bf16_t* dy, const bf16_t* x,
                         long rows, int f, hipStream_t stream) {
  const int most = (f / 8 + BLOCK - 1) / BLOCK;
  silu_mul_bwd_kernel<<<dim3(rows, std::min(most, 4)), dim3(BLOCK), 0,
                        stream>>>(dx, dy, x, f);
}

void launch_lookup_bwd(bf16_t* dw, unsigned char* often, const bf16_t* dy,
                       const long* tokens, int n, long rows, int hidden,
                       hipStream_t stream) {
  by_width(hidden, [&](auto cap) {
    lookup_bwd_kernel<decltype(cap)::value>
        <<<dim3(n), dim3(BLOCK), 0, stream>>>(dw, often, dy, tokens, n, rows,
                                              hidden);
  });
  if (n > OFTEN)
    lookup_bwd_often_kernel<<<dim3(std::min(n, 64),
                                   (hidden + SLICE - 1) / SLICE),
                              dim3(BLOCK), 0, stream>>>(dw, often, dy, tokens,
                                                        n, hidden);
}
