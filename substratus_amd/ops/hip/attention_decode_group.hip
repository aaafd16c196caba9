// Paged decode attention of grouped query heads over a bf16 cache (head sizes
// 64 and 128): one new token per sequence, up to 16 heads of a group at a time
// against their key and value head.
//
// Bound by the K/V stream. Every wave has chunks of 32 keys (two pages) of its
// own: K and V go straight to LDS as they lie in the pages, the next chunk in
// flight, and nothing waits for other waves until the end, where the two
// waves' results are merged. Pieces of a row are permuted by the row against
// bank conflicts. Heads are the matrix instructions' columns:
//   S^T = K Q^T   a lane has four consecutive keys, twice, of one head: a
//                 head's maximum takes two exchanges
//   O^T = V^T P^T the keys a lane holds weights of are the keys its share of
//                 the inner dimension stands for; V^T is read by transposing
//                 LDS reads of the same keys, so weights never move
//
// us on a MI355X, merging of shares included, from the kernel whose waves
// share a chunk of 32 keys with a barrier (groups of 4, 8, 16) or a wave per
// head (others) to this one:
//   64 sequences of 625 to 2500 keys, 32 heads on 8 of 128   148 -> 94 (4.4 TB/s)
//   256 of 150 to 600, the same                              127 -> 85
//   1 of 4000, the same                                     28.5 -> 12.3
//   32 of 250 to 1000, 128 heads on 8 of 64                 28.8 -> 16.9
//   128 of 300 to 1200, 71 heads on 1 of 64                  206 -> 28
// Four waves (one workgroup per CU): 96, 98, 10.9, 20.4, 25; one: 95, 86, 14.8,
// 17.9, 27, with weights in two bf16 parts. Three, which keep all their bits,
// cost 1 % (the last shape 6 %).
#include "attention_order.h"
#include "rows_gemm.h"

namespace {

constexpr int NW = 2;             // waves
constexpr int PAGE = 16;
constexpr int CH = 2 * PAGE;      // keys of a chunk
constexpr float LOG2E = 1.44269504088896340736f;
constexpr float NONE = -1e30f;    // "no key yet": finite, so differences are too

DEV_INLINE unsigned pack2(float lo, float hi) {
  return pack_bf16x2(lo, hi);
}

DEV_INLINE unsigned lds_address(const void* p) {
  return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
}

// Eight transposing reads and the wait for them. The compiler's own form
// first waits for all loads in flight to LDS.
DEV_INLINE void read_transposed(uint2v (&r)[8], const unsigned (&at)[8]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %1, %9\n\t"
      "ds_read_b64_tr_b16 %2, %10\n\tds_read_b64_tr_b16 %3, %11\n\t"
      "ds_read_b64_tr_b16 %4, %12\n\tds_read_b64_tr_b16 %5, %13\n\t"
      "ds_read_b64_tr_b16 %6, %14\n\tds_read_b64_tr_b16 %7, %15\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]),
        "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
      : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "v"(at[4]),
        "v"(at[5]), "v"(at[6]), "v"(at[7])
      : "memory");
}

template <int D>
__global__ __launch_bounds__(NW * WAVE, 2)
void attn_group_kernel(bf16_t* __restrict__ out,             // [B, HQ, D]
                       const bf16_t* __restrict__ q,
                       const bf16_t* __restrict__ kc,  // [NB, HKV, 16, D]
                       const bf16_t* __restrict__ vc,
                       const int* __restrict__ block_table,  // [B, max_blocks]
                       const int* __restrict__ seq_lens,
                       int hq, int hkv, int max_blocks, float scale,
                       long q_ld, int nsplit, bool turned, bool ordered,
                       float* __restrict__ part_o,   // [B, HQ, NS, D]
                       float* __restrict__ part_ml) {  // [B, HQ, NS, 2]
  constexpr int RC = D / 8;                      // 16-byte pieces of a row
  constexpr int HALF = CH * RC;                  // of a chunk's K, or V
  constexpr int LOADS = HALF / WAVE;             // of either
  constexpr int KS = D / 32, DT = D / 16;
  constexpr int ROWS = WAVE / RC;                // rows of one load
  // one array: beside a second one the compiler guards every LDS read against
  // the direct loads in flight, and waits for them
  __shared__ alignas(16) uint4v s_all[NW * 2 * 2 * HALF];

  const int in_group = hq / hkv, parts = (in_group + 15) / 16;
  int b = blockIdx.x, part = blockIdx.y, split = blockIdx.z, n;
  if (turned) {                   // (no more groups than sequences)
    b += part;
    if (b >= (int)gridDim.x) b -= gridDim.x;
  }
  if (ordered) {
    const int bsz = gridDim.x, at_lane = length_at_lane(seq_lens, bsz);
    if (unlike_lengths(at_lane, max_blocks * PAGE)) {
      const Turn turn = turn_of(hkv * parts, nsplit);
      part = turn.head;
      split = turn.split;
      b = sequence_at(at_lane, bsz, max_blocks * PAGE, turn.sequence);
    }
    n = __builtin_amdgcn_readlane(at_lane, b);
  } else {
    n = __builtin_amdgcn_readfirstlane(seq_lens[b]);
  }
  const int kvh = part / parts, h0 = part % parts * 16;
  const int head0 = kvh * in_group + h0, heads = min(16, in_group - h0);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE;
  const int lo = lane & 15, g = lane >> 4;
  const int pages = (n + PAGE - 1) / PAGE;
  const int chunks = (n + CH - 1) / CH;
  const int first = split * NW + wave, step = nsplit * NW;
  const int mine = first < chunks ? (chunks - first + step - 1) / step : 0;
  uint4v* ring = s_all + wave * 2 * 2 * HALF;
  // page numbers come by scalar loads, which the counted waits do not see
  const auto* bt = (const __attribute__((address_space(4))) int*)(
      block_table + (long)b * max_blocks);

  // the lane's place in a load: piece lane % RC of row lane / RC; the row's
  // permutation depends on the row alone
  const int lr = lane / RC, lp = lane % RC;
  auto load = [&](int buf, int i) {
    const int c = first + i * step;
    // past the last page: that page again, whose keys are masked
    const long p0 = ((long)bt[min(2 * c, pages - 1)] * hkv + kvh) * PAGE * D;
    const long p1 = ((long)bt[min(2 * c + 1, pages - 1)] * hkv + kvh) *
                    PAGE * D;
    uint4v* to = ring + buf * 2 * HALF;
    #pragma unroll
    for (int t = 0; t < LOADS; ++t) {
      const int row = t * ROWS + lr;             // of the chunk
      const long at = (t < LOADS / 2 ? p0 : p1) + (row % PAGE) * D +
                      (lp ^ (row & (RC - 1))) * 8;
      load_to_lds<16>(kc + at, to + t * WAVE);
    }
    #pragma unroll
    for (int t = 0; t < LOADS; ++t) {
      const int row = t * ROWS + lr;
      const long at = (t < LOADS / 2 ? p0 : p1) + (row % PAGE) * D +
                      (lp ^ (row & (RC - 1))) * 8;
      load_to_lds<16>(vc + at, to + HALF + t * WAVE);
    }
  };
  if (mine > 0) load(0, 0);
  if (mine > 1) load(1, 1);

  // queries: lane = head (zeros past the last), 8 consecutive elements
  short8 qf[KS];
  #pragma unroll
  for (int c = 0; c < KS; ++c)
    qf[c] = lo < heads
        ? *reinterpret_cast<const short8*>(
              q + (long)b * q_ld + (long)(head0 + lo) * D + c * 32 +
              g * 8)
        : (short8){0, 0, 0, 0, 0, 0, 0, 0};
  // there before the loop, so that it never waits for them
  #pragma unroll
  for (int c = 0; c < KS; ++c) asm volatile("" : "+v"(qf[c]));

  const float scale2 = scale * LOG2E;
  float m = NONE, l = 0.f;
  float4v o[DT];
  #pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = (float4v){0.f, 0.f, 0.f, 0.f};
  auto use = [&](int buf, int i) {
    const uint4v* k = ring + buf * 2 * HALF;
    uint4v* v = ring + buf * 2 * HALF + HALF;
    const int key0 = (first + i * step) * CH;
    float p[8];
    float mx = NONE;
    #pragma unroll
    for (int s = 0; s < 2; ++s) {
      float4v acc = {0.f, 0.f, 0.f, 0.f};
      const int row = s * PAGE + lo;
      #pragma unroll
      for (int c = 0; c < KS; ++c)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(
                short8, k[row * RC + ((c * 4 + g) ^ (row & (RC - 1)))]),
            qf[c], acc, 0, 0, 0);
      #pragma unroll
      for (int e = 0; e < 4; ++e) {
        p[s * 4 + e] = key0 + s * PAGE + g * 4 + e < n ? acc[e] * scale2
                                                       : -INFINITY;
        mx = fmaxf(mx, p[s * 4 + e]);
      }
    }
    mx = across_from<16>(mx, Larger{});
    const float mn = fmaxf(m, mx);
    const float keep = __builtin_amdgcn_exp2f(m - mn);
    m = mn;
    float sum = 0.f;
    #pragma unroll
    for (int e = 0; e < 8; ++e) {
      p[e] = __builtin_amdgcn_exp2f(p[e] - mn);  // exp2(-inf) is 0
      sum += p[e];
    }
    l = l * keep + sum;                          // of the lane's own keys
    if (!__all(keep == 1.f)) {
      #pragma unroll
      for (int t = 0; t < DT; ++t) o[t] *= keep;
    }
    // weights as three parts, which hold all of their 24 bits
    short8 parts[3];
    #pragma unroll
    for (int w = 0; w < 3; ++w) {
      uint4v u;
      #pragma unroll
      for (int e = 0; e < 4; ++e) {
        u[e] = pack2(p[2 * e], p[2 * e + 1]);
        const float2 b = unpack_bf16x2(u[e]);
        p[2 * e] -= b.x;
        p[2 * e + 1] -= b.y;
      }
      parts[w] = __builtin_bit_cast(short8, u);
    }
    // a cache's own values past the last key may be anything, and times a
    // weight of zero still be no number
    if (key0 + CH > n) {
      for (int e = (n - key0) * RC + lane; e < HALF; e += WAVE)
        v[e] = (uint4v){0, 0, 0, 0};
      wait_lds_reads();
    }
    #pragma unroll
    for (int t0 = 0; t0 < DT; t0 += 4) {
      uint2v r[8];
      unsigned at[8];
      #pragma unroll
      for (int e = 0; e < 8; ++e) {
        // the lane's place in a transposing read: four columns of a key
        const int row = (e & 1) * PAGE + g * 4 + (lo >> 2);
        const int col = (t0 + e / 2) * 16 + (lo & 3) * 4;
        at[e] = lds_address(v + row * RC + ((col / 8) ^ (row & (RC - 1)))) +
                col % 8 * 2;
      }
      read_transposed(r, at);
      #pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint4v w = {r[2 * t][0], r[2 * t][1], r[2 * t + 1][0],
                          r[2 * t + 1][1]};
        const short8 vt = __builtin_bit_cast(short8, w);
        #pragma unroll
        for (int w = 0; w < 3; ++w)
          o[t0 + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              vt, parts[w], o[t0 + t], 0, 0, 0);
      }
    }
  };
  for (int i = 0; i < mine; i += 2) {
    #pragma unroll
    for (int s = 0; s < 2; ++s)
      if (i + s < mine) {
        if (i + s + 1 < mine) wait_loads<2 * LOADS>();
        else wait_loads<0>();
        use(s, i + s);
        if (i + s + 2 < mine) {
          wait_lds_reads();
          load(s, i + s + 2);
        }
      }
  }
  __syncthreads();

  // merge: [wave][head][D + 2], the last two being maximum and sum
  float* red = reinterpret_cast<float*>(s_all);
  constexpr int LD = D + 4;
  l = across_from<16>(l, Plus{});
  float* w = red + (wave * 16 + lo) * LD;
  #pragma unroll
  for (int t = 0; t < DT; ++t)
    *reinterpret_cast<float4v*>(&w[t * 16 + g * 4]) = o[t];
  if (g == 0) { w[D] = m; w[D + 1] = l; }
  __syncthreads();
  for (int e = threadIdx.x; e < heads * (D / 4); e += NW * WAVE) {
    const int h = e / (D / 4), d = e % (D / 4) * 4;
    float M = NONE, L = 0.f;
    #pragma unroll
    for (int i = 0; i < NW; ++i) M = fmaxf(M, red[(i * 16 + h) * LD + D]);
    float4v sum = {0.f, 0.f, 0.f, 0.f};
    #pragma unroll
    for (int i = 0; i < NW; ++i) {
      const float* r = red + (i * 16 + h) * LD;
      const float f = __builtin_amdgcn_exp2f(r[D] - M);
      L += f * r[D + 1];
      sum += f * *reinterpret_cast<const float4v*>(&r[d]);
    }
    const long head = (long)b * hq + head0 + h;
    if (nsplit == 1) {
      const float inv = L > 0.f ? 1.f / L : 0.f;
      *reinterpret_cast<uint2*>(out + head * D + d) =
          make_uint2(pack2(sum[0] * inv, sum[1] * inv),
                     pack2(sum[2] * inv, sum[3] * inv));
    } else {
      const long at = head * nsplit + split;
      *reinterpret_cast<float4v*>(part_o + at * D + d) = sum;
      if (d == 0) {
        // the merging kernel's maxima are natural logarithms
        part_ml[at * 2] = L > 0.f ? M / LOG2E : -INFINITY;
        part_ml[at * 2 + 1] = L;
      }
    }
  }
}

}  // namespace

bool attn_group_takes(int hq, int hkv, int d, long q_ld, const void* q,
                      const void* kc, const void* vc) {
  auto ok = [](const void* p) {
    return reinterpret_cast<uintptr_t>(p) % 16 == 0;
  };
  return hq > hkv && (d == 64 || d == 128) && q_ld % 8 == 0 && ok(q) &&
         ok(kc) && ok(vc);
}

void launch_attn_group(bf16_t* out, const bf16_t* q, const bf16_t* kc,
                       const bf16_t* vc, const int* block_table,
                       const int* seq_lens, int bsz, int hq, int hkv, int d,
                       int max_blocks, float scale, long q_ld, int nsplit,
                       float* part_o, float* part_ml, hipStream_t stream) {
  const int parts = (hq / hkv + 15) / 16;
  // sequences first, as parts of a group read the same keys (see
  // attention_decode_heads.hip; us, 71 heads on 1, 200 x 516 keys, heads first 31.4,
  // now 23.8; 64 x 32 on 8 x 1500, all of them, 83 and 76.5). Where a part is all of
  // a group, long sequences before short ones, heads first then: 32 on 8, unlike, 64
  // x 2500 89.6 -> 80.8, 40 x 2000 55.8 -> 49.4. And groups begin at sequences of
  // their own then, where these are a multiple of eight: an eighth of the chip would
  // have all groups of the same ones, and eighths with long ones end last. 32 on 8,
  // unlike, 24 x 2500 46.6 -> 43.9, 40 x 2500 69.0 -> 65.2, 48 x 2500 80.8 -> 73.0, 72 x
  // 2500 113.9 -> 103.9, 104 x 1500 95.5 -> 91.8; 16 x 2500 30.1 -> 31.3, so not of so
  // few; all of them 40 x 100 12.7 -> 13.2, longer ones the same.
  const dim3 grid(bsz, hkv * parts, nsplit), block(NW * WAVE);
  const bool turned = parts == 1 && bsz % 8 == 0 && bsz > 16 && bsz >= hkv;
  const bool ordered =
      parts == 1 && orders_sequences(bsz, max_blocks, nsplit,
                                     (long)bsz * hkv * nsplit,
                                     d == 128 ? 2 : 4);
  if (d == 128) {
    attn_group_kernel<128><<<grid, block, 0, stream>>>(
        out, q, kc, vc, block_table, seq_lens, hq, hkv, max_blocks, scale,
        q_ld, nsplit, turned, ordered, part_o, part_ml);
  } else {
    attn_group_kernel<64><<<grid, block, 0, stream>>>(
        out, q, kc, vc, block_table, seq_lens, hq, hkv, max_blocks, scale,
        q_ld, nsplit, turned, ordered, part_o, part_ml);
  }
}
