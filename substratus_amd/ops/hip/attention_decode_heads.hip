// Paged decode attention, a workgroup per query head and share of a sequence:
// heads that share no keys, and grouped ones over an fp8 cache for which no
// other kernel is made (head sizes 64 and 128).
//
// Bound by the K/V stream, or with few sequences by the chain of loads to its
// end. A row of K or V is 16 (head size 64: 8) lanes wide, in either the same
// eight elements a lane, so a score that those lanes have added up is where its
// weight is needed: lanes of a row keep a softmax of their own, and nothing
// leaves registers before the end. Both of a step's panels and the next step's
// are in flight, page numbers two steps ahead.
//
// Four or eight waves share a sequence, whose results are merged through LDS. us of
// a captured call, second kernel included where there is one, from a kernel that
// waited for V after its scores and took shares of four waves each (each sequence
// seven keys shorter than the one before it, half the longest at least; caches
// from memory):
//   1 sequence of 150, 16 heads of 128      6.3 -> 4.1
//   1 of 800, 40 heads                      8.9 -> 7.9
//   8 of 900, 32 heads                     24.7 -> 20.6 (5.6 TB/s)
//   5 of 1100, 40 heads                    28.5 -> 22.9
//   256 of 620, 32 heads                    319 -> 316  (6.2 TB/s)
//   30 of 700, 12 heads of 64              18.1 -> 13.8
//   40 of 800, fp8, 71 heads on 1 of 64    49.0 -> 28.4
#include "attention_order.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int PAGE = 16;
constexpr int PIECES = 4;         // of K, or V, that a lane has of a step
constexpr float LOG2E = 1.44269504088896340736f;

// Eight elements of a row.
template <bool KV8> struct Piece;
template <> struct Piece<false> {
  uint4v u;
  DEV_INLINE void load(const char* p) { u = nt_load_u4(p); }
  DEV_INLINE void clear() { u = (uint4v){0, 0, 0, 0}; }
  DEV_INLINE void unpack(float (&f)[8]) const {
    #pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float2 v = unpack_bf16x2(u[i]);
      f[2 * i] = v.x;
      f[2 * i + 1] = v.y;
    }
  }
};
template <> struct Piece<true> {
  uint2v u;
  DEV_INLINE void load(const char* p) { u = nt_load_u2(p); }
  DEV_INLINE void clear() { u = (uint2v){0, 0}; }
  DEV_INLINE void unpack(float (&f)[8]) const {
    #pragma unroll
    for (int i = 0; i < 2; ++i) {
      f[4 * i] = fp8_to_f32<0>(u[i]);
      f[4 * i + 1] = fp8_to_f32<1>(u[i]);
      f[4 * i + 2] = fp8_to_f32<2>(u[i]);
      f[4 * i + 3] = fp8_to_f32<3>(u[i]);
    }
  }
};

// v plus another lane's, by a data-parallel move
template <int CTRL>
DEV_INLINE float plus(float v) {
  return v + __uint_as_float(__builtin_amdgcn_update_dpp(
      0u, __float_as_uint(v), CTRL, 0xf, 0xf, true));
}

// The sum over a row's lanes, in all of them: exchanges within pairs, fours,
// eights and sixteens.
template <int LANES>
DEV_INLINE float row_sum(float v) {
  v = plus<0xb1>(v);                      // quad_perm 1 0 3 2
  v = plus<0x4e>(v);                      // quad_perm 2 3 0 1
  v = plus<0x141>(v);                     // row_half_mirror
  if constexpr (LANES == 16) v = plus<0x140>(v);    // row_mirror
  return v;
}

// In which order workgroups go: every sequence's first head, and so on; a sequence's
// heads; or its heads from another one on for each sequence.
enum class Grid { SEQUENCES, HEADS, TURNED };

// ordered: long sequences first where lengths are unlike
template <int D, bool KV8, int WAVES>
__global__ __launch_bounds__(WAVES * WAVE, 4)
void attn_heads_kernel(bf16_t* __restrict__ out,             // [B, HQ, D]
                       const bf16_t* __restrict__ q,
                       const char* __restrict__ kc,    // [NB, HKV, 16, D]
                       const char* __restrict__ vc,
                       const int* __restrict__ block_table,  // [B, max_blocks]
                       const int* __restrict__ seq_lens,
                       int hq, int hkv, int max_blocks, float scale,
                       long q_ld, int nsplit, Grid from, bool ordered,
                       float* __restrict__ part_o,   // [B, HQ, NS, D]
                       float* __restrict__ part_ml) {  // [B, HQ, NS, 2]
  constexpr int LANES = D / 8;                   // of a row
  constexpr int ROWS = WAVE / LANES;             // of a piece of all lanes
  constexpr int KEYS = PIECES * ROWS;            // of a step
  constexpr int SIZE = KV8 ? 1 : 2;
  const bool sequences = from == Grid::SEQUENCES;
  const int bsz = sequences ? gridDim.x : gridDim.y;
  int b = sequences ? blockIdx.x : blockIdx.y, split = blockIdx.z, at_lane = 0;
  int head = sequences ? blockIdx.y : blockIdx.x;
  if (from == Grid::TURNED) head = (head + b) % hq;
  if (ordered) at_lane = length_at_lane(seq_lens, bsz);
  const int group = hq / hkv;
  int kvh = head / group;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE, row = lane / LANES, at = lane % LANES;
  const int* bt = block_table + (long)b * max_blocks;

  // steps of KEYS keys, one page or two, by turns with other waves
  constexpr int PAGES = KEYS / PAGE;
  const int stride = nsplit * WAVES;
  int first = split * WAVES + wave;
  auto page_of = [&](int step, int p) {
    return max_blocks > 0 ? bt[min(step * PAGES + p, max_blocks - 1)] : 0;
  };
  int page[PAGES], next[PAGES];
  auto begin = [&]() {
    #pragma unroll
    for (int p = 0; p < PAGES; ++p) {
      page[p] = page_of(first, p);
      next[p] = page_of(first + stride, p);
    }
  };
  begin();
  int n = seq_lens[b];
  if (ordered && unlike_lengths(at_lane, max_blocks * PAGE)) {
    const Turn turn = turn_of(hq, nsplit);
    head = turn.head;
    kvh = head / group;
    split = turn.split;
    b = sequence_at(at_lane, bsz, max_blocks * PAGE, turn.sequence);
    bt = block_table + (long)b * max_blocks;
    n = __builtin_amdgcn_readlane(at_lane, b);
    first = split * WAVES + wave;
    begin();
  }
  const int steps = (n + KEYS - 1) / KEYS;

  float qf[8];
  {
    const uint4v u = *reinterpret_cast<const uint4v*>(
        q + (long)b * q_ld + (long)head * D + at * 8);
    #pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float2 v = unpack_bf16x2(u[i]);
      qf[2 * i] = v.x * (scale * LOG2E);
      qf[2 * i + 1] = v.y * (scale * LOG2E);
    }
  }
  struct Panels { Piece<KV8> k[PIECES], v[PIECES]; };
  const long own = (long)kvh * PAGE * D * SIZE + (row * D + at * 8) * SIZE;
  const long page_size = (long)hkv * PAGE * D * SIZE;
  auto load = [&](Panels& x, int step, const int (&pages)[PAGES]) {
    #pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int p = i * ROWS / PAGE;
      // a step's second page may be past the last one: the first again
      const bool there = p == 0 || step * PAGES + p < (n + PAGE - 1) / PAGE;
      x.k[i].load(kc + (there ? pages[p] : pages[0]) * page_size + own +
                  i * ROWS % PAGE * D * SIZE);
    }
    #pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int p = i * ROWS / PAGE;
      const bool there = p == 0 || step * PAGES + p < (n + PAGE - 1) / PAGE;
      x.v[i].load(vc + (there ? pages[p] : pages[0]) * page_size + own +
                  i * ROWS % PAGE * D * SIZE);
    }
  };
  float m = -INFINITY, l = 0.f, acc[8];
  #pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = 0.f;
  auto use = [&](Panels& x, int step) {
    const int key = step * KEYS + row;
    float s[PIECES], most = m;
    #pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      float k[8];
      x.k[i].unpack(k);
      float v = qf[0] * k[0];
      #pragma unroll
      for (int j = 1; j < 8; ++j) v = fmaf(qf[j], k[j], v);
      v = row_sum<LANES>(v);
      s[i] = key + i * ROWS < n ? v : -INFINITY;
      most = fmaxf(most, s[i]);
    }
    // no key yet: its weights are zeros, not differences of infinities
    const float base = most == -INFINITY ? 0.f : most;
    const float keep = __builtin_amdgcn_exp2f(m - base);
    m = most;
    l *= keep;
    #pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] *= keep;
    // a cache's own values past the last key may be no numbers
    if ((step + 1) * KEYS > n) {
      #pragma unroll
      for (int i = 0; i < PIECES; ++i)
        if (key + i * ROWS >= n) x.v[i].clear();
    }
    #pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const float w = __builtin_amdgcn_exp2f(s[i] - base);
      float v[8];
      x.v[i].unpack(v);
      l += w;
      #pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] = fmaf(w, v[j], acc[j]);
    }
  };
  Panels a, c;
  auto turn = [&](int step) {
    #pragma unroll
    for (int p = 0; p < PAGES; ++p) next[p] = page_of(step, p);
  };
  if (first < steps) load(a, first, page);
  for (int t = first; t < steps; t += 2 * stride) {
    if (t + stride < steps) {
      load(c, t + stride, next);
      turn(t + 2 * stride);
    }
    use(a, t);
    if (t + stride >= steps) break;
    if (t + 2 * stride < steps) {
      load(a, t + 2 * stride, next);
      turn(t + 3 * stride);
    }
    use(c, t + stride);
  }

  // the rows' softmaxes become one a wave, and the waves' one
  __shared__ float s_o[WAVES][D], s_m[WAVES], s_l[WAVES];
  // Moves between registers are there sooner than shuffles through LDS, but take
  // three instructions each, and with an fp8 cache those are what there is too
  // little of (71 heads on 1, 200 x 300 keys 59.3 us, 65.5 by moves; 64 x 516 32.3
  // and 33.9; bf16, 64 x 12 x 100 of 64 7.6, and 7.1 by moves).
  auto of_rows = [](float v, auto op) {
    if constexpr (!KV8) return across_from<LANES>(v, op);
    #pragma unroll
    for (int off = LANES; off < WAVE; off *= 2)
      v = op(v, __shfl_xor(v, off, WAVE));
    return v;
  };
  const float most = of_rows(m, Larger{});
  const float f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - most);
  l = of_rows(l * f, Plus{});
  #pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = of_rows(acc[j] * f, Plus{});
  if (row == 0) {
    #pragma unroll
    for (int j = 0; j < 8; j += 4)
      *reinterpret_cast<float4*>(&s_o[wave][at * 8 + j]) =
          make_float4(acc[j], acc[j + 1], acc[j + 2], acc[j + 3]);
    if (at == 0) { s_m[wave] = most; s_l[wave] = l; }
  }
  __syncthreads();
  if ((int)threadIdx.x >= D / 2) return;
  float M = -INFINITY, L = 0.f, o0 = 0.f, o1 = 0.f;
  #pragma unroll
  for (int w = 0; w < WAVES; ++w) M = fmaxf(M, s_m[w]);
  const int d = threadIdx.x * 2;
  #pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    const float e =
        s_m[w] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s_m[w] - M);
    L += e * s_l[w];
    o0 += e * s_o[w][d];
    o1 += e * s_o[w][d + 1];
  }
  const long h = (long)b * hq + head;
  if (nsplit == 1) {
    const float inv = L > 0.f ? 1.f / L : 0.f;
    *reinterpret_cast<unsigned*>(out + h * D + d) =
        pack_bf16x2(o0 * inv, o1 * inv);
  } else {
    const long part = h * nsplit + split;
    *reinterpret_cast<float2*>(part_o + part * D + d) = make_float2(o0, o1);
    if (d == 0) {
      // the merging kernel's maxima are natural logarithms
      part_ml[part * 2] = M / LOG2E;
      part_ml[part * 2 + 1] = L;
    }
  }
}

}  // namespace

// Waves of a workgroup, and workgroups that share a sequence: by shapes only, so
// that a captured graph holds them; lengths may be as unlike as the table lets
// them. A CU reads some 55 GB/s, so heads are shared where they would leave CUs
// idle, or where a second round of them would be all but empty: by workgroups of
// four waves, four a CU (eight waves, or more shares than that, cost as much empty
// as they do full). Merging takes 2 us, so the line is where the longest sequence
// that the table has room for has steps that take more: the more heads the round
// has, the later. Alone, eight waves end sooner until there are four heads a CU;
// then four, of which more fit, lose less to sequences shorter than the table. us
// on a MI355X, keys of all, or of one (the others' a twentieth), by shares of four
// waves, and alone by eight:
//   heads x keys          all 1    2    4    8 (eight)   one 1    2    4    8 (eight)
//   64 x 400 of 128         7.3  7.5  6.9  6.7   6.3       6.7  7.2  6.5  6.3   6.6
//   64 x 900               13.0 10.7  8.7  8.4  11.1      12.9 10.5  8.3  8.0  11.0
//   64 x 4000              48.0 30.0 23.1 23.4  44.6      47.0 28.5 18.7 18.4  39.9
//   192 x 900              15.3 16.9 16.7 16.2  15.6      13.0 10.5  8.8  9.4   9.8
//   192 x 4000             58.5 65.6 63.0 63.2  63.3      47.6 29.4 20.1 25.1  40.1
//   256 x 4000             79.2 81.0 80.4 80.2  81.8      53.0 55.4 55.0 55.0  53.0
//   288 x 2000 of 64       30.9 27.0 25.0 24.4  29.1      15.2 12.2 12.6 12.5  13.5
//   384 x 2000 of 64       34.6 31.5 31.3 31.4  31.8      22.1 20.1 19.7 19.5  21.6
//   576 x 2000 of 64       50.0 47.7 44.3 44.6  46.9      15.8 16.6 16.6 18.3  15.5
//   1152 x 150 of 64        8.6 11.5 14.2        10.5       7.0                 9.0
//   1152 x 2000 of 64      89.1 87.6 84.5 84.3  85.1      24.7 26.6 26.6 30.7  27.4
// and where the table has room for 8192 keys, 4544 and 18176 heads x 150 of 64 in
// fp8, alone by four and by eight: 13.8 19.6, 47.5 70.7.
void attn_heads_plan(int bsz, int hq, int d, int max_blocks, int& waves,
                     int& nsplit) {
  const long heads = std::max((long)bsz * hq, 1L);
  const int pages = PIECES * WAVE * 8 / d / PAGE;          // of a step
  const long steps = (max_blocks + pages - 1) / pages;
  const long rest = heads % 256;                           // of the last round
  const bool idle = rest > 0 &&
                    (heads < 256 ? rest <= 232 : heads < 512 && rest <= 96);
  const bool shared = idle && steps * 4 > 40 + rest;
  const long fit = (1024 + heads / 2) / heads;
  waves = shared || heads >= 1024 ? 4 : 8;
  nsplit = !shared ? 1 : std::clamp(fit, 2L, heads < 48 ? 16L : 8L);
}

void launch_attn_heads(bf16_t* out, const bf16_t* q, const void* kc,
                       const void* vc, const int* block_table,
                       const int* seq_lens, int bsz, int hq, int hkv, int d,
                       int max_blocks, float scale, long q_ld, int waves,
                       int nsplit, float* part_o, float* part_ml, bool kv8,
                       hipStream_t stream) {
  // Workgroups go to the eighths of the chip in turn. Sequences first, a sequence's
  // heads come to the same eighth where there is a multiple of eight of them: keys
  // that heads share, and their pages' addresses, come to its caches once, but where
  // lengths are unlike the eighths are, too. Heads first, an eighth reads its own
  // eighth of all pages, and meets the others at few of the memory's channels where
  // lengths are equal; turned by the sequence it does not, and a long sequence has all
  // of the chip. So heads are first where they share no keys, and turned where there
  // are more than the chip holds at a time (four a CU). us, MI355X, sequences first,
  // heads first, turned; keys from a quarter of the most to all, all of them, one of
  // them (the others' a twentieth):
  //   sequences x heads x keys      unlike         all            one (2500)
  //   512 x 32 x 516                             698  764  660
  //   256 x 32 x 516                             387  348  327
  //   64 x 32 x 1500             168  157  158   250  259  239   118   48   48
  //   256 x 12 x 1500 of 64      119  117  117   173  175  174    55   29   29
  //   64 x 16 x 1500 of 64      47.1 44.5 43.8                    51   32   32
  //   20 x 32 x 900             39.1 35.7 35.7  52.9 51.6 52.5
  //   8 x 32 x 2000             36.0 35.4 35.5  45.4 45.9 46.0
  //   8 x 40 x 2000             46.9 44.8 44.8  57.5 57.7 57.7
  //   64 x 71 on 1 x 516, fp8                   33.7 37.3
  // Shares come last: behind each sequence's heads, those of a table's unused room are
  // between those that have keys (4 x 32 x 60 in a table of 4096 6.3 -> 7.9; 4 x 32 x
  // 2000 unlike 21.1 -> 20.2).
  // Long sequences before short ones, heads first then (attention_order.h): 30 x 40
  // x 1100 unlike 74.7 -> 70.5, 64 x 71 on 1 x 1500, fp8, unlike 71.1 -> 61.5.
  const Grid from = hq != hkv || bsz > MOST ? Grid::SEQUENCES
                    : (long)bsz * hq < 1024 ? Grid::HEADS
                                            : Grid::TURNED;
  const dim3 grid = from == Grid::SEQUENCES ? dim3(bsz, hq, nsplit)
                                            : dim3(hq, bsz, nsplit);
  const bool ordered = orders_sequences(bsz, max_blocks, nsplit,
                                        (long)bsz * hq * nsplit, 16 / waves);
  auto go = [&](auto dim, auto fp8, auto w) {
    constexpr int W = decltype(w)::value;
    attn_heads_kernel<decltype(dim)::value, decltype(fp8)::value, W>
        <<<grid, dim3(W * WAVE), 0, stream>>>(
            out, q, reinterpret_cast<const char*>(kc),
            reinterpret_cast<const char*>(vc), block_table, seq_lens, hq, hkv,
            max_blocks, scale, q_ld, nsplit, from, ordered, part_o, part_ml);
  };
  auto sized = [&](auto dim, auto fp8) {
    if (waves == 8) go(dim, fp8, std::integral_constant<int, 8>());
    else go(dim, fp8, std::integral_constant<int, 4>());
  };
  auto typed = [&](auto dim) {
    if (kv8) sized(dim, std::true_type());
    else sized(dim, std::false_type());
  };
  if (d == 128) typed(std::integral_constant<int, 128>());
  else typed(std::integral_constant<int, 64>());
}
