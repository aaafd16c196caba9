// Fused sampling kernel: temperature / top-k /
// top-p + inverse-CDF draw, one workgroup per logits row.
//
// A row is read once, 16 bytes per load, and stays in registers as
// exp(x/T - max): a thread has 8 consecutive logits of every 8192. Thresholds
// are searched over the logits' own ordered bit patterns, by interpolation: top-k
// counts what is not below (one comparison per logit, a wave's count out of its
// mask), top-p adds it up. A step costs one barrier.
//
// Thresholds of bf16 rows of more than 8192 tokens take no steps where they are among
// the 512 largest numbers: the tokens of each of these are counted in LDS.
//
// Bound by vector arithmetic over a row, which one CU has: an operation on every
// logit takes 0.2 us of 32000, its weight 1.5, a step of a search 0.7 to 1, the
// draw's sums in order 5. us on a MI355X, from a search of 4 to 10 steps for every
// threshold and the largest logit found number by number:
//                     greedy      no threshold  top-k 40      top-p .92
//   192 x 32000    6.8 ->  5.5   13.2 -> 12.7   23.5 -> 15.2  22.4 -> 17.1
//   64 x 50272     7.2 ->  5.8   17.8 -> 16.5   33.7 -> 20.6  28.4 -> 22.2
//   256 x 65024   11.7 ->  9.8   36.1 -> 25.6   57.4 -> 32.2  48.8 -> 34.4
//   256 x 1000     4.9 ->  3.7    7.1 ->  6.7   15.1 -> 14.8  18.0 -> 15.5
//   192 x 32000, logits of +-0.1, top-p .92     28.4 -> 25.9 (steps)
//   192 x 32000 in 32 bits   8.1    14.5          24.6           30.7
#include "common.h"

#define SBLOCK 1024
#define SNW (SBLOCK / WAVE)
#define SVEC 8                    // consecutive logits of a thread per round
#define SROUND (SBLOCK * SVEC)
#define RUNS 256                  // runs of tokens that a draw's edges are of
#define LIST 64                   // weights that share 16 bits of a logit
#define SEG 320                   // tokens of a run, at most
#define BINS 512                  // keys below the largest that are counted

namespace {

DEV_INLINE float val(const bf16_t& v) { return bf2f(v); }
DEV_INLINE float val(const float& v) { return v; }

// The high halves of ordered bit patterns: a <= b as floats means that key16(a)
// <= key16(b), of bf16 numbers just then. And the least number that has one.
DEV_INLINE unsigned key16_of(float f) {
  const unsigned b = __float_as_uint(f);
  return (b & 0x80000000u ? ~b : b | 0x80000000u) >> 16;
}
template <class T> DEV_INLINE float number16(unsigned k) {
  const unsigned u = k << 16;
  // (of negative numbers the one whose other bits are set, as keys count)
  return __uint_as_float(u & 0x80000000u ? u ^ 0x80000000u
                         : sizeof(T) == 4 ? ~u : ~u & 0xffff0000u);
}

// Eight logits as they are stored: half the registers of their numbers, if of
// 16 bits. Past the row's end: -inf.
template <class T> struct Eight {
  static constexpr int WORDS = SVEC * sizeof(T) / 4;
  unsigned w[WORDS];

  // VEC: the row is whole 16-byte pieces, of which each is there or not.
  template <bool VEC>
  DEV_INLINE void load(const T* row, int at, int vocab) {
    constexpr int PER = 16 / sizeof(T);
    constexpr unsigned NONE = sizeof(T) == 4 ? 0xff800000u : 0xff80ff80u;
    if constexpr (VEC) {
      #pragma unroll
      for (int p = 0; p < SVEC; p += PER) {
        const uint4v u = *reinterpret_cast<const uint4v*>(
            row + (at + p < vocab ? at + p : 0));
        #pragma unroll
        for (int i = 0; i < 4; ++i)
          w[p / PER * 4 + i] = at + p < vocab ? u[i] : NONE;
      }
    } else {
      #pragma unroll
      for (int i = 0; i < WORDS; ++i) {
        if constexpr (sizeof(T) == 4) {
          w[i] = at + i < vocab ? __float_as_uint(val(row[at + i])) : NONE;
        } else {
          unsigned half[2];
          #pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int from = at + i * 2 + j;
            half[j] = from < vocab
                ? __float_as_uint(val(row[from])) >> 16 : NONE >> 16;
          }
          w[i] = half[0] | half[1] << 16;
        }
      }
    }
  }
  DEV_INLINE float operator[](int j) const {
    if constexpr (sizeof(T) == 4) return __uint_as_float(w[j]);
    return __uint_as_float(j & 1 ? w[j / 2] & 0xffff0000u : w[j / 2] << 16);
  }
};

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
    // as a number of the wave: what follows from it is
    return __uint_as_float(
        __builtin_amdgcn_readfirstlane(__float_as_uint(v)));
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

typedef __attribute__((ext_vector_type(2))) short short2v;
typedef __attribute__((ext_vector_type(2))) unsigned short ushort2v;

// Two bf16 numbers as numbers of 16 bits in the same order: 0 is -inf, USUAL the
// largest that is neither infinite nor NaN (which are above it, of either sign).
// A number's key16_of less that of -inf.
constexpr unsigned USUAL = 0xff00u;
DEV_INLINE ushort2v order16(unsigned w) {
  const short2v s = __builtin_bit_cast(short2v, w);
  const unsigned k =
      w ^ (__builtin_bit_cast(unsigned, (short2v)(s >> 15)) & 0x7fff7fffu);
  return __builtin_bit_cast(ushort2v, k) - (unsigned short)0x807f;
}

// Before a lane: the sums of all lanes ahead of it, by moves to the next lane, the
// second, fourth and eighth of a row, and of whole rows to those behind them.
template <int CTRL, int ROWS>
DEV_INLINE float moved(float v) {
  return __uint_as_float(__builtin_amdgcn_update_dpp(
      0u, __float_as_uint(v), CTRL, ROWS, 0xf, true));
}
DEV_INLINE float sum_upto(float v) {             // a lane's own included
  v += moved<0x111, 0xf>(v);
  v += moved<0x112, 0xf>(v);
  v += moved<0x114, 0xf>(v);
  v += moved<0x118, 0xf>(v);
  v += moved<0x142, 0xa>(v);                     // a row's last to the next row
  v += moved<0x143, 0xc>(v);                     // lane 31 to the upper half
  return v;
}

// What the wave has written to LDS may be read by all of its lanes.
DEV_INLINE void wait_lds() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

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

  // weights for the draw, and before that how many tokens have a key
  constexpr int PART = NR < 4 ? NR : 4;     // rounds whose weights fit LDS
  __shared__ alignas(16) float s_w[PART * SROUND];
  int* bins = reinterpret_cast<int*>(s_w);
  constexpr bool EXACT = sizeof(T) == 2;        // 16 bits are all of a logit
  constexpr bool HALVED = EXACT && NR == 1;
  constexpr bool COUNTED = EXACT && !HALVED;
  if (COUNTED && tid < BINS) bins[tid] = 0;

  // the largest logit; the smallest index of several. NaN is passed over.
  Eight<T> raw[NR];
  float best = -INFINITY, least = INFINITY;
  int besti = 0x7fffffff;
  auto look_at = [&](float v, int i) {
    if (v > best) { best = v; besti = i; }
    least = fminf(least, v > -INFINITY ? v : INFINITY);
  };
  // (read again: kept for the few rows that need it they are short of registers)
  auto look = [&]() {
    for (int i = tid; i < vocab; i += SBLOCK) look_at(val(row[i]), i);
  };
  #pragma unroll
  for (int r = 0; r < NR; ++r)
    raw[r].template load<VEC>(row, r * SROUND + tid * SVEC, vocab);
  // Two numbers an operation where all of a row are finite or -inf, not all -inf:
  // usual. (Of others each is looked at by itself.)
  bool usual = false;
  float top = -INFINITY;
  unsigned mine = 0;
  if constexpr (EXACT) {
    ushort2v most = {0, 0};
    #pragma unroll
    for (int r = 0; r < NR; ++r)
      #pragma unroll
      for (int i = 0; i < Eight<T>::WORDS; ++i)
        most = __builtin_elementwise_max(most, order16(raw[r].w[i]));
    mine = max((unsigned)most[0], (unsigned)most[1]);
    top = totals.most(wave_max(
        mine > USUAL ? INFINITY : number16<T>(mine + key16_of(-INFINITY))));
    usual = top < INFINITY && top > -INFINITY;
  }
  if constexpr (EXACT) {
    if (!usual) look();
  } else {
    #pragma unroll
    for (int r = 0; r < NR; ++r)
      #pragma unroll
      for (int j = 0; j < SVEC; ++j)
        look_at(raw[r][j], r * SROUND + tid * SVEC + j);
  }

  // ---- greedy ---------------------------------------------------------
  if (temp <= 0.f && usual) {
    if (tid == 0) s_tok = 0x7fffffff;
    __syncthreads();
    // zeros of either sign are equal, of other numbers a thread knows its largest
    if (top == 0.f || mine + key16_of(-INFINITY) == key16_of(top)) {
      // read again, which the compiler is not to know: the row kept for this takes
      // registers from all that follows (256 x 65024, no threshold: 39 us for 26).
      // Not one by one: that takes longer than they would.
      int from = tid * SVEC;
      if constexpr (VEC || NR > 4) asm volatile("" : "+v"(from));
      Eight<T> again[NR];
      #pragma unroll
      for (int r = 0; r < NR; ++r) {
        if constexpr (VEC || NR > 4)
          again[r].template load<VEC>(row, r * SROUND + from, vocab);
        else
          again[r] = raw[r];
      }
      #pragma unroll
      for (int r = NR - 1; r >= 0; --r)
        #pragma unroll
        for (int j = SVEC - 1; j >= 0; --j)
          if (again[r][j] == top) besti = r * SROUND + from + j;
      if (besti < vocab) atomicMin(&s_tok, besti);
    }
    __syncthreads();
    if (tid == 0) out[b] = s_tok;
    return;
  }
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
  if (!usual) top = totals.most(wave_max(best));
  const float m = top * inv_t;
  // NaN, and what went past the largest number beside the largest logit: 0. The
  // difference to the largest is rounded once (rounded before it, about a tenth of
  // neighbours in 32 bits would be equal, and thresholds not tell them apart).
  const float past = m == -INFINITY ? m : INFINITY;
  auto weight = [&](float v) {
    const float x = v * inv_t, below = __expf(fmaf(v, inv_t, -m));
    return v == top ? 1.f : x < past ? below : 0.f;
  };
  // of usual ones none is past the largest, and that is 1 as any is (but at an
  // infinite temperature -inf is no number once scaled)
  const bool plain = usual && fabsf(m) < INFINITY && inv_t > 0.f;
  const unsigned first = key16_of(-INFINITY), last = key16_of(top);
  const int k = top_k[b];
  const float p_target = top_p[b];
  const bool some = k > 0 && k < vocab, share = p_target > 0.f &&
                                                p_target < 1.f;
  // Where 512 keys from the largest one down are enough, thresholds are found
  // without steps: one pass counts the tokens of each, and every wave adds them up,
  // eight keys a lane. (With few of a row's numbers within them, or not all usual,
  // steps it is.) us, 192 x 32000, steps -> counts: top-k 40 23.7 -> 15.1, 2000
  // 32.7 -> 15.0, top-p .92 22.3 -> 16.3.
  constexpr int EACH_BIN = BINS / WAVE;
  float tokens[EACH_BIN];
  // (a share of a row whose 512th key still weighs half as much: not there)
  const bool counted =
      COUNTED && plain &&
      (some || (share && weight(number16<T>(max(last, first + BINS) - BINS)) <
                             0.5f));
  if constexpr (COUNTED) {
    if (counted) {
      const unsigned topmost = last - first;
      #pragma unroll
      for (int r = 0; r < NR; ++r) {
        #pragma unroll
        for (int i = 0; i < Eight<T>::WORDS; ++i) {
          const ushort2v u = order16(raw[r].w[i]);
          #pragma unroll
          for (int j = 0; j < 2; ++j)
            if (topmost - u[j] < (unsigned)BINS)
              atomicAdd(&bins[topmost - u[j]], 1);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
      #pragma unroll
      for (int j = 0; j < EACH_BIN; ++j)
        tokens[j] = (float)bins[lane * EACH_BIN + j];
    }
  }
  auto key_at = [&](int i) { return (unsigned)max((int)last - i, (int)first); };

  float e[NR][SVEC];
  auto weigh = [&](auto by) {
    #pragma unroll
    for (int r = 0; r < NR; ++r)
      #pragma unroll
      for (int j = 0; j < SVEC; ++j) {
        e[r][j] = by(raw[r][j]);        // past the row's end: as of -inf
        // a few at a time, or their parts take the registers of the row
        if (j % (NR <= 4 ? 4 : 1) == 0) __builtin_amdgcn_sched_barrier(0);
      }
  };
  if (plain) weigh([&](float v) {
    return v == top ? 1.f : __expf(fmaf(v, inv_t, -m));
  });
  else weigh(weight);
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
  auto count_from = [&](float t) {
    int n = 0;
    #pragma unroll
    for (int r = 0; r < NR; ++r) {
      #pragma unroll
      for (int j = 0; j < SVEC; ++j) n += __popcll(__ballot(e[r][j] >= t));
      __builtin_amdgcn_sched_barrier(0);
    }
    return totals.add((float)n);
  };

  // Two of the 65536 keys of 16 bits between which a threshold lies:
  // measure(weight) holds at lo, not at hi. They are neighbours, or the tokens
  // from lo on, less those from hi on, are no more than FEW. The first `lines` keys
  // are where a line between the logarithms of what was measured at either end, by
  // logits, meets the goal's (but for the third: half way), and an end that stays
  // is moved half way to the goal. From then on what is left is halved: 4 to 10
  // steps in all for most rows, no more than 24. (To go on along the line takes 30
  // and more of rows that it does not fit, as flat ones, or ones with a few tokens
  // far above the rest, and a batch waits for its slowest row. A top-k that leaves
  // much of a row, and top-p of that, fit it least.)
  // Up to 8192 logits of 16 bits cost less to halve than to list: us, 256 rows of
  // 1000, top-k 40, top-p .9, halved 14.2 17.9, by lines throughout 16.7 32.4.
  constexpr float FEW = HALVED ? -1.f : LIST;
  constexpr float MANY = 1e9f;
  const bool large = NR == 1 || (k >= 1024 && k < vocab);
  struct Measured { bool holds; float f, n; };
  struct Ends { unsigned lo, hi; float above; };   // tokens from hi on
  auto search = [&](int lines, auto measure, float goal, float xl, float fl,
                    float fh) {
    unsigned lo = first, hi = last + 1;
    float xh = top, nl = MANY, nh = 0.f;
    int side = 0;
    for (int step = 0; hi - lo > 1 && nl - nh > FEW; ++step) {
      unsigned mid = lo + (hi - lo) / 2;
      if (!HALVED && step < lines) {
        const float x = step == 2
            ? (xl + xh) * 0.5f
            : xl + (xh - xl) * (fl - goal) * __builtin_amdgcn_rcpf(fl - fh);
        mid = min(max(key16_of(x), lo + 1), hi - 1);
      }
      const float x = number16<T>(mid);
      const Measured got = measure(weight(x));
      if (got.holds) {
        lo = mid;
        nl = got.n;
      } else {
        hi = mid;
        nh = got.n;
      }
      if (HALVED || step + 1 >= lines) continue;
      if (got.holds) {
        xl = x;
        fl = __logf(got.f);
        if (side == 1) fh = goal + (fh - goal) * 0.5f;
        side = 1;
      } else {
        xh = x;
        fh = __logf(got.f);
        if (side == 2) fl = goal + (fl - goal) * 0.5f;
        side = 2;
      }
    }
    return Ends{lo, hi, nh};
  };
  // The weights between low and high, sorted out by the first wave's lanes: a
  // lane has one (0: none), how many there are of that and more, and their sum.
  // pick(those) in all threads, or -1 where there are more than LIST.
  __shared__ float s_list[LIST], s_pick;
  __shared__ int s_listed;
  auto between = [&](float low, float high, auto pick) {
    if (tid == 0) s_listed = 0;
    __syncthreads();
    #pragma unroll
    for (int r = 0; r < NR; ++r) {
      #pragma unroll
      for (int j = 0; j < SVEC; ++j)
        if (e[r][j] >= low && e[r][j] < high) {
          const int at = atomicAdd(&s_listed, 1);
          if (at < LIST) s_list[at] = e[r][j];
        }
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    const int listed = s_listed;
    if (listed > LIST) return -1.f;
    if (wave == 0) {
      const float w = lane < listed ? s_list[lane] : 0.f;
      float n = 0.f, sum = 0.f;
      #pragma unroll 4
      for (int i = 0; i < listed; ++i) {
        const float other = __uint_as_float(
            __builtin_amdgcn_readlane(__float_as_uint(w), i));
        n += other >= w ? 1.f : 0.f;
        sum += other >= w ? other : 0.f;
      }
      const float picked = pick(w, n, sum);
      if (lane == 0) s_pick = picked;
    }
    __syncthreads();
    return s_pick;
  };
  // the last weight of [low, high) where holds is true, by halves of its bits
  auto halves = [&](auto holds, float low, float high) {
    unsigned lo = __float_as_uint(low), hi = __float_as_uint(high);
    while (hi - lo > 1) {
      const unsigned mid = lo + (hi - lo) / 2;
      if (holds(__uint_as_float(mid))) lo = mid; else hi = mid;
    }
    return __uint_as_float(lo);
  };
  // The least weight from a key on. Past the last key there is no token: a number
  // as little above the largest logit may weigh no more than that one does.
  auto weight_from = [&](unsigned key) {
    return key > last ? INFINITY : weight(number16<T>(key));
  };

  // The first bin whose sum with those before it passes, or BINS. value(lane's
  // j-th bin) is added up.
  auto first_bin = [&](auto value, auto passes) {
    float own[EACH_BIN], all = 0.f;
    #pragma unroll
    for (int j = 0; j < EACH_BIN; ++j) {
      own[j] = value(j);
      all += own[j];
    }
    float sum = sum_upto(all) - all;
    int at = BINS;
    #pragma unroll
    for (int j = 0; j < EACH_BIN; ++j) {
      sum += own[j];
      if (at == BINS && passes(sum, j)) at = lane * EACH_BIN + j;
    }
    const unsigned long long any = __ballot(at < BINS);
    return any ? __builtin_amdgcn_readlane(at, __ffsll(any) - 1) : BINS;
  };

  // ---- top-k: as many largest as are no more than k with all their equals,
  // ---- the largest and its equals in any case. Measured: tokens
  float thresh = 0.f, floor = -INFINITY;
  if (some) {
    Ends at{};
    int bin = BINS;
    if (counted) {
      bin = first_bin([&](int j) { return tokens[j]; },
                      [&](float n, int) { return n > (float)k; });
      at = Ends{key_at(bin), key_at(bin) + 1, 0.f};
      // a key whose tokens weigh as much as the next one's counts with it
      if (bin > 0 && bin < BINS &&
          !(weight(number16<T>(at.lo)) < weight(number16<T>(at.hi))))
        bin = BINS;
    }
    if (bin == BINS) {
      if (usual) look();
      const float from = HALVED ? 0.f : fmaxf(
          -totals.most(wave_max(-least)), top - 60.f * temp);
      at = search(large ? 1 : 4, [&](float t) {
        const float n = count_from(t);
        return Measured{n > (float)k, fmaxf(n, 0.5f), n};
      }, __logf((float)k + 0.5f), from, __logf((float)vocab), __logf(0.5f));
    }
    if (EXACT && at.hi - at.lo == 1) {
      floor = number16<T>(min(at.hi, last));
      thresh = weight(floor);
    } else {
      floor = number16<T>(at.lo);
      const float low = weight(floor), high = weight_from(at.hi);
      // the smallest that are kept
      float t = between(low, high, [&](float w, float n, float) {
        return -wave_max(w > 0.f && at.above + n <= (float)k ? -w : -high);
      });
      if (t < 0.f) {
        t = halves([&](float t) { return count_from(t) > (float)k; }, low,
                   high);
        t = __uint_as_float(__float_as_uint(t) + 1);
      }
      thresh = fminf(t, 1.f);
    }
  }

  // ---- top-p: the fewest largest weights with that share. Measured: what is
  // ---- left out, which a goal's share of the tokens at most has if each weighs
  // ---- no more than at the first key
  if (share) {
    const float all = sum_from(thresh), goal = p_target * all;
    const float out = all - goal, low = thresh;
    auto enough = [&](float t) { return t < low || sum_from(t) >= goal; };
    constexpr float LESS = 0.135f;              // than what is to be left out
    unsigned lo = 0;
    int bin = BINS;
    if (counted) {
      float w[EACH_BIN];
      #pragma unroll
      for (int j = 0; j < EACH_BIN; ++j)
        w[j] = weight(number16<T>(key_at(lane * EACH_BIN + j)));
      bin = first_bin([&](int j) { return tokens[j] * w[j]; },
                      [&](float s, int j) { return w[j] < low || s >= goal; });
      lo = key_at(bin);
    }
    if (bin == BINS)
      lo = search(large ? 1 : 8, [&](float t) {
        if (t < low) return Measured{true, LESS * out, MANY};
        const float s = sum_from(t);
        return Measured{s >= goal, fmaxf(all - s, 1e-3f * out),
                        s >= goal ? MANY : 0.f};
      }, __logf(out), fmaxf(floor, top - __logf((float)vocab / out) * temp),
         __logf(LESS * out), __logf(all)).lo;
    thresh = fmaxf(low, weight(number16<T>(lo)));
    if constexpr (!EXACT) {
      const float high = weight_from(lo + 1), above = sum_from(high);
      // a sum in another order may be off by its last bits
      const float start = thresh;
      const float t = between(start, high, [&](float w, float, float sum) {
        return wave_max(w > 0.f && above + sum >= goal ? w : start);
      });
      if (t < 0.f || !enough(t) ||
          enough(__uint_as_float(__float_as_uint(t) + 1)))
        thresh = fmaxf(low, halves(enough, thresh, high));
      else
        thresh = fmaxf(low, t);
    }
  }

  // ---- inverse-CDF draw, in token order ---------------------------------
  // Which token a number falls to depends on how sums are rounded: about every
  // two-hundredth draw from thousands of tokens lies that close to an edge. So
  // that a row and a number keep their token, the sum is that of 256 threads
  // over every 256th token, the edges those of 256 runs of tokens, added up
  // from left to right, as they always were.
  __shared__ alignas(16) float s_run[RUNS];
  __shared__ alignas(16) float s_one[SEG];
  const int run = (vocab + RUNS - 1) / RUNS;
  const int from = (tid - RUNS) * run;
  float sum = 0.f;
  #pragma unroll
  for (int r0 = 0; r0 < NR; r0 += PART) {
    if (r0 > 0 || counted) __syncthreads();     // (all have read the bins)
    #pragma unroll
    for (int r = r0; r < NR && r < r0 + PART; ++r) {
      float4 w[2];
      float* f = reinterpret_cast<float*>(w);
      #pragma unroll
      for (int j = 0; j < SVEC; ++j) f[j] = e[r][j] >= thresh ? e[r][j] : 0.f;
      float4* to =
          reinterpret_cast<float4*>(s_w + (r - r0) * SROUND + tid * SVEC);
      to[0] = w[0];
      to[1] = w[1];
    }
    __syncthreads();
    const int base = r0 * SROUND, end = min(vocab, base + PART * SROUND);
    if (tid < RUNS) {
      #pragma unroll 16
      for (int i = base + tid; i < end; i += RUNS) sum += s_w[i - base];
    } else if (tid < 2 * RUNS) {
      const int stop = min(from + run, end);
      #pragma unroll 16
      for (int i = max(from, base); i < stop; ++i) sum += s_w[i - base];
    }
  }
  if (tid < RUNS) {
    sum = wave_sum(sum);
    if (lane == 0) s_tot[0][wave] = sum;
  } else if (tid < 2 * RUNS) {
    s_run[tid - RUNS] = sum;
  }
  if (tid == 0) s_tok = -1;
  __syncthreads();
  if (wave == 0) {
    float z = 0.f;
    #pragma unroll
    for (int q = 0; q < RUNS / WAVE; ++q) z += s_tot[0][q];
    const float goal = uniform[b] * z;
    constexpr int EACH = RUNS / WAVE;
    static_assert(EACH == 4);
    // edges from left to right: every lane goes over all of them, and keeps
    // what there is before its four
    float before = 0.f, upto = 0.f;
    #pragma unroll 8
    for (int l = 0; l < WAVE; ++l) {
      const float4 x = reinterpret_cast<const float4*>(s_run)[l];
      before = lane == l ? upto : before;
      upto = upto + x.x + x.y + x.z + x.w;
    }
    int hit = -1;
    float acc = 0.f;
    #pragma unroll
    for (int q = 0; q < EACH; ++q) {
      const float edge = before + s_run[lane * EACH + q];
      const unsigned long long here = __ballot(goal >= before && goal < edge);
      if (here) {
        const int l = __ffsll(here) - 1;
        hit = l * EACH + q;
        acc = __shfl(before, l, WAVE);
      }
      before = edge;
    }
    if (hit >= 0) {
      // the run's weights, and how many of its sums the goal is not below
      const int first = hit * run, end = min(first + run, vocab);
      for (int i = lane; i < SEG; i += WAVE) {
        float w = 0.f;
        if (first + i < end) {
          if constexpr (NR <= PART) {
            w = s_w[first + i];
          } else {
            w = weight(val(row[first + i]));
            w = w >= thresh ? w : 0.f;
          }
        }
        s_one[i] = w;
      }
      wait_lds();
      int n = 0;
      for (int i = 0; i < run && acc <= goal; i += 16) {
        float4 w[4];
        #pragma unroll
        for (int j = 0; j < 4; ++j)
          w[j] = reinterpret_cast<const float4*>(s_one + i)[j];
        const float* f = reinterpret_cast<const float*>(w);
        #pragma unroll
        for (int j = 0; j < 16; ++j) {
          acc += f[j];
          n += acc <= goal ? 1 : 0;
        }
      }
      // the run's weights, added up one by one to all before them, may end below
      // its edge, to which their sum was added: then its last token is meant
      if (first + n >= end) {
        int kept = -1;
        for (int i = lane; i < run; i += WAVE)
          if (s_one[i] > 0.f) kept = i;
        #pragma unroll
        for (int off = 32; off > 0; off >>= 1)
          kept = max(kept, __shfl_xor(kept, off, WAVE));
        n = kept;
      }
      if (lane == 0 && n >= 0) s_tok = first + n;
    }
  }
  __syncthreads();
  if (s_tok >= 0) {
    if (tid == 0) out[b] = s_tok;
    return;
  }
  // rounding at the very end (goal ~ z): the last token that may be drawn
  int kept = -1;
  for (int i = tid; i < vocab; i += SBLOCK) {
    const float w = weight(val(row[i]));
    if (w > 0.f && w >= thresh) kept = i;
  }
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
