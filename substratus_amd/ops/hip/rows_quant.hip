// y = x w^T of up to 64 rows with a GGUF-quantized weight matrix [n, k], or,
// of a matrix whose first half gates its second, silu(gate) * up, or, of a
// projection of heads, rotated queries, with keys and values appended to the
// cache. Weights as
// models/quant.py lays them out:
//   q4_0, q8_0   scales fp16 [n, k/32]; qs [n, k/2] nibbles (byte i of a block
//                has weights i and i + 16), [n, k] int8
//   q4_K         scales fp16 [n, k/128] (d and dmin of each 256); qs rows: a
//                6-bit scale per 32, a 6-bit minimum per 32, nibbles (byte l
//                of 64 weights has l and l + 32)
//   q6_K         scales fp16 [n, k/256]; qs rows: low nibbles, high pairs of
//                bits, an int8 scale per 16
//
// Bound by reading packed weights and by unpacking them. Unpacked they are
// whole numbers, which bf16 holds exactly, and the matrix cores multiply them
// with x as they are, so that a block's 32-bit sum holds nothing that is taken
// off again (an offset, which is cheap to unpack with, would cost its last bits
// where x is large, and make an infinite x no number). Four bits are bytes that
// count as small 8-bit floating-point numbers, of which one operation converts
// two; six bits go to the top of their bytes, which are then 4 times the number
// with a sign, and are converted like eight bits one by one. Minima need the
// sums of x, which a product with ones gives. One instruction's inner size is
// one block, so its sum is scaled in 32 bits and added up, as in a loop over
// blocks in 32-bit arithmetic.
//
// A workgroup takes 16 weight rows and MR rows of x; its waves share k. A
// stage is 256 columns; weights, scales and x go straight to LDS with
// consecutive lanes on consecutive bytes (see rows_gemm.hip), pieces permuted
// by the row against bank conflicts. Few rows of x: P stages in flight per
// wave; many: one, and more workgroups per CU instead. A single row of x comes as
// such: with three more of no use, stages took half as much LDS again, and two of
// them in flight left a CU fewer workgroups. us of 15360 x 5120, 5120 x 5120, 27648
// x 5120, 5120 x 13824, 12288 x 4096, 22016 x 4096, 32000 x 5120, each from memory,
// four rows, in four waves of wide matrices (of q4_0 and q6_K with one stage in flight)
// -> one, in eight waves (of q4_0 with two stages):
//   q4_0  13.8 6.8 22.5 13.8 9.2 15.3 27.8 -> 13.5 6.5 22.4 12.9 8.2 14.8 26.3
//   q4_K  14.5 7.5 25.5 15.6 9.0 16.4 28.8 -> 14.2 6.8 24.2 15.3 8.8 15.2 27.9
//   q6_K  20.7 10.7 33.7 26.8 12.6 22.6 37.0 -> 20.0 10.9 33.6 27.1 12.1 21.1 36.6
// and of a captured step of 8 layers of 5120, q4_0, 523 -> 503.
// A load takes 8 rows x 128 bytes of weights, where 16 x 64 asked for every
// line twice. q6_K keeps the halves: a row is half a line more than whole ones,
// and what a stage asks for is four kinds of pieces, of which two are less than
// a line. us, weights not in a cache, 15360 x 5120, 5120 x 5120, 27648 x 5120,
// 5120 x 13824, 12288 x 4096, 4096 x 11008, halves -> lines:
//   q4_0  1 row   14.2 7.2 23.2 16.8 10.0 10.9 -> 14.1 7.4 21.8 16.5 10.3 9.5
//   q8_0  3 rows  20.8 10.7 33.5 24.1 13.8 13.1 -> 19.4 10.3 31.6 22.5 12.8 13
//   q4_K  5 rows  18.2 8.6 30.0 24.9 11.6 12.6 -> 17.8 8.7 29.1 23.8 11.5 12.2
//   q6_K  5 rows  5120 x 5120 11.9 -> 15.3, 24 rows 15360 x 5120 35.6 -> 39.2
//
// us on a MI355X with weights partly in a cache, before that, 15360 x 5120,
// 5120 x 5120, 27648 x 5120, 5120 x 13824, from one wave per weight row in
// vector arithmetic (up to 8 rows of x), or from unpacking to bf16 in memory and
// the library (more), to this kernel:
//   q4_0  1 row   20.5  8.5 31.7 15.0 -> 12.9  7.2 20.9 15.3
//         5 rows  55.0 21.5 95.3 47.8 -> 14.1  7.7 22.9 16.9
//        24 rows  81.4 37.8  152 75.9 -> 23.5 12.5 38.7 26.5
//   q8_0  5 rows  55.9 21.2 97.5 46.3 -> 22.2 11.9 36.0 25.7
//        24 rows  82.5 38.8  155 78.9 -> 40.6 20.7 69.9 43.6
//   q4_K  1 row   29.4 12.9 49.4 24.6 -> 12.8  7.3 21.4 16.1
//         5 rows   115 47.7  196  111 -> 15.5  8.6 24.8 18.6
//        24 rows  90.1 37.8  172 84.6 -> 25.9 15.1 43.2 31.4
//   q6_K  1 row   32.7 13.3 57.5 26.8 -> 20.6 11.0 29.9 25.8
//         5 rows   118 40.9  205 90.9 -> 22.4 12.1 31.4 28.6
//        24 rows   523  196  946  479 -> 35.7 18.8 51.9 44.1
// (4-bit numbers with an offset of 24 or 16, which one operation unpacked, took
// 12.6 7.0 20.4 14.4 and 13.3 7.4 22.2 16.6 for one row, 27.5 14.1 50.0 33.3
// and 28.5 14.3 51.2 35.7 for 24.)
// q8_0 with one row stays with the vector kernel (quant_gemv.hip): 20.5, 9.4,
// 33.1, 19.3 there and 19.9, 11.1, 32.2, 23.8 here.
#include "rows_quant.h"

#include <type_traits>

namespace {

typedef _Float16 f16_t;
using std::integral_constant;

constexpr int COLS = 256;         // of a stage
constexpr int TILE = 64;          // 16-byte pieces of 16 rows x 64 bytes

DEV_INLINE short8 vec8(unsigned a, unsigned b, unsigned c, unsigned d) {
  return __builtin_bit_cast(short8, (uint4v){a, b, c, d});
}

DEV_INLINE float half_of(unsigned u) {       // its low 16 bits
  return (float)__builtin_bit_cast(f16_t, (unsigned short)(u & 0xffff));
}

DEV_INLINE float half_at(const uint4v& u, int i) {
  return half_of(u[i >> 1] >> (16 * (i & 1)));
}

DEV_INLINE float byte_at(const uint4v& u, int i) {
  return (float)((u[i >> 2] >> (8 * (i & 3))) & 0xff);
}

// The high halves of two words.
DEV_INLINE unsigned high2(unsigned a, unsigned b) {
  return __builtin_amdgcn_perm(b, a, 0x07060302);
}

// Four signed bytes as bf16, which holds whole numbers up to 256.
DEV_INLINE uint2v unpack4(unsigned v) {
  float f[4];
  #pragma unroll
  for (int i = 0; i < 4; ++i) f[i] = (float)(signed char)(v >> (8 * i) & 0xff);
  return {high2(__float_as_uint(f[0]), __float_as_uint(f[1])),
          high2(__float_as_uint(f[2]), __float_as_uint(f[3]))};
}

template <int ME>
DEV_INLINE void add_scaled(float4v& a, float s, const float4v& v) {
  #pragma unroll
  for (int e = 0; e < ME; ++e) a[e] += s * v[e];
}

// Four numbers of 4 exponent and 3 mantissa bits as 512 times what they are, in
// bf16: one operation converts two. As such numbers bytes below 16 are 0 to 15
// times 2^-9.
DEV_INLINE uint2v unpack_small(unsigned v) {
  return {__builtin_bit_cast(
              unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 512.f,
                                                                  false)),
          __builtin_bit_cast(
              unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 512.f,
                                                                  true))};
}

// Bytes n below 16 as such numbers of n - 8: 0x88 - n or n - 8. A selector of
// 8 and more gives 0 or 255, by the table's own signs below 12, so each half of
// the table undoes what the other one gives there.
DEV_INLINE unsigned minus8(unsigned n) {
  return __builtin_amdgcn_perm(0x7E7D7C84u, 0x7A798788u, n) ^
         __builtin_amdgcn_perm(0xF8F9FA04u, 0x030201FFu, n ^ 0x08080808u);
}

// One result by weights and not by their two parts, whose sums are infinite
// with opposite signs where x is.
DEV_INLINE float dot_q4k(const bf16_t* x, const unsigned char* row,
                         const f16_t* d, int k) {
  float s = 0.f;
  for (int i = 0; i < k; ++i) {
    const unsigned b = row[k / 16 + i / 64 * 32 + i % 32];
    const float w = (float)d[i / 256 * 2] * (float)row[i / 32] *
                        (float)(i & 32 ? b >> 4 : b & 15) -
                    (float)d[i / 256 * 2 + 1] * (float)row[k / 32 + i / 32];
    s += w * bf2f(x[i]);
  }
  return s;
}

// Tiles of 16 rows x 64 bytes in a stage, 16-byte scale rows, loads of both;
// how many times the number unpacked weights are.
template <Quant Q> struct Layout;
template <> struct Layout<Quant::Q4_0> {
  static constexpr int W = 2, S = 1, LOADS = 3, TIMES = 1;
};
template <> struct Layout<Quant::Q8_0> {
  static constexpr int W = 4, S = 1, LOADS = 5, TIMES = 1;
};
template <> struct Layout<Quant::Q4_K> {
  static constexpr int W = 2, S = 2, LOADS = 4, TIMES = 1;
};
template <> struct Layout<Quant::Q6_K> {
  static constexpr int W = 3, S = 1, LOADS = 5, TIMES = 4;   // one to a register
};

// MR: rows of x; ME: of every four, those that are there (MR 4 only); KW
// waves share k, P stages are in flight in each. THIN: a workgroup has eight
// weight rows, and the other eight of an operand are the next 256 columns of the
// same ones, beside those of x (MR 8 at most): a stage is 512 columns.
template <Quant Q, int MR, int ME, int KW, int P, Columns C, bool NORM,
          bool THIN>
// (one row: 80 registers at most, or what a stage needs before its turn takes 118
// and a workgroup's place; 559 us instead of 549 for a step of 8 layers of 5120,
// q4_0. With more rows of x the same costs a tenth, with q4_K's two stages in
// flight up to 6 %.)
__global__ __launch_bounds__(KW * WAVE, ME == 1 && !NORM &&
                                                (Q == Quant::Q4_0 || THIN)
                                            ? 6 : 2)
void rows_quant_kernel(bf16_t* __restrict__ y, const bf16_t* __restrict__ x,
                       const f16_t* __restrict__ scales,
                       const unsigned char* __restrict__ qs, int m, int n,
                       int k, Heads heads, NormOf norm, AddTo add,
                       Undivided of) {
  using L = Layout<Q>;
  constexpr bool K_QUANT = Q == Quant::Q4_K || Q == Quant::Q6_K;
  static_assert(!THIN || (MR <= 8 && !NORM && !paired(C) &&
                          Q != Quant::Q6_K));
  constexpr int HALVES = THIN ? 2 : 1, XW = 2 * HALVES;
  constexpr int FM = (MR + 15) / 16;
  // loads of x, 4 rows x 256 B, XW to a row, or all of a single row (normed x
  // does not go through the ring)
  constexpr bool ONE = ME == 1 && !NORM;
  constexpr int XL = NORM ? 0 : ONE ? 1 : MR / 4 * XW;
  constexpr int WS = L::W * TILE + L::S * 16;    // weights and scales
  constexpr int STAGE = (ONE ? HALVES * 32 : XL * 64) + WS;
  constexpr int LOADS = XL + L::LOADS;
  constexpr int BM = FM * 16, PAD = 1;
  constexpr int RED = (KW * BM * (16 + PAD) + 3) / 4, RING = KW * P * STAGE;
  constexpr int BEFORE = RING > RED ? RING : RED;
  __shared__ alignas(16)
      uint4v s_all[BEFORE + (NORM ? NORM_PIECES + NORM_ROWS + KW : BM / 4)];
  uint4v* s_x = s_all + BEFORE;
  auto squares = reinterpret_cast<float (*)[NORM_ROWS]>(
      s_x + NORM_PIECES + NORM_ROWS);

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE;
  const int lo = lane & 15, g = lane >> 4;
  const int n0 = THIN ? blockIdx.x * 8 : first_column<C>(heads);
  const int half = second_half<C>(n, heads);
  x += (long)blockIdx.y * MR * k;
  m -= blockIdx.y * MR;
  const int nb = k / 32, all = (k + COLS * HALVES - 1) / (COLS * HALVES);
  const int c0 = all * wave / KW, c1 = all * (wave + 1) / KW;
  const int steps = c1 - c0;
  uint4v* ring = s_all + wave * P * STAGE;

  // bytes of a row of weights, of scales
  const long rb = Q == Quant::Q4_0 ? k / 2 : Q == Quant::Q8_0 ? k
      : Q == Quant::Q4_K ? k / 16 + k / 2 : k / 16 * 13;
  const long sb = !K_QUANT ? nb * 2 : Q == Quant::Q4_K ? k / 64 : k / 128;
  // a lane loads 16 bytes of row lane / 4 of a tile, and a word of its scales;
  // of lines of 128 bytes, of row lane / 8 or eight later
  const int row = lane >> 2, piece = (lane & 3) ^ ((row >> 2) & 3);
  const int word = lane & 3;
  const unsigned char* pair[2];
  int in_pair[2];
  #pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = h * 8 + (lane >> 3), from = THIN ? lane >> 3 : r;
    in_pair[h] = (lane & 7) ^ (r >> 1);
    pair[h] = qs + weight_row<C>(n0, from, n, half) * rb;
  }
  const unsigned char* sc = reinterpret_cast<const unsigned char*>(scales);
  // THIN: the half of a stage that rows 8 to 15 are
  const int up = THIN ? row >> 3 : 0, lo_up = THIN ? lo >> 3 : 0;
  const int row_w = THIN ? row & 7 : row, lo_w = THIN ? lo & 7 : lo;
  const unsigned char* wp = qs + weight_row<C>(n0, row_w, n, half) * rb;
  const unsigned char* sp = sc + weight_row<C>(n0, row_w, n, half) * sb;
  const unsigned char* dp = sc + weight_row<C>(n0, lo_w, n, half) * sb;
  const char* xp[XL / XW + 1];
  #pragma unroll
  for (int d = 0; d < (ONE ? 1 : XL / XW); ++d)
    xp[d] = reinterpret_cast<const char*>(
        x + (long)min(d * 4 + (lane >> 4), m - 1) * k);
  static_assert(P == 1 || Q != Quant::Q6_K);
  unsigned short dreg;                           // q6_K: the stage's d
  // the 256 columns that a stage's half has, or the last ones again
  auto of_stage = [&](int c, int h) {
    return THIN ? min(c * 2 + h, k / 256 - 1) : c;
  };
  auto load = [&](int s, int c) {
    uint4v* ws = ring + s * STAGE;
    uint4v* ss = ws + L::W * TILE;
    // past a row's last block: that block again, which nobody reads
    if constexpr (Q == Quant::Q4_0) {
      #pragma unroll
      for (int t = 0; t < 2; ++t)
        load_to_lds<16>(pair[t] + min((c * HALVES + (THIN ? t : 0)) * 8 +
                                          in_pair[t], nb - 1) * 16,
                        ws + t * TILE);
      load_to_lds<4>(sp + min((c * HALVES + up) * 16 + word * 4, nb * 2 - 4),
                     ss);
    } else if constexpr (Q == Quant::Q8_0) {
      #pragma unroll
      for (int t = 0; t < 4; ++t)
        load_to_lds<16>(
            pair[t & 1] + min((c * HALVES + (THIN ? t & 1 : 0)) * 256 +
                                  (t >> 1) * 128 + in_pair[t & 1] * 16,
                              k - 16),
            ws + t * TILE);
      load_to_lds<4>(sp + min((c * HALVES + up) * 16 + word * 4, nb * 2 - 4),
                     ss);
    } else if constexpr (Q == Quant::Q4_K) {
      #pragma unroll
      for (int t = 0; t < 2; ++t)
        load_to_lds<16>(pair[t] + k / 16 + of_stage(c, THIN ? t : 0) * 128 +
                            in_pair[t] * 16,
                        ws + t * TILE);
      // words: scales 0 to 3, 4 to 7, minima 0 to 3, 4 to 7
      load_to_lds<4>(wp + (word & 2) * (k / 64) + of_stage(c, up) * 8 +
                         (word & 1) * 4, ss);
      load_to_lds<4>(dp + of_stage(c, lo_up) * 4, ss + 16);
    } else {
      #pragma unroll
      for (int t = 0; t < 2; ++t)
        load_to_lds<16>(wp + c * 128 + t * 64 + piece * 16, ws + t * TILE);
      load_to_lds<16>(wp + k / 2 + c * 64 + piece * 16, ws + 2 * TILE);
      load_to_lds<4>(wp + k / 4 * 3 + c * 16 + word * 4, ss);
      // two bytes only: words need not be aligned
      dreg = *reinterpret_cast<const unsigned short*>(dp + c * 2);
    }
    uint4v* xs = ws + WS;
    if constexpr (ONE) {
      const int p = c * HALVES * 32 + (lane ^ (lane >> 5) * 4);
      if (THIN || lane < 32)
        load_to_lds<16>(xp[0] + (long)min(p, k / 8 - 1) * 16, xs);
      return;
    }
    #pragma unroll
    for (int d = 0; d < XL; ++d) {
      const int p = (c * XW + d % XW) * 16 +
                    (lo ^ ((lane >> 4) << 2) ^ (d / XW & 3));
      load_to_lds<16>(xp[d / XW] + (long)min(p, k / 8 - 1) * 16, xs + d * 64);
    }
  };

  const short8 ones = vec8(0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u);
  const float4v zero = {0.f, 0.f, 0.f, 0.f};
  // q4_0: lanes of the first 16 weights take low nibbles, the others high ones
  const int down = g >> 1 ? 4 : 0;
  int xr[FM];                                    // the lane's rows of x
  #pragma unroll
  for (int j = 0; j < FM; ++j) {
    const int r = (j * 16 + lo) & (MR - 1);
    xr[j] = ONE ? lo_up * 32 : (r >> 2) * (XW * 64) + lo_up * 128 + (r & 3) * 16;
  }
  const int xsw = ONE ? lo_up * 4
                      : ((lo & 3) << 2) ^
                            (((lo & (MR > 16 ? 15 : MR - 1)) >> 2) & 3);
  // piece i of block b of a row
  auto x_at = [&](int b, int i) {
    return ONE ? (b * 4 + i) ^ xsw
               : (b >> 2) * 64 + (((b * 4 + i) & 15) ^ xsw);
  };
  const int wsw = Q == Quant::Q6_K ? lo >> 2 : lo >> 1;
  const uint4v* x_row = s_x + min(lo & (MR - 1), m - 1) * (k / 8 + 1);
  float4v acc[FM];
  #pragma unroll
  for (int j = 0; j < FM; ++j) acc[j] = zero;

  auto use = [&](int s, int c, auto whole) {
    const uint4v* ws = ring + s * STAGE;
    const uint4v* row = ws + lo * (Q == Quant::Q6_K ? 4 : 8);
    const uint4v* ss = ring + s * STAGE + L::W * TILE;
    const uint4v* xs = ring + s * STAGE + WS;
    const uint4v sv = ss[lo];
    float d = 0.f, dm = 0.f;
    if constexpr (Q == Quant::Q4_K) {
      const unsigned dd = reinterpret_cast<const unsigned*>(ss + 16)[lo];
      d = half_of(dd) / L::TIMES;
      dm = -half_of(dd >> 16);
    }
    if constexpr (Q == Quant::Q6_K) d = half_of(dreg) / L::TIMES;
    // the lane's eight weights of a block, k = 8 g on, out of eight bytes
    auto weights = [&](int b) {
      const int at = Q == Quant::Q4_0 ? b & 3
          : Q == Quant::Q8_0 ? (b & 1) * 2 + (g >> 1)
                             : ((b >> 1) & 1) * 2 + (g >> 1);
      // four blocks of q8_0 are a line
      const int line = Q == Quant::Q8_0 ? (b >> 2) * 2 * TILE : 0;
      const int in = Q == Quant::Q8_0 ? (b >> 1 & 1) * 4 + at
                                      : (b >> 2) * 4 + at;
      const uint2v v = reinterpret_cast<const uint2v*>(
          row + line + (in ^ wsw))[g & 1];
      uint2v w[2];
      #pragma unroll
      for (int h = 0; h < 2; ++h) {
        if constexpr (Q == Quant::Q4_0)
          w[h] = unpack_small(minus8(v[h] >> down & 0x0F0F0F0Fu));
        else if constexpr (Q == Quant::Q8_0)
          w[h] = unpack4(v[h]);
        else
          w[h] = unpack_small((b & 1 ? v[h] >> 4 : v[h]) & 0x0F0F0F0Fu);
      }
      return vec8(w[0][0], w[0][1], w[1][0], w[1][1]);
    };
    #pragma unroll
    for (int b = 0; b < COLS / 32; ++b) {
      if (!decltype(whole)::value && c * HALVES * 8 + b >= nb) break;
      // a stage's second half may have fewer blocks than its first, or none
      const bool there = !THIN || decltype(whole)::value ||
                         (c * 2 + lo_up) * 8 + b < nb;
      if constexpr (Q != Quant::Q6_K) {
        // two blocks at a time: the second's work is done while the first's
        // products are on their way
        if (b & 1) continue;
        const short8 wv[2] = {weights(b), weights(b + 1)};
        #pragma unroll
        for (int j = 0; j < FM; ++j) {
          float4v p[2], sums[2];
          #pragma unroll
          for (int t = 0; t < 2; ++t) {
            const short8 xv = __builtin_bit_cast(
                short8, NORM ? x_row[c * 32 + (b + t) * 4 + g]
                             : xs[xr[j] + x_at(b + t, g)]);
            p[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xv, wv[t], zero, 0,
                                                           0, 0);
            if constexpr (Q == Quant::Q4_K)
              sums[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  xv, ones, zero, 0, 0, 0);
          }
          if (!there) continue;
          #pragma unroll
          for (int t = 0; t < 2; ++t) {
            add_scaled<ME>(acc[j], Q == Quant::Q4_K ? d * byte_at(sv, b + t)
                                                    : half_at(sv, b + t),
                           p[t]);
            if constexpr (Q == Quant::Q4_K)
              add_scaled<ME>(acc[j], dm * byte_at(sv, 8 + b + t), sums[t]);
          }
        }
      } else {
        // a scale per 16 weights: instructions of inner size 16
        const int hf = b >> 2, quarter = b & 3;
        #pragma unroll
        for (int h = 0; h < 2; ++h) {
          const unsigned v = reinterpret_cast<const unsigned*>(
              row + hf * TILE + (((quarter & 1) * 2 + h) ^ wsw))[g];
          const unsigned hv = reinterpret_cast<const unsigned*>(
              row + 2 * TILE + ((hf * 2 + h) ^ wsw))[g];
          const unsigned low = (quarter < 2 ? v << 2 : v >> 2) & 0x3C3C3C3Cu;
          const unsigned high = hv << (6 - 2 * quarter) & 0xC0C0C0C0u;
          const short4v wv = __builtin_bit_cast(
              short4v, unpack4((low | high) ^ 0x80808080u));
          const int si = hf * 8 + quarter * 2 + h;
          const float scale = d * (float)(signed char)(
              (sv[si >> 2] >> (8 * (si & 3))) & 0xff);
          #pragma unroll
          for (int j = 0; j < FM; ++j) {
            const int i = h * 2 + (g >> 1);
            const short4v xv = __builtin_bit_cast(
                short4v, reinterpret_cast<const uint2v*>(
                    NORM ? x_row + c * 32 + b * 4 + i
                         : xs + xr[j] + x_at(b, i))[g & 1]);
            add_scaled<ME>(acc[j], scale,
                           __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
                               xv, wv, zero, 0, 0, 0));
          }
        }
      }
    }
  };

  // a thread ends up with column lo of every ROWSth row from first on
  constexpr int ROWS = KW * WAVE / 16, PER = (BM + ROWS - 1) / ROWS;
  const int first = threadIdx.x / 16, m_here = min(m, MR);
  bf16_t h[PER], weight;
  float* row_squares = reinterpret_cast<float*>(s_all + BEFORE);
  NormRows<KW * WAVE> rows;
  if constexpr (NORM) rows.load(norm, m, k);
  #pragma unroll
  for (int s = 0; s < P; ++s)
    if (s < steps) load(s, c0 + s);
  if constexpr (C == Columns::ADDED) {
    const int at = min(n0 + lo, n - 1);
    #pragma unroll
    for (int f = 0; f < PER; ++f)
      h[f] = add.h[(long)min(first + f * ROWS, m_here - 1) * n + at];
    weight = add.weight[at];
  } else if (!NORM && of.squares != nullptr) {
    // added up here: kept until the end they take registers, and so workgroups of
    // a CU (q4_0, one row, 8 layers of 5120: 568 us instead of 547)
    for (int r = wave; r < m_here; r += KW) {
      RowSquares<3> parts;
      parts.load(of, r);
      const float q = parts.sum(of);
      if (lane == 0) row_squares[r] = q;
    }
  }
  if constexpr (NORM) {
    rows.put(norm, m, k, reinterpret_cast<uint4*>(s_x), squares);
    lds_barrier();
  }
  int i = 0;
  if constexpr (ONE) {
    // places of the ring by number: unrolled, addresses in LDS take registers, ten
    // more than there are of two stages of q4_0
    int slot = 0;
    auto on = [&]() { slot = slot + 1 == P ? 0 : slot + 1; };
    #pragma unroll 1
    for (; i + P < steps; ++i, on()) {      // P stages in flight throughout
      wait_loads<(P - 1) * LOADS>();
      use(slot, c0 + i, integral_constant<bool, true>{});
      wait_lds_reads();
      load(slot, c0 + i + P);
    }
    #pragma unroll 1
    for (; i < steps; ++i, on()) {          // the ring runs dry
      if (P > 1 && i + P == steps) wait_loads<(P - 1) * LOADS>();
      else wait_loads<0>();
      use(slot, c0 + i, integral_constant<bool, K_QUANT && !THIN>{});
    }
  } else {
    for (; i + 2 * P <= steps; i += P) {      // P stages in flight throughout
      #pragma unroll
      for (int s = 0; s < P; ++s) {
        wait_loads<(P - 1) * LOADS>();
        use(s, c0 + i + s, integral_constant<bool, true>{});
        wait_lds_reads();
        load(s, c0 + i + s + P);
      }
    }
    for (; i < steps; i += P) {               // the ring runs dry
      #pragma unroll
      for (int s = 0; s < P; ++s)
        if (i + s < steps) {
          if (i + s + P <= steps) wait_loads<(P - 1) * LOADS>();
          else wait_loads<0>();
          use(s, c0 + i + s, integral_constant<bool, K_QUANT && !THIN>{});
          if (i + s + P < steps) {
            wait_lds_reads();
            load(s, c0 + i + s + P);
          }
        }
    }
  }
  __syncthreads();

  // the waves' shares are added up
  float* red = reinterpret_cast<float*>(s_all);
  #pragma unroll
  for (int j = 0; j < FM; ++j)
    #pragma unroll
    for (int e = 0; e < 4; ++e)
      red[(wave * BM + j * 16 + g * 4 + e) * (16 + PAD) + lo] = acc[j][e];
  __syncthreads();
  const int y_ld = C == Columns::GATED ? n / 2
      : C == Columns::HEADS ? heads.hq * heads.d : n;
  y += (long)blockIdx.y * MR * y_ld;
  if constexpr (C == Columns::HEADS) {
    heads.positions += blockIdx.y * MR;
    heads.slots += blockIdx.y * MR;
  }
  #pragma unroll
  for (int f = 0; f < PER; ++f) {
    const int r = first + f * ROWS, c = lo;
    if (r >= m_here) break;
    float scale = 1.f;
    if constexpr (NORM) scale = norm_scale<KW>(squares, r, k, norm.eps);
    else if (C != Columns::ADDED && of.squares != nullptr)
      scale = undivided_scale(of, row_squares[r], k);
    auto sum = [&](int c) {
      float v = 0.f;
      #pragma unroll
      for (int q = 0; q < KW; ++q) {
        v += red[(q * BM + r) * (16 + PAD) + c];
        if constexpr (THIN) v += red[(q * BM + r + 8) * (16 + PAD) + c + 8];
      }
      if constexpr (Q == Quant::Q4_K && !NORM)
        if (v != v) {
          const long at = weight_row<C>(n0, c, n, half);
          v = dot_q4k(x + (long)r * k, qs + at * rb, scales + at * (sb / 2), k);
        }
      return v * scale;
    };
    if constexpr (C == Columns::GATED) {
      if (c < 8)
        y[(long)r * y_ld + n0 + c] = f2bf(silu_times(sum(c), sum(c + 8)));
    } else if constexpr (C == Columns::HEADS) {
      if (c < 8) finish_heads(y, y_ld, heads, r, n0 + c, sum(c), sum(c + 8));
    } else if constexpr (C == Columns::ADDED) {
      const bool there = (!THIN || c < 8) && n0 + c < n;
      finish_added(add, y, (long)r * y_ld + n0 + c, r, there,
                   there ? bf2f(h[f]) : 0.f,
                   bf2f(weight), there ? sum(c) : 0.f);
    } else {
      if ((!THIN || c < 8) && n0 + c < n)
        y[(long)r * y_ld + n0 + c] = f2bf(sum(c));
    }
  }
}

}  // namespace

// Whether a workgroup has eight weight rows instead of 16: where some CUs would have
// two workgroups and others one, all have two or three half as large. Rows shorter
// than 4096 are read too soon for that to matter, and x, which is read once more,
// counts more from five rows on. us, MI355X, 16 -> eight, 5120 x
// 5120, 5120 x 13824, 6144 x 16384 (4096 rows and fewer, q4_0 of one: 4096 x 11008
// 9.5 -> 11.4; 5120 x 2048, 5 rows 4.9 -> 5.2):
//   q4_0  1 row    7.7 15.9 19.2 ->  7.3 14.6 17.1
//         5 rows   9.0 18.9 22.9 ->  8.7 17.1 20.7
//   q8_0  3 rows   9.9 22.2 28.4 ->  9.8 20.7 25.9
//         5 rows  10.8 23.1 28.3 -> 10.4 21.9 26.3
//   q4_K  1 row    8.3 19.9 22.2 ->  7.6 15.9 18.9
//         5 rows   9.6 23.3 25.7 ->  9.3 19.7 23.3
bool rows_quant_thin(int m, int n, int k, Quant q, bool paired) {
  return m <= 8 && !paired && n > 256 * 16 &&
         n <= (m <= 4 ? 384 : 352) * 16 && k >= 4096 &&
         q != Quant::Q6_K && (m > 1 || q != Quant::Q8_0);
}

// Blocks whose scales come in pairs (k a multiple of 64), or of 256.
bool rows_quant_takes(int m, int n, int k, Quant q, bool gated) {
  const int step = q == Quant::Q4_K || q == Quant::Q6_K ? 256 : 64;
  return m >= 1 && m <= 64 && n >= 1 && k >= step && k % step == 0 &&
         (!gated || n % 16 == 0) && (m > 1 || q != Quant::Q8_0);
}

void launch_rows_quant(bf16_t* y, const bf16_t* x, const void* scales,
                       const unsigned char* qs, int m, int n, int k, Quant q,
                       bool gated, const Heads* heads, const NormOf* norm,
                       const AddTo* add, const Undivided* of,
                       hipStream_t stream) {
  const f16_t* sc = reinterpret_cast<const f16_t*>(scales);
  auto go = [&](auto qc, auto mr, auto me, auto kw, auto p, auto t) {
    constexpr Quant QQ = decltype(qc)::value;
    constexpr int MR = decltype(mr)::value, ME = decltype(me)::value,
                  KW = decltype(kw)::value, P = decltype(p)::value;
    constexpr bool THIN = decltype(t)::value;
    constexpr int ROWS = THIN ? 8 : 16;
    const dim3 grid((n + ROWS - 1) / ROWS, (m + MR - 1) / MR),
        block(KW * WAVE);
    auto kernel = rows_quant_kernel<QQ, MR, ME, KW, P, Columns::PLAIN, false,
                                    THIN>;
    if constexpr (MR <= 8)
      if (add)
        kernel = rows_quant_kernel<QQ, MR, ME, KW, P, Columns::ADDED, false,
                                   THIN>;
    if constexpr (!THIN) {
      auto pick = [&](auto normed) {
        constexpr bool N = decltype(normed)::value;
        return heads ? rows_quant_kernel<QQ, MR, ME, KW, P, Columns::HEADS, N,
                                         false>
               : gated ? rows_quant_kernel<QQ, MR, ME, KW, P, Columns::GATED,
                                           N, false>
                       : rows_quant_kernel<QQ, MR, ME, KW, P, Columns::PLAIN,
                                           N, false>;
      };
      if (!add) kernel = pick(std::false_type{});
      if constexpr (MR == NORM_ROWS)
        if (norm) kernel = pick(std::true_type{});
    }
    kernel<<<grid, block, 0, stream>>>(y, x, sc, qs, m, n, k,
                                       heads ? *heads : Heads{},
                                       norm ? *norm : NormOf{},
                                       add ? *add : AddTo{},
                                       of ? *of : Undivided{});
  };
  auto by_rows = [&](auto qc) {
    constexpr Quant QQ = decltype(qc)::value;
    constexpr integral_constant<int, 1> c1{};
    constexpr integral_constant<int, 4> c4{};
    constexpr integral_constant<int, 8> c8{};
    constexpr integral_constant<int, 16> c16{};
    constexpr integral_constant<int, 32> c32{};
    // Stages in flight for few rows: q6_K's are the largest, q4_0's unpacking
    // pays for none. Little more than a workgroup per CU: eight waves share k
    // instead of four, since a wave's chain of stages is what takes the time.
    // us on a MI355X, 4096 x 14336, 5120 x 13824, four waves -> eight: q4_0 5
    // rows 15.5, 18.9 -> 12.1, 16.3; q4_K 5 rows 15.1, 20.0 -> 13.3, 19.4.
    // 27648 x 5120, q4_0 5 rows: two stages in flight 26.0, one 22.7; eight
    // waves 24.8. A single row has rules of its own, below.
    constexpr bool ONE = QQ == Quant::Q6_K || QQ == Quant::Q4_0;
    constexpr integral_constant<int, ONE ? 1 : 2> some{};
    constexpr integral_constant<int, QQ == Quant::Q6_K ? 1 : 2> one_row{};
    constexpr integral_constant<int, QQ == Quant::Q8_0 ? 4 : 8> waves{};
    const bool few = n <= 384 * 16;
    const bool thin = !norm && rows_quant_thin(m, n, k, QQ, gated || heads);
    constexpr std::false_type no{};
    constexpr std::true_type yes{};
    constexpr bool CAN = QQ != Quant::Q6_K;
    if (thin) {
      if constexpr (CAN) {
        // more waves, or stages in flight, of more rows: 5120 x 5120 of five, q4_0
        // 8.7 us by four waves, 13.0 by eight, 14.3 with two stages
        if constexpr (QQ != Quant::Q8_0) {
          if (m == 1) go(qc, c4, c1, c8, c1, yes);
          else if (m <= 4) go(qc, c4, c4, c4, c1, yes);
          else go(qc, c8, c4, c4, c1, yes);
        } else {
          constexpr integral_constant<int, 2> c2{};
          if (m <= 4) go(qc, c4, c4, c4, c1, yes);
          else go(qc, c8, c4, c2, c2, yes);
        }
      }
    } else if (m == 1) {
      // Eight waves of a row, two stages in flight in each, of q6_K one: all of
      // rows of 4096 at once. Four where rows are short and workgroups many. us,
      // MI355X, four -> eight, 32000 x 2048, 16384 x 3072, 28672 x 3584, 32000 x
      // 4096, 28672 x 4608:
      //   q4_0  10.8 9.2 15.3 18.4 19.1 -> 11.8 9.6 15.6 17.9 18.8
      //   q4_K  10.5 9.4 18.0 18.6 23.8 -> 14.6 10.5 17.8 20.7 22.7
      //   q6_K  14.8 13.8 26.1 29.3 33.6 -> 14.4 13.6 23.8 28.7 31.5
      // of fewer workgroups, 11264 x 2048, q4_0 5.7 -> 5.5.
      const bool four = QQ == Quant::Q4_K ? !few && k <= 4096
                                          : n > 12288 && k < 4096;
      if constexpr (QQ == Quant::Q4_K || QQ == Quant::Q4_0) {
        if (four) go(qc, c4, c1, c4, one_row, no);
        else go(qc, c4, c1, c8, one_row, no);
      } else if constexpr (QQ == Quant::Q6_K) {
        go(qc, c4, c1, c8, one_row, no);
      }
    } else if (m <= 4) {
      if (few) go(qc, c4, c4, waves, some, no);
      else go(qc, c4, c4, c4, some, no);
    } else if (m <= 8) {
      constexpr integral_constant<int, QQ == Quant::Q8_0 ? 2 : 1> one{};
      if (few) go(qc, c8, c4, waves, one, no);
      else go(qc, c8, c4, c4, some, no);
    } else if (m <= 16) {
      go(qc, c16, c4, c4, c1, no);
    } else {
      go(qc, c32, c4, c4, c1, no);
    }
  };
  switch (q) {
    case Quant::Q4_0:
      by_rows(integral_constant<Quant, Quant::Q4_0>{});
      break;
    case Quant::Q8_0:
      by_rows(integral_constant<Quant, Quant::Q8_0>{});
      break;
    case Quant::Q4_K:
      by_rows(integral_constant<Quant, Quant::Q4_K>{});
      break;
    case Quant::Q6_K:
      by_rows(integral_constant<Quant, Quant::Q6_K>{});
      break;
  }
}
