// out = a b^T + bias of bf16 matrices of many rows, with either operand as it
// is or flipped: the products of prompts, and of a training step's forward and
// backward, which need no transposed copy. Or, of a matrix b whose first half
// gates its second, silu(gate) * up: a tile has 128 columns of either then.
//
// Bound by the matrix cores if they are kept busy. A workgroup of eight waves
// takes 256 x 256 outputs, a wave 128 x 64 of them, 64 of the inner dimension
// at a time (or of fewer rows, see below: what follows is of 256). Two waves
// share a SIMD. One multiplies while the other reads its next operands from LDS
// and starts loads from memory; a barrier later they change places (without this
// turn-taking 1.10 instead of 1.33 PFLOP/s at 4096^3). For that a step of 64 is
// cut into four phases of a 64 x 32 quadrant, 16 matrix instructions each:
//
//   phase  1         2         3         4
//   reads  a low     b high    a high    b low of the next step
//   takes  low low   low high  high high high low
//
// Loads go straight to LDS, a quarter of a step per phase, into the place that
// the phase before has read, two steps ahead: 112 KB are in flight, and every
// phase waits for all but the last 12 loads of its thread. Of fewer rows a thread
// has fewer loads of a (N0, N1), and waits for all but a step's (ALL) and those of
// two regions more.
//
// LDS holds per step and half of an operand (a region of 128 rows) lines of 128
// bytes of a row, or, of a flipped operand, lines of 256 bytes of one place of
// the inner dimension, which transposing reads turn. 16-byte pieces are
// permuted within their line against bank conflicts: on the way in, by what a
// lane loads, since what is loaded directly lands in the order of lanes.
//
// A chip of 256 CUs takes 256 tiles at a time. Tiles left over from that share
// the CUs along the inner dimension and leave 32-bit sums to a second kernel. Or
// tiles have fewer rows, 128 to 224, where those of 256 would leave CUs idle or be
// partly empty (plan_of): regions of a's halves are not full then, nothing else
// changes. us, MI355X, from 256 rows: 2331 x 2048 x 2048 35.6 -> 25.8 (128), 6144 x
// 2048 x 2331, both flipped, 60.7 -> 57.4 (192), 2331 x 11264 x 2048 94 -> 88 (224), 908
// x 11264 x 2048, gated, 45 -> 39 (192), 557 x 18176 x 4544, b flipped, 114 -> 93 (192).
// Large ones are bound by power: with random numbers the chip holds 1.5 to 1.7 GHz, at
// 2140 clocks a step of which matrix instructions take 2048 (zeros: 2.4 GHz, 2.1
// PFLOP/s).
//
// TFLOP/s on a MI355X, the library -> this, m x n x k:
//   neither flipped  4165 x 12288 x 4096  1045 -> 1343   (a prompt's products)
//                    4165 x 4096 x 11008   665 -> 1369
//                    4096 x 18176 x 4544  1130 -> 1420
//                    4096 x 4096 x 4096   1411 -> 1369   8192^3 1570 -> 1534
//   b flipped        4096 x 4544 x 18176   693 -> 1325   (gradient of inputs)
//                    4096 x 4544 x 65024   652 -> 1340
//   both flipped     18176 x 4544 x 4096  1011 -> 1280   (of weights)
//                    65024 x 4544 x 4096  1091 -> 1260
// A workgroup's first loads and last stores are some 4 us; workgroups that go
// on to a next tile by themselves, with its loads under way, were no faster.
#include "tile_gemm.h"

#include <algorithm>
#include <type_traits>

#include "rows_gemm.h"

namespace {

constexpr int TILE = 256, STEP = 64;
constexpr int THREADS = 512;
constexpr int REGION = 1024;          // 16-byte pieces of 128 rows x 64
constexpr int LINES = 4;              // tile rows that an XCD takes side by side

// 32-bit raw buffers of 2 GB; what is past their end reads as zero
constexpr int RAW = 0x00020000;
constexpr unsigned PAST = 0xfffffff0u;

DEV_INLINE void barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

DEV_INLINE unsigned lds_address(const void* p) {
  return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
}

DEV_INLINE short8 join(uint2v a, uint2v b) {
  return __builtin_bit_cast(short8, (uint4v){a[0], a[1], b[0], b[1]});
}

// Transposing reads of two fragments of 16 rows x 64, or of two to four with
// addresses of their own, at `AT` bytes past these, and the wait for them. (The
// compiler's own form waits for all direct loads first.)
template <int AT>
DEV_INLINE void read_flipped2(short8 (&f)[2][2], unsigned p) {
  uint2v r[8];
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8 offset:%9\n\t"
      "ds_read_b64_tr_b16 %1, %8 offset:%10\n\t"
      "ds_read_b64_tr_b16 %2, %8 offset:%11\n\t"
      "ds_read_b64_tr_b16 %3, %8 offset:%12\n\t"
      "ds_read_b64_tr_b16 %4, %8 offset:%13\n\t"
      "ds_read_b64_tr_b16 %5, %8 offset:%14\n\t"
      "ds_read_b64_tr_b16 %6, %8 offset:%15\n\t"
      "ds_read_b64_tr_b16 %7, %8 offset:%16\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]),
        "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
      : "v"(p), "i"(AT), "i"(AT + 1024), "i"(AT + 8), "i"(AT + 1032),
        "i"(AT + 8192), "i"(AT + 9216), "i"(AT + 8200), "i"(AT + 9224)
      : "memory");
  #pragma unroll
  for (int q = 0; q < 2; ++q)
    #pragma unroll
    for (int i = 0; i < 2; ++i)
      f[i][q] = join(r[q * 4 + i * 2], r[q * 4 + i * 2 + 1]);
}

template <int AT>
DEV_INLINE void read_flipped(short8 (&f)[2][2], unsigned p0, unsigned p1) {
  uint2v r[8];
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8 offset:%10\n\t"
      "ds_read_b64_tr_b16 %1, %8 offset:%11\n\t"
      "ds_read_b64_tr_b16 %2, %9 offset:%10\n\t"
      "ds_read_b64_tr_b16 %3, %9 offset:%11\n\t"
      "ds_read_b64_tr_b16 %4, %8 offset:%12\n\t"
      "ds_read_b64_tr_b16 %5, %8 offset:%13\n\t"
      "ds_read_b64_tr_b16 %6, %9 offset:%12\n\t"
      "ds_read_b64_tr_b16 %7, %9 offset:%13\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]),
        "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
      : "v"(p0), "v"(p1), "i"(AT), "i"(AT + 1024), "i"(AT + 8192),
        "i"(AT + 9216)
      : "memory");
  #pragma unroll
  for (int q = 0; q < 2; ++q)
    #pragma unroll
    for (int i = 0; i < 2; ++i)
      f[i][q] = join(r[q * 4 + i * 2], r[q * 4 + i * 2 + 1]);
}

template <int AT>
DEV_INLINE void read_flipped(short8 (&f)[3][2], unsigned p0, unsigned p1,
                             unsigned p2) {
  uint2v r[12];
  asm volatile(
      "ds_read_b64_tr_b16 %0, %12 offset:%15\n\t"
      "ds_read_b64_tr_b16 %1, %12 offset:%16\n\t"
      "ds_read_b64_tr_b16 %2, %13 offset:%15\n\t"
      "ds_read_b64_tr_b16 %3, %13 offset:%16\n\t"
      "ds_read_b64_tr_b16 %4, %14 offset:%15\n\t"
      "ds_read_b64_tr_b16 %5, %14 offset:%16\n\t"
      "ds_read_b64_tr_b16 %6, %12 offset:%17\n\t"
      "ds_read_b64_tr_b16 %7, %12 offset:%18\n\t"
      "ds_read_b64_tr_b16 %8, %13 offset:%17\n\t"
      "ds_read_b64_tr_b16 %9, %13 offset:%18\n\t"
      "ds_read_b64_tr_b16 %10, %14 offset:%17\n\t"
      "ds_read_b64_tr_b16 %11, %14 offset:%18\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]),
        "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7]), "=&v"(r[8]), "=&v"(r[9]),
        "=&v"(r[10]), "=&v"(r[11])
      : "v"(p0), "v"(p1), "v"(p2), "i"(AT), "i"(AT + 1024), "i"(AT + 8192),
        "i"(AT + 9216)
      : "memory");
  #pragma unroll
  for (int q = 0; q < 2; ++q)
    #pragma unroll
    for (int i = 0; i < 3; ++i)
      f[i][q] = join(r[q * 6 + i * 2], r[q * 6 + i * 2 + 1]);
}

template <int AT>
DEV_INLINE void read_flipped(short8 (&f)[4][2], unsigned p0, unsigned p1,
                             unsigned p2, unsigned p3) {
  uint2v r[16];
  asm volatile(
      "ds_read_b64_tr_b16 %0, %16 offset:%20\n\t"
      "ds_read_b64_tr_b16 %1, %16 offset:%21\n\t"
      "ds_read_b64_tr_b16 %2, %17 offset:%20\n\t"
      "ds_read_b64_tr_b16 %3, %17 offset:%21\n\t"
      "ds_read_b64_tr_b16 %4, %18 offset:%20\n\t"
      "ds_read_b64_tr_b16 %5, %18 offset:%21\n\t"
      "ds_read_b64_tr_b16 %6, %19 offset:%20\n\t"
      "ds_read_b64_tr_b16 %7, %19 offset:%21\n\t"
      "ds_read_b64_tr_b16 %8, %16 offset:%22\n\t"
      "ds_read_b64_tr_b16 %9, %16 offset:%23\n\t"
      "ds_read_b64_tr_b16 %10, %17 offset:%22\n\t"
      "ds_read_b64_tr_b16 %11, %17 offset:%23\n\t"
      "ds_read_b64_tr_b16 %12, %18 offset:%22\n\t"
      "ds_read_b64_tr_b16 %13, %18 offset:%23\n\t"
      "ds_read_b64_tr_b16 %14, %19 offset:%22\n\t"
      "ds_read_b64_tr_b16 %15, %19 offset:%23\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]),
        "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7]), "=&v"(r[8]), "=&v"(r[9]),
        "=&v"(r[10]), "=&v"(r[11]), "=&v"(r[12]), "=&v"(r[13]),
        "=&v"(r[14]), "=&v"(r[15])
      : "v"(p0), "v"(p1), "v"(p2), "v"(p3), "i"(AT), "i"(AT + 1024),
        "i"(AT + 8192), "i"(AT + 9216)
      : "memory");
  #pragma unroll
  for (int q = 0; q < 2; ++q)
    #pragma unroll
    for (int i = 0; i < 4; ++i)
      f[i][q] = join(r[q * 8 + i * 2], r[q * 8 + i * 2 + 1]);
}

// Where a tile begins: LINES rows of tiles by columns. The last tiles reach
// back instead of over the matrix' end; what two of them have is the same.
template <bool GATED, int T>
DEV_INLINE void tile_of(const TileGemm& g, const TilePlan& p, int tile,
                        int& m0, int& n0) {
  const int per = LINES * p.tiles_n, first = tile / per * LINES;
  const int lines = min(p.tiles_m - first, LINES);
  m0 = min((first + tile % per % lines) * (T * 32), g.m - T * 32);
  const int wide = GATED ? TILE / 2 : TILE;
  n0 = min(tile % per / lines * wide, (GATED ? g.n / 2 : g.n) - wide);
}

// Steps come in pairs, one for each half of LDS; past the end they are zeros.
__host__ __device__ inline int pairs_of(long k) {
  return (int)((k + 2 * STEP - 1) / (2 * STEP));
}

// A piece of work: a tile, or a share of one along the inner dimension.
struct Item {
  int m0, n0, t0, t1;
  int share;                      // -1: the whole tile
};

template <bool GATED, int T>
DEV_INLINE Item item_of(const TileGemm& g, const TilePlan& p, int id) {
  const int pairs = pairs_of(g.k);
  Item it;
  it.t0 = 0;
  it.t1 = 2 * pairs;
  it.share = id - p.whole;
  int tile;
  if (it.share < 0) {
    // an XCD, which has every eighth workgroup, takes a run of tiles
    const int q = p.whole / 8, r = p.whole % 8, xcd = id % 8;
    tile = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + id / 8;
    it.share = -1;
  } else {
    const int part = it.share % p.split;
    tile = p.whole + it.share / p.split;
    it.t0 = 2 * (int)((long)pairs * part / p.split);
    it.t1 = 2 * (int)((long)pairs * (part + 1) / p.split);
    if (p.split == 1) it.share = -1;
  }
  tile_of<GATED, T>(g, p, tile, it.m0, it.n0);
  return it;
}

// Eight outputs of one row.
DEV_INLINE void store(const TileGemm& g, int width, int row, int col,
                      float4v v, float4v w) {
  *reinterpret_cast<uint4*>(g.out + (long)row * width + col) =
      make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]),
                 pack_bf16x2(w[0], w[1]), pack_bf16x2(w[2], w[3]));
}

DEV_INLINE float4v bias_of(const TileGemm& g, int col) {
  if (g.bias == nullptr) return (float4v){0.f, 0.f, 0.f, 0.f};
  const uint2 u = *reinterpret_cast<const uint2*>(g.bias + col);
  const float2 x = unpack_bf16x2(u.x), y = unpack_bf16x2(u.y);
  return (float4v){x.x, x.y, y.x, y.y};
}

// How the pieces of a region's row r are permuted.
DEV_INLINE int a_key(int r) { return r & 7; }
DEV_INLINE int b_key(int r) { return (r & 3) | (r >> 1 & 4); }

// The row and first column of a thread's eight outputs: accumulators (i, 2j)
// and (i, 2j + 1), whose fragments' rows are interleaved by fours for that.
template <int T>
DEV_INLINE int out_row(int tid, int i) {
  return ((tid >> 8) * T + i) * 16 + (tid & 15);
}
DEV_INLINE int out_col(int tid, int j) {
  return (tid >> 6 & 3) * 64 + j * 32 + (tid >> 4 & 3) * 8;
}

// The first of a thread's four columns of accumulator j.
template <bool GATED>
DEV_INLINE int col_of(const TileGemm& g, int n0, int tid, int j) {
  if constexpr (GATED)
    return n0 + (tid >> 6 & 3) * 32 + (tid >> 4 & 3) * 8 + (j & 1) * 4 +
           (j >> 1) * (g.n / 2);
  return n0 + out_col(tid, j >> 1) + (j & 1) * 4;
}

DEV_INLINE float4v gate(float4v a, float4v u) {
  float4v v;
  #pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = silu_times(a[e], u[e]);
  return v;
}

// The gelu of rounded numbers, as gelu_kernel has it: a pass over memory less. us,
// MI355X, 18176 x 4544, product and gelu -> one kernel: 700 rows 108.6 -> 105.9,
// 2000 280.5 -> 266.3, 8000 996 -> 938.
DEV_INLINE float4v gelu(float4v a) {
  float4v v;
  #pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = gelu_of(bf2f(f2bf(a[e])));
  return v;
}

// T: fragments of 16 rows that a wave has, the first half of them (one more of
// odd numbers) in the low regions.
template <bool FA, bool FB, bool GATED, bool GELU, int T>
__global__ __launch_bounds__(THREADS, 2)
void tile_gemm_kernel(TileGemm g, TilePlan plan, float4v* __restrict__ shares) {
  // [two steps][a low, a high, b low, b high]
  __shared__ alignas(1024) uint4 s[2 * 4 * REGION];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE, lo = lane & 15, gr = lane >> 4;
  const int wm = wave >> 2, wn = wave & 3;
  static_assert(!GATED || !FB);
  const Item it = item_of<GATED, T>(g, plan, blockIdx.x);
  constexpr int LOW = (T + 1) / 2, HIGH = T - LOW;
  // loads of a thread, of a region: two of 128 rows, or of a flipped operand's
  constexpr int ROWS[4] = {FA ? 4 : LOW, FA ? 4 : HIGH, 4, 4};  // of either half
  constexpr int N0 = (ROWS[0] + 1) / 2, N1 = (ROWS[1] + 1) / 2, NB = 2;
  constexpr int ALL = N0 + N1 + 2 * NB;

  // Loads: KBs of a region, 8 lines of 128 bytes each of rows, of a flipped operand
  // 4 lines of 256. Of regions of fewer rows than 128 the first ones of either half
  // are there; a wave that has none left takes its own again. off: from the low
  // region's first byte on.
  const int piece_f = lane & 15, piece_r = lane & 7;
  // a KB's place in a region of rows, in eights of them
  auto kb_of = [&](int rows, int p) {
    const int kb = rows == 4 ? wave * 2 + p : p == 0 || wave >= 4 ? wave
                                                                  : 8 + wave;
    return kb / (2 * rows) * 8 + kb % (2 * rows);
  };
  unsigned off[4][2];
  #pragma unroll
  for (int e = 0; e < 4; ++e)
    #pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int r = kb_of(ROWS[e], p) * 8 + (lane >> 3);
      const int line = (wave * 2 + p) * 4 + (lane >> 4);
      const int qa = piece_f ^ ((line & 3) << 1);
      const int qb = piece_f ^ ((line & 3) << 2);
      if (e < 2) {
        off[e][p] = FA
            ? (unsigned)(line * g.a_ld + (qa >> 3) * (T * 16) + (qa & 7) * 8) *
                  2u
            : (unsigned)(((r >> 6) * (T * 16) + (r & 63)) * g.a_ld) * 2u +
                  (piece_r ^ a_key(r)) * 16;
        if (FA && (qa & 7) >= 2 * (e == 0 ? LOW : HIGH)) off[e][p] = PAST;
      } else {
        off[e][p] = FB
            ? (unsigned)(line * g.b_ld + (qb >> 2) * 64 + (qb & 3) * 8) * 2u
            : (unsigned)((GATED ? r : (r >> 5) * 64 + (r & 31)) * g.b_ld) *
                      2u +
                  (piece_r ^ b_key(r)) * 16;
      }
    }
  const long a_step = (FA ? g.a_ld : 1) * STEP * 2;
  const long b_step = (FB ? g.b_ld : 1) * STEP * 2;
  const int a_high = (FA ? 1 : g.a_ld) * (LOW * 16) * 2;
  const int b_high = (FB ? 1 : g.b_ld) * (GATED ? g.n / 2 : 32) * 2;
  // What is loaded, two steps ahead of what is multiplied: by buffer loads,
  // whose only vector operand is the offset.
  int lt = it.t0;
  const char* la = reinterpret_cast<const char*>(
      g.a + it.m0 * (FA ? 1 : g.a_ld)) + lt * a_step;
  const char* lb = reinterpret_cast<const char*>(
      g.b + it.n0 * (FB ? 1 : g.b_ld)) + lt * b_step;
  // WHOLE: the step is known to be one of the inner dimension's whole ones
  auto load = [&](auto whole, int buf, int region) {
    const auto from = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(region < 2 ? la : lb), 0, 0x80000000u, RAW);
    const int high = region & 1 ? (region < 2 ? a_high : b_high) : 0;
    constexpr int LOADS[4] = {N0, N1, NB, NB};
    uint4* to = s + (buf * 4 + region) * REGION;
    const bool flipped = region < 2 ? FA : FB;
    #pragma unroll
    for (int p = 0; p < LOADS[region]; ++p) {
      unsigned o = off[region][p];
      const int kb = flipped ? wave * 2 + p : kb_of(ROWS[region], p);
      if constexpr (!decltype(whole)::value) {
        const int r = kb * 8 + (lane >> 3);
        const int at = flipped
            ? kb * 4 + (lane >> 4)
            : (piece_r ^ (region < 2 ? a_key(r) : b_key(r))) * 8;
        if (at >= g.k - lt * STEP) o = PAST;
      }
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          from,
          (__attribute__((address_space(3))) unsigned int*)(to + kb * 64),
          16, o, high, 0, 0);
    }
  };
  auto advance = [&]() {
    ++lt;
    la += a_step;
    lb += b_step;
  };

  float4v acc[T][4];
  short8 al[LOW][2], ah[HIGH][2], bl[2][2][2], bh[2][2];

  // flipped: a lane's place in a transposing read of the first fragment
  const int place16 = ((gr * 8 + (lo >> 2)) * 16) * 16;
  const unsigned base = lds_address(s);
  const unsigned at_a = base + place16 + (lo & 1) * 8 +
      (((wm * 8 + ((lo & 3) >> 1)) ^ ((lo >> 2) << 1)) * 16);
  const unsigned at_b = base + place16 +
      (((wn * 4 + (lo & 3)) ^ ((lo >> 2) << 2)) * 16);
  auto read_a = [&](auto buf, auto half, auto& f) {
    constexpr int BUF = decltype(buf)::value, H = decltype(half)::value;
    constexpr int COUNT = sizeof(f) / sizeof(f[0]);
    if constexpr (FA) {
      const unsigned p = at_a + BUF * 4 * REGION * 16;
      if constexpr (COUNT == 4)
        read_flipped<H * REGION * 16>(f, p, p ^ 32, p ^ 64, p ^ 96);
      else if constexpr (COUNT == 3)
        read_flipped<H * REGION * 16>(f, p, p ^ 32, p ^ 64);
      else
        read_flipped<H * REGION * 16>(f, p, p ^ 32);
    } else {
      const uint4* r = s + (BUF * 4 + H) * REGION + (wm * 64 + lo) * 8;
      #pragma unroll
      for (int i = 0; i < COUNT; ++i)
        #pragma unroll
        for (int q = 0; q < 2; ++q)
          f[i][q] = *reinterpret_cast<const short8*>(
              r + i * 128 + ((q * 4 + gr) ^ (lo & 7)));
    }
  };
  auto read_b = [&](auto buf, auto half, short8 (&f)[2][2]) {
    constexpr int BUF = decltype(buf)::value, H = decltype(half)::value;
    if constexpr (FB) {
      const unsigned p = at_b + BUF * 4 * REGION * 16;
      read_flipped2<(2 + H) * REGION * 16>(f, p);
    } else {
      const uint4* r = s + (BUF * 4 + 2 + H) * REGION +
                       (wn * 32 + (lo >> 2) * 8 + (lo & 3)) * 8;
      #pragma unroll
      for (int i = 0; i < 2; ++i)
        #pragma unroll
        for (int q = 0; q < 2; ++q)
          f[i][q] = *reinterpret_cast<const short8*>(
              r + i * 32 + ((q * 4 + gr) ^ (lo & 7)));
    }
  };
  // the phase's reads are done, and so are the loads of the next one's, behind
  // which no more than N were issued
  auto turn = [&](auto n) {
    wait_lds_reads();
    wait_loads<decltype(n)::value>();
    barrier();
  };
  auto take = [&](int i0, int j0, const auto& fa, const short8 (&f)[2][2]) {
    #pragma unroll
    for (int q = 0; q < 2; ++q)
      #pragma unroll
      for (int i = 0; i < (int)(sizeof(fa) / sizeof(fa[0])); ++i)
        #pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i0 + i][j0 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              f[j][q], fa[i][q], acc[i0 + i][j0 + j], 0, 0, 0);
    barrier();
  };
  using std::integral_constant;
  constexpr integral_constant<int, 0> low{};
  constexpr integral_constant<int, 1> high{};
  auto step = [&](auto buf, auto whole) {
    constexpr int B = decltype(buf)::value;
    constexpr integral_constant<int, B ^ 1> other{};
    read_a(buf, low, al);
    load(whole, B, 2);
    turn(integral_constant<int, ALL + N1 + NB>{});
    take(0, 0, al, bl[B]);
    read_b(buf, high, bh);
    load(whole, B, 0);
    turn(integral_constant<int, ALL + NB + N0>{});
    take(0, 2, al, bh);
    read_a(buf, high, ah);
    load(whole, B, 3);
    turn(integral_constant<int, ALL + N0 + NB>{});
    take(LOW, 2, ah, bh);
    read_b(other, low, bl[B ^ 1]);
    load(whole, B, 1);
    advance();
    turn(integral_constant<int, ALL + NB + N1>{});
    take(LOW, 0, ah, bl[B]);
  };
  constexpr std::true_type whole{};
  constexpr std::false_type any{};

  #pragma unroll
  for (int t = 0; t < 2; ++t) {
    load(any, t, 2);
    load(any, t, 0);
    load(any, t, 3);
    load(any, t, 1);
    advance();
  }
  #pragma unroll
  for (int i = 0; i < T; ++i)
    #pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (float4v){0.f, 0.f, 0.f, 0.f};
  wait_loads<ALL + NB + N1>();
  barrier();
  read_b(low, low, bl[0]);
  wait_lds_reads();
  barrier();
  if (wm == 1) barrier();         // half of the waves run half a phase behind
  const int pairs = (it.t1 - it.t0) / 2;
  // pairs whose loads, a pair ahead, are all of whole steps
  const int hot = min(pairs - 1, (g.k / STEP - it.t0) / 2 - 1);
  int t = 0;
  #pragma unroll 1
  for (; t < hot; ++t) {
    step(low, whole);
    step(high, whole);
  }
  #pragma unroll 1
  for (; t < pairs; ++t) {        // loads past the end are zeros
    step(low, any);
    step(high, any);
  }
  if (wm == 0) barrier();
  wait_loads<0>();                // no load outlives its workgroup's LDS

  const int tid = threadIdx.x;
  if (it.share >= 0) {
    float4v* to = shares + (long)it.share * (4 * T * THREADS) + tid;
    #pragma unroll
    for (int i = 0; i < T; ++i)
      #pragma unroll
      for (int j = 0; j < 4; ++j) to[(i * 4 + j) * THREADS] = acc[i][j];
    return;
  }
  const int n = GATED ? g.n / 2 : g.n;
  float4v add[4];
  #pragma unroll
  for (int j = 0; j < 4; ++j)
    add[j] = bias_of(g, col_of<GATED>(g, it.n0, tid, j));
  #pragma unroll
  for (int i = 0; i < T; ++i) {
    const int row = it.m0 + out_row<T>(tid, i);
    #pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] += add[j];
    if constexpr (GELU) {
      #pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = gelu(acc[i][j]);
    }
    if constexpr (GATED) {
      store(g, n, row, col_of<true>(g, it.n0, tid, 0),
            gate(acc[i][0], acc[i][2]), gate(acc[i][1], acc[i][3]));
    } else {
      #pragma unroll
      for (int j = 0; j < 2; ++j)
        store(g, n, row, it.n0 + out_col(tid, j), acc[i][2 * j],
              acc[i][2 * j + 1]);
    }
  }
}

// The shares of the tiles left over are added up, 32 rows of a tile per workgroup.
template <bool GATED, bool GELU, int T>
__global__ __launch_bounds__(THREADS)
void tile_sum_kernel(TileGemm g, TilePlan plan,
                     const float4v* __restrict__ shares) {
  int m0, n0;
  tile_of<GATED, T>(g, plan, plan.whole + blockIdx.x, m0, n0);
  const int tid = threadIdx.x, i = blockIdx.y;
  const float4v* from = shares +
      (long)blockIdx.x * plan.split * (4 * T * THREADS) + i * 4 * THREADS +
      tid;
  float4v v[4];
  #pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = from[j * THREADS];
  #pragma unroll 4
  for (int p = 1; p < plan.split; ++p)
    #pragma unroll
    for (int j = 0; j < 4; ++j)
      v[j] += from[(long)p * 4 * T * THREADS + j * THREADS];
  #pragma unroll
  for (int j = 0; j < 4; ++j) v[j] += bias_of(g, col_of<GATED>(g, n0, tid, j));
  if constexpr (GELU) {
    #pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = gelu(v[j]);
  }
  const int row = m0 + out_row<T>(tid, i);
  if constexpr (GATED) {
    store(g, g.n / 2, row, col_of<true>(g, n0, tid, 0), gate(v[0], v[2]),
          gate(v[1], v[3]));
  } else {
    #pragma unroll
    for (int j = 0; j < 2; ++j)
      store(g, g.n, row, n0 + out_col(tid, j), v[2 * j], v[2 * j + 1]);
  }
}

}  // namespace

// A tile's offsets within an operand fit 32 bits, 16-byte pieces of it lie
// within a row.
bool tile_gemm_takes(long m, long n, long k, long a_ld, long b_ld,
                     bool a_flipped, bool b_flipped, bool gated) {
  if (gated && (a_flipped || b_flipped || n % 16 != 0 ||
                (n / 2 + TILE) * b_ld * 2 >= (1L << 31)))
    return false;
  auto fits = [&](long rows, long ld, bool flipped) {
    return ld % 8 == 0 && (flipped ? rows % 8 == 0 && ld >= rows
                                   : k % 8 == 0 && ld >= k) &&
           ld < (1L << 21);
  };
  return m >= TILE && n >= TILE && k > STEP && n % 8 == 0 &&
         m < (1L << 30) && n < (1L << 30) && k < (1L << 30) &&
         fits(m, a_ld, a_flipped) && fits(n, b_ld, b_flipped);
}

// us on a MI355X, by a fit of 2055 products of 260 to 6000 rows with matrices of 2048
// to 28672 rows and columns, tiles of 128 to 256 rows, a pass over memory before each
// (rms 8 %): a step of a tile where all CUs have one, and where few do (the chip holds
// a higher clock then); what a round, all rounds and the sum of shares begin and end
// with; a tile's share's way through memory. Of the five heights the plan's is 0.6 %
// slower than the best, 256 rows by themselves 5 %. A step of fewer rows reads LDS, and
// turns a flipped operand, for longer than it multiplies. Bytes are not counted, which
// bound products of few rows: 256 x 22016 x 4096, gated, is planned at 58 us and takes
// 67.7 (the library and its gate 78.3).
static TilePlan plan_of(long m, long n, long k, int rows, bool a_flipped,
                        bool b_flipped) {
  TilePlan p;
  p.rows = rows;
  p.tiles_m = (int)((m + rows - 1) / rows);
  p.tiles_n = (int)((n + TILE - 1) / TILE);
  const long tiles = (long)p.tiles_m * p.tiles_n;
  const long steps = 2 * pairs_of(k);
  const long rest = tiles % 256, rounds = tiles / 256;
  constexpr double STEP_US[3][5] = {{0.843, 0.958, 1.083, 1.188, 1.301},
                                    {1.035, 1.161, 1.265, 1.343, 1.398},
                                    {1.028, 1.162, 1.314, 1.443, 1.540}};
  const double step =
      STEP_US[a_flipped ? 2 : b_flipped ? 1 : 0][rows / 32 - 4];
  auto busy = [&](long tiles) { return 0.78 + 0.22 * tiles / 256.; };
  const double full = 2.4 + rounds * (steps * step + 5.5);
  p.whole = (int)tiles;
  p.split = 1;
  p.us = full + (rest ? steps * step * busy(rest) + 5.5 : 0.);
  for (int s = 2; rest && rest * s <= 256 && steps / s >= 4; ++s) {
    const double us = full + (steps + s - 1) / s * step * busy(rest * s) + 5.5 +
                      rest * s * rows * (0.0127 / 32);
    if (us < p.us) {
      p.us = us;
      p.whole = (int)(tiles - rest);
      p.split = s;
    }
  }
  return p;
}

// Fewer rows turn a flipped operand once more for the same result, and such tiles take
// longer than planned where no CU was idle before, or where shares keep all busy. By
// what 256 rows take over what fewer do, MI355X, 2647 products of 256 to 8192 rows:
//   both flipped   128 rows instead of shares of 256  12 of 0.84 to 1.03 (2048 x 4096 x
//                  5000 84.6 and 100.6 us), of more shares 0.89 to 1.05; several rounds
//                  0.93 to 1.12 (5120 x 5120 x 6000 264 and 284); a single round
//                  instead of one with fewer tiles 1.22 (128), 1.05 (192): only that
//   b flipped      128 rows instead of shares 0.92, 0.96, 1.09; two shares of 160 rows
//                  9 of 0.88 to 0.95, of 192 28 of 0.85 to 1.06: neither; three and
//                  more 1.15 and 1.11, of 224 rows 1.04
//   neither        1.03 to 1.2 in every group
TilePlan tile_gemm_plan(long m, long n, long k, bool a_flipped,
                        bool b_flipped) {
  const TilePlan high = plan_of(m, n, k, TILE, a_flipped, b_flipped);
  TilePlan best = high;
  for (int rows = 128; rows < TILE; rows += 32) {
    const TilePlan p = plan_of(m, n, k, rows, a_flipped, b_flipped);
    if (a_flipped ? high.split > 1 || p.tiles_m * (long)p.tiles_n > 256
                  : b_flipped && ((rows == 128 && high.split > 1) ||
                                  (rows < 224 && p.split == 2)))
      continue;
    if (p.us < (best.rows == TILE ? 0.97 : 1.) * best.us) best = p;
  }
  return best;
}

// Whether the library's product would take longer. What that takes is no smooth
// function of sizes: it has products that it is tuned for, whose neighbours take up to
// twice as long. So this goes by planned PFLOP/s, and where the lines lie by what all
// products beyond them gain together. The library's time over this one's, MI355X, 4060
// products of models of 768 to 8192 columns by 256 to 8192 rows, operands from memory:
//   neither flipped   in three and more shares from 0.95 on 138 of 0.95 to 2.24, 1.22
//                     on average; others from 1.0 on 556 of 0.89 to 2.17, 1.07 (from
//                     0.9 on 43 more, 1.02; 3330 x 2048 x 5632, of those, lost in a
//                     model, 0.91). Tiles of 256 rows in whole rounds stay, 51 of 0.93
//                     to 1.05; two shares of 8192 columns whose inner size it is tuned
//                     for, 15 of 0.81 to 1.06 (10 of other widths and such inner sizes
//                     1.13); and tiles of fewer rows where 256 would leave a quarter
//                     of the CUs idle and plan less than 1.0, 52 of 0.92 to 1.23, 1.03
//                     together (2048 x 4096 x 4096 1.05; 60 that plan more go, 1.04)
//   b flipped         in three and more shares from 0.7 on 350 of 0.93 to 3.15, 1.50;
//                     others from 0.85 on 359 of 0.87 to 1.86, 1.14. Two shares of 8192
//                     columns and up to 1023 rows stay, 24 of 0.78 to 1.05, others of
//                     a multiple of that below 1.15, 7 of 0.87 to 1.02, and where
//                     tiles of 256 rows would take up to three quarters of their
//                     rounds' CUs, 132 of 0.81 to 1.53, 0.98 on average
//   both flipped      from 0.5 on 502 of 0.84 to 1.57, 1.18; of rows by 32 from 0.55
//                     on 572 of 0.75 to 1.65, 1.10 (below that 2048 x 2048 x 3072
//                     0.86); not where a quarter and more of the steps' places is
//                     empty and the library has no such places (288 tokens: 29 of 0.71
//                     to 1.30, 0.94)
//   gated             from 0.5 on 140 of 1.00 to 1.63 over the product and the pass
//                     that gates it, 1.16
// Lines 128 bytes longer change the two shares of 8192 columns by up to 5 %, the
// library's as well: not where the operands lie is what keeps them there.
bool tile_gemm_pays(long m, long n, long k, bool a_flipped, bool b_flipped,
                    bool gated) {
  const TilePlan p = tile_gemm_plan(m, n, k, a_flipped, b_flipped);
  const double rate = 2e-9 * m * n * k / p.us;        // PFLOP/s
  if (gated) return rate >= 0.5;
  if (a_flipped) {
    const long empty = 2 * pairs_of(k) * STEP - k;
    return k % 32 == 0 ? rate >= 0.55 && 4 * empty < k : rate >= 0.5;
  }
  const TilePlan whole = plan_of(m, n, k, TILE, false, b_flipped);
  const long high = whole.tiles_m * (long)whole.tiles_n;
  const bool idle = 4 * high <= 3 * ((high + 255) / 256 * 256);
  const bool halves = p.whole == 0 && p.split == 2 && n % 8192 == 0;
  if (b_flipped)
    return rate >= (p.split > 2 ? 0.7 : n % 8192 == 0 && m < 1024 ? 1.15 : 0.85) &&
           !(whole.split == 1 && idle) && !(halves && m < 1024);
  if (p.split > 2) return rate >= 0.95;
  const bool even = m % TILE == 0 && n % TILE == 0 && high % 256 == 0;
  const bool fewer = p.split == 1 && (whole.split == 1 || whole.whole == 0);
  return rate >= 1. && !even && !(halves && k % 4096 == 0) &&
         !(fewer && idle && 2e-9 * m * n * k / whole.us < 1.);
}

void launch_tile_gemm(const TileGemm& g, const TilePlan& plan, float* shares,
                      hipStream_t stream) {
  float4v* sh = reinterpret_cast<float4v*>(shares);
  const dim3 grid(plan.whole + plan.rest() * plan.split);
  auto go = [&](auto t) {
    constexpr int T = decltype(t)::value;
    auto kernel = g.gated ? tile_gemm_kernel<false, false, true, false, T>
        : g.gelu ? tile_gemm_kernel<false, false, false, true, T>
        : g.a_flipped
            ? (g.b_flipped ? tile_gemm_kernel<true, true, false, false, T>
                           : tile_gemm_kernel<true, false, false, false, T>)
            : (g.b_flipped ? tile_gemm_kernel<false, true, false, false, T>
                           : tile_gemm_kernel<false, false, false, false, T>);
    kernel<<<grid, dim3(THREADS), 0, stream>>>(g, plan, sh);
    if (plan.split > 1) {
      auto sum = g.gated ? tile_sum_kernel<true, false, T>
                 : g.gelu ? tile_sum_kernel<false, true, T>
                          : tile_sum_kernel<false, false, T>;
      sum<<<dim3(plan.rest(), T), dim3(THREADS), 0, stream>>>(g, plan, sh);
    }
  };
  switch (plan.rows / 32) {
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 5: go(std::integral_constant<int, 5>{}); break;
    case 6: go(std::integral_constant<int, 6>{}); break;
    case 7: go(std::integral_constant<int, 7>{}); break;
    default: go(std::integral_constant<int, 8>{});
  }
}
