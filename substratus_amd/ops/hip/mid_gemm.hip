// y = x w^T + bias of 17 to 256 rows with a bf16 weight matrix [n, k], as decode
// steps of larger batches and short prompts need it; or silu(gate) * up of a
// matrix whose first half gates its second; or, of a projection of heads, rotated
// queries, with keys and values appended to the cache (rows_gemm.h).
//
// Bound by reading the weights once and the rows of x once per workgroup: tiles
// are about as wide as they are high, so that either is half of it, and as many
// workgroups as CUs share the inner dimension, whose 32-bit sums a second kernel
// adds up. Stages of 64 columns go straight to LDS, 96 to 128 KB in flight per CU
// (of one workgroup that has most of LDS, or of two). A load takes 8 rows x 128
// bytes: with 16 rows x 64 bytes every cache line came twice, 128 x 4544 x 18176
// in 64 us instead of 51. Four waves that shared the inner dimension instead,
// without barriers, were no faster at either; nor are more stages in flight,
// operands read half a stage ahead, or 256 columns a workgroup.
//
// us on a MI355X, from the library's product to this one:
//   rows     n x k: 4096 x 4096    4096 x 11008   4544 x 18176   8192 x 8192
//   17              13.1 -> 11.8    30.6 -> 21.3   117 -> 35.3   30.2 -> 29.9
//   64              14.9 -> 13.3    34.2 -> 25.6   155 -> 40.9   33.2 -> 32.1
//   128             24.3 -> 19.2    59.9 -> 31.1   150 -> 46.8   48.0 -> 39.0
//   192             32.6 -> 21.4    81.1 -> 39.0   124 -> 70.9   64.8 -> 54.1
//   256             22.4 -> 23.8    49.6 -> 43.8   142 -> 77.5   78.0 -> 60.2
#include "mid_gemm.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int WAVES = 4;
constexpr int STEP = 64;          // columns of a stage
constexpr int TILE = 128;         // 16-byte pieces of 16 rows x 64 columns

DEV_INLINE void barrier() {
  wait_lds_reads();
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Weight tile t's first column, and how much later its second eight are.
template <Columns C>
DEV_INLINE int column_of(int t, const Heads& heads) {
  if constexpr (!paired(C)) return t * 16;
  const int at = t * 8;
  if constexpr (C == Columns::HEADS) {
    const int half = heads.d / 2;
    return at + at / half * half;
  }
  return at;
}

// Four columns c to c + 3 of tile t, row r, and, unless they are stored as they
// are, the four that go with them, eight later in the tile.
template <Columns C>
DEV_INLINE void finish(const MidGemm& a, const Heads& heads, int r, int t, int c,
                       float4v u, float4v v) {
  const int n0 = column_of<C>(t, heads), half = C == Columns::HEADS
      ? heads.d / 2 : a.n / 2;
  if constexpr (!paired(C)) {
    const int col = n0 + c;
    if (col >= a.n) return;
    if (a.bias != nullptr) {
      #pragma unroll
      for (int e = 0; e < 4; ++e) u[e] += bf2f(a.bias[min(col + e, a.n - 1)]);
    }
    if constexpr (C == Columns::GELU) {
      #pragma unroll
      for (int e = 0; e < 4; ++e) u[e] = gelu_of(bf2f(f2bf(u[e])));
    }
    bf16_t* to = a.y + r * a.y_ld + col;
    if (a.quads) {
      *reinterpret_cast<uint2*>(to) =
          make_uint2(pack_bf16x2(u[0], u[1]), pack_bf16x2(u[2], u[3]));
      return;
    }
    #pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col + e < a.n) to[e] = f2bf(u[e]);
    return;
  }
  if (a.bias != nullptr) {
    #pragma unroll
    for (int e = 0; e < 4; ++e) {
      u[e] += bf2f(a.bias[n0 + c + e]);
      v[e] += bf2f(a.bias[n0 + c + e + half]);
    }
  }
  #pragma unroll
  for (int e = 0; e < 4; ++e) {
    if constexpr (C == Columns::GATED)
      a.y[r * a.y_ld + n0 + c + e] = f2bf(silu_times(u[e], v[e]));
    else
      finish_heads(a.y, a.y_ld, heads, r, n0 + c + e, u[e], v[e]);
  }
}

// F: tiles of 16 rows of x, N: of weights; P stages of 64 columns of both in LDS.
// SPREAD: workgroups begin at different places of their shares
template <Columns C, int F, int N, int P, bool SPREAD>
__global__ __launch_bounds__(WAVES * WAVE, (N + F) * 2 * P <= 80 ? 2 : 1)
void mid_gemm_kernel(MidGemm a, Heads heads, float* __restrict__ part) {
  constexpr int STAGE = (N + F) * TILE;
  constexpr int LOADS = (N + F) * 2 / WAVES;     // a wave's, of a stage
  static_assert((N + F) % 2 == 0);
  // waves share rows of x, too, where there are enough
  constexpr int WM = F >= 4 ? 2 : 1;
  constexpr int WN = WAVES / WM, FW = F / WM, NW = N / WN;
  static_assert(FW * WM == F && NW * WN == N);
  __shared__ alignas(16) uint4 s_all[P * STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE, lo = lane & 15, g = lane >> 4;
  const int wm = wave % WM, wn = wave / WM;
  // blocks of rows of the same columns go to the same XCD, which has every
  // eighth workgroup
  const int cols = gridDim.x / a.blocks;
  const int q = blockIdx.x / (8 * a.blocks), rest = min(cols - q * 8, 8);
  const int in = blockIdx.x - q * 8 * a.blocks;
  const int ct = q * 8 + in % rest, r0 = in / rest * F * 16;
  const int last = (a.n + 15) / 16 - 1;
  const int all = (a.k + STEP - 1) / STEP;
  const int i0 = (int)((long)all * blockIdx.y / gridDim.y);
  const int steps = (int)((long)all * (blockIdx.y + 1) / gridDim.y) - i0;
  // Those of an XCD stay close to each other, so that rows of x come to its cache
  // once (128 x 8192 x 28672 110 us, spread over the whole share 137).
  const int first = SPREAD && steps > 0
      ? (ct % 8 * 4 + ct / 8 * (a.m > 64 ? 1 : 3)) % steps : 0;
  auto in_share = [&](int i) {
    return SPREAD && i + first >= steps ? i + first - steps : i + first;
  };
  // A load is 8 rows x 128 bytes, whole cache lines (64 of 16 rows each: lines
  // came twice, 35 % slower). A row's pieces are permuted by the row against
  // bank conflicts.
  const char* from[LOADS];
  int piece[LOADS];
  #pragma unroll
  for (int l = 0; l < LOADS; ++l) {
    const int id = wave * LOADS + l, t = id / 2;
    const int row = id % 2 * 8 + lane / 8;
    const int n0 = column_of<C>(min(ct * N + min(t, N - 1), last), heads);
    const int half = C == Columns::HEADS ? heads.d / 2 : a.n / 2;
    const bf16_t* p = t < N
        ? a.w + (long)weight_row<C>(n0, row, a.n, half) * a.k
        : a.x + min(r0 + (t - N) * 16 + row, a.m - 1) * a.x_ld;
    piece[l] = (lane % 8) ^ (row >> 1 & 7);
    from[l] = reinterpret_cast<const char*>(p + (long)i0 * STEP);
  }
  const int over = a.k / 8 - i0 * 8 - 1;         // a row's last piece from here
  auto load = [&](int i) {
    uint4* to = s_all + i % P * STAGE + wave * LOADS * 64;
    const int at = in_share(i) * 8;
    #pragma unroll
    for (int l = 0; l < LOADS; ++l)
      load_to_lds<16>(from[l] + min(at + piece[l], over) * 16, to + l * 64);
  };
  float4v acc[NW][FW];
  #pragma unroll
  for (int j = 0; j < NW; ++j)
    #pragma unroll
    for (int f = 0; f < FW; ++f) acc[j][f] = (float4v){0.f, 0.f, 0.f, 0.f};
  auto use = [&](int i) {
    const uint4* s = s_all + i % P * STAGE + lo * 8;
    const bool half = (i0 + in_share(i)) * STEP + STEP > a.k;
    #pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int at = (c * 4 + g) ^ (lo >> 1);
      short8 wf[NW], xf[FW];
      #pragma unroll
      for (int j = 0; j < NW; ++j)
        wf[j] = *reinterpret_cast<const short8*>(s + (wn * NW + j) * TILE + at);
      #pragma unroll
      for (int f = 0; f < FW; ++f)
        xf[f] = *reinterpret_cast<const short8*>(
            s + (N + wm * FW + f) * TILE + at);
      if (c == 1 && half) break;
      #pragma unroll
      for (int j = 0; j < NW; ++j)
        #pragma unroll
        for (int f = 0; f < FW; ++f)
          acc[j][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              wf[j], xf[f], acc[j][f], 0, 0, 0);
    }
  };
  #pragma unroll
  for (int i = 0; i < P - 1; ++i)
    if (i < steps) load(i);
  int i = 0;
  for (; i + P - 1 < steps; ++i) {
    wait_loads<(P - 2) * LOADS>();  // this step's, of all waves; and all have
    barrier();                      // read what the next load takes the place of
    load(i + P - 1);
    use(i);
  }
  for (; i < steps; ++i) {
    wait_loads<0>();
    barrier();
    use(i);
  }

  #pragma unroll
  for (int f = 0; f < FW; ++f) {
    const int r = r0 + (wm * FW + f) * 16 + lo;
    #pragma unroll
    for (int j = 0; j < NW; ++j) {
      const int t = ct * N + wn * NW + j;
      const bool there = r < a.m && t <= last;
      if (gridDim.y > 1) {
        if (there)
          *reinterpret_cast<float4v*>(
              part + ((long)blockIdx.y * a.m + r) * (last + 1) * 16 + t * 16 +
              g * 4) = acc[j][f];
        continue;
      }
      float4v other = {0.f, 0.f, 0.f, 0.f};
      if constexpr (paired(C))
        #pragma unroll
        for (int e = 0; e < 4; ++e)
          other[e] = __shfl_xor(acc[j][f][e], 32, WAVE);
      if (there && (!paired(C) || g < 2))
        finish<C>(a, heads, r, t, g * 4, acc[j][f], other);
    }
  }
}

// Workgroups' shares of the inner dimension, added up.
template <Columns C>
__global__ __launch_bounds__(256)
void mid_sum_kernel(MidGemm a, Heads heads, const float* __restrict__ part,
                    int splits) {
  constexpr int PER = paired(C) ? 2 : 4;
  const int tiles = (a.n + 15) / 16;
  const long id = (long)blockIdx.x * 256 + threadIdx.x;
  const int r = id / (tiles * PER), e = id % (tiles * PER);
  if (r >= a.m) return;
  const int t = e / PER, c = e % PER * 4;
  const long step = (long)a.m * tiles * 16;
  const float* p = part + (long)r * tiles * 16 + t * 16 + c;
  float4v u = {0.f, 0.f, 0.f, 0.f}, v = u;
  #pragma unroll 4
  for (int s = 0; s < splits; ++s) {
    u += *reinterpret_cast<const float4v*>(p + s * step);
    if constexpr (paired(C))
      v += *reinterpret_cast<const float4v*>(p + s * step + 8);
  }
  finish<C>(a, heads, r, t, c, u, v);
}

// The same, of a whole row to a workgroup, which adds them to the residual stream
// and makes the norm that follows of it: bound by a launch and its first loads, and
// a norm of its own has both again, besides the row's way through memory. The row
// is rounded as the product and the norm round it.
template <int BLOCK, int QUADS>
__global__ __launch_bounds__(BLOCK)
void mid_norm_kernel(MidGemm a, MidNorm norm, const float* __restrict__ part,
                     int splits) {
  __shared__ float scratch[BLOCK / WAVE];
  const int r = blockIdx.x, wide = (a.n + 15) / 16 * 16;
  const long step = (long)a.m * wide, row = (long)r * a.n;
  float4v keep[QUADS], w[QUADS];
  float squares = 0.f;
  auto quad = [](const bf16_t* p) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    const float2 x = unpack_bf16x2(u.x), y = unpack_bf16x2(u.y);
    return (float4v){x.x, x.y, y.x, y.y};
  };
  #pragma unroll
  for (int q = 0; q < QUADS; ++q) {
    const int c = (q * BLOCK + threadIdx.x) * 4;
    if (c >= a.n) break;
    const float4v h = quad(norm.h + row + c);
    w[q] = quad(norm.weight + c);
    const float* p = part + (long)r * wide + c;
    float4v u = {0.f, 0.f, 0.f, 0.f};
    #pragma unroll 4
    for (int s = 0; s < splits; ++s)
      u += *reinterpret_cast<const float4v*>(p + s * step);
    if (a.bias != nullptr) u += quad(a.bias + c);
    #pragma unroll
    for (int e = 0; e < 4; ++e) {
      u[e] = h[e] + bf2f(f2bf(u[e]));
      squares += u[e] * u[e];
    }
    const uint2 to = make_uint2(pack_bf16x2(u[0], u[1]),
                                pack_bf16x2(u[2], u[3]));
    *reinterpret_cast<uint2*>(norm.total + row + c) = to;
    const float2 x = unpack_bf16x2(to.x), y = unpack_bf16x2(to.y);
    keep[q] = (float4v){x.x, x.y, y.x, y.y};
  }
  const float inv = rsqrtf(
      block_sum<BLOCK / WAVE>(squares, scratch) / (float)a.n + norm.eps);
  #pragma unroll
  for (int q = 0; q < QUADS; ++q) {
    const int c = (q * BLOCK + threadIdx.x) * 4;
    if (c >= a.n) break;
    const float4v v = keep[q];
    *reinterpret_cast<uint2*>(a.y + row + c) = make_uint2(
        pack_bf16x2(v[0] * inv * w[q][0], v[1] * inv * w[q][1]),
        pack_bf16x2(v[2] * inv * w[q][2], v[3] * inv * w[q][3]));
  }
}

}  // namespace

bool mid_gemm_takes(long m, long n, long k, bool paired) {
  return m >= 1 && m <= 256 && n >= 16 && k >= STEP && k % 32 == 0 &&
         n < (1L << 24) && k < (1L << 24) && (!paired || n % 16 == 0);
}

// The tiles and shares that take least: some 5 us of launch and first loads, the
// weights at 5.3 TB/s, a stage of a CU at 38 GB/s, and the sums' kernel and way
// through memory. Within a seventh of what 900 products were measured to take.
MidPlan mid_gemm_plan(long m, long n, long k) {
  MidPlan best{};
  best.us = 1e30;
  const long steps = (k + STEP - 1) / STEP;
  const long blocks = (m + 127) / 128, per = (m + blocks - 1) / blocks;
  const int rows = per <= 32 ? 32 : per <= 64 ? 64 : per <= 96 ? 96 : 128;
  const double weights = n * k * 2 / 5.3e6;
  for (int tiles = 4; tiles <= 8; tiles += 4) {
    const long groups = (n + tiles * 16 - 1) / (tiles * 16) * blocks;
    for (int s = 1; s <= 16 && s <= steps; ++s) {
      const long rounds = (groups * s + 255) / 256;
      const double load = rounds * ((steps + s - 1) / s) *
                          ((tiles + rows / 16) * 2.048 / 38.);
      const double sum = s > 1 ? 3. + s * m * n * 8 / 7e6 : 0.;
      const double us = 4.5 + std::max(weights, load) + sum;
      if (us < best.us) best = {rows, tiles, s, us};
    }
  }
  return best;
}

// Whether the library's product would take longer, by an estimate fitted to what
// it took: a launch, the weights at 10 TB/s, the products at 2 PFLOP/s, and what a
// tile takes along the inner dimension, which is shared where there are few columns
// and by rows up to 128; nearly half as much again where rows of the weights do not
// begin on lines of 512 bytes. A paired product saves a launch and a pass. Where
// matrices are wide and rows many the library has tiles for the chip, and sums of
// few numbers cannot be shared. Long sums of more than 32 rows take it a fifth
// longer at least, but for 256, which are whole tiles. Of rows of a multiple of 4 KB
// it takes a fifth longer in paired products, as its CUs all read the same of the
// memory's channels (64 x 28672 x 4096 54.4 us, and 45.9 here; 32 x 22016 x 4096 46.1,
// and 37.0; 64 x 57344 x 8192 182 and 176; 120 x 10880 x 8192 62.3 and 49.9; 151 x 6016
// x 10240 92.8 and 61.4), but for rows of a multiple of 32 KB (48 x 8192 x 16384 62, and
// 70 here), and with more than 64 rows the shortest and the longest (69 x 6144 x 2048
// 13.1 and 15.3, 96 x 13824 x 16384 118 and 137), narrow matrices of few rows or
// of short ones (96 x 2464 x 4096 12.8 and 16.3; but 108 x 2112 x 6144 38.9 and 19.7),
// and of 129 to 192 rows widths whose second round of tiles is nearly empty (135 x 4288
// x 6144 29.2 and 33.3, 132 x 4352 x 8192 35.2 and 40.2). Of 3700 products that a fifth more
// would take from it 1003 stay, 470 slower by more than 3 % here; of the others 65 are,
// and together they are 1.15 times as fast. Up to 96 rows whose shares begin on whole
// 4 KB of rows of a multiple of 16 KB stay with it: of 8192 x 8192 32 to 40 us either
// way, of 128 rows 48, and 39 here. What nothing is shared of begins and ends 2 us
// sooner (55 x 11264 x 2048, gated: 16 us, the library 21).
// Of 7795 products (17 to 256 rows, 250 to 20000 x 512 to 32768, an eighth of them
// sizes of models, a quarter paired) this takes 0.75 of the library's time on
// average, where 0.72 is the least of either; 30 take longer than the library's, by
// 3 to 16 %, none of those of models. us on a MI355X, measured and (estimated), the
// library's and ours:
//   32 x 8192 x 8192   30 38 (32 42)     160 x 4096 x 11008   71  39 (53 43)
//   64 x 4544 x 4544   28 17 (23 17)     128 x 4544 x 18176  151  48 (67 48)
//   64 x 4096 x 11008  34 28 (39 27)     208 x 6144 x 4096    27  36 (24 37)
//   64 x 4096 x 4096   15 13 (16 16)     224 x 5120 x 13824  111  62 (90 74)
//   96 x 768 x 3072   7.8 10 (10 11)      80 x 10240 x 8192   75  42 (48 43)
// Of such rows the widest are taken by up to 64 in any case, up to inner sizes where
// memory is all that either waits for (20 x 44032 x 16384 260 us, and 267 here; 32 x
// 57344 x 8192, gated, 171 and 176): 20 x 32000 x 2048 33.4 us, and 26.1 here, 64 x
// 32000 x 4096 61.6 and 50.7, 64 x 128256 x 4096 210 and 191, 48 x 29760 x 12288 174
// and 130, 20 x 28672 x 4096, gated, 56.7 and 47.3. More rows lose what there is to
// gain (96 x 48000 x 6144 146 and 143), or are two blocks, which read the weights
// twice (130 x 32000 x 4096 65 and 93). Nor are those of more than 32 rows whose
// second round of 256 workgroups is all but empty, where rows are of 4 KB (64 x 33328 x
// 2048 40.5 us, and 53.4 here; 48 x 36864 x 2048, gated, 41.7 and 46.3) or of more than
// 16 (64 x 38272 x 10240 158 and 175; but 34 x 33216 x 4096 88.8 and 73.5, 57 x 37824 x
// 8192 169 and 150), and of rows of 16 KB the narrowest and widest (24 x 27648 x 8192
// 116 and 96, 20 x 22016 x 8192 87.3 and 70.3, but 32 x 16384 x 8192 55.8 and 58.0, 20 x
// 57344 x 8192 164 and 188; of 33 to 64 rows the last alone take 175 to 179 either way,
// and steps of llama2-70b are 2 to 3 % shorter with it: 40 rows 990 -> 955). Of 2100
// products 22 are slower by more than 3 %, by 7 at most, and they are 1.17 times as
// fast; of the others 233 would be.
// A norm that adds up the shares saves a launch: 3.5 us of a product that would have
// been this one's (64 x 4096 x 4096 16.1 -> 13.8 us, 64 x 4096 x 14336 37.1 -> 33.9,
// 256 x 4096 x 11008 47.2 -> 43.8; of 8070 of those widths none slower by more than
// 1 %, 1.10 times as fast on average). For its sake products leave the library, too,
// from a product and a norm of its own, weights from memory: 96 x 4096 x 4096 25.8 ->
// 19.2 us, 128 28.3 -> 21.3, 144 25.7 -> 21.5, 96 x 2048 x 5632 19.0 -> 14.2, 192 23.5
// -> 19.2. But not of more than 64 rows where the estimates are not near enough: short
// ones whose results are a round of the library's small tiles (69 x 2560 x 3072 13.7
// -> 15.9, 104 x 1984 x 3840 14.8 -> 18.3), wide ones (68 x 11648 x 3712 37.3 -> 40.8,
// 144 x 8640 x 6272 50.9 -> 65.0, 162 x 5120 x 8192 42.8 -> 45.3, 231 x 6656 x 12288
// 86.5 -> 91.3), but for the longest, of which the library has few tiles (256 x 5632 x
// 24576 292 -> 134). Of 6000 products that 3.5 us more would take from the library
// 5383 are, 1.19 times as fast, 39 slower by more than 3 % (of 5000 others 4497, 1.19,
// 30; most 5 to 10 %, a few of some 170 rows and 5500 columns up to 24: 179 x 5440 x
// 3456 26.0 -> 34.3); of the rest 196 would be.
bool mid_gemm_pays(long m, long n, long k, bool paired, bool normed) {
  if (m <= 16 || m > 256 || k < (paired ? 1024 : 2048) ||
      (m > 96 && n > 12288))
    return false;
  if (m <= 64 && n >= 16000 && k % 2048 == 0 && k <= (paired ? 6144 : 12288) &&
      !(m > 32 && n > 32768 && n <= 45056 && (k == 2048 || k > 8192)) &&
      (k != 8192 || (m <= 32 ? n > 16384 && n <= 32768
                             : n >= 24576 && n <= 57344)))
    return true;
  if (!paired && k < 3072) return false;
  const double few = std::min(1., n / 4500.);
  const double inner = m > 128 ? 1.5e-3 + 1.7e-3 * few : .6e-3 + .6e-3 * few;
  const double work = n * k * 2 / 1e7 + k * inner + m * n * k * 2 / 2e9;
  const bool round =
      k <= 6144 ? m > 144 : n <= 5120 ? m > 192 : n > 6144 || m <= 160;
  const bool same = paired && k % 2048 == 0 &&
                    (m <= 64     ? k % 16384 != 0
                     : n <= 2800 ? m > 96 && k > 4096 && k < 16384
                     : n <= 8300 ? k > 2048 && k < 16384 &&
                                       (m <= 128 || n <= 4096 || round)
                     : m <= 128  ? k < 8192 || (n <= 12288 && k < 16384)
                                 : m > 144 && k < 8192);
  const double library =
      (m > 128 ? 1. : 6.6) + work * (k % 256 ? 1.45 : same ? 1.2 : 1.);
  const bool longer = m > 32 && m < 256 && n <= 10240 &&
                      k >= (m > 128 ? 12288 : 8192);
  const MidPlan plan = mid_gemm_plan(m, n, k);
  const long share = ((k + STEP - 1) / STEP + plan.splits - 1) / plan.splits;
  const bool in_step = !(paired || normed) && m <= 96 && k % 8192 == 0 &&
                       share % 32 == 0;
  const double theirs = library * (longer ? 1.2 : 1.);
  const bool tiles = n <= 2816 && k <= 4096 && m * n > 130000 && m * n <= 262144;
  const bool near =
      m <= 64 || k > 16384 ? true
      : tiles              ? false
      : m <= 128           ? n <= 10240
      : k <= 4096          ? n <= 8192
      : k <= 8448          ? n <= (m > 192 ? 8192 : 4096)
                           : n <= 5120;
  const bool saved = normed && near && plan.splits > 1 &&
                     (m <= 64 || n >= 1536 || k > 4096);
  const double pass = saved ? 3.5
                      : !paired ? 0. : n >= 4096 && k >= 2048 ? 2. : 1.;
  const double ours = plan.us * (in_step ? 1.25 : 1.) -
                      (plan.splits > 1 ? 0. : 2.);
  return ours < theirs + pass;
}

bool mid_norm_takes(long m, long n, long k) {
  return mid_gemm_takes(m, n, k, false) && n % 4 == 0 && n <= 16384 &&
         mid_gemm_plan(m, n, k).splits > 1;
}

// Whether workgroups begin at different places of the inner dimension. Where they all
// read the same columns, and rows are a multiple of a large power of two of bytes, or
// nearly, they meet at few of the memory's channels. us, from the start -> spread:
// 64 x 8192 x 8192 40.8 -> 31.7, 64 x 28672 x 4096, gated, 53.2 -> 45.4, 64 x 57344 x
// 8192, gated, 181 -> 176, 64 x 4096 x 14336 34.6 -> 30.1, 64 x 4096 x 11008 27.6 ->
// 25.9, 128 x 8192 x 8192 45.2 -> 38.5, 128 x 22016 x 4096, gated, 56.5 -> 53.3. Rows
// of other lengths, and many long ones, of which x is no longer read by all at the
// same time, lose 2 to 6 %: 64 x 6656 x 17920 55.5 -> 57.1, 224 x 4544 x 18176 77.4 ->
// 82.7, 160 x 8192 x 28672 158 -> 166.
static bool mid_gemm_spreads(int m, int k) {
  return k % 2048 == 0 && (m <= 64 || k <= 8192) ||
         k % 256 == 0 && m <= 64 && k <= 12288;
}

void launch_mid_gemm(const MidGemm& given, const MidPlan& plan,
                     const Heads* heads, bool gated, bool gelu,
                     const MidNorm* norm, float* part, hipStream_t stream) {
  MidGemm a = given;
  a.blocks = (a.m + plan.rows - 1) / plan.rows;
  a.quads = a.n % 4 == 0 && a.y_ld % 4 == 0 &&
            reinterpret_cast<uintptr_t>(a.y) % 8 == 0;
  const Heads h = heads ? *heads : Heads{};
  const int tiles = (a.n + 15) / 16;
  auto launch = [&](auto f, auto n, auto p) {
    constexpr int F = decltype(f)::value, N = decltype(n)::value,
                  P = decltype(p)::value;
    auto pick = [&](auto spread) {
      constexpr bool S = decltype(spread)::value;
      return heads ? mid_gemm_kernel<Columns::HEADS, F, N, P, S>
             : gated ? mid_gemm_kernel<Columns::GATED, F, N, P, S>
             : gelu ? mid_gemm_kernel<Columns::GELU, F, N, P, S>
                    : mid_gemm_kernel<Columns::PLAIN, F, N, P, S>;
    };
    auto kernel = mid_gemm_spreads(a.m, a.k) ? pick(std::true_type{})
                                             : pick(std::false_type{});
    kernel<<<dim3((tiles + N - 1) / N * a.blocks, plan.splits), WAVES * WAVE,
             0, stream>>>(a, h, part);
  };
  using std::integral_constant;
  auto wide = [&](auto f) {
    constexpr int F = decltype(f)::value;
    constexpr integral_constant<int, 4> c4{};
    constexpr integral_constant<int, 8> c8{};
    if (plan.tiles == 4) launch(f, c4, integral_constant<int, F == 2 ? 6 : F <= 4 ? 5 : F == 6 ? 4 : 3>{});
    else launch(f, c8, integral_constant<int, F == 2 ? 4 : F == 4 ? 3 : F == 6 ? 5 : 4>{});
  };
  if (plan.rows == 32) wide(integral_constant<int, 2>{});
  else if (plan.rows == 64) wide(integral_constant<int, 4>{});
  else if (plan.rows == 96) wide(integral_constant<int, 6>{});
  else wide(integral_constant<int, 8>{});
  if (norm) {
    auto kernel = a.n <= 2048 ? mid_norm_kernel<512, 1>
                  : a.n <= 4096 ? mid_norm_kernel<1024, 1>
                  : a.n <= 8192 ? mid_norm_kernel<1024, 2>
                                : mid_norm_kernel<1024, 4>;
    const dim3 block(a.n <= 2048 ? 512 : 1024);
    kernel<<<dim3(a.m), block, 0, stream>>>(a, *norm, part, plan.splits);
  } else if (plan.splits > 1) {
    auto sum = heads ? mid_sum_kernel<Columns::HEADS>
               : gated ? mid_sum_kernel<Columns::GATED>
               : gelu ? mid_sum_kernel<Columns::GELU>
                       : mid_sum_kernel<Columns::PLAIN>;
    const long quads = (long)a.m * tiles * (heads || gated ? 2 : 4);
    sum<<<dim3((quads + 255) / 256), 256, 0, stream>>>(a, h, part,
                                                       plan.splits);
  }
}
