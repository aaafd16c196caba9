// y = x w^T + bias of at most 64 rows with a bf16 weight matrix [n, k], as
// single tokens of a small batch need it; or, of a matrix whose first half
// gates its second, silu(gate) * up; or, of a projection of heads, rotated
// queries, with keys and values appended to the cache.
//
// Bound by reading the weights once. A workgroup takes 16 weight rows; its
// four waves share k. A wave's loads go straight to LDS, 8 rows x 128
// contiguous bytes each, whole cache lines, with consecutive lanes on consecutive
// 16-byte pieces: loaded in the order of the matrix operands, where consecutive
// lanes have different rows, every lane is a cache lookup of its own, and that,
// not memory, sets the pace (4.5 TB/s). (16 rows x 64 bytes: half lines, 8 x 12288
// x 4096 21.2 us instead of 19.7, 16 rows of it 25.9 instead of 21.8, 48 x 2048 x
// 2048 8.3 instead of 7.2.) x takes the same way, since by registers
// its rows would cost the lookups that the weights no longer do. A stage is 64
// columns; four are in flight per wave and waited for one by one (64 KB, two
// workgroups per CU). Pieces are permuted by the row, so that operand reads
// meet no bank conflicts.
//
// us on a MI355X, from the library's product to this one:
//   1 x 6144 x 2048    12.3 -> 7.1     8 x 12288 x 4096   28.2 -> 18.5
//   1 x 2048 x 2048    10.8 -> 3.6     8 x 4096 x 4096    15.4 -> 8.0
//   1 x 11264 x 2048   16.1 -> 9.7     8 x 22016 x 4096   52.8 -> 33.1
//   1 x 2048 x 5632    11.2 -> 6.2     8 x 4096 x 11008   37.7 -> 17.4
// (5.0 to 5.8 TB/s where the matrix is large). 8 and 16 waves, or 32 rows of
// weights, are slower: fewer workgroups per CU.
//
// With 17 to 64 rows a wave has two to four operand tiles of x, and every
// workgroup reads all of x: that, not the weights, then sets the pace, so it
// pays for matrices of few rows only, of which the library's tiles make too
// few workgroups.
//   20 x 3072 x 2048   11.8 -> 6.4     48 x 3072 x 2048   11.7 -> 8.5
//   32 x 2048 x 2048   11.2 -> 6.5     64 x 2048 x 2048   11.6 -> 9.9
//   32 x 4096 x 4096   14.2 -> 12.7    64 x 2304 x 768    7.2 -> 4.4
// Four stages in flight instead of two, and eight waves, are 2 to 10% slower
// at these.
#include "rows_gemm.h"

#include <type_traits>

namespace {

constexpr int KW = 4;             // waves, which share k
constexpr int U = 2;              // 32-column chunks of a stage
constexpr int TILE = 64;          // 16-byte pieces of 16 rows x 32 columns
constexpr int PAD = 4;

// FM: tiles of 16 rows of x; P: stages in flight. THIN: a workgroup has eight
// weight rows, and the other eight of an operand are the next 64 columns of the
// same ones, beside those of x: the rows of x are eight at most then. X8: of its 16
// rows of x only eight are loaded. SPREAD: workgroups begin at different places of
// their shares.
template <Columns C, bool NORM, int FM, int P, bool THIN, bool X8,
          bool SPREAD = false>
__global__ __launch_bounds__(KW * WAVE, 2)
void rows_gemm_kernel(bf16_t* __restrict__ y, const bf16_t* __restrict__ x,
                      const bf16_t* __restrict__ w,
                      const bf16_t* __restrict__ bias, int m, int n, int k,
                      long x_ld, long y_ld, Heads heads, NormOf norm,
                      AddTo add, Undivided of) {
  // (normed x does not go through the ring)
  static_assert(!NORM || FM == 1);
  static_assert(!THIN || (FM == 1 && !NORM && !paired(C)));
  static_assert(!X8 || (FM == 1 && !NORM && !THIN));
  // of a stage, 8 rows x 64 columns
  constexpr int LOADS = NORM ? U : X8 ? U + 1 : U + U * FM;
  constexpr int STAGE = LOADS * TILE;
  constexpr int RING = KW * P * STAGE;
  // one array: beside a second one the compiler guards every LDS read against
  // the direct loads in flight, and waits for them
  __shared__ alignas(16)
      uint4 s_all[RING + (NORM ? NORM_PIECES + NORM_ROWS + KW
                               : FM == 1 ? 4 : 0)];
  uint4* s_x = s_all + RING;
  auto squares = reinterpret_cast<float (*)[NORM_ROWS]>(
      s_x + NORM_PIECES + NORM_ROWS);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE;
  const int lo = lane & 15, g = lane >> 4;
  const int n0 = THIN ? blockIdx.x * 8 : first_column<C>(heads);
  const int half = second_half<C>(n, heads);
  // shares begin on whole cache lines, of THIN on two
  constexpr int LINES = THIN ? 2 : 1, CHUNKS = U * LINES;     // of a stage
  const int chunks = k / 32, lines = (chunks + CHUNKS - 1) / CHUNKS;
  const int c0 = lines * wave / KW * CHUNKS;
  const int c1 = min(lines * (wave + 1) / KW * CHUNKS, chunks);
  const int steps = (c1 - c0 + CHUNKS - 1) / CHUNKS;
  uint4* ring = s_all + wave * P * STAGE;
  const int begin = SPREAD && steps > 0
      ? (int)(blockIdx.x * 5 % (unsigned)steps) : 0;
  auto in_share = [&](int i) {
    return SPREAD && i + begin >= steps ? i + begin - steps : i + begin;
  };

  // a load is 8 rows x 128 bytes: of a tile's row lane / 8, or eight later
  const int row = lane >> 3;
  const char *wp[2], *xp[FM][2];
  int piece[2];
  #pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = h * 8 + row, from = THIN ? row : r;
    const int at = c0 * 32 + (THIN ? h * 64 : 0);
    piece[h] = (lane & 7) ^ (r >> 1);
    wp[h] = reinterpret_cast<const char*>(
        w + (long)weight_row<C>(n0, from, n, half) * k + at);
    #pragma unroll
    for (int f = 0; f < FM; ++f)
      xp[f][h] = reinterpret_cast<const char*>(
          x + min(f * 16 + from, m - 1) * x_ld + at);
  }
  const int end = (c1 - c0) * 4 - 1;             // the share's last piece
  auto load = [&](int s, int i) {
    uint4* to = ring + s * STAGE;
    i = in_share(i);
    #pragma unroll
    for (int h = 0; h < 2; ++h) {
      // a stage may be half of one: then its last piece comes again
      const unsigned at = THIN ? (unsigned)(i * 16 + piece[h]) * 16
                               : (unsigned)min(i * 8 + piece[h], end) * 16;
      load_to_lds<16>(wp[h] + at, to + h * TILE);
      if constexpr (!NORM) {
        if constexpr (X8)
          if (h == 1) continue;
        #pragma unroll
        for (int f = 0; f < FM; ++f)
          load_to_lds<16>(xp[f][h] + at, to + (2 + f * 2 + h) * TILE);
      }
    }
  };
  float4v acc[FM];
  #pragma unroll
  for (int f = 0; f < FM; ++f) acc[f] = (float4v){0.f, 0.f, 0.f, 0.f};
  auto step = [&](int s, int i, bool more) {
    const int at = in_share(i);
    short8 wf[U], xf[U][FM];
    #pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint4* t = ring + s * STAGE + lo * 8 + ((u * 4 + g) ^ (lo >> 1));
      wf[u] = *reinterpret_cast<const short8*>(t);
      #pragma unroll
      for (int f = 0; f < FM; ++f)
        xf[u][f] = *reinterpret_cast<const short8*>(
            NORM ? s_x + min(lo, m - 1) * (k / 8 + 1) +
                       min(c0 + at * U + u, c1 - 1) * 4 + g
            : X8 ? ring + s * STAGE + 2 * TILE + (lo & 7) * 8 +
                       ((u * 4 + g) ^ (lo >> 1 & 3))
                 : t + (2 + f * 2) * TILE);
    }
    if (more) {
      wait_lds_reads();
      load(s, i + P);
    }
    #pragma unroll
    for (int u = 0; u < U; ++u)
      if (THIN || c0 + at * U + u < c1) {
        #pragma unroll
        for (int f = 0; f < FM; ++f)
          acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              wf[u], xf[u][f], acc[f], 0, 0, 0);
      }
  };
  // a thread ends up with column c of rows from row on
  const int c = threadIdx.x % 16, first = threadIdx.x / 16;
  bf16_t h[FM], weight;
  // rows that are still to be divided: a wave adds up the squares of every fourth
  constexpr bool DIVIDES = FM == 1 && !NORM && C != Columns::ADDED;
  const bool divided = DIVIDES && of.squares != nullptr;
  float* row_squares = reinterpret_cast<float*>(s_all + RING);
  RowSquares<2> parts[DIVIDES ? 16 / KW : 1];
  NormRows<KW * WAVE> rows;
  if constexpr (NORM) rows.load(norm, m, k);
  #pragma unroll
  for (int s = 0; s < P; ++s)
    if (s < steps) load(s, s);
  if constexpr (C == Columns::ADDED) {
    const int at = min(n0 + c, n - 1);
    #pragma unroll
    for (int f = 0; f < FM; ++f)
      h[f] = add.h[(long)min(first + f * 16, m - 1) * n + at];
    weight = add.weight[at];
  }
  if constexpr (DIVIDES) {
    // waited for at the end (added up here, 643 us instead of 616 for a step of
    // 16 layers of 2048, one row)
    #pragma unroll
    for (int i = 0; i < 16 / KW; ++i)
      if (divided && wave + i * KW < m) parts[i].load(of, wave + i * KW);
  }
  if constexpr (NORM) {
    rows.put(norm, m, k, s_x, squares);
    lds_barrier();
  }
  int i = 0;
  for (; i + 2 * P <= steps; i += P) {      // P stages in flight throughout
    #pragma unroll
    for (int s = 0; s < P; ++s) {
      wait_loads<(P - 1) * LOADS>();
      step(s, i + s, true);
    }
  }
  for (; i < steps; i += P) {               // the ring runs dry
    #pragma unroll
    for (int s = 0; s < P; ++s)
      if (i + s < steps) {
        if (i + s + P <= steps) wait_loads<(P - 1) * LOADS>();
        else wait_loads<0>();
        step(s, i + s, i + s + P < steps);
      }
  }
  __syncthreads();

  // the waves' shares are added up; a lane has four columns of one row
  constexpr int ROWS = FM * 16;
  static_assert(KW * ROWS * (16 + PAD) <= RING * 4);
  float* red = reinterpret_cast<float*>(s_all);
  #pragma unroll
  for (int f = 0; f < FM; ++f)
    *reinterpret_cast<float4v*>(
        &red[(wave * ROWS + f * 16 + lo) * (16 + PAD) + g * 4]) = acc[f];
  if constexpr (DIVIDES) {
    #pragma unroll
    for (int i = 0; i < 16 / KW; ++i)
      if (divided && wave + i * KW < m) {
        const float q = parts[i].sum(of);
        if (lane == 0) row_squares[wave + i * KW] = q;
      }
  }
  __syncthreads();
  #pragma unroll
  for (int f = 0; f < FM; ++f) {
    const int r = first + f * 16;
    if (r >= m) break;
    float scale = 1.f;
    if constexpr (NORM) scale = norm_scale<KW>(squares, r, k, norm.eps);
    else if (divided) scale = undivided_scale(of, row_squares[r], k);
    auto sum = [&](int c) {
      float v = 0.f;
      #pragma unroll
      for (int q = 0; q < KW; ++q) {
        v += red[(q * ROWS + r) * (16 + PAD) + c];
        if constexpr (THIN) v += red[(q * ROWS + r + 8) * (16 + PAD) + c + 8];
      }
      v *= scale;
      if (bias != nullptr) v += bf2f(bias[weight_row<C>(n0, c, n, half)]);
      return v;
    };
    if constexpr (C == Columns::GATED) {
      if (c < 8) y[r * y_ld + n0 + c] = f2bf(silu_times(sum(c), sum(c + 8)));
    } else if constexpr (C == Columns::HEADS) {
      if (c < 8) finish_heads(y, y_ld, heads, r, n0 + c, sum(c), sum(c + 8));
    } else if constexpr (C == Columns::ADDED) {
      const bool there = (!THIN || c < 8) && n0 + c < n;
      finish_added(add, y, r * y_ld + n0 + c, r, there, there ? bf2f(h[f]) : 0.f,
                   bf2f(weight), there ? sum(c) : 0.f);
    } else {
      if ((!THIN || c < 8) && n0 + c < n)
        y[r * y_ld + n0 + c] = stored<C>(sum(c));
    }
  }
}

}  // namespace

// Rows begin on 16-byte pieces; offsets within a row fit 32 bits.
bool rows_gemm_takes(int m, int n, int k, bool gated) {
  return m >= 1 && m <= 64 && n >= 1 && k >= 32 && k % 32 == 0 &&
         (!gated || n % 16 == 0);
}

// Whether the library's product of 17 to 64 rows takes longer, and mid_gemm.hip's:
// every workgroup, 16 columns, reads all rows here, which costs less than few
// tiles, or shares and their sums, where there are not many columns or they are
// short. us, the library, mid_gemm, this, MI355X, weights from memory (17 to 64
// rows, 512 to 16384 x 768 to 5632 measured):
//   17 rows   4096 x 4096 13.4 11.8 9.3     8192 x 3072 18.4 15.2 13.4
//   32        8192 x 2048 13.6 12.2 10.3   12288 x 2048 15.8 14.2 14.7
//   48        4096 x 4096 13.7 12.6 12.6    5120 x 2048 12.7 11.9 11.7
//             8192 x 2048 14.3 12.7 12.3   10240 x 2048 16.2 15.7 16.6
//   64        4096 x 3072 16.1 12.7 12.2    4096 x 4096 15.2 13.3 14.5
//             8192 x 1024 12.0  9.1  8.7    8192 x 2048 14.0 13.4 14.1
// paired: the library's needs a launch more, gated 17 x 8192 x 4096 18.7 20.4 15.3.
bool rows_gemm_pays(int m, int n, int k, bool paired) {
  if (m <= 16) return true;
  if (n <= 4096) return k <= (m <= 48 || n <= 1024 ? 4096 : 3072);
  if (n > 8192) return n <= 12288 && k <= 2048 && m <= 32;
  if (k <= (m <= 48 ? 2048 : 1024)) return true;
  return n > 6144 && m <= 32 && k <= (paired ? 4096 : 3072);
}

// Whether a workgroup has eight weight rows instead of 16. A CU takes in some 45
// GB/s, so the ones that have most of a matrix are what takes the time: eight rows
// instead of 16 up to 2048, three times eight instead of two of 16 from 4096 to
// 6144. (Between and past them it is as many rows either way, and x once more; of
// those wider ones rows of up to 2048 end before it matters.) us, MI355X, 16 ->
// eight, of one and eight rows:
//   768 x 3072   4.6  5.2 ->  3.6  4.2     4608 x 18432  41.6 45.2 -> 34.8 40.7
//   2048 x 2048  4.7  4.8 ->  4.1  4.2     5120 x 5120   13.7 15.3 -> 12.1 13.7
//   2048 x 5632  8.6  8.4 ->  6.5  6.8     6144 x 2560    8.1      ->  7.7
//   2560 x 10240  14 14.9 -> 13.5 16.4     6144 x 16384  44.7 47.2 -> 41.8 43.6
//   3584 x 18944  26 27.1 -> 26.0 32.3     5632 x 768     4.1  4.2 ->  4.4  4.5
bool rows_gemm_thin(int m, int n, int k, bool paired) {
  return m <= 8 && !paired && k % 128 == 0 &&
         (n <= 2048 || (n > 4096 && n <= 6144 && k > 2048));
}

// Whether workgroups begin at different columns: all at the same they meet at few of
// the memory's channels, of lengths that depend on how addresses are spread over them.
// us: 8 x 4096 x 11008 19.3 -> 17.4, 8 x 4096 x 8192 16.2 -> 13.7, 8 x 8192 x 8192 28.3
// -> 25.4, 8 x 32000 x 8192 95.9 -> 92.6; 1 x 9216 x 8448 30.8 -> 31.0. Against that
// stands the arithmetic of the loads' addresses. Of 1, 4, 8 and 16 rows and 4096 columns
// and more, at lengths of a multiple of 256, time with it over time without, on average
// (least, most): up to 4096 1.010 (0.98, 1.05) of 261 products, to 8192 1.003 (0.96,
// 1.04) of 160, in this range 0.965 (0.85, 1.03) of 88 (8192 0.91, 11008 0.94, of 49
// others 1.002), to 16384 0.995 (0.94, 1.02) of 43, longer 0.967 (0.75, 1.04) of 70; of
// other lengths 1.010 (0.88, 1.08) of 156. (A step of 8 rows and 8 layers of llama2-7b:
// with all products like this 827 -> 837, with this range 829 -> 816.)
static bool rows_gemm_spreads(int n, int k) {
  return n >= 4096 && k >= 8192 && k < 12288 && k % 256 == 0;
}

// heads: null, or what is done with the columns instead of storing them (n is
// a multiple of 16 then, like gated's)
void launch_rows_gemm(bf16_t* y, const bf16_t* x, const bf16_t* w,
                      const bf16_t* bias, int m, int n, int k, long x_ld,
                      long y_ld, bool gated, bool gelu, const Heads* heads,
                      const NormOf* norm, const AddTo* add,
                      const Undivided* of, hipStream_t stream) {
  auto launch = [&](auto normed, auto tiles, auto stages, auto thin,
                    auto eight) {
    constexpr bool N = decltype(normed)::value, T = decltype(thin)::value,
                   X = decltype(eight)::value;
    constexpr int F = decltype(tiles)::value, S = decltype(stages)::value;
    auto kernel = rows_gemm_kernel<Columns::PLAIN, N, F, S, T, X>;
    if constexpr (!T) {
      if (heads) kernel = rows_gemm_kernel<Columns::HEADS, N, F, S, T, X>;
      else if (gated) kernel = rows_gemm_kernel<Columns::GATED, N, F, S, T, X>;
    }
    if constexpr (!N)
      if (gelu) kernel = rows_gemm_kernel<Columns::GELU, N, F, S, T, X>;
    if constexpr (!N && F == 1)
      if (add) kernel = rows_gemm_kernel<Columns::ADDED, N, F, S, T, X>;
    if constexpr (!N && !T && F == 1)
      if (!(heads || gated || gelu) && rows_gemm_spreads(n, k))
        kernel = add ? rows_gemm_kernel<Columns::ADDED, N, F, S, T, X, true>
                     : rows_gemm_kernel<Columns::PLAIN, N, F, S, T, X, true>;
    constexpr int ROWS = T ? 8 : 16;
    kernel<<<dim3((n + ROWS - 1) / ROWS), dim3(KW * WAVE), 0, stream>>>(
        y, x, w, bias, m, n, k, x_ld, y_ld, heads ? *heads : Heads{},
        norm ? *norm : NormOf{}, add ? *add : AddTo{},
        of ? *of : Undivided{});
  };
  using std::integral_constant;
  constexpr std::false_type no{};
  constexpr std::true_type yes{};
  constexpr integral_constant<int, 1> one{};
  constexpr integral_constant<int, 2> two{};
  constexpr integral_constant<int, 3> three{};
  constexpr integral_constant<int, 4> four{};
  if (norm) launch(yes, one, four, no, no);
  else if (rows_gemm_thin(m, n, k, gated || heads))
    launch(no, one, four, yes, no);
  else if (m <= 8) launch(no, one, four, no, yes);
  else if (m <= 16) launch(no, one, four, no, no);
  else if (m <= 32) launch(no, two, two, no, no);
  else if (m <= 48) launch(no, three, two, no, no);
  else launch(no, four, two, no, no);
}
