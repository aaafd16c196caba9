// Grouped products (group_gemm.h) of packed rows, few to a group: experts of a
// decode step, up to 64 rows of one in a tile.
//
// Bound by reading the weights once. A workgroup has 16 of a matrix' rows (tiles
// of 16 rows of x) or 32, and its four waves share the inner dimension; a wave's
// loads go straight to LDS, 8 rows x 128 contiguous bytes with consecutive lanes
// on consecutive pieces (loaded in the order of the matrix operands every lane is
// a cache lookup of its own; 16 rows x 64 bytes are half cache lines, and 48 rows
// take 37.3 us instead of 35.1). A stage is 64 columns of the weights and of the
// 16 to 64 rows that a tile really has.
//
// us on a MI355X, 32 experts, 6 a row, 2048 -> 1408 and back, from operands loaded
// in their own order to this:
//   1 row     14.4 -> 10.4 (3.3 TB/s)    13.0 -> 10.2
//   10 rows   35.4 -> 32.2 (5.2)         35.8 -> 34.1
//   48 rows   41.1 -> 35.1 (5.3)         42.5 -> 34.0
//   128 rows  49.3 -> 38.4 (4.8)         50.0 -> 38.8
//   300 rows  62.9 -> 55.4               65.0 -> 53.9
//   500 rows  89.0 -> 73.3               86.2 -> 71.8
#include "../rows_gemm.h"
#include "group_gemm.h"

namespace {

constexpr int KW = 4;             // waves, which share k
constexpr int TILE = 64;          // 16-byte pieces of 16 rows x 32 columns
constexpr int PAD = 4;
constexpr int KC = 32;
constexpr int U = 2;              // chunks of a stage

// How rows are taken: F tiles of 16 with N of the weights', P stages in flight.
template <int F_, int N_, int P_> struct How {
  static constexpr int F = F_, N = N_, P = P_;
  static constexpr int PIECES = KW * P * U * (N + F) * TILE;     // of LDS
};

template <class H, Act ACT, class Y>
DEV_INLINE void rows_of_group(const GroupGemm<bf16_t, Y>& a, const Tile& t,
                              uint4* s_all) {
  constexpr int F = H::F, N = H::N, P = H::P;
  constexpr int TILES = N + F, STAGE = U * TILES * TILE, LOADS = U * TILES;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE, lo = lane & 15, g = lane >> 4;
  // shares begin on whole cache lines
  const int n0 = blockIdx.x * N * 16, chunks = a.k / KC;
  const int pairs = (chunks + 1) / 2;
  const int c0 = pairs * wave / KW * 2;
  const int c1 = min(pairs * (wave + 1) / KW * 2, chunks);
  const int steps = (c1 - c0 + U - 1) / U;
  uint4* ring = s_all + wave * P * STAGE;

  // a load is 8 rows x 128 bytes: of a tile's row lane / 8, or eight later.
  // Pieces are permuted by the row against bank conflicts.
  const char *wp[N][2], *xp[F][2];
  int piece[2];
  #pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = h * 8 + (lane >> 3);
    piece[h] = (lane & 7) ^ (row >> 1);
    #pragma unroll
    for (int f = 0; f < N; ++f)
      wp[f][h] = reinterpret_cast<const char*>(
          a.w + ((long)t.g * a.n + min(n0 + f * 16 + row, a.n - 1)) * a.k +
          c0 * KC);
    #pragma unroll
    for (int f = 0; f < F; ++f) {
      const int r = min(t.r0 + f * 16 + row, t.r1 - 1);
      xp[f][h] = reinterpret_cast<const char*>(
          a.x + (long)(a.src != nullptr ? a.src[r] : r) * a.x_ld + c0 * KC);
    }
  }
  const int end = (c1 - c0) * 4 - 1;             // the share's last piece
  auto load = [&](int s, int i) {
    uint4* to = ring + s * STAGE;
    #pragma unroll
    for (int h = 0; h < 2; ++h) {
      // a stage may be half of one: then its last piece comes again
      const unsigned at = (unsigned)min(i * 8 + piece[h], end) * 16;
      #pragma unroll
      for (int f = 0; f < N; ++f)
        load_to_lds<16>(wp[f][h] + at, to + (f * 2 + h) * TILE);
      #pragma unroll
      for (int f = 0; f < F; ++f)
        load_to_lds<16>(xp[f][h] + at, to + ((N + f) * 2 + h) * TILE);
    }
  };
  float4v acc[N][F];
  #pragma unroll
  for (int j = 0; j < N; ++j)
    #pragma unroll
    for (int f = 0; f < F; ++f) acc[j][f] = (float4v){0.f, 0.f, 0.f, 0.f};
  auto step = [&](int s, int i, bool more) {
    short8 wf[U][N], xf[U][F];
    #pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint4* p = ring + s * STAGE + lo * 8 + ((u * 4 + g) ^ (lo >> 1));
      #pragma unroll
      for (int f = 0; f < N; ++f)
        wf[u][f] = *reinterpret_cast<const short8*>(p + f * 2 * TILE);
      #pragma unroll
      for (int f = 0; f < F; ++f)
        xf[u][f] = *reinterpret_cast<const short8*>(p + (N + f) * 2 * TILE);
    }
    if (more) {
      wait_lds_reads();
      load(s, i + P);
    }
    #pragma unroll
    for (int u = 0; u < U; ++u)
      if (c0 + i * U + u < c1) {
        #pragma unroll
        for (int j = 0; j < N; ++j)
          #pragma unroll
          for (int f = 0; f < F; ++f)
            acc[j][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                wf[u][j], xf[u][f], acc[j][f], 0, 0, 0);
      }
  };
  #pragma unroll
  for (int s = 0; s < P; ++s)
    if (s < steps) load(s, s);
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

  // the waves' shares are added up; a thread has four columns of one row
  constexpr int ROWS = F * 16, LD = N * 16 + PAD;
  static_assert(KW * ROWS * LD <= H::PIECES * 4);
  float* red = reinterpret_cast<float*>(s_all);
  #pragma unroll
  for (int j = 0; j < N; ++j)
    #pragma unroll
    for (int f = 0; f < F; ++f)
      *reinterpret_cast<float4v*>(
          &red[(wave * ROWS + f * 16 + lo) * LD + j * 16 + g * 4]) = acc[j][f];
  __syncthreads();
  for (int e = threadIdx.x; e < ROWS * N * 4; e += KW * WAVE) {
    const int r = e / (N * 4), c = e % (N * 4) * 4;
    float4v v = {0.f, 0.f, 0.f, 0.f};
    #pragma unroll
    for (int q = 0; q < KW; ++q)
      v += *reinterpret_cast<const float4v*>(&red[(q * ROWS + r) * LD + c]);
    store4<ACT>(a, t, t.r0 + r, n0 + c, v);
  }
}

// MAX: times 16 rows that a tile may have
template <class Y, Act ACT, int MAX>
__global__ __launch_bounds__(KW * WAVE, 2)
void group_gemm_rows_kernel(GroupGemm<bf16_t, Y> a) {
  constexpr int N = MAX == 1 ? 1 : 2;
  using One = std::conditional_t<MAX == 1, How<1, N, 4>, How<1, N, 3>>;
  using Two = How<2, N, 2>;
  // one array: beside a second one the compiler guards every LDS read against
  // the direct loads in flight, and waits for them
  using Three = How<3, N, 2>;
  using Four = How<4, N, 1>;
  constexpr int LARGEST = MAX > 2 ? Three::PIECES : One::PIECES;
  __shared__ alignas(16) uint4 s_all[LARGEST];
  static_assert(MAX == 1 || Two::PIECES <= LARGEST);
  const Tile t = tile_of(a, blockIdx.y, 0, MAX * 16);
  if (t.r1 <= t.r0) return;
  const int tiles = (t.r1 - t.r0 + 15) / 16;     // of the rows there are
  if (MAX == 1 || tiles == 1) {
    rows_of_group<One, ACT>(a, t, s_all);
  } else if constexpr (MAX > 1) {
    if (MAX == 2 || tiles == 2) {
      rows_of_group<Two, ACT>(a, t, s_all);
    } else if constexpr (MAX > 2) {
      if (tiles == 3) rows_of_group<Three, ACT>(a, t, s_all);
      else rows_of_group<Four, ACT>(a, t, s_all);
    }
  }
}

}  // namespace

// Pieces of rows are known to be aligned; stages are of whole chunks.
template <class Y>
bool group_gemm_rows_takes(const GroupGemm<bf16_t, Y>& a, int tile) {
  return a.tiles != nullptr && tile <= 64 && a.k % KC == 0 && a.k >= 4 * KC &&
         a.tail == 0;
}

template <class Y>
void launch_group_gemm_rows(const GroupGemm<bf16_t, Y>& a, int tile,
                            hipStream_t stream) {
  by_act(a.act, [&](auto act) {
    constexpr Act ACT = decltype(act)::value;
    auto kernel = tile == 16 ? group_gemm_rows_kernel<Y, ACT, 1>
                  : tile == 32 ? group_gemm_rows_kernel<Y, ACT, 2>
                               : group_gemm_rows_kernel<Y, ACT, 4>;
    const int wide = tile == 16 ? 16 : 32;
    kernel<<<dim3((a.n + wide - 1) / wide, a.max_tiles), KW * WAVE, 0, stream>>>(a);
  });
}

#define INSTANTIATE(Y)                                                       \
  template bool group_gemm_rows_takes<Y>(const GroupGemm<bf16_t, Y>&, int);  \
  template void launch_group_gemm_rows<Y>(const GroupGemm<bf16_t, Y>&, int,  \
                                          hipStream_t);
INSTANTIATE(bf16_t)
INSTANTIATE(float)
