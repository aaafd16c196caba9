// Grouped products (group_gemm.h) of packed rows, few to a group: experts of a
// decode step, up to 32 rows of one in a tile.
//
// Bound by reading the weights once. A workgroup has 16 of a matrix' rows (tiles
// of 16 rows of x) or 32 (tiles of up to 32), and its four waves share the inner
// dimension; a wave's loads go straight to LDS, 16 rows x 64 contiguous bytes
// with consecutive lanes on consecutive pieces (loaded in the order of the matrix
// operands every lane is a cache lookup of its own). A stage is 64 columns of the
// weights and of the 16 or 32 rows that a tile really has.
//
// us on a MI355X, 32 experts, 6 a row, 2048 -> 1408 and back, from operands loaded
// in their own order to this:
//   1 row     14.4 -> 10.3 (3.4 TB/s)    13.0 -> 9.9
//   10 rows   35.4 -> 31.4 (5.3)         35.8 -> 34.1
//   48 rows   41.1 -> 37.3 (5.0)         42.5 -> 38.8
//   64 rows   42.0 -> 39.0
//   100 rows  43.4 -> 43.7
// Tiles of 48 and 64 rows read more of x than of weights and are no faster so
// (128 rows 49.3, 50.6): those stay with the other kernel. 48 rows, 16 and 64
// columns a workgroup: 38.0 43.7, 41.3 39.4.
#include "../rows_gemm.h"
#include "group_gemm.h"

namespace {

constexpr int KW = 4;             // waves, which share k
constexpr int TILE = 64;          // 16-byte pieces of 16 rows x 32 columns
constexpr int PAD = 4;
constexpr int KC = 32;

// How rows are taken: F tiles of 16 with N of the weights', U chunks a stage, P
// stages in flight.
template <int F_, int N_, int U_, int P_> struct How {
  static constexpr int F = F_, N = N_, U = U_, P = P_;
  static constexpr int PIECES = KW * P * U * (N + F) * TILE;     // of LDS
};

template <class H, Act ACT, class Y>
DEV_INLINE void rows_of_group(const GroupGemm<bf16_t, Y>& a, const Tile& t,
                              uint4* s_all) {
  constexpr int F = H::F, N = H::N, U = H::U, P = H::P;
  constexpr int TILES = N + F, STAGE = U * TILES * TILE, LOADS = U * TILES;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE, lo = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * N * 16, chunks = a.k / KC;
  const int c0 = chunks * wave / KW, c1 = chunks * (wave + 1) / KW;
  const int steps = (c1 - c0 + U - 1) / U;
  uint4* ring = s_all + wave * P * STAGE;

  // a lane loads 16 bytes of row lane / 4 of a tile, permuted by the row
  // against bank conflicts
  const int row = lane >> 2, piece = (lane & 3) ^ ((row >> 2) & 3);
  const char* wp[N];
  #pragma unroll
  for (int f = 0; f < N; ++f)
    wp[f] = reinterpret_cast<const char*>(
        a.w + ((long)t.g * a.n + min(n0 + f * 16 + row, a.n - 1)) * a.k) +
        piece * 16;
  const char* xp[F];
  #pragma unroll
  for (int f = 0; f < F; ++f) {
    const int r = min(t.r0 + f * 16 + row, t.r1 - 1);
    xp[f] = reinterpret_cast<const char*>(
        a.x + (long)(a.src != nullptr ? a.src[r] : r) * a.x_ld) + piece * 16;
  }
  auto load = [&](int s, int i) {
    #pragma unroll
    for (int u = 0; u < U; ++u) {
      // a stage may be half of one: then its last chunk comes twice
      const unsigned at = (unsigned)min(c0 + i * U + u, c1 - 1) * 64;
      uint4* to = ring + s * STAGE + u * TILES * TILE;
      #pragma unroll
      for (int f = 0; f < N; ++f) load_to_lds<16>(wp[f] + at, to + f * TILE);
      #pragma unroll
      for (int f = 0; f < F; ++f)
        load_to_lds<16>(xp[f] + at, to + (N + f) * TILE);
    }
  };
  const int at = lo * 4 + (g ^ ((lo >> 2) & 3));
  float4v acc[N][F];
  #pragma unroll
  for (int j = 0; j < N; ++j)
    #pragma unroll
    for (int f = 0; f < F; ++f) acc[j][f] = (float4v){0.f, 0.f, 0.f, 0.f};
  auto step = [&](int s, int i, bool more) {
    short8 wf[U][N], xf[U][F];
    #pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint4* p = ring + s * STAGE + u * TILES * TILE + at;
      #pragma unroll
      for (int f = 0; f < N; ++f)
        wf[u][f] = *reinterpret_cast<const short8*>(p + f * TILE);
      #pragma unroll
      for (int f = 0; f < F; ++f)
        xf[u][f] = *reinterpret_cast<const short8*>(p + (N + f) * TILE);
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
  using One = std::conditional_t<MAX == 1, How<1, N, 2, 4>, How<1, N, 2, 3>>;
  using Two = How<2, N, 2, 2>;
  // one array: beside a second one the compiler guards every LDS read against
  // the direct loads in flight, and waits for them
  __shared__ alignas(16)
      uint4 s_all[MAX > 1 && Two::PIECES > One::PIECES ? Two::PIECES
                                                        : One::PIECES];
  const Tile t = tile_of(a, blockIdx.y, 0, MAX * 16);
  if (t.r1 <= t.r0) return;
  if (MAX == 1 || t.r1 - t.r0 <= 16)             // rows that there are
    rows_of_group<One, ACT>(a, t, s_all);
  else if constexpr (MAX > 1)
    rows_of_group<Two, ACT>(a, t, s_all);
}

}  // namespace

// Pieces of rows are known to be aligned; stages are of whole chunks.
template <class Y>
bool group_gemm_rows_takes(const GroupGemm<bf16_t, Y>& a, int tile) {
  return a.tiles != nullptr && tile <= 32 && a.k % KC == 0 && a.k >= 4 * KC &&
         a.tail == 0;
}

template <class Y>
void launch_group_gemm_rows(const GroupGemm<bf16_t, Y>& a, int tile,
                            hipStream_t stream) {
  by_act(a.act, [&](auto act) {
    constexpr Act ACT = decltype(act)::value;
    auto kernel = tile == 16 ? group_gemm_rows_kernel<Y, ACT, 1>
                             : group_gemm_rows_kernel<Y, ACT, 2>;
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
