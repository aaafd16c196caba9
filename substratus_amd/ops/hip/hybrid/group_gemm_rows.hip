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
//
// Where rows are not packed, but have their groups' numbers (ids), a workgroup
// looks through all of these for its group's rows: a step's choices are a few
// hundred, which each of its waves has in registers after one load, and nothing
// waits for a kernel that packs them. Weights wait for that: asked for ahead of it
// they are also asked for where a group has no rows (8 experts of 1536 x 1536, 16
// rows of one 17.4 us, 11.0 now), and x behind two stages' weights is late (packed,
// 64 experts of 2048 x 512, 128 rows 88.4, 82.1; listed, of unlike groups, no more
// than 3 % either way).
#include "../rows_gemm.h"
#include "group_gemm.h"

#include <algorithm>
#include <climits>

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

constexpr int IDS = 512;          // that are looked through, at most

// list: of rows that are not packed, t's numbers are places in it.
template <class H, Act ACT, bool LISTED, class Y>
DEV_INLINE void rows_of_group(const GroupGemm<bf16_t, Y>& a, const Tile& t,
                              uint4* s_all, const int* list) {
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
      int r = min(t.r0 + f * 16 + row, t.r1 - 1);
      if constexpr (LISTED) {
        r = list[r];
        if (a.top > 0) r /= a.top;
      } else if (a.src != nullptr) {
        r = a.src[r];
      }
      xp[f][h] =
          reinterpret_cast<const char*>(a.x + (long)r * a.x_ld + c0 * KC);
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
    if constexpr (LISTED) {
      if (r < t.r1) store4<ACT>(a, Tile{t.g, 0, INT_MAX}, list[r], n0 + c, v);
    } else {
      store4<ACT>(a, t, t.r0 + r, n0 + c, v);
    }
  }
}

// A lane's ids, of every wave's rows.
struct Ids {
  int id[IDS / WAVE];
  DEV_INLINE void load(const int* ids, int n) {
    #pragma unroll
    for (int i = 0; i < IDS / WAVE; ++i)
      id[i] = ids[min(i * WAVE + (int)threadIdx.x % WAVE, n - 1)];
  }
  // Rows of group g, in order: those from the `from`th on, up to `most`, to a
  // wave's list. Returns how many there are in all.
  DEV_INLINE int list(int n, int g, int from, int most, int* to) const {
    const int lane = threadIdx.x % WAVE;
    int count = 0;
    #pragma unroll
    for (int i = 0; i < IDS / WAVE; ++i) {
      const bool mine = i * WAVE + lane < n && id[i] == g;
      const unsigned long long all = __ballot(mine);
      const int at = count - from + __builtin_amdgcn_mbcnt_hi(
          (unsigned)(all >> 32),
          __builtin_amdgcn_mbcnt_lo((unsigned)all, 0));
      if (mine && at >= 0 && at < most) to[at] = i * WAVE + lane;
      count += __popcll(all);
    }
    return count;
  }
};

// MAX: times 16 rows that a tile may have; LISTED: rows by their ids
template <class Y, Act ACT, int MAX, bool LISTED>
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
  constexpr int T = MAX * 16;
  constexpr int LIST = T / 4;                    // pieces of a wave's
  __shared__ alignas(16) uint4 s_all[LARGEST + (LISTED ? KW * LIST : 0)];
  static_assert(MAX == 1 || Two::PIECES <= LARGEST);
  int* list = reinterpret_cast<int*>(s_all + LARGEST +
                                     threadIdx.x / WAVE * LIST);
  auto run = [&](const Tile& t) {
    const int tiles = (t.r1 - t.r0 + 15) / 16;   // of the rows there are
    if (MAX == 1 || tiles == 1) {
      rows_of_group<One, ACT, LISTED>(a, t, s_all, list);
    } else if constexpr (MAX > 1) {
      if (MAX == 2 || tiles == 2) {
        rows_of_group<Two, ACT, LISTED>(a, t, s_all, list);
      } else if constexpr (MAX > 2) {
        if (tiles == 3) rows_of_group<Three, ACT, LISTED>(a, t, s_all, list);
        else rows_of_group<Four, ACT, LISTED>(a, t, s_all, list);
      }
    }
  };
  if constexpr (LISTED) {
    // As many workgroups as rows, where that is less than groups: a group's first
    // row has them.
    const bool by_row = a.m < a.groups;
    const int g = by_row ? a.ids[blockIdx.y] : (int)blockIdx.y;
    for (int from = 0;; from += T) {
      Ids ids;
      ids.load(a.ids, a.m);
      const int rows = ids.list(a.m, g, from, T, list) - from;
      wait_lds_reads();                          // the list is written
      if (rows <= 0 || (by_row && from == 0 && list[0] != (int)blockIdx.y))
        return;
      run(Tile{g, 0, min(rows, T)});
      if (rows <= T) return;
      __syncthreads();
    }
  } else {
    const Tile t = tile_of(a, blockIdx.y, 0, T);
    if (t.r1 > t.r0) run(t);
  }
}

}  // namespace

// Tiles of 32 where ones of 16 would do: workgroups of 32 columns instead of 16 are
// half as many, and what it takes to begin one and to add up its waves' shares counts
// more than rows that are not there. us of both products, gated, weights from memory,
// MI355X, packed 16 -> packed 32 -> 32 by ids: 32 experts of 2048 x 1408, 6 a row, 1, 4,
// 16, 32 rows 29.7 64.9 100.9 106.9 -> 28.7 62.5 99.3 100.9 -> 26.5 64.1 98.1 100.8; of
// 4096 x 2048, 8 a row, 1, 4, 24 rows 80.4 193.4 275.1 -> 79.1 181.6 271.6 -> 76.5
// 182.8 269.6; 64 of 2048 x 1408, 8, 16 and 64 rows 114 149 202 -> 114 145 190 -> 116
// 143; 8 of 4096 x 1408, 2 a row, 4 and 16 rows 40.5 57 -> 41.4 54.8 -> 39.5 53.4.
// Shorter rows are another kernel's with tiles of 16 (64 of 2048 x 512, 4 a row, 16
// rows 54.2 -> 58.8).
int group_gemm_rows_tile(int tile, int k, int n) {
  return tile == 16 && k % KC == 0 && n % KC == 0 && std::min(k, n) > 1280
      ? 32 : tile;
}

// A workgroup's columns.
static int columns(int tile) { return tile == 16 ? 16 : 32; }

// Pieces of rows are known to be aligned; stages are of whole chunks. Where rows are
// short and there are workgroups for the chip many times over, what it takes to
// begin one and to add up its waves' shares counts: 16 columns of up to 1280 long
// rows, or 32 of up to 128, cost more than the kernel of 64. Its time over this
// one's, MI355X, 16 to 64 experts, 1 to 32 rows each in tiles of 16 (of 32 and 64):
//   inner size             128        256         512         768     1024  1408
//   up to 1024 workgroups  - (0.94-   0.98-1.30   1.06-1.45   1.16-   1.3-  1.3-
//                          1.27)      (1.2-1.4)   (1.4-1.7)   1.6     1.6   1.6
//   more                   - (0.76-   0.55-0.98   0.67-1.26   0.77-   0.85- 0.92-
//                          1.06)      (1.0-1.2)   (0.9-1.7)   1.18    1.38  1.25
template <class Y>
bool group_gemm_rows_takes(const GroupGemm<bf16_t, Y>& a, int tile) {
  if ((a.tiles == nullptr && a.ids == nullptr) || tile > 64 || a.k % KC != 0 ||
      a.k < 4 * KC || a.tail != 0 ||
      (a.ids != nullptr && (a.m > IDS || tile > 32)))
    return false;
  const long blocks = (long)(a.n + columns(tile) - 1) / columns(tile) * a.max_tiles;
  return blocks <= 1024 || a.k > (tile == 16 ? 1280 : 128);
}

// Looking for one's rows takes longer than to be told, in every workgroup, and a kernel
// that packs 3 us (4.5 in a step). us of two products, MI355X, packed -> not, by tiles
// of 32, of 1, 4, 16, 32, 64 rows: 32 experts of 2048 x 1408, 6 a row 28.7 62.5 99.3
// 100.9 104 -> 26.5 64.1 98.1 100.8 104.3 (4864 workgroups, 64 rows: 1.9 M); of 4096 x
// 2048, 8 a row, 24 rows 271.6 -> 269.6 (8192: 1.6 M); 8 of 2048 x 1408, 2 a row 17.3
// 27.1 33.6 34.1 35.4 -> 14.6 24.1 30.9 31.6 33.1; 16 of 512 x 256, 2 a row, tiles of
// 16, 4 and 48 rows 10.5 12.1 -> 8.2 9. Tiles of 64 wait for their rows at the start of
// every stage: 74 -> 97.
bool group_gemm_ids_pay(int rows, int n, int n2, int groups, int tile) {
  const int wide = columns(tile);
  return tile <= 32 &&
         (long)((n + wide - 1) / wide + (n2 + wide - 1) / wide) * groups *
                 rows <= 2000000;
}

template <class Y>
void launch_group_gemm_rows(const GroupGemm<bf16_t, Y>& a, int tile,
                            hipStream_t stream) {
  by_act(a.act, [&](auto act) {
    constexpr Act ACT = decltype(act)::value;
    const int wide = columns(tile);
    auto go = [&](auto listed, int tiles) {
      constexpr bool L = decltype(listed)::value;
      auto kernel = tile == 16 ? group_gemm_rows_kernel<Y, ACT, 1, L>
                               : group_gemm_rows_kernel<Y, ACT, 2, L>;
      if constexpr (!L)
        if (tile == 64) kernel = group_gemm_rows_kernel<Y, ACT, 4, L>;
      kernel<<<dim3((a.n + wide - 1) / wide, tiles), KW * WAVE, 0, stream>>>(
          a);
    };
    if constexpr (std::is_same_v<Y, bf16_t> && ACT != Act::GATE &&
                  ACT != Act::SIDE)
      if (a.ids != nullptr) {
        go(std::true_type{}, std::min(a.m, a.groups));
        return;
      }
    go(std::false_type{}, a.max_tiles);
  });
}

#define INSTANTIATE(Y)                                                       \
  template bool group_gemm_rows_takes<Y>(const GroupGemm<bf16_t, Y>&, int);  \
  template void launch_group_gemm_rows<Y>(const GroupGemm<bf16_t, Y>&, int,  \
                                          hipStream_t);
INSTANTIATE(bf16_t)
INSTANTIATE(float)
