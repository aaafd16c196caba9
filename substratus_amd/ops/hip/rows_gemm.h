// What products of a few rows with a weight matrix share (rows_gemm.hip for
// bf16 weights, rows_quant.hip for GGUF blocks).
#pragma once

#include "common.h"

typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) short short4v;
typedef __attribute__((ext_vector_type(4))) float float4v;

#define LDS_LOAD_ARGS(g, lds)                                        \
  (const __attribute__((address_space(1))) unsigned int*)(g),        \
      (__attribute__((address_space(3))) unsigned int*)(lds)

// SZ bytes of every lane go from its address to lds + lane * SZ.
template <int SZ>
DEV_INLINE void load_to_lds(const void* g, void* lds) {
  static_assert(SZ == 16 || SZ == 4);
  if constexpr (SZ == 16)
    __builtin_amdgcn_global_load_lds(LDS_LOAD_ARGS(g, lds), 16, 0, 0);
  else
    __builtin_amdgcn_global_load_lds(LDS_LOAD_ARGS(g, lds), 4, 0, 0);
}

// Until no more than the N loads issued last are in flight.
template <int N>
DEV_INLINE void wait_loads() {
  static_assert(N < 64);
  asm volatile("s_waitcnt vmcnt(%0)" :: "i"(N) : "memory");
}

// What was read from LDS is in registers: its place may be loaded over.
DEV_INLINE void wait_lds_reads() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// What becomes of a workgroup's 16 columns.
//   PLAIN  they are stored
//   GELU   they are rounded, and what is stored is their gelu
//   GATED  eight gate another eight, which begin half a matrix later
//   HEADS  of a fused projection of query, key and value heads: eight are
//          rotated with another eight, half a head later; queries are stored,
//          keys and values go to the paged cache
//   ADDED  they are added to the residual stream (AddTo)
enum class Columns { PLAIN, GATED, HEADS, GELU, ADDED };

// Whether a workgroup has eight columns and another eight that go with them.
constexpr bool paired(Columns c) {
  return c == Columns::GATED || c == Columns::HEADS;
}

// For HEADS: what launch_rope_kv_append takes.
struct Heads {
  const int* positions;
  const int* slots;
  void* k_cache;              // [blocks, hkv, block_size, d]
  void* v_cache;
  int hq, hkv, d, block_size;
  float ln_theta;
  bool turned;                // else keys and queries stay as they are
  bool kv8;                   // the cache is fp8
};

// A workgroup's first column, and how much later its second eight are.
template <Columns C>
DEV_INLINE int first_column(const Heads& heads) {
  const int at = blockIdx.x * (paired(C) ? 8 : 16);
  if constexpr (C == Columns::HEADS) {
    const int half = heads.d / 2;
    return at + at / half * half;
  }
  return at;
}

template <Columns C>
DEV_INLINE int second_half(int n, const Heads& heads) {
  return C == Columns::HEADS ? heads.d / 2 : n / 2;
}

// What becomes of a product that is added to the residual stream h, whose RMSNorm
// the next product takes: sum = h + the columns, rounded, y = sum * weight, and
// each workgroup's part of every row's squares. A row's 1/deviation only scales
// the results of that product, which adds the parts up while its first weights
// are on their way (Undivided): no launch for the norm, and nothing of it is made
// by every workgroup. us of a captured decode step on a MI355X, from a launch for
// each norm of 5 rows and more, and NormOf's of fewer, to this: 890 -> 848 (8
// rows, 8 layers of 4096), 685 -> 653 (5 rows, 6 layers of 5120, q4_K), 600 -> 568
// (1 row, 8 layers of 5120, q4_0), 620 -> 617 (1 row, 16 layers of 2048).
struct AddTo {
  const bf16_t *h, *weight;     // [m, n], [n]
  bf16_t* sum;                  // [m, n]
  float* squares;               // [m, workgroups]
};
struct Undivided {
  const float* squares;         // [m, parts], or null: nothing is divided
  int parts;                    // a multiple of 4
  float eps;
};

// A row's sum of squares, by a wave. Asked for behind a workgroup's first weights.
template <int PER>
struct RowSquares {
  float4 v[PER];
  float rest;

  DEV_INLINE void load(const Undivided& of, int r) {
    const float* row = of.squares + (long)r * of.parts;
    const int at = threadIdx.x % WAVE * 4;
    #pragma unroll
    for (int i = 0; i < PER; ++i)
      if (i * 256 < of.parts)
        v[i] = *reinterpret_cast<const float4*>(
            row + min(at + i * 256, of.parts - 4));
    rest = 0.f;
    for (int j = at + PER * 256; j < of.parts; j += 256) {
      const float4 u = *reinterpret_cast<const float4*>(row + j);
      rest += u.x + u.y + (u.z + u.w);
    }
  }
  DEV_INLINE float sum(const Undivided& of) const {
    const int at = threadIdx.x % WAVE * 4;
    float s = rest;
    #pragma unroll
    for (int i = 0; i < PER; ++i)
      if (at + i * 256 < of.parts) s += v[i].x + v[i].y + (v[i].z + v[i].w);
    return wave_sum(s);
  }
};

DEV_INLINE float undivided_scale(const Undivided& of, float squares, int k) {
  return rsqrtf(squares / (float)k + of.eps);
}

// x as the norm of a sum, made by the product itself, where what is added has to be
// summed over ranks first: RMS of h + delta, which
// the first workgroup stores in sum. A row's 1/deviation only scales its
// results, so a workgroup multiplies (h + delta) * weight, rounded like a
// normed row, and scales at the end; it sums squares meanwhile. On a MI355X, us
// of a decode step with a launch for each norm -> in the products: 737 -> 688
// (1 row, 16 layers of 2048), 630 -> 614 (1 row, 8 layers of 5120, q4_0). Every
// workgroup makes all of x: more than 8192 numbers of it would take LDS from
// other workgroups.
struct NormOf {
  const bf16_t *delta, *h, *weight;
  bf16_t* sum;
  float eps;
};

constexpr int NORM_ROWS = 4;            // of x, at most
constexpr int NORM_PIECES = 1024;       // 16-byte pieces of x in LDS, at most

// A thread's pieces of h + delta on their way, loaded before a workgroup's
// first weights so that their wait is not the weights'. A row of x in LDS is
// a piece longer than k, against bank conflicts.
template <int THREADS>
struct NormRows {
  static constexpr int PER = (NORM_PIECES + THREADS - 1) / THREADS;
  uint4 h[PER], d[PER], w[PER];

  DEV_INLINE void load(const NormOf& n, int m, int k) {
    const int row = k / 8, all = m * row;
    #pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int p = min((int)threadIdx.x + i * THREADS, all - 1);
      h[i] = reinterpret_cast<const uint4*>(n.h)[p];
      d[i] = reinterpret_cast<const uint4*>(n.delta)[p];
      w[i] = reinterpret_cast<const uint4*>(n.weight)[p % row];
    }
  }

  // x to LDS, and each wave's sum of squares of every row
  DEV_INLINE void put(const NormOf& n, int m, int k, uint4* x,
                      float (*squares)[NORM_ROWS]) {
    const int row = k / 8, all = m * row;
    float ss[NORM_ROWS] = {0.f, 0.f, 0.f, 0.f};
    #pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int p = (int)threadIdx.x + i * THREADS;
      if (p >= all) break;
      const unsigned a[4] = {h[i].x, h[i].y, h[i].z, h[i].w};
      const unsigned b[4] = {d[i].x, d[i].y, d[i].z, d[i].w};
      const unsigned c[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
      unsigned s[4], o[4];
      float q = 0.f;
      #pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float2 x0 = unpack_bf16x2(a[j]), x1 = unpack_bf16x2(b[j]);
        s[j] = pack_bf16x2(x0.x + x1.x, x0.y + x1.y);
        const float2 v = unpack_bf16x2(s[j]), g = unpack_bf16x2(c[j]);
        q += v.x * v.x + v.y * v.y;
        o[j] = pack_bf16x2(v.x * g.x, v.y * g.y);
      }
      const int r = p / row;
      #pragma unroll
      for (int e = 0; e < NORM_ROWS; ++e) ss[e] += r == e ? q : 0.f;
      x[p + r] = make_uint4(o[0], o[1], o[2], o[3]);
      if (blockIdx.x == 0)
        reinterpret_cast<uint4*>(n.sum)[p] = make_uint4(s[0], s[1], s[2],
                                                        s[3]);
    }
    #pragma unroll
    for (int e = 0; e < NORM_ROWS; ++e) ss[e] = wave_sum(ss[e]);
    if (threadIdx.x % WAVE == 0) {
      #pragma unroll
      for (int e = 0; e < NORM_ROWS; ++e)
        squares[threadIdx.x / WAVE][e] = ss[e];
    }
  }
};

template <int WAVES>
DEV_INLINE float norm_scale(const float (*squares)[NORM_ROWS], int r, int k,
                            float eps) {
  float s = 0.f;
  #pragma unroll
  for (int w = 0; w < WAVES; ++w) s += squares[w][r];
  return rsqrtf(s / (float)k + eps);
}

// LDS is written by all waves, and no load has to have arrived.
DEV_INLINE void lds_barrier() {
  wait_lds_reads();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

inline bool norm_rows_take(long m, long k) {
  return m <= NORM_ROWS && k % 8 == 0 && m * (k / 8) <= NORM_PIECES;
}

// The weight row behind row r of the 16 that a workgroup from column n0 on
// multiplies.
template <Columns C>
DEV_INLINE int weight_row(int n0, int r, int n, int half) {
  if constexpr (paired(C)) return n0 + (r & 7) + (r >> 3) * half;
  return min(n0 + r, n - 1);
}

// A pair of a head's columns of row r: what rope_kv_append_kernel (rope.hip)
// does with them after their product is rounded.
DEV_INLINE void finish_heads(bf16_t* y, long y_ld, const Heads& heads, int r,
                             int col, float a, float b) {
  const int half = heads.d / 2, j = col % heads.d;
  int head = col / heads.d;
  float x1 = bf2f(f2bf(a)), x2 = bf2f(f2bf(b));
  if (heads.turned && head < heads.hq + heads.hkv) {
    float s, c;
    const float pos = (float)heads.positions[r];
    const float inv_freq = __expf(-(float)j / (float)half * heads.ln_theta);
    __sincosf(pos * inv_freq, &s, &c);
    const float r1 = x1 * c - x2 * s;
    x2 = x2 * c + x1 * s;
    x1 = r1;
  }
  if (head < heads.hq) {
    y[r * y_ld + col] = f2bf(x1);
    y[r * y_ld + col + half] = f2bf(x2);
    return;
  }
  head -= heads.hq;
  const bool key = head < heads.hkv;
  if (!key) head -= heads.hkv;
  const int slot = heads.slots[r];
  const long at = (((long)(slot / heads.block_size) * heads.hkv + head) *
                       heads.block_size + slot % heads.block_size) *
                      heads.d + j;
  void* cache = key ? heads.k_cache : heads.v_cache;
  if (heads.kv8) {
    unsigned char* to = reinterpret_cast<unsigned char*>(cache) + at;
    to[0] = f32_to_fp8(x1);
    to[half] = f32_to_fp8(x2);
  } else {
    bf16_t* to = reinterpret_cast<bf16_t*>(cache) + at;
    to[0] = f2bf(x1);
    to[half] = f2bf(x2);
  }
}

bool rows_gemm_thin(int m, int n, int k, bool paired);
void launch_rows_gemm(bf16_t* y, const bf16_t* x, const bf16_t* w,
                      const bf16_t* bias, int m, int n, int k, long x_ld,
                      long y_ld, bool gated, bool gelu, const Heads* heads,
                      const NormOf* norm, const AddTo* add,
                      const Undivided* of, hipStream_t stream);

DEV_INLINE float silu_times(float g, float u) {
  return g / (1.f + __expf(-g)) * u;
}

// One of a row's 16 columns that a workgroup adds, the others in the lanes beside
// it (past the last one h and v are 0).
DEV_INLINE void finish_added(const AddTo& add, bf16_t* y, long at, int r,
                             bool there, float h, float weight, float v) {
  const float s = bf2f(f2bf(h + bf2f(f2bf(v))));
  if (there) {
    add.sum[at] = f2bf(s);
    y[at] = f2bf(s * weight);
  }
  const float squares = group16_sum(s * s);
  if (threadIdx.x % 16 == 0)
    add.squares[(long)r * gridDim.x + blockIdx.x] = squares;
}

// A column as it is stored. Rounded before its gelu, as gelu_kernel has it, so
// the bits are that kernel's: a launch less. us, MI355X, product and gelu ->
// one kernel: 1 x 3072 x 768 5.4 -> 3.4, 32 rows 6.4 -> 4.2, 64 rows 7.4 -> 5.3;
// 1 x 18176 x 4544 33.4 -> 31.3, 16 rows 37.6 -> 35.4; 4 x 32768 x 8192 100.3 ->
// 97.6.
template <Columns C>
DEV_INLINE bf16_t stored(float v) {
  return f2bf(C == Columns::GELU ? gelu_of(bf2f(f2bf(v))) : v);
}
