// Attention of prompt portions over the paged bf16 cache (which already holds
// the portion's own keys and values), with a distance bias, a chunk mask,
// unequal key and value head sizes, a gated output, and softmax or sigmoid
// weights; the formulas are in attention_ctx.hip. Rows of a portion carry
// their absolute positions, so a prompt can be cut anywhere.
//
// A step's chain (products of scores, weights, products of values, the barrier) is what
// bounds it: 3 us of a wave alone on its SIMD, 4.5 of two; memory and the matrix cores
// wait. The structure is that of attention_v5.hip: every wave owns 32 query rows
// kept in registers, 64 keys per step go through LDS, S^T = K Q^T leaves a
// lane with scores of its own query row only, and softmax stays in registers.
// Differences:
//   * K and V rows are gathered through the block table, page numbers one
//     step ahead of the rows they point at;
//   * a step's biases depend only on i - j: one window of the bias row per
//     step and workgroup in LDS;
//   * the weights enter the second product as bf16 high and low parts, i.e.
//     with 16 mantissa bits, so softmax weights keep more than bf16 carries;
//   * keys and values may also lie unpaged, projected for this step from what
//     the cache holds (FLAT), with a key part that all heads share;
//   * where tiles of the most rows are too few for the chip, two waves share 32 rows
//     and take every other 32 keys; their sums meet in LDS at the end;
//   * where those are too few, too, workgroups share a tile's keys, merged by
//     attn_ctx_merge;
//   * V is staged with keys 4..7 and 8..11 of every 16 exchanged, which is
//     the order in which the score accumulators hold them: weights need no
//     lane exchange before the second product.
#include "attention_ctx.h"

#include <algorithm>

typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) short short4v;
typedef __attribute__((ext_vector_type(16))) float float16v;

namespace {

constexpr int CH = 64;          // keys per step
constexpr int PAGE = 16;

DEV_INLINE short4v tr16_read(const short* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) short4v*)p);
}

// KK: 16-wide steps of the key size; DC: 32-wide tiles of the value size
enum Kind {
  PLAIN,
  CAP,        // scores are capped
  SIGMOID,    // weights are sigmoids: no maximum, no sum
};

// SH: waves that share their 32 query rows, each a part of a step's keys
template <int KK, int DC, int WAVES, int SH, bool FLAT, Kind KIND>
__global__ __launch_bounds__(WAVES * WAVE)
void attn_ctx_prefill_kernel(AttnCtx<bf16_t> a, int splits,
                             float* __restrict__ part_o,
                             float* __restrict__ part_ml) {
  constexpr int THREADS = WAVES * WAVE;
  constexpr int RW = WAVES / SH;            // waves of unlike rows
  constexpr int QT = RW * 32;               // query rows per workgroup
  constexpr int NS = CH / 32 / SH;          // a wave's keys of a step, by 32
  constexpr int KROW = KK * 16 + 8;         // padded LDS row, in elements
  constexpr int BW = QT + CH - 1;           // distances met in one step
  constexpr int LK = (CH * KK * 2 + THREADS - 1) / THREADS;
  constexpr int LV = (CH * DC * 4 + THREADS - 1) / THREADS;
  static_assert(BW <= THREADS, "one bias per thread");

  __shared__ alignas(16) short s_k[2][CH][KROW];
  __shared__ alignas(16) short s_v[2][DC][CH / 32][2][2][16][16];
  __shared__ float s_b[2][THREADS];

  // longest rows first, of all entries or of each
  const bool each = SH > 1 && a.by_entry;
  const int e = SH == 1 ? blockIdx.x : each ? blockIdx.z : blockIdx.y;
  const int head = SH > 1 ? blockIdx.x : blockIdx.y;
  const int place = each ? gridDim.y - 1 - blockIdx.y
                         : gridDim.z - 1 - blockIdx.z;
  const int tile = place / splits, split = place % splits;
  if (SH > 1 && e >= a.entries) return;
  const Entry en = entry_of(a.seq_start, e);
  const int q0_tile = tile * QT;
  if (q0_tile >= en.n) return;
  const int kvh = head / (a.heads / a.kv_heads);
  const int* bt = FLAT ? nullptr : a.block_table + (long)e * a.max_blocks;
  const int kd = a.dim - a.shared;               // a head's own key elements

  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
  const int lo5 = lane & 31, hi = lane >> 5;
  const int pos0 = a.positions[en.row0];
  const int total = pos0 + en.n;                 // keys in the cache
  const int from = FLAT ? flat_from(a.window, pos0) : 0;
  const long flat0 = FLAT ? (long)a.ctx_start[e] - from : 0;
  const int qa0 = pos0 + q0_tile;                // first position of the tile
  const int part_of = SH > 1 ? wave / RW : 0;    // which of a step's keys
  const int rw = SH > 1 ? wave % RW : wave;
  const int qw0 = qa0 + rw * 32;                 // first position of the wave
  const bool wave_live = qw0 < total;
  const int qpos = qw0 + lo5;
  const int row = min(q0_tile + rw * 32 + lo5, en.n - 1);
  const int lo = first_seen(a, qpos), lo_wave = first_seen(a, qw0);
  const int hi_wave = min(qw0 + 31, total - 1);
  // lo of the wave's last row: keys at or above it are inside every range
  const int lo_last = first_seen(a, qw0 + 31);
  const Pieces part(a.keep, first_seen(a, qa0),
                    (min(qa0 + QT, total) + CH - 1) / CH, CH);

  short8 qreg[KK];
  {
    const bf16_t* qp = a.q + (long)(en.row0 + row) * a.q_ld +
                       (long)head * a.dim;
    #pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const int d = kk * 16 + hi * 8;
      qreg[kk] = d < a.dim ? *reinterpret_cast<const short8*>(qp + d)
                           : (short8){0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  float m = -INFINITY, l = 0.f;
  if (a.sink != nullptr && part_of == 0 && splits == 1) {
    m = a.sink[head] * LOG2E;
    l = 1.f;
  }
  float16v o_t[DC];
  #pragma unroll
  for (int c = 0; c < DC; ++c) o_t[c] = (float16v){};

  const float scale2 = a.scale * LOG2E;
  const float cap2 = a.cap * LOG2E;
  const float cscale = a.cap > 0.f ? 2.f * scale2 / a.cap : 0.f;
  int pgk[LK], pgv[LV];                          // page bases, -1: no key
  uint4 st_k[LK], st_v[LV];
  float st_b = 0.f;
  const float fall1 = a.r1 != nullptr ? a.r1[head] : 0.f;
  const float fall2 = a.r1 != nullptr ? a.r2[head] : 0.f;
  const float wb2 = KIND == SIGMOID ? a.wbias[head] * LOG2E : 0.f;

  auto pages = [&](int it) {
    const int st = part.at(it);
    #pragma unroll
    for (int i = 0; i < LK; ++i) {
      const int key = st * CH + (i * THREADS + tid) / (KK * 2);
      pgk[i] = it < part.n && key >= from && key < total &&
               key < st * CH + CH
          ? (FLAT ? key : bt[key / PAGE]) : -1;
    }
    #pragma unroll
    for (int i = 0; i < LV; ++i) {
      const int key = st * CH + (i * THREADS + tid) / (DC * 4);
      pgv[i] = it < part.n && key >= from && key < total &&
               key < st * CH + CH
          ? (FLAT ? key : bt[key / PAGE]) : -1;
    }
  };
  auto stage_load = [&](int it) {
    const int st = part.at(it);
    #pragma unroll
    for (int i = 0; i < LK; ++i) {
      const int f = i * THREADS + tid;
      const int r = f / (KK * 2), d = f % (KK * 2) * 8;
      st_k[i] = make_uint4(0, 0, 0, 0);
      if constexpr (FLAT) {
        const long at = flat0 + pgk[i];
        if (pgk[i] >= 0 && d < a.dim)
          st_k[i] = *reinterpret_cast<const uint4*>(
              d < kd ? a.kc + at * a.v_ld + (long)head * kd + d
                     : a.kr + at * a.shared + d - kd);
      } else if (pgk[i] >= 0 && d < a.dim)
        st_k[i] = *reinterpret_cast<const uint4*>(
            a.kc + (((long)pgk[i] * a.kv_heads + kvh) * PAGE +
                    (st * CH + r) % PAGE) * a.dim + d);
    }
    #pragma unroll
    for (int i = 0; i < LV; ++i) {
      const int f = i * THREADS + tid;
      const int r = f / (DC * 4), d = f % (DC * 4) * 8;
      st_v[i] = make_uint4(0, 0, 0, 0);
      if constexpr (FLAT) {
        if (pgv[i] >= 0 && d < a.vdim)
          st_v[i] = *reinterpret_cast<const uint4*>(
              a.vc + (flat0 + pgv[i]) * a.v_ld + (long)head * a.vdim + d);
      } else if (pgv[i] >= 0 && d < a.vdim)
        st_v[i] = *reinterpret_cast<const uint4*>(
            a.vc + (((long)pgv[i] * a.kv_heads + kvh) * PAGE +
                    (st * CH + r) % PAGE) * a.v_ld + d);
    }
    if (!FLAT && a.bias != nullptr)
      st_b = a.bias[(long)head * a.nbias +
                    min(max(qa0 - (st * CH + CH - 1) + tid, 0), a.nbias - 1)];
  };
  // nothing is worked out from what was loaded before this: it would be waited for
  // ahead of a step's products
  auto stage_write = [&](int it, int buf) {
    #pragma unroll
    for (int i = 0; i < LK; ++i) {
      const int f = i * THREADS + tid;
      const int r = f / (KK * 2), d = f % (KK * 2) * 8;
      if (r < CH) *reinterpret_cast<uint4*>(&s_k[buf][r][d]) = st_k[i];
    }
    #pragma unroll
    for (int i = 0; i < LV; ++i) {
      const int f = i * THREADS + tid;
      const int r = f / (DC * 4), col = f % (DC * 4) * 8;
      if (r < CH) {
        // bits 2 and 3 of the key exchanged
        const int kx = (r & 3) | (r & 4) << 1 | (r & 8) >> 1;
        const int ir = ((kx & 8) ? 8 : 0) + ((col % 32) / 16) * 4 + (kx & 3);
        *reinterpret_cast<uint4*>(
            &s_v[buf][col / 32][r / 32][(r % 32) / 16][(kx >> 2) & 1][ir]
                [col % 16]) = st_v[i];
      }
    }
    if constexpr (FLAT) return;                  // distances change nothing
    float b = st_b * LOG2E;
    if (a.r1 != nullptr) {
      const int n = qa0 - (part.at(it) * CH + CH - 1) + tid;
      b -= fall1 * __builtin_amdgcn_logf(1.f + fall2 * (float)max(n, 0));
    }
    if constexpr (KIND == SIGMOID) b += wb2;
    s_b[buf][tid] = b;
  };

  const int it0 = part.n * split / splits, it1 = part.n * (split + 1) / splits;
  pages(it0);
  stage_load(it0);
  pages(it0 + 1);
  stage_write(it0, 0);
  __syncthreads();

  for (int it = it0; it < it1; ++it) {
    const int cur = (it - it0) & 1;
    if (it + 1 < it1) {
      stage_load(it + 1);
      pages(it + 2);
    }
    const int kbase = part.at(it) * CH + part_of * NS * 32;
    if (wave_live && kbase <= hi_wave &&
        (kbase + NS * 32 > lo_wave || kbase < a.keep)) {
      const int sc0 = part_of * NS;
      float16v sacc[NS];
      #pragma unroll
      for (int sc = 0; sc < NS; ++sc) {
        sacc[sc] = (float16v){};
        #pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          const short8 ka = *reinterpret_cast<const short8*>(
              &s_k[cur][(sc0 + sc) * 32 + lo5][kk * 16 + hi * 8]);
          sacc[sc] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              ka, qreg[kk], sacc[sc], 0, 0, 0);
        }
      }
      float sv[NS][16];
      const float* bw =
          &s_b[cur][rw * 32 + lo5 + CH - 1 - 4 * hi - sc0 * 32];
      #pragma unroll
      for (int sc = 0; sc < NS; ++sc)
        #pragma unroll
        for (int r = 0; r < 16; ++r)
          sv[sc][r] = (KIND == CAP ? cap2 * tanh_exp2(sacc[sc][r] * cscale)
                                   : sacc[sc][r] * scale2) +
                      (FLAT ? 0.f : bw[-(sc * 32 + (r & 3) + 8 * (r >> 2))]);
      // steps inside every row's range need no mask
      if (kbase < lo_last || kbase + NS * 32 - 1 > qw0 || qw0 + 31 >= total) {
        #pragma unroll
        for (int sc = 0; sc < NS; ++sc)
          #pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int kpos =
                kbase + sc * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi;
            if (!(kpos <= qpos && (kpos >= lo || kpos < a.keep) &&
                  qpos < total))
              sv[sc][r] = -INFINITY;
          }
      }
      if constexpr (KIND != SIGMOID) {
        float mloc = -INFINITY;
        #pragma unroll
        for (int sc = 0; sc < NS; ++sc)
          #pragma unroll
          for (int r = 0; r < 16; ++r) mloc = fmaxf(mloc, sv[sc][r]);
        mloc = across<32>(mloc, Larger{});
        // the running maximum moves only when a score exceeds it by 2^8
        if (!__all(mloc == -INFINITY || mloc - m <= 8.f)) {
          const float mn = fmaxf(m, mloc);
          const float keep = m == -INFINITY ? 0.f
                                            : __builtin_amdgcn_exp2f(m - mn);
          m = mn;
          l *= keep;
          #pragma unroll
          for (int c = 0; c < DC; ++c)
            #pragma unroll
            for (int r = 0; r < 16; ++r) o_t[c][r] *= keep;
        }
      }
      // -inf less this is -inf: a weight of 0
      const float mf = m == -INFINITY ? 0.f : m;
      float sum = 0.f;
      #pragma unroll
      for (int sc = 0; sc < NS; ++sc) {
        #pragma unroll
        for (int g = 0; g < 2; ++g) {
          unsigned wh[4], wl[4];
          #pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float s0 = sv[sc][8 * g + 2 * i];
            const float s1 = sv[sc][8 * g + 2 * i + 1];
            float p0, p1;
            if constexpr (KIND == SIGMOID) {
              p0 = sigmoid_exp2(s0);
              p1 = sigmoid_exp2(s1);
            } else {
              p0 = __builtin_amdgcn_exp2f(s0 - mf);
              p1 = __builtin_amdgcn_exp2f(s1 - mf);
              sum += p0 + p1;
            }
            wh[i] = cvt_pk_bf16(p0, p1);
            const float2 back = unpack_bf16x2(wh[i]);
            wl[i] = cvt_pk_bf16(p0 - back.x, p1 - back.y);
          }
          const short8 ph = *reinterpret_cast<const short8*>(wh);
          const short8 pl = *reinterpret_cast<const short8*>(wl);
          #pragma unroll
          for (int c = 0; c < DC; ++c) {
            const short4v v0 =
                tr16_read(&s_v[cur][c][sc0 + sc][g][0][0][0] + lane * 4);
            const short4v v1 =
                tr16_read(&s_v[cur][c][sc0 + sc][g][1][0][0] + lane * 4);
            short8 vt;
            #pragma unroll
            for (int j = 0; j < 4; ++j) { vt[j] = v0[j]; vt[4 + j] = v1[j]; }
            o_t[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vt, ph, o_t[c],
                                                             0, 0, 0);
            o_t[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vt, pl, o_t[c],
                                                             0, 0, 0);
          }
        }
      }
      if constexpr (KIND != SIGMOID) l += across<32>(sum, Plus{});
    }
    if (it + 1 < it1) stage_write(it + 1, cur ^ 1);
    __syncthreads();
  }

  if constexpr (SH > 1) {
    // the second wave's sums join the first's, 32 columns at a time
    static_assert(SH == 2 && sizeof(s_k) >= RW * WAVE * 16 * sizeof(float) &&
                  sizeof(s_b) >= RW * WAVE * 2 * sizeof(float));
    float* s_o = reinterpret_cast<float*>(s_k) + rw * 16 * WAVE + lane;
    float* s_m = &s_b[0][0] + rw * 2 * WAVE + lane;
    float mine = 1.f, other = 1.f;
    if constexpr (KIND != SIGMOID) {
      if (part_of == 1) { s_m[0] = m; s_m[WAVE] = l; }
      __syncthreads();
      if (part_of == 0) {
        const float m1 = s_m[0], mn = fmaxf(m, m1);
        mine = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
        other = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - mn);
        l = l * mine + s_m[WAVE] * other;
        m = mn;
      }
    }
    #pragma unroll
    for (int c = 0; c < DC; ++c) {
      if (part_of == 1) {
        #pragma unroll
        for (int r = 0; r < 16; ++r) s_o[r * WAVE] = o_t[c][r];
      }
      __syncthreads();
      if (part_of == 0) {
        #pragma unroll
        for (int r = 0; r < 16; ++r)
          o_t[c][r] = o_t[c][r] * mine + s_o[r * WAVE] * other;
      }
      __syncthreads();
    }
  }

  if (wave_live && qpos < total && part_of == 0) {
    const long r = en.row0 + row;
    if (!FLAT && splits > 1) {
      const long at = (r * a.heads + head) * splits + split;
      #pragma unroll
      for (int c = 0; c < DC; ++c)
        #pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const int d0 = c * 32 + 8 * rr + 4 * hi;
          if (d0 >= a.vdim) continue;
          float o[4];
          #pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = o_t[c][rr * 4 + j];
          stv<4>(part_o + at * a.vdim + d0, o);
        }
      if (hi == 0 && KIND != SIGMOID) {
        part_ml[at * 2] = m;
        part_ml[at * 2 + 1] = l;
      }
      return;
    }
    float f = KIND == SIGMOID ? a.mult : a.mult / l;
    if (!(FLAT && a.gate_each) && a.gate != nullptr)
      f *= sigmoid_f(bf2f(a.gate[r * a.g_ld + head]));
    bf16_t* op = a.out + r * a.out_ld + (long)head * a.vdim;
    #pragma unroll
    for (int c = 0; c < DC; ++c) {
      #pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int d0 = c * 32 + 8 * rr + 4 * hi;
        if (d0 < a.vdim) {
          float o[4];
          #pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = o_t[c][rr * 4 + j] * f;
          if (FLAT && a.gate_each && a.gate != nullptr) {
            float g[4];
            ldv<4>(a.gate + r * a.g_ld + (long)head * a.vdim + d0, g);
            #pragma unroll
            for (int j = 0; j < 4; ++j) o[j] *= sigmoid_f(g[j]);
          }
          if (a.quads) {
            stv<4>(op + d0, o);
          } else {
            #pragma unroll
            for (int j = 0; j < 4; ++j) st1(op + d0 + j, o[j]);
          }
        }
      }
    }
  }
}

}  // namespace

bool attn_ctx_prefill_supported(int dim, int vdim, int block_size) {
  return dim % 8 == 0 && vdim % 8 == 0 && dim <= 256 && vdim <= 256 &&
         block_size == PAGE;
}

// Tiles of half the height, whose last of a portion is half full on average.
static long halves_of(int entries, long rows, int heads, int vdim) {
  return heads * (rows / (vdim <= 128 ? 128 : 64) + entries);
}

// Whether two waves share their rows. Tiles are half as high then, and as many again;
// the longest one's steps, one after another, are what a launch takes when the tiles
// are too few for the chip: with more than three quarters of the CUs at work the
// halves are no gain. us, MI355X, heads of 128, one wave and two: 900 rows x 16 heads
// (64 tiles) 67.0 and 49.5, portions of 900, 483 behind 1001, 741, 324 behind 1003
// (176) 109.1 and 77.9, 2900 rows (192) 172 and 138; 8 x 300 rows (256) 32.2 and 36.7,
// 6 x 2000 (768) 256 and 299. Heads of 64: 900 rows x 32 58.4 and 42.4, 4 x 500 behind
// 1500 (256) 125 and 133; of 256: 8 x 300 rows x 8 (192 tiles of 128) 49.7 and 40.2.
// Keys that are not paged are each head's own, and tiles of half the height read them
// twice as often: there more than half of the CUs at work are enough (keys of 192,
// six portions of up to 480 rows x 16, 192 tiles: 57.0 and 63.4).
// A step of 64 keys that is the only one is no chain, but 64 columns are few to add
// up: 58 rows of 128 x 64 heads 9.4 and 10.2, 14 of 64 x 4 heads 7.8 and 7.4. Behind a
// window chains are of one length, and a second round takes as long as the first; a CU
// has room for two workgroups of 64 columns, which make none: 2214 and 2682 rows of 256
// x 8 heads (288 and 336 tiles) 59.2 and 65.8, 55.2 and 68.5, 1973 of 64 x 16 (304) 88
// and 61.
bool attn_ctx_prefill_shared(int entries, long rows, int heads, int vdim,
                             int span, bool window, bool flat) {
  return halves_of(entries, rows, heads, vdim) <=
             (flat ? 256 : window && vdim > 64 ? 280 : 384) &&
         (vdim <= 64 || span > CH);
}

// Workgroups that share a tile's keys: those of few tiles, where a step of 64 keys takes
// 3 us and what follows (a launch, for the host, too; the shares' sums written and read)
// less than the steps saved; no more workgroups than CUs. us, MI355X, one and by
// shares, heads of 128, 16 of them: 100 rows behind 2000 96.1 and 29.5, 30 behind 3000
// 132 and 28.9, 500 behind 3500 170 and 65.7, 3 x 100 behind 600 41.3 and 28.0 (900
// rows, 49.8 and 41.3 by two shares, stay whole: the cost is a little high there);
// heads of 64, 32 of 8: 33.3 and 29.6 of 3 x 100; of 256, 8 of 1: 63.0 and 32.8.
int attn_ctx_prefill_splits(int entries, long rows, int heads, int vdim,
                            int span) {
  const int tile = vdim <= 128 ? 256 : 128;
  if (!attn_ctx_prefill_shared(entries, rows, heads, vdim, span, false, false))
    return 1;
  const long blocks = std::max(1L, heads * (4 * rows / tile + entries) / 2);
  const int steps = (span + CH - 1) / CH;
  auto cost = [&](long s) {
    return (steps + s - 1) / s * 3. +
           (s > 1 ? 14. + (double)rows * heads * s * vdim * (8 / 4e6) : 0.);
  };
  int best = 1;
  for (int s = 2; s <= 16 && blocks * s <= 256; ++s)
    if (cost(s) < cost(best)) best = s;
  return best;
}

// Where waves share rows workgroups are few, and go to XCDs, engines and CUs in turn.
// Those of an entry that has more rows than others, at equal distances with a power of
// two in them, would meet the same few CUs, which have two then while others have none:
// 127, 775, 127 and 127 rows of 256 x 8 heads 152 us. So an entry's come one after
// another (80 us), or, of more than CUs, whose longest should be the first of all,
// entries and one that there is not in turn, if they are even in number.
void launch_attn_ctx_prefill(const AttnCtx<bf16_t>& given, int entries,
                             long rows, int max_len, int span, int splits,
                             float* part_o, float* part_ml,
                             hipStream_t stream) {
  AttnCtx<bf16_t> a = given;
  a.entries = entries;
  a.by_entry = halves_of(entries, rows, a.heads, a.vdim) <= 256;
  auto with = [&](auto kk, auto dc, auto waves, auto sh) {
    constexpr int W = decltype(waves)::value, SH = decltype(sh)::value;
    constexpr int K = decltype(kk)::value, D = decltype(dc)::value;
    const int tiles = (max_len + W / SH * 32 - 1) / (W / SH * 32) * splits;
    // none of no rows or entries: such a launch is refused
    const int odd = tiles | (tiles > 0 && entries > 1);
    const dim3 grid =
        SH == 1      ? dim3(entries, a.heads, tiles)
        : a.by_entry ? dim3(a.heads, odd, entries)
                     : dim3(a.heads, entries > 0 ? entries | 1 : 0, tiles);
    const dim3 block(W * WAVE);
    if (a.ctx_start != nullptr)
      attn_ctx_prefill_kernel<K, D, W, SH, true, PLAIN>
          <<<grid, block, 0, stream>>>(a, splits, part_o, part_ml);
    else if (a.wbias != nullptr)
      attn_ctx_prefill_kernel<K, D, W, SH, false, SIGMOID>
          <<<grid, block, 0, stream>>>(a, splits, part_o, part_ml);
    else if (a.cap > 0.f)
      attn_ctx_prefill_kernel<K, D, W, SH, false, CAP>
          <<<grid, block, 0, stream>>>(a, splits, part_o, part_ml);
    else
      attn_ctx_prefill_kernel<K, D, W, SH, false, PLAIN>
          <<<grid, block, 0, stream>>>(a, splits, part_o, part_ml);
  };
  auto go = [&](auto kk, auto dc, auto waves) {
    if (splits > 1 ||
        attn_ctx_prefill_shared(entries, rows, a.heads, a.vdim, span,
                                a.window > 0 && a.window + a.keep <= span,
                                a.ctx_start != nullptr))
      with(kk, dc, waves, std::integral_constant<int, 2>{});
    else
      with(kk, dc, waves, std::integral_constant<int, 1>{});
  };
  using std::integral_constant;
  auto by_dc = [&](auto kk) {
    if (a.vdim <= 64)
      go(kk, integral_constant<int, 2>{}, integral_constant<int, 8>{});
    else if (a.vdim <= 128)
      go(kk, integral_constant<int, 4>{}, integral_constant<int, 8>{});
    else
      go(kk, integral_constant<int, 8>{}, integral_constant<int, 4>{});
  };
  if (a.dim <= 64) by_dc(integral_constant<int, 4>{});
  else if (a.dim <= 96) by_dc(integral_constant<int, 6>{});
  else if (a.dim <= 128) by_dc(integral_constant<int, 8>{});
  else if (a.dim <= 192) by_dc(integral_constant<int, 12>{});
  else by_dc(integral_constant<int, 16>{});
}
