// Common CDNA4 (gfx950) kernel helpers.
//
// Wave width is 64 on CDNA4 (guide §1) — hard-coded; every warp-style idiom
// below is 64-wide. bf16 data moves as packed uint/uint4 (8×bf16 = 16 B per
// lane per load) for full coalescing (guide §5 common-mistake #2).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#define WAVE 64
#define DEV_INLINE __device__ __forceinline__

typedef __hip_bfloat16 bf16_t;

// clang ext_vector (not HIP_vector_type) — required by
// __builtin_nontemporal_load, which rejects class types.
typedef __attribute__((ext_vector_type(4))) unsigned int uint4v;

DEV_INLINE uint4v nt_load_u4(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const uint4v*>(p));
}

typedef __attribute__((ext_vector_type(2))) unsigned int uint2v;

DEV_INLINE uint2v nt_load_u2(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const uint2v*>(p));
}

// OCP fp8 e4m3 <-> f32 via the gfx950 hardware converts (OCP semantics on
// gfx950 — matches torch.float8_e4m3fn).
template <int SEL>
DEV_INLINE float fp8_to_f32(unsigned int word) {
  return __builtin_amdgcn_cvt_f32_fp8(word, SEL);  // sel must be constant
}

DEV_INLINE unsigned char f32_to_fp8(float x) {
  return (unsigned char)(__builtin_amdgcn_cvt_pk_fp8_f32(x, x, 0, false) &
                         0xFF);
}

DEV_INLINE float bf2f(bf16_t x) { return __bfloat162float(x); }
DEV_INLINE bf16_t f2bf(float x) { return __float2bfloat16(x); }

// Unpack a uint holding 2 bf16 into 2 floats.
DEV_INLINE float2 unpack_bf16x2(unsigned int u) {
  float2 r;
  r.x = __uint_as_float((u & 0xffffu) << 16);
  r.y = __uint_as_float(u & 0xffff0000u);
  return r;
}

DEV_INLINE unsigned int pack_bf16x2(float lo, float hi) {
  bf16_t a = f2bf(lo), b = f2bf(hi);
  unsigned short ua = *reinterpret_cast<unsigned short*>(&a);
  unsigned short ub = *reinterpret_cast<unsigned short*>(&b);
  return (unsigned int)ua | ((unsigned int)ub << 16);
}

// --- wave-level reductions (64 lanes) -------------------------------------
// op, which is symmetric, of a lane's number and that of the lane OFF away: by
// moves between registers, where __shfl_xor goes through LDS. 4 away only where
// lanes 8 away have equal numbers (a row of 16 lanes turned by four). Lanes must
// be there: all of a wave for 32 and 16, of a row of 16 for the others. ns of a
// sum over a wave that waits for the one before it: 178 -> 52.
template <int OFF, class Op>
DEV_INLINE float across(float v, Op op) {
  const unsigned u = __float_as_uint(v);
  if constexpr (OFF == 32) {
    const auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return op(__uint_as_float(s[0]), __uint_as_float(s[1]));
  } else if constexpr (OFF == 16) {
    const auto s = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return op(__uint_as_float(s[0]), __uint_as_float(s[1]));
  } else {
    static_assert(OFF == 8 || OFF == 4 || OFF == 2 || OFF == 1);
    constexpr int CTRL = OFF == 8 ? 0x128       // row_ror 8
                       : OFF == 4 ? 0x124       // row_ror 4
                       : OFF == 2 ? 0x4e        // quad_perm 2 3 0 1
                                  : 0xb1;       // quad_perm 1 0 3 2
    return op(v, __uint_as_float(__builtin_amdgcn_update_dpp(
                     0u, u, CTRL, 0xf, 0xf, true)));
  }
}

// The number of the lane OFF away.
template <int OFF>
DEV_INLINE float from_lane(float v) {
  const unsigned u = __float_as_uint(v);
  if constexpr (OFF >= 16) {
    static_assert(OFF == 32 || OFF == 16);
    const bool up = threadIdx.x & OFF;
    if constexpr (OFF == 32) {
      const auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false);
      return __uint_as_float(up ? s[0] : s[1]);
    } else {
      const auto s = __builtin_amdgcn_permlane16_swap(u, u, false, false);
      return __uint_as_float(up ? s[0] : s[1]);
    }
  } else if constexpr (OFF == 4) {              // 7 away, of which 3 back
    const unsigned t =
        __builtin_amdgcn_update_dpp(0u, u, 0x141, 0xf, 0xf, true);
    return __uint_as_float(
        __builtin_amdgcn_update_dpp(0u, t, 0x1b, 0xf, 0xf, true));
  } else {
    constexpr int CTRL = OFF == 8 ? 0x128 : OFF == 2 ? 0x4e : 0xb1;
    static_assert(OFF == 8 || OFF == 2 || OFF == 1);
    return __uint_as_float(
        __builtin_amdgcn_update_dpp(0u, u, CTRL, 0xf, 0xf, true));
  }
}

struct Plus {
  DEV_INLINE float operator()(float a, float b) const { return a + b; }
};
struct Larger {
  DEV_INLINE float operator()(float a, float b) const { return fmaxf(a, b); }
};

// Of the lanes FROM, 2 FROM and so on to 32 away, in this order.
template <int FROM, class Op>
DEV_INLINE float across_from(float v, Op op) {
  static_assert(FROM == 8 || FROM == 16 || FROM == 32);
  if constexpr (FROM == 8) v = across<8>(v, op);
  if constexpr (FROM <= 16) v = across<16>(v, op);
  return across<32>(v, op);
}

// Within 16-lane groups (used by 16-lanes-per-token layouts).
template <class Op>
DEV_INLINE float group16(float v, Op op) {
  return across<1>(across<2>(across<4>(across<8>(v, op), op), op), op);
}

DEV_INLINE float group16_sum(float v) { return group16(v, Plus{}); }

template <class Op>
DEV_INLINE float wave_all(float v, Op op) {
  return group16(across<16>(across<32>(v, op), op), op);
}

DEV_INLINE float wave_sum(float v) { return wave_all(v, Plus{}); }
DEV_INLINE float wave_max(float v) { return wave_all(v, Larger{}); }

// --- block-level reductions over NW waves via LDS --------------------------
// Caller provides __shared__ float scratch[NW]; result valid in all threads.
template <int NW>
DEV_INLINE float block_sum(float v, float* scratch) {
  int wave = threadIdx.x / WAVE;
  v = wave_sum(v);
  if ((threadIdx.x & (WAVE - 1)) == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
  #pragma unroll
  for (int i = 0; i < NW; ++i) total += scratch[i];
  return total;
}

template <int NW>
DEV_INLINE float block_max(float v, float* scratch) {
  int wave = threadIdx.x / WAVE;
  v = wave_max(v);
  if ((threadIdx.x & (WAVE - 1)) == 0) scratch[wave] = v;
  __syncthreads();
  float m = -INFINITY;
  #pragma unroll
  for (int i = 0; i < NW; ++i) m = fmaxf(m, scratch[i]);
  return m;
}

// v / 2 (1 + tanh(t)) is v / (1 + exp(-2 t)): a fraction of tanhf's instructions,
// and nothing is lost where 1 + tanh(t) is all but zero. Over all bf16 numbers up
// to 20 the largest relative error after rounding was 1 (zeros for numbers), is
// 0.00386, half a step. At the end of a product of 4165 x 18176 x 4544 tanhf took
// 48 us, this 37; gelu by itself of its result 80, 66.
DEV_INLINE float gelu_of(float v) {
  const float c = 2.f * 0.7978845608028654f;  // 2 sqrt(2/pi)
  return v / (1.f + __expf(-c * (v + 0.044715f * v * v * v)));
}

#define HIP_CHECK_KERNEL()                                            \
  do {                                                                \
    hipError_t e_ = hipGetLastError();                                \
    if (e_ != hipSuccess)                                             \
      TORCH_CHECK(false, "HIP kernel launch failed: ", hipGetErrorString(e_)); \
  } while (0)
