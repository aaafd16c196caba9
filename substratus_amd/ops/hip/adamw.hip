// Fused AdamW: m/v update + decoupled weight decay + bias-corrected param
// update in one pass. bf16 params and grads, fp32 optimizer state; pure HBM
// streaming (reads p,g,m,v; writes p,m,v → 12 B in / 10 B out per element).
// Up to 40 tensors a launch: a model's small tensors cost a launch each
// otherwise, 5 us on a MI355X for a norm's weights.
//
// gscale folds gradient clipping into the update (g := g * gscale), so the
// trainer never runs a separate foreach_mul over every grad (~10 ms/step at
// falcon-7b scale). It may be given as the gradients' norm on the device,
// which no one has to wait for.
// 1.12e9 parameters in 27 tensors on a MI355X: 27 launches 4.97 ms, this one
// 4.75 ms (5.2 TB/s).
#include "common.h"
#include "optimizer.h"
#include <algorithm>
#include <vector>

namespace {

constexpr int OPT_BLOCK = 256;
constexpr long ADAMW_CHUNK = 8192;    // elements a workgroup
constexpr long NORM_CHUNK = 32768;

DEV_INLINE const OptTensor& tensor_of(const OptTensors& all) {
  int i = 0;
  while (i + 1 < all.count && (int)blockIdx.x >= all.t[i + 1].block) ++i;
  return all.t[i];
}

}  // namespace

// min(1, clip / (norm + 1e-6)) in 64 bits; 1 where the norm is no number
DEV_INLINE float clip_scale(const float* norm, double clip) {
  const double s = clip / ((double)*norm + 1e-6);
  return s < 1.0 ? (float)s : 1.f;
}

__global__ __launch_bounds__(OPT_BLOCK) void adamw_kernel(
    OptTensors all, float lr, float beta1, float beta2, float eps, float wd,
    float bc1, float bc2, float gscale, const float* __restrict__ norm,
    double clip) {
  const OptTensor& at = tensor_of(all);
  const long lo = ((int)blockIdx.x - at.block) * ADAMW_CHUNK;
  const long n = min(at.n - lo, ADAMW_CHUNK), n4 = n / 4;
  bf16_t* p = reinterpret_cast<bf16_t*>(at.p) + lo;
  const bf16_t* g = reinterpret_cast<const bf16_t*>(at.g) + lo;
  float* m = at.m + lo;
  float* v = at.v + lo;
  if (norm) gscale = clip_scale(norm, clip);
  uint2* p2 = reinterpret_cast<uint2*>(p);
  const uint2* g2 = reinterpret_cast<const uint2*>(g);
  float4* m4 = reinterpret_cast<float4*>(m);
  float4* v4 = reinterpret_cast<float4*>(v);
  #pragma unroll 2
  for (int i = threadIdx.x; i < n4; i += OPT_BLOCK) {
    uint2 pu = p2[i], gu = g2[i];
    float2 pf0 = unpack_bf16x2(pu.x), pf1 = unpack_bf16x2(pu.y);
    float2 gf0 = unpack_bf16x2(gu.x), gf1 = unpack_bf16x2(gu.y);
    float4 mf = m4[i], vf = v4[i];
    float pv[4] = {pf0.x, pf0.y, pf1.x, pf1.y};
    float gv[4] = {gf0.x * gscale, gf0.y * gscale,
                   gf1.x * gscale, gf1.y * gscale};
    float mv[4] = {mf.x, mf.y, mf.z, mf.w};
    float vv[4] = {vf.x, vf.y, vf.z, vf.w};
    #pragma unroll
    for (int j = 0; j < 4; ++j) {
      mv[j] = beta1 * mv[j] + (1.f - beta1) * gv[j];
      vv[j] = beta2 * vv[j] + (1.f - beta2) * gv[j] * gv[j];
      float denom = sqrtf(vv[j] / bc2) + eps;
      pv[j] = pv[j] * (1.f - lr * wd) - lr * (mv[j] / bc1) / denom;
    }
    m4[i] = make_float4(mv[0], mv[1], mv[2], mv[3]);
    v4[i] = make_float4(vv[0], vv[1], vv[2], vv[3]);
    p2[i].x = pack_bf16x2(pv[0], pv[1]);
    p2[i].y = pack_bf16x2(pv[2], pv[3]);
  }
  // tail
  for (int i = n4 * 4 + threadIdx.x; i < n; i += OPT_BLOCK) {
    float gj = bf2f(g[i]) * gscale;
    float mj = beta1 * m[i] + (1.f - beta1) * gj;
    float vj = beta2 * v[i] + (1.f - beta2) * gj * gj;
    m[i] = mj; v[i] = vj;
    float pj = bf2f(p[i]) * (1.f - lr * wd) -
               lr * (mj / bc1) / (sqrtf(vj / bc2) + eps);
    p[i] = f2bf(pj);
  }
}

// Sums of squares, a share per workgroup: 2.2 GB of gradients in
// 27 tensors, MI355X: torch's norms 1.09 ms in 54 launches, this 0.38 ms (5.9
// TB/s) in one; 0.34 and 0.14 ms for 0.7 GB.
__global__ __launch_bounds__(OPT_BLOCK) void square_sum_kernel(
    float* __restrict__ shares, OptTensors all) {
  __shared__ float scratch[OPT_BLOCK / WAVE];
  const OptTensor& at = tensor_of(all);
  const long lo = ((int)blockIdx.x - at.block) * NORM_CHUNK;
  const long n = min(at.n - lo, NORM_CHUNK);
  const bf16_t* g = reinterpret_cast<const bf16_t*>(at.g) + lo;
  const uint4* gv = reinterpret_cast<const uint4*>(g);
  float s = 0.f;
  #pragma unroll 4
  for (int i = threadIdx.x; i < n / 8; i += OPT_BLOCK) {
    const uint4 u = gv[i];
    const unsigned int w[4] = {u.x, u.y, u.z, u.w};
    #pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float2 f = unpack_bf16x2(w[j]);
      s += f.x * f.x + f.y * f.y;
    }
  }
  for (int i = n / 8 * 8 + threadIdx.x; i < n; i += OPT_BLOCK) {
    const float f = bf2f(g[i]);
    s += f * f;
  }
  s = block_sum<OPT_BLOCK / WAVE>(s, scratch);
  if (threadIdx.x == 0) shares[blockIdx.x] = s;
}

// The root of all shares' sum, in 64 bits, by one workgroup.
__global__ __launch_bounds__(1024) void norm_kernel(
    float* __restrict__ norm, const float* __restrict__ shares, long n) {
  __shared__ double part[1024 / WAVE];
  double s = 0.;
  for (long i = threadIdx.x; i < n; i += 1024) s += (double)shares[i];
  #pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, WAVE);
  if (threadIdx.x % WAVE == 0) part[threadIdx.x / WAVE] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < 1024 / WAVE; ++i) s += part[i];
    *norm = (float)sqrt(s);
  }
}

// fp32-param variant (small models / master weights).
__global__ void adamw_kernel_f32(float* __restrict__ p,
                                 const float* __restrict__ g,
                                 float* __restrict__ m, float* __restrict__ v,
                                 long n, float lr, float beta1, float beta2,
                                 float eps, float wd, float bc1, float bc2,
                                 float gscale) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n;
       i += (long)gridDim.x * blockDim.x) {
    float gj = g[i] * gscale;
    float mj = beta1 * m[i] + (1.f - beta1) * gj;
    float vj = beta2 * v[i] + (1.f - beta2) * gj * gj;
    m[i] = mj; v[i] = vj;
    p[i] = p[i] * (1.f - lr * wd) - lr * (mj / bc1) / (sqrtf(vj / bc2) + eps);
  }
}

namespace {

// go(tensors, workgroups) for launches of OPT_MOST tensors
template <class F>
void by_launch(const std::vector<OptTensor>& given, long chunk, F go) {
  OptTensors all;
  all.count = 0;
  long blocks = 0;
  for (size_t i = 0; i < given.size(); ++i) {
    const long more = (given[i].n + chunk - 1) / chunk;
    // a launch's threads are counted in 32 bits
    const bool full = all.count == OPT_MOST ||
                      (all.count > 0 && blocks + more > (1L << 23));
    if (full) {
      go(all, blocks);
      all.count = 0;
      blocks = 0;
    }
    if (more == 0) continue;
    all.t[all.count] = given[i];
    all.t[all.count++].block = (int)blocks;
    blocks += more;
  }
  if (all.count) go(all, blocks);
}

}  // namespace

void launch_adamw(const std::vector<OptTensor>& given, float lr, float beta1,
                  float beta2, float eps, float wd, int step, float gscale,
                  const float* norm, double clip, hipStream_t stream) {
  float bc1 = 1.f - powf(beta1, (float)step);
  float bc2 = 1.f - powf(beta2, (float)step);
  by_launch(given, ADAMW_CHUNK, [&](const OptTensors& all, long blocks) {
    adamw_kernel<<<dim3(blocks), dim3(OPT_BLOCK), 0, stream>>>(
        all, lr, beta1, beta2, eps, wd, bc1, bc2, gscale, norm, clip);
  });
}

long grad_norm_shares(const std::vector<OptTensor>& given) {
  long n = 0;
  for (const OptTensor& t : given) n += (t.n + NORM_CHUNK - 1) / NORM_CHUNK;
  return n;
}

void launch_grad_norm(float* norm, float* shares,
                      const std::vector<OptTensor>& given,
                      hipStream_t stream) {
  long done = 0;
  by_launch(given, NORM_CHUNK, [&](const OptTensors& all, long blocks) {
    square_sum_kernel<<<dim3(blocks), dim3(OPT_BLOCK), 0, stream>>>(
        shares + done, all);
    done += blocks;
  });
  norm_kernel<<<dim3(1), dim3(1024), 0, stream>>>(norm, shares, done);
}

void launch_adamw_f32(float* p, const float* g, float* m, float* v, long n,
                      float lr, float beta1, float beta2, float eps, float wd,
                      int step, float gscale, hipStream_t stream) {
  float bc1 = 1.f - powf(beta1, (float)step);
  float bc2 = 1.f - powf(beta2, (float)step);
  int grid = (int)std::min((n + 255) / 256, (long)8192);
  adamw_kernel_f32<<<dim3(std::max(grid, 1)), dim3(256), 0, stream>>>(
      p, g, m, v, n, lr, beta1, beta2, eps, wd, bc1, bc2, gscale);
}
