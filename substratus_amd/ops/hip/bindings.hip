// Python bindings for the CDNA4 HIP kernel library (substratus_amd._C).
// Validation lives here; kernels are thin and trusting.
#include <torch/extension.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/cuda/CUDAContext.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/core/DeviceGuard.h>
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include "optimizer.h"
#include "rows_quant.h"
#include "mid_gemm.h"
#include "tile_gemm.h"

typedef __hip_bfloat16 bf16_t;

// launchers (defined in the .hip translation units)
void launch_rms_norm(bf16_t*, const bf16_t*, const bf16_t*, long, int, float, hipStream_t);
void launch_rms_norm_residual(bf16_t*, bf16_t*, const bf16_t*, const bf16_t*, long, int, float, hipStream_t);
void launch_layer_norm(bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*, long, int, float, hipStream_t);
void launch_silu_mul(bf16_t*, const bf16_t*, long, int, hipStream_t);
void launch_gelu(bf16_t*, const bf16_t*, long, hipStream_t);
void launch_rope_kv_append(bf16_t*, bf16_t*, const bf16_t*, const int*, void*, void*, const int*, int, int, int, int, int, float, bool, long, long, long, hipStream_t);
void launch_rope_split_append(bf16_t*, bf16_t*, bf16_t*, const bf16_t*, const int*, void*, void*, const int*, long, int, int, int, int, float, bool, hipStream_t);
void launch_paged_attn_decode(bf16_t*, const bf16_t*, const void*, const void*, const int*, const int*, int, int, int, int, int, int, float, long, int, float*, float*, bool, bool, int, hipStream_t);
bool paged_attn_grouped(int, int, int, long, const void*, const void*, const void*, bool);
int paged_attn_plan(int, int, int, int, int, bool, int&);
bool paged_attn_decode_supported(int, int);
void launch_attn_prefill(bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*, const int*, int, int, int, int, int, float, hipStream_t, float*);
bool attn_prefill_supported(int);
void launch_attn_v5(bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*, const int*, int, int, int, int, int, float, hipStream_t, float*);
bool attn_v5_supported(int);
void launch_attn_bwd_dq(bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*, const float*, const float*, const int*, int, int, int, int, int, float, hipStream_t);
void launch_attn_bwd_dkv(float*, float*, const bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*, const float*, const float*, const int*, int, int, int, int, int, float, hipStream_t);
void launch_attn_bwd_delta(float*, const bf16_t*, const bf16_t*, long, int, hipStream_t);
bool attn_bwd_supported(int);
void launch_attn_prefill_probe(int, bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*, const int*, int, int, int, int, float, hipStream_t);
void launch_mfma_probe(float*, const bf16_t*, const bf16_t*, hipStream_t);
void launch_mfma32_probe(float*, const bf16_t*, const bf16_t*, hipStream_t);
bool train_norm_takes(int);
int train_norm_shares(long);
void launch_add_norm_fwd(bf16_t*, bf16_t*, float*, const bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*, long, int, float, bool, hipStream_t);
void launch_add_norm_bwd(bf16_t*, bf16_t*, bf16_t*, float*, const bf16_t*, const bf16_t*, const bf16_t*, const float*, const bf16_t*, long, int, bool, hipStream_t);
void launch_rope_split(bf16_t*, bf16_t*, bf16_t*, const bf16_t*, const float*, const float*, long, int, int, int, int, hipStream_t);
void launch_rope_join(bf16_t*, const bf16_t*, const float*, const float*, const float*, const float*, long, int, int, int, int, hipStream_t);
void launch_lookup_bwd(bf16_t*, unsigned char*, const bf16_t*, const long*, int, long, int, hipStream_t);
void launch_silu_mul_bwd(bf16_t*, const bf16_t*, const bf16_t*, long, int, hipStream_t);
void launch_softmax_sample(long*, const bf16_t*, const float*, const int*, const float*, const float*, int, int, hipStream_t);
void launch_softmax_sample(long*, const float*, const float*, const int*, const float*, const float*, int, int, hipStream_t);
void launch_cross_entropy(float*, bf16_t*, const bf16_t*, const long*, long, int, long, float*, hipStream_t);
void launch_adamw(const std::vector<OptTensor>&, float, float, float, float, float, int, float, const float*, double, hipStream_t);
long grad_norm_shares(const std::vector<OptTensor>&);
void launch_grad_norm(float*, float*, const std::vector<OptTensor>&, hipStream_t);
void launch_adamw_f32(float*, const float*, float*, float*, long, float, float, float, float, float, int, float, hipStream_t);
void launch_quant_gemv(bf16_t*, const bf16_t*, const void*, const unsigned char*, int, int, int, bool, hipStream_t);
bool rows_gemm_takes(int, int, int, bool);
bool rows_gemm_pays(int, int, int, bool);
void launch_dequant(bf16_t*, const void*, const unsigned char*, long, int, bool, hipStream_t);
void launch_dequant_k(bf16_t*, const void*, const unsigned char*, int, int, bool, hipStream_t);
int decode_gemm_splitk(int, int);
bool decode_gemm_supported(int, int, int);
void launch_decode_gemm(bf16_t*, const bf16_t*, const bf16_t*, float*, int, int, int, int, hipStream_t);
int mfma_gemm_splitk(int, int, int);
bool mfma_gemm_supported(int, int, int);
void launch_mfma_gemm(bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*, float*, int, int, int, int, hipStream_t);
int wstream_splitk(int, int);
bool wstream_supported(int, int, int);
void launch_wstream_gemm(bf16_t*, const bf16_t*, const bf16_t*, float*, int, int, int, int, hipStream_t);

namespace {

// The current device's; of products and training ops, which torch's own do on
// whatever device their operands are, the operands' (a guard in each).
inline hipStream_t stream() {
  return at::cuda::getCurrentCUDAStream().stream();
}

inline bf16_t* bf(torch::Tensor& t) {
  return reinterpret_cast<bf16_t*>(t.data_ptr<at::BFloat16>());
}
inline const bf16_t* bfc(const torch::Tensor& t) {
  return reinterpret_cast<const bf16_t*>(t.data_ptr<at::BFloat16>());
}

// [ntok, h, d] tensors may be views of a fused qkv projection: inner two
// dims contiguous, token-row stride arbitrary (saves the decode path three
// elementwise copies per layer)
void check_bf16_rows(const torch::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), name, " must be on GPU");
  TORCH_CHECK(t.scalar_type() == torch::kBFloat16, name, " must be bf16");
  TORCH_CHECK(t.dim() == 3 && t.stride(2) == 1 &&
                  t.stride(1) == t.size(2),
              name, " must be [n, h, d] with contiguous rows");
}

void check_bf16(const torch::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), name, " must be on GPU");
  TORCH_CHECK(t.scalar_type() == torch::kBFloat16, name, " must be bf16");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}

bool aligned16(const torch::Tensor& t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

void post_launch_check(const char* op) {
  hipError_t e = hipGetLastError();
  TORCH_CHECK(e == hipSuccess, op, ": HIP launch failed: ", hipGetErrorString(e));
}

// Whether values are all that is asked of an op on these (None among them): 2; 1
// but for function modes; 0. Asked for every product and by every backward: 0.7
// us here, 1.4 (6.5 the first time in a thread) in Python.
int plain_tensors(const py::args& tensors) {
  using c10::DispatchKey;
  constexpr c10::DispatchKeySet wrapped({
      DispatchKey::Python, DispatchKey::Batched, DispatchKey::FuncTorchBatched,
      DispatchKey::FuncTorchGradWrapper, DispatchKey::Functionalize});
  for (const auto& o : tensors) {
    if (o.is_none()) continue;
    if (!THPVariable_CheckExact(o.ptr())) return 0;
    const at::Tensor& t = THPVariable_Unpack(o.ptr());
    if (t.layout() != at::kStrided || t.key_set().has_any(wrapped) ||
        (t.key_set().has(DispatchKey::ADInplaceOrView) &&
         t._fw_grad(0).defined()))
      return 0;
  }
  if (at::autocast::is_autocast_enabled(at::kCUDA) ||
      torch::jit::tracer::isTracing() ||
      c10::impl::tls_is_dispatch_key_included(
          DispatchKey::FuncTorchDynamicLayerFrontMode) ||
      c10::impl::TorchDispatchModeTLS::any_modes_set())
    return 0;
  return at::impl::PythonTorchFunctionTLS::stack_len() > 0 ? 1 : 2;
}

// bf16, contiguous, of n elements and on 16-byte boundaries
void check_rows(const torch::Tensor& t, long n, const char* name) {
  check_bf16(t, name);
  TORCH_CHECK(t.numel() == n, name, " has ", t.numel(), " elements, not ", n);
  TORCH_CHECK(aligned16(t), name, " must be on a 16-byte boundary");
}

void check_rows32(const torch::Tensor& t, long n, const char* name) {
  TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kFloat &&
                  t.is_contiguous() && aligned16(t) && t.numel() == n,
              name, " must be ", n, " contiguous floats on GPU");
}

// y = norm(h + d1 + d2), sum = h + d1 + d2 (d1, d2 and with them sum may be
// absent; without bias it is RMS)
void add_norm_fwd(torch::Tensor y, c10::optional<torch::Tensor> sum,
                  torch::Tensor stats, torch::Tensor h,
                  c10::optional<torch::Tensor> d1,
                  c10::optional<torch::Tensor> d2, torch::Tensor w,
                  c10::optional<torch::Tensor> b, double eps) {
  const c10::DeviceGuard guard(h.device());
  const long n = h.numel(), hidden = w.numel();
  TORCH_CHECK(n > 0 && train_norm_takes(hidden) && n % hidden == 0,
              "width ", hidden, " not taken");
  check_rows(y, n, "y"); check_rows(h, n, "h"); check_rows(w, hidden, "w");
  TORCH_CHECK(d1.has_value() == sum.has_value() && (d1 || !d2), "operands");
  if (d1) { check_rows(*d1, n, "d1"); check_rows(*sum, n, "sum"); }
  if (d2) check_rows(*d2, n, "d2");
  if (b) check_rows(*b, hidden, "b");
  check_rows32(stats, 2 * (n / hidden), "stats");
  launch_add_norm_fwd(bf(y), sum ? bf(*sum) : nullptr,
                      stats.data_ptr<float>(), bfc(h), d1 ? bfc(*d1) : nullptr,
                      d2 ? bfc(*d2) : nullptr, bfc(w), b ? bfc(*b) : nullptr,
                      n / hidden, hidden, (float)eps, !b, stream());
  post_launch_check("add_norm_fwd");
}

// db tells LayerNorm from RMS
void add_norm_bwd(torch::Tensor dh, torch::Tensor dw,
                  c10::optional<torch::Tensor> db, torch::Tensor dy,
                  c10::optional<torch::Tensor> dres, torch::Tensor x,
                  torch::Tensor stats, torch::Tensor w) {
  const c10::DeviceGuard guard(x.device());
  const long n = x.numel(), hidden = w.numel();
  TORCH_CHECK(n > 0 && train_norm_takes(hidden) && n % hidden == 0,
              "width ", hidden, " not taken");
  check_rows(dh, n, "dh"); check_rows(dy, n, "dy"); check_rows(x, n, "x");
  check_rows(w, hidden, "w"); check_rows(dw, hidden, "dw");
  if (dres) check_rows(*dres, n, "dres");
  if (db) check_rows(*db, hidden, "db");
  check_rows32(stats, 2 * (n / hidden), "stats");
  auto shares = torch::empty(
      {(db ? 2 : 1) * train_norm_shares(n / hidden) * hidden},
      stats.options());
  launch_add_norm_bwd(bf(dh), bf(dw), db ? bf(*db) : nullptr,
                      shares.data_ptr<float>(), bfc(dy),
                      dres ? bfc(*dres) : nullptr, bfc(x),
                      stats.data_ptr<float>(), bfc(w), n / hidden, hidden,
                      !db, stream());
  post_launch_check("add_norm_bwd");
}

void check_angles(const c10::optional<torch::Tensor>& c,
                  const c10::optional<torch::Tensor>& s, long rows,
                  long length, long d) {
  // a head's threads have to divide a workgroup's
  TORCH_CHECK(d == 16 || d == 32 || d == 64 || d == 128 || d == 256,
              "head_dim ", d, " not taken");
  TORCH_CHECK(rows > 0 && length > 0 && rows % length == 0, "rows");
  TORCH_CHECK(c.has_value() == s.has_value(), "angles");
  if (c) {
    check_rows32(*c, length * (d / 2), "cos");
    check_rows32(*s, length * (d / 2), "sin");
  }
}

// qkv rows into q, k, v, turned by the angles of row % length (none: copied)
void rope_split(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                torch::Tensor qkv, c10::optional<torch::Tensor> c,
                c10::optional<torch::Tensor> s, long length) {
  const c10::DeviceGuard guard(qkv.device());
  TORCH_CHECK(q.dim() == 3 && k.dim() == 3, "q, k are [rows, heads, d]");
  const long rows = q.size(0), hq = q.size(1), hkv = k.size(1), d = q.size(2);
  check_angles(c, s, rows, length, d);
  check_rows(q, rows * hq * d, "q"); check_rows(k, rows * hkv * d, "k");
  check_rows(v, rows * hkv * d, "v");
  check_rows(qkv, rows * (hq + 2 * hkv) * d, "qkv");
  launch_rope_split(bf(q), bf(k), bf(v), bfc(qkv),
                    c ? c->data_ptr<float>() : nullptr,
                    s ? s->data_ptr<float>() : nullptr, rows, length, hq, hkv,
                    d, stream());
  post_launch_check("rope_split");
}

void rope_join(torch::Tensor dqkv, torch::Tensor dq, torch::Tensor dk,
               torch::Tensor dv, c10::optional<torch::Tensor> c,
               c10::optional<torch::Tensor> s, long length) {
  const c10::DeviceGuard guard(dqkv.device());
  TORCH_CHECK(dq.dim() == 3 && dk.dim() == 3, "q, k are [rows, heads, d]");
  const long rows = dq.size(0), hq = dq.size(1), hkv = dk.size(1);
  const long d = dq.size(2);
  check_angles(c, s, rows, length, d);
  check_rows(dq, rows * hq * d, "dq");
  check_rows32(dk, rows * hkv * d, "dk");
  check_rows32(dv, rows * hkv * d, "dv");
  check_rows(dqkv, rows * (hq + 2 * hkv) * d, "dqkv");
  launch_rope_join(bf(dqkv), bfc(dq), dk.data_ptr<float>(),
                   dv.data_ptr<float>(), c ? c->data_ptr<float>() : nullptr,
                   s ? s->data_ptr<float>() : nullptr, rows, length, hq, hkv,
                   d, stream());
  post_launch_check("rope_join");
}

// dw, zero before, gets the sums of dy's rows at tokens, which are rows of dw.
void lookup_bwd(torch::Tensor dw, torch::Tensor dy, torch::Tensor tokens) {
  const c10::DeviceGuard guard(dw.device());
  const long n = tokens.numel(), hidden = dw.size(1);
  TORCH_CHECK(dw.dim() == 2 && n > 0 && n < (1L << 30) &&
              train_norm_takes(hidden), "width ", hidden, " not taken");
  TORCH_CHECK(tokens.is_cuda() && tokens.scalar_type() == torch::kLong &&
              tokens.is_contiguous(), "tokens must be int64 on GPU");
  check_rows(dw, dw.numel(), "dw"); check_rows(dy, n * hidden, "dy");
  auto often = torch::empty({n}, tokens.options().dtype(torch::kByte));
  launch_lookup_bwd(bf(dw), often.data_ptr<unsigned char>(), bfc(dy),
                    tokens.data_ptr<long>(), n, dw.size(0), hidden, stream());
  post_launch_check("lookup_bwd");
}

void silu_mul_bwd(torch::Tensor dx, torch::Tensor dy, torch::Tensor x) {
  const c10::DeviceGuard guard(x.device());
  const long f = x.size(-1) / 2, n = x.numel();
  TORCH_CHECK(n > 0 && f % 8 == 0 && x.size(-1) == 2 * f,
              "width must be a multiple of 16");
  check_rows(x, n, "x"); check_rows(dx, n, "dx"); check_rows(dy, n / 2, "dy");
  launch_silu_mul_bwd(bf(dx), bfc(dy), bfc(x), n / (2 * f), f, stream());
  post_launch_check("silu_mul_bwd");
}

void rms_norm(torch::Tensor out, torch::Tensor x, torch::Tensor w, double eps) {
  check_bf16(out, "out"); check_bf16(x, "x"); check_bf16(w, "w");
  int hidden = x.size(-1);
  TORCH_CHECK(hidden % 8 == 0, "hidden must be a multiple of 8");
  TORCH_CHECK(hidden <= 16384, "hidden > 16384 unsupported (register cache)");
  long rows = x.numel() / hidden;
  launch_rms_norm(bf(out), bfc(x), bfc(w), rows, hidden, (float)eps, stream());
  post_launch_check("rms_norm");
}

void rms_norm_residual(torch::Tensor out, torch::Tensor residual,
                       torch::Tensor x, torch::Tensor w, double eps) {
  check_bf16(out, "out"); check_bf16(residual, "residual");
  check_bf16(x, "x"); check_bf16(w, "w");
  int hidden = x.size(-1);
  TORCH_CHECK(hidden % 8 == 0, "hidden must be a multiple of 8");
  TORCH_CHECK(hidden <= 16384, "hidden > 16384 unsupported (register cache)");
  long rows = x.numel() / hidden;
  launch_rms_norm_residual(bf(out), bf(residual), bfc(x), bfc(w), rows,
                           hidden, (float)eps, stream());
  post_launch_check("rms_norm_residual");
}

void layer_norm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                torch::Tensor b, double eps) {
  check_bf16(out, "out"); check_bf16(x, "x"); check_bf16(w, "w");
  check_bf16(b, "b");
  int hidden = x.size(-1);
  TORCH_CHECK(hidden % 8 == 0, "hidden must be a multiple of 8");
  long rows = x.numel() / hidden;
  launch_layer_norm(bf(out), bfc(x), bfc(w), bfc(b), rows, hidden, (float)eps,
                    stream());
  post_launch_check("layer_norm");
}

void silu_mul(torch::Tensor out, torch::Tensor x) {
  const c10::DeviceGuard guard(x.device());
  check_bf16(out, "out"); check_bf16(x, "x");
  int f = out.size(-1);
  TORCH_CHECK(x.size(-1) == 2 * f, "x last dim must be 2*out last dim");
  TORCH_CHECK(f % 8 == 0, "intermediate size must be a multiple of 8");
  long rows = out.numel() / f;
  launch_silu_mul(bf(out), bfc(x), rows, f, stream());
  post_launch_check("silu_mul");
}

void gelu_tanh(torch::Tensor out, torch::Tensor x) {
  check_bf16(out, "out"); check_bf16(x, "x");
  TORCH_CHECK(x.numel() % 8 == 0, "numel must be a multiple of 8");
  launch_gelu(bf(out), bfc(x), x.numel(), stream());
  post_launch_check("gelu_tanh");
}

bool cache_kv8(const torch::Tensor& t, const char* name) {
  if (t.scalar_type() == torch::kBFloat16) return false;
  TORCH_CHECK(t.scalar_type() == torch::kFloat8_e4m3fn, name,
              " cache must be bf16 or float8_e4m3fn");
  return true;
}

void rope_kv_append(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                    torch::Tensor positions, torch::Tensor k_cache,
                    torch::Tensor v_cache, torch::Tensor slots, double theta) {
  check_bf16_rows(q, "q"); check_bf16_rows(k, "k"); check_bf16_rows(v, "v");
  const bool kv8 = cache_kv8(k_cache, "k");
  TORCH_CHECK(cache_kv8(v_cache, "v") == kv8, "cache dtypes must match");
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous());
  TORCH_CHECK(positions.scalar_type() == torch::kInt, "positions must be int32");
  TORCH_CHECK(slots.scalar_type() == torch::kInt, "slots must be int32");
  int ntok = q.size(0), hq = q.size(1), d = q.size(2);
  int hkv = k.size(1);
  int block_size = k_cache.size(2);
  TORCH_CHECK(k_cache.size(1) == hkv && k_cache.size(3) == d, "cache shape");
  TORCH_CHECK(d % 8 == 0 && (d / 2) % 8 == 0, "head_dim constraints");
  launch_rope_kv_append(bf(q), bf(k), bfc(v), positions.data_ptr<int>(),
                        k_cache.data_ptr(), v_cache.data_ptr(),
                        slots.data_ptr<int>(), ntok,
                        hq, hkv, d, block_size, (float)theta, kv8,
                        q.stride(0), k.stride(0), v.stride(0), stream());
  post_launch_check("rope_kv_append");
}

void paged_attn_decode(torch::Tensor out, torch::Tensor q,
                       torch::Tensor k_cache, torch::Tensor v_cache,
                       torch::Tensor block_table, torch::Tensor seq_lens,
                       double scale) {
  check_bf16(out, "out"); check_bf16_rows(q, "q");
  const bool kv8 = cache_kv8(k_cache, "k");
  TORCH_CHECK(cache_kv8(v_cache, "v") == kv8, "cache dtypes must match");
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous());
  TORCH_CHECK(block_table.scalar_type() == torch::kInt, "block_table int32");
  TORCH_CHECK(seq_lens.scalar_type() == torch::kInt, "seq_lens int32");
  TORCH_CHECK(block_table.is_contiguous() && seq_lens.is_contiguous());
  int bsz = q.size(0), hq = q.size(1), d = q.size(2);
  int hkv = k_cache.size(1), block_size = k_cache.size(2);
  int max_blocks = block_table.size(1);
  TORCH_CHECK(paged_attn_decode_supported(d, block_size),
              "paged_attn_decode: unsupported head_dim ", d, " / block_size ",
              block_size);
  TORCH_CHECK(hq % hkv == 0, "hq must be divisible by hkv");
  const bool grouped = paged_attn_grouped(
      hq, hkv, d, q.stride(0), q.data_ptr(), k_cache.data_ptr(),
      v_cache.data_ptr(), kv8);
  int waves;
  const int nsplit = paged_attn_plan(bsz, hq, hkv, d, max_blocks, grouped,
                                     waves);
  float *po = nullptr, *pml = nullptr;
  torch::Tensor part_o, part_ml;
  if (nsplit > 1) {
    auto opts = q.options().dtype(torch::kFloat);
    part_o = torch::empty({bsz, hq, nsplit, d}, opts);
    part_ml = torch::empty({bsz, hq, nsplit, 2}, opts);
    po = part_o.data_ptr<float>();
    pml = part_ml.data_ptr<float>();
  }
  launch_paged_attn_decode(bf(out), bfc(q), k_cache.data_ptr(),
                           v_cache.data_ptr(),
                           block_table.data_ptr<int>(),
                           seq_lens.data_ptr<int>(), bsz, hq, hkv, d,
                           max_blocks, block_size, (float)scale, q.stride(0),
                           nsplit, po, pml, kv8, grouped, waves, stream());
  post_launch_check("paged_attn_decode");
}

void attn_prefill(torch::Tensor out, torch::Tensor q, torch::Tensor k,
                  torch::Tensor v, torch::Tensor seq_start, long max_len,
                  double scale) {
  check_bf16(out, "out"); check_bf16(q, "q"); check_bf16(k, "k");
  check_bf16(v, "v");
  TORCH_CHECK(seq_start.scalar_type() == torch::kInt, "seq_start int32");
  int hq = q.size(1), d = q.size(2), hkv = k.size(1);
  int num_seqs = seq_start.size(0) - 1;
  TORCH_CHECK(attn_prefill_supported(d), "unsupported head_dim ", d);
  TORCH_CHECK(hq % hkv == 0, "hq must be divisible by hkv");
  launch_attn_prefill(bf(out), bfc(q), bfc(k), bfc(v),
                      seq_start.data_ptr<int>(), num_seqs, (int)max_len, hq,
                      hkv, d, (float)scale, stream(), nullptr);
  post_launch_check("attn_prefill");
}

void attn_v5(torch::Tensor out, torch::Tensor q, torch::Tensor k,
             torch::Tensor v, torch::Tensor seq_start, long max_len,
             double scale, c10::optional<torch::Tensor> lse) {
  check_bf16(out, "out"); check_bf16(q, "q"); check_bf16(k, "k");
  check_bf16(v, "v");
  TORCH_CHECK(seq_start.scalar_type() == torch::kInt, "seq_start int32");
  int hq = q.size(1), d = q.size(2), hkv = k.size(1);
  int num_seqs = seq_start.size(0) - 1;
  TORCH_CHECK(attn_v5_supported(d), "unsupported head_dim ", d);
  TORCH_CHECK(hq % hkv == 0, "hq must be divisible by hkv");
  float* lp = nullptr;
  if (lse.has_value()) {
    TORCH_CHECK(lse->scalar_type() == torch::kFloat, "lse f32");
    lp = lse->data_ptr<float>();
  }
  launch_attn_v5(bf(out), bfc(q), bfc(k), bfc(v),
                 seq_start.data_ptr<int>(), num_seqs, (int)max_len, hq,
                 hkv, d, (float)scale, stream(), lp);
  post_launch_check("attn_v5");
}

// forward with saved log2-domain LSE (training path)
void attn_train_fwd(torch::Tensor out, torch::Tensor lse, torch::Tensor q,
                    torch::Tensor k, torch::Tensor v,
                    torch::Tensor seq_start, long max_len, double scale) {
  check_bf16(out, "out"); check_bf16(q, "q"); check_bf16(k, "k");
  check_bf16(v, "v");
  TORCH_CHECK(lse.scalar_type() == torch::kFloat, "lse must be f32");
  TORCH_CHECK(seq_start.scalar_type() == torch::kInt, "seq_start int32");
  int hq = q.size(1), d = q.size(2), hkv = k.size(1);
  int num_seqs = seq_start.size(0) - 1;
  TORCH_CHECK(attn_prefill_supported(d), "unsupported head_dim ", d);
  TORCH_CHECK(hq % hkv == 0, "hq must be divisible by hkv");
  TORCH_CHECK(lse.numel() == q.size(0) * hq, "lse shape");
  launch_attn_prefill(bf(out), bfc(q), bfc(k), bfc(v),
                      seq_start.data_ptr<int>(), num_seqs, (int)max_len, hq,
                      hkv, d, (float)scale, stream(),
                      lse.data_ptr<float>());
  post_launch_check("attn_train_fwd");
}

void attn_train_bwd(torch::Tensor dq, torch::Tensor dk, torch::Tensor dv,
                    torch::Tensor q, torch::Tensor k, torch::Tensor v,
                    torch::Tensor out, torch::Tensor dout,
                    torch::Tensor lse, torch::Tensor delta,
                    torch::Tensor seq_start, long max_len, double scale) {
  check_bf16(dq, "dq");
  TORCH_CHECK(dk.scalar_type() == torch::kFloat &&
              dv.scalar_type() == torch::kFloat,
              "dk/dv are f32 accumulators (GQA heads atomically add)");
  check_bf16(q, "q"); check_bf16(k, "k"); check_bf16(v, "v");
  check_bf16(out, "out"); check_bf16(dout, "dout");
  TORCH_CHECK(lse.scalar_type() == torch::kFloat &&
              delta.scalar_type() == torch::kFloat, "lse/delta f32");
  TORCH_CHECK(seq_start.scalar_type() == torch::kInt, "seq_start int32");
  int hq = q.size(1), d = q.size(2), hkv = k.size(1);
  int num_seqs = seq_start.size(0) - 1;
  TORCH_CHECK(attn_bwd_supported(d), "unsupported head_dim ", d);
  TORCH_CHECK(hq % hkv == 0, "hq must be divisible by hkv");
  launch_attn_bwd_delta(delta.data_ptr<float>(), bfc(dout), bfc(out),
                        (long)q.size(0) * hq, d, stream());
  launch_attn_bwd_dq(bf(dq), bfc(q), bfc(k), bfc(v), bfc(dout),
                     lse.data_ptr<float>(), delta.data_ptr<float>(),
                     seq_start.data_ptr<int>(), num_seqs, (int)max_len, hq,
                     hkv, d, (float)scale, stream());
  launch_attn_bwd_dkv(dk.data_ptr<float>(), dv.data_ptr<float>(), bfc(q),
                      bfc(k), bfc(v), bfc(dout), lse.data_ptr<float>(),
                      delta.data_ptr<float>(), seq_start.data_ptr<int>(),
                      num_seqs, (int)max_len, hq, hkv, d, (float)scale,
                      stream());
  post_launch_check("attn_train_bwd");
}


void attn_prefill_probe(long variant, torch::Tensor out, torch::Tensor q,
                        torch::Tensor k, torch::Tensor v,
                        torch::Tensor seq_start, long max_len, double scale) {
  check_bf16(out, "out"); check_bf16(q, "q"); check_bf16(k, "k");
  check_bf16(v, "v");
  int hq = q.size(1), hkv = k.size(1);
  TORCH_CHECK(q.size(2) == 128, "probe is D=128 only");
  launch_attn_prefill_probe((int)variant, bf(out), bfc(q), bfc(k), bfc(v),
                            seq_start.data_ptr<int>(),
                            seq_start.size(0) - 1, (int)max_len, hq, hkv,
                            (float)scale, stream());
  post_launch_check("attn_prefill_probe");
}

void mfma_gemm(torch::Tensor y, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias,
               c10::optional<torch::Tensor> part, long splitk) {
  check_bf16(y, "y"); check_bf16(x, "x"); check_bf16(w, "w");
  int m = x.size(0), k = x.size(1), n = w.size(0);
  TORCH_CHECK(w.size(1) == k, "shape mismatch");
  TORCH_CHECK(mfma_gemm_supported(m, n, k), "unsupported mfma_gemm shape ",
              m, "x", n, "x", k);
  const bf16_t* bp = nullptr;
  if (bias.has_value()) { check_bf16(*bias, "bias"); bp = bfc(*bias); }
  float* pp = nullptr;
  if (splitk > 1) {
    TORCH_CHECK(part.has_value() &&
                part->numel() >= splitk * (long)m * n, "part too small");
    pp = part->data_ptr<float>();
  }
  launch_mfma_gemm(bf(y), bfc(x), bfc(w), bp, pp, m, n, k, (int)splitk,
                   stream());
  post_launch_check("mfma_gemm");
}

long mfma_gemm_pick_splitk(long m, long n, long k) {
  if (!mfma_gemm_supported((int)m, (int)n, (int)k)) return 0;
  return mfma_gemm_splitk((int)m, (int)n, (int)k);
}

bool tile_gemm_good(long m, long n, long k, long a_ld, long b_ld,
                    bool a_flipped, bool b_flipped, bool gated) {
  return tile_gemm_takes(m, n, k, a_ld, b_ld, a_flipped, b_flipped, gated) &&
         tile_gemm_pays(m, n, k, a_flipped, b_flipped, gated);
}

// y = x w^T + bias, at most 64 rows of x, or up to 256 where that is faster than
// the library and than tile_gemm; gated: y has half the columns, silu(first half) *
// second half; gelu: gelu of rounded columns
bool mid_gemm_good(long m, long n, long k, bool paired) {
  return mid_gemm_takes(m, n, k, paired) && mid_gemm_pays(m, n, k, paired) &&
         !tile_gemm_good(m, n, k, k, k, false, false, paired);
}

bool rows_gemm_good(long m, long n, long k, bool paired) {
  return rows_gemm_takes((int)m, (int)n, (int)k, paired) &&
         rows_gemm_pays((int)m, (int)n, (int)k, paired);
}

// Whether a product's shares are best added up by the norm that follows it.
bool mid_norm_good(long m, long n, long k) {
  return mid_norm_takes(m, n, k) && mid_gemm_pays(m, n, k, false, true) &&
         !rows_gemm_good(m, n, k, false) &&
         !tile_gemm_good(m, n, k, k, k, false, false, false);
}

// Whether the library's product of these few rows would take longer.
bool few_rows_good(long m, long n, long k, bool paired) {
  return rows_gemm_good(m, n, k, paired) || mid_gemm_good(m, n, k, paired);
}

bool rows_gemm_ok(long m, long n, long k, bool gated) {
  return mid_gemm_good(m, n, k, gated) ||
         rows_gemm_takes((int)m, (int)n, (int)k, gated);
}

// Where the columns of a projection of heads go: queries to q [rows, hq, d],
// keys and values to the paged caches.
Heads heads_of(const torch::Tensor& q, const torch::Tensor& positions,
               const torch::Tensor& k_cache, const torch::Tensor& v_cache,
               const torch::Tensor& slots, double theta) {
  check_bf16(q, "q");
  TORCH_CHECK(q.dim() == 3 && q.size(2) % 16 == 0, "q must be [rows, hq, d]");
  const bool kv8 = cache_kv8(k_cache, "k");
  TORCH_CHECK(cache_kv8(v_cache, "v") == kv8, "cache dtypes must match");
  TORCH_CHECK(k_cache.is_cuda() && v_cache.is_cuda() &&
              k_cache.is_contiguous() && v_cache.is_contiguous() &&
              k_cache.dim() == 4 && k_cache.sizes() == v_cache.sizes() &&
              k_cache.size(3) == q.size(2), "cache shape");
  for (const auto& t : {positions, slots})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kInt &&
                t.is_contiguous() && t.numel() == q.size(0),
                "positions and slots must be an int32 of each row");
  return {positions.data_ptr<int>(), slots.data_ptr<int>(),
          k_cache.data_ptr(), v_cache.data_ptr(), (int)q.size(1),
          (int)k_cache.size(1), (int)q.size(2), (int)k_cache.size(2),
          theta > 0. ? logf((float)theta) : 0.f, theta > 0., kv8};
}

// rope_kv_append of fused rows qkv, whose heads come out as rows of their own
void rope_split_append(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                       torch::Tensor qkv, torch::Tensor positions,
                       torch::Tensor k_cache, torch::Tensor v_cache,
                       torch::Tensor slots, double theta) {
  const Heads h = heads_of(q, positions, k_cache, v_cache, slots, theta);
  const long rows = q.size(0), kv = rows * h.hkv * h.d;
  TORCH_CHECK(rows > 0 && 256 % (h.d / 16) == 0 && h.d <= 128,
              "head_dim ", h.d, " not taken");
  check_rows(q, rows * h.hq * h.d, "q");
  check_rows(k, kv, "k"); check_rows(v, kv, "v");
  check_rows(qkv, q.numel() + 2 * kv, "qkv");
  TORCH_CHECK(aligned16(k_cache) && aligned16(v_cache), "misaligned cache");
  launch_rope_split_append(bf(q), bf(k), bf(v), bfc(qkv), h.positions,
                           h.k_cache, h.v_cache, h.slots, rows, h.hq, h.hkv,
                           h.d, h.block_size, (float)theta, h.kv8, stream());
  post_launch_check("rope_split_append");
}

void rows_gemm_to(torch::Tensor y, torch::Tensor x, torch::Tensor w,
                  c10::optional<torch::Tensor> bias, bool gated,
                  const Heads* heads, const NormOf* norm = nullptr,
                  bool gelu = false, const AddTo* add = nullptr,
                  const Undivided* of = nullptr,
                  const MidNorm* after = nullptr) {
  const c10::DeviceGuard guard(x.device());
  check_bf16(y, "y"); check_bf16(w, "w");
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == torch::kBFloat16 &&
              x.dim() == 2 && x.stride(1) == 1 &&
              (x.stride(0) % 8 == 0 || x.size(0) == 1),
              "x must be bf16 rows that begin on 16-byte pieces");
  const int m = x.size(0), k = x.size(1), n = w.size(0);
  const int cols = heads ? n - 2 * heads->hkv * heads->d : gated ? n / 2 : n;
  TORCH_CHECK(w.dim() == 2 && w.size(1) == k && y.size(0) == m &&
              y.numel() == (long)m * cols, "rows_gemm: shape mismatch");
  const bool many = after || !(norm || add || of) &&
                                 !rows_gemm_good(m, n, k, gated || heads) &&
                                 mid_gemm_good(m, n, k, gated || heads);
  TORCH_CHECK(many || rows_gemm_takes(m, n, k, gated || heads),
              "rows_gemm: unsupported shape ", m, "x", n, "x", k);
  TORCH_CHECK(m <= 16 || !(add || of), "rows_gemm: too many rows");
  TORCH_CHECK(!after || mid_norm_takes(m, n, k), "rows_gemm: no shares");
  TORCH_CHECK(aligned16(x) && aligned16(w), "rows_gemm: misaligned operand");
  const bf16_t* bp = nullptr;
  if (bias.has_value()) {
    check_bf16(*bias, "bias");
    TORCH_CHECK(bias->numel() == n, "bias size");
    bp = bfc(*bias);
  }
  if (many) {
    const MidPlan plan = mid_gemm_plan(m, n, k);
    torch::Tensor part;
    if (plan.shares(m, n))
      part = torch::empty({plan.shares(m, n)},
                          x.options().dtype(torch::kFloat));
    launch_mid_gemm({bf(y), bfc(x), bfc(w), bp, m, n, k, x.stride(0), cols},
                    plan, heads, gated, gelu, after,
                    plan.shares(m, n) ? part.data_ptr<float>() : nullptr,
                    stream());
  } else {
    launch_rows_gemm(bf(y), bfc(x), bfc(w), bp, m, n, k, x.stride(0), cols,
                     gated, gelu, heads, norm, add, of, stream());
  }
  post_launch_check("rows_gemm");
}

void rows_gemm(torch::Tensor y, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias, bool gated, bool gelu) {
  TORCH_CHECK(!gated || !gelu, "rows_gemm: one activation");
  rows_gemm_to(y, x, w, bias, gated, nullptr, nullptr, gelu);
}

// a b^T + bias for operands of many rows as they are stored: a [m, k], or [k, m]
// if flipped; b [n, k], or [k, n]. gated: silu(first half) * second half.
torch::Tensor tile_gemm(torch::Tensor a, torch::Tensor b,
                        c10::optional<torch::Tensor> bias, bool a_flipped,
                        bool b_flipped, bool gated, bool gelu) {
  const c10::DeviceGuard guard(a.device());
  for (const auto& t : {a, b})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kBFloat16 &&
                    t.dim() == 2 && t.stride(1) == 1 && aligned16(t),
                "operands must be bf16 rows on 16-byte boundaries");
  const long m = a.size(a_flipped), k = a.size(!a_flipped);
  const long n = b.size(b_flipped);
  TORCH_CHECK(b.size(!b_flipped) == k, "inner dimensions differ");
  TORCH_CHECK(!gelu || !(gated || a_flipped || b_flipped),
              "tile_gemm: gelu is of rows by rows, and the one activation");
  TORCH_CHECK(tile_gemm_takes(m, n, k, a.stride(0), b.stride(0), a_flipped,
                              b_flipped, gated),
              "tile_gemm: unsupported shape ", m, "x", n, "x", k);
  if (bias) check_rows(*bias, n, "bias");
  const TilePlan plan = tile_gemm_plan(m, n, k, a_flipped, b_flipped);
  auto out = torch::empty({m, gated ? n / 2 : n}, a.options());
  torch::Tensor shares;
  if (plan.shares())
    shares = torch::empty({plan.shares()}, a.options().dtype(torch::kFloat));
  launch_tile_gemm({bf(out), bfc(a), bfc(b), bias ? bfc(*bias) : nullptr,
                    (int)m, (int)n, (int)k, a.stride(0), b.stride(0),
                    a_flipped, b_flipped, gated, gelu},
                   plan, plan.shares() ? shares.data_ptr<float>() : nullptr,
                   stream());
  post_launch_check("tile_gemm");
  return out;
}

// A projection of heads with rope_kv_append of what comes out: rotated queries
// in q, keys and values in the caches.
void rows_heads(torch::Tensor q, torch::Tensor x, torch::Tensor w,
                c10::optional<torch::Tensor> bias, torch::Tensor positions,
                torch::Tensor k_cache, torch::Tensor v_cache,
                torch::Tensor slots, double theta) {
  const Heads heads = heads_of(q, positions, k_cache, v_cache, slots, theta);
  rows_gemm_to(q, x, w, bias, false, &heads);
}

Quant quant_of(const std::string& name) {
  if (name == "q4_0") return Quant::Q4_0;
  if (name == "q8_0") return Quant::Q8_0;
  if (name == "q4_K") return Quant::Q4_K;
  TORCH_CHECK(name == "q6_K", "unknown quantization ", name);
  return Quant::Q6_K;
}

bool quant_rows_ok(long m, long n, long k, const std::string& quant,
                   bool gated) {
  return rows_quant_takes((int)m, (int)n, (int)k, quant_of(quant), gated);
}

void quant_rows_to(torch::Tensor y, torch::Tensor x, torch::Tensor scales,
                   torch::Tensor qs, const std::string& quant, bool gated,
                   const Heads* heads, const NormOf* norm = nullptr,
                   const AddTo* add = nullptr,
                   const Undivided* of = nullptr) {
  const c10::DeviceGuard guard(x.device());
  check_bf16(y, "y"); check_bf16(x, "x");
  TORCH_CHECK(scales.scalar_type() == torch::kHalf, "scales must be fp16");
  TORCH_CHECK(qs.scalar_type() == torch::kByte, "qs must be uint8");
  TORCH_CHECK(scales.is_contiguous() && qs.is_contiguous());
  const Quant q = quant_of(quant);
  const int m = x.size(0), k = x.size(1), n = qs.size(0);
  const int cols = heads ? n - 2 * heads->hkv * heads->d : gated ? n / 2 : n;
  TORCH_CHECK(y.size(0) == m && y.numel() == (long)m * cols &&
              scales.size(0) == n, "quant_rows: shape mismatch");
  TORCH_CHECK(rows_quant_takes(m, n, k, q, gated || heads),
              "quant_rows: unsupported shape ", m, "x", n, "x", k);
  TORCH_CHECK(m <= 8 || !(add || of), "quant_rows: too many rows");
  // what is not aligned to the kernel's loads is copied to where it is
  if (!aligned16(x)) x = x.clone();
  if (!aligned16(qs)) qs = qs.clone();
  if (!aligned16(scales)) scales = scales.clone();
  launch_rows_quant(bf(y), bfc(x), scales.data_ptr(),
                    qs.data_ptr<unsigned char>(), m, n, k, q, gated, heads,
                    norm, add, of, stream());
  post_launch_check("quant_rows");
}

// y = x w^T of a quantized weight matrix, at most 64 rows of x; gated as above
void quant_rows(torch::Tensor y, torch::Tensor x, torch::Tensor scales,
                torch::Tensor qs, const std::string& quant, bool gated) {
  quant_rows_to(y, x, scales, qs, quant, gated, nullptr);
}

// The products above of RMS(h + delta) weight as x; sum = h + delta. Heads
// where a cache is given.
NormOf norm_of(const torch::Tensor& sum, const torch::Tensor& delta,
               const torch::Tensor& h, const torch::Tensor& weight,
               double eps) {
  const long k = weight.numel();
  TORCH_CHECK(h.dim() == 2 && h.size(1) == k && h.size(0) > 0 &&
              norm_rows_take(h.size(0), k), "normed rows: unsupported shape");
  check_rows(weight, k, "norm weight");
  check_rows(h, h.numel(), "h"); check_rows(delta, h.numel(), "delta");
  check_rows(sum, h.numel(), "sum");
  return {bfc(delta), bfc(h), bfc(weight),
          const_cast<bf16_t*>(bfc(sum)), (float)eps};
}

struct Where {
  c10::optional<torch::Tensor> positions, k_cache, v_cache, slots;
  double theta;
  Heads heads;
  const Heads* of(const torch::Tensor& q) {
    if (!positions) return nullptr;
    heads = heads_of(q, *positions, *k_cache, *v_cache, *slots, theta);
    return &heads;
  }
};

// In how many parts a product that is added leaves a row's squares.
long rows_added_parts(long m, long n, long k) {
  return n / (rows_gemm_thin((int)m, (int)n, (int)k, false) ? 8 : 16);
}

long quant_added_parts(long m, long n, long k, const std::string& quant) {
  return n / (rows_quant_thin((int)m, (int)n, (int)k, quant_of(quant), false)
                  ? 8 : 16);
}

// A product that is added to the residual stream: total = h + its rows, y =
// total * weight, and every row's squares in parts.
AddTo add_of(const torch::Tensor& y, const torch::Tensor& total,
             const torch::Tensor& squares, const torch::Tensor& h,
             const torch::Tensor& weight, long parts) {
  const long n = weight.numel();
  TORCH_CHECK(h.dim() == 2 && h.size(1) == n && n % 64 == 0 &&
              y.dim() == 2 && y.sizes() == h.sizes(), "added rows: shapes");
  check_rows(weight, n, "norm weight");
  check_rows(h, h.numel(), "h"); check_rows(total, h.numel(), "total");
  TORCH_CHECK(squares.is_cuda() && squares.is_contiguous() &&
              squares.scalar_type() == torch::kFloat &&
              squares.numel() == h.size(0) * parts, "squares");
  return {bfc(h), bfc(weight), const_cast<bf16_t*>(bfc(total)),
          squares.data_ptr<float>()};
}

// Rows x that are an RMSNorm's but for the division by its deviations.
Undivided undivided_of(const torch::Tensor& x, const torch::Tensor& squares,
                       double eps) {
  TORCH_CHECK(x.dim() == 2 && squares.dim() == 2 && squares.is_cuda() &&
              squares.is_contiguous() && aligned16(squares) &&
              squares.scalar_type() == torch::kFloat &&
              squares.size(0) == x.size(0) && squares.size(1) % 4 == 0,
              "squares");
  return {squares.data_ptr<float>(), (int)squares.size(1), (float)eps};
}

void rows_added(torch::Tensor y, torch::Tensor total, torch::Tensor squares,
                torch::Tensor x, torch::Tensor w,
                c10::optional<torch::Tensor> bias, torch::Tensor h,
                torch::Tensor weight) {
  const AddTo add =
      add_of(y, total, squares, h, weight,
             rows_added_parts(x.size(0), w.size(0), w.size(1)));
  rows_gemm_to(y, x, w, bias, false, nullptr, nullptr, false, &add);
}

// A product that is added to the residual stream, total = h + its rows, and the
// RMSNorm of that, y.
void mid_normed(torch::Tensor y, torch::Tensor total, torch::Tensor x,
                torch::Tensor w, c10::optional<torch::Tensor> bias,
                torch::Tensor h, torch::Tensor weight, double eps) {
  const long n = weight.numel();
  TORCH_CHECK(h.dim() == 2 && h.size(1) == n && y.sizes() == h.sizes() &&
              w.dim() == 2 && w.size(0) == n, "normed: shapes");
  check_rows(weight, n, "norm weight");
  check_rows(h, h.numel(), "h"); check_rows(total, h.numel(), "total");
  check_rows(y, h.numel(), "y");
  if (bias) check_rows(*bias, n, "bias");
  const MidNorm after{bfc(h), bfc(weight), const_cast<bf16_t*>(bfc(total)),
                      (float)eps};
  rows_gemm_to(y, x, w, bias, false, nullptr, nullptr, false, nullptr, nullptr,
               &after);
}

void rows_scaled(torch::Tensor y, torch::Tensor x, torch::Tensor squares,
                 double eps, torch::Tensor w,
                 c10::optional<torch::Tensor> bias, bool gated,
                 c10::optional<torch::Tensor> positions,
                 c10::optional<torch::Tensor> k_cache,
                 c10::optional<torch::Tensor> v_cache,
                 c10::optional<torch::Tensor> slots, double theta) {
  Where where{positions, k_cache, v_cache, slots, theta};
  const Undivided of = undivided_of(x, squares, eps);
  rows_gemm_to(y, x, w, bias, gated, where.of(y), nullptr, false, nullptr,
               &of);
}

void quant_added(torch::Tensor y, torch::Tensor total, torch::Tensor squares,
                 torch::Tensor x, torch::Tensor scales, torch::Tensor qs,
                 const std::string& quant, torch::Tensor h,
                 torch::Tensor weight) {
  const AddTo add = add_of(y, total, squares, h, weight,
                           quant_added_parts(x.size(0), qs.size(0),
                                             x.size(1), quant));
  quant_rows_to(y, x, scales, qs, quant, false, nullptr, nullptr, &add);
}

void quant_scaled(torch::Tensor y, torch::Tensor x, torch::Tensor squares,
                  double eps, torch::Tensor scales, torch::Tensor qs,
                  const std::string& quant, bool gated,
                  c10::optional<torch::Tensor> positions,
                  c10::optional<torch::Tensor> k_cache,
                  c10::optional<torch::Tensor> v_cache,
                  c10::optional<torch::Tensor> slots, double theta) {
  Where where{positions, k_cache, v_cache, slots, theta};
  const Undivided of = undivided_of(x, squares, eps);
  quant_rows_to(y, x, scales, qs, quant, gated, where.of(y), nullptr, nullptr,
                &of);
}

void rows_normed(torch::Tensor y, torch::Tensor sum, torch::Tensor delta,
                 torch::Tensor h, torch::Tensor norm, double eps,
                 torch::Tensor w, c10::optional<torch::Tensor> bias,
                 bool gated, c10::optional<torch::Tensor> positions,
                 c10::optional<torch::Tensor> k_cache,
                 c10::optional<torch::Tensor> v_cache,
                 c10::optional<torch::Tensor> slots, double theta) {
  Where where{positions, k_cache, v_cache, slots, theta};
  const NormOf of = norm_of(sum, delta, h, norm, eps);
  rows_gemm_to(y, h, w, bias, gated, where.of(y), &of);
}

void quant_normed(torch::Tensor y, torch::Tensor sum, torch::Tensor delta,
                  torch::Tensor h, torch::Tensor norm, double eps,
                  torch::Tensor scales, torch::Tensor qs,
                  const std::string& quant, bool gated,
                  c10::optional<torch::Tensor> positions,
                  c10::optional<torch::Tensor> k_cache,
                  c10::optional<torch::Tensor> v_cache,
                  c10::optional<torch::Tensor> slots, double theta) {
  Where where{positions, k_cache, v_cache, slots, theta};
  const NormOf of = norm_of(sum, delta, h, norm, eps);
  quant_rows_to(y, h, scales, qs, quant, gated, where.of(y), &of);
}

// rows_heads of a quantized weight matrix
void quant_heads(torch::Tensor q, torch::Tensor x, torch::Tensor scales,
                 torch::Tensor qs, const std::string& quant,
                 torch::Tensor positions, torch::Tensor k_cache,
                 torch::Tensor v_cache, torch::Tensor slots, double theta) {
  const Heads heads = heads_of(q, positions, k_cache, v_cache, slots, theta);
  quant_rows_to(q, x, scales, qs, quant, false, &heads);
}

void quant_gemv_k(torch::Tensor y, torch::Tensor x, torch::Tensor scales,
                  torch::Tensor qs, bool q6) {
  const int m = x.size(0), k = x.size(1);
  TORCH_CHECK(m >= 1 && m <= 8, "quant_gemv_k is the M<=8 decode path");
  TORCH_CHECK(k % 256 == 0, "K must be a multiple of 256 (K-quants)");
  quant_rows(y, x, scales, qs, q6 ? "q6_K" : "q4_K", false);
}

void dequant_k(torch::Tensor out, torch::Tensor scales, torch::Tensor qs,
               bool q6) {
  check_bf16(out, "out");
  TORCH_CHECK(scales.scalar_type() == torch::kHalf, "scales must be fp16");
  TORCH_CHECK(qs.scalar_type() == torch::kByte, "qs must be uint8");
  int n = out.size(0), k = out.size(1);
  TORCH_CHECK(k % 256 == 0, "K must be a multiple of 256 (K-quants)");
  launch_dequant_k(bf(out), scales.data_ptr(),
                   qs.data_ptr<unsigned char>(), n, k, q6, stream());
  post_launch_check("dequant_k");
}

// The same of several bf16 tensors, their gradients scaled by
// min(1, clip / (norm + 1e-6)) where a norm on the device is given.
void adamw_steps(std::vector<torch::Tensor> ps, std::vector<torch::Tensor> gs,
                 std::vector<torch::Tensor> ms, std::vector<torch::Tensor> vs,
                 double lr, double beta1, double beta2, double eps, double wd,
                 long step, double gscale, c10::optional<torch::Tensor> norm,
                 double clip) {
  std::vector<OptTensor> all;
  TORCH_CHECK(!ps.empty() && gs.size() == ps.size() &&
              ms.size() == ps.size() && vs.size() == ps.size(),
              "as many of each");
  const c10::DeviceGuard guard(ps[0].device());
  for (size_t i = 0; i < ps.size(); ++i) {
    const long n = ps[i].numel();
    check_bf16(ps[i], "parameter");
    check_rows(gs[i], n, "gradient");
    check_rows32(ms[i], n, "moment");
    check_rows32(vs[i], n, "moment");
    TORCH_CHECK(aligned16(ps[i]), "parameter must be on a 16-byte boundary");
    all.push_back({ps[i].data_ptr(), gs[i].data_ptr(),
                   ms[i].data_ptr<float>(), vs[i].data_ptr<float>(), n, 0});
  }
  if (norm) check_rows32(*norm, 1, "norm");
  launch_adamw(all, (float)lr, (float)beta1, (float)beta2, (float)eps,
               (float)wd, (int)step, (float)gscale,
               norm ? norm->data_ptr<float>() : nullptr, clip, stream());
  post_launch_check("adamw_steps");
}

// The 2-norm of all tensors as one vector, in 32 bits on the device.
torch::Tensor grad_norm(std::vector<torch::Tensor> gs) {
  TORCH_CHECK(!gs.empty(), "no gradients");
  const c10::DeviceGuard guard(gs[0].device());
  std::vector<OptTensor> all;
  for (auto& g : gs) {
    check_rows(g, g.numel(), "gradient");
    all.push_back({nullptr, g.data_ptr(), nullptr, nullptr, g.numel(), 0});
  }
  auto opts = gs[0].options().dtype(torch::kFloat);
  auto norm = torch::empty({}, opts);
  auto shares = torch::empty({grad_norm_shares(all)}, opts);
  launch_grad_norm(norm.data_ptr<float>(), shares.data_ptr<float>(), all,
                   stream());
  post_launch_check("grad_norm");
  return norm;
}

torch::Tensor mfma32_probe(torch::Tensor a, torch::Tensor b) {
  check_bf16(a, "a"); check_bf16(b, "b");
  TORCH_CHECK(a.size(0) == 32 && a.size(1) == 16 &&
              b.size(0) == 16 && b.size(1) == 32, "probe is 32x16 x 16x32");
  auto d = torch::empty({32, 32}, a.options().dtype(torch::kFloat));
  launch_mfma32_probe(d.data_ptr<float>(), bfc(a), bfc(b), stream());
  post_launch_check("mfma32_probe");
  return d;
}

torch::Tensor mfma_probe(torch::Tensor a, torch::Tensor b) {
  check_bf16(a, "a"); check_bf16(b, "b");
  TORCH_CHECK(a.size(0) == 16 && a.size(1) == 32 && b.size(0) == 32 &&
              b.size(1) == 16, "probe shapes: a[16,32] b[32,16]");
  auto out = torch::empty({16, 16}, a.options().dtype(torch::kFloat));
  launch_mfma_probe(out.data_ptr<float>(), bfc(a), bfc(b), stream());
  post_launch_check("mfma_probe");
  return out;
}

void softmax_sample(torch::Tensor out, torch::Tensor logits,
                    torch::Tensor temperature, torch::Tensor top_k,
                    torch::Tensor top_p, torch::Tensor uniform) {
  TORCH_CHECK(out.scalar_type() == torch::kLong, "out must be int64");
  int bsz = logits.size(0), vocab = logits.size(1);
  TORCH_CHECK((size_t)vocab * logits.element_size() <= 160 * 1024 - 4096,
              "vocab too large for LDS staging: ", vocab);
  auto go = [&](auto* data) {
    launch_softmax_sample(out.data_ptr<long>(), data,
                          temperature.data_ptr<float>(),
                          top_k.data_ptr<int>(), top_p.data_ptr<float>(),
                          uniform.data_ptr<float>(), bsz, vocab, stream());
  };
  if (logits.scalar_type() == torch::kFloat) {   // models served in 32 bits
    TORCH_CHECK(logits.is_cuda() && logits.is_contiguous(),
                "logits must be contiguous on GPU");
    go(static_cast<const float*>(logits.data_ptr<float>()));
  } else {
    check_bf16(logits, "logits");
    go(bfc(logits));
  }
  post_launch_check("softmax_sample");
}

void cross_entropy_fwd_bwd(torch::Tensor loss, torch::Tensor dlogits,
                           torch::Tensor logits, torch::Tensor targets,
                           long ignore_index) {
  const c10::DeviceGuard guard(logits.device());
  check_bf16(dlogits, "dlogits"); check_bf16(logits, "logits");
  TORCH_CHECK(loss.scalar_type() == torch::kFloat, "loss must be fp32");
  TORCH_CHECK(targets.scalar_type() == torch::kLong, "targets must be int64");
  long rows = logits.size(0);
  int vocab = logits.size(1);
  TORCH_CHECK(vocab % 8 == 0, "vocab must be a multiple of 8");
  TORCH_CHECK(targets.is_cuda() && targets.numel() == rows,
              "targets: one of each row, on GPU");
  targets = targets.contiguous();
  auto nvalid = torch::empty({1}, loss.options());
  launch_cross_entropy(loss.data_ptr<float>(), bf(dlogits), bfc(logits),
                       targets.data_ptr<long>(), rows, vocab, ignore_index,
                       nvalid.data_ptr<float>(), stream());
  post_launch_check("cross_entropy_fwd_bwd");
}

void adamw_step(torch::Tensor p, torch::Tensor g, torch::Tensor m,
                torch::Tensor v, double lr, double beta1, double beta2,
                double eps, double wd, long step, double gscale) {
  TORCH_CHECK(p.is_cuda() && p.is_contiguous());
  TORCH_CHECK(m.scalar_type() == torch::kFloat && v.scalar_type() == torch::kFloat);
  long n = p.numel();
  TORCH_CHECK(g.numel() == n && m.numel() == n && v.numel() == n);
  if (p.scalar_type() == torch::kBFloat16) {
    TORCH_CHECK(g.scalar_type() == torch::kBFloat16);
    launch_adamw({{p.data_ptr(), g.data_ptr(), m.data_ptr<float>(),
                   v.data_ptr<float>(), n, 0}},
                 (float)lr, (float)beta1, (float)beta2, (float)eps, (float)wd,
                 (int)step, (float)gscale, nullptr, 0., stream());
  } else {
    TORCH_CHECK(p.scalar_type() == torch::kFloat && g.scalar_type() == torch::kFloat);
    launch_adamw_f32(p.data_ptr<float>(), g.data_ptr<float>(),
                     m.data_ptr<float>(), v.data_ptr<float>(), n, (float)lr,
                     (float)beta1, (float)beta2, (float)eps, (float)wd,
                     (int)step, (float)gscale, stream());
  }
  post_launch_check("adamw_step");
}

void quant_gemv(torch::Tensor y, torch::Tensor x, torch::Tensor scales,
                torch::Tensor qs, bool q8) {
  check_bf16(y, "y"); check_bf16(x, "x");
  TORCH_CHECK(scales.scalar_type() == torch::kHalf, "scales must be fp16");
  TORCH_CHECK(qs.scalar_type() == torch::kByte, "qs must be uint8");
  TORCH_CHECK(scales.is_contiguous() && qs.is_contiguous());
  int m = x.size(0), k = x.size(1), n = y.size(1);
  TORCH_CHECK(m >= 1 && m <= 8, "quant_gemv supports M in [1,8], got ", m);
  TORCH_CHECK(k % 32 == 0, "K must be a multiple of 32");
  if (rows_quant_takes(m, n, k, q8 ? Quant::Q8_0 : Quant::Q4_0, false)) {
    quant_rows(y, x, scales, qs, q8 ? "q8_0" : "q4_0", false);
    return;
  }
  launch_quant_gemv(bf(y), bfc(x), scales.data_ptr(),
                    qs.data_ptr<unsigned char>(), m, n, k, q8, stream());
  post_launch_check("quant_gemv");
}

void dequant(torch::Tensor out, torch::Tensor scales, torch::Tensor qs,
             bool q8) {
  check_bf16(out, "out");
  TORCH_CHECK(scales.scalar_type() == torch::kHalf && qs.scalar_type() == torch::kByte);
  long n = out.size(0);
  int k = out.size(1);
  launch_dequant(bf(out), scales.data_ptr(), qs.data_ptr<unsigned char>(),
                 n, k, q8, stream());
  post_launch_check("dequant");
}

void decode_gemm(torch::Tensor y, torch::Tensor x, torch::Tensor w) {
  check_bf16(y, "y"); check_bf16(x, "x"); check_bf16(w, "w");
  int m = x.size(0), k = x.size(1), n = w.size(0);
  TORCH_CHECK(w.size(1) == k && y.size(0) == m && y.size(1) == n);
  TORCH_CHECK(decode_gemm_supported(m, n, k),
              "decode_gemm unsupported shape M=", m, " N=", n, " K=", k);
  const int splitk = decode_gemm_splitk(n, k);
  auto part = torch::empty({splitk, 256, n},
                           x.options().dtype(torch::kFloat));
  launch_decode_gemm(bf(y), bfc(x), bfc(w), part.data_ptr<float>(), m, n, k,
                     splitk, stream());
  post_launch_check("decode_gemm");
}

bool decode_gemm_ok(long m, long n, long k) {
  return decode_gemm_supported((int)m, (int)n, (int)k);
}

// Y[M, N] = X[M, K] · W^T with W repacked fragment-linear
// (ops.wstream_repack); wstream_gemm.hip
void wstream_gemm(torch::Tensor y, torch::Tensor x, torch::Tensor wp,
                  long n_, long k_) {
  check_bf16(y, "y"); check_bf16(x, "x"); check_bf16(wp, "wp");
  const int m = x.size(0), k = (int)k_, n = (int)n_;
  TORCH_CHECK(x.size(1) == k && y.size(0) == m && y.size(1) == n);
  TORCH_CHECK(wp.numel() == (long)n * k, "packed W size mismatch");
  TORCH_CHECK(wstream_supported(m, n, k),
              "wstream_gemm unsupported shape M=", m, " N=", n, " K=", k);
  const int splitk = wstream_splitk(n, k);
  torch::Tensor part;
  float* pp = nullptr;
  if (splitk > 1) {
    part = torch::empty({splitk, 256, n}, x.options().dtype(torch::kFloat));
    pp = part.data_ptr<float>();
  }
  launch_wstream_gemm(bf(y), bfc(x), bfc(wp), pp, m, n, k, splitk, stream());
  post_launch_check("wstream_gemm");
}

bool wstream_ok(long m, long n, long k) {
  return wstream_supported((int)m, (int)n, (int)k);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("decode_gemm", &decode_gemm);
  m.def("decode_gemm_ok", &decode_gemm_ok);
  m.def("wstream_gemm", &wstream_gemm);
  m.def("wstream_ok", &wstream_ok);
  m.def("rows_gemm", &rows_gemm, py::arg("y"), py::arg("x"), py::arg("w"),
        py::arg("bias"), py::arg("gated"), py::arg("gelu") = false);
  m.def("tile_gemm", &tile_gemm, py::arg("a"), py::arg("b"), py::arg("bias"),
        py::arg("a_flipped"), py::arg("b_flipped"), py::arg("gated") = false,
        py::arg("gelu") = false);
  m.def("tile_gemm_good", &tile_gemm_good);
  m.def("tile_gemm_rows", [](long m, long n, long k, bool a_flipped,
                             bool b_flipped) {
    return tile_gemm_plan(m, n, k, a_flipped, b_flipped).rows;
  });
  m.def("rows_heads", &rows_heads);
  m.def("rows_normed", &rows_normed);
  m.def("quant_normed", &quant_normed);
  m.def("rows_added", &rows_added);
  m.def("rows_added_parts", &rows_added_parts);
  m.def("quant_added_parts", &quant_added_parts);
  m.def("rows_scaled", &rows_scaled);
  m.def("quant_added", &quant_added);
  m.def("quant_scaled", &quant_scaled);
  m.def("norm_rows_take", &norm_rows_take);
  m.def("rope_split_append", &rope_split_append);
  m.def("quant_heads", &quant_heads);
  m.def("rows_gemm_ok", &rows_gemm_ok);
  m.def("mid_gemm_good", &mid_gemm_good);
  m.def("mid_norm_good", &mid_norm_good);
  m.def("mid_normed", &mid_normed);
  m.def("few_rows_good", &few_rows_good);
  m.def("quant_rows", &quant_rows);
  m.def("quant_rows_ok", &quant_rows_ok);
  m.def("quant_gemv", &quant_gemv);
  m.def("dequant", &dequant);
  m.def("add_norm_fwd", &add_norm_fwd);
  m.def("add_norm_bwd", &add_norm_bwd);
  m.def("train_norm_takes", &train_norm_takes);
  m.def("rope_split", &rope_split);
  m.def("rope_join", &rope_join);
  m.def("silu_mul_bwd", &silu_mul_bwd);
  m.def("lookup_bwd", &lookup_bwd);
  m.def("rms_norm", &rms_norm);
  m.def("rms_norm_residual", &rms_norm_residual);
  m.def("layer_norm", &layer_norm);
  m.def("silu_mul", &silu_mul);
  m.def("gelu_tanh", &gelu_tanh);
  m.def("rope_kv_append", &rope_kv_append);
  m.def("plain_tensors", &plain_tensors);
  m.def("paged_attn_plan", [](int bsz, int hq, int hkv, int d, int max_blocks,
                              bool grouped) {
    int waves;
    const int nsplit = paged_attn_plan(bsz, hq, hkv, d, max_blocks, grouped,
                                       waves);
    return py::make_tuple(nsplit, waves);
  });
  m.def("paged_attn_decode", &paged_attn_decode);
  m.def("attn_prefill", &attn_prefill);
  m.def("attn_train_fwd", &attn_train_fwd);
  m.def("mfma_gemm", &mfma_gemm);
  m.def("quant_gemv_k", &quant_gemv_k);
  m.def("mfma32_probe", &mfma32_probe);
  m.def("attn_v5", &attn_v5);
  m.def("dequant_k", &dequant_k);
  m.def("mfma_gemm_pick_splitk", &mfma_gemm_pick_splitk);
  m.def("attn_train_bwd", &attn_train_bwd);
  m.def("mfma_probe", &mfma_probe);
  m.def("attn_prefill_probe", &attn_prefill_probe);
  m.def("softmax_sample", &softmax_sample);
  m.def("cross_entropy_fwd_bwd", &cross_entropy_fwd_bwd);
  m.def("adamw_step", &adamw_step);
  m.def("adamw_steps", &adamw_steps);
  m.def("grad_norm", &grad_norm);
}
