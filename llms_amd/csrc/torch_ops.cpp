// torch_ops.cpp — the thin PyTorch-ROCm custom ops over the C ABI of
// include/llms_amd_fp.h. Each op allocates its output (and, for the bf16
// calls that split k across workgroups, the workspace) with torch on the
// tensor's device, takes torch's current HIP stream, and hands plain pointers,
// row strides and sizes to the C ABI; a nonzero fp_status becomes a
// c10::Error (RuntimeError in Python). No computation happens here.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include "llms_amd_fp.h"

namespace {

void check_status(int st, const char* fn) {
  TORCH_CHECK(st == FP_OK, fn, " failed: ", fp_status_string(st), " (fp_status ", st, ")");
}

void check_2d(const at::Tensor& t, const char* name, at::ScalarType dt) {
  TORCH_CHECK(t.dim() == 2, name, " must be 2-D, got ", t.dim(), "-D");
  TORCH_CHECK(t.scalar_type() == dt, name, " must be ", c10::toString(dt), ", got ",
              c10::toString(t.scalar_type()));
  TORCH_CHECK(t.size(1) <= 1 || t.stride(1) == 1, name, " must have unit inner stride");
  TORCH_CHECK(t.is_cuda(), name, " must be a HIP device tensor");
}

// Every tensor of a call lives on x's device (the kernels dereference all of
// them there; a host pointer would fault the GPU).
void check_same_device(const at::Tensor& x, const at::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda() && t.device() == x.device(), name, " must be on ", x.device(),
              ", got ", t.device());
}

// A weight [N, K] of the call: K columns (the x row length), on x's device.
void check_weight(const at::Tensor& x, const at::Tensor& w, const char* name) {
  TORCH_CHECK(w.size(1) == x.size(1), name, " has ", w.size(1), " columns, x has K = ",
              x.size(1));
  check_same_device(x, w, name);
}

// Per-row int8 scales of weight q: contiguous 1-D fp32, one per row, on x's
// device.
void check_scale(const at::Tensor& x, const at::Tensor& s, const at::Tensor& q, const char* name) {
  TORCH_CHECK(s.dim() == 1 && s.scalar_type() == at::kFloat && s.is_contiguous(), name,
              " must be a contiguous 1-D float32 tensor");
  TORCH_CHECK(s.size(0) == q.size(0), name, " has ", s.size(0), " rows, q has ", q.size(0));
  check_same_device(x, s, name);
}

// Gate and up weights of one call have the same shape.
void check_pair(const at::Tensor& g, const at::Tensor& u, const char* gn, const char* un) {
  TORCH_CHECK(g.sizes() == u.sizes(), gn, " ", g.sizes(), " and ", un, " ", u.sizes(),
              " must have the same shape");
}

void* cur_stream(const at::Tensor& t) {
  return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// Split-k workspace for a bf16 call, from torch's caching allocator on the
// current stream (empty when the call does not split).
at::Tensor workspace(const at::Tensor& x, int64_t M, int64_t N, int64_t K, bool gate_up) {
  const int64_t bytes = fp_workspace_bytes(M, N, K, gate_up ? 1 : 0);
  return at::empty({bytes}, x.options().dtype(at::kByte));
}

// Workspace for an int8 call: the fp32 partials where k is split across
// workgroups, empty otherwise (int8 weights are never expanded to bf16).
at::Tensor workspace_w8(const at::Tensor& x, int64_t M, int64_t N, int64_t K, bool gate_up) {
  const int64_t bytes = fp_workspace_bytes_w8(M, N, K, gate_up ? 1 : 0);
  return at::empty({bytes}, x.options().dtype(at::kByte));
}

at::Tensor qkv(const at::Tensor& x, const at::Tensor& w, int64_t n_q, int64_t n_k) {
  check_2d(x, "x", at::kBFloat16);
  check_2d(w, "W_qkv", at::kBFloat16);
  check_weight(x, w, "W_qkv");
  const c10::DeviceGuard guard(x.device());
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  at::Tensor y = at::empty({M, N}, x.options());
  at::Tensor ws = workspace(x, M, N, K, false);
  check_status(fp_qkv_bf16_ws(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), y.data_ptr(),
                              y.stride(0), M, n_q, n_k, K, ws.numel() ? ws.data_ptr() : nullptr,
                              ws.numel(), cur_stream(x)),
               "fp_qkv_bf16_ws");
  return y;
}

at::Tensor gate_up_silu(const at::Tensor& x, const at::Tensor& wg, const at::Tensor& wu) {
  check_2d(x, "x", at::kBFloat16);
  check_2d(wg, "Wg", at::kBFloat16);
  check_2d(wu, "Wu", at::kBFloat16);
  check_weight(x, wg, "Wg");
  check_weight(x, wu, "Wu");
  check_pair(wg, wu, "Wg", "Wu");
  const c10::DeviceGuard guard(x.device());
  const int64_t M = x.size(0), K = x.size(1), N = wg.size(0);
  at::Tensor y = at::empty({M, N}, x.options());
  at::Tensor ws = workspace(x, M, N, K, true);
  check_status(fp_gate_up_silu_bf16_ws(x.data_ptr(), x.stride(0), wg.data_ptr(), wg.stride(0),
                                       wu.data_ptr(), wu.stride(0), y.data_ptr(), y.stride(0), M,
                                       N, K, ws.numel() ? ws.data_ptr() : nullptr, ws.numel(),
                                       cur_stream(x)),
               "fp_gate_up_silu_bf16_ws");
  return y;
}

at::Tensor qkv_w8(const at::Tensor& x, const at::Tensor& q, const at::Tensor& s, int64_t n_q,
                  int64_t n_k) {
  check_2d(x, "x", at::kBFloat16);
  check_2d(q, "q", at::kChar);
  check_weight(x, q, "q");
  check_scale(x, s, q, "scale");
  const c10::DeviceGuard guard(x.device());
  const int64_t M = x.size(0), K = x.size(1), N = q.size(0);
  at::Tensor y = at::empty({M, N}, x.options());
  at::Tensor ws = workspace_w8(x, M, N, K, false);
  check_status(fp_qkv_w8_ws(x.data_ptr(), x.stride(0), (const int8_t*)q.data_ptr(), q.stride(0),
                            s.data_ptr<float>(), y.data_ptr(), y.stride(0), M, n_q, n_k, K,
                            ws.numel() ? ws.data_ptr() : nullptr, ws.numel(), cur_stream(x)),
               "fp_qkv_w8_ws");
  return y;
}

at::Tensor gate_up_silu_w8(const at::Tensor& x, const at::Tensor& qg, const at::Tensor& sg,
                           const at::Tensor& qu, const at::Tensor& su) {
  check_2d(x, "x", at::kBFloat16);
  check_2d(qg, "qg", at::kChar);
  check_2d(qu, "qu", at::kChar);
  check_weight(x, qg, "qg");
  check_weight(x, qu, "qu");
  check_pair(qg, qu, "qg", "qu");
  check_scale(x, sg, qg, "sg");
  check_scale(x, su, qu, "su");
  const c10::DeviceGuard guard(x.device());
  const int64_t M = x.size(0), K = x.size(1), N = qg.size(0);
  at::Tensor y = at::empty({M, N}, x.options());
  at::Tensor ws = workspace_w8(x, M, N, K, true);
  check_status(fp_gate_up_silu_w8_ws(x.data_ptr(), x.stride(0), (const int8_t*)qg.data_ptr(),
                                     qg.stride(0), sg.data_ptr<float>(),
                                     (const int8_t*)qu.data_ptr(), qu.stride(0),
                                     su.data_ptr<float>(), y.data_ptr(), y.stride(0), M, N, K,
                                     ws.numel() ? ws.data_ptr() : nullptr, ws.numel(),
                                     cur_stream(x)),
               "fp_gate_up_silu_w8_ws");
  return y;
}

at::Tensor linear(const at::Tensor& x, const at::Tensor& w) {
  check_2d(x, "x", at::kBFloat16);
  check_2d(w, "W", at::kBFloat16);
  check_weight(x, w, "W");
  const c10::DeviceGuard guard(x.device());
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  at::Tensor y = at::empty({M, N}, x.options());
  at::Tensor ws = workspace(x, M, N, K, false);
  check_status(fp_linear_bf16_ws(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0),
                                 y.data_ptr(), y.stride(0), M, N, K,
                                 ws.numel() ? ws.data_ptr() : nullptr, ws.numel(), cur_stream(x)),
               "fp_linear_bf16_ws");
  return y;
}

at::Tensor linear_w8(const at::Tensor& x, const at::Tensor& q, const at::Tensor& s) {
  check_2d(x, "x", at::kBFloat16);
  check_2d(q, "q", at::kChar);
  check_weight(x, q, "q");
  check_scale(x, s, q, "scale");
  const c10::DeviceGuard guard(x.device());
  const int64_t M = x.size(0), K = x.size(1), N = q.size(0);
  at::Tensor y = at::empty({M, N}, x.options());
  at::Tensor ws = workspace_w8(x, M, N, K, false);
  check_status(fp_linear_w8_ws(x.data_ptr(), x.stride(0), (const int8_t*)q.data_ptr(), q.stride(0),
                               s.data_ptr<float>(), y.data_ptr(), y.stride(0), M, N, K,
                               ws.numel() ? ws.data_ptr() : nullptr, ws.numel(), cur_stream(x)),
               "fp_linear_w8_ws");
  return y;
}

// ---- RMSNorm prologue fused with the projections ----

void check_gamma(const at::Tensor& x, const at::Tensor& gamma) {
  TORCH_CHECK(gamma.dim() == 1 && gamma.scalar_type() == at::kBFloat16 && gamma.is_contiguous(),
              "norm weight must be a contiguous 1-D bfloat16 tensor");
  TORCH_CHECK(gamma.size(0) == x.size(1), "norm weight has ", gamma.size(0),
              " elements, x has K = ", x.size(1));
  check_same_device(x, gamma, "norm weight");
}

// Workspace for a fused-norm call: what the library asks for (enough for any
// pointers and strides of the shape).
at::Tensor norm_workspace(const at::Tensor& x, int64_t M, int64_t N, int64_t K, bool gate_up,
                          bool int8) {
  const int64_t bytes = fp_rmsnorm_workspace_bytes(M, N, K, gate_up ? 1 : 0, int8 ? 1 : 0);
  return at::empty({bytes}, x.options().dtype(at::kByte));
}

at::Tensor rmsnorm_qkv(const at::Tensor& x, const at::Tensor& gamma, double eps,
                       const at::Tensor& w, int64_t n_q, int64_t n_k) {
  check_2d(x, "x", at::kBFloat16);
  check_2d(w, "W_qkv", at::kBFloat16);
  check_weight(x, w, "W_qkv");
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  check_gamma(x, gamma);
  const c10::DeviceGuard guard(x.device());
  at::Tensor y = at::empty({M, N}, x.options());
  at::Tensor ws = norm_workspace(x, M, N, K, false, false);
  check_status(fp_rmsnorm_qkv_bf16(x.data_ptr(), x.stride(0), gamma.data_ptr(), (float)eps,
                                   w.data_ptr(), w.stride(0), y.data_ptr(), y.stride(0), M, n_q,
                                   n_k, K, ws.data_ptr(), ws.numel(), cur_stream(x)),
               "fp_rmsnorm_qkv_bf16");
  return y;
}

at::Tensor rmsnorm_gate_up_silu(const at::Tensor& x, const at::Tensor& gamma, double eps,
                                const at::Tensor& wg, const at::Tensor& wu) {
  check_2d(x, "x", at::kBFloat16);
  check_2d(wg, "Wg", at::kBFloat16);
  check_2d(wu, "Wu", at::kBFloat16);
  check_weight(x, wg, "Wg");
  check_weight(x, wu, "Wu");
  check_pair(wg, wu, "Wg", "Wu");
  const int64_t M = x.size(0), K = x.size(1), N = wg.size(0);
  check_gamma(x, gamma);
  const c10::DeviceGuard guard(x.device());
  at::Tensor y = at::empty({M, N}, x.options());
  at::Tensor ws = norm_workspace(x, M, N, K, true, false);
  check_status(fp_rmsnorm_gate_up_silu_bf16(x.data_ptr(), x.stride(0), gamma.data_ptr(),
                                            (float)eps, wg.data_ptr(), wg.stride(0),
                                            wu.data_ptr(), wu.stride(0), y.data_ptr(),
                                            y.stride(0), M, N, K, ws.data_ptr(), ws.numel(),
                                            cur_stream(x)),
               "fp_rmsnorm_gate_up_silu_bf16");
  return y;
}

at::Tensor rmsnorm_qkv_w8(const at::Tensor& x, const at::Tensor& gamma, double eps,
                          const at::Tensor& q, const at::Tensor& s, int64_t n_q, int64_t n_k) {
  check_2d(x, "x", at::kBFloat16);
  check_2d(q, "q", at::kChar);
  check_weight(x, q, "q");
  check_scale(x, s, q, "scale");
  const int64_t M = x.size(0), K = x.size(1), N = q.size(0);
  check_gamma(x, gamma);
  const c10::DeviceGuard guard(x.device());
  at::Tensor y = at::empty({M, N}, x.options());
  at::Tensor ws = norm_workspace(x, M, N, K, false, true);
  check_status(fp_rmsnorm_qkv_w8(x.data_ptr(), x.stride(0), gamma.data_ptr(), (float)eps,
                                 (const int8_t*)q.data_ptr(), q.stride(0), s.data_ptr<float>(),
                                 y.data_ptr(), y.stride(0), M, n_q, n_k, K, ws.data_ptr(),
                                 ws.numel(), cur_stream(x)),
               "fp_rmsnorm_qkv_w8");
  return y;
}

at::Tensor rmsnorm_gate_up_silu_w8(const at::Tensor& x, const at::Tensor& gamma, double eps,
                                   const at::Tensor& qg, const at::Tensor& sg,
                                   const at::Tensor& qu, const at::Tensor& su) {
  check_2d(x, "x", at::kBFloat16);
  check_2d(qg, "qg", at::kChar);
  check_2d(qu, "qu", at::kChar);
  check_weight(x, qg, "qg");
  check_weight(x, qu, "qu");
  check_pair(qg, qu, "qg", "qu");
  check_scale(x, sg, qg, "sg");
  check_scale(x, su, qu, "su");
  const int64_t M = x.size(0), K = x.size(1), N = qg.size(0);
  check_gamma(x, gamma);
  const c10::DeviceGuard guard(x.device());
  at::Tensor y = at::empty({M, N}, x.options());
  at::Tensor ws = norm_workspace(x, M, N, K, true, true);
  check_status(fp_rmsnorm_gate_up_silu_w8(x.data_ptr(), x.stride(0), gamma.data_ptr(),
                                          (float)eps, (const int8_t*)qg.data_ptr(), qg.stride(0),
                                          sg.data_ptr<float>(), (const int8_t*)qu.data_ptr(),
                                          qu.stride(0), su.data_ptr<float>(), y.data_ptr(),
                                          y.stride(0), M, N, K, ws.data_ptr(), ws.numel(),
                                          cur_stream(x)),
               "fp_rmsnorm_gate_up_silu_w8");
  return y;
}

// ---- the attention layer between its projections ----

// q [B, T, n] as rows b*T + t of a row stride the kernels take; -1 if not.
int64_t token_rows(const at::Tensor& t, int64_t B, int64_t T, int64_t n) {
  if (t.dim() != 3 || t.size(0) != B || t.size(1) != T || t.size(2) != n || t.stride(2) != 1)
    return -1;
  const int64_t ld = T > 1 ? t.stride(1) : B > 1 ? t.stride(0) : n;
  if (B > 1 && t.stride(0) != T * ld) return -1;
  return ld >= n && ld % 4 == 0 && (uintptr_t)t.data_ptr() % 8 == 0 ? ld : -1;
}

// q, k, v: the projection's flat outputs. q_gamma, k_gamma: the QK-norm
// weights, or absent where q and k are normalised already. Returns the
// attention output [B, T, n_heads * D], or an empty 1-D tensor, with nothing
// launched and nothing written, where the kernels do not take the call (types,
// devices, sizes, strides): the caller then runs the torch form, which also
// raises the errors of invalid calls.
at::Tensor attention(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                     const c10::optional<at::Tensor>& q_gamma,
                     const c10::optional<at::Tensor>& k_gamma, double q_eps, double k_eps,
                     const at::Tensor& cos, const at::Tensor& sin, at::Tensor cache_k,
                     at::Tensor cache_v, int64_t n_heads, int64_t start_pos,
                     const c10::optional<at::Tensor>& pos) {
  const auto none = [&] { return at::empty({0}, q.options()); };
  const auto bf16_here = [&](const at::Tensor& t) {
    return t.scalar_type() == at::kBFloat16 && t.device() == q.device() &&
           t.layout() == at::kStrided && !t.is_neg();
  };
  for (const at::Tensor* t : {&q, &k, &v, &cos, &sin, (const at::Tensor*)&cache_k,
                              (const at::Tensor*)&cache_v})
    if (!bf16_here(*t)) return none();
  // torch refuses to write an inference tensor outside inference mode
  if (!c10::InferenceMode::is_enabled() && (cache_k.is_inference() || cache_v.is_inference()))
    return none();
  if (!q.is_cuda() || q.dim() != 3 || cache_k.dim() != 4 || cache_v.dim() != 4) return none();
  const int64_t B = q.size(0), T = q.size(1), Hk = cache_k.size(1), S = cache_k.size(2);
  const int64_t D = cache_k.size(3);
  if (B < 1 || T < 1 || Hk < 1 || n_heads < 1 || n_heads % Hk != 0) return none();
  if (cache_v.sizes() != cache_k.sizes() || cache_k.size(0) < B || cache_k.stride(3) != 1 ||
      cache_v.stride(3) != 1)
    return none();
  fp_attention_args a{};
  a.ldq = token_rows(q, B, T, n_heads * D);
  a.ldk = token_rows(k, B, T, Hk * D);
  a.ldv = token_rows(v, B, T, Hk * D);
  if (a.ldq < 0 || a.ldk < 0 || a.ldv < 0) return none();
  for (const at::Tensor* t : {&cos, &sin})
    if (t->dim() != 2 || t->size(0) != T || t->size(1) != D || t->stride(1) != 1) return none();
  if (q_gamma.has_value() != k_gamma.has_value()) return none();
  if (q_gamma.has_value()) {
    for (const at::Tensor* t : {&*q_gamma, &*k_gamma})
      if (!bf16_here(*t) || t->dim() != 1 || t->size(0) != D || t->stride(0) != 1) return none();
    a.q_gamma = q_gamma->data_ptr(), a.k_gamma = k_gamma->data_ptr();
  }
  int64_t keys = S;
  if (pos.has_value()) {
    if (pos->dim() != 0 || pos->scalar_type() != at::kLong || pos->device() != q.device())
      return none();
    a.pos_dev = pos->data_ptr<int64_t>();
  } else {
    if (start_pos < 0 || start_pos + T > S) return none();
    a.pos = start_pos;
    keys = start_pos + T;
  }
  a.q = q.data_ptr(), a.k = k.data_ptr(), a.v = v.data_ptr();
  a.cos = cos.data_ptr(), a.sin = sin.data_ptr();
  a.ld_cos = T > 1 ? cos.stride(0) : D, a.ld_sin = T > 1 ? sin.stride(0) : D;
  a.cache_k = cache_k.data_ptr(), a.cache_v = cache_v.data_ptr();
  // a dimension of one element may carry any stride
  const auto sd = [](const at::Tensor& t, int64_t i) { return t.size(i) > 1 ? t.stride(i) : 0; };
  a.k_s_b = sd(cache_k, 0), a.k_s_h = sd(cache_k, 1), a.k_s_p = S > 1 ? cache_k.stride(2) : D;
  a.v_s_b = sd(cache_v, 0), a.v_s_h = sd(cache_v, 1), a.v_s_p = S > 1 ? cache_v.stride(2) : D;
  a.B = B, a.T = T, a.n_heads = n_heads, a.n_kv_heads = Hk, a.head_dim = D, a.cache_len = S;
  a.q_eps = (float)q_eps, a.k_eps = (float)k_eps;
  const c10::DeviceGuard guard(q.device());
  const int64_t bytes = fp_attention_workspace_bytes(B, T, n_heads, Hk, D, keys);
  if (bytes <= 0) return none();
  at::Tensor y = at::empty({B, T, n_heads * D}, q.options());
  at::Tensor ws = at::empty({bytes}, q.options().dtype(at::kByte));
  a.y = y.data_ptr();
  const int st = fp_attention_bf16(&a, ws.data_ptr(), bytes, cur_stream(q));
  // sizes, strides and alignments that the kernels do not take: nothing ran
  if (st == FP_ERR_SHAPE || st == FP_ERR_STRIDE) return none();
  check_status(st, "fp_attention_bf16");
  for (at::Tensor* t : {&cache_k, &cache_v})
    if (!t->is_inference()) t->unsafeGetTensorImpl()->bump_version();
  return y;
}

std::tuple<at::Tensor, at::Tensor> quantize_w8(const at::Tensor& w) {
  check_2d(w, "W", at::kBFloat16);
  const c10::DeviceGuard guard(w.device());
  const int64_t N = w.size(0), K = w.size(1);
  at::Tensor q = at::empty({N, K}, w.options().dtype(at::kChar));
  at::Tensor s = at::empty({N}, w.options().dtype(at::kFloat));
  check_status(fp_quantize_w8_per_row(w.data_ptr(), w.stride(0), (int8_t*)q.data_ptr(),
                                      q.stride(0), s.data_ptr<float>(), N, K, cur_stream(w)),
               "fp_quantize_w8_per_row");
  return {q, s};
}

}  // namespace

TORCH_LIBRARY(llms_amd, m) {
  m.def("qkv(Tensor x, Tensor w_qkv, int n_q, int n_k) -> Tensor");
  m.def("gate_up_silu(Tensor x, Tensor wg, Tensor wu) -> Tensor");
  m.def("qkv_w8(Tensor x, Tensor q, Tensor scale, int n_q, int n_k) -> Tensor");
  m.def("gate_up_silu_w8(Tensor x, Tensor qg, Tensor sg, Tensor qu, Tensor su) -> Tensor");
  m.def("linear(Tensor x, Tensor w) -> Tensor");
  m.def("linear_w8(Tensor x, Tensor q, Tensor scale) -> Tensor");
  m.def("rmsnorm_qkv(Tensor x, Tensor gamma, float eps, Tensor w, int n_q, int n_k) -> Tensor");
  m.def("rmsnorm_gate_up_silu(Tensor x, Tensor gamma, float eps, Tensor wg, Tensor wu) -> Tensor");
  m.def("rmsnorm_qkv_w8(Tensor x, Tensor gamma, float eps, Tensor q, Tensor scale, int n_q, "
        "int n_k) -> Tensor");
  m.def("rmsnorm_gate_up_silu_w8(Tensor x, Tensor gamma, float eps, Tensor qg, Tensor sg, "
        "Tensor qu, Tensor su) -> Tensor");
  m.def("attention(Tensor q, Tensor k, Tensor v, Tensor? q_gamma, Tensor? k_gamma, float q_eps, "
        "float k_eps, Tensor cos, Tensor sin, Tensor(a!) cache_k, Tensor(b!) cache_v, "
        "int n_heads, int start_pos, Tensor? pos) -> Tensor");
  m.def("quantize_w8(Tensor w) -> (Tensor, Tensor)");
}

TORCH_LIBRARY_IMPL(llms_amd, CUDA, m) {
  m.impl("qkv", qkv);
  m.impl("gate_up_silu", gate_up_silu);
  m.impl("qkv_w8", qkv_w8);
  m.impl("gate_up_silu_w8", gate_up_silu_w8);
  m.impl("linear", linear);
  m.impl("linear_w8", linear_w8);
  m.impl("rmsnorm_qkv", rmsnorm_qkv);
  m.impl("rmsnorm_gate_up_silu", rmsnorm_gate_up_silu);
  m.impl("rmsnorm_qkv_w8", rmsnorm_qkv_w8);
  m.impl("rmsnorm_gate_up_silu_w8", rmsnorm_gate_up_silu_w8);
  m.impl("attention", attention);
  m.impl("quantize_w8", quantize_w8);
}
