// fp_api.hip — the extern "C" entry points of include/llms_amd_fp.h:
// argument validation (before any launch), regime dispatch and the
// per-row int8 quantisation kernel.
#include "llms_amd_fp.h"

#include "fp_common.h"
#include "fp_launch.h"

namespace fp {

namespace {

// One workgroup per weight row: absmax reduction, then quantise the row.
__global__ __launch_bounds__(256) void quantize_w8_kernel(const uint16_t* w, int64_t ldw,
                                                          int8_t* q, int64_t ldq, float* scale,
                                                          int64_t K) {
  const int64_t r = blockIdx.x;
  const uint16_t* wr = w + r * ldw;
  float mx = 0.f;
  for (int64_t k = threadIdx.x; k < K; k += blockDim.x) mx = fmaxf(mx, fabsf(bf16_bits_to_f32(wr[k])));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
  __shared__ float part[4];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
  const float s = mx / 127.0f;
  if (threadIdx.x == 0) scale[r] = s;
  int8_t* qr = q + r * ldq;
  for (int64_t k = threadIdx.x; k < K; k += blockDim.x) {
    float v = 0.f;
    if (s > 0.f) v = fminf(fmaxf(rintf(bf16_bits_to_f32(wr[k]) / s), -127.f), 127.f);
    qr[k] = (int8_t)(int)v;
  }
}

// The same with the row in registers, 16 bytes per load (one pass over memory
// instead of two of 2-byte loads). A row that starts off a 16-byte boundary is
// cut into chunks at those boundaries, the partial ones at its two ends read and
// stored by elements, so loads are aligned for any K and stride; the int8 chunks
// are stored as they fall, 8 bytes at any address. Bit-identical (a maximum, and
// the same division and rounding per element). Measured on MI355X, 12288 x 4096
// 103.9 -> 37.9 us (4.0 TB/s), 6409 x 10234 134 -> 62.6, 9728 x 2560 38.7 -> 20.7.
// NV chunks of 8 elements per thread: rows of up to 2048 NV - 7 elements.
template <int NV>
__global__ __launch_bounds__(256) void quantize_w8_row_kernel(const uint16_t* w, int64_t ldw,
                                                              int8_t* q, int64_t ldq, float* scale,
                                                              int K) {
  const int64_t r = blockIdx.x;
  const uint16_t* wr = w + r * ldw;
  const int off = (int)((reinterpret_cast<uintptr_t>(wr) & 15) / 2);  // elements past a boundary
  u32x4 v[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int k = ((int)threadIdx.x + 256 * i) * 8 - off;  // element of the chunk's first
    v[i] = u32x4{0u, 0u, 0u, 0u};
    if (k >= 0 && k + 8 <= K) {
      v[i] = ld16(wr + k);
    } else if (k < K) {  // the row's two ends
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (k + e >= 0 && k + e < K) v[i][e / 2] |= (uint32_t)wr[k + e] << (16 * (e & 1));
    }
  }
  float mx = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int d = 0; d < 4; ++d)
      mx = fmaxf(mx, fmaxf(fabsf(bf16_bits_to_f32(v[i][d] & 0xffffu)), fabsf(bf16_bits_to_f32(v[i][d] >> 16))));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  __shared__ float part[4];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
  const float s = mx / 127.0f;
  if (threadIdx.x == 0) scale[r] = s;
  int8_t* qr = q + r * ldq;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int k = ((int)threadIdx.x + 256 * i) * 8 - off;
    if (k >= K) continue;
    uint32_t b[2] = {0u, 0u};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t h = e & 1 ? v[i][e / 2] >> 16 : v[i][e / 2] & 0xffffu;
      float f = 0.f;
      if (s > 0.f) f = fminf(fmaxf(rintf(bf16_bits_to_f32(h) / s), -127.f), 127.f);
      b[e / 4] |= (uint32_t)(uint8_t)(int8_t)(int)f << (8 * (e % 4));
    }
    if (k >= 0 && k + 8 <= K) {
      __builtin_memcpy(qr + k, b, 8);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (k + e >= 0 && k + e < K) qr[k + e] = (int8_t)(b[e / 4] >> (8 * (e % 4)));
    }
  }
}

inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// rc is the hipError_t of the launch (hipGetLastError right after it).
int launch_status(int rc) {
  if (rc == (int)hipSuccess) return FP_OK;
  const hipError_t e = (hipError_t)rc;
  if (e == hipErrorNoBinaryForGpu || e == hipErrorInvalidDeviceFunction) return FP_ERR_DEVICE;
  return FP_ERR_LAUNCH;
}

template <bool GATEUP, bool W8>
int run(const StreamArgs& a, bool aligned, hipStream_t s) {
  if (a.M == 0) return FP_OK;
  const int rc = (a.M <= kStreamMaxM) ? launch_stream<GATEUP, W8>(a, aligned, s)
                                      : launch_tiled<GATEUP, W8>(a, aligned, s);
  return launch_status(rc);
}

inline int64_t round_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

// int8 calls always dequantise in registers (or once per workgroup into
// LDS in the prefill tiles); no bf16 copy of the weights is ever written.
// With a workspace, the calls whose plan splits k across at least 4
// workgroups (gemm_split_plan: Qwen3 down and o at row counts between 65 and 1792, 8B QKV at 129-256)
// run that split on the int8 weights (gemm_kernel dequantising in registers,
// fp32 partials in the workspace, the fixed-order reduce). Excluded: the
// shapes the int8 split-K tiles take (splitk8_shape) and those the
// in-register prefill tiles take unsplit (gemm8_shape). Measured on MI355X
// against the unsplit dispatch: 8B QKV at 256 rows 44.1 -> 30.9 us, 4B down
// at 128 40.5 -> 26.9 us, 8B down at 256 66.2 -> 46.9 us, 8B o at 256 34.0 ->
// 26.7 us.
inline GemmSplit split8_plan(int64_t M, int64_t N, int64_t K, bool gateup) {
  const GemmSplit none{-1, 1};
  if (K % 64 != 0 || M < 48) return none;
  if (splitk8_shape(M, N, K, gateup) || gemm8_shape(M, N, K, gateup)) return none;
  const GemmSplit p = gemm_split_plan(M, N, K, gateup);
  return p.nsplit >= 4 ? p : none;
}

template <bool GATEUP>
int run_w8(const StreamArgs& a, bool aligned, void* ws, int64_t ws_bytes, hipStream_t s) {
  if (a.M == 0) return FP_OK;
  const GemmSplit p8 = split8_plan(a.M, a.N, a.K, GATEUP);
  if (aligned && p8.tile >= 0 && ws) {
    StreamArgs b = a;
    b.ws = (float*)ws;
    b.ws_floats = ws_bytes / 4;
    if (gemm_split_ws_floats(p8, a.M, a.N, a.K, GATEUP) <= b.ws_floats &&
        gemm_supported(b, true, true))
      return launch_status(launch_gemm_split<GATEUP, true>(b, p8, s));
  }
  StreamArgs b = a;
  b.ws = nullptr;
  b.ws_floats = 0;
  return run<GATEUP, true>(b, aligned, s);
}

int64_t w8_workspace_bytes(int64_t M, int64_t N, int64_t K, bool gateup) {
  if (M < 1 || N < 1 || K < 1) return 0;
  const GemmSplit p8 = split8_plan(M, N, K, gateup);
  return p8.tile >= 0 ? 4 * gemm_split_ws_floats(p8, M, N, K, gateup) : 0;
}

// Where the rows kernel, if it takes the call, also normalises. Every one of its
// workgroups (N / 8 of them) repeats the norm of all the rows behind two barriers,
// which costs more with each element of x and each round of workgroups, while a
// launch of rmsnorm_kernel costs 1-3.5 us once and lets the plain dispatch choose
// its kernel (int8 from 2 rows: fp_xpanel.hip). Graph of 2-24 weight sets, us, in
// the rows kernel / as its own launch:
//   one bf16 row: 4B QKV 8.70 / 9.17, gate-up 18.05 / 18.85, 8B 10.89 / 12.50, 32.19
//   / 34.13. A tied head's thousands of workgroups repeat it too often (151936 x
//   2560 120 / 109; 43871 x 2048 33.2 / 31.8) but for the longest rows (96529 x 4096
//   122.7 / 124.9).
//   one round of workgroups (N <= 2048): two bf16 rows, 1596 x 2048 5.21 / 5.84,
//   gate-up 711 x 2560 6.71 / 7.45, 1779 x 3072 6.49 / 7.12, but 270 x 3072 5.80
//   / 5.39; int8 949 x 3072 4.58 / 5.59, two rows, gate-up 755 x 2048 7.40 / 8.22 (the
//   kernel takes K in chunks of 1024: 1668 x 1536 7.67 / 7.40), four rows 885 x 1024
//   5.02 / 5.38.
//   more rounds: two bf16 rows 4B QKV 10.94 / 10.37, gate-up 22.32 / 20.35, 0.6B (K =
//   1024) 5.14 / 5.97, 6.60 / 7.28, 3731 x 1536 6.39 / 6.93; one int8 row 0.6B 4.33 /
//   5.27, 5.49 / 5.95, 3416 x 4096 7.38 / 7.77, 4B 8.37 / 8.54, gate-up 16.24 / 13.55,
//   8B 9.84 / 9.67, 23.96 / 22.12; two 4B 10.21 / 9.46, 20.69 / 19.29; three and four
//   14.3-14.8 / 9.4-9.6, 29.7-31.2 / 19.3-19.4.
template <bool GATEUP, bool W8>
bool norm_in_rows(int64_t M, int64_t N, int64_t K) {
  const int64_t x = M * K;
  if (N > 32768) return !W8 && !GATEUP && M == 1 && K > 3072;
  if (!W8) {
    if (M == 1 || x <= 2048) return true;
    if (N <= 2048) return x <= (GATEUP || N > 1024 ? 8192 : 5120);
    return !GATEUP && N <= 4096 && x <= 3072;
  }
  if (M <= 2 && x <= (GATEUP ? 2048 : 2560)) return true;
  if constexpr (GATEUP) return N <= 2048 && M > 1 && K % 1024 == 0 && K <= (M == 2 ? 3072 : 2048);
  if (M == 1) return N <= 4096 && K <= 4096;
  return N <= 2048 && K <= (M == 2 ? 3072 : 1024);
}

// RMSNorm prologue + projection: one launch on the rows kernel (x normalised
// while it is staged in LDS) where norm_in_rows says so or no workspace is
// there, else the norm into the workspace and the plain dispatch on the
// normalised rows (any split workspace follows them).
// xaligned: x rows and K fit the vector path; waligned: the weights do.
template <bool GATEUP, bool W8>
int run_norm(StreamArgs a, bool xaligned, bool waligned, void* ws, int64_t ws_bytes,
             hipStream_t s) {
  if (a.M == 0) return FP_OK;
  const bool galigned = al16(a.gamma);
  const int64_t xn_bytes = round_up(a.M * a.K * 2, 256);
  const bool room = ws && ws_bytes >= xn_bytes;
  if (rows_supported<W8>(a, xaligned && waligned && galigned) &&
      (!room || norm_in_rows<GATEUP, W8>(a.M, a.N, a.K)))
    return launch_status(launch_rows<GATEUP, W8>(a, s));
  if (!ws || ws_bytes < xn_bytes) return FP_ERR_WORKSPACE;
  uint16_t* xn = (uint16_t*)ws;
  int rc = launch_rmsnorm(a.x, a.ldx, a.gamma, a.eps, xn, a.M, a.K,
                          xaligned && galigned && a.K % 8 == 0, s);
  if (rc) return launch_status(rc);
  StreamArgs b = a;
  b.x = xn;
  b.ldx = a.K;
  b.gamma = nullptr;
  const bool baligned = waligned && a.K % (W8 ? 16 : 8) == 0;
  if constexpr (W8) return run_w8<GATEUP>(b, baligned, (char*)ws + xn_bytes, ws_bytes - xn_bytes, s);
  b.ws = (float*)((char*)ws + xn_bytes);
  b.ws_floats = (ws_bytes - xn_bytes) / 4;
  return run<GATEUP, false>(b, baligned, s);
}

int check_norm(float eps, void* ws, int64_t ws_bytes) {
  if (!(eps >= 0.f) || eps > 3.0e38f) return FP_ERR_SHAPE;
  if (ws_bytes < 0 || (ws && !al16(ws))) return FP_ERR_WORKSPACE;
  return FP_OK;
}

int check_common(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldy) {
  if (M < 0 || N < 1 || K < 1) return FP_ERR_SHAPE;
  // grid.x = ceil(N / 16) must fit a 32-bit grid dimension; M tiles likewise.
  if (N > (int64_t)1 << 34 || M > (int64_t)1 << 34) return FP_ERR_SHAPE;
  if (ldx < K || ldy < N) return FP_ERR_STRIDE;
  return FP_OK;
}

// B, T, heads and head size of an attention call: sizes that keep every grid
// (in threads) and row index within 32 bits.
int check_attention(int64_t B, int64_t T, int64_t Hq, int64_t Hk, int64_t D) {
  if (B < 1 || T < 1 || Hk < 1 || Hq < Hk || Hq % Hk != 0 || (D != 64 && D != 128))
    return FP_ERR_SHAPE;
  if (B > 65535 || Hq > 65535 || B * Hk > 65535 || T > (int64_t)1 << 24 ||
      B * T > (int64_t)1 << 27 || B * T * (Hq + 2 * Hk) > (int64_t)1 << 27)
    return FP_ERR_SHAPE;
  return FP_OK;
}

// A dimension of a strided layout, in elements.
struct Dim {
  int64_t size, stride;
};

// Elements from the first to the last, if every dimension's stride passes over
// all that the smaller ones reach (inner: the contiguous elements below them);
// else -1: two indices may be one element.
template <int N>
int64_t nested_extent(Dim (&d)[N], int64_t inner) {
  for (int i = 1; i < N; ++i)
    for (int j = i; j > 0 && d[j].stride < d[j - 1].stride; --j) {
      const Dim t = d[j];
      d[j] = d[j - 1], d[j - 1] = t;
    }
  int64_t extent = inner;
  for (const Dim& x : d) {
    if (x.size <= 1) continue;
    if (x.stride < extent) return -1;
    extent += (x.size - 1) * x.stride;
  }
  return extent;
}

// Whether a call could write one cache element for two (sequence, head,
// position) or as a key and as a value, or write what it reads as q, k or v:
// its workgroups run in no order. Keys and values may interleave (a cache
// [B][S][2][heads][D]) when their strides are the same.
bool attention_overlaps(const fp_attention_args& g) {
  const int64_t D = g.head_dim;
  Dim k[] = {{g.B, g.k_s_b}, {g.n_kv_heads, g.k_s_h}, {g.cache_len, g.k_s_p}};
  Dim v[] = {{g.B, g.v_s_b}, {g.n_kv_heads, g.v_s_h}, {g.cache_len, g.v_s_p}};
  const auto same = [](int64_t size, int64_t a, int64_t b) { return size <= 1 || a == b; };
  const bool alike = same(g.B, g.k_s_b, g.v_s_b) && same(g.n_kv_heads, g.k_s_h, g.v_s_h) &&
                     same(g.cache_len, g.k_s_p, g.v_s_p);
  const int64_t ek = nested_extent(k, D), ev = nested_extent(v, D);
  if (ek < 0 || ev < 0) return true;
  const uintptr_t kp = (uintptr_t)g.cache_k, vp = (uintptr_t)g.cache_v;
  const auto meet = [](uintptr_t a, int64_t na, uintptr_t b, int64_t nb) {
    return a < b + 2 * (uintptr_t)nb && b < a + 2 * (uintptr_t)na;
  };
  if (meet(kp, ek, vp, ev)) {
    Dim kv[] = {{2, (int64_t)(kp < vp ? vp - kp : kp - vp) / 2}, k[0], k[1], k[2]};
    if (!alike || nested_extent(kv, D) < 0) return true;
  }
  const int64_t last = g.B * g.T - 1;
  const struct { const void* p; int64_t n; } in[] = {{g.q, last * g.ldq + g.n_heads * D},
                                                     {g.k, last * g.ldk + g.n_kv_heads * D},
                                                     {g.v, last * g.ldv + g.n_kv_heads * D}};
  for (const auto& i : in)
    if (meet(kp, ek, (uintptr_t)i.p, i.n) || meet(vp, ev, (uintptr_t)i.p, i.n)) return true;
  return false;
}

}  // namespace

int rmsnorm_qkv_args(const void* x, int64_t ldx, const void* gamma, float eps, const void* w,
                     int64_t ldw, const void* y, int64_t ldy, int64_t M, int64_t n_q, int64_t n_k,
                     int64_t K) {
  if (n_q < 1 || n_k < 0) return FP_ERR_SHAPE;
  int st = check_common(M, n_q + 2 * n_k, K, ldx, ldy);
  if (st) return st;
  if (ldw < K) return FP_ERR_STRIDE;
  if ((st = check_norm(eps, nullptr, 0))) return st;
  if (M > 0 && (!x || !gamma || !w || !y)) return FP_ERR_NULL;
  return FP_OK;
}

}  // namespace fp

using fp::StreamArgs;

extern "C" {

const char* fp_status_string(int status) {
  switch (status) {
    case FP_OK: return "ok";
    case FP_ERR_NULL: return "a required pointer is NULL";
    case FP_ERR_SHAPE: return "shape out of range or inconsistent (M, N, K, n_q, n_k)";
    case FP_ERR_STRIDE: return "row stride smaller than the row length";
    case FP_ERR_LAUNCH: return "HIP kernel launch failed";
    case FP_ERR_DEVICE: return "no gfx950 code object for the current device";
    case FP_ERR_WORKSPACE: return "workspace missing, too small or not 16-byte aligned, or a negative workspace size";
    case FP_ERR_SCRATCH: return "the call needs more than the library's static scratch (FP_SCRATCH_BYTES); use the workspace entry point";
    default: return "unknown fp_status";
  }
}

int fp_abi_version(void) { return (1 << 16) | 6; }

int64_t fp_workspace_bytes(int64_t M, int64_t N, int64_t K, int gate_up) {
  if (M < 1 || N < 1 || K < 1) return 0;
  const fp::GemmSplit p = fp::gemm_split_plan_bf16(M, N, K, gate_up != 0);
  return 4 * fp::gemm_split_ws_floats(p, M, N, K, gate_up != 0);
}

int fp_qkv_bf16_ws(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y, int64_t ldy,
                   int64_t M, int64_t n_q, int64_t n_k, int64_t K, void* workspace,
                   int64_t workspace_bytes, void* stream) {
  if (n_q < 1 || n_k < 0) return FP_ERR_SHAPE;
  const int64_t N = n_q + 2 * n_k;
  int st = fp::check_common(M, N, K, ldx, ldy);
  if (st) return st;
  if (ldw < K) return FP_ERR_STRIDE;
  if (workspace_bytes < 0 || (workspace && !fp::al16(workspace))) return FP_ERR_WORKSPACE;
  if (M == 0) return FP_OK;
  if (!x || !w || !y) return FP_ERR_NULL;
  StreamArgs a{(const uint16_t*)x, ldx, w, ldw, nullptr, 0, nullptr, nullptr,
               (uint16_t*)y, ldy, M, N, K, (float*)workspace, workspace_bytes / 4};
  const bool aligned = (K % 8 == 0) && (ldx % 8 == 0) && (ldw % 8 == 0) &&
                       fp::al16(x) && fp::al16(w);
  return fp::run<false, false>(a, aligned, (hipStream_t)stream);
}

int fp_qkv_bf16(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y, int64_t ldy,
                int64_t M, int64_t n_q, int64_t n_k, int64_t K, void* stream) {
  return fp_qkv_bf16_ws(x, ldx, w, ldw, y, ldy, M, n_q, n_k, K, nullptr, 0, stream);
}

int fp_gate_up_silu_bf16_ws(const void* x, int64_t ldx, const void* wg, int64_t ldwg,
                            const void* wu, int64_t ldwu, void* y, int64_t ldy, int64_t M,
                            int64_t N, int64_t K, void* workspace, int64_t workspace_bytes,
                            void* stream) {
  int st = fp::check_common(M, N, K, ldx, ldy);
  if (st) return st;
  if (ldwg < K || ldwu < K) return FP_ERR_STRIDE;
  if (workspace_bytes < 0 || (workspace && !fp::al16(workspace))) return FP_ERR_WORKSPACE;
  if (M == 0) return FP_OK;
  if (!x || !wg || !wu || !y) return FP_ERR_NULL;
  StreamArgs a{(const uint16_t*)x, ldx, wg, ldwg, wu, ldwu, nullptr, nullptr,
               (uint16_t*)y, ldy, M, N, K, (float*)workspace, workspace_bytes / 4};
  const bool aligned = (K % 8 == 0) && (ldx % 8 == 0) && (ldwg % 8 == 0) && (ldwu % 8 == 0) &&
                       fp::al16(x) && fp::al16(wg) && fp::al16(wu);
  return fp::run<true, false>(a, aligned, (hipStream_t)stream);
}

int fp_gate_up_silu_bf16(const void* x, int64_t ldx, const void* wg, int64_t ldwg,
                         const void* wu, int64_t ldwu, void* y, int64_t ldy,
                         int64_t M, int64_t N, int64_t K, void* stream) {
  return fp_gate_up_silu_bf16_ws(x, ldx, wg, ldwg, wu, ldwu, y, ldy, M, N, K, nullptr, 0,
                                 stream);
}

int64_t fp_workspace_bytes_w8(int64_t M, int64_t N, int64_t K, int gate_up) {
  return fp::w8_workspace_bytes(M, N, K, gate_up != 0);
}

int fp_qkv_w8_ws(const void* x, int64_t ldx, const int8_t* q, int64_t ldq, const float* scale,
                 void* y, int64_t ldy, int64_t M, int64_t n_q, int64_t n_k, int64_t K,
                 void* workspace, int64_t workspace_bytes, void* stream) {
  if (n_q < 1 || n_k < 0) return FP_ERR_SHAPE;
  const int64_t N = n_q + 2 * n_k;
  int st = fp::check_common(M, N, K, ldx, ldy);
  if (st) return st;
  if (ldq < K) return FP_ERR_STRIDE;
  if (workspace_bytes < 0 || (workspace && !fp::al16(workspace))) return FP_ERR_WORKSPACE;
  if (M == 0) return FP_OK;
  if (!x || !q || !scale || !y) return FP_ERR_NULL;
  StreamArgs a{(const uint16_t*)x, ldx, q, ldq, nullptr, 0, scale, nullptr,
               (uint16_t*)y, ldy, M, N, K};
  const bool aligned = (K % 16 == 0) && (ldx % 8 == 0) && (ldq % 16 == 0) &&
                       fp::al16(x) && fp::al16(q);
  return fp::run_w8<false>(a, aligned, workspace, workspace_bytes, (hipStream_t)stream);
}

int fp_qkv_w8(const void* x, int64_t ldx, const int8_t* q, int64_t ldq, const float* scale,
              void* y, int64_t ldy, int64_t M, int64_t n_q, int64_t n_k, int64_t K,
              void* stream) {
  return fp_qkv_w8_ws(x, ldx, q, ldq, scale, y, ldy, M, n_q, n_k, K, nullptr, 0, stream);
}

int fp_gate_up_silu_w8_ws(const void* x, int64_t ldx, const int8_t* qg, int64_t ldqg,
                          const float* sg, const int8_t* qu, int64_t ldqu, const float* su,
                          void* y, int64_t ldy, int64_t M, int64_t N, int64_t K,
                          void* workspace, int64_t workspace_bytes, void* stream) {
  int st = fp::check_common(M, N, K, ldx, ldy);
  if (st) return st;
  if (ldqg < K || ldqu < K) return FP_ERR_STRIDE;
  if (workspace_bytes < 0 || (workspace && !fp::al16(workspace))) return FP_ERR_WORKSPACE;
  if (M == 0) return FP_OK;
  if (!x || !qg || !sg || !qu || !su || !y) return FP_ERR_NULL;
  StreamArgs a{(const uint16_t*)x, ldx, qg, ldqg, qu, ldqu, sg, su,
               (uint16_t*)y, ldy, M, N, K};
  const bool aligned = (K % 16 == 0) && (ldx % 8 == 0) && (ldqg % 16 == 0) &&
                       (ldqu % 16 == 0) && fp::al16(x) && fp::al16(qg) && fp::al16(qu);
  return fp::run_w8<true>(a, aligned, workspace, workspace_bytes, (hipStream_t)stream);
}

int fp_gate_up_silu_w8(const void* x, int64_t ldx, const int8_t* qg, int64_t ldqg,
                       const float* sg, const int8_t* qu, int64_t ldqu, const float* su,
                       void* y, int64_t ldy, int64_t M, int64_t N, int64_t K, void* stream) {
  return fp_gate_up_silu_w8_ws(x, ldx, qg, ldqg, sg, qu, ldqu, su, y, ldy, M, N, K, nullptr, 0,
                               stream);
}

int fp_linear_bf16(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y, int64_t ldy,
                   int64_t M, int64_t N, int64_t K, void* stream) {
  return fp_qkv_bf16(x, ldx, w, ldw, y, ldy, M, N, 0, K, stream);
}

int fp_linear_bf16_ws(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y,
                      int64_t ldy, int64_t M, int64_t N, int64_t K, void* workspace,
                      int64_t workspace_bytes, void* stream) {
  return fp_qkv_bf16_ws(x, ldx, w, ldw, y, ldy, M, N, 0, K, workspace, workspace_bytes, stream);
}

int fp_linear_w8(const void* x, int64_t ldx, const int8_t* q, int64_t ldq, const float* scale,
                 void* y, int64_t ldy, int64_t M, int64_t N, int64_t K, void* stream) {
  return fp_qkv_w8(x, ldx, q, ldq, scale, y, ldy, M, N, 0, K, stream);
}

int fp_linear_w8_ws(const void* x, int64_t ldx, const int8_t* q, int64_t ldq, const float* scale,
                    void* y, int64_t ldy, int64_t M, int64_t N, int64_t K, void* workspace,
                    int64_t workspace_bytes, void* stream) {
  return fp_qkv_w8_ws(x, ldx, q, ldq, scale, y, ldy, M, N, 0, K, workspace, workspace_bytes,
                      stream);
}

int64_t fp_rmsnorm_workspace_bytes(int64_t M, int64_t N, int64_t K, int gate_up, int int8) {
  if (M < 1 || N < 1 || K < 1) return 0;
  const bool w8 = int8 != 0;
  // Room for the normalised rows always: decode-sized calls usually run as
  // one launch and leave it unused, but take the two-launch path when a
  // pointer or stride misses the 16-byte alignment of that launch. There the
  // plain dispatch (bf16 M <= 2, int8 M <= 4) needs no further workspace.
  int64_t b = fp::round_up(M * K * 2, 256);
  if (M <= (w8 ? fp::kRowsMaxM : 2) && K % (w8 ? 16 : 8) == 0 && fp::rows_fit(M, K, w8, true))
    return b;
  if (w8) return b + fp::w8_workspace_bytes(M, N, K, gate_up != 0);
  return b + 4 * fp::gemm_split_ws_floats(fp::gemm_split_plan_bf16(M, N, K, gate_up != 0), M, N,
                                          K, gate_up != 0);
}

int fp_rmsnorm_qkv_bf16(const void* x, int64_t ldx, const void* gamma, float eps, const void* w,
                        int64_t ldw, void* y, int64_t ldy, int64_t M, int64_t n_q, int64_t n_k,
                        int64_t K, void* workspace, int64_t workspace_bytes, void* stream) {
  int st = fp::rmsnorm_qkv_args(x, ldx, gamma, eps, w, ldw, y, ldy, M, n_q, n_k, K);
  if (st) return st;
  if ((st = fp::check_norm(eps, workspace, workspace_bytes))) return st;
  if (M == 0) return FP_OK;
  const int64_t N = n_q + 2 * n_k;
  StreamArgs a{(const uint16_t*)x, ldx, w, ldw, nullptr, 0, nullptr, nullptr, (uint16_t*)y, ldy,
               M, N, K, nullptr, 0, (const uint16_t*)gamma, eps};
  const bool xal = K % 8 == 0 && ldx % 8 == 0 && fp::al16(x);
  const bool wal = ldw % 8 == 0 && fp::al16(w);
  return fp::run_norm<false, false>(a, xal, wal, workspace, workspace_bytes, (hipStream_t)stream);
}

int fp_rmsnorm_gate_up_silu_bf16(const void* x, int64_t ldx, const void* gamma, float eps,
                                 const void* wg, int64_t ldwg, const void* wu, int64_t ldwu,
                                 void* y, int64_t ldy, int64_t M, int64_t N, int64_t K,
                                 void* workspace, int64_t workspace_bytes, void* stream) {
  int st = fp::check_common(M, N, K, ldx, ldy);
  if (st) return st;
  if (ldwg < K || ldwu < K) return FP_ERR_STRIDE;
  if ((st = fp::check_norm(eps, workspace, workspace_bytes))) return st;
  if (M == 0) return FP_OK;
  if (!x || !gamma || !wg || !wu || !y) return FP_ERR_NULL;
  StreamArgs a{(const uint16_t*)x, ldx, wg, ldwg, wu, ldwu, nullptr, nullptr, (uint16_t*)y, ldy,
               M, N, K, nullptr, 0, (const uint16_t*)gamma, eps};
  const bool xal = K % 8 == 0 && ldx % 8 == 0 && fp::al16(x);
  const bool wal = ldwg % 8 == 0 && ldwu % 8 == 0 && fp::al16(wg) && fp::al16(wu);
  return fp::run_norm<true, false>(a, xal, wal, workspace, workspace_bytes, (hipStream_t)stream);
}

int fp_rmsnorm_qkv_w8(const void* x, int64_t ldx, const void* gamma, float eps, const int8_t* q,
                      int64_t ldq, const float* scale, void* y, int64_t ldy, int64_t M,
                      int64_t n_q, int64_t n_k, int64_t K, void* workspace,
                      int64_t workspace_bytes, void* stream) {
  if (n_q < 1 || n_k < 0) return FP_ERR_SHAPE;
  const int64_t N = n_q + 2 * n_k;
  int st = fp::check_common(M, N, K, ldx, ldy);
  if (st) return st;
  if (ldq < K) return FP_ERR_STRIDE;
  if ((st = fp::check_norm(eps, workspace, workspace_bytes))) return st;
  if (M == 0) return FP_OK;
  if (!x || !gamma || !q || !scale || !y) return FP_ERR_NULL;
  StreamArgs a{(const uint16_t*)x, ldx, q, ldq, nullptr, 0, scale, nullptr, (uint16_t*)y, ldy,
               M, N, K, nullptr, 0, (const uint16_t*)gamma, eps};
  const bool xal = K % 16 == 0 && ldx % 8 == 0 && fp::al16(x);
  const bool wal = ldq % 16 == 0 && fp::al16(q);
  return fp::run_norm<false, true>(a, xal, wal, workspace, workspace_bytes, (hipStream_t)stream);
}

int fp_rmsnorm_gate_up_silu_w8(const void* x, int64_t ldx, const void* gamma, float eps,
                               const int8_t* qg, int64_t ldqg, const float* sg, const int8_t* qu,
                               int64_t ldqu, const float* su, void* y, int64_t ldy, int64_t M,
                               int64_t N, int64_t K, void* workspace, int64_t workspace_bytes,
                               void* stream) {
  int st = fp::check_common(M, N, K, ldx, ldy);
  if (st) return st;
  if (ldqg < K || ldqu < K) return FP_ERR_STRIDE;
  if ((st = fp::check_norm(eps, workspace, workspace_bytes))) return st;
  if (M == 0) return FP_OK;
  if (!x || !gamma || !qg || !sg || !qu || !su || !y) return FP_ERR_NULL;
  StreamArgs a{(const uint16_t*)x, ldx, qg, ldqg, qu, ldqu, sg, su, (uint16_t*)y, ldy,
               M, N, K, nullptr, 0, (const uint16_t*)gamma, eps};
  const bool xal = K % 16 == 0 && ldx % 8 == 0 && fp::al16(x);
  const bool wal = ldqg % 16 == 0 && ldqu % 16 == 0 && fp::al16(qg) && fp::al16(qu);
  return fp::run_norm<true, true>(a, xal, wal, workspace, workspace_bytes, (hipStream_t)stream);
}

int64_t fp_attention_workspace_bytes(int64_t B, int64_t T, int64_t n_heads, int64_t n_kv_heads,
                                     int64_t head_dim, int64_t keys) {
  if (fp::check_attention(B, T, n_heads, n_kv_heads, head_dim) || keys < 1) return 0;
  return fp::attn_workspace_bytes(B, T, n_heads, n_kv_heads, head_dim, keys);
}

int fp_attention_bf16(const fp_attention_args* g, void* workspace, int64_t workspace_bytes,
                      void* stream) {
  if (!g) return FP_ERR_NULL;
  const int64_t D = g->head_dim, S = g->cache_len, T = g->T;
  int st = fp::check_attention(g->B, T, g->n_heads, g->n_kv_heads, D);
  if (st) return st;
  if (S < 1 || S > (int64_t)1 << 30) return FP_ERR_SHAPE;
  if (!g->pos_dev && (g->pos < 0 || g->pos + T > S)) return FP_ERR_SHAPE;
  if (!(g->q_eps >= 0.f) || !(g->k_eps >= 0.f)) return FP_ERR_SHAPE;
  if (g->ldq < g->n_heads * D || g->ldk < g->n_kv_heads * D || g->ldv < g->n_kv_heads * D ||
      g->ld_cos < D || g->ld_sin < D || g->k_s_p < D || g->v_s_p < D || g->k_s_b < 0 ||
      g->k_s_h < 0 || g->v_s_b < 0 || g->v_s_h < 0)
    return FP_ERR_STRIDE;
  const int64_t any4 = g->ldq | g->ldk | g->ldv;
  const int64_t any8 = g->k_s_b | g->k_s_h | g->k_s_p | g->v_s_b | g->v_s_h | g->v_s_p;
  if ((any4 & 3) || (any8 & 7)) return FP_ERR_STRIDE;
  constexpr int64_t kLim = (int64_t)1 << 31;
  if ((S + 64) * g->k_s_p * 2 >= kLim || (S + 64) * g->v_s_p * 2 >= kLim) return FP_ERR_SHAPE;
  if (!g->q || !g->k || !g->v || !g->cos || !g->sin || !g->cache_k || !g->cache_v || !g->y)
    return FP_ERR_NULL;
  if (!g->q_gamma != !g->k_gamma) return FP_ERR_NULL;
  const auto al8 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7) == 0; };
  if (!al8(g->q) || !al8(g->k) || !al8(g->v) || !al8(g->q_gamma) || !al8(g->k_gamma) ||
      !al8(g->y) || !fp::al16(g->cache_k) || !fp::al16(g->cache_v))
    return FP_ERR_STRIDE;
  if (fp::attention_overlaps(*g)) return FP_ERR_STRIDE;
  const int64_t keys = g->pos_dev ? S : g->pos + T;
  if (!workspace || !fp::al16(workspace) ||
      workspace_bytes < fp::attn_workspace_bytes(g->B, T, g->n_heads, g->n_kv_heads, D, keys))
    return FP_ERR_WORKSPACE;
  fp::AttnArgs a{};
  a.q = (const uint16_t*)g->q, a.k = (const uint16_t*)g->k, a.v = (const uint16_t*)g->v;
  a.ldq = g->ldq, a.ldk = g->ldk, a.ldv = g->ldv;
  a.gq = (const uint16_t*)g->q_gamma, a.gk = (const uint16_t*)g->k_gamma;
  a.epsq = g->q_eps, a.epsk = g->k_eps;
  a.cos = (const uint16_t*)g->cos, a.sin = (const uint16_t*)g->sin;
  a.ldc = g->ld_cos, a.lds = g->ld_sin;
  a.ck = (uint16_t*)g->cache_k, a.cv = (uint16_t*)g->cache_v;
  a.ckb = g->k_s_b, a.ckh = g->k_s_h, a.cks = g->k_s_p;
  a.cvb = g->v_s_b, a.cvh = g->v_s_h, a.cvs = g->v_s_p;
  a.y = (uint16_t*)g->y;
  a.B = (int)g->B, a.T = (int)T, a.Hq = (int)g->n_heads, a.Hk = (int)g->n_kv_heads, a.S = (int)S;
  a.pos = g->pos;
  a.pos_dev = g->pos_dev;
  return fp::launch_status(fp::launch_attention(a, D, keys, workspace, (hipStream_t)stream));
}

int fp_quantize_w8_per_row(const void* w, int64_t ldw, int8_t* q, int64_t ldq, float* scale,
                           int64_t N, int64_t K, void* stream) {
  if (N < 0 || K < 1 || N > ((int64_t)1 << 31) - 1) return FP_ERR_SHAPE;
  if (ldw < K || ldq < K) return FP_ERR_STRIDE;
  if (N == 0) return FP_OK;
  if (!w || !q || !scale) return FP_ERR_NULL;
  const dim3 grid((unsigned)N), block(256);
  const hipStream_t hs = (hipStream_t)stream;
  const uint16_t* wp = (const uint16_t*)w;
  // Two passes for rows of more than 8 chunks per thread, bases off an element
  // boundary, and short rows, where only a few of a workgroup's threads would hold a
  // chunk of 8 and each divides 8 times (300 shapes, one pass against two: K of 50-99
  // 1.3-1.7 of the time, 500-649 1.1-1.3, 950-1099 0.97-1.02, 1500 0.76).
  if (K > 8 * 2048 - 7 || K < 1024 || (reinterpret_cast<uintptr_t>(w) & 1))
    hipLaunchKernelGGL(fp::quantize_w8_kernel, grid, block, 0, hs, wp, ldw, q, ldq, scale, K);
  else if (K <= 2048 - 7)
    hipLaunchKernelGGL(fp::quantize_w8_row_kernel<1>, grid, block, 0, hs, wp, ldw, q, ldq, scale, (int)K);
  else if (K <= 2 * 2048 - 7)
    hipLaunchKernelGGL(fp::quantize_w8_row_kernel<2>, grid, block, 0, hs, wp, ldw, q, ldq, scale, (int)K);
  else if (K <= 3 * 2048 - 7)
    hipLaunchKernelGGL(fp::quantize_w8_row_kernel<3>, grid, block, 0, hs, wp, ldw, q, ldq, scale, (int)K);
  else if (K <= 5 * 2048 - 7)
    hipLaunchKernelGGL(fp::quantize_w8_row_kernel<5>, grid, block, 0, hs, wp, ldw, q, ldq, scale, (int)K);
  else
    hipLaunchKernelGGL(fp::quantize_w8_row_kernel<8>, grid, block, 0, hs, wp, ldw, q, ldq, scale, (int)K);
  return fp::launch_status((int)hipGetLastError());
}

}  // extern "C"
