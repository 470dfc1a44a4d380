// fp_attn.hip — what follows the QKV projection in an attention layer, up to
// the o projection: QK-norm, RoPE, the KV-cache write and causal softmax
// attention over the cache (reference src/kernels/fused_qkv.py:242-282), as
// two or three launches instead of ~45 torch ones.
//
//   - attn_prep_kernel: RMS-normalises (fp32 statistics) and rotates every q
//     and k head at torch's rounding points, writes q to the workspace and the
//     new k and v rows into the cache.
//   - attn_rows_kernel (T * group <= 64 query rows per kv head: decode and
//     spec-verify) and attn_tiles_kernel (prompts): attention of the q rows of
//     one kv head's group over that head's keys. The GQA group's heads are
//     packed into the row dimension, so a key is read once for all of them and
//     never expanded. Keys may be split over workgroups (fp32 partials).
//   - attn_combine_kernel: sums the partials of a split in split order.
//
// Both attention kernels compute S^T = K Q^T with keys as the A operand of
// v_mfma_f32_16x16x32_bf16, so that a lane's accumulators are four keys of one
// query row (column lane % 16): a row's softmax statistics then live in its
// lane column, and its probabilities are already the B operand of
// O^T = V^T P^T, whose 32-wide k index is any fixed order of the keys: lane
// group g takes keys 4g .. 4g+3 and 16 + 4g .. 16 + 4g+3. V^T comes out of the
// row-major V rows in LDS by ds_read_b64_tr_b16 in that same order.
//
// Precision: scores are exact bf16 products summed in fp32, softmax is in
// fp32, and the fp32 probabilities enter the matrix core as three bf16 parts
// (p = hi + mid + lo to within 2^-27 p), so p.V is a sum of fp32-precise
// products as in an fp32 matmul. Where a V tile holds an infinity or a NaN the
// mid and lo parts (zero for many p) meet V with those entries zeroed, so that
// inf * p stays inf.
//
// Every output's sums run in a fixed order (it depends on the sizes only).
//
// Measured on MI355X, Qwen3-4B heads (32 over 8 of 128), the torch form against
// this one: one token at position 2047, the whole attention layer called
// eagerly 313 -> 43 us (kernels alone 200 -> 33, of which the two projections
// 16); a 1000-token prompt 701 -> 127 us (the core 620 -> 55, attn_tiles_kernel
// 45: 8.2 GFLOP of visible pairs, which the three parts of p make 16.4, and the
// softmax's VALU work about as much again); a 4-layer graph decode step with
// the tied head 1468 -> 553 us. Against 64 bits the layer's error is unchanged.
#include "fp_common.h"
#include "fp_launch.h"
#include "fp_norm.h"

namespace fp {

namespace {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* lds_s16x4_t;

constexpr int kAttnMaxSplit = 64;  // one lane per split in attn_combine_kernel
constexpr float kLog2e = 1.4426950408889634f;

constexpr int vmcnt_imm(int v) { return (v & 15) | (7 << 4) | (15 << 8) | ((v >> 4) << 14); }

// 16 bytes per lane from base + voff into LDS at dst + 16 * lane; bytes at or
// past nbytes read as zero.
__device__ __forceinline__ void load_lds16(const void* base, int nbytes, lds_ptr_t dst,
                                           uint32_t voff) {
  constexpr int kRsrcFlags = 0x00020000;  // raw buffer, 32-bit data format
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, nbytes, kRsrcFlags), dst, 16,
      voff, 0, 0, 0);
}
__device__ __forceinline__ u32x4 load_buf16(const void* base, int nbytes, uint32_t voff) {
  constexpr int kRsrcFlags = 0x00020000;
  return __builtin_amdgcn_raw_buffer_load_b128(
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, nbytes, kRsrcFlags), voff,
      0, 0);
}

// First position of the call's tokens (a device position far outside any cache
// stays outside, within 32-bit arithmetic).
__device__ __forceinline__ int first_pos(const AttnArgs& a) {
  constexpr int64_t kFar = 1 << 30;
  const int64_t p = a.pos_dev ? *a.pos_dev : a.pos;
  return (int)(p < -kFar ? -kFar : p > kFar ? kFar : p);
}

// Sum over the LPH (8 or 16) consecutive lanes of a head.
template <int LPH>
__device__ __forceinline__ float head_sum(float v) {
  v += dpp_f32<0xb1>(v);                            // quad_perm [1,0,3,2]
  v += dpp_f32<0x4e>(v);                            // quad_perm [2,3,0,1]
  v += dpp_f32<0x141>(v);                           // row_half_mirror: sums of 8
  if constexpr (LPH == 16) v += dpp_f32<0x140>(v);  // row_mirror: sums of 16
  return v;
}

// One head row per LPH = D / 8 lanes: lane j holds elements 4j .. 4j+3 of the
// first half and of the second, so a rotate-half pair sits in one lane.
// gamma NULL: no norm (the caller has normalised q and k).
template <int D>
__global__ __launch_bounds__(256) void attn_prep_kernel(AttnArgs a) {
  constexpr int LPH = D / 8;
  const int heads = a.Hq + 2 * a.Hk;
  const int64_t items = (int64_t)a.B * a.T * heads;
  int64_t item = (int64_t)blockIdx.x * (256 / LPH) + threadIdx.x / LPH;
  const bool live = item < items;  // dead lanes stay for the cross-lane sums
  if (!live) item = items - 1;
  const int j = threadIdx.x % LPH;
  const int64_t m = item / heads;
  const int h = (int)(item - m * heads);
  const int64_t b = m / a.T, t = m - b * a.T;
  const bool isq = h < a.Hq, isk = !isq && h < a.Hq + a.Hk;
  const int hk = isk ? h - a.Hq : h - a.Hq - a.Hk;  // cache head of k and v
  const uint16_t* src = isq   ? a.q + m * a.ldq + (int64_t)h * D
                        : isk ? a.k + m * a.ldk + (int64_t)hk * D
                              : a.v + m * a.ldv + (int64_t)hk * D;
  u32x2 lo = *reinterpret_cast<const u32x2*>(src + 4 * j);
  u32x2 hi = *reinterpret_cast<const u32x2*>(src + D / 2 + 4 * j);
  const uint16_t* g = isq ? a.gq : a.gk;
  if (isq || isk) {
    uint32_t x[8] = {lo.x & 0xffffu, lo.x >> 16, lo.y & 0xffffu, lo.y >> 16,
                     hi.x & 0xffffu, hi.x >> 16, hi.y & 0xffffu, hi.y >> 16};
    if (g) {
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float f = bf16_bits_to_f32(x[e]);
        s += __fmul_rn(f, f);
      }
      const float r = rms_scale(head_sum<LPH>(s), D, isq ? a.epsq : a.epsk);
      const u32x2 gl = *reinterpret_cast<const u32x2*>(g + 4 * j);
      const u32x2 gh = *reinterpret_cast<const u32x2*>(g + D / 2 + 4 * j);
      const uint32_t gb[8] = {gl.x & 0xffffu, gl.x >> 16, gl.y & 0xffffu, gl.y >> 16,
                              gh.x & 0xffffu, gh.x >> 16, gh.y & 0xffffu, gh.y >> 16};
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = norm_bf16(x[e], gb[e], r);
    }
    // RoPE, each product and the sum rounded to bf16 as torch's bf16 ops do
    const uint16_t* cr = a.cos + t * a.ldc;
    const uint16_t* sr = a.sin + t * a.lds;
    uint32_t y[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x1 = bf16_bits_to_f32(x[e]), x2 = bf16_bits_to_f32(x[4 + e]);
      const int d = 4 * j + e;
      const float c1 = bf16_bits_to_f32(cr[d]), c2 = bf16_bits_to_f32(cr[D / 2 + d]);
      const float s1 = bf16_bits_to_f32(sr[d]), s2 = bf16_bits_to_f32(sr[D / 2 + d]);
      y[e] = f32_to_bf16_bits(round_bf16(__fmul_rn(x1, c1)) + round_bf16(__fmul_rn(-x2, s1)));
      y[4 + e] = f32_to_bf16_bits(round_bf16(__fmul_rn(x2, c2)) + round_bf16(__fmul_rn(x1, s2)));
    }
    lo = u32x2{y[0] | (y[1] << 16), y[2] | (y[3] << 16)};
    hi = u32x2{y[4] | (y[5] << 16), y[6] | (y[7] << 16)};
  }
  uint16_t* dst;
  if (isq) {
    dst = a.qn + (m * a.Hq + h) * D;
  } else {
    const int64_t p = first_pos(a) + t;
    if (p < 0 || p >= a.S) return;  // a device position outside the cache
    dst = isk ? a.ck + b * a.ckb + hk * a.ckh + p * a.cks : a.cv + b * a.cvb + hk * a.cvh + p * a.cvs;
  }
  if (!live) return;
  *reinterpret_cast<u32x2*>(dst + 4 * j) = lo;
  *reinterpret_cast<u32x2*>(dst + D / 2 + 4 * j) = hi;
}

// ---- shared pieces of the two attention kernels ---------------------------

// Row stride of the partial planes' statistics: {m, l} per row.
__device__ __forceinline__ int64_t part_row(const AttnArgs& a, int split, int bh, int64_t rr) {
  return ((int64_t)split * a.B * a.Hk + bh) * ((int64_t)a.T * (a.Hq / a.Hk)) + rr;
}

// 32 keys' probabilities of one row column (p[0]: keys 4g .. 4g+3, p[1]: keys
// 16 + 4g ..) as three bf16 B operands, p = f[0] + f[1] + f[2].
__device__ __forceinline__ void split_p(const f32x4& p0, const f32x4& p1, u32x4 f[3]) {
  const float p[8] = {p0[0], p0[1], p0[2], p0[3], p1[0], p1[1], p1[2], p1[3]};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float x = p[2 * i], y = p[2 * i + 1];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const uint32_t h = cvt_bf16x2(x, y);
      f[c][i] = h;
      if (c < 2) {
        x -= __uint_as_float(h << 16);  // exact
        y -= __uint_as_float(h & 0xffff0000u);
      }
    }
  }
}

// Whether any of the eight bf16 is an infinity or a NaN: both halves' |x|
// compared with 0x7f80 through the carry of 0x7fff - that.
__device__ __forceinline__ bool nonfinite8(u32x4 v) {
  uint32_t any = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) any |= ((v[i] & 0x7fff7fffu) + 0x00800080u);
  return (any & 0x80008000u) != 0;
}
// The same with those entries replaced by zero.
__device__ __forceinline__ u32x4 zero_nonfinite8(u32x4 v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t bad = ((v[i] & 0x7fff7fffu) + 0x00800080u) & 0x80008000u;
    // 0x8000 -> 0xffff in each half
    v[i] &= ~((bad >> 15) * 0xffffu);
  }
  return v;
}

// A operand of V^T for d block dt and keys {4g .. 4g+3, 16 + 4g ..} of 32 V
// rows in LDS (row stride D * 2 bytes, 16-byte chunk c of row r at
// c ^ (r & (D / 8 - 1)): two passes over the banks, the least for 512 bytes).
template <int D>
__device__ __forceinline__ u32x4 read_vt(const char* rows, int dt, int li, int grp) {
  constexpr int CM = D / 8 - 1;
  const int key = 4 * grp + (li >> 2), c = 2 * dt + ((li & 3) >> 1), half = (li & 1) * 8;
  u32x4 out;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int r = key + 16 * s;
    const char* p = rows + r * (D * 2) + ((c ^ (r & CM)) * 16) + half;
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)p);
    const u32x2 w = __builtin_bit_cast(u32x2, v);
    out[2 * s] = w.x;
    out[2 * s + 1] = w.y;
  }
  return out;
}

// max / sum over the four lane groups that share a row column (xor 16, 32).
__device__ __forceinline__ float col_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 16));
  return fmaxf(v, __shfl_xor(v, 32));
}
__device__ __forceinline__ float col_sum(float v) {
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// ---- decode and verify ----------------------------------------------------
//
// Latency-bound: a few MB of cache per call. A workgroup takes one kv head of
// one sequence, 16 * RT query rows (token t, group head h at row t * G + h)
// and one contiguous range of 32-key chunks; its four waves take chunks w,
// w + 4, ... of the range (so 128 keys keep every wave busy), each with the
// next chunk's keys in registers and values in its own LDS buffer while it
// computes, and the waves' softmax states are merged through LDS in wave order.
template <int D, int RT>
__global__ __launch_bounds__(256) void attn_rows_kernel(AttnArgs a) {
  constexpr int NW = 4, KC = 32;
  constexpr int DK = D / 32, DT = D / 16;      // k-steps of q.k, d blocks of p.V
  constexpr int RPI = 1024 / (D * 2);          // V rows per load instruction
  constexpr int NV = KC / RPI, NK = 2 * DK;    // V and K load instructions per chunk
  constexpr int CH = D / 8;                    // 16-byte chunks per row
  __shared__ __attribute__((aligned(1024))) char sV0[NW][KC * D * 2];
  __shared__ __attribute__((aligned(1024))) char sV1[NW][KC * D * 2];
  __shared__ float sM[NW][16 * RT], sL[NW][16 * RT];

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int li = lane & 15, grp = lane >> 4;
  const int G = a.Hq / a.Hk, rows = a.T * G;
  const int bh = blockIdx.y, b = bh / a.Hk, kh = bh - b * a.Hk;
  const int row0 = blockIdx.z * 16 * RT;
  const int p0 = first_pos(a), pend = p0 + a.T;
  const int end = pend < 0 ? 0 : pend < a.S ? pend : a.S;  // keys in the cache
  // this split's chunks
  const int nc = (end + KC - 1) / KC;
  const int per = (nc + a.nsplit - 1) / a.nsplit;
  const int c_lo = (int)blockIdx.x * per;
  const int c_hi = c_lo + per < nc ? c_lo + per : nc;

  // q rows of this lane's columns (clamped: rows past the last are not stored)
  u32x4 qf[RT][DK];
  int lim[RT];  // last visible key (none past the cache's end)
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    int rr = row0 + rt * 16 + li;
    if (rr >= rows) rr = rows - 1;
    const int t = rr / G, h = kh * G + (rr - t * G);
    lim[rt] = p0 + t < a.S ? p0 + t : a.S - 1;
    const uint16_t* qp = a.qn + (((int64_t)b * a.T + t) * a.Hq + h) * D + 8 * grp;
#pragma unroll
    for (int i = 0; i < DK; ++i) qf[rt][i] = ld16(qp + 32 * i);
  }

  const uint16_t* kb = a.ck + b * a.ckb + kh * a.ckh;
  const uint16_t* vb = a.cv + b * a.cvb + kh * a.cvh;
  const int kbytes = end > 0 ? (int)(((int64_t)(end - 1) * a.cks + D) * 2) : 0;
  const int vbytes = end > 0 ? (int)(((int64_t)(end - 1) * a.cvs + D) * 2) : 0;
  const uint32_t kstep = (uint32_t)(a.cks * 2), vstep = (uint32_t)(a.cvs * 2);
  const uint32_t koff = (uint32_t)li * kstep + 16 * grp;
  const int vr = lane / CH;
  auto issue = [&](u32x4 (&kf)[2][DK], char* sv, int c) {
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int r = n * RPI + vr;
      load_lds16(vb, vbytes, (lds_ptr_t)(sv + n * 1024),
                 (uint32_t)(c * KC + r) * vstep + (uint32_t)(((lane % CH) ^ (r & (CH - 1))) * 16));
    }
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < DK; ++i)
        kf[kt][i] = load_buf16(kb, kbytes, koff + (uint32_t)(c * KC + 16 * kt) * kstep + 64 * i);
  };

  const float sc = kLog2e / sqrtf((float)D);
  f32x4 o[DT][RT];
  float mx[RT], sum[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    mx[rt] = -INFINITY;
    sum[rt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  auto compute = [&](u32x4 (&kf)[2][DK], const char* sv, int c) {
    f32x4 s[2][RT];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        s[kt][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < DK; ++i) s[kt][rt] = mfma16(kf[kt][i], qf[rt][i], s[kt][rt]);
      }
    u32x4 pf[RT][3];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float m = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool vis = c * KC + kt * 16 + 4 * grp + r <= lim[rt];
          s[kt][rt][r] = vis ? s[kt][rt][r] * sc : -INFINITY;
          m = fmaxf(m, s[kt][rt][r]);
        }
      const float mn = fmaxf(mx[rt], col_max(m));
      const float base = mn == -INFINITY ? 0.f : mn;
      const float al = exp2_fast(mx[rt] - base);
      mx[rt] = mn;
      float l = 0.f;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[kt][rt][r] = exp2_fast(s[kt][rt][r] - base);
          l += s[kt][rt][r];
        }
      sum[rt] = sum[rt] * al + l;
      split_p(s[0][rt], s[1][rt], pf[rt]);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt][rt] *= al;
    }
    u32x4 vt[DT];
    bool bad = false;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      vt[dt] = read_vt<D>(sv, dt, li, grp);
      bad |= nonfinite8(vt[dt]);
    }
    const bool any = __any(bad);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) o[dt][rt] = mfma16(vt[dt], pf[rt][0], o[dt][rt]);
      if (__builtin_expect(any, 0)) vt[dt] = zero_nonfinite8(vt[dt]);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        o[dt][rt] = mfma16(vt[dt], pf[rt][1], o[dt][rt]);
        o[dt][rt] = mfma16(vt[dt], pf[rt][2], o[dt][rt]);
      }
    }
  };

  // chunk c_lo + wave + 4 i of this wave, the next one's loads in flight
  u32x4 k0[2][DK], k1[2][DK];
  int c = c_lo + wave;
  if (c < c_hi) issue(k0, sV0[wave], c);
  while (c < c_hi) {
    if (c + NW < c_hi) {
      issue(k1, sV1[wave], c + NW);
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(NK + NV));
    } else {
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    }
    compute(k0, sV0[wave], c);
    c += NW;
    if (c >= c_hi) break;
    if (c + NW < c_hi) {
      issue(k0, sV0[wave], c + NW);
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(NK + NV));
    } else {
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    }
    compute(k1, sV1[wave], c);
    c += NW;
  }

  // Merge the waves' states in wave order. Row block rt's sums go over the
  // wave's own V buffer rt (free now: the same 32 D bytes x 2 per 16 rows),
  // 16-byte chunk q of row r at q ^ r, so 16 rows' stores spread over the banks.
  static_assert(RT <= 2 && 16 * D * 4 == KC * D * 2, "row sums fit the V buffers");
  auto slot = [&](int w, int r, int q) -> f32x4* {
    char* base = r < 16 ? sV0[w] : sV1[w];
    return reinterpret_cast<f32x4*>(base + (r & 15) * (D * 4) + ((q ^ (r & 15)) * 16));
  };
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const float l = col_sum(sum[rt]);
    if (grp == 0) {
      sM[wave][rt * 16 + li] = mx[rt];
      sL[wave][rt * 16 + li] = l;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      *slot(wave, rt * 16 + li, dt * 4 + grp) = o[dt][rt];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 16 * RT * (D / 4); i += NW * kWave) {
    const int r = i / (D / 4), d = (i % (D / 4)) * 4, rr = row0 + r;
    if (rr >= rows) continue;
    float m = sM[0][r];
#pragma unroll
    for (int w = 1; w < NW; ++w) m = fmaxf(m, sM[w][r]);
    const float base = m == -INFINITY ? 0.f : m;
    float l = 0.f;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float e = exp2_fast(sM[w][r] - base);
      l += e * sL[w][r];
      v += *slot(w, r, d / 4) * e;
    }
    if (a.nsplit > 1) {
      const int64_t pr = part_row(a, blockIdx.x, bh, rr);
      *reinterpret_cast<f32x4*>(a.part + pr * D + d) = v;
      if (d == 0) *reinterpret_cast<f32x2*>(a.stat + pr * 2) = f32x2{m, l};
    } else {
      const int t = rr / G, h = kh * G + (rr - t * G);
      uint16_t* yp = a.y + (((int64_t)b * a.T + t) * a.Hq + h) * D + d;
      *reinterpret_cast<u32x2*>(yp) = u32x2{pack_bf16x2(v[0] / l, v[1] / l), pack_bf16x2(v[2] / l, v[3] / l)};
    }
  }
}

// ---- prompts --------------------------------------------------------------
//
// A workgroup takes one kv head of one sequence and 64 * RT query rows (token
// t, group head h at row t * G + h; wave w rows 16 RT w ..), and walks its
// keys in tiles of 64 shared by the four waves: K by LDS DMA, V through
// registers (checked for infinities and NaN on the way), both double-buffered,
// one barrier per tile. Within a head, row tiles with the most keys start first.
template <int D, int RT>
__global__ __launch_bounds__(256, 2) void attn_tiles_kernel(AttnArgs a, int n_rt) {
  constexpr int NW = 4, KT = 64;
  constexpr int DK = D / 32, DT = D / 16;
  constexpr int RPI = 1024 / (D * 2);
  constexpr int NL = KT / RPI / NW;            // load instructions per wave, tile and operand
  constexpr int CH = D / 8;
  __shared__ __attribute__((aligned(1024))) char sK0[KT * D * 2];
  __shared__ __attribute__((aligned(1024))) char sK1[KT * D * 2];
  __shared__ __attribute__((aligned(1024))) char sV0[KT * D * 2];
  __shared__ __attribute__((aligned(1024))) char sV1[KT * D * 2];
  __shared__ int sBad[2][NW];

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int li = lane & 15, grp = lane >> 4;
  const int G = a.Hq / a.Hk, rows = a.T * G;
  const int bh = blockIdx.y, b = bh / a.Hk, kh = bh - b * a.Hk;
  const int tile = n_rt - 1 - (int)blockIdx.x;
  const int row0 = tile * 64 * RT + wave * 16 * RT;  // this wave's first row
  const int p0 = first_pos(a);
  // keys this workgroup's last row sees
  int last = (tile + 1) * 64 * RT - 1;
  if (last >= rows) last = rows - 1;
  const int pend = p0 + last / G + 1;
  const int end = pend < 0 ? 0 : pend < a.S ? pend : a.S;
  const int nt = (end + KT - 1) / KT;
  const int per = (nt + a.nsplit - 1) / a.nsplit;
  const int t_lo = (int)blockIdx.z * per;
  const int t_hi = t_lo + per < nt ? t_lo + per : nt;

  u32x4 qf[RT][DK];
  int lim[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    int rr = row0 + rt * 16 + li;
    if (rr >= rows) rr = rows - 1;
    const int t = rr / G, h = kh * G + (rr - t * G);
    lim[rt] = p0 + t < a.S ? p0 + t : a.S - 1;
    const uint16_t* qp = a.qn + (((int64_t)b * a.T + t) * a.Hq + h) * D + 8 * grp;
#pragma unroll
    for (int i = 0; i < DK; ++i) qf[rt][i] = ld16(qp + 32 * i);
  }
  // the wave's first and last visible key over its rows (uniform)
  int lim_lo = p0 + (row0 < rows ? row0 : rows - 1) / G;
  if (lim_lo >= a.S) lim_lo = a.S - 1;
  const int lim_hi = p0 + (row0 + 16 * RT - 1 < rows ? row0 + 16 * RT - 1 : rows - 1) / G;

  const uint16_t* kb = a.ck + b * a.ckb + kh * a.ckh;
  const uint16_t* vb = a.cv + b * a.cvb + kh * a.cvh;
  const int kbytes = end > 0 ? (int)(((int64_t)(end - 1) * a.cks + D) * 2) : 0;
  const int vbytes = end > 0 ? (int)(((int64_t)(end - 1) * a.cvs + D) * 2) : 0;
  const uint32_t kstep = (uint32_t)(a.cks * 2), vstep = (uint32_t)(a.cvs * 2);
  uint32_t koff[NL], voff[NL];
#pragma unroll
  for (int n = 0; n < NL; ++n) {
    const int r = (wave * NL + n) * RPI + lane / CH;
    const uint32_t ch = (uint32_t)(((lane % CH) ^ (r & (CH - 1))) * 16);
    koff[n] = (uint32_t)r * kstep + ch;
    voff[n] = (uint32_t)r * vstep + ch;
  }
  // each tile's rows through a buffer that starts at the tile and ends with the
  // last key, so that the lane offset alone tells whether a row is past it
  auto issue_k = [&](char* sk, int kt) {
    const int off = (int)((uint32_t)(kt * KT) * kstep);
#pragma unroll
    for (int n = 0; n < NL; ++n)
      load_lds16((const char*)kb + off, kbytes - off, (lds_ptr_t)(sk + (wave * NL + n) * 1024),
                 koff[n]);
  };
  u32x4 vr[NL];
  auto load_v = [&](int kt) {
    const int off = (int)((uint32_t)(kt * KT) * vstep);
#pragma unroll
    for (int n = 0; n < NL; ++n) vr[n] = load_buf16((const char*)vb + off, vbytes - off, voff[n]);
  };
  auto store_v = [&](char* sv, int st) {
    bool bad = false;
#pragma unroll
    for (int n = 0; n < NL; ++n) {
      *reinterpret_cast<u32x4*>(sv + (wave * NL + n) * 1024 + lane * 16) = vr[n];
      bad |= nonfinite8(vr[n]);
    }
    const int any = __any(bad) ? 1 : 0;
    if (lane == 0) sBad[st][wave] = any;
  };

  const float sc = kLog2e / sqrtf((float)D);
  f32x4 o[DT][RT];
  float mx[RT], sum[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    mx[rt] = -INFINITY;
    sum[rt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  auto compute = [&](const char* sk, const char* sv, int st, int kt) {
    if (kt * KT > lim_hi) return;  // every key hidden from every row
    f32x4 s[4][RT];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) s[n][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < DK; ++i) {
        const int r = n * 16 + li;
        const u32x4 kf = *reinterpret_cast<const u32x4*>(
            sk + r * (D * 2) + (((4 * i + grp) ^ (r & (CH - 1))) * 16));
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) s[n][rt] = mfma16(kf, qf[rt][i], s[n][rt]);
      }
    }
    const bool mask = kt * KT + KT - 1 > lim_lo;  // uniform
    u32x4 pf[RT][2][3];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float m = -INFINITY;
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[n][rt][r] *= sc;
          if (mask && kt * KT + n * 16 + 4 * grp + r > lim[rt]) s[n][rt][r] = -INFINITY;
          m = fmaxf(m, s[n][rt][r]);
        }
      const float mn = fmaxf(mx[rt], col_max(m));
      const float base = mn == -INFINITY ? 0.f : mn;
      const float al = exp2_fast(mx[rt] - base);
      float l = 0.f;
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[n][rt][r] = exp2_fast(s[n][rt][r] - base);
          l += s[n][rt][r];
        }
      sum[rt] = sum[rt] * al + l;
      if (__any(mn != mx[rt])) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[dt][rt] *= al;
      }
      mx[rt] = mn;
      split_p(s[0][rt], s[1][rt], pf[rt][0]);
      split_p(s[2][rt], s[3][rt], pf[rt][1]);
    }
    const bool any = (sBad[st][0] | sBad[st][1] | sBad[st][2] | sBad[st][3]) != 0;
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        u32x4 vt = read_vt<D>(sv + n * 32 * D * 2, dt, li, grp);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) o[dt][rt] = mfma16(vt, pf[rt][n][0], o[dt][rt]);
        if (__builtin_expect(any, 0)) vt = zero_nonfinite8(vt);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          o[dt][rt] = mfma16(vt, pf[rt][n][1], o[dt][rt]);
          o[dt][rt] = mfma16(vt, pf[rt][n][2], o[dt][rt]);
        }
      }
  };

  if (t_lo < t_hi) {
    issue_k(sK0, t_lo);
    load_v(t_lo);
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    store_v(sV0, 0);
    __syncthreads();
    for (int kt = t_lo; kt < t_hi; kt += 2) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int k = kt + u;
        if (k >= t_hi) break;
        const bool more = k + 1 < t_hi;
        if (more) {
          issue_k(u ? sK0 : sK1, k + 1);
          load_v(k + 1);
        }
        compute(u ? sK1 : sK0, u ? sV1 : sV0, u, k);
        if (more) {
          __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
          store_v(u ? sV0 : sV1, u ^ 1);
          __syncthreads();
        }
      }
    }
  }

#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const float l = col_sum(sum[rt]);
    const int rr = row0 + rt * 16 + li;
    if (rr >= rows) continue;
    if (a.nsplit > 1) {
      const int64_t pr = part_row(a, blockIdx.z, bh, rr);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        *reinterpret_cast<f32x4*>(a.part + pr * D + dt * 16 + 4 * grp) = o[dt][rt];
      if (grp == 0) *reinterpret_cast<f32x2*>(a.stat + pr * 2) = f32x2{mx[rt], l};
    } else {
      const int t = rr / G, h = kh * G + (rr - t * G);
      uint16_t* yp = a.y + (((int64_t)b * a.T + t) * a.Hq + h) * D + 4 * grp;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        *reinterpret_cast<u32x2*>(yp + dt * 16) =
            u32x2{pack_bf16x2(o[dt][rt][0] / l, o[dt][rt][1] / l),
                  pack_bf16x2(o[dt][rt][2] / l, o[dt][rt][3] / l)};
    }
  }
}

// One output row per workgroup: lane s of each wave holds split s's statistics
// (at most 64 splits), so the weights take one load and a few lane exchanges;
// then each group of D / 4 threads sums every NG-th split's partials and the
// groups' sums are added in group order (one serial chain over the splits ran
// 7-8 us for 16 splits of 32 rows, this 3).
template <int D>
__global__ __launch_bounds__(256) void attn_combine_kernel(AttnArgs a) {
  constexpr int LPR = D / 4, NG = 256 / LPR;
  __shared__ __attribute__((aligned(16))) f32x4 part[NG][LPR];
  const int rows = a.T * (a.Hq / a.Hk);
  const int64_t total = (int64_t)a.B * a.Hk * rows, i = blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1), grp = threadIdx.x / LPR, q = threadIdx.x % LPR;
  const bool has = lane < a.nsplit;
  f32x2 st = {-INFINITY, 0.f};
  if (has) st = *reinterpret_cast<const f32x2*>(a.stat + (lane * total + i) * 2);
  float m = st.x;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) m = fmaxf(m, __shfl_xor(m, off));
  const float base = m == -INFINITY ? 0.f : m;
  const float e = has ? exp2_fast(st.x - base) : 0.f;
  const float l = wave_sum(has ? e * st.y : 0.f);
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int n = 0; n < kAttnMaxSplit / NG; ++n) {
    const int s = n * NG + grp;
    const float w = __shfl(e, s);  // every lane takes part in the exchange
    if (s < a.nsplit)
      v += *reinterpret_cast<const f32x4*>(a.part + (s * total + i) * D + q * 4) * w;
  }
  part[grp][q] = v;
  __syncthreads();
  if (grp != 0) return;
#pragma unroll
  for (int g = 1; g < NG; ++g) v += part[g][q];
  const int bh = (int)(i / rows), b = bh / a.Hk, kh = bh - b * a.Hk;
  const int rr = (int)(i - (int64_t)bh * rows), G = a.Hq / a.Hk;
  const int t = rr / G, h = kh * G + (rr - t * G);
  uint16_t* yp = a.y + (((int64_t)b * a.T + t) * a.Hq + h) * D + q * 4;
  *reinterpret_cast<u32x2*>(yp) = u32x2{pack_bf16x2(v[0] / l, v[1] / l), pack_bf16x2(v[2] / l, v[3] / l)};
}

// The attention kernel's shape for a call.
struct AttnPlan {
  bool rows;   // attn_rows_kernel (else attn_tiles_kernel)
  int rt;      // 16-row blocks per wave
  int n_rt;    // row groups (rows) or row tiles
  int nsplit;  // key ranges
};

constexpr int kAttnRowsMax = 64;    // query rows per kv head of attn_rows_kernel
constexpr int kAttnGroups = 512;    // workgroups a call aims at (two per CU)

// S: the keys a call may see (an int position: start + T; a device position:
// the whole cache). Splits: as many key ranges as give about two workgroups
// per CU, none shorter than 128 keys (attn_rows_kernel: one chunk per wave)
// or 256 (attn_tiles_kernel: four tiles).
AttnPlan attn_plan(int64_t B, int64_t T, int64_t Hq, int64_t Hk, int64_t S) {
  AttnPlan p;
  const int64_t rows = T * (Hq / Hk);
  p.rows = rows <= kAttnRowsMax;
  if (p.rows) {
    p.rt = rows <= 16 ? 1 : 2;
    p.n_rt = (int)((rows + 16 * p.rt - 1) / (16 * p.rt));
  } else {
    p.rt = B * Hk * ((rows + 127) / 128) >= kAttnGroups ? 2 : 1;
    p.n_rt = (int)((rows + 64 * p.rt - 1) / (64 * p.rt));
  }
  const int64_t groups = B * Hk * p.n_rt, unit = p.rows ? 128 : 256;
  int64_t ns = kAttnGroups / groups, most = (S + unit - 1) / unit;
  ns = ns < most ? ns : most;
  ns = ns < kAttnMaxSplit ? ns : kAttnMaxSplit;
  p.nsplit = (int)(ns < 1 ? 1 : ns);
  return p;
}

inline int64_t up256(int64_t v) { return (v + 255) / 256 * 256; }

template <int D>
int launch_attn_d(AttnArgs a, int64_t S, hipStream_t s) {
  const int64_t heads = (int64_t)a.B * a.T * (a.Hq + 2 * a.Hk), hpb = 256 / (D / 8);
  hipLaunchKernelGGL(attn_prep_kernel<D>, dim3((unsigned)((heads + hpb - 1) / hpb)), dim3(256), 0, s, a);
  int e = (int)hipGetLastError();
  if (e) return e;
  const AttnPlan p = attn_plan(a.B, a.T, a.Hq, a.Hk, S);
  a.nsplit = p.nsplit;
  const unsigned bh = (unsigned)(a.B * a.Hk);
  if (p.rows) {
    const dim3 grid((unsigned)p.nsplit, bh, (unsigned)p.n_rt);
    if (p.rt == 1) hipLaunchKernelGGL((attn_rows_kernel<D, 1>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((attn_rows_kernel<D, 2>), grid, dim3(256), 0, s, a);
  } else {
    const dim3 grid((unsigned)p.n_rt, bh, (unsigned)p.nsplit);
    if (p.rt == 1) hipLaunchKernelGGL((attn_tiles_kernel<D, 1>), grid, dim3(256), 0, s, a, p.n_rt);
    else hipLaunchKernelGGL((attn_tiles_kernel<D, 2>), grid, dim3(256), 0, s, a, p.n_rt);
  }
  e = (int)hipGetLastError();
  if (e || p.nsplit == 1) return e;
  hipLaunchKernelGGL(attn_combine_kernel<D>, dim3((unsigned)((int64_t)a.B * a.T * a.Hq)), dim3(256), 0, s, a);
  return (int)hipGetLastError();
}

}  // namespace

int64_t attn_workspace_bytes(int64_t B, int64_t T, int64_t Hq, int64_t Hk, int64_t D, int64_t S) {
  const AttnPlan p = attn_plan(B, T, Hq, Hk, S);
  const int64_t rows = B * T * Hq;
  int64_t b = up256(rows * D * 2);
  if (p.nsplit > 1) b += up256(rows * p.nsplit * 8) + rows * p.nsplit * D * 4;
  return b;
}

int launch_attention(AttnArgs a, int64_t D, int64_t S, void* ws, hipStream_t s) {
  const AttnPlan p = attn_plan(a.B, a.T, a.Hq, a.Hk, S);
  const int64_t rows = (int64_t)a.B * a.T * a.Hq;
  char* w = (char*)ws;
  a.qn = (uint16_t*)w;
  w += up256(rows * D * 2);
  a.stat = (float*)w;
  if (p.nsplit > 1) w += up256(rows * p.nsplit * 8);
  a.part = (float*)w;
  return D == 128 ? launch_attn_d<128>(a, S, s) : launch_attn_d<64>(a, S, s);
}

}  // namespace fp
