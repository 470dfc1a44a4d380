// fp_stream.hip — weight-streaming fused projections for the decode /
// spec-verify regime (M <= 64), where every weight byte is used once per call
// and the HBM stream of W is the whole cost.
//
// Memory pattern first: every weight load instruction reads whole 128-byte
// lines — 8 weight rows x 128 B per wave instruction (half-line requests cost
// ~25% of the achieved bandwidth on MI355X). The MFMA mapping is built
// around that:
//   - A workgroup owns a tile of 8 weight rows (for gate-up: the same 8 rows
//     of Wg and of Wu). In a load, lane l reads 16 B of row (l & 7) at chunk
//     c = 4*((l >> 3) & 1) + (l >> 4) of a 128 B line, i.e. rows 0..7 land in
//     MFMA rows i = l & 15 as two halves: MFMA row i holds weight row (i & 7),
//     line half (i >> 3).
//   - v_mfma_f32_16x16x32_bf16 then runs twice per load with two B operands
//     (x for the first and for the second half of the line); MFMA rows 0..7
//     of the first product and rows 8..15 of the second are the wanted partial
//     sums, the other halves are discarded. The MFMA pipe is ~90% idle in this
//     regime, so the doubled MFMA count is free; x^T (M <= 16*MT columns,
//     zero-padded) is the B operand.
//   - K is split across the NW waves of the workgroup, interleaved by k-block.
//     Each wave double-buffers U k-blocks of loads in registers.
//   - x is read from L2 per k-block.
//   - The NW partial tiles are summed through LDS in fixed wave order; the
//     epilogue (bf16 store, or silu(g)*u) runs in registers, so the fp32
//     intermediate never reaches HBM and results are bit-reproducible.
#include "fp_common.h"
#include "fp_launch.h"

namespace fp {

namespace {

// x vectors per lane per k-block: one per (line half, 8-element sub-chunk);
// packed (XP): one per sub-chunk, lanes 0..7 carrying half 0 and lanes 8..15
// half 1 (needs M <= 8).
template <bool W8, bool XP>
constexpr int x_vectors() { return (W8 ? 2 : 1) * (XP ? 1 : 2); }

template <int MT, bool GATEUP, bool W8, bool XP>
struct Frag {
  static constexpr int XV = x_vectors<W8, XP>();
  u32x4 a0;                               // 16 B of a weight line (8 bf16 or 16 int8)
  u32x4 a1;                               // same for the up weights (gate-up only)
  u32x4 xb[MT][XV];                       // B operands: 8 bf16 of x per vector
};

// Rotate a 4-dword value by 8 lanes within each row of 16 (DPP row_ror:8):
// lane i receives lane (i + 8) mod 16 of its row.
__device__ __forceinline__ u32x4 ror8(u32x4 v) {
  constexpr int kRowRor8 = 0x128;
  return u32x4{(uint32_t)__builtin_amdgcn_mov_dpp((int)v.x, kRowRor8, 0xf, 0xf, false),
               (uint32_t)__builtin_amdgcn_mov_dpp((int)v.y, kRowRor8, 0xf, 0xf, false),
               (uint32_t)__builtin_amdgcn_mov_dpp((int)v.z, kRowRor8, 0xf, 0xf, false),
               (uint32_t)__builtin_amdgcn_mov_dpp((int)v.w, kRowRor8, 0xf, 0xf, false)};
}

// XP: packed x operand for M <= 8 (one x load per sub-chunk; the B operand of
// line half 1 is the half-0 register rotated by 8 lanes).
template <int NW, int MT, int U, bool GATEUP, bool W8, bool ALIGNED, bool XP = false>
__global__ __launch_bounds__(NW * kWave) void stream_kernel(StreamArgs a) {
  static_assert(!XP || MT == 1, "packed x needs M <= 8");
  using F = Frag<MT, GATEUP, W8, XP>;
  constexpr int XV = F::XV;
  constexpr int SV = W8 ? 2 : 1;           // 8-element sub-chunks per lane per line half
  constexpr int KB = W8 ? 128 : 64;        // k elements per k-block (one 128 B line)
  constexpr int CK = KB / 8;               // k elements per 16-byte chunk of the line
  constexpr int NM = GATEUP ? 2 : 1;       // weight matrices
  constexpr int NACC = 2 * MT * NM;        // [half][matrix][mt]

  const int lane = threadIdx.x & (kWave - 1);
  // (unaligned rows: as a scalar, for the uniform branches of load_block)
  const int wave = ALIGNED ? (int)(threadIdx.x / kWave)
                           : __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int li = lane & 15;                // MFMA row (A) / column (B)
  const int grp = lane >> 4;               // MFMA k-group
  const int64_t n0 = (int64_t)blockIdx.x * 8;
  const int64_t row = n0 + (lane & 7);     // weight row this lane loads
  const int chunk = 4 * ((lane >> 3) & 1) + grp;
  const bool row_ok = row < a.N;
  const int64_t K = a.K;
  // k-blocks of the main loop; for unaligned rows the whole ones only, and the
  // one that crosses the row's end comes after the loop (with its element reads
  // inside the loop the compiler kept the buffers in scratch memory)
  const int64_t nkb = ALIGNED ? (K + KB - 1) / KB : K / KB;

  const int64_t rsafe = row_ok ? row : 0;
  const char* w0row = (const char*)a.w0 + rsafe * a.ldw0 * (W8 ? 1 : 2);
  const char* w1row = GATEUP ? (const char*)a.w1 + rsafe * a.ldw1 * (W8 ? 1 : 2) : nullptr;
  float s0 = 0.f, s1 = 0.f;
  if constexpr (W8) {
    s0 = row_ok ? a.s0[row] : 0.f;
    if constexpr (GATEUP) s1 = row_ok ? a.s1[row] : 0.f;
  }
  const float n128s0 = -128.f * s0;
  const float n128s1 = -128.f * s1;

  // x rows this lane feeds into the B operands (column li of each m-subtile;
  // packed: column li & 7, line half li >> 3).
  const uint16_t* xrow[MT];
  bool xok[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = XP ? (li & 7) : mt * 16 + li;
    xok[mt] = m < a.M;
    xrow[mt] = a.x + (int64_t)(xok[mt] ? m : 0) * a.ldx;
  }
  const int xhalf = XP ? (li >> 3) : 0;

  // k-blocks of this wave: wave, wave + NW, ...
  const int64_t nmine = nkb > wave ? (nkb - wave + NW - 1) / NW : 0;

  // First k of the 8 x values group grp supplies to the MFMA of line half h,
  // sub-chunk s (int8 lines carry two 8-element sub-chunks per lane).
  auto xk = [&](int64_t kb, int h, int s) -> int64_t {
    return kb * KB + h * (KB / 2) + grp * CK + s * 8;
  };

  auto load_block = [&](F& f, int64_t j) {
    const bool live = j < nmine;
    const int64_t kb = wave + j * NW;
    const int64_t kw = kb * KB + chunk * CK;
    const u32x4 z{0, 0, 0, 0};
    if constexpr (!ALIGNED) {
      // plain loads of any alignment, without a branch per load (rows and
      // columns past the last are row 0 again, never stored)
      if (!live) return;
      f.a0 = ld16_any(w0row + kw * (W8 ? 1 : 2));
      if constexpr (GATEUP) f.a1 = ld16_any(w1row + kw * (W8 ? 1 : 2));
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int v = 0; v < XV; ++v)
          f.xb[mt][v] = ld16_any(xrow[mt] + xk(kb, XP ? xhalf : v / SV, XP ? v : v % SV));
      return;
    }
    if constexpr (W8) {
      f.a0 = (live && row_ok) ? load_w_i8x16<ALIGNED>((const int8_t*)w0row, kw, K) : z;
      if constexpr (GATEUP)
        f.a1 = (live && row_ok) ? load_w_i8x16<ALIGNED>((const int8_t*)w1row, kw, K) : z;
    } else {
      f.a0 = (live && row_ok) ? load_w_bf16x8<ALIGNED>((const uint16_t*)w0row, kw, K) : z;
      if constexpr (GATEUP)
        f.a1 = (live && row_ok) ? load_w_bf16x8<ALIGNED>((const uint16_t*)w1row, kw, K) : z;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < XV; ++v) {
        // packed: v = sub-chunk, half from the lane; else v = h * SV + s
        const int h = XP ? xhalf : v / SV;
        const int s = XP ? v : v % SV;
        f.xb[mt][v] = (live && xok[mt]) ? load_bf16x8<ALIGNED>(xrow[mt], xk(kb, h, s), K) : z;
      }
  };

  // B operand for line half h, sub-chunk s of m-subtile mt.
  auto xfrag = [&](const F& f, int mt, int h, int s) -> u32x4 {
    if constexpr (XP) return h == 0 ? f.xb[mt][s] : ror8(f.xb[mt][s]);
    return f.xb[mt][h * SV + s];
  };

  f32x4 acc[NACC];
#pragma unroll
  for (int i = 0; i < NACC; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // accumulator of (line half h, matrix mat, m-subtile mt)
  auto A = [&](int h, int mat, int mt) -> f32x4& { return acc[(h * NM + mat) * MT + mt]; };

  auto compute_block = [&](const F& f) {
#pragma unroll
    for (int mat = 0; mat < NM; ++mat) {
      const u32x4 w = mat == 0 ? f.a0 : f.a1;
      if constexpr (W8) {
        const float s = mat == 0 ? s0 : s1;
        const float n128s = mat == 0 ? n128s0 : n128s1;
        const u32x4 wlo = dequant8(w.x, w.y, s, n128s);
        const u32x4 whi = dequant8(w.z, w.w, s, n128s);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            A(h, mat, mt) = mfma16(wlo, xfrag(f, mt, h, 0), A(h, mat, mt));
            A(h, mat, mt) = mfma16(whi, xfrag(f, mt, h, 1), A(h, mat, mt));
          }
      } else {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int h = 0; h < 2; ++h) A(h, mat, mt) = mfma16(w, xfrag(f, mt, h, 0), A(h, mat, mt));
      }
    }
  };

  const int64_t nchunks = (nmine + U - 1) / U;
  F fa[U], fb[U];
  auto load_chunk = [&](F* f, int64_t c) {
#pragma unroll
    for (int j = 0; j < U; ++j) load_block(f[j], c * U + j);
  };
  auto compute_chunk = [&](const F* f, int64_t c) {
#pragma unroll
    for (int j = 0; j < U; ++j)
      if (c * U + j < nmine) compute_block(f[j]);
  };

  // Prologue: two chunks of weight loads in flight before anything waits. (A
  // lambda: written out here the compiler orders the address arithmetic otherwise,
  // and calls of 3-4 us take 8-11% longer.)
  auto prologue = [&]() {
    if (nchunks > 0) load_chunk(fa, 0);
    if (nchunks > 1) load_chunk(fb, 1);
  };
  prologue();
  // Steady state: while one chunk is consumed the other is in flight; a
  // consumed buffer is refilled with the chunk two ahead.
  for (int64_t c = 0; c < nchunks; c += 2) {
    compute_chunk(fa, c);
    if (c + 2 < nchunks) load_chunk(fa, c + 2);
    if (c + 1 >= nchunks) break;
    compute_chunk(fb, c + 1);
    if (c + 3 < nchunks) load_chunk(fb, c + 3);
  }

  // The k-block that crosses the row's end: the last one of its wave.
  if constexpr (!ALIGNED) {
    if (nkb * KB < K && wave == (int)(nkb % NW)) {
      F f;
      const int64_t kw = nkb * KB + chunk * CK;
      if constexpr (W8) {
        f.a0 = load_i8x16<false>((const int8_t*)w0row, kw, K);
        if constexpr (GATEUP) f.a1 = load_i8x16<false>((const int8_t*)w1row, kw, K);
      } else {
        f.a0 = load_bf16x8<false>((const uint16_t*)w0row, kw, K);
        if constexpr (GATEUP) f.a1 = load_bf16x8<false>((const uint16_t*)w1row, kw, K);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int v = 0; v < XV; ++v)
          f.xb[mt][v] = load_bf16x8<false>(xrow[mt], xk(nkb, XP ? xhalf : v / SV, XP ? v : v % SV), K);
      compute_block(f);
    }
  }

  // Fixed-order cross-wave reduction through LDS.
  __shared__ f32x4 red[NW > 1 ? NW - 1 : 1][NACC][kWave];
  if constexpr (NW > 1) {
    if (wave > 0) {
#pragma unroll
      for (int i = 0; i < NACC; ++i) red[wave - 1][i][lane] = acc[i];
    }
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int w = 0; w < NW - 1; ++w)
#pragma unroll
      for (int i = 0; i < NACC; ++i) acc[i] += red[w][i][lane];
  }

  // D lane layout: MFMA rows 4*grp + r (r = 0..3), column li. Lanes 0..31
  // hold rows 0..7 (line half 0 of weight rows 0..7) of the first product;
  // lanes 32..63 hold rows 8..15 (half 1 of the same weight rows) of the
  // second. Output row n0 + 4*grp + r (grp < 2) = half 0 (lane) + half 1
  // (lane + 32).
  float sum[NM][MT][4];
#pragma unroll
  for (int mat = 0; mat < NM; ++mat)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float hi = __shfl_down(A(1, mat, mt)[r], 32);
        sum[mat][mt][r] = A(0, mat, mt)[r] + hi;
      }
  if (lane >= 32) return;

  const int64_t nb = n0 + 4 * grp;
  const bool vec_ok = (nb + 3 < a.N) && ((a.ldy & 3) == 0) &&
                      ((reinterpret_cast<uintptr_t>(a.y) & 7) == 0);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = mt * 16 + li;
    if (m >= a.M) continue;
    uint32_t hb[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (GATEUP)
        hb[r] = gate_up_silu_bits(sum[0][mt][r], sum[1][mt][r]);
      else
        hb[r] = f32_to_bf16_bits(sum[0][mt][r]);
    }
    uint16_t* yrow = a.y + (int64_t)m * a.ldy;
    if (vec_ok) {
      *reinterpret_cast<u32x2*>(yrow + nb) = u32x2{hb[0] | (hb[1] << 16), hb[2] | (hb[3] << 16)};
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (nb + r < a.N) yrow[nb + r] = (uint16_t)hb[r];
    }
  }
}

template <int NW, int MT, int U, bool GATEUP, bool W8, bool XP = false>
int launch_stream_cfg(const StreamArgs& a, bool aligned, hipStream_t s) {
  const dim3 grid((unsigned)((a.N + 7) / 8));
  const dim3 block(NW * kWave);
  if (aligned)
    hipLaunchKernelGGL((stream_kernel<NW, MT, U, GATEUP, W8, true, XP>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((stream_kernel<NW, MT, U, GATEUP, W8, false, XP>), grid, block, 0, s, a);
  return (int)hipGetLastError();
}

template <int NW, int MT, int U, bool GATEUP, bool W8>
int launch_stream_aligned(const StreamArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((stream_kernel<NW, MT, U, GATEUP, W8, true>), dim3((unsigned)((a.N + 7) / 8)),
                     dim3(NW * kWave), 0, s, a);
  return (int)hipGetLastError();
}

}  // namespace

// Configurations measured on MI355X (Qwen3-4B shapes, 36 cycled weight sets):
// 4 waves per 8-row tile with interleaved k-blocks; packed x for M <= 8; the
// gate-up kernel (two weight streams) keeps 4 k-blocks per buffer in flight,
// QKV 2 (QKV's 3x smaller grid is latency-bound and prefers occupancy).
template <bool GATEUP, bool W8>
int launch_stream(const StreamArgs& a, bool aligned, hipStream_t s) {
  // int8 at 2-16 rows with K <= 2560: x staged once per workgroup, all weight
  // loads in flight (fp_xpanel.hip)
  if (W8 && xpanel8_shape(a.M, a.N, a.K, GATEUP) && splitk_supported(a, aligned, true))
    return launch_xpanel8<GATEUP>(a, s);
  // int8 from a few rows: split-K tiles dequantising in registers (fp_splitk.hip)
  if (W8 && splitk8_shape(a.M, a.N, a.K, GATEUP) && splitk_supported(a, aligned, true))
    return launch_splitk<GATEUP, true>(a, s);
  // one or a few rows: contiguous row streaming (fp_rows.hip)
  if (rows_supported<W8>(a, aligned)) return launch_rows<GATEUP, W8>(a, s);
  // bf16 against large weights with a caller workspace: k split across
  // workgroups (fp_gemm.hip)
  GemmSplit sp;
  if (!W8 && use_gemm_split(a, aligned, GATEUP, &sp)) return launch_gemm_split<GATEUP, false>(a, sp, s);
  // bf16 with a nearly full round of small staged tiles (from 48 rows
  // against large weights): fp_gemm.hip
  if (!W8 && small_round_tile(a.M, a.N, a.K, GATEUP) >= 0 && gemm_supported(a, aligned, false))
    return launch_gemm<GATEUP, false>(a, s);
  // bf16 outputs of more than 8192 columns from 33 rows: whole rounds of the
  // prefill tiles (one box, us, 64 rows, against the 32-row split-K tiles:
  // 151936 x 2560 247.8 -> 180.6, 32000 x 2560 55.0 -> 39.6; 190 drawn shapes of 33-64
  // rows, 8193-40000 outputs, K = 512-4096: 0.79 of the time at the median, 1.04 at most)
  if (!W8 && !GATEUP && a.N > kSplitkSmallN && a.M > 32 && gemm_supported(a, aligned, false))
    return launch_gemm<GATEUP, false>(a, s);
  // bf16 from 3 rows, wide gate-up from 4 or 6: split-K tiles (fp_splitk.hip)
  const int64_t wrows = GATEUP ? 2 * a.N : a.N;
  // (wide gate-up from fewer rows: 4 with K > 3072, 6 below. One box, µs,
  // stream -> split-K tiles: Qwen3-8B M = 4 34.0 -> 33.2, M = 6 35.1 -> 32.8,
  // M = 7 36.3-37.4 -> 33.0, M = 3 33.0 -> 34.0; Qwen3-4B M = 7 21.0 -> 20.2,
  // M = 6 even, M = 4 19.3 -> 20.1; other wide outputs, 151936 x 2560 at 3
  // rows 135.8 -> 118.4, 32000 x 4096 at 4 rows 52.9 -> 44.3)
  const int64_t min_m = GATEUP && wrows > kSplitkSmallN ? (a.K > 3072 ? 4 : 6) : kSplitkMinM;
  if (!W8 && a.M >= min_m && splitk_supported(a, aligned, false))
    return launch_splitk<GATEUP, false>(a, s);
  // More x rows than a wave's registers stream well (rows or K that the kernels
  // above do not take): the general tiles from 33 rows, and from 9 for unaligned
  // gate-up over at least 8192 weight rows, whose 32-row tiles fill the chip. One
  // box, us, stream / 32 x 32 tiles: gate-up N = 9700, K = 2541 at 16 (int8), 20,
  // 40 rows 55 / 44, 78 / 38, 121 / 51, N = 4800 at 4, 16 rows 32 / 38, 47 / 39; 6100
  // columns, K = 3001 at 16 rows 36 / 37, 2541 columns at 20, 64 rows 30 / 37, 69 / 37.
  // Aligned rows of a long K with up to two workgroups of 8 rows per CU stream on to
  // 64 rows (700 drawn shapes; stream / tiles: int8 171 x 3856 at 33 rows 14.6 / 37.4,
  // 1030 x 2768 at 40 12.5 / 28.0, gate-up 1827 x 3808 at 45 20.4 / 46.5, bf16 173 x 3856
  // at 35 14.5 / 27.1; a shorter K, bf16 gate-up 2282 x 976 at 63 rows 17.3 / 10.1).
  const int64_t stream_k = GATEUP ? (a.N > 2048 ? 1300 : W8 ? 600 : 800)
                                  : (a.N > 2048 ? 800 : W8 ? 320 : 600);
  const bool stream_on = aligned && a.N <= 4096 && a.K >= stream_k;
  if ((a.M > 32 && !stream_on) ||
      (!aligned && GATEUP && a.M > 8 && wrows >= kSplitkSmallN))
    return launch_tiled<GATEUP, W8>(a, aligned, s);
  // (int8 dequantisation needs registers of its own: 2 k-blocks per buffer)
  constexpr int U8 = (GATEUP && !W8) ? 4 : 2;
  if (a.M <= 8) return launch_stream_cfg<4, 1, U8, GATEUP, W8, true>(a, aligned, s);
  if (a.M <= 16) return launch_stream_cfg<4, 1, 2, GATEUP, W8>(a, aligned, s);
  if (a.M <= 32) return launch_stream_cfg<4, 2, 2, GATEUP, W8>(a, aligned, s);
  if (a.M <= 48) return launch_stream_aligned<4, 3, 2, GATEUP, W8>(a, s);
  return launch_stream_aligned<4, 4, 1, GATEUP, W8>(a, s);
}

template int launch_stream<false, false>(const StreamArgs&, bool, hipStream_t);
template int launch_stream<true, false>(const StreamArgs&, bool, hipStream_t);
template int launch_stream<false, true>(const StreamArgs&, bool, hipStream_t);
template int launch_stream<true, true>(const StreamArgs&, bool, hipStream_t);

}  // namespace fp
