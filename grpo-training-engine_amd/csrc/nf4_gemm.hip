// NF4 (+ bias, + LoRA) linear for batches of more than 64 rows on gfx950: one
// MFMA GEMM launch that decodes the 4-bit weight in registers and applies the
// reference epilogue in the kernel.  Restates _lora_forward_kernel
// (src/triton_kernels/lora_forward.py:107-260) for any M:
//   acc = sum_k x[m,k] * bf16(code[q(n,k)] * absmax)   (float32 accumulation)
//   v = bf16(acc); v = bf16(v + bias[n])                (:243-247)
//   t = bf16(x A^T)  (rank r <= 32)                     (:210-236)
//   u = bf16(bf16(t . B[n, :]) * bf16(scaling)); y = bf16(v + u)   (:249-257)
//
//  * Tile: a workgroup (4 waves) owns 128 rows m x 128 columns n; wave w owns
//    all 128 rows x columns 32 w .. 32 w + 31 as 8 x 2 tiles of
//    v_mfma_f32_16x16x32_bf16 (A = x rows from LDS, B = W rows decoded in the
//    wave's registers).  Two workgroups per CU (80 KiB of LDS each).
//  * Stage = 128 K values.  Lane (n = lane % 16, group g = lane / 16) of a
//    column tile holds the 32 nibbles [32 g, 32 g + 32) of its weight row (one
//    16-byte load) and their absmax (blocksize >= 32); per stage it builds the
//    block's bf16 codebook bf16(code[j] * absmax) in registers and decodes
//    8 K values per MFMA with v_perm byte lookups (nf4_decode.hpp), in the
//    order [0,2,4,6,1,3,5,7]; x is staged in LDS permuted the same way.
//  * x is double-buffered in LDS: stage s + 1's x and weights are loaded while
//    stage s's MFMAs run; one barrier per stage.
//  * LoRA: wave w also multiplies rows 32 w .. 32 w + 31 by A (one or two
//    16-rank column tiles; A is bf16, no decode).  After the K loop t goes to
//    LDS in bf16 and t . B[n, :] is one more MFMA per output tile (K = 32
//    ranks, ranks >= r zero).
//  * Output: the bf16 tile passes through LDS so every thread stores 16-byte
//    row chunks.
//  * Edges: rows >= M read row M - 1 and are not stored; columns >= N read
//    row N - 1 of W and are not stored; a last stage past K (K % 128 != 0)
//    stages zero x (its weight loads are clamped into the row).
//  * Workgroup -> tile: the dispatcher places workgroup i on XCD i mod 8; the
//    tiles, column tile by column tile, are cut into 8 equal runs and run x
//    goes to the ids = x mod 8, so the row tiles of a column tile read its
//    weights through one L2 and every XCD gets the same number of tiles.
//
// bf16 with K % 128 == 0, r <= 16 and blocksize >= 64 runs nf4_gemm_k2 (below) instead:
// with the tile and slices that its time model picks it was slower at 2 of 560 measured
// shapes of 65 .. 4096 rows (224 x 4608 x 3584 6 %, 1024 x 1536 x 8960 3 %), at the median
// 0.77 of the time, its SiLU form 0.68 .. 0.93.
#include <algorithm>
#include <type_traits>

#include "lds_dma.hpp"
#include "linear_parts.hpp"
#include "nf4_decode.hpp"

using namespace grpo;

namespace {

constexpr int GM_BM = 128;            // rows per workgroup
constexpr int GM_BN = 128;            // columns per workgroup
constexpr int GM_KS = 128;            // K values per stage
constexpr int GM_T = 256;             // threads (4 waves)
constexpr int GM_XS = GM_KS + 8;      // LDS row stride of a staged x stage (elements)
constexpr int GM_TS = 32 + 8;         // LDS row stride of t (elements)
constexpr int GM_OS = GM_BN + 8;      // LDS row stride of the output tile (elements)
constexpr int GM_RT = GM_BM / 16;     // row tiles per wave
constexpr int GM_MAX_R = 32;
constexpr size_t GM_LDS =
    (size_t)(2 * GM_BM * GM_XS + GM_BM * GM_TS) * 2;  // 79,872 bytes
static_assert(GM_BM * GM_OS <= 2 * GM_BM * GM_XS, "output tile reuses the x stages");
constexpr int GM_PS = GM_BN + 4;      // LDS row stride of a float32 partial-sum tile
static_assert(GM_BM * GM_PS * 2 <= 2 * GM_BM * GM_XS, "partial-sum tile reuses the x stages");

struct GemmArgs {
  const uint16_t* x;
  int64_t ldx;
  const uint8_t* w;
  const float* absmax;
  const float* code16;
  int bs_shift;
  int64_t wrow0;         // weight row of output column 0 (of segment 0)
  // Up to 4 segments: consecutive column ranges [seg_end[s-1], seg_end[s]) of
  // one stacked weight and of y, each with its own bias and LoRA pair (the
  // q|k|v projections of one launch); seg_tile[s] = first column tile of
  // segment s (seg_tile[nseg..4] = NT).
  int nseg;
  int seg_end[MAXSEG];
  int seg_tile[MAXSEG + 1];
  const uint16_t* bias[MAXSEG];  // [N_s] or null
  const uint16_t* la[MAXSEG];    // [r][K] (r > 0)
  const uint16_t* lb[MAXSEG];    // [N_s][r] (r > 0)
  int r;
  float scaling;
  uint16_t* y;
  int64_t ldy;
  int M, N, K;
  int MT, NT;  // row and column tiles
  int nst;     // stages
  int kst;     // stages per K slice (gridDim.y slices)
  bool yvec;   // 16-byte stores of y rows (y aligned, ldy and N multiples of 8)
  bool lbvec;  // 16-byte loads of B rows (lb aligned, r % 8 == 0)
  // K split over gridDim.y slices: float32 partial sums part[slice][m][n]
  // (slice stride psl, row stride ldp) and, from column tile 0, the LoRA t
  // partials tpart[slice][m][16] (slice stride tsl); the epilogue then runs in
  // the finish kernel.  part == null: one slice, epilogue in this kernel.
  float* part;
  int64_t ldp, psl;
  float* tpart;  // segment s at tpart + s * tseg
  int64_t tsl, tseg;
  int silu_I;    // SILU kernels: I (y = act [M, I], row stride ldy)
};

// TC: LoRA rank tiles of 16 (0: no LoRA, 1: r <= 16, 2: r <= 32).  F16: x,
// the weight values, LoRA, bias and y in float16 instead of bf16 (the
// reference's float16 X_DTYPE / LORA_DTYPE, lora_forward.py:141-143, 745-749).
// SILU: the MLP's gate|up projection of the stacked [2I, K] weight (no bias,
// no LoRA) with act = bf16(bf16(silu(g)) * u) applied in the epilogue: the
// tile's columns are 64 gate columns j0 .. j0 + 63 (waves 0, 1) and the same
// 64 up columns (waves 2, 3), and y is act [M, I].
template <int TC, bool F16, bool SILU = false>
__global__ void __launch_bounds__(GM_T, 2) nf4_gemm_mfma(GemmArgs p) {
  constexpr bool LORA = TC > 0;
  static_assert(!SILU || (TC == 0 && !F16), "gate|up + SiLU: bf16, no LoRA");
  extern __shared__ __align__(16) uint16_t lds[];
  uint16_t* const ts = lds + 2 * GM_BM * GM_XS;  // t [128][GM_TS] bf16
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 15, lg = lane >> 4;
  // Tiles t = nt * MT + mt in order, in 8 contiguous runs of equal length
  // (+-1): run x goes to the workgroups with ids = x mod 8, which the
  // dispatcher places on one XCD, so the row tiles of a column tile share
  // that tile's weights through one L2 and every XCD gets the same work.
  const int b = blockIdx.x, run = b & 7, T = p.MT * p.NT;
  const int t = ((run * T) >> 3) + (b >> 3);
  if (t >= (((run + 1) * T) >> 3)) return;  // past the end of this run
  const int nt = t / p.MT, mt = t - nt * p.MT;
  // the segment of column tile nt (uniform per workgroup) and its columns
  const int seg = (nt >= p.seg_tile[1]) + (nt >= p.seg_tile[2]) + (nt >= p.seg_tile[3]);
  const int c0 = seg > 0 ? sel4(p.seg_end[0], p.seg_end[1], p.seg_end[2], p.seg_end[3],
                                seg - 1) : 0;
  const int N = sel4(p.seg_end[0], p.seg_end[1], p.seg_end[2], p.seg_end[3], seg) - c0;
  const uint16_t* const sbias = sel4(p.bias[0], p.bias[1], p.bias[2], p.bias[3], seg);
  const uint16_t* const sla = sel4(p.la[0], p.la[1], p.la[2], p.la[3], seg);
  const uint16_t* const slb = sel4(p.lb[0], p.lb[1], p.lb[2], p.lb[3], seg);
  const int lt = nt - sel4(p.seg_tile[0], p.seg_tile[1], p.seg_tile[2], p.seg_tile[3], seg);
  const int m0 = mt * GM_BM, n0 = lt * GM_BN;  // n0: column within the segment

  float code[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) code[j] = p.code16[j];

  // x staging: thread (row r0 + 16 u, chunk c) for u < 8; 16 threads per row
  const int r0 = tid >> 4, c8 = 8 * (tid & 15);
  const uint16_t* xr[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) xr[u] = p.x + (int64_t)min(m0 + r0 + 16 * u, p.M - 1) * p.ldx;
  // weight rows of this lane's two column tiles
  const uint8_t* wr[2];
  int64_t we[2];
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    const int n = min(n0 + 32 * wave + 16 * ct + ln, N - 1);
    if (SILU) {  // gate row j (waves 0, 1) or up row I + j (waves 2, 3)
      const int j = min(lt * (GM_BN / 2) + 32 * (wave & 1) + 16 * ct + ln, p.silu_I - 1);
      we[ct] = ((int64_t)(wave >> 1) * p.silu_I + j) * p.K;
    } else {
      we[ct] = (p.wrow0 + c0 + n) * p.K;
    }
    wr[ct] = p.w + we[ct] / 2;
  }
  // LoRA A rows: rank 16 tc + ln of this lane.  Ranks >= r read rank r - 1:
  // their t columns are finite and meet zero B entries, so they add nothing
  // (no select, which the compiler turns into a predicated load).
  const uint16_t* ar[LORA ? TC : 1];
#pragma unroll
  for (int tc = 0; tc < TC; ++tc) ar[tc] = sla + (int64_t)min(16 * tc + ln, p.r - 1) * p.K;

  uint4 xv[8];
  uint4 wv[2];
  float av[2];
  auto load_stage = [&](int st) __attribute__((always_inline)) {
    const int k0 = st * GM_KS;
    const int kx = min(k0 + c8, p.K - 8);
#pragma unroll
    for (int u = 0; u < 8; ++u) xv[u] = *reinterpret_cast<const uint4*>(xr[u] + kx);
    const int kc = min(k0 + 32 * lg, p.K - 32);
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
      wv[ct] = *reinterpret_cast<const uint4*>(wr[ct] + kc / 2);
      av[ct] = p.absmax[(we[ct] + kc) >> p.bs_shift];
    }
  };
  auto store_x = [&](int st) __attribute__((always_inline)) {
    uint16_t* buf = lds + (st & 1) * GM_BM * GM_XS;
    const bool kin = st * GM_KS + c8 < p.K;
#pragma unroll
    for (int u = 0; u < 8; ++u)
      *reinterpret_cast<uint4*>(buf + (r0 + 16 * u) * GM_XS + c8) =
          kin ? deinterleave8(xv[u]) : make_uint4(0, 0, 0, 0);
  };

  f32x4_t acc[GM_RT][2];
#pragma unroll
  for (int rt = 0; rt < GM_RT; ++rt) acc[rt][0] = acc[rt][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  f32x4_t tacc[2][LORA ? TC : 1];  // [row tile of the wave's 32 rows][rank tile]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int tc = 0; tc < TC; ++tc) tacc[i][tc] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int st0 = blockIdx.y * p.kst, st1 = min(p.nst, st0 + p.kst);
  load_stage(st0);
  store_x(st0);
  __syncthreads();
  for (int st = st0; st < st1; ++st) {
    // This stage's LoRA A loads go out before the next stage's prefetch (loads
    // retire in order) and are used after the stage's weight MFMAs.
    uint4 la4[LORA ? TC : 1][4];
    if (LORA) {
      const int kc = min(st * GM_KS + 32 * lg, p.K - 32);
#pragma unroll
      for (int tc = 0; tc < TC; ++tc)
#pragma unroll
        for (int s = 0; s < 4; ++s)
          la4[tc][s] = *reinterpret_cast<const uint4*>(ar[tc] + kc + 8 * s);
    }
    const uint4 wc0 = wv[0], wc1 = wv[1];
    const float ac0 = av[0], ac1 = av[1];
    // The prefetch is unconditional (the last stage re-reads itself): after a
    // conditional load the compiler waits for every load with vmcnt(0).
    const bool more = st + 1 < st1;
    load_stage(min(st + 1, st1 - 1));
    // keep the loads here, ahead of this stage's MFMAs
    __builtin_amdgcn_sched_barrier(0);
    const uint16_t* buf = lds + (st & 1) * GM_BM * GM_XS + ln * GM_XS + 32 * lg;
    const Lut t0 = make_lut<F16>(code, ac0), t1 = make_lut<F16>(code, ac1);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      uint4 a[GM_RT];
#pragma unroll
      for (int rt = 0; rt < GM_RT; ++rt)
        a[rt] = *reinterpret_cast<const uint4*>(buf + rt * 16 * GM_XS + 8 * s);
      const uint4 b0 = decode8(word(wc0, s), t0);
      const uint4 b1 = decode8(word(wc1, s), t1);
#pragma unroll
      for (int rt = 0; rt < GM_RT; ++rt) {
        acc[rt][0] = mfma16x16x32_e<F16>(a[rt], b0, acc[rt][0]);
        acc[rt][1] = mfma16x16x32_e<F16>(a[rt], b1, acc[rt][1]);
      }
    }
    if (LORA) {
      // rows 32 w .. 32 w + 31 of this wave times the A ranks (ranks >= r zero)
      const uint16_t* tb = buf + 32 * wave * GM_XS;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const uint4 a0 = *reinterpret_cast<const uint4*>(tb + 8 * s);
        const uint4 a1 = *reinterpret_cast<const uint4*>(tb + 16 * GM_XS + 8 * s);
#pragma unroll
        for (int tc = 0; tc < TC; ++tc) {
          const uint4 lb = deinterleave8(la4[tc][s]);
          tacc[0][tc] = mfma16x16x32_e<F16>(a0, lb, tacc[0][tc]);
          tacc[1][tc] = mfma16x16x32_e<F16>(a1, lb, tacc[1][tc]);
        }
      }
    }
    if (more) store_x(st + 1);
    __syncthreads();
  }

  if (p.part) {
    // K slice: float32 partial sums (and column tile 0's LoRA t partials).
    // The tile passes through LDS (the x stages are free after the loop's last
    // barrier) so every thread stores 16-byte row chunks (N % 16 == 0 here).
    float* const ps = reinterpret_cast<float*>(lds);  // [128][GM_PS]
#pragma unroll
    for (int rt = 0; rt < GM_RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          ps[(rt * 16 + 4 * lg + q) * GM_PS + 32 * wave + 16 * ct + ln] = acc[rt][ct][q];
    __syncthreads();
    float* pp = p.part + blockIdx.y * p.psl + c0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int c = tid + GM_T * i, row = c >> 5, c4 = 4 * (c & 31);
      const int m = m0 + row, n = n0 + c4;
      if (m < p.M && n < N)
        *reinterpret_cast<float4*>(pp + (int64_t)m * p.ldp + n) =
            *reinterpret_cast<const float4*>(ps + row * GM_PS + c4);
    }
    if (LORA && lt == 0) {
      float* tp = p.tpart + blockIdx.y * p.tsl + seg * p.tseg;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int m = m0 + 32 * wave + 16 * i + 4 * lg + q;
          if (m < p.M) tp[(int64_t)m * 16 + ln] = tacc[i][0][q];
        }
    }
    return;
  }

  // ---- epilogue
  f32x4_t u[GM_RT][2];
  if (LORA) {
    // t rows 32 w + 16 i + 4 lg + q, ranks 16 tc + ln, rounded to bf16
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int tc = 0; tc < 2; ++tc)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          ts[(32 * wave + 16 * i + 4 * lg + q) * GM_TS + 16 * tc + ln] =
              tc < TC ? f2e<F16>(tacc[i][tc < TC ? tc : 0][q]) : (uint16_t)0;
    // B rows: ranks 8 lg .. 8 lg + 7 of column n (ranks >= r zero)
    uint4 bv[2];
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
      const int n = min(n0 + 32 * wave + 16 * ct + ln, N - 1);
      const uint16_t* br = slb + (int64_t)n * p.r;
      if (p.lbvec) {
        bv[ct] = 8 * lg < p.r ? *reinterpret_cast<const uint4*>(br + 8 * lg)
                              : make_uint4(0, 0, 0, 0);
      } else {
        uint32_t h[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) h[j] = 8 * lg + j < p.r ? br[8 * lg + j] : 0u;
        bv[ct] = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16),
                            h[6] | (h[7] << 16));
      }
    }
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < GM_RT; ++rt) {
      const uint4 tv = *reinterpret_cast<const uint4*>(ts + (rt * 16 + ln) * GM_TS + 8 * lg);
#pragma unroll
      for (int ct = 0; ct < 2; ++ct)
        u[rt][ct] = mfma16x16x32_e<F16>(tv, bv[ct], f32x4_t{0.f, 0.f, 0.f, 0.f});
    }
  }
  float bias[2] = {0.f, 0.f};
  if (sbias) {
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
      bias[ct] = e2f<F16>(sbias[min(n0 + 32 * wave + 16 * ct + ln, N - 1)]);
  }
  const float sc = round_e<F16>(p.scaling);
  // bf16 tile [128][GM_OS] in the x stage buffers (free after the loop's last barrier)
  uint16_t* os = lds;
#pragma unroll
  for (int rt = 0; rt < GM_RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v = round_e<F16>(acc[rt][ct][q]);
        if (sbias) v = round_e<F16>(v + bias[ct]);
        if (LORA) v = round_e<F16>(v + round_e<F16>(round_e<F16>(u[rt][ct][q]) * sc));
        os[(rt * 16 + 4 * lg + q) * GM_OS + 32 * wave + 16 * ct + ln] = f2e<F16>(v);
      }
  __syncthreads();
  if (SILU) {
    // act columns j0 .. j0 + 63: thread (row r0 + 32 i, 8 columns 8 (tid % 8)),
    // the gate values at tile columns 0..63, the up values at 64..127
    const int j0 = lt * (GM_BN / 2), rs = tid >> 3, cc = 8 * (tid & 7);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = rs + 32 * i, m = m0 + row;
      if (m >= p.M || j0 + cc >= p.silu_I) continue;
      const uint4 gv = *reinterpret_cast<const uint4*>(os + row * GM_OS + cc);
      const uint4 uv = *reinterpret_cast<const uint4*>(os + row * GM_OS + 64 + cc);
      const uint32_t gw[4] = {gv.x, gv.y, gv.z, gv.w}, uw[4] = {uv.x, uv.y, uv.z, uv.w};
      uint32_t o[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float r2[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float g = h ? bf_hi(gw[q]) : bf_lo(gw[q]);
          const float u = h ? bf_hi(uw[q]) : bf_lo(uw[q]);
          r2[h] = round_bf(g * (1.f / (1.f + expf(-g)))) * u;  // as silu_mul_kernel
        }
        o[q] = pack_bf2(r2[0], r2[1]);
      }
      uint16_t* dst = p.y + (int64_t)m * p.ldy + j0 + cc;
      if (p.yvec) {
        *reinterpret_cast<uint4*>(dst) = make_uint4(o[0], o[1], o[2], o[3]);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) dst[j] = (uint16_t)(o[j >> 1] >> (16 * (j & 1)));
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = r0 + 16 * i, m = m0 + row, n = n0 + c8;
    if (m >= p.M || n >= N) continue;
    const uint4 v = *reinterpret_cast<const uint4*>(os + row * GM_OS + c8);
    uint16_t* dst = p.y + (int64_t)m * p.ldy + c0 + n;
    if (p.yvec) {
      *reinterpret_cast<uint4*>(dst) = v;
    } else {
      const uint32_t h[4] = {v.x, v.y, v.z, v.w};
      for (int j = 0; j < 8 && n + j < N; ++j)
        dst[j] = (uint16_t)(h[j >> 1] >> (16 * (j & 1)));
    }
  }
}

// Epilogue of a K-split GEMM: y[m, n] from the partial sums, a workgroup per
// 16 rows x 64 columns, a thread per (row, four columns): every thread's
// partial sums go out at once (one memory round trip).  The LoRA t of the 16
// rows is summed once into LDS (slice order, as every consumer sums them) and
// the 64 columns' LoRA B rows are staged in LDS once (the per-row finish of
// the decode batches loads them for every row: 32 bytes of B per output).
constexpr int FR_ROWS = 16, FR_COLS = 64;

__global__ void __launch_bounds__(256) nf4_finish_rows(LinParts o, uint16_t* __restrict__ y,
                                                       int64_t ldy) {
  __shared__ float ts[FR_ROWS][MAXSEG * 16];
  __shared__ uint4 lbs[FR_COLS * 2];  // B rows (r == 16, 16-byte aligned): two halves per column
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * FR_ROWS, c0 = blockIdx.x * FR_COLS;
  const int rows = min(FR_ROWS, o.M - m0);
  const int row = tid >> 4, n = c0 + 4 * (tid & 15);
  const int m = m0 + row;
  Fetch4<> f;  // lin_fetch4 without the B rows (staged below)
  if (m < o.M && n < o.N) {
    const float4* p = reinterpret_cast<const float4*>(o.part + (int64_t)m * o.N + n);
    const int64_t stride = (int64_t)o.M * o.N / 4;
#pragma unroll
    for (int k = 0; k < MAX_SLICES; ++k)
      if (k < o.S) f.part[k] = p[k * stride];
    f.seg = lin_seg(o, n);
    f.nl = n - (f.seg > 0 ? sel_seg(o.seg_end, f.seg - 1) : 0);
    const uint16_t* bias = sel_seg(o.bias, f.seg);
    if (bias && o.bias_vec) f.bias = *reinterpret_cast<const uint2*>(bias + f.nl);
  }
  if (o.r > 0) {
    const int per_row = o.nseg * 4;
    const int64_t stride = (int64_t)o.nseg * o.M * 4;  // float4s per slice
    for (int i = tid; i < rows * per_row; i += 256) {
      const int rr = i / per_row, it = i - rr * per_row;
      const int seg = it >> 2, q = it & 3;
      const float4* p =
          reinterpret_cast<const float4*>(o.tpart + ((int64_t)seg * o.M + m0 + rr) * 16) + q;
      float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
      for (int k = 0; k < o.S; ++k) {
        const float4 v = p[k * stride];
        acc.x += v.x;
        acc.y += v.y;
        acc.z += v.z;
        acc.w += v.w;
      }
      float* t = &ts[rr][seg * 16 + 4 * q];
      t[0] = round_bf(acc.x);
      t[1] = round_bf(acc.y);
      t[2] = round_bf(acc.z);
      t[3] = round_bf(acc.w);
    }
    if (o.lb_vec && tid < FR_COLS * 2) {
      const int col = min(c0 + (tid >> 1), o.N - 1);
      const int seg = lin_seg(o, col);
      const int nl = col - (seg > 0 ? sel_seg(o.seg_end, seg - 1) : 0);
      lbs[tid] = reinterpret_cast<const uint4*>(sel_seg(o.lb, seg) + (int64_t)nl * 16)[tid & 1];
    }
  }
  __syncthreads();
  if (m >= o.M || n >= o.N) return;
  if (o.r > 0 && o.lb_vec) {
#pragma unroll
    for (int j = 0; j < 8; ++j) f.lb[j] = lbs[8 * (tid & 15) + j];
  }
  float v[4];
  lin_finish4(o, ts[row], f, v);
  uint16_t* yr = y + (int64_t)m * ldy + n;
  if (aligned8(yr)) {
    *reinterpret_cast<uint2*>(yr) = make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c) yr[c] = f2bf(v[c]);
  }
}

// ------------------------------------------------- K in steps of 128, bf16 --
//
// The same linear for K % 128 == 0 and r <= 16 on the ring of gemm16.hip: x comes to LDS
// by global_load_lds in stages of 32 K values, four in flight, and the weight is
// decoded once per workgroup (not once per 32-column wave) into LDS, in the piece order
// its operand reads want.
//  * Superstage = 128 K values = four stages. Its packed bytes (16 rows x 64 bytes per
//    1 KiB piece), absmax (one per row and stage) and LoRA A rows come to LDS too,
//    into a ring of three: the one being decoded, the next and the one being fetched.
//  * Step st multiplies stage st, decodes stage st + 2 (a thread: 8 or 16 nibbles of
//    one row, whose codebook is built once per two stages: an absmax block has 64
//    values at least), fetches stage st + 3 of x and a quarter of the
//    superstage after next. The decoded stages alternate between two LDS slots: the
//    slot written in step st was read before its barrier. Every wait counts loads.
//  * LoRA: x A^T is one more MFMA column of the tile, its rows shared out among the
//    waves; t passes through LDS once and its product with B is one MFMA per tile.
//  * SILU: the four column tiles of a wave are gate, gate, up, up of the same 32
//    columns, so a lane ends with both factors of 8 activation columns.
//  * KS = 2: two K groups of waves, each with rings of its own, halve the chain of
//    steps of a small launch; they exchange halves of their sums through LDS.
// Bound by the vector ALUs' decode beside the MFMAs (about 90 vector instructions per
// stage and wave against 16 MFMAs of 16 cycles on the 128 x 128 tile), and below one
// workgroup per CU by the chain of a step (LDS, decode, barrier: 0.32 us per 64 K
// values at 64 x 64). Against nf4_gemm_mfma, us at 511 rows: 2048 x 1536, r 16: 28.2 ->
// 13.9; 1536 x 1536, r 16: 24.1 -> 13.3; gate|up 2 x 8960 x 1536: 64.6 -> 51.9; 1536 x
// 8960: 37.5 -> 36.6; 4608 x 3584, r 16: 55.5 -> 45.1; at 2048 rows: 39.2 -> 27.1, 38.2
// -> 25.9, 177.7 -> 155.3, 111.6 -> 91.5, 158.1 -> 136.4.
struct K2Args {
  const uint16_t* x;
  int64_t ldx;
  const uint8_t* w;
  const float* absmax;
  const float* code16;
  int bs_shift;
  int nseg;
  int seg_end[MAXSEG];
  int seg_tile[MAXSEG + 1];
  const uint16_t* bias[MAXSEG];
  const uint16_t* la[MAXSEG];
  const uint16_t* lb[MAXSEG];
  int r;
  float scaling;
  uint16_t* y;
  int64_t ldy;
  int M, K;
  int MT, NT;
  int nss;  // superstages
  int kst;  // superstages per K slice (gridDim.y slices)
  bool yvec, lbvec;  // 16-byte stores of y, 16-byte loads of LoRA B
  float* part;  // K slices: part[slice][m][n] (slice stride psl, row stride ldp)
  int64_t ldp, psl;
  float* tpart;  // LoRA t partials [slice][16] at segment stride tseg
  int64_t tsl, tseg;
  int silu_I;
};

enum K2Mode { K2_OUT, K2_PART, K2_SILU };

template <K2Mode MODE, bool LORA, int RM, int RN, int WM, int WN, int KS>
struct K2Shape {
  static constexpr int BM = 16 * RM * WM, BN = 16 * RN * WN, W = WM * WN, T = 64 * W;
  static constexpr int TA = BM / 16, TB = BN / 16;     // pieces of a stage of x, of the weight
  static constexpr int LDA = TA / W, LDX = LDA + LORA; // x, x and LoRA A loads per wave and step
  static constexpr int EW = TB / W, EA = 1, E = EW + EA;  // other loads per wave and superstage
  static constexpr int TPR = T / BN;                   // threads per weight row
  static constexpr int ST = (TA + LORA) * 1024, SB = TB * 1024;  // bytes of a stage
  static constexpr int RAW = TB * 1024 + 8 * BN;       // a superstage's packed bytes, absmax
  static constexpr int XS = 4 * ST, BS = 2 * SB, LDS = XS + BS + 3 * RAW;  // of a K group
  // exchange of two K groups: sums from 0, t sums from XT, then t
  static constexpr int XT = W * RM * RN * 1024;
  static constexpr int TS = XT + (LORA ? 2 * W * (RM / WN > 0 ? RM / WN : 1) * 1024 : 0);
  static_assert(KS == 1 || (KS == 2 && TS + (LORA ? BM * 64 : 0) <= 2 * LDS), "exchange");
  static constexpr int ex(int j) { return ((j & 3) + 1) * E / 4 - (j & 3) * E / 4; }
  static_assert(TA % W == 0 && TB % W == 0 && (!LORA || W == 4) && BN / 32 <= W && TPR >= 1 && 4 % TPR == 0, "");
};

template <K2Mode MODE, bool LORA, int RM, int RN, int WM, int WN, int KS>
__global__ void __launch_bounds__(64 * WM * WN * KS, 2) nf4_gemm_k2(K2Args p) {
  using S = K2Shape<MODE, LORA, RM, RN, WM, WN, KS>;
  constexpr int BN = S::BN, W = S::W, RH = RM / 2, NIB = 32 / S::TPR;
  constexpr bool SILU = MODE == K2_SILU;
  static_assert(!SILU || (RN == 4 && !LORA), "gate, gate, up, up");
  extern __shared__ __align__(16) char smem0[];
  // K group of this wave, thread and wave in the group
  const int grp = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / S::T);
  const int tid = threadIdx.x % S::T, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  char* const smem = smem0 + grp * S::LDS;
  const int ln = lane & 15, lg = lane >> 4;
  const int bx = blockIdx.x, run = bx & 7, T = p.MT * p.NT;
  const int t = ((run * T) >> 3) + (bx >> 3);
  if (t >= (((run + 1) * T) >> 3)) return;  // past the end of this run
  const int nt = t / p.MT, mt = t - nt * p.MT;
  const int seg = (nt >= p.seg_tile[1]) + (nt >= p.seg_tile[2]) + (nt >= p.seg_tile[3]);
  const int c0 = seg > 0 ? sel4(p.seg_end[0], p.seg_end[1], p.seg_end[2], p.seg_end[3],
                                seg - 1) : 0;
  const int N = sel4(p.seg_end[0], p.seg_end[1], p.seg_end[2], p.seg_end[3], seg) - c0;
  const uint16_t* const sbias = sel4(p.bias[0], p.bias[1], p.bias[2], p.bias[3], seg);
  const uint16_t* const sla = sel4(p.la[0], p.la[1], p.la[2], p.la[3], seg);
  const uint16_t* const slb = sel4(p.lb[0], p.lb[1], p.lb[2], p.lb[3], seg);
  const int lt = nt - sel4(p.seg_tile[0], p.seg_tile[1], p.seg_tile[2], p.seg_tile[3], seg);
  const int m0 = mt * S::BM, n0 = lt * (SILU ? BN / 2 : BN);

  // weight row (of the whole stacked weight) of row i of piece pb
  auto wrow = [&](int pb, int i) __attribute__((always_inline)) {
    const int g = pb / RN, j = pb % RN;
    if (SILU) {
      const int a = n0 + 32 * g + 8 * (i >> 2) + 4 * (j & 1) + (i & 3);
      return (j >> 1) * p.silu_I + min(a, p.silu_I - 1);
    }
    return c0 + min(n0 + 16 * RN * g + 4 * RN * (i >> 2) + 4 * j + (i & 3), N - 1);
  };
  // superstages of this workgroup, of this group (the second's may be none: its loads
  // then repeat valid ones)
  const int wss0 = blockIdx.y * p.kst, wnss = min(p.nss, wss0 + p.kst) - wss0;
  const int lss = KS == 1 ? wnss : (wnss + 1) >> 1;  // of the longer group
  const int nst = 4 * (grp == 0 ? lss : wnss - lss), last = max(nst, 4) - 1;
  const int64_t k0 = 128 * (int64_t)min(wss0 + grp * lss, p.nss - 1);
  const uint32_t lb0 = lds_address(smem);

  // x: this wave's pieces of a stage
  const int prow = lane >> 2, pch = (lane & 3) ^ ((prow >> 1) & 3);
  const char* const xb = reinterpret_cast<const char*>(p.x + (int64_t)m0 * p.ldx + k0);
  uint32_t xoff[S::LDA];
#pragma unroll
  for (int i = 0; i < S::LDA; ++i)
    xoff[i] = min(16 * (wave * S::LDA + i) + prow, p.M - 1 - m0) * (uint32_t)(2 * p.ldx) + 16 * pch;
  auto fetch_x = [&](int st, int i) __attribute__((always_inline)) {
    dma16(lb0 + (st & 3) * S::ST + (wave * S::LDA + i) * 1024, xoff[i],
          xb + 64 * (int64_t)min(st, last));
  };
  // packed weight: piece e W + wave, 16 rows x 64 bytes, chunk ^ (row / 4 % 4)
  const int wch = (lane & 3) ^ ((prow >> 2) & 3);
  uint32_t woff[S::EW];
#pragma unroll
  for (int e = 0; e < S::EW; ++e)
    woff[e] = (uint32_t)wrow(e * W + wave, prow) * (uint32_t)(p.K / 2) + 16 * wch;
  const char* const wb = reinterpret_cast<const char*>(p.w) + k0 / 2;
  // LoRA A of a stage: this wave's 256 bytes (4 rows), ranks >= r repeat rank r - 1
  const int lrow = 4 * wave + (lane >> 4), lch = ((lane >> 2) & 3) ^ ((lrow >> 1) & 3);
  const uint32_t loff =
      LORA ? min(lrow, p.r - 1) * (uint32_t)(2 * p.K) + 16 * lch + 4 * (lane & 3) : 0;
  const char* const lab = reinterpret_cast<const char*>(sla) + 2 * k0;
  auto fetch_l = [&](int st) __attribute__((always_inline)) {
    if (LORA)
      dma4(lb0 + (st & 3) * S::ST + S::TA * 1024 + wave * 256, loff,
           lab + 64 * (int64_t)min(st, last));
  };
  // absmax: 64 values of the superstage's half id % 2, rows 64 (id / 2) + lane of the
  // piece order (id = wave, modulo what there is)
  const int aid = wave % (BN / 32), arho = 64 * (aid >> 1) + lane;
  const uint32_t aidx = (uint32_t)wrow(arho >> 4, arho & 15) * (uint32_t)p.K + (uint32_t)k0 +
                        64 * (aid & 1);
  constexpr int OA = S::TB * 1024;  // absmax in a raw slot: [half][row]
  auto fetch_raw = [&](int ss, int e) __attribute__((always_inline)) {
    const uint32_t slot = lb0 + S::XS + S::BS + (ss % 3) * S::RAW;
    const int sc = min(ss, last >> 2);
    if (e < S::EW)
      dma16(slot + (e * W + wave) * 1024, woff[e], wb + 64 * (int64_t)sc);
    else
      dma4(slot + OA + ((aid & 1) * BN + 64 * (aid >> 1)) * 4,
           ((aidx + 128u * sc) >> p.bs_shift) * 4, p.absmax);
  };
  // the extra loads of phase j: raw loads [j E / 4, (j + 1) E / 4) of superstage ss
  auto extras = [&](int ss, auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
#pragma unroll
    for (int e = j * S::E / 4; e < (j + 1) * S::E / 4; ++e) fetch_raw(ss, e);
  };

  float code[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) code[j] = load_uniform(p.code16 + j);
  const int rho = tid / S::TPR, sub = tid % S::TPR, dr = rho & 15;
  const int wread = (rho >> 4) * 1024 + dr * 64 + (16 / S::TPR) * sub, wsw = (dr >> 2) & 3;
  char* const bw = smem + S::XS + (rho >> 4) * 1024 + dr * 64;
  Lut lut;
  uint32_t raw[NIB / 8];
  float am = 0.f;
  // packed nibbles and absmax of stage d (j = d % 4) of this thread
  auto take = [&](int d, int j) __attribute__((always_inline)) {
    const char* const slot = smem + S::XS + S::BS + ((d >> 2) % 3) * S::RAW;
    const char* const q = slot + wread + 16 * (j ^ wsw);
    if constexpr (NIB == 16) {
      const uint2 v = *reinterpret_cast<const uint2*>(q);
      raw[0] = v.x;
      raw[1] = v.y;
    } else if constexpr (NIB == 32) {
      const uint4 v = *reinterpret_cast<const uint4*>(q);
      raw[0] = v.x;
      raw[1] = v.y;
      raw[2] = v.z;
      raw[3] = v.w;
    } else {
      raw[0] = *reinterpret_cast<const uint32_t*>(q);
    }
    if (!(j & 1)) am = *reinterpret_cast<const float*>(slot + OA + ((j >> 1) * BN + rho) * 4);
  };
  auto decode = [&](int d, int j) __attribute__((always_inline)) {
    if (!(j & 1)) lut = make_lut(code, am);  // an absmax block is two stages at least
#pragma unroll
    for (int c = 0; c < NIB / 8; ++c) {
      const int ch = sub * (NIB / 8) + c;
      *reinterpret_cast<uint4*>(bw + (d & 1) * S::SB + 16 * (ch ^ ((dr >> 1) & 3))) =
          interleave8(decode8(raw[c], lut));
    }
  };

  // ---- prologue: superstages 0 and 1, stages 0 .. 2 of x, the first half of
  // superstage 2 (in the order the steps before step 0 would have used)
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
#pragma unroll
  for (int e = 0; e < S::E; ++e) fetch_raw(0, e);
#pragma unroll
  for (int e = 0; e < S::E; ++e) fetch_raw(1, e);
#pragma unroll
  for (int st = 0; st < 3; ++st) {
#pragma unroll
    for (int i = 0; i < S::LDA; ++i) fetch_x(st, i);
    fetch_l(st);
    if (st == 1) extras(2, I0{});
    if (st == 2) extras(2, I1{});
  }
  constexpr int PRE = 3 * S::LDX + S::ex(0) + S::ex(1);  // loads after the raw ones
  wait_vm<PRE + S::E>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  take(0, 0);
  decode(0, 0);
  take(1, 1);
  decode(1, 1);

  const int wm = wave / WN, wn = wave % WN;
  const int off = ln * 64 + 16 * (lg ^ ((ln >> 1) & 3));
  const char* const la = smem + wm * RM * 1024 + off;
  const char* const lbp = smem + S::XS + wn * RN * 1024 + off;
  f32x4_t acc[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  constexpr int RT = RM / WN > 0 ? RM / WN : 1;  // row tiles of t per wave
  f32x4_t tacc[LORA ? RT : 1];
#pragma unroll
  for (int i = 0; i < (LORA ? RT : 1); ++i) tacc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  uint4 a0[RH], a1[RH], b0[RN], b1[RN], l0 = make_uint4(0, 0, 0, 0), l1 = l0;
  auto read = [&](const char* q, auto& x) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < (int)(sizeof(x) / 16); ++i)
      x[i] = *reinterpret_cast<const uint4*>(q + i * 1024);
  };
  auto read_l = [&](int st, uint4& l) __attribute__((always_inline)) {
    if (LORA)
      l = *reinterpret_cast<const uint4*>(smem + (st & 3) * S::ST + S::TA * 1024 + off);
  };
  // x A^T of row tile i (static) in the wave that has it
  auto mul_t = [&](int i, const uint4& a, const uint4& l) __attribute__((always_inline)) {
    if (LORA && i / RT == wn) tacc[i % RT] = mfma16x16x32(l, a, tacc[i % RT]);
  };
  wait_vm_lds<PRE - S::LDX>();  // stage 0 of x, and this wave's decoded values
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  read(lbp, b0);
  read(la, a0);
  read_l(0, l0);

  // step st, j = (st + 2) % 4 the phase of the stage that it decodes
  auto step = [&](int st, auto jc, uint4 (&bc)[RN], uint4& lc, uint4 (&bn)[RN], uint4& lnx)
                  __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
    __builtin_amdgcn_sched_barrier(0);
    take(st + 2, j);
    read(la + (st & 3) * S::ST + RH * 1024, a1);
#pragma unroll
    for (int i = 0; i < RH; ++i) {
#pragma unroll
      for (int q = 0; q < RN; ++q) acc[i][q] = mfma16x16x32(bc[q], a0[i], acc[i][q]);
      mul_t(i, a0[i], lc);
    }
    // stage st + 1 of x has landed, and every wave's LDS work is done: its reads of
    // the slots written next, its decoded values of stage st + 1
    wait_vm_lds<S::ex(j + 2) + S::LDX + S::ex(j + 3)>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(lbp + ((st + 1) & 1) * S::SB, bn);
    read(la + ((st + 1) & 3) * S::ST, a0);
    read_l(st + 1, lnx);
    decode(st + 2, j);
#pragma unroll
    for (int i = 0; i < RH; ++i) {
#pragma unroll
      for (int q = 0; q < RN; ++q) acc[RH + i][q] = mfma16x16x32(bc[q], a1[i], acc[RH + i][q]);
      mul_t(RH + i, a1[i], lc);
    }
#pragma unroll
    for (int i = 0; i < S::LDA; ++i) fetch_x(st + 3, i);
    fetch_l(st + 3);
    extras(((st + 2) >> 2) + 2, jc);
  };
  for (int st = 0; st < nst; st += 4) {
    step(st, I2{}, b0, l0, b1, l1);
    step(st + 1, I3{}, b1, l1, b0, l0);
    step(st + 2, I0{}, b0, l0, b1, l1);
    step(st + 3, I1{}, b1, l1, b0, l0);
  }
  if (KS > 1 && nst < 4 * lss)  // the longer group's last four barriers
#pragma unroll
    for (int i = 0; i < 4; ++i) __builtin_amdgcn_s_barrier();
  wait_vm<0>();
  if (LORA) {  // ranks >= r, which repeat rank r - 1, must not reach a product with 0
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (4 * lg + e >= p.r) tacc[i][e] = 0.f;
  }

  // Row tiles that this wave finishes: with two K groups half of them, whose other
  // partial sum comes through LDS from the same wave of the other group.
  constexpr int NR = KS == 1 ? RM : RH;
  const int rt0 = wm * RM + (KS == 1 ? 0 : grp * RH);
  f32x4_t fin[NR][RN];
  uint16_t* const ts = reinterpret_cast<uint16_t*>(smem0 + (KS == 1 ? 0 : S::TS));
  if constexpr (KS == 1) {
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int q = 0; q < RN; ++q) fin[i][q] = acc[i][q];
    if (LORA) __syncthreads();  // every wave is past its last read of the rings
  } else {
    f32x4_t* const xs = reinterpret_cast<f32x4_t*>(smem0) + lane;
    f32x4_t* const xt = reinterpret_cast<f32x4_t*>(smem0 + S::XT) + lane;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RH; ++i)
#pragma unroll
      for (int q = 0; q < RN; ++q) {
        xs[((grp * W + wave) * RH * RN + i * RN + q) * 64] = grp == 0 ? acc[RH + i][q] : acc[i][q];
        fin[i][q] = grp == 0 ? acc[i][q] : acc[RH + i][q];
      }
    if (LORA)
#pragma unroll
      for (int i = 0; i < RT; ++i) xt[((grp * W + wave) * RT + i) * 64] = tacc[i];
    __syncthreads();
    const int og = 1 - grp;
#pragma unroll
    for (int i = 0; i < RH; ++i)
#pragma unroll
      for (int q = 0; q < RN; ++q) fin[i][q] += xs[((og * W + wave) * RH * RN + i * RN + q) * 64];
    if (LORA)
#pragma unroll
      for (int i = 0; i < RT; ++i) tacc[i] += xt[((og * W + wave) * RT + i) * 64];
  }

  const int nl = n0 + wn * 16 * RN + 4 * RN * lg;  // this lane's first column
  if constexpr (MODE == K2_PART) {
    float* const pp = p.part + blockIdx.y * p.psl + c0;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int m = m0 + (rt0 + i) * 16 + ln;
      if (m >= p.M) continue;
#pragma unroll
      for (int q = 0; q < RN; ++q)
        if (nl + 4 * q < N)  // N % 16 == 0
          *reinterpret_cast<float4*>(pp + (int64_t)m * p.ldp + nl + 4 * q) =
              make_float4(fin[i][q][0], fin[i][q][1], fin[i][q][2], fin[i][q][3]);
    }
    if (LORA && lt == 0 && grp == 0) {
      float* const tp = p.tpart + blockIdx.y * p.tsl + seg * p.tseg;
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const int m = m0 + (wm * RM + wn * RT + i) * 16 + ln;
        if (wn * RT + i < RM && m < p.M)
          *reinterpret_cast<float4*>(tp + (int64_t)m * 16 + 4 * lg) =
              make_float4(tacc[i][0], tacc[i][1], tacc[i][2], tacc[i][3]);
      }
    }
  } else if constexpr (SILU) {
    const int a = n0 + 32 * wn + 8 * lg;  // act columns a .. a + 7
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int m = m0 + (rt0 + i) * 16 + ln;
      uint32_t o[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float r2[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int e = 2 * q + h;
          const float gv = round_bf(fin[i][e >> 2][e & 3]);
          const float uv = round_bf(fin[i][2 + (e >> 2)][e & 3]);
          r2[h] = round_bf(gv * (1.f / (1.f + expf(-gv)))) * uv;  // as silu_mul_kernel
        }
        o[q] = pack_bf2(r2[0], r2[1]);
      }
      if (m < p.M && a < p.silu_I) {  // I % 8 == 0
        uint16_t* const d = p.y + (int64_t)m * p.ldy + a;
        if (p.yvec) {
          *reinterpret_cast<uint4*>(d) = make_uint4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) d[e] = (uint16_t)(o[e >> 1] >> (16 * (e & 1)));
        }
      }
    }
  } else {
    uint4 low[RN];
    if (LORA) {
      // t [BM][32], ranks >= 16 zero
#pragma unroll
      for (int i = 0; i < RT; ++i)
        if (grp == 0 && wn * RT + i < RM) {
          uint16_t* d = ts + ((wm * RM + wn * RT + i) * 16 + ln) * 32 + 4 * lg;
          *reinterpret_cast<uint2*>(d) = make_uint2(pack_bf2(tacc[i][0], tacc[i][1]),
                                                    pack_bf2(tacc[i][2], tacc[i][3]));
          *reinterpret_cast<uint2*>(d + 16) = make_uint2(0, 0);
        }
#pragma unroll
      for (int q = 0; q < RN; ++q) {
        const int col = min(n0 + wn * 16 * RN + 4 * RN * (ln >> 2) + 4 * q + (ln & 3), N - 1);
        const uint16_t* br = slb + (int64_t)col * p.r;
        low[q] = make_uint4(0, 0, 0, 0);
        if (p.lbvec) {
          if (8 * lg < p.r) low[q] = *reinterpret_cast<const uint4*>(br + 8 * lg);
        } else {
          uint32_t v[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = 8 * lg + e < p.r ? br[8 * lg + e] : 0u;
          low[q] = make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16),
                              v[6] | (v[7] << 16));
        }
      }
      __syncthreads();
    }
    float bias[4 * RN];
    if (sbias) {
#pragma unroll
      for (int e = 0; e < 4 * RN; ++e) bias[e] = bf2f(sbias[min(nl + e, N - 1)]);
    }
    const float sc = round_bf(p.scaling);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int row = (rt0 + i) * 16 + ln, m = m0 + row;
      uint4 tv;
      if (LORA) tv = *reinterpret_cast<const uint4*>(ts + row * 32 + 8 * lg);
      uint32_t o[2 * RN];
#pragma unroll
      for (int q = 0; q < RN; ++q) {
        f32x4_t u{0.f, 0.f, 0.f, 0.f};
        if (LORA) u = mfma16x16x32(low[q], tv, u);
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = round_bf(fin[i][q][e]);
          if (sbias) v[e] = round_bf(v[e] + bias[4 * q + e]);
          if (LORA) v[e] = round_bf(v[e] + round_bf(round_bf(u[e]) * sc));
        }
        o[2 * q] = pack_bf2(v[0], v[1]);
        o[2 * q + 1] = pack_bf2(v[2], v[3]);
      }
      if (m < p.M) {
        uint16_t* const d = p.y + (int64_t)m * p.ldy + c0 + nl;
        if (p.yvec) {  // segment ends % 8 == 0
#pragma unroll
          for (int h = 0; h < RN / 2; ++h)
            if (nl + 8 * h < N)
              *reinterpret_cast<uint4*>(d + 8 * h) =
                  make_uint4(o[4 * h], o[4 * h + 1], o[4 * h + 2], o[4 * h + 3]);
        } else {
#pragma unroll
          for (int e = 0; e < 4 * RN; ++e)
            if (nl + e < N) d[e] = (uint16_t)(o[e >> 1] >> (16 * (e & 1)));
        }
      }
    }
  }
}

// Tiles of nf4_gemm_k2 (ks K groups) and their time model in us: a round of workgroups
// costs `fixed` and, per step, `step` alone on a CU, `more` for each further one that fits
// (occ, occ_l with LoRA), `lora` with LoRA. Over 560 shapes of 65 .. 4096 rows, each
// measured with every tile and up to 13 slice counts, its r.m.s. error is 8 %; what it
// picks is within 1 % of the best one at 90 % of them, within 13 % at all.
struct K2Tile {
  int bm, bn, ks, occ, occ_l;
  double fixed, step, more, lora;
};
constexpr K2Tile K2_TILE[] = {{256, 256, 1, 1, 1, 10.2, 0.75, 0.0, 0.0},
                              {128, 128, 1, 2, 2, 3.9, 0.38, 0.21, 0.06},
                              {64, 128, 2, 1, 1, 3.4, 0.47, 0.0, 0.02},
                              {64, 64, 2, 2, 1, 1.8, 0.32, 0.22, 0.04},
                              {128, 128, 2, 1, 1, 5.1, 0.58, 0.0, 0.05}};
// Which tiles a form is built for.
constexpr bool k2_has(int tile, K2Mode mode, bool lora) {
  return tile == 0 ? !lora && mode != K2_PART : (mode != K2_SILU || tile == 1 || tile == 4);
}

// The tile for the segments' columns (SILU: I columns of half a tile each) in S K
// slices of kss superstages, and its time in us. Rounds are counted on the XCD with the
// most workgroups, ceil(tiles / 8) in every slice, over its 32 CUs: 28 tiles in 9 slices
// are 252 workgroups, but 36 on four of the XCDs, and take two rounds (128 x 3584 x
// 18944: 55.8 us, in 8 slices 39.2). A split also writes float32 partial sums, reads them
// back and launches the finish (3.2 us; 1.4 us per million sums, with LoRA 3.3 us per
// million outputs).
int k2_tile(int M, int nseg, const int* seg_end, int kss, int S, bool lora, K2Mode mode,
            double* us) {
  int best = -1;
  for (int i = 0; i < 5; ++i) {
    if (!k2_has(i, mode, lora)) continue;
    const K2Tile& c = K2_TILE[i];
    int64_t nt = 0;
    for (int s = 0, start = 0; s < nseg; start = seg_end[s], ++s)
      nt += cdiv(seg_end[s] - start, mode == K2_SILU ? c.bn / 2 : c.bn);
    const int64_t tiles = cdiv(cdiv(M, c.bm) * nt, 8) * S;  // of an XCD
    const int occ = lora ? c.occ_l : c.occ;
    auto round = [&](int64_t per_cu) {
      return c.fixed + 4 * (double)cdiv(kss, c.ks) *
                           (c.step + (lora ? c.lora : 0.0) + (double)(per_cu - 1) * c.more);
    };
    const int64_t full = tiles / (32 * occ), rem = tiles % (32 * occ);
    double t = 3.5 + (double)full * round(occ) + (rem ? round(cdiv(rem, 32)) : 0.0);
    if (S > 1) {
      const double outs = (double)M * seg_end[nseg - 1];
      t += 3.2 + outs * (S * 1.4e-6 + (lora ? 3.3e-6 : 0.0));
    }
    if (best < 0 || t < *us) best = i, *us = t;
  }
  return best;
}

bool k2_shape(int K, int r, int64_t wrows, int blocksize) {
  return K % 128 == 0 && r <= 16 && blocksize >= 64 && wrows * K < (1ll << 32);
}

template <K2Mode MODE, bool LORA, int RM, int RN, int WM, int WN, int KS>
int k2_go(const K2Args& a, unsigned slices, hipStream_t st) {
  using S = K2Shape<MODE, LORA, RM, RN, WM, WN, KS>;
  static_assert(KS * S::LDS <= 160 * 1024, "LDS");
  constexpr auto kern = nf4_gemm_k2<MODE, LORA, RM, RN, WM, WN, KS>;
  if (int rc = allow_dynamic_lds<kern, KS * S::LDS>()) return rc;
  kern<<<dim3(8u * (unsigned)cdiv((int64_t)a.MT * a.NT, 8), slices), KS * S::T, KS * S::LDS,
         st>>>(a);
  return launch_check("nf4_gemm_k2");
}

template <K2Mode MODE, bool LORA>
int k2_pick(const K2Args& a, int tile, unsigned slices, hipStream_t st) {
  if constexpr (k2_has(0, MODE, LORA))
    if (tile == 0) return k2_go<MODE, LORA, 8, 4, 2, 4, 1>(a, slices, st);
  if constexpr (k2_has(2, MODE, LORA))
    if (tile == 2) return k2_go<MODE, LORA, 2, 4, 2, 2, 2>(a, slices, st);
  if constexpr (k2_has(3, MODE, LORA))
    if (tile == 3) return k2_go<MODE, LORA, 2, 2, 2, 2, 2>(a, slices, st);
  if (tile == 4) return k2_go<MODE, LORA, 4, 4, 2, 2, 2>(a, slices, st);
  return k2_go<MODE, LORA, 4, 4, 2, 2, 1>(a, slices, st);
}

bool pow2(int v) { return v > 0 && (v & (v - 1)) == 0; }


bool gemm_ok(int M, int N, int K, int r, int blocksize) {
  return M >= 1 && N >= 1 && K >= 32 && K % 32 == 0 && r >= 0 && r <= GM_MAX_R &&
         pow2(blocksize) && blocksize >= 32;
}

}  // namespace

namespace grpo {

bool nf4_gemm_ok(int M, int N, int K, int r, int blocksize) {
  return gemm_ok(M, N, K, r, blocksize);
}

GemmPlan nf4_gemm_plan(int M, int K, int r, int blocksize, int nseg, const int* seg_end) {
  const int nst = (int)cdiv(K, GM_KS);
  GemmPlan pl{1, nst, 0, 0};
  const int64_t mt = cdiv(M, GM_BM);
  int64_t tiles = 0;
  bool split_ok = r <= 16 && nseg >= 1 && nseg <= MAXSEG;
  for (int s = 0, start = 0; s < nseg; start = seg_end[s], ++s) {
    tiles += mt * cdiv(seg_end[s] - start, GM_BN);
    split_ok = split_ok && seg_end[s] % 16 == 0;
  }
  if (!split_ok || nst < 6) return pl;
  const int N = seg_end[nseg - 1];
  if (k2_shape(K, r, N, blocksize)) {
    // The ring kernel (nf4_gemm_k2): the slice count of the least estimated time, of one
    // N-column segment, so that a size query without the segments gives the same.
    double best = 0.0;
    for (int S = 1; S <= std::min(MAX_SLICES, nst / 3); ++S) {
      const int kst = (int)cdiv(nst, S), slices = (int)cdiv(nst, kst);
      double t = 0.0;
      k2_tile(M, 1, &N, kst, slices, r > 0, slices > 1 ? K2_PART : K2_OUT, &t);
      if (S == 1 || t < best) {
        best = t;
        pl.S = slices;
        pl.kst = kst;
      }
    }
    if (pl.S > 1) {
      pl.part_bytes = (size_t)pl.S * M * N * 4;
      pl.tpart_bytes = r > 0 ? (size_t)pl.S * nseg * M * 16 * 4 : 0;
    }
    return pl;
  }
  // Time model (us) of S K slices, from measurements on MI355X: a workgroup
  // stage (128 K values) takes about 2.2 us whatever the tile count (its loads'
  // latency), 512 workgroups run at once; a split adds the float32 partial
  // sums (written and read back, ~4 TB/s), the finish launch and, with LoRA,
  // the finish's per-output rank sums (~2 ns per 1000 outputs).
  const double outs = (double)M * N;
  auto est = [&](int S, int* kst, int* slices) {
    *kst = (int)cdiv(nst, S);
    *slices = (int)cdiv(nst, *kst);
    double t = (double)cdiv(tiles * *slices, 512) * *kst * 2.2;
    if (*slices > 1) t += *slices * outs * 8.0 / 4e6 + 4.0 + (r > 0 ? outs * 2e-6 : 0.0);
    return t;
  };
  double best = 0.0;
  for (int S = 1; S <= std::min(MAX_SLICES, nst / 3); ++S) {
    int kst, slices;
    const double t = est(S, &kst, &slices);
    if (S == 1 || t < best) {
      best = t;
      pl.S = slices;
      pl.kst = kst;
    }
  }
  if (pl.S > 1) {
    pl.part_bytes = (size_t)pl.S * M * N * 4;
    pl.tpart_bytes = r > 0 ? (size_t)pl.S * nseg * M * 16 * 4 : 0;
  }
  return pl;
}

int nf4_gemm_launch(const uint16_t* x, int64_t ldx, const uint8_t* w, int64_t wrow0,
                    const float* absmax, const float* code16, int blocksize,
                    const GemmSegs& sg, int r, float scaling, uint16_t* y, int64_t ldy, int M,
                    int K, hipStream_t st, const GemmSplit* split, bool f16) {
  if (M < 0 || K < 0 || r < 0 || wrow0 < 0) return einval("negative dimension");
  if (sg.nseg < 1 || sg.nseg > MAXSEG) return einval("nseg must be in [1, 4]");
  int NT = 0, prev = 0;
  for (int s = 0; s < sg.nseg; ++s) {
    if (sg.seg_end[s] <= prev) return einval("segment ends must increase");
    if (!gemm_ok(M, sg.seg_end[s] - prev, K, r, blocksize)) {
      set_error("shape not supported by the NF4 GEMM (K %% 32 == 0, r <= 32, power-of-two "
                "blocksize >= 32)");
      return GRPO_EUNSUPPORTED;
    }
    NT += (int)cdiv(sg.seg_end[s] - prev, GM_BN);
    prev = sg.seg_end[s];
  }
  const int N = prev;
  if (M == 0) return GRPO_OK;
  if (!x || !w || !absmax || !code16 || !y) return einval("null pointer");
  if (ldx < K || ldx % 8 != 0 || !aligned16(x)) return einval("x rows must be 16-byte aligned");
  if (!aligned16(w)) return einval("w must be 16-byte aligned");
  if (ldy < N) return einval("ldy smaller than N");
  GemmArgs a{};
  a.x = x;
  a.ldx = ldx;
  a.w = w;
  a.absmax = absmax;
  a.code16 = code16;
  a.bs_shift = __builtin_ctz((unsigned)blocksize);
  a.wrow0 = wrow0;
  a.nseg = sg.nseg;
  a.yvec = aligned16(y) && ldy % 8 == 0;
  a.lbvec = r > 0 && r % 8 == 0;
  for (int s = 0, tile = 0; s < MAXSEG; ++s) {
    const bool on = s < sg.nseg;
    a.seg_end[s] = on ? sg.seg_end[s] : N;
    a.seg_tile[s] = on ? tile : NT;
    if (on) {
      const int ns = sg.seg_end[s] - (s > 0 ? sg.seg_end[s - 1] : 0);
      tile += (int)cdiv(ns, GM_BN);
      a.bias[s] = sg.bias[s];
      a.la[s] = r > 0 ? sg.la[s] : nullptr;
      a.lb[s] = r > 0 ? sg.lb[s] : nullptr;
      if (r > 0 && (!sg.la[s] || !sg.lb[s])) return einval("r > 0 needs lora_a and lora_b");
      if (r > 0 && !aligned16(sg.la[s])) return einval("lora_a must be 16-byte aligned");
      a.yvec = a.yvec && sg.seg_end[s] % 8 == 0;
      a.lbvec = a.lbvec && aligned16(sg.lb[s]);
    }
  }
  a.seg_tile[MAXSEG] = NT;
  a.r = r;
  a.scaling = scaling;
  a.y = y;
  a.ldy = ldy;
  a.M = M;
  a.N = N;
  a.K = K;
  a.MT = (int)cdiv(M, GM_BM);
  a.NT = NT;
  a.nst = (int)cdiv(K, GM_KS);
  a.kst = a.nst;
  unsigned slices = 1;
  if (split && split->S > 1) {
    if (r > 16) return einval("a K-split NF4 GEMM takes r <= 16");
    if (f16) return einval("a K-split NF4 GEMM is bf16 only");
    if (!split->part || (r > 0 && !split->tpart)) return einval("null partial-sum buffer");
    a.kst = split->kst;
    slices = (unsigned)split->S;
    if ((int64_t)(slices - 1) * a.kst >= a.nst) return einval("empty K slice");
    a.part = split->part;
    a.ldp = split->ldp;
    a.psl = split->psl;
    a.tpart = split->tpart;
    a.tsl = split->tsl;
    a.tseg = split->tseg;
  }
  if (!f16 && wrow0 == 0 && k2_shape(K, r, N, blocksize) && ldx < (1 << 22)) {
    K2Args k{};
    k.x = x;
    k.ldx = ldx;
    k.w = w;
    k.absmax = absmax;
    k.code16 = code16;
    k.bs_shift = a.bs_shift;
    k.nseg = sg.nseg;
    k.r = r;
    k.scaling = scaling;
    k.y = y;
    k.ldy = ldy;
    k.M = M;
    k.K = K;
    k.nss = a.nst;
    k.kst = a.kst;
    k.lbvec = a.lbvec;
    k.yvec = a.yvec;
    k.part = a.part;
    k.ldp = a.ldp;
    k.psl = a.psl;
    k.tpart = a.tpart;
    k.tsl = a.tsl;
    k.tseg = a.tseg;
    double us = 0.0;
    const int tile = k2_tile(M, sg.nseg, sg.seg_end, k.kst, (int)slices, r > 0,
                             slices > 1 ? K2_PART : K2_OUT, &us);
    k.MT = (int)cdiv(M, K2_TILE[tile].bm);
    for (int s = 0; s < MAXSEG; ++s) {
      k.seg_end[s] = a.seg_end[s];
      k.bias[s] = a.bias[s];
      k.la[s] = a.la[s];
      k.lb[s] = a.lb[s];
      k.seg_tile[s] = k.NT;
      if (s < sg.nseg)
        k.NT += (int)cdiv(sg.seg_end[s] - (s > 0 ? sg.seg_end[s - 1] : 0), K2_TILE[tile].bn);
    }
    for (int s = sg.nseg; s <= MAXSEG; ++s) k.seg_tile[s] = k.NT;
    if (slices > 1)
      return r > 0 ? k2_pick<K2_PART, true>(k, tile, slices, st)
                   : k2_pick<K2_PART, false>(k, tile, slices, st);
    return r > 0 ? k2_pick<K2_OUT, true>(k, tile, 1, st) : k2_pick<K2_OUT, false>(k, tile, 1, st);
  }
  const dim3 grid(8u * (unsigned)cdiv((int64_t)a.MT * a.NT, 8), slices);
  const int tc = r > 16 ? 2 : (r > 0 ? 1 : 0);
  int rc = GRPO_OK;
  auto go = [&](auto tag) {
    constexpr auto kern = decltype(tag)::value;
    if (!(rc = allow_dynamic_lds<kern, (int)GM_LDS>())) kern<<<grid, GM_T, GM_LDS, st>>>(a);
  };
  using KernT = void (*)(GemmArgs);
  if (f16) {
    if (tc == 2) go(std::integral_constant<KernT, nf4_gemm_mfma<2, true>>{});
    else if (tc == 1) go(std::integral_constant<KernT, nf4_gemm_mfma<1, true>>{});
    else go(std::integral_constant<KernT, nf4_gemm_mfma<0, true>>{});
  } else {
    if (tc == 2) go(std::integral_constant<KernT, nf4_gemm_mfma<2, false>>{});
    else if (tc == 1) go(std::integral_constant<KernT, nf4_gemm_mfma<1, false>>{});
    else go(std::integral_constant<KernT, nf4_gemm_mfma<0, false>>{});
  }
  return rc ? rc : launch_check("nf4_gemm_mfma");
}

int nf4_gemm_finish(const grpo_linear_parts_t* h, uint16_t* y, int64_t ldy, hipStream_t st) {
  LinParts o;
  if (int rc = make_parts(h, &o)) return rc;
  if (!y) return einval("null y");
  if (ldy < o.N) return einval("ldy smaller than N");
  nf4_finish_rows<<<dim3((unsigned)cdiv(o.N, FR_COLS), (unsigned)cdiv(o.M, FR_ROWS)), 256, 0,
                    st>>>(o, y, ldy);
  return launch_check("nf4_finish_rows");
}

bool nf4_gemm_silu_ok(int M, int I, int K, int blocksize) {
  return I >= 8 && I % 8 == 0 && gemm_ok(M, 2 * I, K, 0, blocksize);
}

int nf4_gemm_silu_launch(const uint16_t* x, int64_t ldx, const uint8_t* w, const float* absmax,
                         const float* code16, int blocksize, int I, int K, int M, uint16_t* act,
                         int64_t lda, hipStream_t st) {
  if (M < 0 || I < 0 || K < 0) return einval("negative dimension");
  if (M == 0 || I == 0) return GRPO_OK;
  if (!nf4_gemm_silu_ok(M, I, K, blocksize)) {
    set_error("shape not supported by the NF4 GEMM's gate|up SiLU form (I %% 8 == 0, K %% 32 "
              "== 0, power-of-two blocksize >= 32)");
    return GRPO_EUNSUPPORTED;
  }
  if (!x || !w || !absmax || !code16 || !act) return einval("null pointer");
  if (ldx < K || ldx % 8 != 0 || !aligned16(x)) return einval("x rows must be 16-byte aligned");
  if (!aligned16(w)) return einval("w must be 16-byte aligned");
  if (lda < I) return einval("lda smaller than I");
  GemmArgs a{};
  a.x = x;
  a.ldx = ldx;
  a.w = w;
  a.absmax = absmax;
  a.code16 = code16;
  a.bs_shift = __builtin_ctz((unsigned)blocksize);
  a.nseg = 1;
  a.M = M;
  a.K = K;
  a.MT = (int)cdiv(M, GM_BM);
  a.NT = (int)cdiv(I, GM_BN / 2);
  for (int s = 0; s < MAXSEG; ++s) {
    a.seg_end[s] = 2 * I;
    a.seg_tile[s] = s == 0 ? 0 : a.NT;
  }
  a.seg_tile[MAXSEG] = a.NT;
  a.y = act;
  a.ldy = lda;
  a.yvec = aligned16(act) && lda % 8 == 0;
  a.nst = a.kst = (int)cdiv(K, GM_KS);
  a.silu_I = I;
  if (k2_shape(K, 0, 2 * (int64_t)I, blocksize) && ldx < (1 << 22)) {
    K2Args k{};
    k.x = x;
    k.ldx = ldx;
    k.w = w;
    k.absmax = absmax;
    k.code16 = code16;
    k.bs_shift = a.bs_shift;
    k.nseg = 1;
    k.y = act;
    k.ldy = lda;
    k.M = M;
    k.K = K;
    k.nss = k.kst = a.nst;
    k.silu_I = I;
    k.yvec = a.yvec;
    double us = 0.0;
    const int tile = k2_tile(M, 1, &I, k.nss, 1, false, K2_SILU, &us);
    k.MT = (int)cdiv(M, K2_TILE[tile].bm);
    k.NT = (int)cdiv(I, K2_TILE[tile].bn / 2);
    for (int s = 0; s < MAXSEG; ++s) {
      k.seg_end[s] = 2 * I;
      k.seg_tile[s] = s == 0 ? 0 : k.NT;
    }
    k.seg_tile[MAXSEG] = k.NT;
    return k2_pick<K2_SILU, false>(k, tile, 1, st);
  }
  const dim3 grid(8u * (unsigned)cdiv((int64_t)a.MT * a.NT, 8));
  constexpr auto kern = nf4_gemm_mfma<0, false, true>;
  if (int rc = allow_dynamic_lds<kern, (int)GM_LDS>()) return rc;
  kern<<<grid, GM_T, GM_LDS, st>>>(a);
  return launch_check("nf4_gemm_mfma (gate|up SiLU)");
}

}  // namespace grpo

extern "C" int grpo_nf4_gemm_supported(int M, int N, int K, int r, int blocksize) {
  return gemm_ok(M, N, K, r, blocksize) ? 1 : 0;
}

extern "C" int grpo_nf4_gemm_tile(int M, int N, int K, int r, int blocksize, int silu, int* rows,
                                  int* cols, int* k_groups, int* slices) {
  const int64_t wrows = silu ? 2 * (int64_t)N : N;
  if (!rows || !cols || !k_groups || !slices || wrows > INT32_MAX || (silu && r != 0) ||
      !gemm_ok(M, (int)wrows, K, r, blocksize) || !k2_shape(K, r, wrows, blocksize))
    return 0;
  GemmPlan pl{1, (int)cdiv(K, GM_KS), 0, 0};
  if (!silu) pl = nf4_gemm_plan(M, K, r, blocksize, 1, &N);
  double us = 0.0;
  const K2Tile& t = K2_TILE[k2_tile(M, 1, &N, pl.kst, pl.S, r > 0,
                                    silu ? K2_SILU : (pl.S > 1 ? K2_PART : K2_OUT), &us)];
  *rows = t.bm;
  *cols = t.bn;
  *k_groups = t.ks;
  *slices = pl.S;
  return 1;
}

namespace {

int gemm_one(const void* x, int64_t ldx, const uint8_t* w, const float* absmax,
             const float* code16, int blocksize, const void* bias, const void* lora_a,
             const void* lora_b, int r, float scaling, void* y, int64_t ldy, int M, int N, int K,
             grpo_stream_t stream, bool f16) {
  if (N < 0) return einval("negative dimension");
  if (N == 0) return GRPO_OK;
  GemmSegs sg{};
  sg.nseg = 1;
  sg.seg_end[0] = N;
  sg.bias[0] = static_cast<const uint16_t*>(bias);
  sg.la[0] = static_cast<const uint16_t*>(lora_a);
  sg.lb[0] = static_cast<const uint16_t*>(lora_b);
  return nf4_gemm_launch(static_cast<const uint16_t*>(x), ldx, w, 0, absmax, code16, blocksize,
                         sg, r, scaling, static_cast<uint16_t*>(y), ldy, M, K,
                         as_stream(stream), nullptr, f16);
}

}  // namespace

extern "C" int grpo_nf4_gemm(const void* x, int64_t ldx, const uint8_t* w, const float* absmax,
                             const float* code16, int blocksize, const void* bias,
                             const void* lora_a, const void* lora_b, int r, float scaling,
                             void* y, int64_t ldy, int M, int N, int K, grpo_stream_t stream) {
  return gemm_one(x, ldx, w, absmax, code16, blocksize, bias, lora_a, lora_b, r, scaling, y, ldy,
                  M, N, K, stream, false);
}

extern "C" int grpo_nf4_gemm_f16(const void* x, int64_t ldx, const uint8_t* w,
                                 const float* absmax, const float* code16, int blocksize,
                                 const void* bias, const void* lora_a, const void* lora_b, int r,
                                 float scaling, void* y, int64_t ldy, int M, int N, int K,
                                 grpo_stream_t stream) {
  return gemm_one(x, ldx, w, absmax, code16, blocksize, bias, lora_a, lora_b, r, scaling, y, ldy,
                  M, N, K, stream, true);
}
