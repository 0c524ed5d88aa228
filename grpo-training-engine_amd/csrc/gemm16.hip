// 16-bit GEMM C = A B^T (both operands contiguous along K) for gfx950 with the
// rounding points and the LoRA term of the NF4 + LoRA linear in its epilogue;
// the training step's products over a weight dequantized once per call.
//
//  * Stage = 32 K values of the tile's rows of A and B, brought to LDS by
//    global_load_lds (16 bytes per lane, no registers), four stages in a ring:
//    two are in flight while one is multiplied and the next one's operands are read.
//    A stage is 1 KiB pieces of 16 rows x 64 bytes; in a piece, row w's four 16-byte
//    chunks are stored at chunk ^ (w / 2 % 4), which the loading lane chooses
//    by its global address, so that both the 64-byte row segments of a load
//    are contiguous and the 16 rows of an operand read fall on different banks.
//  * The waves' tiles: 16 RM rows x 16 RN columns of v_mfma_f32_16x16x32, the rows
//    of B in the A position, so a lane ends with columns of one row of C. B's rows
//    are dealt to the pieces so that these are 4 RN consecutive columns.
//  * A step's MFMAs are split into the two halves of the wave's rows: during the
//    first half the second half's operands are read, then comes the step's one
//    barrier (the next stage has landed), and during the second half the
//    next stage's operands are read and the stage three ahead is fetched, one
//    load after each row of MFMAs (loads and waits: lds_dma.hpp).
//  * Tiles go to the XCDs in eight equal runs, in groups of a few rows of tiles,
//    so that the tiles that run together on an XCD share operands in its L2.
//
// Bound: the matrix cores and the power they draw at the large tile, LDS reads
// (one 16-byte operand per 2..2.7 MFMAs) at the small ones, and load latency
// where a shape has fewer tiles than CUs. Measured on random normal bf16, without
// the LoRA term: 8192 x 3584 x 3584 176.9 us = 1189 TFLOP/s (the GEMM library 176.3;
// 211.8 with the fetches issued together behind the barrier), 4096 x 8960 x 1536 118
// us (116), 8192 x 512 x 3584 35.5 us (32.6), 2092 x 1536 x 1536 18.1 us (19.0), 256 x
// 1024 x 1024 5.4 us (19.3). The library's products need one more pass over C for
// each of bias, LoRA term and sum.
#include "gemm16.hpp"
#include "lds_dma.hpp"

#include <algorithm>

namespace grpo {
namespace {

constexpr int PIECE = 512;  // elements of a piece (16 rows x 32)
constexpr int RING = 4;

struct Args {
  Gemm16 g;
  int MT, NT;
  bool lowvec;  // 16-byte loads of low's rows
};

// RM x RN tiles of 16 x 16 per wave, WM x WN waves, GROUP rows of tiles.
template <bool F16, Gemm16Mode MODE, int RM, int RN, int WM, int WN, int GROUP>
__global__ void __launch_bounds__(64 * WM * WN, 2) gemm16_kernel(Args p) {
  constexpr int BM = 16 * RM * WM, BN = 16 * RN * WN, W = WM * WN;
  constexpr int TA = BM / 16, TB = BN / 16, LD = (TA + TB) / W, RH = RM / 2;
  static_assert((TA + TB) % W == 0 && RM % 2 == 0 && RN % 2 == 0, "whole pieces and halves");
  constexpr int ST = (TA + TB) * PIECE;
  extern __shared__ __align__(16) uint16_t lds[];  // [RING][ST]
  const Gemm16& g = p.g;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 15, lg = lane >> 4;
  const int bx = blockIdx.x, run = bx & 7;
  const int64_t T = (int64_t)p.MT * p.NT;
  const int t = (int)((run * T) >> 3) + (bx >> 3);
  if (t >= (int)(((run + 1) * T) >> 3)) return;  // past the end of this run
  const int grp = t / (GROUP * p.NT), rem = t - grp * GROUP * p.NT;
  const int rows = min(GROUP, p.MT - grp * GROUP);
  const int nt = rem / rows, mt = grp * GROUP + rem - nt * rows;
  const int m0 = mt * BM, n0 = nt * BN;

  // this wave's pieces of a stage: byte offsets from the tile's first row (rows
  // past the end repeat the last one and are not stored)
  const int prow = lane >> 2, pch = (lane & 3) ^ ((prow >> 1) & 3);
  const char* const ab = reinterpret_cast<const char*>(g.a + (int64_t)m0 * g.lda);
  const char* const bb = reinterpret_cast<const char*>(g.b + (int64_t)n0 * g.ldb);
  uint32_t voff[LD];
  const char* base[LD];
#pragma unroll
  for (int i = 0; i < LD; ++i) {
    const int pc = wave * LD + i, pb = pc - TA;
    const bool isa = pc < TA;
    const int brow = (pb / RN) * 16 * RN + (prow >> 2) * 4 * RN + 4 * (pb % RN) + (prow & 3);
    const uint32_t row = isa ? min(16 * pc + prow, g.M - 1 - m0) : min(brow, g.N - 1 - n0);
    base[i] = isa ? ab : bb;
    voff[i] = row * (uint32_t)(2 * (isa ? g.lda : g.ldb)) + 16 * pch;
  }
  const int nst = g.K / 32;
  const uint32_t lbase =
      lds_address(lds) + wave * LD * PIECE * 2;
  // stages past the end repeat the last one into slots that are not multiplied
  auto fetch = [&](int st, int i) __attribute__((always_inline)) {
    dma16(lbase + (st % RING) * (ST * 2) + i * PIECE * 2, voff[i],
          base[i] + 64 * (int64_t)min(st, nst - 1));
  };
#pragma unroll
  for (int st = 0; st < RING - 1; ++st)
#pragma unroll
    for (int i = 0; i < LD; ++i) fetch(st, i);

  const int wm = wave / WN, wn = wave % WN;
  const int nw = n0 + wn * 16 * RN;  // this wave's first column
  // the rank-r operand (row i of tile j: column 4 RN (i / 4) + 4 j + i % 4) and
  // the bias of this lane's columns, loaded with the first stages
  uint4 low[RN];
#pragma unroll
  for (int j = 0; j < RN; ++j) {
    const int col = min(nw + 4 * RN * (ln >> 2) + 4 * j + (ln & 3), g.N - 1);
    const uint16_t* q = g.low + col * g.ldl;
    low[j] = make_uint4(0, 0, 0, 0);
    if (p.lowvec) {
      if (8 * lg < g.r) low[j] = *reinterpret_cast<const uint4*>(q + 8 * lg);
    } else {
      uint32_t v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = 8 * lg + i < g.r ? q[8 * lg + i] : 0u;
      low[j] = make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16),
                          v[6] | (v[7] << 16));
    }
  }
  const int nl = nw + 4 * RN * lg;  // this lane's first column
  uint32_t bias[2 * RN];
  if (MODE == GEMM16_LORA && g.bias) {
#pragma unroll
    for (int i = 0; i < 2 * RN; ++i)
      bias[i] = g.bias[min(nl + 2 * i, g.N - 1)] | (uint32_t)g.bias[min(nl + 2 * i + 1, g.N - 1)]
                                                       << 16;
  }

  const int off = ln * 32 + 8 * (lg ^ ((ln >> 1) & 3));
  const uint16_t* const la = lds + wm * RM * PIECE + off;
  const uint16_t* const lb = lds + (TA + wn * RN) * PIECE + off;
  f32x4_t acc[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  uint4 a0[RH], a1[RH], b0[RN], b1[RN];
  auto read = [&](const uint16_t* q, auto& x) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < (int)(sizeof(x) / 16); ++i)
      x[i] = *reinterpret_cast<const uint4*>(q + i * PIECE);
  };
  wait_vm<(RING - 2) * LD>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  read(lb, b0);
  read(la, a0);
  auto step = [&](int st, uint4 (&bc)[RN], uint4 (&bn)[RN]) __attribute__((always_inline)) {
    const int cur = (st % RING) * ST, nxt = ((st + 1) % RING) * ST;
    __builtin_amdgcn_sched_barrier(0);
    read(la + cur + RH * PIECE, a1);
#pragma unroll
    for (int i = 0; i < RH; ++i)
#pragma unroll
      for (int j = 0; j < RN; ++j) acc[i][j] = mfma16x16x32_e<F16>(bc[j], a0[i], acc[i][j]);
#pragma unroll
    for (int i = 0; i < RH; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one operand read,
      __builtin_amdgcn_sched_group_barrier(0x8, RN, 0);   // one row of MFMAs
    }
    __builtin_amdgcn_sched_barrier(0);
    // stage st + 1 has landed for every wave, and every wave's reads of stage
    // st - 1 (whose slot is filled next) have been used
    wait_vm<(RING - 3) * LD>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(lb + nxt, bn);
    read(la + nxt, a0);
#pragma unroll
    for (int i = 0; i < RH; ++i) {
#pragma unroll
      for (int j = 0; j < RN; ++j)
        acc[RH + i][j] = mfma16x16x32_e<F16>(bc[j], a1[i], acc[RH + i][j]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = i * LD / RH; q < (i + 1) * LD / RH; ++q) fetch(st + RING - 1, q);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int st = 0;
  for (; st + 2 <= nst; st += 2) {
    step(st, b0, b1);
    step(st + 1, b1, b0);
  }
  if (st < nst) step(st, b0, b1);
  wait_vm<0>();  // nothing lands after the workgroup's end

  const float sc = MODE == GEMM16_LORA ? round_e<F16>(g.scaling) : 1.f;
#pragma unroll
  for (int i = 0; i < RM; ++i) {
    const int m = m0 + (wm * RM + i) * 16 + ln;
    const uint4 tv = *reinterpret_cast<const uint4*>(g.t + (int64_t)min(m, g.M - 1) * 32 + 8 * lg);
    uint32_t o[2 * RN];
#pragma unroll
    for (int j = 0; j < RN; ++j) {
      const f32x4_t u = mfma16x16x32_e<F16>(low[j], tv, f32x4_t{0.f, 0.f, 0.f, 0.f});
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[q] = round_e<F16>(acc[i][j][q]);
        float w = round_e<F16>(u[q]);
        if (MODE == GEMM16_LORA) {
          if (g.bias)
            v[q] = round_e<F16>(
                v[q] + e2f<F16>((uint16_t)(bias[2 * j + (q >> 1)] >> (16 * (q & 1)))));
          w = round_e<F16>(w * sc);
        }
        v[q] += w;
      }
      o[2 * j] = pack_e2<F16>(v[0], v[1]);
      o[2 * j + 1] = pack_e2<F16>(v[2], v[3]);
    }
    if (m < g.M) {
      uint16_t* d = g.c + (int64_t)m * g.ldc + nl;
#pragma unroll
      for (int h = 0; h < RN / 2; ++h)
        if (nl + 8 * h < g.N)  // N % 8 == 0
          *reinterpret_cast<uint4*>(d + 8 * h) =
              make_uint4(o[4 * h], o[4 * h + 1], o[4 * h + 2], o[4 * h + 3]);
    }
  }
}

template <bool F16, Gemm16Mode MODE, int RM, int RN, int WM, int WN, int GROUP>
int go(Args a, hipStream_t st) {
  constexpr int BM = 16 * RM * WM, BN = 16 * RN * WN, LDS = RING * (BM + BN) * 64;
  constexpr auto kern = gemm16_kernel<F16, MODE, RM, RN, WM, WN, GROUP>;
  a.MT = (int)cdiv(a.g.M, BM);
  a.NT = (int)cdiv(a.g.N, BN);
  if (int rc = allow_dynamic_lds<kern, LDS>()) return rc;
  const int64_t blocks = 8 * cdiv((int64_t)a.MT * a.NT, 8);
  kern<<<dim3((unsigned)blocks), 64 * WM * WN, LDS, st>>>(a);
  return launch_check("gemm16");
}

// Microseconds per stage of each tile, measured: alone on a CU, and per tile of
// a full chip. The tile with the least time for its count per CU runs:
// 256 x 256 once the chip is full of them (1189 TFLOP/s; 837 with 128 x 128),
// the smaller ones where a larger tile would leave CUs without work (2092 x 1536 x
// 1536: 33.1, 18.1, 22.0 and 28.0 us with the four tiles; 662 rows: 31.4, 12.5, 9.5
// and 9.7; 256 x 1024 x 1024: 22.4, 8.9, 6.5 and 5.4).
constexpr struct {
  int bm, bn;
  double alone, full;
} TILE[4] = {{256, 256, 0.70, 0.79},
             {128, 128, 0.32, 0.281},
             {64, 128, 0.198, 0.231},
             {64, 64, 0.165, 0.136}};

int tile_of(int M, int N) {
  int best = 0;
  double least = 0.0;
  for (int i = 0; i < 4; ++i) {
    const int64_t tiles = cdiv(M, TILE[i].bm) * cdiv(N, TILE[i].bn);
    const double us = std::max(TILE[i].alone, TILE[i].full * (double)cdiv(tiles, 256));
    if (i == 0 || us < least) best = i, least = us;
  }
  return best;
}

template <bool F16, Gemm16Mode MODE>
int pick(const Args& a, hipStream_t st) {
  switch (tile_of(a.g.M, a.g.N)) {
    case 0: return go<F16, MODE, 8, 4, 2, 4, 4>(a, st);
    case 1: return go<F16, MODE, 4, 4, 2, 2, 8>(a, st);
    case 2: return go<F16, MODE, 2, 4, 2, 2, 8>(a, st);
    default: return go<F16, MODE, 2, 2, 2, 2, 8>(a, st);
  }
}

}  // namespace

bool gemm16_ok(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb) {
  return M >= 1 && N >= 8 && N % 8 == 0 && K >= 32 && K % 32 == 0 && lda < (1 << 22) &&
         ldb < (1 << 22) && cdiv(M, 64) * cdiv(N, 64) < (1ll << 30);
}

int gemm16_launch(const Gemm16& g, Gemm16Mode mode, bool f16, hipStream_t st) {
  if (!gemm16_ok(g.M, g.N, g.K, g.lda, g.ldb)) {
    set_error("shape not supported by the 16-bit GEMM (N %% 8 == 0, K %% 32 == 0)");
    return GRPO_EUNSUPPORTED;
  }
  if (!g.a || !g.b || !g.c || !g.t || !g.low) return einval("null pointer");
  if (!aligned16(g.a) || !aligned16(g.b) || !aligned16(g.c) || !aligned16(g.t) || g.lda % 8 ||
      g.ldb % 8 || g.ldc % 8)
    return einval("GEMM rows must be 16-byte aligned");
  if (g.lda < g.K || g.ldb < g.K || g.ldc < g.N || g.ldl < g.r || g.r < 1 || g.r > 32)
    return einval("row stride too small or rank outside [1, 32]");
  const Args a{g, 0, 0, g.r % 8 == 0 && g.ldl % 8 == 0 && aligned16(g.low)};
  if (mode == GEMM16_ADD)
    return f16 ? pick<true, GEMM16_ADD>(a, st) : pick<false, GEMM16_ADD>(a, st);
  return f16 ? pick<true, GEMM16_LORA>(a, st) : pick<false, GEMM16_LORA>(a, st);
}

}  // namespace grpo

extern "C" int grpo_gemm16_tile(int M, int N, int* rows, int* cols) {
  using namespace grpo;
  if (M < 1 || N < 1 || !rows || !cols) return einval("bad GEMM dimensions");
  *rows = TILE[tile_of(M, N)].bm;
  *cols = TILE[tile_of(M, N)].bn;
  return GRPO_OK;
}
