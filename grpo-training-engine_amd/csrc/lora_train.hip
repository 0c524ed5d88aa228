// The NF4 + LoRA linear for training batches on gfx950, forward and backward.
// Restates _lora_forward_kernel (src/triton_kernels/lora_forward.py:107-260) and
// FusedLoRAFunction.backward (:761-930); every rounding point is the 16-bit type's
// (bf16 or float16), sums are float32:
//   xa = dt(x A^T)                    gi = dt(dt(g * dt(s)) B)
//   grad_A = dt(gi^T x)               grad_B = dt(dt(g * dt(s))^T xa)
//   grad_x = dt(dt(g W) + dt(gi A))   y = dt(dt(dt(x W^T) [+ bias]) + dt(dt(t B^T) * dt(s)))
//
// The weight is decoded once per call, not once per row tile: from about 5 million
// outputs (fewer where the decoding GEMM's ring kernel does not run) the two passes over
// N x K 16-bit values cost less than the decode repeated; the backward, which needs the
// weight transposed, always takes them.
// The products of rank r are bound by one read of x and g (M x K and M x N
// 16-bit values), so they are MFMA tiles fed straight from global memory in the
// row-major layout the caller has: no transposed or scaled copies are written.
//  * train_prep_kernel: what the products need, in one launch of independent
//    workgroups. x A^T and (g s) B (contraction over the row): a workgroup owns 16
//    rows, its 8 waves take 64-column steps round-robin and meet in LDS. The
//    weight in 16 bits, row-major or transposed. A transposed with its ranks
//    padded to 32.
//  * gemm16 (gemm16.hip): x W^T and g W with the LoRA term in the epilogue.
//  * lora_wgrad_kernel (contraction over rows m): a lane loads 8 rows x 8
//    columns and transposes pairs with v_perm, so eight MFMAs cover 128 columns x
//    32 rows per wave step; the row range is cut into slices that leave float32
//    partial sums, added in slice order by lora_sum_kernel.
// Measured at 8192 rows, N = K = 3584, r = 16 (bf16; x and g are 58.7 MB each):
// backward's preparation 32 us (x, g and the weight: 4.6 TB/s), weight gradients
// 24 us (4.9 TB/s) + sums 6, forward's preparation 21 us, the two GEMMs 183 and 180
// us. Forward and backward of q, k, v, o: 2199 us as torch products over the
// dequantized weight (scaled, transposed and added copies 595 us, rank-r GEMMs
// 490), 1382 with library GEMMs between these kernels and a pass over the result
// for the LoRA term (23-48 us each), 1222 with the term in the GEMM's epilogue.
#include <algorithm>

#include "gemm16.hpp"
#include "nf4_decode.hpp"

using namespace grpo;

namespace {

constexpr int LT_MAX_R = 32;

// ------------------------------------------------------------ dequantize --

struct DequantJob {
  const uint8_t* w;
  const float* absmax;
  const float* code16;
  uint16_t* out;  // [N][K], or [K][N] transposed
  int N, K, bs_shift;
  int blocks;     // workgroups
};

__device__ __forceinline__ void load_code(const float* code16, float (&code)[16]) {
#pragma unroll
  for (int j = 0; j < 16; ++j) code[j] = load_uniform(code16 + j);
}

// Row-major: a thread decodes 8 nibbles at a time, so a wave stores 1 KiB runs.
constexpr int DQ_PER = 8 * 512 * 4;  // values per workgroup

template <bool F16>
__device__ __forceinline__ void dequant_rows(const DequantJob& j, int b) {
  float code[16];
  load_code(j.code16, code);
  const int64_t total = (int64_t)j.N * j.K;  // a multiple of 32
  int64_t e[4];
  uint32_t wv[4];
  float a[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    e[i] = (int64_t)b * DQ_PER + 8 * (threadIdx.x + 512 * i);
    const int64_t ec = min(e[i], total - 8);
    wv[i] = *reinterpret_cast<const uint32_t*>(j.w + ec / 2);
    a[i] = j.absmax[ec >> j.bs_shift];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint4 v = interleave8(decode8(wv[i], make_lut<F16>(code, a[i])));
    if (e[i] < total) *reinterpret_cast<uint4*>(j.out + e[i]) = v;
  }
}

// Transposed, out[k][n] = dt(code[q(n, k)] * absmax): a workgroup decodes 128
// rows n x 128 columns k (a thread: one row, 32 nibbles of one absmax block) and
// turns the tile over in LDS.
constexpr int DT = 128, DT_LD = DT + 8;

template <bool F16>
__device__ __forceinline__ void dequant_tile_t(const DequantJob& j, int b, uint16_t* t) {
  const int kt = (j.K + DT - 1) / DT;
  const int tid = threadIdx.x, n0 = (b / kt) * DT, k0 = (b % kt) * DT;
  {
    const int nl = tid & (DT - 1), kl = 32 * (tid / DT);
    const int n = min(n0 + nl, j.N - 1), k = min(k0 + kl, j.K - 32);
    const int64_t e = (int64_t)n * j.K + k;
    const uint4 wv = *reinterpret_cast<const uint4*>(j.w + e / 2);
    const float a = j.absmax[e >> j.bs_shift];
    float code[16];
    load_code(j.code16, code);
    const Lut lut = make_lut<F16>(code, a);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint4 v = decode8(word(wv, q), lut);  // elements [0,2,4,6,1,3,5,7]
      const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int el = i < 4 ? 2 * i : 2 * (i - 4) + 1;
        t[(kl + 8 * q + el) * DT_LD + nl] = (uint16_t)(d[i >> 1] >> (16 * (i & 1)));
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < DT * DT / 8 / 512; ++i) {
    const int c = tid + 512 * i, kl = c / (DT / 8), nl = 8 * (c % (DT / 8));
    const int k = k0 + kl, n = n0 + nl;
    if (k < j.K && n < j.N)  // N % 8 == 0
      *reinterpret_cast<uint4*>(j.out + (int64_t)k * j.N + n) =
          *reinterpret_cast<const uint4*>(t + kl * DT_LD + nl);
  }
}

template <bool F16>
__global__ void __launch_bounds__(512) nf4_dequant_t_kernel(DequantJob j) {
  __shared__ __align__(16) uint16_t t[DT * DT_LD];
  dequant_tile_t<F16>(j, blockIdx.x, t);
}

// ------------------------------------------------------------ x A^T, g B --

struct RowsJob {
  const uint16_t* src;  // [M][C], row stride ld
  int64_t ld;
  const uint16_t* low;  // bt: B [C][r]; else A [r][C]
  int C;
  uint16_t* rows;       // [Mp][32] (ranks >= r zero) or null
  uint16_t* cols;       // [16 TC][Mp] (rows m >= M zero) or null
};

// One launch: workgroups [0, rows) run job 0, the next `rows` job 1 (a job
// without src: none), then dequant.blocks, then those that transpose A.
struct PrepArgs {
  RowsJob job[2];  // job 0: x A^T, job 1: dt(g s) B
  int M, Mp, r, rows;
  float scaling;
  DequantJob dequant;
  const uint16_t* la;  // A [r][K]
  uint16_t* at;        // [K][32] (ranks >= r zero)
  int K;
};

template <bool F16>
__device__ __forceinline__ uint4 scale8(uint4 v, float s) {
  const uint32_t d[4] = {v.x, v.y, v.z, v.w};
  uint32_t o[4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
    o[q] = pack_e2<F16>(e2f<F16>((uint16_t)d[q]) * s, e2f<F16>((uint16_t)(d[q] >> 16)) * s);
  return make_uint4(o[0], o[1], o[2], o[3]);
}

__device__ __forceinline__ uint4 keep(bool on, uint4 v) {
  return make_uint4(on ? v.x : 0u, on ? v.y : 0u, on ? v.z : 0u, on ? v.w : 0u);
}

// One job's product for rows m0 .. m0 + 15: wave w takes the 64-column steps w,
// w + 8, ...; lane (row ln, group lg) the columns c0 + 16 lg .. + 15.
template <int TC, bool F16, bool BT>
__device__ __forceinline__ void rows_product(const RowsJob& j, const PrepArgs& p, int m0, int wave,
                                             int ln, int lg, f32x4_t (&acc)[TC]) {
  const float sc = BT ? round_e<F16>(p.scaling) : 1.f;
  const uint16_t* const xr = j.src + (int64_t)min(m0 + ln, p.M - 1) * j.ld;
  int rk[TC];  // ranks >= r repeat rank r - 1; their results are not used
#pragma unroll
  for (int tc = 0; tc < TC; ++tc) rk[tc] = min(16 * tc + ln, p.r - 1);
  for (int c0 = 64 * wave; c0 < j.C; c0 += 512) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int c = c0 + 16 * lg + 8 * h;
      const bool on = c < j.C;  // C % 8 == 0
      const int cc = on ? c : 0;
      uint4 a = keep(on, *reinterpret_cast<const uint4*>(xr + cc));
      uint4 b[TC];
#pragma unroll
      for (int tc = 0; tc < TC; ++tc) {
        if (BT) {
          const uint16_t* q = j.low + (int64_t)cc * p.r + rk[tc];
          uint32_t v[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) v[i] = q[i * p.r];
          b[tc] = make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16),
                             v[6] | (v[7] << 16));
        } else {
          b[tc] = *reinterpret_cast<const uint4*>(j.low + (int64_t)rk[tc] * j.C + cc);
        }
        b[tc] = keep(on, b[tc]);
      }
      if (BT) a = scale8<F16>(a, sc);
#pragma unroll
      for (int tc = 0; tc < TC; ++tc) acc[tc] = mfma16x16x32_e<F16>(a, b[tc], acc[tc]);
    }
  }
}

template <int TC, bool F16>
__device__ __forceinline__ void rows_tile(const PrepArgs& p, int b, float* red) {
  constexpr int LD = 16 * TC + 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 15, lg = lane >> 4;
  const bool bt = b >= p.rows;
  const RowsJob j = bt ? p.job[1] : p.job[0];
  if (!j.src) return;
  const int m0 = 16 * (bt ? b - p.rows : b);
  f32x4_t acc[TC];
#pragma unroll
  for (int tc = 0; tc < TC; ++tc) acc[tc] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (bt)
    rows_product<TC, F16, true>(j, p, m0, wave, ln, lg, acc);
  else
    rows_product<TC, F16, false>(j, p, m0, wave, ln, lg, acc);
#pragma unroll
  for (int tc = 0; tc < TC; ++tc)
#pragma unroll
    for (int q = 0; q < 4; ++q) red[(16 * wave + 4 * lg + q) * LD + 16 * tc + ln] = acc[tc][q];
  __syncthreads();
  // one value per thread, the eight waves' sums in wave order; consecutive
  // threads: consecutive rows of one rank, so the transposed form leaves in runs
  const int row = tid & 15, rank = tid >> 4, m = m0 + row;
  uint16_t v = 0;
  if (rank < p.r && m < p.M) {
    float s = red[row * LD + rank];
#pragma unroll
    for (int w = 1; w < 8; ++w) s += red[(16 * w + row) * LD + rank];
    v = f2e<F16>(s);
  }
  if (j.rows) j.rows[(int64_t)m * 32 + rank] = v;  // m < Mp: Mp % 16 == 0
  if (j.cols && rank < 16 * TC) j.cols[(int64_t)rank * p.Mp + m] = v;
}

template <int TC, bool F16, bool TR>
__global__ void __launch_bounds__(512) train_prep_kernel(PrepArgs p) {
  __shared__ __align__(16) char lds[TR ? DT * DT_LD * 2 : 8 * 16 * (16 * TC + 1) * 4];
  static_assert(8 * 16 * (16 * TC + 1) * 4 <= DT * DT_LD * 2, "both uses fit");
  int b = blockIdx.x;
  if (b < 2 * p.rows) {
    rows_tile<TC, F16>(p, b, reinterpret_cast<float*>(lds));
    return;
  }
  b -= 2 * p.rows;
  if (b < p.dequant.blocks) {
    if (TR)
      dequant_tile_t<F16>(p.dequant, b, reinterpret_cast<uint16_t*>(lds));
    else
      dequant_rows<F16>(p.dequant, b);
    return;
  }
  // thread (column k, ranks 8 c .. 8 c + 7)
  const int i = (b - p.dequant.blocks) * 512 + threadIdx.x, k = i >> 2, c = 8 * (i & 3);
  if (k >= p.K) return;
  uint32_t v[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) v[q] = c + q < p.r ? p.la[(int64_t)(c + q) * p.K + k] : 0u;
  *reinterpret_cast<uint4*>(p.at + (int64_t)k * 32 + c) =
      make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16),
                 v[6] | (v[7] << 16));
}

// ------------------------------------------------- gradients of A and B --

constexpr int WG_C = 128;  // columns per workgroup

struct WgradArgs {
  const uint16_t* g;  // [M][N]: grad_B[n][r] = sum_m dt(g s)[m][n] xa[m][r]
  int64_t ldg;
  const uint16_t* x;  // [M][K]: grad_A[r][k] = sum_m gi[m][r] x[m][k]
  int64_t ldx;
  const uint16_t* xat;  // [16 TC][Mp]
  const uint16_t* git;  // [16 TC][Mp]
  int M, Mp, N, K, r, tn;  // tn: column tiles of g (0: no grad_B)
  float scaling;
  int steps;   // 32-row steps per slice
  float* pb;   // [S][N][r] partial sums, or null: dt results to gb and ga
  float* pa;   // [S][r][K]
  uint16_t* gb;
  uint16_t* ga;
};

template <int TC, bool F16>
__global__ void __launch_bounds__(256) lora_wgrad_kernel(WgradArgs p) {
  constexpr int LD = 16 * TC + 1;
  __shared__ float red[2][WG_C * LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 15, lg = lane >> 4;
  const bool isg = (int)blockIdx.x < p.tn;
  const int c0 = (isg ? blockIdx.x : blockIdx.x - p.tn) * WG_C;
  const int C = isg ? p.N : p.K;
  const int64_t ld = isg ? p.ldg : p.ldx;
  const uint16_t* const src = isg ? p.g : p.x;
  const uint16_t* const low = isg ? p.xat : p.git;
  const float sc = round_e<F16>(p.scaling);
  const int c = c0 + 8 * ln;
  const bool con = c < C;  // C % 8 == 0
  const uint16_t* const sc0 = src + (con ? c : 0);
  f32x4_t acc[8][TC];
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int tc = 0; tc < TC; ++tc) acc[j][tc] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int s1 = min((int)(blockIdx.y + 1) * p.steps, p.Mp / 32);
  for (int st = blockIdx.y * p.steps + wave; st < s1; st += 4) {
    const int m = 32 * st + 8 * lg;
    uint4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int mi = min(m + i, p.M - 1);
      v[i] = *reinterpret_cast<const uint4*>(sc0 + (int64_t)mi * ld);
    }
    uint4 b[TC];
#pragma unroll
    for (int tc = 0; tc < TC; ++tc)
      b[tc] = *reinterpret_cast<const uint4*>(low + (int64_t)(16 * tc + ln) * p.Mp + m);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[i] = keep(con && m + i < p.M, v[i]);  // no 0 * inf from rows past the end
      if (isg) v[i] = scale8<F16>(v[i], sc);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t sel = j & 1 ? 0x07060302u : 0x05040100u;
      const uint4 a = make_uint4(perm(word(v[1], j >> 1), word(v[0], j >> 1), sel),
                                 perm(word(v[3], j >> 1), word(v[2], j >> 1), sel),
                                 perm(word(v[5], j >> 1), word(v[4], j >> 1), sel),
                                 perm(word(v[7], j >> 1), word(v[6], j >> 1), sel));
#pragma unroll
      for (int tc = 0; tc < TC; ++tc) acc[j][tc] = mfma16x16x32_e<F16>(a, b[tc], acc[j][tc]);
    }
  }
  // tile j's row 4 lg + q is column 8 (4 lg + q) + j; waves added as (0 + 2) + (1 + 3)
  auto at = [&](int j, int tc, int q) __attribute__((always_inline)) {
    return (8 * (4 * lg + q) + j) * LD + 16 * tc + ln;
  };
  if (wave >= 2) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int tc = 0; tc < TC; ++tc)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[wave - 2][at(j, tc, q)] = acc[j][tc][q];
  }
  __syncthreads();
  if (wave < 2) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int tc = 0; tc < TC; ++tc)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[wave][at(j, tc, q)] += acc[j][tc][q];
  }
  __syncthreads();
  for (int i = tid; i < WG_C * p.r; i += 256) {
    // grad_B runs over ranks, grad_A over columns
    const int col = isg ? i / p.r : i & (WG_C - 1), rank = isg ? i - col * p.r : i / WG_C;
    if (c0 + col >= C) continue;
    const float s = red[0][col * LD + rank] + red[1][col * LD + rank];
    const int64_t o = isg ? (int64_t)(c0 + col) * p.r + rank : (int64_t)rank * C + c0 + col;
    if (p.pb)
      (isg ? p.pb : p.pa)[(int64_t)blockIdx.y * C * p.r + o] = s;
    else
      (isg ? p.gb : p.ga)[o] = f2e<F16>(s);
  }
}

struct SumArgs {
  const float* pb;  // [S][nb]
  const float* pa;  // [S][na]
  uint16_t* gb;
  uint16_t* ga;
  int64_t nb, na;  // values of each (multiples of 8)
  int S;
};

// Four values per thread, slices in order.
template <bool F16>
__global__ void __launch_bounds__(256) lora_sum_kernel(SumArgs p) {
  int64_t e = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
  const bool isb = e < p.nb;
  if (!isb) e -= p.nb;
  const int64_t n = isb ? p.nb : p.na;
  if (e >= n) return;
  const float* src = (isb ? p.pb : p.pa) + e;
  float4 s = *reinterpret_cast<const float4*>(src);
  for (int k = 1; k < p.S; ++k) {
    const float4 v = *reinterpret_cast<const float4*>(src + k * n);
    s.x += v.x;
    s.y += v.y;
    s.z += v.z;
    s.w += v.w;
  }
  *reinterpret_cast<uint2*>((isb ? p.gb : p.ga) + e) =
      make_uint2(pack_e2<F16>(s.x, s.y), pack_e2<F16>(s.z, s.w));
}

// ----------------------------------------------------------------- host --

int64_t pad32(int64_t m) { return (m + 31) / 32 * 32; }

// Row slices of the weight gradients: enough workgroups for two per CU, each
// slice at least one 32-row step per wave.
int wgrad_slices(int M, int N, int K) {
  const int64_t tiles = cdiv(N, WG_C) + cdiv(K, WG_C), steps = pad32(M) / 32;
  int64_t s = std::min<int64_t>(std::max<int64_t>(1, 640 / tiles), std::max<int64_t>(1, steps / 4));
  s = std::min<int64_t>(s, 32);
  return (int)cdiv(steps, cdiv(steps, s));
}

// Workspace of either direction (byte offsets): the 16-bit weight, t or gi by
// rows, x A^T and gi by columns, A by columns, the partial sums.
struct TrainWs {
  size_t w, rows, xat, git, at, pb, pa, total;
};

TrainWs train_ws(int M, int N, int K, int r) {
  const size_t Mp = (size_t)pad32(M), R = r > 16 ? 32 : 16;
  const int S = wgrad_slices(M, N, K);
  TrainWs w{};
  size_t o = 0;
  auto take = [&](size_t n) {
    const size_t at = o;
    o += (n + 255) / 256 * 256;
    return at;
  };
  w.w = take((size_t)N * K * 2);
  w.rows = take(Mp * 32 * 2);
  w.xat = take(R * Mp * 2);
  w.git = take(R * Mp * 2);
  w.at = take((size_t)K * 32 * 2);
  w.pb = take(S > 1 ? (size_t)S * N * r * 4 : 0);
  w.pa = take(S > 1 ? (size_t)S * K * r * 4 : 0);
  w.total = o;
  return w;
}

template <bool F16, bool TR>
int launch_prep(const PrepArgs& a, hipStream_t st) {
  const unsigned grid = 2u * a.rows + a.dequant.blocks + (a.at ? (unsigned)cdiv(a.K, 128) : 0u);
  if (a.r > 16) train_prep_kernel<2, F16, TR><<<grid, 512, 0, st>>>(a);
  else train_prep_kernel<1, F16, TR><<<grid, 512, 0, st>>>(a);
  return launch_check("train_prep");
}

bool train_ok(int M, int N, int K, int r, int blocksize) {
  return M >= 1 && r >= 1 && r <= LT_MAX_R && blocksize >= 32 &&
         (blocksize & (blocksize - 1)) == 0 && N % 32 == 0 && K % 32 == 0 &&
         gemm16_ok(M, N, K, K, K) && gemm16_ok(M, K, N, N, N);
}

struct TrainCall {
  const uint16_t* x;
  int64_t ldx;
  const uint8_t* w;
  const float* absmax;
  const float* code16;
  int bs_shift;
  const uint16_t* la;
  const uint16_t* lb;
  int r;
  float scaling;
  int M, N, K;
  char* ws;
  hipStream_t st;
};

template <bool F16>
int run_forward(const TrainCall& c, const uint16_t* bias, uint16_t* y, int64_t ldy) {
  const TrainWs o = train_ws(c.M, c.N, c.K, c.r);
  uint16_t* const wd = reinterpret_cast<uint16_t*>(c.ws + o.w);
  uint16_t* const rows = reinterpret_cast<uint16_t*>(c.ws + o.rows);
  PrepArgs a{};
  a.M = c.M;
  a.Mp = (int)pad32(c.M);
  a.r = c.r;
  a.job[0] = RowsJob{c.x, c.ldx, c.la, c.K, rows, nullptr};
  a.rows = a.Mp / 16;
  a.dequant = DequantJob{c.w, c.absmax, c.code16, wd, c.N, c.K, c.bs_shift,
                         (int)cdiv((int64_t)c.N * c.K, DQ_PER)};
  if (int rc = launch_prep<F16, false>(a, c.st)) return rc;
  Gemm16 g{};
  g.a = c.x;
  g.lda = c.ldx;
  g.b = wd;
  g.ldb = c.K;
  g.c = y;
  g.ldc = ldy;
  g.M = c.M;
  g.N = c.N;
  g.K = c.K;
  g.t = rows;
  g.low = c.lb;
  g.ldl = c.r;
  g.bias = bias;
  g.r = c.r;
  g.scaling = c.scaling;
  return gemm16_launch(g, GEMM16_LORA, F16, c.st);
}

template <bool F16>
int run_backward(const TrainCall& c, const uint16_t* grad, int64_t ldg, uint16_t* grad_x,
                 int64_t ldgx, uint16_t* grad_a, uint16_t* grad_b) {
  const TrainWs o = train_ws(c.M, c.N, c.K, c.r);
  const int Mp = (int)pad32(c.M), S = wgrad_slices(c.M, c.N, c.K);
  uint16_t* const wt = reinterpret_cast<uint16_t*>(c.ws + o.w);
  uint16_t* const rows = reinterpret_cast<uint16_t*>(c.ws + o.rows);
  uint16_t* const xat = reinterpret_cast<uint16_t*>(c.ws + o.xat);
  uint16_t* const git = reinterpret_cast<uint16_t*>(c.ws + o.git);
  uint16_t* const at = reinterpret_cast<uint16_t*>(c.ws + o.at);
  PrepArgs a{};
  a.M = c.M;
  a.Mp = Mp;
  a.r = c.r;
  a.scaling = c.scaling;
  a.rows = Mp / 16;
  a.K = c.K;
  if (grad_b) a.job[0] = RowsJob{c.x, c.ldx, c.la, c.K, nullptr, xat};
  if (grad_x || grad_a)
    a.job[1] = RowsJob{grad, ldg, c.lb, c.N, grad_x ? rows : nullptr, grad_a ? git : nullptr};
  if (grad_x) {
    a.dequant = DequantJob{c.w, c.absmax, c.code16, wt, c.N, c.K, c.bs_shift,
                           (int)(cdiv(c.N, DT) * cdiv(c.K, DT))};
    a.la = c.la;
    a.at = at;
  }
  if (int rc = launch_prep<F16, true>(a, c.st)) return rc;
  if (grad_x) {
    Gemm16 g{};
    g.a = grad;
    g.lda = ldg;
    g.b = wt;
    g.ldb = c.N;
    g.c = grad_x;
    g.ldc = ldgx;
    g.M = c.M;
    g.N = c.K;
    g.K = c.N;
    g.t = rows;
    g.low = at;
    g.ldl = 32;
    g.r = c.r;
    if (int rc = gemm16_launch(g, GEMM16_ADD, F16, c.st)) return rc;
  }
  if (!grad_a && !grad_b) return GRPO_OK;
  WgradArgs w{};
  w.g = grad;
  w.ldg = ldg;
  w.x = c.x;
  w.ldx = c.ldx;
  w.xat = xat;
  w.git = git;
  w.M = c.M;
  w.Mp = Mp;
  w.N = c.N;
  w.K = c.K;
  w.r = c.r;
  w.tn = grad_b ? (int)cdiv(c.N, WG_C) : 0;
  w.scaling = c.scaling;
  w.steps = (int)cdiv(Mp / 32, S);
  w.gb = grad_b;
  w.ga = grad_a;
  if (S > 1) {
    w.pb = reinterpret_cast<float*>(c.ws + o.pb);
    w.pa = reinterpret_cast<float*>(c.ws + o.pa);
  }
  const dim3 grid((unsigned)(w.tn + (grad_a ? cdiv(c.K, WG_C) : 0)), (unsigned)S);
  if (c.r > 16) lora_wgrad_kernel<2, F16><<<grid, 256, 0, c.st>>>(w);
  else lora_wgrad_kernel<1, F16><<<grid, 256, 0, c.st>>>(w);
  if (int rc = launch_check("lora_wgrad")) return rc;
  if (S == 1) return GRPO_OK;
  const SumArgs sa{w.pb, w.pa, grad_b, grad_a, grad_b ? (int64_t)c.N * c.r : 0,
                   grad_a ? (int64_t)c.K * c.r : 0, S};
  lora_sum_kernel<F16><<<(unsigned)cdiv(sa.nb + sa.na, 1024), 256, 0, c.st>>>(sa);
  return launch_check("lora_sum");
}

// The checks both directions share.
int train_check(const void* x, int64_t ldx, const uint8_t* w, const float* absmax,
                const float* code16, int blocksize, const void* lora_a, const void* lora_b, int r,
                int M, int N, int K, void* workspace, size_t workspace_bytes) {
  if (!train_ok(M, N, K, r, blocksize)) {
    set_error("shape not supported by the NF4 + LoRA training kernels (N %% 32 == 0, K %% 32 == "
              "0, 1 <= r <= 32, power-of-two blocksize >= 32)");
    return GRPO_EUNSUPPORTED;
  }
  if (!x || !w || !absmax || !code16 || !lora_a || !lora_b || !workspace)
    return einval("null pointer");
  if (ldx < K || ldx % 8 || ldx >= (1 << 22) || !aligned16(x))
    return einval("x rows must be 16-byte aligned");
  if (!aligned16(w) || !aligned16(lora_a) || !aligned16(workspace))
    return einval("w, lora_a and the workspace must be 16-byte aligned");
  if (workspace_bytes < train_ws(M, N, K, r).total) {
    set_error("workspace too small");
    return GRPO_EWORKSPACE;
  }
  return GRPO_OK;
}

TrainCall train_call(const void* x, int64_t ldx, const uint8_t* w, const float* absmax,
                     const float* code16, int blocksize, const void* lora_a, const void* lora_b,
                     int r, float scaling, int M, int N, int K, void* workspace,
                     grpo_stream_t stream) {
  return TrainCall{static_cast<const uint16_t*>(x), ldx, w, absmax, code16,
                   __builtin_ctz((unsigned)blocksize), static_cast<const uint16_t*>(lora_a),
                   static_cast<const uint16_t*>(lora_b), r, scaling, M, N, K,
                   static_cast<char*>(workspace), as_stream(stream)};
}

}  // namespace

extern "C" int grpo_nf4_dequant_t(const uint8_t* w, const float* absmax, const float* code16,
                                  void* out, int N, int K, int blocksize, int f16,
                                  grpo_stream_t stream) {
  if (N < 0 || K < 0) return einval("negative dimension");
  if (N == 0 || K == 0) return GRPO_OK;
  if (!w || !absmax || !code16 || !out) return einval("null pointer");
  if (blocksize < 32 || (blocksize & (blocksize - 1)) || K % 32 || N % 8) {
    set_error("transposed dequantization needs a power-of-two blocksize >= 32, K %% 32 == 0 and "
              "N %% 8 == 0");
    return GRPO_EUNSUPPORTED;
  }
  if (!aligned16(w) || !aligned16(out)) return einval("w and out must be 16-byte aligned");
  const DequantJob j{w, absmax, code16, static_cast<uint16_t*>(out), N, K,
                     __builtin_ctz((unsigned)blocksize), (int)(cdiv(N, DT) * cdiv(K, DT))};
  if (f16) nf4_dequant_t_kernel<true><<<j.blocks, 512, 0, as_stream(stream)>>>(j);
  else nf4_dequant_t_kernel<false><<<j.blocks, 512, 0, as_stream(stream)>>>(j);
  return launch_check("nf4_dequant_t");
}

extern "C" size_t grpo_nf4_lora_train_workspace_bytes(int M, int N, int K, int r, int blocksize) {
  return train_ok(M, N, K, r, blocksize) ? train_ws(M, N, K, r).total : 0;
}

extern "C" int grpo_nf4_lora_train_forward(const void* x, int64_t ldx, const uint8_t* w,
                                           const float* absmax, const float* code16,
                                           int blocksize, const void* bias, const void* lora_a,
                                           const void* lora_b, int r, float scaling, void* y,
                                           int64_t ldy, int M, int N, int K, int f16,
                                           void* workspace, size_t workspace_bytes,
                                           grpo_stream_t stream) {
  if (int rc = train_check(x, ldx, w, absmax, code16, blocksize, lora_a, lora_b, r, M, N, K,
                           workspace, workspace_bytes))
    return rc;
  if (!y) return einval("null pointer");
  if (ldy < N || ldy % 8 || !aligned16(y)) return einval("y rows must be 16-byte aligned");
  const TrainCall c = train_call(x, ldx, w, absmax, code16, blocksize, lora_a, lora_b, r, scaling,
                                 M, N, K, workspace, stream);
  const uint16_t* const b = static_cast<const uint16_t*>(bias);
  uint16_t* const o = static_cast<uint16_t*>(y);
  return f16 ? run_forward<true>(c, b, o, ldy) : run_forward<false>(c, b, o, ldy);
}

extern "C" int grpo_nf4_lora_train_backward(const void* x, int64_t ldx, const void* grad,
                                            int64_t ldg, const uint8_t* w, const float* absmax,
                                            const float* code16, int blocksize,
                                            const void* lora_a, const void* lora_b, int r,
                                            float scaling, int M, int N, int K, int f16,
                                            void* grad_x, int64_t ldgx, void* grad_a,
                                            void* grad_b, void* workspace,
                                            size_t workspace_bytes, grpo_stream_t stream) {
  if (int rc = train_check(x, ldx, w, absmax, code16, blocksize, lora_a, lora_b, r, M, N, K,
                           workspace, workspace_bytes))
    return rc;
  if (!grad_x && !grad_a && !grad_b) return GRPO_OK;
  if (!grad) return einval("null pointer");
  if (ldg < N || ldg % 8 || ldg >= (1 << 22) || !aligned16(grad))
    return einval("grad rows must be 16-byte aligned");
  if (grad_x && (ldgx < K || ldgx % 8 || !aligned16(grad_x)))
    return einval("grad_x rows must be 16-byte aligned");
  if (!aligned16(grad_a) || !aligned16(grad_b))
    return einval("the adapters' gradients must be 16-byte aligned");
  const TrainCall c = train_call(x, ldx, w, absmax, code16, blocksize, lora_a, lora_b, r, scaling,
                                 M, N, K, workspace, stream);
  const uint16_t* const g = static_cast<const uint16_t*>(grad);
  auto u = [](void* q) { return static_cast<uint16_t*>(q); };
  return f16 ? run_backward<true>(c, g, ldg, u(grad_x), ldgx, u(grad_a), u(grad_b))
             : run_backward<false>(c, g, ldg, u(grad_x), ldgx, u(grad_a), u(grad_b));
}
