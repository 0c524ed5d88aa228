// The rank-r side of the NF4 + LoRA linear in training for gfx950: the
// products x A^T and (g s) B, the adapters' gradients, and the LoRA term's
// addition to a product of the base weight.  Restates the LoRA parts of
// _lora_forward_kernel (src/triton_kernels/lora_forward.py:210-257) and of
// FusedLoRAFunction.backward (:761-930); every rounding point is the 16-bit
// type's (bf16 or float16), sums are float32:
//   xa = dt(x A^T)                    gi = dt(dt(g * dt(s)) B)
//   grad_A = dt(gi^T x)               grad_B = dt(dt(g * dt(s))^T xa)
//   grad_x = dt(dt(g W) + dt(gi A))   y = dt(dt(x W^T [+ bias]) + dt(dt(t B^T) * dt(s)))
//
// All of them are bound by one read of x and g (M x K and M x N 16-bit values);
// the r <= 32 columns on the other side make the arithmetic small, so every
// product is MFMA tiles fed straight from global memory in the row-major
// layout the caller has: no transposed or scaled copies are written.
//  * lora_rows_kernel (contraction over the row, x A^T and (g s) B): a
//    workgroup owns 16 or 32 rows, its 8 waves take 64-column steps round-robin
//    and meet in LDS.
//  * lora_wgrad_kernel (contraction over rows m): a lane loads 8 rows x 8
//    columns and transposes pairs with v_perm, so eight MFMAs cover 128 columns x
//    32 rows per wave step; the row range is cut into slices that leave float32
//    partial sums, added in slice order by lora_sum_kernel (or by the add kernel's
//    extra workgroups).
//  * lora_add_kernel: the M x N product is read and rewritten once, the rank-r
//    product on MFMAs with the wide operand in the A position, so a lane holds 16
//    consecutive columns of one row (two 16-byte accesses).
// Measured at 8192 rows, N = K = 3584, r = 16 (bf16; x and g are 58.7 MB each):
// rows 25.8 us and weight gradients 24.0 us (4.5 and 4.9 TB/s of x and g), add 33
// us (3.6 TB/s), against about 300 us for the same results as torch products,
// which wrote scaled, transposed and added copies of g and x (327 us of strided
// copies, 268 us of adds and 490 us of rank-r GEMMs over the four projections of
// a layer: 2199 us forward and backward, 1382 with these kernels).
#include <algorithm>

#include "common.hpp"
#include "nf4_decode.hpp"

using namespace grpo;

namespace {

constexpr int LT_MAX_R = 32;

// ------------------------------------------------- dequantize, transposed --

// WT[k][n] = dt(code[q(n, k)] * absmax): the [K, N] form of nf4_dequant_vec's
// output (bound by its 2-byte writes: 10.2 us at 3584 x 3584, 2.5 TB/s written;
// nf4_dequant_vec takes 10.8).  The transposed weight makes grad_x = g W a product
// of two K-contiguous operands, which the GEMM library runs in 144 us at 8192 rows
// where the row-major weight takes 168.  A workgroup decodes 64 rows n x 128 columns k (a thread: one row, 32
// nibbles of one absmax block) and turns the tile over in LDS.
constexpr int DT_N = 64, DT_K = 128, DT_LD = DT_N + 8;

template <bool F16>
__global__ void __launch_bounds__(256) nf4_dequant_t_kernel(const uint8_t* __restrict__ w,
                                                            const float* __restrict__ absmax,
                                                            const float* __restrict__ code16,
                                                            uint16_t* __restrict__ out, int N,
                                                            int K, int bs_shift) {
  __shared__ __align__(16) uint16_t t[DT_K * DT_LD];
  const int tid = threadIdx.x;
  const int n0 = blockIdx.y * DT_N, k0 = blockIdx.x * DT_K;
  {
    const int nl = tid & 63, kl = 32 * (tid >> 6);
    const int n = min(n0 + nl, N - 1), k = min(k0 + kl, K - 32);
    const int64_t e = (int64_t)n * K + k;
    const uint4 wv = *reinterpret_cast<const uint4*>(w + e / 2);
    const float a = absmax[e >> bs_shift];
    float code[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) code[j] = code16[j];
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
  for (int i = 0; i < DT_K * DT_N / 8 / 256; ++i) {
    const int c = tid + 256 * i, kl = c >> 3, nl = 8 * (c & 7);
    const int k = k0 + kl, n = n0 + nl;
    if (k < K && n < N)  // N % 8 == 0
      *reinterpret_cast<uint4*>(out + (int64_t)k * N + n) =
          *reinterpret_cast<const uint4*>(t + kl * DT_LD + nl);
  }
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

struct RowsArgs {
  RowsJob job[2];  // job 0: x A^T, job 1: dt(g s) B
  int M, Mp, r;
  float scaling;
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

// One job's product over the columns c0 + 16 lg .. + 15 of this lane's rows.
template <int TC, bool F16, int RT, bool BT>
__device__ __forceinline__ void rows_product(const RowsJob& j, const RowsArgs& p, int m0, int wave,
                                             int ln, int lg, f32x4_t (&acc)[RT][TC]) {
  const float sc = BT ? round_e<F16>(p.scaling) : 1.f;
  const uint16_t* xr[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) xr[t] = j.src + (int64_t)min(m0 + 16 * t + ln, p.M - 1) * j.ld;
  int rk[TC];  // ranks >= r repeat rank r - 1; their results are not used
#pragma unroll
  for (int tc = 0; tc < TC; ++tc) rk[tc] = min(16 * tc + ln, p.r - 1);
  for (int c0 = 64 * wave; c0 < j.C; c0 += 512) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int c = c0 + 16 * lg + 8 * h;
      const bool on = c < j.C;  // C % 8 == 0
      const int cc = on ? c : 0;
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
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        uint4 a = keep(on, *reinterpret_cast<const uint4*>(xr[t] + cc));
        if (BT) a = scale8<F16>(a, sc);
#pragma unroll
        for (int tc = 0; tc < TC; ++tc) acc[t][tc] = mfma16x16x32_e<F16>(a, b[tc], acc[t][tc]);
      }
    }
  }
}

template <int TC, bool F16, int RT>
__global__ void __launch_bounds__(512) lora_rows_kernel(RowsArgs p) {
  constexpr int LD = 16 * TC + 1;
  __shared__ float red[8][16 * RT][LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 15, lg = lane >> 4;
  const int m0 = blockIdx.x * 16 * RT;
  const bool bt = blockIdx.y != 0;
  const RowsJob j = bt ? p.job[1] : p.job[0];
  if (!j.src) return;
  f32x4_t acc[RT][TC];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int tc = 0; tc < TC; ++tc) acc[t][tc] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (bt)
    rows_product<TC, F16, RT, true>(j, p, m0, wave, ln, lg, acc);
  else
    rows_product<TC, F16, RT, false>(j, p, m0, wave, ln, lg, acc);
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int tc = 0; tc < TC; ++tc)
#pragma unroll
      for (int q = 0; q < 4; ++q) red[wave][16 * t + 4 * lg + q][16 * tc + ln] = acc[t][tc][q];
  __syncthreads();
  // the eight waves' sums in wave order; consecutive threads: consecutive rows
  // of one rank, so the transposed form leaves in runs
  for (int i = tid; i < 16 * RT * 32; i += 512) {
    const int row = i & (16 * RT - 1), rank = i / (16 * RT), m = m0 + row;
    uint16_t v = 0;
    if (rank < p.r && m < p.M) {
      float s = red[0][row][rank];
#pragma unroll
      for (int w = 1; w < 8; ++w) s += red[w][row][rank];
      v = f2e<F16>(s);
    }
    if (m < p.Mp) {
      if (j.rows) j.rows[(int64_t)m * 32 + rank] = v;
      if (j.cols && rank < 16 * TC) j.cols[(int64_t)rank * p.Mp + m] = v;
    }
  }
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
__device__ __forceinline__ void sum_slices(const SumArgs& p, int64_t i) {
  int64_t e = 4 * i;
  const bool isb = e < p.nb;
  if (!isb) e -= p.nb;
  const int64_t n = isb ? p.nb : p.na;
  if (e >= n) return;
  const float* src = (isb ? p.pb : p.pa) + e;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int k = 0; k < p.S; ++k) {
    const float4 v = *reinterpret_cast<const float4*>(src + k * n);
    s.x += v.x;
    s.y += v.y;
    s.z += v.z;
    s.w += v.w;
  }
  *reinterpret_cast<uint2*>((isb ? p.gb : p.ga) + e) =
      make_uint2(pack_e2<F16>(s.x, s.y), pack_e2<F16>(s.z, s.w));
}

// ------------------------------------------------- adding the LoRA term --

struct AddArgs {
  const uint16_t* t;    // [M][32] rows of t or gi, ranks >= r zero
  const uint16_t* low;  // FWD: B [C][r]; else A [r][C]
  const uint16_t* bias; // FWD: [C] or null
  const uint16_t* src;  // [M][C] the base product
  uint16_t* out;        // [M][C] (may be src)
  int64_t lds, ldo;
  int M, C, r;
  float scaling;
  int rows;             // rows per workgroup (a multiple of 16)
  int tiles_c, blocks;  // workgroups of the add; the rest run sum_slices
};

template <bool FWD, bool F16>
__device__ __forceinline__ void add_tile(const AddArgs& p, int bx) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ln = lane & 15, lg = lane >> 4;
  const int c0 = (bx % p.tiles_c) * 256 + 64 * wave, m0 = (bx / p.tiles_c) * p.rows;
  // MFMA row i of tile j is column c0 + 16 (i / 4) + 4 j + i % 4: a lane ends
  // with columns c0 + 16 lg .. + 15 of row m0 + ln
  uint4 a[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int col = min(c0 + 16 * (ln >> 2) + 4 * j + (ln & 3), p.C - 1);
    uint32_t v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int rank = 8 * lg + i, rr = min(rank, p.r - 1);
      const uint16_t e = FWD ? p.low[(int64_t)col * p.r + rr] : p.low[(int64_t)rr * p.C + col];
      v[i] = rank < p.r ? e : 0u;
    }
    a[j] = make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16),
                      v[6] | (v[7] << 16));
  }
  const int c = c0 + 16 * lg;
  const bool on[2] = {c < p.C, c + 8 < p.C};  // C % 8 == 0
  float bias[16];
  if (FWD && p.bias) {
#pragma unroll
    for (int i = 0; i < 16; ++i) bias[i] = e2f<F16>(p.bias[min(c + i, p.C - 1)]);
  }
  const float sc = FWD ? round_e<F16>(p.scaling) : 1.f;
  const int m1 = min(m0 + p.rows, p.M);
  for (int mb = m0; mb < m1; mb += 16) {
    const int m = mb + ln, mc = min(m, p.M - 1);
    const uint16_t* s = p.src + (int64_t)mc * p.lds + c;
    uint4 sv[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
      sv[h] = on[h] ? *reinterpret_cast<const uint4*>(s + 8 * h) : make_uint4(0, 0, 0, 0);
    const uint4 tv = *reinterpret_cast<const uint4*>(p.t + (int64_t)mc * 32 + 8 * lg);
    uint32_t o[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4_t u = mfma16x16x32_e<F16>(a[j], tv, f32x4_t{0.f, 0.f, 0.f, 0.f});
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int e = 4 * j + q;
        v[q] = e2f<F16>((uint16_t)(word(sv[e >> 3], (e >> 1) & 3) >> (16 * (e & 1))));
        float uq = round_e<F16>(u[q]);
        if (FWD) {
          if (p.bias) v[q] = round_e<F16>(v[q] + bias[e]);
          uq = round_e<F16>(uq * sc);
        }
        v[q] += uq;
      }
      o[2 * j] = pack_e2<F16>(v[0], v[1]);
      o[2 * j + 1] = pack_e2<F16>(v[2], v[3]);
    }
    if (m < p.M) {
      uint16_t* d = p.out + (int64_t)m * p.ldo + c;
      if (on[0]) *reinterpret_cast<uint4*>(d) = make_uint4(o[0], o[1], o[2], o[3]);
      if (on[1]) *reinterpret_cast<uint4*>(d + 8) = make_uint4(o[4], o[5], o[6], o[7]);
    }
  }
}

template <bool FWD, bool F16>
__global__ void __launch_bounds__(256) lora_add_kernel(AddArgs p, SumArgs s) {
  if ((int)blockIdx.x < p.blocks)
    add_tile<FWD, F16>(p, blockIdx.x);
  else
    sum_slices<F16>(s, (int64_t)(blockIdx.x - p.blocks) * 256 + threadIdx.x);
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

struct TrainWs {  // byte offsets into the workspace
  size_t rows, xat, git, pb, pa, total;
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
  w.rows = take(Mp * 32 * 2);
  w.xat = take(R * Mp * 2);
  w.git = take(R * Mp * 2);
  w.pb = take(S > 1 ? (size_t)S * N * r * 4 : 0);
  w.pa = take(S > 1 ? (size_t)S * K * r * 4 : 0);
  w.total = o;
  return w;
}

template <bool F16>
int launch_rows(const RowsArgs& a, int jobs, hipStream_t st) {
  // 32 rows per workgroup once 16-row workgroups would pass four per CU
  const bool wide = cdiv(a.Mp, 16) * jobs > 1024;
  const dim3 grid((unsigned)cdiv(a.Mp, wide ? 32 : 16), (unsigned)jobs);
  if (a.r > 16) {
    if (wide) lora_rows_kernel<2, F16, 2><<<grid, 512, 0, st>>>(a);
    else lora_rows_kernel<2, F16, 1><<<grid, 512, 0, st>>>(a);
  } else {
    if (wide) lora_rows_kernel<1, F16, 2><<<grid, 512, 0, st>>>(a);
    else lora_rows_kernel<1, F16, 1><<<grid, 512, 0, st>>>(a);
  }
  return launch_check("lora_rows");
}

AddArgs add_args(const uint16_t* t, const void* low, const void* bias, const void* src,
                 int64_t lds, void* out, int64_t ldo, int M, int C, int r, float scaling) {
  AddArgs a{};
  a.t = t;
  a.low = static_cast<const uint16_t*>(low);
  a.bias = static_cast<const uint16_t*>(bias);
  a.src = static_cast<const uint16_t*>(src);
  a.out = static_cast<uint16_t*>(out);
  a.lds = lds;
  a.ldo = ldo;
  a.M = M;
  a.C = C;
  a.r = r;
  a.scaling = scaling;
  a.tiles_c = (int)cdiv(C, 256);
  // 64 rows per workgroup while that leaves fewer than 2048 of them
  a.rows = cdiv(M, 64) * a.tiles_c > 2048 ? 128 : 64;
  if (cdiv(M, 64) * a.tiles_c < 512) a.rows = 16;
  a.blocks = a.tiles_c * (int)cdiv(M, a.rows);
  return a;
}

bool train_ok(int M, int N, int K, int r) {
  return M >= 0 && N >= 8 && K >= 8 && N % 8 == 0 && K % 8 == 0 && r >= 1 && r <= LT_MAX_R;
}

int train_unsupported() {
  set_error("shape not supported by the LoRA training kernels (N %% 8 == 0, K %% 8 == 0, "
            "1 <= r <= 32)");
  return GRPO_EUNSUPPORTED;
}

template <bool F16>
int run_backward(const uint16_t* x, int64_t ldx, const uint16_t* g, int64_t ldg,
                 const uint16_t* la, const uint16_t* lb, int r, float scaling, int M, int N, int K,
                 uint16_t* grad_x, int64_t ldgx, uint16_t* grad_a, uint16_t* grad_b, char* ws,
                 hipStream_t st) {
  const TrainWs o = train_ws(M, N, K, r);
  const int Mp = (int)pad32(M), S = wgrad_slices(M, N, K);
  uint16_t* const rows = reinterpret_cast<uint16_t*>(ws + o.rows);
  uint16_t* const xat = reinterpret_cast<uint16_t*>(ws + o.xat);
  uint16_t* const git = reinterpret_cast<uint16_t*>(ws + o.git);
  RowsArgs ra{};
  ra.M = M;
  ra.Mp = Mp;
  ra.r = r;
  ra.scaling = scaling;
  if (grad_b) ra.job[0] = RowsJob{x, ldx, la, K, nullptr, xat};
  if (grad_x || grad_a)
    ra.job[1] = RowsJob{g, ldg, lb, N, grad_x ? rows : nullptr, grad_a ? git : nullptr};
  if (int rc = launch_rows<F16>(ra, 2, st)) return rc;
  SumArgs sa{};
  if (grad_a || grad_b) {
    WgradArgs w{};
    w.g = g;
    w.ldg = ldg;
    w.x = x;
    w.ldx = ldx;
    w.xat = xat;
    w.git = git;
    w.M = M;
    w.Mp = Mp;
    w.N = N;
    w.K = K;
    w.r = r;
    w.tn = grad_b ? (int)cdiv(N, WG_C) : 0;
    w.scaling = scaling;
    w.steps = (int)cdiv(Mp / 32, S);
    w.gb = grad_b;
    w.ga = grad_a;
    if (S > 1) {
      w.pb = reinterpret_cast<float*>(ws + o.pb);
      w.pa = reinterpret_cast<float*>(ws + o.pa);
      sa = SumArgs{w.pb, w.pa, grad_b, grad_a, grad_b ? (int64_t)N * r : 0,
                   grad_a ? (int64_t)K * r : 0, S};
    }
    const dim3 grid((unsigned)(w.tn + (grad_a ? cdiv(K, WG_C) : 0)), (unsigned)S);
    if (r > 16) lora_wgrad_kernel<2, F16><<<grid, 256, 0, st>>>(w);
    else lora_wgrad_kernel<1, F16><<<grid, 256, 0, st>>>(w);
    if (int rc = launch_check("lora_wgrad")) return rc;
  }
  const unsigned sum_blocks = (unsigned)cdiv(cdiv(sa.nb + sa.na, 4), 256);
  AddArgs a{};
  if (grad_x) a = add_args(rows, la, nullptr, grad_x, ldgx, grad_x, ldgx, M, K, r, 1.f);
  if (a.blocks + sum_blocks == 0) return GRPO_OK;
  lora_add_kernel<false, F16><<<a.blocks + sum_blocks, 256, 0, st>>>(a, sa);
  return launch_check("lora_add");
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
  const dim3 grid((unsigned)cdiv(K, DT_K), (unsigned)cdiv(N, DT_N));
  const int shift = __builtin_ctz((unsigned)blocksize);
  hipStream_t st = as_stream(stream);
  if (f16)
    nf4_dequant_t_kernel<true><<<grid, 256, 0, st>>>(w, absmax, code16,
                                                     static_cast<uint16_t*>(out), N, K, shift);
  else
    nf4_dequant_t_kernel<false><<<grid, 256, 0, st>>>(w, absmax, code16,
                                                      static_cast<uint16_t*>(out), N, K, shift);
  return launch_check("nf4_dequant_t");
}

extern "C" size_t grpo_lora_train_workspace_bytes(int M, int N, int K, int r) {
  return M > 0 && train_ok(M, N, K, r) ? train_ws(M, N, K, r).total : 0;
}

extern "C" int grpo_lora_forward_add(const void* x, int64_t ldx, const void* lora_a,
                                     const void* lora_b, const void* bias, int r, float scaling,
                                     void* y, int64_t ldy, int M, int N, int K, int f16,
                                     void* workspace, size_t workspace_bytes,
                                     grpo_stream_t stream) {
  if (!train_ok(M, N, K, r)) return train_unsupported();
  if (M == 0) return GRPO_OK;
  if (!x || !lora_a || !lora_b || !y || !workspace) return einval("null pointer");
  if (ldx < K || ldx % 8 || !aligned16(x)) return einval("x rows must be 16-byte aligned");
  if (ldy < N || ldy % 8 || !aligned16(y)) return einval("y rows must be 16-byte aligned");
  if (!aligned16(lora_a) || !aligned16(workspace))
    return einval("lora_a and workspace must be 16-byte aligned");
  const int Mp = (int)pad32(M);
  if (workspace_bytes < (size_t)Mp * 64) {
    set_error("workspace too small");
    return GRPO_EWORKSPACE;
  }
  uint16_t* const rows = static_cast<uint16_t*>(workspace);
  RowsArgs ra{};
  ra.M = M;
  ra.Mp = Mp;
  ra.r = r;
  ra.job[0] = RowsJob{static_cast<const uint16_t*>(x), ldx, static_cast<const uint16_t*>(lora_a),
                      K, rows, nullptr};
  hipStream_t st = as_stream(stream);
  if (int rc = f16 ? launch_rows<true>(ra, 1, st) : launch_rows<false>(ra, 1, st)) return rc;
  const AddArgs a = add_args(rows, lora_b, bias, y, ldy, y, ldy, M, N, r, scaling);
  if (f16) lora_add_kernel<true, true><<<a.blocks, 256, 0, st>>>(a, SumArgs{});
  else lora_add_kernel<true, false><<<a.blocks, 256, 0, st>>>(a, SumArgs{});
  return launch_check("lora_add");
}

extern "C" int grpo_lora_backward(const void* x, int64_t ldx, const void* grad, int64_t ldg,
                                  const void* lora_a, const void* lora_b, int r, float scaling,
                                  int M, int N, int K, int f16, void* grad_x, int64_t ldgx,
                                  void* grad_a, void* grad_b, void* workspace,
                                  size_t workspace_bytes, grpo_stream_t stream) {
  if (!train_ok(M, N, K, r)) return train_unsupported();
  if (M == 0) return einval("M > 0 required");
  if (!grad_x && !grad_a && !grad_b) return GRPO_OK;
  if (!x || !grad || !lora_a || !lora_b || !workspace) return einval("null pointer");
  if (ldx < K || ldx % 8 || !aligned16(x)) return einval("x rows must be 16-byte aligned");
  if (ldg < N || ldg % 8 || !aligned16(grad)) return einval("grad rows must be 16-byte aligned");
  if (grad_x && (ldgx < K || ldgx % 8 || !aligned16(grad_x)))
    return einval("grad_x rows must be 16-byte aligned");
  if (!aligned16(lora_a) || !aligned16(workspace) || !aligned16(grad_a) || !aligned16(grad_b))
    return einval("lora_a, the gradients and the workspace must be 16-byte aligned");
  if (workspace_bytes < train_ws(M, N, K, r).total) {
    set_error("workspace too small");
    return GRPO_EWORKSPACE;
  }
  auto u = [](const void* q) { return static_cast<const uint16_t*>(q); };
  auto v = [](void* q) { return static_cast<uint16_t*>(q); };
  hipStream_t st = as_stream(stream);
  char* ws = static_cast<char*>(workspace);
  return f16 ? run_backward<true>(u(x), ldx, u(grad), ldg, u(lora_a), u(lora_b), r, scaling, M, N,
                                  K, v(grad_x), ldgx, v(grad_a), v(grad_b), ws, st)
             : run_backward<false>(u(x), ldx, u(grad), ldg, u(lora_a), u(lora_b), r, scaling, M, N,
                                   K, v(grad_x), ldgx, v(grad_a), v(grad_b), ws, st);
}
