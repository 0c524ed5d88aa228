// Paged GQA attention of a prompt chunk for gfx950: many rows of ONE sequence (one
// block table), row m over the sequence's first lens[m] tokens, bf16 output. The
// attention part of the reference's prefill forward (src/triton_kernels/paged_kv.py:
// 547-586 runs a transformers forward), with the decode kernel's arithmetic
// (paged_attention.hip): float32 scores in the log2 domain, online softmax,
// P.V as V.P_hi + V.P_lo on bf16 MFMA (P = P_hi + P_lo within 2^-17 |P|), out =
// bf16(O / max(sum, 1e-6)).
//
// The decode kernel gives every row a workgroup of its own, which reads that row's
// whole context: 512 rows read the shared K/V 512 times, ten of sixteen MFMA columns
// idle, and a second launch merges the splits. Here 16 rows are the 16 columns:
//  * A wave owns one query head of 16 rows; a workgroup the same rows for HW
//    heads of one KV head, CS times: its CS groups of waves take the 32-token parts
//    of each step and meet in LDS at the end, so that the longest chain (the last
//    rows, over the whole context) is a CS-th as long. A wave's step is bound by its
//    instruction issue (about 450 for 32 tokens, 1.3 us), and a chunk has fewer waves
//    than the chip has SIMDs (three heads, two parts: 15.7 us; four parts 13.1).
//  * K and V of a step (16 KiB per part) come to LDS by global_load_lds, one step
//    ahead; a token's sixteen 16-byte chunks are stored at chunk ^ (token % 16), so that
//    the score operand's reads (16 tokens, one chunk) spread over the banks.
//  * S^T = K Q^T leaves lane (row ln, group lg) with the scores of tokens 4 lg + r of
//    both 16-token tiles, which is the operand P^T of the next product if its
//    contraction index (lg, e) means token 16 (e / 4) + 4 lg + e % 4: P never leaves
//    the lane. V's operand is read as rows and its pairs are turned with v_perm.
//  * A token that only some of the 16 rows attend has P = 0 in the others. Where its V is
//    not finite (an overflow, a slot never written) it is taken out of the product and
//    the rows that do attend it are set to NaN.
// Bound by that issue and, for short contexts, by the launch and the first loads (7.1
// us at 128 rows, 0.4 of them for the look at values that are not finite). 512 rows
// after nothing, 12 query and 2 KV heads: 11.5 us against 29.1 for the decode kernel and
// its merge; after 4000 tokens 55 us against 164.
#include <algorithm>

#include "lds_dma.hpp"

using namespace grpo;

namespace {

constexpr int PD = 128;            // head dim
constexpr int PBS = 16;            // block size
constexpr int PART_B = 32 * PD * 2 * 2;  // bytes of 32 tokens of K and V
constexpr int RING = 2;
constexpr float LOG2E = 1.4426950408889634f;

struct PrefillArgs {
  const uint16_t* q;
  int64_t qsb, qsh;
  const uint16_t* kc;
  const uint16_t* vc;
  int64_t num_blocks;
  const int32_t* bt;
  const int32_t* lens;
  uint16_t* out;  // [M][Hq][128]
  int M, Hq, Hkv, max_blocks;
  float scale;
};

// Largest value of each row of 16 lanes, of the first row for the whole wave (the
// rows hold the same values): DPP moves, no LDS round trips.
__device__ __forceinline__ int max16(int v) {
#define STEP_MAX(ctrl) v = max(v, __builtin_amdgcn_update_dpp(0, v, ctrl, 0xF, 0xF, false))
  STEP_MAX(0xB1);   // quad_perm xor 1
  STEP_MAX(0x4E);   // quad_perm xor 2
  STEP_MAX(0x141);  // row_half_mirror
  STEP_MAX(0x140);  // row_mirror
#undef STEP_MAX
  return __builtin_amdgcn_readfirstlane(v);
}

__device__ __forceinline__ uint32_t word(const uint4& v, int i) {
  return i == 0 ? v.x : (i == 1 ? v.y : (i == 2 ? v.z : v.w));
}

__device__ __forceinline__ uint4 keep(uint32_t mask, const uint4& v) {
  return make_uint4(v.x & mask, v.y & mask, v.z & mask, v.w & mask);
}
// All ones in the halves of d that are an infinity or NaN (exponent bits all set).
__device__ __forceinline__ uint32_t inf_mask(uint32_t d) {
  return ((d & 0x7F80u) == 0x7F80u ? 0xFFFFu : 0u) |
         ((d & 0x7F800000u) == 0x7F800000u ? 0xFFFF0000u : 0u);
}
// Per half the larger of m and of v's bits in mask.
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u16x2 max_halves(u16x2 m, uint32_t mask, const uint4& v) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, word(v, i) & mask));
  return m;
}
// Of V's rows (a token each, 8 dims) the operand V^T of the dims 8 (..) + i.
__device__ __forceinline__ uint4 turned(const uint4 (&v)[8], int i) {
  const uint32_t sel = (i & 1) ? 0x07060302u : 0x05040100u;
  return make_uint4(perm(word(v[1], i >> 1), word(v[0], i >> 1), sel),
                    perm(word(v[3], i >> 1), word(v[2], i >> 1), sel),
                    perm(word(v[5], i >> 1), word(v[4], i >> 1), sel),
                    perm(word(v[7], i >> 1), word(v[6], i >> 1), sel));
}

// HW heads per workgroup, CS parts of a step (32 tokens each): CS HW waves.
template <int HW, int CS>
__global__ void __launch_bounds__(64 * CS * HW) prefill_attn_kernel(PrefillArgs p) {
  touch_kernargs<sizeof(PrefillArgs)>();
  constexpr int STEP = 32 * CS, STEP_BLK = STEP / PBS, STEP_B = CS * PART_B;
  constexpr int PIECES = STEP_B / 1024;
  constexpr int W = CS * HW, LD = (PIECES + W - 1) / W;
  extern __shared__ __align__(16) char lds[];  // [RING][STEP_B]; the waves' merge afterwards
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 15, lg = lane >> 4;
  const int part = wave / HW;
  const int GQ = p.Hq / p.Hkv, ng = (GQ + HW - 1) / HW;
  const int kvh = blockIdx.y / ng, hk = (blockIdx.y - kvh * ng) * HW + wave % HW;
  const int head = kvh * GQ + min(hk, GQ - 1);
  const int m = ((int)(gridDim.x - 1 - blockIdx.x)) * 16 + ln;  // the longest rows first
  const int mc = min(m, p.M - 1);
  const int cap = p.max_blocks * PBS;
  const int len_v = p.lens[mc];
  // The ids of 64 blocks, one per lane (reloaded every 64 blocks), as indexes of
  // (block, KV head) in the caches; ids out of range read block 0 (their tokens are
  // masked and their V cleared).
  int tb_v = p.bt[min(lane, p.max_blocks - 1)];
  uint4 qf[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    qf[i] = *reinterpret_cast<const uint4*>(p.q + (int64_t)mc * p.qsb + (int64_t)head * p.qsh +
                                            8 * lg + 32 * i);
  uint64_t okm = 0, okm_before = 0;  // valid ids of this and the previous 64 blocks
  int tb, win = 0;
  auto take_table = [&]() __attribute__((always_inline)) {
    const bool ok = tb_v >= 0 && tb_v < p.num_blocks;
    okm = __builtin_amdgcn_ballot_w64(ok);
    tb = (ok ? tb_v : 0) * p.Hkv + kvh;
  };
  const int len = m < p.M ? max(0, min(len_v, cap)) : 0;
  const int most = max16(len), least = -max16(m < p.M ? -len : -cap);
  const int nblk = (most + PBS - 1) / PBS, nstep = (most + STEP - 1) / STEP;
  const int row4 = lane >> 4, slot = lane & 15;
  const uint32_t lbase = lds_address(lds);
  // Piece pc of a step: tokens 4 (pc % 8) .. + 3 of K (pc / 8 even) or V of part pc / 16.
  // Blocks past the rows' contexts read the last one (its tokens are masked).
  uint32_t voff[LD];
#pragma unroll
  for (int i = 0; i < LD; ++i) {
    const int t = 4 * (min(wave + W * i, PIECES - 1) & 3) + row4;
    voff[i] = t * (PD * 2) + 16 * (slot ^ t);
  }
  auto fetch = [&](int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      const int pc = min(wave + W * i, PIECES - 1);  // waves repeat the last piece to a whole LD
      const int b = min(STEP_BLK * st + 2 * (pc >> 4) + ((pc >> 2) & 1), nblk - 1);
      const int64_t at = __builtin_amdgcn_readlane(tb, b & 63);
      const char* const base = reinterpret_cast<const char*>((pc >> 3) & 1 ? p.vc : p.kc);
      dma16(lbase + (st % RING) * STEP_B + pc * 1024, voff[i], base + at * (PBS * PD * 2));
    }
  };

  const float sl2 = p.scale * LOG2E;
  float m_run = -INFINITY, l_run = 0.f;  // of row ln
  f32x4_t oacc[8];                       // O[row ln][8 (4 lg + q) + i] in oacc[i][q]
#pragma unroll
  for (int i = 0; i < 8; ++i) oacc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  take_table();
  // Wait for q here: at its first use the compiler, which does not count the
  // fetches, would wait for all of them, in every step.
#pragma unroll
  for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(qf[i].x), "+v"(qf[i].y), "+v"(qf[i].z), "+v"(qf[i].w));
  if (nstep > 0) fetch(0);
  for (int st = 0; st < nstep; ++st) {
    wait_vm<0>();  // step st has landed
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // The slot filled now was read a step ago: every wave is past that. The last step
    // fetches nothing (the slots hold what it and the step before it read).
    if (st + 1 < nstep) {
      if ((st + 1) / (64 / STEP_BLK) != win) {
        win = (st + 1) / (64 / STEP_BLK);
        tb_v = p.bt[min(64 * win + lane, p.max_blocks - 1)];
        okm_before = okm;
        take_table();
      }
      fetch(st + 1);
    }
    const int t0 = STEP * st + 32 * part;
    if (t0 >= most) continue;
    const uint64_t okw = st / (64 / STEP_BLK) == win ? okm : okm_before;
    const int b0 = STEP_BLK * st + 2 * part;
    const bool ok0 = (okw >> (min(b0, nblk - 1) & 63)) & 1;
    const bool ok1 = (okw >> (min(b0 + 1, nblk - 1) & 63)) & 1;
    const char* const kb = lds + (st % RING) * STEP_B + part * PART_B;
    const char* const vb = kb + PART_B / 2;
    f32x4_t s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      s[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint4 kf = *reinterpret_cast<const uint4*>(
            kb + (16 * t + ln) * (PD * 2) + 16 * ((lg + 4 * i) ^ ln));
        s[t] = mfma16x16x32(kf, qf[i], s[t]);
      }
    }
    uint4 v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int t = 16 * (e >> 2) + 4 * lg + (e & 3);
      v[e] = *reinterpret_cast<const uint4*>(vb + t * (PD * 2) + 16 * (ln ^ (t & 15)));
    }
    float sv[8], bmax = -INFINITY;
#pragma unroll
    for (int e = 0; e < 8; ++e) sv[e] = s[e >> 2][e & 3] * sl2;
    if (t0 + 32 > least || !(ok0 && ok1)) {  // some row ends here, or a block is missing
      const uint32_t z[2] = {ok0 ? ~0u : 0u, ok1 ? ~0u : 0u};
      u16x2 top{0, 0};  // largest exponent of the tokens that some row does not attend
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int t = t0 + 16 * (e >> 2) + 4 * lg + (e & 3);
        const bool on = t < len && z[e >> 2];
        sv[e] = on ? sv[e] : -INFINITY;
        v[e] = keep(z[e >> 2], v[e]);
        top = max_halves(top, t < least ? 0u : 0x7F807F80u, v[e]);
      }
      // A value that is not finite, in a token that some row does not attend: 0 times it
      // would be NaN. It leaves V; the rows that attend its token become NaN there.
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(max(top.x, top.y) == 0x7F80u) != 0, 0)) {
        uint32_t one[4] = {0, 0, 0, 0};  // 1 (bf16) for the tokens that the row attends
        uint4 w[8];                      // ... and for the values that leave V
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int t = t0 + 16 * (e >> 2) + 4 * lg + (e & 3);
          one[e >> 1] |= t < len ? 0x3F80u << (16 * (e & 1)) : 0u;
          const uint4 f = keep(t >= least ? ~0u : 0u,
                               make_uint4(inf_mask(v[e].x), inf_mask(v[e].y), inf_mask(v[e].z),
                                          inf_mask(v[e].w)));
          w[e] = keep(0x3F803F80u, f);
          v[e] = make_uint4(v[e].x & ~f.x, v[e].y & ~f.y, v[e].z & ~f.z, v[e].w & ~f.w);
        }
        const uint4 b = make_uint4(one[0], one[1], one[2], one[3]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const f32x4_t n = mfma16x16x32(turned(w, i), b, f32x4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
          for (int q = 0; q < 4; ++q) oacc[i][q] = n[q] > 0.f ? NAN : oacc[i][q];
        }
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) bmax = fmaxf(bmax, sv[e]);
    bmax = pair32_max(pair16_max(bmax));
    const float m_new = fmaxf(m_run, bmax);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;  // no token yet: every P is 0
    const float corr = __builtin_amdgcn_exp2f(m_run - m_use);
    float pv[8], ps = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      pv[e] = __builtin_amdgcn_exp2f(sv[e] - m_use);
      ps += pv[e];
    }
    l_run = l_run * corr + pair32_sum(pair16_sum(ps));
    m_run = m_new;
    uint32_t ph[4], pl[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      ph[q] = pack_bf2(pv[2 * q], pv[2 * q + 1]);
      pl[q] = pack_bf2(pv[2 * q] - bf_lo(ph[q]), pv[2 * q + 1] - bf_hi(ph[q]));
    }
    if (__builtin_amdgcn_ballot_w64(corr != 1.f)) {
#pragma unroll
      for (int i = 0; i < 8; ++i) oacc[i] *= corr;
    }
    const uint4 bh = make_uint4(ph[0], ph[1], ph[2], ph[3]);
    const uint4 bl = make_uint4(pl[0], pl[1], pl[2], pl[3]);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint4 a = turned(v, i);
      oacc[i] = mfma16x16x32(a, bh, oacc[i]);
      oacc[i] = mfma16x16x32(a, bl, oacc[i]);
    }
  }
  wait_vm<0>();
  __syncthreads();  // every wave is past its last read of the ring

  // The other parts' waves hand (max, sum, O) to the first part's: 34 values per lane,
  // strided by lane.
  float* const x = reinterpret_cast<float*>(lds) + (size_t)(wave % HW) * 34 * 64 + lane;
  constexpr int XP = HW * 34 * 64;  // values of a part
  if (part > 0) {
    float* const w = x + (size_t)(part - 1) * XP;
    w[0] = m_run;
    w[64] = l_run;
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) w[64 * (2 + 4 * i + q)] = oacc[i][q];
  }
  __syncthreads();
  if (part > 0) return;
  float M = m_run, f[CS], den = 0.f;
#pragma unroll
  for (int c = 1; c < CS; ++c) M = fmaxf(M, x[(c - 1) * XP]);
#pragma unroll
  for (int c = 0; c < CS; ++c) {
    const float mx = c ? x[(c - 1) * XP] : m_run;
    f[c] = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mx - M);
    den += f[c] * (c ? x[(c - 1) * XP + 64] : l_run);
  }
  den = fmaxf(den, 1e-6f);
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float o = f[0] * oacc[i][q];
#pragma unroll
      for (int c = 1; c < CS; ++c) o += f[c] * x[(c - 1) * XP + 64 * (2 + 4 * i + q)];
      oacc[i][q] = o / den;
    }
  if (m >= p.M || hk >= GQ) return;
  uint16_t* const o = p.out + ((int64_t)m * p.Hq + head) * PD;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *reinterpret_cast<uint4*>(o + 8 * (4 * lg + q)) =
        make_uint4(pack_bf2(oacc[0][q], oacc[1][q]), pack_bf2(oacc[2][q], oacc[3][q]),
                   pack_bf2(oacc[4][q], oacc[5][q]), pack_bf2(oacc[6][q], oacc[7][q]));
}

template <int HW, int CS>
int go(const PrefillArgs& a, hipStream_t st) {
  constexpr int LDS = RING * CS * PART_B;
  static_assert((CS - 1) * HW * 34 * 64 * 4 <= LDS, "the merge fits the ring");
  constexpr auto kern = prefill_attn_kernel<HW, CS>;
  if (int rc = allow_dynamic_lds<kern, LDS>()) return rc;
  const dim3 grid((unsigned)cdiv(a.M, 16), (unsigned)(a.Hkv * cdiv(a.Hq / a.Hkv, HW)));
  kern<<<grid, 64 * CS * HW, LDS, st>>>(a);
  return launch_check("prefill_attn");
}

// Heads per workgroup and parts of a step. Two heads in four parts while every workgroup
// has a CU of its own (128 KiB of LDS), else up to four heads in two parts: 512 rows of
// 12 / 2 heads 11.2 us against 14.7, of 28 / 4 heads 21.4 against 15.2 (each 0.4 more since
// the look at values that are not finite).
struct Form {
  int heads, parts;
};
Form form_of(int M, int Hq, int Hkv) {
  const int gq = Hq / Hkv;
  if (cdiv(M, 16) * Hkv * cdiv(gq, 2) <= 256) return {std::min(gq, 2), 4};
  return {gq > 2 ? 4 : gq, 2};
}

bool prefill_ok(int Hq, int Hkv, int D, int block_size) {
  return Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && D == PD && block_size == PBS &&
         (int64_t)Hq < 65536;
}

}  // namespace

extern "C" int grpo_paged_attn_prefill_supported(int Hq, int Hkv, int D, int block_size) {
  return prefill_ok(Hq, Hkv, D, block_size) ? 1 : 0;
}

extern "C" int grpo_paged_attn_prefill_plan(int M, int Hq, int Hkv, int* heads, int* parts) {
  if (M < 1 || !heads || !parts || !prefill_ok(Hq, Hkv, PD, PBS))
    return einval("bad attention dimensions");
  const Form f = form_of(M, Hq, Hkv);
  *heads = f.heads;
  *parts = f.parts;
  return GRPO_OK;
}

extern "C" int grpo_paged_attn_prefill(const void* q, int64_t q_stride_b, int64_t q_stride_h,
                                       const void* k_cache, const void* v_cache,
                                       int64_t num_blocks, const int32_t* block_table,
                                       const int32_t* lens, void* out, int M, int Hq, int Hkv,
                                       int D, int block_size, int max_blocks, float scale,
                                       grpo_stream_t stream) {
  if (M < 0 || max_blocks < 1 || num_blocks < 1) return einval("bad attention dimensions");
  if (!prefill_ok(Hq, Hkv, D, block_size)) {
    set_error("shape not supported by the prefill attention (head_dim 128, block size 16, Hq a "
              "multiple of Hkv)");
    return GRPO_EUNSUPPORTED;
  }
  if (M == 0) return GRPO_OK;
  if (!q || !k_cache || !v_cache || !block_table || !lens || !out) return einval("null pointer");
  if (!aligned16(q) || q_stride_b % 8 || q_stride_h % 8 || !aligned16(k_cache) ||
      !aligned16(v_cache) || !aligned16(out))
    return einval("q rows, the caches and out must be 16-byte aligned");
  const PrefillArgs a{static_cast<const uint16_t*>(q), q_stride_b, q_stride_h,
                      static_cast<const uint16_t*>(k_cache),
                      static_cast<const uint16_t*>(v_cache), num_blocks, block_table, lens,
                      static_cast<uint16_t*>(out), M, Hq, Hkv, max_blocks, scale};
  hipStream_t st = as_stream(stream);
  const Form f = form_of(M, Hq, Hkv);
  if (f.parts == 4) return f.heads == 1 ? go<1, 4>(a, st) : go<2, 4>(a, st);
  if (f.heads == 1) return go<1, 2>(a, st);
  return f.heads == 2 ? go<2, 2>(a, st) : go<4, 2>(a, st);
}
