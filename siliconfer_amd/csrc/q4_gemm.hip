// q4_gemm.hip — int4 prefill GEMM on CDNA4 MFMA (gfx950).
//
// Y[m, n] = sum_k X[m, k] * (q[n,k] - z[n,g(k)]) * s[n,g(k)], fp32 accumulation:
// the reference's q4_gemm_sym / q4_gemm_asym
// (/root/reference/siliconfer/kernels/neon/q4_gemm.cpp:12-51), which loop the
// GEMV over the T rows and re-stream W for each; here W is read once per
// 128-row block of X. Both kernels fold each scale group's fp32 partial into
// the result once, with the group's fp16 scale: y = sum_g s_g * sum_{k in g}
// x_k (q_k - z), the reference's own grouping (q4_gemv.cpp:136).
//
// Two kernels:
//  * k_q4_gemm_rows (q4_gemm_rows.h; groups of 32, 64 or a multiple of 128):
//    16-bit activations as they are, fp32 ones as two bf16 halves that a first
//    launch writes to the workspace (sf_q4_matmul only).
//  * k_q4_gemm (fp32 activations through sf_q4_gemm, whose workspace holds no
//    halves, and the other multiples of 32): staging threads dequantize the W
//    tile once into LDS as the integers q - z (exact in fp16 and bf16); fp32
//    activations are split into bf16 high and low parts (two MFMAs); 128 x 128
//    per 512 threads (2 x 4 waves of 64 x 32), K steps of 64 through two padded
//    LDS buffers with each step's global loads three steps ahead in registers;
//    the output goes back through LDS as whole row segments.
// When the tile grid is too small to fill the GPU, K is split across
// workgroups into an fp32 workspace and summed by a second kernel in a fixed
// order.
#include <limits.h>
#include <math.h>

#include "q4_gemm_rows.h"
#include "q4_gemv_blk.h"
#include "sf_common.h"

bool sf_gemm_rows_f16(const sf_gemm::RowsArgs &a, const sf_gemm::RowsGroupArgs *group, bool asym, int rb, int kw,
                      hipStream_t s);
bool sf_gemm_rows_bf16(const sf_gemm::RowsArgs &a, const sf_gemm::RowsGroupArgs *group, bool asym, int rb, int kw,
                      hipStream_t s);
bool sf_gemm_rows_f32(const sf_gemm::RowsArgs &a, const sf_gemm::RowsGroupArgs *group, bool asym, int rb, int kw,
                      hipStream_t s);

namespace {

using sf_gemm::bf16x8_t;
using sf_gemm::float16_t;
using sf_gemm::half8_t;

constexpr int BM = 128, BN = 128, BK = 64;
constexpr int kGemmGemvRows = 16;  // sf_q4_gemm runs up to this many rows as 8-row batch GEMVs
constexpr int LDS_PITCH = BK + 8;  // bf16 elements per LDS row (+16 B breaks bank conflicts)
constexpr int NTHREADS = 512;      // 8 waves: two per SIMD, so one's VALU overlaps another's MFMA
constexpr int KPT = BM * BK / NTHREADS;  // 16 elements of X (and of W) staged per thread per step
constexpr int WAVE_M = 64, WAVE_N = 32;  // wave tile: 2 x 1 MFMA 32x32 tiles
constexpr int OUT_PITCH = WAVE_N + 4;    // fp32 pitch of a wave's output tile staged in LDS
static_assert(BN * BK / NTHREADS == KPT, "X and W staging shares must match");
static_assert((BM / WAVE_M) * (BN / WAVE_N) * 64 == NTHREADS, "wave grid must cover the tile");

__device__ __forceinline__ uint32_t hi_pair(uint32_t a, uint32_t b) {
  // top 16 bits of a (low half) and of b (high half)
  return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

// One thread's share of the X tile: row tid/4, KPT consecutive k starting at
// KPT*(tid%4). Loaded into registers as raw bits; loads are unconditional
// (clamped in-bounds address; K is a multiple of 32) so they stay in flight,
// and rows or k past the end are zeroed when the registers are staged.
template <int XDT>
struct XRegs {
  static constexpr int NQ = KPT * (XDT == SF_F32 ? 4 : 2) / 16;  // 16-byte loads
  u32x4 v[NQ];
  bool ok;
};

template <int XDT>
__device__ __forceinline__ void load_x(XRegs<XDT> &r, const void *X, int M, int K, int m, int k) {
  r.ok = m < M && k < K;
  const size_t esz = XDT == SF_F32 ? 4 : 2;
  const u32x4 *p =
      (const u32x4 *)((const char *)X + ((size_t)min(m, M - 1) * K + min(k, K - KPT)) * esz);
#pragma unroll
  for (int i = 0; i < XRegs<XDT>::NQ; ++i) r.v[i] = p[i];
}

// Split 2 fp32 values into (hi pair, lo pair) of bf16: hi = truncation, lo = rest.
__device__ __forceinline__ void split2(float a, float b, uint32_t &hi, uint32_t &lo) {
  const uint32_t ua = sf_bitcast<uint32_t>(a) & 0xFFFF0000u;
  const uint32_t ub = sf_bitcast<uint32_t>(b) & 0xFFFF0000u;
  const float ra = a - sf_bitcast<float>(ua);
  const float rb = b - sf_bitcast<float>(ub);
  hi = hi_pair(ua, ub);
  lo = hi_pair(sf_bitcast<uint32_t>(ra), sf_bitcast<uint32_t>(rb));
}

// Write the thread's KPT activations to the LDS tiles: fp16 / bf16 as they
// are, fp32 as bf16 high and low parts.
template <int XDT>
__device__ __forceinline__ void store_x(const XRegs<XDT> &r, uint16_t *xs_hi, uint16_t *xs_lo,
                                        int lrow, int lk) {
  u32x4 *dh = (u32x4 *)(xs_hi + lrow * LDS_PITCH + lk);
  const uint32_t keep = r.ok ? 0xFFFFFFFFu : 0u;
  if constexpr (XDT != SF_F32) {
#pragma unroll
    for (int i = 0; i < KPT / 8; ++i) dh[i] = r.v[i] & keep;
  } else {
    u32x4 *dl = (u32x4 *)(xs_lo + lrow * LDS_PITCH + lk);
#pragma unroll
    for (int i = 0; i < KPT / 8; ++i) {  // 8 activations per 16-byte LDS store
      float f[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = sf_bitcast<float>(r.v[2 * i + j / 4][j % 4] & keep);
      u32x4 h4, l4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t hp, lp;
        split2(f[2 * j], f[2 * j + 1], hp, lp);
        h4[j] = hp;
        l4[j] = lp;
      }
      dh[i] = h4;
      dl[i] = l4;
    }
  }
}

// One thread's share of the W tile: KPT = 16 codes of row n from k (two
// dwords of the blob's unit: k-pieces k and k + 8 of the same MFMA slice sit in
// lanes 16 apart), and the raw scale / zero-point bits of that (row, group);
// converted at staging (a step never straddles a group: g is a multiple of 32
// and KPT divides 32).
struct WRegs {
  u32x2 w;
  uint32_t sbits, zbyte;
  bool ok;
};

template <bool ASYM>
__device__ __forceinline__ void load_w(WRegs &r, const uint8_t *__restrict__ wq,
                                       const f16 *__restrict__ st, const uint8_t *__restrict__ zt,
                                       int N, int K, int G, int g, int n, int k) {
  r.ok = n < N && k < K;
  const int nc = min(n, N - 1), kc = min(k, K - KPT);
  const int nb = (K + 127) >> 7, kb = kc & 127;
  const uint8_t *unit = wq + ((size_t)(nc >> 4) * nb + (kc >> 7)) * 1024;
  const int lane = ((kb & 31) >> 3) * 16 + (nc & 15);
  r.w.x = *(const uint32_t *)(unit + lane * 16 + (kb >> 5) * 4);
  r.w.y = *(const uint32_t *)(unit + (lane + 16) * 16 + (kb >> 5) * 4);
  const size_t cell = (size_t)(nc >> 3) * G + kc / g;
  r.sbits = ((const uint16_t *)st)[cell * 8 + (nc & 7)];
  if constexpr (ASYM) r.zbyte = zt[cell * 4 + ((nc & 7) >> 1)];
}

// Store the thread's KPT weights as the integers q - z (fp16 when MT is
// SF_F16, else bf16; zero past the matrix) and, from the threads at the start
// of a 32-k half, the row's scale for that half into the scale table.
template <bool ASYM, int MT>
__device__ __forceinline__ void store_w(const WRegs &r, uint16_t *ws, uint16_t *ss, int lrow,
                                        int lk) {
  u32x4 *d = (u32x4 *)(ws + lrow * LDS_PITCH + lk);
  // row n's zero-point nibble: the low one for even n, the high one for odd n
  // (offset-binary symmetric codes have z = 8)
  uint32_t z = 8u;
  if constexpr (ASYM) z = (r.zbyte >> (4 * (lrow & 1))) & 15u;
  const uint32_t keep = r.ok ? 0xFFFFFFFFu : 0u;
#pragma unroll
  for (int i = 0; i < KPT / 8; ++i) {  // dword i holds k = 8i .. 8i+7, code e at 4(e/2) + 16(e%2)
    const uint32_t dw = i == 0 ? r.w.x : r.w.y;
    u32x4 o;
#pragma unroll
    for (int b = 0; b < 4; ++b) {  // pair (k = 8i + 2b, 8i + 2b + 1) in the two 16-bit halves
      const uint32_t pq = (dw >> (4 * b)) & 0x000F000Fu;
      if constexpr (MT == SF_F16) {
        // 1024 + q as fp16, minus (1024 + z): exact
        const half2_t v = sf_bitcast<half2_t>(pq | 0x64006400u) +
                          sf_bitcast<half2_t>((0xE400u | z) * 0x10001u);
        o[b] = sf_bitcast<uint32_t>(v);
      } else {
        const float f0 = (float)(int)((pq & 0xFu) - z), f1 = (float)(int)((pq >> 16) - z);
        o[b] = hi_pair(sf_bitcast<uint32_t>(f0), sf_bitcast<uint32_t>(f1));
      }
    }
    d[i] = o & keep;
  }
  if ((lk & 31) == 0) ss[lrow * 2 + (lk >> 5)] = (uint16_t)r.sbits;
}

// GK: the group size's shape, fixed at compile time so the per-group folds
// are straight-line code: 0 = 32 (two groups per K step), 1 = 64 (one per
// step), 2 = a multiple of 128 (a group spans several steps; a test per
// step), 3 = any other multiple of 32 (a test per 16-k slice).
template <int XDT, bool ASYM, int GK>
__global__ void __launch_bounds__(NTHREADS, 2)
k_q4_gemm(const uint8_t *__restrict__ wq, const f16 *__restrict__ st,
          const uint8_t *__restrict__ zt, const void *__restrict__ X, void *__restrict__ Y,
          int ydt, float *__restrict__ y32, const void *__restrict__ bias, int bdt,
          float *__restrict__ part, int M, int N, int K, int G, int g, int ksplit,
          int steps_per_split, bool vec) {
  constexpr bool XSPLIT = XDT == SF_F32;             // fp32 activations: bf16 hi + lo
  constexpr int MT = XDT == SF_F16 ? SF_F16 : SF_BF16;  // MFMA operand type
  constexpr int XB = BM * LDS_PITCH, WB = BN * LDS_PITCH;  // one LDS buffer of each tile
  constexpr int SB = BN * 2;                               // scales: 2 halves of the step per row
  constexpr int SMEM_U16 = 2 * XB * (XSPLIT ? 2 : 1) + 2 * WB + 2 * SB;
  constexpr int NWAVES = NTHREADS / 64;
  constexpr int OUT_U16 = NWAVES * WAVE_M * OUT_PITCH * 2;
  __shared__ __attribute__((aligned(16))) uint16_t smem[SMEM_U16 > OUT_U16 ? SMEM_U16 : OUT_U16];
  uint16_t *const xs_hi = smem;
  uint16_t *const xs_lo = smem + 2 * XB;  // used only when XSPLIT
  uint16_t *const ws = smem + 2 * XB * (XSPLIT ? 2 : 1);
  uint16_t *const ss = ws + 2 * WB;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  constexpr int WGN = BN / WAVE_N;  // waves across the tile's columns
  const int wm = (wave / WGN) * WAVE_M, wn = (wave % WGN) * WAVE_N;  // wave tile origin
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int split = blockIdx.z;
  const int nsteps_total = (K + BK - 1) / BK;
  const int s0 = split * steps_per_split;
  const int s1 = min(s0 + steps_per_split, nsteps_total);

  // staging assignment: row tid / (BK / KPT), KPT consecutive k
  const int lrow = tid / (BK / KPT), lk = (tid % (BK / KPT)) * KPT;

  float16_t acc[2], gp[2];  // the result, and the current scale group's partial
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = gp[i][r] = 0.f;

  // Loads past the split's last step re-read that step (in bounds, unused), so
  // every load is unconditional and stays in flight.
  auto load = [&](int step, XRegs<XDT> &xr, WRegs &wr) {
    const int k = min(step, s1 - 1) * BK + lk;
    load_x<XDT>(xr, X, M, K, m0 + lrow, k);
    load_w<ASYM>(wr, wq, st, zt, N, K, G, g, n0 + lrow, k);
  };
  auto store = [&](int step, const XRegs<XDT> &xr, const WRegs &wr) {
    const int b = step & 1;
    store_x<XDT>(xr, xs_hi + b * XB, xs_lo + (XSPLIT ? b * XB : 0), lrow, lk);
    store_w<ASYM, MT>(wr, ws + b * WB, ss + b * SB, lrow, lk);
  };
  // a lane's accumulators all belong to output column c: one scale per group
  auto fold = [&](float sc) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][r] = fmaf(gp[i][r], sc, acc[i][r]);
  };
  const float16_t zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f,
                            0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // one K step; `fresh`: the step starts a scale group (its first MFMAs take
  // a zero accumulator), `last`: the step ends one (fold after it)
  auto compute_step = [&](int step, bool fresh, bool last) {
    const int b = step & 1;
    const uint16_t *xh = xs_hi + b * XB, *xl = xs_lo + (XSPLIT ? b * XB : 0);
    const uint16_t *wt = ws + b * WB;
    const int c = wn + (lane & 31);
    const int kb = step * BK;
#pragma unroll
    for (int kk = 0; kk < BK; kk += 16) {
      // a group starts here: the slice's MFMAs take a zero accumulator
      const bool zc = GK == 3 ? (kk % 32 == 0 && ((kb + kk) % g == 0 || (kk == 0 && step == s0)))
                              : (kk == 0 && fresh) || (GK == 0 && kk == 32);
      const int kofs = kk + (lane >> 5) * 8;
      u32x4 ah[2], al[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = wm + i * 32 + (lane & 31);
        ah[i] = *(const u32x4 *)(xh + r * LDS_PITCH + kofs);
        if constexpr (XSPLIT) al[i] = *(const u32x4 *)(xl + r * LDS_PITCH + kofs);
      }
      const u32x4 bw = *(const u32x4 *)(wt + c * LDS_PITCH + kofs);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float16_t cin = zc ? zero16 : gp[i];
        if constexpr (MT == SF_F16) {
          gp[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sf_bitcast<half8_t>(ah[i]),
                                                         sf_bitcast<half8_t>(bw), cin, 0, 0, 0);
        } else {
          gp[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(sf_bitcast<bf16x8_t>(ah[i]),
                                                          sf_bitcast<bf16x8_t>(bw), cin, 0, 0, 0);
          if constexpr (XSPLIT)
            gp[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(sf_bitcast<bf16x8_t>(al[i]),
                                                            sf_bitcast<bf16x8_t>(bw), gp[i], 0, 0, 0);
        }
      }
      // a group ends after this 16-k slice: scale the partial once
      const bool end = GK == 3 ? (kk % 32 == 16 && ((kb + kk + 16) % g == 0 ||
                                                    (kk == BK - 16 && step == s1 - 1)))
                               : (GK == 0 && kk == 16) || (kk == BK - 16 && last);
      if (end) fold((float)sf_bitcast<f16>(ss[b * SB + c * 2 + (kk >> 5)]));
    }
  };
  // g = 32 / 64: every step starts and ends its groups; g >= 128: a group
  // spans g / 64 steps (and a split's last step closes its open group)
  auto compute = [&](int step) {
    if constexpr (GK < 2 || GK == 3) {
      compute_step(step, true, true);  // (GK 3 decides per slice)
    } else {
      const int spg = g / BK;
      const bool fresh = step % spg == 0 || step == s0;
      const bool last = (step + 1) % spg == 0 || step == s1 - 1;
      if (fresh && last) compute_step(step, true, true);
      else if (fresh) compute_step(step, true, false);
      else if (last) compute_step(step, false, true);
      else compute_step(step, false, false);
    }
  };

  // Pipeline: three register stages of global loads (a step's loads are issued
  // three steps before it is staged) and two LDS buffers, one barrier per step.
  // At the top of the loop for step s: LDS buffer s&1 holds step s, xb/wb hold
  // step s+1, xc/wc step s+2, xa/wa step s+3. Staging is unconditional (past
  // the end it re-stages the last step into the buffer no one reads again), so
  // it shares a basic block with the MFMAs and the two can interleave.
  if (s0 < s1) {
    XRegs<XDT> xa, xb, xc;
    WRegs wa, wb, wc;
    load(s0, xa, wa);
    load(s0 + 1, xb, wb);
    load(s0 + 2, xc, wc);
    store(s0, xa, wa);
    __syncthreads();
    load(s0 + 3, xa, wa);
    for (int s = s0; s < s1; s += 3) {
      store(s + 1, xb, wb);
      compute(s);
      __syncthreads();
      if (s + 1 >= s1) break;
      load(s + 4, xb, wb);
      store(s + 2, xc, wc);
      compute(s + 1);
      __syncthreads();
      if (s + 2 >= s1) break;
      load(s + 5, xc, wc);
      store(s + 3, xa, wa);
      compute(s + 2);
      __syncthreads();
      if (s + 3 >= s1) break;
      load(s + 6, xa, wa);
    }
  }

  // Output. acc[i][r] is C[row][col] with row = 8*(r/4) + 4*(lane/32) + r%4,
  // col = lane % 32 within MFMA tile i: a lane holds one column, so each wave
  // stages its WAVE_M x WAVE_N tile in LDS and writes it back as row segments
  // of 8 values per lane (16-byte stores, whole cache lines per instruction).
  __syncthreads();  // every wave is done with the operand buffers
  float *ot = (float *)smem + wave * WAVE_M * OUT_PITCH;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      ot[(i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * OUT_PITCH + (lane & 31)] = acc[i][r];
  __syncthreads();
  constexpr int SEGS = WAVE_N / 8;  // 8-column segments per row
#pragma unroll 2
  for (int it = 0; it < WAVE_M * SEGS / 64; ++it) {
    const int seg = it * 64 + lane;
    const int rl = seg / SEGS, cl = (seg % SEGS) * 8;
    const int row = m0 + wm + rl, col = n0 + wn + cl;
    if (row >= M || col >= N) continue;
    float v[8];
    {
      const float4_t a = *(const float4_t *)(ot + rl * OUT_PITCH + cl);
      const float4_t c = *(const float4_t *)(ot + rl * OUT_PITCH + cl + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = a[e];
        v[4 + e] = c[e];
      }
    }
    const int nv = min(8, N - col);
    const size_t idx = (size_t)row * N + col;
    if (ksplit > 1) {
      float *dst = part + (size_t)split * M * N + idx;
      if (vec && nv == 8) {
        ((float4_t *)dst)[0] = float4_t{v[0], v[1], v[2], v[3]};
        ((float4_t *)dst)[1] = float4_t{v[4], v[5], v[6], v[7]};
      } else {
        for (int e = 0; e < nv; ++e) dst[e] = v[e];
      }
      continue;
    }
    if (bias) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int cc = min(col + e, N - 1);
        v[e] += sf_gemm::bias_at(bias, bdt, cc);
      }
    }
    sf_gemm::store8(v, nv, vec, y32, Y, ydt, idx);
  }
}

// Sum of the K-split partials in split order (deterministic), plus bias, to
// the outputs; 8 consecutive elements per thread.
__global__ void __launch_bounds__(256)
k_splitk_reduce(const float *__restrict__ part, void *__restrict__ Y, int ydt, float *__restrict__ y32,
                const void *__restrict__ bias, int bdt, int M, int N, int ksplit, bool vec) {
  const size_t MN = (size_t)M * N;
  const size_t n8 = (MN + 7) / 8;
  for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n8;
       t += (size_t)gridDim.x * blockDim.x) {
    const size_t idx = t * 8;
    const int row = (int)(idx / N), col = (int)(idx - (size_t)row * N);
    float v[8];
    int nv = 8;
    if (vec) {  // N % 8 == 0: the 8 elements are in one row
      float4_t a = {0.f, 0.f, 0.f, 0.f}, c = a;
      for (int s = 0; s < ksplit; ++s) {
        a += ((const float4_t *)(part + (size_t)s * MN + idx))[0];
        c += ((const float4_t *)(part + (size_t)s * MN + idx))[1];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = a[e];
        v[4 + e] = c[e];
      }
    } else {
      nv = (int)min((size_t)8, MN - idx);
      for (int e = 0; e < 8; ++e) {
        v[e] = 0.f;
        if (e < nv)
          for (int s = 0; s < ksplit; ++s) v[e] += part[(size_t)s * MN + idx + e];
      }
    }
    if (vec) {
      if (bias)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int cc = col + e;
          v[e] += sf_gemm::bias_at(bias, bdt, cc);
        }
      sf_gemm::store8(v, 8, true, y32, Y, ydt, idx);
    } else {
      for (int e = 0; e < nv; ++e) {
        float o = v[e];
        const size_t id = idx + e;
        if (bias) {
          const int cc = (int)(id % N);
          o += sf_gemm::bias_at(bias, bdt, cc);
        }
        if (y32) y32[id] = o;
        if (Y) {
          if (ydt == SF_BF16) ((uint16_t *)Y)[id] = sf_f32_to_bf16(o);
          else if (ydt == SF_F16) ((f16 *)Y)[id] = (f16)o;
          else ((float *)Y)[id] = o;
        }
      }
    }
  }
}

// fp32 activations as two bf16 halves, 8 values a thread: high = the top 16
// bits, low = the rest rounded to nearest (|error| <= 2^-17 of the value).
__global__ void __launch_bounds__(256)
k_split_f32(const float *__restrict__ x, uint16_t *__restrict__ hi, uint16_t *__restrict__ lo, size_t n8) {
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= n8) return;
  const u32x4 v0 = ((const u32x4 *)x)[2 * t], v1 = ((const u32x4 *)x)[2 * t + 1];
  u32x4 h, l;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t a = j < 2 ? v0[2 * j] : v1[2 * j - 4], b = j < 2 ? v0[2 * j + 1] : v1[2 * j - 3];
    h[j] = hi_pair(a, b);
    l[j] = sf_gemm::pk_bf16(sf_bitcast<float>(a) - sf_bitcast<float>(a & 0xFFFF0000u),
                            sf_bitcast<float>(b) - sf_bitcast<float>(b & 0xFFFF0000u));
  }
  ((u32x4 *)hi)[t] = h;
  ((u32x4 *)lo)[t] = l;
}

const void *split_rows(const float *x, void *halves, int M, int K, hipStream_t s) {
  uint16_t *xs = (uint16_t *)halves;
  const size_t n = (size_t)M * K;
  k_split_f32<<<(unsigned)((n / 8 + 255) / 256), 256, 0, s>>>(x, xs, xs + n, n / 8);
  return xs;
}

// K split count: enough (tile, split) workgroups to give every CU one, each
// split keeping at least 4 K steps.
int choose_ksplit(int M, int N, int K) {
  const int tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  const int steps = (K + BK - 1) / BK;
  int s = 1;
  while (tiles * s * 2 <= 256 && steps / (s * 2) >= 4 && s < 8) s *= 2;
  return s;
}

// Shapes k_q4_gemm_rows takes: groups of 32, 64 or a multiple of 128, and
// activations (fp32: both halves) within a buffer resource's 2 GB range. fp32
// rows no more than the grid's 65535 of its 64-row tiles; k_q4_gemm's hold 128,
// and so do the tiles that 16-bit rows take at such counts.
bool rows_takes(int M, int K, int g, int xdt) {
  return (g == 32 || g == 64 || g % 128 == 0) && (xdt != SF_F32 || M <= 65535 * 64) &&
         (size_t)M * K * (xdt == SF_F32 ? 4 : 2) <= 0x7FFFFFFFu;
}

// The tile of k_q4_gemm_rows: rb row blocks of 32, kw K groups of waves. A
// tile's time per step goes as its conversion (c) plus its row blocks; up to
// one workgroup a CU it stands alone (two K groups overlap its latencies:
// 0.6), up to four they share the CU's SIMDs round by round, above that they
// average out. c = 4 row blocks' worth, bf16 (a dearer conversion) 6. Against
// the best of all tiles for 17..2048 rows on ten matrices from 896 x 896 to
// 14336 x 4096 in fp16, bf16 with zero-points and fp32 the choice loses 2.6% on
// average. Examples (us, 32 / 64 / 96 / 128 rows a tile): 2048 rows on
// 4096 x 11008, fp16 - / 195 / - / 169; 512 on 4864 x 896, bf16 with zero-points
// 16.0 / 14.8 / 13.4 / 15.3 (96 rows: 228 workgroups, one round).
void rows_tile(int M, int N, int K, int xdt, int ks, int *rb, int *kw) {
  const bool f32 = xdt == SF_F32;
  const int tn = (N + 127) / 128 * ks, pairs = (K + 127) / 128 / ks;
  float best = 0.f;
  for (int b = 1; b <= (f32 ? 2 : 4) && (b == 1 || 32 * (b - 1) < M); ++b) {
    const float w = (float)((M + 32 * b - 1) / (32 * b) * tn) / 256.f;  // workgroups per CU
    const int k = w <= 1.f && pairs >= 6 && !(f32 && b > 1) ? 2 : 1;
    const float f = k == 2 ? 0.6f : w <= 1.f ? 1.f : w <= 4.f ? 0.9f * ceilf(w) : 0.7f * w;
    const float cost = f * ((xdt == SF_BF16 ? 6.f : 4.f) + b * (f32 ? 2 : 1));
    if (b == 1 || cost < best) {
      best = cost;
      *rb = b;
      *kw = k;
    }
  }
}

// A weight as a RowsSeg whose columns begin at output column `col`.
sf_gemm::RowsSeg rows_seg(const void *blob, const void *bias, int bdt, int N, int K, int g, bool asym,
                          int tile, int col) {
  BlobLayout L;
  sf_blob_layout(N, K, g, asym, &L);
  const uint8_t *w = (const uint8_t *)blob;
  return {w, (const f16 *)(w + L.s_off), asym ? w + L.z_off : nullptr, bias, bdt, N, 0, tile, col};
}

constexpr sf_gemm::RowsSeg kNoSeg = {nullptr, nullptr, nullptr, nullptr, 0, 0, 0, INT_MAX, 0};

sf_gemm::RowsArgs rows_args(const void *blob, const void *x, void *y, float *y32, const void *bias, float *part,
                            int ydt, int bdt, int M, int N, int K, int g, bool asym, int ks, bool vec) {
  const int pairs = (K + 127) / 128;
  return {rows_seg(blob, bias, bdt, N, K, g, asym, 0, 0), x, y, y32, part, ydt, M, K, N,
          K / g, g, ks, (pairs + ks - 1) / ks, (N + 127) / 128, vec};
}

int rows_run(const sf_gemm::RowsArgs &a, int xdt, bool asym, int rb, int kw, hipStream_t s,
             const sf_gemm::RowsGroupArgs *group = nullptr) {
  const bool built = xdt == SF_F32   ? sf_gemm_rows_f32(a, group, asym, rb, kw, s)
                     : xdt == SF_F16 ? sf_gemm_rows_f16(a, group, asym, rb, kw, s)
                                     : sf_gemm_rows_bf16(a, group, asym, rb, kw, s);
  return built ? SF_OK : sf_fail(SF_EUNSUPPORTED, "no GEMM tile of %d row blocks, %d K groups", rb, kw);
}

int splitk_reduce(const float *part, void *y, int y_dtype, float *y_f32, const void *bias, int bias_dtype,
                  int M, int N, int ksplit, bool vec, hipStream_t s) {
  const size_t n8 = ((size_t)M * N + 7) / 8;
  unsigned rg = (unsigned)((n8 + 255) / 256);
  if (rg > 65535u * 16u) rg = 65535u * 16u;
  k_splitk_reduce<<<rg, 256, 0, s>>>(part, y, y_dtype, y_f32, bias, bias_dtype, M, N, ksplit, vec);
  return sf_check_launch("split-K reduce");
}

// How sf_q4_matmul runs a shape.
struct MatmulPlan {
  enum { GEMV, GEMM, ROWS } route;
  int ks, rb, kw;
  size_t parts, halves, bytes;  // workspace: K-split partials, then the fp32 rows' halves
};

// Rows on the GEMV in slices of 8, or on the tile kernels. Up to 8 rows the
// GEMV is ahead where it takes them in one pass with every weight in flight
// (fp16, 4096 x 11008, 8 rows: 10.9 us against 15.4); where its waves loop over
// K (bf16 with groups below 128 at K of about 9000 and more: 4096 x 11008 with
// zero-points 19.9-23.2 us at 1-8 rows against 16.6-17.0, symmetric 14.5 at
// one row, 17.3 at eight, against 16.4) the rows kernel takes zero-points and
// 7 or 8 rows. fp32 rows too long for the GEMV's LDS go to the rows kernel
// (4096 x 4096, 3-16 rows: 21.6-22.0 us on k_q4_gemm, 13.7-14.5).
// 9 to 16 rows stream the weights twice on the GEMV: ahead up to K = 4096 on
// matrices under 32 M weights (4096 x 4096, 12 rows: 9.7 us against 11.2),
// behind above (11008 x 4096: 16.7 against 13.9; 1024 x 8192: 14.0 against 11.3).
// A residual (bias == y_f32: each output adds its own previous value) is the
// GEMV's form; the tile kernels and the split-K reduce take a bias per column.
void matmul_plan(int M, int N, int K, int g, bool asym, int xdt, bool residual, MatmulPlan *p) {
  *p = {MatmulPlan::GEMM, 1, 1, 1, 0, 0, 0};
  if (g % 32) return;
  if (residual) {
    p->route = MatmulPlan::GEMV;
    return;
  }
  sf_gemv::BlkPlan b;
  const bool fits = sf_gemv::plan_blk(M < 8 ? M : 8, N, K, g, xdt, sf_gemv::PRE_NONE, false, &b);
  const bool rows = rows_takes(M, K, g, xdt);
  bool gemv = false;
  if (M <= 8) gemv = fits && !(rows && b.kc && xdt == SF_BF16 && g < 128 && (asym || M > 6));
  else if (M <= kGemmGemvRows)
    gemv = fits && (xdt == SF_F32 || !rows || (K <= 4096 && (size_t)N * K < (size_t)1 << 25));
  if (gemv) {
    p->route = MatmulPlan::GEMV;
    return;
  }
  if (!rows) {
    p->bytes = sf_q4_gemm_workspace_bytes(M, N, K, g);
    return;
  }
  p->route = MatmulPlan::ROWS;
  // K splits while they bring at most two 32-row workgroups per CU and each
  // keeps four units of K (mean loss against the best split count 0.9%)
  const int t32 = (M + 31) / 32 * ((N + 127) / 128), pairs = (K + 127) / 128;
  while (t32 * p->ks * 2 <= 512 && pairs / (2 * p->ks) >= 4 && p->ks < 8) p->ks *= 2;
  rows_tile(M, N, K, xdt, p->ks, &p->rb, &p->kw);
  p->parts = p->ks > 1 ? sf_align256((size_t)p->ks * M * N * sizeof(float)) : 0;
  p->halves = xdt == SF_F32 ? (size_t)M * K * 4 : 0;
  p->bytes = p->parts + p->halves;
}

}  // namespace

int sf_q4_anyg(const void *blob, const void *x, int x_dtype, void *y, int y_dtype, float *y_f32,
               const void *bias, int bias_dtype, int M, int N, int K, int g, int has_zeros, void *stream);

extern "C" size_t sf_q4_gemm_workspace_bytes(int M, int N, int K, int group_size) {
  if (M <= 0 || N <= 0 || K <= 0 || group_size <= 0 || group_size % 32) return 0;
  const int s = choose_ksplit(M, N, K);
  return s > 1 ? (size_t)s * M * N * sizeof(float) : 0;
}

static int gemm_check(const void *blob, const void *x, int x_dtype, const void *y, int y_dtype,
                      const float *y_f32, const void *bias, int bias_dtype, int M, int N, int K,
                      int group_size) {
  SF_REQUIRE(M > 0 && N > 0 && K > 0 && group_size > 0, SF_EINVAL,
             "invalid shape M=%d N=%d K=%d group_size=%d", M, N, K, group_size);
  SF_REQUIRE(K % group_size == 0, SF_EINVAL, "in_features must be divisible by group_size");
  SF_REQUIRE(blob && x && (y || y_f32), SF_EINVAL, "null pointer argument");
  SF_REQUIRE(x_dtype == SF_F16 || x_dtype == SF_BF16 || x_dtype == SF_F32, SF_EINVAL,
             "bad activation dtype %d", x_dtype);
  SF_REQUIRE(y_dtype == SF_F16 || y_dtype == SF_BF16 || y_dtype == SF_F32, SF_EINVAL,
             "bad output dtype %d", y_dtype);
  SF_REQUIRE(!bias || bias_dtype == SF_F16 || bias_dtype == SF_BF16 || bias_dtype == SF_F32,
             SF_EINVAL, "bad bias dtype %d", bias_dtype);
  SF_REQUIRE(((uintptr_t)blob & 255) == 0 && ((uintptr_t)x & 15) == 0, SF_EINVAL,
             "blob must be 256-byte aligned and X 16-byte aligned");
  return SF_OK;
}

// M rows as batch GEMVs of 8.
static int gemv_slices(const void *blob, const void *x, int x_dtype, void *y, int y_dtype, float *y_f32,
                       const void *bias, int bias_dtype, int M, int N, int K, int group_size,
                       int has_zeros, void *stream) {
  const size_t xsz = x_dtype == SF_F32 ? 4 : 2, ysz = y_dtype == SF_F32 ? 4 : 2;
  for (int m0 = 0; m0 < M; m0 += 8) {
    const int mb = M - m0 < 8 ? M - m0 : 8;
    const int rc = sf_q4_gemv(blob, (const char *)x + (size_t)m0 * K * xsz, x_dtype,
                              y ? (char *)y + (size_t)m0 * N * ysz : nullptr, y_dtype,
                              y_f32 ? y_f32 + (size_t)m0 * N : nullptr,
                              bias && bias == (const void *)y_f32 ? y_f32 + (size_t)m0 * N : bias, bias_dtype,
                              mb, N, K, group_size, has_zeros, stream);
    if (rc) return rc;
  }
  return SF_OK;
}

// The GEMM launch; `partials` leaves a split shape's K-split partials in the
// workspace (no reduce launch, no output) for a consumer that sums them in
// split order itself.
static int q4_gemm_impl(const void *blob, const void *x, int x_dtype, void *y, int y_dtype,
                        float *y_f32, const void *bias, int bias_dtype, int M, int N, int K,
                        int group_size, int has_zeros, void *workspace, size_t workspace_bytes,
                        void *stream, bool partials) {
  const int bad = gemm_check(blob, x, x_dtype, partials ? blob : y, y_dtype, y_f32, bias, bias_dtype, M, N, K,
                             group_size);
  if (bad) return bad;
  if (group_size % 32)  // a group boundary inside an MFMA's k: the any-group-size kernel
    return sf_q4_anyg(blob, x, x_dtype, y, y_dtype, y_f32, bias, bias_dtype, M, N, K, group_size,
                      has_zeros, stream);
  // Up to 16 rows: batch GEMVs of 8 rows (the reference's GEMM is a loop of
  // GEMVs too); sf_q4_matmul chooses between them and the tile kernels.
  // y_f32 passed as the bias too is the GEMV's per-row residual form, not a
  // per-column bias: such a call stays here.
  if (!partials && M <= kGemmGemvRows && !(bias && bias == (const void *)y_f32)) {
    sf_gemv::BlkPlan p;
    if (sf_gemv::plan_blk(M < 8 ? M : 8, N, K, group_size, x_dtype, sf_gemv::PRE_NONE, false, &p))
      return gemv_slices(blob, x, x_dtype, y, y_dtype, y_f32, bias, bias_dtype, M, N, K, group_size,
                         has_zeros, stream);
  }
  BlobLayout L;
  sf_blob_layout(N, K, group_size, has_zeros, &L);
  const int ksplit = choose_ksplit(M, N, K);
  if (ksplit > 1) {
    const size_t need = (size_t)ksplit * M * N * sizeof(float);
    SF_REQUIRE(workspace && workspace_bytes >= need, SF_EINVAL,
               "GEMM workspace too small: %zu < %zu", workspace_bytes, need);
  }
  const int nsteps = (K + BK - 1) / BK;
  const int steps_per_split = (nsteps + ksplit - 1) / ksplit;
  const uint8_t *w = (const uint8_t *)blob;
  const f16 *st = (const f16 *)(w + L.s_off);
  const uint8_t *zt = has_zeros ? w + L.z_off : nullptr;
  hipStream_t s = (hipStream_t)stream;
  dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM, ksplit);
  float *part = (float *)workspace;
  // 16-byte output stores need rows of whole 16-byte multiples and aligned bases
  const bool vec = N % 8 == 0 && ((uintptr_t)y & 15) == 0 && ((uintptr_t)y_f32 & 15) == 0 &&
                   ((uintptr_t)part & 15) == 0;
  if (x_dtype != SF_F32 && rows_takes(M, K, group_size, x_dtype)) {
    int rb, kw;
    rows_tile(M, N, K, x_dtype, ksplit, &rb, &kw);
    const int rr = rows_run(rows_args(blob, x, y, y_f32, bias, part, y_dtype, bias_dtype, M, N, K, group_size,
                                      has_zeros, ksplit, vec),
                            x_dtype, has_zeros, rb, kw, s);
    if (rr) return rr;
  } else {
#define SF_GEMM_LAUNCH(XD, AS)                                                               \
  do {                                                                                       \
    if (group_size == 32)                                                                    \
      k_q4_gemm<XD, AS, 0><<<grid, NTHREADS, 0, s>>>(w, st, zt, x, y, y_dtype, y_f32, bias,  \
                                                     bias_dtype, part, M, N, K, L.G,         \
                                                     group_size, ksplit, steps_per_split, vec); \
    else if (group_size == 64)                                                               \
      k_q4_gemm<XD, AS, 1><<<grid, NTHREADS, 0, s>>>(w, st, zt, x, y, y_dtype, y_f32, bias,  \
                                                     bias_dtype, part, M, N, K, L.G,         \
                                                     group_size, ksplit, steps_per_split, vec); \
    else if (group_size % 64)                                                                \
      k_q4_gemm<XD, AS, 3><<<grid, NTHREADS, 0, s>>>(w, st, zt, x, y, y_dtype, y_f32, bias,  \
                                                     bias_dtype, part, M, N, K, L.G,         \
                                                     group_size, ksplit, steps_per_split, vec); \
    else                                                                                     \
      k_q4_gemm<XD, AS, 2><<<grid, NTHREADS, 0, s>>>(w, st, zt, x, y, y_dtype, y_f32, bias,  \
                                                     bias_dtype, part, M, N, K, L.G,         \
                                                     group_size, ksplit, steps_per_split, vec); \
  } while (0)
#define SF_GEMM_X(AS)                                  \
  do {                                                 \
    if (x_dtype == SF_BF16) SF_GEMM_LAUNCH(SF_BF16, AS); \
    else if (x_dtype == SF_F16) SF_GEMM_LAUNCH(SF_F16, AS); \
    else SF_GEMM_LAUNCH(SF_F32, AS);                   \
  } while (0)
  if (has_zeros) SF_GEMM_X(true);
  else SF_GEMM_X(false);
#undef SF_GEMM_X
#undef SF_GEMM_LAUNCH
  }
  int rc = sf_check_launch(partials ? "sf_q4_gemm_partials" : "sf_q4_gemm");
  if (rc || ksplit == 1 || partials) return rc;
  return splitk_reduce(part, y, y_dtype, y_f32, bias, bias_dtype, M, N, ksplit, vec, s);
}

extern "C" int sf_q4_gemm(const void *blob, const void *x, int x_dtype, void *y, int y_dtype,
                          float *y_f32, const void *bias, int bias_dtype, int M, int N, int K,
                          int group_size, int has_zeros, void *workspace, size_t workspace_bytes,
                          void *stream) {
  return q4_gemm_impl(blob, x, x_dtype, y, y_dtype, y_f32, bias, bias_dtype, M, N, K, group_size,
                      has_zeros, workspace, workspace_bytes, stream, false);
}

extern "C" int sf_q4_gemm_splits(int M, int N, int K, int group_size) {
  if (M <= 0 || N <= 0 || K <= 0 || group_size <= 0 || K % group_size || group_size % 32) return 0;
  return choose_ksplit(M, N, K);
}

extern "C" int sf_q4_gemm_partials(const void *blob, const void *x, int x_dtype, int M, int N,
                                   int K, int group_size, int has_zeros, void *workspace,
                                   size_t workspace_bytes, void *stream) {
  const int s = sf_q4_gemm_splits(M, N, K, group_size);
  SF_REQUIRE(s > 1, SF_EINVAL,
             "sf_q4_gemm_partials: M=%d N=%d K=%d group_size=%d runs unsplit (use sf_q4_gemm)", M,
             N, K, group_size);
  return q4_gemm_impl(blob, x, x_dtype, nullptr, SF_F32, nullptr, nullptr, SF_F32, M, N, K,
                      group_size, has_zeros, workspace, workspace_bytes, stream, true);
}

// The larger of the plans that has_zeros chooses between (a residual needs none).
extern "C" size_t sf_q4_matmul_workspace_bytes(int M, int N, int K, int group_size, int x_dtype) {
  if (M <= 0 || N <= 0 || K <= 0 || group_size <= 0 || K % group_size) return 0;
  if (x_dtype != SF_F16 && x_dtype != SF_BF16 && x_dtype != SF_F32) return 0;
  size_t bytes = 0;
  for (int i = 0; i < (M <= kGemmGemvRows ? 2 : 1); ++i) {
    MatmulPlan p;
    matmul_plan(M, N, K, group_size, i & 1, x_dtype, false, &p);
    if (p.bytes > bytes) bytes = p.bytes;
  }
  return bytes;
}

extern "C" size_t sf_q4_rows_workspace_bytes(int max_rows, int N, int K, int group_size, int x_dtype) {
  size_t bytes = 0;
  for (int m = 0; m < max_rows; ++m) {
    const int M = m + 1;
    const size_t a = sf_q4_matmul_workspace_bytes(M, N, K, group_size, x_dtype);
    const size_t b = sf_q4_gemm_workspace_bytes(M, N, K, group_size);
    if (a > bytes) bytes = a;
    if (b > bytes) bytes = b;
  }
  return bytes;
}

extern "C" int sf_q4_matmul(const void *blob, const void *x, int x_dtype, void *y, int y_dtype,
                            float *y_f32, const void *bias, int bias_dtype, int M, int N, int K,
                            int group_size, int has_zeros, void *workspace, size_t workspace_bytes,
                            void *stream) {
  const int bad = gemm_check(blob, x, x_dtype, y, y_dtype, y_f32, bias, bias_dtype, M, N, K, group_size);
  if (bad) return bad;
  MatmulPlan p;
  matmul_plan(M, N, K, group_size, has_zeros, x_dtype, bias && bias == (const void *)y_f32, &p);
  if (p.route == MatmulPlan::GEMV)
    return gemv_slices(blob, x, x_dtype, y, y_dtype, y_f32, bias, bias_dtype, M, N, K, group_size,
                       has_zeros, stream);
  if (p.route == MatmulPlan::GEMM)
    return sf_q4_gemm(blob, x, x_dtype, y, y_dtype, y_f32, bias, bias_dtype, M, N, K, group_size,
                      has_zeros, workspace, workspace_bytes, stream);
  SF_REQUIRE(p.bytes == 0 || (workspace && workspace_bytes >= p.bytes), SF_EINVAL,
             "matmul workspace too small: %zu < %zu", workspace_bytes, p.bytes);
  SF_REQUIRE(p.bytes == 0 || ((uintptr_t)workspace & 15) == 0, SF_EINVAL,
             "matmul workspace must be 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  if (x_dtype == SF_F32) x = split_rows((const float *)x, (char *)workspace + p.parts, M, K, s);
  const bool vec = N % 8 == 0 && ((uintptr_t)y & 15) == 0 && ((uintptr_t)y_f32 & 15) == 0;
  const int rr = rows_run(rows_args(blob, x, y, y_f32, bias, (float *)workspace, y_dtype, bias_dtype, M, N, K,
                                    group_size, has_zeros, p.ks, vec),
                          x_dtype, has_zeros, p.rb, p.kw, s);
  if (rr) return rr;
  const int rc = sf_check_launch("sf_q4_matmul");
  if (rc || p.ks == 1) return rc;
  return splitk_reduce((const float *)workspace, y, y_dtype, y_f32, bias, bias_dtype, M, N, p.ks, vec, s);
}

// One k_q4_gemm_rows launch for several weights on the same rows. Taken where
// they go to the rows kernel with no K split (a split's partials have one
// weight's layout), and no weight's K sum runs longer than in a launch of its
// own, which splits K or has two K groups for a small weight (1024 x 4096, 300
// rows: error against 64 bits 7.4e-8 by itself, 1.07e-7 in an unsplit group);
// else the caller runs them one by one.
static bool group_plan(int op, int n, const int *Ns, int M, int K, int g, int xdt, MatmulPlan *p, int *tiles) {
  if (n < 1 || n > 3 || !Ns || M <= kGemmGemvRows || K <= 0 || g <= 0 || K % g || !rows_takes(M, K, g, xdt))
    return false;
  if (op == SF_GROUP_SWIGLU && (n > 2 || (n == 1 ? Ns[0] % 2 : Ns[0] != Ns[1]))) return false;
  long long t = 0, cols = 0;
  for (int i = 0; i < n; ++i) {
    if (Ns[i] <= 0) return false;
    t += (Ns[i] + 127) / 128;
    cols += Ns[i];
  }
  if (op == SF_GROUP_SWIGLU) t = (cols / 2 + 63) / 64;
  if (t > (1 << 20) || cols > INT_MAX) return false;
  *tiles = (int)t;
  matmul_plan(M, *tiles * 128, K, g, false, xdt, false, p);
  if (p->route != MatmulPlan::ROWS || p->ks != 1) return false;
  for (int i = 0; i < n; ++i) {
    MatmulPlan own;
    matmul_plan(M, Ns[i], K, g, false, xdt, false, &own);
    if (own.ks != 1 || own.kw > p->kw) return false;
  }
  return true;
}

extern "C" int sf_q4_matmul_group_supported(int op, int n, const int *Ns, int M, int K, int group_size,
                                            int x_dtype, size_t *workspace_bytes) {
  MatmulPlan p;
  int tiles;
  if (op != SF_GROUP_CONCAT && op != SF_GROUP_SWIGLU) return 0;
  if (x_dtype != SF_F16 && x_dtype != SF_BF16 && x_dtype != SF_F32) return 0;
  if (!group_plan(op, n, Ns, M, K, group_size, x_dtype, &p, &tiles)) return 0;
  if (workspace_bytes) *workspace_bytes = p.bytes;
  return 1;
}

extern "C" int sf_q4_matmul_group(int op, int n, const void *const *blobs, const int *Ns,
                                  const void *const *biases, const int *bias_dtypes, const void *x,
                                  int x_dtype, void *y, int y_dtype, int M, int K, int group_size,
                                  int has_zeros, void *workspace, size_t workspace_bytes, void *stream) {
  size_t need = 0;
  SF_REQUIRE(blobs && Ns && sf_q4_matmul_group_supported(op, n, Ns, M, K, group_size, x_dtype, &need),
             SF_EUNSUPPORTED, "no grouped launch for op=%d n=%d M=%d K=%d group_size=%d", op, n, M, K, group_size);
  SF_REQUIRE(op == SF_GROUP_CONCAT || !biases, SF_EUNSUPPORTED, "the SwiGLU form takes no biases");
  SF_REQUIRE(!biases || bias_dtypes, SF_EINVAL, "null pointer argument");
  int width = 0;
  for (int i = 0; i < n; ++i) {
    const void *bias = biases ? biases[i] : nullptr;
    const int bad = gemm_check(blobs[i], x, x_dtype, y, y_dtype, nullptr, bias, bias ? bias_dtypes[i] : 0, M,
                               Ns[i], K, group_size);
    if (bad) return bad;
    width += Ns[i];
  }
  SF_REQUIRE(need == 0 || (workspace && workspace_bytes >= need && ((uintptr_t)workspace & 15) == 0), SF_EINVAL,
             "matmul workspace too small or not 16-byte aligned: %zu < %zu", workspace_bytes, need);
  MatmulPlan p;
  int tiles;
  group_plan(op, n, Ns, M, K, group_size, x_dtype, &p, &tiles);
  hipStream_t s = (hipStream_t)stream;
  if (x_dtype == SF_F32) x = split_rows((const float *)x, workspace, M, K, s);
  sf_gemm::RowsGroupArgs a{rows_args(blobs[0], x, y, nullptr, nullptr, nullptr, y_dtype, 0, M, Ns[0], K, group_size,
                                     has_zeros, 1, true),
                           {kNoSeg, kNoSeg},
                           false};
  a.tiles = tiles;
  if (op == SF_GROUP_SWIGLU) {
    const int I = n == 1 ? Ns[0] / 2 : Ns[0];
    a.swiglu = true;
    a.ld = I;
    a.more[0] = n == 1 ? a.seg : rows_seg(blobs[1], nullptr, 0, I, K, group_size, has_zeros, 0, 0);
    a.seg.N = a.more[0].N = I;
    a.more[0].n_off = n == 1 ? I : 0;
  } else {
    a.ld = width;
    int tile = 0, col = 0;
    for (int i = 0; i < n; ++i) {
      (i ? a.more[i - 1] : a.seg) = rows_seg(blobs[i], biases ? biases[i] : nullptr, bias_dtypes && biases ? bias_dtypes[i] : 0,
                          Ns[i], K, group_size, has_zeros, tile, col);
      tile += (Ns[i] + 127) / 128;
      col += Ns[i];
      a.vec = a.vec && Ns[i] % 8 == 0;
    }
  }
  a.vec = a.vec && a.ld % 8 == 0 && ((uintptr_t)y & 15) == 0;
  const int rr = rows_run(a, x_dtype, has_zeros, p.rb, p.kw, s, &a);
  return rr ? rr : sf_check_launch("sf_q4_matmul_group");
}
