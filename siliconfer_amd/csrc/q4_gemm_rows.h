// q4_gemm_rows.h — int4 prefill GEMM whose waves own 32 columns and every row
// of the tile (gfx950).
#pragma once

#include <atomic>
#include <type_traits>

#include "q4_gemv_blk.h"
#include "sf_common.h"

namespace sf_gemm {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;

// Wait until at most n vector-memory operations of this wave are outstanding
// (gfx9 s_waitcnt: vmcnt in bits 3:0 and 15:14; exp and lgkm left at their maxima).
#define SF_WAIT_VM(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | (7 << 4) | (15 << 8))
// Wait for this wave's LDS operations (vm and exp left at their maxima).
#define SF_WAIT_LGKM0() __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4))

// One weight of a call (n_off: its first row inside the blob).
struct RowsSeg {
  const uint8_t *wq;   // blob: codes
  const f16 *st;       // scales
  const uint8_t *zt;   // zero-points (asymmetric)
  const void *bias;
  int bdt, N, n_off, tile, col;  // tile: its first column tile; col: its first output column
};

struct RowsArgs {
  RowsSeg seg;
  const void *x;       // activations [M][K] (fp32: the bf16 high rows, then the low rows)
  void *y;
  float *y32;
  float *part;
  int ydt, M, K, ld, G, g, ksplit, pairs_per_split, tiles;  // ld: outputs a row
  bool vec;
};

// Several weights (unused: tile past every column tile), or swiglu: seg gate,
// more[0] up, y = silu(gate) * up. A single weight's kernel is not passed these.
struct RowsGroupArgs : RowsArgs {
  RowsSeg more[2];
  bool swiglu;
};

// One output value's bias.
__device__ __forceinline__ float bias_at(const void *bias, int bdt, int c) {
  return bdt == SF_F32 ? ((const float *)bias)[c]
         : bdt == SF_F16 ? (float)((const f16 *)bias)[c]
                         : sf_bf16_to_f32(((const uint16_t *)bias)[c]);
}

// Write 8 consecutive outputs (nv of them in range) to the fp32 copy and / or
// the output in its dtype; 16-byte stores when `vec` (row pitch and bases
// allow it) and all 8 are in range.
__device__ __forceinline__ void store8(const float (&v)[8], int nv, bool vec, float *y32, void *Y,
                                       int ydt, size_t idx) {
  auto f32 = [&](float *d) {
    if (vec && nv == 8) {
      ((float4_t *)d)[0] = float4_t{v[0], v[1], v[2], v[3]};
      ((float4_t *)d)[1] = float4_t{v[4], v[5], v[6], v[7]};
    } else {
      for (int e = 0; e < nv; ++e) d[e] = v[e];
    }
  };
  if (y32) f32(y32 + idx);
  if (!Y) return;
  if (ydt == SF_F32) {
    f32((float *)Y + idx);
    return;
  }
  uint16_t b[8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    b[e] = ydt == SF_BF16 ? sf_f32_to_bf16(v[e]) : sf_bitcast<uint16_t>((f16)v[e]);
  uint16_t *d = (uint16_t *)Y + idx;
  if (vec && nv == 8) {
    u32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = (uint32_t)b[2 * e] | ((uint32_t)b[2 * e + 1] << 16);
    *(u32x4 *)d = w;
  } else {
    for (int e = 0; e < nv; ++e) d[e] = b[e];
  }
}

__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
  const float2_t f = {a, b};
  return sf_bitcast<uint32_t>(__builtin_convertvector(f, bf16x2_t));
}

// One byte of v to fp32 in one instruction (SDWA source selects): the byte's
// signed value, or its low nibble as a two's complement int4 over 16.
#define SF_SBYTE_F32(out, v, B)                                                                   \
  asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_" #B \
      : "=v"(out)                                                                              \
      : "v"(v))
#define SF_NIB_F32(out, v, B)                                                                  \
  asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_" #B \
      : "=v"(out)                                                                           \
      : "v"(v))

// The bf16 B operand of 8 codes (one dword of a unit lane; nibble i is k
// element 2 i for i < 4, else 2 (i - 4) + 1). Symmetric: (code - 8) / 16, the
// flipped nibble read as two's complement, 14 VALU instructions (the 16 goes
// into the group's scale, exactly). With a zero-point, 19: the nibbles go one to
// a byte, ((b ^ 0x80) - z) ^ 0x80 makes the byte the two's complement of b - z
// with no borrow between bytes (0x80 + b - z stays in 0x71..0x8F), and each
// byte converts in one instruction; code - z is exact in bf16.
template <bool ASYM>
__device__ __forceinline__ u32x4 dequant_bf16(uint32_t d, uint32_t z) {
  float e0, e1, e2, e3, o0, o1, o2, o3;
  if constexpr (ASYM) {
    const uint32_t zz = z * 0x01010101u;
    const uint32_t e = (((d & 0x0F0F0F0Fu) ^ 0x80808080u) - zz) ^ 0x80808080u;
    const uint32_t o = ((((d >> 4) & 0x0F0F0F0Fu) ^ 0x80808080u) - zz) ^ 0x80808080u;
    SF_SBYTE_F32(e0, e, 0);
    SF_SBYTE_F32(e1, e, 1);
    SF_SBYTE_F32(e2, e, 2);
    SF_SBYTE_F32(e3, e, 3);
    SF_SBYTE_F32(o0, o, 0);
    SF_SBYTE_F32(o1, o, 1);
    SF_SBYTE_F32(o2, o, 2);
    SF_SBYTE_F32(o3, o, 3);
  } else {
    const uint32_t e = d ^ 0x88888888u, o = e >> 4;
    SF_NIB_F32(e0, e, 0);
    SF_NIB_F32(e1, e, 1);
    SF_NIB_F32(e2, e, 2);
    SF_NIB_F32(e3, e, 3);
    SF_NIB_F32(o0, o, 0);
    SF_NIB_F32(o1, o, 1);
    SF_NIB_F32(o2, o, 2);
    SF_NIB_F32(o3, o, 3);
  }
  return u32x4{pk_bf16(e0, e2), pk_bf16(o0, o2), pk_bf16(e1, e3), pk_bf16(o1, o3)};
}

// 16 bytes per lane from a buffer resource straight into LDS (lane i's bytes
// at dst + 16 i; past the resource: zeros).
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t rs, uint8_t *dst, uint32_t voff,
                                           uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)dst, 16, voff, soff, 0, 0);
}

constexpr int R_BN = 128, R_BK = 64, R_SLOTS = 4, R_PITCH = R_BN + 4;
// dynamic LDS: per K group of waves, four slots of the tile's A rows for one
// K step; reused for the other groups' sums and the output
template <int XM, int RB, int KW>
constexpr int rows_lds_bytes() {
  const int slots = KW * R_SLOTS * RB * (XM == SF_F32 ? 2 : 1) * 32 * 128;
  const int sums = (KW - 1) * RB * 16 * 1024, out = (RB > 1 ? 2 : 1) * 32 * R_PITCH * 4;
  return slots > sums ? (slots > out ? slots : out) : (sums > out ? sums : out);
}

// Y = X . dequant(W)^T: a workgroup takes 32 RB rows by 128 columns, four waves
// of 32 columns each over all its rows (v_mfma_f32_32x32x16).
//  * W never touches LDS: a wave loads its own columns' codes (two 16-byte
//    loads a lane per 128 k, the blob's order) two pairs of steps ahead and
//    turns them into the exact integers q - z in registers, once for all RB row
//    blocks, so no code is converted twice in a workgroup and the conversion
//    (9 / 14 / 19 VALU instructions per 8 codes, fp16 / bf16 / bf16 with
//    zero-points) spreads over RB MFMAs.
//  * X goes straight into LDS (buffer loads ... lds), K steps of 64, four
//    slots, three steps ahead, one bare barrier a step in front of the last row
//    block, whose operands are already in registers.
//  * Each scale group's fp32 partial is folded with its fp16 scale once per
//    group (y = sum_g s_g sum_k x_k (q_k - z)), one row block behind its MFMAs.
//    fp32 activations: X holds bf16 high rows, then low rows; two MFMAs an
//    operand.
//  * Up to three weights a launch on the same rows (q|k|v): column tiles of each,
//    side by side in one output. A small weight's tiles fill the last round of
//    a large one's, the rows are split into halves once and nothing
//    concatenates afterwards: the 8B attention layer over 1500 rows 415 -> 350 us,
//    its MLP over 333 rows 318 -> 297 (fp32 both). swiglu: waves 0, 1 take 64 gate columns and waves
//    2, 3 the same columns of up, and the output tile is silu(gate) * up.
//  * KW = 2: a second set of four waves takes the other half of the K steps and
//    the sums meet in LDS (two waves a SIMD without a second output tile).
// The kernel it replaced staged converted codes through LDS with separate
// convert waves, 128 x 128 tiles only. Measured (us a call, before -> after;
// fp32 results but for the first): 2048 rows on 4096 x 11008, bf16 223 -> 164
// (1126 TFLOP/s; torch's bf16 matmul of 8192^3 reaches 1308 on this card), fp16
// 234 -> 173; 512 on 11008 x 4096, fp16 85 -> 58; 48 there 26.1 -> 16.4; 512 on
// 4864 x 896, bf16 with zero-points 15.9 -> 14.3, fp16 15.3 -> 13.4. fp32 against
// the in-kernel split of k_q4_gemm: 333 on 11008 x 4096 189 -> 79. Behind that
// kernel by 1-7%: bf16 with zero-points at K of 8192 and more and 96-333 rows
// (333 on 4096 x 14336: 74.4 -> 78.0), and 7 units of K on wide weights and
// 200-333 rows (333 on 9728 x 896 15.5 -> 16.2: two K groups take 8 units' time).
// What bounds it at the large end (2048 rows on 4096 x 11008, bf16, counters):
// MFMAs busy 55% of the SIMD cycles and VALU issue 43%, no bank conflicts, at
// the 1.9 GHz that the card holds under this mix. Tried and not kept: eight row
// blocks (one wave a SIMD: 234), slot rings of eight with four code sets and a
// pinned MFMA / VALU interleave (4% slower over the sweep), 256 columns a
// workgroup (the same).
template <int XM, bool ASYM, int GK, int RB, int KW, bool GRP>
__global__ void __launch_bounds__(256 * KW, KW == 1 ? 2 : 1)
k_q4_gemm_rows(const std::conditional_t<GRP, RowsGroupArgs, RowsArgs> a) {
  constexpr bool SPLIT = XM == SF_F32, F16 = XM == SF_F16;
  constexpr int NF = RB * (SPLIT ? 2 : 1);  // 32-row blocks in LDS
  constexpr int STAGE = NF * 32 * 128;
  constexpr int NG = GK == 0 ? 2 : 1;       // groups per K step
  constexpr int NSP = GK == 0 ? 4 : GK == 1 ? 2 : 1;  // groups per pair of steps
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);  // the wave's columns
  const int kg = KW == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);  // its K group
  uint8_t *const smem = lds + kg * R_SLOTS * STAGE;
  const int l32 = lane & 31, h = lane >> 5;
  const int m0 = blockIdx.y * (32 * RB), bx = blockIdx.x;
  const int split = blockIdx.z;
  const int M = a.M, K = a.K, G = a.G;
  // The wave's weight (one for the workgroup but for swiglu). Every candidate is
  // read with the other arguments and selected: an indexed argument would be a
  // second memory round trip in front of the first load (512 rows on 4864 x 896
  // 12.9 us against 12.2, and 37 rows on 11008 x 4096 16.3 against 15.8; 15.6
  // with one weight's arguments only, so that has its own code).
  RowsSeg sg = a.seg;
  bool swiglu = false;
  if constexpr (GRP) {
    swiglu = a.swiglu;
    const bool s1st = swiglu ? wave >= 2 : bx >= a.more[0].tile, s2nd = !swiglu && bx >= a.more[1].tile;
#define SF_SEG(f) sg.f = s2nd ? a.more[1].f : s1st ? a.more[0].f : sg.f
    SF_SEG(wq); SF_SEG(st); SF_SEG(zt); SF_SEG(bias); SF_SEG(bdt); SF_SEG(N); SF_SEG(n_off); SF_SEG(tile); SF_SEG(col);
#undef SF_SEG
  } else {
    sg.n_off = sg.tile = sg.col = 0;
  }
  const int N = sg.N;
  const int nblk = (K + 127) >> 7;
  // this wave's K steps [s0, s1): the split's pairs dealt to the K groups in
  // contiguous runs; every group runs nst steps (those past s1 add zeros)
  const int p0 = split * a.pairs_per_split, p1 = min(p0 + a.pairs_per_split, nblk);
  const int ppg = (max(p1 - p0, 0) + KW - 1) / KW;
  const int nst = 2 * ppg;
  const int s0 = 2 * (p0 + kg * ppg);
  const int s1 = min(min(s0 + nst, 2 * p1), (K + R_BK - 1) / R_BK);

  // ---- A rows: wave w loads LDS rows 8 (w NF + i) .. + 7, i < NF, 128 bytes
  // (64 k) a row; row r's 16-byte piece p sits in place p ^ ((r / 2) % 8), so
  // that 16 rows of one piece (two rows span the 64 banks) touch every bank
  // once; each lane fetches the piece that belongs in its place. Rows past M
  // repeat row M - 1 (never stored). Rows and lim keep every load inside X. The
  // resource ends 1 KB behind it (at most at kPastEnd): the range check takes the
  // vector offset against the size minus the scalar offset (step * 128), which
  // must not wrap where one row of 2 K bytes is all there is and the last
  // prefetch is up to 2 (K / 128 + 1) + 3 steps in (holding the scalar offset
  // back instead costs the loop 1%).
  constexpr uint32_t kPastEnd = 0x80000000u;
  const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
      (void *)a.x, 0, min((uint32_t)((SPLIT ? 2 : 1) * M * K * 2) + 1024u, kPastEnd), 0x00020000);
  uint32_t voff[NF];
  int lim[NF < 2 ? 1 : 2];  // K steps whose piece lies inside K (a last step of 32 k has four)
#pragma unroll
  for (int i = 0; i < NF; ++i) {
    const int lr = 8 * (wave * NF + i) + (lane >> 3);
    const int piece = (lane & 7) ^ ((lr >> 1) & 7);
    const int half = lr / (32 * RB);
    const int row = min(m0 + lr - half * 32 * RB, M - 1) + half * M;
    voff[i] = (uint32_t)row * (uint32_t)(K * 2) + piece * 16;
    if (i < 2) lim[i] = (K + R_BK - 1 - piece * 8) / R_BK;  // (the piece alternates with i)
  }
#pragma unroll
  for (int i = 0; i < (NF < 2 ? 1 : 2); ++i) lim[i] = min(lim[i], s1);
  // steps past the last read past the resource: zeros, no memory access
  auto issue = [&](int step, int slot) {
#pragma unroll
    for (int i = 0; i < NF; ++i)
      load_lds16(xrs, smem + slot * STAGE + (wave * NF + i) * 1024,
                 step < lim[NF < 2 ? 0 : i & 1] ? voff[i] : kPastEnd, step * (R_BK * 2));
  };

  // ---- B: the lane's column; a pair of steps is one unit (128 k)
  const int wc = swiglu ? 64 * bx + 32 * (wave & 1) : R_BN * (bx - sg.tile) + 32 * wave;
  const int n = min(wc + l32, N - 1) + sg.n_off;
  const uint8_t *wp = sg.wq + (size_t)(n >> 4) * nblk * 1024 + (h * 16 + (n & 15)) * 16;
  const f16 *sp = sg.st + (size_t)(n >> 3) * G * 8 + (n & 7);
  const uint8_t *zp = ASYM ? sg.zt + (size_t)(n >> 3) * G * 4 + ((n & 7) >> 1) : nullptr;
  const int zsh = 4 * (n & 1);
  struct Pair {
    u32x4 lo, hi;
    f16 s[NSP];
    uint8_t z[ASYM ? NSP : 1];
  };
  const int gpp = GK == 2 ? a.g >> 7 : 1;  // pairs per group
  auto load_pair = [&](int pair, Pair &p) {
    const int u = min(pair, nblk - 1);  // past the end: the last unit again (its operands meet zeros)
    p.lo = *(const u32x4 *)(wp + (size_t)u * 1024);
    p.hi = *(const u32x4 *)(wp + (size_t)u * 1024 + 512);
#pragma unroll
    for (int q = 0; q < NSP; ++q) {
      const int gi = min(GK == 2 ? u / gpp : u * NSP + q, G - 1);
      p.s[q] = sp[(size_t)gi * 8];
      if constexpr (ASYM) p.z[q] = zp[(size_t)gi * 4];
    }
  };
  const sf_gemv::DequantConsts dk;
  // slice kk's operand of step parity `par` of a pair
  auto convert = [&](const Pair &p, int par, int kk) -> u32x4 {
    const uint32_t d = (kk & 1) ? p.hi[2 * par + (kk >> 1)] : p.lo[2 * par + (kk >> 1)];
    uint32_t z = 8u;
    if constexpr (ASYM) z = ((uint32_t)p.z[GK == 0 ? 2 * par + (kk >> 1) : GK == 1 ? par : 0] >> zsh) & 15u;
    if constexpr (F16) return sf_gemv::dequant_f16(d, z, dk);
    else return dequant_bf16<ASYM>(d, z);
  };
  constexpr float SMUL = F16 || ASYM ? 1.f : 16.f;
  auto scale = [&](const Pair &p, int par, int q) -> float {
    return SMUL * (float)p.s[GK == 0 ? 2 * par + q : GK == 1 ? par : 0];
  };

  const float16_t zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f,
                            0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float16_t acc[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) acc[r] = zero16;

  // A operand of row block rb, slice kk: row l32, piece 2 kk + h
  uint32_t aoff[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) aoff[kk] = l32 * 128 + (((2 * kk + h) ^ ((l32 >> 1) & 7)) << 4);
  struct AOps {
    u32x4 v[SPLIT ? 2 : 1][4];
  };
  auto read_a = [&](int slot, int rb, AOps &o) {
#pragma unroll
    for (int hl = 0; hl < (SPLIT ? 2 : 1); ++hl)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        o.v[hl][kk] = *(const u32x4 *)(smem + slot * STAGE + (hl * RB + rb) * 4096 + aoff[kk]);
  };
  auto mfma = [&](const u32x4 &x, const u32x4 &w, const float16_t &c) -> float16_t {
    if constexpr (F16)
      return __builtin_amdgcn_mfma_f32_32x32x16_f16(sf_bitcast<half8_t>(x), sf_bitcast<half8_t>(w), c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_32x32x16_bf16(sf_bitcast<bf16x8_t>(x), sf_bitcast<bf16x8_t>(w), c, 0, 0, 0);
  };

  Pair pr[2];
  u32x4 b[2][4];
  AOps af[2];
  // Group partials. GK 0 / 1 (a step ends its groups): two sets, a row block's
  // fold one block behind its MFMAs. GK 2: one per row block, folded in the
  // odd steps (a group is a whole number of pairs of steps).
  constexpr int NP = GK == 2 ? RB : 2;
  float16_t gp[NP][NG];
  float sc[2][NG] = {};  // the groups' scales (by step parity)
  auto fold = [&](int r, const float16_t (&g)[NG], const float (&f)[NG]) {
#pragma unroll
    for (int q = 0; q < NG; ++q)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[r][e] = fmaf(g[q][e], f[q], acc[r][e]);
  };

  if (nst > 0) {
    load_pair(s0 >> 1, pr[0]);
    load_pair((s0 >> 1) + 1, pr[1]);
    issue(s0, 0);
    issue(s0 + 1, 1);
    issue(s0 + 2, 2);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) b[0][kk] = convert(pr[0], 0, kk);
    SF_WAIT_VM(2 * NF);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read_a(0, 0, af[0]);
#pragma unroll
    for (int r = 0; r < NP; ++r)
#pragma unroll
      for (int q = 0; q < NG; ++q) gp[r][q] = zero16;
    for (int j = 0; j < nst; j += 4) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (u == 2 && j + 2 >= nst) break;
        const int step = s0 + j + u, par = u & 1;
#pragma unroll
        for (int q = 0; q < NG; ++q) sc[par][q] = step < s1 ? scale(pr[u >> 1], par, q) : 0.f;
        issue(step + 3, (u + 3) & 3);
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          const int t = (u * RB + r) & 1;
          if (r == RB - 1) {
            SF_WAIT_VM(2 * NF);
            SF_WAIT_LGKM0();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            read_a((u + 1) & 3, 0, af[t ^ 1]);
          } else {
            read_a(u, r + 1, af[t ^ 1]);
          }
          const int gi = GK == 2 ? r : t;
          if (GK == 2 && !par && r == 0) fold(RB - 1, gp[RB - 1], sc[1]);
#pragma unroll
          for (int kk = 0; kk < 4; ++kk) {
            const int q = GK == 0 ? kk >> 1 : 0;
            const bool open = GK == 0 ? !(kk & 1) : kk == 0 && (GK == 1 || !par);
            gp[gi][q] = mfma(af[t].v[0][kk], b[par][kk], open ? zero16 : gp[gi][q]);
            if constexpr (SPLIT) gp[gi][q] = mfma(af[t].v[1][kk], b[par][kk], gp[gi][q]);
          }
          // fold the row block before this one (r = 0: the last one of the step
          // before; all zero in front of the first step)
          if constexpr (GK != 2) {
            if (r == 0) fold(RB - 1, gp[t ^ 1], sc[par ^ 1]);
            else fold(r - 1, gp[t ^ 1], sc[par]);
          } else if (par && r > 0) {
            fold(r - 1, gp[r - 1], sc[1]);
          }
          // the next step's B operands, spread over the row blocks
#pragma unroll
          for (int kk = 0; kk < 4; ++kk)
            if (kk * RB / 4 == r)
              b[par ^ 1][kk] = par ? convert(pr[(u >> 1) ^ 1], 0, kk) : convert(pr[u >> 1], 1, kk);
        }
        if (par) load_pair((step >> 1) + 2, pr[u >> 1]);
      }
    }
    fold(RB - 1, gp[GK == 2 ? RB - 1 : 1], sc[1]);  // the last row block of the last (odd) step
  }

  // ---- every load landed and every wave done with the slots: the K groups'
  // sums, added in group order
  SF_WAIT_VM(0);
  __syncthreads();
  if constexpr (KW > 1) {
    float *sums = (float *)lds;
    const int t = tid & 255;
    if (kg > 0) {
#pragma unroll
      for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int e = 0; e < 16; ++e) sums[(((kg - 1) * RB + r) * 16 + e) * 256 + t] = acc[r][e];
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int q = 0; q < KW - 1; ++q)
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[r][e] += sums[((q * RB + r) * 16 + e) * 256 + t];
    }
    __syncthreads();  // sums read before the output is staged over them
  }

  // ---- output, one 32-row block at a time through LDS (two blocks in turn):
  // whole 128-column row segments, 8 columns a thread
  const int n0 = R_BN * (bx - sg.tile), cl = (tid & 15) * 8, col = n0 + cl, nv = min(8, N - col);
  float *y32 = a.y32;
  void *y = a.y;
  float bv[8] = {};
  if (a.ksplit > 1) {
    y32 = a.part + (size_t)split * M * N;  // one weight: ld = N
    y = nullptr;
  } else if (!swiglu && sg.bias) {
    for (int e = 0; e < 8; ++e) bv[e] = bias_at(sg.bias, sg.bdt, min(col + e, N - 1));
  }
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    float *ot = (float *)lds + (r & 1) * 32 * R_PITCH;
    if (kg == 0) {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        ot[(8 * (e >> 2) + 4 * h + (e & 3)) * R_PITCH + 32 * wave + l32] = acc[r][e];
    }
    __syncthreads();
    if (swiglu) {  // columns 0..63 of the tile: gate, 64..127: up
      const int rl = tid >> 3, sl = (tid & 7) * 8, sc0 = 64 * bx + sl, sv = min(8, N - sc0);
      const int row = m0 + 32 * r + rl;
      if (rl < 32 && row < M && sv > 0) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
          v[e] = sf_silu_mul(ot[rl * R_PITCH + sl + e], ot[rl * R_PITCH + 64 + sl + e]);
        store8(v, sv, a.vec, y32, y, a.ydt, (size_t)row * a.ld + sc0);
      }
      continue;
    }
#pragma unroll
    for (int rl = tid >> 4; rl < 32; rl += 16 * KW) {
      const int row = m0 + 32 * r + rl;
      const float4_t x0 = *(const float4_t *)(ot + rl * R_PITCH + cl);
      const float4_t x1 = *(const float4_t *)(ot + rl * R_PITCH + cl + 4);
      float v[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = x0[e] + bv[e];
        v[4 + e] = x1[e] + bv[4 + e];
      }
      if (row < M && nv > 0) store8(v, nv, a.vec, y32, y, a.ydt, (size_t)row * (GRP ? a.ld : N) + sg.col + col);
    }
  }
}

template <int XM, bool ASYM, int GK, int RB, int KW, bool GRP>
void rows_launch(const std::conditional_t<GRP, RowsGroupArgs, RowsArgs> &a, hipStream_t s) {
  constexpr int lds = rows_lds_bytes<XM, RB, KW>();
  if constexpr (lds > 64 * 1024) {  // raise the dynamic LDS limit once per variant
    static std::atomic<bool> raised{false};
    if (!raised.load(std::memory_order_acquire)) {
      (void)hipFuncSetAttribute((const void *)k_q4_gemm_rows<XM, ASYM, GK, RB, KW, GRP>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      raised.store(true, std::memory_order_release);
    }
  }
  const dim3 grid(a.tiles, (a.M + 32 * RB - 1) / (32 * RB), a.ksplit);
  k_q4_gemm_rows<XM, ASYM, GK, RB, KW, GRP><<<grid, 256 * KW, lds, s>>>(a);
}

// The tiles built: rb row blocks of 32 (1..4; fp32 halves up to 2) by kw K
// groups of waves (1 or 2; two fp32 row blocks 1). group: a itself, if it is one.
template <int XM>
bool rows_dispatch(const RowsArgs &a, const RowsGroupArgs *group, bool asym, int rb, int kw, hipStream_t s) {
#define SF_RL(AS, GKV, RBV, KWV)                  \
  if (rb == RBV && kw == KWV) {                   \
    if (group) rows_launch<XM, AS, GKV, RBV, KWV, true>(*group, s); \
    else rows_launch<XM, AS, GKV, RBV, KWV, false>(a, s);        \
    return true;                                  \
  }
#define SF_RR(AS, GKV)                            \
  do {                                            \
    SF_RL(AS, GKV, 1, 1) SF_RL(AS, GKV, 1, 2) SF_RL(AS, GKV, 2, 1)                             \
    if constexpr (XM != SF_F32) {                                                              \
      SF_RL(AS, GKV, 2, 2) SF_RL(AS, GKV, 3, 1) SF_RL(AS, GKV, 3, 2)                           \
      SF_RL(AS, GKV, 4, 1) SF_RL(AS, GKV, 4, 2)                                                \
    }                                                                                          \
    return false;                                 \
  } while (0)
#define SF_RG(AS)                                 \
  do {                                            \
    if (a.g == 32) SF_RR(AS, 0);                  \
    if (a.g == 64) SF_RR(AS, 1);                  \
    SF_RR(AS, 2);                                 \
  } while (0)
  if (asym) SF_RG(true);
  SF_RG(false);
#undef SF_RG
#undef SF_RR
#undef SF_RL
}

}  // namespace sf_gemm
