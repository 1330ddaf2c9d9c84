// Small-batch (2..8 tokens) Q4_K, Q6_K and Q8_0 linear layer on the matrix cores, register-resident form: the decode step of a few sequences
// with ONE launch per linear layer (no activation pre-pass, no slice reduction launch).
//
// The arithmetic is that of gemm_q4k_nb (cai_gemm_nb.hip): A operand = sc_j * q (exact in f16), B operand = the activations
// of up to 8 tokens, scaled per (token, 256-block) by a power of two and split hi + lo into two f16 = the 16 columns of
// v_mfma_f32_16x16x32_f16, one more MFMA per row set and super-block for the - dmin * mn_j * sum_j(x) term
// (Q4_K: neural/neuralgguf.pas:472-514); for Q6_K that of gemm_q6k_nb: one v_mfma_f32_16x16x16_f16 a scale group of 16 weights, activations
// as the rows of the result, so that a lane multiplies by the scale it loaded itself; for Q8_0 that of gemm_blk_nb, the same with one
// v_mfma_f32_16x16x32_f16 a block.  What differs is who holds what:
//   * a WAVE owns two super-blocks (512 columns) of EVERY row its work-group walks, so the B operands of its 16 MFMA steps
//     never change: it reads its 8 x 512 activations as fp32 once, applies the RMSNorm gain, finds the block scales, splits
//     hi + lo and keeps the operands in 64 registers for the whole launch - no activation planes in memory, no LDS traffic
//     in the product loop, no barrier before the first product;
//   * a work-group = the waves that together cover the columns (7 waves for 3584) walks 32-row pairs of row sets; per pair
//     every wave leaves its share in LDS, and after up to 16 pairs the waves meet and each finishes every n-th pair: adds the shares in wave
//     order, 1/rms of the token (sums of squares exchanged through LDS), bias, residual, or SwiGLU when the two
//     row sets of a pair are 16 up rows and their 16 gate rows - written once, as fp32, where the next launch reads them;
//   * a width of more than 16 super-blocks (the 18944-wide down projection) is cut into column slices = work-groups of
//     blockIdx.y; the slices' shares meet in a partial buffer and the LAST slice work-group of a row group to arrive (an
//     arrival counter, as in the attention merge) adds them in slice order with bias and residual.
// What bounds it: the arithmetic of the operands (two waves a SIMD, 250 instructions an item of 32 rows and a super-block) beside the requests, of which more on their
// way are slower.  us a launch, 8 tokens, a meeting per pair, addresses by lane and up to three items on their way | this: 7B gate|up 27.4 | 23.0, down 20.1 | 17.5
// (Q6_K 25.2 | 22.5), q|k|v 12.5 | 11.3, o 9.8 | 8.5, Q6_K head 121 | 106; alone the meetings were 1.2 of gate|up's, a second item on its way cost 2.5, requests past the
// last item 0.5.
// Fixed orders everywhere: the result does not depend on timing.
#include "cai_internal.hpp"
#include "cai_gemv_common.hpp"
#include <algorithm>
#include <type_traits>

namespace cai {

namespace {
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t uint2_t __attribute__((ext_vector_type(2)));

constexpr int RA_TK = 8;         // tokens per launch
constexpr int RA_NW = 8;         // waves per work-group at most
constexpr int RA_SBW = 2;        // super-blocks of a row per wave
constexpr int RA_SMAX = RA_NW * RA_SBW;   // super-blocks per column slice at most
constexpr int RA_BB = 144;       // bytes of a Q4_K super-block
constexpr int RA_B6 = 192;       // bytes of a Q6_K record of codes (16 scales and d lie in planes of their own)
constexpr int RA_PART_BATCH = 8; // slices of an element the last arriver requests at once (times 2 elements, times 2 for SwiGLU)
constexpr int RA_XLD = RA_SBW * 256 + 8;          // halfs per operand column in LDS (+8: 16 columns x 16-byte reads tile the banks)
constexpr int RA_PAIRS = 16;      // pairs that a wave leaves its shares of before the waves meet (a KB each, over its operand columns)
constexpr int RA_WAVE_LDS = 16 * RA_XLD * 2 + 16 * 16 * 2 + RA_SBW * RA_TK * 4 + 192;   // = 17408 bytes per wave

struct RaSeg { const uint8_t* w; const uint8_t* aux; const uint8_t* aux2; const float* bias; int rows; int y_off; int pair_end; };   // pair_end: cumulative 32-row pairs

struct RaParams {
  RaSeg seg[3]; int n_seg;                       // up to three matrices of equal width share a launch (q | k | v)
  float eps;                                     // RMSNorm of the activations (when a gain is given): 1/rms is applied to the result
  int swiglu_half;                               // > 0: rows [0, half) are up, [half, 2 half) gate; pair p = up rows 16 p.. + gate rows half + 16 p..
  float* y; long long y_stride; const float* residual;   // residual: laid out like y (may be y itself)
  int n_slices;
  float* part; long long part_stride;            // n_slices > 1: part[(slice * n_tok + t) * part_stride + y_off + row]
  unsigned* counters;                            // n_slices > 1: one arrival counter per row group (blockIdx.x), wrapping to 0
  unsigned long long* timeline;                  // stamps of this launch's work-groups (null: none)
};

__device__ __forceinline__ void ra_part_store(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float ra_part_load(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// The weight operand of one MFMA step from two quant dwords (8 bytes, low or high nibbles): with K = 0x64006400 the halfs of
// (d & 0x000f000f) | K are 1024 + the low nibbles of bytes 0 and 2, those of (d & 0x00f000f0) | K are 1024 + 16 x the high
// nibbles of the same bytes (no shift needed); d >> 8 gives bytes 1 and 3.  One packed fma each turns them into the exact
// halfs sc * q: (1024 + q) * sc - 1024 * sc, or (1024 + 16 q) * (sc / 16) - 64 * sc.  The order in which the 8 weights land in
// the operand (bytes 0, 2, 1, 3 of the first dword, then of the second) is the order the activation operand is built in.
// (written as a bit-field insert into a register copy of K - (d & M) | (K & ~M) - so that it is ONE instruction, v_bfi_b32:
// with two literal constants the and and the or stay separate.)
template <bool HIGH> __device__ __forceinline__ half8_t ra_weights(uint32_t d0, uint32_t d1, half2_t s2, half2_t c2, uint32_t kreg)
{
  constexpr uint32_t M = HIGH ? 0x00f000f0u : 0x000f000fu;
  const uint32_t e0 = d0 >> 8, e1 = d1 >> 8;
  const half2_t a0 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, (d0 & M) | (kreg & ~M)), s2, c2);
  const half2_t a1 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, (e0 & M) | (kreg & ~M)), s2, c2);
  const half2_t a2 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, (d1 & M) | (kreg & ~M)), s2, c2);
  const half2_t a3 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, (e1 & M) | (kreg & ~M)), s2, c2);
  return half8_t{a0.x, a0.y, a1.x, a1.y, a2.x, a2.y, a3.x, a3.y};
}
__device__ __forceinline__ half2_t ra_halves(float a, float b)
{
  typedef float float2_t __attribute__((ext_vector_type(2)));
  return __builtin_convertvector((float2_t{a, b}), half2_t);
}
// all-reduce over the 16 lanes of a row: lane ^ 1, lane ^ 2, then the mirror images within 8 and within 16
#define RA_DPP(v, ctrl) __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, (v)), (ctrl), 0xf, 0xf, false))
__device__ __forceinline__ float ra_row_max(float v)
{
  v = fmaxf(v, RA_DPP(v, 0xb1)); v = fmaxf(v, RA_DPP(v, 0x4e)); v = fmaxf(v, RA_DPP(v, 0x141)); v = fmaxf(v, RA_DPP(v, 0x140));
  return v;
}
__device__ __forceinline__ float ra_row_sum(float v)
{
  v += RA_DPP(v, 0xb1); v += RA_DPP(v, 0x4e); v += RA_DPP(v, 0x141); v += RA_DPP(v, 0x140);
  return v;
}
// all-reduce over each half of a row (8 lanes)
__device__ __forceinline__ float ra_oct_sum(float v)
{
  v += RA_DPP(v, 0xb1); v += RA_DPP(v, 0x4e); v += RA_DPP(v, 0x141);
  return v;
}
}  // namespace

// v_mfma_f32_16x16x32_f16: lane (m = lane % 16, kg = lane / 16) supplies 8 consecutive k of row m (A) / column m (B); the
// 16 x 16 result has rows 4 kg .. 4 kg + 3 of column m in this lane.  The order of k inside a super-block is free (both
// operands follow it) and is chosen for the weight requests: the four kg lanes of a row ask for 64 contiguous quant bytes per
// request (bytes 16 kg .. + 15, then 64 + 16 kg .. + 15).  With g = kg / 2 and c1 = kg % 2 lane kg owns weights
// 16 c1 .. 16 c1 + 15 of sub-blocks 2 g + 4 c + nib (c = request, nib = low / high nibbles), step t = 4 c + 2 nib + j takes
// the 8 of them at 8 j (in the order 0, 2, 1, 3, 4, 6, 5, 7: see ra_weights).  For the min term lane kg stands for the two sub-blocks 2 g + 4 c1, + 1 (each lane pair kg, kg ^ 1
// holds the halves of four sub-blocks' activations, so their sums are one exchange away).
// (what the first requests need travels as leading scalar arguments, preloaded in scalar registers)
// Q6_K: see gemm_q6k_nb for which bytes make which group; the operands of group g are columns 16 g + 4 kg .. + 3, in the order 0, 2, 1, 3.
// HH: 16-row sets per unit of rows (2: pairs - what SwiGLU needs and what long walks take; 1 halves the unit, for products
// with fewer pairs than compute units or an uneven number per work-group).  GAIN: the activations carry an RMSNorm gain.  HQ: four tokens, or
// two times four, are converted (2 sequences of a 7B shape 318 -> 308 us of four layers; as a branch of one kernel eight lost 1 %).
#define RA_ARGS const float* hsrc, const long long hstride, const float* hgain, const int hcols, const int hntok, const int hnpairs, const int hS
template <int QT, int HH, bool GAIN, int HQ>
__device__ __forceinline__ void ra_body(RA_ARGS, const int bx, const int n_bx, const RaParams& p)      // row group bx of n_bx
{
  // per wave RA_WAVE_LDS bytes: the operand columns [16][RA_XLD] halfs while the activations are converted (each wave converts
  // and reads back only its own columns: no work-group barrier), their sub-block sums [16][16] halfs and 1 / scale [2][8]; once
  // the operands are in registers the first 16 KB are the wave's shares of its pairs: [RA_PAIRS][32 lanes][8]
  extern __shared__ __align__(16) unsigned char ra_dyn[];
  __shared__ float ssq_s[RA_SMAX][RA_TK];
  const unsigned long long tl0 = timeline_now();
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, kg = lane >> 4, g = kg >> 1, c1 = kg & 1;
  const int K = hcols, nsb = K >> 8;
  const int slice = blockIdx.y, sb0 = slice * hS, nS = min(hS, nsb - sb0);
  const int nwa = (nS + RA_SBW - 1) / RA_SBW;                              // waves of this work-group with columns to cover
  const int nsw = max(0, min(RA_SBW, nS - RA_SBW * wave));                  // super-blocks of this wave
  const int sbw0 = sb0 + min(RA_SBW * wave, nS - 1);                        // its first one (an idle wave re-reads the last)
  constexpr bool Q6 = QT == CAI_Q6_K, Q8 = QT == CAI_Q8_0, Q4 = QT == CAI_Q4_K;
  const int npw = bx < hnpairs ? (hnpairs - bx + n_bx - 1) / n_bx : 0;   // pairs of this work-group
  const int nq = RA_SBW * npw;                                              // (pair, super-block) items of a wave
  const int tok = n & (RA_TK - 1), tokc = min(tok, hntok - 1);
  const bool tok_on = tok < hntok;
  const bool lo_col = n >= RA_TK;

  // rows of a pair: plain matrices take 32 consecutive rows of a segment, SwiGLU 16 up rows and their 16 gate rows
  auto locate = [&](int pair, const RaSeg*& sg, int& r0, int& r1) __attribute__((always_inline)) {
    int sgi = 0, t0 = 0;
    if (p.n_seg > 1 && pair >= p.seg[0].pair_end) { sgi = 1; t0 = p.seg[0].pair_end; }
    if (p.n_seg > 2 && pair >= p.seg[1].pair_end) { sgi = 2; t0 = p.seg[1].pair_end; }
    sg = &p.seg[sgi];
    if (p.swiglu_half > 0) { r0 = 16 * pair; r1 = p.swiglu_half + 16 * pair; }
    else { r0 = (pair - t0) * 16 * HH; r1 = r0 + 16; }
  };

  struct W4 { uint4 h[HH], q[HH][2]; };
  struct W6 { u32x4_t ql[HH][2], qh[HH], sc[HH]; uint32_t d[HH]; };
  struct W8 { u32x4_t q[HH][4], sc[HH]; };
  using WRegs = std::conditional_t<Q6, W6, std::conditional_t<Q8, W8, W4>>;
  // Weights of item q = (pair q / 2, super-block q % 2 of this wave): for the rows n of both row sets the header and this
  // lane's 2 x 16 quant bytes.  Loads are never under a branch.
  // A scalar base and an offset that a lane keeps for the whole launch (row sets are whole, so no row is clamped).
  constexpr int WB = Q6 ? RA_B6 : Q8 ? 256 : RA_BB;
  uint32_t w_off = (uint32_t)(n * nsb) * WB + 16 * kg, h_off = (uint32_t)(n * nsb) * (Q4 ? WB : 16), d_off = (uint32_t)(n * nsb) * 2;
  auto load_w = [&](int q, WRegs& r) __attribute__((always_inline)) {
    asm volatile("" : "+v"(w_off), "+v"(h_off), "+v"(d_off));      // (32-bit offsets beside a scalar base: kept as 64-bit sums the addresses were the registers that spilled)
    const int qc = max(min(q, nq - 1), 0);
    const int pair = min(bx + (qc >> 1) * n_bx, hnpairs - 1), sb = sbw0 + min(qc & 1, max(nsw, 1) - 1);
    const RaSeg* sg; int r0, r1; locate(pair, sg, r0, r1);
#pragma unroll
    for (int hh = 0; hh < HH; hh++) {
      const int64_t b = (int64_t)(hh ? r1 : r0) * nsb + sb;
      const uint8_t* blk = sg->w + b * WB + w_off;
      if constexpr (Q6) {
        r.ql[hh][0] = *reinterpret_cast<const u32x4_t*>(blk);
        r.ql[hh][1] = *reinterpret_cast<const u32x4_t*>(blk + 64);
        r.qh[hh] = *reinterpret_cast<const u32x4_t*>(blk + 128);
        r.sc[hh] = *reinterpret_cast<const u32x4_t*>(sg->aux + b * 16 + h_off);
        r.d[hh] = *reinterpret_cast<const uint16_t*>(sg->aux2 + b * 2 + d_off);
      } else if constexpr (Q8) {           // 256 codes; the scales of their eight blocks
#pragma unroll
        for (int i = 0; i < 4; i++) r.q[hh][i] = *reinterpret_cast<const u32x4_t*>(blk + 64 * i);
        r.sc[hh] = *reinterpret_cast<const u32x4_t*>(sg->aux + b * 16 + h_off);
      } else {
        r.h[hh] = *reinterpret_cast<const uint4*>(sg->w + b * WB + h_off);
        r.q[hh][0] = *reinterpret_cast<const uint4*>(blk + 16);
        r.q[hh][1] = *reinterpret_cast<const uint4*>(blk + 80);
      }
    }
  };
  WRegs wa, wb;

  // ---- this wave's activations: 8 tokens x its super-blocks, requested before the first weights ----
  // Requests in memory order: lane (r = lane / 16, i = lane % 16) asks for floats 64 m + 4 i .. + 3 (m = 0..3) of super-block j
  // of tokens r and 4 + r, so a request covers 256 contiguous bytes of each of four tokens (in operand order a request would
  // touch 64 different cache lines).  A 16-lane row then holds whole (token, block)s: scale and sums are row-local reductions.
  unsigned char* wl = ra_dyn + (size_t)wave * RA_WAVE_LDS;
  _Float16* xw = reinterpret_cast<_Float16*>(wl);                          // [16 columns][RA_XLD]
  _Float16* sxw = xw + 16 * RA_XLD;                                        // [16 columns][16 sub-blocks]
  float* sinvw = reinterpret_cast<float*>(sxw + 16 * 16);                  // [RA_SBW][8 tokens]
  const int rr = lane >> 4, ii = lane & 15;
  float4 xr[RA_SBW][HQ][4];
#pragma unroll
  for (int j = 0; j < RA_SBW; j++)
#pragma unroll
    for (int hq = 0; hq < HQ; hq++) {
      const float* px = hsrc + (int64_t)min(4 * hq + rr, hntok - 1) * hstride + (int64_t)(sbw0 + min(j, max(nsw, 1) - 1)) * 256 + 4 * ii;
#pragma unroll
      for (int m = 0; m < 4; m++) xr[j][hq][m] = *reinterpret_cast<const float4*>(px + 64 * m);
    }
  float4 gr[RA_SBW][4];
#pragma unroll
  for (int j = 0; j < RA_SBW; j++) {
    const float* pg = (GAIN ? hgain : hsrc) + (int64_t)(sbw0 + min(j, max(nsw, 1) - 1)) * 256 + 4 * ii;    // (no gain: any readable address, the values are not used)
#pragma unroll
    for (int m = 0; m < 4; m++) gr[j][m] = *reinterpret_cast<const float4*>(pg + 64 * m);
  }
  load_w(0, wa); load_w(1, wb);
  timeline_put(p.timeline, 0, tl0); timeline_stamp(p.timeline, 1);

#pragma unroll
  for (int j = 0; j < RA_SBW; j++)
#pragma unroll
    for (int hq = 0; hq < 2; hq++) {
      const int t8 = 4 * hq + rr;                 // the row's token
      if (hq >= HQ) {                              // four absent tokens: zeros
#pragma unroll
        for (int m = 0; m < 4; m++) {
          *reinterpret_cast<uint2*>(xw + t8 * RA_XLD + j * 256 + 64 * m + 4 * ii) = make_uint2(0u, 0u);
          *reinterpret_cast<uint2*>(xw + (8 + t8) * RA_XLD + j * 256 + 64 * m + 4 * ii) = make_uint2(0u, 0u);
          if (Q4 && (ii & 7) == 0) sxw[t8 * 16 + j * 8 + 2 * m + (ii >> 3)] = sxw[(8 + t8) * 16 + j * 8 + 2 * m + (ii >> 3)] = (_Float16)0.0f;
        }
        if (ii == 0) { sinvw[j * RA_TK + t8] = 0.0f; if (j < nsw) ssq_s[RA_SBW * wave + j][t8] = 0.0f; }
        continue;
      }
      float v[4][4];
      float amax = 0.0f, ss = 0.0f;
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const float4 a = xr[j][hq][m], gq = gr[j][m];
        const float raw[4] = {a.x, a.y, a.z, a.w}, gg[4] = {gq.x, gq.y, gq.z, gq.w};
#pragma unroll
        for (int u = 0; u < 4; u++) { v[m][u] = GAIN ? raw[u] * gg[u] : raw[u]; amax = fmaxf(amax, fabsf(v[m][u])); ss = fmaf(raw[u], raw[u], ss); }
      }
      amax = ra_row_max(amax); ss = ra_row_sum(ss);
      if (j == 0 && hq == 0) timeline_stamp_after(p.timeline, 2, amax);
      int e = 0;
      if (amax > 0.0f && amax < 3.0e38f) { int ex; frexpf(amax, &ex); e = 14 - ex; }   // amax * 2^e in [2^13, 2^14)
      e = max(-60, min(60, e));
      const bool on = t8 < hntok;
      const float s = on ? ldexpf(1.0f, e) : 0.0f;      // (an absent token's columns: zeros)
#pragma unroll
      for (int m = 0; m < 4; m++) {
        // vs = h + l to 22 bits, both parts rounded two at a time (v_cvt_pk_f16_f32: the pair comes out packed, and
        // in the operand's order - inside a group of 8 that order is 0, 2, 1, 3, 4, 6, 5, 7 (ra_weights): the middle two of every four
        // swap); l = vs - h is exact in fp32
        float vs[4], sm = 0.0f;
#pragma unroll
        for (int u = 0; u < 4; u++) { vs[u] = v[m][u] * s; sm += vs[u]; }
        const half2_t h02 = ra_halves(vs[0], vs[2]), h13 = ra_halves(vs[1], vs[3]);
        const half2_t l02 = ra_halves(fmaf((float)h02.x, -1.0f, vs[0]), fmaf((float)h02.y, -1.0f, vs[2])), l13 = ra_halves(fmaf((float)h13.x, -1.0f, vs[1]), fmaf((float)h13.y, -1.0f, vs[3]));      // (one v_fma_mix_f32 each)
        *reinterpret_cast<uint2*>(xw + t8 * RA_XLD + j * 256 + 64 * m + 4 * ii) = make_uint2(__builtin_bit_cast(uint32_t, h02), __builtin_bit_cast(uint32_t, h13));
        *reinterpret_cast<uint2*>(xw + (8 + t8) * RA_XLD + j * 256 + 64 * m + 4 * ii) = make_uint2(__builtin_bit_cast(uint32_t, l02), __builtin_bit_cast(uint32_t, l13));
        // sub-block 2 m + i / 8 of the block: the sum of 8 lanes' values, / 32, hi + lo
        if constexpr (!Q4) continue;
        sm = ra_oct_sum(sm) * 0.03125f;
        const _Float16 qh = (_Float16)sm, ql = (_Float16)(sm - (float)qh);
        if ((ii & 7) == 0) { sxw[t8 * 16 + j * 8 + 2 * m + (ii >> 3)] = qh; sxw[(8 + t8) * 16 + j * 8 + 2 * m + (ii >> 3)] = ql; }
      }
      if (ii == 0) {
        sinvw[j * RA_TK + t8] = on ? ldexpf(1.0f, -e) : 0.0f;
        if (j < nsw) ssq_s[RA_SBW * wave + j][t8] = ss;
      }
    }
  __builtin_amdgcn_wave_barrier();    // LDS operations of a wave complete in order: its own columns are there
  // the operands in MFMA order: column n, this lane's 8 k of every step
  half8_t Bx[Q6 ? 1 : RA_SBW][8]; half4_t Xg[Q6 ? RA_SBW : 1][16]; half2_t bm[RA_SBW]; float4 sinv4[RA_SBW];
#pragma unroll
  for (int j = 0; j < RA_SBW; j++) {
    if constexpr (Q6) {
#pragma unroll
      for (int gi = 0; gi < 16; gi++) Xg[j][gi] = *reinterpret_cast<const half4_t*>(xw + n * RA_XLD + j * 256 + 16 * gi + 4 * kg);
    } else if constexpr (Q8) {             // block t: what the exchange of halves below leaves in this lane, weights 16 c1 + 8 g .. + 7
#pragma unroll
      for (int t = 0; t < 8; t++) Bx[j][t] = *reinterpret_cast<const half8_t*>(xw + n * RA_XLD + j * 256 + 32 * t + 16 * c1 + 8 * g);
    } else {
#pragma unroll
      for (int t = 0; t < 8; t++)
        Bx[j][t] = *reinterpret_cast<const half8_t*>(xw + n * RA_XLD + j * 256 + 64 * g + 16 * c1 + 128 * (t >> 2) + 32 * ((t >> 1) & 1) + 8 * (t & 1));
      bm[j] = *reinterpret_cast<const half2_t*>(sxw + n * 16 + j * 8 + 2 * g + 4 * c1);    // sub-blocks 2 g + 4 c1, + 1
    }
    sinv4[j] = *reinterpret_cast<const float4*>(sinvw + j * RA_TK + 4 * c1);      // row 4 kg + i of a result: token (4 kg + i) % 8
  }
  __builtin_amdgcn_wave_barrier();    // (the region is written again as the wave's shares of a pair)
  timeline_stamp_after(p.timeline, 3, sinv4[RA_SBW - 1].x);
  timeline_stamp(p.timeline, 4);
  // what a wave adds to the rows of the first pair that it finishes (bias, residual) is requested before the walk; from a harmless address when there is none
  struct Extra { float4 bias[HH], res[HH]; };
  auto prefetch = [&](int i, Extra& f) __attribute__((always_inline)) {
    const int pair = min(bx + min(i, max(npw, 1) - 1) * n_bx, hnpairs - 1);
    const RaSeg* sg; int r0, r1; locate(pair, sg, r0, r1);
#pragma unroll
    for (int hh = 0; hh < HH; hh++) {
      const int row = (hh ? r1 : r0) + 4 * kg;
      const float* bp = sg->bias ? sg->bias + row : reinterpret_cast<const float*>(sg->w);
      const float* rp = p.residual ? p.residual + (int64_t)tokc * p.y_stride + sg->y_off + row : p.y;
      f.bias[hh] = *reinterpret_cast<const float4*>(bp);
      f.res[hh] = *reinterpret_cast<const float4*>(rp);
    }
  };
  Extra ex;
  float acc[HH][4];
  const _Float16 k1024 = (_Float16)1024.0f, kz = (_Float16)0.0f;
  uint32_t kreg = 0x64006400u;                 // 1024.0 twice, kept in a register the compiler cannot fold (see ra_weights)
  asm volatile("" : "+v"(kreg));

  auto compute = [&](const WRegs& r, const int j) __attribute__((always_inline)) {
    if (j == 0) {
#pragma unroll
      for (int hh = 0; hh < HH; hh++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[hh][i] = 0.0f;
    }
    if (j >= nsw) return;
    if constexpr (Q6) {
      const float4_t z4 = {0.0f, 0.0f, 0.0f, 0.0f};
      const half2_t o2 = {(_Float16)(-1056.0f), (_Float16)(-1056.0f)};   // 1024 + q - 1056 = q - 32
#pragma unroll
      for (int hh = 0; hh < HH; hh++) {
        // dword kg of every 16-byte chunk: ql chunks 0..7 in lq[0..7], qh chunks 0..3 in hq[0..3]
        uint32_t lq[8], hq[4];
#pragma unroll
        for (int a = 0; a < 3; a++) {
          const u32x4_t v = a < 2 ? r.ql[hh][a] : r.qh[hh];
          const uint2_t t02 = __builtin_amdgcn_permlane32_swap(v.x, v.z, false, false);
          const uint2_t t13 = __builtin_amdgcn_permlane32_swap(v.y, v.w, false, false);
          const uint2_t u01 = __builtin_amdgcn_permlane16_swap(t02.x, t13.x, false, false);
          const uint2_t u23 = __builtin_amdgcn_permlane16_swap(t02.y, t13.y, false, false);
          uint32_t* dst = a < 2 ? lq + 4 * a : hq;
          dst[0] = u01.x; dst[1] = u01.y; dst[2] = u23.x; dst[3] = u23.y;
        }
        const float d = __half2float(__ushort_as_half((unsigned short)r.d[hh]));
        const uint32_t scw[4] = {r.sc[hh].x, r.sc[hh].y, r.sc[hh].z, r.sc[hh].w};
        float gs[4] = {0.0f, 0.0f, 0.0f, 0.0f}, s_before = 0.0f;
        float4_t c_before = z4;            // (a result is taken while the next product runs)
#pragma unroll
        for (int gi = 0; gi < 16; gi++) {
          const int nh = gi >> 3, jq = (gi >> 1) & 3, h = gi & 1;
          const uint32_t lo = (lq[4 * nh + 2 * (jq & 1) + h] >> (4 * (jq >> 1))) & 0x0f0f0f0fu;
          const uint32_t hf = hq[2 * nh + h];
          const uint32_t hi = (jq == 0 ? (hf << 4) : jq == 1 ? (hf << 2) : jq == 2 ? hf : (hf >> 2)) & 0x30303030u;
          const uint32_t c = lo | hi;
          const half2_t w02 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, c, 0x04020400u)) + o2;
          const half2_t w13 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, c, 0x04030401u)) + o2;
          const half4_t W = {w02.x, w02.y, w13.x, w13.y};
          const float4_t C = __builtin_amdgcn_mfma_f32_16x16x16f16(Xg[j][gi], W, z4, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; i++) gs[i] = gi ? fmaf(s_before, c_before[i], gs[i]) : 0.0f;
          s_before = (float)(int)(int8_t)((scw[gi >> 2] >> (8 * (gi & 3))) & 0xffu);
          c_before = C;
        }
        const float si[4] = {sinv4[j].x, sinv4[j].y, sinv4[j].z, sinv4[j].w};
#pragma unroll
        for (int i = 0; i < 4; i++) acc[hh][i] = fmaf(si[i] * d, fmaf(s_before, c_before[i], gs[i]), acc[hh][i]);
      }
    } else if constexpr (Q8) {
      const float4_t z4 = {0.0f, 0.0f, 0.0f, 0.0f};
      const half2_t o2 = {(_Float16)(-1152.0f), (_Float16)(-1152.0f)};   // 1024 + (code + 128) - 1152
#pragma unroll
      for (int hh = 0; hh < HH; hh++) {
        float gs[4] = {0.0f, 0.0f, 0.0f, 0.0f}, s_before = 0.0f;
        float4_t c_before = z4;            // (a result is taken while the next product runs)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          // lanes kg 0, 1 asked for block 2 i, kg 2, 3 for block 2 i + 1: the halves change places, and each block is in all four
          const u32x4_t v = r.q[hh][i];
          const uint2_t xz = __builtin_amdgcn_permlane32_swap(v.x, v.z, false, false);
          const uint2_t yw = __builtin_amdgcn_permlane32_swap(v.y, v.w, false, false);
          const uint32_t scw = i == 0 ? r.sc[hh].x : i == 1 ? r.sc[hh].y : i == 2 ? r.sc[hh].z : r.sc[hh].w;
#pragma unroll
          for (int e = 0; e < 2; e++) {
            const uint32_t c0 = (e ? xz.y : xz.x) ^ 0x80808080u, c1w = (e ? yw.y : yw.x) ^ 0x80808080u;
            const half2_t a = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, c0, 0x04020400u)) + o2, b = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, c0, 0x04030401u)) + o2;
            const half2_t c = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, c1w, 0x04020400u)) + o2, d = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, c1w, 0x04030401u)) + o2;
            const half8_t W = {a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
            const float ds = __half2float(__ushort_as_half((unsigned short)(e ? scw >> 16 : scw & 0xffffu)));
            const float4_t C = __builtin_amdgcn_mfma_f32_16x16x32_f16(Bx[j][2 * i + e], W, z4, 0, 0, 0);
#pragma unroll
            for (int k = 0; k < 4; k++) gs[k] = i + e ? fmaf(s_before, c_before[k], gs[k]) : 0.0f;
            s_before = ds; c_before = C;
          }
        }
        const float si[4] = {sinv4[j].x, sinv4[j].y, sinv4[j].z, sinv4[j].w};
#pragma unroll
        for (int k = 0; k < 4; k++) acc[hh][k] = fmaf(si[k], fmaf(s_before, c_before[k], gs[k]), acc[hh][k]);
      }
    } else {
    float4_t C[HH], Cm[HH];
    half2_t s2[HH][4], c2[HH][4];
#pragma unroll
    for (int hh = 0; hh < HH; hh++) {
      // 6-bit scales / mins (neural/neuralgguf.pas:448-464), one per byte: sub-blocks 0..3 and 4..7
      const uint4 h = r.h[hh];
      const uint32_t sc_lo = h.y & 0x3f3f3f3fu, sc_hi = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u);
      const uint32_t mn_lo = h.z & 0x3f3f3f3fu, mn_hi = ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u);
      const uint32_t scq[2] = {sc_lo >> (16 * g), sc_hi >> (16 * g)};       // bytes 0, 1 = sub-blocks 2 g + 4 c, + 1
      const uint32_t mnp = (c1 ? mn_hi : mn_lo) >> (16 * g);                // sub-blocks 2 g + 4 c1, + 1
      const half2_t mnh = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, mnp, 0x04010400u)) - half2_t{k1024, k1024};
#pragma unroll
      for (int c = 0; c < 2; c++) {
        // low nibbles: (sc, -1024 sc); high nibbles arrive as 16 q: (sc / 16, -64 sc) - all exact in f16
        const half2_t sch = (__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, scq[c], 0x04010400u)) - half2_t{k1024, k1024}) * half2_t{(_Float16)1.0f, (_Float16)0.0625f};
        const half2_t cch = sch * half2_t{(_Float16)(-1024.0f), (_Float16)(-1024.0f)};
        s2[hh][2 * c] = half2_t{sch.x, sch.x}; s2[hh][2 * c + 1] = half2_t{sch.y, sch.y};
        c2[hh][2 * c] = half2_t{cch.x, cch.x}; c2[hh][2 * c + 1] = half2_t{cch.y, cch.y};
      }
      // - dmin * mn * (sum of the sub-block's activations): k = this lane's two sub-blocks, the other six k stay zero
      const half8_t Am = {mnh.x, mnh.y, kz, kz, kz, kz, kz, kz}, Bm = {bm[j].x, bm[j].y, kz, kz, kz, kz, kz, kz};
      const float4_t z4 = {0.0f, 0.0f, 0.0f, 0.0f};
      Cm[hh] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Bm, Am, z4, 0, 0, 0);
      C[hh] = z4;
    }
#pragma unroll
    for (int t = 0; t < 8; t++) {
      const int c = t >> 2, nib = (t >> 1) & 1, jj = t & 1;      // request, nibble, dword pair
#pragma unroll
      for (int hh = 0; hh < HH; hh++) {
        const uint4& qq = r.q[hh][c];
        const uint32_t d0 = jj ? qq.z : qq.x, d1 = jj ? qq.w : qq.y;
        const half8_t A = nib ? ra_weights<true>(d0, d1, s2[hh][2 * c + 1], c2[hh][2 * c + 1], kreg) : ra_weights<false>(d0, d1, s2[hh][2 * c], c2[hh][2 * c], kreg);
        C[hh] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Bx[j][t], A, C[hh], 0, 0, 0);
      }
    }
#pragma unroll
    for (int hh = 0; hh < HH; hh++) {
      const uint32_t dd = r.h[hh].x;
      const float d = __half2float(__ushort_as_half((unsigned short)(dd & 0xffffu))), dmin = __half2float(__ushort_as_half((unsigned short)(dd >> 16))) * 32.0f;
      const float si[4] = {sinv4[j].x, sinv4[j].y, sinv4[j].z, sinv4[j].w};
#pragma unroll
      for (int i = 0; i < 4; i++) acc[hh][i] += si[i] * (d * C[hh][i] - dmin * Cm[hh][i]);
    }
    }
  };

  // ---- end of a pair: every wave leaves its share (column t hi + column 8 + t lo) ----
  auto share = [&](int i) __attribute__((always_inline)) {
    const int slot = i % RA_PAIRS;
    if (nsw > 0) {     // result row 4 kg + i = token (4 kg + i) % 8, hi (kg < 2) or lo: they meet across kg ^ 2; column n = weight row n
#pragma unroll
      for (int hh = 0; hh < HH; hh++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const uint32_t v = __builtin_bit_cast(uint32_t, acc[hh][k]);
          const uint2_t hl = __builtin_amdgcn_permlane32_swap(v, v, false, false);
          const uint32_t hi = hl.x, lo = hl.y;      // (of an element in place __builtin_bit_cast takes the first)
          const float t = __builtin_bit_cast(float, hi) + __builtin_bit_cast(float, lo);
          if (kg < 2) reinterpret_cast<float*>(wl)[(slot * 32 + (n >> 2) * 8 + 4 * kg + k) * 8 + 4 * hh + (n & 3)] = t;
        }
    }
  };
  // ---- one wave finishes the rows of a pair ----
  auto finish = [&](int i, const Extra& f) __attribute__((always_inline)) {
    const int slot = i % RA_PAIRS;
    if (lo_col) return;
    float t8[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    for (int w = 0; w < nwa; w++) {       // wave order: fixed
      const float* src = reinterpret_cast<const float*>(ra_dyn + (size_t)w * RA_WAVE_LDS) + (slot * 32 + kg * 8 + n) * 8;
      const float4 a = *reinterpret_cast<const float4*>(src);
      t8[0] += a.x; t8[1] += a.y; t8[2] += a.z; t8[3] += a.w;
      if constexpr (HH == 2) { const float4 b = *reinterpret_cast<const float4*>(src + 4); t8[4] += b.x; t8[5] += b.y; t8[6] += b.z; t8[7] += b.w; }
    }
    if (!tok_on) return;
    const int pair = bx + i * n_bx;
    const RaSeg* sg; int r0, r1; locate(pair, sg, r0, r1);
    if (p.n_slices > 1) {     // a slice's share of the rows (finished by the last slice to arrive, below)
#pragma unroll
      for (int hh = 0; hh < HH; hh++) {
        float* dst = p.part + ((int64_t)slice * hntok + tok) * p.part_stride + sg->y_off + (hh ? r1 : r0) + 4 * kg;
#pragma unroll
        for (int k = 0; k < 4; k++) ra_part_store(dst + k, t8[4 * hh + k]);
      }
      return;
    }
    float inv = 1.0f;
    if (GAIN) {   // (a product with a gain is one slice: the work-group has seen the whole row, and its waves have met since)
      float t = 0.0f;
      for (int sb = 0; sb < nS; sb++) t += ssq_s[sb][tok];     // fixed order
      inv = 1.0f / sqrtf(t / (float)K + p.eps);
    }
    if (HH == 2 && p.swiglu_half > 0) {
      const int col = 16 * pair + 4 * kg;       // rows r0 + 4 kg .. + 3 (up) and r1 + 4 kg .. + 3 (gate)
      const float bu[4] = {f.bias[0].x, f.bias[0].y, f.bias[0].z, f.bias[0].w}, bg[4] = {f.bias[HH - 1].x, f.bias[HH - 1].y, f.bias[HH - 1].z, f.bias[HH - 1].w};
      float o[4];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        float up = inv * t8[k], gate = inv * t8[4 + k];
        if (sg->bias) { up += bu[k]; gate += bg[k]; }
        o[k] = silu_mul(up, gate);
      }
      *reinterpret_cast<float4*>(p.y + (int64_t)tok * p.y_stride + col) = make_float4(o[0], o[1], o[2], o[3]);
      return;
    }
#pragma unroll
    for (int hh = 0; hh < HH; hh++) {
      const int row = (hh ? r1 : r0) + 4 * kg;
      const float bb[4] = {f.bias[hh].x, f.bias[hh].y, f.bias[hh].z, f.bias[hh].w}, rr[4] = {f.res[hh].x, f.res[hh].y, f.res[hh].z, f.res[hh].w};
      float vv[4];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        vv[k] = inv * t8[4 * hh + k];
        if (sg->bias) vv[k] += bb[k];
        if (p.residual) vv[k] += rr[k];
      }
      *reinterpret_cast<float4*>(p.y + (int64_t)tok * p.y_stride + sg->y_off + row) = make_float4(vv[0], vv[1], vv[2], vv[3]);
    }
  };

  const int nwb = blockDim.x >> 6;
  for (int i0 = 0; i0 < npw; i0 += RA_PAIRS) {
    const int i1 = min(npw, i0 + RA_PAIRS);
    prefetch(i0 + wave, ex);
    for (int i = i0; i < min(i1, npw - 1); i++) {
      compute(wa, 0); load_w(2 * i + 2, wa);
      compute(wb, 1); load_w(2 * i + 3, wb);
      share(i);
    }
    if (i1 == npw) { compute(wa, 0); compute(wb, 1); share(npw - 1); }
    __syncthreads();
    for (int i = i0 + wave; i < i1; i += nwb) {
      if (i != i0 + wave) prefetch(i, ex);
      finish(i, ex);
    }
    if (i1 < npw) __syncthreads();      // (the slots are written again)
  }
  timeline_stamp(p.timeline, 5);
  if (p.n_slices > 1) {
    // the slices of a row group meet (shares stored and read at agent scope); the last to arrive adds them in slice order
    const bool last = arrives_last(p.counters + bx, (unsigned)p.n_slices);
    timeline_stamp(p.timeline, 6);
    if (!last) { timeline_stamp(p.timeline, 7); return; }
    // the elements EB at a time: all slices' shares of a batch of elements (and their bias and residual) are requested before
    // the first addition; the additions run in slice order
    const int rpu = 16 * HH;                                  // rows per unit
    const int total = npw * rpu * hntok;
    const int64_t sstep = (int64_t)hntok * p.part_stride;     // from one slice's share of an element to the next
    constexpr int EB = 2;
    for (int e0 = threadIdx.x; e0 < total; e0 += EB * blockDim.x) {
      const float* src[EB]; float bias[EB], res[EB], sum[EB]; int64_t out[EB]; bool on[EB];
#pragma unroll
      for (int b = 0; b < EB; b++) {
        const int e = min(e0 + b * (int)blockDim.x, total - 1);
        on[b] = e0 + b * (int)blockDim.x < total;
        const int rl = e % rpu, t = (e / rpu) % hntok, i = (e / rpu) / hntok;
        const RaSeg* sg; int r0, r1; locate(bx + i * n_bx, sg, r0, r1);
        src[b] = p.part + (int64_t)t * p.part_stride + sg->y_off + r0 + rl;
        out[b] = (int64_t)t * p.y_stride + sg->y_off + r0 + rl;
        bias[b] = sg->bias ? sg->bias[r0 + rl] : 0.0f;
        res[b] = p.residual ? p.residual[out[b]] : 0.0f;
        sum[b] = 0.0f;
      }
      for (int s0 = 0; s0 < p.n_slices; s0 += RA_PART_BATCH) {
        float ps[EB][RA_PART_BATCH];
#pragma unroll
        for (int b = 0; b < EB; b++)
#pragma unroll
          for (int u = 0; u < RA_PART_BATCH; u++) ps[b][u] = ra_part_load(src[b] + (int64_t)min(s0 + u, p.n_slices - 1) * sstep);
#pragma unroll
        for (int b = 0; b < EB; b++)
#pragma unroll
          for (int u = 0; u < RA_PART_BATCH; u++) if (s0 + u < p.n_slices) sum[b] += ps[b][u];
      }
#pragma unroll
      for (int b = 0; b < EB; b++) if (on[b]) p.y[out[b]] = sum[b] + bias[b] + res[b];
    }
  }
  timeline_stamp(p.timeline, 7);
}

template <int QT, int HH, bool GAIN, int HQ>
__global__ __launch_bounds__(64 * RA_NW) void gemm_ra(RA_ARGS, const RaParams p)
{
  ra_body<QT, HH, GAIN, HQ>(hsrc, hstride, hgain, hcols, hntok, hnpairs, hS, blockIdx.x, gridDim.x, p);
}
// Normed products over the same activations whose matrices are of both types (attn_q and attn_k beside the attn_v of a mixed file): the first
// hn4 work-groups take the Q4_K rows in pairs of row sets, the others the Q6_K rows.  Both launches by themselves spend most of their time on
// the activations (7B shape, eight sequences: 11.1 + 11.2 us, 12.9 here).
template <int HQ>
__global__ __launch_bounds__(64 * RA_NW) void gemm_ra_two(RA_ARGS, const int hnpairs6, const int hn4, const RaParams p, const RaParams p6)
{
  if ((int)blockIdx.x < hn4) ra_body<CAI_Q4_K, 2, true, HQ>(hsrc, hstride, hgain, hcols, hntok, hnpairs, hS, blockIdx.x, hn4, p);
  else ra_body<CAI_Q6_K, 1, true, HQ>(hsrc, hstride, hgain, hcols, hntok, hnpairs6, hS, blockIdx.x - hn4, gridDim.x - hn4, p6);
}

// ------------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------------
namespace {
struct RaWs { float* part = nullptr; size_t cap_part = 0; unsigned* counters = nullptr; int generation = 0; };
RaWs g_ra;
constexpr int RA_COUNTERS = 1024;

// How a product over nsb super-blocks and `pairs` row pairs is cut: column slices of S super-blocks (work-groups of
// ceil(S / 2) waves; a CU holds 8 such waves) and gx row groups, so that all work-groups are resident at once and the
// longest walk (pairs of a work-group) is shortest; fewer slices at equal length.
bool ra_geometry(int nsb, int pairs, int& S, int& n_slices, int& gx)
{
  const int n_cu = ctx().n_cu;
  const int ns_min = (nsb + RA_SMAX - 1) / RA_SMAX;
  float best = 3.0e38f;
  // (a width that fits one slice stays one: no partial results at all)
  for (int ns = ns_min; ns <= (ns_min == 1 ? 1 : std::min(nsb, ns_min + 8)); ns++) {
    const int s = (nsb + ns - 1) / ns;
    if ((nsb + s - 1) / s != ns) continue;
    const int nw = (s + RA_SBW - 1) / RA_SBW;
    const int slots = n_cu * (RA_NW / nw);
    const int g = std::max(1, std::min(pairs, std::min(slots / ns, RA_COUNTERS)));
    // every wave takes two super-blocks of each pair of its work-group: the walk is as long as the pairs per work-group
    const float cost = (float)((pairs + g - 1) / g) + 0.05f * (float)ns;
    if (cost < best) { best = cost; S = s; n_slices = ns; gx = g; }
  }
  return best < 3.0e38f;
}
}  // namespace

void ra_release()
{
  if (g_ra.part) (void)hipFree(g_ra.part);
  if (g_ra.counters) (void)hipFree(g_ra.counters);
  const int gen = g_ra.generation + 1;
  g_ra = RaWs(); g_ra.generation = gen;
}
int ra_ws_generation() { return g_ra.generation; }

// Partial buffer (floats) and arrival counters of the sliced products (never inside a stream capture).
int ra_reserve(size_t part_floats)
{
  if (!g_ra.counters) {
    CAI_HIP(hipMalloc((void**)&g_ra.counters, RA_COUNTERS * sizeof(unsigned)));
    CAI_HIP(hipMemsetAsync(g_ra.counters, 0, RA_COUNTERS * sizeof(unsigned), ctx().stream));
    CAI_HIP(hipStreamSynchronize(ctx().stream));
    g_ra.generation++;
  }
  if (part_floats > g_ra.cap_part) {
    CAI_HIP(hipStreamSynchronize(ctx().stream));
    if (g_ra.part) (void)hipFree(g_ra.part);
    g_ra.part = nullptr; g_ra.cap_part = 0;
    CAI_HIP(hipMalloc((void**)&g_ra.part, part_floats * sizeof(float)));
    g_ra.cap_part = part_floats; g_ra.generation++;
  }
  return CAI_OK;
}

// Floats of partial buffer a product of `rows` outputs over `cols` columns may need for 8 tokens (0: it is one slice)
size_t ra_part_floats(int64_t rows, int64_t cols)
{
  const int nsb = (int)(cols >> 8);
  if (nsb <= RA_SMAX) return 0;
  const int ns_max = (nsb + RA_SMAX - 1) / RA_SMAX + 8;
  return (size_t)ns_max * RA_TK * (size_t)((rows + 3) / 4 * 4);
}

// Whether ra_gemm takes these matrices: Q4_K, Q6_K or Q8_0, one width of whole super-blocks, whole 16-row sets,
// one column slice when the product carries an RMSNorm or SwiGLU.
bool ra_supported(const cai_qw_s* const* ws, int n_w, bool normed, int swiglu_half)
{
  if (n_w < 1 || n_w > 3 || (swiglu_half > 0 && n_w != 1)) return false;
  for (int i = 0; i < n_w; i++) {
    const cai_qw_s* w = ws[i];
    if ((w->qtype != CAI_Q4_K && w->qtype != CAI_Q6_K && w->qtype != CAI_Q8_0) || w->cols != ws[0]->cols || w->cols % 256 || w->cols < 256 || w->rows % 16) return false;
  }
  if (swiglu_half > 0 && (ws[0]->rows != 2 * (int64_t)swiglu_half || swiglu_half % 16)) return false;
  // a product with an RMSNorm or SwiGLU must be one column slice (its finishing wave needs the whole row's sum of squares and
  // both halves' rows); measured on 5120 columns a sliced form with those exchanged through memory lost to the plane form
  const int nsb = (int)(ws[0]->cols >> 8);
  return !((normed || swiglu_half > 0) && nsb > RA_SMAX);
}

static int ra_check(const cai_qw_s* const* ws, const int* y_off, int n_w, const float* x, int64_t x_stride, const float* gain, const float* y, int64_t y_stride, const float* residual)
{
  if ((x_stride & 3) || (reinterpret_cast<uintptr_t>(x) & 15) || (gain && (reinterpret_cast<uintptr_t>(gain) & 15)))
    return set_error(CAI_ERR_INVALID, "small-batch product (register form): activations must be 16-byte aligned rows");
  if ((y_stride & 3) || (reinterpret_cast<uintptr_t>(y) & 15) || (residual && (reinterpret_cast<uintptr_t>(residual) & 15)))
    return set_error(CAI_ERR_INVALID, "small-batch product (register form): results must be 16-byte aligned rows");
  for (int i = 0; i < n_w; i++)
    if ((y_off[i] & 3) || (ws[i]->bias && (reinterpret_cast<uintptr_t>(ws[i]->bias) & 15)))
      return set_error(CAI_ERR_INVALID, "small-batch product (register form): output offsets and biases must be 16-byte aligned");
  return CAI_OK;
}
static RaSeg ra_seg(const cai_qw_s* w, int y_off, int end) { return RaSeg{w->data, w->aux, w->qtype == CAI_Q6_K ? qw_aux2(w) : nullptr, w->bias, (int)w->rows, y_off, end}; }
static int ra_two(const cai_qw_s* const* ws, const int* y_off, int n_w, int n_tok, const float* x, int64_t x_stride, const float* gain, float eps, float* y, int64_t y_stride)
{
  int rc = ra_check(ws, y_off, n_w, x, x_stride, gain, y, y_stride, nullptr);
  if (rc) return rc;
  RaParams p[2] = {};
  int units[2] = {0, 0};        // pairs of row sets of Q4_K, row sets of Q6_K
  for (int i = 0; i < n_w; i++) {
    const int six = ws[i]->qtype == CAI_Q6_K;
    units[six] += (int)(ws[i]->rows / (six ? 16 : 32));
    p[six].seg[p[six].n_seg++] = ra_seg(ws[i], y_off[i], units[six]);
  }
  for (RaParams& q : p) { q.eps = eps; q.y = y; q.y_stride = y_stride; q.n_slices = 1; }
  const int nsb = (int)(ws[0]->cols >> 8), nw = (nsb + RA_SBW - 1) / RA_SBW, all = units[0] + units[1], slots = std::max(2, ctx().n_cu * (RA_NW / nw));
  const int n4 = all <= slots ? units[0] : std::max(1, std::min(slots - 1, (int)((int64_t)slots * units[0] / all))), n6 = all <= slots ? units[1] : std::max(1, std::min(units[1], slots - n4));
  p[0].timeline = p[1].timeline = timeline_next(n4 + n6);
  auto launch = [&](auto kern, bool& attr_done) -> int {
    if (!attr_done) { CAI_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, RA_NW * RA_WAVE_LDS)); attr_done = true; }
    hipLaunchKernelGGL(kern, dim3(n4 + n6), dim3(64 * nw), (size_t)nw * RA_WAVE_LDS, ctx().stream, x, (long long)x_stride, gain, (int)ws[0]->cols, n_tok, units[0], nsb, units[1], n4, p[0], p[1]);
    return CAI_OK;
  };
  static bool attr_done[2] = {false, false};
  if ((rc = n_tok <= 4 ? launch(gemm_ra_two<1>, attr_done[0]) : launch(gemm_ra_two<2>, attr_done[1]))) return rc;
  return CAI_OK;
}

// y[t][y_off_i + r] = W_i (gain . x_t) / rms(x_t) + bias_i [+ residual]   for t < n_tok <= 8, or, with swiglu_half > 0,
// y[t][r] = up_r * silu(gate_r) of the one matrix [up; gate].  x: fp32 rows of x_stride floats (16-byte aligned).
int ra_gemm(const cai_qw_s* const* ws, const int* y_off, int n_w, int n_tok, const float* x, int64_t x_stride, const float* gain, float eps,
            int swiglu_half, float* y, int64_t y_stride, const float* residual)
{
  if (n_tok < 1 || n_tok > RA_TK || !ra_supported(ws, n_w, gain != nullptr, swiglu_half))
    return set_error(CAI_ERR_UNSUPPORTED, "small-batch product (register form): %d matrices, %d tokens", n_w, n_tok);
  if (gain && swiglu_half == 0 && !residual) {
    bool four = false, six = false, other = false;
    for (int i = 0; i < n_w; i++) {
      (ws[i]->qtype == CAI_Q6_K ? six : four) = true;
      other = other || ws[i]->qtype == CAI_Q8_0 || (ws[i]->qtype == CAI_Q4_K && ws[i]->rows % 32);
    }
    if (four && six && !other) return ra_two(ws, y_off, n_w, n_tok, x, x_stride, gain, eps, y, y_stride);
  }
  for (int i = 1; i < n_w; i++)
    if (ws[i]->qtype != ws[0]->qtype) {      // (one type after the other)
      int rc = ra_gemm(ws, y_off, i, n_tok, x, x_stride, gain, eps, swiglu_half, y, y_stride, residual);
      return rc ? rc : ra_gemm(ws + i, y_off + i, n_w - i, n_tok, x, x_stride, gain, eps, swiglu_half, y, y_stride, residual);
    }
  { int rc = ra_check(ws, y_off, n_w, x, x_stride, gain, y, y_stride, residual); if (rc) return rc; }
  RaParams p{};
  p.n_seg = n_w; p.eps = eps; p.swiglu_half = swiglu_half; p.y = y; p.y_stride = y_stride; p.residual = residual;
  const int cols = (int)ws[0]->cols, nsb = cols >> 8;
  // units of 32 rows (pairs of row sets), or of 16 where that shortens the longest walk (a wave takes 2 x HH items per unit)
  int HH = 2, S = 0, n_slices = 0, gx = 0, units = 0;
  {
    int u2 = 0, u1 = 0;
    for (int i = 0; i < n_w; i++) { u2 += swiglu_half > 0 ? swiglu_half / 16 : (int)(ws[i]->rows / 32); u1 += (int)(ws[i]->rows / 16); }
    bool whole_pairs = true;
    for (int i = 0; i < n_w; i++) whole_pairs = whole_pairs && ws[i]->rows % 32 == 0;
    int S2 = 0, ns2 = 0, g2 = 0, S1 = 0, ns1 = 0, g1 = 0;
    if (!ra_geometry(nsb, u2, S2, ns2, g2) || !ra_geometry(nsb, u1, S1, ns1, g1))
      return set_error(CAI_ERR_UNSUPPORTED, "small-batch product (register form): width %d", cols);
    units = u2; S = S2; n_slices = ns2; gx = g2;
    if (swiglu_half == 0 && (!whole_pairs || (u1 + g1 - 1) / g1 < 2 * ((u2 + g2 - 1) / g2))) { HH = 1; units = u1; S = S1; n_slices = ns1; gx = g1; }
  }
  int cum = 0; int64_t width = 0;
  for (int i = 0; i < n_w; i++) {
    cum += swiglu_half > 0 ? swiglu_half / 16 : (int)(ws[i]->rows / (16 * HH));
    p.seg[i] = ra_seg(ws[i], y_off[i], cum);
    width = std::max<int64_t>(width, y_off[i] + ws[i]->rows);
  }
  p.n_slices = n_slices;
  if (n_slices > 1) {
    p.part_stride = (width + 3) / 4 * 4;
    if ((size_t)n_slices * n_tok * p.part_stride > g_ra.cap_part || !g_ra.counters)
      return set_error(CAI_ERR_STATE, "small-batch product (register form): workspace not reserved (%d slices x %d tokens x %lld)", n_slices, n_tok, (long long)p.part_stride);
    p.part = g_ra.part; p.counters = g_ra.counters;
  }
  const int nw = (S + RA_SBW - 1) / RA_SBW;
  p.timeline = timeline_next(gx * n_slices);
  const dim3 grid(gx, n_slices), block(64 * nw);
  const size_t lds = (size_t)nw * RA_WAVE_LDS;
#define RA_LAUNCH(QTv, HHv, GAINv, HQv) do { \
    static bool attr_done = false; \
    if (!attr_done) { CAI_HIP(hipFuncSetAttribute((const void*)gemm_ra<QTv, HHv, GAINv, HQv>, hipFuncAttributeMaxDynamicSharedMemorySize, RA_NW * RA_WAVE_LDS)); attr_done = true; } \
    hipLaunchKernelGGL((gemm_ra<QTv, HHv, GAINv, HQv>), grid, block, lds, ctx().stream, x, (long long)x_stride, gain, cols, n_tok, units, S, p); } while (0)
#define RA_FORM(QTv, HQv) do { \
    if (HH == 2 && gain) RA_LAUNCH(QTv, 2, true, HQv); \
    else if (HH == 2) RA_LAUNCH(QTv, 2, false, HQv); \
    else if (gain) RA_LAUNCH(QTv, 1, true, HQv); \
    else RA_LAUNCH(QTv, 1, false, HQv); } while (0)
#define RA_TYPE(QTv) do { if (n_tok <= 4) RA_FORM(QTv, 1); else RA_FORM(QTv, 2); } while (0)
  if (ws[0]->qtype == CAI_Q6_K) RA_TYPE(CAI_Q6_K);
  else if (ws[0]->qtype == CAI_Q8_0) RA_TYPE(CAI_Q8_0);
  else RA_TYPE(CAI_Q4_K);
#undef RA_TYPE
#undef RA_FORM
#undef RA_LAUNCH
  return CAI_OK;
}

}  // namespace cai
