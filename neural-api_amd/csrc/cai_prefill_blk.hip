// Multi-token (prompt) linear layer on the matrix cores for the 32-weight block types, Q8_0 and Q4_0 (one f16 scale per
// block: neural/neuralgguf.pas:389-441, 811-845; resident as a quants plane and a scales plane), dense or grouped by
// expert for a mixture-of-experts prompt (wiring: neural/neuralpretrained.pas:15331-15388).
//
// Accuracy contract as for the Q4_K prompt kernel: the result equals single-token linear layers to fp32 level.  The codes
// (signed bytes, nibble - 8) are exact in f16; an activation is a power-of-two scaled pair of halfs hi + lo (22 bits);
// products accumulate in fp32 on v_mfma_f32_32x32x16_f16; the block scale d multiplies the block's sum in fp32.
//
// d belongs to a weight ROW and a block, so the weights are the B operand (columns of the result = 32 weight rows) and the
// activations the A operand (rows = 32 tokens): lane (n, kg) then holds 16 results of ONE weight row n and d is a value it
// loaded itself - 16 FMAs fold a block's 32 x 32 sums into the running result, no exchange through LDS.  The order of the
// contraction index inside a block is free as long as both operands agree: a lane takes a CONTIGUOUS piece of each block
// (Q8_0: bytes 16 kg .. + 15, two steps of 8; Q4_0: bytes 8 kg .. + 7, low nibbles = weights 8 kg .. + 7 then high nibbles
// = weights 16 + 8 kg .. + 7), so the two lanes of a row read whole 32- / 16-byte blocks and a row's 256 columns are one
// contiguous run.
//
// Two forms: work-groups with a large tile of their own (gemm_blk_tile), and, where there are too few of those to fill the chip,
// work-groups whose waves share one small tile and cut its width (gemm_blk_cut).  Both bring their operands into LDS with
// asynchronous copies along the rows.
#include "cai_internal.hpp"
#include "cai_gemv_common.hpp"
#include "cai_blocks_raw.hpp"
#include "cai_async_copy.hpp"
#include <algorithm>
#include <type_traits>

namespace cai {

namespace {

typedef _Float16 half2_b __attribute__((ext_vector_type(2)));
typedef _Float16 half8_b __attribute__((ext_vector_type(8)));
typedef float float16_b __attribute__((ext_vector_type(16)));
typedef float f32x4_b __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_b __attribute__((ext_vector_type(4)));   // (arrays of HIP's uint4 struct end up in scratch memory)

struct BlkGemmParams {
  const uint8_t* q; const uint8_t* d; const float* bias;
  int rows, cols;                       // rows of ONE matrix (of one expert's window for a bank)
  const _Float16* xhi; const _Float16* xlo; const float* sinv;   // activation planes [x row][cols], scale per x row
  int n_tok;
  float* y; int64_t y_stride; const float* residual;
  int n_row_groups, n_tok_tiles;
  // grouped by expert: a table of token tiles built on the device (expert, first sorted position, count; count 0 = unused)
  const int32_t* tile_tab; const int32_t* perm;   // perm: sorted position -> slot (token * top_k + rank)
  int x_div;                            // activation row of a slot = slot / x_div; result row = slot
  int64_t expert_rows;
  // dense launches: up to two more matrices of the same type and width (q | k | v) - row groups [seg_end[i], ...) belong to
  // matrix i + 1, whose rows land y_off2[i] columns into a y row
  int n_seg; int seg_end[2];
  const uint8_t* q2[2]; const uint8_t* d2[2]; const float* bias2[2]; int rows2[2]; int y_off2[2];
  // types with minima: a weight is d * code + m16 of its sixteen; s16 = sums of sixteen activations [x row][cols / 16] in the planes' scale
  const float* m16; const float* s16;
  float post;                           // the results' last factor (gemm_blk_cut)
};

// eight codes (two dwords) -> eight exact halfs, negated or not.  Q8_0: signed bytes; Q4_0: (nibble - 8), low or high nibbles of the bytes
template <int QT>
__device__ __forceinline__ half8_b codes8(uint32_t w0, uint32_t w1, int high, bool neg = false)
{
  uint32_t a, b; _Float16 off;
  if (QT == CAI_Q8_0) { a = w0 ^ 0x80808080u; b = w1 ^ 0x80808080u; off = (_Float16)(-1152.0f); }   // byte + 128 as 1024 + u, minus 1152
  else { a = (high ? (w0 >> 4) : w0) & 0x0f0f0f0fu; b = (high ? (w1 >> 4) : w1) & 0x0f0f0f0fu; off = (_Float16)(-1032.0f); }
  const half2_b o2 = {off, off};
  auto half_pair = [&](uint32_t v, uint32_t sel) {
    const half2_b h = __builtin_bit_cast(half2_b, __builtin_amdgcn_perm(0x64646464u, v, sel));
    return neg ? -o2 - h : h + o2;
  };
  const half2_b h0 = half_pair(a, 0x04010400u), h1 = half_pair(a, 0x04030402u), h2 = half_pair(b, 0x04010400u), h3 = half_pair(b, 0x04030402u);
  return half8_b{h0.x, h0.y, h1.x, h1.y, h2.x, h2.y, h3.x, h3.y};
}

typedef uint32_t uint2_b __attribute__((ext_vector_type(2)));

}  // namespace

// ------------------------------------------------------------------------------------------
// Large tiles.  NW waves, 32 NW weight rows x TT * 32 tokens: eight, or four in half the LDS, so that a CU holds two work-groups which wait, start and
// end independently of each other.  Chunks of 64 columns - token planes, quants, scales, all copied along
// the rows from memory into LDS - are requested DEPTH - 1 chunks ahead of the one that is multiplied; the waves meet once a chunk.
// A wave holds 64 rows x 16 TT tokens: what it reads of a chunk from LDS (activations of its tokens, quants of its rows) takes less
// time than its products, which 32 rows x all tokens does not.  A tile of at most 32 tokens (an expert's run, a short prompt) is
// neither staged nor multiplied in its other half.
// What bounds it: a chunk's products (2048 cycles of a SIMD at TT = 4), the folds and codes (about 1800 cycles of VALU) and the LDS
// reads overlap only in part between the two waves of a SIMD (1.65 us a chunk; without copies 1.4, without folds 1.5, with neither
// and no codes 1.1).  Operands requested one block ahead, and folds issued between the next block's products, changed nothing.
// 37888 x 3584 Q8_0, 2048 tokens: 1721 us in tiles of 256 x 64 that staged through registers -> 1273 (TT = 4); 3584 x 18944: 1358 -> 718.
// Gate | up and down of 64 experts (2048 x 2048, 2048 x 1024), 2040 slots: 199 us a layer -> 149 (82 to read the banks once): with tiles
// of 64 slots instead of 32 an expert's rows come from memory once.
// ------------------------------------------------------------------------------------------
constexpr int blk_depth(int TT, int NW) { return TT == 2 && NW == 8 ? 4 : 3; }      // chunks in LDS
template <int QT, int TT, bool ODD, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_blk_tile(const BlkGemmParams p)
{
  extern __shared__ __align__(16) unsigned char bl_smem[];
  constexpr int NTOK = TT * 32, ROWS = 32 * NW, DEPTH = blk_depth(TT, NW), WROW = QT == CAI_Q8_0 ? 64 : 32;
  constexpr int PLANE = NTOK * 128, XB = 2 * PLANE, WB = ROWS * WROW, DB = ROWS * 4, SLOT = XB + WB + (ODD ? 2 : 1) * DB;
  constexpr int XC = NTOK / (8 * NW), WC = WROW / 32, COPIES = 2 * XC + WC + (ODD ? 2 : 1);      // a wave's copies of a chunk
  __shared__ int s_yrow[NTOK];
  __shared__ float s_sinv[NTOK];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, kg = lane >> 5;
  int rg, ttile, first, n_here, expert = 0;
  if (p.tile_tab) {
    ttile = blockIdx.x / p.n_row_groups; rg = blockIdx.x % p.n_row_groups;
    expert = p.tile_tab[3 * ttile]; first = p.tile_tab[3 * ttile + 1]; n_here = p.tile_tab[3 * ttile + 2];
    if (n_here <= 0) return;            // (uniform: the whole work-group leaves)
  } else {
    // linear id = rg_lo + 8 * (tt + n_tok_tiles * rg_hi): the token tiles of a row group share id mod 8, i.e. one XCD and its L2
    const int L = blockIdx.x;
    rg = (L & 7) + 8 * ((L >> 3) / p.n_tok_tiles); ttile = (L >> 3) % p.n_tok_tiles;
    if (rg >= p.n_row_groups) return;
    first = ttile * NTOK; n_here = min(NTOK, p.n_tok - first);
  }
  const bool one = TT == 2 && n_here <= 32;              // half a tile: the other half is neither staged nor multiplied
  const int x_n = !one ? XC : 8 * wave < 32 ? 1 : 0;     // of a wave's XC copies of token rows (8 (NW i + wave) and on) those that are made
  static_assert(XC == 1 || 8 * NW >= 32, "of half a tile a wave has one copy at most");
  const uint8_t* qbase = p.q; const uint8_t* dbase = p.d; const float* bias = p.bias; int rows = p.rows, yo = 0, rgl = rg;   // this work-group's matrix (uniform)
  if (p.n_seg > 1 && rg >= p.seg_end[0]) { qbase = p.q2[0]; dbase = p.d2[0]; bias = p.bias2[0]; rows = p.rows2[0]; yo = p.y_off2[0]; rgl = rg - p.seg_end[0]; }
  if (p.n_seg > 2 && rg >= p.seg_end[1]) { qbase = p.q2[1]; dbase = p.d2[1]; bias = p.bias2[1]; rows = p.rows2[1]; yo = p.y_off2[1]; rgl = rg - p.seg_end[1]; }
  const int R0 = rgl * ROWS, K = p.cols, nb32 = K >> 5, n_chunks = (nb32 + 1) >> 1;
  const int64_t bank_row = (int64_t)expert * p.expert_rows;
  auto x_row = [&](int m) { const int t = first + min(m, n_here - 1); return p.perm ? p.perm[t] / p.x_div : t; };   // rows past the end repeat the last token; their results are not written
  if (threadIdx.x < NTOK) {
    const int t = first + min((int)threadIdx.x, n_here - 1);
    s_yrow[threadIdx.x] = p.perm ? p.perm[t] : t; s_sinv[threadIdx.x] = p.sinv[x_row(threadIdx.x)];
  }
  // this lane's part of the copies: copy 8 i + wave takes 8 token rows (128 bytes a plane), 16 or 32 weight rows, 64 rows' scales
  uint32_t xo[XC], wo[WC], xcut = 0, wcut = 0;
#pragma unroll
  for (int i = 0; i < XC; i++) {
    const int t = 8 * (NW * i + wave) + (lane >> 3);
    const uint32_t piece = (uint32_t)((lane & 7) ^ ((t >> 1) & 7));
    xo[i] = (uint32_t)x_row(t) * (uint32_t)K * 2u + 16u * piece;
    if (ODD && piece >= 4) xcut |= 1u << i;
  }
  const int rlast = rows - 1 - R0;         // tail rows: the last one again, not written
#pragma unroll
  for (int i = 0; i < WC; i++) {
    if constexpr (QT == CAI_Q8_0) {
      const int t = 16 * (NW * i + wave) + (lane >> 2); const uint32_t piece = (uint32_t)((lane & 3) ^ ((t >> 2) & 3));
      wo[i] = (uint32_t)min(t, rlast) * (uint32_t)K + 16u * piece; if (ODD && piece >= 2) wcut |= 1u << i;
    }
    else {
      const int t = 32 * (NW * i + wave) + (lane >> 1); const uint32_t piece = (uint32_t)((lane & 1) ^ ((t >> 3) & 1));
      wo[i] = (uint32_t)min(t, rlast) * (uint32_t)(K / 2) + 16u * piece; if (ODD && piece) wcut |= 1u << i;
    }
  }
  const uint32_t dof = (uint32_t)min(64 * (wave & (NW / 2 - 1)) + lane, rlast) * (uint32_t)(nb32 * 2);     // (the upper half of the waves repeats the lower: every wave counts the same copies)
  const uint8_t* const qb = qbase + (bank_row + R0) * (int64_t)nb32 * (WROW / 2);
  const uint8_t* const db = dbase + (bank_row + R0) * (int64_t)nb32 * 2;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)bl_smem;
  auto copy = [&](int c, int slot) {
    const uint32_t dst = lds0 + (uint32_t)(slot * SLOT);
    const bool half = ODD && c == n_chunks - 1;        // one block is left: the chunk's second half repeats the first and is not used
    const char* const xh = reinterpret_cast<const char*>(p.xhi) + (int64_t)c * 128;
    const char* const xl = reinterpret_cast<const char*>(p.xlo) + (int64_t)c * 128;
#pragma unroll
    for (int i = 0; i < XC; i++)
      if (i < x_n) {
        const uint32_t o = xo[i] - (half && (xcut >> i & 1) ? 64u : 0u);
        copy16_to_lds(dst + 1024 * (NW * i + wave), o, xh);
        copy16_to_lds(dst + PLANE + 1024 * (NW * i + wave), o, xl);
      }
#pragma unroll
    for (int i = 0; i < WC; i++) copy16_to_lds(dst + XB + 1024 * (NW * i + wave), wo[i] - (half && (wcut >> i & 1) ? WROW / 2u : 0u), qb + (int64_t)c * WROW);
    if constexpr (ODD) {
      copy2_to_lds(dst + XB + WB + 256 * (wave & (NW / 2 - 1)), dof, db + (int64_t)c * 4);
      copy2_to_lds(dst + XB + WB + DB + 256 * (wave & (NW / 2 - 1)), dof, db + (int64_t)c * 4 + (half ? 0 : 2));
    } else copy4_to_lds(dst + XB + WB + 256 * (wave & (NW / 2 - 1)), dof, db + (int64_t)c * 4);
  };

  const float16_b zero16 = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  // RW row tiles x TW token tiles of a wave, from row tile r0 and token tile t0 of the work-group's on
  auto body = [&](auto rw_, auto tw_, int r0, int t0) {
    constexpr int RW = rw_, TW = tw_;
    // Runs of up to 16 tokens - all there are in a mixture's prompt of 9 to 16, whose slots went one by one through walks with short sums
    // before - take their sums in two steps of eight chunks, as the cut tiles do: logits 3 to 10 % further from 64 bits in one chain (width 2048
    // and 4096, eight experts), nearer than the walks so.  For all tiles a prompt of 255 tokens over 64 experts took 4549 us instead of 4475.
    constexpr bool STEPS = RW == 1;
    const bool steps = STEPS && n_here <= 16;
    float16_b Y[RW][TW], Z[STEPS ? RW : 1][STEPS ? TW : 1];
#pragma unroll
    for (int rt = 0; rt < RW; rt++)
#pragma unroll
      for (int tt = 0; tt < TW; tt++)
#pragma unroll
        for (int v = 0; v < 16; v++) { Y[rt][tt][v] = 0.0f; if constexpr (STEPS) Z[rt][tt][v] = 0.0f; }
    auto use = [&](int slot, bool half) {
      const unsigned char* const s0 = bl_smem + slot * SLOT;
      const unsigned char* const sx = s0 + (32 * t0 + n) * 128;
      const unsigned char* const sw = s0 + XB + (32 * r0 + n) * WROW;
      uint32_t dw[RW];
#pragma unroll
      for (int rt = 0; rt < RW; rt++) {
        dw[rt] = *reinterpret_cast<const uint32_t*>(s0 + XB + WB + 4 * (32 * (r0 + rt) + n));
        if constexpr (ODD) dw[rt] |= *reinterpret_cast<const uint32_t*>(s0 + XB + WB + DB + 4 * (32 * (r0 + rt) + n)) << 16;
      }
#pragma unroll
      for (int b = 0; b < 2; b++) {
        if (ODD && b && half) break;
        half8_b A[TW][4], W[RW][2];
#pragma unroll
        for (int s = 0; s < 2; s++) {
          // Q8_0: the lane's k of step s are columns 16 kg + 8 s .. of the block; Q4_0: 16 s + 8 kg ..
          const int c = 4 * b + (QT == CAI_Q8_0 ? 2 * kg + s : 2 * s + kg);
#pragma unroll
          for (int tt = 0; tt < TW; tt++) {
            const unsigned char* const a = sx + tt * 4096 + 16 * (c ^ ((n >> 1) & 7));
            A[tt][2 * s] = *reinterpret_cast<const half8_b*>(a); A[tt][2 * s + 1] = *reinterpret_cast<const half8_b*>(a + PLANE);
          }
        }
#pragma unroll
        for (int rt = 0; rt < RW; rt++) {
          const unsigned char* const w = sw + rt * 32 * WROW;
          if constexpr (QT == CAI_Q8_0) {
            const u32x4_b q = *reinterpret_cast<const u32x4_b*>(w + 16 * ((2 * b + kg) ^ ((n >> 2) & 3)));
            W[rt][0] = codes8<QT>(q.x, q.y, 0); W[rt][1] = codes8<QT>(q.z, q.w, 0);
          } else {
            const uint2 q = *reinterpret_cast<const uint2*>(w + 16 * (b ^ ((n >> 3) & 1)) + 8 * kg);
            W[rt][0] = codes8<QT>(q.x, q.y, 0); W[rt][1] = codes8<QT>(q.x, q.y, 1);
          }
        }
#pragma unroll
        for (int rt = 0; rt < RW; rt++) {
          const float dv = __half2float(__ushort_as_half((unsigned short)(b ? (dw[rt] >> 16) : (dw[rt] & 0xffffu))));
          float16_b C[TW];
#pragma unroll
          for (int k = 0; k < 4; k++)
#pragma unroll
            for (int tt = 0; tt < TW; tt++) C[tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[tt][k], W[rt][k >> 1], k == 0 ? zero16 : C[tt], 0, 0, 0);
#pragma unroll
          for (int tt = 0; tt < TW; tt++)
#pragma unroll
            for (int v = 0; v < 16; v++) Y[rt][tt][v] = fmaf(dv, C[tt][v], Y[rt][tt][v]);
        }
      }
    };
#pragma unroll
    for (int i = 0; i < DEPTH - 1; i++) if (i < n_chunks) copy(i, i);
    int slot = 0;
    for (int c = 0; c < n_chunks; c++) {
      const int left = n_chunks - 1 - c;               // chunks behind this one
      if (left >= DEPTH - 2) { if (x_n == XC) wait_copies<(DEPTH - 2) * COPIES>(); else wait_copies<(DEPTH - 2) * (COPIES - 2)>(); }
      else wait_copies<0>();
      __builtin_amdgcn_s_waitcnt(0xC07F);              // lgkmcnt(0): this wave's reads of the slot that is filled next (and the row tables, the first time)
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (left >= DEPTH - 1) copy(c + DEPTH - 1, slot == 0 ? DEPTH - 1 : slot - 1);
      use(slot, ODD && left == 0);
      slot = slot + 1 == DEPTH ? 0 : slot + 1;
      if constexpr (STEPS)
        if (steps && (c & 7) == 7)
#pragma unroll
          for (int rt = 0; rt < RW; rt++)
#pragma unroll
            for (int tt = 0; tt < TW; tt++)
#pragma unroll
              for (int v = 0; v < 16; v++) { Z[rt][tt][v] += Y[rt][tt][v]; Y[rt][tt][v] = 0.0f; }
    }
    // ---- write: the lane holds weight row n and tokens 8 g + 4 kg + i of each tile: the 32 lanes of a half-wave store 32
    // consecutive outputs of one token row ----
#pragma unroll
    for (int tt = 0; tt < TW; tt++)
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int m = 32 * (t0 + tt) + 8 * (v >> 2) + 4 * kg + (v & 3);
        if (m >= n_here) continue;
        const float si = s_sinv[m];
        const int64_t o = (int64_t)s_yrow[m] * p.y_stride + yo;
#pragma unroll
        for (int rt = 0; rt < RW; rt++) {
          const int row = R0 + 32 * (r0 + rt) + n;
          if (row >= rows) continue;
          float y = Y[rt][tt][v];
          if constexpr (STEPS) y += Z[rt][tt][v];
          y *= si;
          if (bias) y += bias[bank_row + row];
          if (p.residual) y += p.residual[o + row];
          p.y[o + row] = y;
        }
      }
  };
  if constexpr (TT == 2) {
    if (one) { body(std::integral_constant<int, 1>(), std::integral_constant<int, 1>(), wave, 0); return; }
  }
  body(std::integral_constant<int, 2>(), std::integral_constant<int, TT / 2>(), 2 * (wave & (NW / 2 - 1)), TT / 2 * (wave / (NW / 2)));
}

// ------------------------------------------------------------------------------------------
// Few tiles: the waves of a work-group share ONE tile of 32 RT rows x 32 tokens and cut its width; their sums meet in LDS at the end.
// Each wave copies chunks of 64 columns (token planes, quants, scales) along the rows into LDS of its own, one chunk ahead of the one
// it multiplies, so there is no barrier before the end.  An operand load straight from memory touches 32 rows, a line each, and takes
// four times the cycles of the same bytes read along the rows: that form, also cut, took 15.2 us where this one takes 10.7.
// Sums are taken in two steps: one chain over a wave's share of 18944 columns is 1.9e-7 off 64 bits, two short ones 1.2e-7, as the
// one-token kernels are (1 % of the time).
// What bounds it: the copies, 66 KB/us into one CU.  576 x 1536, 37 tokens, with the pre-pass of the activations: 23.1 us as 10 uncut
// tiles of 128 x 32 -> 10.7; 64 x 2048, 255 tokens: 27 -> 14; 2048 x 2048, 255: 31 -> 17.
// Places in LDS: 16-byte piece c of token row t (128 bytes a plane) at c ^ (t / 2 % 8), of Q8_0 weight row n (64 bytes) at c ^ (n / 4 % 4),
// of Q4_0 row n (32 bytes) at c ^ (n / 8 % 2): the lanes of a read pass then meet different banks.
// ------------------------------------------------------------------------------------------
// FINE (panels of the stored streams, and up to 16 tokens of Q8_0 and Q4_0: what went through the 32-bit walks otherwise): the lo halves and the
// minima are summed apart from the large parts.  A matrix instruction that adds them to the block's sum rounds it once more each, and cuts what
// lies below the largest of its products off downwards (so every second block goes in with its sign changed): 1.04e-7 off 64 bits for Q2_K and 0.91e-7 for Q3_K at width 512, where the walk of
// eight tokens is 0.96e-7 and 0.88e-7; apart 0.80e-7 both (3584: 1.28e-7 -> 0.95e-7, walk 1.52e-7) for 3 to 5 % of the time.  Q8_0, nine
// tokens: 0.92e-7 -> 0.82e-7 at 512, walk 0.99e-7; at 3584 1.06e-7 -> 0.97e-7, walk 1.07e-7, and with activations that spread over decades
// 1.14e-7 -> 1.04e-7, walk 1.05e-7.
template <int QT, int RT, int NW, bool ODD, bool FINE = false, bool MIN = false>     // ODD: rows of an odd number of blocks (scales that are not aligned to 4 bytes, a last chunk of one block)
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_blk_cut(const BlkGemmParams p)
{
  extern __shared__ __align__(16) unsigned char bl_smem[];
  constexpr int WROW = QT == CAI_Q8_0 ? 64 : 32, NV = RT * 16;                 // quant bytes of a row's chunk; values of a lane
  constexpr int XB = 8192, WB = 32 * WROW, DB = ODD ? 512 : 256, MB = RT * WB + XB + DB, SLOT = MB + (MIN ? 512 + 512 * RT : 0);          // a chunk: planes hi, lo; quants; scales
  constexpr int COPIES = 8 + RT * WB / 1024 + (ODD ? 2 : 1) + (MIN ? 2 + 2 * RT : 0);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, kg = lane >> 5;
  const int L = blockIdx.x;
  const int rg = (L & 7) + 8 * ((L >> 3) / p.n_tok_tiles), ttile = (L >> 3) % p.n_tok_tiles;
  if (rg >= p.n_row_groups) return;
  const int first = ttile * 32;
  const uint8_t* qbase = p.q; const uint8_t* dbase = p.d; const float* bias = p.bias; int rows = p.rows, yo = 0, rgl = rg;   // this work-group's matrix (uniform)
  if (p.n_seg > 1 && rg >= p.seg_end[0]) { qbase = p.q2[0]; dbase = p.d2[0]; bias = p.bias2[0]; rows = p.rows2[0]; yo = p.y_off2[0]; rgl = rg - p.seg_end[0]; }
  if (p.n_seg > 2 && rg >= p.seg_end[1]) { qbase = p.q2[1]; dbase = p.d2[1]; bias = p.bias2[1]; rows = p.rows2[1]; yo = p.y_off2[1]; rgl = rg - p.seg_end[1]; }
  const int R0 = rgl * 32 * RT, K = p.cols, nb32 = K >> 5;
  const int n_chunks = (nb32 + 1) >> 1, c0 = n_chunks * wave / NW, c1 = n_chunks * (wave + 1) / NW;     // this wave's chunks
  // this lane's part of the copies; rows and tokens past the end repeat the last one and are not written
  uint32_t xo[4], wo[RT * WB / 1024], xcut = 0, wcut = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int t = 8 * i + (lane >> 3);
    const uint32_t piece = (uint32_t)((lane & 7) ^ ((t >> 1) & 7));
    xo[i] = (uint32_t)min(first + t, p.n_tok - 1) * (uint32_t)K * 2u + 16u * piece;
    if (ODD && piece >= 4) xcut |= 1u << i;
  }
  const int rlast = rows - 1 - R0;
#pragma unroll
  for (int i = 0; i < RT * WB / 1024; i++) {
    if constexpr (QT == CAI_Q8_0) {
      const int t = 16 * i + (lane >> 2); const uint32_t piece = (uint32_t)((lane & 3) ^ ((t >> 2) & 3));
      wo[i] = (uint32_t)min(t, rlast) * (uint32_t)K + 16u * piece; if (ODD && piece >= 2) wcut |= 1u << i;
    }
    else {
      const int t = 32 * i + (lane >> 1); const uint32_t piece = (uint32_t)((lane & 1) ^ ((t >> 3) & 1));
      wo[i] = (uint32_t)min(t, rlast) * (uint32_t)(K / 2) + 16u * piece; if (ODD && piece) wcut |= 1u << i;
    }
  }
  const uint32_t dof = (uint32_t)min(RT == 2 ? lane : n, rlast) * (uint32_t)(nb32 * 2);
  const uint8_t* const qb = qbase + (int64_t)R0 * nb32 * (WROW / 2);
  const uint8_t* const db = dbase + (int64_t)R0 * nb32 * 2;
  // (MIN) lanes of a copy: token n, sixteen 2 i + kg; rows: RT = 2 row `lane`, sixteen i, RT = 1 row n, sixteen i + kg
  const uint32_t sof = MIN ? (uint32_t)min(first + n, p.n_tok - 1) * (uint32_t)(K / 4) + 4u * (uint32_t)kg : 0u;
  const uint32_t mof = MIN ? (uint32_t)min(RT == 2 ? lane : n, rlast) * (uint32_t)(K / 4) + (RT == 2 ? 0u : 4u * (uint32_t)kg) : 0u;
  const char* const mb = MIN ? reinterpret_cast<const char*>(p.m16) + (int64_t)R0 * (K / 4) : nullptr;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)bl_smem + (uint32_t)(wave * 2 * SLOT);
  auto copy = [&](int c, int slot) {
    const uint32_t dst = lds0 + (uint32_t)(slot * SLOT);
    const bool half = ODD && c == n_chunks - 1;        // one block is left: the chunk's second half repeats the first and is not used
    const char* const xh = reinterpret_cast<const char*>(p.xhi) + (int64_t)c * 128;
    const char* const xl = reinterpret_cast<const char*>(p.xlo) + (int64_t)c * 128;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t o = xo[i] - (half && (xcut >> i & 1) ? 64u : 0u);
      copy16_to_lds(dst + 1024 * i, o, xh); copy16_to_lds(dst + 4096 + 1024 * i, o, xl);
    }
#pragma unroll
    for (int i = 0; i < RT * WB / 1024; i++) copy16_to_lds(dst + XB + 1024 * i, wo[i] - (half && (wcut >> i & 1) ? WROW / 2u : 0u), qb + (int64_t)c * WROW);
    if constexpr (ODD) {
      copy2_to_lds(dst + XB + RT * WB, dof, db + (int64_t)c * 4);
      copy2_to_lds(dst + XB + RT * WB + 256, dof, db + (int64_t)c * 4 + (half ? 0 : 2));
    } else copy4_to_lds(dst + XB + RT * WB, dof, db + (int64_t)c * 4);
    if constexpr (MIN) {                   // [sixteen of the chunk][token or row]; past the width (the last chunk of ODD) the ones before again
#pragma unroll
      for (int i = 0; i < 2; i++) copy4_to_lds(dst + MB + 256 * i, sof + (uint32_t)(8 * i), reinterpret_cast<const char*>(p.s16) + (int64_t)c * 16 - (half && i ? 8 : 0));
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (RT == 2 || (i & 1) == 0)
          copy4_to_lds(dst + MB + 512 + 256 * (RT == 2 ? i : i >> 1), mof + (uint32_t)(4 * i), mb + (int64_t)c * 16 - (half && i >= 2 ? 8 : 0));
    }
  };
  float16_b Y[RT], Z[RT], U[RT];           // sums of eight (RT = 2: sixteen) blocks, sums of those: see the comment above; FINE: the small parts
#pragma unroll
  for (int rt = 0; rt < RT; rt++)
#pragma unroll
    for (int v = 0; v < 16; v++) Y[rt][v] = Z[rt][v] = U[rt][v] = 0.0f;
  const float16_b zero16 = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  const unsigned char* const mine = bl_smem + wave * 2 * SLOT;
  auto use = [&](int slot, bool half) {
    const unsigned char* const s0 = mine + slot * SLOT;
    uint32_t dw[RT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
      dw[rt] = *reinterpret_cast<const uint32_t*>(s0 + XB + RT * WB + 4 * (32 * rt + n));
      if constexpr (ODD) dw[rt] |= *reinterpret_cast<const uint32_t*>(s0 + XB + RT * WB + 256 + 4 * (32 * rt + n)) << 16;
    }
#pragma unroll
    for (int b = 0; b < 2; b++) {
      if (ODD && b && half) break;
      const bool neg = FINE && b;           // (the second block's products and scale change sign, and with it the side to which the small ones are cut off)
      half8_b A[4], W[RT][2];
#pragma unroll
      for (int s = 0; s < 2; s++) {
        // Q8_0: the lane's k of step s are columns 16 kg + 8 s .. of the block; Q4_0: 16 s + 8 kg ..
        const int c = 4 * b + (QT == CAI_Q8_0 ? 2 * kg + s : 2 * s + kg);
        const unsigned char* const a = s0 + n * 128 + 16 * (c ^ ((n >> 1) & 7));
        A[2 * s] = *reinterpret_cast<const half8_b*>(a); A[2 * s + 1] = *reinterpret_cast<const half8_b*>(a + 4096);
      }
#pragma unroll
      for (int rt = 0; rt < RT; rt++) {
        const unsigned char* const w = s0 + XB + rt * WB + n * WROW;
        if constexpr (QT == CAI_Q8_0) {
          const u32x4_b q = *reinterpret_cast<const u32x4_b*>(w + 16 * ((2 * b + kg) ^ ((n >> 2) & 3)));
          W[rt][0] = codes8<QT>(q.x, q.y, 0, neg); W[rt][1] = codes8<QT>(q.z, q.w, 0, neg);
        } else {
          const uint2 q = *reinterpret_cast<const uint2*>(w + 16 * (b ^ ((n >> 3) & 1)) + 8 * kg);
          W[rt][0] = codes8<QT>(q.x, q.y, 0, neg); W[rt][1] = codes8<QT>(q.x, q.y, 1, neg);
        }
      }
#pragma unroll
      for (int rt = 0; rt < RT; rt++) {
        const float dh = __half2float(__ushort_as_half((unsigned short)(b ? (dw[rt] >> 16) : (dw[rt] & 0xffffu)))), dv = neg ? -dh : dh;
        float16_b C = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[0], W[rt][0], zero16, 0, 0, 0);
        if constexpr (FINE) {
          float16_b D = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[1], W[rt][0], zero16, 0, 0, 0);
          C = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[2], W[rt][1], C, 0, 0, 0);
          D = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[3], W[rt][1], D, 0, 0, 0);
#pragma unroll
          for (int v = 0; v < 16; v++) { Y[rt][v] = fmaf(dv, C[v], Y[rt][v]); U[rt][v] = fmaf(dv, D[v], U[rt][v]); }
        } else {
#pragma unroll
          for (int k = 1; k < 4; k++) C = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[k], W[rt][k >> 1], C, 0, 0, 0);
#pragma unroll
          for (int v = 0; v < 16; v++) Y[rt][v] = fmaf(dv, C[v], Y[rt][v]);
        }
      }
      if constexpr (MIN)
#pragma unroll
        for (int e = 0; e < 2; e++) {
          const int g16 = 2 * b + e;
          const float* const sp = reinterpret_cast<const float*>(s0 + MB) + 32 * g16 + 4 * kg;
          const float* const mp = reinterpret_cast<const float*>(s0 + MB + 512);
          f32x4_b sv[4];
#pragma unroll
          for (int g = 0; g < 4; g++) sv[g] = *reinterpret_cast<const f32x4_b*>(sp + 8 * g);
#pragma unroll
          for (int rt = 0; rt < RT; rt++) {
            const float m = mp[32 * RT * g16 + 32 * rt + n];
#pragma unroll
            for (int v = 0; v < 16; v++) U[rt][v] = fmaf(m, sv[v >> 2][v & 3], U[rt][v]);
          }
        }
    }
  };
  if (c0 < c1) copy(c0, 0);
  for (int c = c0; c < c1; c++) {
    const int slot = (c - c0) & 1;
    if (c + 1 < c1) {
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the last reads of the other slot
      copy(c + 1, slot ^ 1);
      wait_copies<COPIES>();
    } else wait_copies<0>();
    use(slot, ODD && c == n_chunks - 1);
    if (((c - c0) & (RT == 1 ? 3 : 7)) == (RT == 1 ? 3 : 7))
#pragma unroll
      for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int v = 0; v < 16; v++) { Z[rt][v] += Y[rt][v]; Y[rt][v] = 0.0f; }
  }
  __syncthreads();                         // (every wave's copies have been waited for)
  float* const sacc = reinterpret_cast<float*>(bl_smem);     // [wave][RT 16][64 lanes]
#pragma unroll
  for (int rt = 0; rt < RT; rt++)
#pragma unroll
    for (int v = 0; v < 16; v++) sacc[(wave * NV + rt * 16 + v) * 64 + lane] = FINE ? Z[rt][v] + (Y[rt][v] + U[rt][v]) : Z[rt][v] + Y[rt][v];
  __syncthreads();
  // wave w sums the values w, w + NW, ...: the lane's value v of row tile rt is weight row n and token 8 (v / 4) + 4 kg + v % 4
#pragma unroll
  for (int j0 = 0; j0 < NV; j0 += NW) {
    const int j = j0 + wave, v = j & 15, rt = j >> 4;
    if (j >= NV) break;
    float y = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; w++) y += sacc[(w * NV + j) * 64 + lane];
    const int t = first + 8 * (v >> 2) + 4 * kg + (v & 3), row = R0 + 32 * rt + n;
    if (t >= p.n_tok || row >= rows) continue;
    const int64_t o = (int64_t)t * p.y_stride + yo + row;
    if constexpr (MIN)
      if (!(fabsf(y) < __builtin_inff())) {         // an infinity among the activations: its two parts may differ in sign, the weight's own counts
        float sum = 0.0f; bool any = false;
        for (int k = 0; k < K; k++) {
          const float x = (float)p.xhi[(int64_t)t * K + k] + (float)p.xlo[(int64_t)t * K + k];
          if (fabsf(x) < __builtin_inff()) continue;
          const int64_t at = (int64_t)row * K + k;
          const float d = (float)__builtin_bit_cast(_Float16, reinterpret_cast<const uint16_t*>(dbase)[at >> 5]);
          sum += fmaf(d, (float)reinterpret_cast<const int8_t*>(qbase)[at], p.m16[at >> 4]) * x; any = true;
        }
        if (any) y = sum;
      }
    y *= p.sinv[t] * p.post;
    if (bias) y += bias[row];
    if (p.residual) y += p.residual[o];
    p.y[o] = y;
  }
}

// ------------------------------------------------------------------------------------------
// The products of a short prompt's layers, whose activations stay planes from product to product (launch_gemm_blk_short): what finishes 32
// outputs of a token scales them by a power of two of their largest and leaves them in the order of the matrix operands, with the sum of their
// squares; the norm's gain is multiplied in by the writer, its root divided by at the end of the reader.  So a layer has 5 launches instead of 10 - the rotated
// K and the V go into the cache from the product that makes them, and the attention leaves planes too - and a
// wave requests its operands straight into registers, one contiguous KB an instruction, all of a short width at once: a width of 2048 comes in
// one round trip, where the cut tiles above take one a chunk of 64 columns and stage them in LDS.
//   planes: tile of 16 tokens, block of 32 columns, [64 lanes][8 halfs]; scales and squares: tile, block, [16 tokens].
// A work-group's waves cut the width of 16 tokens x 32 rows (PAIR: 32 up rows and their 32 gate rows) and meet in LDS at the end, a result a thread.  hi and lo
// are summed apart, every second block with its sign changed, in chains of eight blocks (FINE above).
// What bounds it: a launch, a round trip and the requests themselves, which touch a line a row of weights: 14 a chunk (the scales one by one, eight
// bytes of a row) took 11.2 us for the down product of the 135M shape (576 x 1536, 37 tokens), 9 a chunk 8.2; tiles of 32 tokens 10.2.  Results that
// left as single halfs cost gate | up 1.7 us.  A layer of that prompt, kernels alone, us: q | k | v 5.4, attention 6.5, o 4.8, gate | up with
// SwiGLU 6.8, down 8.0 = 32; with launches of their own for the append (2.8) and the attention's planes (2.3) 36 and 1201 -> 1080 a prompt; with rows between
// the products 51 (four pre-passes of 4.1, products 5.2, 4.5, 5.4 and 9.4).
// ------------------------------------------------------------------------------------------
struct BlkShortParams {
  const uint8_t* q[3]; const uint8_t* d[3]; const float* bias[3]; int rows[3]; int y_off[3]; int seg_end[2]; int n_seg;     // up to three matrices of one type and width
  int cols, n_tok, n_row_groups, n_tok_tiles, half;   // half > 0: rows [0, half) are up, [half, 2 half) gate
  BlkPlanes x; int normed; float eps;                 // (x.squares are read where the rows are normed)
  float* y; int64_t y_stride; const float* residual;
  BlkPlanes out; const float* gain;                   // planes of the results, times a gain (out.hi null: none)
  KvRows kv;                                          // the second and third matrix are K and V: their results go into the cache (kv.k null: to y)
};
constexpr int BS_NW = 8;
template <int QT, bool PAIR, bool TWICE, bool KV>       // TWICE: two work-groups a CU; KV: results of the second and third matrix go into the cache (a form of its own: 2 % of the others' time)
__global__ __launch_bounds__(64 * BS_NW) __attribute__((amdgpu_waves_per_eu(TWICE ? 4 : 2, TWICE ? 4 : 2))) void gemm_blk_short(const BlkShortParams p)
{
  constexpr int NW = BS_NW, RT = PAIR ? 4 : 2, P = TWICE ? (PAIR ? 1 : 2) : PAIR ? 3 : 4;      // row tiles of 16; chunks of 64 columns on their way to a wave
  __shared__ float sums[NW][RT * 4][64];
  __shared__ float s_sq[NW][16];
  __shared__ __align__(16) _Float16 s_out[2][512];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15, kg = lane >> 4;
  const int L = blockIdx.x, rg = (L & 7) + 8 * ((L >> 3) / p.n_tok_tiles), tile = (L >> 3) % p.n_tok_tiles;     // (the token tiles of a row group share an XCD and its L2)
  if (rg >= p.n_row_groups) return;
  int sg = 0, rgl = rg;
  if (p.n_seg > 1 && rg >= p.seg_end[0]) { sg = 1; rgl = rg - p.seg_end[0]; }
  if (p.n_seg > 2 && rg >= p.seg_end[1]) { sg = 2; rgl = rg - p.seg_end[1]; }
  const float* const bias = p.bias[sg];
  const int rows = p.rows[sg], R0 = rgl * 32, K = p.cols, nb32 = K >> 5, n_chunks = (nb32 + 1) >> 1;
  const int c0 = n_chunks * wave / NW, c1 = n_chunks * (wave + 1) / NW;
  const _Float16 *const xh = p.x.hi + (int64_t)tile * nb32 * 512 + lane * 8, *const xl = p.x.lo + (int64_t)tile * nb32 * 512 + lane * 8;
  const float* const xs = p.x.scale + (int64_t)tile * nb32 * 16 + 4 * kg;
  // A request touches sixteen rows, a line each, so a chunk of a row is shared out over the four lanes of the row and changes hands in registers:
  // (Q8_0) 16 bytes a lane, (Q4_0) 8; the two scales of a row, of row tile kg.
  auto row_of = [&](int rt) { return (PAIR && rt >= 2 ? (int64_t)p.half : 0) + min(R0 + 16 * (rt & 1) + n, rows - 1); };     // rows past the end: the last one again, not written
  const uint8_t* wq[RT];
#pragma unroll
  for (int rt = 0; rt < RT; rt++) wq[rt] = p.q[sg] + row_of(rt) * (QT == CAI_Q8_0 ? K : K / 2) + (QT == CAI_Q8_0 ? 16 : 8) * kg;
  const uint8_t* const wd = p.d[sg] + (kg & 2 ? row_of(RT == 4 ? 2 + (kg & 1) : kg & 1) : row_of(kg & 1)) * (nb32 * 2);
  const bool odd = nb32 & 1;
  typedef std::conditional_t<QT == CAI_Q8_0, u32x4_b, uint2_b> Quants;
  struct Chunk { half8_b h[2], l[2]; f32x4_b sc[2]; Quants w[RT]; uint32_t d; };
  auto fetch = [&](int c, Chunk& x) {
#pragma unroll
    for (int b = 0; b < 2; b++) {                       // (behind the last block of an odd number of them: that one again, not used)
      const int kb = min(2 * c + b, nb32 - 1);
      x.h[b] = *reinterpret_cast<const half8_b*>(xh + kb * 512); x.l[b] = *reinterpret_cast<const half8_b*>(xl + kb * 512);
      x.sc[b] = *reinterpret_cast<const f32x4_b*>(xs + kb * 16);
    }
    // the last chunk of an odd number of blocks: the lanes of its second half stay on the first
    const int back = odd && 2 * c + 1 >= nb32 && kg >= 2 ? (QT == CAI_Q8_0 ? 32 : 16) : 0;
#pragma unroll
    for (int rt = 0; rt < RT; rt++) x.w[rt] = *reinterpret_cast<const Quants*>(wq[rt] + c * (QT == CAI_Q8_0 ? 64 : 32) - back);
    if (odd) x.d = *reinterpret_cast<const uint16_t*>(wd + c * 4) | (uint32_t)*reinterpret_cast<const uint16_t*>(wd + min(2 * c + 1, nb32 - 1) * 2) << 16;
    else x.d = *reinterpret_cast<const uint32_t*>(wd + c * 4);
  };
  Chunk r[P];
#pragma unroll
  for (int i = 0; i < P; i++) if (c0 + i < c1) fetch(c0 + i, r[i]);
  // what finishes this thread's result - row R0 + tid % 32, token tid / 32 - is requested behind them
  const int tl = tid >> 5, t = tile * 16 + tl, row = R0 + (tid & 31), rc = min(row, rows - 1);
  const int64_t at_y = (int64_t)min(t, p.n_tok - 1) * p.y_stride + p.y_off[sg] + rc;
  const float res = p.residual ? p.residual[at_y] : 0.0f, bs = bias ? bias[rc] : 0.0f, bs2 = PAIR && bias ? bias[p.half + rc] : 0.0f, gain = p.gain ? p.gain[rc] : 1.0f;
  const int hd = KV ? p.kv.head_dim : 1, pos = KV ? p.kv.pos[min(t, p.n_tok - 1)] : 0;
  float sn = 0.0f, cs = 1.0f;
  auto rotation = [&]() { if (KV && sg == 1 && p.kv.theta) sincosf((float)pos * p.kv.theta[(rc % hd) >> 1], &sn, &cs); };
  if (!TWICE) rotation();                               // (behind the requests, in front of what they bring; two work-groups a CU lack the registers)
  if (p.normed) {                                       // sums of squares: token tid % 16, a 32nd of the blocks
    float ss = 0.0f;
    for (int kb = tid >> 4; kb < nb32; kb += 4 * NW) ss += p.x.squares[((int64_t)tile * nb32 + kb) * 16 + n];
    ss += __shfl_xor(ss, 16); ss += __shfl_xor(ss, 32);
    if (kg == 0) s_sq[wave][n] = ss;
  }
  const f32x4_b zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4_b Y[RT], Z[RT], U[RT];
#pragma unroll
  for (int rt = 0; rt < RT; rt++) Y[rt] = Z[rt] = U[rt] = zero;
  auto use = [&](const Chunk& x, bool half) {
    uint32_t d[4];                                      // of each row tile, in all lanes of a row
    {
      const uint2_b a = __builtin_amdgcn_permlane16_swap(x.d, x.d, false, false);         // tiles 0 0 2 2, 1 1 3 3
      const uint2_b e = __builtin_amdgcn_permlane32_swap(a.x, a.x, false, false), o = __builtin_amdgcn_permlane32_swap(a.y, a.y, false, false);
      d[0] = e.x; d[2] = e.y; d[1] = o.x; d[3] = o.y;
    }
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
      uint32_t w0[2], w1[2];                            // a block's eight codes of this lane
      if constexpr (QT == CAI_Q8_0) {
        // lanes kg 0, 1 asked for block 0, kg 2, 3 for block 1: the halves change places, and each block is in all four
        const uint2_b xz = __builtin_amdgcn_permlane32_swap(x.w[rt].x, x.w[rt].z, false, false), yw = __builtin_amdgcn_permlane32_swap(x.w[rt].y, x.w[rt].w, false, false);
        w0[0] = xz.x; w1[0] = yw.x; w0[1] = xz.y; w1[1] = yw.y;
      } else {
        const uint2_b xx = __builtin_amdgcn_permlane32_swap(x.w[rt].x, x.w[rt].x, false, false), yy = __builtin_amdgcn_permlane32_swap(x.w[rt].y, x.w[rt].y, false, false);
        const int sh = kg & 2 ? 4 : 0;
        w0[0] = xx.x >> sh; w1[0] = yy.x >> sh; w0[1] = xx.y >> sh; w1[1] = yy.y >> sh;
      }
#pragma unroll
      for (int b = 0; b < 2; b++) {
        if (b && half) break;
        const half8_b W = codes8<QT>(w0[b], w1[b], 0, b);
        const float dh = __half2float(__ushort_as_half((unsigned short)(b ? d[rt] >> 16 : d[rt] & 0xffffu))), dv = b ? -dh : dh;
        const f32x4_b C = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.h[b], W, zero, 0, 0, 0), D = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.l[b], W, zero, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) { const float f = dv * x.sc[b][i]; Y[rt][i] = fmaf(f, C[i], Y[rt][i]); U[rt][i] = fmaf(f, D[i], U[rt][i]); }
      }
    }
  };
  for (int c = c0; c < c1; c += P) {
#pragma unroll
    for (int i = 0; i < P; i++) {
      if (c + i >= c1) break;
      use(r[i], 2 * (c + i) + 1 >= nb32);
      if (c + i + P < c1) fetch(c + i + P, r[i]);
      if (((c + i - c0) & 3) == 3)
#pragma unroll
        for (int rt = 0; rt < RT; rt++) { Z[rt] += Y[rt]; Y[rt] = zero; }
    }
  }
#pragma unroll
  for (int rt = 0; rt < RT; rt++)
#pragma unroll
    for (int i = 0; i < 4; i++) sums[wave][rt * 4 + i][lane] = Z[rt][i] + (Y[rt][i] + U[rt][i]);
  __syncthreads();
  // lane (n, kg) of a sum: row n of the tile, tokens 4 kg + i
  const int from = (tl >> 2) * 16 + (tid & 15), v = ((tid >> 4) & 1) * 4 + (tl & 3);
  float y = 0.0f, gate = 0.0f, inv = 1.0f;
#pragma unroll
  for (int w = 0; w < NW; w++) { y += sums[w][v][from]; if (PAIR) gate += sums[w][PAIR ? 8 + v : 0][from]; }
  if (p.normed) {
    float ss = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; w++) ss += s_sq[w][tl];
    inv = 1.0f / sqrtf(ss / (float)K + p.eps);
  }
  y = y * inv + bs;
  if constexpr (PAIR) y = silu_mul(y, gate * inv + bs2);
  else {
    y += res;
    if (KV && sg > 0) {                                 // two neighbouring lanes hold a pair of K
      if (TWICE) rotation();
      const float mate = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, y), 0xb1, 0xf, 0xf, false));
      if (sg == 1 && p.kv.theta) y = row & 1 ? sn * mate + cs * y : cs * y - sn * mate;
      const int64_t o = ((int64_t)(rc / hd) * p.kv.max_ctx + pos) * hd + rc % hd;
      void* const c = sg == 1 ? p.kv.k : p.kv.v;
      if (t < p.n_tok && row < rows) { if (p.kv.half) reinterpret_cast<__half*>(c)[o] = __float2half_rn(y); else reinterpret_cast<float*>(c)[o] = y; }
      return;
    }
    if (t < p.n_tok && row < rows) p.y[at_y] = y;
  }
  if (!p.out.hi) return;
  // (rows in whole blocks of 32: the lanes of a half-wave are one of them)
  const float x = y * gain;
  float m = finite_abs(x), ss = y * y;
#define BS_DPP(z, ctrl) __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, (z)), (ctrl), 0xf, 0xf, false))
  m = fmaxf(m, BS_DPP(m, 0xb1)); m = fmaxf(m, BS_DPP(m, 0x4e)); m = fmaxf(m, BS_DPP(m, 0x141)); m = fmaxf(m, BS_DPP(m, 0x140));
  ss += BS_DPP(ss, 0xb1); ss += BS_DPP(ss, 0x4e); ss += BS_DPP(ss, 0x141); ss += BS_DPP(ss, 0x140);
#undef BS_DPP
  m = fmaxf(m, __shfl_xor(m, 16)); ss += __shfl_xor(ss, 16);
  const int e = plane_exponent(m);
  _Float16 h, l; split_plane(x * ldexpf(1.0f, e), h, l);
  // (the work-group's results are one block of the planes: it leaves as whole lines; tokens past the end are its padding)
  const int at = plane_place(QT == CAI_Q8_0, tl, tid & 31);
  s_out[0][at] = h; s_out[1][at] = l;
  const int64_t blk = (int64_t)tile * (rows >> 5) + (R0 >> 5);
  if ((tid & 31) == 0) { p.out.scale[blk * 16 + tl] = ldexpf(1.0f, -e); p.out.squares[blk * 16 + tl] = ss; }
  __syncthreads();
  if (wave < 2) reinterpret_cast<u32x4_b*>((wave ? p.out.lo : p.out.hi) + blk * 512)[lane] = reinterpret_cast<const u32x4_b*>(s_out[wave])[lane];
}

// Float rows times a gain (or as they are) as such planes, with their sums of squares: the stream in front of the first layer, and what the attention leaves.  Eight
// lanes a block.
template <int QT>
__global__ __launch_bounds__(256) void blk_planes_kernel(const float* __restrict__ x, const float* __restrict__ gain, int K, int n4, BlkPlanes o)
{
  const int id = blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;
  if (id >= n4) return;                    // (whole blocks: K is a multiple of 32)
  const f32x4_b v = *reinterpret_cast<const f32x4_b*>(x + (int64_t)t * K + 4 * id), one = {1.0f, 1.0f, 1.0f, 1.0f}, g = gain ? *reinterpret_cast<const f32x4_b*>(gain + 4 * id) : one;
  float m = 0.0f, ss = 0.0f, u[4];
#pragma unroll
  for (int i = 0; i < 4; i++) { u[i] = v[i] * g[i]; m = fmaxf(m, finite_abs(u[i])); ss = fmaf(v[i], v[i], ss); }
#pragma unroll
  for (int d = 4; d; d >>= 1) { m = fmaxf(m, __shfl_xor(m, d)); ss += __shfl_xor(ss, d); }
  const int e = plane_exponent(m);
  const float s = ldexpf(1.0f, e);
  typedef _Float16 half4_b __attribute__((ext_vector_type(4)));
  half4_b h, l;
#pragma unroll
  for (int i = 0; i < 4; i++) { _Float16 a, b; split_plane(u[i] * s, a, b); h[i] = a; l[i] = b; }
  const int64_t blk = (int64_t)(t >> 4) * (K >> 5) + (id >> 3), at = blk * 512 + plane_place(QT == CAI_Q8_0, t & 15, 4 * (id & 7));
  *reinterpret_cast<half4_b*>(o.hi + at) = h; *reinterpret_cast<half4_b*>(o.lo + at) = l;
  if ((id & 7) == 0) { o.scale[blk * 16 + (t & 15)] = ldexpf(1.0f, -e); o.squares[blk * 16 + (t & 15)] = ss; }
}

// ------------------------------------------------------------------------------------------
// Grouping of a prompt's (token, rank) slots by expert: perm lists the slots expert by expert, tile_tab cuts each expert's
// run into token tiles of at most `tile` slots.  One work-group; the order of the slots inside an expert's run depends on
// the arrival of LDS atomics, which does not matter: every result row is computed from its own activation row only.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void moe_group_kernel(const int32_t* expert, int n_slots, int n_experts, int tile, int max_tiles,
                                                         int32_t* perm, int32_t* tile_tab)
{
  __shared__ int cnt[512], off[512], cur[512], w_slots[8], w_tiles[8];
  for (int e = threadIdx.x; e < n_experts; e += blockDim.x) { cnt[e] = 0; cur[e] = 0; }
  __syncthreads();
  for (int s = threadIdx.x; s < n_slots; s += blockDim.x) atomicAdd(&cnt[min(max(expert[s], 0), n_experts - 1)], 1);
  __syncthreads();
  // a thread an expert (up to 512): its first slot and its first tile are sums over the experts before it (2040 slots of 64 experts: one
  // thread that walked the experts 8.4 us, so 4.6)
  const int e = threadIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = e < n_experts ? cnt[e] : 0, nt = (n + tile - 1) / tile;
  int so = n, to = nt;
  for (int d = 1; d < 64; d <<= 1) {
    const int a = __shfl_up(so, d, 64), b = __shfl_up(to, d, 64);
    if (lane >= d) { so += a; to += b; }
  }
  if (lane == 63 && wave < 8) { w_slots[wave] = so; w_tiles[wave] = to; }
  __syncthreads();
  so -= n; to -= nt;
  int all = 0;
  for (int w = 0; w < 8; w++) { if (w < wave) { so += w_slots[w]; to += w_tiles[w]; } all += w_tiles[w]; }
  if (e < n_experts) {
    off[e] = so;
    for (int k = 0; k < nt; k++) { int32_t* const t = tile_tab + 3 * (to + k); t[0] = e; t[1] = so + k * tile; t[2] = min(tile, n - k * tile); }
  }
  for (int t = all + threadIdx.x; t < max_tiles; t += blockDim.x) { tile_tab[3 * t] = 0; tile_tab[3 * t + 1] = 0; tile_tab[3 * t + 2] = 0; }
  __syncthreads();
  for (int s = threadIdx.x; s < n_slots; s += blockDim.x) {
    const int e = min(max(expert[s], 0), n_experts - 1);
    perm[off[e] + atomicAdd(&cur[e], 1)] = s;
  }
}

namespace {

template <void (*KERNEL)(BlkGemmParams)>
int launch_lds(int grid, int threads, size_t lds, const BlkGemmParams& p)
{
  static bool attr_done = false;
  if (!attr_done) {
    CAI_HIP(hipFuncSetAttribute((const void*)KERNEL, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_done = true;
  }
  hipLaunchKernelGGL(KERNEL, dim3(grid), dim3(threads), lds, ctx().stream, p);
  return CAI_OK;
}

// Row groups of `rows` weight rows (every matrix starts one of its own) x n_tiles token tiles
int blk_grid(BlkGemmParams& p, int rows, int n_tiles)
{
  p.n_row_groups = (p.rows + rows - 1) / rows;
  for (int i = 1; i < p.n_seg; i++) { p.seg_end[i - 1] = p.n_row_groups; p.n_row_groups += (p.rows2[i - 1] + rows - 1) / rows; }
  p.n_tok_tiles = n_tiles;
  return p.tile_tab ? n_tiles * p.n_row_groups : 8 * n_tiles * ((p.n_row_groups + 7) / 8);
}

template <int QT, bool ODD>
int launch_blk(const BlkGemmParams& p0, int n_tiles_grouped)
{
  BlkGemmParams p = p0;
  constexpr size_t WROW = QT == CAI_Q8_0 ? 64 : 32;                                    // quant bytes of a row's chunk
  auto tile = [&](auto tt_, auto nw_, int n_tiles) {
    constexpr int TT = tt_, NW = nw_;
    return launch_lds<gemm_blk_tile<QT, TT, ODD, NW>>(blk_grid(p, 32 * NW, n_tiles), 64 * NW, blk_depth(TT, NW) * (TT * 8192 + 32 * NW * (WROW + (ODD ? 8 : 4))), p);
  };
  auto cut = [&](auto rt_, auto nw_) {
    constexpr int RT = rt_, NW = nw_;
    const int grid = blk_grid(p, 32 * RT, (p.n_tok + 31) / 32), lds = NW * 2 * (8192 + RT * 32 * WROW + (ODD ? 512 : 256));
    if (p.n_tok <= 16) return launch_lds<gemm_blk_cut<QT, RT, NW, ODD, true>>(grid, 64 * NW, lds, p);
    return launch_lds<gemm_blk_cut<QT, RT, NW, ODD>>(grid, 64 * NW, lds, p);
  };
  typedef std::integral_constant<int, 1> One; typedef std::integral_constant<int, 2> Two; typedef std::integral_constant<int, 3> Three;
  typedef std::integral_constant<int, 4> Four; typedef std::integral_constant<int, 7> Seven; typedef std::integral_constant<int, 8> Eight;
  // An expert's runs: 128 x 64, two work-groups a CU, us as 256 x 64 : 128 x 64: 255 tokens to 64 experts of which few are chosen (45 tiles of 64 slots), gate | up
  // of 2048 x 2048 88 : 82, down of 2048 x 1024 52 : 47; whole prompts, four layers of width 2048, 32 experts of 1024: 17 tokens 540 : 480, 100 tokens 641 : 580,
  // 700 1906 : 1767, 2048 4818 : 4433; eight of 1536 at width 4096, 2048 tokens 6120 : 5640; Q4_0, 255 tokens 764 : 748, eight of 2048 at 3072, 1024 tokens 2775 : 2565.
  // (Two chunks in LDS and three work-groups a CU: the same to 4 % slower; 256 x 64 with two chunks and two work-groups 2 to 3 % slower than with one.)
  if (p.tile_tab) return tile(Two(), Four(), n_tiles_grouped);
  // A form's time is its rounds over the chip times what a round takes, in ns a column (Q8_0; with a full chip): cut tiles of 32 rows
  // 3.0, of 64 rows 4.6 (one work-group a CU) or 9.0 (three waves, two work-groups a CU: better from the second round on, 6144 x 2048
  // and 255 tokens 34.2 us against 35.5), tiles of 256 x 64 18 (13 if half empty), of 256 x 128 27.  At the lines, with the pre-pass:
  //   2048 x 2048:  128 tokens  32 rows 13.5  64 rows 16.0     255: 20.3, 17.4     1024:  64 rows 51.5  256 x 64 51.7
  //   6144 x 2048:  511 tokens  64 rows 59.8  256 x 64 51.4   1024: 256 x 64 96, 256 x 128 77
  //   3072 x 576:   511 tokens  64 rows 18.9  256 x 64 21.6   1024: 30.4, 24.8
  const int n_cu = ctx().n_cu, tok32 = (p.n_tok + 31) / 32;
  auto groups = [&](int rows) {
    int g = (p.rows + rows - 1) / rows;
    for (int i = 1; i < p.n_seg; i++) g += (p.rows2[i - 1] + rows - 1) / rows;
    return (int64_t)g;
  };
  auto rounds = [](int64_t wgs, int n) { return (double)((wgs + n - 1) / n); };
  if (groups(32) * tok32 <= n_cu) return cut(One(), Seven());
  if (groups(64) * tok32 <= n_cu) return cut(Two(), Four());
  // 128 x 64 of four waves takes 0.6 of the time of 256 x 64 while a CU has one of them (two: all of it), so where they fill the chip once and cut tiles
  // go into a second round by more than half: with the pre-pass, cut : 128 x 64
  //   2048 x 2048, 1024 tokens 49.5 : 38.5   4096 x 4096, 511: 75.3 : 62.2   14336 x 4096, 100: 64.1 : 57.2   4096 x 14336, 511: 253 : 190
  //   (6144 x 2048, 255, a round and a half: 33.0 : 34.6)
  if (groups(64) * tok32 > 3 * n_cu && groups(128) * ((p.n_tok + 63) / 64) <= n_cu) return tile(Two(), Four(), (p.n_tok + 63) / 64);
  const double c64 = 9.0 * rounds(groups(64) * tok32, 2 * n_cu);
  const double t64 = (p.n_tok <= 32 ? 13.0 : 18.0) * rounds(groups(256) * ((p.n_tok + 63) / 64), n_cu);
  const double t128 = 27.0 * rounds(groups(256) * ((p.n_tok + 127) / 128), n_cu);
  if (c64 <= t64 && c64 <= t128) return cut(Two(), Three());
  return t128 <= t64 ? tile(Four(), Eight(), (p.n_tok + 127) / 128) : tile(Two(), Eight(), (p.n_tok + 63) / 64);
}

int launch_blk(const cai_qw_s* w, const BlkGemmParams& p0, int n_tiles_grouped)
{
  auto go = [&](const BlkGemmParams& p) {
    const bool odd = (p.cols >> 5) & 1;
    if (w->qtype == CAI_Q8_0) return odd ? launch_blk<CAI_Q8_0, true>(p, n_tiles_grouped) : launch_blk<CAI_Q8_0, false>(p, n_tiles_grouped);
    return odd ? launch_blk<CAI_Q4_0, true>(p, n_tiles_grouped) : launch_blk<CAI_Q4_0, false>(p, n_tiles_grouped);
  };
  if (p0.tile_tab) return go(p0);
  const int64_t most = blk_piece(p0.cols);
  for (int64_t t = 0; t < p0.n_tok; t += most) {
    BlkGemmParams p = p0;
    p.n_tok = (int)std::min<int64_t>(most, p0.n_tok - t);
    p.xhi += t * p0.cols; p.xlo += t * p0.cols; p.sinv += t; p.y += t * p0.y_stride;
    if (p.residual) p.residual += t * p0.y_stride;
    const int rc = go(p);
    if (rc) return rc;
  }
  return CAI_OK;
}

// ------------------------------------------------------------------------------------------
// Types kept as their stored stream (Q2_K, Q3_K, Q4_1, Q5_0, Q5_1): a panel of rows at a time is rewritten as signed bytes with an f16 scale
// a block of 32 - and, for the types with minima, a float a sixteen - and multiplied by the kernel above.  Codes and scales are exact:
// Q5_0 q - 16; Q4_1, Q5_1 q - 8, q - 16 with m + 8 d, m + 16 d; Q3_K (32 - scale) * q with -d; Q2_K, all doubled, scale * (2 q - c) with c d scale - 2 dmin min,
// c the whole number of 0 .. 6 next to 2 dmin min / (d scale).
// (Codes about zero: with q from 0 up the two parts of a sum cancel, and its error doubles.)
// In place of passes of eight tokens through the float walk, bound by its VALU work: 18944 x 3584 with 200 tokens Q3_K 2282 -> 186 us,
// Q4_1 1321 -> 269, with 16 tokens 183 -> 77, 106 -> 95; 3584 x 3584 with 16 tokens 52 -> 26, 39 -> 31.  Rewriting takes about 2 bytes of
// memory traffic a weight (40 us of the first), the minima half the time of the products; up to eight tokens the walk is one pass and stays.
// ------------------------------------------------------------------------------------------
template <int QT>
__global__ __launch_bounds__(256) void raw_expand_kernel(const uint8_t* __restrict__ raw, int64_t row_bytes, int n_rows, int runs, int8_t* __restrict__ q, uint16_t* __restrict__ d, float* __restrict__ m16)
{
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (id >= (int64_t)n_rows * runs) return;
  const int row = (int)(id / runs), run = (int)(id % runs);
  const uint8_t* const base = raw + row * row_bytes;
  uint32_t out[4]; float m = 0.0f; uint16_t dh;
  auto put = [&](int t, int v) { const uint32_t byte = (uint32_t)(v & 255) << (8 * (t & 3)); out[t >> 2] = (t & 3) ? out[t >> 2] | byte : byte; };
  constexpr int BB = raw_block_bytes(QT);
  if constexpr (raw_block_elems(QT) == 32) {
    const uint8_t* const blk = base + (int64_t)(run >> 1) * BB;
    const int half = run & 1;
    uint32_t qs[4];
    raw_load16<QT == CAI_Q5_0 ? 2 : 4>(blk + (QT == CAI_Q4_1 ? 4 : QT == CAI_Q5_0 ? 6 : 8), qs);
    dh = *reinterpret_cast<const uint16_t*>(blk);
    const uint32_t qh = QT == CAI_Q4_1 ? 0u : (QT == CAI_Q5_0 ? raw_u32_a2(blk + 2) : *reinterpret_cast<const uint32_t*>(blk + 4)) >> (16 * half);
#pragma unroll
    for (int t = 0; t < 16; t++) {
      const int b = raw_byte(qs, t), nib = half ? (b >> 4) : (b & 15);
      put(t, QT == CAI_Q4_1 ? nib - 8 : (nib | (int)(((qh >> t) & 1u) << 4)) - 16);
    }
    if constexpr (QT != CAI_Q5_0) m = fmaf(raw_half(blk), QT == CAI_Q4_1 ? 8.0f : 16.0f, raw_half(blk + 2));
  } else {
    const uint8_t* const blk = base + (int64_t)(run >> 4) * BB;
    const int r = run & 15, sh = 2 * ((r >> 1) & 3);
    uint32_t qs[4];
    if constexpr (QT == CAI_Q2_K) {
      const int sc = blk[r] & 15, mn = blk[r] >> 4;
      const float ds = raw_half(blk + 80) * (float)sc, dm = raw_half(blk + 82) * (float)(2 * mn);
      const int c = (int)fminf(fmaxf(rintf(dm / ds), 0.0f), 6.0f);      // (0 / 0 counts as 0)
      raw_load16<4>(blk + 16 + (r >> 3) * 32 + 16 * (r & 1), qs);
      dh = *reinterpret_cast<const uint16_t*>(blk + 80);
#pragma unroll
      for (int t = 0; t < 16; t++) put(t, sc * (2 * ((raw_byte(qs, t) >> sh) & 3) - c));
      m = fmaf(ds, (float)c, -dm);
    } else {
      const int sc = -q3k_scale(blk + 96, r), bit = r >> 1;
      uint32_t hm[4];
      raw_load16<2>(blk + 32 + (r >> 3) * 32 + 16 * (r & 1), qs);
      raw_load16<2>(blk + 16 * (r & 1), hm);
      dh = *reinterpret_cast<const uint16_t*>(blk + 108) ^ 0x8000u;
#pragma unroll
      for (int t = 0; t < 16; t++) put(t, sc * (((raw_byte(qs, t) >> sh) & 3) - ((((raw_byte(hm, t) >> bit) & 1) ^ 1) << 2)));
    }
  }
  *reinterpret_cast<uint4*>(q + id * 16) = make_uint4(out[0], out[1], out[2], out[3]);
  if ((run & 1) == 0) d[id >> 1] = dh;
  if constexpr (QT == CAI_Q2_K || QT == CAI_Q4_1 || QT == CAI_Q5_1) m16[id] = m;
}

// sums of sixteen neighbours of the activation planes
__global__ __launch_bounds__(256) void plane_sums_kernel(const _Float16* __restrict__ hi, const _Float16* __restrict__ lo, int64_t n, float* __restrict__ s16)
{
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;      // eight values each
  if (id >= n) return;
  const half8_b h = *reinterpret_cast<const half8_b*>(hi + id * 8), l = *reinterpret_cast<const half8_b*>(lo + id * 8);
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; i++) s += (float)h[i] + (float)l[i];
  s += __shfl_xor(s, 1);
  if ((id & 1) == 0) s16[id >> 1] = s;
}

struct RawWs { uint8_t* q = nullptr; float* s16 = nullptr; size_t q_cap = 0, s_cap = 0; };
RawWs g_raw;
constexpr int64_t RAW_PANEL = (int64_t)64 << 20;       // weights of a panel: its bytes stay in the last-level cache between the two launches

constexpr bool raw_has_minima(int qt) { return qt == CAI_Q2_K || qt == CAI_Q4_1 || qt == CAI_Q5_1; }
int64_t raw_panel(const cai_qw_s* w) { return std::min((w->rows + 63) / 64 * 64, std::max<int64_t>(64, RAW_PANEL / w->cols / 64 * 64)); }
int64_t raw_piece(const cai_qw_s* w) { return std::min<int64_t>(4096, blk_piece(w->cols)); }     // (4096: the sums of sixteen are bounded)

template <int QT>
int launch_raw(const cai_qw_s* w, const BlkGemmParams& p0)
{
  constexpr bool MIN = raw_has_minima(QT);
  const int64_t K = w->cols, rows = w->rows, panel = raw_panel(w);
  hipStream_t st = ctx().stream;
  if (MIN) {
    const int64_t n8 = (int64_t)p0.n_tok * K / 8;
    hipLaunchKernelGGL(plane_sums_kernel, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, st, p0.xhi, p0.xlo, n8, g_raw.s16);
  }
  const int64_t row_bytes = K / raw_block_elems(QT) * raw_block_bytes(QT);
  const int n_cu = ctx().n_cu, tok32 = (p0.n_tok + 31) / 32;
  for (int64_t r0 = 0; r0 < rows; r0 += panel) {
    BlkGemmParams p = p0;
    const int n = (int)std::min(panel, rows - r0), runs = (int)(K / 16);
    uint16_t* const d = reinterpret_cast<uint16_t*>(g_raw.q + panel * K);
    float* const m16 = reinterpret_cast<float*>(g_raw.q + panel * K / 16 * 17);
    hipLaunchKernelGGL(raw_expand_kernel<QT>, dim3((unsigned)(((int64_t)n * runs + 255) / 256)), dim3(256), 0, st, w->data + r0 * row_bytes, row_bytes, n, runs, (int8_t*)g_raw.q, d, m16);
    p.q = g_raw.q; p.d = reinterpret_cast<const uint8_t*>(d); p.rows = n; p.m16 = m16; p.s16 = g_raw.s16;
    if (p.bias) p.bias += r0;
    p.y += r0;
    if (p.residual) p.residual += r0;
    auto cut = [&](auto rt_, auto nw_, auto odd_) {
      constexpr int RT = rt_, NW = nw_; constexpr bool ODD = odd_;
      return launch_lds<gemm_blk_cut<CAI_Q8_0, RT, NW, ODD, true, MIN>>(blk_grid(p, 32 * RT, tok32), 64 * NW, NW * 2 * (8192 + RT * 2048 + (ODD ? 512 : 256) + (MIN ? 512 + 512 * RT : 0)), p);
    };
    // (always cut tiles, whose sums are short chains: 0.95e-7 off 64 bits at width 3584, the float walk of eight tokens a pass 1.5e-7; large tiles 2e-7)
    auto form = [&](auto odd_) {
      if ((int64_t)((n + 31) / 32) * tok32 <= n_cu) return cut(std::integral_constant<int, 1>(), std::integral_constant<int, 6>(), odd_);
      if ((int64_t)((n + 63) / 64) * tok32 <= n_cu || MIN) return cut(std::integral_constant<int, 2>(), std::integral_constant<int, 4>(), odd_);
      return cut(std::integral_constant<int, 2>(), std::integral_constant<int, 3>(), odd_);
    };
    const int rc = (K >> 5) & 1 ? form(std::true_type()) : form(std::false_type());
    if (rc) return rc;
  }
  return CAI_OK;
}

}  // namespace

bool gemm_blk_supported(const cai_qw_s* w) { return (w->qtype == CAI_Q8_0 || w->qtype == CAI_Q4_0) && w->cols % 32 == 0 && w->cols <= BLK_MAX_COLS; }

// Dense: y[t][rows] = W x[t] (+ bias) (+ residual) for the n_tok prepared activation rows.
int launch_gemm_blk(const cai_qw_s* w, const _Float16* xhi, const _Float16* xlo, const float* sinv, int n_tok, float* y, int64_t y_stride,
                    const float* residual)
{
  if (!gemm_blk_supported(w)) return set_error(CAI_ERR_UNSUPPORTED, "prompt gemm: weight type %d", w->qtype);
  BlkGemmParams p{};
  p.q = w->data; p.d = w->aux; p.bias = w->bias; p.rows = (int)w->rows; p.cols = (int)w->cols;
  p.xhi = xhi; p.xlo = xlo; p.sinv = sinv; p.n_tok = n_tok; p.y = y; p.y_stride = y_stride; p.residual = residual;
  p.x_div = 1; p.expert_rows = 0; p.post = 1.0f;
  return launch_blk(w, p, 0);
}

// Up to three matrices of one type and width in one launch: y[t][y_off[i] + r] = (W_i x[t])[r] (+ bias_i)
bool gemm_blk_multi_supported(const cai_qw_s* const* ws, int n_w)
{
  if (n_w < 1 || n_w > 3 || !gemm_blk_supported(ws[0])) return false;
  for (int i = 1; i < n_w; i++) if (ws[i]->qtype != ws[0]->qtype || ws[i]->cols != ws[0]->cols) return false;
  return true;
}
int launch_gemm_blk_multi(const cai_qw_s* const* ws, const int* y_off, int n_w, const _Float16* xhi, const _Float16* xlo, const float* sinv,
                          int n_tok, float* y, int64_t y_stride)
{
  if (!gemm_blk_multi_supported(ws, n_w)) return set_error(CAI_ERR_UNSUPPORTED, "prompt gemm: %d matrices in one launch", n_w);
  const cai_qw_s* w = ws[0];
  BlkGemmParams p{};
  p.q = w->data; p.d = w->aux; p.bias = w->bias; p.rows = (int)w->rows; p.cols = (int)w->cols;
  p.xhi = xhi; p.xlo = xlo; p.sinv = sinv; p.n_tok = n_tok; p.y = y + y_off[0]; p.y_stride = y_stride; p.residual = nullptr;
  p.x_div = 1; p.expert_rows = 0; p.post = 1.0f; p.n_seg = n_w;
  for (int i = 1; i < n_w; i++) { p.q2[i - 1] = ws[i]->data; p.d2[i - 1] = ws[i]->aux; p.bias2[i - 1] = ws[i]->bias; p.rows2[i - 1] = (int)ws[i]->rows; p.y_off2[i - 1] = y_off[i] - y_off[0]; }
  return launch_blk(w, p, 0);
}

// Whether the products of a layer go through gemm_blk_short: all of them of one type, in whole blocks of 32 rows where their results become planes, and each
// of at most two work-groups of 16 tokens x 32 rows a CU.  Beyond that the tiles that share their operands are faster than the launches they
// need.  Prompts, us, one product after the other | this way: six layers of 2048 / ffn 5632 in Q8_0, 24 tokens (352 work-groups of gate | up) 574 | 550, 64 tokens (704)
// 684 | 649 .. 728; eight of 1024 / 4096, 64 tokens (512) 610 | 577, 100 (896) 693 | 701; four of 4096 / 14336, 24 tokens (896) 768 | 809; twelve of
// 576 / 1536, 37 tokens (144) 576 | 525 (Q4_0 653 | 512), 128 (384) 661 | 603.  Up to one work-group a CU registers for three or four chunks a wave, past that for two work-groups:
// 1024 / 4096, 64 tokens 591 | 577, 24 tokens 501 | 515.
bool blk_short_wanted(const cai_qw_s* wq, const cai_qw_s* wk, const cai_qw_s* wv, const cai_qw_s* wo, const cai_qw_s* wgu, const cai_qw_s* wd, int n_tok)
{
  const cai_qw_s* ws[6] = {wq, wk, wv, wo, wgu, wd};
  for (const cai_qw_s* w : ws)
    if (!w || !gemm_blk_supported(w) || w->qtype != wq->qtype || prompt_route(w, n_tok) != 2) return false;
  if (wo->rows % 32 || wgu->rows % 64 || wd->rows != wo->rows || wd->cols * 2 != wgu->rows || wq->cols != wo->rows || wk->cols != wq->cols || wv->cols != wq->cols || wgu->cols != wo->rows || wo->cols != wq->rows) return false;
  const int64_t tiles = (n_tok + 15) / 16, most = 2 * ctx().n_cu;
  return ((wq->rows + 31) / 32 + (wk->rows + 31) / 32 + (wv->rows + 31) / 32) * tiles <= most && wo->rows / 32 * tiles <= most && wd->cols / 32 * tiles <= most;
}

// y[t][y_off[i] + r] = (W_i x[t])[r] (+ bias_i) (+ residual), or with half > 0 (one matrix of 2 half rows) up * silu(gate), which only out receives; eps >= 0: x is the
// stream, to be normed; out: planes of the results times a gain, for the next product
int launch_gemm_blk_short(const cai_qw_s* const* ws, const int* y_off, int n_w, const BlkPlanes& x, float eps, int n_tok, float* y, int64_t y_stride, const float* residual, int half,
                          const BlkPlanes& out, const float* gain, const KvRows& kv)
{
  const cai_qw_s* w = ws[0];
  if (!gemm_blk_multi_supported(ws, n_w) || (half && (n_w != 1 || !out.hi || w->rows != 2 * (int64_t)half || half % 32)) || (out.hi && (n_w != 1 || w->rows % 32)))
    return set_error(CAI_ERR_UNSUPPORTED, "short prompt: %d matrices of %lld rows", n_w, (long long)w->rows);
  BlkShortParams p{};
  p.cols = (int)w->cols; p.n_tok = n_tok; p.n_tok_tiles = (n_tok + 15) / 16; p.half = half; p.x = x; p.normed = eps >= 0.0f; p.eps = eps;
  p.y = y; p.y_stride = y_stride; p.residual = residual; p.out = out; p.gain = gain; p.n_seg = n_w; p.kv = kv;
  for (int i = 0; i < n_w; i++) { p.q[i] = ws[i]->data; p.d[i] = ws[i]->aux; p.bias[i] = ws[i]->bias; p.rows[i] = half ? half : (int)ws[i]->rows; p.y_off[i] = y_off[i]; }
  for (int i = 0; i < n_w; i++) { if (i) p.seg_end[i - 1] = p.n_row_groups; p.n_row_groups += (p.rows[i] + 31) / 32; }
  const dim3 grid(8 * p.n_tok_tiles * ((p.n_row_groups + 7) / 8)), blk(64 * BS_NW);
  const bool twice = p.n_row_groups * p.n_tok_tiles > ctx().n_cu;
#define SHORT_T(QT, PAIR, KV) do { if (twice) hipLaunchKernelGGL((gemm_blk_short<QT, PAIR, true, KV>), grid, blk, 0, ctx().stream, p); \
                                   else hipLaunchKernelGGL((gemm_blk_short<QT, PAIR, false, KV>), grid, blk, 0, ctx().stream, p); } while (0)
#define SHORT(QT) do { if (half) SHORT_T(QT, true, false); else if (kv.k) SHORT_T(QT, false, true); else SHORT_T(QT, false, false); } while (0)
  if (w->qtype == CAI_Q8_0) SHORT(CAI_Q8_0); else SHORT(CAI_Q4_0);
#undef SHORT
#undef SHORT_T
  return CAI_OK;
}
int launch_blk_planes(const cai_qw_s* w, const float* x, const float* gain, int n_tok, const BlkPlanes& o)      // for products with w
{
  const int K = (int)w->cols;
  const dim3 grid((K / 4 + 255) / 256, n_tok);
  if (w->qtype == CAI_Q8_0) hipLaunchKernelGGL(blk_planes_kernel<CAI_Q8_0>, grid, dim3(256), 0, ctx().stream, x, gain, K, K / 4, o);
  else hipLaunchKernelGGL(blk_planes_kernel<CAI_Q4_0>, grid, dim3(256), 0, ctx().stream, x, gain, K, K / 4, o);
  return CAI_OK;
}

// Two sets of planes, of whole tiles of 16 tokens; grown, never inside a capture (prompts are not captured)
struct ShortWs { BlkPlanes p[2]; size_t cap[2] = {0, 0}; };
static ShortWs g_short;
void blk_short_release()
{
  for (BlkPlanes& b : g_short.p) { void* q[] = {b.hi, b.lo, b.scale, b.squares}; for (void* v : q) if (v) (void)hipFree(v); }
  g_short = ShortWs();
}
int blk_short_planes(int n_tok, int width0, int width1, BlkPlanes (&out)[2])
{
  const size_t tok = (size_t)(n_tok + 15) / 16 * 16, need[2] = {tok * width0, tok * width1};
  for (int i = 0; i < 2; i++) {
    if (need[i] > g_short.cap[i]) {
      CAI_HIP(hipStreamSynchronize(ctx().stream));
      BlkPlanes& b = g_short.p[i];
      void* q[] = {b.hi, b.lo, b.scale, b.squares};
      for (void* v : q) if (v) (void)hipFree(v);
      b = BlkPlanes(); g_short.cap[i] = 0;
      const size_t n = std::max(need[i], (size_t)128 * (i ? width1 : width0));
      CAI_HIP(hipMalloc((void**)&b.hi, n * 2)); CAI_HIP(hipMalloc((void**)&b.lo, n * 2)); CAI_HIP(hipMalloc((void**)&b.scale, n / 8)); CAI_HIP(hipMalloc((void**)&b.squares, n / 8));
      g_short.cap[i] = n;
    }
    out[i] = g_short.p[i];
  }
  return CAI_OK;
}

bool gemm_raw_supported(const cai_qw_s* w)
{
  return (w->qtype == CAI_Q2_K || w->qtype == CAI_Q3_K || w->qtype == CAI_Q4_1 || w->qtype == CAI_Q5_0 || w->qtype == CAI_Q5_1) && w->cols <= BLK_MAX_COLS;
}
void raw_release()
{
  if (g_raw.q) (void)hipFree(g_raw.q);
  if (g_raw.s16) (void)hipFree(g_raw.s16);
  g_raw = RawWs();
}
// bytes of a panel (code 1, f16 scale 1 / 16, float minimum 4 / 16 a weight) and floats of a piece's sums: the larger of what need[] holds and this
void raw_needs(const cai_qw_s* w, int n_tok, size_t (&need)[2])
{
  if (!gemm_raw_supported(w)) return;
  need[0] = std::max(need[0], (size_t)raw_panel(w) * w->cols * 21 / 16);
  if (raw_has_minima(w->qtype)) need[1] = std::max(need[1], (size_t)std::min<int64_t>(n_tok, raw_piece(w)) * w->cols / 16);
}
int raw_reserve(const size_t (&need)[2])      // (prompts are not captured: the buffers may move between two of them)
{
  if (need[0] > g_raw.q_cap || need[1] > g_raw.s_cap) CAI_HIP(hipStreamSynchronize(ctx().stream));
  if (need[0] > g_raw.q_cap) {
    if (g_raw.q) (void)hipFree(g_raw.q);
    g_raw.q = nullptr; g_raw.q_cap = 0;
    CAI_HIP(hipMalloc((void**)&g_raw.q, need[0])); g_raw.q_cap = need[0];
  }
  if (need[1] > g_raw.s_cap) {
    if (g_raw.s16) (void)hipFree(g_raw.s16);
    g_raw.s16 = nullptr; g_raw.s_cap = 0;
    CAI_HIP(hipMalloc((void**)&g_raw.s16, need[1] * 4)); g_raw.s_cap = need[1];
  }
  return CAI_OK;
}
int launch_gemm_raw(const cai_qw_s* w, const _Float16* xhi, const _Float16* xlo, const float* sinv, int n_tok, float* y, int64_t y_stride, const float* residual)
{
  if (!gemm_raw_supported(w)) return set_error(CAI_ERR_UNSUPPORTED, "prompt gemm: weight type %d", w->qtype);
  size_t need[2] = {0, 0};
  raw_needs(w, n_tok, need);
  const int rc0 = raw_reserve(need); if (rc0) return rc0;
  const int64_t most = raw_piece(w);
  for (int64_t t = 0; t < n_tok; t += most) {
    BlkGemmParams p{};
    p.bias = w->bias; p.cols = (int)w->cols; p.x_div = 1; p.post = w->qtype == CAI_Q2_K ? 0.5f : 1.0f;
    p.n_tok = (int)std::min<int64_t>(most, n_tok - t);
    p.xhi = xhi + t * w->cols; p.xlo = xlo + t * w->cols; p.sinv = sinv + t; p.y = y + t * y_stride; p.y_stride = y_stride;
    p.residual = residual ? residual + t * y_stride : nullptr;
    int rc;
    switch (w->qtype) {
      case CAI_Q2_K: rc = launch_raw<CAI_Q2_K>(w, p); break;
      case CAI_Q3_K: rc = launch_raw<CAI_Q3_K>(w, p); break;
      case CAI_Q4_1: rc = launch_raw<CAI_Q4_1>(w, p); break;
      case CAI_Q5_0: rc = launch_raw<CAI_Q5_0>(w, p); break;
      default: rc = launch_raw<CAI_Q5_1>(w, p); break;
    }
    if (rc) return rc;
  }
  return CAI_OK;
}

// Token tiles of the grouped launches: every expert may end with a partial tile
constexpr int MOE_TILE = 64;
int moe_group_max_tiles(int n_slots, int n_experts) { return (n_slots + MOE_TILE - 1) / MOE_TILE + n_experts; }

int launch_moe_group(const int32_t* expert, int n_slots, int n_experts, int32_t* perm, int32_t* tile_tab)
{
  if (n_experts > 512) return set_error(CAI_ERR_UNSUPPORTED, "moe grouping: %d experts (up to 512)", n_experts);
  hipLaunchKernelGGL(moe_group_kernel, dim3(1), dim3(1024), 0, ctx().stream, expert, n_slots, n_experts, MOE_TILE, moe_group_max_tiles(n_slots, n_experts), perm, tile_tab);
  return CAI_OK;
}

// Grouped: slot s (a token's rank-th expert) takes activation row s / x_div through the rows [e * expert_rows, + expert_rows)
// of the bank, e the slot's expert; the result goes to row s of y.
int launch_gemm_blk_grouped(const cai_qw_s* bank, int64_t expert_rows, const _Float16* xhi, const _Float16* xlo, const float* sinv, int x_div,
                            int n_slots, int n_experts, const int32_t* perm, const int32_t* tile_tab, float* y, int64_t y_stride)
{
  if (!gemm_blk_supported(bank)) return set_error(CAI_ERR_UNSUPPORTED, "grouped prompt gemm: weight type %d", bank->qtype);
  if (expert_rows <= 0 || bank->rows != expert_rows * n_experts) return set_error(CAI_ERR_INVALID, "grouped prompt gemm: bank of %lld rows is not %d windows of %lld", (long long)bank->rows, n_experts, (long long)expert_rows);
  if ((int64_t)((n_slots - 1) / x_div + 1) * bank->cols >= ((int64_t)1 << 31)) return set_error(CAI_ERR_UNSUPPORTED, "grouped prompt gemm: %d slots of width %lld", n_slots, (long long)bank->cols);
  BlkGemmParams p{};
  p.q = bank->data; p.d = bank->aux; p.bias = bank->bias; p.rows = (int)expert_rows; p.cols = (int)bank->cols;
  p.xhi = xhi; p.xlo = xlo; p.sinv = sinv; p.n_tok = n_slots; p.y = y; p.y_stride = y_stride; p.residual = nullptr;
  p.tile_tab = tile_tab; p.perm = perm; p.x_div = x_div; p.expert_rows = expert_rows;
  const int tiles = moe_group_max_tiles(n_slots, n_experts);
  return launch_blk(bank, p, tiles);
}

}  // namespace cai
