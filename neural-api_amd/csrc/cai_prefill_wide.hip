// Prompt products on wide tiles: BM weight rows x BN tokens per work-group, the activations of 64 columns at a time copied straight
// from memory into LDS while the 64 columns before them are multiplied.
//
// Accuracy contract of the other prompt kernels: the weights' integers (Q4_K, Q5_K: 6-bit scale times code, at most 63 * 31) are exact
// f16 operands, an activation is a power-of-two scaled pair of halfs hi + lo, products accumulate in 32 bits, d and dmin multiply the
// sums of a super-block in 32 bits.
//
// What bounds it: every useful product is two MFMAs (hi and lo), so the 2.5 PFLOP/s of the matrix cores are 1.25 useful.  A tile of
// 32 rows x 32 tokens x 16 columns takes its activations from LDS (2 x 1 KB) and its weights from registers, where they have to be
// made from nibbles first; with 64 x 64 per wave both are shared by two tiles, which leaves LDS (128 B a cycle) three quarters busy at
// the full MFMA rate, and the vector instructions that make the weights run beside the MFMAs of the SIMD's other wave.
// The weights are the B operand: a lane then holds results of ONE row, and that row's d and dmin are values it loaded itself.
#include "cai_layered.hpp"
#include "cai_gemv_common.hpp"
#include "cai_async_copy.hpp"
#include <algorithm>

namespace cai {

namespace {

typedef _Float16 half2_w __attribute__((ext_vector_type(2)));
typedef _Float16 half8_w __attribute__((ext_vector_type(8)));
typedef float float16_w __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_w __attribute__((ext_vector_type(4)));

struct WideParams {
  const uint8_t* w; const float* bias; int rows, cols;
  const _Float16* xhi; const _Float16* xlo; const _Float16* sxhi; const _Float16* sxlo; const float* sinv;
  int n_tok;
  float* y; int64_t y_stride; const float* residual;
  int n_row_groups, n_tok_tiles;
  int n_seg; int seg_end[2];                 // up to two more matrices of one type and width (q | k | v)
  const uint8_t* w2[2]; const float* bias2[2]; int rows2[2]; int y_off2[2];
  int swiglu_half;
  // The first n_whole tiles are one work-group each; the width of the others is cut into n_splits slices, which leave their sums in
  // part[tile - n_whole][slice][token of the tile][row of the tile]
  int n_whole, n_splits; float* part;
  int sum_wide;                              // gemm_wide_sum: four rows of a result lie on 16 bytes, and so do their bias and residual
};

__device__ __forceinline__ void wide_store(const WideParams& p, const float* bias, int64_t o, int row, float v)
{
  if (bias) v += bias[row];
  if (p.residual) v += p.residual[o];
  p.y[o] = v;
}
__device__ __forceinline__ void wide_store_pair(const WideParams& p, const float* bias, int64_t o, int row, float up, float gate)
{
  if (bias) { up += bias[row]; gate += bias[p.swiglu_half + row]; }
  p.y[o] = silu_mul(up, gate);
}

// tile -> row group and token tile.  The token tiles of a row group share id mod 8 (one XCD, whose L2 serves the re-reads of its weights)
// as far as there are eight row groups.
__device__ __forceinline__ void wide_tile(const WideParams& p, int i, int& rg, int& tt)
{
  const int whole8 = p.n_row_groups & ~7, body = whole8 * p.n_tok_tiles;
  if (i < body) { rg = (i & 7) + 8 * ((i >> 3) / p.n_tok_tiles); tt = (i >> 3) % p.n_tok_tiles; }
  else { const int j = i - body, r = p.n_row_groups - whole8; rg = whole8 + j % r; tt = j / r; }
}

__device__ __forceinline__ half2_w pk_codes(uint32_t v, uint32_t sel, half2_w s2, half2_w c2)
{
  return __builtin_elementwise_fma(__builtin_bit_cast(half2_w, __builtin_amdgcn_perm(0x64646464u, v, sel)), s2, c2);   // (1024 + q) * sc - 1024 * sc
}

}  // namespace

// 256 rows x 64 TT tokens, eight waves as 4 (rows) x 2 (tokens) of 64 rows x 32 TT tokens: one work-group per CU, two waves per SIMD.
// Everything the loop reads from memory is copied into LDS ahead of its use - activations (4 bytes a value) and nibbles of 64 columns
// into one of three buffers, the headers of the super-blocks and the block sums one super-block ahead - so that the loop holds no load
// whose arrival the compiler would wait for, and the waits count the copies.  The copies are what costs most beside the MFMAs: with 128
// rows a work-group needs 32 KB of activations for half the products, 37888 x 3584 x 2048 tokens took 1370 us instead of 1213
// (useful 398 and 458 TFLOP/s; a library product of 4096 f16 rows, the same MFMAs, takes 874 us).  x 511 tokens, by launch: 286 us beside 7.6 for the
// planes and 8.3 for the sums of cut tiles, the kernel of narrow tiles 369; 3584 x 18944 143 + 24 + 8.5 us, 229 + 24.
template <int QT, int TT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_wide_pf(const WideParams p)
{
  constexpr int BM = 256, BN = 64 * TT, RT = 2;
  constexpr int BB = QT == CAI_Q5_K ? 176 : 144, HB = QT == CAI_Q5_K ? 48 : 16;   // bytes of a super-block, of what lies before its nibbles
  constexpr int PLANE = BN * 128, BUF = 2 * PLANE;      // activations: [token][64 halfs] of a plane; hi | lo
  constexpr int XCOP = BUF / 1024 / 8;                  // 1 KB copies per wave and step
  constexpr int QBUF = BM * 32, HBUF = BM * HB, SXBUF = 2 * BN * 16;
  constexpr int HCOP = HB / 16 == 1 ? 1 : 2;            // copies per wave of headers and block sums (uniform over the waves: see copy_h)
  extern __shared__ __align__(1024) unsigned char wide_smem[];
  constexpr int QOFS = 3 * BUF, HOFS = QOFS + 3 * QBUF, SOFS = HOFS + 2 * HBUF;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, kg = lane >> 5, wr = wave & 3, wt = wave >> 2;
  const bool cut = (int)blockIdx.x >= p.n_whole;
  const int n_cut = p.n_row_groups * p.n_tok_tiles - p.n_whole, ci = cut ? ((int)blockIdx.x - p.n_whole) % n_cut : 0, slice = cut ? ((int)blockIdx.x - p.n_whole) / n_cut : 0;
  int rg, ttile; wide_tile(p, cut ? p.n_whole + ci : (int)blockIdx.x, rg, ttile);
  const uint8_t* wbase = p.w; const float* bias = p.bias; int rows = p.rows, yo = 0, rgl = rg;
  if (p.n_seg > 1 && rg >= p.seg_end[0]) { wbase = p.w2[0]; bias = p.bias2[0]; yo = p.y_off2[0]; rgl = rg - p.seg_end[0]; rows = p.rows2[0]; }
  if (p.n_seg > 2 && rg >= p.seg_end[1]) { wbase = p.w2[1]; bias = p.bias2[1]; yo = p.y_off2[1]; rgl = rg - p.seg_end[1]; rows = p.rows2[1]; }
  const int half = p.swiglu_half;             // rows 0..127 of the tile are up rows, 128..255 their gate rows
  const int R0 = half ? rgl * (BM / 2) : rgl * BM, T0 = ttile * BN;
  const int K = p.cols, nsb_all = K >> 8, nb32 = K >> 5;
  const int sb0 = cut ? nsb_all * slice / p.n_splits : 0, sb1 = cut ? nsb_all * (slice + 1) / p.n_splits : nsb_all;
  const int n_steps = 4 * (sb1 - sb0);
  auto tile_row = [&](int r) { return half ? min(R0 + (r & 127), half - 1) + (r >> 7) * half : min(R0 + r, rows - 1); };   // rows past the end: the last again

  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)wide_smem;
  uint32_t voff[XCOP];                        // activations: token rows past the end repeat the last token
#pragma unroll
  for (int i = 0; i < XCOP; i++) {
    // slot s of token row t holds columns 8 (s ^ ((t >> 1) & 7)) ..: sixteen neighbouring rows (128 bytes each) then cover all 64 banks
    // when one column group is read
    const int t = ((wave * XCOP + i) % (BN / 8)) * 8 + (lane >> 3), chunk = (lane & 7) ^ ((t >> 1) & 7);
    voff[i] = ((uint32_t)min(T0 + t, p.n_tok - 1) * (uint32_t)K + (uint32_t)chunk * 8u) * 2u;
  }
  const _Float16* const xplane = wave * XCOP >= BN / 8 ? p.xlo : p.xhi;        // a wave's copies are of one plane
  // nibbles: 32 bytes a row and step, one 16-byte piece per thread; the halves trade places in every second eight rows (banks)
  const uint32_t row_bytes = (uint32_t)(nsb_all * BB);
  const uint32_t qoff = (uint32_t)tile_row(tid >> 1) * row_bytes + (uint32_t)(HB + 16 * ((tid & 1) ^ ((tid >> 4) & 1)));
  // headers (HB bytes a row) and block sums (waves 4..7, the last round)
  uint32_t hoff[HCOP];
#pragma unroll
  for (int i = 0; i < HCOP; i++) {
    const int P = min(i * 512 + tid, HBUF / 16 - 1);
    hoff[i] = (uint32_t)tile_row(P / (HB / 16)) * row_bytes + (uint32_t)(P % (HB / 16)) * 16u;
  }
  const uint32_t soff = ((uint32_t)min(T0 + (tid & 255) % BN, p.n_tok - 1) * (uint32_t)nb32) * 2u;
  auto copy_x = [&](int step, int b) {        // past the last step the last one again, into a buffer nobody reads
    const int st = min(step, n_steps - 1), col = sb0 * 256 + st * 64;
#pragma unroll
    for (int i = 0; i < XCOP; i++) copy16_to_lds(lds0 + (uint32_t)(b * BUF + (wave * XCOP + i) * 1024), voff[i], xplane + col);
    copy16_to_lds(lds0 + (uint32_t)(QOFS + b * QBUF + wave * 1024), qoff, wbase + (int64_t)(sb0 + (st >> 2)) * BB + (st & 3) * 32);
  };
  auto copy_h = [&](int sb) {                 // HCOP copies per wave: waves 4..7 take the block sums in the round that the headers leave to them
    const int b = (sb - sb0) & 1, s = min(sb, sb1 - 1);
    const uint8_t* const blk = wbase + (int64_t)s * BB;
    if constexpr (HCOP == 2) copy16_to_lds(lds0 + (uint32_t)(HOFS + b * HBUF + wave * 1024), hoff[0], blk);
    if (wave < 4) copy16_to_lds(lds0 + (uint32_t)(HOFS + b * HBUF + (HCOP - 1) * 8192 + wave * 1024), hoff[HCOP - 1], blk);
    else {                                    // (of 64 tokens twice: every wave issues the same number of copies)
      const int k = (wave - 4) % (2 * BN / 64);
      copy16_to_lds(lds0 + (uint32_t)(SOFS + b * SXBUF + k * 1024), soff, (k < BN / 64 ? p.sxhi : p.sxlo) + s * 8);
    }
  };
  // operand of k-step (hl, t): columns 32 hl + 16 kg + 8 t .. + 7 of the 64
  uint32_t xa[4];
#pragma unroll
  for (int s = 0; s < 4; s++) xa[s] = (uint32_t)((wt * 32 * TT + n) * 128 + (((4 * (s >> 1) + 2 * kg + (s & 1)) ^ ((n >> 1) & 7)) << 4));
  const int lr0 = half ? wr * 32 + n : wr * 64 + n, lrs = half ? 128 : 32;     // row of the tile: lr0 + rt * lrs

  float16_w Y[RT][TT], C[RT][TT];
  const float16_w zero16 = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int rt = 0; rt < RT; rt++)
#pragma unroll
    for (int tt = 0; tt < TT; tt++) Y[rt][tt] = zero16;
  half8_w Xh[2][TT], Xl[2][TT], W[2][RT];
  u32x4_w h[RT], e[RT], q[RT], qn[RT];        // header, Q5_K: the lane's 16 bytes of fifth bits; 16 bytes of nibbles of this step and the next
  auto request = [&](int s, int b) {
    const unsigned char* const xb = wide_smem + b * BUF;
#pragma unroll
    for (int tt = 0; tt < TT; tt++) {
      Xh[s & 1][tt] = *reinterpret_cast<const half8_w*>(xb + xa[s] + tt * 4096);
      Xl[s & 1][tt] = *reinterpret_cast<const half8_w*>(xb + xa[s] + PLANE + tt * 4096);
    }
  };
  auto read_q = [&](int b, u32x4_w (&r)[RT]) {
#pragma unroll
    for (int rt = 0; rt < RT; rt++) r[rt] = *reinterpret_cast<const u32x4_w*>(wide_smem + QOFS + b * QBUF + (lr0 + rt * lrs) * 32 + ((kg ^ ((n >> 3) & 1)) << 4));
  };
  auto read_h = [&](int b) {
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
      h[rt] = *reinterpret_cast<const u32x4_w*>(wide_smem + HOFS + b * HBUF + (lr0 + rt * lrs) * HB);
      if constexpr (QT == CAI_Q5_K) e[rt] = *reinterpret_cast<const u32x4_w*>(wide_smem + HOFS + b * HBUF + (lr0 + rt * lrs) * HB + 16 + 16 * kg);
    }
  };
  auto make = [&](int c, int s) {
    const int hl = s >> 1, t = s & 1;
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
      uint32_t sc, mn; q4k_scale_pair(h[rt].y, h[rt].z, h[rt].w, c, sc, mn);
      const _Float16 f = (_Float16)(float)((sc >> (8 * hl)) & 0xffu), m = (_Float16)(-1024.0f) * f;
      const half2_w s2 = {f, f}, c2 = {m, m};
      uint32_t a = q[rt][2 * t], b = q[rt][2 * t + 1];
      if (hl) { a >>= 4; b >>= 4; }
      a &= 0x0f0f0f0fu; b &= 0x0f0f0f0fu;
      if constexpr (QT == CAI_Q5_K) { a |= ((e[rt][2 * t] >> (2 * c + hl)) & 0x01010101u) << 4; b |= ((e[rt][2 * t + 1] >> (2 * c + hl)) & 0x01010101u) << 4; }
      const half2_w w0 = pk_codes(a, 0x04010400u, s2, c2), w1 = pk_codes(a, 0x04030402u, s2, c2), w2 = pk_codes(b, 0x04010400u, s2, c2), w3 = pk_codes(b, 0x04030402u, s2, c2);
      W[s & 1][rt] = half8_w{w0.x, w0.y, w1.x, w1.y, w2.x, w2.y, w3.x, w3.y};
    }
  };

  copy_h(sb0); copy_x(0, 0); copy_x(1, 1);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0070);         // vmcnt(0) lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  read_h(0); read_q(0, q);
  request(0, 0); make(0, 0);

  // The meeting of the waves lies in the MIDDLE of a step of 64 columns: by then the copies of the next step have had a step's time, and
  // the operands of its first k-step are requested and made before this step's last products are issued, so no wave starts a step with
  // nothing to multiply.
  int buf = 0, step = 0;                      // buffer of the current step
  for (int sb = sb0; sb < sb1; sb++) {
#pragma unroll
    for (int c = 0; c < 4; c++, step++) {
      const int nbuf = buf == 2 ? 0 : buf + 1;
#pragma unroll
      for (int s = 0; s < 4; s++) {
        if (s < 3) request(s + 1, buf); else request(0, nbuf);
        if (s == 2) read_q(nbuf, qn);
        __builtin_amdgcn_sched_barrier(0);
        if (s < 3) make(c, s + 1);
        else {
#pragma unroll
          for (int rt = 0; rt < RT; rt++) q[rt] = qn[rt];
          if (c < 3) make(c + 1, 0);
        }
#pragma unroll
        for (int tt = 0; tt < TT; tt++)
#pragma unroll
          for (int rt = 0; rt < RT; rt++) C[rt][tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(Xh[s & 1][tt], W[s & 1][rt], c == 0 && s == 0 ? zero16 : C[rt][tt], 0, 0, 0);
#pragma unroll
        for (int tt = 0; tt < TT; tt++)
#pragma unroll
          for (int rt = 0; rt < RT; rt++) C[rt][tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(Xl[s & 1][tt], W[s & 1][rt], C[rt][tt], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (s == 1) {
          // The next step's copies have to be there; newer than they are, in the second step of a super-block, the HCOP copies of the next
          // one's headers.
          asm volatile("" ::: "memory");
          if (c == 1) __builtin_amdgcn_s_waitcnt(0x0F70 | HCOP); else __builtin_amdgcn_s_waitcnt(0x0F70);
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
          copy_x(step + 2, buf == 0 ? 2 : buf - 1);      // (the buffer of the step before: every wave is past it)
          if (c == 0) copy_h(sb + 1);
          asm volatile("" ::: "memory");
        }
      }
      buf = nbuf;
    }
    // + d * (codes) - dmin * (minima); the eight minima meet the block sums hi in the lower k, lo in the upper
    const int hb = (sb - sb0) & 1;
    half8_w M[RT]; float d[RT], dm[RT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
      const uint32_t m0 = h[rt].z & 0x3f3f3f3fu, m1 = ((h[rt].w >> 4) & 0x0f0f0f0fu) | ((h[rt].z >> 2) & 0x30303030u);
      const half2_w one = {(_Float16)1.0f, (_Float16)1.0f}, off = {(_Float16)(-1024.0f), (_Float16)(-1024.0f)};
      const half2_w a0 = pk_codes(m0, 0x04010400u, one, off), a1 = pk_codes(m0, 0x04030402u, one, off), a2 = pk_codes(m1, 0x04010400u, one, off), a3 = pk_codes(m1, 0x04030402u, one, off);
      M[rt] = half8_w{a0.x, a0.y, a1.x, a1.y, a2.x, a2.y, a3.x, a3.y};
      d[rt] = __half2float(__ushort_as_half((unsigned short)(h[rt].x & 0xffffu))); dm[rt] = -32.0f * __half2float(__ushort_as_half((unsigned short)(h[rt].x >> 16)));
    }
    read_h(hb ^ 1);                           // the next super-block's (past the last one its own again, not used)
    const unsigned char* const sxb = wide_smem + SOFS + hb * SXBUF + kg * BN * 16 + (wt * 32 * TT + n) * 16;
#pragma unroll
    for (int tt = 0; tt < TT; tt++) {
      const half8_w S = *reinterpret_cast<const half8_w*>(sxb + tt * 512);
#pragma unroll
      for (int rt = 0; rt < RT; rt++) {
        const float16_w Cm = __builtin_amdgcn_mfma_f32_32x32x16_f16(S, M[rt], zero16, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 16; v++) Y[rt][tt][v] = fmaf(dm[rt], Cm[v], fmaf(d[rt], C[rt][tt][v], Y[rt][tt][v]));
      }
    }
    make(0, 0);
  }

  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0070);         // copies past the last step still write into the buffers, which have to be this work-group's until then
  asm volatile("" ::: "memory");

  // ---- write: the lane holds row n of each row tile and tokens 8 g + 4 kg + i of each token tile ----
  if (cut) {
    float* const out = p.part + ((int64_t)ci * p.n_splits + slice) * (BN * BM) + lr0;
#pragma unroll
    for (int tt = 0; tt < TT; tt++)
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int tl = (wt * TT + tt) * 32 + 8 * (v >> 2) + 4 * kg + (v & 3);
        if (T0 + tl >= p.n_tok) continue;
#pragma unroll
        for (int rt = 0; rt < RT; rt++) out[tl * BM + rt * lrs] = Y[rt][tt][v];
      }
    return;
  }
#pragma unroll
  for (int tt = 0; tt < TT; tt++)
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int t = T0 + (wt * TT + tt) * 32 + 8 * (v >> 2) + 4 * kg + (v & 3);
      if (t >= p.n_tok) continue;
      const float si = p.sinv[t];
      if (half) {
        const int row = R0 + lr0;
        if (row < half) wide_store_pair(p, bias, (int64_t)t * p.y_stride + row, row, Y[0][tt][v] * si, Y[1][tt][v] * si);
      } else {
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
          const int row = R0 + lr0 + rt * lrs;
          if (row < rows) wide_store(p, bias, (int64_t)t * p.y_stride + yo + row, row, Y[rt][tt][v] * si);
        }
      }
    }
}

// The slices of a cut tile, added in order, and its results: a work-group takes eight tokens, a thread four rows of two of them (four up rows and
// their gate rows of one).  What it reads was written on other XCDs, so it is bound by those round trips: eight slices are requested at once, and what is
// added to the sums in front of them (one slice after another: 3584 rows x 511 tokens in four slices 12.0 us, 8.3 so).
template <int BN>
__global__ __launch_bounds__(256) void gemm_wide_sum(const WideParams p)
{
  constexpr int BM = 256, AT_ONCE = 8;
  const int ci = blockIdx.x, tid = threadIdx.x;
  int rg, ttile; wide_tile(p, p.n_whole + ci, rg, ttile);
  const float* bias = p.bias; int rows = p.rows, yo = 0, rgl = rg;
  if (p.n_seg > 1 && rg >= p.seg_end[0]) { bias = p.bias2[0]; yo = p.y_off2[0]; rgl = rg - p.seg_end[0]; rows = p.rows2[0]; }
  if (p.n_seg > 2 && rg >= p.seg_end[1]) { bias = p.bias2[1]; yo = p.y_off2[1]; rgl = rg - p.seg_end[1]; rows = p.rows2[1]; }
  const int half = p.swiglu_half, r = half ? 4 * (tid & 31) : 4 * (tid & 63), row = half ? rgl * (BM / 2) + r : rgl * BM + r;
  int tl[2], last = p.n_tok - 1 - ttile * BN;                        // tokens of the tile
  tl[0] = blockIdx.y * 8 + (half ? tid >> 5 : tid >> 6); tl[1] = tl[0] + (half ? 0 : 4);
  float si[2]; float4 extra[2];
  const bool wide = p.sum_wide && row < (half ? half : rows);
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int t = ttile * BN + min(tl[u], last);
    si[u] = p.sinv[t];
    extra[u] = wide && p.residual ? *reinterpret_cast<const float4*>(p.residual + (int64_t)t * p.y_stride + yo + row) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
  const float* src = p.part + (int64_t)ci * p.n_splits * (BN * BM);
  const float* at[2] = {src + min(tl[0], last) * BM + r, src + min(tl[1], last) * BM + r + (half ? BM / 2 : 0)};
  float4 v[2] = {make_float4(0.0f, 0.0f, 0.0f, 0.0f), make_float4(0.0f, 0.0f, 0.0f, 0.0f)};
  for (int s = 0; s < p.n_splits; s += AT_ONCE) {
    float4 a[AT_ONCE][2];
#pragma unroll
    for (int k = 0; k < AT_ONCE; k++)
      if (k < 4 || s + 4 < p.n_splits)                               // (uniform)
#pragma unroll
        for (int u = 0; u < 2; u++) a[k][u] = *reinterpret_cast<const float4*>(at[u] + (int64_t)min(s + k, p.n_splits - 1) * (BN * BM));
#pragma unroll
    for (int k = 0; k < AT_ONCE; k++)
      if (s + k < p.n_splits)
#pragma unroll
        for (int u = 0; u < 2; u++) { v[u].x += a[k][u].x; v[u].y += a[k][u].y; v[u].z += a[k][u].z; v[u].w += a[k][u].w; }
  }
#pragma unroll
  for (int u = 0; u < 2; u++) { v[u].x *= si[u]; v[u].y *= si[u]; v[u].z *= si[u]; v[u].w *= si[u]; }
  if (half) {
    const int t = ttile * BN + tl[0];
    if (t >= p.n_tok) return;
    const float up[4] = {v[0].x, v[0].y, v[0].z, v[0].w}, gate[4] = {v[1].x, v[1].y, v[1].z, v[1].w};
#pragma unroll
    for (int i = 0; i < 4; i++) if (row + i < half) wide_store_pair(p, bias, (int64_t)t * p.y_stride + row + i, row + i, up[i], gate[i]);
    return;
  }
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int t = ttile * BN + tl[u];
    if (t >= p.n_tok) continue;
    const int64_t o = (int64_t)t * p.y_stride + yo + row;
    if (wide) {
      float4 b = bias ? *reinterpret_cast<const float4*>(bias + row) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (bias) { v[u].x += b.x; v[u].y += b.y; v[u].z += b.z; v[u].w += b.w; }
      if (p.residual) { v[u].x += extra[u].x; v[u].y += extra[u].y; v[u].z += extra[u].z; v[u].w += extra[u].w; }
      *reinterpret_cast<float4*>(p.y + o) = v[u];
    } else {
      const float w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
      for (int i = 0; i < 4; i++) if (row + i < rows) wide_store(p, bias, o + i, row + i, w[i]);
    }
  }
}

// partial sums of products whose width is cut over work-groups: allocated once for any product (no more than one slice of a tile per CU), given
// back with the other prompt buffers.  All prompt work runs on the one stream of the library under its lock, so one buffer serves every decoder.
static float* g_wide_part = nullptr;
static int wide_reserve()
{
  if (!g_wide_part) CAI_HIP(hipMalloc((void**)&g_wide_part, (size_t)ctx().n_cu * 256 * 128 * sizeof(float)));
  return CAI_OK;
}
void wide_release() { if (g_wide_part) (void)hipFree(g_wide_part); g_wide_part = nullptr; }

namespace {
template <int QT, int TT>
int go_wide(const WideParams& p)
{
  constexpr int BN = 64 * TT, HB = QT == CAI_Q5_K ? 48 : 16;
  constexpr size_t lds = 3 * BN * 256 + 3 * 256 * 32 + 2 * 256 * HB + 2 * 2 * BN * 16;
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  static bool raised = false;
  if (!raised) { CAI_HIP(hipFuncSetAttribute((const void*)gemm_wide_pf<QT, TT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)); raised = true; }
  const int n_cut = p.n_row_groups * p.n_tok_tiles - p.n_whole;
  hipLaunchKernelGGL((gemm_wide_pf<QT, TT>), dim3(p.n_whole + n_cut * p.n_splits), dim3(512), lds, ctx().stream, p);
  if (n_cut) hipLaunchKernelGGL(gemm_wide_sum<BN>, dim3(n_cut, (std::min(BN, p.n_tok) + 7) / 8), dim3(256), 0, ctx().stream, p);
  return CAI_OK;
}
}  // namespace

// Wide tiles or those of 128 rows x 32 tokens (gemm_q4k_pf), whose work-groups walk the whole width: for n_w matrices of one type and
// width together.  The lines, us of a call by tiles of that kernel | super-blocks of the width, Q4_K, 256 CUs, that kernel -> this one:
//   many tiles (4 per CU on): 37888 x 3584 x 511 tokens 358 -> 300, x 2048 1540 -> 1213; 28672 x 1024 x 200 48.1 -> 46.0;
//   long widths: 3584 x 18944 x 20 152 -> 47, x 511 253 -> 184, 4608 x 3584 x 256 47 -> 40, 3584 x 3584 x 511 54 -> 49;
//   few tiles: 2048 x 2048 x 20 22.1 -> 17.0, x 200 24.8 -> 21.7 (the width is cut; nothing to cut below eight super-blocks, for Q5_K four);
//   in between that kernel is the faster one: 11264 x 2048 x 200 42.1, here 43.6; 4096 x 1024 x 200 15.9 and 20.1;
//   one token tile of it that fills the chip: 37888 x 3584 x 20 44, here 61 (a tile takes 64 tokens).
bool gemm_wide_wanted(const cai_qw_s* const* ws, int n_w, int n_tok)
{
  const cai_qw_s* w = ws[0];
  int64_t rows_all = 0;
  for (int i = 0; i < n_w; i++) {
    if (!wide_offsets_fit(n_tok, ws[i]->cols, ws[i]->data_bytes)) return false;
    rows_all += ws[i]->rows;
  }
  if ((w->qtype != CAI_Q4_K && w->qtype != CAI_Q5_K) || w->cols % 256 || n_tok <= 16) return false;
  const int n_cu = ctx().n_cu, nsb = (int)(w->cols >> 8);
  const int64_t tiles = (rows_all + 127) / 128 * ((n_tok + 31) / 32);
  if (n_tok <= 32 && tiles >= n_cu) return false;
  const bool q5 = w->qtype == CAI_Q5_K;
  return tiles >= 4 * n_cu || nsb >= (q5 ? 8 : 10) || (nsb >= (q5 ? 4 : 8) && tiles < n_cu);
}

int launch_gemm_wide(const cai_qw_s* const* ws, const int* y_off, int n_w, const _Float16* xhi, const _Float16* xlo, const _Float16* sxhi,
                     const _Float16* sxlo, const float* sinv, int n_tok, float* y, int64_t y_stride, const float* residual, int swiglu_half)
{
  constexpr int BM = 256;
  WideParams p{};
  p.w = ws[0]->data; p.bias = ws[0]->bias; p.rows = (int)ws[0]->rows; p.cols = (int)ws[0]->cols;
  p.xhi = xhi; p.xlo = xlo; p.sxhi = sxhi; p.sxlo = sxlo; p.sinv = sinv; p.n_tok = n_tok; p.y = y + y_off[0]; p.y_stride = y_stride; p.residual = residual;
  p.n_seg = n_w; p.swiglu_half = swiglu_half;
  for (int i = 0; i < n_w; i++) {        // every matrix starts a row group of its own
    if (i > 0) { p.seg_end[i - 1] = p.n_row_groups; p.w2[i - 1] = ws[i]->data; p.bias2[i - 1] = ws[i]->bias; p.rows2[i - 1] = (int)ws[i]->rows; p.y_off2[i - 1] = y_off[i] - y_off[0]; }
    p.n_row_groups += (int)((ws[i]->rows + BM - 1) / BM);
  }
  if (swiglu_half) p.n_row_groups = (swiglu_half + BM / 2 - 1) / (BM / 2);
  // One tile per CU and round; the tiles that do not fill a round are cut along the width so that they do.  64 or 128 tokens per tile:
  // whichever takes less time, counted in super-blocks of a 128-token tile (5.8 us of a CU by itself; of 64 tokens 3.7 us), with two of
  // them for the sums of cut tiles.
  const int slots = ctx().n_cu, nsb = p.cols >> 8;
  float best = 0.0f; int BN = 0;
  for (int bn = 128; bn >= 64; bn /= 2) {
    const int tt = (n_tok + bn - 1) / bn, tiles = p.n_row_groups * tt, left = tiles % slots;
    const bool cut = left && 2 * left <= slots;
    const int sp = cut ? std::min(slots / left, nsb) : 1;
    const float unit = bn == 128 ? 1.0f : 0.64f;
    const float t = unit * ((tiles / slots) * nsb + (left ? (nsb + sp - 1) / sp : 0)) + (cut ? 2.0f : 0.0f);
    if (!BN || t < best) { best = t; BN = bn; p.n_tok_tiles = tt; p.n_splits = sp; p.n_whole = cut ? tiles - left : tiles; }
  }
  const int n_cut = p.n_row_groups * p.n_tok_tiles - p.n_whole;
  if (n_cut) {
    if (n_cut * p.n_splits > slots) return set_error(CAI_ERR_INVALID, "prompt gemm: %d tiles cut into %d slices for %d work-groups", n_cut, p.n_splits, slots);
    const int rc = wide_reserve(); if (rc) return rc;
    p.part = g_wide_part;
    uintptr_t low = (uintptr_t)p.y | (uintptr_t)residual | (uintptr_t)(y_stride * 4);
    for (int i = 0; i < n_w; i++) low |= (uintptr_t)ws[i]->bias | (uintptr_t)(ws[i]->rows * 4) | (uintptr_t)(i ? p.y_off2[i - 1] : 0) * 4;
    p.sum_wide = !swiglu_half && (low & 15) == 0;
  }
  const bool q5 = ws[0]->qtype == CAI_Q5_K;
  const int rc = BN == 128 ? (q5 ? go_wide<CAI_Q5_K, 2>(p) : go_wide<CAI_Q4_K, 2>(p)) : (q5 ? go_wide<CAI_Q5_K, 1>(p) : go_wide<CAI_Q4_K, 1>(p));
  if (rc) return rc;
  return CAI_OK;
}

}  // namespace cai
