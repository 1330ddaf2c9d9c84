// Linear layers over bfloat16 weights: streaming kernels for up to sixteen bfloat16 or eight float activation rows (decode) and a
// matrix-core kernel for more (prompts and mixed batches).
//
// Weights are row-major [out][padded in], the padding zero.  Activations are bfloat16 (matrix cores multiply bfloat16 with
// 32-bit sums) or float; with float activations the weights are widened exactly and every product and sum is 32-bit (the
// 16x16x4 float form of the matrix cores).  What follows the product runs in its epilogue on the 32-bit sums: bias and
// activation, act(gate) * up of a gated pair, or the residual update with the Dynamic Tanh before and after it - that norm
// has no statistics, so a sublayer needs no launch besides its products and its mixer - or a result's scaled and gated joining.  The
// streaming kernel takes float rows (the stream's) through an RMS norm itself, and runs two products in one launch.  The matrix-core kernel also runs over a
// bank of equal matrices with a list of activation rows for each (mixtures of experts).
#include "cai_lin_epilogue.hpp"
#include "cai_async_copy.hpp"

#include <algorithm>
#include <string.h>

namespace cai {

// ------------------------------------------------------------------------------------------
// Decode, every product in 32 bits: float activations, an RMS norm on the way, two products in one, bfloat16 rows of more than 8192 columns and one or two
// (run_lin) of smaller matrices.
// NB activation rows.  A wave owns R weight rows (of a gated matrix R / 2 outputs) or, with ksplit > 1, every ksplit-th
// 512-wide turn of them; the activations are staged in LDS as float in panels, the weights stream past once.
// GV_RMS: the activations are the float stream, RMS-normed on the way (the gain while they are staged, the root at the end), and the
// work-groups from q.blocks on do the same for a second matrix with a gain of its own.
// GV_PAIR: two products over the same outputs, both joined to the stream.
// ------------------------------------------------------------------------------------------
constexpr int GV_WAVES = 8;
constexpr int GV_LDS = 16384;              // most floats of staged activations (a launch asks for what its width needs)
enum { GV_PLAIN = 0, GV_RMS = 1, GV_PAIR = 2 };
struct GvSecond {                          // the second matrix of GV_RMS and GV_PAIR, and what the norm needs
  const uint16_t* W = nullptr; const void* x = nullptr; int n_rows = 0, ldw = 0; int64_t ldx = 0; LinEpi e;
  int blocks = 0, width = 0; float eps = 0.0f; const float *gain = nullptr, *gain2 = nullptr;
  void *normed = nullptr, *normed2 = nullptr; int64_t ldn = 0;   // the normed rows themselves (null: not)
};

template <typename AT, int NB, int R, int KIND>
__global__ __launch_bounds__(64 * GV_WAVES) void gemv_bf16(const uint16_t* __restrict__ W, const void* __restrict__ xv, int n_rows, int ldw, int64_t ldx, int ksplit, LinEpi e, GvSecond q)
{
  // one row: as much as its width needs (more work-groups fit a CU); several rows: a fixed array, its layout known at compile time
  extern __shared__ float xs_dyn[];
  __shared__ float xs_fix[NB == 1 ? 1 : GV_LDS];
  float* const xs = NB == 1 ? xs_dyn : xs_fix;
  __shared__ float part[GV_WAVES][R * NB];
  __shared__ float sq[GV_WAVES][NB];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ks = wave % ksplit;
  int block = blockIdx.x, n_blocks = q.blocks;             // (of this matrix)
  const float* gain = q.gain;
  if constexpr (KIND == GV_RMS) {
    if (block >= q.blocks) { block -= q.blocks; n_blocks = gridDim.x - q.blocks; W = q.W; n_rows = q.n_rows; e = q.e; gain = q.gain2; q.normed = q.normed2; }
  }
  const int grp = block * (GV_WAVES / ksplit) + wave / ksplit;
  constexpr int PANEL = GV_LDS / NB / 512 * 512;
  const bool glu = KIND == GV_PLAIN && e.mode == EPI_GLU;
  float ss[NB];                            // sums of squares of the rows
#pragma unroll
  for (int b = 0; b < NB; b++) ss[b] = 0.0f;

  // (read past the caches' replacement beside the ring kernel's, or they push out what that leaves there - a recurrent layer's state: a token of eight
  // such layers of width 2048 452 -> 423 us, of width 4096 914 -> 868)
  auto weights = [](const uint16_t* at) -> u32x4 {
    if constexpr (KIND == GV_PLAIN && sizeof(AT) == 2) return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(at));
    else return *reinterpret_cast<const u32x4*>(at);
  };
  // lane i * NB + b ends with the sum of row i, activation b (of the first wave of a split row)
  auto product = [&](const uint16_t* __restrict__ M, const void* __restrict__ xw, const int ld, const int64_t lx) -> float {
    const AT* x = reinterpret_cast<const AT*>(xw);
    const uint16_t* row[R];
#pragma unroll
    for (int i = 0; i < R; i++) {
      int r = glu ? glu_row(grp * (R / 2) + i % (R / 2 > 0 ? R / 2 : 1), i / (R / 2 > 0 ? R / 2 : 1)) : grp * R + i;
      row[i] = M + (int64_t)min(r, n_rows - 1) * ld;
    }
    float acc[R][NB];
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
      for (int b = 0; b < NB; b++) acc[i][b] = 0.0f;
    for (int p0 = 0; p0 < ld; p0 += PANEL) {
      const int pk = min(PANEL, ld - p0), pk512 = (pk + 511) / 512 * 512;
      // eight weights a turn ahead of the staging: the first requests are out while the activations arrive
      u32x4 w0[R];
      const int k_first = ks * 512 + lane * 8;
#pragma unroll
      for (int i = 0; i < R; i++) w0[i] = weights(row[i] + p0 + (k_first < pk ? k_first : 0));
      if (p0) __syncthreads();
#pragma unroll
      for (int b = 0; b < NB; b++)
        for (int k = threadIdx.x * 8; k < pk512; k += 64 * GV_WAVES * 8) {
          float v[8];
          if constexpr (KIND == GV_RMS) {
            const float* xf = reinterpret_cast<const float*>(xw) + b * lx;
            const int c = p0 + k;
            if (c + 8 <= q.width && (lx & 3) == 0) {
              const f32x4 a = *reinterpret_cast<const f32x4*>(xf + c), d = *reinterpret_cast<const f32x4*>(xf + c + 4);
              const f32x4 ga = *reinterpret_cast<const f32x4*>(gain + c), gd = *reinterpret_cast<const f32x4*>(gain + c + 4);
#pragma unroll
              for (int j = 0; j < 4; j++) { ss[b] = fmaf(a[j], a[j], ss[b]); ss[b] = fmaf(d[j], d[j], ss[b]); v[j] = a[j] * ga[j]; v[4 + j] = d[j] * gd[j]; }
            } else {
#pragma unroll
              for (int j = 0; j < 8; j++) { const float a = c + j < q.width ? xf[c + j] : 0.0f; ss[b] = fmaf(a, a, ss[b]); v[j] = c + j < q.width ? a * gain[c + j] : 0.0f; }
            }
          } else if (k < pk) {
            if constexpr (sizeof(AT) == 2) {
              const u32x4 u = *reinterpret_cast<const u32x4*>(x + b * lx + p0 + k);
#pragma unroll
              for (int j = 0; j < 4; j++) { v[2 * j] = bf16_lo(u[j]); v[2 * j + 1] = bf16_hi(u[j]); }
            } else {
              const f32x4 a = *reinterpret_cast<const f32x4*>(x + b * lx + p0 + k), c = *reinterpret_cast<const f32x4*>(x + b * lx + p0 + k + 4);
#pragma unroll
              for (int j = 0; j < 4; j++) { v[j] = a[j]; v[4 + j] = c[j]; }
            }
          } else {
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = 0.0f;
          }
          // a turn of 512 values is kept as two halves of 256 (four values a lane each), so that a wave's 16-byte reads are contiguous
          float* o = xs + b * PANEL + (k >> 9) * 512 + ((k >> 3) & 63) * 4;
          *reinterpret_cast<f32x4*>(o) = f32x4{v[0], v[1], v[2], v[3]};
          *reinterpret_cast<f32x4*>(o + 256) = f32x4{v[4], v[5], v[6], v[7]};
        }
      if constexpr (KIND == GV_RMS) {
        if (p0 + PANEL >= ld)
#pragma unroll
          for (int b = 0; b < NB; b++) { const float t = wave_sum(ss[b]); if (lane == 63) sq[wave][b] = t; }
      }
      __syncthreads();
      for (int k0 = ks * 512; k0 < pk512; k0 += ksplit * 512) {
        u32x4 w1[R];
        const int kn = k0 + ksplit * 512 + lane * 8;
#pragma unroll
        for (int i = 0; i < R; i++) w1[i] = weights(row[i] + p0 + (kn < pk ? kn : 0));
#pragma unroll
        for (int b = 0; b < NB; b++) {
          const f32x4 xa = *reinterpret_cast<const f32x4*>(xs + b * PANEL + k0 + lane * 4);
          const f32x4 xb = *reinterpret_cast<const f32x4*>(xs + b * PANEL + k0 + 256 + lane * 4);
#pragma unroll
          for (int i = 0; i < R; i++) {
            float s = acc[i][b];
            s = fmaf(bf16_lo(w0[i][0]), xa[0], s); s = fmaf(bf16_hi(w0[i][0]), xa[1], s);
            s = fmaf(bf16_lo(w0[i][1]), xa[2], s); s = fmaf(bf16_hi(w0[i][1]), xa[3], s);
            s = fmaf(bf16_lo(w0[i][2]), xb[0], s); s = fmaf(bf16_hi(w0[i][2]), xb[1], s);
            s = fmaf(bf16_lo(w0[i][3]), xb[2], s); s = fmaf(bf16_hi(w0[i][3]), xb[3], s);
            acc[i][b] = s;
          }
        }
#pragma unroll
        for (int i = 0; i < R; i++) w0[i] = w1[i];
      }
    }
    float mine = 0.0f;
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const float t = wave_sum(acc[i][b]);
        const float s = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, t), 63));
        if (lane == i * NB + b) mine = s;
      }
    if (ksplit > 1) {
      if (lane < R * NB) part[wave][lane] = mine;
      __syncthreads();
      if (ks == 0 && lane < R * NB) for (int j = 1; j < ksplit; j++) mine += part[wave + j][lane];
    }
    return mine;
  };

  float mine = product(W, xv, ldw, ldx);
  const int i = lane / NB, b = lane % NB;
  if constexpr (KIND == GV_PAIR) {
    __syncthreads();
    const float second = product(q.W, q.x, q.ldw, q.ldx);
    if (ks == 0 && i < R && grp * R + i < n_rows) join_two(e, mine, q.e, second, grp * R + i, b);
    return;
  }
  if constexpr (KIND == GV_RMS) {
    auto root = [&](int r) {
      float t = 0.0f;
#pragma unroll
      for (int w = 0; w < GV_WAVES; w++) t += sq[w][r];
      return 1.0f / sqrtf(t / (float)q.width + q.eps);
    };
    mine *= root(b);
    for (int r = block; q.normed && r < NB; r += n_blocks) {   // the first work-groups leave a normed row each
      const float inv = root(r);
      const float* xf = reinterpret_cast<const float*>(xv) + r * ldx;
#pragma unroll 4
      for (int k = threadIdx.x; k < q.ldn; k += 64 * GV_WAVES) put_act<AT>(q.normed, r * q.ldn + k, k < q.width ? xf[k] * inv * gain[k] : 0.0f);
    }
  }
  if (ks != 0) return;
  if (glu) {
    const float up = __shfl(mine, lane + R / 2 * NB);
    const int j = grp * (R / 2) + i;
    if (i < R / 2 && glu_row(j, 0) < n_rows) put_act<AT>(e.h, b * e.ldh + j, glu_pair(e.glu, e.limit, mine, up));
  } else if (i < R && grp * R + i < n_rows) {
    if constexpr (KIND == GV_RMS) { if (e.mode == EPI_SPLIT) epi_as<AT, EPI_SPLIT>(e, grp * R + i, b, mine); else epi_as<AT, EPI_STORE>(e, grp * R + i, b, mine); }
    else epi_one<AT>(e, grp * R + i, b, mine);
  }
}

// ------------------------------------------------------------------------------------------
// Decode over bfloat16 activations, and their shortest prompts: the matrix cores multiply eight weight rows (twice: a tile has sixteen) and up to
// 16 activation rows (lanes past the last one repeat it; what they make is not read), so a weight costs no more at sixteen rows than at one, and
// what is left is the stream of weights.  A work-group owns MC_H rows (of a gated matrix so many gate and up rows) at a time, its KS waves every
// KS-th slot of 256 columns of them.  A wave copies its slots (two rows of 512 bytes a request; requests of 64 bytes a row, the shape of the
// operands, reached half the rate) into a ring of its own in LDS without meeting anyone, and keeps its part of the activations in registers from
// tile to tile.  16-byte chunk q of row r lies at q ^ r, which makes the operand reads conflict-free.  The sums of a tile meet once, in one of two
// areas in turn.  Weights are read past the caches' replacement ("nt"): a step's do not fit the memory-side cache, and kept there one by one
// they push each other out.
// A matrix instruction cuts what lies below the largest of its products off downwards, and a chain of them does so again at the size of the running
// sum: whole chains were 1.4 (512 columns) to 2.3 times (8192) as far off 64 bits as the 32-bit walk above.  So each starts from zero, every second one
// with its activations' sign changed, the difference of two joins a 64-bit sum, and the waves' parts are added in 64 bits: 0.89 times the walk's distance
// at 512 columns, 0.73 at 2048, 0.62 at 8192 (5.3e-8; one instruction or two, 64 columns: 0.99, all products positive 1.02), for 2 to 4 % of the time.
// Per launch at 4 rows, us, by the 32-bit walk | whole chains | here (the last two from the trace of a step, whose launches wait for what they read):
// 11264 x 2048 gated 14.2 | 11.0 | 11.2; 2048 x 5632 10.9 | 9.3 | 9.5; 6200 x 2048 9.2 | 8.7 | 9.0; 32768 x 2048 33.7 | 25.8 | 26.9 (5.0 TB/s).
// Sixteen rows a tile: 128 work-groups for 2048 rows, 9.9 for 2048 x 5632; a ring of one slot loses 2 % of a step; without "nt" 13.2 and 10.6 (whole chains).
// ------------------------------------------------------------------------------------------
constexpr int MC_WAVES = 8, MC_ROWS = 16, MC_H = 8, MC_SLOT = MC_H * 512, MC_SLOTS = 4;      // (at most MC_SLOTS slots of a row a wave)
constexpr int mc_depth(int sb) { return sb < 2 ? 2 : sb; }  // slots of a wave's ring: a tile's, and the next one's where that is one
template <bool GLU, int SB>
__global__ __launch_bounds__(64 * MC_WAVES) void gemv_bf16_mc(const uint16_t* __restrict__ W, const bf16_t* __restrict__ x, int n_rows, int ldw, int64_t ldx, int n_tok, int n_tiles, LinEpi e)
{
  constexpr int T = GLU ? 2 : 1, DEPTH = mc_depth(SB), COPIES = MC_H / 2;
  extern __shared__ u32x4 mc_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), KS = blockDim.x >> 6;
  const int r = lane & 15, c = lane >> 4, hi = lane >> 5;
  const int slots = (ldw + 255) >> 8, mine = wave < slots ? (slots - wave + KS - 1) / KS : 0;       // slots of a row, of this wave
  float* const parts = reinterpret_cast<float*>(mc_lds) + KS * (DEPTH * MC_SLOT / 4);
  const int part_len = n_tok * T * 16;                                                              // of one wave: [token][row]
  const char* const ring = reinterpret_cast<const char*>(mc_lds) + wave * (DEPTH * MC_SLOT);
  const uint32_t ring0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) u32x4*)mc_lds + wave * (DEPTH * MC_SLOT);
  auto first_row = [](int tile, int t) { return !GLU ? tile * MC_H : (tile >> 1) * 32 + t * 16 + (tile & 1) * MC_H; };
  // the next slot to request: slot q_s of this wave, of part q_t of tile q_tile
  int q_tile = blockIdx.x, q_t = 0, q_s = 0, q_ring = 0;
  auto request = [&]() {
    const int row0 = first_row(q_tile, q_t), k0 = (wave + q_s * KS) * 256, chunks = min(32, (ldw - k0) >> 3);
    const char* const base = reinterpret_cast<const char*>(W + (int64_t)row0 * ldw + k0);
    const int last = n_rows - 1 - row0;
#pragma unroll
    for (int i = 0; i < COPIES; i++) {
      const int row = 2 * i + hi;
      copy16_to_lds_once(ring0 + q_ring * MC_SLOT + i * 1024, (uint32_t)(min(row, last) * ldw * 2 + min((lane & 31) ^ row, chunks - 1) * 16), base);
    }
    q_ring = q_ring + 1 == DEPTH ? 0 : q_ring + 1;
    if (++q_s == mine) { q_s = 0; if (++q_t == T) { q_t = 0; q_tile += gridDim.x; } }
  };
  int ahead = 0;
  if (mine) {
#pragma unroll
    for (int i = 0; i < DEPTH; i++) if (q_tile < n_tiles) { request(); ahead++; }
  }
  u32x4 b[SB][8];
#pragma unroll
  for (int s = 0; s < SB; s++)
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int k = min((wave + s * KS) * 256 + u * 32, ldw - 32);
      b[s][u] = *reinterpret_cast<const u32x4*>(x + min(r, n_tok - 1) * ldx + k + c * 8);
      if (u & 1) b[s][u] ^= 0x80008000u;
    }
  int at = 0, parity = 0;
  for (int tile = blockIdx.x, turn = 0; tile < n_tiles; tile += gridDim.x, turn++) {
    double sum[T][4] = {};
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
      for (int s = 0; s < SB; s++)
        if (s < mine) {
          if (ahead == DEPTH) wait_copies<(DEPTH - 1) * COPIES>(); else wait_copies<0>();
          const char* const slot = ring + at * MC_SLOT;
          u32x4 w[8];
#pragma unroll
          for (int u = 0; u < 8; u++) { const int row = r & (MC_H - 1); w[u] = *reinterpret_cast<const u32x4*>(slot + row * 512 + (((u * 4 + c) ^ row) << 4)); }
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot has been read
          at = at + 1 == DEPTH ? 0 : at + 1;
          if (q_tile < n_tiles) request(); else ahead--;
          const int left = (ldw - (wave + s * KS) * 256) >> 5;       // (even: rows are padded to 64 columns)
          auto pair = [&](int u) {
            const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
            const f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[u]), __builtin_bit_cast(bf16x8, b[s][u]), zero, 0, 0, 0);
            const f32x4 n = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[u + 1]), __builtin_bit_cast(bf16x8, b[s][u + 1]), zero, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; q++) sum[t][q] += (double)(d[q] - n[q]);
          };
          if (left >= 8) {
#pragma unroll
            for (int u = 0; u < 8; u += 2) pair(u);
          } else {
#pragma unroll
            for (int u = 0; u < 8; u += 2) if (u < left) pair(u);
          }
        }
    float* const area = parts + parity * KS * part_len;
    parity ^= 1;
    if (r < n_tok)
#pragma unroll
      for (int t = 0; t < T; t++)
        *reinterpret_cast<f32x4*>(area + wave * part_len + r * (T * 16) + t * 16 + c * 4) = f32x4{(float)sum[t][0], (float)sum[t][1], (float)sum[t][2], (float)sum[t][3]};
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // (no wait for the copies on their way)
    // (another wave's turn from tile to tile: a result's own loads wait for the copies requested before them)
    for (int o = (tid + turn * 64) & (blockDim.x - 1); o < MC_H * n_tok; o += blockDim.x) {
      const int i = o & (MC_H - 1), tok = o / MC_H, n = first_row(tile, 0) + i;
      const float* p = area + tok * (T * 16) + i;
      double v = 0.0, up = 0.0;
      for (int w = 0; w < KS; w++) { v += p[w * part_len]; if (GLU) up += p[w * part_len + 16]; }
      if constexpr (GLU) put_act<bf16_t>(e.h, tok * e.ldh + tile * MC_H + i, glu_pair(e.glu, e.limit, (float)v, (float)up));
      else if (n < n_rows) epi_one<bf16_t>(e, n, tok, (float)v);
    }
  }
}

// ------------------------------------------------------------------------------------------
// Prompts: C^T tile = W tile x activations^T on the matrix cores; a lane ends with four consecutive outputs of one token.
// Both operand tiles are 128 bytes deep per row (64 bfloat16 or 32 floats), DEPTH of them in LDS; the 16-byte chunks of a row
// are stored at chunk ^ (row & 7), which makes the fragment reads conflict-free.  bfloat16 tiles are copied into LDS asynchronously,
// DEPTH - 1 steps ahead, with one meeting of the waves a step; float ones are widened on the way, through registers.
// Bound by the matrix cores and the fragment reads of a step together: sixteen waves of 64 x 32 overlap them better than four of
// 64 x 64 (whole prompt of 2048 tokens through four layers of width 2048: 2798 us with four waves and staging through registers -> 2546).
// ------------------------------------------------------------------------------------------
template <typename AT, int BM, int BN, int WM, int WN, bool BANK, int MODE, int DEPTH = 2>   // MODE: e.mode (one epilogue a kernel: with all of them the accumulators would leave their registers)
__global__ __launch_bounds__(64 * WM * WN) void gemm_bf16(const uint16_t* __restrict__ W, const AT* __restrict__ X, int n_rows, int ldw, int64_t ldx, int n_tok, int tiles_m, int n_tiles, LinEpi e, BankList l)
{
  constexpr int NT = 64 * WM * WN;
  constexpr int BK = 128 / (int)sizeof(AT);          // elements per row of a tile
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  constexpr int CA = BM * 8 / NT, CW = BN * 8 / NT;  // 16-byte chunks per thread
  static_assert(CA >= 1 && CW >= 1 && BM * 8 % NT == 0 && BN * 8 % NT == 0 && TN % 2 == 0, "tile shape");
  extern __shared__ u32x4 gm_lds[];                 // DEPTH slots of BM + BN rows of 128 bytes
  u32x4* const sx_ = gm_lds; u32x4* const sw_ = gm_lds + BM * 8;
  constexpr int SLOT = (BM + BN) * 8;
  // consecutive work-groups go to different XCDs: give each XCD a contiguous run of tiles, token tiles fastest, so that the
  // work-groups of an XCD share weight rows in its L2
  int tile;
  {
    const int xcd = blockIdx.x & 7, per = n_tiles >> 3, rem = n_tiles & 7;
    tile = xcd * per + min(xcd, rem) + (blockIdx.x >> 3);
  }
  int m0 = tile % tiles_m * BM;
  const int n0 = tile / tiles_m * BN;
  if constexpr (BANK) {                    // n_rows: of one matrix; the token tile is a run of places of the order
    const int tm = tile % tiles_m;
    if (tm >= *l.n_tiles) return;
    const int32_t* tl = l.tiles + 3 * tm;
    W += (int64_t)tl[0] * n_rows * ldw;
    m0 = tl[1]; n_tok = m0 + tl[2];
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN * (BM / WM), wn = wave % WN * (BN / WN);
  const AT* xp[CA]; const uint16_t* wp[CW];
#pragma unroll
  for (int i = 0; i < CA; i++) {
    const int c = tid + i * NT;
    int t = min(m0 + (c >> 3), n_tok - 1);
    if constexpr (BANK) { if (l.div) t = l.order[t] / l.div; }
    xp[i] = X + (int64_t)t * ldx + ((c ^ (c >> 3)) & 7) * (16 / sizeof(AT));
  }
#pragma unroll
  for (int i = 0; i < CW; i++) { const int c = tid + i * NT; wp[i] = W + (int64_t)min(n0 + (c >> 3), n_rows - 1) * ldw + ((c ^ (c >> 3)) & 7) * (16 / sizeof(AT)); }
  f32x4 acc[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; j++)
#pragma unroll
    for (int i = 0; i < TM; i++) acc[j][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int fr = lane & 15, fc = lane >> 4;
  const int nk = ldw / BK;
  auto multiply = [&](int s) {
    const u32x4 *const sx = sx_ + s * SLOT, *const sw = sw_ + s * SLOT;
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
      u32x4 fx[TM], fw[TN];
#pragma unroll
      for (int i = 0; i < TM; i++) { const int r = wm + i * 16 + fr; fx[i] = sx[r * 8 + ((kk * 4 + fc) ^ (r & 7))]; }
#pragma unroll
      for (int j = 0; j < TN; j++) { const int r = wn + j * 16 + fr; fw[j] = sw[r * 8 + ((kk * 4 + fc) ^ (r & 7))]; }
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int i = 0; i < TM; i++) {
          if constexpr (sizeof(AT) == 2) {
            acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fw[j]), __builtin_bit_cast(bf16x8, fx[i]), acc[j][i], 0, 0, 0);
          } else {
            // the k index a lane group contributes at step q is 4 * group + q of the 16-wide block, for both operands alike
            const f32x4 a = __builtin_bit_cast(f32x4, fw[j]), b = __builtin_bit_cast(f32x4, fx[i]);
#pragma unroll
            for (int q = 0; q < 4; q++) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q], b[q], acc[j][i], 0, 0, 0);
          }
        }
    }
  };
  if constexpr (sizeof(AT) == 2) {
    // the copies of step kt + DEPTH - 1 go out as soon as every wave has read the slot they fill
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) u32x4*)gm_lds;
    auto copy = [&](int kt) {
      const uint32_t dst = lds0 + (uint32_t)(kt % DEPTH * SLOT * 16 + wave * 1024);
#pragma unroll
      for (int i = 0; i < CA; i++) copy16_to_lds(dst + i * NT * 16, xp[i] + kt * BK);
#pragma unroll
      for (int i = 0; i < CW; i++) copy16_to_lds(dst + BM * 128 + i * NT * 16, wp[i] + kt * BK);
    };
#pragma unroll
    for (int i = 0; i < DEPTH - 1; i++) if (i < nk) copy(i);
    for (int kt = 0; kt < nk; kt++) {
      if (kt + DEPTH - 1 <= nk) wait_copies<(DEPTH - 2) * (CA + CW)>(); else wait_copies<0>();
      __builtin_amdgcn_s_waitcnt(0xC07F);              // lgkmcnt(0): this wave's reads of the slot that is filled next
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (kt + DEPTH - 1 < nk) copy(kt + DEPTH - 1);
      multiply(kt % DEPTH);
    }
  } else {
    u32x4 rx[CA], rw[CW];
    auto fetch = [&](int k) {
#pragma unroll
      for (int i = 0; i < CA; i++) rx[i] = *reinterpret_cast<const u32x4*>(xp[i] + k);
#pragma unroll
      for (int i = 0; i < CW; i++) {
        const uint2 u = *reinterpret_cast<const uint2*>(wp[i] + k);
        rw[i] = u32x4{u.x << 16, u.x & 0xffff0000u, u.y << 16, u.y & 0xffff0000u};
      }
    };
    auto stash = [&](int s) {
#pragma unroll
      for (int i = 0; i < CA; i++) { const int c = tid + i * NT; sx_[s * SLOT + c] = rx[i]; }
#pragma unroll
      for (int i = 0; i < CW; i++) { const int c = tid + i * NT; sw_[s * SLOT + c] = rw[i]; }
    };
    fetch(0); stash(0);
    __syncthreads();
    for (int kt = 0; kt < nk; kt++) {
      const int s = kt & 1;
      if (kt + 1 < nk) fetch((kt + 1) * BK);
      multiply(s);
      if (kt + 1 < nk) stash(s ^ 1);
      __syncthreads();
    }
  }
  const bool whole = (e.ldy & 3) == 0 && (e.ldh & 3) == 0 && (e.ld0 & 3) == 0 && (e.ldg & 3) == 0 && (e.split & 3) == 0;
  if constexpr (MODE == EPI_RESIDUAL && !BANK) {
    // outputs in the outer loop: their bias and norm factors are requested once (for every token again, behind stores they might alias, they
    // are half of the epilogue), and the stream of all the tokens before the first is changed
    if (whole) {
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const int n = n0 + wn + j * 16 + fc * 4;
        if (n >= n_rows) continue;
        if (n + 3 >= n_rows) {
          for (int i = 0; i < TM; i++) {
            const int t = m0 + wm + i * 16 + fr;
#pragma unroll
            for (int q = 0; q < 4; q++) if (t < n_tok && n + q < n_rows) epi_as<AT, MODE>(e, n + q, t, acc[j][i][q]);
          }
          continue;
        }
        const DytFour post = dyt_four(e.post, n), next = dyt_four(e.next, n);
        const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
        f32x4 bias = zero;
        if (e.bias) bias = *reinterpret_cast<const f32x4_any*>(e.bias + n);
        constexpr int P = TM * TN < 16 ? TM : 2;         // (tokens at once: with more the largest tile's sums leave their registers)
#pragma unroll
        for (int i0 = 0; i0 < TM; i0 += P) {
          f32x4 x[P], x0[P];
#pragma unroll
          for (int i = 0; i < P; i++) {
            const int64_t t = min(m0 + wm + (i0 + i) * 16 + fr, n_tok - 1);
            x[i] = e.fresh ? zero : *reinterpret_cast<const f32x4*>(e.y + t * e.ldy + n);
            x0[i] = e.add0 ? *reinterpret_cast<const f32x4*>(e.add0 + t * e.ld0 + n) : zero;
          }
#pragma unroll
          for (int i = 0; i < P; i++) {
            const int64_t t = m0 + wm + (i0 + i) * 16 + fr;
            x[i] += dyt(e.post, post, acc[j][i0 + i] + bias);
            if (e.add0) x[i] += x0[i];
            if (t >= n_tok) continue;
            *reinterpret_cast<f32x4*>(e.y + t * e.ldy + n) = x[i];
            if (e.h) put_four<AT>(e.h, t * e.ldh + n, dyt(e.next, next, x[i]));
          }
        }
      }
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < TM; i++) {
    int t = m0 + wm + i * 16 + fr;
    if (t >= n_tok) continue;
    float scale = 1.0f;
    if constexpr (BANK) {
      const int at = l.order[t];
      if (MODE == EPI_GLU || MODE == EPI_SPLIT) scale = l.scale[at]; else t = at;
    }
    if constexpr (MODE == EPI_GLU) {
#pragma unroll
      for (int j = 0; j < TN; j += 2) {
        const int n = n0 + wn + j * 16;                // block of 16 gate rows; its up rows are the next fragment
        if (n >= n_rows) continue;
        const int o = (n >> 1) + fc * 4;
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = glu_pair(e.glu, e.limit, acc[j][i][q], acc[j + 1][i][q]);
        if constexpr (BANK) {
#pragma unroll
          for (int q = 0; q < 4; q++) v[q] *= scale;
        }
        put_four<AT>(e.h, (int64_t)t * e.ldh + o, f32x4{v[0], v[1], v[2], v[3]});
      }
      continue;
    }
    if constexpr (BANK && MODE == EPI_SPLIT) {           // (split 0, rows in whole fours)
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const int n = n0 + wn + j * 16 + fc * 4;
        if (n >= n_rows) continue;
        put_four<AT>(e.h, (int64_t)t * e.ldh + n, lin_act_four(acc[j][i], e.act, e.limit) * scale);
      }
      continue;
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const int n = n0 + wn + j * 16 + fc * 4;
      if (n >= n_rows) continue;
      if (n + 3 < n_rows && whole) epi_four<AT, MODE>(e, n, t, acc[j][i]);
      else {
#pragma unroll
        for (int q = 0; q < 4; q++) if (n + q < n_rows) epi_as<AT, MODE>(e, n + q, t, acc[j][i][q]);
      }
    }
  }
}

template <typename AT, int BM, int BN, int WM, int WN, int MODE, int DEPTH>
static int run_gemm_mode(const cai_qw_s* w, const AT* x, int64_t ldx, int n_tok, const LinEpi& e)
{
  constexpr size_t lds = (size_t)DEPTH * (BM + BN) * 128;
  if constexpr (lds > 65536) {
    static bool attr_done = false;
    if (!attr_done) {
      CAI_HIP(hipFuncSetAttribute((const void*)gemm_bf16<AT, BM, BN, WM, WN, false, MODE, DEPTH>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      attr_done = true;
    }
  }
  const int tm = (n_tok + BM - 1) / BM, tn = ((int)w->rows + BN - 1) / BN;
  hipLaunchKernelGGL((gemm_bf16<AT, BM, BN, WM, WN, false, MODE, DEPTH>), dim3(tm * tn), dim3(64 * WM * WN), lds, ctx().stream,
                     (const uint16_t*)w->data, x, (int)w->rows, (int)w->ld, ldx, n_tok, tm, tm * tn, e, BankList{});
  return CAI_OK;
}
template <typename AT, int BM, int BN, int WM, int WN, int DEPTH = 2>
static int run_gemm(const cai_qw_s* w, const AT* x, int64_t ldx, int n_tok, const LinEpi& e)
{
#define GEMM(MODE) case MODE: return run_gemm_mode<AT, BM, BN, WM, WN, MODE, DEPTH>(w, x, ldx, n_tok, e)
  switch (e.mode) { GEMM(EPI_STORE); GEMM(EPI_GLU); GEMM(EPI_RESIDUAL); GEMM(EPI_SPLIT); GEMM(EPI_JOIN); }
#undef GEMM
  return CAI_OK;
}

template <typename AT, int BM, int BN>
static void run_bank(const cai_qw_s* w, int mat_rows, const AT* x, int64_t ldx, const BankList& l, const LinEpi& e)
{
  const int tm = l.max_tiles, tn = (mat_rows + BN - 1) / BN;
#define GEMM(MODE) case MODE: hipLaunchKernelGGL((gemm_bf16<AT, BM, BN, 2, 2, true, MODE>), dim3(tm * tn), dim3(256), (size_t)2 * (BM + BN) * 128, ctx().stream, \
                              (const uint16_t*)w->data, x, mat_rows, (int)w->ld, ldx, 0, tm, tm * tn, e, l); break
  switch (e.mode) { GEMM(EPI_STORE); GEMM(EPI_GLU); GEMM(EPI_SPLIT); }
#undef GEMM
}

int launch_lin_bank(const cai_qw_s* w, int mat_rows, int act_t, const void* x, int64_t ldx, const BankList& l, const LinEpi& e)
{
  CAI_REQUIRE(w->qtype == CAI_BF16 && mat_rows >= 1 && w->rows % mat_rows == 0 && ldx >= w->ld && l.max_tiles >= 1, "bf16 bank: matrices of %d rows of %lld, activation rows of %lld", mat_rows, (long long)w->rows, (long long)ldx);
  CAI_REQUIRE(e.mode == EPI_STORE || (e.mode == EPI_GLU && mat_rows % 32 == 0) || (e.mode == EPI_SPLIT && e.split == 0 && !e.bias && mat_rows % 4 == 0 && e.ldh % 4 == 0), "bf16 bank: a gated matrix needs whole blocks of 32 rows, another one of 4");
  CAI_REQUIRE(l.tile == BANK_TILE || l.tile == BANK_TILE_MAX, "bf16 bank: runs of %d places", l.tile);
  if (act_t == ACT_T_BF16) {
    if (l.tile == BANK_TILE_MAX) run_bank<bf16_t, BANK_TILE_MAX, 128>(w, mat_rows, (const bf16_t*)x, ldx, l, e);
    else run_bank<bf16_t, BANK_TILE, 64>(w, mat_rows, (const bf16_t*)x, ldx, l, e);
  } else if (l.tile == BANK_TILE_MAX) run_bank<float, BANK_TILE_MAX, 128>(w, mat_rows, (const float*)x, ldx, l, e);
  else run_bank<float, BANK_TILE, 64>(w, mat_rows, (const float*)x, ldx, l, e);
  CAI_HIP(hipGetLastError());
  return CAI_OK;
}

// four rows a wave once that still leaves every CU eight waves; fewer rows, then a split of the row, for small matrices
struct GvShape { bool four; int ks; };
static GvShape gv_shape(int rows, int turns, bool glu)
{
  const int want = ctx().n_cu * 8;
  const bool four = rows / 4 >= want;
  const int groups = glu ? (four ? (rows / 2 + 1) / 2 : rows / 2) : (rows + (four ? 3 : 1)) / (four ? 4 : 2);
  int ks = 1;
  while (ks < GV_WAVES && ks * 2 <= turns && groups * ks * 2 <= want * 2) ks *= 2;
  return {four, ks};
}
static int gv_blocks(int rows, const GvShape& s, bool glu)
{
  const int groups = glu ? (s.four ? (rows / 2 + 1) / 2 : rows / 2) : (rows + (s.four ? 3 : 1)) / (s.four ? 4 : 2), per = GV_WAVES / s.ks;
  return (groups + per - 1) / per;
}
static int gv_turns(const cai_qw_s* w) { return ((int)w->ld + 511) / 512; }

template <typename AT, int NB, int KIND>
static void run_gemv(const cai_qw_s* w, const void* x, int64_t ldx, const LinEpi& e, const GvShape& s, int blocks, int turns, const GvSecond& q)
{
  const dim3 grid(blocks), blk(64 * GV_WAVES);
  const size_t lds = NB == 1 ? (size_t)std::min(GV_LDS, turns * 512) * 4 : 0;
  if (s.four) hipLaunchKernelGGL((gemv_bf16<AT, NB, 4, KIND>), grid, blk, lds, ctx().stream, (const uint16_t*)w->data, x, (int)w->rows, (int)w->ld, ldx, s.ks, e, q);
  else hipLaunchKernelGGL((gemv_bf16<AT, NB, 2, KIND>), grid, blk, lds, ctx().stream, (const uint16_t*)w->data, x, (int)w->rows, (int)w->ld, ldx, s.ks, e, q);
}
template <typename AT, int KIND>
static void run_gemv_rows(int n_tok, const cai_qw_s* w, const void* x, int64_t ldx, const LinEpi& e, const GvShape& s, int blocks, int turns, const GvSecond& q)
{
  switch (n_tok) {
    case 1: run_gemv<AT, 1, KIND>(w, x, ldx, e, s, blocks, turns, q); break;
    case 2: run_gemv<AT, 2, KIND>(w, x, ldx, e, s, blocks, turns, q); break;
    case 3: run_gemv<AT, 3, KIND>(w, x, ldx, e, s, blocks, turns, q); break;
    case 4: run_gemv<AT, 4, KIND>(w, x, ldx, e, s, blocks, turns, q); break;
    case 5: run_gemv<AT, 5, KIND>(w, x, ldx, e, s, blocks, turns, q); break;
    case 6: run_gemv<AT, 6, KIND>(w, x, ldx, e, s, blocks, turns, q); break;
    case 7: run_gemv<AT, 7, KIND>(w, x, ldx, e, s, blocks, turns, q); break;
    default: run_gemv<AT, 8, KIND>(w, x, ldx, e, s, blocks, turns, q); break;
  }
}

template <bool GLU, int SB>
static int run_mc(const cai_qw_s* w, const bf16_t* x, int64_t ldx, int n_tok, const LinEpi& e, int ks)
{
  constexpr int T = GLU ? 2 : 1;
  auto lds_of = [](int waves, int rows) { return (size_t)waves * (mc_depth(SB) * MC_SLOT + 2 * rows * T * 16 * 4); };
  static bool attr_done = false;
  if (!attr_done) {
    CAI_HIP(hipFuncSetAttribute((const void*)gemv_bf16_mc<GLU, SB>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_of(MC_WAVES, MC_ROWS)));
    attr_done = true;
  }
  const int tiles = ((int)w->rows + T * MC_H - 1) / (T * MC_H);
  const size_t lds = lds_of(ks, n_tok);
  // as many as a CU holds at once: sixteen waves of the registers of one slot of a row a wave, eight of more (147 registers and up).  Twice that many
  // work-groups began anew half way: width 4096, one to eight rows of 4096 outputs 12.1 .. 14.6 us a launch, 11.2 .. 12.3 with what fits; 18720 outputs 30.2 | 28.6
  const int per_cu = std::min((int)(160 * 1024 / lds), (SB == 1 ? 16 : 8) / ks);
  hipLaunchKernelGGL((gemv_bf16_mc<GLU, SB>), dim3(std::min(tiles, std::max(1, per_cu) * ctx().n_cu)), dim3(64 * ks), lds, ctx().stream,
                     (const uint16_t*)w->data, x, (int)w->rows, (int)w->ld, ldx, n_tok, tiles, e);
  return CAI_OK;
}
static int run_gemv_mc(const cai_qw_s* w, const bf16_t* x, int64_t ldx, int n_tok, const LinEpi& e)
{
  const int slots = ((int)w->ld + 255) / 256;
  int ks = 1;
  while (ks < MC_WAVES && ks < slots) ks *= 2;
#define MC(SB) return e.mode == EPI_GLU ? run_mc<true, SB>(w, x, ldx, n_tok, e, ks) : run_mc<false, SB>(w, x, ldx, n_tok, e, ks)
  switch ((slots + ks - 1) / ks) { case 1: MC(1); case 2: MC(2); case 3: MC(3); default: MC(4); }
#undef MC
}

// The tiles (tokens x outputs, waves) of a product over `depth` bfloat16 columns of more rows than the walks take.
// Large tiles, by rounds over the chip: 256 x 256 by sixteen waves or 256 x 128 by sixteen, one work-group a CU, or 128 x 128 by eight, two a
// CU.  A full round takes 57, 32 and 37 us (at a depth of 2048), one of 128 x 128 with at most a work-group a CU 28.  Products alone, us,
// 256 x 256 | 256 x 128 | 128 x 128 by eight: 11264 rows, 1024 tokens 56 | 65 | 59, 2048: 113 | 105 | 108; 6200 rows, 1024 tokens 49 | 34 | 34, 2048: 57 | 67 | 67;
// without the first: 11264 rows, 300 tokens 30.8 | 31.9, 640: 57.1 | 35.6; 32800 rows, 128 tokens 57.6 | 43.9; 49152 rows, 100: 61.1 | 50.4.
// One round of 256 x 256 wants more than three fifths of the CUs (11264 rows over 256 columns, 700 tokens, 132 tiles: 23.6 | 18.8), and up to a depth of 512, where its start
// and end are half of it, a second round of the others that is three quarters full (11264 rows over 256, 900 tokens, not so: 25.1 | 22.5) or a gated product, which writes a quarter as much
// (12800 rows over 256, 900 tokens 13.4 | 15.0).
// Where one round of 128 x 128 covers everything, sixteen waves and copies three steps ahead (a CU has one work-group): 2048 x 2048, 2048 tokens 33 | 24 (256 x 128 |
// here), 2048 x 5632 75 | 54, 6200 x 2048, 512 tokens 29 (64 x 64) | 21, 11264 x 2048, 256 tokens 23 | 21; up to two tiles of 64 x 64 a CU those take less
// (2048 rows, 1024 tokens 16 | 20; 6200 rows, 256: 15 | 18.5), and a little past that: a CU holds three of them at once, so up to three a CU are one round.  64 x 64 | 128 x 128,
// 3072 rows, 700 tokens (2.06 a CU), depth 256 5.7 | 8.1, 512: 7.5 | 8.6, 1024: 11.8 | 12.3, 2048: 19.6 | 20.6, 4096: 34.5 | 35.5, 6400: 52.9 | 50.6; 4096 rows, 700 tokens (2.75 a CU) 6.2 | 7.6, 8.6 | 9.2, 12.8 |
// 13.4, 1536: 18.1 | 17.4, 2048: 22.4 | 21.6.  (The weights are what a first pass waits for: from HBM instead of a cache 128 x 128 is 0.8 to 0.95 times 64 x 64 from two a CU and a depth of 768
// on, but a small model's stay in the cache.)
// Against 256 x 128, 128 x 128 by eight and the small tiles alone, over 2889 sizes of eight depths from 256 to 5632, plain and gated, weights in the 256 MB cache, and 2512 with them in HBM:
// 0.945 to 0.990 times on average of a depth, never more than 1.01 times but for six sizes (1.015 to 1.056); by the times of a depth of 2048 whatever the depth is, up to 1.26 (1.41 with
// the weights in L2).
// What holds a tile's step up is neither the copies by themselves (128 x 128 steps alone 0.39 us, here 0.55), the fragment reads (two groups of waves with half
// the columns each, a quarter fewer, took the same) nor their order (a half step's read while the half before is multiplied: the same).
// Small tiles: a step is a hundred nanoseconds of work and a round trip to memory is a microsecond, so copies go out several steps ahead, as
// far as the LDS of the work-groups that share a CU allows (two slots: 5632 columns, 162 tokens 46 us a product of 2048 rows, six 20).  Whole prompt through
// four layers, us, two slots | these: width 2048, 20 tokens 884 | 569, 100: 962 | 687, 250: 1045 | 805, 400: 1116 | 976; 1024, 64: 653 | 496; 512, 250: 500 | 472.
// 64 x 64 with four and with six slots: 833, 854 at 250 tokens; 32 x 64 with four and with eight: within 2 %.
enum { TILES_32, TILES_64, TILES_128_16, TILES_128_8, TILES_256_128, TILES_256 };
static int lin_tiles(int64_t n_rows, int64_t depth, int n_tok, bool gated, int64_t n_cu)
{
  auto tiles = [&](int bm, int bn) { return (int64_t)((n_tok + bm - 1) / bm) * ((n_rows + bn - 1) / bn); };
  const int64_t small = tiles(128, 128), large = tiles(256, 128), huge = tiles(256, 256);
  if (n_tok > 64 && small <= n_cu && 4 * tiles(64, 64) > (depth > 4096 ? 8 : depth > 1024 ? 9 : 12) * n_cu) return TILES_128_16;
  if (n_tok > 64 && small >= n_cu) {
    const int64_t left = small % (2 * n_cu), t_small = 37 * (small / (2 * n_cu)) + (left == 0 ? 0 : left <= n_cu && small > n_cu ? 28 : 37);
    const int64_t t_large = 32 * ((large + n_cu - 1) / n_cu), t_huge = 57 * ((huge + n_cu - 1) / n_cu);
    if (t_huge < t_large && t_huge < t_small && 5 * huge > 3 * n_cu && (depth > 512 || gated || 4 * large > 7 * n_cu)) return TILES_256;
    return t_large <= t_small ? TILES_256_128 : TILES_128_8;
  }
  return n_tok > 32 && tiles(64, 64) >= n_cu ? TILES_64 : TILES_32;
}
// For the tests of the rule; host only, not part of the interface in caihip.h.
extern "C" int cai_bf16_tiles(int rows, int cols, int n_tok, int gated)
{
  CAI_ENTER();
  CAI_REQUIRE(rows >= 1 && cols >= 1 && n_tok >= 1, "cai_bf16_tiles: bad argument");
  return lin_tiles(rows, (cols + LIN_PAD - 1) / LIN_PAD * LIN_PAD, n_tok, gated != 0, ctx().n_cu);
}

template <typename AT>
static int run_lin(const cai_qw_s* w, const AT* x, int64_t ldx, int n_tok, const LinEpi& e)
{
  if constexpr (sizeof(AT) == 2) {
    // The 32-bit walk costs more with every row, this form hardly.  Of fewer than 8192 outputs (the walk's two-row form) one and two rows are the walk's, and up to
    // four between 2048 and 4096 columns, where a wave has two slots a tile and the walk one panel.  us a launch, walk | here: 2048 x 5632, one row 7.5 | 8.9, two
    // 8.25 | 9.1, three 10.8 | 9.3; 6200 x 2048 7.3 | 8.6, 7.95 | 8.65; 2048 x 2048 4.8 | 4.9, 5.0 | 5.0, three 6.05 | 5.0; 4096 x 4096 9.3 | 11.2, 10.55 | 11.3,
    // 11.0 | 11.4, four 11.65 | 11.5, eight 16.9 | 12.3; 18720 x 4096, one row 35.7 | 28.6; 32768 x 2048 27.7 | 26.8
    const bool few_outputs = (int)w->rows / 4 < ctx().n_cu * 8;
    const bool walk = few_outputs && (n_tok <= 2 || (n_tok <= 4 && w->ld > 2048 && w->ld <= 4096));
    if (!walk && n_tok <= MC_ROWS && w->ld <= 256 * MC_WAVES * MC_SLOTS) return run_gemv_mc(w, x, ldx, n_tok, e);
  }
  if (n_tok <= LIN_FEW) {
    const bool glu = e.mode == EPI_GLU;
    const GvShape s = gv_shape((int)w->rows, gv_turns(w), glu);
    run_gemv_rows<AT, GV_PLAIN>(n_tok, w, x, ldx, e, s, gv_blocks((int)w->rows, s, glu), gv_turns(w), GvSecond());
    return CAI_OK;
  }
  if constexpr (sizeof(AT) == 2)
    switch (lin_tiles(w->rows, w->ld, n_tok, e.mode == EPI_GLU, ctx().n_cu)) {
      case TILES_128_16: return run_gemm<AT, 128, 128, 4, 4, 4>(w, x, ldx, n_tok, e);
      case TILES_256: return run_gemm<AT, 256, 256, 4, 4, 2>(w, x, ldx, n_tok, e);
      case TILES_256_128: return run_gemm<AT, 256, 128, 4, 4, 3>(w, x, ldx, n_tok, e);
      case TILES_128_8: return run_gemm<AT, 128, 128, 2, 4>(w, x, ldx, n_tok, e);
      case TILES_64: return run_gemm<AT, 64, 64, 2, 2, 3>(w, x, ldx, n_tok, e);
      default: return run_gemm<AT, 32, 64, 2, 2, 6>(w, x, ldx, n_tok, e);
    }
  auto tiles = [&](int bm, int bn) { return (int64_t)((n_tok + bm - 1) / bm) * ((w->rows + bn - 1) / bn); };
  if (n_tok > 64 && tiles(128, 128) >= ctx().n_cu) return run_gemm<AT, 128, 128, 2, 2>(w, x, ldx, n_tok, e);
  if (n_tok > 32 && tiles(64, 64) >= ctx().n_cu) return run_gemm<AT, 64, 64, 2, 2>(w, x, ldx, n_tok, e);
  return run_gemm<AT, 32, 64, 2, 2>(w, x, ldx, n_tok, e);
}

int launch_lin_rms(int act_t, const float* x, int64_t ldx, int width, float eps, int n_tok, const RmsLin& a, const RmsLin* b)
{
  CAI_REQUIRE(n_tok >= 1 && n_tok <= LIN_FEW && a.w->cols == width && (!b || b->w->cols == width), "normed bf16 products: %d rows of %d columns", n_tok, width);
  auto mode_ok = [](const LinEpi& e) { return e.mode == EPI_STORE || e.mode == EPI_SPLIT; };
  CAI_REQUIRE(mode_ok(a.e) && (!b || mode_ok(b->e)), "normed bf16 products: an epilogue of another kind");
  CAI_REQUIRE(!b || !a.normed || !b->normed || a.ldn == b->ldn, "normed bf16 products: rows of two strides");
  const GvShape s = gv_shape((int)a.w->rows + (b ? (int)b->w->rows : 0), gv_turns(a.w), false);
  GvSecond q;
  q.blocks = gv_blocks((int)a.w->rows, s, false); q.width = width; q.eps = eps; q.gain = a.gain; q.normed = a.normed; q.ldn = a.ldn;
  int blocks = q.blocks;
  if (b) {
    q.W = (const uint16_t*)b->w->data; q.n_rows = (int)b->w->rows; q.e = b->e; q.gain2 = b->gain; q.normed2 = b->normed;
    if (b->normed) q.ldn = b->ldn;
    blocks += gv_blocks((int)b->w->rows, s, false);
  }
  if (act_t == ACT_T_BF16) run_gemv_rows<bf16_t, GV_RMS>(n_tok, a.w, x, ldx, a.e, s, blocks, gv_turns(a.w), q);
  else run_gemv_rows<float, GV_RMS>(n_tok, a.w, x, ldx, a.e, s, blocks, gv_turns(a.w), q);
  CAI_HIP(hipGetLastError());
  return CAI_OK;
}

int launch_lin_pair(int act_t, int n_tok, const cai_qw_s* w, const void* x, int64_t ldx, const LinEpi& e, const cai_qw_s* w2, const void* x2, int64_t ldx2, const LinEpi& e2)
{
  CAI_REQUIRE(n_tok >= 1 && n_tok <= LIN_FEW && w->rows == w2->rows && ldx >= w->ld && ldx2 >= w2->ld, "pair of bf16 products: %d rows, %lld and %lld outputs", n_tok, (long long)w->rows, (long long)w2->rows);
  CAI_REQUIRE(e.mode == EPI_JOIN && e2.mode == EPI_JOIN && e.y == e2.y && e.ldy == e2.ldy, "pair of bf16 products: both join one stream");
  const GvShape s = gv_shape((int)w->rows, std::min(gv_turns(w), gv_turns(w2)), false);
  GvSecond q;
  q.W = (const uint16_t*)w2->data; q.x = x2; q.ldw = (int)w2->ld; q.ldx = ldx2; q.e = e2;
  const int blocks = gv_blocks((int)w->rows, s, false), turns = std::max(gv_turns(w), gv_turns(w2));
  if (act_t == ACT_T_BF16) run_gemv_rows<bf16_t, GV_PAIR>(n_tok, w, x, ldx, e, s, blocks, turns, q);
  else run_gemv_rows<float, GV_PAIR>(n_tok, w, x, ldx, e, s, blocks, turns, q);
  CAI_HIP(hipGetLastError());
  return CAI_OK;
}

int launch_lin(const cai_qw_s* w, int act_t, const void* x, int64_t ldx, int n_tok, const LinEpi& e)
{
  CAI_REQUIRE(w->qtype == CAI_BF16 && n_tok >= 1 && ldx >= w->ld, "bf16 linear layer: %lld columns need activation rows of %lld, got %lld", (long long)w->cols, (long long)w->ld, (long long)ldx);
  CAI_REQUIRE(e.mode != EPI_GLU || w->rows % 32 == 0, "bf16 linear layer: a gated matrix needs whole blocks of 32 rows");
  const int rc = act_t == ACT_T_BF16 ? run_lin<bf16_t>(w, (const bf16_t*)x, ldx, n_tok, e) : run_lin<float>(w, (const float*)x, ldx, n_tok, e);
  if (rc) return rc;
  CAI_HIP(hipGetLastError());
  return CAI_OK;
}

// ------------------------------------------------------------------------------------------
// float columns [col0, col0 + cols) of x -> padded activation rows of the chosen type
// ------------------------------------------------------------------------------------------
template <typename AT>
__global__ __launch_bounds__(256) void pack_rows_kernel(const float* x, int64_t ldx, int64_t col0, int cols, void* out, int64_t ldo)
{
  const int t = blockIdx.y;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < ldo; i += gridDim.x * 256)
    put_act<AT>(out, t * ldo + i, i < cols ? x[t * ldx + col0 + i] : 0.0f);
}
int launch_pack_rows(const float* x, int64_t ldx, int64_t col0, int cols, int n_tok, int act_t, void* out, int64_t ldo)
{
  const dim3 grid((unsigned)std::min<int64_t>((ldo + 255) / 256, 32), n_tok);
  if (act_t == ACT_T_BF16) hipLaunchKernelGGL(pack_rows_kernel<bf16_t>, grid, dim3(256), 0, ctx().stream, x, ldx, col0, cols, out, ldo);
  else hipLaunchKernelGGL(pack_rows_kernel<float>, grid, dim3(256), 0, ctx().stream, x, ldx, col0, cols, out, ldo);
  CAI_HIP(hipGetLastError());
  return CAI_OK;
}

__global__ __launch_bounds__(256) void bf16_rows_kernel(const uint16_t* w, int64_t ld, int64_t cols, int64_t row0, float* out)
{
  const int64_t r = blockIdx.y;
  for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < cols; i += (int64_t)gridDim.x * 256)
    out[r * cols + i] = __builtin_bit_cast(float, (uint32_t)w[(row0 + r) * ld + i] << 16);
}
int bf16_dequant_rows(const cai_qw_s* w, int64_t row0, int64_t n_rows, float* out)
{
  for (int64_t r = 0; r < n_rows; r += 32768)
    hipLaunchKernelGGL(bf16_rows_kernel, dim3((unsigned)std::min<int64_t>((w->cols + 255) / 256, 32), (unsigned)std::min<int64_t>(n_rows - r, 32768)), dim3(256), 0, ctx().stream,
                       (const uint16_t*)w->data, w->ld, w->cols, row0 + r, out + r * w->cols);
  CAI_HIP(hipGetLastError());
  return CAI_OK;
}

// the stand-alone products (cai_qgemv, cai_qgemm) take unpadded float rows
static float* g_pack = nullptr; static size_t g_pack_cap = 0;
void bf16_release() { if (g_pack) (void)hipFree(g_pack); g_pack = nullptr; g_pack_cap = 0; }
int bf16_linear_f32(const cai_qw_s* w, const float* x, int64_t ldx, int n_tok, float* y, int64_t ldy, int act)
{
  const size_t need = (size_t)n_tok * w->ld;
  if (g_pack_cap < need) {
    CAI_HIP(hipStreamSynchronize(ctx().stream));
    bf16_release();
    CAI_HIP(hipMalloc((void**)&g_pack, need * 4));
    g_pack_cap = need;
  }
  int rc = launch_pack_rows(x, ldx, 0, (int)w->cols, n_tok, ACT_T_F32, g_pack, w->ld);
  if (rc) return rc;
  LinEpi e; e.y = y; e.ldy = ldy; e.bias = w->bias; e.act = act;
  return launch_lin(w, ACT_T_F32, g_pack, w->ld, n_tok, e);
}

}  // namespace cai

using namespace cai;

// One product over bfloat16 activation rows by itself, as a layered decoder's sublayers run it, on host memory: the rows of x are rounded to
// bfloat16.  gated: w holds blocks of 16 gate and 16 up rows, y[t][rows / 2] = relu(gate) * up rounded to bfloat16.  For the tests of the
// products (whole models bound them by a few percent only); not part of the interface in caihip.h.
extern "C" int cai_bf16_rows(cai_qw_t w, const float* x, int n_tok, int gated, float* y)
{
  CAI_ENTER();
  CAI_READY();
  CAI_REQUIRE(w && x && y && n_tok >= 1 && w->qtype == CAI_BF16, "cai_bf16_rows: bad argument");
  const hipStream_t st = ctx().stream;
  const int64_t outs = gated ? w->rows / 2 : w->rows;
  const size_t xb = (size_t)n_tok * w->cols * 4, hb = (size_t)n_tok * w->ld * 2, yb = (size_t)n_tok * outs * 4;
  auto round = [](size_t b) { return (b + 255) / 256 * 256; };
  char* d = nullptr;
  CAI_HIP(hipMalloc((void**)&d, round(xb) + round(hb) + yb));
  char* const dh = d + round(xb); char* const dy = dh + round(hb);
  hipError_t err = hipMemcpyAsync(d, x, xb, hipMemcpyHostToDevice, st);
  int rc = err == hipSuccess ? launch_pack_rows((const float*)d, w->cols, 0, (int)w->cols, n_tok, ACT_T_BF16, dh, w->ld) : CAI_OK;
  LinEpi e; e.bias = w->bias;
  if (gated) { e.mode = EPI_GLU; e.h = dy; e.ldh = outs; } else { e.y = (float*)dy; e.ldy = outs; }
  if (err == hipSuccess && !rc) rc = launch_lin(w, ACT_T_BF16, dh, w->ld, n_tok, e);
  if (err == hipSuccess && !rc) err = hipMemcpyAsync(y, dy, gated ? yb / 2 : yb, hipMemcpyDeviceToHost, st);
  if (err == hipSuccess) err = hipStreamSynchronize(st);
  (void)hipFree(d);
  if (err != hipSuccess) return hip_fail(err, "cai_bf16_rows", __FILE__, __LINE__);
  if (gated && !rc) {                      // (widened in place, from the last)
    const uint16_t* h = reinterpret_cast<const uint16_t*>(y);
    for (int64_t i = (int64_t)n_tok * outs; i-- > 0;) { const uint32_t v = (uint32_t)h[i] << 16; memcpy(y + i, &v, 4); }
  }
  return rc;
}
