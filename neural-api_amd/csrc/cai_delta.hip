// Gated delta rule with short convolutions: prompt kernels (convolution and unit norms, the scan, the gated output norm) and a
// one-launch decode kernel.
//
// Per head a float state S [dim][vdim] (rows padded to four columns, the padding stays zero); one token does  S <- diag(g) S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q.
// With S' = diag(g) S the read-out is  o = S'^T q + (q . k) u, so both products with S' are taken together and the second
// reduction is off the dependent chain.  Everything that touches the state is 32-bit.
#include "cai_layered.hpp"
#include "cai_recurrent.hpp"

namespace cai {

// ------------------------------------------------------------------------------------------
// prompt pass 1: q and k unit vectors (q scaled), v, decay, write strength, q . k.
// A wave owns one unit - the q and k channels of a key head, 256 channels of v, 256 decays, the write strengths - over eight
// consecutive rows; the convolution slides over them, so each input is fetched once (TAPS = 4; other lengths look back per row).  Where the eight rows
// are of one portion, all of them are requested before the first is convolved: row by row it was eight round trips (2048 rows of 8 + 16 heads of 128:
// 29 us, now 22).
// ------------------------------------------------------------------------------------------
constexpr int PREP_ROWS = 8;

template <int TAPS, int ND>                // ND: runs of 64 channels of a key head
__global__ __launch_bounds__(256) void delta_prep_kernel(const DeltaDims d, const DeltaIn in, const DeltaW w, const float* hist, const int64_t h_elems, const StepRows r, const DeltaBuf b)
{
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r0 = blockIdx.x * PREP_ROWS, r1 = min(r0 + PREP_ROWS, r.n_rows);
  const int C = d.channels(), kw = d.kv_heads * d.dim, vw = d.heads * d.vdim, bw = d.heads + d.kv_heads;
  const int gw = d.channel_decay ? d.heads * d.dim : d.heads;
  const int nv = (vw + 255) / 256, ng = (gw + 255) / 256;
  int unit = blockIdx.y * 4 + wave;
  const bool one = TAPS && r1 - r0 == PREP_ROWS && r.first[r0] == r.first[r1 - 1];
  if (unit < d.kv_heads) {
    const int g = unit, c0 = g * d.dim;
    const float qs = rsqrtf((float)d.dim);
    ConvWindow<TAPS ? TAPS : 2> wq, wk;
    // unit vectors and their product from a row's convolved channels
    auto finish = [&](int row, const float (&q)[4], const float (&k)[4]) {
      float sq = 0.0f, sk = 0.0f, dot = 0.0f;
#pragma unroll
      for (int i = 0; i < ND; i++) { sq = fmaf(q[i], q[i], sq); sk = fmaf(k[i], k[i], sk); dot = fmaf(q[i], k[i], dot); }
      const float nq = qs / sqrtf(wave_total(sq) + 1e-6f), nk = 1.0f / sqrtf(wave_total(sk) + 1e-6f);
      dot = wave_total(dot) * nq * nk;
#pragma unroll
      for (int i = 0; i < ND; i++) {
        const int c = lane + 64 * i;
        if (c < d.dim) { b.q[(int64_t)row * kw + c0 + c] = q[i] * nq; b.k[(int64_t)row * kw + c0 + c] = k[i] * nk; }
      }
      if (lane == 0) b.beta[(int64_t)row * bw + d.heads + g] = dot;
    };
    if constexpr (TAPS != 0) {
      if (one) {
        float qi[PREP_ROWS][ND], ki[PREP_ROWS][ND];
        const float* const p0 = in.proj + r0 * in.ldp + c0;
#pragma unroll
        for (int u = 0; u < PREP_ROWS; u++)
#pragma unroll
          for (int i = 0; i < ND; i++) { const int c = min(lane + 64 * i, d.dim - 1); qi[u][i] = p0[u * in.ldp + in.oq + c]; ki[u][i] = p0[u * in.ldp + in.ok + c]; }
        const int pos = r.pos[r0], back = r0 - r.first[r0];
        const float* const ring = hist + r.slot[r0] * h_elems;
        wq.taps(w.cq, c0, lane, d.dim); wk.taps(w.ck, c0, lane, d.dim);
        wq.history(in.proj + r0 * in.ldp + in.oq, in.ldp, back, pos, ring, C, 0, c0, lane, d.dim);
        wk.history(in.proj + r0 * in.ldp + in.ok, in.ldp, back, pos, ring, C, kw, c0, lane, d.dim);
#pragma unroll
        for (int u = 0; u < PREP_ROWS; u++) {
          float q[4], k[4];
#pragma unroll
          for (int i = 0; i < ND; i++) { const bool in_head = lane + 64 * i < d.dim; q[i] = wq.step(i, in_head ? qi[u][i] : 0.0f); k[i] = wk.step(i, in_head ? ki[u][i] : 0.0f); }
          finish(r0 + u, q, k);
        }
        return;
      }
    }
    if (TAPS) { wq.taps(w.cq, c0, lane, d.dim); wk.taps(w.ck, c0, lane, d.dim); }
    for (int row = r0; row < r1; row++) {
      const int pos = r.pos[row], back = row - r.first[row];
      const float* ring = hist + r.slot[row] * h_elems;
      const float* p = in.proj + row * in.ldp;
      if (TAPS && (row == r0 || back == 0)) {
        wq.history(p + in.oq, in.ldp, back, pos, ring, C, 0, c0, lane, d.dim);
        wk.history(p + in.ok, in.ldp, back, pos, ring, C, kw, c0, lane, d.dim);
      }
      float q[4], k[4];
#pragma unroll
      for (int i = 0; i < ND; i++) { const int c = lane + 64 * i; q[i] = c < d.dim ? p[in.oq + c0 + c] : 0.0f; k[i] = c < d.dim ? p[in.ok + c0 + c] : 0.0f; }
#pragma unroll
      for (int i = 0; i < ND; i++) {
        const int c = lane + 64 * i;
        if (TAPS) { q[i] = wq.step(i, q[i]); k[i] = wk.step(i, k[i]); }
        else if (c < d.dim) {
          q[i] = conv_silu(p + in.oq, in.ldp, back, pos, ring, C, 0, w.cq, d.taps, c0 + c);
          k[i] = conv_silu(p + in.ok, in.ldp, back, pos, ring, C, kw, w.ck, d.taps, c0 + c);
        }
      }
      finish(row, q, k);
    }
    return;
  }
  unit -= d.kv_heads;
  if (unit < nv) {
    const int c0 = unit * 256, n = min(256, vw - c0);
    ConvWindow<TAPS ? TAPS : 2> wv;
    if constexpr (TAPS != 0) {
      if (one) {
        float vi[PREP_ROWS][4];
        const float* const p0 = in.proj + r0 * in.ldp + in.ov;
#pragma unroll
        for (int u = 0; u < PREP_ROWS; u++)
#pragma unroll
          for (int i = 0; i < 4; i++) vi[u][i] = p0[u * in.ldp + c0 + min(lane + 64 * i, n - 1)];
        const int pos = r.pos[r0], back = r0 - r.first[r0];
        wv.taps(w.cv, c0, lane, n);
        wv.history(p0, in.ldp, back, pos, hist + r.slot[r0] * h_elems, C, 2 * kw, c0, lane, n);
#pragma unroll
        for (int u = 0; u < PREP_ROWS; u++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const int c = lane + 64 * i;
            const float v = wv.step(i, c < n ? vi[u][i] : 0.0f);
            if (c < n) b.v[(int64_t)(r0 + u) * vw + c0 + c] = v;
          }
        return;
      }
    }
    if (TAPS) wv.taps(w.cv, c0, lane, n);
    for (int row = r0; row < r1; row++) {
      const int pos = r.pos[row], back = row - r.first[row];
      const float* ring = hist + r.slot[row] * h_elems;
      const float* p = in.proj + row * in.ldp + in.ov;
      if (TAPS && (row == r0 || back == 0)) wv.history(p, in.ldp, back, pos, ring, C, 2 * kw, c0, lane, n);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int c = lane + 64 * i;
        if (TAPS) { const float v = wv.step(i, c < n ? p[c0 + c] : 0.0f); if (c < n) b.v[(int64_t)row * vw + c0 + c] = v; }
        else if (c < n) b.v[(int64_t)row * vw + c0 + c] = conv_silu(p, in.ldp, back, pos, ring, C, 2 * kw, w.cv, d.taps, c0 + c);
      }
    }
    return;
  }
  unit -= nv;
  if (unit < ng) {
    for (int i = 0; i < 4; i++) {
      const int c = unit * 256 + lane + 64 * i;
      if (c >= gw) continue;
      const float bias = w.dt_bias[c], rate = w.rate[d.channel_decay ? c / d.dim : c];
#pragma unroll
      for (int u = 0; u < PREP_ROWS; u++) {
        const int row = min(r0 + u, r1 - 1);
        const float z = d.rank_a ? b.za[(int64_t)row * gw + c] : in.proj[row * in.ldp + in.oa + c];
        b.g[(int64_t)row * gw + c] = expf(rate * softplus_f(z + bias));
      }
    }
    return;
  }
  if (unit == ng)
    for (int row = r0; row < r1; row++)
      for (int h = lane; h < d.heads; h += 64) b.beta[(int64_t)row * bw + h] = sigmoid_f(in.proj[row * in.ldp + in.ob + h]);
}

// ------------------------------------------------------------------------------------------
// prompt pass 2 for short portions: the scan.  A wave owns four columns of one head's state: 16 lanes a column, RPL rows a lane (rows
// 64 j + 4 (lane & 15) + i), in registers for the whole portion.  Tokens are staged through LDS 16 at a time, the next block
// requested before the current one is walked; the walk itself has no barrier.
// ------------------------------------------------------------------------------------------
constexpr int SCAN_TB = 16;
template <int RPL, bool CH>
__global__ __launch_bounds__(256) void delta_scan_kernel(const DeltaDims d, float* state, const int64_t s_elems, const StepRows r, const DeltaBuf b)
{
  constexpr int DP = RPL * 16;
  __shared__ f32x4 sq[SCAN_TB][DP / 4], sk[SCAN_TB][DP / 4], sg[CH ? SCAN_TB : 1][CH ? DP / 4 : 1];
  __shared__ float sv[SCAN_TB][16], so[SCAN_TB][16], sgs[SCAN_TB], sb[SCAN_TB], sqk[SCAN_TB];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c0 = blockIdx.x * 16, h = blockIdx.y;
  const int32_t* en = r.ent + 4 * blockIdx.z;
  const int slot = en[0], row0 = en[1], n = en[2], pos0 = en[3];
  const int g = h / (d.heads / d.kv_heads), kw = d.kv_heads * d.dim, vw = d.heads * d.vdim, gw = d.heads * d.dim, bw = d.heads + d.kv_heads;
  const int rg = lane & 15, cl = wave * 4 + (lane >> 4), col = c0 + cl;
  const int dvp = d.vdim_p();
  float* Sg = state + slot * s_elems + (int64_t)h * d.dim * dvp;
  float S[RPL];
#pragma unroll
  for (int j = 0; j < RPL; j++) {
    const int rr = (j >> 2) * 64 + rg * 4 + (j & 3);
    S[j] = pos0 > 0 && rr < d.dim && col < d.vdim ? Sg[(int64_t)rr * dvp + col] : 0.0f;
  }
  float nq[RPL], nk[RPL], ng[CH ? RPL : 1], nv, nb, nqk, ngs;
  auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < RPL; i++) {
      const int e = tid + 256 * i, t = t0 + e / DP, c = e % DP;
      const bool ok = t < n && c < d.dim;
      const int64_t rw = row0 + (ok ? t : 0);
      const int cc = ok ? c : 0;
      nq[i] = b.q[rw * kw + g * d.dim + cc]; nk[i] = b.k[rw * kw + g * d.dim + cc];
      if (CH) ng[i] = b.g[rw * gw + h * d.dim + cc];
      if (!ok) { nq[i] = 0.0f; nk[i] = 0.0f; }
    }
    {
      const int t = t0 + (tid >> 4), c = c0 + (tid & 15);
      nv = t < n && c < d.vdim ? b.v[(int64_t)(row0 + t) * vw + h * d.vdim + c] : 0.0f;
    }
    if (tid < SCAN_TB) {
      const int64_t rw = row0 + min(t0 + tid, n - 1);
      nb = b.beta[rw * bw + h]; nqk = b.beta[rw * bw + d.heads + g];
      if (!CH) ngs = b.g[rw * d.heads + h];
    }
  };
  fetch(0);
  for (int t0 = 0; t0 < n; t0 += SCAN_TB) {
#pragma unroll
    for (int i = 0; i < RPL; i++) {
      const int e = tid + 256 * i, t = e / DP, c = e % DP;
      reinterpret_cast<float*>(sq[t])[c] = nq[i]; reinterpret_cast<float*>(sk[t])[c] = nk[i];
      if (CH) reinterpret_cast<float*>(sg[t])[c] = ng[i];
    }
    sv[tid >> 4][tid & 15] = nv;
    if (tid < SCAN_TB) { sb[tid] = nb; sqk[tid] = nqk; if (!CH) sgs[tid] = ngs; }
    __syncthreads();
    if (t0 + SCAN_TB < n) fetch(t0 + SCAN_TB);
    const int nt = min(SCAN_TB, n - t0);
    auto token = [&](int t) {
      float ks = 0.0f, qd = 0.0f;
      f32x4 kf[RPL / 4];
#pragma unroll
      for (int j = 0; j < RPL / 4; j++) {
        kf[j] = sk[t][j * 16 + rg];
        const f32x4 qf = sq[t][j * 16 + rg];
        f32x4 gf;
        if (CH) gf = sg[t][j * 16 + rg];
        else { const float s = sgs[t]; gf = f32x4{s, s, s, s}; }
#pragma unroll
        for (int i = 0; i < 4; i++) {
          S[j * 4 + i] *= gf[i];
          ks = fmaf(S[j * 4 + i], kf[j][i], ks); qd = fmaf(S[j * 4 + i], qf[i], qd);
        }
      }
      ks = row16_total(ks); qd = row16_total(qd);
      const float u = sb[t] * (sv[t][cl] - ks);
#pragma unroll
      for (int j = 0; j < RPL / 4; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) S[j * 4 + i] = fmaf(kf[j][i], u, S[j * 4 + i]);
      if (rg == 0) so[t][cl] = fmaf(sqk[t], u, qd);
    };
    if (nt == SCAN_TB) {
#pragma unroll 4
      for (int t = 0; t < SCAN_TB; t++) token(t);
    } else for (int t = 0; t < nt; t++) token(t);
    __syncthreads();
    {
      const int t = tid >> 4, c = c0 + (tid & 15);
      if (t < nt && c < d.vdim) b.o[(int64_t)(row0 + t0 + t) * vw + h * d.vdim + c] = so[t][tid & 15];
    }
  }
#pragma unroll
  for (int j = 0; j < RPL; j++) {
    const int rr = (j >> 2) * 64 + rg * 4 + (j & 3);
    if (rr < d.dim && col < dvp) Sg[(int64_t)rr * dvp + col] = S[j];
  }
}

// ------------------------------------------------------------------------------------------
// prompt pass 2 for long portions: the same recurrence in chunks of 16 tokens, on the float matrix cores (32-bit throughout).
//
// With P_t the product of the decays of the chunk's tokens up to t, D_ts that of the tokens after s up to t, and S the state
// before the chunk, the writes u of a chunk solve a unit lower triangular system,
//     u_t = beta_t (v_t - S^T (P_t k_t) - sum_{s<t} A_ts u_s),   A_ts = k_t . D_ts k_s,
// so with T = (I + diag(beta) A)^-1 diag(beta):   U = T V - (T [P k]) S =: U0 - W S.   Then
//     o_t = S^T (P_t q_t) + sum_{s<=t} (q_t . D_ts k_s) u_s,      S <- P_16 S + sum_s (D_16,s k_s) u_s^T.
// Everything before "S" is made for all chunks at once (first kernel); the second kernel walks the chunks of a sequence with a
// 16-column slice of the state in registers.  Decays enter only as running products, never as quotients or differences of
// logarithms, so strong decay costs no accuracy.
//
// The first kernel leaves a chunk's factors of one head as the walk's matrix operands, a record of 1 KB blocks [64 lanes][4 floats]
// (fr = lane % 16, fg = lane / 16; everything past the portion's end or a width is zero):
//     block j                 - W,    token fr, channels 16 j + 4 fg ..      (tiles of them)
//     block tiles + j         P q,    token fr, channels 16 j + 4 fg ..
//     block 2 tiles + j       D_16 k, tokens 4 fg .., channel 16 j + fr
//     block 3 tiles           q D k,  token fr, writing tokens 4 fg ..
//     block 3 tiles + 1 + c   U0,     tokens 4 fg .., value column 16 c + fr
// so that the walk, whose chain of 128 chunks is what a prompt of 2048 tokens waits for, requests one contiguous KB an instruction
// and puts it into a product as it comes.  Read from arrays by row instead, with the masks, decays and signs applied in the walk (18 requests
// and 70 more vector instructions a chunk), 16 heads of 128 x 128 took 157 us for 2048 tokens; now 96 (128 work-groups).
// ------------------------------------------------------------------------------------------
constexpr int CHUNK = DELTA_CHUNK;

// The chunks of a launch and their records: all of a step as listed, or (chunks null) of every entry those from `first` on, `most` records each
struct DeltaPass { const int32_t *chunks, *chunk0; int first, most; };

template <bool CH>
__global__ __launch_bounds__(256) void delta_chunk_kernel(const DeltaDims d, const StepRows r, const DeltaBuf b, const DeltaPass p)
{
  extern __shared__ float lds[];
  __shared__ float sA[CHUNK][CHUNK + 1], sQ[CHUNK][CHUNK + 1], sP[CH ? 1 : 4][CHUNK][CHUNK + 1];
  __shared__ f32x4 sT[CHUNK][CHUNK / 4];
  __shared__ float sbeta[CHUNK], sg1[CHUNK], sdot[CHUNK], sz[CHUNK];      // sdot: q . k, later (one decay a head) the running products of the decays
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), fr = lane & 15, fg = lane >> 4;
  const int32_t* en = r.ent + 4 * (p.chunks ? p.chunks[2 * blockIdx.x] : (int)blockIdx.x / p.most);
  const int t0 = p.chunks ? p.chunks[2 * blockIdx.x + 1] : (p.first + (int)blockIdx.x % p.most) * CHUNK, nt = min(CHUNK, en[2] - t0), h = blockIdx.y;
  if (nt <= 0) return;                     // (whole work-groups: an entry that ends before the pass does)
  const int64_t row0 = en[1] + t0;
  const int g = h / (d.heads / d.kv_heads), kw = d.kv_heads * d.dim, vw = d.heads * d.vdim, gw = d.heads * d.dim, bw = d.heads + d.kv_heads;
  const int dp = (d.dim + 15) & ~15, DS = dp + 4, tiles = delta_tiles(d);
  float *sk = lds, *sq = lds + CHUNK * DS, *sg = lds + 2 * CHUNK * DS;       // sg: channel decays
  for (int e = tid; e < CHUNK * dp; e += 256) {
    const int t = e / dp, c = e - t * dp;
    const bool ok = t < nt && c < d.dim;
    const int64_t rw = row0 + (ok ? t : 0); const int cc = ok ? c : 0;
    const float k = b.k[rw * kw + g * d.dim + cc], q = b.q[rw * kw + g * d.dim + cc];
    sk[t * DS + c] = ok ? k : 0.0f; sq[t * DS + c] = ok ? q : 0.0f;
    if (CH) { const float x = b.g[rw * gw + h * d.dim + cc]; sg[t * DS + c] = ok ? x : 1.0f; }
  }
  if (tid < CHUNK) {
    const bool ok = tid < nt; const int64_t rw = row0 + (ok ? tid : 0);
    sbeta[tid] = ok ? b.beta[rw * bw + h] : 0.0f; sdot[tid] = ok ? b.beta[rw * bw + d.heads + g] : 0.0f;
    sg1[tid] = !CH && ok ? b.g[rw * d.heads + h] : 1.0f;
  }
  __syncthreads();
  if (CH) {
    // thread (s, 16 channel lanes): running product of the decays after s
    const int s = tid >> 4, cl = tid & 15;
    float a[CHUNK], o[CHUNK];
#pragma unroll
    for (int t = 0; t < CHUNK; t++) a[t] = o[t] = 0.0f;
    for (int c = cl; c < dp; c += 16) {
      const float ks = sk[s * DS + c];
      float e = ks;
#pragma unroll
      for (int t = 1; t < CHUNK; t++) {
        e = t > s ? e * sg[t * DS + c] : e;
        a[t] = fmaf(sk[t * DS + c], e, a[t]); o[t] = fmaf(sq[t * DS + c], e, o[t]);
      }
    }
#pragma unroll
    for (int t = 0; t < CHUNK; t++) {
      const float x = row16_total(a[t]), y = row16_total(o[t]);
      if (cl == 0) { sA[t][s] = t > s ? x : 0.0f; sQ[t][s] = t > s ? y : t == s ? sdot[t] : 0.0f; }
    }
    __syncthreads();
    // the factors of the three products, each in its place: k times the decays behind it, q and k (in place of the decays) times those up to it
    for (int c = tid; c < 16 * tiles; c += 256) {
      float p = 1.0f;
      if (c < dp) {
        float z = 1.0f, k[CHUNK], gr[CHUNK];
#pragma unroll
        for (int t = CHUNK - 1; t >= 0; t--) {
          gr[t] = sg[t * DS + c]; k[t] = sk[t * DS + c];
          sk[t * DS + c] = k[t] * z;
          z *= gr[t];
        }
#pragma unroll
        for (int t = 0; t < CHUNK; t++) {
          p *= gr[t];
          sq[t * DS + c] *= p; sg[t * DS + c] = k[t] * p;
        }
      }
      b.gt[((int64_t)blockIdx.x * d.heads + h) * (16 * tiles) + c] = p;
    }
  } else {
    // K K^T and Q K^T, half of the width by each of two waves
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const float* am = wave & 1 ? sq : sk;
    for (int kt = wave >> 1; kt < dp / 16; kt += 2) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(am + fr * DS + kt * 16 + fg * 4), y = *reinterpret_cast<const f32x4*>(sk + fr * DS + kt * 16 + fg * 4);
#pragma unroll
      for (int i = 0; i < 4; i++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], y[i], acc, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) sP[wave][fg * 4 + i][fr] = acc[i];
    __syncthreads();
    const int t = tid >> 4, s = tid & 15;
    float e = t >= s ? 1.0f : 0.0f;
#pragma unroll
    for (int x = 1; x < CHUNK; x++) e *= x > s && x <= t ? sg1[x] : 1.0f;
    sA[t][s] = t > s ? e * (sP[0][t][s] + sP[2][t][s]) : 0.0f;
    sQ[t][s] = e * (sP[1][t][s] + sP[3][t][s]);
    if (tid < CHUNK) {
      float p = 1.0f, z = 1.0f;
#pragma unroll
      for (int x = 0; x < CHUNK; x++) { p *= x <= tid ? sg1[x] : 1.0f; z *= x > tid ? sg1[x] : 1.0f; }
      sdot[tid] = p; sz[tid] = z;
      if (tid == CHUNK - 1) b.gt[(int64_t)blockIdx.x * d.heads + h] = p;
    }
  }
  __syncthreads();
  f32x4* const rec = reinterpret_cast<f32x4*>(b.rec) + ((int64_t)blockIdx.x * d.heads + h) * (64 * delta_record_blocks(d)) + lane;
  if (tid < CHUNK) {                       // column tid of T by forward substitution
    float c[CHUNK];
#pragma unroll
    for (int t = 0; t < CHUNK; t++) {
      float x = t == tid ? 1.0f : 0.0f;
#pragma unroll
      for (int s = 0; s < t; s++) x = fmaf(-sA[t][s], c[s], x);
      c[t] = x * sbeta[t];
      reinterpret_cast<float*>(sT[t])[tid] = c[t];
    }
  }
  // the factors that do not need T, while wave 0 substitutes
  for (int j = wave; j < 2 * tiles + 1; j += 4) {
    f32x4 x = {0.0f, 0.0f, 0.0f, 0.0f};
    const int ct = j < tiles ? j : j - tiles;
    if (j == 2 * tiles) {
#pragma unroll
      for (int i = 0; i < 4; i++) x[i] = sQ[fr][fg * 4 + i];
    } else if (ct * 16 < dp) {
      if (j < tiles) {
        x = *reinterpret_cast<const f32x4*>(sq + fr * DS + ct * 16 + fg * 4);
        if (!CH) x *= sdot[fr];
      } else
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = CH ? sk[(fg * 4 + i) * DS + ct * 16 + fr] : sk[(fg * 4 + i) * DS + ct * 16 + fr] * sz[fg * 4 + i];
    }
    rec[64 * (tiles + j)] = x;
  }
  __syncthreads();
  const f32x4 tf = sT[fr][fg];
  for (int ct = wave; ct < tiles; ct += 4) {             // W = T [P k]: channels as rows, tokens as columns of the result
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    if (ct * 16 < dp)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int s = fg * 4 + i, c = ct * 16 + fr;
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(CH ? sg[s * DS + c] : sk[s * DS + c] * sdot[s], tf[i], acc, 0, 0, 0);
      }
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = fr < nt ? -acc[i] : 0.0f;
    rec[64 * ct] = acc;
  }
  for (int ct = wave; ct * 16 < d.vdim; ct += 4) {       // U0 = T V
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const int c = ct * 16 + fr;
    float x[4];
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = fg * 4 + i < nt && c < d.vdim ? b.v[(row0 + fg * 4 + i) * vw + h * d.vdim + c] : 0.0f;
#pragma unroll
    for (int i = 0; i < 4; i++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(tf[i], x[i], acc, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = fg * 4 + i < nt ? acc[i] : 0.0f;
    rec[64 * (3 * tiles + 1 + ct)] = acc;
  }
}

// The walk: one work-group per (16 value columns, head, entry).  Waves 0 .. NW - 1 hold the state - wave w the key rows of tiles
// w TPW .. as matrix-core result registers, which are at the same time an operand of the products with S - and wave NW makes
// the output: it contributes U0 to the sum of a chunk's writes and finishes the previous chunk's rows of o while the others are a
// chunk further.  One barrier a chunk; the partial sums live in LDS for three chunks.
// What bounds it: the chain from chunk to chunk - 8 products, their parts through LDS (a third of the time), 8 products: 1700 cycles, 130 of
// them waiting for the other waves.  U0 as the start of a state wave's sums and U handed to wave NW took 102 us where this takes 96, factors
// five chunks ahead 92 to 98, the read-out in front of the barrier or around it 98 to 100.
template <int NW, int TPW, bool CH, bool WHOLE>      // WHOLE: the value width is a multiple of sixteen
__global__ __launch_bounds__(64 * (NW + 1)) void delta_walk_kernel(const DeltaDims d, float* state, const int64_t s_elems, const StepRows r, const DeltaBuf b, const DeltaPass p)
{
  constexpr int TILES = NW * TPW;
  __shared__ f32x4 pu[3][NW + 1][64], po[3][NW][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), fr = lane & 15, fg = lane >> 4;
  // consecutive work-groups go to different XCDs; the column slices of a head read the same chunk data, so with heads in whole
  // eights every head stays on one XCD (and in its L2)
  const int slices = (d.vdim + 15) / 16;
  const int h = d.heads % 8 == 0 ? (blockIdx.x & 7) + 8 * ((blockIdx.x >> 3) / slices) : blockIdx.x / slices;
  const int slice = d.heads % 8 == 0 ? (blockIdx.x >> 3) % slices : blockIdx.x % slices, col = slice * 16 + fr;
  const int32_t* en = r.ent + 4 * blockIdx.y;
  const int skip = p.first * CHUNK, slot = en[0], row0 = en[1] + skip, n = min(en[2] - skip, p.most * CHUNK), pos0 = en[3] + skip, ch0 = p.chunks ? p.chunk0[blockIdx.y] : (int)blockIdx.y * p.most;
  if (n <= 0) return;
  const int vw = d.heads * d.vdim, dvp = d.vdim_p(), blocks = delta_record_blocks(d);
  const int nc = (n + CHUNK - 1) / CHUNK;
  const f32x4* const rec = reinterpret_cast<const f32x4*>(b.rec) + ((int64_t)ch0 * d.heads + h) * (64 * blocks);
  const int64_t step = (int64_t)d.heads * (64 * blocks);
  auto total = [&](int it) -> f32x4 {                    // a chunk's writes: U0 and every wave's part of - W S
    f32x4 x[NW];
#pragma unroll
    for (int v = 0; v < NW; v++) x[v] = pu[it][v][lane];
    x[0] += pu[it][NW][lane];
#pragma unroll
    for (int m = NW / 2; m; m >>= 1)
#pragma unroll
      for (int v = 0; v < m; v++) x[v] += x[v + m];
    return x[0];
  };
  if (wave == NW) {
    struct Out { f32x4 u0, qk; };
    auto fetch = [&](int c, Out& x) {
      const f32x4* p = rec + min(c, nc - 1) * step;
      x.u0 = p[64 * (3 * TILES + 1 + slice) + lane]; x.qk = p[64 * (3 * TILES) + lane];
    };
    f32x4 qk_last;
    float* const ob = b.o + (int64_t)(row0 + fr) * vw + h * d.vdim + slice * 16 + fg * 4;     // token fr, columns 4 fg ..
    auto finish = [&](int c, int it, bool last) {        // rows of o of chunk c (parts it)
      f32x4 o = po[it][0][lane];
#pragma unroll
      for (int v = 1; v < NW; v++) o += po[it][v][lane];
      const f32x4 u = total(it);
#pragma unroll
      for (int i = 0; i < 4; i++) o = __builtin_amdgcn_mfma_f32_16x16x4f32(u[i], qk_last[i], o, 0, 0, 0);
      float* const p = ob + (int64_t)c * CHUNK * vw;
      if (WHOLE && !last) *reinterpret_cast<f32x4_any*>(p) = o;
      else if (c * CHUNK + fr < n)
#pragma unroll
        for (int i = 0; i < 4; i++) if (slice * 16 + fg * 4 + i < d.vdim) p[i] = o[i];
    };
    auto chunk = [&](int c, const Out& x, int it) {
      pu[it][NW][lane] = x.u0;
      __syncthreads();
      finish(c - 1, (it + 2) % 3, false);
      qk_last = x.qk;
    };
    // (all stores of the loop are without a condition: a store that may not have happened makes every wait for a chunk's factors wait for
    // the stores behind them too, and this wave then holds up the others: 110 us)
    Out xa, xb, xc;
    fetch(0, xa); fetch(1, xb); fetch(2, xc);
    pu[0][NW][lane] = xa.u0;
    qk_last = xa.qk;
    __syncthreads();
    for (int c = 1; c < nc; c += 3) {
      fetch(c + 2, xa); chunk(c, xb, 1);
      if (c + 1 >= nc) break;
      fetch(c + 3, xb); chunk(c + 1, xc, 2);
      if (c + 2 >= nc) break;
      fetch(c + 4, xc); chunk(c + 2, xa, 0);
    }
    __syncthreads();
    finish(nc - 1, (nc - 1) % 3, true);
    return;
  }
  float* Sg = state + slot * s_elems + (int64_t)h * d.dim * dvp;
  f32x4 S[TPW];
#pragma unroll
  for (int j = 0; j < TPW; j++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int c = (wave * TPW + j) * 16 + fg * 4 + i;
      S[j][i] = pos0 > 0 && c < d.dim && col < d.vdim ? Sg[(int64_t)c * dvp + col] : 0.0f;
    }
  // a chunk's factors are requested two chunks ahead
  struct In { f32x4 w[TPW], q[TPW], k[TPW], tot[CH ? TPW : 1]; };
  const f32x4* const mine = rec + 64 * TPW * wave + lane;
  const float* const tot = CH ? b.gt + ((int64_t)ch0 * d.heads + h) * (16 * TILES) + 16 * TPW * wave + 4 * fg : b.gt + (int64_t)ch0 * d.heads + h;
  const int tstep = CH ? d.heads * (16 * TILES) : d.heads;
  auto fetch = [&](int c, In& x) {
    const int cc = min(c, nc - 1);
    const f32x4* const p = mine + cc * step;
    const float* const t = tot + (int64_t)cc * tstep;
#pragma unroll
    for (int j = 0; j < TPW; j++) x.w[j] = p[64 * j];
    if (CH)
#pragma unroll
      for (int j = 0; j < TPW; j++) x.tot[j] = *reinterpret_cast<const f32x4*>(t + 16 * j);
    else x.tot[0][0] = *t;
#pragma unroll
    for (int j = 0; j < TPW; j++) { x.q[j] = p[64 * (TILES + j)]; x.k[j] = p[64 * (2 * TILES + j)]; }
  };
  auto chunk = [&](const In& x, int it) {
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 u[2] = {zero, zero}, o = zero;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < TPW; j++) u[(i * TPW + j) & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[j][i], S[j][i], u[(i * TPW + j) & 1], 0, 0, 0);
    pu[it][wave][lane] = u[0] + u[1];
    __syncthreads();
    const f32x4 t = total(it);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < TPW; j++)        // the read-out with the state before the chunk, columns as rows of the result, while the sums arrive
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(S[j][i], x.q[j][i], o, 0, 0, 0);
    po[it][wave][lane] = o;
#pragma unroll
    for (int j = 0; j < TPW; j++) S[j] *= CH ? x.tot[CH ? j : 0] : f32x4{x.tot[0][0], x.tot[0][0], x.tot[0][0], x.tot[0][0]};
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < TPW; j++) S[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[j][i], t[i], S[j], 0, 0, 0);
  };
  // (the scheduling barriers keep a chunk's requests in front of the chunk that is worked on: they are used two chunks later)
  In xa, xb, xc;
  fetch(0, xa); fetch(1, xb);
  for (int c = 0;; c += 3) {
    fetch(c + 2, xc);
    __builtin_amdgcn_sched_barrier(0);
    chunk(xa, 0);
    if (c + 1 >= nc) break;
    fetch(c + 3, xa);
    __builtin_amdgcn_sched_barrier(0);
    chunk(xb, 1);
    if (c + 2 >= nc) break;
    fetch(c + 4, xb);
    __builtin_amdgcn_sched_barrier(0);
    chunk(xc, 2);
    if (c + 3 >= nc) break;
  }
  __syncthreads();                         // the last chunk's read-outs are there
#pragma unroll
  for (int j = 0; j < TPW; j++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int c = (wave * TPW + j) * 16 + fg * 4 + i;
      if (c < d.dim && col < dvp) Sg[(int64_t)c * dvp + col] = S[j][i];
    }
}

// ------------------------------------------------------------------------------------------
// prompt pass 3: per row and head RMS norm, gain, gate; then the row's raw inputs into the ring if the portion's last taps reach it
// ------------------------------------------------------------------------------------------
template <typename AT, int NV>             // NV: runs of 64 columns of a head
__global__ __launch_bounds__(256) void delta_finish_kernel(const DeltaDims d, const DeltaIn in, const DeltaW w, float* hist, const int64_t h_elems, const StepRows r, const DeltaBuf b, AT* out, const int64_t ldo)
{
  const int row = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int vw = d.heads * d.vdim;
  const float* p = in.proj + row * in.ldp;
  const float* gate = d.rank_g ? b.zg + (int64_t)row * vw : p + in.og;
  // four heads of a wave requested together (heads past the last one: that again, not written)
  constexpr int AT_ONCE = 4;
  for (int h0 = wave; h0 < d.heads; h0 += 4 * AT_ONCE) {
    float o[AT_ONCE][NV], z[AT_ONCE][NV], gain[NV];
#pragma unroll
    for (int k = 0; k < AT_ONCE; k++)
#pragma unroll
      for (int i = 0; i < NV; i++) {
        const int at = min(h0 + 4 * k, d.heads - 1) * d.vdim + min(lane + 64 * i, d.vdim - 1);
        o[k][i] = b.o[(int64_t)row * vw + at]; z[k][i] = gate[at];
      }
#pragma unroll
    for (int i = 0; i < NV; i++) gain[i] = w.norm[min(lane + 64 * i, d.vdim - 1)];
#pragma unroll
    for (int k = 0; k < AT_ONCE; k++) {
      const int h = h0 + 4 * k;
      if (h >= d.heads) break;
      float s = 0.0f;
#pragma unroll
      for (int i = 0; i < NV; i++) if (lane + 64 * i < d.vdim) s = fmaf(o[k][i], o[k][i], s);
      const float inv = 1.0f / sqrtf(wave_total(s) / (float)d.vdim + d.eps);
#pragma unroll
      for (int i = 0; i < NV; i++) {
        const int c = lane + 64 * i;
        if (c >= d.vdim) continue;
        const float sg = sigmoid_f(z[k][i]);
        out[row * ldo + h * d.vdim + c] = (AT)(o[k][i] * inv * gain[i] * (d.sigmoid_gate ? sg : z[k][i] * sg));
      }
    }
  }
  if (r.last[row] - row < d.taps) {
    const int kw = d.kv_heads * d.dim, C = d.channels();
    float* ring = hist + r.slot[row] * h_elems + (int64_t)(r.pos[row] % d.taps) * C;
    for (int c = threadIdx.x; c < kw; c += 256) { ring[c] = p[in.oq + c]; ring[kw + c] = p[in.ok + c]; }
    for (int c = threadIdx.x; c < vw; c += 256) ring[2 * kw + c] = p[in.ov + c];
  }
}

// ------------------------------------------------------------------------------------------
// decode: one token of each entry, one work-group per (head, row): low-rank seconds, convolutions, unit norms, decay, the state
// update, output norm and gate.
// What bounds it: round trips (a state of 64 KB is 1 us of a CU).  Everything is requested before the first value is used, in the order of its use - what lies at
// known places, then what needs the row's slot and position, the state last - and without a condition that would make a wait count the state's
// requests too.  (Taps and low-rank rows requested as they came to their use: four rows of 16 heads 9.6 us, 8.2 so.)
// TAPS: of the convolutions (0: any number, requested one after another, and heads of more than 128 channels, whose four a lane take too many registers).
// ------------------------------------------------------------------------------------------
constexpr int SINGLE_LOW = 2, SINGLE_QUADS = 13 * 16;      // low-rank rows a quad has requested ahead; quads of waves 3 .. 15
template <typename AT, int RPT, int TAPS>
__global__ __launch_bounds__(1024) void delta_single_kernel(const DeltaDims d, const DeltaIn in, const DeltaW w, const uint16_t* a2, const int lda2, const uint16_t* g2, const int ldg2,
                                                            float* state, const int64_t s_elems, float* hist, const int64_t h_elems, const StepRows r, AT* out, const int64_t ldo, const int ct_log)
{
  __shared__ float sq[256], sk[256], sg[256], sv[256], sgate[256], so[256];
  __shared__ f32x4 su[32];
  __shared__ float sra[512], srg[512];
  __shared__ float red[2][16][128];
  __shared__ float sc[1];
  const int h = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pos = r.pos[row], slot = r.slot[row];
  const int hg = d.heads / d.kv_heads, g = h / hg, kw = d.kv_heads * d.dim, C = d.channels();
  // a thread holds four consecutive columns of RPT rows; CT threads a row, RG rows side by side
  const int CT = 1 << ct_log, CP = CT * 4, RG = 1024 >> ct_log, ct = tid & (CT - 1), rg = tid >> ct_log;
  const int dvp = d.vdim_p();
  float* Sg = state + slot * s_elems + (int64_t)h * d.dim * dvp;
  const float* p = in.proj + row * in.ldp;
  float* ring = hist + slot * h_elems;
  float* ring_now = ring + (int64_t)(pos % d.taps) * C;
  const float ra = tid < d.rank_a ? p[in.oa + tid] : 0.0f, rgv = tid < d.rank_g ? p[in.og + tid] : 0.0f;      // (ranks of at most 512)
  const float beta_z = p[in.ob + h];

  // q (wave 0), k (wave 1) and v (wave 2): channels lane + 64 i of the head; the other waves: low-rank rows of decay and gate, four lanes a row
  const int oc = wave == 0 ? in.oq : wave == 1 ? in.ok : in.ov, hc = wave == 0 ? 0 : wave == 1 ? kw : 2 * kw, n_ch = wave == 2 ? d.vdim : d.dim, c0h = wave == 2 ? h * d.vdim : g * d.dim;
  const float* const cw = wave == 0 ? w.cq : wave == 1 ? w.ck : w.cv;
  constexpr int T = TAPS ? TAPS : 2, NC = TAPS ? 2 : 4;
  float x[NC], taps[NC][T], past[NC][T - 1], gain[NC];
  const int nd = d.channel_decay ? d.dim : 1, quad = (tid - 192) >> 2, ql = tid & 3;
  const bool ahead = d.rank_a && d.rank_g && d.rank_a <= 128 && d.rank_g <= 128 && nd + d.vdim <= SINGLE_LOW * SINGLE_QUADS;
  u32x4 low_m[SINGLE_LOW][4]; float low_b[SINGLE_LOW];
  if (wave < 3) {
#pragma unroll
    for (int i = 0; i < NC; i++) {
      const int c = c0h + min(lane + 64 * i, n_ch - 1);
      x[i] = p[oc + c];
      if constexpr (TAPS != 0)
#pragma unroll
        for (int k = 0; k < T; k++) taps[i][k] = cw[c * T + k];
      gain[i] = w.norm[min(lane + 64 * i, d.vdim - 1)];
    }
  } else if (ahead) {
#pragma unroll
    for (int u = 0; u < SINGLE_LOW; u++) {
      const int i = min(quad + u * SINGLE_QUADS, nd + d.vdim - 1);
      const uint16_t* m = i < nd ? a2 + (int64_t)(h * nd + i) * lda2 : g2 + (int64_t)(h * d.vdim + i - nd) * ldg2;
      const int ld = i < nd ? lda2 : ldg2;
#pragma unroll
      for (int k = 0; k < 4; k++) low_m[u][k] = *reinterpret_cast<const u32x4*>(m + (ql * 8 + 32 * k < ld ? ql * 8 + 32 * k : 0));
      low_b[u] = w.dt_bias[h * nd + min(i, nd - 1)];
    }
  }
  const float rate = w.rate[h];
  asm volatile("" ::: "memory");
  if (TAPS != 0 && wave < 3)
#pragma unroll
    for (int i = 0; i < NC; i++)
#pragma unroll
      for (int j = 1; j < T; j++) past[i][j - 1] = ring[(int64_t)((pos + T - j) % T) * C + hc + c0h + min(lane + 64 * i, n_ch - 1)];
  asm volatile("" ::: "memory");
  f32x4 S[RPT];
  auto load_state = [&](int c0) {
#pragma unroll
    for (int j = 0; j < RPT; j++) S[j] = *reinterpret_cast<const f32x4*>(Sg + (unsigned)(min(rg + j * RG, d.dim - 1) * dvp + min(c0 + ct * 4, dvp - 4)));
  };
  auto keep_state = [&](int c0) {                        // what this thread holds of a state that there is
#pragma unroll
    for (int j = 0; j < RPT; j++)
      if (!(pos > 0 && rg + j * RG < d.dim && c0 + ct * 4 < dvp)) S[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  };
  load_state(0);
  asm volatile("" ::: "memory");
  if (tid < d.rank_a) sra[tid] = ra;
  if (tid < d.rank_g) srg[tid] = rgv;
  if (d.rank_a || d.rank_g) {                            // (waits for LDS only: the other requests stay on their way)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  if (wave < 3) {
    float v[NC], s = 0.0f;
#pragma unroll
    for (int i = 0; i < NC; i++) {
      const int c = lane + 64 * i;
      v[i] = 0.0f;
      if (c >= n_ch) continue;
      if constexpr (TAPS != 0) {
        float t = fmaf(taps[i][T - 1], x[i], 0.0f);
#pragma unroll
        for (int j = 1; j < T; j++) t = fmaf(taps[i][T - 1 - j], j <= pos ? past[i][j - 1] : 0.0f, t);
        v[i] = t * sigmoid_f(t);
      } else v[i] = conv_silu(p + oc, in.ldp, 0, pos, ring, C, hc, cw, d.taps, c0h + c);
      s = fmaf(v[i], v[i], s);
    }
    if (wave < 2) {                                      // unit norm
      const float nrm = (wave ? 1.0f : rsqrtf((float)d.dim)) / sqrtf(wave_total(s) + 1e-6f);
      float* dst = wave ? sk : sq;
#pragma unroll
      for (int i = 0; i < NC; i++) dst[lane + 64 * i] = v[i] * nrm;
    } else
#pragma unroll
      for (int i = 0; i < NC; i++) if (lane + 64 * i < n_ch) sv[lane + 64 * i] = v[i];
    if (wave == 2 || h % hg == 0)
#pragma unroll
      for (int i = 0; i < NC; i++) if (lane + 64 * i < n_ch) ring_now[hc + c0h + lane + 64 * i] = x[i];
  } else {                                               // decay and gate
    auto part = [&](float s, const u32x4 u, const float* v, int rank, int i) {      // (columns beyond the rank are zero in the matrix, the vector is guarded)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (i + 2 * j < rank) s = fmaf(bf16_lo(u[j]), v[i + 2 * j], s);
        if (i + 2 * j + 1 < rank) s = fmaf(bf16_hi(u[j]), v[i + 2 * j + 1], s);
      }
      return s;
    };
    auto quad_sum = [](float s) { s += __shfl_xor(s, 1); return s + __shfl_xor(s, 2); };
    auto low = [&](const uint16_t* m, int ld, const float* v, int rank, int rw) {
      float s = 0.0f;
      const uint16_t* mr = m + (int64_t)rw * ld;
      for (int i = ql * 8; i < rank; i += 32) s = part(s, *reinterpret_cast<const u32x4*>(mr + i), v, rank, i);
      return quad_sum(s);
    };
    auto put = [&](int i, float z) {
      if (ql != 0) return;
      if (i < nd) sg[i] = expf(rate * softplus_f(z));
      else { const float s = sigmoid_f(z); sgate[i - nd] = d.sigmoid_gate ? s : z * s; }
    };
    if (ahead) {
#pragma unroll
      for (int u = 0; u < SINGLE_LOW; u++) {
        const int i = quad + u * SINGLE_QUADS;
        if (i >= nd + d.vdim) break;                     // (whole quads)
        const bool decay = i < nd;
        const float* v = decay ? sra : srg;
        const int rank = decay ? d.rank_a : d.rank_g;
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; k++) s = part(s, low_m[u][k], v, rank, ql * 8 + 32 * k);
        s = quad_sum(s);
        put(i, decay ? s + low_b[u] : s);
      }
    } else
      for (int i = quad; i < nd + d.vdim; i += SINGLE_QUADS) {
        if (i < nd) {
          const int c = h * nd + i;
          put(i, (d.rank_a ? low(a2, lda2, sra, d.rank_a, c) : p[in.oa + c]) + w.dt_bias[c]);
        } else {
          const int c = h * d.vdim + i - nd;
          put(i, d.rank_g ? low(g2, ldg2, srg, d.rank_g, c) : p[in.og + c]);
        }
      }
  }
  __syncthreads();
  if (wave == 0) {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < NC; i++) s = fmaf(sq[lane + 64 * i], sk[lane + 64 * i], s);
    s = wave_total(s);
    if (lane == 0) sc[0] = s;
  }
  const float beta = sigmoid_f(beta_z);
  for (int c0 = 0; c0 < d.vdim; c0 += CP) {
    if (c0) load_state(c0);
    keep_state(c0);
    f32x4 ks = {0.0f, 0.0f, 0.0f, 0.0f}, qd = ks;
#pragma unroll
    for (int j = 0; j < RPT; j++) {
      const int rr = rg + j * RG;
      if (rr >= d.dim) continue;
      const float gr = sg[d.channel_decay ? rr : 0], kr = sk[rr], qr = sq[rr];
#pragma unroll
      for (int i = 0; i < 4; i++) { S[j][i] *= gr; ks[i] = fmaf(S[j][i], kr, ks[i]); qd[i] = fmaf(S[j][i], qr, qd[i]); }
    }
    for (int m = CT; m < 64; m <<= 1) {
#pragma unroll
      for (int i = 0; i < 4; i++) { ks[i] += __shfl_xor(ks[i], m); qd[i] += __shfl_xor(qd[i], m); }
    }
    if (lane < CT) { *reinterpret_cast<f32x4*>(&red[0][wave][ct * 4]) = ks; *reinterpret_cast<f32x4*>(&red[1][wave][ct * 4]) = qd; }
    __syncthreads();
    if (tid < 2 * CP) {
      const int which = tid >= CP, c = which ? tid - CP : tid;
      float a = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; i++) a += red[which][i][c];
      if (which) { if (c0 + c < d.vdim) so[c0 + c] = a; }
      else reinterpret_cast<float*>(su)[c] = c0 + c < d.vdim ? beta * (sv[c0 + c] - a) : 0.0f;
    }
    __syncthreads();
    const f32x4 u = su[ct];
    if (tid < CP && c0 + tid < d.vdim) so[c0 + tid] = fmaf(sc[0], reinterpret_cast<float*>(su)[tid], so[c0 + tid]);
#pragma unroll
    for (int j = 0; j < RPT; j++) {
      const int rr = rg + j * RG;
      if (rr >= d.dim || c0 + ct * 4 >= dvp) continue;
      const float kr = sk[rr];
#pragma unroll
      for (int i = 0; i < 4; i++) S[j][i] = fmaf(kr, u[i], S[j][i]);
      *reinterpret_cast<f32x4*>(Sg + (unsigned)(rr * dvp + c0 + ct * 4)) = S[j];
    }
  }
  __syncthreads();
  if (wave == 0) {
    float o[NC], s = 0.0f;
#pragma unroll
    for (int i = 0; i < NC; i++) { const int c = lane + 64 * i; o[i] = c < d.vdim ? so[c] : 0.0f; s = fmaf(o[i], o[i], s); }
    const float inv = 1.0f / sqrtf(wave_total(s) / (float)d.vdim + d.eps);
#pragma unroll
    for (int i = 0; i < NC; i++) {
      const int c = lane + 64 * i;
      if (c < d.vdim) out[row * ldo + h * d.vdim + c] = (AT)(o[i] * inv * gain[i] * sgate[c]);
    }
  }
}

int delta_prep(const DeltaDims& d, const DeltaIn& in, const DeltaW& w, const SeqPool::StateRun& st, const StepRows& r, const DeltaBuf& b)
{
  const int gw = d.channel_decay ? d.heads * d.dim : d.heads;
  const int units = d.kv_heads + (d.heads * d.vdim + 255) / 256 + (gw + 255) / 256 + 1;
  const dim3 grid((r.n_rows + PREP_ROWS - 1) / PREP_ROWS, (units + 3) / 4);
#define PREP(TAPS, ND) hipLaunchKernelGGL((delta_prep_kernel<TAPS, ND>), grid, dim3(256), 0, ctx().stream, d, in, w, st.hist, st.h_elems, r, b)
#define PREP_N(TAPS) do { if (d.dim <= 64) PREP(TAPS, 1); else if (d.dim <= 128) PREP(TAPS, 2); else PREP(TAPS, 4); } while (0)
  if (d.taps == 4) PREP_N(4); else PREP_N(0);
#undef PREP_N
#undef PREP
  CAI_HIP(hipGetLastError());
  return CAI_OK;
}

int delta_scan(const DeltaDims& d, const SeqPool::StateRun& st, const StepRows& r, const DeltaBuf& b)
{
  const dim3 grid((d.vdim + 15) / 16, d.heads, r.n_ent), blk(256);
  auto s = ctx().stream;
#define SCAN(RPL) do { if (d.channel_decay) hipLaunchKernelGGL((delta_scan_kernel<RPL, true>), grid, blk, 0, s, d, st.S, st.s_elems, r, b); \
                       else hipLaunchKernelGGL((delta_scan_kernel<RPL, false>), grid, blk, 0, s, d, st.S, st.s_elems, r, b); } while (0)
  if (d.dim <= 64) SCAN(4); else if (d.dim <= 128) SCAN(8); else SCAN(16);
#undef SCAN
  CAI_HIP(hipGetLastError());
  return CAI_OK;
}

static int delta_pass(const DeltaDims& d, const SeqPool::StateRun& st, const StepRows& r, const DeltaBuf& b, const DeltaPass& p, int n_chunks)
{
  auto s = ctx().stream;
  const size_t lds = (size_t)(d.channel_decay ? 3 : 2) * CHUNK * (((d.dim + 15) & ~15) + 4) * 4;
  const dim3 g1(n_chunks, d.heads), g2((d.vdim + 15) / 16 * d.heads, r.n_ent), blk(256);
  if (d.channel_decay) hipLaunchKernelGGL(delta_chunk_kernel<true>, g1, blk, lds, s, d, r, b, p);
  else hipLaunchKernelGGL(delta_chunk_kernel<false>, g1, blk, lds, s, d, r, b, p);
#define WALK_C(NW, N, CH) do { if (d.vdim % 16 == 0) hipLaunchKernelGGL((delta_walk_kernel<NW, N, CH, true>), g2, dim3(64 * (NW + 1)), 0, s, d, st.S, st.s_elems, r, b, p); \
                               else hipLaunchKernelGGL((delta_walk_kernel<NW, N, CH, false>), g2, dim3(64 * (NW + 1)), 0, s, d, st.S, st.s_elems, r, b, p); } while (0)
#define WALK(NW, N) do { if (d.channel_decay) WALK_C(NW, N, true); else WALK_C(NW, N, false); } while (0)
  switch (delta_tiles(d)) { case 4: WALK(4, 1); break; case 8: WALK(4, 2); break; default: WALK(8, 2); break; }
#undef WALK_C
#undef WALK
  CAI_HIP(hipGetLastError());
  return CAI_OK;
}

int delta_chunked(const DeltaDims& d, const SeqPool::StateRun& st, const StepRows& r, const DeltaBuf& b, const int32_t* chunks, int n_chunks, const int32_t* chunk0, int longest)
{
  const int64_t room = b.rec_floats / ((int64_t)d.heads * delta_record_blocks(d) * 256);      // chunks whose records b.rec holds: one of every entry at least
  if (n_chunks <= room) return delta_pass(d, st, r, b, DeltaPass{chunks, chunk0, 0, n_chunks}, n_chunks);
  if (room < r.n_ent) return set_error(CAI_ERR_STATE, "delta rule: records of %lld chunks for %d sequences", (long long)room, r.n_ent);
  // passes over time, all entries together: they walk side by side as in one pass
  const int most = (int)(room / r.n_ent);
  for (int first = 0; first < longest; first += most) {
    const int rc = delta_pass(d, st, r, b, DeltaPass{nullptr, nullptr, first, most}, r.n_ent * most);
    if (rc) return rc;
  }
  return CAI_OK;
}

int delta_finish(const DeltaDims& d, const DeltaIn& in, const DeltaW& w, const SeqPool::StateRun& st, const StepRows& r, const DeltaBuf& b, int act_t, void* out, int64_t ldo)
{
#define FINISH(AT, NV) hipLaunchKernelGGL((delta_finish_kernel<AT, NV>), dim3(r.n_rows), dim3(256), 0, ctx().stream, d, in, w, st.hist, st.h_elems, r, b, (AT*)out, ldo)
#define FINISH_N(AT) do { if (d.vdim <= 64) FINISH(AT, 1); else if (d.vdim <= 128) FINISH(AT, 2); else FINISH(AT, 4); } while (0)
  if (act_t == ACT_T_BF16) FINISH_N(bf16_t); else FINISH_N(float);
#undef FINISH_N
#undef FINISH
  CAI_HIP(hipGetLastError());
  return CAI_OK;
}

int delta_single(const DeltaDims& d, const DeltaIn& in, const DeltaW& w, const SeqPool::StateRun& st, const StepRows& r, int act_t, void* out, int64_t ldo)
{
  const int ct_log = d.vdim > 64 ? 5 : d.vdim > 32 ? 4 : 3, rgs = 1024 >> ct_log, rpt = (d.dim + rgs - 1) / rgs;
  const dim3 grid(d.heads, r.n_rows), blk(1024);
  const uint16_t* a2 = w.a2 ? (const uint16_t*)w.a2->data : nullptr; const uint16_t* g2 = w.g2 ? (const uint16_t*)w.g2->data : nullptr;
  const int la = w.a2 ? (int)w.a2->ld : 0, lg = w.g2 ? (int)w.g2->ld : 0;
  auto s = ctx().stream;
#define SINGLE(AT, N, TAPS) hipLaunchKernelGGL((delta_single_kernel<AT, N, TAPS>), grid, blk, 0, s, d, in, w, a2, la, g2, lg, st.S, st.s_elems, st.hist, st.h_elems, r, (AT*)out, ldo, ct_log)
  const bool ahead = d.taps == 4 && d.dim <= 128 && d.vdim <= 128;      // (four rows of the state a thread at most then)
#define SINGLE_N(AT) do { if (ahead && rpt <= 2) SINGLE(AT, 2, 4); else if (ahead) SINGLE(AT, 4, 4); else if (rpt <= 2) SINGLE(AT, 2, 0); else if (rpt <= 4) SINGLE(AT, 4, 0); else SINGLE(AT, 8, 0); } while (0)
  if (act_t == ACT_T_BF16) SINGLE_N(bf16_t); else SINGLE_N(float);
#undef SINGLE_N
#undef SINGLE
  CAI_HIP(hipGetLastError());
  return CAI_OK;
}

}  // namespace cai
