// Distribution pipeline ahead of the samplers, on the device, so that a sampled (non-greedy) decode does not read
// the vocabulary-sized logits row back (TChatEngine.GenerateFromIds, neural/neuralchatengine.pas:1374-1396, 1495-1501):
//   softmax -> history penalty in the probability domain (neural/neuralvolume.pas:5335-5376)
//           -> temperature in the probability domain (neural/neuraldecode.pas:4710-4754)
//           -> the m most probable tokens in descending order: the prefix every sampler of the reference draws from
//              (TNNetSamplerBase.SelectTopCandidates / SortTokenArray, neural/neuralvolume.pas:5171-5196; the nucleus
//              sampler starts from a 256-wide prefix itself, 4548-4562).
// The draw stays with the host and its own random generator: it gets m (token, probability) pairs instead of the row.
//
// The row is cut into at most 256 slices, one work-group each, and every stage that needs a number of the whole row is a launch
// boundary: slice maxima and sums -> [penalised probabilities] -> last values and a histogram of their leading 12 bits -> the few
// values at or above the bin that holds the m-th largest -> their ranking, by one work-group up to 32 candidates and sixteen for more.
// What bounds it is launches (five, four without a penalty), not bytes: a 152k row with penalties, temperature and 40 candidates takes 44 us a call, 284 as
// one work-group that walked the row ten times out of L2 at the 40 GB/s one compute unit gets.
#include "cai_internal.hpp"
#include <algorithm>
#include <string.h>

namespace cai {

constexpr int SMP_T = 1024;       // threads of the ranking work-group
constexpr int SMP_MAX_M = 1024;
constexpr int SL_T = 256;         // threads of a slice's work-group
constexpr int SL_MAX = 256;       // slices: a thread of a work-group folds one slice's number
constexpr int SMP_BINS = 4096;
constexpr int RANK_MAX = 2048;    // values ranked by comparison with each other; more go through a radix select first
constexpr int RANK_WG = 16;       // work-groups that share the ranking

template <int NT>
__device__ __forceinline__ float smp_max(float v, float* red)
{
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = red[0];
#pragma unroll
  for (int w = 1; w < NT / 64; w++) r = fmaxf(r, red[w]);
  return r;
}

template <int NT>
__device__ __forceinline__ float smp_sum(float v, float* red)
{
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = 0.0f;
#pragma unroll
  for (int w = 0; w < NT / 64; w++) r += red[w];
  return r;
}

// exclusive prefix sum over the work-group in thread order; *total gets the sum
template <int NT>
__device__ __forceinline__ int smp_excl_scan(int v, int* red, int* total)
{
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int inc = v;
  for (int o = 1; o < 64; o <<= 1) { const int t = __shfl_up(inc, o, 64); if (lane >= o) inc += t; }
  __syncthreads();
  if (lane == 63) red[w] = inc;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int i = 0; i < NT / 64; i++) { const int t = red[i]; if (i < w) before += t; all += t; }
  *total = all;
  return before + inc - v;
}

// the bin (0 .. 4095) in which the `need`-th largest value lies, top bins first, and how many of its values are needed; every thread
// gets both
template <int NT>
__device__ __forceinline__ void smp_crossing(const int* hist, int need, int* redi, int* sel)
{
  constexpr int PER = SMP_BINS / NT;
  const int b0 = SMP_BINS - 1 - PER * (int)threadIdx.x;
  int own[PER], sum = 0, total;
#pragma unroll
  for (int k = 0; k < PER; k++) { own[k] = hist[b0 - k]; sum += own[k]; }
  int acc = smp_excl_scan<NT>(sum, redi, &total);
  if (acc < need && need <= acc + sum) {        // exactly one thread: the crossing lies in its bins
#pragma unroll
    for (int k = 0; k < PER; k++) {
      if (acc < need && need <= acc + own[k]) { sel[0] = b0 - k; sel[1] = need - acc; }
      acc += own[k];
    }
  }
  __syncthreads();
}

struct SampleParams {
  const float* logits; int n;
  const int32_t* hist_ids; const int32_t* hist_counts; int n_hist;
  float repetition, frequency, presence, temperature;
  int m;
  int slice, n_slices;               // values of a slice (a multiple of 256); slices
  int penalty;                       // some token of the history lies in the row and a penalty is set
  float* val;                        // [n] probabilities on the way
  float* cand_v; int32_t* cand_t;    // [n_slices][slice] the slice's values in reach of the m largest, in token order
  int* bins;                         // [4096] values per leading 12 bits
  float *st_max, *st_sum, *st_tot, *st_pmax, *st_sum2; int* st_cnt;   // [256] per slice
  int32_t* tok_out; float* p_out;    // host memory
};

// the same clamps as the host row soft-max (a NaN counts as far below the maximum)
__device__ __forceinline__ float smp_exp(float v, float mx) { return expf(fminf(fmaxf(v - mx, -4000.0f), 4000.0f)); }

// maximum of the row and 1 / sum of its exponentials (0 where the sum is: the row then stays as the exponentials are)
__device__ __forceinline__ void smp_row_stats(const SampleParams& p, float* red, float& mx, float& inv)
{
  const int g = threadIdx.x;
  const float own = g < p.n_slices ? p.st_max[g] : -3.0e38f, s = g < p.n_slices ? p.st_sum[g] : 0.0f;
  mx = smp_max<SL_T>(own, red);
  const float sum = smp_sum<SL_T>(s * smp_exp(own, mx), red);
  inv = sum > 0.0f ? 1.0f / sum : 0.0f;
}

__global__ __launch_bounds__(SL_T) void candidates_stats_kernel(const SampleParams p)
{
  __shared__ float red[SL_T / 64];
  const int i0 = blockIdx.x * p.slice, len = min(p.slice, p.n - i0);
  for (int b = blockIdx.x * SL_T + threadIdx.x; b < SMP_BINS; b += p.n_slices * SL_T) p.bins[b] = 0;
  float mx = -3.0e38f;
  for_strided8(p.logits + i0, threadIdx.x, len, SL_T, [&](float v, int) { mx = fmaxf(mx, v); });
  mx = smp_max<SL_T>(mx, red);
  float sum = 0.0f;
  for_strided8(p.logits + i0, threadIdx.x, len, SL_T, [&](float v, int) { sum += smp_exp(v, mx); });
  sum = smp_sum<SL_T>(sum, red);
  if (threadIdx.x == 0) { p.st_max[blockIdx.x] = mx; p.st_sum[blockIdx.x] = sum; }
}

// probabilities with the history penalty: p^r, * exp(-(f * count + presence)) on the distinct context tokens
__global__ __launch_bounds__(SL_T) void candidates_penalty_kernel(const SampleParams p)
{
  __shared__ float red[SL_T / 64];
  const int i0 = blockIdx.x * p.slice, len = min(p.slice, p.n - i0);
  float mx, inv;
  smp_row_stats(p, red, mx, inv);
  float* val = p.val + i0;
  for_strided8(p.logits + i0, threadIdx.x, len, SL_T, [&](float v, int i) { const float e = smp_exp(v, mx); val[i] = inv > 0.0f ? e * inv : e; });
  __syncthreads();
  for (int k = threadIdx.x; k < p.n_hist; k += SL_T) {
    const int t = p.hist_ids[k] - i0;
    if (t < 0 || t >= len) continue;
    float v = val[t];
    if (p.repetition != 1.0f && v > 0.0f) v = powf(v, p.repetition);
    if (p.frequency != 0.0f || p.presence != 0.0f) v *= expf(-(p.frequency * (float)p.hist_counts[k] + p.presence));
    val[t] = v;
  }
  __syncthreads();
  float tot = 0.0f, top = 0.0f;
  for_strided8(val, threadIdx.x, len, SL_T, [&](float v, int) { tot += v; top = fmaxf(top, v); });
  tot = smp_sum<SL_T>(tot, red);
  top = smp_max<SL_T>(top, red);
  if (threadIdx.x == 0) { p.st_tot[blockIdx.x] = tot; p.st_pmax[blockIdx.x] = top; }
}

// last values: the probabilities, or with a temperature exp(ln(max(p, 1e-30)) / T - ln(max p) / T) still to be divided by its sum
__global__ __launch_bounds__(SL_T) void candidates_value_kernel(const SampleParams p)
{
  __shared__ float red[SL_T / 64];
  __shared__ int bins[SMP_BINS];
  const int i0 = blockIdx.x * p.slice, len = min(p.slice, p.n - i0), g = threadIdx.x;
  for (int b = g; b < SMP_BINS; b += SL_T) bins[b] = 0;
  float mx = 0.0f, inv = 0.0f, tot = 0.0f, pm;
  if (p.penalty) {
    tot = smp_sum<SL_T>(g < p.n_slices ? p.st_tot[g] : 0.0f, red);
    pm = smp_max<SL_T>(g < p.n_slices ? p.st_pmax[g] : 0.0f, red);
    if (tot > 0.0f) pm = pm / tot;
  } else {
    smp_row_stats(p, red, mx, inv);
    pm = inv;                                   // the maximum's exponential is 1
  }
  const bool warm = p.temperature != 1.0f && pm > 0.0f;
  const float lm = logf(fmaxf(pm, 1e-30f)), inv_t = 1.0f / fmaxf(p.temperature, 1e-6f);
  __syncthreads();
  float sum2 = 0.0f;
  const float* src = p.penalty ? p.val + i0 : p.logits + i0;
  for_strided8(src, g, len, SL_T, [&](float v, int i) {
    if (p.penalty) { if (tot > 0.0f) v = v / tot; }
    else { v = smp_exp(v, mx); if (inv > 0.0f) v *= inv; }
    if (warm) { v = expf(logf(fmaxf(v, 1e-30f)) * inv_t - lm * inv_t); sum2 += v; }
    p.val[i0 + i] = v;
    atomicAdd(&bins[__float_as_uint(v) >> 20], 1);
  });
  sum2 = smp_sum<SL_T>(sum2, red);
  if (g == 0) p.st_sum2[blockIdx.x] = warm ? sum2 : -1.0f;      // (< 0: nothing to divide by)
  __syncthreads();
  for (int b = g; b < SMP_BINS; b += SL_T) { const int c = bins[b]; if (c) atomicAdd(&p.bins[b], c); }
}

// the slice's values that can be among the m largest, in token order
__global__ __launch_bounds__(SL_T) void candidates_reach_kernel(const SampleParams p)
{
  __shared__ float red[SL_T / 64];
  __shared__ int redi[SL_T / 64];
  __shared__ int sel[2];
  const int i0 = blockIdx.x * p.slice, g = threadIdx.x, per = p.slice / SL_T;
  const float s2 = g < p.n_slices ? p.st_sum2[g] : 0.0f;
  const bool warm = !(p.st_sum2[0] < 0.0f);
  float inv = smp_sum<SL_T>(s2, red);
  inv = warm ? 1.0f / (inv <= 0.0f ? 1.0f : inv) : 1.0f;
  smp_crossing<SL_T>(p.bins, min(p.m, p.n), redi, sel);
  // A division by the sum keeps the order but can make neighbours equal, and equal ones go by token: a quotient rounds two steps of its
  // dividend together at most, and with the rounding of the reciprocal values up to four steps below the bin are still in reach.  Where the quotients lose bits to the end of the number range everything is.
  uint32_t floor_bits = (uint32_t)sel[0] << 20;
  floor_bits = warm && __uint_as_float(floor_bits) * inv < 1.0e-36f ? 0u : floor_bits < 4u ? 0u : floor_bits - 4u;
  int mine = 0, total;
  const int j0 = g * per;
  for (int k = 0; k < per; k++) mine += i0 + j0 + k < p.n && __float_as_uint(p.val[i0 + j0 + k]) >= floor_bits;
  int at = smp_excl_scan<SL_T>(mine, redi, &total);
  for (int k = 0; mine > 0 && k < per; k++) {
    const int i = i0 + j0 + k;
    if (i >= p.n) break;
    const float v = p.val[i];
    if (__float_as_uint(v) >= floor_bits) { p.cand_v[i0 + at] = v * inv; p.cand_t[i0 + at] = i; at++; }
  }
  if (g == 0) p.st_cnt[blockIdx.x] = total;
}

// descending probability, equal ones by token.  Every work-group gathers the whole list (a few thousand values from the L2) and ranks its
// share of it: the comparisons, not the gathering, were the time of one work-group (of 152064 logits,
// a whole call: 1000 candidates 185 -> 59 us, 256 65 -> 48, 40 46.8 -> 44.2; up to about 32 there is little to compare, and one is enough: 5 42.4, 42.3).
__global__ __launch_bounds__(SMP_T) void candidates_rank_kernel(const SampleParams p)
{
  __shared__ int redi[SMP_T / 64];
  __shared__ int hist[SMP_BINS];
  __shared__ int cnt[SL_MAX], start[SL_MAX];
  __shared__ int sel[2];
  __shared__ int n_gt;
  __shared__ float cp[RANK_MAX];
  __shared__ int32_t ct[RANK_MAX];
  __shared__ uint16_t mine[RANK_MAX];
  __shared__ int n_own;
  const int tid = threadIdx.x, m = min(p.m, p.n);
  const int own = tid < p.n_slices ? p.st_cnt[tid] : 0;
  int total;
  const int before = smp_excl_scan<SMP_T>(own, redi, &total);
  if (tid < SL_MAX) { cnt[tid] = own; start[tid] = before; }
  if (tid == 0) n_gt = 0;
  __syncthreads();
  if (total <= RANK_MAX) {
    for (int s = tid >> 6; s < p.n_slices; s += SMP_T / 64)      // a wave per slice
      for (int j = tid & 63; j < cnt[s]; j += 64) { cp[start[s] + j] = p.cand_v[s * p.slice + j]; ct[start[s] + j] = p.cand_t[s * p.slice + j]; }
  } else {
    // many equal or nearly equal values: the m-th largest exactly, 12 + 12 + 8 bits at a time
    const int slots = p.n_slices * p.slice;
    uint32_t prefix = 0, mask = 0;
    int need = m;                                // still to be taken at or below the current prefix
    const int shifts[3] = {20, 8, 0};
    const uint32_t widths[3] = {0xFFFu, 0xFFFu, 0xFFu};
    for (int lvl = 0; lvl < 3; lvl++) {
      for (int b = tid; b < SMP_BINS; b += SMP_T) hist[b] = 0;
      __syncthreads();
      for_strided8(p.cand_v, tid, slots, SMP_T, [&](float v, int i) {
        const uint32_t u = __float_as_uint(v);
        const int s = i / p.slice;
        if (i - s * p.slice < cnt[s] && (u & mask) == prefix) atomicAdd(&hist[(u >> shifts[lvl]) & widths[lvl]], 1);
      });
      __syncthreads();
      smp_crossing<SMP_T>(hist, need, redi, sel);
      prefix |= (uint32_t)sel[0] << shifts[lvl]; mask |= widths[lvl] << shifts[lvl];
      need = sel[1];
      __syncthreads();
    }
    // everything above it (any order), then `need` of its copies in token order
    for_strided8(p.cand_v, tid, slots, SMP_T, [&](float v, int i) {
      const int s = i / p.slice;
      if (i - s * p.slice < cnt[s] && __float_as_uint(v) > prefix) { const int k = atomicAdd(&n_gt, 1); cp[k] = v; ct[k] = p.cand_t[i]; }
    });
    __syncthreads();
    const int base = n_gt;                       // = m - need
    const int chunk = (slots + SMP_T - 1) / SMP_T, c0 = tid * chunk, c1 = min(slots, c0 + chunk);
    int ties = 0;
    for (int i = c0; i < c1; i++) { const int s = i / p.slice; ties += i - s * p.slice < cnt[s] && __float_as_uint(p.cand_v[i]) == prefix; }
    int all, rank = smp_excl_scan<SMP_T>(ties, redi, &all);
    for (int i = c0; ties > 0 && rank < need && i < c1; i++) {
      const int s = i / p.slice;
      if (i - s * p.slice < cnt[s] && __float_as_uint(p.cand_v[i]) == prefix) { cp[base + rank] = p.cand_v[i]; ct[base + rank] = p.cand_t[i]; rank++; }
    }
    total = m;
  }
  __syncthreads();
  // This work-group's share: the tokens of one residue (the order of the list is not the same in every work-group).  Eight neighbouring
  // lanes rank a value together.
  if (tid == 0) n_own = 0;
  __syncthreads();
  for (int e = tid; e < total; e += SMP_T) if ((unsigned)ct[e] % gridDim.x == blockIdx.x) mine[atomicAdd(&n_own, 1)] = (uint16_t)e;
  __syncthreads();
  for (int o = tid >> 3; o < n_own; o += SMP_T / 8) {
    const int e = mine[o], t = ct[e];
    const float v = cp[e];
    const uint32_t u = __float_as_uint(v);       // (values are not negative, so their bits order like they do; a NaN is the largest and has a rank like any other)
    int rank = 0;
    for (int j = tid & 7; j < total; j += 8) { const uint32_t w = __float_as_uint(cp[j]); rank += w > u || (w == u && ct[j] < t); }
    rank += __shfl_xor(rank, 1); rank += __shfl_xor(rank, 2); rank += __shfl_xor(rank, 4);
    if ((tid & 7) == 0 && rank < m) { p.tok_out[rank] = t; p.p_out[rank] = v; }
  }
}

// host arrays in, host arrays out; the row itself is a device pointer
int run_candidates(const float* logits_dev, int n, const int32_t* hist_ids, const int32_t* hist_counts, int n_hist,
                   float repetition, float frequency, float presence, float temperature, int m,
                   int32_t* tokens_out, float* probs_out, int* count_out)
{
  Context& c = ctx();
  if (n < 1 || m < 1 || m > SMP_MAX_M) return set_error(CAI_ERR_INVALID, "candidates: %d tokens wanted from a row of %d (1..%d)", m, n, SMP_MAX_M);
  if (n_hist < 0 || (n_hist > 0 && (!hist_ids || !hist_counts))) return set_error(CAI_ERR_INVALID, "candidates: history of %d tokens without its arrays", n_hist);
  if (m > n) m = n;
  SampleParams p{};
  p.logits = logits_dev; p.n = n; p.repetition = repetition; p.frequency = frequency; p.presence = presence; p.temperature = temperature; p.m = m;
  if (repetition != 1.0f || frequency != 0.0f || presence != 0.0f)
    for (int k = 0; k < n_hist && !p.penalty; k++) p.penalty = hist_ids[k] >= 0 && hist_ids[k] < n;
  // four values per thread of a slice (149 work-groups for a 152k row) until there are 256 slices
  p.slice = std::max(4 * SL_T, ((n + SL_MAX - 1) / SL_MAX + SL_T - 1) / SL_T * SL_T);
  p.n_slices = (n + p.slice - 1) / p.slice;
  const size_t slots = (size_t)p.n_slices * p.slice;
  int rc = ensure_stage(&c.stage_out, &c.stage_out_cap, (3 * slots + SMP_BINS + 6 * SL_MAX) * 4); if (rc) return rc;
  p.val = (float*)c.stage_out; p.cand_v = p.val + slots; p.cand_t = (int32_t*)(p.cand_v + slots);
  p.bins = (int*)(p.cand_t + slots);
  p.st_max = (float*)(p.bins + SMP_BINS); p.st_sum = p.st_max + SL_MAX; p.st_tot = p.st_sum + SL_MAX; p.st_pmax = p.st_tot + SL_MAX;
  p.st_sum2 = p.st_pmax + SL_MAX; p.st_cnt = (int*)(p.st_sum2 + SL_MAX);
  // host side: [tokens 1024 | probabilities 1024 | history ids | history counts]; the last launch writes the first two where they lie
  const size_t hist = p.penalty ? (size_t)n_hist : 0;
  if ((rc = ensure_host_stage((2 * (size_t)SMP_MAX_M + 2 * hist) * 4))) return rc;
  int32_t* h = (int32_t*)c.h_stage;
  p.tok_out = h; p.p_out = (float*)(h + SMP_MAX_M);
  if (p.penalty) {
    if ((rc = ensure_stage(&c.stage_in, &c.stage_in_cap, 2 * hist * 4))) return rc;
    memcpy(h + 2 * SMP_MAX_M, hist_ids, hist * 4); memcpy(h + 2 * SMP_MAX_M + hist, hist_counts, hist * 4);
    CAI_HIP(hipMemcpyAsync(c.stage_in, h + 2 * SMP_MAX_M, 2 * hist * 4, hipMemcpyHostToDevice, c.stream));
    p.hist_ids = (const int32_t*)c.stage_in; p.hist_counts = p.hist_ids + hist; p.n_hist = n_hist;
  }
  const dim3 grid(p.n_slices), block(SL_T);
  hipLaunchKernelGGL(candidates_stats_kernel, grid, block, 0, c.stream, p);
  if (p.penalty) hipLaunchKernelGGL(candidates_penalty_kernel, grid, block, 0, c.stream, p);
  hipLaunchKernelGGL(candidates_value_kernel, grid, block, 0, c.stream, p);
  hipLaunchKernelGGL(candidates_reach_kernel, grid, block, 0, c.stream, p);
  hipLaunchKernelGGL(candidates_rank_kernel, dim3(m > 32 ? RANK_WG : 1), dim3(SMP_T), 0, c.stream, p);
  CAI_HIP(hipGetLastError());
  CAI_HIP(hipStreamSynchronize(c.stream));
  memcpy(tokens_out, h, (size_t)m * 4);
  memcpy(probs_out, h + SMP_MAX_M, (size_t)m * 4);
  if (count_out) *count_out = m;
  return CAI_OK;
}

}  // namespace cai

using namespace cai;

extern "C" int cai_sample_candidates(const float* logits, int n, const int32_t* hist_ids, const int32_t* hist_counts, int n_hist,
                                     float repetition, float frequency, float presence, float temperature, int m,
                                     int32_t* tokens_out, float* probs_out, int* count_out, int flags)
{
  CAI_ENTER();
  CAI_READY();
  CAI_REQUIRE(logits && tokens_out && probs_out, "cai_sample_candidates: null argument");
  CAI_REQUIRE(n >= 1 && m >= 1 && m <= SMP_MAX_M, "cai_sample_candidates: %d candidates from a row of %d (1..%d)", m, n, SMP_MAX_M);
  Context& c = ctx();
  const float* row = logits;
  if (!(flags & CAI_X_DEVICE)) {
    // the row travels into a private device buffer behind the scratch areas run_candidates lays out
    int rc = ensure_stage(&c.stage_sample, &c.stage_sample_cap, (size_t)n * 4); if (rc) return rc;
    CAI_HIP(hipMemcpyAsync(c.stage_sample, logits, (size_t)n * 4, hipMemcpyHostToDevice, c.stream));
    row = (const float*)c.stage_sample;
  }
  return run_candidates(row, n, hist_ids, hist_counts, n_hist, repetition, frequency, presence, temperature, m, tokens_out, probs_out, count_out);
}
