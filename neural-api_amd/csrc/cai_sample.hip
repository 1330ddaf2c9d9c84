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
// boundary: slice maxima and sums (and the history, out of pinned memory) -> penalised probabilities and the largest of each group of 4 to 64 -> last values, and
// the few whose probability is at or above the bin that holds the m-th largest of those maxima -> their ranking, by the third launch's last work-group up to
// 128 candidates and by a launch of sixteen for more.
// What bounds it is launches and round trips, not bytes.  us a call, five launches and a copy with a histogram of the last values, waiting for the end of the stream | this: 40 of 152064
// behind a history of 512, penalties and temperature 44.4 | 29.9; without penalties 36.1 | 27.7; 5 of 152064 42.1 | 27.8; 300 of 50000 behind 3000 54.0 | 37; 905 of 152064 57.6 | 41.
#include "cai_router.hpp"
#include <algorithm>
#include <string.h>

namespace cai {

constexpr int SMP_T = 1024;       // threads of the ranking work-group
constexpr int SMP_MAX_M = 1024;
constexpr int SL_T = 256;         // threads of a slice's work-group
constexpr int SL_MAX = 256;       // slices: a thread of a work-group folds one slice's number
constexpr int SMP_BINS = 4096;
constexpr int TOP_MAX = 8192;     // maxima of groups
constexpr int RANK_MAX = 2048;    // values ranked by comparison with each other; more go through a radix select first
constexpr int SMP_FOLD_M = 128;   // candidates that the third launch ranks itself: 32.5 us a call for 128; a launch of sixteen work-groups 35.4 for 200, 36.7 for 500
constexpr int RANK_WG = 16;       // work-groups that share the ranking

template <int NT>
__device__ __forceinline__ float smp_max(float v, float* red)
{
  v = wave_max(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = red[0];
#pragma unroll
  for (int w = 1; w < NT / 64; w++) r = fmaxf(r, red[w]);
  return r;
}

template <int NT>
__device__ __forceinline__ float smp_sum(float v, float* red)
{
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = v;
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
  int inc = v;                                   // (wave_sum's steps leave every lane the sum up to itself)
#define STEP(ctrl, rows) inc += __builtin_amdgcn_update_dpp(0, inc, ctrl, rows, 0xf, true);
  STEP(0x111, 0xf) STEP(0x112, 0xf) STEP(0x114, 0xf) STEP(0x118, 0xf) STEP(0x142, 0xa) STEP(0x143, 0xc)
#undef STEP
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
  for (int k = 0; k < PER; k += 4) {
    const int4 t = *reinterpret_cast<const int4*>(hist + b0 - k - 3);
    own[k] = t.w; own[k + 1] = t.z; own[k + 2] = t.y; own[k + 3] = t.x;
    sum += t.x + t.y + t.z + t.w;
  }
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
  int32_t* hist_ids; int32_t* hist_counts; int n_hist;      // ... behind each other
  const int32_t* hist_src;           // pinned host memory
  float repetition, frequency, presence, temperature;
  int m;
  int slice, n_slices;               // values of a slice (a multiple of 256); slices
  float* val;                        // [n] probabilities on the way
  float* cand_v; int32_t* cand_t;    // [n_slices][slice] the slice's values in reach of the m largest, in token order
  uint32_t* top; int n_top, groups;  // bits of the maxima of the slices' groups of values (`groups` of every slice), or of a short row's values themselves
  float *st_max, *st_sum, *st_tot, *st_pmax, *st_sum2; int* st_cnt;   // [256] per slice
  int32_t* tok_out; float* p_out;    // host memory
  HostSignal done;                   // set where the last work-group of the third launch ranks
};

// where the e-th value in reach lies: in the last slice that starts at or before it
__device__ __forceinline__ int smp_slot(const int* start, int e, int slice)
{
  int s = 0;
#pragma unroll
  for (int step = SL_MAX / 2; step > 0; step >>= 1) if (start[s + step] <= e) s += step;
  return s * slice + e - start[s];
}
// A value and its token as one number: descending values, equal ones by token.  (Values are not negative, so their bits order like they do; a NaN is the largest and has
// a place like any other.)
__device__ __forceinline__ uint64_t smp_key(float v, int32_t t) { return (uint64_t)__float_as_uint(v) << 32 | ~(uint32_t)t; }
__device__ __forceinline__ int32_t smp_token(uint64_t k) { return (int32_t)~(uint32_t)k; }
__device__ __forceinline__ float smp_value(uint64_t k) { return __uint_as_float((uint32_t)(k >> 32)); }
// the place of a key among `total`, by eight neighbouring lanes
__device__ __forceinline__ int smp_rank(const uint64_t* key, int total, uint64_t own)
{
  int rank = 0;
#pragma unroll 8
  for (int j = threadIdx.x & 7; j < total; j += 8) rank += key[j] > own;
  rank += __shfl_xor(rank, 1); rank += __shfl_xor(rank, 2); rank += __shfl_xor(rank, 4);
  return rank;
}

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

// A slice of up to HELD x 256 values stays in registers over a launch
constexpr int HELD = 8;
// the work-groups behind the slices': the history, 8 x SL_T words each (as a copy of the stream's own it was one more launch)
constexpr int HIST_PER = 8 * SL_T;
__global__ __launch_bounds__(SL_T) void candidates_stats_kernel(const SampleParams p)
{
  __shared__ float red[SL_T / 64];
  if ((int)blockIdx.x >= p.n_slices) {
    const int i0 = ((int)blockIdx.x - p.n_slices) * HIST_PER + threadIdx.x, n = 2 * p.n_hist;
    int32_t t[8];
#pragma unroll
    for (int u = 0; u < 8; u++) t[u] = __hip_atomic_load(p.hist_src + min(i0 + u * SL_T, n - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
#pragma unroll
    for (int u = 0; u < 8; u++) if (i0 + u * SL_T < n) p.hist_ids[i0 + u * SL_T] = t[u];
    return;
  }
  const int i0 = blockIdx.x * p.slice, len = min(p.slice, p.n - i0);
  const float* x = p.logits + i0;
  float mx = -3.0e38f, sum = 0.0f, t[HELD];
#pragma unroll
  for (int u = 0; u < HELD; u++) { t[u] = x[min((int)threadIdx.x + u * SL_T, len - 1)]; mx = fmaxf(mx, t[u]); }
  for_strided8(x, threadIdx.x + HELD * SL_T, len, SL_T, [&](float v, int) { mx = fmaxf(mx, v); });
  mx = smp_max<SL_T>(mx, red);
#pragma unroll
  for (int u = 0; u < HELD; u++) if ((int)threadIdx.x + u * SL_T < len) sum += smp_exp(t[u], mx);
  for_strided8(x, threadIdx.x + HELD * SL_T, len, SL_T, [&](float v, int) { sum += smp_exp(v, mx); });
  sum = smp_sum<SL_T>(sum, red);
  if (threadIdx.x == 0) { p.st_max[blockIdx.x] = mx; p.st_sum[blockIdx.x] = sum; }
}

// Probabilities with the history penalty: p^r, * exp(-(f * count + presence)) on the distinct context tokens.  What follows keeps their order, but for its
// rounding, so the largest ones of groups of values, found here, tell the next launch where the m-th largest lies (a histogram of the row by atomics: 8.7 us of launch, 5.5 so).
template <bool SHORT>                            // slices of up to HELD x 256 values
__global__ __launch_bounds__(SL_T) void candidates_penalty_kernel(const SampleParams p)
{
  __shared__ float red[SL_T / 64];
  __shared__ float held[SHORT ? HELD * SL_T : 1];
  const int i0 = blockIdx.x * p.slice, len = min(p.slice, p.n - i0), tid = threadIdx.x;
  constexpr int ID = 4;
  int id[ID], count[ID];                         // (the first of the history on their way beside the row)
  float t[HELD];
#pragma unroll
  for (int u = 0; u < ID; u++) if (p.n_hist) { const int k = min(tid + u * SL_T, p.n_hist - 1); id[u] = p.hist_ids[k]; count[u] = p.hist_counts[k]; }
  if (SHORT) {
#pragma unroll
    for (int u = 0; u < HELD; u++) t[u] = p.logits[i0 + min(tid + u * SL_T, len - 1)];
  }
  float mx, inv;
  smp_row_stats(p, red, mx, inv);
  float* const out = p.val + i0;
  float* const val = SHORT ? held : out;
  auto prob = [&](float v) { const float e = smp_exp(v, mx); return inv > 0.0f ? e * inv : e; };
  if (SHORT) {
#pragma unroll
    for (int u = 0; u < HELD; u++) if (tid + u * SL_T < len) held[tid + u * SL_T] = prob(t[u]);
  } else
    for_strided8(p.logits + i0, tid, len, SL_T, [&](float v, int i) { out[i] = prob(v); });
  if (p.n_hist) {
    __syncthreads();
    auto penalise = [&](int t, int c) {
      float v = val[t];
      if (p.repetition != 1.0f && v > 0.0f) v = powf(v, p.repetition);
      if (p.frequency != 0.0f || p.presence != 0.0f) v *= expf(-(p.frequency * (float)c + p.presence));
      val[t] = v;
    };
#pragma unroll
    for (int u = 0; u < ID; u++) { const int j = id[u] - i0; if (tid + u * SL_T < p.n_hist && j >= 0 && j < len) penalise(j, count[u]); }
    for (int k = tid + ID * SL_T; k < p.n_hist; k += SL_T) { const int j = p.hist_ids[k] - i0; if (j >= 0 && j < len) penalise(j, p.hist_counts[k]); }
    __syncthreads();
  }
  float tot = 0.0f, top = 0.0f;
  uint32_t own = 0;
  for_strided8(val, tid, len, SL_T, [&](float v, int i) {
    tot += v; top = fmaxf(top, v); own = max(own, __float_as_uint(v));
    if (SHORT) out[i] = v;
  });
  tot = smp_sum<SL_T>(tot, red);
  top = smp_max<SL_T>(top, red);
  if (tid == 0) { p.st_tot[blockIdx.x] = tot; p.st_pmax[blockIdx.x] = top; }
  if (p.groups == 0) return;
  // groups of SL_T / groups neighbouring threads: 16, 4 or 1
  if (p.groups <= SL_T / 4) { own = max(own, (uint32_t)__shfl_xor((int)own, 1)); own = max(own, (uint32_t)__shfl_xor((int)own, 2)); }
  if (p.groups <= SL_T / 16) { own = max(own, (uint32_t)__shfl_xor((int)own, 4)); own = max(own, (uint32_t)__shfl_xor((int)own, 8)); }
  const int of = SL_T / p.groups;
  if (tid % of == 0) p.top[blockIdx.x * p.groups + tid / of] = own;
}

// The last step of a probability v of a row with the sum tot (0: it is 1) and the largest probability of logarithm lm: itself, or warmed or cooled and still to be
// divided by the row's sum.
__host__ __device__ inline float smp_last(float v, float tot, bool warm, float lm, float inv_t)
{
  if (tot > 0.0f) v = v / tot;
  return warm ? expf(logf(fmaxf(v, 1e-30f)) * inv_t - lm * inv_t) : v;
}
__host__ __device__ inline float smp_bits_float(uint32_t u) { return __builtin_bit_cast(float, u); }
// The bits from which on a probability is in reach of the m largest, where the m-th largest of the groups' maxima lies in `bin` (its leading 12 bits).
// The steps after the maxima keep the order but can make neighbours equal, and equal ones go by token.  A quotient rounds two steps of its dividend together at
// most: four steps below the bin are still in reach.  With a temperature a whole bin is, 6 % of the value at least: 0.06 / T of the exponent, whose own
// errors are 3e-5 / T (of logarithms up to 69) and 1e-6.  Everything is (0) where the row has no finite sum, where what lies below would meet the logarithm's floor, and where the m-th
// value itself, divided by the row's sum, would have lost bits to the end of the number range (what is smaller may: it stays smaller).  That sum is at most n, and up to T = 1 at
// most 1 / (the largest probability), since (v / top)^(1 / T) <= v / top.  Of 152064 values at T = 0.1 this reaches to an m-th value 9 nats below the first (a call 26 us; with everything in
// reach 350).
__host__ __device__ inline uint32_t smp_reach_floor(int bin, bool warm, float tot, float pm, float lm, float inv_t, float temperature, int n, bool divided)
{
  const uint32_t at = (uint32_t)bin << 20, slack = warm ? 1u << 20 : 4u, low = at < slack ? 0u : at - slack;
  const float quotient = tot > 0.0f ? smp_bits_float(low) / tot : smp_bits_float(low);
  bool clear;
  if (warm) {
    const float sum = temperature < 1.0f ? fminf((float)n, 1.0f / pm) : (float)n;
    clear = tot < 3.0e38f && quotient > 1.0e-30f && temperature < 1000.0f && smp_last(smp_bits_float(at), tot, warm, lm, inv_t) > 1.0e-40f * sum;
  } else
    clear = !divided || quotient > 1.2e-38f;
  return clear ? low : 0u;
}

// Last values: the probabilities, or with a temperature exp(ln(max(p, 1e-30)) / T - ln(max p) / T) still to be divided by its sum.  The slice's values that
// can be among the m largest are kept in token order.  FOLDED: the work-group that arrives last ranks them and
// leaves them to the host, or a token of -1 if they are more than it takes; a launch less, and the host reads the flag before the end of the stream.  Where all values of a
// row are in reach every work-group knows that they are too many: nothing is handed over, and the first one tells the host at once.
constexpr int FOLD_MAX = 512;
template <typename T> __device__ __forceinline__ void part_put(T* q, T v) { __hip_atomic_store(q, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename T> __device__ __forceinline__ T part_get(const T* q) { return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <bool FOLDED>
__global__ __launch_bounds__(SL_T) void candidates_reach_kernel(const SampleParams p)
{
  __shared__ float red[SL_T / 64];
  __shared__ int redi[SL_T / 64];
  __shared__ int sel[2];
  __shared__ alignas(16) int bins[SMP_BINS];
  const int i0 = blockIdx.x * p.slice, g = threadIdx.x, per = p.slice / SL_T, j0 = i0 + g * per;
  float v[4];                                    // (a slice has four values a thread at least; past the row any values)
#pragma unroll
  for (int k = 0; k < 4; k++) v[k] = p.val[j0 + k];
  const float own_tot = g < p.n_slices ? p.st_tot[g] : 0.0f, own_max = g < p.n_slices ? p.st_pmax[g] : 0.0f;
  // where the m-th largest of the maxima lies: at least as many values lie there or above
  constexpr int TOPS = 12;
  uint32_t t[TOPS];
#pragma unroll
  for (int u = 0; u < TOPS; u++) t[u] = p.top[min(g + u * SL_T, p.n_top - 1)];
#pragma unroll
  for (int b = 0; b < SMP_BINS / SL_T / 4; b++) reinterpret_cast<int4*>(bins)[g + b * SL_T] = int4{0, 0, 0, 0};
  __syncthreads();
#pragma unroll
  for (int u = 0; u < TOPS; u++) if (g + u * SL_T < p.n_top) atomicAdd(&bins[t[u] >> 20], 1);
  for_strided8(reinterpret_cast<const float*>(p.top), g + TOPS * SL_T, p.n_top, SL_T, [&](float w, int) { atomicAdd(&bins[__float_as_uint(w) >> 20], 1); });
  float pm, tot = 0.0f;
  if (p.n_hist) {
    tot = smp_sum<SL_T>(own_tot, red);
    pm = smp_max<SL_T>(own_max, red);
    if (tot > 0.0f) pm = pm / tot;
  } else {
    float mx;
    smp_row_stats(p, red, mx, pm);              // the maximum's exponential is 1
  }
  const bool warm = p.temperature != 1.0f && pm > 0.0f;
  const float lm = logf(fmaxf(pm, 1e-30f)), inv_t = 1.0f / fmaxf(p.temperature, 1e-6f);
  auto last = [&](float v) { return smp_last(v, tot, warm, lm, inv_t); };
  smp_crossing<SL_T>(bins, min(p.m, p.n), redi, sel);      // (behind the barriers of the sums)
  const uint32_t floor_bits = smp_reach_floor(sel[0], warm, tot, pm, lm, inv_t, p.temperature, p.n, p.n_hist > 0);
  const bool whole = FOLDED && floor_bits == 0u && p.n > FOLD_MAX;
  if (whole && blockIdx.x == 0) {
    if (g == 0) host_store(p.tok_out, (int32_t)-1);
    host_signal(p.done, 1);
  }
  int mine = 0, total;
  float sum2 = 0.0f;
#pragma unroll
  for (int k = 0; k < 4; k++) if (j0 + k < p.n) { mine += __float_as_uint(v[k]) >= floor_bits; if (warm) sum2 += last(v[k]); }
  for (int k = 4; k < per && j0 + k < p.n; k++) { const float t = p.val[j0 + k]; mine += __float_as_uint(t) >= floor_bits; if (warm) sum2 += last(t); }
  sum2 = smp_sum<SL_T>(sum2, red);
  int at = smp_excl_scan<SL_T>(mine, redi, &total);
  if (!warm) sum2 = -1.0f;                       // (< 0: nothing to divide by)
  auto put = [&](auto* q, auto v) { if (FOLDED && !whole) part_put(q, v); else *q = v; };
  if (g == 0) { put(p.st_sum2 + blockIdx.x, sum2); put(p.st_cnt + blockIdx.x, total); }
  for (int k = 0; mine > 0 && k < per && j0 + k < p.n; k++) {
    const float t = p.val[j0 + k];
    if (__float_as_uint(t) >= floor_bits) { put(p.cand_v + i0 + at, last(t)); put(p.cand_t + i0 + at, (int32_t)(j0 + k)); at++; }
  }
  if constexpr (FOLDED) {
    __shared__ int start[SL_MAX];
    __shared__ uint64_t key[FOLD_MAX], place[SMP_FOLD_M];
    if (whole || !arrives_last(p.done.arrive, gridDim.x)) return;
    const int m = min(p.m, p.n), own = g < p.n_slices ? part_get(p.st_cnt + g) : 0;
    float inv = smp_sum<SL_T>(g < p.n_slices ? part_get(p.st_sum2 + g) : 0.0f, red);
    inv = !warm ? 1.0f : 1.0f / (inv <= 0.0f ? 1.0f : inv);
    start[g] = smp_excl_scan<SL_T>(own, redi, &total);
    __syncthreads();
    if (total <= FOLD_MAX) {
      for (int e = g; e < total; e += SL_T) {
        const int j = smp_slot(start, e, p.slice);
        key[e] = smp_key(part_get(p.cand_v + j) * inv, part_get(p.cand_t + j));
      }
      __syncthreads();
      for (int e = g >> 3; e < total; e += SL_T / 8) {
        const uint64_t k = key[e];
        const int rank = smp_rank(key, total, k);
        if ((g & 7) == 0 && rank < m) place[rank] = k;
      }
      __syncthreads();
      for (int r = g; r < m; r += SL_T) { host_store(p.tok_out + r, smp_token(place[r])); host_store(p.p_out + r, smp_value(place[r])); }
    } else if (g == 0) host_store(p.tok_out, (int32_t)-1);
    host_signal(p.done, 1);
  }
}

// descending probability, equal ones by token.  Every work-group gathers the whole list (a few thousand values from the L2) and ranks its
// share of it: the comparisons, not the gathering, were the time of one work-group (1000 candidates of 152064, a whole call, 185 -> 59 us).  Where the third launch left more
// than it takes (equal values in reach) up to 32 wanted are found by one work-group.
__global__ __launch_bounds__(SMP_T) void candidates_rank_kernel(const SampleParams p)
{
  __shared__ int redi[SMP_T / 64];
  __shared__ float redf[SMP_T / 64];
  __shared__ alignas(16) int hist[SMP_BINS];
  __shared__ int cnt[SL_MAX], start[SL_MAX];
  __shared__ int sel[2];
  __shared__ int n_gt;
  __shared__ uint64_t key[RANK_MAX];
  __shared__ uint16_t mine[RANK_MAX];
  __shared__ int n_own;
  const int tid = threadIdx.x, m = min(p.m, p.n);
  const int own = tid < p.n_slices ? p.st_cnt[tid] : 0;
  float inv = smp_sum<SMP_T>(tid < p.n_slices ? p.st_sum2[tid] : 0.0f, redf);
  inv = p.st_sum2[0] < 0.0f ? 1.0f : 1.0f / (inv <= 0.0f ? 1.0f : inv);
  int total;
  const int before = smp_excl_scan<SMP_T>(own, redi, &total);
  if (tid < SL_MAX) { cnt[tid] = own; start[tid] = before; }
  if (tid == 0) n_gt = 0;
  __syncthreads();
  if (total <= RANK_MAX) {
    for (int e = tid; e < total; e += SMP_T) { const int j = smp_slot(start, e, p.slice); key[e] = smp_key(p.cand_v[j] * inv, p.cand_t[j]); }
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
        const uint32_t u = __float_as_uint(v * inv);
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
      if (i - s * p.slice < cnt[s] && __float_as_uint(v * inv) > prefix) { const int k = atomicAdd(&n_gt, 1); key[k] = smp_key(v * inv, p.cand_t[i]); }
    });
    __syncthreads();
    const int base = n_gt;                       // = m - need
    const int chunk = (slots + SMP_T - 1) / SMP_T, c0 = tid * chunk, c1 = min(slots, c0 + chunk);
    int ties = 0;
    for (int i = c0; i < c1; i++) { const int s = i / p.slice; ties += i - s * p.slice < cnt[s] && __float_as_uint(p.cand_v[i] * inv) == prefix; }
    int all, rank = smp_excl_scan<SMP_T>(ties, redi, &all);
    for (int i = c0; ties > 0 && rank < need && i < c1; i++) {
      const int s = i / p.slice;
      if (i - s * p.slice < cnt[s] && __float_as_uint(p.cand_v[i] * inv) == prefix) { key[base + rank] = smp_key(p.cand_v[i] * inv, p.cand_t[i]); rank++; }
    }
    total = m;
  }
  __syncthreads();
  // This work-group's share: the tokens of one residue (the order of the list is not the same in every work-group).  Eight neighbouring
  // lanes rank a value together.
  if (tid == 0) n_own = 0;
  __syncthreads();
  for (int e = tid; e < total; e += SMP_T) if ((unsigned)smp_token(key[e]) % gridDim.x == blockIdx.x) mine[atomicAdd(&n_own, 1)] = (uint16_t)e;
  __syncthreads();
  for (int o = tid >> 3; o < n_own; o += SMP_T / 8) {
    const uint64_t k = key[mine[o]];
    const int rank = smp_rank(key, total, k);
    if ((tid & 7) == 0 && rank < m) { p.tok_out[rank] = smp_token(k); p.p_out[rank] = smp_value(k); }
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
  bool penalty = false;              // some token of the history lies in the row and a penalty is set
  if (repetition != 1.0f || frequency != 0.0f || presence != 0.0f)
    for (int k = 0; k < n_hist && !penalty; k++) penalty = hist_ids[k] >= 0 && hist_ids[k] < n;
  // four values per thread of a slice (149 work-groups for a 152k row) until there are 256 slices
  p.slice = std::max(4 * SL_T, ((n + SL_MAX - 1) / SL_MAX + SL_T - 1) / SL_T * SL_T);
  p.n_slices = (n + p.slice - 1) / p.slice;
  const size_t slots = (size_t)p.n_slices * p.slice;
  int rc = ensure_stage(&c.stage_out, &c.stage_out_cap, (3 * slots + TOP_MAX + 6 * SL_MAX) * 4); if (rc) return rc;
  p.val = (float*)c.stage_out; p.cand_v = p.val + slots; p.cand_t = (int32_t*)(p.cand_v + slots);
  // groups of 64 values of an ordinary slice, or of 16 or 4 where there would not be twice as many of them as are wanted; the values themselves of short rows
  p.groups = n <= TOP_MAX ? 0 : p.n_slices * 16 >= 2 * m ? 16 : p.n_slices * 64 >= 2 * m ? 64 : 256;
  p.top = p.groups ? (uint32_t*)(p.cand_t + slots) : (uint32_t*)p.val;
  p.n_top = p.groups ? p.n_slices * p.groups : n;
  p.st_max = (float*)((uint32_t*)(p.cand_t + slots) + TOP_MAX); p.st_sum = p.st_max + SL_MAX; p.st_tot = p.st_sum + SL_MAX; p.st_pmax = p.st_tot + SL_MAX;
  p.st_sum2 = p.st_pmax + SL_MAX; p.st_cnt = (int*)(p.st_sum2 + SL_MAX);
  // host side: [tokens 1024 | probabilities 1024 | history ids | history counts]; the last launch writes the first two where they lie
  const size_t hist = penalty ? (size_t)n_hist : 0;
  if ((rc = ensure_host_stage((2 * (size_t)SMP_MAX_M + 2 * hist) * 4))) return rc;
  int32_t* h = (int32_t*)c.h_stage;
  p.tok_out = h; p.p_out = (float*)(h + SMP_MAX_M);
  if (hist) {
    if ((rc = ensure_stage(&c.stage_in, &c.stage_in_cap, 2 * hist * 4))) return rc;
    memcpy(h + 2 * SMP_MAX_M, hist_ids, hist * 4); memcpy(h + 2 * SMP_MAX_M + hist, hist_counts, hist * 4);
    p.hist_src = h + 2 * SMP_MAX_M; p.hist_ids = (int32_t*)c.stage_in; p.hist_counts = p.hist_ids + hist; p.n_hist = n_hist;
  }
  const dim3 grid(p.n_slices), block(SL_T);
  hipLaunchKernelGGL(candidates_stats_kernel, dim3(p.n_slices + (2 * hist + HIST_PER - 1) / HIST_PER), block, 0, c.stream, p);
  if (p.slice <= HELD * SL_T) hipLaunchKernelGGL(candidates_penalty_kernel<true>, grid, block, 0, c.stream, p);
  else hipLaunchKernelGGL(candidates_penalty_kernel<false>, grid, block, 0, c.stream, p);
  bool ranked = false;
  if (m <= SMP_FOLD_M) {
    p.done = host_signal_next();
    hipLaunchKernelGGL(candidates_reach_kernel<true>, grid, block, 0, c.stream, p);
    CAI_HIP(hipGetLastError());
    if ((rc = host_signal_wait(p.done))) return rc;
    ranked = h[0] >= 0;
  } else
    hipLaunchKernelGGL(candidates_reach_kernel<false>, grid, block, 0, c.stream, p);
  if (!ranked) {
    hipLaunchKernelGGL(candidates_rank_kernel, dim3(m > 32 ? RANK_WG : 1), dim3(SMP_T), 0, c.stream, p);
    CAI_HIP(hipGetLastError());
    CAI_HIP(hipStreamSynchronize(c.stream));
  }
  memcpy(tokens_out, h, (size_t)m * 4);
  memcpy(probs_out, h + SMP_MAX_M, (size_t)m * 4);
  if (count_out) *count_out = m;
  return CAI_OK;
}

}  // namespace cai

using namespace cai;

// For the tests of the rule; host only, not part of the interface in caihip.h: the bits from which on values are in reach (0: all), in a row whose largest probability is pm and whose
// values are, with a history, probabilities times tot.
extern "C" int cai_candidates_floor(int bin, float tot, float pm, float temperature, int n, int divided)
{
  CAI_ENTER();
  CAI_REQUIRE(bin >= 0 && bin < SMP_BINS && n >= 1, "cai_candidates_floor: bad argument");
  const bool warm = temperature != 1.0f && pm > 0.0f;
  return (int)smp_reach_floor(bin, warm, tot, pm, logf(fmaxf(pm, 1e-30f)), 1.0f / fmaxf(temperature, 1e-6f), temperature, n, divided != 0);
}

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
