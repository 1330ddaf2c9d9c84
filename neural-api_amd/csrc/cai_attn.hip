// KV cache + cached grouped-query decode attention for gfx950.
//
// Layer semantics (TNNetFusedSDPA; neural/neural.cl:2354-2499): the token row is [Q | K | V]; K and V are
// appended to a head-major cache (row (g, p) at (g*MaxCtx + p)*Dk), then for each query head h (KV head
// g = h / group) out_h = softmax(q_h . K_g / sqrt(Dk)) V_g over the live rows [jStart, len).
//
// Device formulation: split-K over the key axis; a slice of the live rows per work-group, and the slices of a head merged by the last of its work-groups to
// arrive (the per-head kernel: 8.0 + 4.9 -> 9.8 us on the 7B shape) or by a small second kernel, one work-group per query head (the kernels of a whole group of heads: merged in place 37.7 us on
// the 32B shape, 21.5 + 5 so).  RoPE of q and of the new k row and the cache append happen inside the split kernel.  Two split kernels:
//   attn_group_kernel       one work-group per (slice, KV head) serves the whole group of query heads, so K and V are
//                           fetched once; three phases per slice (scores -> LDS, softmax, value sum).  Used when the
//                           grid fills the chip by itself (long caches, several sequences, prompt ingestion).
//   attn_split_head_kernel  one work-group per (slice, QUERY head), online softmax in registers; the G heads of a
//                           group re-read the slice from L2.  G times more work-groups: the better one for one
//                           sequence with a short cache.
// Cache element types: fp32, IEEE half, or int8 codes with one fp32 scale per cached row (neural/neural.cl:2501-2687).
#include "cai_internal.hpp"
#include "cai_gemv_common.hpp"

namespace cai {

template <typename T> __device__ __forceinline__ float kv_to_float(T v);
template <> __device__ __forceinline__ float kv_to_float<float>(float v) { return v; }
template <> __device__ __forceinline__ float kv_to_float<__half>(__half v) { return __half2float(v); }
template <typename T> __device__ __forceinline__ T kv_from_float(float v);
template <> __device__ __forceinline__ float kv_from_float<float>(float v) { return v; }
template <> __device__ __forceinline__ __half kv_from_float<__half>(float v) { return __float2half_rn(v); }


// VW (2 or 4) consecutive cache elements with one load, kept as they lie until they are used: a conversion beside the load would wait for it
// before the next goes out
template <int VW, typename KV_T> struct RowVec;
template <> struct RowVec<2, float> { typedef float type __attribute__((ext_vector_type(2), aligned(4))); };
template <> struct RowVec<4, float> { typedef float type __attribute__((ext_vector_type(4), aligned(4))); };
template <> struct RowVec<2, __half> { using type = uint32_t; };
template <> struct RowVec<4, __half> { using type = uint2; };
template <> struct RowVec<2, int8_t> { using type = uint16_t; };
template <> struct RowVec<4, int8_t> { using type = uint32_t; };
template <int VW, typename KV_T> using row_vec = typename RowVec<VW, KV_T>::type;
template <int VW, typename KV_T>
__device__ __forceinline__ void row_floats(const row_vec<VW, KV_T>& r, float* o)
{
  if constexpr (sizeof(KV_T) == 4) {
#pragma unroll
    for (int i = 0; i < VW; i++) o[i] = r[i];
  } else if constexpr (sizeof(KV_T) == 2) {
    if constexpr (VW == 2) { const __half2 h = __builtin_bit_cast(__half2, r); o[0] = __low2float(h); o[1] = __high2float(h); }
    else {
      const __half2 h = __builtin_bit_cast(__half2, r.x), g = __builtin_bit_cast(__half2, r.y);
      o[0] = __low2float(h); o[1] = __high2float(h); o[2] = __low2float(g); o[3] = __high2float(g);
    }
  } else {
#pragma unroll
    for (int i = 0; i < VW; i++) o[i] = (float)((int)((uint32_t)r << (24 - 8 * i)) >> 24);
  }
}
// sum / maximum over each row of 16 lanes, in every lane of it
#define ROW_ROR(v, n) __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, (v)), 0x120 + (n), 0xf, 0xf, false))
__device__ __forceinline__ float row16_sum(float v) { v += ROW_ROR(v, 8); v += ROW_ROR(v, 4); v += ROW_ROR(v, 2); v += ROW_ROR(v, 1); return v; }
__device__ __forceinline__ float row16_max(float v) { v = fmaxf(v, ROW_ROR(v, 8)); v = fmaxf(v, ROW_ROR(v, 4)); v = fmaxf(v, ROW_ROR(v, 2)); v = fmaxf(v, ROW_ROR(v, 1)); return v; }

// max over each half-wave (32 lanes), result in every lane of that half
__device__ __forceinline__ float half_wave_allmax(float v)
{
  for (int o = 16; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// One cached row of an int8 cache from DS elements per lane of a half-wave (neural/neural.cl:2549-2578): the maximum
// over FINITE magnitudes, zero codes and unit scale when that maximum is zero or denormal, else scale = max / 127 and
// code = clamp(rint(v * (1/max) * 127)), NaN -> 0.  Lanes beyond the head width pass zeros.  On return v[] holds the
// codes as floats.  ROW16: 16 lanes hold the row.
template <int DS, bool ROW16 = false> __device__ __forceinline__ float quantise_row_i8(float (&v)[DS])
{
  float m = 0.0f;
#pragma unroll
  for (int i = 0; i < DS; i++) {
    const float a = fabsf(v[i]);
    if (__builtin_bit_cast(uint32_t, a) <= 0x7F7FFFFFu) m = fmaxf(m, a);
  }
  m = ROW16 ? row16_max(m) : half_wave_allmax(m);
  const bool usable = __builtin_bit_cast(uint32_t, m) >= 0x00800000u;
  const float recip = usable ? 1.0f / m : 0.0f;
#pragma unroll
  for (int i = 0; i < DS; i++) {
    float scaled = v[i] * recip * 127.0f;
    if (!usable || __builtin_bit_cast(uint32_t, fabsf(v[i])) > 0x7F800000u) scaled = 0.0f;
    v[i] = fminf(fmaxf(rintf(scaled), -127.0f), 127.0f);
  }
  return usable ? m / 127.0f : 1.0f;
}

struct AttnParams {
  float* qkv; int64_t qkv_stride;
  void* kc; void* vc;          // base of [seq][layer][kv_head][max_ctx][hd]
  int64_t seq_elems, layer_off; // element offsets
  int q_heads, kv_heads, hd, max_ctx;
  int window; float softcap; float inv_sqrt;
  const float* theta;          // hd/2 frequencies or null
  const int32_t* pos;          // [seq]
  int split_len, n_splits;
  float* part;                 // [seq][q_head][split][hd+2]
  float* out; int64_t out_stride;
  int seq0;                    // cache sequence index of activation row 0
  int seq_mul;                 // 1: activation row s uses cache sequence seq0 + s; 0: all rows share sequence seq0 (prompt)
  int appended;                // 1: the K,V rows of this step are already in the cache (prompt ingestion)
  float* part_override;        // split partials buffer when more rows than cache sequences are in flight
  float* ksc; float* vsc;      // int8 caches: row scales [seq][layer][kv_head][max_ctx]
  int64_t seq_rows, layer_row_off;
  int64_t scale_row0;          // the per-head kernel: row of the scales where this layer of sequence seq0 begins
  int evict_sinks, evict_cap;  // cap > 0: only the first `sinks` positions and the latest cap - sinks stay cached
  const float* qn_gain; const float* kn_gain; float qk_eps;   // full-width RMSNorm of q and of k applied while they are read (null: rows are used as they are)
  unsigned* merge_cnt;         // decode steps: arrival counters [seq][head]; the work-group that completes the last slice merges (null: a merge launch follows)
  unsigned long long* timeline; // stamps of this launch's work-groups (null: none)
};
struct PlanesParams : AttnParams { BlkPlanes planes; bool planes_q8 = true; };      // a prompt's rows whose results leave as planes (planes.hi null: as rows)

typedef _Float16 ph4_t __attribute__((ext_vector_type(4)));
typedef _Float16 ph8_t __attribute__((ext_vector_type(8)));

// A result of row t, column c of w, whose neighbours of a block of 32 columns are in the neighbouring lanes
__device__ __forceinline__ void out_plane(const BlkPlanes& o, bool q8_0, int t, int c, int w, float y)
{
  float m = finite_abs(y);
#pragma unroll
  for (int k = 1; k < 32; k <<= 1) m = fmaxf(m, __shfl_xor(m, k));
  const int e = plane_exponent(m);
  _Float16 h, l; split_plane(y * ldexpf(1.0f, e), h, l);
  const int64_t blk = (int64_t)(t >> 4) * (w >> 5) + (c >> 5), at = blk * 512 + plane_place(q8_0, t & 15, c & 31);
  o.hi[at] = h; o.lo[at] = l;
  if ((c & 31) == 0) o.scale[blk * 16 + (t & 15)] = ldexpf(1.0f, -e);
}
// Four of them, c .. c + 3: eight neighbouring lanes hold a block
__device__ __forceinline__ void out_plane4(const BlkPlanes& o, bool q8_0, int t, int c, int w, const float (&y)[4])
{
  float m = fmaxf(fmaxf(finite_abs(y[0]), finite_abs(y[1])), fmaxf(finite_abs(y[2]), finite_abs(y[3])));
#pragma unroll
  for (int k = 1; k < 8; k <<= 1) m = fmaxf(m, __shfl_xor(m, k));
  const int e = plane_exponent(m);
  ph4_t h, l;
#pragma unroll
  for (int i = 0; i < 4; i++) { _Float16 a, b; split_plane(y[i] * ldexpf(1.0f, e), a, b); h[i] = a; l[i] = b; }
  const int64_t blk = (int64_t)(t >> 4) * (w >> 5) + (c >> 5), at = blk * 512 + plane_place(q8_0, t & 15, c & 31);
  *reinterpret_cast<ph4_t*>(o.hi + at) = h; *reinterpret_cast<ph4_t*>(o.lo + at) = l;
  if ((c & 31) == 0) o.scale[blk * 16 + (t & 15)] = ldexpf(1.0f, -e);
}

// ---- merge of the split partials inside the split kernels ----
// The slices of a head (or of a KV head's group of heads) finish in any order on any XCD.  Each work-group writes its partial
// through to memory (agent-scope stores: the XCDs' L2 caches are not coherent with one another inside a launch), waits for the
// stores to be acknowledged and then counts itself in; the one that counts last reads all partials back at agent scope and
// writes the finished rows.  The counter wraps to zero on the last arrival, so it needs no clearing between launches.  No
// cache-wide fence is involved (a __threadfence per work-group measured several times the merge launch it saves).
__device__ __forceinline__ float lane_value(float v, int lane) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane)); }
__device__ __forceinline__ void part_store(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float part_load(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// The slices of head qh of sequence `seq`; every thread of the work-group calls it after its partial stores
__device__ __forceinline__ void merge_if_last(const AttnParams& p, int seq, int qh, int s_first, int n_active, int counter)
{
  const bool last = arrives_last(p.merge_cnt + counter, (unsigned)n_active);
  timeline_stamp(p.timeline, 6);
  if (!last) return;
  // One round trip per MB slices: every thread requests its value of each slice, lane u of every wave the maximum and the sum of slice u.  The
  // slices are folded in order with a running maximum; what that scales by depends on the maxima alone, so lane u works it out for slice u
  // and the fold reads it from there (every thread by itself, two exponentials a slice: half a microsecond at ten slices).
  constexpr int MB = 12;                  // (at most the 16 lanes of a row)
  const int hd = p.hd, lane = threadIdx.x & 63;
  const float* const pt = p.part + (((int64_t)seq * p.q_heads + qh) * p.n_splits + s_first) * (hd + 2);
  for (int o = threadIdx.x; o - lane < hd; o += blockDim.x) {      // (whole waves)
    const int d = min(o, hd - 1);
    float A = 0.0f, L = 0.0f, M = -1e30f;
    for (int s0 = 0; s0 < n_active; s0 += MB) {
      float v[MB];
      const float* pu = pt + (int64_t)min(s0 + min(lane, MB - 1), n_active - 1) * (hd + 2);
      const float mu = part_load(pu + hd), lu = part_load(pu + hd + 1);
#pragma unroll
      for (int u = 0; u < MB; u++) v[u] = part_load(pt + (int64_t)min(s0 + u, n_active - 1) * (hd + 2) + d);
      const bool on = s0 + lane < n_active && lane < MB && lu > 0.0f;
      float top = on ? mu : -1e30f;                                            // the running maximum up to this lane's slice
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int t = __builtin_bit_cast(int, top);
        top = fmaxf(top, __builtin_bit_cast(float, k == 0 ? __builtin_amdgcn_update_dpp(t, t, 0x111, 0xf, 0xf, false) : k == 1 ? __builtin_amdgcn_update_dpp(t, t, 0x112, 0xf, 0xf, false)
                                                 : k == 2 ? __builtin_amdgcn_update_dpp(t, t, 0x114, 0xf, 0xf, false) : __builtin_amdgcn_update_dpp(t, t, 0x118, 0xf, 0xf, false)));   // row_shr
      }
      top = fmaxf(top, M);
      const float before = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, M), __builtin_bit_cast(int, top), 0x111, 0xf, 0xf, false));
      const float c0 = expf(before - top), c1 = on ? expf(mu - top) : 0.0f;
#pragma unroll
      for (int u = 0; u < MB; u++) {
        if (lane_value(on ? 1.0f : 0.0f, u) != 0.0f) {
          const float e0 = lane_value(c0, u), e1 = lane_value(c1, u);
          A = fmaf(v[u], e1, A * e0); L = fmaf(lane_value(lu, u), e1, L * e0);
        }
      }
      M = lane_value(top, MB - 1);
    }
    if (o < hd) p.out[(int64_t)seq * p.out_stride + qh * hd + d] = L > 0.0f ? A * (1.0f / L) : 0.0f;
  }
}

// Where the row of stream position `pos` lives and which rows are live.  Without eviction: slot = pos, rows
// [j_start, pos] (j_start > 0 under a sliding window).  With sink + recent-window eviction (TNNetStreamingDecoder.
// EnableEviction, neural/neuraldecode.pas:1257-1276) the cache holds positions [0, sinks) and the latest cap - sinks;
// instead of shifting rows on every token the recent part is a ring: slot = sinks + (pos - sinks) mod (cap - sinks),
// and all cap rows are live.  Keys keep the rotation of their own position, the query that of `pos`.
struct LiveRows { int slot, len, j_start; };
__device__ __forceinline__ LiveRows live_rows(const AttnParams& p, int pos)
{
  LiveRows r;
  if (p.evict_cap > 0 && pos >= p.evict_cap) {
    r.slot = p.evict_sinks + (pos - p.evict_sinks) % (p.evict_cap - p.evict_sinks); r.len = p.evict_cap; r.j_start = 0;
  } else {
    r.slot = pos; r.len = pos + 1;
    r.j_start = (p.window > 0 && r.len > p.window) ? r.len - p.window : 0;
  }
  return r;
}

// ---- split kernel: RoPE (neural/neural.cl:1517-1542) + KV append (2354-2379) + one slice of the cached decode
//      (2406-2499), all query heads of a KV head in ONE work-group, so K and V are fetched once.
//
//      16 lanes x 8 elements cover a row, a wave holds 4 rows, the work-group 16 rows per pass; every load is 16
//      contiguous bytes per lane and a wave's load is 4 whole rows.  Three phases like the reference kernel, but per
//      slice: (1) scores of the slice into LDS (dot products reduced over 16 lanes with DPP), (2) slice maximum,
//      exp-shift and sum per head, (3) the value sum.  The query heads are taken HC at a time (q and the accumulators
//      live in registers: 8*HC each); a second chunk of heads re-reads the slice from cache.  The slice partial
//      (sum_j e_j V_j, max, sum e_j) goes to the merge kernel, or straight to the output when the live range fits one
//      slice. ----
template <typename KV_T> struct Row8;
template <> struct Row8<float>  { float4 a, b; };
template <> struct Row8<__half> { uint4 a; };
template <> struct Row8<int8_t> { uint2 a; };

__device__ __forceinline__ void load8(const float* s, Row8<float>& r) { r.a = reinterpret_cast<const float4*>(s)[0]; r.b = reinterpret_cast<const float4*>(s)[1]; }
__device__ __forceinline__ void load8(const __half* s, Row8<__half>& r) { r.a = *reinterpret_cast<const uint4*>(s); }
__device__ __forceinline__ void load8(const int8_t* s, Row8<int8_t>& r) { r.a = *reinterpret_cast<const uint2*>(s); }
__device__ __forceinline__ void unpack8(const Row8<float>& r, float (&v)[8])
{
  v[0] = r.a.x; v[1] = r.a.y; v[2] = r.a.z; v[3] = r.a.w; v[4] = r.b.x; v[5] = r.b.y; v[6] = r.b.z; v[7] = r.b.w;
}
__device__ __forceinline__ void unpack8(const Row8<__half>& r, float (&v)[8])
{
  const uint32_t w[4] = {r.a.x, r.a.y, r.a.z, r.a.w};
#pragma unroll
  for (int i = 0; i < 4; i++) { const __half2 h = __builtin_bit_cast(__half2, w[i]); v[2 * i] = __low2float(h); v[2 * i + 1] = __high2float(h); }
}
__device__ __forceinline__ void unpack8(const Row8<int8_t>& r, float (&v)[8])
{
  const int w[2] = {(int)r.a.x, (int)r.a.y};
#pragma unroll
  for (int i = 0; i < 2; i++) {
    v[4 * i] = (float)((w[i] << 24) >> 24); v[4 * i + 1] = (float)((w[i] << 16) >> 24);
    v[4 * i + 2] = (float)((w[i] << 8) >> 24); v[4 * i + 3] = (float)(w[i] >> 24);
  }
}

// wave64 maximum / sum in every lane: DPP steps inside the vector unit (row_shr within rows of 16, row_bcast15 / row_bcast31,
// total in lane 63, broadcast through a scalar register) instead of six trips through the LDS crossbar
__device__ __forceinline__ float wave_allmax(float v)
{
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x111, 0xf, 0xf, false)));
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x112, 0xf, 0xf, false)));
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x114, 0xf, 0xf, false)));
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x118, 0xf, 0xf, false)));
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x142, 0xa, 0xf, false)));
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x143, 0xc, 0xf, false)));
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ __forceinline__ float wave_allsum(float v)
{
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wave_sum(v)), 63));
}
// gfx950 row swaps (a row = 16 lanes).  row_swap16: rows 1, 3 of x change places with rows 0, 2 of y, i.e. x = (x0 y0 x2 y2),
// y = (x1 y1 x3 y3); row_swap32: the upper half of x with the lower half of y, i.e. x = (x0 x1 y0 y1), y = (x2 x3 y2 y3).
// Written as instructions: through the builtins this compiler read BOTH results from the first register (sums came out as
// 2 x the first result).  The instruction needs two idle cycles after a vector write of its operands, which the compiler
// cannot see inside the statement: the s_nop provides them.
__device__ __forceinline__ void row_swap16(float& x, float& y) { asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(x), "+v"(y)); }
__device__ __forceinline__ void row_swap32(float& x, float& y) { asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(x), "+v"(y)); }
// sum over each aligned group of 16 lanes, result in every lane of the group
__device__ __forceinline__ float row16_allsum(float v)
{
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xb1, 0xf, 0xf, true));   // lane ^ 1
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4e, 0xf, 0xf, true));   // lane ^ 2
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, true));  // 7 - lane within 8
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xf, 0xf, true));  // 15 - lane within 16
  return v;
}

template <int HC, typename KV_T, int NPF>     // NPF: passes in flight per lane
__global__ __launch_bounds__(256) void attn_group_kernel(const int32_t* hpos, const float* hqkv, const float* htheta, const long long hqkv_stride,
                                                         const int hheads, const int hgeo, const int hsl, const AttnParams p)
{
  // (leading scalar arguments arrive preloaded in scalar registers: position, q | k | v row and frequencies are requested without
  //  a round trip to the argument block; hheads = query heads | KV heads << 16, hgeo = slices | head width << 16, hsl = slice length)
  const unsigned long long tl0 = timeline_now();
  const int h_q_heads = hheads & 0xffff, h_kv_heads = hheads >> 16, h_n_splits = hgeo & 0xffff, h_hd = hgeo >> 16;
  extern __shared__ __align__(16) float lds[];
  constexpr bool I8 = sizeof(KV_T) == 1;
  const int G = h_q_heads / h_kv_heads, n_chunks = (G + HC - 1) / HC;
  const int split = blockIdx.x % h_n_splits, g = blockIdx.x / h_n_splits, seq = blockIdx.y;
  const int pos = hpos[seq];
  const LiveRows lr = live_rows(p, pos);
  const int len = lr.len, j_start = lr.j_start, slot = lr.slot;
  const int s_begin = max(j_start, split * hsl), s_end = min(len, (split + 1) * hsl);
  if (s_begin >= s_end) return;   // whole work-group leaves together, before any barrier
  const int s_first = j_start / hsl, s_last = (len - 1) / hsl;
  const int n_active = s_last - s_first + 1;
  const int n_rows = s_end - s_begin, n_pass = (n_rows + 15) >> 4;

  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, r = lane >> 4, c = lane & 15, rr = 4 * w + r;
  const int hd = h_hd, qw = h_q_heads * hd, kw = h_kv_heads * hd, SL = hsl;
  const int d0 = 8 * c;
  const bool lane_on = d0 < hd;
  const int dl = lane_on ? d0 : 0;
  const float* row = hqkv + (int64_t)seq * hqkv_stride;
  const int64_t cache_seq = seq * p.seq_mul + p.seq0;
  KV_T* kc = reinterpret_cast<KV_T*>(p.kc) + cache_seq * p.seq_elems + p.layer_off + (int64_t)g * p.max_ctx * hd;
  KV_T* vc = reinterpret_cast<KV_T*>(p.vc) + cache_seq * p.seq_elems + p.layer_off + (int64_t)g * p.max_ctx * hd;
  float* ksc = nullptr; float* vsc = nullptr;
  if (I8) { const int64_t r0 = cache_seq * p.seq_rows + p.layer_row_off + (int64_t)g * p.max_ctx; ksc = p.ksc + r0; vsc = p.vsc + r0; }

  float* sq = lds;                          // rotated q [G][128]
  float* sS = sq + G * 128;                 // scores [G][SL]
  constexpr int PW = HC > 4 ? 8 : 4;
  float* sP = sS + G * SL;                  // softmax weights [chunk][SL][PW]
  float* sred = sP + n_chunks * SL * PW;    // per-wave value sums [4][HC][128]
  float* sML = sred + 4 * HC * 128;         // slice maximum [G], slice sum [G]

  Row8<KV_T> ring[NPF];
  float rsc[NPF];
  auto issue = [&](const KV_T* base, const float* scales, int slot, int t) {
    const int j = min(s_begin + 16 * t + rr, s_end - 1);
    load8(base + (int64_t)j * hd + dl, ring[slot]);     // lanes beyond the head width re-read its start; q is zero there
    if (I8) rsc[slot] = scales[j];
  };
  auto prime = [&](const KV_T* base, const float* scales) {
#pragma unroll
    for (int u = 0; u < NPF; u++) { rsc[u] = 0.0f; issue(base, scales, u, u); }   // (never conditional: passes beyond the slice re-read its last row, unused)
  };
  const bool owns_new = !p.appended && slot >= s_begin && slot < s_end;
  // Requests return in the order they were issued: the group's q pairs and frequencies (two turns of the work-group cover up to
  // eight 128-wide heads) go out first, the cached rows behind them, so that the rotation runs while the rows are on their way.
  const int n_qp = G * (hd >> 1);
  float qx0[2], qx1[2], qth[2];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int e = min(tid + 256 * u, n_qp - 1), h = e / (hd >> 1), i = e % (hd >> 1);
    const float* qh = row + (g * G + h) * hd;
    qx0[u] = qh[2 * i]; qx1[u] = qh[2 * i + 1]; qth[u] = htheta ? htheta[i] : 0.0f;
  }
  if (!owns_new) prime(kc, ksc);
  timeline_put(p.timeline, 0, tl0);
  timeline_stamp(p.timeline, 1);

  // rotated q of the group's heads -> LDS
  for (int e = tid; e < n_qp; e += 256) {
    const int h = e / (hd >> 1), i = e % (hd >> 1);
    const int u = (e - tid) >> 8;
    float x0, x1, th;
    if (u < 2) { x0 = u ? qx0[1] : qx0[0]; x1 = u ? qx1[1] : qx1[0]; th = u ? qth[1] : qth[0]; }
    else { const float* qh = row + (g * G + h) * hd; x0 = qh[2 * i]; x1 = qh[2 * i + 1]; th = htheta ? htheta[i] : 0.0f; }
    if (htheta) {
      float sn, cs; sincosf((float)pos * th, &sn, &cs);
      const float y0 = cs * x0 - sn * x1, y1 = sn * x0 + cs * x1;
      x0 = y0; x1 = y1;
    }
    sq[h * 128 + 2 * i] = x0; sq[h * 128 + 2 * i + 1] = x1;
  }
  // the work-group whose slice holds `pos` appends the new row: wave 0, one half-wave each for K and V
  if (owns_new && w == 0) {
    const int l32 = lane & 31, is_v = lane >> 5, e0 = 4 * l32;
    const float* src = row + qw + (is_v ? kw : 0) + g * hd;
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      const int d = e0 + i;
      float x0 = d < hd ? src[d] : 0.0f, x1 = d + 1 < hd ? src[d + 1] : 0.0f;
      if (htheta && !is_v && d < hd) {
        float sn, cs; sincosf((float)pos * htheta[d >> 1], &sn, &cs);
        const float y0 = cs * x0 - sn * x1, y1 = sn * x0 + cs * x1;
        x0 = y0; x1 = y1;
      }
      v[i] = x0; v[i + 1] = x1;
    }
    KV_T* dst = (is_v ? vc : kc) + (int64_t)slot * hd;
    if constexpr (I8) {
      const float scale = quantise_row_i8<4>(v);
#pragma unroll
      for (int i = 0; i < 4; i++) if (e0 + i < hd) dst[e0 + i] = (int8_t)v[i];
      if (l32 == 0) (is_v ? vsc : ksc)[slot] = scale;
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++) if (e0 + i < hd) dst[e0 + i] = kv_from_float<KV_T>(v[i]);
    }
  }
  __syncthreads();      // q is staged; the appended row is visible to this work-group's loads
  if (owns_new) prime(kc, ksc);
  timeline_stamp(p.timeline, 4);

  // ---- phase 1: scores of the slice ----
  for (int ch = 0; ch < n_chunks; ch++) {
    const int h0 = ch * HC;
    if (ch > 0) prime(kc, ksc);
    float q[HC][8];
#pragma unroll
    for (int hh = 0; hh < HC; hh++)
#pragma unroll
      for (int i = 0; i < 8; i++) q[hh][i] = (lane_on && h0 + hh < G) ? sq[(h0 + hh) * 128 + d0 + i] : 0.0f;
    for (int t0 = 0; t0 < n_pass; t0 += NPF) {
#pragma unroll
      for (int u = 0; u < NPF; u++) {
        const int t = t0 + u;
        if (t < n_pass) {
          float v[8];
          unpack8(ring[u], v);
          const float rs = rsc[u];
          if (t + NPF < n_pass) issue(kc, ksc, u, t + NPF);
          float sv = 0.0f;
#pragma unroll
          for (int hh = 0; hh < HC; hh++) {
            float a = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; i++) a = fmaf(q[hh][i], v[i], a);
            a = row16_allsum(a);
            if (c == hh) sv = a;
          }
          const int rl = 16 * t + rr;
          if (rl < n_rows && c < HC && h0 + c < G) {
            sS[(h0 + c) * SL + rl] = sv * (I8 ? rs * p.inv_sqrt : p.inv_sqrt);
          }
        }
      }
    }
  }
  prime(vc, vsc);        // the first value rows travel while the softmax runs
  __syncthreads();
  timeline_stamp(p.timeline, 5);

  // ---- phase 2: slice maximum, exp-shift and sum per head (wave w takes heads w, w+4, ..) ----
  for (int h = w; h < G; h += 4) {
    float m = -1e30f;
    if (p.softcap > 0.0f)
      for (int rl = lane; rl < n_rows; rl += 64) sS[h * SL + rl] = p.softcap * tanhf(sS[h * SL + rl] / p.softcap);
    for (int rl = lane; rl < n_rows; rl += 64) m = fmaxf(m, sS[h * SL + rl]);
    m = wave_allmax(m);
    float l = 0.0f;
    for (int rl = lane; rl < n_rows; rl += 64) {
      const float e = expf(sS[h * SL + rl] - m);
      l += e;
      sP[((h / HC) * SL + rl) * PW + h % HC] = I8 ? e * vsc[s_begin + rl] : e;
    }
    l = wave_allsum(l);
    if (lane == 0) { sML[h] = m; sML[G + h] = l; }
  }
  __syncthreads();

  timeline_stamp(p.timeline, 6);
  // ---- phase 3: value sums ----
  for (int ch = 0; ch < n_chunks; ch++) {
    const int h0 = ch * HC;
    if (ch > 0) prime(vc, vsc);
    float acc[HC][8];
#pragma unroll
    for (int hh = 0; hh < HC; hh++)
#pragma unroll
      for (int i = 0; i < 8; i++) acc[hh][i] = 0.0f;
    for (int t0 = 0; t0 < n_pass; t0 += NPF) {
#pragma unroll
      for (int u = 0; u < NPF; u++) {
        const int t = t0 + u;
        if (t < n_pass) {
          float v[8];
          unpack8(ring[u], v);
          if (t + NPF < n_pass) issue(vc, vsc, u, t + NPF);
          const int rl = 16 * t + rr;
          float pf[PW];
#pragma unroll
          for (int k4 = 0; k4 < PW; k4 += 4) {
            float4 pw = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (rl < n_rows) pw = *reinterpret_cast<const float4*>(sP + ((int64_t)ch * SL + rl) * PW + k4);
            pf[k4] = pw.x; pf[k4 + 1] = pw.y; pf[k4 + 2] = pw.z; pf[k4 + 3] = pw.w;
          }
#pragma unroll
          for (int hh = 0; hh < HC; hh++)
#pragma unroll
            for (int i = 0; i < 8; i++) acc[hh][i] = fmaf(pf[hh], v[i], acc[hh][i]);
        }
      }
    }
    // The wave's 4 row groups (rows of 16 lanes), then the 4 waves.  A transposing sum: the row-swap instructions of gfx950 turn
    // two registers into (row 0+1 | 2+3 of the first, of the second), then four into one whose row r holds the total of value
    // 4 q + r - (r0 + r1) + (r2 + r3) as a butterfly over lanes ^16, ^32 would give, in 1.5 instructions per value instead of
    // two LDS-crossbar permutes and two additions, and with one store per four values (the butterfly form took 3.8 of the
    // launch's 15 us at batch 8).
#pragma unroll
    for (int q4 = 0; q4 < 2 * HC; q4++) {
      float s2[2];
#pragma unroll
      for (int hf = 0; hf < 2; hf++) {
        const int n = 4 * q4 + 2 * hf;
        float x = acc[n >> 3][n & 7], y = acc[(n + 1) >> 3][(n + 1) & 7];
        row_swap16(x, y);
        s2[hf] = x + y;                 // rows: x0+x1 | y0+y1 | x2+x3 | y2+y3
      }
      row_swap32(s2[0], s2[1]);
      const float tot = s2[0] + s2[1];  // row r: total of value 4 q4 + r
      const int n = 4 * q4 + r;
      if (lane_on) sred[(w * HC + (n >> 3)) * 128 + d0 + (n & 7)] = tot;
    }
    __syncthreads();
    for (int o = tid; o < HC * hd; o += 256) {
      const int hh = o / hd, d = o % hd, h = h0 + hh;
      if (h < G) {
        const float A = (sred[(0 * HC + hh) * 128 + d] + sred[(1 * HC + hh) * 128 + d]) + (sred[(2 * HC + hh) * 128 + d] + sred[(3 * HC + hh) * 128 + d]);
        const float M = sML[h], Ls = sML[G + h];
        const int qh = g * G + h;
        if (n_active == 1) {
          p.out[(int64_t)seq * p.out_stride + qh * hd + d] = Ls > 0.0f ? A * (1.0f / Ls) : 0.0f;
        } else {
          float* pt = p.part + (((int64_t)seq * h_q_heads + qh) * h_n_splits + split) * (hd + 2);
          pt[d] = A;
          if (d == 0) { pt[hd] = M; pt[hd + 1] = Ls; }
        }
      }
    }
    __syncthreads();
  }
  timeline_stamp(p.timeline, 7);
}

// ---- the same split on the matrix cores: half-precision cache, 128-wide heads, groups of up to 16 query heads.
//      The VALU form above spends its time on instructions (8 conversions, 8 fused multiply-adds per head and a 4-step lane
//      reduction per head for every 16 bytes of K), one wave per SIMD.  Here a wave requests ALL its rows of the slice at once
//      (16-row tiles w, w + NW, ..: TPW tiles of K and of V, 16 KB in flight per wave) and the products are
//        S[row][head]  = K . q^T      v_mfma_f32_16x16x32_f16, K rows straight from memory as the A operand (lane = row,
//                                     16 bytes = 8 of the 32 contraction slots), q split hi + lo into two f16 planes in LDS;
//        O[head][dim] += P^T . V      the result registers of the first product (lane = head, 4 rows each of two tiles) ARE
//                                     the A operand of a 32-row step; P is scaled by 1024 and split hi + lo (its low part
//                                     stays clear of the f16 subnormal range); V goes through LDS as it arrives (row-major,
//                                     16-byte stores) and comes back as 32-bit words = two neighbouring dims of one row, so
//                                     that one byte permute per word pair builds the operand of the even and of the odd dims.
//      Every wave keeps its own maximum and sum per head; the four waves meet once, in LDS, and the slice partial has the
//      same form as above.  Same contract and tolerance as the VALU kernels (1e-5 against the oracle). ----
constexpr int GM_LD = 136;                         // halfs per staged row (128 + pad: 16-byte aligned, 4 rows apart = 16 banks apart)
constexpr int GM_FIXED = 2 * 16 * GM_LD * 2 + 512 + 1024;  // q hi | q lo | new K,V row | per-wave maximum and sum
constexpr int gm_lds_bytes(int tpw, int nw) { return GM_FIXED + nw * tpw * 16 * GM_LD * 2; }

// TPW 16-row tiles per wave, NW waves: 2 x 4 (slices of up to 128 rows) or 2 x 8 (up to 256: two waves per SIMD overlap each
// other's dependent LDS / matrix-core / soft-max chains)
// KV_T = int8_t: the codes become f16 exactly on their way into the operands (byte ^ 0x80 under a 0x64 exponent byte = 1152 + code,
// one packed subtraction: 1.25 instructions per element), the K row scale multiplies the finished score and the V row scale the
// soft-max weight before its hi + lo split, as in the VALU kernels (neural/neural.cl:2639-2640, 2683-2684).
__device__ __forceinline__ ph8_t gm_codes_to_halfs(uint32_t w0, uint32_t w1)
{
  typedef _Float16 gh2_t __attribute__((ext_vector_type(2)));
  const uint32_t x0 = w0 ^ 0x80808080u, x1 = w1 ^ 0x80808080u, K = 0x64646464u;
  const gh2_t off = {(_Float16)1152.0f, (_Float16)1152.0f};
  const gh2_t a = __builtin_bit_cast(gh2_t, __builtin_amdgcn_perm(K, x0, 0x04010400u)) - off, b = __builtin_bit_cast(gh2_t, __builtin_amdgcn_perm(K, x0, 0x04030402u)) - off;
  const gh2_t c = __builtin_bit_cast(gh2_t, __builtin_amdgcn_perm(K, x1, 0x04010400u)) - off, d = __builtin_bit_cast(gh2_t, __builtin_amdgcn_perm(K, x1, 0x04030402u)) - off;
  return ph8_t{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}
template <int TPW, int NW, typename KV_T>
__global__ __launch_bounds__(64 * NW) void attn_group_mfma_kernel(const int32_t* hpos, const float* hqkv, const float* htheta, const long long hqkv_stride,
                                                              const int hheads, const int hgeo, const int hsl, const AttnParams p)
{
  const unsigned long long tl0 = timeline_now();
  const int h_q_heads = hheads & 0xffff, h_kv_heads = hheads >> 16, h_n_splits = hgeo & 0xffff;
  constexpr int hd = 128;
  constexpr bool I8 = sizeof(KV_T) == 1;
  extern __shared__ __align__(16) unsigned char glds[];
  _Float16* sqh = reinterpret_cast<_Float16*>(glds);
  _Float16* sql = sqh + 16 * GM_LD;
  _Float16* snew = sql + 16 * GM_LD;                           // [K | V][128] (int8: the codes as bytes, then the two row scales at byte 256)
  float* sML = reinterpret_cast<float*>(snew + 256);           // [wave][head][maximum, sum]
  constexpr int REGION = TPW * 16 * GM_LD * 2;                 // bytes of a wave's V tiles (later: its [head][128] float sums)
  const int G = h_q_heads / h_kv_heads;
  const int split = blockIdx.x % h_n_splits, g = blockIdx.x / h_n_splits, seq = blockIdx.y;
  const int pos = hpos[seq];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, n16 = lane & 15, kg = lane >> 4;
  const int qw = h_q_heads * hd, kw = h_kv_heads * hd;
  const float* row = hqkv + (int64_t)seq * hqkv_stride;
  // the group's q pairs and frequencies do not depend on the position: requested behind it, before anything waits
  float qx0[2], qx1[2], qth[2];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int e = tid + 64 * NW * u, h = min(e >> 6, G - 1), i = e & 63;
    const float* qh = row + (g * G + h) * hd;
    qx0[u] = qh[2 * i]; qx1[u] = qh[2 * i + 1]; qth[u] = htheta ? htheta[i] : 0.0f;
  }
  const int SL = hsl, base = split * SL;
  const int64_t cache_seq = seq * p.seq_mul + p.seq0;
  KV_T* kc = reinterpret_cast<KV_T*>(p.kc) + cache_seq * p.seq_elems + p.layer_off + (int64_t)g * p.max_ctx * hd;
  KV_T* vc = reinterpret_cast<KV_T*>(p.vc) + cache_seq * p.seq_elems + p.layer_off + (int64_t)g * p.max_ctx * hd;
  float* ksc = nullptr; float* vsc = nullptr;
  if (I8) { const int64_t r0 = cache_seq * p.seq_rows + p.layer_row_off + (int64_t)g * p.max_ctx; ksc = p.ksc + r0; vsc = p.vsc + r0; }
  // contraction slots of a lane group: half cache dims 32 s + 8 kg .., int8 cache dims 32 kg + 8 s .. (a lane's 32 codes of a row are
  // two 16-byte requests)
  constexpr int KCH = I8 ? 2 : 4;          // 16-byte requests per lane and K tile
  // The wave's first K tile is requested before the position is known (its rows exist whatever the position: the slice lies
  // inside the cache; rows past the live range are masked), so the stream starts while the position is still on its way.
  uint4 kreg[TPW][4], vreg[TPW][4];
  {
    const int j = min(base + 16 * w + n16, p.max_ctx - 1);
#pragma unroll
    for (int s4 = 0; s4 < KCH; s4++) kreg[0][s4] = *reinterpret_cast<const uint4*>(kc + (int64_t)j * hd + (I8 ? 32 * kg + 16 * s4 : 32 * s4 + 8 * kg));
  }
  const LiveRows lr = live_rows(p, pos);
  const int len = lr.len, j_start = lr.j_start, slot = lr.slot;
  const int s_begin = max(j_start, base), s_end = min(len, base + SL);
  if (s_begin >= s_end) return;   // whole work-group leaves together, before any barrier
  const int s_first = j_start / SL, s_last = (len - 1) / SL;
  const int n_active = s_last - s_first + 1;

  // the work-group whose slice holds `pos` appends the new row (wave 0, one half-wave each for K and V): its raw elements are
  // requested here, in front of the cached rows (requests return in order)
  const bool owns_new = !p.appended && slot >= s_begin && slot < s_end;
  float nraw[4] = {0.0f, 0.0f, 0.0f, 0.0f}, nth[2] = {0.0f, 0.0f};
  if (owns_new && w == 0) {
    const int l32 = lane & 31, is_v = lane >> 5, e0 = 4 * l32;
    const float* src = row + qw + (is_v ? kw : 0) + g * hd + e0;
#pragma unroll
    for (int i = 0; i < 4; i++) nraw[i] = src[i];
    if (htheta) { nth[0] = htheta[e0 >> 1]; nth[1] = htheta[(e0 >> 1) + 1]; }
  }
  // int8: the scales of the rows whose scores this lane will hold (rows 4 kg .. 4 kg + 3 of every tile), in front of the rows
  float ks4[TPW][4], vs4[TPW][4];
#pragma unroll
  for (int t = 0; t < TPW; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int j = min(base + 16 * (w + NW * t) + 4 * kg + i, s_end - 1);
      ks4[t][i] = I8 ? ksc[j] : 1.0f; vs4[t][i] = I8 ? vsc[j] : 1.0f;
    }
  // every other row of the wave's tiles, K first (the first product starts while V is still on its way).
  // Rows past the live range repeat its last row and are masked below.
#pragma unroll
  for (int t = 1; t < TPW; t++) {
    const int j = min(base + 16 * (w + NW * t) + n16, s_end - 1);
#pragma unroll
    for (int s4 = 0; s4 < KCH; s4++) kreg[t][s4] = *reinterpret_cast<const uint4*>(kc + (int64_t)j * hd + (I8 ? 32 * kg + 16 * s4 : 32 * s4 + 8 * kg));
  }
  // V rows as they lie in memory: half cache 4 rows x 256 bytes per request, int8 cache 8 rows x 128 bytes
  constexpr int VCH = I8 ? 2 : 4, VROWS = I8 ? 8 : 4;
  const int vrow = I8 ? lane >> 3 : kg, vcol = I8 ? 16 * (lane & 7) : 8 * n16;
#pragma unroll
  for (int t = 0; t < TPW; t++)
#pragma unroll
    for (int i = 0; i < VCH; i++) {
      const int j = min(base + 16 * (w + NW * t) + VROWS * i + vrow, s_end - 1);
      vreg[t][i] = *reinterpret_cast<const uint4*>(vc + (int64_t)j * hd + vcol);
    }
  timeline_put(p.timeline, 0, tl0);
  timeline_stamp(p.timeline, 1);

  // rotated q of the group's heads as two f16 planes in LDS (wave w takes heads w, w + NW, ..; rows G .. 15 are zero)
#pragma unroll
  for (int u = 0; u < 16 / NW; u++) {
    const int h = w + NW * u, i = lane;
    _Float16 h0 = 0, h1 = 0, l0 = 0, l1 = 0;
    if (h < G) {
      float x0, x1, th;
      if (u < 2) { x0 = qx0[u]; x1 = qx1[u]; th = qth[u]; }
      else { const float* qh = row + (g * G + h) * hd; x0 = qh[2 * i]; x1 = qh[2 * i + 1]; th = htheta ? htheta[i] : 0.0f; }
      if (htheta) {
        float sn, cs; sincosf((float)pos * th, &sn, &cs);
        const float y0 = cs * x0 - sn * x1, y1 = sn * x0 + cs * x1;
        x0 = y0; x1 = y1;
      }
      split_f16(x0, h0, l0); split_f16(x1, h1, l1);
    }
    sqh[h * GM_LD + 2 * i] = h0; sqh[h * GM_LD + 2 * i + 1] = h1;
    sql[h * GM_LD + 2 * i] = l0; sql[h * GM_LD + 2 * i + 1] = l1;
  }
  // the new row: rotated, rounded to the cache's precision (int8: quantised, neural/neural.cl:2501-2580), stored, and kept in LDS for
  // this work-group's own products (its requests for that row went out before the store)
  if (owns_new && w == 0) {
    const int l32 = lane & 31, is_v = lane >> 5, e0 = 4 * l32;
    KV_T* dst = (is_v ? vc : kc) + (int64_t)slot * hd;
    float v4[4];
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      float x0 = nraw[i], x1 = nraw[i + 1];
      if (htheta && !is_v) {
        float sn, cs; sincosf((float)pos * nth[i >> 1], &sn, &cs);
        const float y0 = cs * x0 - sn * x1, y1 = sn * x0 + cs * x1;
        x0 = y0; x1 = y1;
      }
      v4[i] = x0; v4[i + 1] = x1;
    }
    if constexpr (I8) {
      const float scale = quantise_row_i8<4>(v4);
      int8_t* sb = reinterpret_cast<int8_t*>(snew);
#pragma unroll
      for (int i = 0; i < 4; i++) { dst[e0 + i] = (int8_t)v4[i]; sb[is_v * 128 + e0 + i] = (int8_t)v4[i]; }
      if (l32 == 0) { (is_v ? vsc : ksc)[slot] = scale; reinterpret_cast<float*>(snew + 128)[is_v] = scale; }
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const __half r = __float2half_rn(v4[i]);
        dst[e0 + i] = r; snew[is_v * 128 + e0 + i] = __builtin_bit_cast(_Float16, r);
      }
    }
  }
  __syncthreads();
  timeline_stamp(p.timeline, 4);

  ph8_t qh8[4], ql8[4];
#pragma unroll
  for (int s4 = 0; s4 < 4; s4++) {
    qh8[s4] = *reinterpret_cast<const ph8_t*>(sqh + n16 * GM_LD + (I8 ? 32 * kg + 8 * s4 : 32 * s4 + 8 * kg));
    ql8[s4] = *reinterpret_cast<const ph8_t*>(sql + n16 * GM_LD + (I8 ? 32 * kg + 8 * s4 : 32 * s4 + 8 * kg));
  }
  if (owns_new) {
    // the new row from LDS in place of what memory held; rows past the live range may be memory that was never written (the
    // new row's slot before this step): their V registers are cleared, 0 x NaN would poison the sums
    const int rs = slot - base;
#pragma unroll
    for (int t = 0; t < TPW; t++) {
      const int r0 = 16 * (w + NW * t);
      if (rs >= r0 && rs < r0 + 16) {
        const unsigned char* sb = reinterpret_cast<const unsigned char*>(snew);
        if (n16 == rs - r0) {
#pragma unroll
          for (int s4 = 0; s4 < KCH; s4++) kreg[t][s4] = *reinterpret_cast<const uint4*>(sb + (I8 ? 32 * kg + 16 * s4 : 2 * (32 * s4 + 8 * kg)));
        }
#pragma unroll
        for (int i = 0; i < VCH; i++)
          if (VROWS * i + vrow == rs - r0) vreg[t][i] = *reinterpret_cast<const uint4*>(sb + (I8 ? 128 + vcol : 2 * (128 + vcol)));
        if (I8) {
#pragma unroll
          for (int i = 0; i < 4; i++)
            if (4 * kg + i == rs - r0) { ks4[t][i] = reinterpret_cast<const float*>(snew + 128)[0]; vs4[t][i] = reinterpret_cast<const float*>(snew + 128)[1]; }
        }
      }
#pragma unroll
      for (int i = 0; i < VCH; i++)
        if (base + r0 + VROWS * i + vrow >= s_end) vreg[t][i] = make_uint4(0u, 0u, 0u, 0u);
    }
  }

  // ---- scores of the wave's rows, maximum, weights ----
  typedef float gf4_t __attribute__((ext_vector_type(4)));
  gf4_t C[TPW];
#pragma unroll
  for (int t = 0; t < TPW; t++) {
    C[t] = gf4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s4 = 0; s4 < 4; s4++) {
      ph8_t a;
      if constexpr (I8) {
        const uint4 kq = kreg[t][s4 >> 1];
        a = (s4 & 1) ? gm_codes_to_halfs(kq.z, kq.w) : gm_codes_to_halfs(kq.x, kq.y);
      } else a = __builtin_bit_cast(ph8_t, kreg[t][s4]);
      C[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qh8[s4], C[t], 0, 0, 0);
      C[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, ql8[s4], C[t], 0, 0, 0);
    }
  }
  // lane (n16, kg) holds head n16 of rows 4 kg .. 4 kg + 3 of every tile
  float m_w = -1e30f;
  bool ok[TPW][4];
#pragma unroll
  for (int t = 0; t < TPW; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int j = base + 16 * (w + NW * t) + 4 * kg + i;
      float sc = C[t][i] * (I8 ? ks4[t][i] * p.inv_sqrt : p.inv_sqrt);
      if (p.softcap > 0.0f) sc = p.softcap * tanhf(sc / p.softcap);
      ok[t][i] = j >= s_begin && j < s_end;
      C[t][i] = sc;
      if (ok[t][i]) m_w = fmaxf(m_w, sc);
    }
  m_w = fmaxf(m_w, __shfl_xor(m_w, 16, 64));
  m_w = fmaxf(m_w, __shfl_xor(m_w, 32, 64));
  float l_w = 0.0f;
#pragma unroll
  for (int t = 0; t < TPW; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) { C[t][i] = ok[t][i] ? expf(C[t][i] - m_w) : 0.0f; l_w += C[t][i]; }
  l_w += __shfl_xor(l_w, 16, 64);
  l_w += __shfl_xor(l_w, 32, 64);
  timeline_stamp(p.timeline, 5);

  // ---- value sums ----
  unsigned char* region = glds + GM_FIXED + w * REGION;
  _Float16* sV = reinterpret_cast<_Float16*>(region);
#pragma unroll
  for (int t = 0; t < TPW; t++)
#pragma unroll
    for (int i = 0; i < VCH; i++) {
      if constexpr (I8) {
        const uint4 vq = vreg[t][i];
        _Float16* dstv = sV + (16 * t + 8 * i + vrow) * GM_LD + vcol;
        *reinterpret_cast<ph8_t*>(dstv) = gm_codes_to_halfs(vq.x, vq.y);
        *reinterpret_cast<ph8_t*>(dstv + 8) = gm_codes_to_halfs(vq.z, vq.w);
      } else *reinterpret_cast<uint4*>(sV + (16 * t + 4 * i + kg) * GM_LD + 8 * n16) = vreg[t][i];
    }
  gf4_t Oe[4], Oo[4];
#pragma unroll
  for (int u = 0; u < 4; u++) { Oe[u] = gf4_t{0.0f, 0.0f, 0.0f, 0.0f}; Oo[u] = gf4_t{0.0f, 0.0f, 0.0f, 0.0f}; }
#pragma unroll
  for (int b = 0; b < TPW / 2; b++) {
    // contraction slot e of this lane group = row 4 kg + (e & 3) of tile 2 b + (e >> 2), in both operands
    ph8_t ph, pl;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int t = 2 * b + (e >> 2), i = e & 3;
      const float pe = I8 ? (ok[t][i] ? C[t][i] * vs4[t][i] : 0.0f) : C[t][i];      // (a dead row's scale is whatever memory holds)
      _Float16 hv, lv; split_f16(pe * 1024.0f, hv, lv); ph[e] = hv; pl[e] = lv;
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      uint32_t wv[8];
#pragma unroll
      for (int e = 0; e < 8; e++)
        wv[e] = *reinterpret_cast<const uint32_t*>(sV + (16 * (2 * b + (e >> 2)) + 4 * kg + (e & 3)) * GM_LD + 32 * u + 2 * n16);
      uint4 va, vb;       // column n16 of the even dims 32 u + 2 n16 and of the odd dims 32 u + 2 n16 + 1
      va.x = __builtin_amdgcn_perm(wv[1], wv[0], 0x05040100u); vb.x = __builtin_amdgcn_perm(wv[1], wv[0], 0x07060302u);
      va.y = __builtin_amdgcn_perm(wv[3], wv[2], 0x05040100u); vb.y = __builtin_amdgcn_perm(wv[3], wv[2], 0x07060302u);
      va.z = __builtin_amdgcn_perm(wv[5], wv[4], 0x05040100u); vb.z = __builtin_amdgcn_perm(wv[5], wv[4], 0x07060302u);
      va.w = __builtin_amdgcn_perm(wv[7], wv[6], 0x05040100u); vb.w = __builtin_amdgcn_perm(wv[7], wv[6], 0x07060302u);
      const ph8_t a8 = __builtin_bit_cast(ph8_t, va), b8 = __builtin_bit_cast(ph8_t, vb);
      Oe[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ph, a8, Oe[u], 0, 0, 0);
      Oe[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pl, a8, Oe[u], 0, 0, 0);
      Oo[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ph, b8, Oo[u], 0, 0, 0);
      Oo[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pl, b8, Oo[u], 0, 0, 0);
    }
  }
  timeline_stamp(p.timeline, 6);
  // ---- meeting of the waves: lane (n16, kg) holds heads 4 kg .. 4 kg + 3, dims 32 u + 2 n16 (+ 1) ----
  float* sO = reinterpret_cast<float*>(region);       // [head][128], over the wave's own V tiles (all read by now)
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (4 * kg + i < G) {
#pragma unroll
      for (int u = 0; u < 4; u++) *reinterpret_cast<float2*>(sO + (4 * kg + i) * 128 + 32 * u + 2 * n16) = make_float2(Oe[u][i], Oo[u][i]);
    }
  if (kg == 0) { sML[(w * 16 + n16) * 2] = m_w; sML[(w * 16 + n16) * 2 + 1] = l_w; }
  __syncthreads();
  for (int o = tid; o < G * hd; o += 64 * NW) {
    const int h = o >> 7, d = o & 127;
    float mw[NW], lw[NW], ow[NW];
#pragma unroll
    for (int k = 0; k < NW; k++) {
      mw[k] = sML[(k * 16 + h) * 2]; lw[k] = sML[(k * 16 + h) * 2 + 1];
      ow[k] = reinterpret_cast<const float*>(glds + GM_FIXED + k * REGION)[h * 128 + d];
    }
    float M = mw[0];
#pragma unroll
    for (int k = 1; k < NW; k++) M = fmaxf(M, mw[k]);
    float A = 0.0f, Ls = 0.0f;
#pragma unroll
    for (int k4 = 0; k4 < NW; k4 += 4) {      // fixed order: groups of four waves
      float e[4];
#pragma unroll
      for (int k = 0; k < 4; k++) e[k] = lw[k4 + k] > 0.0f ? expf(mw[k4 + k] - M) : 0.0f;
      A += (ow[k4] * e[0] + ow[k4 + 1] * e[1]) + (ow[k4 + 2] * e[2] + ow[k4 + 3] * e[3]);
      Ls += (lw[k4] * e[0] + lw[k4 + 1] * e[1]) + (lw[k4 + 2] * e[2] + lw[k4 + 3] * e[3]);
    }
    A *= 1.0f / 1024.0f;
    const int qh = g * G + h;
    if (n_active == 1) {
      p.out[(int64_t)seq * p.out_stride + qh * hd + d] = Ls > 0.0f ? A * (1.0f / Ls) : 0.0f;
    } else {
      float* pt = p.part + (((int64_t)seq * h_q_heads + qh) * h_n_splits + split) * (hd + 2);
      pt[d] = A;
      if (d == 0) { pt[hd] = M; pt[hd + 1] = Ls; }
    }
  }
  timeline_stamp(p.timeline, 7);
}

// ---- merge of the split partials: one work-group per query head.  Four quarter-groups of head_dim threads each take every
//      fourth slice (all their loads go out together: one round trip for up to 32 slices per quarter), fold them with a running
//      maximum, and meet in LDS. ----
template <int MR, bool PLANES>      // slices per quarter and round trip: 12, or 32 for long caches (130k rows = 508 slices: 4 dependent rounds instead of 11)
__global__ __launch_bounds__(512) void attn_merge_kernel(const int32_t* hpos, const float* hpart, float* hout, const long long hout_stride,
                                                         const int hheads, const int hgeo, const int hsl, const std::conditional_t<PLANES, PlanesParams, AttnParams> p)
{
  const int h_q_heads = hheads & 0xffff, h_n_splits = hgeo & 0xffff, h_hd = hgeo >> 16;     // (preloaded leading arguments, as in the split kernels)
  const int qh = blockIdx.x, seq = blockIdx.y;
  const int hd = h_hd;
  __shared__ float qA[4][128], qM[4], qL[4];
  const int quarter = threadIdx.x >> 7, d = threadIdx.x & 127;
  // Without a sliding window the first live slice is slice 0 whatever the position: the first round of partials (4 MR slices) is
  // requested before the position has arrived and masked by the slice count afterwards (a partial past the live range is
  // whatever an earlier step left there: it is selected away, never used in arithmetic).
  const bool ahead = p.window <= 0 && d < hd;
  const float* pt0 = hpart + ((int64_t)seq * h_q_heads + qh) * h_n_splits * (hd + 2);
  float v[MR], ms[MR], ls[MR];
  if (ahead) {
#pragma unroll
    for (int u = 0; u < MR; u++) {
      const float* ps = pt0 + (int64_t)min(quarter + 4 * u, h_n_splits - 1) * (hd + 2);
      v[u] = ps[d]; ms[u] = ps[hd]; ls[u] = ps[hd + 1];
    }
  }
  const LiveRows lr = live_rows(p, hpos[seq]);
  const int s_first = lr.j_start / hsl, s_last = (lr.len - 1) / hsl;
  const int n_active = s_last - s_first + 1;
  if (n_active == 1) return;                       // the split kernel already wrote the final row
  const float* pt = pt0 + (int64_t)s_first * (hd + 2);
  float A = 0.0f, L = 0.0f, M = -1e30f;
  if (d < hd) {
    for (int s0 = quarter; s0 < n_active; s0 += 4 * MR) {
      if (!(ahead && s0 == quarter)) {
#pragma unroll
        for (int u = 0; u < MR; u++) {
          const float* ps = pt + (int64_t)min(s0 + 4 * u, n_active - 1) * (hd + 2);
          v[u] = ps[d]; ms[u] = ps[hd]; ls[u] = ps[hd + 1];
        }
      }
#pragma unroll
      for (int u = 0; u < MR; u++) {
        if (s0 + 4 * u < n_active && ls[u] > 0.0f) {
          const float mn = fmaxf(M, ms[u]), c0 = expf(M - mn), c1 = expf(ms[u] - mn);
          A = fmaf(v[u], c1, A * c0); L = fmaf(ls[u], c1, L * c0); M = mn;
        }
      }
    }
    qA[quarter][d] = A;
    if (d == 0) { qM[quarter] = M; qL[quarter] = L; }
  }
  __syncthreads();
  if (quarter == 0 && d < hd) {
    const float Mx = fmaxf(fmaxf(qM[0], qM[1]), fmaxf(qM[2], qM[3]));
    float At = 0.0f, Lt = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const float e = qL[k] > 0.0f ? expf(qM[k] - Mx) : 0.0f;
      At = fmaf(qA[k][d], e, At); Lt = fmaf(qL[k], e, Lt);
    }
    const float y = Lt > 0.0f ? At * (1.0f / Lt) : 0.0f;
    if constexpr (PLANES) out_plane(p.planes, p.planes_q8, seq, qh * hd + d, h_q_heads * hd, y);
    else hout[(int64_t)seq * hout_stride + qh * hd + d] = y;
  }
}

// ---- short caches: one work-group per (split, QUERY head).  The G heads of a group each re-read the slice (from
//      L2: their work-groups are numbered so that they land on the same XCD), but no work-group loops over heads:
//      with one wave per SIMD that loop is a chain of dependent DPP/exp/LDS latencies and dominated the step.
//      Running state lives in registers; LDS is used once, for the meeting of the groups of 16 lanes. ----
// What bounds it is round trips to memory, one after another: the step's q | k | v, the frequencies and the first 64 or 128 rows of the slice are
// requested unconditionally and before anything waits, the rows before the position has arrived (a slice begins where it begins unless a
// sliding window cuts it; rows past the live range are read as they lie and dropped).  With requests under branches and rows turned to floats
// beside them it was four to eight round trips: 28 / 4 heads of 128, 600 float rows 10.0 us a launch (7.8 here), eight sequences of 200 half
// rows 15.5 (8.9), 9 / 3 heads of 64 and 100 float rows 7.4 (4.8).
// The leading scalar arguments are all that these first requests need: they arrive preloaded in scalar registers (see the Makefile), and
// the rest of the parameter block is fetched while the requests are on their way.  hk, hv: this layer's keys and values of activation row 0's
// sequence, hseq_planes: planes of max_ctx rows from one sequence to the next (0: all activation rows share one), hheads = query heads | KV heads << 16, hgeo =
// slices | head width << 16, hsl = rows of a slice.
// QN: q and k carry an RMS norm over their whole rows, whose first 2048 elements are among the first requests (16 / 16 heads of 128: 8.7 -> 8.1 us a launch).
// 16 lanes hold a row: of NV x 16 VW elements lane l has VW from 16 VW i + VW l on.  What is not waiting is instructions, one wave a SIMD: with
// 32 lanes a row, sums of five steps and two scalar reads, 64 rows cost 1.5 us (0.5 here); sine and cosine are worked out once a wave
// and not once a group, the exponentials of the meeting once a lane.  More waves (8, 16 a work-group) took longer to start and to meet
// (100 half rows of 128: 5.5 us with four, 6.3, 9.6; 200: 7.2, 7.2, 9.6).  NCH: chunks of 64 rows on their way at once.
// MODE: a step's rows as they are, with the norms of whole q and k rows, or a prompt's rows whose results leave as planes.
constexpr int HEAD_PLAIN = 0, HEAD_NORMED = 1, HEAD_PLANES = 2;
// (a trait, and no enumerator in the kernel's signature: an enumeration without a name is numbered differently for host and device, and so is the kernel's)
template <int MODE> struct HeadParams { using type = AttnParams; };
template <> struct HeadParams<HEAD_PLANES> { using type = PlanesParams; };
template <int VW, int NV, typename KV_T, int NCH, int MODE>
__global__ __launch_bounds__(256) void attn_split_head_kernel(const int32_t* hpos, const float* hqkv, const void* hk, const void* hv, const int hqkv_stride,
                                                                  const int hheads, const int hgeo, const int hsl, const int hmax_ctx, const int hseq_planes, const typename HeadParams<MODE>::type p)
{
  constexpr bool QN = MODE == HEAD_NORMED;
  constexpr int DS = VW * NV, NG = 16;         // groups of 16 lanes, four waves: row j of the slice belongs to group j % NG
  const unsigned long long tl0 = timeline_now();
  const int q_heads = hheads & 0xffff, kv_heads = hheads >> 16, n_splits = hgeo & 0xffff, hd = hgeo >> 16;
  const int G = q_heads / kv_heads;
  // linear id = item_lo + 8 * (h + G * item_hi), item = split + n_splits * kv_head: consecutive ids rotate over the XCDs, and a sequence
  // starts on the XCD behind the last one's (four items a sequence would leave half of the chip idle)
  const int L = blockIdx.x, seq = blockIdx.y, n_items = n_splits * kv_heads;
  const int item = ((L - seq * n_items) & 7) + 8 * ((L >> 3) / G), h = (L >> 3) % G;
  if (item >= n_items) return;
  const int split = item % n_splits, g = item / n_splits;
  // (a vector load: a scalar one would be waited for together with the parameter block, in front of the requests for the rows)
  int lane0 = 0;
  asm volatile("" : "+v"(lane0));
  const int pos_v = hpos[seq + lane0];
  const int tid = threadIdx.x, grp = tid >> 4, l16 = tid & 15;
  const int qw = q_heads * hd, kw = kv_heads * hd;
  int dc[NV]; bool in_row[NV];                // (lanes beyond the head width read its last elements; the values are dropped)
#pragma unroll
  for (int i = 0; i < NV; i++) { const int d = 16 * VW * i + VW * l16; in_row[i] = d < hd; dc[i] = min(d, hd - VW); }
  const float* row = hqkv + (int64_t)seq * hqkv_stride;
  using FV = row_vec<VW, float>;
  using CV = row_vec<VW, KV_T>;
  const float* const qp = row + (g * G + h) * hd; const float* const kp = row + qw + g * hd; const float* const vp = kp + kw;
  FV qv[NV], kv[NV], vv[NV];
#pragma unroll
  for (int i = 0; i < NV; i++) { qv[i] = *reinterpret_cast<const FV*>(qp + dc[i]); kv[i] = *reinterpret_cast<const FV*>(kp + dc[i]); vv[i] = *reinterpret_cast<const FV*>(vp + dc[i]); }

  float tq[QN ? 8 : 1], tk[QN ? 8 : 1];      // the first 2048 elements of the whole rows of q and k
  if constexpr (QN) {
#pragma unroll
    for (int u = 0; u < 8; u++) { tq[u] = row[min(tid + 256 * u, qw - 1)]; tk[u] = row[qw + min(tid + 256 * u, kw - 1)]; }
  }

  const int64_t plane_row = ((int64_t)seq * hseq_planes + g) * hmax_ctx;
  KV_T* const kc = reinterpret_cast<KV_T*>(const_cast<void*>(hk)) + plane_row * hd;
  KV_T* const vc = reinterpret_cast<KV_T*>(const_cast<void*>(hv)) + plane_row * hd;
  // int8 cache: codes enter the dot products as they are; the K row scale multiplies the finished score and the V row
  // scale the softmax weight (neural/neural.cl:2639-2640, 2683-2684), so nothing is dequantised per element
  constexpr bool I8 = sizeof(KV_T) == 1;
  constexpr int PCH = 4;
  struct Chunk { CV k[PCH][NV], v[PCH][NV]; float ks[PCH], vs[PCH]; };
  Chunk ch[NCH];
  auto load_k = [&](Chunk& ch, int j0, int last) {
#pragma unroll
    for (int c = 0; c < PCH; c++)
#pragma unroll
      for (int i = 0; i < NV; i++) ch.k[c][i] = *reinterpret_cast<const CV*>(kc + (int64_t)min(j0 + NG * c, last) * hd + dc[i]);
  };
  auto load_v = [&](Chunk& ch, int j0, int last) {
#pragma unroll
    for (int c = 0; c < PCH; c++)
#pragma unroll
      for (int i = 0; i < NV; i++) ch.v[c][i] = *reinterpret_cast<const CV*>(vc + (int64_t)min(j0 + NG * c, last) * hd + dc[i]);
  };
  const int split_len = hsl & 0xffff, row0 = split * split_len;
  const bool ahead = !(hsl >> 16);                               // no sliding window
  const int last0 = ahead ? min(row0 + split_len, hmax_ctx) - 1 : row0;   // (a window's first rows are asked for again once the position is known)
#pragma unroll
  for (int n = 0; n < NCH; n++) load_k(ch[n], row0 + grp + n * NG * PCH, last0);
  const float th = (p.theta ? p.theta : row)[min(tid & 63, (hd >> 1) - 1)];      // lane a turns pair a (no rotation: any readable address)
#pragma unroll
  for (int n = 0; n < NCH; n++) load_v(ch[n], row0 + grp + n * NG * PCH, last0);
  float* const ksc = p.ksc + plane_row + p.scale_row0; float* const vsc = p.vsc + plane_row + p.scale_row0;      // (int8 only)
  auto load_scales = [&](Chunk& ch, int j0, int last) {
    if constexpr (I8) {
#pragma unroll
      for (int c = 0; c < PCH; c++) { const int j = min(j0 + NG * c, last); ch.ks[c] = ksc[j]; ch.vs[c] = vsc[j]; }
    }
  };
#pragma unroll
  for (int n = 0; n < NCH; n++) load_scales(ch[n], row0 + grp + n * NG * PCH, last0);
  FV qg[NV], kg[NV];
  if constexpr (QN) {
#pragma unroll
    for (int i = 0; i < NV; i++) { qg[i] = *reinterpret_cast<const FV*>(p.qn_gain + (g * G + h) * hd + dc[i]); kg[i] = *reinterpret_cast<const FV*>(p.kn_gain + g * hd + dc[i]); }
  }
  __builtin_amdgcn_sched_barrier(0);      // (nothing waits before the last of these requests is out)
  const int pos = __builtin_amdgcn_readfirstlane(pos_v);
  const LiveRows lr = live_rows(p, pos);
  const int len = lr.len, j_start = lr.j_start, slot = lr.slot;
  const int s_begin = max(j_start, row0), s_end = min(len, row0 + split_len);
  if (s_begin >= s_end) return;   // whole work-group leaves together, before any barrier
  const int s_first = j_start / split_len, s_last = (len - 1) / split_len;
  const int n_active = s_last - s_first + 1;
  timeline_put(p.timeline, 0, tl0);
  timeline_stamp(p.timeline, 1);
  auto load_chunk = [&](Chunk& ch, int j0) { load_k(ch, j0, s_end - 1); load_v(ch, j0, s_end - 1); load_scales(ch, j0, s_end - 1); };
  if (!ahead)
#pragma unroll
    for (int n = 0; n < NCH; n++) load_chunk(ch[n], s_begin + grp + n * NG * PCH);
  const bool owns_new = !p.appended && slot >= s_begin && slot < s_end;
  const int skip = owns_new ? slot : -1;        // the row being appended: what lies in the cache there is stale

  // Full-width RMSNorm of q and k (neural/neuralpretrained.pas:16511-16530) folded into this kernel: every work-group
  // sums the squares of the whole q and k rows itself (same order as the stand-alone kernel: strided per thread, wave
  // totals, (w0 + w1) + (w2 + w3)) and scales the elements it reads.
  float inv_q = 1.0f, inv_k = 1.0f;
  if constexpr (QN) {
    __shared__ float nred[8];
    {
      float sq = 0.0f, sk = 0.0f;
#pragma unroll
      for (int u = 0; u < 8; u++) { if (tid + 256 * u < qw) sq = fmaf(tq[u], tq[u], sq); if (tid + 256 * u < kw) sk = fmaf(tk[u], tk[u], sk); }
      for_strided8(row, tid + 2048, qw, 256, [&](float v, int) { sq = fmaf(v, v, sq); });
      for_strided8(row + qw, tid + 2048, kw, 256, [&](float v, int) { sk = fmaf(v, v, sk); });
      sq = wave_sum(sq); sk = wave_sum(sk);
      if ((tid & 63) == 63) { nred[tid >> 6] = sq; nred[4 + (tid >> 6)] = sk; }
    }
    __syncthreads();
    inv_q = 1.0f / sqrtf(((nred[0] + nred[1]) + (nred[2] + nred[3])) / (float)qw + p.qk_eps);
    inv_k = 1.0f / sqrtf(((nred[4] + nred[5]) + (nred[6] + nred[7])) / (float)kw + p.qk_eps);
  }
  float rs[DS / 2], rc[DS / 2];
  {
    float sn = 0.0f, cs = 1.0f;
    if (p.theta) sincosf((float)pos * th, &sn, &cs);       // (one pair a lane, and from there to the lanes that need it)
#pragma unroll
    for (int i = 0; i < DS / 2; i++) {
      const int from = (dc[2 * i / VW] + 2 * i % VW) << 1;       // 4 bytes a lane
      rs[i] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(from, __builtin_bit_cast(int, sn)));
      rc[i] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(from, __builtin_bit_cast(int, cs)));
    }
  }
  // raw elements -> RMSNorm gain of QN -> optional rotation
  auto finish_rot = [&](const FV (&raw)[NV], const FV (&gain)[NV], float inv, float (&o)[DS]) {
#pragma unroll
    for (int i = 0; i < DS; i += 2) {
      const int n = i / VW, e = i % VW;
      float x0 = raw[n][e], x1 = raw[n][e + 1];
      if constexpr (QN) { x0 = gain[n][e] * (x0 * inv); x1 = gain[n][e + 1] * (x1 * inv); }
      if (!in_row[n]) x0 = x1 = 0.0f;
      o[i] = x0; o[i + 1] = x1;
      if (p.theta) { o[i] = rc[i / 2] * x0 - rs[i / 2] * x1; o[i + 1] = rs[i / 2] * x0 + rc[i / 2] * x1; }
    }
  };
  float q[DS], acc[DS], m = -1e30f, l = 0.0f;
  finish_rot(qv, qg, inv_q, q);
#pragma unroll
  for (int i = 0; i < DS; i++) acc[i] = 0.0f;
  // a lane's part of a score, VW elements a chain (one of 8 for two of 4: 2 % further from 64 bits)
  auto dot_of = [&](const float (&k)[DS]) {
    float d[NV];
#pragma unroll
    for (int n = 0; n < NV; n++) {
      d[n] = q[VW * n] * k[VW * n];
#pragma unroll
      for (int e = 1; e < VW; e++) d[n] = fmaf(q[VW * n + e], k[VW * n + e], d[n]);
    }
    return NV == 2 ? d[0] + d[NV - 1] : d[0];
  };
  auto score = [&](float dot, float k_scale) {
    const float s = row16_sum(dot) * (I8 ? k_scale * p.inv_sqrt : p.inv_sqrt);
    return p.softcap > 0.0f ? p.softcap * tanhf(s / p.softcap) : s;
  };
  // The work-group whose slice holds the new row has it in registers: its first group starts from it, and the group's first head appends it
  if (owns_new) {
    float knew[DS], vnew[DS], knew_s = 1.0f, vnew_s = 1.0f;
    finish_rot(kv, kg, inv_k, knew);
#pragma unroll
    for (int i = 0; i < DS; i++) vnew[i] = in_row[i / VW] ? vv[i / VW][i % VW] : 0.0f;
    if constexpr (I8) { knew_s = quantise_row_i8<DS, true>(knew); vnew_s = quantise_row_i8<DS, true>(vnew); }
    if (h == 0 && grp == 0) {
#pragma unroll
      for (int i = 0; i < DS; i++)
        if (in_row[i / VW]) {
          const int64_t at = (int64_t)slot * hd + dc[i / VW] + i % VW;
          if constexpr (I8) { kc[at] = (int8_t)knew[i]; vc[at] = (int8_t)vnew[i]; }
          else { kc[at] = kv_from_float<KV_T>(knew[i]); vc[at] = kv_from_float<KV_T>(vnew[i]); }
        }
      if constexpr (I8) if (l16 == 0) { ksc[slot] = knew_s; vsc[slot] = vnew_s; }
    }
    if constexpr (!I8)
#pragma unroll
      for (int i = 0; i < DS; i++) { knew[i] = kv_to_float<KV_T>(kv_from_float<KV_T>(knew[i])); vnew[i] = kv_to_float<KV_T>(kv_from_float<KV_T>(vnew[i])); }
    const float s = score(dot_of(knew), knew_s);
    if (grp == 0) {
      m = s; l = 1.0f;
#pragma unroll
      for (int i = 0; i < DS; i++) acc[i] = I8 ? vnew_s * vnew[i] : vnew[i];
    }
  }
  timeline_stamp_after(p.timeline, 4, q[0]);
  auto reduce_chunk = [&](const Chunk& ch, int j0) {
    float sc[PCH], cmax = -1e30f;
#pragma unroll
    for (int c = 0; c < PCH; c++) {
      float kf[DS];
#pragma unroll
      for (int i = 0; i < NV; i++) row_floats<VW, KV_T>(ch.k[c][i], kf + VW * i);
      sc[c] = row16_sum(dot_of(kf)) * (I8 ? ch.ks[c] * p.inv_sqrt : p.inv_sqrt);       // (q is 0 beyond the head width)
    }
    if (p.softcap > 0.0f) {
#pragma unroll
      for (int c = 0; c < PCH; c++) sc[c] = p.softcap * tanhf(sc[c] / p.softcap);
    }
    bool live[PCH];
#pragma unroll
    for (int c = 0; c < PCH; c++) {
      const int j = j0 + NG * c;
      live[c] = j < s_end && j != skip;
      if (!live[c]) sc[c] = -1e30f;           // (whatever a row that is not live holds ends here and at its values below)
      cmax = fmaxf(cmax, sc[c]);
    }
    const float mn = fmaxf(m, cmax), corr = expf(m - mn);
    float lsum = 0.0f;
#pragma unroll
    for (int i = 0; i < DS; i++) acc[i] *= corr;
#pragma unroll
    for (int c = 0; c < PCH; c++) {
      const float pj = live[c] ? expf(sc[c] - mn) : 0.0f;
      lsum += pj;
      const float pv = I8 ? (live[c] ? pj * ch.vs[c] : 0.0f) : pj;
      float vf[DS];
#pragma unroll
      for (int i = 0; i < NV; i++) row_floats<VW, KV_T>(live[c] ? ch.v[c][i] : CV{}, vf + VW * i);
#pragma unroll
      for (int i = 0; i < DS; i++) acc[i] = fmaf(pv, vf[i], acc[i]);
    }
    l = l * corr + lsum; m = mn;
  };
  for (int b = s_begin; b < s_end; b += NCH * NG * PCH) {
#pragma unroll
    for (int n = 0; n < NCH; n++)
      if (b + n * NG * PCH < s_end) {
        reduce_chunk(ch[n], b + grp + n * NG * PCH);
        if (b + (n + NCH) * NG * PCH < s_end) load_chunk(ch[n], b + grp + (n + NCH) * NG * PCH);
      }
  }

  // ---- meeting of the groups ----
  timeline_stamp(p.timeline, 5);
  __shared__ float sm[NG], sl[NG];
  __shared__ __attribute__((aligned(16))) float sacc[NG][16 * DS];
  if (l16 == 0) { sm[grp] = m; sl[grp] = l; }
#pragma unroll
  for (int i = 0; i < DS; i++) sacc[grp][16 * VW * (i / VW) + VW * l16 + i % VW] = acc[i];
  __syncthreads();
  if ((tid & ~63) < hd) {                                    // (whole waves)
    const int d = min(tid, hd - 1), lane = tid & 63;
    const float mw = lane < NG ? sm[lane] : -1e30f, lw = lane < NG ? sl[lane] : 0.0f;      // group `lane`'s maximum and sum
    const float M = lane_value(row16_max(mw), 0);      // (the groups are one row of lanes)
    const float ew = lw > 0.0f ? expf(mw - M) : 0.0f;
    // (four short sums: one of sixteen is up to 15 % further from 64 bits, 30 rows of 64 1.39e-7 instead of 1.16e-7)
    float Lp[4] = {0.0f, 0.0f, 0.0f, 0.0f}, Ap[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < NG; w++) {
      const float e = lane_value(ew, w);
      Lp[w & 3] = fmaf(lane_value(lw, w), e, Lp[w & 3]); Ap[w & 3] = fmaf(sacc[w][d], e, Ap[w & 3]);
    }
    const float Ls = (Lp[0] + Lp[1]) + (Lp[2] + Lp[3]), A = (Ap[0] + Ap[1]) + (Ap[2] + Ap[3]);
    const int qh = g * G + h;
    if (tid < hd && n_active == 1) {
      const float y = Ls > 0.0f ? A * (1.0f / Ls) : 0.0f;
      if constexpr (MODE == HEAD_PLANES) out_plane(p.planes, p.planes_q8, seq, qh * hd + d, q_heads * hd, y);
      else p.out[(int64_t)seq * p.out_stride + qh * hd + d] = y;
    } else if (tid < hd) {
      float* pt = p.part + (((int64_t)seq * p.q_heads + qh) * p.n_splits + split) * (hd + 2);
      if (p.merge_cnt) { part_store(pt + d, A); if (d == 0) { part_store(pt + hd, M); part_store(pt + hd + 1, Ls); } }
      else { pt[d] = A; if (d == 0) { pt[hd] = M; pt[hd + 1] = Ls; } }
    }
  }
  if (n_active > 1 && p.merge_cnt) merge_if_last(p, seq, g * G + h, s_first, n_active, seq * p.kv_heads * 8 + g * G + h);
  timeline_stamp(p.timeline, 7);
}

template <typename KV_T>
static int launch_split_head(const PlanesParams& p0, int n_seq, hipStream_t st)
{
  PlanesParams p = p0;
  const int G = p.q_heads / p.kv_heads;
  const int items = p.n_splits * p.kv_heads;
  const dim3 grid(8 * G * ((items + 7) / 8), n_seq);
  p.timeline = timeline_next((int)(grid.x * grid.y));
  const int hheads = p.q_heads | p.kv_heads << 16, hgeo = p.n_splits | p.hd << 16, hsl = p.split_len | (p.window > 0 ? 1 << 16 : 0);
  const int64_t seq_planes = p.seq_mul && n_seq > 1 ? p.seq_elems / ((int64_t)p.hd * p.max_ctx) : 0, qkv_stride = n_seq > 1 ? p.qkv_stride : 0;
  if (p.q_heads > 0xffff || p.kv_heads > 0x7fff || p.n_splits > 0xffff || p.split_len > 0xffff || seq_planes > 0x7fffffff || qkv_stride > 0x7fffffff)
    return set_error(CAI_ERR_UNSUPPORTED, "attention: %d query heads, %d slices of %d rows, rows of %lld", p.q_heads, p.n_splits, p.split_len, (long long)qkv_stride);
  if (p.hd > 128) return set_error(CAI_ERR_UNSUPPORTED, "attention: head_dim %d > 128", p.hd);
  const int64_t at = (p.seq0 * p.seq_elems + p.layer_off) * (int64_t)sizeof(KV_T);
  const void* hk = (const char*)p.kc + at; const void* hv = (const char*)p.vc + at;
  p.scale_row0 = p.seq0 * p.seq_rows + p.layer_row_off;
  auto put = [&](auto kern, const auto& params) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, p.pos, (const float*)p.qkv, hk, hv, (int)qkv_stride, hheads, hgeo, hsl, p.max_ctx, (int)seq_planes, params);
  };
  auto go = [&](auto vw, auto nv) {
    constexpr int VW = decltype(vw)::value, NV = decltype(nv)::value;
    // a slice of up to 64 rows is one chunk; longer ones have 128 rows on their way (256: 0.1 us less at 200 rows, 0.5 more at 100)
    constexpr int LONG = 2;
    auto of = [&](auto mode) {
      constexpr int MODE = decltype(mode)::value;
      const typename HeadParams<MODE>::type& q = p;
      if (p.split_len <= 64) put(attn_split_head_kernel<VW, NV, KV_T, 1, MODE>, q); else put(attn_split_head_kernel<VW, NV, KV_T, LONG, MODE>, q);
    };
    if (p.qn_gain) of(std::integral_constant<int, HEAD_NORMED>());
    else if (p.planes.hi) of(std::integral_constant<int, HEAD_PLANES>());
    else of(std::integral_constant<int, HEAD_PLAIN>());
  };
  using std::integral_constant;
  if (p.hd > 64) go(integral_constant<int, 4>(), integral_constant<int, 2>());       // (widths past 64 are whole fours, all are even)
  else if (p.hd % 4 == 0) go(integral_constant<int, 4>(), integral_constant<int, 1>());
  else go(integral_constant<int, 2>(), integral_constant<int, 2>());
  return CAI_OK;
}

template <typename KV_T, int NPF>
static void launch_group_t(const AttnParams& p0, const dim3 grid, size_t lds, int hc, hipStream_t st)
{
  AttnParams p = p0;
  p.timeline = timeline_next((int)(grid.x * grid.y));
  switch (hc) {
#define CAI_GROUP_ARGS p.pos, (const float*)p.qkv, p.theta, (long long)p.qkv_stride, p.q_heads | p.kv_heads << 16, p.n_splits | p.hd << 16, p.split_len, p
    case 1: hipLaunchKernelGGL((attn_group_kernel<1, KV_T, NPF>), grid, dim3(256), lds, st, CAI_GROUP_ARGS); break;
    case 2: hipLaunchKernelGGL((attn_group_kernel<2, KV_T, NPF>), grid, dim3(256), lds, st, CAI_GROUP_ARGS); break;
    case 3: hipLaunchKernelGGL((attn_group_kernel<3, KV_T, NPF>), grid, dim3(256), lds, st, CAI_GROUP_ARGS); break;
    case 4: hipLaunchKernelGGL((attn_group_kernel<4, KV_T, NPF>), grid, dim3(256), lds, st, CAI_GROUP_ARGS); break;
    case 5: hipLaunchKernelGGL((attn_group_kernel<5, KV_T, NPF>), grid, dim3(256), lds, st, CAI_GROUP_ARGS); break;
    case 6: hipLaunchKernelGGL((attn_group_kernel<6, KV_T, NPF>), grid, dim3(256), lds, st, CAI_GROUP_ARGS); break;
    case 7: hipLaunchKernelGGL((attn_group_kernel<7, KV_T, NPF>), grid, dim3(256), lds, st, CAI_GROUP_ARGS); break;
    default: hipLaunchKernelGGL((attn_group_kernel<8, KV_T, NPF>), grid, dim3(256), lds, st, CAI_GROUP_ARGS); break;
#undef CAI_GROUP_ARGS
  }
}

template <typename KV_T>
static int launch_group(const AttnParams& p, int n_seq, hipStream_t st)
{
  const int G = p.q_heads / p.kv_heads;
  constexpr int hc_max = 8;    // query heads held in registers per pass
  const int n_chunks = (G + hc_max - 1) / hc_max, hc = (G + n_chunks - 1) / n_chunks;
  const dim3 grid(p.n_splits * p.kv_heads, n_seq);
  const size_t lds = (size_t)(G * 128 + G * p.split_len + n_chunks * p.split_len * (hc > 4 ? 8 : 4) + 4 * hc * 128 + 2 * G) * sizeof(float);
  if (lds > 64 * 1024) return set_error(CAI_ERR_UNSUPPORTED, "attention: %d query heads per KV head need %zu bytes of LDS", G, lds);
  // Several work-groups per CU: a shallow load ring frees registers for more resident waves (5 instead of 3 per SIMD),
  // which hides the phase changes of one work-group behind the streaming of the others.  A grid of about one work-group
  // per CU has nothing to overlap with and keeps the deep ring.
  if ((int)(grid.x * grid.y) >= 3 * ctx().n_cu) launch_group_t<KV_T, 2>(p, grid, lds, hc, st);
  else launch_group_t<KV_T, (sizeof(KV_T) == 4 ? 4 : 8)>(p, grid, lds, hc, st);
  return CAI_OK;
}

// Which kernel attends: one work-group per (slice, query head), or per (slice, KV head) with the whole group of query heads, that one on vector
// instructions or on the matrix cores (half and int8 rows of 128; CAIHIP_ATTN_GROUP_MFMA=0 keeps the vector form).
enum { ATTN_PER_HEAD = 0, ATTN_GROUPED = 1, ATTN_GROUPED_CORES = 2 };
static int attn_form(const cai_kv_s* kv, int q_heads, int n_seq, int split_len, int n_splits, bool prompt_rows, bool normed)
{
  static const bool cores_on = []() { const char* e = getenv("CAIHIP_ATTN_GROUP_MFMA"); return !(e && e[0] == '0'); }();
  const int group_min = ctx().n_cu;   // smallest grid that fills the chip with one work-group per (slice, KV head)
  // (a cache short enough to be ONE slice may be up to 2048 rows long: the grouped kernel's per-slice score arrays in LDS are
  // sized for ordinary slices, the per-head kernel keeps its state in registers)
  if ((kv->head_dim & 7) != 0 || split_len > 256 || (int64_t)n_seq * kv->kv_heads * n_splits < group_min) return ATTN_PER_HEAD;
  const bool cores = cores_on && kv->dtype != CAI_KV_F32 && kv->head_dim == 128 && q_heads / kv->kv_heads <= 16;
  // Where both can run, the per-head kernel saves the merge launch, and the norm launch of normed q and k; the grouped one reads a row once for
  // all its heads.  us of a layer of a decoding step, per head minus grouped, least and most over 4 to 32 KV heads, one to eight sequences and
  // slices of 32 to 256 rows (one slice of 256: the same):
  //   float rows, and half and int8 rows of 64: up to 512 work-groups per head -8.9 .. +0.1 (one query head a KV head, two); half and int8 rows of 64 with a
  //     query head a KV head, up to 2048 -20 .. -0.1
  //   half and int8 rows of 128 (grouped: on the matrix cores), a query head a KV head: slices of up to 64 rows, 1024 work-groups -5.1 .. -0.1 (2048: -1.4 ..
  //     +0.4); int8 slices of 256, up to 2048, -2.8 .. +0.1; others -1.5 .. +3.5; two query heads a KV head -1.2 .. +2.6
  //   the same with normed q and k: up to 512 work-groups -5.2 .. +0.3, slices of 64 up to 2048 -6.1 .. -0.5, the others -2.1 .. +7.7
  const int64_t wgs = (int64_t)n_seq * q_heads * n_splits;
  const bool alone = q_heads == kv->kv_heads;         // heads that share nothing
  bool per_head;
  if (!cores) per_head = wgs <= 512 || (alone && kv->dtype != CAI_KV_F32 && wgs <= 2048);
  else if (normed) per_head = wgs <= 512 || (alone && split_len <= 64 && wgs <= 2048);
  else per_head = alone && (split_len <= 64 ? wgs <= 1024 : kv->dtype == CAI_KV_I8 && split_len > 128 && n_splits > 1 && wgs <= 2048);
  if (per_head && !prompt_rows && n_splits <= 16) return ATTN_PER_HEAD;
  return cores ? ATTN_GROUPED_CORES : ATTN_GROUPED;
}
template <typename KV_T>
static int launch_group_mfma(const AttnParams& p0, int n_seq, hipStream_t st)
{
  AttnParams p = p0;
  const dim3 grid(p.n_splits * p.kv_heads, n_seq);
  p.timeline = timeline_next((int)(grid.x * grid.y));
  if (p.q_heads > 0xffff || p.kv_heads > 0x7fff || p.n_splits > 0xffff) return set_error(CAI_ERR_UNSUPPORTED, "attention: %d query heads, %d slices", p.q_heads, p.n_splits);
  const int hheads = p.q_heads | p.kv_heads << 16, hgeo = p.n_splits | p.hd << 16;
#define CAI_GM_LAUNCH(TPWv, NWv) do { \
    static bool attr_done = false;      /* up to 80 KB of dynamic LDS */ \
    if (!attr_done) { CAI_HIP(hipFuncSetAttribute((const void*)attn_group_mfma_kernel<TPWv, NWv, KV_T>, hipFuncAttributeMaxDynamicSharedMemorySize, gm_lds_bytes(TPWv, NWv))); attr_done = true; } \
    hipLaunchKernelGGL((attn_group_mfma_kernel<TPWv, NWv, KV_T>), grid, dim3(64 * NWv), gm_lds_bytes(TPWv, NWv), st, p.pos, (const float*)p.qkv, p.theta, (long long)p.qkv_stride, hheads, hgeo, p.split_len, p); } while (0)
  // slices of up to 128 rows: four waves; longer ones: eight (32B shape at 8.2k rows, slices of 256: 177.5 tok/s with four waves
  // of four tiles, 180.8 with eight waves of two at batch 1; 693.7 against 698.0 at batch 8)
  if (p.split_len <= 128) CAI_GM_LAUNCH(2, 4);
  else CAI_GM_LAUNCH(2, 8);
#undef CAI_GM_LAUNCH
  return CAI_OK;
}

// Prompt ingestion: rotate the K rows of n_tok tokens at their positions and write K,V into sequence `seq`.
template <typename KV_T>
__device__ __forceinline__ void kv_append_row(const AttnParams& p)
{
  const int b = blockIdx.x;
  const float* row = p.qkv + (int64_t)b * p.qkv_stride;
  const int pos = p.pos[b], slot = live_rows(p, pos).slot;
  const int hd = p.hd, qw = p.q_heads * hd, kw = p.kv_heads * hd;
  KV_T* kc = reinterpret_cast<KV_T*>(p.kc) + (int64_t)p.seq0 * p.seq_elems + p.layer_off;
  KV_T* vc = reinterpret_cast<KV_T*>(p.vc) + (int64_t)p.seq0 * p.seq_elems + p.layer_off;
  for (int i = threadIdx.x; i < (kw >> 1); i += 256) {
    const int e = 2 * i, g = e / hd, d = e % hd;
    float x0 = row[qw + e], x1 = row[qw + e + 1];
    if (p.theta) {
      const float angle = (float)pos * p.theta[d >> 1];
      float sn, cs; sincosf(angle, &sn, &cs);
      const float y0 = cs * x0 - sn * x1, y1 = sn * x0 + cs * x1;
      x0 = y0; x1 = y1;
    }
    KV_T* dst = kc + ((int64_t)g * p.max_ctx + slot) * hd + d;
    dst[0] = kv_from_float<KV_T>(x0); dst[1] = kv_from_float<KV_T>(x1);
  }
  for (int i = threadIdx.x; i < kw; i += 256) {
    const int g = i / hd, d = i % hd;
    vc[((int64_t)g * p.max_ctx + slot) * hd + d] = kv_from_float<KV_T>(row[qw + kw + i]);
  }
}
template <typename KV_T>
__global__ __launch_bounds__(256) void kv_append_rows_kernel(const AttnParams p) { kv_append_row<KV_T>(p); }

// The same for an int8 cache: one half-wave per (token, KV head, K|V) row, quantised with the decode step's rule.
template <int DS>
__global__ __launch_bounds__(256) void kv_append_rows_i8_kernel(const AttnParams p)
{
  const int b = blockIdx.x, hw = threadIdx.x >> 5, l32 = threadIdx.x & 31;
  const float* row = p.qkv + (int64_t)b * p.qkv_stride;
  const int pos = p.pos[b], slot = live_rows(p, pos).slot;
  const int hd = p.hd, qw = p.q_heads * hd, kw = p.kv_heads * hd;
  const int d0 = l32 * DS;
  for (int item = hw; item < 2 * p.kv_heads; item += 8) {      // uniform per half-wave; both halves of a wave loop alike
    const int g = item >> 1, is_v = item & 1;
    const float* src = row + qw + (is_v ? kw : 0) + g * hd;
    float v[DS];
    if (DS >= 2) {
#pragma unroll
      for (int i = 0; i < DS; i += 2) {
        const int d = d0 + i;
        float x0 = d < hd ? src[d] : 0.0f, x1 = d + 1 < hd ? src[d + 1] : 0.0f;
        if (p.theta && !is_v && d < hd) {
          float sn, cs; sincosf((float)pos * p.theta[d >> 1], &sn, &cs);
          const float y0 = cs * x0 - sn * x1, y1 = sn * x0 + cs * x1;
          x0 = y0; x1 = y1;
        }
        v[i] = x0; v[i + (DS > 1 ? 1 : 0)] = x1;
      }
    } else {
      const int d = d0;
      const float own = d < hd ? src[d] : 0.0f, mate = (d ^ 1) < hd ? src[d ^ 1] : 0.0f;
      v[0] = own;
      if (p.theta && !is_v && d < hd) {
        float sn, cs; sincosf((float)pos * p.theta[d >> 1], &sn, &cs);
        v[0] = (d & 1) ? (sn * mate + cs * own) : (cs * own - sn * mate);
      }
    }
    const float scale = quantise_row_i8<DS>(v);
    const int64_t srow = (int64_t)p.seq0 * p.seq_rows + p.layer_row_off + (int64_t)g * p.max_ctx + slot;
    int8_t* dst = reinterpret_cast<int8_t*>(is_v ? p.vc : p.kc) + (int64_t)p.seq0 * p.seq_elems + p.layer_off + ((int64_t)g * p.max_ctx + slot) * hd;
#pragma unroll
    for (int i = 0; i < DS; i++) if (d0 + i < hd) dst[d0 + i] = (int8_t)v[i];
    if (l32 == 0) (is_v ? p.vsc : p.ksc)[srow] = scale;
  }
}

// ------------------------------------------------------------------------------------------
// Prompt ingestion on the matrix cores: every prompt token attends over the cached rows up to its own position.
//
// prompt_rows_kernel: the rotated K and the V of the chunk's tokens into the cache, and what the products read: q and the cached rows of the layer's
// range as planes of halfs (a float or dequantised row two of them, hi + lo), the rows in the order of the matrix operands, so that a wave takes
// an operand of a tile of 32 rows with one request of a whole KB.
// attn_prompt_kernel: a work-group = (query head, 32 consecutive tokens); its four waves take every fourth tile of the tokens' range, each with sums of
// its own, and fold them through LDS at the end.  Per tile and wave:
//   S^T[row][token] = K . q^T   on v_mfma_f32_32x32x16_f16: the result lane holds ONE token column, so the running
//                               maximum, the normaliser and the rescaling of the output are per-lane scalars, and the
//                               result registers of k-step s are exactly the B operand of step s of the next product;
//   O^T[dim][token] += V^T . P^T   with P split hi + lo into two f16 (22 bits), like q; a float cache is split too.
// Same arithmetic as the decode kernels up to the order of the sums (tests: < 1e-4 of token-at-a-time ingestion).
// A pair of halfs ends at 65504 and loses bits below 2^-14, so heads of 64, whose per-row kernel holds floats, scale every operand by a power of
// two first: q per token and head, the rows of a float cache each (int8 codes are exact halfs; their scales count as the row's), the weights
// times the value rows' scales per token and tile, whose sums are then added to O as floats; over a half cache only q and, by 2^14, the
// weights.  9 / 3 heads, float cache, six layers of a 511-token prompt: 593 us without, 630; values of 1e-5 were 7e-5 off and such past 65504 NaN.
// What bounds it: a CU takes in 85 KB/us, an operand pair of a tile of a float cache is 32 KB for 1536 cycles of products.
// Before, four heads of a group shared tiles that every work-group converted itself, V transposed by two-byte stores, one wave a SIMD and three of
// four without a head where a KV head has one.  511 tokens of 28 / 4 heads, float rows: 39.5 us and 11.7 for adding two pieces, 18.7 now (6.6 without any tile,
// 11.3 with one a wave); 255 of 16 / 16: 20.5 + 5.3, 10.2; rows and planes 8.3, 8.5.  512 behind 4096 cached rows, three layers, whole prompt:
// 28 / 4 heads 1088, 646; 16 / 16 1759, 542; 9 / 3 of 64 478, 326.
// ------------------------------------------------------------------------------------------
typedef float pf16_t __attribute__((ext_vector_type(16)));

struct PromptParams {
  const float* qkv; int64_t qkv_stride;      // rows [Q | K | V]
  _Float16* qhi; _Float16* qlo;              // [token][q_heads * HD] rotated q, hi + lo
  int head0, heads;                          // the launch's KV heads
  int tile0, n_tiles;                        // the tiles of 32 cached rows that the chunk's tokens see
  _Float16* planes;                          // [head0 + ..][tile0 + ..] PromptShape::TILE halfs
  float* rsc;                                // PromptShape::ROWS: likewise [K 32 | V 32] what a row's planes are to be multiplied by
  void* kc; void* vc;                        // this sequence's layer plane: [kv_head][max_ctx][HD]
  const float* ksc; const float* vsc;        // int8 cache: row scales of the same plane, [kv_head][max_ctx]
  int q_heads, kv_heads, max_ctx, n_tok, window;
  float softcap, inv_sqrt;
  const float* theta; int pos0;              // token t: position pos0 + t of the sequence
  float* out; int64_t out_stride;
  float* part;                               // [token][q_head][K split][HD + 2]: unnormalised sums, maximum, normaliser
  float* qsc;                                // HD = 64: [token][q_head] what the head's planes are to be multiplied by
  BlkPlanes planes_out; bool planes_q8;      // the results leave as planes of the next product (planes_out.hi null: as rows)
};

template <typename KV_T, int HD> struct PromptShape {
  static constexpr bool I8 = sizeof(KV_T) == 1;          // int8 rows: HD = 128: dequantised (code * row scale)
  static constexpr bool SC = HD == 64;                   // every operand holds what a float holds, whatever its size: see the comment above
  static constexpr bool ROWS = SC && sizeof(KV_T) != 2;  // row scales
  static constexpr int NP = (SC ? sizeof(KV_T) == 4 : sizeof(KV_T) != 2) ? 2 : 1;      // planes of K and V
  static constexpr int PLANE = 32 * HD, TILE = 2 * NP * PLANE;      // halfs: K's planes [step of 16 dims][lane][8], V's [step of 16 rows][32 dims][lane][8]
};

constexpr int PA_KT_MIN = 8;     // K tiles (of 32 cached rows) a split takes at least: two a wave
constexpr int PA_KS_MAX = 8;     // splits of a token tile's K range at most
// K tiles a token tile walks and the number of work-groups (blockIdx.z) they are cut over: a short prompt behind many rows
// (few token tiles) still fills the chip; the merge kernel adds the pieces.
__device__ __forceinline__ void prompt_k_range(const PromptParams& p, int t0, int n_ks, int& jt0, int& jt1, int& splits)
{
  const int pos_first = p.pos0 + t0, pos_last = p.pos0 + min(t0 + 31, p.n_tok - 1);
  const int j_lo = (p.window > 0 && pos_first + 1 > p.window) ? pos_first + 1 - p.window : 0;
  jt0 = j_lo >> 5; jt1 = pos_last >> 5;
  splits = max(1, min(n_ks, (jt1 - jt0 + 1) / PA_KT_MIN));
}

// rotated q of token t (neural/neural.cl:1517-1542) as two f16 planes
template <int HD>
__device__ __forceinline__ void prompt_q_row(const PromptParams& p, const int t)
{
  const int qw = p.q_heads * HD;
  const float* row = p.qkv + (int64_t)t * p.qkv_stride;
  const int pos = p.pos0 + t;
  for (int e = threadIdx.x; e < (qw >> 1); e += 256) {
    const int d = (2 * e) & (HD - 1);
    float x0 = row[2 * e], x1 = row[2 * e + 1];
    if (p.theta) {
      float sn, cs; sincosf((float)pos * p.theta[d >> 1], &sn, &cs);
      const float y0 = cs * x0 - sn * x1, y1 = sn * x0 + cs * x1;
      x0 = y0; x1 = y1;
    }
    _Float16 h0, h1, l0, l1;
    if constexpr (HD == 64) {               // (32 neighbouring lanes hold a head)
      float m = fmaxf(finite_abs(x0), finite_abs(x1));
#pragma unroll
      for (int off = 1; off < 32; off <<= 1) m = fmaxf(m, __shfl_xor(m, off));
      const int ex = plane_exponent(m);
      split_plane(ldexpf(x0, ex), h0, l0); split_plane(ldexpf(x1, ex), h1, l1);
      if ((e & 31) == 0) p.qsc[(int64_t)t * p.q_heads + (e >> 5)] = ldexpf(1.0f, -ex);
    } else { split_f16(x0, h0, l0); split_f16(x1, h1, l1); }
    p.qhi[(int64_t)t * qw + 2 * e] = h0; p.qhi[(int64_t)t * qw + 2 * e + 1] = h1;
    p.qlo[(int64_t)t * qw + 2 * e] = l0; p.qlo[(int64_t)t * qw + 2 * e + 1] = l1;
  }
}

// Work-groups 0 .. n_tiles * heads - 1: 32 cached rows of a KV head each, those of the chunk from its K and V (an int8 cache has them already);
// the others (with the first heads): a token's q.
template <typename KV_T, int HD>
__global__ __launch_bounds__(256) void prompt_rows_kernel(const PromptParams p)
{
  using S = PromptShape<KV_T, HD>;
  constexpr int E = HD / 8, DT = HD / 32, LDF = HD + 4;
  __shared__ __align__(16) float sv[32 * LDF];
  const int tiles = p.n_tiles * p.heads, tid = threadIdx.x;
  if ((int)blockIdx.x >= tiles) { prompt_q_row<HD>(p, blockIdx.x - tiles); return; }
  const int g = p.head0 + blockIdx.x % p.heads, jt = p.tile0 + blockIdx.x / p.heads;
  const int64_t place = (int64_t)(blockIdx.x % p.heads) * p.n_tiles + blockIdx.x / p.heads;
  const int pos0 = p.pos0, last = pos0 + p.n_tok - 1;
  const int r = tid >> 3, d0 = (tid & 7) * E, j = 32 * jt + r;     // E consecutive elements of a cached row
  const bool live = j <= last;
  const int64_t at = ((int64_t)g * p.max_ctx + min(j, last)) * HD + d0;
  float k[E], v[E], ks = 1.0f, vs = 1.0f;
  if constexpr (S::I8) {
    const int8_t *kq = reinterpret_cast<const int8_t*>(p.kc) + at, *vq = reinterpret_cast<const int8_t*>(p.vc) + at;
    ks = p.ksc[(int64_t)g * p.max_ctx + min(j, last)]; vs = p.vsc[(int64_t)g * p.max_ctx + min(j, last)];
#pragma unroll
    for (int i = 0; i < E; i += 4) {
      const int a = *reinterpret_cast<const int*>(kq + i), b = *reinterpret_cast<const int*>(vq + i);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        k[i + u] = (float)((a << (24 - 8 * u)) >> 24) * (S::ROWS ? 1.0f : ks);      // (codes are exact halfs)
        v[i + u] = (float)((b << (24 - 8 * u)) >> 24) * (S::ROWS ? 1.0f : vs);
      }
    }
  } else {
    KV_T ko[E], vo[E];
    if (live && j >= pos0) {
      const float *kr = p.qkv + (int64_t)(j - pos0) * p.qkv_stride + (int64_t)p.q_heads * HD + g * HD + d0, *vr = kr + p.kv_heads * HD;
      KV_T *kd = reinterpret_cast<KV_T*>(p.kc) + at, *vd = reinterpret_cast<KV_T*>(p.vc) + at;
#pragma unroll
      for (int i = 0; i < E; i += 4) { *reinterpret_cast<float4*>(k + i) = *reinterpret_cast<const float4*>(kr + i); *reinterpret_cast<float4*>(v + i) = *reinterpret_cast<const float4*>(vr + i); }
      if (p.theta)
#pragma unroll
        for (int i = 0; i < E; i += 2) {
          float sn, cs; sincosf((float)j * p.theta[(d0 + i) >> 1], &sn, &cs);
          const float y0 = cs * k[i] - sn * k[i + 1], y1 = sn * k[i] + cs * k[i + 1];
          k[i] = y0; k[i + 1] = y1;
        }
#pragma unroll
      for (int i = 0; i < E; i++) { ko[i] = kv_from_float<KV_T>(k[i]); vo[i] = kv_from_float<KV_T>(v[i]); k[i] = kv_to_float(ko[i]); v[i] = kv_to_float(vo[i]); }
#pragma unroll
      for (int i = 0; i < E * (int)sizeof(KV_T) / 16; i++) { reinterpret_cast<uint4*>(kd)[i] = reinterpret_cast<const uint4*>(ko)[i]; reinterpret_cast<uint4*>(vd)[i] = reinterpret_cast<const uint4*>(vo)[i]; }
    } else {
#pragma unroll
      for (int i = 0; i < E * (int)sizeof(KV_T) / 16; i++) {
        reinterpret_cast<uint4*>(ko)[i] = reinterpret_cast<const uint4*>(reinterpret_cast<const KV_T*>(p.kc) + at)[i];
        reinterpret_cast<uint4*>(vo)[i] = reinterpret_cast<const uint4*>(reinterpret_cast<const KV_T*>(p.vc) + at)[i];
      }
#pragma unroll
      for (int i = 0; i < E; i++) { k[i] = kv_to_float(ko[i]); v[i] = kv_to_float(vo[i]); }
    }
  }
  if (!live) {                                // rows behind the last one hold what an earlier sequence left: not multiplied, not even by zero
#pragma unroll
    for (int i = 0; i < E; i++) k[i] = v[i] = 0.0f;
    ks = vs = 0.0f;
  }
  if constexpr (S::ROWS) {                    // (the eight threads of a row are neighbours)
    if (!S::I8) {
      float mk = 0.0f, mv = 0.0f;
#pragma unroll
      for (int i = 0; i < E; i++) { mk = fmaxf(mk, finite_abs(k[i])); mv = fmaxf(mv, finite_abs(v[i])); }
#pragma unroll
      for (int off = 1; off < 8; off <<= 1) { mk = fmaxf(mk, __shfl_xor(mk, off)); mv = fmaxf(mv, __shfl_xor(mv, off)); }
      const int ek = plane_exponent(mk), ev = plane_exponent(mv);
#pragma unroll
      for (int i = 0; i < E; i++) { k[i] = ldexpf(k[i], ek); v[i] = ldexpf(v[i], ev); }
      ks = ldexpf(1.0f, -ek); vs = ldexpf(1.0f, -ev);
    }
    if ((tid & 7) == 0) { float* s = p.rsc + place * 64 + r; s[0] = ks; s[32] = vs; }
  }
  auto split = [](float x, _Float16& h, _Float16& l) { if (S::SC) split_plane(x, h, l); else split_f16(x, h, l); };
  _Float16* tile = p.planes + place * S::TILE;
#pragma unroll
  for (int i8 = 0; i8 < E; i8 += 8) {         // dims d0 + i8 .. + 7: step d / 16, lane half (d / 8) % 2, row r
    ph8_t h, l;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      if (S::NP == 2) { _Float16 a, b; split(k[i8 + i], a, b); h[i] = a; l[i] = b; }
      else h[i] = (_Float16)k[i8 + i];
    }
    const int d = d0 + i8, o = ((d >> 4) * 64 + ((d >> 3) & 1) * 32 + r) * 8;
    *reinterpret_cast<ph8_t*>(tile + o) = h;
    if (S::NP == 2) *reinterpret_cast<ph8_t*>(tile + S::PLANE + o) = l;
  }
#pragma unroll
  for (int i = 0; i < E; i += 4) *reinterpret_cast<float4*>(&sv[r * LDF + d0 + i]) = *reinterpret_cast<const float4*>(v + i);
  __syncthreads();
  tile += S::NP * S::PLANE;
  for (int f = tid; f < 2 * DT * 64; f += 256) {      // lane (n, kg) of step s2, dims 32 dt + n: the rows that the weights' registers hold (below)
    const int lane = f & 63, dt = (f >> 6) % DT, s2 = (f >> 6) / DT, n = lane & 31, kg = lane >> 5;
    ph8_t h, l;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float x = sv[(16 * s2 + 8 * (i >> 2) + 4 * kg + (i & 3)) * LDF + 32 * dt + n];
      if (S::NP == 2) { _Float16 a, b; split(x, a, b); h[i] = a; l[i] = b; }
      else h[i] = (_Float16)x;
    }
    *reinterpret_cast<ph8_t*>(tile + 8 * f) = h;
    if (S::NP == 2) *reinterpret_cast<ph8_t*>(tile + S::PLANE + 8 * f) = l;
  }
}

constexpr int PA_LDO = 33;     // floats per output dimension in LDS (32 tokens + 1)

template <typename KV_T, int HD>
__global__ __launch_bounds__(256, 2) void attn_prompt_kernel(const PromptParams p)
{
  using S = PromptShape<KV_T, HD>;
  constexpr bool SC = S::SC, ROWS = S::ROWS;
  constexpr int NP = S::NP, STEPS = HD / 16, DT = HD / 32, LDQ = HD + 8;      // (LDQ: rows stay 16-byte aligned for the 8-half operand reads)
  constexpr int Q_B = 2 * 32 * LDQ * 2, O_B = 4 * HD * PA_LDO * 4;
  __shared__ __align__(16) unsigned char lds[Q_B > O_B ? Q_B : O_B];          // q's planes [2][32][LDQ] halfs; then the waves' sums [4][HD][PA_LDO]
  __shared__ float sM[4][32], sL[4][32];
  _Float16* sQ = reinterpret_cast<_Float16*>(lds);
  float* sO = reinterpret_cast<float*>(lds);
  const int G = p.q_heads / p.kv_heads, head = p.head0 * G + blockIdx.x, g = blockIdx.x / G;      // (g: of the launch's)
  const int t0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * 32;                 // the longest ranges first
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, n = lane & 31, kg = lane >> 5;
  const int tok = t0 + n;
  const int pos_n = tok < p.n_tok ? p.pos0 + tok : -1;
  const int jstart_n = (p.window > 0 && pos_n + 1 > p.window) ? pos_n + 1 - p.window : 0;
  // the tile's range of cached rows (tokens are consecutive positions of one sequence) and this work-group's share of it
  int jt_first, jt_last, splits;
  prompt_k_range(p, t0, (int)gridDim.z, jt_first, jt_last, splits);
  const int ks = blockIdx.z;
  if (ks >= splits) return;                       // (uniform: the whole work-group leaves before any barrier)
  {
    const int per = (jt_last - jt_first + 1 + splits - 1) / splits;
    const int a = jt_first + ks * per;
    jt_last = min(jt_last, a + per - 1); jt_first = a;
  }
  // The operands of the wave's next tile are requested as soon as the registers of the current one are free: K's run behind the weights and the second
  // product, V's behind the next tile's first product.
  const _Float16* planes = p.planes + ((int64_t)g * p.n_tiles - p.tile0) * S::TILE + 8 * lane;
  const float* scales = ROWS ? p.rsc + ((int64_t)g * p.n_tiles - p.tile0) * 64 + 4 * kg : nullptr;
  ph8_t K[NP][STEPS], V[NP][2 * DT];
  float4 rk[ROWS ? 4 : 1], rv[ROWS ? 4 : 1];
  auto load_k = [&](int jt) __attribute__((always_inline)) {
    if (jt > jt_last) return;
#pragma unroll
    for (int s = 0; s < STEPS; s++)
#pragma unroll
      for (int q = 0; q < NP; q++) K[q][s] = *reinterpret_cast<const ph8_t*>(planes + (int64_t)jt * S::TILE + q * S::PLANE + 512 * s);
    if constexpr (ROWS)
#pragma unroll
      for (int i = 0; i < 4; i++) rk[i] = *reinterpret_cast<const float4*>(scales + (int64_t)jt * 64 + 8 * i);
  };
  auto load_v = [&](int jt) __attribute__((always_inline)) {
    if (jt > jt_last) return;
#pragma unroll
    for (int s = 0; s < 2 * DT; s++)
#pragma unroll
      for (int q = 0; q < NP; q++) V[q][s] = *reinterpret_cast<const ph8_t*>(planes + (int64_t)jt * S::TILE + (NP + q) * S::PLANE + 512 * s);
    if constexpr (ROWS)
#pragma unroll
      for (int i = 0; i < 4; i++) rv[i] = *reinterpret_cast<const float4*>(scales + (int64_t)jt * 64 + 32 + 8 * i);
  };
  constexpr int QN = 2 * 32 * (HD / 8) / 256;
  ph8_t qr[QN];
#pragma unroll
  for (int i = 0; i < QN; i++) {
    const int u = tid + 256 * i, q = u / (32 * (HD / 8)), r = u / (HD / 8) % 32, c = u % (HD / 8);
    qr[i] = *reinterpret_cast<const ph8_t*>((q ? p.qlo : p.qhi) + (int64_t)min(t0 + r, p.n_tok - 1) * (p.q_heads * HD) + head * HD + 8 * c);
  }
  load_k(jt_first + wave);
#pragma unroll
  for (int i = 0; i < QN; i++) {
    const int u = tid + 256 * i, r = u / (HD / 8) % 64, c = u % (HD / 8);
    *reinterpret_cast<ph8_t*>(sQ + r * LDQ + 8 * c) = qr[i];
  }
  const float qs = SC ? p.qsc[(int64_t)min(tok, p.n_tok - 1) * p.q_heads + head] * p.inv_sqrt : p.inv_sqrt;
  load_v(jt_first + wave);
  pf16_t O[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int v = 0; v < 16; v++) O[dt][v] = 0.0f;
  float m_run = -1e30f, l_run = 0.0f;
  __syncthreads();

  for (int jt = jt_first + wave; jt <= jt_last; jt += 4) {
    // ---- S^T = K . q^T ----
    pf16_t C;
#pragma unroll
    for (int v = 0; v < 16; v++) C[v] = 0.0f;
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
      const ph8_t qh = *reinterpret_cast<const ph8_t*>(sQ + n * LDQ + 16 * s + 8 * kg), ql = *reinterpret_cast<const ph8_t*>(sQ + (32 + n) * LDQ + 16 * s + 8 * kg);
      C = __builtin_amdgcn_mfma_f32_32x32x16_f16(K[0][s], qh, C, 0, 0, 0);
      C = __builtin_amdgcn_mfma_f32_32x32x16_f16(K[0][s], ql, C, 0, 0, 0);
      if (NP == 2) C = __builtin_amdgcn_mfma_f32_32x32x16_f16(K[NP - 1][s], qh, C, 0, 0, 0);
    }
    // ---- this token's column: mask, running maximum, weights ----
    float tmax = -1e30f;
    bool ok[16];
    auto of_row = [](const float4* r, int v) { const float4 x = r[ROWS ? v >> 2 : 0]; return (v & 3) == 0 ? x.x : (v & 3) == 1 ? x.y : (v & 3) == 2 ? x.z : x.w; };
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int krow = jt * 32 + 8 * (v >> 2) + 4 * kg + (v & 3);
      float sc = C[v] * (ROWS ? of_row(rk, v) * qs : qs);
      if (p.softcap > 0.0f) sc = p.softcap * tanhf(sc / p.softcap);
      ok[v] = krow <= pos_n && krow >= jstart_n;
      C[v] = sc;
      if (ok[v]) tmax = fmaxf(tmax, sc);
    }
    __builtin_amdgcn_sched_barrier(0);        // (moved up, the requests would take registers of their own)
    load_k(jt + 4);
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float m_new = fmaxf(m_run, tmax), corr = expf(m_run - m_new);
    float psum = 0.0f;
#pragma unroll
    for (int v = 0; v < 16; v++) { C[v] = ok[v] ? (SC && !ROWS ? 16384.0f : 1.0f) * expf(C[v] - m_new) : 0.0f; psum += C[v]; }   // (half cache: weights of 2^-39 on stay)
    psum += __shfl_xor(psum, 32, 64);
    l_run = l_run * corr + psum; m_run = m_new;
    if (__builtin_amdgcn_ballot_w64(corr != 1.0f)) {      // (after the first tiles a new maximum is rare: the whole wave skips the rescaling)
#pragma unroll
      for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int v = 0; v < 16; v++) O[dt][v] *= corr;
    }
    // row scales: the weights take them, and a power of two per token and tile brings the largest to 2^13
    float back = 1.0f;
    pf16_t T[ROWS ? DT : 1];
    if constexpr (ROWS) {
      float wmax = 0.0f;
#pragma unroll
      for (int v = 0; v < 16; v++) { C[v] = ok[v] ? C[v] * of_row(rv, v) : 0.0f; wmax = fmaxf(wmax, finite_abs(C[v])); }
      wmax = fmaxf(wmax, __shfl_xor(wmax, 32, 64));
      const int e = plane_exponent(wmax);
      back = ldexpf(1.0f, -e);
#pragma unroll
      for (int v = 0; v < 16; v++) C[v] = ldexpf(C[v], e);
#pragma unroll
      for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int v = 0; v < 16; v++) T[dt][v] = 0.0f;
    }
    // ---- O^T += V^T . P^T ----
    // The score registers 8 s2 .. 8 s2 + 7 of a lane are cached rows 16 s2 + 4 kg + (0..3) and 16 s2 + 8 + 4 kg + (0..3): taken as
    // the eight k of a 16-deep step, with the value operand holding the same two groups of four rows (the order of the
    // rows inside a step is free as long as both operands agree).
#pragma unroll
    for (int s2 = 0; s2 < 2; s2++) {
      ph8_t ph, pl;
#pragma unroll
      for (int i = 0; i < 8; i++) { _Float16 hv, lv; split_f16(C[8 * s2 + i], hv, lv); ph[i] = hv; pl[i] = lv; }
#pragma unroll
      for (int dt = 0; dt < DT; dt++) {
        pf16_t& A = ROWS ? T[ROWS ? dt : 0] : O[dt];
        A = __builtin_amdgcn_mfma_f32_32x32x16_f16(V[0][s2 * DT + dt], ph, A, 0, 0, 0);
        A = __builtin_amdgcn_mfma_f32_32x32x16_f16(V[0][s2 * DT + dt], pl, A, 0, 0, 0);
        if (NP == 2) A = __builtin_amdgcn_mfma_f32_32x32x16_f16(V[NP - 1][s2 * DT + dt], ph, A, 0, 0, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    load_v(jt + 4);
    if constexpr (ROWS)
#pragma unroll
      for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int v = 0; v < 16; v++) O[dt][v] = fmaf(T[dt][v], back, O[dt][v]);
  }

  // ---- the waves' sums, in wave order: a wave without a row of the token (a normaliser of exactly 0) leaves nothing, one that met a score that is not a number or
  // infinite (a normaliser that is not a number) makes the token's result that too ----
  if (kg == 0) { sM[wave][n] = m_run; sL[wave][n] = l_run; }
  __syncthreads();                                // (and q has been read)
  {
    const float M = fmaxf(fmaxf(sM[0][n], sM[1][n]), fmaxf(sM[2][n], sM[3][n])), c = expf(m_run - M);
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int v = 0; v < 16; v++) sO[(wave * HD + 32 * dt + 8 * (v >> 2) + 4 * kg + (v & 3)) * PA_LDO + n] = l_run == 0.0f ? 0.0f : O[dt][v] * c;
  }
  __syncthreads();
  const int r = tid >> 3, t = t0 + r;
  if (t >= p.n_tok) return;
  const float M = fmaxf(fmaxf(sM[0][r], sM[1][r]), fmaxf(sM[2][r], sM[3][r]));
  float L = 0.0f;
#pragma unroll
  for (int w = 0; w < 4; w++) if (sL[w][r] != 0.0f) L = fmaf(sL[w][r], expf(sM[w][r] - M), L);
  const float inv = splits > 1 ? 1.0f : L == 0.0f ? 0.0f : 1.0f / L;          // a piece leaves unnormalised sums, maximum and normaliser; prompt_merge_kernel adds the pieces
  float* dst = splits > 1 ? p.part + (((int64_t)t * p.q_heads + head) * gridDim.z + ks) * (HD + 2) : p.out + (int64_t)t * p.out_stride + head * HD;
#pragma unroll
  for (int i = 0; i < HD / 32; i++) {
    const int d = 32 * i + 4 * (tid & 7);
    float a[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      a[u] = 0.0f;
#pragma unroll
      for (int w = 0; w < 4; w++) a[u] += sO[(w * HD + d + u) * PA_LDO + r];
      a[u] *= inv;
    }
    if (splits > 1) { *reinterpret_cast<float2*>(dst + d) = make_float2(a[0], a[1]); *reinterpret_cast<float2*>(dst + d + 2) = make_float2(a[2], a[3]); }      // (records of HD + 2 floats: 8-byte aligned only)
    else if (p.planes_out.hi) out_plane4(p.planes_out, p.planes_q8, t, head * HD + d, p.q_heads * HD, a);
    else *reinterpret_cast<float4*>(dst + d) = make_float4(a[0], a[1], a[2], a[3]);
  }
  if (splits > 1 && (tid & 7) == 0) { dst[HD] = M; dst[HD + 1] = L; }
}

// out[token][head] = sum of the K splits of a token tile, folded with a running maximum in split order (a tile walked by one
// work-group was written by it and is left alone)
template <int HD>
__global__ __launch_bounds__(512) void prompt_merge_kernel(const PromptParams p, int n_ks)
{
  const int tok = blockIdx.x, head = blockIdx.y * 4 + (threadIdx.x >> 7), d = threadIdx.x & 127;   // four heads per work-group
  int jt0, jt1, splits;
  prompt_k_range(p, (tok >> 5) << 5, n_ks, jt0, jt1, splits);
  if (splits <= 1 || head >= p.q_heads || d >= HD) return;
  const float* pt = p.part + (((int64_t)tok * p.q_heads + head) * n_ks) * (HD + 2);
  float M = -1e30f, L = 0.0f, A = 0.0f;
  float ms[PA_KS_MAX], ls[PA_KS_MAX], as[PA_KS_MAX];                     // all requests first (a split past the count repeats the last one; not used)
#pragma unroll
  for (int s = 0; s < PA_KS_MAX; s++) { const int sc = min(s, splits - 1); ms[s] = pt[sc * (HD + 2) + HD]; ls[s] = pt[sc * (HD + 2) + HD + 1]; as[s] = pt[sc * (HD + 2) + d]; }
#pragma unroll
  for (int s = 0; s < PA_KS_MAX; s++) {
    if (s < splits && ls[s] != 0.0f) {      // (a piece that is not a number stays one)
      const float mn = fmaxf(M, ms[s]), c0 = expf(M - mn), c1 = expf(ms[s] - mn);
      A = A * c0 + as[s] * c1; L = L * c0 + ls[s] * c1; M = mn;
    }
  }
  const float y = L == 0.0f ? 0.0f : A * (1.0f / L);
  if (p.planes_out.hi) out_plane(p.planes_out, p.planes_q8, tok, head * HD + d, p.q_heads * HD, y);
  else p.out[(int64_t)tok * p.out_stride + head * HD + d] = y;
}

// Whether n prompt rows of this cache go to the matrix-core prompt kernel (it needs no per-slice partial results).
// Heads of 128: from 8 rows on.  Heads of 64: from 256 on, where the per-row kernel's reads of the cache outgrow its launch (first chunks of
// 9 / 3 heads, a whole prompt through six layers, float cache: 128 tokens 383 us per row, 395 here (with operands that were not scaled
// yet); 256: 929, 486; 511: 1317, 630; 1500: 4313, 1878; int8 6698, 1873; 8 / 8 heads, three layers, 200 tokens: 261, 272).
bool attn_prompt_is_flash(const cai_kv_s* kv, int n)
{
  static const int flash_on = []() { const char* e = getenv("CAIHIP_PROMPT_FLASH"); return e ? atoi(e) : 1; }();
  return flash_on && kv->evict_cap == 0 && ((kv->head_dim == 128 && n >= 8) || (kv->head_dim == 64 && n >= 256));
}

bool attn_rows_for_product(const cai_kv_s* kv, int seq, int layer, int n, const float* theta, const int32_t* pos, KvRows& out)
{
  if (kv->dtype == CAI_KV_I8 || kv->evict_cap > 0 || (kv->head_dim & 1) || attn_prompt_is_flash(kv, n)) return false;      // (those take them by themselves, or quantise whole rows)
  const size_t at = ((size_t)seq * kv->seq_elems() + (size_t)layer * kv->layer_elems()) * kv->elem();
  out.k = (char*)kv->k + at; out.v = (char*)kv->v + at; out.half = kv->dtype == CAI_KV_F16; out.head_dim = kv->head_dim; out.max_ctx = kv->max_ctx;
  out.theta = theta; out.pos = pos;
  return true;
}

int launch_attn_step(cai_kv_s* kv, int layer, float* qkv, int64_t qkv_stride, int n_seq, int q_heads, int window,
                     float softcap, const float* theta, const int32_t* pos_dev, float* out, int64_t out_stride, int seq0,
                     int prompt_rows, float* prompt_part, const float* qn_gain, const float* kn_gain, float qk_eps, AttnOnPlanes* on_planes)
{
  Context& c = ctx();
  if (layer < 0 || layer >= kv->n_layers) return set_error(CAI_ERR_INVALID, "attention: layer %d of %d", layer, kv->n_layers);
  if (n_seq < 1 || seq0 < 0 || seq0 + (prompt_rows ? 1 : n_seq) > kv->n_seq) return set_error(CAI_ERR_INVALID, "attention: %d sequences, cache holds %d", n_seq, kv->n_seq);
  if (q_heads % kv->kv_heads) return set_error(CAI_ERR_INVALID, "attention: %d query heads not a multiple of %d KV heads", q_heads, kv->kv_heads);
  if (q_heads > kv->part_q_heads) return set_error(CAI_ERR_INVALID, "attention: %d query heads exceed the cache's scratch (%d)", q_heads, kv->part_q_heads);
  PlanesParams p{};
  p.qkv = qkv; p.qkv_stride = qkv_stride; p.kc = kv->k; p.vc = kv->v;
  p.seq_elems = kv->seq_elems(); p.layer_off = (int64_t)layer * kv->layer_elems();
  p.q_heads = q_heads; p.kv_heads = kv->kv_heads; p.hd = kv->head_dim; p.max_ctx = kv->max_ctx;
  p.window = window; p.softcap = softcap; p.inv_sqrt = kv->score_mul / sqrtf((float)kv->head_dim);
  p.theta = theta; p.pos = pos_dev;
  if (kv->geo_rows > 0) {   // the caller chose a length bucket: it must cover the rows the host knows to be in use
    int needed = 0;
    for (int s0 = 0; s0 < (prompt_rows ? 1 : n_seq); s0++) needed = std::max(needed, kv->len_at(seq0 + s0, layer) + (prompt_rows ? n_seq : 1));
    if (needed > kv->geo_rows) return set_error(CAI_ERR_STATE, "attention: launch geometry covers %d rows, %d are in use", kv->geo_rows, needed);
  }
  kv_geometry(kv, kv->geo_rows, &p.split_len, &p.n_splits);
  p.part = prompt_rows ? prompt_part : kv->part; p.out = out; p.out_stride = out_stride; p.seq0 = seq0;
  p.seq_mul = prompt_rows ? 0 : 1; p.appended = prompt_rows ? 1 : 0;
  p.evict_sinks = kv->evict_sinks; p.evict_cap = kv->evict_cap;
  p.ksc = kv->ks; p.vsc = kv->vs; p.seq_rows = kv->seq_rows(); p.layer_row_off = (int64_t)layer * kv->layer_rows();
  int rc;
  const int form = attn_form(kv, q_heads, n_seq, p.split_len, p.n_splits, prompt_rows != 0, qn_gain != nullptr);
  const bool grouped = form != ATTN_PER_HEAD;
  // The per-head kernel merges its slices itself (one work-group per head does a head's merge).  A prompt has more rows in
  // flight than the counters cover, and in the per-KV-head kernel the last arriver would fold a whole group of heads over
  // many slices alone (32B shape, 33 slices x 5 heads: 37.7 us against 30.7 us with the merge launch): those keep the launch.
  p.merge_cnt = (prompt_rows || grouped) ? nullptr : kv->merge_cnt;
  if (qn_gain) {
    // q and k norms over the whole rows: the per-head decode kernel applies them while it reads its operands; the
    // other kernels find the rows normalised in place
    const int qw = q_heads * kv->head_dim, kw = kv->kv_heads * kv->head_dim;
    if (!prompt_rows && !grouped) { p.qn_gain = qn_gain; p.kn_gain = kn_gain; p.qk_eps = qk_eps; }
    else if ((rc = launch_rmsnorm_pair(qkv, qn_gain, qw, kn_gain, kw, n_seq, qk_eps, qkv_stride))) return rc;
  }
  // prompts over a 128- or 64-wide cache: matrix-core kernel, 32 tokens of a head per work-group
  const bool flash = prompt_rows == 1 && attn_prompt_is_flash(kv, n_seq);
  if (on_planes && on_planes->planes.hi && (flash || (!grouped && p.hd % 32 == 0))) { p.planes = on_planes->planes; p.planes_q8 = on_planes->q8_0; on_planes->planes_done = true; }
  if (on_planes && on_planes->appended) {}      // (by the product that made them)
  else if (prompt_rows && kv->dtype == CAI_KV_I8) {
    if (p.hd <= 32) hipLaunchKernelGGL(kv_append_rows_i8_kernel<1>, dim3(n_seq), dim3(256), 0, c.stream, p);
    else if (p.hd <= 64) hipLaunchKernelGGL(kv_append_rows_i8_kernel<2>, dim3(n_seq), dim3(256), 0, c.stream, p);
    else hipLaunchKernelGGL(kv_append_rows_i8_kernel<4>, dim3(n_seq), dim3(256), 0, c.stream, p);
  } else if (prompt_rows && !flash) {        // (prompt_rows_kernel appends by itself)
    if (kv->dtype == CAI_KV_F16) hipLaunchKernelGGL(kv_append_rows_kernel<__half>, dim3(n_seq), dim3(256), 0, c.stream, p);
    else hipLaunchKernelGGL(kv_append_rows_kernel<float>, dim3(n_seq), dim3(256), 0, c.stream, p);
  }
  if (flash) {
    if (kv->prompt_end < n_seq || kv->prompt_end > kv->max_ctx) return set_error(CAI_ERR_STATE, "attention: a prompt of %d rows ends at row %d of %d", n_seq, kv->prompt_end, kv->max_ctx);
    const int pos0 = kv->prompt_end - n_seq, tok_tiles = (n_seq + 31) / 32;
    const int tile0 = window > 0 && pos0 + 1 > window ? (pos0 + 1 - window) / 32 : 0, n_tiles = (kv->prompt_end + 31) / 32 - tile0;      // a window's rows, not the cache's
    // K splits per token tile: a work-group takes a CU's half, so the range is cut where that shortens (rounds of work-groups) / splits by a fifth or more, and
    // never to less than two tiles a wave.  Three layers of the 28 / 4 heads shape, whole prompts: 16 tokens behind 4096 rows 387 us uncut, 249 in eight; 300 behind 7000
    // 855, 699 in three; 64 behind 2000 325, 277; a single tile a wave (a limit of four tiles a work-group) changes nothing at 28 / 4.
    int n_ks = 1;
    auto rounds = [&](int k) { return (tok_tiles * q_heads * k + 2 * c.n_cu - 1) / (2 * c.n_cu) / (double)k; };
    for (int k = 2; k <= std::min(PA_KS_MAX, n_tiles / PA_KT_MIN); k++) if (rounds(k) <= 0.8 * rounds(n_ks)) n_ks = k;
    // One piece of memory: q's planes, their scales, the cached rows' planes (as large as the rows are as floats or halfs) and scales, the pieces' sums.  Tiles are counted up to a
    // power of two, so that the chunks of a long prompt find it large enough.  The planes hold the rows of one layer and sequence, of as many KV heads at a time as 512 MB take
    // (eight of 128 behind 65536 float or int8 rows), so that a cache that leaves little room beside it can be filled.
    const int np = p.hd == 64 ? (kv->dtype == CAI_KV_F32 ? 2 : 1) : (kv->dtype == CAI_KV_F16 ? 1 : 2);
    int most = 16; while (most < n_tiles) most *= 2;
    most = std::min(most, (kv->max_ctx + 31) / 32);
    const size_t q_b = (size_t)n_seq * q_heads * p.hd * 2, s_b = ((size_t)n_seq * q_heads * 4 + 255) / 256 * 256;
    const size_t head_b = (size_t)most * (4 * np * 32 * p.hd);
    const int at_once = (int)std::min<size_t>(kv->kv_heads, std::max<size_t>(1, ((size_t)512 << 20) / head_b)), turns = (kv->kv_heads + at_once - 1) / at_once, heads = (kv->kv_heads + turns - 1) / turns;
    const size_t t_b = heads * head_b, r_b = (size_t)most * heads * 256;
    const size_t need = 2 * q_b + s_b + t_b + r_b + (n_ks > 1 ? (size_t)n_seq * q_heads * n_ks * (p.hd + 2) * 4 : 0);
    if (need > kv->pq_cap) {
      CAI_HIP(hipStreamSynchronize(c.stream));
      if (kv->pq) (void)hipFree(kv->pq);
      kv->pq = nullptr; kv->pq_cap = 0;
      CAI_HIP(hipMalloc(&kv->pq, need));
      kv->pq_cap = need;
    }
    PromptParams pp{};
    char* ws = (char*)kv->pq;
    pp.qkv = qkv; pp.qkv_stride = qkv_stride; pp.qhi = (_Float16*)ws; pp.qlo = (_Float16*)(ws + q_b);
    pp.qsc = (float*)(ws + 2 * q_b); pp.planes = (_Float16*)(ws + 2 * q_b + s_b); pp.rsc = (float*)(ws + 2 * q_b + s_b + t_b); pp.part = (float*)(ws + 2 * q_b + s_b + t_b + r_b);
    const size_t plane = ((size_t)seq0 * kv->seq_elems() + (size_t)layer * kv->layer_elems()) * kv->elem();
    pp.kc = (char*)kv->k + plane; pp.vc = (char*)kv->v + plane;
    if (kv->dtype == CAI_KV_I8) {
      const size_t rows0 = (size_t)seq0 * kv->seq_rows() + (size_t)layer * kv->layer_rows();
      pp.ksc = kv->ks + rows0; pp.vsc = kv->vs + rows0;
    }
    pp.q_heads = q_heads; pp.kv_heads = kv->kv_heads; pp.max_ctx = kv->max_ctx; pp.n_tok = n_seq; pp.tile0 = tile0; pp.n_tiles = n_tiles; pp.window = window;
    pp.softcap = softcap; pp.inv_sqrt = p.inv_sqrt; pp.theta = theta; pp.pos0 = pos0; pp.planes_out = p.planes; pp.planes_q8 = p.planes_q8; pp.out = out; pp.out_stride = out_stride;
    const int G = q_heads / kv->kv_heads;
    auto go = [&](auto hd_) {
      constexpr int HD = hd_;
      auto both = [&](auto kv_) {
        using KV_T = decltype(kv_);
        for (pp.head0 = 0; pp.head0 < kv->kv_heads; pp.head0 += heads) {
          pp.heads = std::min(heads, kv->kv_heads - pp.head0);
          hipLaunchKernelGGL((prompt_rows_kernel<KV_T, HD>), dim3(n_tiles * pp.heads + (pp.head0 ? 0 : n_seq)), dim3(256), 0, c.stream, pp);
          hipLaunchKernelGGL((attn_prompt_kernel<KV_T, HD>), dim3(pp.heads * G, tok_tiles, n_ks), dim3(256), 0, c.stream, pp);
        }
      };
      if (kv->dtype == CAI_KV_F16) both(__half()); else if (kv->dtype == CAI_KV_I8) both(int8_t()); else both(float());
      if (n_ks > 1) hipLaunchKernelGGL(prompt_merge_kernel<HD>, dim3(n_seq, (q_heads + 3) / 4), dim3(512), 0, c.stream, pp, n_ks);
    };
    if (p.hd == 64) go(std::integral_constant<int, 64>()); else go(std::integral_constant<int, 128>());
    return CAI_OK;
  }
  // one work-group per (slice, KV head) serving the whole group of query heads, or one per (slice, query head)
  // (the first fetches K and V once but has G times fewer work-groups: it needs a grid that fills the chip by itself)
  if (form == ATTN_GROUPED_CORES)
    rc = kv->dtype == CAI_KV_I8 ? launch_group_mfma<int8_t>(p, n_seq, c.stream) : launch_group_mfma<__half>(p, n_seq, c.stream);
  else if (grouped)
    rc = kv->dtype == CAI_KV_I8 ? launch_group<int8_t>(p, n_seq, c.stream) : kv->dtype == CAI_KV_F16 ? launch_group<__half>(p, n_seq, c.stream) : launch_group<float>(p, n_seq, c.stream);
  else
    rc = kv->dtype == CAI_KV_I8 ? launch_split_head<int8_t>(p, n_seq, c.stream) : kv->dtype == CAI_KV_F16 ? launch_split_head<__half>(p, n_seq, c.stream) : launch_split_head<float>(p, n_seq, c.stream);
  if (rc) return rc;
  if (p.n_splits > 1 && !p.merge_cnt)
  {
    auto merge = [&](auto kern, const auto& params) {
      hipLaunchKernelGGL(kern, dim3(q_heads, n_seq), dim3(512), 0, c.stream, p.pos, (const float*)p.part, p.out, (long long)p.out_stride,
                         p.q_heads | p.kv_heads << 16, p.n_splits | p.hd << 16, p.split_len, params);
    };
    const AttnParams& rows = p;
    if (p.planes.hi) { if (p.n_splits > 96) merge(attn_merge_kernel<32, true>, p); else merge(attn_merge_kernel<12, true>, p); }
    else if (p.n_splits > 96) merge(attn_merge_kernel<32, false>, rows);
    else merge(attn_merge_kernel<12, false>, rows);
  }
  return CAI_OK;
}

// ------------------------------------------------------------------------------------------
// cache lifetime
// ------------------------------------------------------------------------------------------
int kv_bucket_rows(const cai_kv_s* kv, int needed_rows)
{
  if (kv->evict_cap > 0) return 0;                       // a rolling cache is short by construction: its own geometry
  int rows = 1024;
  while (rows < needed_rows && rows < kv->max_ctx) rows *= 2;
  return rows >= kv->max_ctx ? 0 : rows;
}

void kv_geometry(const cai_kv_s* kv, int rows, int* split_len, int* n_splits)
{
  if (rows <= 0 || rows > kv->max_ctx) rows = kv->max_ctx;
  // few, fat slices: every extra slice costs the merging work-group another device-coherent load round,
  // while one CU sustains only ~20 GB/s, so a slice should stay under ~100 KB
  constexpr int sl_max = 256;
  int sl = (rows + 15) / 16; sl = (sl + 31) / 32 * 32; if (sl < 32) sl = 32; if (sl > sl_max) sl = sl_max;
  // From 8192 rows on the grouped kernel (K and V fetched once for all query heads of a KV head) is the fast one, but it needs
  // about one work-group per CU: with few KV heads the slices are halved until slices x KV heads fill the chip.  7B shape, 4 KV
  // heads, 7000 rows: 256-row slices take the per-head kernel at 31.8 us per launch, 128-row slices the grouped one at 23.3
  // (445 -> 494 tok/s); at 4096 rows both forms take the same time and the longer slices stay.
  if (rows >= 8192 && (kv->head_dim & 7) == 0)
    while (sl > 64 && kv->kv_heads * ((rows + sl - 1) / sl) < ctx().n_cu) sl /= 2;
  // a head's whole K (or V) plane of at most 64 KB is one slice: a single work-group streams it in a few microseconds and
  // the merge launch disappears (small models at short contexts are bound by launches, not by bytes)
  constexpr int single_bytes = 65536;
  if ((int64_t)rows * kv->head_dim * (kv->dtype == CAI_KV_F16 ? 2 : kv->dtype == CAI_KV_I8 ? 1 : 4) <= single_bytes) sl = (rows + 31) / 32 * 32;
  *split_len = sl; *n_splits = (rows + sl - 1) / sl;
}

static __global__ void iota_kernel(int32_t* __restrict__ dst, int n)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = i;
}

int kv_alloc(cai_kv_s* kv, int n_seq, int n_layers, int kv_heads, int head_dim, int max_ctx, int dtype, bool positions)
{
  if (n_seq < 1 || n_layers < 1 || kv_heads < 1 || head_dim < 2 || (head_dim & 1) || (head_dim > 64 && (head_dim & 3)) || head_dim > 128 || max_ctx < 1)
    return set_error(CAI_ERR_INVALID, "kv cache: bad geometry seq=%d layers=%d kv_heads=%d head_dim=%d max_ctx=%d", n_seq, n_layers, kv_heads, head_dim, max_ctx);
  if (dtype != CAI_KV_F32 && dtype != CAI_KV_F16 && dtype != CAI_KV_I8) return set_error(CAI_ERR_INVALID, "kv cache: dtype %d", dtype);
  kv->n_seq = n_seq; kv->n_layers = n_layers; kv->kv_heads = kv_heads; kv->head_dim = head_dim; kv->max_ctx = max_ctx; kv->dtype = dtype;
  kv->len.assign((size_t)n_seq * n_layers, 0);
  kv->geo_rows = 0;
  kv_geometry(kv, 0, &kv->split_len, &kv->n_splits);
  kv->n_splits_alloc = kv->n_splits;
  for (int rows = 1024; rows < max_ctx; rows *= 2) { int sl, ns; kv_geometry(kv, rows, &sl, &ns); kv->n_splits_alloc = std::max(kv->n_splits_alloc, ns); }
  const size_t bytes = (size_t)kv->seq_elems() * n_seq * kv->elem();
  // (the kernels index slices generically; the bound keeps the per-row scratch of prompts and windows - one partial result per
  // slice and query head - within reason: 131072 rows are 512 slices)
  if (kv->n_splits > 512) return set_error(CAI_ERR_UNSUPPORTED, "kv cache: max_ctx %d needs %d slices of %d rows (limit 512: 131072 rows)", max_ctx, kv->n_splits, kv->split_len);
  CAI_HIP(hipMalloc(&kv->k, bytes));
  CAI_HIP(hipMalloc(&kv->v, bytes));
  CAI_HIP(hipMemsetAsync(kv->k, 0, bytes, ctx().stream));
  CAI_HIP(hipMemsetAsync(kv->v, 0, bytes, ctx().stream));
  if (dtype == CAI_KV_I8) {
    const size_t sb = (size_t)kv->seq_rows() * n_seq * sizeof(float);
    CAI_HIP(hipMalloc(&kv->ks, sb));
    CAI_HIP(hipMalloc(&kv->vs, sb));
    CAI_HIP(hipMemsetAsync(kv->ks, 0, sb, ctx().stream));
    CAI_HIP(hipMemsetAsync(kv->vs, 0, sb, ctx().stream));
  }
  kv->part_q_heads = kv_heads * 8;
  CAI_HIP(hipMalloc(&kv->part, (size_t)n_seq * kv->part_q_heads * kv->n_splits_alloc * (head_dim + 2) * sizeof(float)));
  CAI_HIP(hipMalloc(&kv->d_len, sizeof(int32_t) * ((size_t)n_seq + (positions ? max_ctx : 0))));
  if (positions) {
    kv->d_iota = kv->d_len + n_seq;
    hipLaunchKernelGGL(iota_kernel, dim3((max_ctx + 255) / 256), dim3(256), 0, ctx().stream, kv->d_iota, max_ctx);
  }
  CAI_HIP(hipMalloc((void**)&kv->merge_cnt, sizeof(unsigned) * n_seq * kv->part_q_heads));
  CAI_HIP(hipMemsetAsync(kv->merge_cnt, 0, sizeof(unsigned) * n_seq * kv->part_q_heads, ctx().stream));
  CAI_HIP(hipStreamSynchronize(ctx().stream));
  return CAI_OK;
}

void kv_free(cai_kv_s* kv)
{
  if (kv->k) (void)hipFree(kv->k);
  if (kv->v) (void)hipFree(kv->v);
  if (kv->ks) (void)hipFree(kv->ks);
  if (kv->vs) (void)hipFree(kv->vs);
  kv->ks = kv->vs = nullptr;
  if (kv->pq) (void)hipFree(kv->pq);
  kv->pq = nullptr; kv->pq_cap = 0;
  if (kv->part) (void)hipFree(kv->part);
  if (kv->d_len) (void)hipFree(kv->d_len);
  if (kv->merge_cnt) (void)hipFree(kv->merge_cnt);
  kv->merge_cnt = nullptr; kv->d_iota = nullptr;
  kv->k = kv->v = nullptr; kv->part = nullptr; kv->d_len = nullptr;
}

// Deep copy of the live rows of one sequence (TNNetDecoderSessionSnapshot, neural/neuraldecode.pas:1089-1142).
int kv_snapshot(cai_kv_s* kv, int seq, cai_kv_snap_s** out)
{
  cai_kv_snap_s* s = new cai_kv_snap_s();
  auto drop = [&](int code) { cai_kv_snap_destroy(s); return code; };   // every error path releases what the snapshot holds so far
  s->n_layers = kv->n_layers; s->kv_heads = kv->kv_heads; s->head_dim = kv->head_dim; s->dtype = kv->dtype;
  s->evict_sinks = kv->evict_sinks; s->evict_cap = kv->evict_cap;
  s->len.resize(kv->n_layers);
  int rows = 0;
  for (int l = 0; l < kv->n_layers; l++) { s->len[l] = kv->len_at(seq, l); rows = std::max(rows, kv->live(s->len[l])); }
  s->rows = rows;
  if (rows > 0) {
    const size_t bytes = (size_t)kv->n_layers * kv->kv_heads * rows * kv->head_dim * kv->elem();
    if (hipMalloc(&s->k, bytes) != hipSuccess || hipMalloc(&s->v, bytes) != hipSuccess)
      return (void)hipGetLastError(), drop(set_error(CAI_ERR_NOMEM, "kv snapshot: out of device memory (%zu bytes)", 2 * bytes));
    const size_t row_b = (size_t)kv->head_dim * kv->elem();
    for (int which = 0; which < 2; which++) {
      const char* src = (const char*)(which ? kv->v : kv->k) + (size_t)seq * kv->seq_elems() * kv->elem();
      char* dst = (char*)(which ? s->v : s->k);
      // [layer*kv_heads] planes of max_ctx rows -> planes of `rows` rows
      const hipError_t e = hipMemcpy2DAsync(dst, (size_t)rows * row_b, src, (size_t)kv->max_ctx * row_b, (size_t)rows * row_b,
                                            (size_t)kv->n_layers * kv->kv_heads, hipMemcpyDeviceToDevice, ctx().stream);
      if (e != hipSuccess) return drop(hip_fail(e, "kv snapshot copy", __FILE__, __LINE__));
    }
    if (kv->dtype == CAI_KV_I8) {     // the row scales travel with the codes
      const size_t sb = (size_t)kv->n_layers * kv->kv_heads * rows * sizeof(float);
      if (hipMalloc(&s->ks, sb) != hipSuccess || hipMalloc(&s->vs, sb) != hipSuccess)
        return (void)hipGetLastError(), drop(set_error(CAI_ERR_NOMEM, "kv snapshot: out of device memory (%zu bytes)", 2 * sb));
      for (int which = 0; which < 2; which++) {
        const hipError_t e = hipMemcpy2DAsync(which ? s->vs : s->ks, (size_t)rows * 4, (which ? kv->vs : kv->ks) + (size_t)seq * kv->seq_rows(), (size_t)kv->max_ctx * 4,
                                              (size_t)rows * 4, (size_t)kv->n_layers * kv->kv_heads, hipMemcpyDeviceToDevice, ctx().stream);
        if (e != hipSuccess) return drop(hip_fail(e, "kv snapshot copy", __FILE__, __LINE__));
      }
    }
    { const hipError_t e = hipStreamSynchronize(ctx().stream); if (e != hipSuccess) return drop(hip_fail(e, "kv snapshot sync", __FILE__, __LINE__)); }
  }
  *out = s;
  return CAI_OK;
}

int kv_restore(cai_kv_s* kv, int seq, const cai_kv_snap_s* s)
{
  if (s->n_layers != kv->n_layers || s->kv_heads != kv->kv_heads || s->head_dim != kv->head_dim)
    return set_error(CAI_ERR_INVALID, "kv restore: snapshot geometry differs from the cache");
  if (s->dtype != kv->dtype) return set_error(CAI_ERR_INVALID, "kv restore: snapshot element type differs from the cache (mode must match)");
  if (s->evict_sinks != kv->evict_sinks || s->evict_cap != kv->evict_cap)
    return set_error(CAI_ERR_INVALID, "kv restore: snapshot was taken under eviction (%d sinks, cap %d), the cache runs (%d, %d)", s->evict_sinks, s->evict_cap, kv->evict_sinks, kv->evict_cap);
  if (s->rows > kv->max_ctx) return set_error(CAI_ERR_INVALID, "kv restore: snapshot holds %d rows, cache %d", s->rows, kv->max_ctx);
  if (s->rows > 0) {
    const size_t row_b = (size_t)kv->head_dim * kv->elem();
    for (int which = 0; which < 2; which++) {
      char* dst = (char*)(which ? kv->v : kv->k) + (size_t)seq * kv->seq_elems() * kv->elem();
      const char* src = (const char*)(which ? s->v : s->k);
      CAI_HIP(hipMemcpy2DAsync(dst, (size_t)kv->max_ctx * row_b, src, (size_t)s->rows * row_b, (size_t)s->rows * row_b,
                               (size_t)kv->n_layers * kv->kv_heads, hipMemcpyDeviceToDevice, ctx().stream));
    }
    if (kv->dtype == CAI_KV_I8)
      for (int which = 0; which < 2; which++)
        CAI_HIP(hipMemcpy2DAsync((which ? kv->vs : kv->ks) + (size_t)seq * kv->seq_rows(), (size_t)kv->max_ctx * 4, which ? s->vs : s->ks, (size_t)s->rows * 4,
                                 (size_t)s->rows * 4, (size_t)kv->n_layers * kv->kv_heads, hipMemcpyDeviceToDevice, ctx().stream));
    CAI_HIP(hipStreamSynchronize(ctx().stream));
  }
  for (int l = 0; l < kv->n_layers; l++) kv->len_at(seq, l) = s->len[l];
  return CAI_OK;
}

// Sequence dst becomes a copy of sequence src (the cache-forking step of a beam search: every survivor continues from its
// parent's rows, neural/neuraldecode.pas:1436-1449): the live rows of every (layer, KV head) plane move device to device, on
// the library's stream, without a snapshot in between.
int kv_fork(cai_kv_s* kv, int src, int dst)
{
  if (src == dst) return CAI_OK;
  int rows = 0;
  for (int l = 0; l < kv->n_layers; l++) rows = std::max(rows, kv->live(kv->len_at(src, l)));
  if (rows > 0) {
    const size_t row_b = (size_t)kv->head_dim * kv->elem(), seq_b = (size_t)kv->seq_elems() * kv->elem();
    for (int which = 0; which < 2; which++) {
      char* base = (char*)(which ? kv->v : kv->k);
      CAI_HIP(hipMemcpy2DAsync(base + dst * seq_b, (size_t)kv->max_ctx * row_b, base + src * seq_b, (size_t)kv->max_ctx * row_b, (size_t)rows * row_b,
                               (size_t)kv->n_layers * kv->kv_heads, hipMemcpyDeviceToDevice, ctx().stream));
    }
    if (kv->dtype == CAI_KV_I8)
      for (int which = 0; which < 2; which++) {
        float* base = which ? kv->vs : kv->ks;
        CAI_HIP(hipMemcpy2DAsync(base + (size_t)dst * kv->seq_rows(), (size_t)kv->max_ctx * 4, base + (size_t)src * kv->seq_rows(), (size_t)kv->max_ctx * 4,
                                 (size_t)rows * 4, (size_t)kv->n_layers * kv->kv_heads, hipMemcpyDeviceToDevice, ctx().stream));
      }
  }
  for (int l = 0; l < kv->n_layers; l++) kv->len_at(dst, l) = kv->len_at(src, l);
  return CAI_OK;
}

}  // namespace cai

// ------------------------------------------------------------------------------------------
// C ABI
// ------------------------------------------------------------------------------------------
using namespace cai;

extern "C" int cai_kv_create(int n_layers, int kv_heads, int head_dim, int max_ctx, int kv_dtype, cai_kv_t* out)
{
  CAI_ENTER();
  CAI_READY();
  CAI_REQUIRE(out, "cai_kv_create: null out");
  cai_kv_s* kv = new cai_kv_s();
  const int rc = kv_alloc(kv, 1, n_layers, kv_heads, head_dim, max_ctx, kv_dtype, true);
  if (rc) { kv_free(kv); delete kv; return rc; }
  *out = kv;
  return CAI_OK;
}

extern "C" int cai_kv_destroy(cai_kv_t kv)
{
  CAI_ENTER();
  if (!kv) return CAI_OK;
  (void)hipStreamSynchronize(ctx().stream);
  kv_free(kv); delete kv;
  return CAI_OK;
}

extern "C" int cai_kv_reset(cai_kv_t kv)
{
  CAI_ENTER();
  CAI_REQUIRE(kv, "cai_kv_reset: null cache");
  std::fill(kv->len.begin(), kv->len.end(), 0);
  return CAI_OK;
}

extern "C" int cai_kv_truncate(cai_kv_t kv, int n)
{
  CAI_ENTER();
  CAI_REQUIRE(kv, "cai_kv_truncate: null cache");
  CAI_REQUIRE(n >= 0, "cai_kv_truncate: negative length %d", n);
  for (int l : kv->len)
    if (l > n && kv->evict_cap > 0 && l > kv->evict_cap) return set_error(CAI_ERR_STATE, "cai_kv_truncate: %d tokens streamed under eviction, the rows before %d are gone", l, l - (kv->evict_cap - kv->evict_sinks));
  for (auto& l : kv->len) if (l > n) l = n;
  return CAI_OK;
}

// Sink + recent-window eviction (TNNetStreamingDecoder.EnableEviction / DisableEviction, neural/neuraldecode.pas:5722-5735).
int cai::kv_set_eviction(cai_kv_s* kv, int sinks, int recent)
{
  const int cap = sinks + recent;
  if (sinks < 0 || recent < 0 || (cap > 0 && recent < 1)) return set_error(CAI_ERR_INVALID, "eviction: %d sink tokens, recent window %d", sinks, recent);
  if (cap > kv->max_ctx) return set_error(CAI_ERR_INVALID, "eviction: %d sinks + %d recent exceed the cache's %d rows", sinks, recent, kv->max_ctx);
  // rows sit at slot = position until the stream passes the cap, so the policy may change freely before that
  const int limit = std::min(kv->evict_cap > 0 ? kv->evict_cap : kv->max_ctx, cap > 0 ? cap : kv->max_ctx);
  for (int n : kv->len)
    if (n > limit) return set_error(CAI_ERR_STATE, "eviction: a sequence already holds %d tokens, past the %d the change allows", n, limit);
  kv->evict_sinks = cap > 0 ? sinks : 0; kv->evict_cap = cap;
  return CAI_OK;
}

extern "C" int cai_kv_set_eviction(cai_kv_t kv, int sink_tokens, int recent_window)
{
  CAI_ENTER();
  CAI_REQUIRE(kv, "cai_kv_set_eviction: null cache");
  return kv_set_eviction(kv, sink_tokens, recent_window);
}

extern "C" int cai_kv_rows(cai_kv_t kv, int layer, int* rows_out)
{
  CAI_ENTER();
  CAI_REQUIRE(kv && rows_out, "cai_kv_rows: null argument");
  CAI_REQUIRE(layer >= 0 && layer < kv->n_layers, "cai_kv_rows: layer %d of %d", layer, kv->n_layers);
  *rows_out = kv->live(kv->len_at(0, layer));
  return CAI_OK;
}

extern "C" int cai_kv_len(cai_kv_t kv, int layer, int* len_out)
{
  CAI_ENTER();
  CAI_REQUIRE(kv && len_out, "cai_kv_len: null argument");
  CAI_REQUIRE(layer >= 0 && layer < kv->n_layers, "cai_kv_len: layer %d of %d", layer, kv->n_layers);
  *len_out = kv->len_at(0, layer);
  return CAI_OK;
}

extern "C" int cai_kv_snapshot(cai_kv_t kv, cai_kv_snap_t* out)
{
  CAI_ENTER();
  CAI_READY();
  CAI_REQUIRE(kv && out, "cai_kv_snapshot: null argument");
  return kv_snapshot(kv, 0, out);
}

extern "C" int cai_kv_restore(cai_kv_t kv, cai_kv_snap_t snap)
{
  CAI_ENTER();
  CAI_READY();
  CAI_REQUIRE(kv && snap, "cai_kv_restore: null argument");
  return kv_restore(kv, 0, snap);
}

extern "C" int cai_kv_snap_destroy(cai_kv_snap_t s)
{
  CAI_ENTER();
  if (!s) return CAI_OK;
  if (s->net) net_snap_free(s->net);
  if (s->k) (void)hipFree(s->k);
  if (s->v) (void)hipFree(s->v);
  if (s->ks) (void)hipFree(s->ks);
  if (s->vs) (void)hipFree(s->vs);
  delete s;
  return CAI_OK;
}

// one layer of sequence 0 <-> packed host rows; dir 0 = device to host
static int kv_layer_copy(cai_kv_s* kv, int layer, int len, void* k, void* v, float* ks, float* vs, int to_device)
{
  if (len == 0) return CAI_OK;
  const size_t row_b = (size_t)kv->head_dim * kv->elem();
  const hipMemcpyKind kind = to_device ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost;
  auto copy2d = [&](char* dev, char* host, size_t unit) -> hipError_t {
    return to_device ? hipMemcpy2DAsync(dev, (size_t)kv->max_ctx * unit, host, (size_t)len * unit, (size_t)len * unit, (size_t)kv->kv_heads, kind, ctx().stream)
                     : hipMemcpy2DAsync(host, (size_t)len * unit, dev, (size_t)kv->max_ctx * unit, (size_t)len * unit, (size_t)kv->kv_heads, kind, ctx().stream);
  };
  CAI_HIP(copy2d((char*)kv->k + (size_t)layer * kv->layer_elems() * kv->elem(), (char*)k, row_b));
  CAI_HIP(copy2d((char*)kv->v + (size_t)layer * kv->layer_elems() * kv->elem(), (char*)v, row_b));
  if (kv->dtype == CAI_KV_I8) {
    CAI_HIP(copy2d((char*)(kv->ks + (size_t)layer * kv->layer_rows()), (char*)ks, 4));
    CAI_HIP(copy2d((char*)(kv->vs + (size_t)layer * kv->layer_rows()), (char*)vs, 4));
  }
  CAI_HIP(hipStreamSynchronize(ctx().stream));
  return CAI_OK;
}

extern "C" int cai_kv_export_layer(cai_kv_t kv, int layer, void* k, void* v, float* k_scales, float* v_scales)
{
  CAI_ENTER();
  CAI_READY();
  CAI_REQUIRE(kv && k && v, "cai_kv_export_layer: null argument");
  CAI_REQUIRE(layer >= 0 && layer < kv->n_layers, "cai_kv_export_layer: layer %d of %d", layer, kv->n_layers);
  CAI_REQUIRE(kv->dtype != CAI_KV_I8 || (k_scales && v_scales), "cai_kv_export_layer: an int8 cache needs the scale outputs");
  return kv_layer_copy(kv, layer, kv->live(kv->len_at(0, layer)), k, v, k_scales, v_scales, 0);
}

extern "C" int cai_kv_import_layer(cai_kv_t kv, int layer, int len, const void* k, const void* v, const float* k_scales, const float* v_scales)
{
  CAI_ENTER();
  CAI_READY();
  CAI_REQUIRE(kv && (len == 0 || (k && v)), "cai_kv_import_layer: null argument");
  CAI_REQUIRE(layer >= 0 && layer < kv->n_layers, "cai_kv_import_layer: layer %d of %d", layer, kv->n_layers);
  CAI_REQUIRE(len >= 0 && len <= kv->max_ctx && (kv->evict_cap == 0 || len <= kv->evict_cap), "cai_kv_import_layer: %d rows, cache holds %d", len, kv->evict_cap ? kv->evict_cap : kv->max_ctx);
  CAI_REQUIRE(kv->dtype != CAI_KV_I8 || len == 0 || (k_scales && v_scales), "cai_kv_import_layer: an int8 cache needs the row scales");
  const int rc = kv_layer_copy(kv, layer, len, const_cast<void*>(k), const_cast<void*>(v), const_cast<float*>(k_scales), const_cast<float*>(v_scales), 1);
  if (rc) return rc;
  kv->len_at(0, layer) = len;
  return CAI_OK;
}

extern "C" int cai_attn_decode(cai_kv_t kv, int layer, const float* qkv, int q_heads, int window, float softcap,
                               float* out, int flags)
{
  CAI_ENTER();
  CAI_READY();
  CAI_REQUIRE(kv && qkv && out, "cai_attn_decode: null argument");
  CAI_REQUIRE(layer >= 0 && layer < kv->n_layers, "cai_attn_decode: layer %d of %d", layer, kv->n_layers);
  CAI_REQUIRE(q_heads > 0 && q_heads % kv->kv_heads == 0, "cai_attn_decode: %d query heads vs %d KV heads", q_heads, kv->kv_heads);
  Context& c = ctx();
  const int len = kv->len_at(0, layer);
  if (len >= kv->max_ctx && kv->evict_cap == 0) return set_error(CAI_ERR_STATE, "cai_attn_decode: cache full (%d rows)", kv->max_ctx);
  const int hd = kv->head_dim;
  const size_t in_b = (size_t)(q_heads + 2 * kv->kv_heads) * hd * sizeof(float), out_b = (size_t)q_heads * hd * sizeof(float);
  // The kernels below only read the row (no norm and no rotation in place here), so a device row is used where it lies: its copy
  // and the upload of the position below were two more launches (40 / 8 heads x 128 behind 8191 int8 rows: 29.4 us with both,
  // 24.1 without).  It is still copied where the wide loads need an alignment that it lacks,
  // and where the result is written over it, which would race with work-groups that have yet to read their part.
  float* d_out = out;
  int rc;
  if (!(flags & CAI_Y_DEVICE)) { rc = ensure_stage(&c.stage_out, &c.stage_out_cap, out_b); if (rc) return rc; d_out = (float*)c.stage_out; }
  const char *x0 = (const char*)qkv, *y0 = (const char*)d_out;
  float* d_qkv = const_cast<float*>(qkv);
  if (!(flags & CAI_X_DEVICE) || ((uintptr_t)qkv & 15) || (x0 < y0 + out_b && y0 < x0 + in_b)) {
    rc = ensure_stage(&c.stage_in, &c.stage_in_cap, in_b); if (rc) return rc;
    CAI_HIP(hipMemcpyAsync(c.stage_in, qkv, in_b, (flags & CAI_X_DEVICE) ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, c.stream));
    d_qkv = (float*)c.stage_in;
  }
  // The kernels read the position through a pointer (a captured step moves it on the device): here it is an entry of the cache's
  // table of positions instead of an upload of four bytes.  A rolling cache counts past the table.
  const int32_t* d_pos = kv->d_iota && len < kv->max_ctx ? kv->d_iota + len : kv->d_len;
  if (d_pos == kv->d_len) {
    c.h_small[0] = len;
    CAI_HIP(hipMemcpyAsync(kv->d_len, c.h_small, sizeof(int32_t), hipMemcpyHostToDevice, c.stream));
  }
  kv->geo_rows = kv_bucket_rows(kv, len + 1);
  (void)hipGetLastError();      // what an earlier call of this thread left is no error of these launches
  rc = launch_attn_step(kv, layer, d_qkv, 0, 1, q_heads, window, softcap, nullptr, d_pos, d_out, 0, 0, 0, nullptr);
  if (rc) return rc;
  CAI_HIP(hipGetLastError());
  if (flags & CAI_Y_DEVICE) {
    // The signal behind the row says that launches can read it: memory of this card.  A row anywhere else (pinned, managed, a peer's) is there for the host
    // when the stream has ended.  40 / 8 heads x 128 behind 8191 int8 rows: 24.1 us with hipStreamSynchronize, 22.1 with the signal (the question
    // about the address is asked while the kernels run).
    hipPointerAttribute_t at{};
    const bool known = hipPointerGetAttributes(&at, out) == hipSuccess;
    if (!known) (void)hipGetLastError();      // (the question's)
    if (known && at.type == hipMemoryTypeDevice && at.device == c.device) {
      const HostSignal done = host_signal_next();
      launch_host_signal(done);
      CAI_HIP(hipGetLastError());
      rc = host_signal_wait(done); if (rc) return rc;
    } else CAI_HIP(hipStreamSynchronize(c.stream));
  } else {
    const HostCopy res = {out, d_out, out_b};
    rc = fetch_to_host(&res, 1); if (rc) return rc;
  }
  kv->len_at(0, layer) = len + 1;
  return CAI_OK;
}

// The kernel (ATTN_PER_HEAD, ATTN_GROUPED, ATTN_GROUPED_CORES) that a decoding step of n_seq sequences over caches of `rows` rows takes.  For the tests of the
// kernels, which say by it what they reach; host only, not part of the interface in caihip.h.
extern "C" int cai_attn_form(int n_seq, int q_heads, int kv_heads, int head_dim, int rows, int kv_dtype, int normed)
{
  CAI_ENTER();
  CAI_REQUIRE(n_seq >= 1 && kv_heads >= 1 && q_heads >= kv_heads && head_dim >= 2 && rows >= 1, "cai_attn_form: bad argument");
  cai_kv_s kv;
  kv.kv_heads = kv_heads; kv.head_dim = head_dim; kv.max_ctx = rows; kv.dtype = kv_dtype;
  int split_len, n_splits;
  kv_geometry(&kv, 0, &split_len, &n_splits);
  return attn_form(&kv, q_heads, n_seq, split_len, n_splits, false, normed != 0);
}
