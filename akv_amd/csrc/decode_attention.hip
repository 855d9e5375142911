// GQA decode attention with attention sinks over compacted page-one indices
// (gfx950, MFMA).  The consumer of the Drop + Reposition metadata: one decode
// step reads each request's keys through kv_indptr / kv_indices (full layers)
// or the window-limited indices (sliding-window layers) and normalises with a
// per-head sink logit:
//   o_h = sum_j exp(s_hj) v_j / (sum_j exp(s_hj) + exp(sink_h)),
//   s_hj = scale * q_h . k_j
// which equals the reference's o * sigmoid(lse - sink)
// (akv/system/sglang/srt/layers/attention/context_backend.py:254-272).
//
// Split-K: workgroup = (chunk of keys, KV head, request), in passes of 256
// keys: D / 16 waves of 4096 / D keys each.  A wave brings all its keys of a
// pass at once -- slots, then K into registers in the operand layout and V
// straight into its own LDS tile -- so a pass is two round trips, whatever its
// length, and needs no barrier.  S^T[keys x 16 heads] = K . Q^T on
// v_mfma_f32_16x16x32_bf16 (the group's q heads padded to 16), one softmax
// step per pass, then O^T[D x 16] += V^T . P^T, where P^T is already in the
// B-operand layout of the second MFMA (a lane's keys 4 (l/16) + i of two
// 16-key tiles) and V^T comes from ds_read_b64_tr_b16.  The waves' results
// meet in LDS at the end.  A combine kernel merges the chunks and the sink;
// when every request fits one chunk (a sliding-window layer) the first kernel
// applies the sink itself and the combine is not launched.
//
// MFMA 16x16x32 bf16 lane layout (verified on gfx950): lane l supplies
// A[l%16][k(l, i)] and B[k(l, i)][l%16], i < 8, and holds D[4(l/16)+i][l%16].
#include <algorithm>
#include <cmath>
#include <mutex>

#include "common.h"

namespace akv {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) u32x4 global_u32x4;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kPass = 256;  // keys of a workgroup's pass
constexpr float kLog2e = 1.4426950408889634f;

struct AttnArgs {
  const __bf16* q;
  int64_t q_stride_b, q_stride_h;
  const __bf16* k;
  const __bf16* v;
  int64_t k_stride_slot, k_stride_head, v_stride_slot, v_stride_head;
  const int32_t* kv_indptr;
  const int32_t* kv_indices;
  const float* sinks;
  const int32_t* gate;  // compaction status word, or nullptr
  float scale_log2;  // scale * log2(e)
  void* out;
  int32_t out_f32;
  int64_t out_stride_b, out_stride_h;
  int32_t n_requests, q_heads, kv_heads, group, chunks;
  int32_t max_passes;  // passes per workgroup with which `chunks` chunks hold max_len keys
  // the grid: chunks fastest, then heads or requests; its chunks turn by one
  // every 2^turn_shift (request, head) pairs, and again every 4 and 32 times that
  int32_t heads_last, turn_shift;
  int32_t q_vectors;   // q rows are 16-byte aligned
  float* partial;  // [B][Hkv][chunks][16][D + 2]  (o..., m, l)
};

// Passes of a workgroup: up to four where that still leaves eight workgroups
// per CU (a quarter of the partial results).
constexpr int32_t kMaxPasses = 4;
constexpr int64_t kEnoughGroups = 8 * 256;

// Keys of a chunk of a request of `len` keys in a batch of `total`.  The host
// knows a bound of the longest request only, which may be far off (a captured
// graph's, a context length); the batch itself says how many workgroups its
// keys can feed.  Both kernels compute it.
__device__ __forceinline__ int32_t chunk_keys_of(const AttnArgs& a, int32_t len, int32_t total) {
  int32_t passes = 1;
  while (passes < a.max_passes && (static_cast<int64_t>(total) * a.kv_heads >= kEnoughGroups * 2 * passes * kPass ||
                                   len > static_cast<int64_t>(a.chunks) * passes * kPass))
    passes *= 2;
  // one chunk of two passes rather than two of one
  if (passes == 1 && a.max_passes > 1 && len <= 2 * kPass) passes = 2;
  // equal chunks, in whole waves of keys
  const uint32_t most = passes * kPass, n = (static_cast<uint32_t>(len) + most - 1) / most;
  return n > 1 ? ((static_cast<uint32_t>(len) + n - 1) / n + 63) / 64 * 64 : most;
}

// The V rows of keys past a chunk's end: their weights are 0, and 0 times
// whatever a real row holds (infinities) need not be 0.
static __device__ __attribute__((aligned(16))) const uint32_t zero_row[64] = {};

// 16-byte chunk c of V row r sits at chunk c ^ swz(r) of its LDS row: distinct
// bank groups for the 8 rows of a transposing read, a chunk pair stays adjacent.
template <int D>
__device__ __forceinline__ int swz(int r) { return D == 64 ? r & 6 : (r & 7) << 1; }

// Bound by the HBM's random rows: 32 GPT-OSS requests of ~20k keys (1.31 GB)
// take 252 us with the combine, 5.2 TB/s, where a large copy reaches 4.9 (read
// + write); with one wave per 256 keys, 16 at a time, they took 267.  Four
// requests of 1-6k keys, where the chain of round trips counts, take 12 us
// against 22; a 128-key window 4.3 against 9.3.  The next pass's slots arrive
// with this pass's rows (12 Llama-3 requests and the like 2-8%).
//
// The grid follows the host's bound, so its live workgroups must not depend
// on where they stand in it: workgroups go round robin to the XCDs and, by what
// the times show, within an XCD to its shader engines, so a grid whose first chunks are the live (or
// the long) ones would keep to a few of them.  Its chunks therefore turn from
// pair to pair, at the period of the XCDs and at 4 and 32 times that, and a
// request's chunks are equally long.  Without both, and with passes from the
// bound: 64 GPT-OSS requests of 2000 keys at a bound of 32768 took 372 us (52
// now), 300 of 1100 at 1100 232 (156), 128 of 100-8000 218 (133).  Chunks
// fastest and then heads, so neighbouring workgroups read different rows;
// where there are few chunks (kFewChunks), requests before heads: 256 x 1000
// keys of all heads side by side 4.4 TB/s, of different requests 5.5; with 20
// chunks it is 0.4-1% slower, and 5% for ragged requests.  A chunk's heads one
// after the other on one XCD measured 4% slower (295 against 284 us for the
// decode step).
template <int D>
__global__ void __launch_bounds__(4 * D, 4) decode_attention_partial_kernel(const AttnArgs a) {
  constexpr int kWaves = D / 16;
  constexpr int kKeys = kPass / kWaves;       // keys of a wave's pass: 64 / 32
  constexpr int kTiles = kKeys / 16;          // 16-key tiles
  constexpr int kSteps = D / 32;              // MFMA k-steps over the head dim
  constexpr int kDTiles = D / 16;
  constexpr int kChunks = D / 8;              // 16-byte chunks of a row
  constexpr int kRows = 64 / kChunks;         // V rows of one wave-wide load
  constexpr int kOut = D + 4;                 // floats of an O row in LDS (padded: no bank conflicts)
  constexpr int kWaveBytes = kKeys * D * 2 > 16 * kOut * 4 ? kKeys * D * 2 : 16 * kOut * 4;
  __shared__ __attribute__((aligned(16))) char tiles[kWaves][kWaveBytes];
  __shared__ float s_m[kWaves][16], s_l[kWaves][16];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = a.heads_last ? blockIdx.y : blockIdx.z;
  const int g = a.heads_last ? blockIdx.z : blockIdx.y;
  const uint32_t pair = (blockIdx.z * gridDim.y + blockIdx.y) >> a.turn_shift;
  const uint32_t turn = pair + (pair >> 2) + (pair >> 5);
  int chunk = blockIdx.x + turn % a.chunks;
  if (chunk >= a.chunks) chunk -= a.chunks;
  const int64_t begin = a.kv_indptr[b];
  const int32_t len = max(a.kv_indptr[b + 1] - a.kv_indptr[b], 0);
  const int32_t total = a.kv_indptr[a.n_requests] - a.kv_indptr[0];
  // a closed gate stops the workgroup before its key indices and rows
  if (gated(a.gate)) return;
  const int32_t chunk_keys = chunk_keys_of(a, len, total);
  const int64_t c0 = static_cast<int64_t>(chunk) * chunk_keys;
  // an empty chunk is not read by the combine; with one chunk the output is 0
  if (c0 >= len && a.chunks > 1) return;
  const int n = static_cast<int>(len - c0 < chunk_keys ? (len > c0 ? len - c0 : 0) : chunk_keys);
  const int32_t* idx = a.kv_indices + begin + c0;
  const int col = lane & 15;   // head within the group (B / D layout column)
  const int quad = lane >> 4;  // 0..3

  // Q^T operand: lane supplies q[head col][dims 32 st + 8 quad + i]
  bf16x8 qop[kSteps];
  {
    // columns past the group repeat its last head; they are never stored
    const __bf16* qrow = a.q + static_cast<int64_t>(b) * a.q_stride_b +
                         static_cast<int64_t>(g * a.group + (col < a.group ? col : a.group - 1)) * a.q_stride_h + 8 * quad;
#pragma unroll
    for (int st = 0; st < kSteps; ++st) {
      if (a.q_vectors) {
        qop[st] = __builtin_bit_cast(bf16x8, *((const global_u32x4*)(qrow + 32 * st)));
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) qop[st][i] = qrow[32 * st + i];
      }
    }
  }
  const char* kbase = reinterpret_cast<const char*>(a.k + static_cast<int64_t>(g) * a.k_stride_head + 8 * quad);
  const char* vbase = reinterpret_cast<const char*>(a.v + static_cast<int64_t>(g) * a.v_stride_head);
  const int64_t k_slot = 2 * a.k_stride_slot, v_slot = 2 * a.v_stride_slot;

  f32x4 acc[kDTiles];
#pragma unroll
  for (int t = 0; t < kDTiles; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;
  __bf16* vt = reinterpret_cast<__bf16*>(tiles[wave]);

  // the slot of this lane's key of a pass (keys past the end: the last one's)
  auto slot_at = [&](int t0) {
    const int mine = t0 + (lane & (kKeys - 1));
    return idx[mine < n ? mine : n - 1];
  };
  int32_t next = wave * kKeys < n ? slot_at(wave * kKeys) : 0;
  for (int t0 = wave * kKeys; t0 < n; t0 += kPass) {
    const int32_t slot = next;
    u32x4 k[kTiles][kSteps];
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
      const char* row = kbase + __shfl(slot, 16 * j + col) * k_slot;
#pragma unroll
      for (int st = 0; st < kSteps; ++st) k[j][st] = *((const global_u32x4*)(row + 64 * st));
    }
#pragma unroll
    for (int u = 0; u < kKeys / kRows; ++u) {
      const int r = u * kRows + lane / kChunks;
      const int c = (lane % kChunks) ^ swz<D>(r);
      const char* row = vbase + __shfl(slot, r) * v_slot;
      if (t0 + r >= n) row = reinterpret_cast<const char*>(zero_row);
      __builtin_amdgcn_global_load_lds(row + 16 * c, (lds_void*)(vt + u * kRows * D), 16, 0, 0);
    }
    // the next pass's slots come in with these rows
    if (t0 + kPass < n) next = slot_at(t0 + kPass);
    // ---- S^T = K . Q^T; lane holds S^T[keys 16 j + 4 quad + i][head col]
    f32x4 p[kTiles];
    float top = -INFINITY;
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int st = 0; st < kSteps; ++st)
        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, k[j][st]), qop[st], s, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[j][i] = t0 + 16 * j + 4 * quad + i < n ? s[i] * a.scale_log2 : -INFINITY;
        top = fmaxf(top, p[j][i]);
      }
    }
    top = fmaxf(top, __shfl_xor(top, 16));
    top = fmaxf(top, __shfl_xor(top, 32));
    const float m_new = fmaxf(m_run, top);
    const float corr = m_new == -INFINITY ? 1.f : exp2f(m_run - m_new);
    float row = 0.f;
#pragma unroll
    for (int j = 0; j < kTiles; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[j][i] = m_new == -INFINITY ? 0.f : exp2f(p[j][i] - m_new);
        row += p[j][i];
      }
    row += __shfl_xor(row, 16);
    row += __shfl_xor(row, 32);
    l_run = l_run * corr + row;
    m_run = m_new;
#pragma unroll
    for (int t = 0; t < kDTiles; ++t) acc[t] *= corr;
    // ---- O^T += V^T . P^T, once this wave's V rows have landed
    __builtin_amdgcn_s_waitcnt(0);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int jj = 0; jj < kTiles / 2; ++jj) {
      const bf16x4 p0 = __builtin_convertvector(p[2 * jj], bf16x4), p1 = __builtin_convertvector(p[2 * jj + 1], bf16x4);
      const bf16x8 pop = __builtin_shufflevector(p0, p1, 0, 1, 2, 3, 4, 5, 6, 7);
      // transposing read: lane col of group quad receives V[key][16 t + col]
      // for keys 32 jj + 4 quad + i, then 16 keys on; its source is row
      // key0 + col / 4, dims 16 t + 4 (col % 4) .. + 3
      const int r0 = 32 * jj + 4 * quad + (col >> 2), r1 = r0 + 16;
#pragma unroll
      for (int t = 0; t < kDTiles; ++t) {
        const int c = 2 * t + ((col & 3) >> 1), h = 4 * (col & 1);
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vt + r0 * D + 8 * (c ^ swz<D>(r0)) + h));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vt + r1 * D + 8 * (c ^ swz<D>(r1)) + h));
        const bf16x8 vop = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vop, pop, acc[t], 0, 0, 0);
      }
    }
    // this pass's reads are done (lgkmcnt 0) before the next pass's rows are
    // asked into their place: its slots are here already, so nothing else waits
    __builtin_amdgcn_s_waitcnt(0xc07f);
    asm volatile("" ::: "memory");
  }

  // the waves meet: O rows [head][dim] over their V tiles, m and l beside them
  // (every lane of a column carries that head's m and l)
  float* om = reinterpret_cast<float*>(tiles[wave]);
#pragma unroll
  for (int t = 0; t < kDTiles; ++t) *reinterpret_cast<f32x4*>(om + col * kOut + 16 * t + 4 * quad) = acc[t];
  if (quad == 0) {
    s_m[wave][col] = m_run;
    s_l[wave][col] = l_run;
  }
  __syncthreads();
  for (int u = threadIdx.x; u < a.group * (D / 4); u += 64 * kWaves) {
    const int hl = u / (D / 4), d = 4 * (u % (D / 4));
    float m = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) m = fmaxf(m, s_m[w][hl]);
    float l = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      // a wave without keys carries m = -inf, l = 0 and O = 0
      const float sw = s_m[w][hl] == -INFINITY ? 0.f : exp2f(s_m[w][hl] - m);
      l += s_l[w][hl] * sw;
      o += *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(tiles[w]) + hl * kOut + d) * sw;
    }
    if (a.chunks > 1) {
      // a partial row is D + 2 floats: 8-byte aligned
      float* ph = a.partial + (((static_cast<int64_t>(b) * a.kv_heads + g) * a.chunks + chunk) * 16 + hl) * (D + 2);
      *reinterpret_cast<f32x2_t*>(ph + d) = f32x2_t{o[0], o[1]};
      *reinterpret_cast<f32x2_t*>(ph + d + 2) = f32x2_t{o[2], o[3]};
      if (d == 0) *reinterpret_cast<f32x2_t*>(ph + D) = f32x2_t{m, l};
      continue;
    }
    // one chunk holds every key: normalise with the sink here (the combine's
    // arithmetic for a single partial)
    const int head = g * a.group + hl;
    const float sink = a.sinks ? a.sinks[head] * kLog2e : -INFINITY;
    const bool valid = m != -INFINITY;
    const float mt = valid ? fmaxf(sink, m) : sink;
    float lt = (a.sinks && mt != -INFINITY) ? exp2f(sink - mt) : 0.f;
    const float sw = valid ? exp2f(m - mt) : 0.f;
    lt += valid ? l * sw : 0.f;
    const int64_t at = static_cast<int64_t>(b) * a.out_stride_b + static_cast<int64_t>(head) * a.out_stride_h + d;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float r = lt > 0.f ? (valid ? o[i] * sw : 0.f) / lt : 0.f;
      if (a.out_f32)
        static_cast<float*>(a.out)[at + i] = r;
      else
        static_cast<__bf16*>(a.out)[at + i] = static_cast<__bf16>(r);
    }
  }
}

// One workgroup per (request, q head): merge chunk partials and the sink.
// kCombineThreads threads in ways of D / 4 lanes (four dims per lane: two
// 8-byte loads per chunk, as a partial row of D + 2 floats is 8-byte
// aligned); each way folds every ways-th chunk with an online
// (max, sum) merge -- the loads of one chunk do not wait on the previous
// one -- and the ways meet in LDS.
constexpr int kCombineThreads = 256;

template <int D>
__global__ void __launch_bounds__(kCombineThreads) decode_attention_combine_kernel(const AttnArgs a) {
  constexpr int kLanes = D / 4;
  constexpr int kWays = kCombineThreads / kLanes;
  __shared__ float s_m[kWays], s_l[kWays];
  __shared__ __attribute__((aligned(16))) float s_o[kWays][D];
  const int b = blockIdx.x;
  const int h = blockIdx.y;
  const int g = h / a.group;
  const int hl = h - g * a.group;
  const int dl = threadIdx.x % kLanes;
  const int way = threadIdx.x / kLanes;
  const int32_t len = max(a.kv_indptr[b + 1] - a.kv_indptr[b], 0);
  const int32_t total = a.kv_indptr[a.n_requests] - a.kv_indptr[0];
  if (gated(a.gate)) return;
  // keys past max_len (a caller error) are not read: the partials stop there
  const uint32_t chunk_keys = chunk_keys_of(a, len, total);
  const int want = (static_cast<uint32_t>(len) + chunk_keys - 1) / chunk_keys;
  const int used = want < a.chunks ? want : a.chunks;
  const float* base = a.partial + (static_cast<int64_t>(b) * a.kv_heads + g) * a.chunks * 16 * (D + 2);
  float m = -INFINITY, l = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  for (int c = way; c < used; c += kWays) {
    const float* pc = base + (c * 16 + hl) * (D + 2);
    const float mc = pc[D];
    const float lc = pc[D + 1];
    // a partial row is D + 2 floats: 8-byte aligned, so two 8-byte loads
    const f32x2_t lo = *reinterpret_cast<const f32x2_t*>(pc + 4 * dl);
    const f32x2_t hi = *reinterpret_cast<const f32x2_t*>(pc + 4 * dl + 2);
    const f32x4 oc = {lo.x, lo.y, hi.x, hi.y};
    // an empty chunk carries m = -inf and no o values
    const bool valid = mc != -INFINITY;
    const float mn = valid ? fmaxf(m, mc) : m;
    const float ws = valid ? exp2f(m - mn) : 1.f;
    const float wc = valid ? exp2f(mc - mn) : 0.f;
    l = l * ws + (valid ? lc : 0.f) * wc;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = o[i] * ws + (valid ? oc[i] : 0.f) * wc;
    m = mn;
  }
  *reinterpret_cast<f32x4*>(&s_o[way][4 * dl]) = o;
  if (dl == 0) {
    s_m[way] = m;
    s_l[way] = l;
  }
  __syncthreads();
  if (threadIdx.x >= D) return;
  const int d = threadIdx.x;
  float mt = a.sinks ? a.sinks[h] * kLog2e : -INFINITY;
#pragma unroll
  for (int w = 0; w < kWays; ++w) mt = fmaxf(mt, s_m[w]);
  float lt = (a.sinks && mt != -INFINITY) ? exp2f(a.sinks[h] * kLog2e - mt) : 0.f;
  float ot = 0.f;
#pragma unroll
  for (int w = 0; w < kWays; ++w) {
    if (s_m[w] == -INFINITY) continue;
    const float sw = exp2f(s_m[w] - mt);
    lt += s_l[w] * sw;
    ot += s_o[w][d] * sw;
  }
  const float r = lt > 0.f ? ot / lt : 0.f;
  const int64_t at = static_cast<int64_t>(b) * a.out_stride_b + static_cast<int64_t>(h) * a.out_stride_h + d;
  if (a.out_f32)
    static_cast<float*>(a.out)[at] = r;
  else
    static_cast<__bf16*>(a.out)[at] = static_cast<__bf16>(r);
}

int64_t chunks_for(int64_t max_len, int64_t keys) { return max_len <= 0 ? 1 : (max_len + keys - 1) / keys; }

// The passes that the bound allows, and two for requests of up to two passes'
// keys rather than a second launch.
int32_t max_passes_for(int64_t requests, int64_t kv_heads, int64_t max_len) {
  int32_t passes = 1;
  while (passes < kMaxPasses &&
         requests * kv_heads * chunks_for(max_len, 2 * passes * kPass) >= kEnoughGroups)
    passes *= 2;
  if (passes == 1 && max_len <= 2 * kPass) passes = 2;
  return passes;
}

constexpr int32_t kFewChunks = 8;

// Split-K scratch of akv_decode_attention_noalloc: a file-scope device array,
// one per GPU, held until the process ends.  Host code never passes the
// array's name to a kernel (on the host it is only a stand-in for the
// symbol): it uses the per-device address hipGetSymbolAddress returns.
constexpr int64_t kScratchBytes = 32ll << 20;
static __device__ __align__(256) float scratch[kScratchBytes / sizeof(float)];

constexpr int kMaxDevices = 64;
std::mutex scratch_mutex;
void* scratch_ptr[kMaxDevices] = {};

// The current device's scratch address, looked up once per device with that
// device current.
int scratch_address(void** out) {
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess)
    return fail(AKV_EHIP, "akv_decode_attention_noalloc: hipGetDevice failed: %s", hipGetErrorString(err));
  if (dev < 0 || dev >= kMaxDevices)
    return fail(AKV_EINVAL, "akv_decode_attention_noalloc: device %d beyond %d", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (!scratch_ptr[dev]) {
    void* p = nullptr;
    err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess || !p)
      return fail(AKV_EHIP, "akv_decode_attention_noalloc: hipGetSymbolAddress(scratch) failed: %s",
                  hipGetErrorString(err));
    scratch_ptr[dev] = p;
  }
  *out = scratch_ptr[dev];
  return AKV_OK;
}

}  // namespace
}  // namespace akv

extern "C" int64_t akv_decode_attention_workspace_bytes(int32_t n_requests, int32_t kv_heads,
                                                         int32_t head_dim, int64_t max_len) {
  using namespace akv;
  if (n_requests < 0 || kv_heads <= 0 || head_dim <= 0 || max_len < 0) return -1;
  return static_cast<int64_t>(n_requests) * kv_heads * chunks_for(max_len, kPass) * 16 * (head_dim + 2) * 4;
}

extern "C" int akv_decode_attention(const void* q, int64_t q_stride_b, int64_t q_stride_h, const void* k_buffer,
                                    const void* v_buffer, int64_t k_stride_slot, int64_t k_stride_head,
                                    int64_t v_stride_slot, int64_t v_stride_head, int32_t n_requests,
                                    int32_t q_heads, int32_t kv_heads, int32_t head_dim,
                                    const int32_t* kv_indptr, const int32_t* kv_indices, const float* sinks,
                                    float scale, void* out, int32_t out_dtype, int64_t out_stride_b,
                                    int64_t out_stride_h, int64_t max_len, void* workspace,
                                    int64_t workspace_bytes, const int32_t* status, void* stream) {
  using namespace akv;
  if (n_requests < 0 || max_len < 0) return fail(AKV_EINVAL, "akv_decode_attention: negative size");
  if (n_requests == 0) return AKV_OK;
  if (head_dim != 64 && head_dim != 128)
    return fail(AKV_EINVAL, "akv_decode_attention: head_dim %d (supported: 64, 128)", head_dim);
  if (kv_heads <= 0 || q_heads <= 0 || q_heads % kv_heads != 0 || q_heads / kv_heads > 16)
    return fail(AKV_EINVAL, "akv_decode_attention: %d q heads over %d KV heads (group <= 16)", q_heads,
                kv_heads);
  if (out_dtype != AKV_BF16 && out_dtype != AKV_F32)
    return fail(AKV_EINVAL, "akv_decode_attention: output must be bf16 or f32");
  if (!q || !k_buffer || !v_buffer || !kv_indptr || !kv_indices || !out || !workspace)
    return fail(AKV_EINVAL, "akv_decode_attention: null device pointer");
  if ((k_stride_slot | k_stride_head | v_stride_slot | v_stride_head) % 8 != 0 ||
      ((reinterpret_cast<uintptr_t>(k_buffer) | reinterpret_cast<uintptr_t>(v_buffer)) & 15) != 0)
    return fail(AKV_EINVAL, "akv_decode_attention: K/V rows must be 16-byte aligned");
  if (n_requests > 65535 || kv_heads > 65535)
    return fail(AKV_EINVAL, "akv_decode_attention: batch too large");
  const int64_t need = akv_decode_attention_workspace_bytes(n_requests, kv_heads, head_dim, max_len);
  if (workspace_bytes < need)
    return fail(AKV_EINVAL, "akv_decode_attention: workspace holds %lld bytes, needs %lld",
                static_cast<long long>(workspace_bytes), static_cast<long long>(need));
  AttnArgs a{};
  a.q = static_cast<const __bf16*>(q);
  a.q_stride_b = q_stride_b;
  a.q_stride_h = q_stride_h;
  a.k = static_cast<const __bf16*>(k_buffer);
  a.v = static_cast<const __bf16*>(v_buffer);
  a.k_stride_slot = k_stride_slot;
  a.k_stride_head = k_stride_head;
  a.v_stride_slot = v_stride_slot;
  a.v_stride_head = v_stride_head;
  a.kv_indptr = kv_indptr;
  a.kv_indices = kv_indices;
  a.sinks = sinks;
  a.gate = status;
  a.scale_log2 = scale * kLog2e;
  a.out = out;
  a.out_f32 = out_dtype == AKV_F32;
  a.out_stride_b = out_stride_b;
  a.out_stride_h = out_stride_h;
  a.n_requests = n_requests;
  a.q_heads = q_heads;
  a.kv_heads = kv_heads;
  a.group = q_heads / kv_heads;
  a.max_passes = max_passes_for(n_requests, kv_heads, max_len);
  a.chunks = static_cast<int32_t>(chunks_for(max_len, a.max_passes * kPass));
  a.heads_last = a.chunks < kFewChunks;
  // 2^e chunks (times an odd number) of 2^(3-e) pairs are one round of the XCDs
  a.turn_shift = 3 - std::min(3, __builtin_ctz(static_cast<uint32_t>(a.chunks)));
  a.q_vectors = ((q_stride_b | q_stride_h) % 8 == 0) && (reinterpret_cast<uintptr_t>(q) & 15) == 0;
  a.partial = static_cast<float*>(workspace);
  hipStream_t st = as_stream(stream);
  const unsigned heads = static_cast<unsigned>(kv_heads), requests = static_cast<unsigned>(n_requests);
  const dim3 grid(static_cast<unsigned>(a.chunks), a.heads_last ? requests : heads, a.heads_last ? heads : requests);
  if (head_dim == 64)
    hipLaunchKernelGGL(decode_attention_partial_kernel<64>, grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL(decode_attention_partial_kernel<128>, grid, dim3(512), 0, st, a);
  int rc = check_launch("akv_decode_attention (partial)");
  if (rc || a.chunks == 1) return rc;
  const dim3 merge(n_requests, q_heads);
  if (head_dim == 64)
    hipLaunchKernelGGL(decode_attention_combine_kernel<64>, merge, dim3(kCombineThreads), 0, st, a);
  else
    hipLaunchKernelGGL(decode_attention_combine_kernel<128>, merge, dim3(kCombineThreads), 0, st, a);
  return check_launch("akv_decode_attention (combine)");
}

extern "C" int64_t akv_decode_attention_noalloc_max_bytes(void) { return akv::kScratchBytes; }

extern "C" int akv_decode_attention_noalloc(const void* q, int64_t q_stride_b, int64_t q_stride_h,
                                            const void* k_buffer, const void* v_buffer, int64_t k_stride_slot,
                                            int64_t k_stride_head, int64_t v_stride_slot, int64_t v_stride_head,
                                            int32_t n_requests, int32_t q_heads, int32_t kv_heads,
                                            int32_t head_dim, const int32_t* kv_indptr, const int32_t* kv_indices,
                                            const float* sinks, float scale, void* out, int32_t out_dtype,
                                            int64_t out_stride_b, int64_t out_stride_h, int64_t max_len,
                                            const int32_t* status, void* stream) {
  using namespace akv;
  const int64_t need = akv_decode_attention_workspace_bytes(n_requests, kv_heads > 0 ? kv_heads : 1,
                                                            head_dim > 0 ? head_dim : 1, max_len);
  if (need > kScratchBytes)
    return fail(AKV_EINVAL,
                "akv_decode_attention_noalloc: the split-K partials need %lld bytes, the static scratch holds "
                "%lld (%d requests x %d KV heads x max_len %lld)",
                static_cast<long long>(need), static_cast<long long>(kScratchBytes), n_requests, kv_heads,
                static_cast<long long>(max_len));
  if (n_requests <= 0) return akv_decode_attention(q, q_stride_b, q_stride_h, k_buffer, v_buffer, k_stride_slot,
                                                   k_stride_head, v_stride_slot, v_stride_head, n_requests,
                                                   q_heads, kv_heads, head_dim, kv_indptr, kv_indices, sinks,
                                                   scale, out, out_dtype, out_stride_b, out_stride_h, max_len,
                                                   nullptr, 0, status, stream);
  void* ws = nullptr;
  const int rc = scratch_address(&ws);
  if (rc) return rc;
  return akv_decode_attention(q, q_stride_b, q_stride_h, k_buffer, v_buffer, k_stride_slot, k_stride_head,
                              v_stride_slot, v_stride_head, n_requests, q_heads, kv_heads, head_dim, kv_indptr,
                              kv_indices, sinks, scale, out, out_dtype, out_stride_b, out_stride_h, max_len, ws,
                              kScratchBytes, status, stream);
}
