// Prefill context attention over occurrence metadata (gfx950, MFMA).
//
// The extend attention the context system launches once per layer
// (akv/system/sglang/srt/layers/attention/context_backend.py:180-251 and the
// position-aware SWA mask of akv/system/sglang.patch:106-237).  For segment s
// the queries are q[qo_indptr[s] .. qo_indptr[s+1]) and the keys are
//   prefix: pool rows kv_indices[kv_indptr[s] .. kv_indptr[s+1]), all visible;
//   extend: the segment's own K/V rows (k_ext/v_ext aligned with q), causal
//           by index (key j visible to query i when j <= i);
// and, with a sliding window W >= 0, a key at position p_k is visible to a
// query at position p_q only when p_q <= p_k + W.  Positions come from
// q_positions (aligned with q) and kv_positions (aligned with kv_indices);
// without them a query's position is prefix_length + i and a prefix key's
// is its index (the native contiguous case).  Sinks add e^{sink} to the
// softmax denominator.  Within a segment positions ascend (the keys of a
// context window are ordered), which lets a workgroup start the prefix and
// extend loops at the first key inside the window.
//
// Workgroup = (block of R / G query tokens, KV head g, segment), KV head
// fastest in the grid (workgroup id mod 8 picks the XCD: with 8 KV heads each
// XCD's L2 serves one head's K/V), with the
// G q heads of the group packed as rows: row r = token * G + head; R = 512
// rows at head_dim 64 (8 waves x 64 rows, 16 for narrow windows; a wave's reads of a K/V tile
// from LDS feed 64 rows), 256 at head_dim 128 (8 waves x 32 rows); one
// workgroup per CU, two waves per SIMD, so every K/V tile a CU stages from
// L2 feeds all of its rows.  Per
// tile of 128 keys (full layers at head_dim 64) or 64 (K and V key-major in
// LDS with XOR-swizzled 16 B chunks, double buffered; the next tile's rows
// stream straight from HBM into LDS with global_load_lds_dwordx4 -- no
// staging registers -- and the slots of the tile after it are fetched, all
// during this tile's math), in 32-key quarters, for a wave's W rows:
//   S^T[32 keys x W rows] = K . Q^T           v_mfma_f32_16x16x32_bf16
//   P^T = 2^(scale log2(e) S^T - m) in bf16   (one fp32 fma per score: Q
//     stays exact -- folding the scale into a bf16 Q costs several times
//     the tolerance once the scores spread over ~40 in the log2 domain)
//   l[rows] += 1^T . P^T                      (row sums of the same bf16 P)
//   O^T[D x W rows] += V^T . P^T              v_mfma_f32_16x16x32_bf16
// Online softmax without per-tile maxima: a row's running maximum m comes
// from exact row maxima (moving only when a quarter exceeds it by 2^8)
// while some row of the wave has seen no key, then stays put.  After each
// tile the weight sums are checked: one past 2^32 is renormalised by a power
// of two; one past 2^64 (a score ~58 above m, or inf) may have overflowed O,
// and the workgroup restarts its keys with exact maxima on every tile.
// P^T leaves the first MFMA in the B-operand layout of the second (any
// consistent split of the 32-long k axis over lanes gives the same product:
// lane l uses keys 4(l/16)+i of two 16-key subtiles); V^T comes from the
// key-major tile through ds_read_b64_tr_b16.  Tiles wholly inside every
// row's causal and window range skip the mask.
//
// Batches whose plain grid leaves CUs idle take the split launch: one
// workgroup per CU with an equal stretch of all key tiles (context_plan.h), and
// a second launch that merges the blocks a stretch boundary cut.
//
// Two instances of each shape: the plain one (head_dim 64 or 128, the group
// a power of two, no logit cap) and the general one, which pads a token's
// rows to a power-of-two group (padding rows keep Q = 0 and store nothing),
// runs heads narrower than the tile with the unloaded dims zero in LDS, and
// caps scaled scores at cap tanh(s / cap) before the mask.
//
// Lane layouts (verified on gfx950): v_mfma_f32_16x16x32_bf16 -- lane l
// supplies A[l%16][k(l,i)], B[k(l,i)][l%16] for i < 8 and holds
// D[4(l/16)+i][l%16]; ds_read_b64_tr_b16 -- within each 16-lane group, lane
// j receives element j%4 of the 8-byte rows read by lanes j/4 + 4i, i < 4.
#include <algorithm>
#include <cmath>

#include "common.h"
#include "context_plan.h"
#include "tile_loop.h"

namespace akv {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) u32x4 global_u32x4;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// 16-row subtiles per wave: 4 at head_dim 64 (each wave's K/V tile reads
// from LDS feed 64 rows), 2 at head_dim 128 (register budget)
constexpr int sub_tiles(int d) { return d == 64 ? 4 : 2; }
// 8 waves: the register budget allows two waves per SIMD, so a workgroup of
// 8 fills the CU alone and its K/V tiles feed twice the rows of two 4-wave
// workgroups (half the tile loads per flop, and twice the math per tile to
// hide each tile's load behind)
constexpr int kWaves = 8;
// (token, head) rows of a block with `sub` row subtiles per wave
constexpr int block_rows(int sub) { return kWaves * 16 * sub; }
constexpr int rows_per_block(int d) { return block_rows(sub_tiles(d)); }
// Blocks of a narrow window (up to kNarrowWindow, 64-dim tiles) may have
// kNarrowSub subtiles per wave (narrow_blocks).
constexpr int kNarrowWindow = 512;
constexpr int kNarrowSub = 1;
constexpr int kThreads = 64 * kWaves;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLazy = 8.f;  // log2-domain slack before an exact maximum moves
constexpr float kBig = 4294967296.f;  // 2^32: a weight sum above it is renormalised
constexpr float kHuge = 18446744073709551616.f;  // 2^64: above it the product may have overflowed

struct CtxArgs {
  const __bf16* q;
  const __bf16* k_ext;
  const __bf16* v_ext;
  const __bf16* k_pool;
  const __bf16* v_pool;
  const void* qo_indptr;
  const void* kv_indptr;
  const void* kv_indices;
  const void* q_pos;
  const void* kv_pos;
  const float* sinks;
  void* out;
  // element strides (checked to fit 32 bits on the host)
  int32_t q_st, q_sh, ke_st, ke_sh, ve_st, ve_sh, kp_ss, kp_sh, vp_ss, vp_sh, o_st, o_sh;
  int32_t indptr_i64;
  int32_t window;
  float scale_log2;
  int32_t out_f32;
  int32_t group, group_shift, tokens_per_block, kv_heads;
  int32_t head_dim;   // head dims in use (<= the kernel's D; the rest are zero)
  float cap, cap_log2;  // logit cap (scores -> cap tanh(score / cap)), cap log2(e)
  // split launch only
  int32_t n_segments;
  int32_t max_shift;    // log2 of the workgroups (what the workspace holds)
  float* partial;       // kPartialFloats per part, two parts per workgroup
};

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

// Maximum over the four lanes col, col+16, col+32, col+48 of each 16-lane
// column group, on the VALU: v_permlane16_swap / v_permlane32_swap exchange
// rows of 16 (32) lanes, so max(swapped pair) = max(own, partner).
// v_max3_f32 / v_max_f32 without the canonicalising moves the compiler adds
// around fmaxf of matrix-core results.  Only the softmax's range uses these
// maxima: a NaN score still reaches the output through exp2 and the MFMAs.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

__device__ __forceinline__ float max2(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

__device__ __forceinline__ float row_max(float x) {
  const uint32_t b = __builtin_bit_cast(uint32_t, x);
  const auto r16 = __builtin_amdgcn_permlane16_swap(b, b, false, false);
  // copy the pair out before the bit casts: a bit cast of a vector element
  // reference reads element 0
  const uint32_t a0 = r16[0], a1 = r16[1];
  x = max2(__builtin_bit_cast(float, a0), __builtin_bit_cast(float, a1));
  const uint32_t c = __builtin_bit_cast(uint32_t, x);
  const auto r32 = __builtin_amdgcn_permlane32_swap(c, c, false, false);
  const uint32_t c0 = r32[0], c1 = r32[1];
  return max2(__builtin_bit_cast(float, c0), __builtin_bit_cast(float, c1));
}

__device__ __forceinline__ u32x4 load16(const __bf16* p) {
  return *((const global_u32x4*)p);
}

// One of the two LDS tile buffers.  They are separate objects, named
// statically in each half of the unrolled tile loop, so the compiler sees
// that this tile's LDS reads never touch the other buffer that the next
// tile's direct loads are filling (no wait on those loads mid-tile in the
// 64-key instances; the rolled quarter loop of the 128-key ones still gets
// a wait before its transposing reads, which measured free).
template <int D, int KEYS>
struct TileLds {
  __bf16 k[KEYS][D];   // key-major K tile, 16 B chunks swizzled per row (swz_k)
  __bf16 v[KEYS][D];   // key-major V tile, read transposed (ds_read_b64_tr_b16), swizzled (swz_v)
  int32_t pos[KEYS];   // key positions relative to the block's first query
};

// Chunk swizzles: logical 16 B chunk c of row r lives at chunk c ^ swz(r).
// K (16 B operand reads, 16 rows per lane group): distinct banks for the 16
// rows of a read.  V (8 B transposed reads, 4 rows x 32 B per 16 lanes, 8
// rows per 32 lanes): bit 0 clear so a row's chunk pair stays adjacent, and
// distinct bank groups for 8 consecutive rows.  At head_dim 64 a row is half
// the 64 banks (rows of opposite parity use opposite halves).
template <int D>
__device__ __forceinline__ int swz_k(int r) { return D == 64 ? (r >> 1) & 7 : r & 15; }
template <int D>
__device__ __forceinline__ int swz_v(int r) { return D == 64 ? r & 6 : (r & 7) << 1; }

typedef __attribute__((address_space(3))) void lds_void;

constexpr int32_t kFar = 1 << 30;  // relative positions are clamped to [-kFar, kFar]

__device__ __forceinline__ int32_t rel_pos(int64_t p, int64_t base) {
  const int64_t r = p - base;
  return static_cast<int32_t>(r < -kFar ? -kFar : (r > kFar ? kFar : r));
}

// Most workgroups of a split launch: one per CU (a power of two).
constexpr int kSplitShift = 8;
constexpr int kSplitGroups = 1 << kSplitShift;
// The split launch keeps a batch's segments one to a lane.
constexpr int kMaxSplitSegments = 64;

// One wave's copy of the batch: lane s holds segment s.
struct BatchPlan {
  int64_t q0, k0;  // this lane's segment: first query, first prefix index
  int32_t q, p;    // queries and prefix keys
  int64_t before;  // cost of the segments before it
  int64_t total;   // one head's cost
  uint64_t live;   // segments with queries
};

template <int D, int KEYS>
__device__ __forceinline__ SplitShape split_shape(const CtxArgs& a) {
  return SplitShape{__builtin_ctz(rows_per_block(D)) - a.group_shift, __builtin_ctz(KEYS)};
}

__device__ __forceinline__ int64_t read_lane(int64_t v, int lane) {
  const uint32_t lo = __builtin_amdgcn_readlane(static_cast<int32_t>(v), lane);
  const uint32_t hi = __builtin_amdgcn_readlane(static_cast<int32_t>(v >> 32), lane);
  return static_cast<int64_t>(static_cast<uint64_t>(hi) << 32 | lo);
}

__device__ __forceinline__ BatchPlan plan_batch(const CtxArgs& a, const SplitShape& sh, int lane) {
  BatchPlan b;
  const bool in = lane < a.n_segments;
  const int s = in ? lane : 0;
  const int64_t q0 = load_index(a.qo_indptr, a.indptr_i64, s), q1 = load_index(a.qo_indptr, a.indptr_i64, s + 1);
  const int64_t k0 = load_index(a.kv_indptr, a.indptr_i64, s), k1 = load_index(a.kv_indptr, a.indptr_i64, s + 1);
  b.q0 = q0;
  b.k0 = k0;
  b.q = in ? static_cast<int32_t>(q1 - q0) : 0;
  b.p = in && a.kv_indices ? static_cast<int32_t>(k1 - k0) : 0;
  const int64_t cost = segment_cost(sh, b.q, b.p);
  int64_t sum = cost;
#pragma nounroll
  for (int off = 1; off < a.n_segments; off <<= 1) {
    const int64_t up = __shfl_up(sum, off);
    if (lane >= off) sum += up;
  }
  b.before = sum - cost;
  b.total = read_lane(sum, a.n_segments - 1);
  b.live = __builtin_amdgcn_ballot_w64(cost > 0);
  return b;
}

// Boundary r of this lane (the lanes' searches run side by side).
__device__ __forceinline__ Place lane_place(const BatchPlan& b, const SplitShape& sh, int32_t heads, int k, int r) {
  auto get = [&](int i, int32_t* q, int32_t* p, int64_t* before) {
    *q = __builtin_amdgcn_readlane(b.q, i);
    *p = __builtin_amdgcn_readlane(b.p, i);
    *before = read_lane(b.before, i);
  };
  return place_of(sh, get, b.live, b.total, heads, k, r);
}

__device__ __forceinline__ int32_t uniform(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ int64_t uniform(int64_t v) {
  const uint32_t lo = uniform(static_cast<int32_t>(v)), hi = uniform(static_cast<int32_t>(v >> 32));
  return static_cast<int64_t>(static_cast<uint64_t>(hi) << 32 | lo);
}

__device__ __forceinline__ Place uniform(const Place& p) {
  return Place{uniform(p.head), uniform(p.seg), uniform(p.block), uniform(p.tile)};
}

__device__ __forceinline__ Place from_lane(const Place& p, int lane) {
  return Place{__builtin_amdgcn_readlane(p.head, lane), __builtin_amdgcn_readlane(p.seg, lane),
               __builtin_amdgcn_readlane(p.block, lane), __builtin_amdgcn_readlane(p.tile, lane)};
}

// Stores a row's normalised output, from its O (4 dims of each of TILES 16-dim
// tiles from dt0 on), weight sum l and maximum m (-inf: the row has seen no
// key), with the sink.
template <int D, bool GEN, int TILES>
__device__ __forceinline__ void store_row(const CtxArgs& a, int g, int r, int32_t t0, int32_t qlen, int64_t qo0,
                                          int quad, int dt0, const f32x4 (&o)[TILES], float l, float m_run) {
  const int G = a.group;
  const int hl = r & ((1 << a.group_shift) - 1);
  float scale = 1.f;
  if (a.sinks) {
    const float sink = a.sinks[g * G + (GEN && hl >= G ? G - 1 : hl)] * kLog2e;
    const float m_f = fmaxf(m_run, sink);
    scale = m_run == -INFINITY ? 0.f : exp2f(m_run - m_f);
    l = l * scale + exp2f(sink - m_f);
  }
  const float inv = l > 0.f ? scale / l : 0.f;
  const int32_t row_token = r >> a.group_shift, row_head = g * G + hl;
  if (t0 + row_token >= qlen || (GEN && hl >= G)) return;
  const int64_t at = (qo0 + t0 + row_token) * a.o_st + static_cast<int64_t>(row_head) * a.o_sh + 16 * dt0 + 4 * quad;
#pragma unroll
  for (int dt = 0; dt < TILES; ++dt) {
    if (GEN && 16 * (dt0 + dt) + 4 * quad >= a.head_dim) continue;
    const f32x4 v = o[dt] * inv;
    if (a.out_f32) {
      *reinterpret_cast<f32x4*>(static_cast<float*>(a.out) + at + 16 * dt) = v;
    } else {
      bf16x4 ob;
#pragma unroll
      for (int i = 0; i < 4; ++i) ob[i] = static_cast<__bf16>(v[i]);
      *reinterpret_cast<bf16x4*>(static_cast<__bf16*>(a.out) + at + 16 * dt) = ob;
    }
  }
}

// A partial result: O of every (16-dim tile, row subtile) as the lanes hold it
// (whole 1 KiB stores), then each row's maximum and weight sum.
constexpr int kPartialO = 32768;  // rows_per_block(D) * D floats, either head_dim
template <int D>
constexpr int64_t partial_floats() { return kPartialO + 2 * rows_per_block(D); }

// Where a stretch starts (tile -1: no such stretch), with its segment's first
// query and query count.  The workspace ends with one for every workgroup.
struct __attribute__((aligned(16))) Cut {
  Place at;
  int64_t q0;
  int32_t q, pad;
};

template <int D>
__device__ __forceinline__ Cut* split_cuts(const CtxArgs& a) {
  return reinterpret_cast<Cut*>(a.partial + (partial_floats<D>() << (a.max_shift + 1)));
}

// A segment's first query and prefix index, its queries and prefix keys.
struct Segment {
  int64_t q0, k0;
  int32_t q, p;
};

template <int D, int KEYS, int SUB>
struct Lds {
  TileLds<D, KEYS>& tile0;
  TileLds<D, KEYS>& tile1;
  int32_t (&rel_rows)[block_rows(SUB)];
  int32_t (&restart)[kRestartWords];  // tile_loop.h
  float2* merge;  // 4 x 16 SUB, split launch only
};

// KEYS keys per tile: 128 for full layers at head_dim 64 (half the tile
// barriers, staging and commits per key), 64 for windowed layers (less of a
// tile outside the window) and at head_dim 128 (measured faster than 128 there)
// GEN: the general instance -- logit caps, heads narrower than D (the dims
// past head_dim zero in the tiles), groups padded to a power of two; the
// plain instance takes none of these checks.
//
// One block of queries of a segment for KV head `g`, over its key tiles
// [it_first, it_stop) (it_stop < 0: to the end; a plain launch's are all of
// them).  All the workgroup's threads call it.  `part`: where a split launch
// keeps a part of a block's result.
template <int D, int KEYS, int SUB, typename IdxT, typename PosT, bool POS, bool GEN, bool SPLIT>
__device__ __forceinline__ void attend(const CtxArgs& a, const Lds<D, KEYS, SUB>& lds, const Segment& sg, int g,
                                       int32_t block, int it_first, int it_stop, float* part) {
  const int it_begin = SPLIT ? it_first : 0;
  constexpr int kSub = SUB;
  constexpr int kKeys = KEYS;
  constexpr int kChunks = D / 8;               // 16 B chunks per key row
  constexpr int kKSteps = D / 32;              // MFMA k-steps over head dims
  constexpr int kDTiles = D / 16;              // O^T row tiles
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: LDS block bases in SGPRs
  const int col = lane & 15;
  const int quad = lane >> 4;
  const int64_t qo0 = sg.q0;
  const int32_t qlen = sg.q;
  const int G = a.group;                         // q heads per KV head
  const int gmask = (1 << a.group_shift) - 1;    // rows per token: G padded to a power of two
  const int T = a.tokens_per_block;
  const int hd = GEN ? a.head_dim : D;
  const bool cap = GEN && a.cap > 0.f;
  // the score's log2-domain multiplier: with a cap the scores are capped
  // (and scaled) before the softmax, which then takes them as they are
  const float mult = cap ? 1.f : a.scale_log2;
  const int32_t t0 = block * T;
  const int64_t kv0 = sg.k0;
  const int32_t plen = sg.p;
  // segment-local views
  const PosT* qpos = static_cast<const PosT*>(a.q_pos) + qo0;
  const PosT* kpos = static_cast<const PosT*>(a.kv_pos) + kv0;
  const IdxT* slots = static_cast<const IdxT*>(a.kv_indices) + kv0;
  const __bf16* kext = a.k_ext + qo0 * a.ke_st + g * a.ke_sh;
  const __bf16* vext = a.v_ext + qo0 * a.ve_st + g * a.ve_sh;
  const __bf16* kpool = a.k_pool + g * a.kp_sh;
  const __bf16* vpool = a.v_pool + g * a.vp_sh;
  const char* kext_b = reinterpret_cast<const char*>(kext);
  const char* vext_b = reinterpret_cast<const char*>(vext);
  const char* kpool_b = reinterpret_cast<const char*>(kpool);
  const char* vpool_b = reinterpret_cast<const char*>(vpool);
  const uint64_t ke_sb = 2u * static_cast<uint32_t>(a.ke_st), ve_sb = 2u * static_cast<uint32_t>(a.ve_st);
  const uint64_t kp_sb = 2u * static_cast<uint32_t>(a.kp_ss), vp_sb = 2u * static_cast<uint32_t>(a.vp_ss);
  auto qpos_of = [&](int32_t i) -> int64_t {  // position of query i of the segment
    if constexpr (POS) return static_cast<int64_t>(qpos[i]);
    return static_cast<int64_t>(plen) + i;
  };
  auto kpos_of = [&](int32_t j) -> int64_t {  // position of prefix key j
    if constexpr (POS) return static_cast<int64_t>(kpos[j]);
    return static_cast<int64_t>(j);
  };
  const int window = SPLIT ? -1 : a.window;  // a split launch has none
  const int64_t qbase = qpos_of(t0);
  const int32_t e_hi = qlen < t0 + T ? qlen : t0 + T;  // extend keys [e_lo, e_hi)
  const int32_t last_rel = rel_pos(qpos_of(e_hi - 1), qbase);

  // keys below qbase - window are outside every row's window
  int32_t p_lo = 0, e_lo = 0;
  if (window >= 0) {
    const int64_t first = qbase - window;
    p_lo = first_at_least(kpos_of, plen, first, lane);
    e_lo = first_at_least(qpos_of, t0, first, lane);
  }
  const int n_pref = (plen - p_lo + kKeys - 1) / kKeys;
  const int n_tiles = n_pref + (e_hi - e_lo + kKeys - 1) / kKeys;
  const int it_end = !SPLIT || it_stop < 0 ? n_tiles : it_stop;
  auto tile_base = [&](int it) -> int32_t {
    return it < n_pref ? p_lo + it * kKeys : e_lo + (it - n_pref) * kKeys;
  };

  // tile staging straight into LDS (global_load_lds_dwordx4: lane l of a
  // wave instruction fills bytes 16 l of a 1 KiB block).  Block b of a tile
  // holds rows kRowsPerBlock b ..; lane l writes row kRowsPerBlock b + l /
  // kChunks at chunk position l % kChunks, i.e. logical chunk (l % kChunks)
  // ^ swz(row) of that key, which it loads.  Each wave fills kBlocksPerWave
  // blocks of K and of V.  Prefix slots are fetched one tile ahead.
  constexpr int kRowsPerBlock = 1024 / (2 * D);
  constexpr int kBlocksPerWave = kKeys / kRowsPerBlock / kWaves;
  static_assert(kBlocksPerWave >= 1 && kBlocksPerWave * kRowsPerBlock * kWaves == kKeys, "tile split over waves");
  static_assert(kThreads >= kKeys, "one thread per key position");
  // slot indices are below 2^32 (a pool of 2^32 slots of one 64-wide bf16
  // head is 512 GiB): int64 indices address rows through their low 32 bits
  uint32_t slot[kBlocksPerWave];
  int64_t preg = 0;  // raw position of key tid of the staged tile
  bool pvalid = false;
  const int my_row = lane / kChunks;   // row within a block
  const int my_pos = lane % kChunks;   // chunk position within the row
  auto fetch_slots = [&](int it) {
    // keys past the prefix read the last prefix row (finite data, masked out)
    const int32_t base = tile_base(it);
#pragma unroll
    for (int u = 0; u < kBlocksPerWave; ++u) {
      const int32_t j = base + (kBlocksPerWave * wave + u) * kRowsPerBlock + my_row;
      slot[u] = static_cast<uint32_t>(slots[j < plen ? j : plen - 1]);
    }
  };
  auto stage = [&](int it, TileLds<D, KEYS>& t) {
    // branch-free: keys past the end read the last valid row (masked out later)
    const bool ext = it >= n_pref;
    const int32_t base = tile_base(it);
#pragma unroll
    for (int u = 0; u < kBlocksPerWave; ++u) {
      const int blk = kBlocksPerWave * wave + u;
      const int r = blk * kRowsPerBlock + my_row;
      const int ck = my_pos ^ swz_k<D>(r), cv = my_pos ^ swz_v<D>(r);
      const char *krow, *vrow;
      if (ext) {
        const int32_t j = base + r;
        const uint64_t off = static_cast<uint32_t>(j < e_hi ? j : e_hi - 1);
        krow = kext_b + off * ke_sb;
        vrow = vext_b + off * ve_sb;
      } else {
        const uint64_t so = slot[u];
        krow = kpool_b + so * kp_sb;
        vrow = vpool_b + so * vp_sb;
      }
      if (!GEN || hd == D) {
        __builtin_amdgcn_global_load_lds(krow + 16 * ck, (lds_void*)(&t.k[blk * kRowsPerBlock][0]), 16, 0, 0);
        __builtin_amdgcn_global_load_lds(vrow + 16 * cv, (lds_void*)(&t.v[blk * kRowsPerBlock][0]), 16, 0, 0);
      } else {
        // narrower heads: chunks past hd are not loaded (they stay zero)
        if (8 * ck < hd)
          __builtin_amdgcn_global_load_lds(krow + 16 * ck, (lds_void*)(&t.k[blk * kRowsPerBlock][0]), 16, 0, 0);
        if (8 * cv < hd)
          __builtin_amdgcn_global_load_lds(vrow + 16 * cv, (lds_void*)(&t.v[blk * kRowsPerBlock][0]), 16, 0, 0);
      }
    }
    // key positions matter only to a window (causal masking is by index)
    if (window >= 0 && tid < kKeys) {
      // loaded now, converted at commit: no wait on the tile's row loads here
      const int32_t j = base + tid;
      const int32_t end = ext ? e_hi : plen;
      pvalid = j < end;
      const int32_t jc = pvalid ? j : end - 1;
      preg = ext ? qpos_of(jc) : kpos_of(jc);
    }
  };
  // positions of the staged tile, then wait for its direct loads (vmcnt) so
  // the barrier that follows publishes the whole tile
  auto commit = [&](TileLds<D, KEYS>& t) {
    // (without a window every key's position reads 0, which the mask admits)
    if (tid < kKeys) t.pos[tid] = window < 0 ? 0 : (pvalid ? rel_pos(preg, qbase) : kFar);
    __builtin_amdgcn_s_waitcnt(0);
  };

  // the first tile's slots are on their way while Q loads
  if (it_begin < n_pref) fetch_slots(it_begin);

  // this lane's rows: row subtile s covers rows group * 16 kSub + 16s + col,
  // row r = (token r >> group_shift, q head g G + r % G); the rows'
  // positions relative to qbase wait in LDS for the masked tiles.  A split
  // launch's short block has 1, 2 or 4 groups of rows; its waves then share
  // the 32-key quarters of each tile (wave w takes row group w % groups and
  // quarters w / groups, w / groups + sharers, ...) and merge at the end.
  int groups = kWaves, sharers = 1;
  if constexpr (SPLIT) {
    const int32_t rows = (qlen - t0 < T ? qlen - t0 : T) << a.group_shift;
    while (groups > 1 && rows <= (groups >> 1) * (16 * kSub)) {
      groups >>= 1;
      sharers <<= 1;
    }
  }
  const int row_group = SPLIT ? wave & (groups - 1) : wave;
  const int share = SPLIT ? wave / groups : 0;
  auto row_of = [&](int s) { return row_group * (16 * kSub) + 16 * s + col; };
  bf16x8 qop[kSub][kKSteps];
#pragma unroll
  for (int s = 0; s < kSub; ++s) {
    const int r = row_of(s);
    const int tl = r >> a.group_shift;
    const int hl = r & gmask;
    const int head = g * G + hl;
    const bool tok = t0 + tl < qlen;
    // rows past the segment are never stored: a split launch, whose pieces are
    // short, repeats its last query there (no branch around the loads), the
    // plain one keeps Q = 0; a padding row (hl >= G) keeps Q = 0
    const int32_t tr = SPLIT && !tok ? qlen - 1 : t0 + tl;
    const bool ok = (SPLIT || tok) && (!GEN || hl < G);
    if (quad == 0) lds.rel_rows[r] = tok ? rel_pos(qpos_of(t0 + tl), qbase) : last_rel;
#pragma unroll
    for (int ks = 0; ks < kKSteps; ++ks) {
      u32x4 w = {0u, 0u, 0u, 0u};
      // head dims past hd are zero
      if (ok && (!GEN || 8 * (4 * ks + quad) < hd))
        w = load16(a.q + (qo0 + tr) * a.q_st + static_cast<int64_t>(head) * a.q_sh + 32 * ks + 8 * quad);
      qop[s][ks] = __builtin_bit_cast(bf16x8, w);
    }
  }

  f32x4 oacc[kDTiles][kSub];
  // per row: the negated running maximum -m (log2 domain; 0 while the row
  // has seen no key) and the running sum of the bf16 weights (4 equal
  // copies); a row with a zero sum has seen no key
  float neg_m[kSub];
  f32x4 lacc[kSub];
  auto clear_rows = [&]() {
#pragma unroll
    for (int s = 0; s < kSub; ++s) {
      neg_m[s] = 0.f;
      lacc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int dt = 0; dt < kDTiles; ++dt) oacc[dt][s] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  clear_rows();
  // some row of this wave has seen no key yet (uniform): tiles take the
  // exact row maxima until every row has a maximum
  bool unset = true;
  // after a restart every tile takes the exact maxima (uniform)
  bool exact_all = false;
  if (tid < kRestartWords) lds.restart[tid] = 0;
  const bf16x8 kOnes = {__bf16(1.f), __bf16(1.f), __bf16(1.f), __bf16(1.f),
                        __bf16(1.f), __bf16(1.f), __bf16(1.f), __bf16(1.f)};

  if (GEN && hd < D) {
    // narrower heads: the tiles' chunks past hd are never loaded; zero them
    // once.  The stores cover every chunk, loaded ones too, so they must
    // land before any wave's direct loads into tile 0: barrier first.
    constexpr int kWords = KEYS * D / 8;  // 16 B chunks per array
    for (int i = tid; i < 4 * kWords; i += kThreads) {
      __bf16* arr = i < kWords ? &lds.tile0.k[0][0] : i < 2 * kWords ? &lds.tile0.v[0][0]
                  : i < 3 * kWords ? &lds.tile1.k[0][0] : &lds.tile1.v[0][0];
      reinterpret_cast<u32x4*>(arr)[i % kWords] = u32x4{0u, 0u, 0u, 0u};
    }
    __syncthreads();
  }
  auto open = [&]() {
    stage(it_begin, lds.tile0);
    if (it_begin + 1 < n_pref) fetch_slots(it_begin + 1);
    commit(lds.tile0);
    __syncthreads();
  };
  open();
  // tile it from cur while tile it + 1 streams into nxt
  auto step = [&](int it, TileLds<D, KEYS>& cur, TileLds<D, KEYS>& nxt) {
    if (it + 1 < it_end) {
      stage(it + 1, nxt);
      if (it + 2 < n_pref) fetch_slots(it + 2);
    }
    const bool ext = it >= n_pref;
    const int32_t base = tile_base(it);
    const int32_t left = (ext ? e_hi : plen) - base;
    const int count = left < kKeys ? left : kKeys;
    // masking is needed for a partial tile, keys past the block's first
    // query (causal), or keys older than the last query's window
    const bool masked = count < kKeys || (ext && base + kKeys - 1 > t0) ||
                        (window >= 0 && __builtin_amdgcn_readfirstlane(cur.pos[0]) < last_rel - window);
    const bool exact = unset || exact_all;

    // The tile in quarters of 32 keys (kk), each complete before the next:
    //   S^T = K . Q^T
    //   P^T = 2^(scale log2(e) S^T - m) in bf16  (the B operand of both products)
    //   l += 1^T . P^T         (row sums of the same bf16 weights on the
    //                           matrix cores: O stays a convex combination)
    //   O^T += V^T . P^T
    // Masked tiles add the mask (masked scores become -inf in place: exp2 ->
    // 0); exact tiles the row maxima (column of S^T: lanes col, col+16,
    // col+32, col+48): a row's maximum moves when the half exceeds it by more
    // than kLazy (a row that has seen no key: on any visible key), scaling O
    // and l by 2^-move.  Both stay runtime branches: a branch-free fast tile
    // lets the scheduler hoist the second half's reads and products into
    // the first half and spill.
    auto half = [&](int kk) {
      f32x4 sh[2][kSub];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int kt = 2 * kk + j;
        const int krow = 16 * kt + col;
#pragma unroll
        for (int ks = 0; ks < kKSteps; ++ks) {
          const bf16x8 kop = __builtin_bit_cast(
              bf16x8, *reinterpret_cast<const u32x4*>(&cur.k[krow][8 * ((4 * ks + quad) ^ swz_k<D>(krow))]));
#pragma unroll
          for (int s = 0; s < kSub; ++s)
            sh[j][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop, qop[s][ks],
                                                               ks == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : sh[j][s], 0, 0, 0);
        }
      }
      if (cap) {
        // capped logits: cap tanh(scale s / cap), in the log2 domain, before
        // the mask (a masked score stays -inf); tanh(x) = 1 - 2 / (1 + e^2x).
        // The cap of SGLang's extend kernel, which the reference hands the
        // layer's cap (akv/system/sglang.patch:2437,2459): scale, then cap.
        // Sinks are not capped.
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int s = 0; s < kSub; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float e2x = __builtin_amdgcn_exp2f(sh[j][s][i] * a.scale_log2 * (2.f / a.cap));
              sh[j][s][i] = a.cap_log2 * (1.f - 2.f * __builtin_amdgcn_rcpf(1.f + e2x));
            }
      }
      if (masked) {
#pragma unroll
        for (int s = 0; s < kSub; ++s) {
          // causal: key index <= the row's token; window: key pos >= row pos - W
          const int r = row_of(s);
          const int32_t climit = ext ? t0 + (r >> a.group_shift) - base : kKeys;
          const int32_t last = climit < count - 1 ? climit : count - 1;
          const int32_t thr = window >= 0 ? lds.rel_rows[r] - window : -kFar - 1;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int k0 = 16 * (2 * kk + j) + 4 * quad;
            const i32x4 kp = *reinterpret_cast<const i32x4*>(&cur.pos[k0]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const bool vis = (k0 + i <= last) & (kp[i] >= thr);
              sh[j][s][i] = vis ? sh[j][s][i] : -INFINITY;
            }
          }
        }
      }
      if (exact) {
#pragma unroll
        for (int s = 0; s < kSub; ++s) {
          // 8 values in 4 three-input maxima, then across the lane groups
          const float m0 = max3(sh[0][s][0], sh[0][s][1], sh[0][s][2]);
          const float m1 = max3(sh[0][s][3], sh[1][s][0], sh[1][s][1]);
          float mx = max3(m0, m1, max3(sh[1][s][2], sh[1][s][3], -INFINITY));
          mx = row_max(mx);  // -inf when the row sees nothing here
          // the half's largest exponent, t - m in the log2 domain
          const float top = fmaf(mx, mult, neg_m[s]);
          const bool seen = lacc[s][0] != 0.f;
          const bool bump = seen ? top > kLazy : mx > -INFINITY;
          if (__builtin_amdgcn_ballot_w64(bump)) {
            const float alpha = bump && seen ? __builtin_amdgcn_exp2f(-top) : 1.f;
            lacc[s] *= alpha;
#pragma unroll
            for (int dt = 0; dt < kDTiles; ++dt) oacc[dt][s] *= alpha;
            neg_m[s] = bump ? -(mx * mult) : neg_m[s];
          }
        }
      }
      bf16x8 pop[kSub];
#pragma unroll
      for (int s = 0; s < kSub; ++s) {
        f32x4 e0, e1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          e0[i] = __builtin_amdgcn_exp2f(fmaf(sh[0][s][i], mult, neg_m[s]));
          e1[i] = __builtin_amdgcn_exp2f(fmaf(sh[1][s][i], mult, neg_m[s]));
        }
        const bf16x4 b0 = __builtin_convertvector(e0, bf16x4);
        const bf16x4 b1 = __builtin_convertvector(e1, bf16x4);
        pop[s] = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
      }
#pragma unroll
      for (int s = 0; s < kSub; ++s) lacc[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kOnes, pop[s], lacc[s], 0, 0, 0);
#pragma unroll
      for (int dt = 0; dt < kDTiles; ++dt) {
        // transposing read: lane col of group quad receives V[key][16dt + col]
        // for keys 32kk + 4 quad + i (i < 4), then 32kk + 16 + 4 quad + i;
        // source lane col supplies row key0 + col / 4, dims 16dt + 4 (col % 4) ..+3
        // (logical element 16dt + 4(col%4) = chunk 2dt + (col%4)/2, half col%2)
        const int vr0 = 32 * kk + 4 * quad + (col >> 2), vr1 = vr0 + 16;
        const int vc = 2 * dt + ((col & 3) >> 1), vh = 4 * (col & 1);
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4*)&cur.v[vr0][8 * (vc ^ swz_v<D>(vr0)) + vh]);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4*)&cur.v[vr1][8 * (vc ^ swz_v<D>(vr1)) + vh]);
        const bf16x8 vop = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int s = 0; s < kSub; ++s)
          oacc[dt][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vop, pop[s], oacc[dt][s], 0, 0, 0);
      }
    };
    if constexpr (SPLIT && kKeys == 64) {
      if (share == 0) half(0);
      if (sharers == 1 || share == 1) half(1);
    } else if constexpr (SPLIT) {
#pragma nounroll
      for (int kk = 0; kk < kKeys / 32; ++kk)
        if ((kk & (sharers - 1)) == share) half(kk);
    } else if constexpr (kKeys == 64) {
      half(0);
      half(1);
    } else {
      // rolled: unrolled, the four quarters' operand reads crowd the registers
#pragma nounroll
      for (int kk = 0; kk < kKeys / 32; ++kk) half(kk);
    }

    // Without maxima the weights' sums are the check: a sum above kBig (a
    // score ~26 above the maximum, or slow growth over many tiles) is
    // renormalised by a power of two (exact); one above kHuge (a score ~58
    // above the maximum, inf included) may have overflowed O: the workgroup
    // restarts its keys with exact maxima on every tile.  NaN sums pass both
    // tests: NaN inputs reach the output.
    bool big = false, huge = false;
#pragma unroll
    for (int s = 0; s < kSub; ++s) {
      big |= lacc[s][0] > kBig;
      huge |= lacc[s][0] > kHuge;
    }
    if (__builtin_amdgcn_ballot_w64(big)) {
      if (!exact && __builtin_amdgcn_ballot_w64(huge)) lds.restart[restart_word(it_begin, it)] = 1;
      // sum -> [1/2, 1): O and the sum by 2^-e, the maximum up by e
#pragma unroll
      for (int s = 0; s < kSub; ++s) {
        const int e = lacc[s][0] > kBig ? __builtin_amdgcn_frexp_expf(lacc[s][0]) : 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) lacc[s][i] = __builtin_amdgcn_ldexpf(lacc[s][i], -e);
#pragma unroll
        for (int dt = 0; dt < kDTiles; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) oacc[dt][s][i] = __builtin_amdgcn_ldexpf(oacc[dt][s][i], -e);
        neg_m[s] -= static_cast<float>(e);
      }
    }
    if (unset) {
      bool none = false;
#pragma unroll
      for (int s = 0; s < kSub; ++s) none |= lacc[s][0] == 0.f;
      unset = __builtin_amdgcn_ballot_w64(none) != 0;
    }
    if (it + 1 < it_end) commit(nxt);
    __syncthreads();
  };
  // a restart starts the keys again from tile 0 with exact maxima; no load is
  // in flight after a barrier and neither buffer is still being read
  run_tiles(
      it_begin, it_end,
      [&](int it, auto half) {
        if constexpr (half == 0)
          step(it, lds.tile0, lds.tile1);
        else
          step(it, lds.tile1, lds.tile0);
      },
      [&](int it) -> bool {
        const volatile int32_t* word = &lds.restart[restart_word(it_begin, it)];
        return !exact_all && __builtin_amdgcn_readfirstlane(*word);
      },
      [&]() {
        exact_all = true;
        unset = true;
        clear_rows();
        if (it_begin < n_pref) fetch_slots(it_begin);
        open();
      });

  if constexpr (SPLIT) {
    // merge the sharers of each row group through the tiles' LDS (free after
    // the last tile's barrier), the upper half into the lower half
    for (int half_sharers = sharers >> 1; half_sharers > 0; half_sharers >>= 1) {
      const bool gives = share >= half_sharers && share < 2 * half_sharers, takes = share < half_sharers;
      const int region = (gives ? share - half_sharers : share) * groups + row_group;  // below 4
      // 16 KB of O, two regions to a tile buffer, and the rows' (m, l)
      f32x4* ro = reinterpret_cast<f32x4*>(region < 2 ? &lds.tile0.k[0][0] : &lds.tile1.k[0][0]) + (region & 1) * 1024;
      float2* rm = lds.merge + region * (16 * kSub);
      if (gives) {
#pragma unroll
        for (int s = 0; s < kSub; ++s) {
#pragma unroll
          for (int dt = 0; dt < kDTiles; ++dt) ro[(dt * kSub + s) * 64 + lane] = oacc[dt][s];
          if (quad == 0) rm[16 * s + col] = float2{lacc[s][0] != 0.f ? -neg_m[s] : -INFINITY, lacc[s][0]};
        }
      }
      __syncthreads();
      if (takes) {
#pragma unroll
        for (int s = 0; s < kSub; ++s) {
          const float2 ml = rm[16 * s + col];
          const float m0 = lacc[s][0] != 0.f ? -neg_m[s] : -INFINITY;
          const float mn = fmaxf(m0, ml.x);
          const float w0 = m0 == -INFINITY ? 0.f : exp2f(m0 - mn), w1 = ml.x == -INFINITY ? 0.f : exp2f(ml.x - mn);
          lacc[s][0] = lacc[s][0] * w0 + ml.y * w1;
          neg_m[s] = mn == -INFINITY ? 0.f : -mn;
#pragma unroll
          for (int dt = 0; dt < kDTiles; ++dt)
            oacc[dt][s] = oacc[dt][s] * w0 + ro[(dt * kSub + s) * 64 + lane] * w1;
        }
      }
      __syncthreads();
    }
    if (share != 0) return;
  }

  // a block whose keys are all here is normalised with the sink and stored; a
  // part of one goes to the workspace
  if (!SPLIT || (it_begin == 0 && it_end == n_tiles)) {
#pragma unroll
    for (int s = 0; s < kSub; ++s) {
      f32x4 o[kDTiles];
#pragma unroll
      for (int dt = 0; dt < kDTiles; ++dt) o[dt] = oacc[dt][s];
      const float l = lacc[s][0];
      store_row<D, GEN, kDTiles>(a, g, row_of(s), t0, qlen, qo0, quad, 0, o, l, l != 0.f ? -neg_m[s] : -INFINITY);
    }
  } else {
#pragma unroll
    for (int s = 0; s < kSub; ++s) {
#pragma unroll
      for (int dt = 0; dt < kDTiles; ++dt)
        reinterpret_cast<f32x4*>(part)[(dt * kSub + s) * kThreads + tid] = oacc[dt][s];
      const float l = lacc[s][0];
      if (quad == 0) {
        part[kPartialO + 2 * row_of(s)] = l != 0.f ? -neg_m[s] : -INFINITY;
        part[kPartialO + 2 * row_of(s) + 1] = l;
      }
    }
  }
}

template <int D, int KEYS, int SUB, typename IdxT, typename PosT, bool POS, bool GEN>
__global__ void __launch_bounds__(kThreads, SUB == 1 ? 4 : 2) context_attention_kernel(const CtxArgs a) {
  __shared__ __attribute__((aligned(16))) TileLds<D, KEYS> tile0, tile1;
  __shared__ int32_t rel_rows[block_rows(SUB)];
  __shared__ int32_t restart[kRestartWords];
  const Lds<D, KEYS, SUB> lds{tile0, tile1, rel_rows, restart, nullptr};
  // KV head fastest: workgroup id mod 8 picks the XCD, so with 8 KV heads
  // every XCD streams one head's K/V through its own L2.  Token blocks run
  // last-first: the last blocks see the most causal keys, and starting them
  // first shortens the tail of the launch.
  const int g = static_cast<int>(blockIdx.x % static_cast<unsigned>(a.kv_heads));
  const int32_t block = static_cast<int32_t>(gridDim.x / static_cast<unsigned>(a.kv_heads) - 1 -
                                             blockIdx.x / static_cast<unsigned>(a.kv_heads));
  const int seg = blockIdx.z;
  const bool i64 = a.indptr_i64;
  Segment sg;
  sg.q0 = load_index(a.qo_indptr, i64, seg);
  sg.q = static_cast<int32_t>(load_index(a.qo_indptr, i64, seg + 1) - sg.q0);
  sg.k0 = load_index(a.kv_indptr, i64, seg);
  // without prefix indices there is no prefix, whatever kv_indptr says
  sg.p = a.kv_indices ? static_cast<int32_t>(load_index(a.kv_indptr, i64, seg + 1) - sg.k0) : 0;
  if (block * a.tokens_per_block >= sg.q) return;
  attend<D, KEYS, SUB, IdxT, PosT, POS, GEN, false>(a, lds, sg, g, block, 0, -1, nullptr);
}

// The split launch: one workgroup per CU, each with an equal stretch of the
// batch's cost line (context_plan.h).  It is for batches whose plain grid
// leaves CUs idle: 200 new tokens over 19441 keys are 32 plain workgroups and
// took 560 us for the GPT-OSS layer, 93 us here and 13 in the merge (the matrix
// cores' share is 52 us; the rest is the cuts, a block's first tile, the parts'
// 28 MB each way and the second launch); six ragged Llama-3 segments (48-624
// queries over 4-14k keys) took 594 us, 437 us here with the merge.
//
// A stretch that starts inside a block leaves that block's part for last: the
// workgroups of an XCD then all begin at their blocks' first keys and walk
// the keys of a segment together.  What the loop carries waits in LDS and the
// arguments are read again for each piece, so the tile loop keeps the scalar
// registers it has in the plain kernel (held in registers, some 80 of them
// spilled to vector lanes inside the tile loop, which cost it 15-25%).
typedef __attribute__((address_space(4))) const CtxArgs kernel_args;

template <int D, int KEYS, typename IdxT, bool GEN>
__global__ void __launch_bounds__(kThreads, 2) context_split_kernel(const CtxArgs args) {
  __shared__ __attribute__((aligned(16))) TileLds<D, KEYS> tile0, tile1;
  __shared__ int32_t rel_rows[rows_per_block(D)];
  __shared__ int32_t restart[kRestartWords];
  __shared__ float2 merge[4 * 16 * sub_tiles(D)];
  __shared__ SplitState state;
  __shared__ Segment segments[kMaxSplitSegments];
  const Lds<D, KEYS, sub_tiles(D)> lds{tile0, tile1, rel_rows, restart, merge};
  {
    const SplitShape shape = split_shape<D, KEYS>(args);
    const int lane = threadIdx.x & 63;
    const BatchPlan plan = plan_batch(args, shape, lane);
    const int k = parts_shift(shape, plan.total, args.kv_heads, args.max_shift);
    const int id = static_cast<int>(blockIdx.x);
    if (plan.total == 0 || (id >> k)) {
      if (threadIdx.x == 0) split_cuts<D>(args)[id].at = Place{0, 0, 0, -1};
      return;
    }
    // workgroup id mod 8 picks the XCD: each XCD gets an eighth of the line
    SplitState s;
    s.rank = k >= 3 ? ((id & 7) << (k - 3)) + (id >> 3) : id;
    s.live = plan.live;
    const Place ends = lane_place(plan, shape, args.kv_heads, k, s.rank + (lane & 1));
    s.first = from_lane(ends, 0);
    s.end = from_lane(ends, 1);
    s.cur = s.first;
    s.last = 0;
    const int32_t qlen = __builtin_amdgcn_readlane(plan.q, s.first.seg);
    if (threadIdx.x == 0)
      split_cuts<D>(args)[s.rank] = Cut{s.first, read_lane(plan.q0, s.first.seg), qlen, 0};
    if (same_block(s.first, s.end) ? s.first.tile == s.end.tile
                                   : s.first.tile > 0 && !next_piece(shape, args.kv_heads, s, qlen))
      return;
    if (threadIdx.x == 0) state = s;
    if (threadIdx.x < kMaxSplitSegments) segments[threadIdx.x] = Segment{plan.q0, plan.k0, plan.q, plan.p};
    __syncthreads();
  }
  kernel_args* kp = (kernel_args*)__builtin_amdgcn_kernarg_segment_ptr();
  for (;;) {
    asm volatile("" : "+s"(kp));
    const CtxArgs& a = *(const CtxArgs*)kp;
    {
      const Place at = uniform(state.cur), end = uniform(state.end);
      const int rank = uniform(state.rank);
      // part 2 rank: the stretch's first block, entered past its first tile;
      // part 2 rank + 1: its last, left before its last tile
      float* part = a.partial + (2 * rank + (at.tile > 0 ? 0 : 1)) * partial_floats<D>();
      const Segment v = segments[at.seg];
      const Segment sg{uniform(v.q0), uniform(v.k0), uniform(v.q), uniform(v.p)};
      attend<D, KEYS, sub_tiles(D), IdxT, int64_t, false, GEN, true>(a, lds, sg, at.head, at.block, at.tile,
                                                                     same_block(at, end) ? end.tile : -1, part);
    }
    SplitState s = state;
    s.cur = uniform(s.cur);
    s.first = uniform(s.first);
    s.end = uniform(s.end);
    s.live = static_cast<uint64_t>(uniform(static_cast<int64_t>(s.live)));
    s.last = uniform(s.last);
    if (!next_piece(split_shape<D, KEYS>(a), a.kv_heads, s, uniform(segments[s.cur.seg].q))) return;
    __syncthreads();
    if (threadIdx.x == 0) state = s;
    __syncthreads();
  }
}

// Merges the parts of each block that a boundary between two stretches cuts.
// Workgroup = (64 / 32 rows of one wave of the main kernel, boundary); the
// block's first boundary does the work.  A wave takes one row subtile and two
// 16-dim tiles, every lane the same rows and dims as in the main kernel, so
// the parts are read in whole 1 KiB accesses, four parts at a time: the cost
// is round trips (the cuts, then the parts), not bandwidth.
constexpr int kCombineDims = 2;  // 16-dim tiles of a wave
template <int D, bool GEN>
__global__ void __launch_bounds__(512) context_combine_kernel(const CtxArgs a) {
  constexpr int kSub = sub_tiles(D);
  constexpr int kAhead = 4;  // parts in flight together (8 and 12: most blocks have fewer, 1-6% slower)
  static_assert(64 * kSub * (D / 16 / kCombineDims) == 512, "one wave per row subtile and pair of dim tiles");
  const int lane = threadIdx.x & 63;
  const int w = uniform(static_cast<int32_t>(threadIdx.x >> 6));
  const int s = w % kSub, dt0 = w / kSub * kCombineDims;
  const int wave = blockIdx.x;
  const int r0 = blockIdx.y + 1;
  // lane i: boundary r0 - 1 + i
  const Cut* cuts = split_cuts<D>(a);
  auto load_cut = [&](int r) {
    const bool in = r < 1 << a.max_shift;
    Cut c = cuts[in ? r : 0];
    if (!in) c.at.tile = -1;
    return c;
  };
  Cut mine = load_cut(r0 - 1 + lane);
  const Place at = from_lane(mine.at, 1), prev = from_lane(mine.at, 0);
  // nothing, or a boundary between two blocks, or not the block's first
  if (at.tile <= 0 || (prev.tile > 0 && same_block(prev, at))) return;
  const int64_t qo0 = read_lane(mine.q0, 1);
  const int32_t qlen = __builtin_amdgcn_readlane(mine.q, 1);
  const int32_t t0 = at.block * a.tokens_per_block;
  if (t0 + ((wave * 16 * kSub) >> a.group_shift) >= qlen) return;  // no rows here (nor a part with them)
  const int row = wave * (16 * kSub) + 16 * s + (lane & 15);
  f32x4 o[kCombineDims];
#pragma unroll
  for (int dt = 0; dt < kCombineDims; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  // the block's parts: its first tiles, up to boundary r0, by the workgroup
  // before it, then one part from each of its boundaries, unless the next
  // boundary lies on the same tile
  int base = r0 - 1, first = 2 * r0 - 1;
  bool more = true;
  while (more) {
    // lane i: boundary base + i and the one after it (lane 63's: not known)
    const int32_t here = base + lane >= r0 && same_block(mine.at, at) ? mine.at.tile : -1;
    const int32_t next = __shfl_down(here, 1);
    more = __builtin_amdgcn_readlane(here, 63) > 0;
    uint64_t parts = __builtin_amdgcn_ballot_w64(here > 0 && lane < 63 && here != next);
    while (parts || first >= 0) {
      f32x4 op[kAhead][kCombineDims];
      float2 ml[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        int slot = 2 * r0 - 1;  // past the last part: the first one again, with no weight
        bool has = true;
        if (first >= 0) {
          first = -1;
        } else if (parts) {
          slot = 2 * (base + __builtin_ctzll(parts));
          parts &= parts - 1;
        } else {
          has = false;
        }
        const float* part = a.partial + slot * partial_floats<D>();
        ml[u] = *reinterpret_cast<const float2*>(part + kPartialO + 2 * row);
        if (!has) ml[u].x = -INFINITY;
#pragma unroll
        for (int dt = 0; dt < kCombineDims; ++dt)
          op[u][dt] = reinterpret_cast<const f32x4*>(part)[((dt0 + dt) * kSub + s) * kThreads + wave * 64 + lane];
      }
      float mn = m;
#pragma unroll
      for (int u = 0; u < kAhead; ++u) mn = fmaxf(mn, ml[u].x);
      const float wo = m == -INFINITY ? 0.f : exp2f(m - mn);
      l *= wo;
#pragma unroll
      for (int dt = 0; dt < kCombineDims; ++dt) o[dt] *= wo;
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        // a row without a key in the part (or no part at all) adds nothing
        const bool none = ml[u].x == -INFINITY;
        const float wu = none ? 0.f : exp2f(ml[u].x - mn);
        l += none ? 0.f : ml[u].y * wu;
#pragma unroll
        for (int dt = 0; dt < kCombineDims; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[dt][i] += none ? 0.f : op[u][dt][i] * wu;
      }
      m = mn;
    }
    base += 63;
    if (more) mine = load_cut(base + lane);
  }
  store_row<D, GEN, kCombineDims>(a, at.head, row, t0, qlen, qo0, lane >> 4, dt0, o, l, m);
}

// SUB 0: the split launch
template <int D, int KEYS, int SUB, typename IdxT, bool GEN>
void launch_pos(int pos, dim3 grid, hipStream_t st, const CtxArgs& a) {
  // pos: 0 none, 1 int32, 2 int64; only a window looks at positions, and
  // neither a split launch nor one of 128-key tiles has one
  if constexpr (SUB == 0) {
    hipLaunchKernelGGL((context_split_kernel<D, KEYS, IdxT, GEN>), grid, dim3(kThreads), 0, st, a);
    if (grid.x > 1)
      hipLaunchKernelGGL((context_combine_kernel<D, GEN>), dim3(kWaves, grid.x - 1), dim3(512), 0, st, a);
  } else {
    if (KEYS == 128 || pos == 0)
      hipLaunchKernelGGL((context_attention_kernel<D, KEYS, SUB, IdxT, int64_t, false, GEN>), grid, dim3(kThreads), 0,
                         st, a);
    if constexpr (KEYS != 128) {
      if (pos == 2)
        hipLaunchKernelGGL((context_attention_kernel<D, KEYS, SUB, IdxT, int64_t, true, GEN>), grid, dim3(kThreads), 0,
                           st, a);
      else if (pos == 1)
        hipLaunchKernelGGL((context_attention_kernel<D, KEYS, SUB, IdxT, int32_t, true, GEN>), grid, dim3(kThreads), 0,
                           st, a);
    }
  }
}

template <int D, int KEYS, int SUB, typename IdxT>
void launch_gen(int pos, dim3 grid, hipStream_t st, const CtxArgs& a) {
  // the general instance for caps, narrower heads and padded groups
  if (a.cap > 0.f || a.head_dim != D || a.group != (1 << a.group_shift))
    launch_pos<D, KEYS, SUB, IdxT, true>(pos, grid, st, a);
  else
    launch_pos<D, KEYS, SUB, IdxT, false>(pos, grid, st, a);
}

template <int D, int KEYS, int SUB>
void launch_idx(bool idx64, int pos, dim3 grid, hipStream_t st, const CtxArgs& a) {
  if (idx64)
    launch_gen<D, KEYS, SUB, int64_t>(pos, grid, st, a);
  else
    launch_gen<D, KEYS, SUB, int32_t>(pos, grid, st, a);
}

// Whether a window takes blocks of a quarter of the rows.  Such a block sees
// few keys outside its rows' windows, and two of them share a CU, which hides
// the latency that a narrow window's few tiles consist of; but there are four
// times as many, and each stages its own window.  Full blocks run in whole
// rounds of 256, counted with the empty ones of a ragged batch's grid (the
// CUs that meet those wait all the same); short ones, 512 at once, even out.
// Times in microseconds, fitted to full | short blocks of one segment with
// GPT-OSS heads at windows 64, 128, 256, 512:
//   1000 tokens (half a round):  18.6 | 11.3, 20.6 | 13.5, 24.4 | 16.4, 32.2 | 22.0
//   2000 (one):                  21.5 | 20.6, 23.4 | 23.3, 27.1 | 29.0, 35.2 | 39.3
//   3000 (one and a half):       39.5 | 30.6, 43.0 | 33.8, 50.8 | 41.7, 66.2 | 57.0
//   8192 (four):                 80.1 | 68.9, 87.7 | 76.7, 103.7 | 94.5, 134.3 | 133.8
// Heads of 32 dims (full blocks load less, short ones still clear their tiles)
// at window 128: 2000 tokens 18.2 | 22.2, 3000 34.2 | 31.5.  512-token blocks
// (group 1), 4096 tokens: 54.7 | 30.8.  Six segments of 33-600 tokens, window
// 128 and 512: 38.4 | 24.0, 63.5 | 40.3.
bool narrow_blocks(int32_t head_dim, int32_t group_shift, int32_t window, int64_t kv_heads, int64_t segments,
                   int64_t max_query_len, int64_t total_queries) {
  if (head_dim > 64 || window < 0 || window > kNarrowWindow) return false;
  const int64_t full = block_rows(sub_tiles(64)) >> group_shift, part = block_rows(kNarrowSub) >> group_shift;
  const int64_t full_blocks = (max_query_len + full - 1) / full * segments;
  int64_t part_blocks = (max_query_len + part - 1) / part * segments;
  // of unequal segments, each leaves half a block empty
  if (total_queries > 0 && total_queries < max_query_len * segments)
    part_blocks = std::min(part_blocks, total_queries / part + (segments + 1) / 2);
  const double full_round = 9. + 11. * head_dim / 64. + 0.027 * window + 0.085 * std::max<int64_t>(0, full - 64);
  const double part_round = 6.3 + 0.02 * window + 0.028 * part;
  return 1.02 * (6. + part_round * std::max(1., part_blocks * kv_heads / 512.)) <
         full_round * ((full_blocks * kv_heads + 255) / 256);
}

void launch_typed(bool split, bool narrow, bool idx64, int pos, dim3 grid, hipStream_t st, const CtxArgs& a) {
  const bool wide = a.head_dim > 64;
  if (split)
    wide ? launch_idx<128, 64, 0>(idx64, pos, grid, st, a) : launch_idx<64, 128, 0>(idx64, pos, grid, st, a);
  else if (wide)
    launch_idx<128, 64, sub_tiles(128)>(idx64, pos, grid, st, a);
  else if (narrow)
    launch_idx<64, 64, kNarrowSub>(idx64, pos, grid, st, a);
  else if (a.window >= 0)
    launch_idx<64, 64, sub_tiles(64)>(idx64, pos, grid, st, a);
  else
    launch_idx<64, 128, sub_tiles(64)>(idx64, pos, grid, st, a);
}

int group_shift_of(int32_t group) {
  int s = 0;
  while ((1 << s) < group) ++s;  // rows per token: the group padded to 2^s
  return s;
}

// Workspace of 2^shift workgroups.
int64_t split_bytes(int32_t head_dim, int shift) {
  return static_cast<int64_t>(8 * (head_dim > 64 ? partial_floats<128>() : partial_floats<64>()) + sizeof(Cut)) << shift;
}

}  // namespace
}  // namespace akv

namespace akv {
namespace {

int run_context_attention(const void* q, int64_t q_stride_t, int64_t q_stride_h, const void* k_ext,
                                     const void* v_ext, int64_t k_ext_stride_t, int64_t k_ext_stride_h,
                                     int64_t v_ext_stride_t, int64_t v_ext_stride_h, const void* k_buffer,
                                     const void* v_buffer, int64_t k_stride_slot, int64_t k_stride_head,
                                     int64_t v_stride_slot, int64_t v_stride_head, int32_t n_segments,
                                     int32_t q_heads, int32_t kv_heads, int32_t head_dim, const void* qo_indptr,
                                     const void* kv_indptr, int32_t indptr_dtype, const void* kv_indices,
                                     int32_t indices_dtype, const void* q_positions, const void* kv_positions,
                                     int32_t positions_dtype, int32_t sliding_window, const float* sinks,
                                     float scale, float logit_cap, void* out, int32_t out_dtype,
                                     int64_t out_stride_t, int64_t out_stride_h, int64_t max_query_len,
                                     int64_t total_queries, bool split, void* workspace, int64_t workspace_bytes, void* stream) {
  if (n_segments < 0 || max_query_len < 0) return fail(AKV_EINVAL, "akv_context_attention: negative size");
  if (n_segments == 0 || max_query_len == 0) return AKV_OK;
  // heads of up to 128 dims in 16-byte chunks: the kernel's 64- or 128-dim
  // tiles with the dims past head_dim zero
  if (head_dim < 8 || head_dim > 128 || head_dim % 8 != 0)
    return fail(AKV_EINVAL, "akv_context_attention: head_dim %d (supported: multiples of 8 up to 128)", head_dim);
  // a block's rows are (token, q head) pairs with the group padded to a
  // power of two (at most 128 q heads per KV head); a row packs its q head
  // into 15 bits
  if (kv_heads <= 0 || q_heads <= 0 || q_heads % kv_heads != 0 || q_heads / kv_heads > 128 || q_heads > 32767)
    return fail(AKV_EINVAL, "akv_context_attention: %d q heads over %d KV heads (at most 128 per KV head)",
                q_heads, kv_heads);
  if (!(logit_cap >= 0.f) || !std::isfinite(logit_cap))
    return fail(AKV_EINVAL, "akv_context_attention: logit_cap must be 0 (none) or positive and finite");
  if (!valid_index_dtype(indptr_dtype) || !valid_index_dtype(indices_dtype) ||
      !valid_index_dtype(positions_dtype))
    return fail(AKV_EINVAL, "akv_context_attention: index vectors must be int32 or int64");
  if (out_dtype != AKV_BF16 && out_dtype != AKV_F32)
    return fail(AKV_EINVAL, "akv_context_attention: output must be bf16 or f32");
  if (split && (sliding_window > 0 || n_segments > kMaxSplitSegments || !workspace ||
                workspace_bytes < split_bytes(head_dim, 0) || (reinterpret_cast<uintptr_t>(workspace) & 15) != 0))
    return fail(AKV_EINVAL, "akv_context_attention_split: needs no window, at most %d segments and %lld aligned bytes",
                kMaxSplitSegments, static_cast<long long>(split_bytes(head_dim, 0)));
  if (!q || !k_ext || !v_ext || !out || !qo_indptr || !kv_indptr)
    return fail(AKV_EINVAL, "akv_context_attention: null device pointer");
  // prefix keys are read from the pools through kv_indices
  if (kv_indices && (!k_buffer || !v_buffer))
    return fail(AKV_EINVAL, "akv_context_attention: prefix indices given without K/V pools");
  if ((q_positions == nullptr) != (kv_positions == nullptr))
    return fail(AKV_EINVAL, "akv_context_attention: needs both query and KV positions or neither");
  const int64_t strides[] = {q_stride_t,    q_stride_h,    k_ext_stride_t, k_ext_stride_h, v_ext_stride_t,
                             v_ext_stride_h, k_stride_slot, k_stride_head,  v_stride_slot,  v_stride_head,
                             out_stride_t,  out_stride_h};
  for (int64_t s : strides) {
    if (s % 8 != 0) return fail(AKV_EINVAL, "akv_context_attention: row strides must be multiples of 8 elements");
    if (s < 0 || s > 0x7fffffffLL) return fail(AKV_EINVAL, "akv_context_attention: strides must fit 31 bits");
  }
  const uintptr_t bases = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_ext) |
                          reinterpret_cast<uintptr_t>(v_ext) | reinterpret_cast<uintptr_t>(k_buffer) |
                          reinterpret_cast<uintptr_t>(v_buffer) | reinterpret_cast<uintptr_t>(out);
  if (bases & 15) return fail(AKV_EINVAL, "akv_context_attention: tensors must be 16-byte aligned");
  if (n_segments > 65535 || kv_heads > 65535)
    return fail(AKV_EINVAL, "akv_context_attention: batch too large");
  // masked scores are -inf before the scale: the softmax needs scale > 0
  if (!(scale > 0.f) || !std::isfinite(scale))
    return fail(AKV_EINVAL, "akv_context_attention: scale must be positive and finite");
  CtxArgs a{};
  a.q = static_cast<const __bf16*>(q);
  a.k_ext = static_cast<const __bf16*>(k_ext);
  a.v_ext = static_cast<const __bf16*>(v_ext);
  a.k_pool = static_cast<const __bf16*>(k_buffer);
  a.v_pool = static_cast<const __bf16*>(v_buffer);
  a.qo_indptr = qo_indptr;
  a.kv_indptr = kv_indptr;
  a.kv_indices = kv_indices;
  a.q_pos = q_positions;
  a.kv_pos = kv_positions;
  a.sinks = sinks;
  a.out = out;
  a.q_st = static_cast<int32_t>(q_stride_t);
  a.q_sh = static_cast<int32_t>(q_stride_h);
  a.ke_st = static_cast<int32_t>(k_ext_stride_t);
  a.ke_sh = static_cast<int32_t>(k_ext_stride_h);
  a.ve_st = static_cast<int32_t>(v_ext_stride_t);
  a.ve_sh = static_cast<int32_t>(v_ext_stride_h);
  a.kp_ss = static_cast<int32_t>(k_stride_slot);
  a.kp_sh = static_cast<int32_t>(k_stride_head);
  a.vp_ss = static_cast<int32_t>(v_stride_slot);
  a.vp_sh = static_cast<int32_t>(v_stride_head);
  a.o_st = static_cast<int32_t>(out_stride_t);
  a.o_sh = static_cast<int32_t>(out_stride_h);
  a.indptr_i64 = indptr_dtype == AKV_I64;
  // as the extend kernel this replaces, a window applies only when it is
  // positive (akv/system/sglang.patch:527-541): 0 means plain causal
  a.window = sliding_window > 0 ? sliding_window : -1;
  a.scale_log2 = scale * kLog2e;
  a.out_f32 = out_dtype == AKV_F32;
  a.group = q_heads / kv_heads;
  a.group_shift = group_shift_of(a.group);
  const int tile_dim = head_dim > 64 ? 128 : 64;
  const bool narrow = narrow_blocks(head_dim, a.group_shift, a.window, kv_heads, n_segments, max_query_len,
                                    total_queries);
  a.tokens_per_block = block_rows(narrow ? kNarrowSub : sub_tiles(tile_dim)) >> a.group_shift;
  a.head_dim = head_dim;
  a.cap = logit_cap;
  a.cap_log2 = logit_cap * kLog2e;
  const int64_t blocks = (max_query_len + a.tokens_per_block - 1) / a.tokens_per_block;
  if (blocks * kv_heads > 0x7fffffffLL) return fail(AKV_EINVAL, "akv_context_attention: queries too long");
  a.kv_heads = kv_heads;
  a.n_segments = n_segments;
  while (split && a.max_shift < kSplitShift && split_bytes(head_dim, a.max_shift + 1) <= workspace_bytes) ++a.max_shift;
  a.partial = static_cast<float*>(workspace);
  const dim3 grid = split ? dim3(1u << a.max_shift)
                          : dim3(static_cast<unsigned>(blocks * kv_heads), 1u, static_cast<unsigned>(n_segments));
  hipStream_t st = as_stream(stream);
  const bool idx64 = indices_dtype == AKV_I64;
  const int pos = q_positions == nullptr || a.window < 0 ? 0 : (positions_dtype == AKV_I64 ? 2 : 1);
  launch_typed(split, narrow, idx64, pos, grid, st, a);
  return check_launch("akv_context_attention");
}

}  // namespace
}  // namespace akv

extern "C" int akv_context_attention_sized(
    const void* q, int64_t q_stride_t, int64_t q_stride_h, const void* k_ext,
    const void* v_ext, int64_t k_ext_stride_t, int64_t k_ext_stride_h, int64_t v_ext_stride_t, int64_t v_ext_stride_h,
    const void* k_buffer, const void* v_buffer, int64_t k_stride_slot, int64_t k_stride_head, int64_t v_stride_slot,
    int64_t v_stride_head, int32_t n_segments, int32_t q_heads, int32_t kv_heads, int32_t head_dim,
    const void* qo_indptr, const void* kv_indptr, int32_t indptr_dtype, const void* kv_indices, int32_t indices_dtype,
    const void* q_positions, const void* kv_positions, int32_t positions_dtype, int32_t sliding_window,
    const float* sinks, float scale, float logit_cap, void* out, int32_t out_dtype, int64_t out_stride_t,
    int64_t out_stride_h, int64_t max_query_len, int64_t total_queries,
    void* stream) {
  return akv::run_context_attention(
      q, q_stride_t, q_stride_h, k_ext, v_ext, k_ext_stride_t, k_ext_stride_h, v_ext_stride_t, v_ext_stride_h, k_buffer,
      v_buffer, k_stride_slot, k_stride_head, v_stride_slot, v_stride_head, n_segments, q_heads, kv_heads, head_dim,
      qo_indptr, kv_indptr, indptr_dtype, kv_indices, indices_dtype, q_positions, kv_positions, positions_dtype,
      sliding_window, sinks, scale, logit_cap, out, out_dtype, out_stride_t, out_stride_h, max_query_len,
      total_queries, false, nullptr, 0, stream);
}

extern "C" int akv_context_attention(
    const void* q, int64_t q_stride_t, int64_t q_stride_h, const void* k_ext,
    const void* v_ext, int64_t k_ext_stride_t, int64_t k_ext_stride_h, int64_t v_ext_stride_t, int64_t v_ext_stride_h,
    const void* k_buffer, const void* v_buffer, int64_t k_stride_slot, int64_t k_stride_head, int64_t v_stride_slot,
    int64_t v_stride_head, int32_t n_segments, int32_t q_heads, int32_t kv_heads, int32_t head_dim,
    const void* qo_indptr, const void* kv_indptr, int32_t indptr_dtype, const void* kv_indices, int32_t indices_dtype,
    const void* q_positions, const void* kv_positions, int32_t positions_dtype, int32_t sliding_window,
    const float* sinks, float scale, float logit_cap, void* out, int32_t out_dtype, int64_t out_stride_t,
    int64_t out_stride_h, int64_t max_query_len,
    void* stream) {
  return akv_context_attention_sized(
      q, q_stride_t, q_stride_h, k_ext, v_ext, k_ext_stride_t, k_ext_stride_h, v_ext_stride_t, v_ext_stride_h, k_buffer,
      v_buffer, k_stride_slot, k_stride_head, v_stride_slot, v_stride_head, n_segments, q_heads, kv_heads, head_dim,
      qo_indptr, kv_indptr, indptr_dtype, kv_indices, indices_dtype, q_positions, kv_positions, positions_dtype,
      sliding_window, sinks, scale, logit_cap, out, out_dtype, out_stride_t, out_stride_h, max_query_len, 0, stream);
}

extern "C" int akv_context_attention_split(
    const void* q, int64_t q_stride_t, int64_t q_stride_h, const void* k_ext,
    const void* v_ext, int64_t k_ext_stride_t, int64_t k_ext_stride_h, int64_t v_ext_stride_t, int64_t v_ext_stride_h,
    const void* k_buffer, const void* v_buffer, int64_t k_stride_slot, int64_t k_stride_head, int64_t v_stride_slot,
    int64_t v_stride_head, int32_t n_segments, int32_t q_heads, int32_t kv_heads, int32_t head_dim,
    const void* qo_indptr, const void* kv_indptr, int32_t indptr_dtype, const void* kv_indices, int32_t indices_dtype,
    const void* q_positions, const void* kv_positions, int32_t positions_dtype, int32_t sliding_window,
    const float* sinks, float scale, float logit_cap, void* out, int32_t out_dtype, int64_t out_stride_t,
    int64_t out_stride_h, int64_t max_query_len,
    void* workspace, int64_t workspace_bytes, void* stream) {
  return akv::run_context_attention(
      q, q_stride_t, q_stride_h, k_ext, v_ext, k_ext_stride_t, k_ext_stride_h, v_ext_stride_t, v_ext_stride_h, k_buffer,
      v_buffer, k_stride_slot, k_stride_head, v_stride_slot, v_stride_head, n_segments, q_heads, kv_heads, head_dim,
      qo_indptr, kv_indptr, indptr_dtype, kv_indices, indices_dtype, q_positions, kv_positions, positions_dtype,
      sliding_window, sinks, scale, logit_cap, out, out_dtype, out_stride_t, out_stride_h, max_query_len,
      0, true, workspace, workspace_bytes, stream);
}

// Which launch: both times estimated in 64-key tiles of a full block (2.0 us,
// at either head_dim), from what the host knows.  The plain grid's workgroups
// run in ceil(groups / CUs) rounds of the longest block (or, of many unequal
// ones, one round more than they fill), after ~12 us; the
// split launch shares all tiles out evenly at ~6% more a tile, plus ~10 us for
// each block a workgroup enters (queries, first tile, result) and ~18 us of
// its own (the cuts, the second launch).  Measured plain / split, us, GPT-OSS
// (64 q / 8 KV heads x 64) | Llama-3 (32 / 8 x 128), new tokens over prefix
// keys: 16 / 1000: 43 / 22 | 38 / 22; 200 / 400: 36 / 37 | 29 / 29; 200 / 1000:
// 50 / 38 | 46 / 34; 800 / 300: 48 / 47 | 42 / 40; 800 / 5000: 182 / 105 | 184 /
// 100; 1500 / 5000: 203 / 174 | 204 / 169; 1800 / 5000: 213 / 206 | 215 / 201
// (the rule says plain); 2040 / 19000 (one full round): 631 / 662 | 642 / 650;
// 3000 / 300: 117 / 141 | 108 / 120; 3000 / 5000: 385 / 352 | 385 / 340; 4096 /
// 19441 (two full rounds): 1294 / 1384 | 1321 / 1360; 6 x 682 / 300: 97 / 103 |
// 77 / 86; 6 x 682 / 1000: 152 / 147 | 138 / 133; 6 x 682 / 5000: 498 / 413 |
// 499 / 400; 32 x 1 / 2000: 76 / 41 | 76 / 56.
extern "C" int64_t akv_context_attention_split_bytes(int32_t n_segments, int32_t q_heads, int32_t kv_heads,
                                                     int32_t head_dim, int32_t sliding_window, int64_t total_queries,
                                                     int64_t max_query_len, int64_t total_prefix) {
  using namespace akv;
  if (n_segments <= 0 || n_segments > kMaxSplitSegments || sliding_window > 0 || kv_heads <= 0 || q_heads < kv_heads ||
      q_heads / kv_heads > 128 || head_dim <= 0 || head_dim > 128 || total_queries <= 0 || max_query_len <= 0)
    return 0;
  const int64_t tokens = rows_per_block(head_dim > 64 ? 128 : 64) >> group_shift_of(q_heads / kv_heads);
  if (total_prefix < 0) return 0;
  const int64_t queries = n_segments == 1 && max_query_len < total_queries ? max_query_len : total_queries;
  // one segment's blocks are known; of several, each leaves half a block empty
  const int64_t most = (std::min(queries, max_query_len) + tokens - 1) / tokens * n_segments;
  const int64_t blocks = n_segments == 1 ? most : std::min(most, queries / tokens + (n_segments + 1) / 2);
  const int64_t groups = blocks * kv_heads, rounds = (groups + kSplitGroups - 1) / kSplitGroups;
  const int64_t prefix = total_prefix / n_segments, own = queries / n_segments / 2;
  // how unequal several prefixes are is not known: for equal ones that fill
  // whole rounds the plain launch is the better one (64 segments of 9-28 queries,
  // 28 / 4 heads x 128, over ~1900 keys: 99 plain, 104 split; 32 of 7-29, 40 / 8
  // heads, over 2268: 100 | 124)
  const int64_t longest = (n_segments == 1 ? prefix : prefix + prefix / 4) + own;
  const double share = static_cast<double>(groups) / kSplitGroups, tiles = (prefix + own) / 64.;
  const double plain = 6. + std::min(rounds * (longest / 64.), (share + 1.) * tiles);
  // more heads than XCDs: an XCD's workgroups walk the keys of several heads
  // (6 x 682 new tokens over 5000 keys, 64 heads x 128: 972 plain, 1018 split)
  const double tile = kv_heads > 8 ? 1.06 * 1.08 : 1.06;
  const double split = tile * share * tiles + 5. * (share + 1.) + 9.;
  if (plain <= split) return 0;
  // no more stretches than the batch can have: a turn of 16 tokens over 1000 keys
  // takes 9 MB, and 69 MB where all CUs work
  const SplitShape shape{__builtin_ctz(static_cast<uint32_t>(tokens)), head_dim > 64 ? 6 : 7};
  const int64_t cost = cost_bound(shape, n_segments, queries, total_prefix);
  return split_bytes(head_dim, parts_shift(shape, cost, kv_heads, kSplitShift));
}
