// Causal varlen prefill attention over the paged BF16 workspace (gfx950).
//
// Reference path: the vLLM FlashAttention call of the FragPack backend
// (fragpack/integrations/vllm/backend.py:560-575, prefill groups :387-444):
// flash_attn_varlen_func(q, k = wk, v = wv, out, cu_seqlens_q, max_seqlen_q,
// seqused_k, max_seqlen_k, softmax_scale, causal=True, block_table).  The
// workspace is what HbmKvStore.gather writes: token-major BF16
// [pages, 128, H, 128]; sequence b's key j lives in page
// block_table[b][j / 128], row j % 128.  Queries are the last
// q_len = cu[b+1] - cu[b] positions of the sequence (causal mask aligned
// bottom-right: query i sees keys j <= i + seqused_k - q_len).
//
// Design (MI355X):
// * One 512-thread workgroup (8 wavefronts) per (256-row query tile, KV head).
//   The 256 rows are T = 256 / G tokens x G query heads of the KV head
//   (head-major), so every K / V tile read serves the whole GQA group and
//   eight waves.  Wave w owns rows 32w .. 32w + 31 as two 16-column MFMA
//   tiles.  Grids that would leave CUs idle, and fresh prompts of few tiles a
//   CU, run two 4-wave workgroups per tile; grids of no more tiles than CUs
//   over long contexts split the keys over the CUs (below; prefill_launch has
//   the rules).
// * Keys stream in 64-key tiles through double-buffered LDS, K and V both
//   key-major and loaded straight from HBM into LDS (buffer_load ... lds, no
//   registers).  K fragments are plain 16-byte reads; V^T fragments come
//   from ds_read_b64_tr_b16 transposing reads.
// * S^T = K Q^T and O^T += V^T P^T with v_mfma_f32_16x16x32_bf16.  The
//   accumulator layout of S^T (lane = query column, 4 consecutive keys per
//   16-lane group) is, after BF16 packing, exactly the B operand of the PV
//   product once the PV contraction visits keys in the matching order
//   {4q..4q+3, 16+4q..16+4q+3} -- P never leaves registers.
// * Online softmax in the log2 domain (exp2), P rounded to BF16 for PV while
//   l sums the fp32 P -- the arithmetic FlashAttention uses.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/fragpack_hip.h"
#include "fp_capi_internal.hpp"
#include "fp_record.hpp"

namespace fp {
namespace {

typedef __bf16 pf_bf16x8 __attribute__((ext_vector_type(8)));
typedef float pf_f32x4 __attribute__((ext_vector_type(4)));

constexpr int kPfQt = 2;           // 16-row query tiles per wavefront
constexpr int kPfWaves = 8;        // wavefronts per workgroup
constexpr int kPfWavesPerEu = 2;
constexpr int kPfXcds = 8;
constexpr int kPfWaveRows = 16 * kPfQt;          // query rows (token x head) per wavefront
constexpr int kPfRows = kPfWaveRows * kPfWaves;  // and per workgroup of 8
constexpr int kPfKeys = 64;        // keys per LDS tile
constexpr int kPfDim = 128;
// K and V tiles in LDS: key-major rows of 256 bytes whose 16-byte chunks are
// XOR-swizzled by the row (chunk c of row r at slot c ^ tile_swizzle(r)): K by
// r % 16, so the fragment reads of 16 consecutive rows cover all banks; V by
// 2 (r % 8), so the 32-byte pieces that 32 lanes of a transposing read take
// from 8 consecutive rows do (swizzled like K they met two to a bank: 135 M
// of 406 M LDS cycles at 4 x 8192 tokens, H 8, G 4, now none).
constexpr int kKRow = 256;
constexpr int kKBytes = kPfKeys * kKRow;   // 16384 (K or V)
constexpr float kLazyMax = 8.f;  // log2 headroom of the softmax reference max

struct PrefillParams {
  const uint16_t* q;
  const uint16_t* wk;
  const uint16_t* wv;
  const int32_t* cu_q;
  const int32_t* seq_k;
  const int32_t* block_table;
  uint16_t* out;
  int64_t q_stride;    // elements between consecutive query tokens
  int64_t out_stride;  // elements between consecutive output tokens
  int64_t bt_stride;
  int64_t num_pages;
  int kvh, group, num_seqs, tiles_per_seq;
  int head_sets;  // heads of a grid row: 8, 4, 2 or 1; negated: its sequences take turns
  float scale_log2;
  int causal;
  // split launches: parts' O, m and l, two slots per workgroup; and per key
  // tile (flattened) and wave the column maxima and whether they may matter
  float* opart;
  float* ml;
  float* tile_max;
  uint8_t* tile_flag;
  int4* ranges;  // two per workgroup, see PfRange
  int64_t tile_cap;  // key tiles these hold (more only if the lengths exceed the host's sizes)
};

__device__ __forceinline__ pf_f32x4 pf_mfma(const uint4& a, const uint4& b, pf_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(pf_bf16x8, a), __builtin_bit_cast(pf_bf16x8, b),
                                                  c, 0, 0, 0);
}

// Two floats -> BF16 pair (x low), round to nearest even: one v_cvt_pk_bf16_f32.
typedef float pf_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 pf_bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_bf16(float x, float y) {
  const pf_f32x2 v = {x, y};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, pf_bf16x2));
}


// Butterfly partners across 16- and 32-lane halves with the gfx950 lane
// swaps (VALU, no LDS round trip): with both operands x, one result holds
// the lane's own value and the other its partner's (lane ^ 16 / lane ^ 32).
__device__ __forceinline__ float pf_xor16_max(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pf_xor32_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pf_xor16_sum(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float pf_xor32_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

typedef __amdgpu_buffer_rsrc_t pf_rsrc_t;
typedef __attribute__((address_space(3))) void* pf_lds_ptr_t;

// A 64-key tile lies in one 128-token page (tiles start at multiples of 64):
// rows key0 .. key0 + 63 of head h are ``kvh * 256`` bytes apart, starting
// at the tile's first row.
__device__ __forceinline__ pf_rsrc_t tile_rsrc(const uint16_t* base, int64_t page, int key0, int h, int kvh,
                                               bool live) {
  const uint16_t* first = base + ((page * 128 + (key0 & 127)) * kvh + h) * kPfDim;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(first), (short)0, live ? 64 * kvh * kPfDim * 2 : 0,
                                           0x00020000);
}

// Transfers a 64-key tile of K and of V straight into LDS (buffer_load ...
// lds): rows of 256 bytes, 16-byte chunk c of row r at slot c ^ swizzle(r).
// Each wave instruction fills 1 KB = four rows, lane L the slot L % 16 of row
// L / 16, so lane L fetches chunk (L % 16) ^ swizzle(row).  ``off`` holds the
// lane's byte offsets in a whole tile; rows past the tile's ``nkeys`` repeat
// its last row: V rows stay finite (their P is 0) and every load stays inside
// the page.
// transfer instructions per wave, tile and operand, four rows each
__host__ __device__ constexpr int tile_loads(int waves) { return kPfKeys / waves / 4; }
template <bool kV>
__device__ __forceinline__ int tile_swizzle(int r) {
  return kV ? 2 * (r & 7) : r & 15;
}
template <int kWaves>
struct TileOffsets {
  int k[tile_loads(kWaves)], v[tile_loads(kWaves)];
};
template <int kWaves>
__device__ __forceinline__ TileOffsets<kWaves> tile_offsets(const PrefillParams& p) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  TileOffsets<kWaves> o;
#pragma unroll
  for (int i = 0; i < tile_loads(kWaves); ++i) {
    const int r = 4 * (tile_loads(kWaves) * w + i) + (lane >> 4), at = r * (p.kvh * kPfDim * 2);
    o.k[i] = at + 16 * ((lane & 15) ^ tile_swizzle<false>(r));
    o.v[i] = at + 16 * ((lane & 15) ^ tile_swizzle<true>(r));
  }
  return o;
}
// 16 bytes per lane into LDS at ``st`` + 16 lane
__device__ __forceinline__ void transfer16(pf_rsrc_t rs, uint8_t* st, int off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (pf_lds_ptr_t)st, 16, off, 0, 0, 0);
}
template <bool kV, int kWaves>
__device__ __forceinline__ void load_one(const PrefillParams& p, int64_t page, int key0, int nkeys, int h, uint8_t* st,
                                         const int* whole, bool live = true) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const pf_rsrc_t rs = tile_rsrc(kV ? p.wv : p.wk, page, key0, h, p.kvh, live);
  int off[tile_loads(kWaves)];
#pragma unroll
  for (int i = 0; i < tile_loads(kWaves); ++i) off[i] = whole[i];
  if (nkeys < kPfKeys) {
#pragma unroll
    for (int i = 0; i < tile_loads(kWaves); ++i) {
      const int r = 4 * (tile_loads(kWaves) * w + i) + (lane >> 4);
      off[i] = min(r, nkeys - 1) * (p.kvh * kPfDim * 2) + 16 * ((lane & 15) ^ tile_swizzle<kV>(r));
    }
  }
#pragma unroll
  for (int i = 0; i < tile_loads(kWaves); ++i)
    transfer16(rs, st + 4 * (tile_loads(kWaves) * w + i) * kKRow, off[i]);
}
template <int kWaves>
__device__ __forceinline__ void load_tile(const PrefillParams& p, int64_t page, int key0, int nkeys, int h,
                                          uint8_t* kst, uint8_t* vst, const TileOffsets<kWaves>& off) {
  load_one<false, kWaves>(p, page, key0, nkeys, h, kst, off.k);
  load_one<true, kWaves>(p, page, key0, nkeys, h, vst, off.v);
}

// Whether a column maximum moves the softmax reference m (-infinity: none yet).
__device__ __forceinline__ bool outgrows(float x, float m, float scale_log2) {
  return x > m && (m == -INFINITY || (x - m) * scale_log2 > kLazyMax);
}

typedef short pf_i16x4 __attribute__((ext_vector_type(4)));

// ds_read_b64_tr_b16 (gfx950): within each 16-lane group, lane i receives
// element i % 4 of the 8-byte pieces addressed by lanes 4 e + i / 4,
// e = 0..3 -- a 4 x 4 transpose of 16-bit elements across lanes.
__device__ __forceinline__ uint2 lds_tr16(const uint8_t* a) {
  const pf_i16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) pf_i16x4*)a);
  return __builtin_bit_cast(uint2, v);
}

// ---------------------------------------------------------------------------
// Split launches, for grids with fewer (query tile, KV head) pairs than CUs: a
// short last chunk of a long prompt, one prompt.  One workgroup per CU; the
// key tiles of all pairs, flattened in (head, sequence, query tile, key tile)
// order, are cut into equal contiguous ranges, so a workgroup may run parts of
// query tiles.  Parts leave O, m and l in fp32 (slot 2 r: a part that
// continues a query tile, 2 r + 1: one that starts it) and
// prefill_merge_kernel merges them.  The ranges of an XCD's workgroups
// (blockIdx % 8) are neighbours and share keys in its L2.
//
// A part starts from the softmax reference that the unsplit kernel would have
// reached at its first key tile, so P rounds to the same BF16 values however
// the work is cut, and only the fp32 sums' order differs.  The reference
// moves only at key tiles where some column outgrows it by 2^kLazyMax; it
// never falls, so such a tile's maximum outgrows a lower bound of it too.
// prefill_max_kernel scores every range (Q K^T only) and keeps the column
// maxima of the tiles that do (few); a part replays them.
constexpr int kPfMinSteps = 4;  // key tiles of a range, at least
constexpr int kPfPartFloats = kPfRows * kPfDim;

// Key tiles of query tile ``i``: exact for causal (bottom-right) and full
// attention; at least one, so that every query tile has an owner.
__device__ __forceinline__ int tile_steps(int i, int qlen, int klen, int T, int causal) {
  const int kend = causal ? min((i + 1) * T, qlen) + max(klen - qlen, 0) : klen;
  return max((kend + kPfKeys - 1) / kPfKeys, 1);
}

// Key tiles of a sequence's first ``nt`` query tiles, in closed form (T is 32,
// 64, 128 or 256): tiles before the last end at key (i + 1) T + shift, i.e.
// after ceil(shift / 64) + (i + 1) T / 64 key tiles, where for T = 32 the even
// tiles' half adds to the shift.
__device__ __forceinline__ int seq_steps(int nt, int qlen, int klen, int T, int causal) {
  if (nt <= 0) return 0;
  const int last = tile_steps(nt - 1, qlen, klen, T, causal);
  const int n = nt - 1;  // tiles before the last
  if (!causal) return nt * last;
  const int shift = max(klen - qlen, 0);
  if (T >= kPfKeys) return n * ((shift + kPfKeys - 1) / kPfKeys) + (T / kPfKeys) * (n * (n + 1) / 2) + last;
  const int odd = n >> 1, even = n - odd;  // tiles 1, 3, .. and 0, 2, ..
  return odd * (1 + (shift + kPfKeys - 1) / kPfKeys) + odd * (odd - 1) / 2 +
         even * ((shift + T + kPfKeys - 1) / kPfKeys) + even * (even - 1) / 2 + last;
}

// A place in the flattened order: key tile ``off`` of query tile ``tile`` of
// (head h, sequence b).
struct PfPlace {
  int h, b, tile, off, steps;  // steps: key tiles of the query tile
  int flat;                    // the place's flattened index
};

struct PfPlan {
  int per_head, per;  // key tiles of a head; of a range
};

__device__ __forceinline__ int seq_tiles(const PrefillParams& p, int qlen, int T) {
  return min((qlen + T - 1) / T, p.tiles_per_seq);
}

// Key tiles of sequence ``b`` (0 past the last one).
__device__ __forceinline__ int lane_seq_steps(const PrefillParams& p, int b, int T) {
  if (b >= p.num_seqs) return 0;
  const int qlen = p.cu_q[b + 1] - p.cu_q[b];
  return seq_steps(seq_tiles(p, qlen, T), qlen, p.seq_k[b], T, p.causal);
}

// The whole wave: lanes take sequences.
__device__ __forceinline__ PfPlan split_plan(const PrefillParams& p, int wgs, int T, int lane) {
  PfPlan r;
  r.per_head = 0;
  for (int b0 = 0; b0 < p.num_seqs; b0 += 64) r.per_head += wave_total<false>(lane_seq_steps(p, b0 + lane, T));
  r.per = max((r.per_head * p.kvh + wgs - 1) / wgs, kPfMinSteps);
  return r;
}

// The place of flattened key tile ``s`` (inside the plan): the sequence by a
// scan over the sequences' totals, the query tile by one over its tiles.
__device__ __forceinline__ PfPlace split_place(const PrefillParams& p, const PfPlan& plan, int s, int T, int lane) {
  PfPlace r;
  r.flat = s;
  r.h = s / plan.per_head;
  int rem = s - r.h * plan.per_head;
  r.b = 0;
  for (int b0 = 0; b0 < p.num_seqs; b0 += 64) {
    const int incl = wave_incl_scan(lane_seq_steps(p, b0 + lane, T));
    const uint64_t past = __ballot(incl > rem);
    if (past) {
      const int l = __builtin_ctzll(past);
      r.b = b0 + l;
      rem -= l ? __builtin_amdgcn_readlane(incl, l - 1) : 0;
      break;
    }
    rem -= __builtin_amdgcn_readlane(incl, 63);
  }
  const int qlen = uniform(p.cu_q[r.b + 1] - p.cu_q[r.b]), klen = uniform(p.seq_k[r.b]);
  for (int i0 = 0;; i0 += 64) {
    const int n = tile_steps(i0 + lane, qlen, klen, T, p.causal), incl = wave_incl_scan(n);
    const uint64_t past = __ballot(incl > rem);
    if (past) {
      const int l = __builtin_ctzll(past);
      r.tile = i0 + l;
      r.steps = __builtin_amdgcn_readlane(n, l);
      r.off = rem - (__builtin_amdgcn_readlane(incl, l) - r.steps);
      return r;
    }
    rem -= __builtin_amdgcn_readlane(incl, 63);
  }
}

__device__ __forceinline__ bool split_next(const PrefillParams& p, PfPlace& at, int T) {
  // the query tile after ``at`` (false past the last)
  at.flat += at.steps - at.off;
  at.off = 0;
  ++at.tile;
  for (;;) {
    const int qlen = uniform(p.cu_q[at.b + 1] - p.cu_q[at.b]);
    if (at.tile < seq_tiles(p, qlen, T)) {
      at.steps = tile_steps(at.tile, qlen, uniform(p.seq_k[at.b]), T, p.causal);
      return true;
    }
    at.tile = 0;
    if (++at.b == p.num_seqs) {
      at.b = 0;
      if (++at.h == p.kvh) return false;
    }
  }
}

// A range as the launch's first kernel leaves it for the others: its first
// place (h -1: none), its key tiles and the plan's range size.
struct PfRange {
  PfPlace at;
  int left, per;
};
__device__ __forceinline__ void put_range(const PrefillParams& p, int rank, const PfRange& r) {
  p.ranges[2 * rank] = make_int4(r.at.h, r.at.b, r.at.tile, r.at.off);
  p.ranges[2 * rank + 1] = make_int4(r.at.steps, r.at.flat, r.left, r.per);
}
__device__ __forceinline__ PfRange get_range(const PrefillParams& p, int rank) {
  const int4 a = p.ranges[2 * rank], b = p.ranges[2 * rank + 1];
  return PfRange{{uniform(a.x), uniform(a.y), uniform(a.z), uniform(a.w), uniform(b.x), uniform(b.y)},
                 uniform(b.z), uniform(b.w)};
}

// Range r of the plan belongs to workgroup (r % per_xcd) * 8 + r / per_xcd.
__device__ __forceinline__ int split_rank() {
  return (int)(blockIdx.x % kPfXcds) * (int)(gridDim.x / kPfXcds) + (int)(blockIdx.x / kPfXcds);
}

template <int kWaves, bool kSplit>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(kPfWavesPerEu))) prefill_kernel(PrefillParams p) {
  // K stages are two separate LDS objects and each trip of the tile loop
  // below names them statically: the counter pass then sees that the next
  // tile's K transfer into one cannot alias this tile's reads of the other
  // (one LDS object with computed stage offsets makes every K read wait for
  // the transfer just issued).  The V stages likewise: reads of the dynamic
  // LDS block are not known to miss the K objects.
  __shared__ __align__(16) uint8_t pf_k0[kKBytes];
  __shared__ __align__(16) uint8_t pf_k1[kKBytes];
  __shared__ __align__(16) uint8_t pf_v0[kKBytes];
  __shared__ __align__(16) uint8_t pf_v1[kKBytes];
  const int T = kPfRows / p.group;  // query tokens per tile
  PfPlace at{0, 0, 0, 0, 0, 0};
  int left = 0, rank = 0;  // key tiles left of the range
  int row0 = 0;            // the workgroup's first row of the query tile
  if constexpr (kSplit) {
    rank = split_rank();
    const PfRange r = get_range(p, rank);
    if (r.at.h < 0) return;
    at = r.at;
    left = r.left;
  } else {
    // Workgroups go to the XCDs in turn.  XCD x takes the heads = x mod
    // head_sets (equal work each), and with fewer heads than XCDs every
    // (8 / head_sets)-th of their query tiles; a sequence's tiles follow each
    // other, longest first (later tiles see more keys under the causal mask).
    // Tiles of one sequence thus spread over all XCDs and CUs: with the
    // sequence as the fastest index a long one among short ones ran on a
    // quarter of the device (prompts of 1000, 37, 2311 and 512 tokens at H 8,
    // G 4: 218 us, 81 in this order, 74 with 4-wave workgroups).
    const int sets = abs(p.head_sets), xcd = (int)blockIdx.x % kPfXcds, share = kPfXcds / sets;
    const int item = (int)blockIdx.x / kPfXcds * share + xcd / sets;
    at.h = xcd % sets + sets * (int)blockIdx.y;
    constexpr int kShares = kPfWaves / kWaves;  // workgroups per query tile
    const int t = item / kShares;
    row0 = item % kShares * (kWaves * kPfWaveRows);
    // Where XCDs share a head, that order gives each XCD every share-th tile,
    // the first ones the longest of every group: sequences of equal length take
    // turns instead (head_sets < 0), which spreads each tile index over the XCDs
    // (prefill_launch has the rule).
    const bool turns = p.head_sets < 0;
    const int width = turns ? p.num_seqs : p.tiles_per_seq, q = t / width, m = t - q * width;
    at.b = turns ? m : q;
    at.tile = p.tiles_per_seq - 1 - (turns ? q : m);
    if (at.b >= p.num_seqs || at.tile < 0) return;
  }
  for (;;) {
  const int h = at.h, b = at.b, qtile = at.tile;
  const int q0 = p.cu_q[b], qlen = p.cu_q[b + 1] - q0;
  const int t0 = qtile * T;
  // (with one query head per KV head a share of a tile is a range of its tokens, else one of its heads)
  const int tok0 = t0 + (p.group == 1 ? row0 : 0), tok1 = p.group == 1 ? tok0 + kWaves * kPfWaveRows : t0 + T;
  if (!kSplit && tok0 >= qlen) return;
  const int klen = p.seq_k[b];
  const int shift = klen - qlen;  // query i sees keys <= i + shift (causal)
  const int32_t* bt = p.block_table + (int64_t)b * p.bt_stride;
  const int seg = kSplit ? min(left, at.steps - at.off) : 0;  // key tiles of this part

  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int j = lane & 15, q4 = lane >> 4;
  // this lane's query columns (tiles qt): row -> (head g, token t)
  int tok[kPfQt], hq[kPfQt];
  bool rvalid[kPfQt];
#pragma unroll
  for (int qt = 0; qt < kPfQt; ++qt) {
    const int row = row0 + 16 * kPfQt * w + 16 * qt + j;
    const int g = row / T, t = row - g * T;
    tok[qt] = t0 + t;
    hq[qt] = h * p.group + g;
    rvalid[qt] = tok[qt] < qlen;
  }
  // Q^T fragments (B operands): lane (j, q4) holds dims 32 ks + 8 q4 .. + 7
  uint4 qf[kPfQt][4];
#pragma unroll
  for (int qt = 0; qt < kPfQt; ++qt) {
    const uint16_t* qrow = p.q + (int64_t)(q0 + (rvalid[qt] ? tok[qt] : 0)) * p.q_stride + (int64_t)hq[qt] * kPfDim;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      qf[qt][ks] = rvalid[qt] ? *reinterpret_cast<const uint4*>(qrow + 32 * ks + 8 * q4) : make_uint4(0u, 0u, 0u, 0u);
  }
  // keys this tile needs: up to the last valid query's causal limit
  const int last_tok = min(tok1, qlen) - 1;
  const int kend = p.causal ? min(klen, last_tok + shift + 1) : klen;
  const int all_tiles = (kend + kPfKeys - 1) / kPfKeys;
  const int it0 = kSplit ? min(at.off, all_tiles) : 0;
  const int ntiles = kSplit ? min(at.off + seg, all_tiles) : all_tiles;  // key tiles [it0, ntiles)
  // causal limit per query column
  int kmax[kPfQt];
#pragma unroll
  for (int qt = 0; qt < kPfQt; ++qt) kmax[qt] = p.causal ? min(klen, tok[qt] + shift + 1) : klen;

  float m[kPfQt], l[kPfQt];
#pragma unroll
  for (int qt = 0; qt < kPfQt; ++qt) {
    m[qt] = -INFINITY;
    l[qt] = 0.f;
  }
  pf_f32x4 o[8][kPfQt];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
#pragma unroll
    for (int qt = 0; qt < kPfQt; ++qt) o[dt][qt] = pf_f32x4{0.f, 0.f, 0.f, 0.f};

  // page ids of the tiles: lane j holds block_table entry 64 pb + j
  int pages = 0, pbase = -1;
  auto page_of = [&](int key0) -> int64_t {
    const int pi = key0 >> 7;
    if ((pi & ~63) != pbase) {
      pbase = pi & ~63;
      pages = pbase + lane < (kend + 127) / 128 ? bt[pbase + lane] : 0;
      // waited for here: where the paths join, the wait would also be for the
      // transfers in flight
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    }
    return __builtin_amdgcn_readlane(pages, pi & 63);
  };
  const TileOffsets<kWaves> offs = tile_offsets<kWaves>(p);
  if (it0 < ntiles)
    load_tile(p, page_of(it0 * kPfKeys), it0 * kPfKeys, min(kPfKeys, kend - it0 * kPfKeys), h, pf_k0, pf_v0, offs);
  if (kSplit && at.off > 0) {
    // the reference at the part's first key tile: the flagged tiles before it
    const int64_t first = (int64_t)at.flat - at.off;
    for (int c0 = 0; c0 < it0; c0 += 64) {
      const bool f = c0 + lane < it0 && first + c0 + lane < p.tile_cap && p.tile_flag[(first + c0 + lane) * kPfWaves + w] != 0;
      // (a batch's loads go out together; past the last flagged tile it repeats that one, which moves nothing)
      constexpr int kBatch = 8;
      uint64_t fl = __ballot(f);
      while (fl) {
        const int cnt = __builtin_popcountll(fl);
        float mt[kBatch][kPfQt];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
          const float* tm = p.tile_max + ((first + c0 + __builtin_ctzll(fl)) * kPfWaves + w) * (16 * kPfQt) + j;
#pragma unroll
          for (int qt = 0; qt < kPfQt; ++qt) mt[k][qt] = tm[16 * qt];
          if (k + 1 < min(cnt, kBatch)) fl &= fl - 1;
        }
        fl &= fl - 1;
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
          bool grow = false;
#pragma unroll
          for (int qt = 0; qt < kPfQt; ++qt) grow |= outgrows(mt[k][qt], m[qt], p.scale_log2);
          if (__ballot(grow) != 0) {
#pragma unroll
            for (int qt = 0; qt < kPfQt; ++qt) m[qt] = fmaxf(m[qt], mt[k][qt]);
          }
        }
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();
  // Nothing in flight at the loop entry (Q and the first tile have landed):
  // without this explicit wait the counter pass, merging the entry path,
  // puts a vmcnt(0) before the first MFMA of every tile, i.e. waits for the
  // next tile's loads right after issuing them.
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  // V fragment lanes: row x = 4 q4 + j / 4 of each 16-row block, byte
  // 8 (j & 1) of the chunk; the chunk's slot term 16 ((j >> 1 & 1) ^ 2 (x % 8))
  const int vx = 4 * q4 + (j >> 2);
  const int vlane = vx * kKRow + 8 * (j & 1), vsw = 16 * (((j >> 1) & 1) ^ tile_swizzle<true>(vx));
  auto tile = [&](int it, const uint8_t* stage, uint8_t* knext, const uint8_t* vstage, uint8_t* vnext)
                  __attribute__((always_inline)) {
    const int key0 = it * kPfKeys;
    const bool more = it + 1 < ntiles;
    if (more)
      load_tile(p, page_of(key0 + kPfKeys), key0 + kPfKeys, min(kPfKeys, kend - key0 - kPfKeys), h, knext, vnext, offs);

    // ---- S^T = K Q^T: s[kt][qt], keys key0 + 16 kt + 4 q4 + r ----
    // The tile runs in halves so that one half's exponentials overlap the
    // other half's MFMAs within the wave: keys 0..31 are scored, then keys
    // 32..63 are scored while P of keys 0..31 is formed (speculatively,
    // against the running max); P of keys 32..63 is formed while the PV
    // product of keys 0..31 runs.
    //
    // Scores stay unscaled (scale > 0 keeps the order); P = exp2(s c - m c)
    // is one FMA and one exp per score.  The reference max m only moves when
    // some column's max outgrows it by more than 2^kLazyMax (log2 domain), so
    // O and l are rescaled on few tiles -- and only then is the speculative P
    // of keys 0..31 recomputed; P <= 2^kLazyMax is exact enough in BF16 and
    // fp32.
    pf_f32x4 s[4][kPfQt];
    auto qk = [&](int kt) {
#pragma unroll
      for (int qt = 0; qt < kPfQt; ++qt) s[kt][qt] = pf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const uint4 kf = *reinterpret_cast<const uint4*>(stage + (16 * kt + j) * kKRow + 16 * ((4 * ks + q4) ^ j));
#pragma unroll
        for (int qt = 0; qt < kPfQt; ++qt) s[kt][qt] = pf_mfma(kf, qf[qt][ks], s[kt][qt]);
      }
    };
    // causal / length mask: only on tiles that reach some column's limit
    // (a wave-uniform branch; other tiles skip the compares)
    int kmin = kmax[0];
#pragma unroll
    for (int qt = 1; qt < kPfQt; ++qt) kmin = min(kmin, kmax[qt]);
    const bool mask_tile = __ballot(key0 + kPfKeys > kmin) != 0;
    auto mask = [&](int kt) {
#pragma unroll
      for (int qt = 0; qt < kPfQt; ++qt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (key0 + 16 * kt + 4 * q4 + r >= kmax[qt]) s[kt][qt][r] = -INFINITY;
    };
    float e[4][kPfQt][4];
    auto expo = [&](int kt, int qt, float nm) {
#pragma unroll
      for (int r = 0; r < 4; ++r) e[kt][qt][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][qt][r], p.scale_log2, nm));
    };
    auto neg_m = [&](int qt) { return m[qt] == -INFINITY ? 0.f : -m[qt] * p.scale_log2; };
    qk(0);
    qk(1);
    if (mask_tile) {
      mask(0);
      mask(1);
    }
    // keys 32..63 scored in four k-steps; after each, a quarter of the
    // exponentials of keys 0..31 (pinned there: they run while the step's
    // MFMAs execute)
    {
      float nm[kPfQt];
#pragma unroll
      for (int qt = 0; qt < kPfQt; ++qt) {
        nm[qt] = neg_m(qt);
        s[2][qt] = s[3][qt] = pf_f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const uint4 k2 = *reinterpret_cast<const uint4*>(stage + (32 + j) * kKRow + 16 * ((4 * ks + q4) ^ j));
        const uint4 k3 = *reinterpret_cast<const uint4*>(stage + (48 + j) * kKRow + 16 * ((4 * ks + q4) ^ j));
#pragma unroll
        for (int qt = 0; qt < kPfQt; ++qt) {
          s[2][qt] = pf_mfma(k2, qf[qt][ks], s[2][qt]);
          s[3][qt] = pf_mfma(k3, qf[qt][ks], s[3][qt]);
        }
        // (kt, qt) pairs ks * kPerStep .. of keys 0..31 (2 kPfQt pairs over
        // the four k-steps): kt = pair / kPfQt
        constexpr int kPerStep = (2 * kPfQt + 3) / 4;
#pragma unroll
        for (int u = 0; u < kPerStep; ++u) {
          const int pr = ks * kPerStep + u, kt = pr / kPfQt, qt = pr % kPfQt;
          if (pr >= 2 * kPfQt) continue;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            e[kt][qt][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][qt][r], p.scale_log2, nm[qt]));
#pragma unroll
          for (int r = 0; r < 4; ++r) asm volatile("" ::"v"(e[kt][qt][r]));  // not sunk into a later block
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (mask_tile) {
      mask(2);
      mask(3);
    }
    float mloc[kPfQt];
#pragma unroll
    for (int qt = 0; qt < kPfQt; ++qt) {
      float mx = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[kt][qt][r]);
      mx = pf_xor32_max(pf_xor16_max(mx));
      mloc[qt] = mx;
    }
    bool grow = false;
#pragma unroll
    for (int qt = 0; qt < kPfQt; ++qt)
      grow |= outgrows(mloc[qt], m[qt], p.scale_log2);
    if (__ballot(grow) != 0) {
#pragma unroll
      for (int qt = 0; qt < kPfQt; ++qt) {
        const float m_new = fmaxf(m[qt], mloc[qt]);
        const float alpha = m[qt] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m[qt] - m_new) * p.scale_log2);
        m[qt] = m_new;
        l[qt] *= alpha;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) o[dt][qt] *= alpha;
        const float nm = neg_m(qt);
        expo(0, qt, nm);
        expo(1, qt, nm);
      }
    }
    // B operand of k-step kk: keys 32 kk + {4 q4 .. 4 q4 + 3} (tile 2 kk) and
    // 32 kk + 16 + {4 q4 ..} (tile 2 kk + 1)
    auto pfrag = [&](int kk, int qt) {
      return make_uint4(pk_bf16(e[2 * kk][qt][0], e[2 * kk][qt][1]), pk_bf16(e[2 * kk][qt][2], e[2 * kk][qt][3]),
                        pk_bf16(e[2 * kk + 1][qt][0], e[2 * kk + 1][qt][1]),
                        pk_bf16(e[2 * kk + 1][qt][2], e[2 * kk + 1][qt][3]));
    };
    uint4 p0[kPfQt];
#pragma unroll
    for (int qt = 0; qt < kPfQt; ++qt) p0[qt] = pfrag(0, qt);
#pragma unroll
    for (int qt = 0; qt < kPfQt; ++qt) {
      const float nm = neg_m(qt);
      expo(2, qt, nm);
      expo(3, qt, nm);
    }
    // ---- O^T += V^T P^T: o[dt][qt], dims 16 dt + 4 q4 + r ----
    // V^T fragment (dims 16 dt + j, keys 32 kk + {4 q4 .. 4 q4 + 3} and
    // 32 kk + 16 + {4 q4 ..}) by two transposing reads: lane (s = j, g = q4)
    // addresses row 32 kk (+ 16) + 4 g + s / 4, dims 16 dt + 4 (s % 4) ..,
    // so lane j receives dim 16 dt + j of rows 32 kk (+ 16) + 4 g + e.
    auto pv = [&](int kk, const uint4 (&pa)[kPfQt]) {
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        // chunk 2 dt + (j >> 1 & 1) of row x = 4 q4 + j / 4 (mod 16) sits at
        // slot chunk ^ 2 (x % 8)
        const uint8_t* base = vstage + (vsw ^ (32 * dt)) + vlane;
        const uint2 lo = lds_tr16(base + 32 * kk * kKRow);
        const uint2 hi = lds_tr16(base + (32 * kk + 16) * kKRow);
        const uint4 vf = make_uint4(lo.x, lo.y, hi.x, hi.y);
#pragma unroll
        for (int qt = 0; qt < kPfQt; ++qt) o[dt][qt] = pf_mfma(vf, pa[qt], o[dt][qt]);
      }
    };
    pv(0, p0);
    {
      uint4 p1[kPfQt];
#pragma unroll
      for (int qt = 0; qt < kPfQt; ++qt) p1[qt] = pfrag(1, qt);
      pv(1, p1);
    }
#pragma unroll
    for (int qt = 0; qt < kPfQt; ++qt) {
      float psum = 0.f;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) psum += e[kt][qt][r];
      l[qt] += psum;
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the next tile has landed
    __syncthreads();
  };
  for (int it = it0; it < ntiles; it += 2) {
    tile(it, pf_k0, pf_k1, pf_v0, pf_v1);
    if (it + 1 < ntiles) tile(it + 1, pf_k1, pf_k0, pf_v1, pf_v0);
  }
  const bool part = kSplit && seg < at.steps;
  const int64_t slot = 2 * rank + (at.off == 0);
  // ---- normalise and store: lane holds dims 16 dt + 4 q4 + r of query j ----
#pragma unroll
  for (int qt = 0; qt < kPfQt; ++qt) {
    float lt = l[qt];
    lt = pf_xor32_sum(pf_xor16_sum(lt));
    if (part) {
      // [wave][dt][qt][lane] x 16 bytes, and (m, l) by row
      float4* po = reinterpret_cast<float4*>(p.opart + slot * kPfPartFloats) + (w * 8 * kPfQt + qt) * 64 + lane;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt)
        po[dt * kPfQt * 64] = make_float4(o[dt][qt][0], o[dt][qt][1], o[dt][qt][2], o[dt][qt][3]);
      if (q4 == 0)
        reinterpret_cast<float2*>(p.ml)[slot * kPfRows + 16 * (kPfQt * w + qt) + j] = make_float2(m[qt], lt);
      continue;
    }
    if (!rvalid[qt]) continue;
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    uint16_t* orow = p.out + (int64_t)(q0 + tok[qt]) * p.out_stride + (int64_t)hq[qt] * kPfDim;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
      *reinterpret_cast<uint2*>(orow + 16 * dt + 4 * q4) =
          make_uint2(pk_bf16(o[dt][qt][0] * inv, o[dt][qt][1] * inv), pk_bf16(o[dt][qt][2] * inv, o[dt][qt][3] * inv));
  }
  if (!kSplit) return;
  left -= seg;
  if (left <= 0 || !split_next(p, at, T)) return;
  }
}

// Column maxima for the parts' references (see above): every range but the
// parts that end their query tile, which none follows.  Grid as the split
// prefill's.  Bound by its steps' latency (K fragments from LDS, one barrier a
// key tile: ~1.1 us, 1.4 with every tile masked and its columns reduced).  200
// tokens over 8192 (H 4, G 8; 9 parts a tile) take 73-77 us in a timed loop; in
// a kernel trace, which adds to each launch, this kernel shows 25, the parts 54
// (14 of launch and first loads, ~7 of replays, 4 of stores, ~1.9 a key tile)
// and the merge 10.
__global__ void __launch_bounds__(64 * kPfWaves) __attribute__((amdgpu_waves_per_eu(kPfWavesPerEu))) prefill_max_kernel(PrefillParams p) {
  // four stages: a step is shorter than a memory round trip, so transfers run
  // three key tiles ahead
  __shared__ __align__(16) uint8_t k0[kKBytes];
  __shared__ __align__(16) uint8_t k1[kKBytes];
  __shared__ __align__(16) uint8_t k2[kKBytes];
  __shared__ __align__(16) uint8_t k3[kKBytes];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int j = lane & 15, q4 = lane >> 4;
  const int T = kPfRows / p.group;
  const PfPlan plan = split_plan(p, gridDim.x, T, lane);
  const int rank = split_rank(), s0 = rank * plan.per;
  int left = min(plan.per, plan.per_head * p.kvh - s0);
  PfPlace at{-1, 0, 0, 0, 0, 0};
  if (left > 0) at = split_place(p, plan, s0, T, lane);
  if (threadIdx.x == 0) put_range(p, rank, PfRange{at, left, plan.per});
  if (left <= 0) return;
  // only the range's last query tile can go on in another range
  if (at.steps - at.off <= left) {
    if (s0 + left >= plan.per_head * p.kvh) return;
    at = split_place(p, plan, s0 + left, T, lane);
    if (at.off == 0) return;
    left = at.off;
    at.flat -= at.off;
    at.off = 0;
  }
  const int h = at.h, b = at.b;
  const int q0 = p.cu_q[b], qlen = p.cu_q[b + 1] - q0, klen = p.seq_k[b], shift = klen - qlen, t0 = at.tile * T;
  const int32_t* bt = p.block_table + (int64_t)b * p.bt_stride;
  const int kend = p.causal ? min(klen, min(t0 + T, qlen) + shift) : klen;
  const int all_tiles = (kend + kPfKeys - 1) / kPfKeys;
  const int it0 = min(at.off, all_tiles), it1 = min(at.off + left, all_tiles);
  if (it0 >= it1) return;
  uint4 qf[kPfQt][4];
  int kmax[kPfQt];
#pragma unroll
  for (int qt = 0; qt < kPfQt; ++qt) {
    const int row = 16 * (kPfQt * w + qt) + j, g = row / T, tok = t0 + row - g * T;
    const uint16_t* qrow = p.q + (int64_t)(q0 + (tok < qlen ? tok : 0)) * p.q_stride + (int64_t)(h * p.group + g) * kPfDim;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      qf[qt][ks] = tok < qlen ? *reinterpret_cast<const uint4*>(qrow + 32 * ks + 8 * q4) : make_uint4(0u, 0u, 0u, 0u);
    kmax[qt] = p.causal ? min(klen, tok + shift + 1) : klen;
  }
  const TileOffsets<kPfWaves> offs = tile_offsets<kPfWaves>(p);
  // A lower bound of each column's reference: key tile 0's maximum, and the
  // later maxima less the headroom (a reference that much below would have
  // moved).  Only a tile that outgrows it can move the reference.  (The
  // headroom a little too wide: rounding must not lift the bound.)
  const float lazy = kLazyMax / p.scale_log2 * 1.0001f;
  float low[kPfQt];
#pragma unroll
  for (int qt = 0; qt < kPfQt; ++qt) low[qt] = -INFINITY;
  int kmin = min(kmax[0], kmax[1]);  // wave-uniform: tiles ending past this key reach some column's limit
#pragma unroll
  for (int o = 32; o; o >>= 1) kmin = min(kmin, __shfl_xor(kmin, o, 64));
  kmin = uniform(kmin);
  // key tile 0 first (its maxima are the first reference), then the range's;
  // step i works on key tile tile_of(i)
  const int n = it1 - it0 + (it0 > 0);
  auto tile_of = [&](int i) { return it0 > 0 ? (i == 0 ? 0 : it0 + i - 1) : i; };
  int pages = 0, pbase = -1;
  auto load = [&](int i, uint8_t* st) __attribute__((always_inline)) {
    // past the last step the transfer moves nothing (so that every step issues the same)
    const int key0 = tile_of(min(i, n - 1)) * kPfKeys, pi = key0 >> 7;
    if ((pi & ~63) != pbase) {
      pbase = pi & ~63;
      pages = pbase + lane < (kend + 127) / 128 ? bt[pbase + lane] : 0;
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    }
    load_one<false, kPfWaves>(p, __builtin_amdgcn_readlane(pages, pi & 63), key0, min(kPfKeys, kend - key0), h, st, offs.k, i < n);
  };
  load(0, k0);
  load(1, k1);
  load(2, k2);
  // flags of 64 key tiles a time, key tile it0 + k in lane k % 64 (a store per
  // step would count among the transfers that the wait below leaves in flight)
  bool flag = false;
  auto put_flags = [&](int k0, int count) __attribute__((always_inline)) {
    const int64_t tile = (int64_t)at.flat + k0 + lane;
    if (lane < count && tile < p.tile_cap) p.tile_flag[tile * kPfWaves + w] = flag;
  };
  auto step = [&](int i, const uint8_t* st, uint8_t* next) __attribute__((always_inline)) {
    static_assert(2 * tile_loads(kPfWaves) == 4, "the wait below");
    __builtin_amdgcn_s_waitcnt(0x0F74);  // vmcnt(4): this step's keys have landed
    __syncthreads();                     // in every wave; and the last step's reads are done
    load(i + 3, next);
    const int it = tile_of(i), key0 = it * kPfKeys;
    pf_f32x4 sc[4][kPfQt];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
      for (int qt = 0; qt < kPfQt; ++qt) sc[kt][qt] = pf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const uint4 kf = *reinterpret_cast<const uint4*>(st + (16 * kt + j) * kKRow + 16 * ((4 * ks + q4) ^ tile_swizzle<false>(j)));
#pragma unroll
        for (int qt = 0; qt < kPfQt; ++qt) sc[kt][qt] = pf_mfma(kf, qf[qt][ks], sc[kt][qt]);
      }
    }
    if (key0 + kPfKeys > kmin) {
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int qt = 0; qt < kPfQt; ++qt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (key0 + 16 * kt + 4 * q4 + r >= kmax[qt]) sc[kt][qt][r] = -INFINITY;
    }
    // the lane's own maxima decide; the columns' are formed where they are kept
    float mx[kPfQt];
    bool grow = false;
#pragma unroll
    for (int qt = 0; qt < kPfQt; ++qt) {
      mx[qt] = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx[qt] = fmaxf(mx[qt], sc[kt][qt][r]);
      grow |= outgrows(mx[qt], low[qt], p.scale_log2);
    }
    const bool keep = __ballot(grow) != 0;
    if (keep) {
#pragma unroll
      for (int qt = 0; qt < kPfQt; ++qt) {
        mx[qt] = pf_xor32_max(pf_xor16_max(mx[qt]));
        low[qt] = fmaxf(low[qt], i == 0 ? mx[qt] : mx[qt] - lazy);
      }
    }
    if (it < it0) return;
    const int k = it - it0;
    if (lane == (k & 63)) flag = keep;
    if ((k & 63) == 63 || i == n - 1) put_flags(k & ~63, (k & 63) + 1);
    const int64_t at_tile = ((int64_t)at.flat + k) * kPfWaves + w;
    if (keep && q4 == 0 && at_tile < p.tile_cap * kPfWaves) {
#pragma unroll
      for (int qt = 0; qt < kPfQt; ++qt) p.tile_max[at_tile * (16 * kPfQt) + 16 * qt + j] = mx[qt];
    }
  };
  for (int i = 0; i < n; i += 4) {
    step(i, k0, k3);
    if (i + 1 < n) step(i + 1, k1, k0);
    if (i + 2 < n) step(i + 2, k2, k1);
    if (i + 3 < n) step(i + 3, k3, k2);
  }
}

// Merges the parts of the query tiles that a split launch cut: grid (ranges -
// 1, 16-row column tiles).  Workgroup (x, y) looks at the start of range r =
// x + 1; if that is the first cut of a query tile, it merges the tile's rows
// 16 y .. 16 y + 15 over its parts (range r - 1's, which starts the tile, and those of ranges
// r, r + 1, .. that continue it), in that order.
constexpr int kPfMergeThreads = 256;
__global__ void __launch_bounds__(kPfMergeThreads) prefill_merge_kernel(PrefillParams p) {
  const int lane = threadIdx.x & 63, sub = threadIdx.x >> 6;
  const int T = kPfRows / p.group, w = (int)blockIdx.y / kPfQt, qt = (int)blockIdx.y % kPfQt;
  const int r = (int)blockIdx.x + 1;
  const PfRange range = get_range(p, r);
  const PfPlace& at = range.at;
  if (at.h < 0 || at.off == 0 || at.off > range.per) return;  // not cut here, or cut before
  const int parts = 1 + (at.steps - at.off + range.per - 1) / range.per;
  const int q0 = p.cu_q[at.b], qlen = p.cu_q[at.b + 1] - q0;
  const int j = lane & 15, q4 = lane >> 4;
  auto slot = [&](int k) -> int64_t { return k == 0 ? 2 * (r - 1) + 1 : 2 * (r + k - 1); };
  const int row = 16 * (kPfQt * w + qt) + j;
  const int g = row / T, tok = at.tile * T + (row - g * T);
  const bool valid = tok < qlen;
  if (__ballot(valid) == 0) return;
  const float2* ml = reinterpret_cast<const float2*>(p.ml) + row;
  float gm = -INFINITY;
#pragma unroll 4
  for (int k = 0; k < parts; ++k) gm = fmaxf(gm, ml[slot(k) * kPfRows].x);
  const float m_use = gm == -INFINITY ? 0.f : gm;
  constexpr int kPer = 8 / (kPfMergeThreads / 64);  // dim tiles of a wave
  float l = 0.f;
  float4 acc[kPer];
#pragma unroll
  for (int d = 0; d < kPer; ++d) acc[d] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 8
  for (int k = 0; k < parts; ++k) {
    const float2 x = ml[slot(k) * kPfRows];
    const float4* po = reinterpret_cast<const float4*>(p.opart + slot(k) * kPfPartFloats) + (w * 8 * kPfQt + qt) * 64 + lane;
    const float wt = __builtin_amdgcn_exp2f((x.x - m_use) * p.scale_log2);
    l += wt * x.y;
#pragma unroll
    for (int d = 0; d < kPer; ++d) {
      const float4 v = po[(kPer * sub + d) * kPfQt * 64];
      acc[d].x += wt * v.x;
      acc[d].y += wt * v.y;
      acc[d].z += wt * v.z;
      acc[d].w += wt * v.w;
    }
  }
  if (!valid) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  uint16_t* orow = p.out + (int64_t)(q0 + tok) * p.out_stride + (int64_t)(at.h * p.group + g) * kPfDim;
#pragma unroll
  for (int d = 0; d < kPer; ++d)
    *reinterpret_cast<uint2*>(orow + 16 * (kPer * sub + d) + 4 * q4) =
        make_uint2(pk_bf16(acc[d].x * inv, acc[d].y * inv), pk_bf16(acc[d].z * inv, acc[d].w * inv));
}

}  // namespace
}  // namespace fp

using namespace fp;

namespace {

// The launch of a call, from the host's sizes (the lengths are on the device:
// upper bounds).  Measured on MI355X, H 8 and G 4 if not said otherwise:
// - 8-wave workgroups, one per 256-row query tile and KV head, each of whose
//   key tiles takes ~1.7 us;
// - 4-wave workgroups, two per query tile (its rows by halves, ~1.3 us a key
//   tile when a CU has one), while the 8-wave ones would leave CUs idle (1024
//   new tokens over 2048: 76 instead of 95 us; but from half the CUs on not for
//   sequences of one or two query tiles over several rows of heads, whose K / V
//   few other tiles share: 8 x 128 over 1000 at H 20, G 1 take 43.6 us with 4
//   waves, 39 with 8, 32 x 64 over 500 at H 5 29.6 and 27.0), and for fresh
//   prompts of up to four query tiles per CU, whose tiles differ in length
//   under the causal mask (2311 tokens 68 us instead of 81, 4 x 1000 59 instead
//   of 69, 2048 x 2 89 instead of 93; with full attention they do not, and 4
//   waves help only past a round: 2 x 2048 at H 16, G 1, 256 tiles, take 71 us
//   with 4 waves and 68 with 8, at H 5, G 4, 320 tiles, 107 and 127).  On
//   full grids of equal tiles they lose, each K / V tile serving half the rows
//   (4 x 1024 over 8192: 598 us, 8 waves 583; 4 x 8192: 2%);
// - the split launch: ~45 us of its own (three kernels, the parts written and
//   read) plus ~2.3 us per key tile of a CU's share, where that beats the
//   longest query tile by 10%: 200 new tokens over 8192 at H 4, G 8 take 76 us
//   instead of 175 (4 waves) or 226 (8).
constexpr int64_t kPfSplitMost = 1 << 16;  // key tiles (1 KB of workspace each)
// The rule in units of 0.1 us, kPfSplitMargin tenths: its own time, per key tile
// of a CU's share, and of the launch that does not split: its own, per key tile.
constexpr int64_t kPfSplitBase = 450, kPfSplitStep = 23, kPfWholeBase = 100, kPfWholeStep = 13, kPfSplitMargin = 9;
// The fewest key tiles of the longest query tile for which it can hold.
constexpr int64_t kPfSplitSteps =
    (10 * kPfSplitBase - kPfSplitMargin * kPfWholeBase) / (kPfSplitMargin * kPfWholeStep) + 1;

struct PfLaunch {
  int64_t tiles;  // query tiles of the longest sequence
  int64_t steps;  // key tiles of all query tiles
  int waves;      // per workgroup
  int split_wgs;  // 0: not split
  // the launch that does not split: heads of a grid row, rows, workgroups of a row
  int head_sets;
  int64_t rows, row_wgs;
  bool tile_major;  // a row's order: sequences take turns
};
// work items of a grid's x dimension (HIP's limit)
constexpr int64_t kPfGridMost = (1LL << 32) - 1;

// The largest of 8, 4, 2, 1 that divides the heads.
int head_sets(int64_t kv_heads) {
  int sets = kPfXcds;
  while (kv_heads % sets) sets /= 2;
  return sets;
}

PfLaunch prefill_launch(int64_t kv_heads, int64_t group, int64_t num_seqs, int64_t total_q, int64_t max_seqlen_q,
                        int64_t max_seqlen_k, bool causal, int64_t device) {
  const int64_t T = kPfRows / group;
  PfLaunch r;
  r.tiles = (max_seqlen_q + T - 1) / T;
  const int64_t cus = device / kPfXcds * kPfXcds, steps = (max_seqlen_k + kPfKeys - 1) / kPfKeys;
  const int64_t most = r.tiles * num_seqs;
  const int64_t all = (total_q > 0 ? std::min(most, total_q / T + num_seqs) : most) * kv_heads;
  r.steps = all * steps;
  const bool fresh = (causal || all > cus) && 2 * max_seqlen_k <= 3 * max_seqlen_q;
  const int sets = head_sets(kv_heads);
  r.waves = 2 * all <= cus || (4 * all <= 3 * cus && (r.tiles > 2 || kv_heads == sets)) || (fresh && all <= 4 * cus)
                ? 4
                : kPfWaves;
  const bool split = all <= cus && 10 * (kPfSplitBase * cus + kPfSplitStep * r.steps) <
                                      kPfSplitMargin * cus * (kPfWholeBase + kPfWholeStep * steps);
  r.split_wgs = total_q > 0 && split && r.steps <= kPfSplitMost ? (int)cus : 0;
  // The most head sets that divide the heads and that the grid's x dimension
  // holds: a row has the query tiles of head_sets heads.
  const int64_t items = most * (kPfWaves / r.waves);
  for (r.head_sets = sets;; r.head_sets /= 2) {
    const int64_t share = kPfXcds / r.head_sets;
    r.rows = kv_heads / r.head_sets;
    r.row_wgs = kPfXcds * ((items + share - 1) / share);
    if (r.head_sets == 1 || r.row_wgs * 64 * r.waves <= kPfGridMost) break;
  }
  // (with one head a row need not fill its last round over the XCDs)
  if (r.row_wgs * 64 * r.waves > kPfGridMost) r.row_wgs = items;
  // Sequences of equal query length take turns where XCDs share a head and CUs
  // get more than one workgroup of unequal tiles, or more than a round (4 x
  // 2048 at H 5, G 4: 114 us, 140 sequence by sequence; 4 x 8192 1306, 1512; 4 x
  // 1024 over 8192 at H 3, G 8 482, 502; 8 x 512 at H 4, G 8 37, 44).  Lengths
  // that differ leave dead tiles at a sequence's end, which would load the XCDs
  // unevenly (4000, 100 and 2000 at H 6, G 4: 215 us, 160).
  r.tile_major = causal && num_seqs > 1 && sets < kPfXcds && total_q == num_seqs * max_seqlen_q &&
                 r.rows * r.row_wgs * (fresh ? kPfWaves : r.waves) > kPfWaves * cus;
  return r;
}

constexpr int64_t kPfSlotFloats = kPfPartFloats + 2 * kPfRows;

// Workspace: parts' O, their (m, l), key tiles' column maxima, their flags.
int64_t prefill_workspace(const PfLaunch& l) {
  return l.split_wgs * (2 * kPfSlotFloats * 4 + 32) + l.steps * (kPfRows * 4 + kPfWaves);
}

}  // namespace

extern "C" int64_t fp_prefill_workspace_bytes(int64_t kv_heads, int64_t group, int64_t num_seqs, int64_t total_q,
                                              int64_t max_seqlen_q, int64_t max_seqlen_k) {
  if (kv_heads < 1 || group < 1 || kPfRows % group || num_seqs < 1 || total_q < 1 || max_seqlen_q < 1) return 0;
  const PfLaunch l = prefill_launch(kv_heads, group, num_seqs, total_q, max_seqlen_q, max_seqlen_k, true, device_cus());
  return l.split_wgs ? prefill_workspace(l) : 0;
}

extern "C" int64_t fp_prefill_workspace_most(int64_t max_seqlen_k, int64_t cus) {
  const int64_t steps = (max_seqlen_k + kPfKeys - 1) / kPfKeys;
  if (steps < kPfSplitSteps) return 0;
  PfLaunch l{};
  l.split_wgs = (int)((cus > 0 ? cus : device_cus()) / kPfXcds * kPfXcds);
  l.steps = std::min(steps * l.split_wgs, kPfSplitMost);  // a split call has at most a query tile per CU
  return prefill_workspace(l);
}

extern "C" int64_t fp_prefill_split_min_keys(void) { return (kPfSplitSteps - 1) * kPfKeys + 1; }

extern "C" int fp_prefill_plan(int64_t kv_heads, int64_t group, int64_t num_seqs, int64_t total_q,
                               int64_t max_seqlen_q, int64_t max_seqlen_k, int causal, int64_t cus, int64_t* plan) {
  FP_CHECK(plan && kv_heads >= 1 && group >= 1 && kPfRows % group == 0 && num_seqs >= 1 && total_q >= 0 &&
               max_seqlen_q >= 1 && max_seqlen_k >= 0,
           "bad prefill sizes");
  const PfLaunch l =
      prefill_launch(kv_heads, group, num_seqs, total_q, max_seqlen_q, max_seqlen_k, causal != 0, cus > 0 ? cus : device_cus());
  plan[0] = l.waves;
  plan[1] = l.split_wgs;
  plan[2] = l.row_wgs;
  plan[3] = l.rows;
  plan[4] = l.tile_major;
  return 0;
}

extern "C" int fp_prefill_attention(const void* q, int64_t q_stride, const void* wk, const void* wv, int64_t num_pages,
                                    int64_t kv_heads, int64_t group, const int32_t* cu_seqlens_q,
                                    const int32_t* seqused_k, const int32_t* block_table, int64_t bt_stride,
                                    int64_t num_seqs, int64_t max_seqlen_q, int64_t max_seqlen_k, double scale,
                                    int causal, void* out, int64_t out_stride, fp_stream_t stream) {
  return fp_prefill_attention_split(q, q_stride, wk, wv, num_pages, kv_heads, group, cu_seqlens_q, seqused_k, block_table,
                                    bt_stride, num_seqs, 0, max_seqlen_q, max_seqlen_k, scale, causal, out, out_stride,
                                    nullptr, 0, stream);
}

extern "C" int fp_prefill_attention_split(const void* q, int64_t q_stride, const void* wk, const void* wv,
                                          int64_t num_pages, int64_t kv_heads, int64_t group,
                                          const int32_t* cu_seqlens_q, const int32_t* seqused_k,
                                          const int32_t* block_table, int64_t bt_stride,
                                          int64_t num_seqs, int64_t total_q, int64_t max_seqlen_q,
                                          int64_t max_seqlen_k, double scale, int causal, void* out,
                                          int64_t out_stride, void* workspace, int64_t workspace_bytes,
                                          fp_stream_t stream) {
  FP_CHECK(num_seqs >= 0 && max_seqlen_q >= 0 && max_seqlen_k >= 0, "negative sizes");
  if (num_seqs == 0 || max_seqlen_q == 0) return 0;
  FP_CHECK(group == 1 || group == 2 || group == 4 || group == 8, "query heads per KV head must be 1, 2, 4 or 8");
  FP_CHECK(kv_heads >= 1 && kv_heads <= 65535, "kv_heads out of range");
  FP_CHECK(q && wk && wv && cu_seqlens_q && seqused_k && block_table && out, "null pointer");
  FP_CHECK(q_stride >= kv_heads * group * kPfDim && out_stride >= kv_heads * group * kPfDim,
           "token strides must cover all query heads");
  FP_CHECK(bt_stride >= (max_seqlen_k + 127) / 128, "block table narrower than max_seqlen_k");
  FP_CHECK(((uintptr_t)q | (uintptr_t)out | (uintptr_t)wk | (uintptr_t)wv) % 16 == 0 && q_stride % 8 == 0 &&
               out_stride % 8 == 0,
           "q / out / workspace must be 16-byte aligned with 8-element token strides");
  const int64_t rows_per_tile = kPfRows / group;
  const int64_t tiles = (max_seqlen_q + rows_per_tile - 1) / rows_per_tile;
  FP_CHECK(tiles * num_seqs < (1LL << 31), "grid too large");
  PrefillParams p{};
  p.q = static_cast<const uint16_t*>(q);
  p.wk = static_cast<const uint16_t*>(wk);
  p.wv = static_cast<const uint16_t*>(wv);
  p.cu_q = cu_seqlens_q;
  p.seq_k = seqused_k;
  p.block_table = block_table;
  p.out = static_cast<uint16_t*>(out);
  p.q_stride = q_stride;
  p.out_stride = out_stride;
  p.bt_stride = bt_stride;
  p.num_pages = num_pages;
  p.kvh = (int)kv_heads;
  p.group = (int)group;
  p.num_seqs = (int)num_seqs;
  p.tiles_per_seq = (int)tiles;
  p.scale_log2 = (float)(scale * 1.4426950408889634);
  p.causal = causal ? 1 : 0;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  // all LDS is static (two K and two V stages, 64 KB)
  const PfLaunch l = prefill_launch(kv_heads, group, num_seqs, total_q, max_seqlen_q, max_seqlen_k, causal != 0, device_cus());
  if (workspace && l.split_wgs > 0) {
    const int64_t slots = 2 * (int64_t)l.split_wgs;
    FP_CHECK(reinterpret_cast<uintptr_t>(workspace) % 16 == 0 && workspace_bytes >= prefill_workspace(l),
             "prefill workspace too small or not 16-byte aligned (see fp_prefill_workspace_bytes)");
    p.opart = static_cast<float*>(workspace);
    p.ml = p.opart + slots * kPfPartFloats;
    p.ranges = reinterpret_cast<int4*>(p.ml + slots * 2 * kPfRows);
    p.tile_max = reinterpret_cast<float*>(p.ranges + slots);
    p.tile_cap = l.steps;
    p.tile_flag = reinterpret_cast<uint8_t*>(p.tile_max + l.steps * kPfRows);
    const dim3 grid((unsigned)l.split_wgs), block(64 * kPfWaves);
    hipLaunchKernelGGL(prefill_max_kernel, grid, block, 0, s, p);
    FP_LAUNCH_CHECK();
    hipLaunchKernelGGL((prefill_kernel<kPfWaves, true>), grid, block, 0, s, p);
    FP_LAUNCH_CHECK();
    hipLaunchKernelGGL(prefill_merge_kernel, dim3((unsigned)(l.split_wgs - 1), kPfWaves * kPfQt), dim3(kPfMergeThreads), 0,
                       s, p);
  } else {
    FP_CHECK(l.row_wgs * 64 * l.waves <= kPfGridMost, "grid too large");
    p.head_sets = l.tile_major ? -l.head_sets : l.head_sets;
    const dim3 grid((unsigned)l.row_wgs, (unsigned)l.rows), block(64 * l.waves);
    if (l.waves == 4)
      hipLaunchKernelGGL((prefill_kernel<4, false>), grid, block, 0, s, p);
    else
      hipLaunchKernelGGL((prefill_kernel<kPfWaves, false>), grid, block, 0, s, p);
  }
  FP_LAUNCH_CHECK();
  return 0;
}
