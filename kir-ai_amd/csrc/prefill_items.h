// Work items of the tile prefill kernels (prefill.hip, prefill256.hip) and the merge of
// items cut into pieces.
//
// `pack` query heads of one kv head share an item's rows: row R is token R / pack, head
// R % pack of the head group, and an item is BM rows of one (sequence, head group).  All heads
// of the group packed (pack = G), a workgroup's rows are a few tokens: nothing is loaded twice,
// short chunks fill the rows, and little of the causal triangle is wasted.  Where that leaves
// compute units idle, fewer heads are packed: the workgroups of one kv head then read the same
// tiles at the same time, and the L2 shares them.  Or (max_pieces > 1) the keys of every item
// are cut into the same number of pieces; a piece leaves unnormalised f32 sums (max, sum,
// outputs) that prefill_merge_kernel combines.  Both are the host's choice; whether a sequence
// is long enough to be cut is seen on the device.
//
// Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2, and one
// compute unit reads only about 32 GB/s past its L2 (a tile kernel consumes 23).  So each XCD
// works on a consecutive range of the items, or pieces, of few (sequence, head group) pairs:
// its workgroups read the same keys at about the same time.
#pragma once

#include <algorithm>

#include "device_common.h"

namespace llh {

constexpr int kPrefillTileKeys = 64;

struct PrefillItem {
  int b, kvh, head0;    // kv head; first query head of the group
  int c0, chunk, ctx;   // first query row, query rows (tokens), context length
  int row0;             // first packed row
  int klo;              // first key any row attends
  int t_begin, t_end;   // keys of this piece: tiles from t_begin (a tile boundary) up to t_end
  int pieces, slot;     // pieces of the item; this piece's first row in the workspace
  bool skip;
  int flags;            // why a skipped sequence is refused
};

// Where an item is cut depends on the CUT >= BM packed rows around it (an aligned group), so
// that workgroups of 128 and of 256 rows cut alike and give the same bits.
//
// A sequence's items (of BM rows), groups (of CUT rows) and the pieces its items are cut into.
template <int BM, int CUT>
__device__ __forceinline__ void prefill_seq(const PrefillArgs &a, int b, int &items, int &groups, int &pieces) {
  items = groups = 0;
  pieces = 1;
  if (b >= a.num_seqs) return;
  const int chunk = a.chunk_starts[b + 1] - a.chunk_starts[b];
  const int ctx = a.context_lens[b];
  if (chunk <= 0 || ctx < chunk) return;
  const int G = a.pack;
  const int rows = chunk * G;
  items = min((rows + BM - 1) / BM, a.q_tiles);
  groups = (items * BM + CUT - 1) / CUT;
  const int first = ctx - chunk + (rows - 1) / CUT * CUT / G;  // the last group's first position
  const int lo = a.window > 0 ? max(0, first - a.window + 1) : 0;
  const int tiles = (ctx - 1) / kPrefillTileKeys - lo / kPrefillTileKeys + 1;
  pieces = tiles >= prefill_cut_tiles(a.max_pieces, a.pool.head_dim) ? a.max_pieces : 1;
}

// Inclusive scan over the wavefront.
__device__ __forceinline__ int wave_scan(int v, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(v, d);
    v += lane >= d ? up : 0;
  }
  return v;
}

// The sequences of a call that may be cut (at most 64), one per lane.  Partial sums lie in the
// workspace by the number of their group among the groups that are cut, in the order (sequence,
// head group, group): [cut group][piece][CUT rows].  The workspace holds ws_pieces pieces, which
// the host's choice of max_pieces keeps below; if the device finds more rows than the call
// declared, nothing is cut.
struct PrefillCuts {
  int items, groups, pieces;
  int cut, cut_end;  // this sequence's cut groups, and their inclusive scan
  int total;         // cut groups in all
};
template <int BM, int CUT>
__device__ __forceinline__ PrefillCuts prefill_cuts(const PrefillArgs &a, int lane) {
  PrefillCuts c;
  prefill_seq<BM, CUT>(a, lane, c.items, c.groups, c.pieces);
  c.cut = c.pieces > 1 ? c.groups * (a.q_heads / a.pack) : 0;
  c.cut_end = wave_scan(c.cut, lane);
  c.total = __builtin_amdgcn_readlane(c.cut_end, 63);
  if ((int64_t)c.total * a.max_pieces > a.ws_pieces) {
    c.pieces = 1;
    c.cut = c.cut_end = c.total = 0;
  }
  return c;
}

// Sequence b's item `tile` (packed rows tile * BM ..) of head group hg: piece `piece` of
// `pieces`.
template <int BM, int CUT>
__device__ __forceinline__ PrefillItem prefill_item_of(const PrefillArgs &a, int b, int hg, int tile, int pieces,
                                                        int piece) {
  PrefillItem it;
  it.b = b;
  it.flags = 0;
  const int G = a.pack;
  it.head0 = hg * G;
  it.kvh = it.head0 / (a.q_heads / a.pool.kv_heads);
  it.c0 = a.chunk_starts[b];
  it.chunk = a.chunk_starts[b + 1] - it.c0;
  it.ctx = a.context_lens[b];
  it.row0 = tile * BM;
  it.pieces = pieces;
  it.slot = 0;
  it.skip = it.chunk <= 0 || it.row0 >= it.chunk * G || it.ctx < it.chunk;
  if (it.skip) return it;
  const int prefix = it.ctx - it.chunk;
  // every key of the chunk's first row through the last must be resident at once: a longer
  // span would alias its own table entries (rows are read modulo max_blocks)
  const int first_lo = a.window > 0 ? max(0, prefix - a.window + 1) : 0;
  if ((int64_t)(it.ctx - first_lo) > (int64_t)a.max_blocks * kFastBlockTokens) {
    it.skip = true;
    it.flags = tile == 0 ? kErrSpan : 0;
    return it;
  }
  // first key and end of the rows from r0 on, n of them
  auto first_key = [&](int r0) { return a.window > 0 ? max(0, prefix + r0 / G - a.window + 1) : 0; };
  auto end_key = [&](int r0, int n) { return prefix + (min(r0 + n, it.chunk * G) - 1) / G + 1; };
  it.klo = first_key(it.row0);
  it.t_begin = it.klo / kPrefillTileKeys * kPrefillTileKeys;
  it.t_end = end_key(it.row0, BM);
  if (pieces > 1) {  // a piece may hold none of this item's tiles: its sums are empty
    const int g0 = it.row0 / CUT * CUT;
    const int t0 = first_key(g0) / kPrefillTileKeys;
    const int tiles = (end_key(g0, CUT) + kPrefillTileKeys - 1) / kPrefillTileKeys - t0;
    it.t_begin = max(it.t_begin, (t0 + piece * tiles / pieces) * kPrefillTileKeys);
    it.t_end = min(it.t_end, (t0 + (piece + 1) * tiles / pieces) * kPrefillTileKeys);
  }
  return it;
}

// The item, or piece, of this workgroup L: number (L % 8) * ceil(N / 8) + L / 8 of N.
// Whole items: N counts q_tiles items for every (sequence, head group), in that order; an XCD
// whose items are whole (sequence, head group) groups takes the last tile of every group first,
// the longest causal reach first.  Pieces (at most 64 sequences, one per lane): N counts the
// pieces there are, ordered (sequence, head group, piece, tile from the last), so ragged
// lengths leave no XCD idle; workgroups past them leave at once.
template <int BM, int CUT>
__device__ __forceinline__ PrefillItem prefill_item(const PrefillArgs &a) {
  const int Hg = a.q_heads / a.pack;  // head groups
  const int L = blockIdx.x;
  PrefillItem none;
  none.skip = true;
  none.flags = 0;
  if (a.max_pieces <= 1) {
    const int n_items = a.q_tiles * Hg * a.num_seqs;
    const int per_xcd = (n_items + 7) / 8;
    int local = L / 8;
    if (per_xcd % a.q_tiles == 0) {
      const int groups = per_xcd / a.q_tiles;
      local = L / 8 % groups * a.q_tiles + (a.q_tiles - 1 - L / 8 / groups);
    }
    const int w = L % 8 * per_xcd + local;
    if (w >= n_items) return none;
    const int grp = w / a.q_tiles;
    return prefill_item_of<BM, CUT>(a, grp / Hg, grp % Hg, w % a.q_tiles, 1, 0);
  }
  const int lane = threadIdx.x & 63;
  const PrefillCuts c = prefill_cuts<BM, CUT>(a, lane);
  const int mine = c.items * c.pieces * Hg;
  const int end = wave_scan(mine, lane);
  const int live = __builtin_amdgcn_readlane(end, 63);
  const int per_xcd = (live + 7) / 8;
  const int w = L % 8 * per_xcd + L / 8;
  if (L / 8 >= per_xcd || w >= live) return none;
  const int b = __ffsll(__ballot(w < end)) - 1;
  const int items = __builtin_amdgcn_readlane(c.items, b);
  const int pieces = __builtin_amdgcn_readlane(c.pieces, b);
  const int groups = __builtin_amdgcn_readlane(c.groups, b);
  const int r = w - __builtin_amdgcn_readlane(end - mine, b);
  const int hg = r / (items * pieces);
  const int q = r % (items * pieces);
  const int tile = items - 1 - q % items;
  const int piece = q / items;
  PrefillItem it = prefill_item_of<BM, CUT>(a, b, hg, tile, pieces, piece);
  const int group = __builtin_amdgcn_readlane(c.cut_end - c.cut, b) + hg * groups + tile * BM / CUT;
  it.slot = (group * pieces + piece) * CUT + tile * BM % CUT;
  return it;
}

// Workgroups of a call: every item whole, and the pieces beyond that of those that are cut.
template <int BM, int CUT>
inline int prefill_grid(const PrefillArgs &a) {
  const long long items = (long long)a.q_tiles * (a.q_heads / a.pack) * a.num_seqs;
  const long long n = a.max_pieces <= 1 ? items : std::min(items * a.max_pieces, items + a.ws_pieces * (CUT / BM));
  return (int)((n + 7) / 8 * 8);
}

// Combines the pieces of every cut item: a workgroup takes kMergeRows packed rows of a cut group
// at a time, each thread four dims of a row, every piece's loads in flight together.
constexpr int kMergeRows = 8;
constexpr int kMergeGrid = 1024;
template <int D, int CUT>
__global__ __launch_bounds__(kMergeRows * D / 4) void prefill_merge_kernel(const PrefillArgs a) {
  typedef __attribute__((ext_vector_type(4))) float f32x4_t;
  const PrefillCuts c = prefill_cuts<CUT, CUT>(a, threadIdx.x & 63);
  const int G = a.pack;
  const int d = threadIdx.x % (D / 4) * 4;
  for (int u = blockIdx.x; u < c.total * (CUT / kMergeRows); u += gridDim.x) {
    const int group = u / (CUT / kMergeRows);
    const int b = __ffsll(__ballot(group < c.cut_end)) - 1;
    const int groups = __builtin_amdgcn_readlane(c.groups, b);
    const int g = group - __builtin_amdgcn_readlane(c.cut_end - c.cut, b);
    const PrefillItem it = prefill_item_of<CUT, CUT>(a, b, g / groups, g % groups, a.max_pieces, 0);
    if (it.skip) continue;
    const int lr = u % (CUT / kMergeRows) * kMergeRows + threadIdx.x / (D / 4);
    const int row = it.row0 + lr;
    if (row >= it.chunk * G) continue;
    const size_t p0 = (size_t)group * a.max_pieces * CUT + lr;
    f32x4_t o[kPrefillMaxPieces];
    float2 ml[kPrefillMaxPieces];
#pragma unroll
    for (int i = 0; i < kPrefillMaxPieces; i++) {
      const size_t p = p0 + (size_t)min(i, a.max_pieces - 1) * CUT;
      ml[i] = a.ws_ml[p];
      o[i] = *reinterpret_cast<const f32x4_t *>(&a.ws_o[p * D + d]);
    }
    float mm = ml[0].x;
#pragma unroll
    for (int i = 1; i < kPrefillMaxPieces; i++) mm = fmaxf(mm, ml[i].x);
    const float mref = mm == -INFINITY ? 0.0f : mm;
    float ll = 0.0f;
    f32x4_t oo = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < kPrefillMaxPieces; i++) {
      const float f = i < a.max_pieces ? __builtin_amdgcn_exp2f(ml[i].x - mref) : 0.0f;
      ll += ml[i].y * f;
      oo += o[i] * f;
    }
    const float inv = ll > 0.0f ? 1.0f / ll : 0.0f;
    const size_t out = ((size_t)(it.c0 + row / G) * a.q_heads + it.head0 + row % G) * D + d;
#pragma unroll
    for (int e = 0; e < 4; e++) a.out[out + e] = f32_to_bf16_rne(gated(oo[e] * inv, a.gate, out + e));
  }
}

template <int D, int BM, int CUT>
hipError_t launch_prefill_merge(const PrefillArgs &a, hipStream_t s) {
  const long long tiles = ((long long)a.q_tiles * BM + CUT - 1) / CUT;
  const long long groups = tiles * (a.q_heads / a.pack) * a.num_seqs;
  const long long units = std::min<long long>(groups, a.ws_pieces / a.max_pieces) * (CUT / kMergeRows);
  PrefillArgs m = a;
  m.q_tiles = (int32_t)tiles;
  hipLaunchKernelGGL((prefill_merge_kernel<D, CUT>), dim3((unsigned)std::min<long long>(units, kMergeGrid)),
                     dim3(kMergeRows * D / 4), 0, s, m);
  return hipGetLastError();
}

}  // namespace llh
