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
// outputs) that prefill_merge_kernel combines.  Both are the host's choice.
//
// Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2, and one
// compute unit reads only about 32 GB/s past its L2 (a tile kernel consumes 23).  So each XCD
// works on a consecutive range of the items, or pieces, of few (sequence, head group) pairs:
// its workgroups read the same keys at about the same time.
#pragma once

#include "device_common.h"

namespace llh {

constexpr int kPrefillTileKeys = 64;

struct PrefillItem {
  int b, kvh, head0;    // kv head; first query head of the group
  int c0, chunk, ctx;   // first query row, query rows (tokens), context length
  int row0;             // first packed row
  int klo;              // first key any row attends
  int t_begin, t_end;   // keys of this piece: tiles from t_begin (a tile boundary) up to t_end
  int pieces, slot;     // pieces of the item; workspace slot of this piece
  bool skip;
  int flags;            // why a skipped sequence is refused
};

// Where an item is cut depends on the CUT >= BM packed rows around it (an aligned group), so
// that workgroups of 128 and of 256 rows cut alike and give the same bits.
//
// A sequence's items and the pieces each is cut into.
template <int BM, int CUT>
__device__ __forceinline__ void prefill_seq(const PrefillArgs &a, int b, int &items, int &pieces) {
  items = 0;
  pieces = 1;
  if (b >= a.num_seqs) return;
  const int chunk = a.chunk_starts[b + 1] - a.chunk_starts[b];
  const int ctx = a.context_lens[b];
  if (chunk <= 0 || ctx < chunk) return;
  const int G = a.pack;
  const int rows = chunk * G;
  items = min((rows + BM - 1) / BM, a.q_tiles);
  const int first = ctx - chunk + (rows - 1) / CUT * CUT / G;  // the last group's first position
  const int lo = a.window > 0 ? max(0, first - a.window + 1) : 0;
  const int tiles = (ctx - 1) / kPrefillTileKeys - lo / kPrefillTileKeys + 1;
  pieces = tiles >= prefill_cut_tiles(a.max_pieces, a.pool.head_dim) ? a.max_pieces : 1;
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
  it.slot = ((b * (a.q_heads / G) + hg) * a.q_tiles + tile) * a.max_pieces + piece;
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
  int items, pieces;
  prefill_seq<BM, CUT>(a, lane, items, pieces);
  const int mine = items * pieces * Hg;
  int end = mine;  // inclusive scan
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(end, d);
    end += lane >= d ? up : 0;
  }
  const int live = __builtin_amdgcn_readlane(end, 63);
  const int per_xcd = (live + 7) / 8;
  const int w = L % 8 * per_xcd + L / 8;
  if (L / 8 >= per_xcd || w >= live) return none;
  const int b = __ffsll(__ballot(w < end)) - 1;
  items = __builtin_amdgcn_readlane(items, b);
  pieces = __builtin_amdgcn_readlane(pieces, b);
  const int r = w - __builtin_amdgcn_readlane(end - mine, b);
  const int q = r % (items * pieces);
  return prefill_item_of<BM, CUT>(a, b, r / (items * pieces), items - 1 - q % items, pieces, q / items);
}

template <int BM>
inline int prefill_grid(const PrefillArgs &a) {
  const int n_items = a.q_tiles * (a.q_heads / a.pack) * a.num_seqs;
  return (n_items * a.max_pieces + 7) / 8 * 8;
}

// Combines the pieces of every cut item: one workgroup per kMergeRows packed rows of one item,
// each thread four dims of a row, every piece's loads in flight together.
constexpr int kMergeRows = 8;
template <int D, int BM, int CUT>
__global__ __launch_bounds__(kMergeRows * D / 4) void prefill_merge_kernel(const PrefillArgs a) {
  typedef __attribute__((ext_vector_type(4))) float f32x4_t;
  const int item = blockIdx.x / (BM / kMergeRows);
  const int grp = item / a.q_tiles;
  const int Hg = a.q_heads / a.pack;
  const int b = grp / Hg;
  int items, pieces;
  prefill_seq<BM, CUT>(a, b, items, pieces);
  const PrefillItem it =
      prefill_item_of<BM, CUT>(a, b, grp % Hg, item % a.q_tiles, pieces, 0);
  if (it.skip || it.pieces <= 1) return;
  const int G = a.pack;
  const int lr = blockIdx.x % (BM / kMergeRows) * kMergeRows + threadIdx.x / (D / 4);
  const int row = it.row0 + lr;
  if (row >= it.chunk * G) return;
  const int d = threadIdx.x % (D / 4) * 4;
  const size_t p0 = (size_t)it.slot * BM + lr;
  f32x4_t o[kPrefillMaxPieces];
  float2 ml[kPrefillMaxPieces];
#pragma unroll
  for (int i = 0; i < kPrefillMaxPieces; i++) {
    const size_t p = p0 + (size_t)min(i, it.pieces - 1) * BM;
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
    const float f = i < it.pieces ? __builtin_amdgcn_exp2f(ml[i].x - mref) : 0.0f;
    ll += ml[i].y * f;
    oo += o[i] * f;
  }
  const float inv = ll > 0.0f ? 1.0f / ll : 0.0f;
  const size_t out = ((size_t)(it.c0 + row / G) * a.q_heads + it.head0 + row % G) * D + d;
#pragma unroll
  for (int e = 0; e < 4; e++) a.out[out + e] = f32_to_bf16_rne(gated(oo[e] * inv, a.gate, out + e));
}

template <int D, int BM, int CUT>
hipError_t launch_prefill_merge(const PrefillArgs &a, hipStream_t s) {
  const int n_items = a.q_tiles * (a.q_heads / a.pack) * a.num_seqs;
  hipLaunchKernelGGL((prefill_merge_kernel<D, BM, CUT>), dim3(n_items * (BM / kMergeRows)), dim3(kMergeRows * D / 4), 0, s,
                     a);
  return hipGetLastError();
}

}  // namespace llh
