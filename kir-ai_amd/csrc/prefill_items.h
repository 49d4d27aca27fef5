// Work items of the tile prefill kernels (prefill.hip, prefill256.hip) and the merge of
// items cut into pieces.
//
// `pack` query heads of one kv head share an item's rows: row R is token R / pack, head
// R % pack of the head group, and an item is BM rows of one (sequence, head group).  All heads
// of the group packed (pack = G), a workgroup's rows are a few tokens: nothing is loaded twice,
// short chunks fill the rows, and little of the causal triangle is wasted.  Where that leaves
// compute units idle, fewer heads are packed: the workgroups of one kv head then read the same
// tiles at the same time, and the L2 shares them.  Or (max_pieces > 1) all heads are packed and
// the keys of every item of a long sequence are cut into max_pieces pieces; a piece leaves
// unnormalised f32 sums (max, sum, outputs), and the last workgroup of an item to finish
// combines them.  The host knows a call's rows but not its context lengths (block-table rows may
// be far wider), so it says how many pieces there may be, and the device sees whether any
// sequence is long enough: if none is, the call runs as if it could not be cut.
//
// Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2, and one
// compute unit reads only about 32 GB/s past its L2 (a tile kernel consumes 23).  So each XCD
// works on a consecutive range of the items, or pieces, of few (sequence, head group) pairs:
// its workgroups read the same keys at about the same time.
#pragma once

#include <algorithm>

#include "arrival.h"
#include "device_common.h"

namespace llh {

constexpr int kPrefillTileKeys = 64;

struct PrefillItem {
  int b, kvh, head0;    // kv head; first query head of the group
  int pack;             // query heads in the rows
  int c0, chunk, ctx;   // first query row, query rows (tokens), context length
  int row0;             // first packed row
  int klo;              // first key any row attends
  int t_begin, t_end;   // keys of this piece: tiles from t_begin (a tile boundary) up to t_end
  int pieces, piece;    // pieces of the item, and this one
  int slot, counter;    // pieces > 1: workspace row of the item's first row, arrival counter
  bool skip;
  int flags;            // why a skipped sequence is refused
};

// Where an item is cut depends on the CUT >= BM packed rows around it (an aligned group), so
// that workgroups of 128 and of 256 rows cut alike and give the same bits.
//
// The sequences of a call that may be cut (at most 64), one per lane: items (of BM rows), groups
// (of CUT rows) and the pieces its items are cut into.  Partial sums lie in the workspace by the
// number of their group among the groups that are cut, in the order (sequence, head group,
// group): [cut group][piece][CUT rows].  The workspace holds ws_pieces pieces, which the host's
// choice of max_pieces keeps below; if the device finds more rows than the call declared,
// nothing is cut.
struct PrefillCuts {
  int c0, chunk, ctx;  // this lane's sequence (as in PrefillItem)
  int items, groups, pieces;
  int cut, cut_end;  // this sequence's cut groups, and their inclusive scan
  int total;         // cut groups in all (0: the other members do not count)
};

// Inclusive scan over the wavefront.
__device__ __forceinline__ int wave_scan(int v, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(v, d);
    v += lane >= d ? up : 0;
  }
  return v;
}

template <int BM, int CUT>
__device__ __forceinline__ PrefillCuts prefill_cuts(const PrefillArgs &a, int lane) {
  PrefillCuts c{0, 0, 0, 0, 0, 1, 0, 0, 0};
  if (lane < a.num_seqs) {
    c.c0 = a.chunk_starts[lane];
    c.chunk = a.chunk_starts[lane + 1] - c.c0;
    c.ctx = a.context_lens[lane];
    const int cut_tiles = prefill_cut_tiles(a.max_pieces, a.pool.head_dim);
    // (a context of fewer tiles is not looked at further)
    if (c.chunk > 0 && c.ctx >= max(c.chunk, (cut_tiles - 1) * kPrefillTileKeys)) {
      const int G = a.cut_pack;
      const int rows = c.chunk * G;
      const int first = c.ctx - c.chunk + (rows - 1) / CUT * CUT / G;  // the last group's first position
      const int lo = a.window > 0 ? max(0, first - a.window + 1) : 0;
      const int tiles = (c.ctx - 1) / kPrefillTileKeys - lo / kPrefillTileKeys + 1;
      c.pieces = tiles >= cut_tiles ? a.max_pieces : 1;
    }
  }
  if (!__any(c.pieces > 1)) return c;
  if (c.chunk > 0 && c.ctx >= c.chunk) {
    c.items = min((c.chunk * a.cut_pack + BM - 1) / BM, a.cut_tiles);
    c.groups = (c.items * BM + CUT - 1) / CUT;
  }
  c.cut = c.pieces > 1 ? c.groups * (a.q_heads / a.cut_pack) : 0;
  c.cut_end = wave_scan(c.cut, lane);
  const int total = __builtin_amdgcn_readlane(c.cut_end, 63);
  c.total = (int64_t)total * a.max_pieces <= a.ws_pieces ? total : 0;
  return c;
}

// Item `tile` (`pack` heads, packed rows tile * BM ..) of head group hg of sequence b, whose chunk
// starts at c0: piece `piece` of `pieces`.
template <int BM, int CUT>
__device__ __forceinline__ PrefillItem prefill_item_of(const PrefillArgs &a, int b, int c0, int chunk, int ctx, int pack,
                                                        int hg, int tile, int pieces, int piece) {
  PrefillItem it;
  it.b = b;
  it.flags = 0;
  it.pack = pack;
  it.head0 = hg * pack;
  it.kvh = it.head0 / (a.q_heads / a.pool.kv_heads);
  it.c0 = c0;
  it.chunk = chunk;
  it.ctx = ctx;
  it.row0 = tile * BM;
  it.pieces = pieces;
  it.piece = piece;
  it.slot = it.counter = 0;
  it.skip = it.chunk <= 0 || it.row0 >= it.chunk * pack || it.ctx < it.chunk;
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
  auto first_key = [&](int r0) { return a.window > 0 ? max(0, prefix + r0 / pack - a.window + 1) : 0; };
  auto end_key = [&](int r0, int n) { return prefix + (min(r0 + n, it.chunk * pack) - 1) / pack + 1; };
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
// Nothing cut: N counts q_tiles items for every (sequence, head group), in that order; an XCD
// whose items are whole (sequence, head group) groups takes the last tile of every group first,
// the longest causal reach first, in runs of a.run tiles.  Else N counts the items and pieces there are, ordered
// (sequence, head group, piece, tile from the last), so ragged lengths leave no XCD idle.
// Workgroups past N leave at once.
template <int BM, int CUT>
__device__ __forceinline__ PrefillItem prefill_item(const PrefillArgs &a) {
  const int L = blockIdx.x;
  PrefillItem none;
  none.skip = true;
  none.flags = 0;
  const int lane = threadIdx.x & 63;
  PrefillCuts c;
  if (a.max_pieces > 1) {
    c = prefill_cuts<BM, CUT>(a, lane);
    if (c.total > 0) {
      const int mine = c.items * c.pieces * (a.q_heads / a.cut_pack);
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
      PrefillItem it = prefill_item_of<BM, CUT>(
          a, b, __builtin_amdgcn_readlane(c.c0, b), __builtin_amdgcn_readlane(c.chunk, b),
          __builtin_amdgcn_readlane(c.ctx, b), a.cut_pack, hg, tile, pieces, q / items);
      const int group = __builtin_amdgcn_readlane(c.cut_end - c.cut, b) + hg * groups + tile * BM / CUT;
      it.slot = group * pieces * CUT + tile * BM % CUT;
      it.counter = group * (CUT / BM) + tile % (CUT / BM);
      return it;
    }
  }
  const int Hg = a.q_heads / a.pack;  // head groups
  const int n_items = a.q_tiles * Hg * a.num_seqs;
  const int per_xcd = (n_items + 7) / 8;
  if (L / 8 >= per_xcd) return none;
  int local = L / 8;
  if (per_xcd % a.q_tiles == 0) {
    const int groups = per_xcd / a.q_tiles;
    const int run = CUT == 128 ? a.run : 1;  // (the head_dim-256 kernel)
    const int whole = a.q_tiles / run * run;  // tiles in whole runs
    const int i = L / 8 - groups * whole;
    if (i < 0) {
      const int j = L / 8 / run;
      local = j % groups * a.q_tiles + (a.q_tiles - 1 - (j / groups * run + L / 8 % run));
    } else {  // the first tiles, too few for a run
      const int rest = a.q_tiles - whole;
      local = i / rest * a.q_tiles + (rest - 1 - i % rest);
    }
  }
  const int w = L % 8 * per_xcd + local;
  if (w >= n_items) return none;
  const int grp = w / a.q_tiles;
  const int b = grp / Hg;
  int c0, chunk, ctx;
  if (a.max_pieces > 1) {  // read already
    c0 = __builtin_amdgcn_readlane(c.c0, b);
    chunk = __builtin_amdgcn_readlane(c.chunk, b);
    ctx = __builtin_amdgcn_readlane(c.ctx, b);
  } else {
    c0 = a.chunk_starts[b];
    chunk = a.chunk_starts[b + 1] - c0;
    ctx = a.context_lens[b];
  }
  return prefill_item_of<BM, CUT>(a, b, c0, chunk, ctx, a.pack, grp % Hg, w % a.q_tiles, 1, 0);
}

// Workgroups of a call: every item whole, or those of a call with cuts: every item and the
// pieces beyond that of those that are cut.
template <int BM, int CUT>
inline int prefill_grid(const PrefillArgs &a) {
  long long n = (long long)a.q_tiles * (a.q_heads / a.pack) * a.num_seqs;
  if (a.max_pieces > 1) {
    const long long items = (long long)a.cut_tiles * (a.q_heads / a.cut_pack) * a.num_seqs;
    n = std::max(n, std::min(items * a.max_pieces, items + a.ws_pieces * (CUT / BM)));
  }
  return (int)((n + 7) / 8 * 8);
}

// A wavefront's sums of ROWS packed rows from `row` on (`live` of them real), dims d .. d + W, from
// its LDS buffer [ROWS][W + kPiecePad]: whole lines, written through the L2 (stores straight from
// the accumulators, 8 bytes a row, made a cut call of 1 x (4096 + 512) tokens, Hq32 / Hkv4, 86 us; 68
// this way).
constexpr int kPiecePad = 2;
template <int D, int CUT, int ROWS, int W>
__device__ __forceinline__ void store_piece(const PrefillArgs &a, const PrefillItem &it, const float *buf, int row,
                                            int live, int d, int lane) {
  constexpr int PER = 128 / W;  // rows per store
  const int r0 = lane / (W / 2), x = lane % (W / 2) * 2;
#pragma unroll
  for (int i = 0; i < ROWS / PER; i++) {
    const int r = i * PER + r0;
    const float2 v = *reinterpret_cast<const float2 *>(&buf[r * (W + kPiecePad) + x]);
    if (r < live)
      st_agent(reinterpret_cast<float2 *>(&a.ws_o[((size_t)it.slot + it.piece * CUT + row + r) * D + d + x]), v);
  }
}
template <int CUT>
__device__ __forceinline__ void store_piece_sums(const PrefillArgs &a, const PrefillItem &it, int row, float m,
                                                 float l) {
  st_agent(&a.ws_ml[(size_t)it.slot + it.piece * CUT + row], make_float2(m, l));
}

// The item's rows from its N pieces, by the workgroup that stored the last of them.
template <int D, int BM, int CUT, int N>
__device__ __forceinline__ void merge_pieces(const PrefillArgs &a, const PrefillItem &it) {
  constexpr int PARTS = D / 128;          // row parts of 128 dims
  constexpr int U = N <= 4 ? 32 / N : 4;  // row parts of a wavefront at a time: 32 loads in flight per lane
  const int lane = threadIdx.x & 63;
  const int parts = min(BM, it.chunk * it.pack - it.row0) * PARTS;
  for (int u0 = (int)(threadIdx.x >> 6) * U; u0 < parts; u0 += (int)(blockDim.x >> 6) * U) {
    const float2 *ml[U];
    const float *o[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int part = min(u0 + u, parts - 1);
      const size_t r = (size_t)it.slot + part / PARTS;
      ml[u] = a.ws_ml + r;
      o[u] = a.ws_o + r * D + part % PARTS * 128;
    }
    float2 out[U];
    float mx[U], sum[U];
    merge_parts<U, N>(ml, CUT, o, (size_t)CUT * D, N, lane, out, mx, sum);
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (u0 + u >= parts) break;
      const int row = it.row0 + (u0 + u) / PARTS;
      const float inv = sum[u] > 0.0f ? 1.0f / sum[u] : 0.0f;
      const size_t at = ((size_t)(it.c0 + row / it.pack) * a.q_heads + it.head0 + row % it.pack) * D +
                        (u0 + u) % PARTS * 128 + 2 * lane;
      a.out[at] = f32_to_bf16_rne(gated(out[u].x * inv, a.gate, at));
      a.out[at + 1] = f32_to_bf16_rne(gated(out[u].y * inv, a.gate, at + 1));
    }
  }
}

// After a piece's sums are stored (all threads of the workgroup call).
template <int D, int BM, int CUT>
__device__ __forceinline__ void finish_piece(const PrefillArgs &a, const PrefillItem &it) {
  if (!last_to_arrive(&a.counters[it.counter], it.pieces)) return;
  if (it.pieces == 2) return merge_pieces<D, BM, CUT, 2>(a, it);
  if (it.pieces == 4) return merge_pieces<D, BM, CUT, 4>(a, it);
  merge_pieces<D, BM, CUT, kPrefillMaxPieces>(a, it);
}

}  // namespace llh
