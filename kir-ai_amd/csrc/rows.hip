// Paged attention of few query rows over many keys, on gfx950 MFMA with split keys.
//
// The query rows that share a kv head -- the G heads of a decode token, or the heads of
// a short prefill chunk -- are packed sixteen to a tile (row r = token * G + head), and
// the keys of a sequence are split over workgroups and, inside one, over its four
// wavefronts.  A wavefront walks units of 64 keys (32 at head_dim 256): it loads the unit's
// K and V straight into MFMA operand registers (every byte is used by one wavefront, so LDS
// would only add a copy), and the next unit's loads are in flight behind the current unit's
// math.  Wavefronts merge in LDS; splits merge in a second launch (decode, whose host knows the
// longest context and so whether there are any) or, where only the block-table width is known, by
// the last workgroup of a tile to arrive, so that short contexts pay for no launch.
//
// It serves
//  * decode steps outside the tuned kernels' shapes (head_dim 128 or 256, 16-token
//    blocks): other group sizes, and int8 / fp8 blocks at head_dim 256 -- the
//    contract of decode_generic_kernel (f32 softmax weights, non-finite scores
//    flagged, a block outside the pool scoring 0);
//  * prefill over int8 / fp8 blocks at head_dim 256, again with f32 weights;
//  * prefill calls of few rows, where a 128-row tile per head would leave most of the
//    chip idle (contract of paged_prefill_kernel: positions [lo(pos), pos]).
// Reference: crates/llm-backend/src/core/native_attention.rs:356-464,707-773.
//
// S^T = K Q^T and O^T += V^T P^T on v_mfma_f32_16x16x32 (A 16 x 32: lane l holds row
// l % 16, k 8 (l / 16) .. +8; B 32 x 16: column l % 16, same k; D: column l % 16, rows
// 4 (l / 16) .. +4).  The rows of a K operand may be any keys, so they are chosen such
// that the scores a lane receives belong to adjacent keys of one block, the keys of one
// load of a V^T row: in step s of 32 keys (blocks 2s, 2s+1), tile j = 0, 1 gives lane
// group g the keys 32 s + 8 g + 4 j + i.  So P^T goes from the accumulators to the B
// operand without leaving its lane.
//
// int8 / fp8 codes enter the MFMA exactly (as bf16); their scales multiply the scores
// and the weights in f32.  PARTS = 3 splits every f32 weight into three bf16 terms
// (24 bits, the whole f32 significand) for three P V products, PARTS = 2 into two terms of the
// pool's own type (bf16: 16 bits; fp16: 22, and 2^-31 of the largest weight at the least);
// PARTS = 1 rounds the weights once, as the tuned 16-bit prefill does.  Beside three terms an
// fp16 element enters as two bf16 terms (8 + 3 bits, exact), so that q stays as it is and small
// weights keep their bits, which fp16 terms would lose below 2^-14.
//
// Bound: the chain lengths -> table entry -> K / V at the start of a workgroup and, in long
// splits, the latency of one unit's loads (one unit in flight per wavefront); HBM traffic
// is each K / V byte once per 16-row tile.  Measured on MI355X: decode, 16 x U[256, 4096]
// tokens, Hq16 / Hkv2, head_dim 256, fp8: 3139 us on the element-wise kernel, 19.7 us here
// (32 MB, 1.6 TB/s); a chunk of 8 tokens over 4099 cached ones, Hq16 / Hkv8, head_dim 128,
// bf16: 119.5 us on 128-row tiles, 14.8 us here (17 MB, 1.1 TB/s; the merge of 17 splits by one
// workgroup takes half of it: with a second launch 12.2, but 8 tokens over none under a table of
// 2048 blocks then 10.2 against 7.4); 2 x (1024 + 250) tokens,
// Hq16 / Hkv2, head_dim 256, int8: 10.6 ms element-wise, 48 us here (197 TFLOP/s: the code
// conversions, repeated by every 16-row tile, bound it).
#include "arrival.h"

namespace llh {

namespace {

constexpr int BT = kFastBlockTokens;
constexpr int TILE = 16;  // packed query rows per tile
constexpr int WAVES = 4;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

template <int OP>
__device__ __forceinline__ f32x4_t mfma16(const u32x4_t &a, const u32x4_t &b, const f32x4_t &c) {
  if constexpr (OP == kF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                    c, 0, 0, 0);
}

__device__ __forceinline__ u32x4_t ld16(const char *p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(p));
}

// Eight codes as eight bf16 elements (exact).
template <int FMT>
__device__ __forceinline__ u32x4_t codes8(uint32_t lo, uint32_t hi) {
  if constexpr (FMT == kInt8)
    return u32x4_t{i8x2_to_bf16(lo, 0), i8x2_to_bf16(lo, 2), i8x2_to_bf16(hi, 0), i8x2_to_bf16(hi, 2)};
  else
    return u32x4_t{fp8x2_to_bf16<false>(lo), fp8x2_to_bf16<true>(lo), fp8x2_to_bf16<false>(hi),
                   fp8x2_to_bf16<true>(hi)};
}

// Two values cut (rounded towards zero) to OP's 16 bits.
template <int OP>
__device__ __forceinline__ uint32_t cut_16(float lo, float hi) {
  if constexpr (OP == kF16)
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(lo, hi));
  else
    return __float_as_uint(lo) >> 16 | (__float_as_uint(hi) & 0xffff0000u);
}

// Eight fp16 elements as eight bf16 terms and the rest, both exact; an infinity or a NaN is all
// in the first.
__device__ __forceinline__ void f16x8_to_bf16(const u32x4_t &w, u32x4_t &hi, u32x4_t &lo) {
#pragma unroll
  for (int x = 0; x < 4; x++) {
    uint32_t h[2], l[2];
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const float v = f16_bits_to_f32(w[x] >> (16 * e) & 0xffffu);
      h[e] = __float_as_uint(v) & 0xffff0000u;
      l[e] = (h[e] & 0x7f800000u) == 0x7f800000u ? 0u : __float_as_uint(v - __uint_as_float(h[e]));
    }
    hi[x] = h[0] >> 16 | h[1];
    lo[x] = l[0] >> 16 | l[1];
  }
}

// The keys of a sequence and their split, the same in every kernel of a call.
struct SeqSplit {
  int c0, chunk, ctx;  // first query row, query rows, context length
  int lo;              // first position any row attends
  int unit0, units;    // units of UK keys
  int per_split, n_splits;
  bool skip;           // nothing to compute (flags: why)
  int flags;
};

template <int UK>
__device__ __forceinline__ SeqSplit seq_split(const RowsArgs &a, int b) {
  SeqSplit s;
  s.flags = 0;
  s.c0 = a.chunk_starts ? a.chunk_starts[b] : b;
  s.chunk = a.chunk_starts ? a.chunk_starts[b + 1] - s.c0 : 1;
  s.ctx = a.context_lens[b];
  const int first = s.ctx - s.chunk;  // position of the first row
  s.lo = a.window > 0 ? max(0, first - a.window + 1) : 0;
  const int span = max(0, s.ctx - s.lo);
  if ((a.max_span > 0 && span > a.max_span) || (a.max_len > 0 && s.ctx > a.max_len)) s.flags = kErrTooManySplits;
  else if ((int64_t)span > (int64_t)a.max_blocks * BT) s.flags = kErrSpan;
  s.skip = s.flags != 0 || s.chunk <= 0 || (a.chunk_starts && s.ctx < s.chunk);
  s.unit0 = s.lo / UK;
  s.units = span > 0 ? (s.ctx - 1) / UK - s.unit0 + 1 : 0;
  s.per_split = s.units <= a.single_units ? a.single_units
                                          : max(a.split_units, (s.units + a.max_splits - 1) / a.max_splits);
  s.n_splits = (s.units + s.per_split - 1) / s.per_split;
  return s;
}

// 1 / (weight sum).  No weight at all (every key masked, or every score -inf) gives the zero
// row of the tile prefill and the reference-order decode, and the NaN (0 / 0) of the vector
// decode kernels in the calls that are theirs too.
__device__ __forceinline__ float row_inv(const RowsArgs &a, float ll) {
  return ll == 0.0f && (a.chunk_starts || a.zero_bad) ? 0.0f : 1.0f / ll;
}

// keys per unit: K and V of a unit take 64 operand registers each in 16-bit formats (32 in
// 8-bit ones)
template <int D>
constexpr int kUnitKeys = D == 256 ? 32 : 64;

// Of a tile's rows, `n` partials from split s0 on, every `stride`-th, by one workgroup at agent
// scope (arrival.h): the output, or (PARTIAL) a partial in the place of split s0.
constexpr int kSplitGroup = 8;
constexpr int kFlatSplits = 24;  // splits merged at once
template <int D, bool PARTIAL>
__device__ __forceinline__ void merge_splits(const RowsArgs &a, const SeqSplit &sq, int b, int kvh, int G, int row0,
                                             int live, int s0, int stride, int n) {
  constexpr int HALVES = D / 128;             // row parts of 128 dims
  constexpr int U = TILE * HALVES / WAVES;    // a wavefront's, all at once: each round is a trip to memory
  const int lane = threadIdx.x & 63;
  for (int u0 = (int)(threadIdx.x >> 6) * U; u0 < live * HALVES; u0 += WAVES * U) {
    const float2 *ml[U];
    const float *o[U];
    size_t place[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int part = min(u0 + u, live * HALVES - 1);
      const int r = row0 + part / HALVES;
      place[u] = (((size_t)b * a.max_rows + r / G) * a.q_heads + kvh * G + r % G) * a.max_splits + s0;
      ml[u] = a.ws_ml + place[u];
      o[u] = a.ws_o + place[u] * D + part % HALVES * 128;
    }
    float2 out[U];
    float mx[U], sum[U];
    merge_parts<U, 8>(ml, stride, o, (size_t)stride * D, n, lane, out, mx, sum);
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (u0 + u >= live * HALVES) break;
      const int half = (u0 + u) % HALVES;
      if constexpr (PARTIAL) {
        st_agent(reinterpret_cast<float2 *>(&a.ws_o[place[u] * D + half * 128]) + lane, out[u]);
        if (half == HALVES - 1 && lane == 0) st_agent(&a.ws_ml[place[u]], make_float2(mx[u], sum[u]));
      } else {
        const int r = row0 + (u0 + u) / HALVES;
        const float inv = row_inv(a, sum[u]);
        const size_t at = ((size_t)(sq.c0 + r / G) * a.q_heads + kvh * G + r % G) * D + half * 128 + 2 * lane;
        a.out[at] = f32_to_bf16_rne(gated(out[u].x * inv, a.gate, at));
        a.out[at + 1] = f32_to_bf16_rne(gated(out[u].y * inv, a.gate, at + 1));
      }
    }
  }
}

template <int D, int FMT, int PARTS>
__global__ __launch_bounds__(64 * WAVES, D == 256 && is16(FMT) ? 1 : 2) void paged_rows_kernel(const RowsArgs a) {
  constexpr bool Q8 = !is16(FMT);
  constexpr bool WIDE16 = FMT == kF16 && PARTS == 3;  // fp16 elements as two bf16 terms
  constexpr int OP = FMT == kF16 && !WIDE16 ? kF16 : kBf16;
  // Two fp16 terms reach 2^-24 at the least: the weights, at most 2^8 (below), are held 2^7 larger.
  constexpr float BIAS = OP == kF16 && PARTS == 2 ? 7.0f : 0.0f;
  constexpr int UK = kUnitKeys<D>;
  constexpr int NT = UK / 16;          // score tiles of 16 keys
  constexpr int NS = UK / 32;          // P V steps of 32 keys
  constexpr int KS = D / 32;           // k-steps of a score
  constexpr int KL = Q8 ? D / 64 : KS; // 16-byte loads of a K operand row
  constexpr int ND = D / 16;           // output tiles
  constexpr int ES = Q8 ? 1 : 2;

  const int Hkv = a.pool.kv_heads;
  const int G = a.q_heads / Hkv;
  // The split is the slowest index.  max_splits follows the longest context there may be, and
  // workgroups go round-robin over the 8 XCDs: with the splits of a tile side by side, the first
  // splits of sequences shorter than that would meet on a few XCDs, between workgroups that leave
  // at once (8 x (384 + 8) tokens, Hq16 / Hkv8, under a table of 2048 blocks: 19.4 us, 11.5 now;
  // decode of 16 x U[500, 2000] tokens, Hq32 / Hkv4, called with a bound of 32768: 96 us, 34.5 now).
  // The sequences are turned by one from split to split, so that one long sequence beside short
  // ones does not keep to half of the XCDs either.
  const int split = blockIdx.z;
  const int b = (blockIdx.y + blockIdx.z) % gridDim.y;
  const int kvh = blockIdx.x % Hkv;
  const int tile = blockIdx.x / Hkv;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15;  // packed query row of the tile; operand row of K and V
  const int g = lane >> 4;    // k group of the operands

  const SeqSplit sq = seq_split<UK>(a, b);
  if (sq.skip) {
    if (sq.flags && tid == 0) atomicOr(a.err, sq.flags);
    return;
  }
  const int rows = min(sq.chunk, a.max_rows) * G;
  const int row0 = tile * TILE;
  if (row0 >= rows || split >= max(sq.n_splits, 1)) return;
  if (sq.units == 0) {  // empty context: zero output (weighted sum of nothing)
    for (int i = tid; i < min(TILE, rows - row0) * D; i += 64 * WAVES) {
      const int r = row0 + i / D;
      a.out[((size_t)(sq.c0 + r / G) * a.q_heads + kvh * G + r % G) * D + i % D] = 0;
    }
    return;
  }

  // this lane's query row (columns past the last repeat it and are never stored)
  const int my_row = min(row0 + col, rows - 1);
  const int my_tok = my_row / G;
  const int first_pos = sq.ctx - sq.chunk;
  const int my_pos = first_pos + my_tok;
  const int my_lo = a.window > 0 ? max(0, my_pos - a.window + 1) : 0;
  // positions of the tile's first and last row bound what it attends
  const int tile_pos0 = first_pos + row0 / G;
  const int tile_pos1 = first_pos + (min(row0 + TILE, rows) - 1) / G;
  const int tile_lo0 = a.window > 0 ? max(0, tile_pos0 - a.window + 1) : 0;

  // units of this split that the tile attends, dealt to the wavefronts in turn
  const int ub = max(sq.unit0 + split * sq.per_split, tile_lo0 / UK);
  const int ue = min(min(sq.unit0 + (split + 1) * sq.per_split, sq.unit0 + sq.units), tile_pos1 / UK + 1);
  const int n = max(0, (ue - ub - wave + WAVES - 1) / WAVES);

  // ---- Q^T operand: k-step ks, this lane's 8 dims of its row ----
  // 16-bit: dims 32 ks + 8 g; 8-bit: a 16-byte K load spans two k-steps, dims
  // 64 (ks / 2) + 16 g + 8 (ks % 2)
  u32x4_t qb[KS];
  {
    const uint16_t *qr = a.q + ((size_t)(sq.c0 + my_tok) * a.q_heads + kvh * G + my_row % G) * D;
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
      qb[ks] = *reinterpret_cast<const u32x4_t *>(qr + (Q8 ? 64 * (ks >> 1) + 16 * g + 8 * (ks & 1) : 32 * ks + 8 * g));
  }
  float c = a.scale_log2e, c_nat = a.scale;
  if constexpr (OP == kF16) {  // the row's q scaled into fp16 (lanes col + 16 g hold its dims)
    uint32_t w[4 * KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int e = 0; e < 4; e++) w[4 * ks + e] = qb[ks][e];
    int mx = bf16_absmax_bits<4 * KS>(w);
    mx = max(mx, __float_as_int(xor16_other(__int_as_float(mx), lane)));
    mx = max(mx, __float_as_int(xor32_other(__int_as_float(mx), lane)));
    const F16Scaling sc = f16_scaling(mx);
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int e = 0; e < 4; e++) qb[ks][e] = bf16x2_to_f16x2(w[4 * ks + e], sc.inv);
    c *= sc.step;
    c_nat *= sc.step;
  }

  f32x4_t oacc[ND];
#pragma unroll
  for (int d = 0; d < ND; d++) oacc[d] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  float m_run = -INFINITY, l_run = 0.0f;
  bool bad = false, nonfinite = false;
  const bool zero_bad = a.zero_bad != 0;

  const int32_t *table = a.tables + (size_t)b * a.max_blocks;
  const int gk = col >> 2;  // lane group whose scores this lane's K operand row feeds
  struct Entries {
    int k[NS], v[NS];
  };
  // block (of the unit) that holds this lane's K rows / V columns, entry i
  auto blk_of = [&](int grp, int i) __attribute__((always_inline)) { return 2 * i + (grp >> 1); };
  auto fetch = [&](int u, Entries &e) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NS; i++) {
      e.k[i] = table[(uint32_t)(u * NT + blk_of(gk, i)) % (uint32_t)a.max_blocks];
      e.v[i] = table[(uint32_t)(u * NT + blk_of(g, i)) % (uint32_t)a.max_blocks];
    }
  };
  // pool block of an entry: block 0 where the unit's block is not attended or lies
  // outside the pool (miss: attended but outside)
  auto resolve = [&](int u, int grp, int i, int e, bool &miss) __attribute__((always_inline)) -> size_t {
    const int pos = (u * NT + blk_of(grp, i)) * BT;
    const bool needed = pos < sq.ctx && pos + BT > tile_lo0;
    const bool ok = e >= 0 && (int64_t)e < a.pool.n_blocks;
    miss = needed && !ok;
    return (size_t)(needed && ok ? e : 0) * Hkv + kvh;
  };
  // byte offsets of this lane's operand rows in a block's K (tile 0) and V (output tile 0)
  const uint32_t k_lane = (8 * (gk & 1) + (col & 3)) * D * ES + 16 * g;
  const uint32_t v_lane = (col * BT + 8 * (g & 1)) * ES;
  u32x4_t kr[NT][KL];
  typedef __attribute__((ext_vector_type(2 * ES))) uint32_t vword_t;  // 8 keys of a V^T row
  vword_t vr[NS][ND];
  // int8: the (K, V) fp16 scale pairs of this lane's 8 keys; fp8: the f32 scales of its block
  u32x4_t sreg[NS][2] = {};
  auto load_k = [&](int u, const Entries &e) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NS; i++) {
      bool miss;
      const size_t bh = resolve(u, gk, i, e.k[i], miss);
      const char *kb = reinterpret_cast<const char *>(a.pool.k) + bh * (BT * D * ES) + k_lane;
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int x = 0; x < KL; x++) kr[2 * i + j][x] = ld16(kb + 4 * j * D * ES + 64 * x);
    }
  };
  auto load_v = [&](int u, const Entries &e, uint32_t &miss) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NS; i++) {
      bool ms;
      const size_t bh = resolve(u, g, i, e.v[i], ms);
      miss = (miss & ~(1u << i)) | (ms ? 1u << i : 0u);
      const char *vb = reinterpret_cast<const char *>(a.pool.v) + bh * (BT * D * ES) + v_lane;
      if constexpr (FMT == kInt8) {
        const u32x4_t *sp = reinterpret_cast<const u32x4_t *>(reinterpret_cast<const uint16_t *>(a.pool.k_scales) +
                                                              int8_scale_index(bh, 8 * (g & 1), BT));
        sreg[i][0] = sp[0];
        sreg[i][1] = sp[1];
      }
      if constexpr (FMT == kFp8) {
        const uint2 t = *reinterpret_cast<const uint2 *>(reinterpret_cast<const uint32_t *>(a.pool.k_scales) +
                                                         fp8_scale_index(bh));
        sreg[i][0][0] = t.x;
        sreg[i][0][1] = t.y;
      }
#pragma unroll
      for (int d = 0; d < ND; d++)
        vr[i][d] = __builtin_nontemporal_load(reinterpret_cast<const vword_t *>(vb + 16 * d * BT * ES));
    }
  };

  // scores of the unit in kr (raw, over this lane's keys: key_of below)
  float sc[4 * NT];
  auto scores = [&]() __attribute__((always_inline)) {
    f32x4_t acc[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) acc[j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int x = 0; x < KL; x++)
#pragma unroll
      for (int j = 0; j < NT; j++) {
        if constexpr (Q8) {
          acc[j] = mfma16<OP>(codes8<FMT>(kr[j][x][0], kr[j][x][1]), qb[2 * x], acc[j]);
          acc[j] = mfma16<OP>(codes8<FMT>(kr[j][x][2], kr[j][x][3]), qb[2 * x + 1], acc[j]);
        } else if constexpr (WIDE16) {
          u32x4_t hi, lo;
          f16x8_to_bf16(kr[j][x], hi, lo);
          acc[j] = mfma16<OP>(hi, qb[x], acc[j]);
          acc[j] = mfma16<OP>(lo, qb[x], acc[j]);
        } else {
          acc[j] = mfma16<OP>(kr[j][x], qb[x], acc[j]);
        }
      }
#pragma unroll
    for (int x = 0; x < 4 * NT; x++) sc[x] = acc[x >> 2][x & 3];
  };
  // position of score x (0 .. 4 NT - 1) of this lane in the unit
  auto key_of = [&](int x) __attribute__((always_inline)) {
    return 32 * (x >> 3) + 8 * g + (x & 7);
  };

  // f32 scale (0: K, 1: V) of score x's key
  auto scale_of = [&](int x, int tensor) __attribute__((always_inline)) {
    if constexpr (FMT == kInt8) {
      const uint32_t pair = sreg[x >> 3][(x >> 2) & 1][x & 3];
      return f16_bits_to_f32(tensor ? pair >> 16 : pair & 0xffffu);
    } else {
      return __uint_as_float(sreg[x >> 3][0][tensor]);
    }
  };

  u32x4_t pb[NS][PARTS];
  auto softmax = [&](int u, uint32_t vmiss) __attribute__((always_inline)) {
    const int base = u * UK;
    float tmax = -INFINITY;
#pragma unroll
    for (int x = 0; x < 4 * NT; x++) {
      float s = sc[x];
      if constexpr (Q8) s *= scale_of(x, 0);
      sc[x] = s;
    }
#pragma unroll
    for (int x = 0; x < 4 * NT; x++) {
      const int p = base + key_of(x);
      const bool miss = vmiss & (1u << (x >> 3));
      const bool on = (p >= my_lo) & (p <= my_pos) & (!miss | zero_bad);
      const float s = miss ? 0.0f : sc[x];
      nonfinite |= on & !(fabsf(s * c_nat) < INFINITY);
      sc[x] = on ? s * c : -INFINITY;
      tmax = fmaxf(tmax, sc[x]);
    }
    tmax = fmaxf(tmax, xor16_other(tmax, lane));
    tmax = fmaxf(tmax, xor32_other(tmax, lane));
    // lazy rescale: the reference max moves only when a row's max grows by more than 8
    const bool grow = tmax > m_run + 8.0f;  // true on a row's first finite unit
    if (__any(grow)) {
      const float nm = grow ? tmax : m_run;
      const float alpha = grow ? fast_exp2(m_run - nm) : 1.0f;
      m_run = nm;
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < ND; d++) oacc[d] *= alpha;
    }
    const float mref = (m_run == -INFINITY ? 0.0f : m_run) - BIAS;
#pragma unroll
    for (int s = 0; s < NS; s++) {
      float p[8];
#pragma unroll
      for (int x = 0; x < 8; x++) {
        p[x] = fast_exp2(sc[8 * s + x] - mref);
        if constexpr (PARTS > 1 || Q8) l_run += p[x];
        // the scale of a slot that is not attended may be anything
        if constexpr (Q8)
          p[x] = ((sc[8 * s + x] == -INFINITY) | ((vmiss >> s & 1u) != 0)) ? 0.0f : p[x] * scale_of(8 * s + x, 1);
      }
      // 16-bit values may be infinite, and such a value times the terms of a positive weight has
      // to be that infinity: the terms are cut, not rounded, so that none is negative, and none
      // is zero where the weight is not.
      constexpr bool CUT = PARTS > 1 && !Q8;
      float least[CUT ? 8 : 1];
      if constexpr (CUT) {
#pragma unroll
        for (int x = 0; x < 8; x++) least[x] = p[x] > 0.0f ? (OP == kF16 ? 0x1p-24f : 0x1p-120f) : 0.0f;
      }
#pragma unroll
      for (int q = 0; q < PARTS; q++) {
#pragma unroll
        for (int x = 0; x < 4; x++) {
          float &p0 = p[2 * x], &p1 = p[2 * x + 1];
          const uint32_t w = CUT && q + 1 < PARTS ? cut_16<OP>(p0, p1) : pack_16<OP>(p0, p1);
          pb[s][q][x] = w;
          if constexpr (PARTS == 1 && !Q8) l_run = dot2_ones_16<OP>(w, l_run);
          if (q + 1 < PARTS) {  // the rest of the weight, exactly
            p0 -= OP == kF16 ? f16_bits_to_f32(w & 0xffffu) : bf16_lo(w);
            p1 -= OP == kF16 ? f16_bits_to_f32(w >> 16) : bf16_hi(w);
            if constexpr (CUT) {
              p0 = fmaxf(p0, least[2 * x]);
              p1 = fmaxf(p1, least[2 * x + 1]);
            }
          }
        }
      }
    }
  };
  auto accumulate = [&](int u, uint32_t vmiss) __attribute__((always_inline)) {
    const int base = u * UK;
    // V slots outside the attended positions may hold anything (0 * NaN is NaN)
    constexpr int PW = Q8 ? 4 : 2;  // elements per word
    vword_t vmask[NS];
#pragma unroll
    for (int i = 0; i < NS; i++) {
      const int p0 = base + 32 * i + 8 * g;
      const bool miss = vmiss & (1u << i);
#pragma unroll
      for (int w = 0; w < 2 * ES; w++) {
        uint32_t mask = 0;
#pragma unroll
        for (int e = 0; e < PW; e++) {
          const int p = p0 + PW * w + e;
          mask |= (!miss & (p >= tile_lo0) & (p < sq.ctx)) ? (Q8 ? 0xffu : 0xffffu) << (32 / PW * e) : 0u;
        }
        vmask[i][w] = mask;
      }
    }
#pragma unroll
    for (int s = 0; s < NS; s++) {
      // output tiles whose independent products hide each other's latency
      constexpr int GRP = WIDE16 ? 2 : 4;
#pragma unroll
      for (int d0 = 0; d0 < ND; d0 += GRP) {
        u32x4_t va[GRP], vl[GRP];
#pragma unroll
        for (int d = 0; d < GRP; d++) {
          const vword_t v = vr[s][d0 + d] & vmask[s];
          if constexpr (Q8) va[d] = codes8<FMT>(v[0], v[1]);
          else if constexpr (WIDE16) f16x8_to_bf16(v, va[d], vl[d]);
          else va[d] = v;
        }
#pragma unroll
        for (int q = 0; q < PARTS; q++) {
#pragma unroll
          for (int d = 0; d < GRP; d++) oacc[d0 + d] = mfma16<OP>(va[d], pb[s][q], oacc[d0 + d]);
          if constexpr (WIDE16) {
#pragma unroll
            for (int d = 0; d < GRP; d++) oacc[d0 + d] = mfma16<OP>(vl[d], pb[s][q], oacc[d0 + d]);
          }
        }
      }
    }
  };

  if (n > 0) {
    Entries e;
    uint32_t vmiss = 0;
    int u = ub + wave;
    fetch(u, e);
    load_k(u, e);
    __builtin_amdgcn_sched_barrier(0);  // K before V, as in the loop
    load_v(u, e, vmiss);
    fetch(n > 1 ? u + WAVES : u, e);
    asm volatile("");  // keeps the compiler from merging these loads with the loop's
    // The last unit is peeled off: loads under a condition would make the compiler
    // wait for every load in flight.
    for (int k = 0; k + 1 < n; k++) {
      bad |= vmiss != 0;
      scores();
      softmax(u, vmiss);
      // the next K loads into the registers this unit's scores have read, and nothing of
      // P V (which waits for V) moves above them
      __builtin_amdgcn_sched_barrier(0);
      load_k(u + WAVES, e);
      __builtin_amdgcn_sched_barrier(0);
      accumulate(u, vmiss);
      __builtin_amdgcn_sched_barrier(0);
      load_v(u + WAVES, e, vmiss);
      u += WAVES;
      fetch(k + 2 < n ? u + WAVES : u, e);
    }
    bad |= vmiss != 0;
    scores();
    softmax(u, vmiss);
    accumulate(u, vmiss);
  }
  if (__any(bad) && lane == 0) atomicOr(a.err, kErrBadBlock);
  if (a.flag_nonfinite && __any(nonfinite) && lane == 0) atomicOr(a.err, kErrNonFinite);

  // ---- merge the four wavefronts ----
  __shared__ __attribute__((aligned(16))) float s_o[WAVES][TILE][D];
  __shared__ float s_m[WAVES][TILE], s_l[WAVES][TILE];
  l_run += xor16_other(l_run, lane);
  l_run += xor32_other(l_run, lane);
  if (g == 0) {
    s_m[wave][col] = m_run - BIAS;
    s_l[wave][col] = l_run;
  }
#pragma unroll
  for (int d = 0; d < ND; d++) *reinterpret_cast<f32x4_t *>(&s_o[wave][col][16 * d + 4 * g]) = oacc[d];
  __syncthreads();
  const int live = min(TILE, rows - row0);
  for (int i = tid; i < live * (D / 4); i += 64 * WAVES) {
    const int r = i / (D / 4);
    const int d = 4 * (i % (D / 4));
    float mm = s_m[0][r];
#pragma unroll
    for (int w = 1; w < WAVES; w++) mm = fmaxf(mm, s_m[w][r]);
    const float mref = mm == -INFINITY ? 0.0f : mm;
    float ll = 0.0f;
    f32x4_t oo = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
      const float f = fast_exp2(s_m[w][r] - mref);
      ll += s_l[w][r] * f;
      oo += *reinterpret_cast<const f32x4_t *>(&s_o[w][r][d]) * f;
    }
    const int tok = (row0 + r) / G;
    const int head = kvh * G + (row0 + r) % G;
    if (sq.n_splits == 1) {
      const float inv = row_inv(a, ll);
      const size_t o = ((size_t)(sq.c0 + tok) * a.q_heads + head) * D + d;
#pragma unroll
      for (int x = 0; x < 4; x++) a.out[o + x] = f32_to_bf16_rne(gated(oo[x] * inv, a.gate, o + x));
    } else {
      const size_t p = (((size_t)b * a.max_rows + tok) * a.q_heads + head) * a.max_splits + split;
      if (a.counters) {
        float2 *o = reinterpret_cast<float2 *>(&a.ws_o[p * D + d]);
        st_agent(o, make_float2(oo[0], oo[1]));
        st_agent(o + 1, make_float2(oo[2], oo[3]));
        if (d == 0) st_agent(&a.ws_ml[p], make_float2(mm, ll));
      } else {
        *reinterpret_cast<f32x4_t *>(&a.ws_o[p * D + d]) = oo;
        if (d == 0) a.ws_ml[p] = make_float2(mm, ll);
      }
    }
  }
  if (sq.n_splits <= 1 || !a.counters) return;
  // The last workgroup of the tile merges the splits.  One compute unit takes about 32 GB/s past
  // its L2, so many splits are first merged in groups, each by the last of its own workgroups,
  // into the place of the group's first split (8 tokens over 16000, head_dim 128: 64 splits at
  // once 31.4 us, in groups 22.7).
  int32_t *counters = &a.counters[((size_t)b * gridDim.x + blockIdx.x) * (1 + kRowsMaxSplits / kSplitGroup)];
  if (sq.n_splits <= kFlatSplits) {
    if (last_to_arrive(counters, sq.n_splits)) merge_splits<D, false>(a, sq, b, kvh, G, row0, live, 0, 1, sq.n_splits);
    return;
  }
  const int group = split / kSplitGroup;
  const int g0 = group * kSplitGroup;
  const int in_group = min(kSplitGroup, sq.n_splits - g0);
  if (!last_to_arrive(&counters[1 + group], in_group)) return;
  if (in_group > 1) merge_splits<D, true>(a, sq, b, kvh, G, row0, live, g0, 1, in_group);
  const int n_groups = (sq.n_splits + kSplitGroup - 1) / kSplitGroup;
  if (!last_to_arrive(counters, n_groups)) return;
  merge_splits<D, false>(a, sq, b, kvh, G, row0, live, 0, kSplitGroup, n_groups);
}

// Merge of the n <= N splits of one (query row, head): every partial row in flight at
// once, the (max, sum) pairs one per lane, split weights through v_readlane.
template <int D, int N>
__device__ __forceinline__ void rows_merge(const RowsArgs &a, size_t prow, size_t orow, int last, int d) {
  const size_t p0 = prow * a.max_splits;
  float o_sp[N];
#pragma unroll
  for (int i = 0; i < N; i++) o_sp[i] = a.ws_o[(p0 + min(i, last)) * D + d];
  const int li = d & 63;
  const float2 ml = a.ws_ml[p0 + min(li, last)];
  const float mx[1] = {li <= last ? ml.x : -INFINITY}, ly[1] = {ml.y};
  float f[1];
  const float ll = merge_weights<1>(mx, ly, li, f);
  float oo = 0.0f;
#pragma unroll
  for (int i = 0; i < N; i++)  // nothing of the places past the last (0 x infinity is NaN)
    oo += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f[0]), i)) * (i <= last ? o_sp[i] : 0.0f);
  const float inv = row_inv(a, ll);
  a.out[orow * D + d] = f32_to_bf16_rne(gated(oo * inv, a.gate, orow * D + d));
}

template <int D, int UK>
__global__ __launch_bounds__(D) void paged_rows_merge_kernel(const RowsArgs a) {
  const int b = blockIdx.y;
  const SeqSplit sq = seq_split<UK>(a, b);
  const int tok = blockIdx.x / a.q_heads;
  if (sq.skip || tok >= sq.chunk || sq.n_splits <= 1) return;
  const size_t prow = (size_t)b * a.max_rows * a.q_heads + blockIdx.x;  // row of the partials
  const size_t orow = (size_t)sq.c0 * a.q_heads + blockIdx.x;           // and of the output
  const int last = sq.n_splits - 1;
  const int d = threadIdx.x;
  if (last < 8) return rows_merge<D, 8>(a, prow, orow, last, d);
  if (last < 16) return rows_merge<D, 16>(a, prow, orow, last, d);
  if (last < 32) return rows_merge<D, 32>(a, prow, orow, last, d);
  return rows_merge<D, kRowsMaxSplits>(a, prow, orow, last, d);
}

template <int D, int FMT, int PARTS>
hipError_t launch_rows_t(const RowsArgs &a, hipStream_t s, void *hu, LaunchHook hook) {
  const unsigned tiles = (unsigned)(((long long)a.max_rows * (a.q_heads / a.pool.kv_heads) + TILE - 1) / TILE);
  if (hook) hook(hu, 0, s);
  hipLaunchKernelGGL((paged_rows_kernel<D, FMT, PARTS>), dim3(tiles * a.pool.kv_heads, a.num_seqs, a.max_splits),
                     dim3(64 * WAVES), 0, s, a);
  hipError_t e = hipGetLastError();
  if (hook) hook(hu, 1, s);
  if (e != hipSuccess || a.max_splits <= 1 || a.counters) return e;
  hipLaunchKernelGGL((paged_rows_merge_kernel<D, kUnitKeys<D>>), dim3(a.max_rows * a.q_heads, a.num_seqs), dim3(D), 0,
                     s, a);
  return hipGetLastError();
}

// 16-bit pools: PARTS by the caller's need.  The vector decode kernels keep a maximum per four
// tokens, whose weights are exact more often than under this kernel's one per unit: two terms
// keep a decode step's error below theirs (short contexts, against f64: bf16, vector 0.00174, one
// term 0.00184; fp16, 0.00165 and 0.00166).
template <int D, int FMT>
hipError_t launch_rows_16(const RowsArgs &a, bool exact_weights, hipStream_t s, void *hu, LaunchHook hook) {
  if (exact_weights) return launch_rows_t<D, FMT, 3>(a, s, hu, hook);
  if constexpr (D == kFastHeadDim)
    if (!a.chunk_starts) return launch_rows_t<D, FMT, 2>(a, s, hu, hook);
  return launch_rows_t<D, FMT, 1>(a, s, hu, hook);
}

template <int D>
hipError_t launch_rows_d(const RowsArgs &a, bool exact_weights, hipStream_t s, void *hu, LaunchHook hook) {
  switch (a.pool.format) {
    case kBf16:
      return launch_rows_16<D, kBf16>(a, exact_weights, s, hu, hook);
    case kF16:
      return launch_rows_16<D, kF16>(a, exact_weights, s, hu, hook);
    case kInt8:
      return launch_rows_t<D, kInt8, 3>(a, s, hu, hook);
    case kFp8:
      return launch_rows_t<D, kFp8, 3>(a, s, hu, hook);
  }
  return hipErrorInvalidValue;
}

}  // namespace

int rows_unit_keys(int head_dim) { return head_dim == 256 ? 32 : 64; }

hipError_t launch_rows(const RowsArgs &a, bool exact_weights, hipStream_t s, void *hu, LaunchHook hook) {
  if (a.max_splits < 1 || a.max_splits > kRowsMaxSplits || a.max_rows < 1) return hipErrorInvalidValue;
  return a.pool.head_dim == 256 ? launch_rows_d<256>(a, exact_weights, s, hu, hook)
                                : launch_rows_d<128>(a, exact_weights, s, hu, hook);
}

}  // namespace llh
