"""The packed-row kernel (rows.hip): decode steps at head_dim 128 / 256 outside the tuned
kernels' shapes and short prefill chunks, against the oracle's per-head loop (crates/llm-backend/src/core/
native_attention.rs:707-773) on the pool the GPU holds.

It keeps f32 softmax weights, so its outputs are held to more than the parity bar: the
bf16 rounding of the f32 result (2^-9 of the value; 2^-8 allowed) plus 2e-5 for the f32
sums (scores of a few units: 2^-24 x about 10 terms' error, times values up to 5)."""
import math

import numpy as np
import pytest

import llm_hip
import oracle
from helpers import from_dev_bf16, to_dev
from llm_hip import workloads
from test_gpu_decode import build_case, oracle_decode

pytestmark = pytest.mark.gpu

BT = 16
FMTS = {"bf16": llm_hip.KV_BF16, "f16": llm_hip.KV_F16, "int8": llm_hip.KV_INT8, "fp8": llm_hip.KV_FP8_E4M3}
# lengths at the edges of blocks, of units of 32 and 64 keys, of one and several splits
EDGES = [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 129, 255, 256, 257, 511, 700]


def assert_f32_weights(out, ref, what):
    g = oracle.bf16_to_f32(out.ravel())
    r = ref.ravel()
    bad = ~(np.abs(g - r) <= np.abs(r) * 2.0**-8 + 2e-5)
    assert not bad.any(), f"{what}: {bad.sum()} of {r.size}, worst {np.abs(g - r)[bad].max():.3e}"


def decode(ctx, pool, lens, tables, q, Hq, D, window, scale, gate=None, noalloc=False):
    import torch

    out = torch.full((len(lens) * Hq * D,), 0x7FC0, dtype=torch.int16, device="cuda")
    desc = ctx.decode_desc(to_dev(lens), to_dev(tables), Hq, int(lens.max()), window,
                           gate=None if gate is None else to_dev(gate))
    before = ctx.metrics()["generic_decode_calls"]
    (ctx.paged_decode_noalloc if noalloc else ctx.paged_decode)(pool, desc, to_dev(q), out, scale)
    torch.cuda.synchronize()
    assert ctx.metrics()["generic_decode_calls"] == before + 1
    return from_dev_bf16(out)


@pytest.mark.parametrize("window", [0, 1, 100])
@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("D,Hq,Hkv", [(256, 8, 4), (256, 20, 1), (256, 6, 2), (128, 12, 4), (128, 34, 2)])
def test_rows_decode(ctx, D, Hq, Hkv, fmt, window):
    """Groups of 2, 20 (two tiles), 3 and 17; every edge length, empty included."""
    lens = np.array(EDGES, np.int32)
    batch = workloads.paged_batch(lens, BT, 0.10, 7 + D + Hq)
    pool, q = build_case(ctx, batch, Hq, Hkv, FMTS[fmt], 50 + Hq, head_dim=D)
    scale = 1.0 / math.sqrt(D)
    out = decode(ctx, pool, lens, batch.tables, q, Hq, D, window, scale)
    assert ctx.device_errors() == 0, ctx.last_error()
    ref = oracle_decode(pool, batch, FMTS[fmt], Hq, Hkv, window, q, scale, head_dim=D)
    assert_f32_weights(out, ref, f"D{D} {Hq}/{Hkv} {fmt} W{window}")
    # the no-allocation entry gives the same bits from its own scratch
    assert np.array_equal(out, decode(ctx, pool, lens, batch.tables, q, Hq, D, window, scale, noalloc=True))


@pytest.mark.parametrize("fmt", ["int8", "fp8"])
def test_rows_decode_many_splits_and_gate(ctx, fmt):
    """The head_dim-256 group of 8 over quantised blocks, gated: one long sequence (the
    merge's 64 splits, several units per wavefront) beside short ones."""
    D, Hq, Hkv = 256, 16, 2
    lens = np.array([17000, 3, 4000], np.int32)
    batch = workloads.paged_batch(lens, BT, 0.10, 11)
    pool, q = build_case(ctx, batch, Hq, Hkv, FMTS[fmt], 12, head_dim=D)
    gate = oracle.normal_bf16(99, q.size)
    out = decode(ctx, pool, lens, batch.tables, q, Hq, D, 0, 0.0625, gate=gate)
    assert ctx.device_errors() == 0, ctx.last_error()
    ref = oracle_decode(pool, batch, FMTS[fmt], Hq, Hkv, 0, q, 0.0625, head_dim=D)
    g = oracle.bf16_to_f32(gate).astype(np.float64)
    assert_f32_weights(out, (ref.ravel() / (1.0 + np.exp(-g))).astype(np.float32), fmt)


def test_rows_decode_flags(ctx):
    """The reference-order kernel's flags: a block outside the pool scores 0 with a zero
    value, a non-finite score and a length beyond the call's bound are flagged."""
    D, Hq, Hkv = 256, 8, 4
    lens = np.array([40, 200], np.int32)
    batch = workloads.paged_batch(lens, BT, 0.10, 21)
    pool, q = build_case(ctx, batch, Hq, Hkv, llm_hip.KV_BF16, 22, head_dim=D)
    tables = batch.tables.copy()
    tables[1, 3] = batch.n_blocks + 4
    out = decode(ctx, pool, lens, tables, q, Hq, D, 0, 0.0625)
    assert ctx.device_errors() == llm_hip.ERR_FLAG_BAD_BLOCK
    assert np.array_equal(out, decode(ctx, pool, lens, tables, q, Hq, D, 0, 0.0625))
    ctx.device_errors()
    opool = oracle.Pool.from_raw(llm_hip.KV_BF16, BT, Hkv, D, batch.n_blocks, pool.raw())
    _, k, v = opool.gather_f32(batch.tables[1], 0, 200)
    k, v = (x.reshape(200, Hkv, D).astype(np.float64) for x in (k, v))
    k[48:64] = v[48:64] = 0.0
    qf = oracle.bf16_to_f32(q).reshape(2, Hq, D)[1].astype(np.float64)
    for h in range(Hq):
        s = k[:, h // 2] @ qf[h] * 0.0625
        p = np.exp(s - s.max())
        ref = (p / p.sum()) @ v[:, h // 2]
        assert_f32_weights(out.reshape(2, Hq, D)[1, h], ref.astype(np.float32), f"bad block, head {h}")
    qi = q.copy()
    qi.reshape(2, Hq, D)[1, 5, 7] = 0x7F80  # an infinite query element
    decode(ctx, pool, lens, batch.tables, qi, Hq, D, 0, 0.0625)
    assert ctx.device_errors() & llm_hip.ERR_FLAG_NON_FINITE
    import torch

    desc = ctx.decode_desc(to_dev(lens), to_dev(batch.tables), Hq, 100)  # 200 > 100
    o = torch.zeros(2 * Hq * D, dtype=torch.int16, device="cuda")
    ctx.paged_decode(pool, desc, to_dev(q), o, 0.0625)
    torch.cuda.synchronize()
    assert ctx.device_errors() == llm_hip.ERR_FLAG_TOO_MANY_SPLITS


@pytest.mark.parametrize("window", [0, 33])
@pytest.mark.parametrize("D,Hq,Hkv,fmt", [(128, 16, 8, "bf16"), (128, 8, 1, "f16"), (128, 6, 2, "int8"),
                                          (128, 8, 2, "fp8"), (256, 16, 2, "bf16"), (256, 8, 4, "f16"),
                                          (256, 16, 2, "int8"), (256, 12, 4, "fp8")])
def test_rows_prefill(ctx, opts, D, Hq, Hkv, fmt, window):
    """Short ragged chunks (an empty one included) over prefixes at unit and split edges: the
    packed-row kernel, the 128-row-tile kernel on the same call, and -- under graph capture,
    where no scratch may be taken -- the latter again; all against the oracle."""
    import torch

    from helpers import assert_parity

    # few keys (a window of 33) at head_dim 256: packed rows only below 32 row tiles
    chunk = [3, 0, 1, 2, 5] if D == 256 and window else [8, 0, 1, 13, 5]
    prefix = [0, 40, 2100, 243, 507]
    lens = np.array([p + c for p, c in zip(prefix, chunk)], np.int32)
    batch = workloads.paged_batch(lens, BT, 0.10, 31)
    pool, _ = build_case(ctx, batch, Hq, Hkv, FMTS[fmt], 32, head_dim=D)
    starts = np.concatenate([[0], np.cumsum(chunk)]).astype(np.int32)
    T = int(starts[-1])
    q = oracle.normal_bf16(35, T * Hq * D)
    gate = oracle.normal_bf16(36, T * Hq * D)
    scale = 1.0 / math.sqrt(D)
    keep = [to_dev(a) for a in (starts, batch.seq_lens, batch.tables, q, gate)]
    out = torch.zeros(T * Hq * D, dtype=torch.int16, device="cuda")
    desc = ctx.prefill_desc(keep[0], keep[1], keep[2], Hq, max(chunk), window, total_q_rows=T, gate=keep[4])
    opool = oracle.Pool.from_raw(FMTS[fmt], BT, Hkv, D, batch.n_blocks, pool.raw())
    st, ref = opool.prefill(Hq, starts, batch.seq_lens, batch.tables, window, q, scale, threads=16)
    assert st == oracle.OK
    ref = ref.ravel() / (1.0 + np.exp(-oracle.bf16_to_f32(gate).astype(np.float64)))
    stream = torch.cuda.Stream()
    before = ctx.route_calls()["rows_prefill"]
    with torch.cuda.stream(stream):
        ctx.paged_prefill(pool, desc, keep[3], out, scale, stream=stream)
    stream.synchronize()
    assert ctx.route_calls()["rows_prefill"] == before + 1
    rows = from_dev_bf16(out)
    assert_parity(rows, ref.astype(np.float32), what="packed rows")
    if D == 256 and fmt in ("int8", "fp8"):  # no tile kernel: packed rows always, f32 weights
        assert_f32_weights(rows, ref.astype(np.float32), "packed rows")
    opts(llm_hip.OPT_PREFILL_HEADS_PER_WG, 1)
    out.zero_()
    ctx.paged_prefill(pool, desc, keep[3], out, scale)
    torch.cuda.synchronize()
    rows_only = D == 256 and fmt in ("int8", "fp8")
    assert ctx.route_calls()["rows_prefill"] == before + 1 + rows_only
    tiles = from_dev_bf16(out)
    assert_parity(tiles, ref.astype(np.float32), what="128-row tiles")
    opts(llm_hip.OPT_PREFILL_HEADS_PER_WG, 0)
    bytes0 = ctx.metrics()["workspace_bytes"]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        ctx.paged_prefill(pool, desc, keep[3], out, scale, stream=torch.cuda.current_stream())
    assert ctx.metrics()["workspace_bytes"] == bytes0
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert_parity(from_dev_bf16(out), ref.astype(np.float32), what="captured")
    assert ctx.device_errors() == 0, ctx.last_error()
    ctx.release_stream(stream)


@pytest.mark.parametrize("fmt", FMTS)
def test_rows_decode_group_of_eight(ctx, opts, fmt):
    """Groups of eight at head_dim 128, which the planner gives to the packed-row kernel,
    against the vector kernels (forced) and the oracle: edge lengths, one long sequence,
    a window."""
    from helpers import assert_parity
    from test_gpu_decode import run_decode

    Hq, Hkv, D = 32, 4, 128
    lens = np.array(EDGES + [5000], np.int32)
    batch = workloads.paged_batch(lens, BT, 0.10, 61)
    pool, q = build_case(ctx, batch, Hq, Hkv, FMTS[fmt], 62, head_dim=D)
    for window in (0, 100):
        ref = oracle_decode(pool, batch, FMTS[fmt], Hq, Hkv, window, q, 0.088, head_dim=D)
        outs = {}
        for kernel in ("auto", "split", "stream"):
            opts(llm_hip.OPT_DECODE_KERNEL, kernel)
            before = ctx.route_calls()["rows_decode"]
            outs[kernel] = run_decode(ctx, pool, batch, q, Hq, window, 0.088)
            assert ctx.route_calls()["rows_decode"] - before == (kernel == "auto"), kernel
            assert_parity(outs[kernel], ref, what=f"{fmt} W{window} {kernel}")
            assert_parity(outs["auto"], oracle.bf16_to_f32(outs[kernel]), what=f"{fmt} W{window} rows, {kernel}")
    assert ctx.device_errors() == 0, ctx.last_error()


@pytest.mark.parametrize("fmt,tiles", [("bf16", 256), ("f16", 256), ("int8", 64), ("fp8", 64)])
def test_rows_decode_group_of_four_rule(ctx, fmt, tiles):
    """Groups of four at head_dim 128 take the packed-row kernel from `tiles` (sequence, kv head)
    pairs up and up to 512 attended tokens: one below and at either line, and a window of that
    length over longer contexts; each against the oracle."""
    from helpers import assert_parity
    from test_gpu_decode import run_decode

    Hq, Hkv, D = 32, 8, 128
    n = tiles // Hkv
    for seqs, longest, window, rows in ((n, 512, 0, 1), (n - 1, 512, 0, 0), (n, 513, 0, 0), (n, 800, 512, 1),
                                        (n, 800, 513, 0)):
        lens = np.resize(np.array(EDGES[:-2] + [longest], np.int32), seqs)
        lens[0] = longest
        batch = workloads.paged_batch(lens, BT, 0.10, 65)
        pool, q = build_case(ctx, batch, Hq, Hkv, FMTS[fmt], 66, head_dim=D)
        before = ctx.route_calls()["rows_decode"]
        out = run_decode(ctx, pool, batch, q, Hq, window, 0.088)
        what = f"{fmt} {seqs} x {longest} W{window}"
        assert ctx.route_calls()["rows_decode"] - before == rows, what
        assert_parity(out, oracle_decode(pool, batch, FMTS[fmt], Hq, Hkv, window, q, 0.088, head_dim=D), what=what)
    assert ctx.device_errors() == 0, ctx.last_error()


def test_rows_decode_no_weight_as_the_vector_kernels(ctx, opts):
    """Every score of a group of eight -inf (q . k overflows), or +inf: NaN rows from the
    packed-row kernel and the vector kernel alike, split or not; the other heads' rows stay."""
    import torch

    Hq, Hkv, D = 32, 4, 128
    lens = np.array([20, 700, 3000, 90, 40], np.int32)
    batch = workloads.paged_batch(lens, BT, 0.0, 71)
    pool = ctx.pool(llm_hip.KV_BF16, BT, Hkv, D, batch.n_blocks)
    ids = torch.arange(batch.n_blocks, dtype=torch.int32, device="cuda")
    k = torch.ones(batch.n_blocks, BT, Hkv, D, dtype=torch.bfloat16, device="cuda")
    ctx.write_blocks(pool, ids, k.view(torch.int16), k.view(torch.int16))
    q = torch.full((lens.size, Hq, D), 0.5, dtype=torch.bfloat16, device="cuda")
    q[:, 3] = -3e38  # 128 of them: beyond f32
    q[:, 17] = 3e38
    outs = {}
    desc = ctx.decode_desc(to_dev(lens), to_dev(batch.tables), Hq, int(lens.max()))
    for kernel in ("auto", "split"):
        opts(llm_hip.OPT_DECODE_KERNEL, kernel)
        out = torch.zeros(lens.size, Hq, D, dtype=torch.bfloat16, device="cuda")
        ctx.paged_decode(pool, desc, q.view(torch.int16), out.view(torch.int16), 0.088)
        torch.cuda.synchronize()
        outs[kernel] = out.cpu()
    nan = torch.zeros(lens.size, Hq, D, dtype=torch.bool)
    nan[:, [3, 17]] = True
    for kernel, out in outs.items():
        assert torch.equal(out.isnan(), nan), kernel
        assert (out[~nan] == 1).all(), kernel
    assert ctx.device_errors() == 0, ctx.last_error()


@pytest.mark.parametrize("window", [0, 1500])
@pytest.mark.parametrize("D,Hq,Hkv,fmt,chunk,prefix", [
    (128, 32, 4, "bf16", [300, 0, 130, 1], [1500, 10, 900, 2000]),   # all heads packed, cut; ragged
    (128, 6, 2, "f16", [700], [800]),                                # odd group, cut
    (128, 16, 2, "int8", [200, 200], [1300, 1300]),
    (256, 16, 2, "bf16", [150, 90], [1500, 30]),                     # one sequence too short to cut
    (256, 8, 4, "f16", [400], [1000]),
])
def test_prefill_cut_items(ctx, opts, D, Hq, Hkv, fmt, chunk, prefix, window):
    """Prefill calls that fill less than half the chip cut their items' keys into pieces:
    sampled rows against the oracle, and every row against the same call under capture,
    where items stay whole."""
    import torch

    from helpers import assert_parity

    opts(llm_hip.OPT_PREFILL_HEADS_PER_WG, 2)
    lens = np.array([p + c for p, c in zip(prefix, chunk)], np.int32)
    batch = workloads.paged_batch(lens, BT, 0.10, 71)
    pool, _ = build_case(ctx, batch, Hq, Hkv, FMTS[fmt], 72, head_dim=D)
    starts = np.concatenate([[0], np.cumsum(chunk)]).astype(np.int32)
    T = int(starts[-1])
    q = oracle.normal_bf16(75, T * Hq * D)
    scale = 1.0 / math.sqrt(D)
    keep = [to_dev(a) for a in (starts, batch.seq_lens, batch.tables, q)]
    out = torch.zeros(T * Hq * D, dtype=torch.int16, device="cuda")
    desc = ctx.prefill_desc(keep[0], keep[1], keep[2], Hq, max(chunk), window, total_q_rows=T)
    stream = torch.cuda.Stream()
    before = ctx.route_calls()["cut_prefill"]
    ctx.paged_prefill(pool, desc, keep[3], out, scale, stream=stream)
    stream.synchronize()
    assert ctx.route_calls()["cut_prefill"] == before + 1
    cut = from_dev_bf16(out)
    assert ctx.metrics()["workspace_bytes"] > 0
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        ctx.paged_prefill(pool, desc, keep[3], out, scale, stream=torch.cuda.current_stream())
    out.zero_()
    graph.replay()
    torch.cuda.synchronize()
    whole = from_dev_bf16(out)
    assert_parity(cut, oracle.bf16_to_f32(whole), what="cut against whole")
    assert not np.array_equal(cut, whole), "nothing was cut"
    opool = oracle.Pool.from_raw(FMTS[fmt], BT, Hkv, D, batch.n_blocks, pool.raw())
    qr = q.reshape(T, Hq * D)
    rows = sorted({r for b in range(len(chunk)) for r in (starts[b], starts[b] + 17, starts[b + 1] - 1)
                   if starts[b] <= r < starts[b + 1]})
    for r in rows:
        b = int(np.searchsorted(starts, r, side="right") - 1)
        n = np.array([prefix[b] + r - starts[b] + 1], np.int32)
        st, ref = opool.decode(Hq, n, batch.tables[b:b + 1], window, qr[r], scale, threads=16)
        assert st == oracle.OK
        assert_parity(cut.reshape(T, Hq * D)[r], ref, what=f"row {r}")
    assert ctx.device_errors() == 0, ctx.last_error()
    ctx.release_stream(stream)


def prefill_call(ctx, fmt, D, Hq, Hkv, chunk, prefix, seed, max_chunk=None, table_blocks=None):
    """(batch, pool, q, out, desc) of a ragged prefill call on the device; table_blocks: row
    width of the block tables (default: the longest context's)."""
    import torch

    lens = np.array([p + c for p, c in zip(prefix, chunk)], np.int32)
    batch = workloads.paged_batch(lens, BT, 0.10, seed)
    pool, _ = build_case(ctx, batch, Hq, Hkv, fmt, seed + 1, head_dim=D)
    tables = batch.tables
    if table_blocks is not None:
        tables = np.full((lens.size, table_blocks), -1, np.int32)
        tables[:, :batch.tables.shape[1]] = batch.tables
    starts = np.concatenate([[0], np.cumsum(chunk)]).astype(np.int32)
    T = int(starts[-1])
    q = to_dev(oracle.normal_bf16(seed + 2, T * Hq * D))
    desc = ctx.prefill_desc(to_dev(starts), to_dev(batch.seq_lens), to_dev(tables), Hq, max_chunk or max(chunk),
                            total_q_rows=T)
    return batch, pool, q, torch.zeros_like(q), desc


@pytest.mark.parametrize("D,Hq,Hkv,n,chunk", [(128, 32, 4, 32, 481), (256, 16, 2, 64, 449)])
def test_prefill_scratch_is_bounded_and_its_own(ctx, opts, D, Hq, Hkv, n, chunk):
    """One long chunk beside many single tokens, cut into pieces, with a tight and a loose bound on
    the chunks, between replays of a decode captured on the same stream: the decode's workspace stays
    where it is, and the prefill's scratch is made once, a fixed number of rows per compute unit."""
    import torch

    from helpers import assert_parity

    stream = torch.cuda.Stream()
    lens = np.array([3000, 70, 900], np.int32)
    batch = workloads.paged_batch(lens, BT, 0.10, 101)
    pool, q = build_case(ctx, batch, 16, 8, llm_hip.KV_BF16, 102)
    d_q = to_dev(q)
    d_out = torch.zeros_like(d_q)
    desc = ctx.decode_desc(to_dev(lens), to_dev(batch.tables), 16, 3000)
    ctx.paged_decode(pool, desc, d_q, d_out, 0.088, stream=stream)
    stream.synchronize()
    want = d_out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        ctx.paged_decode(pool, desc, d_q, d_out, 0.088, stream=torch.cuda.current_stream())

    def replay():
        d_out.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        stream.synchronize()
        assert torch.equal(d_out, want)

    replay()
    m0 = ctx.metrics()
    chunks = [1] * n
    chunks[n // 2] = chunk
    outs, used = [], []
    for max_chunk in (chunk, 4096):
        _, ppool, pq, pout, pdesc = prefill_call(ctx, llm_hip.KV_BF16, D, Hq, Hkv, chunks, [2100] * n, 103, max_chunk)
        ctx.paged_prefill(ppool, pdesc, pq, pout, 0.088, stream=stream)
        stream.synchronize()
        replay()
        outs.append(pout.clone())
        used.append(ctx.metrics()["workspace_bytes"] - m0["workspace_bytes"])
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert 0 < used[0] <= cus * (2 * 256 * 130 * 4 + 2 * 16 * 258 * 4) and used[1] == used[0], used
    assert torch.equal(*outs)
    g2 = torch.cuda.CUDAGraph()  # under capture the items stay whole
    with torch.cuda.graph(g2, stream=stream):
        ctx.paged_prefill(ppool, pdesc, pq, pout, 0.088, stream=torch.cuda.current_stream())
    pout.zero_()
    g2.replay()
    torch.cuda.synchronize()
    assert_parity(from_dev_bf16(outs[0]), oracle.bf16_to_f32(from_dev_bf16(pout)), what="cut against whole")
    assert not torch.equal(outs[0], pout), "nothing was cut"
    replay()
    m1 = ctx.metrics()
    assert m1["device_errors"] == m0["device_errors"] and ctx.device_errors() == 0, ctx.last_error()
    ctx.release_stream(stream)
    assert ctx.metrics()["workspace_bytes"] < m1["workspace_bytes"] - used[0] + 1


# groups that the packed-row kernel serves in place of the reference-order kernel (f32 weights),
# and of the vector kernels (8 and 4 at head_dim 128); sequences enough for the rules
ROW_GROUPS = [(256, 8, 4, 2), (128, 12, 4, 2), (128, 32, 4, 5), (128, 32, 8, 32)]


def one_pool(ctx, fmt, D, Hkv, k, v):
    """A pool whose blocks 0 .. hold the rows k, v ([n][Hkv][D] f32, exact in bf16), whole blocks."""
    n = k.shape[0] // BT
    pool = ctx.pool(fmt, BT, Hkv, D, n)
    rows = [to_dev(oracle.f32_to_bf16(x.astype(np.float32).ravel())) for x in (k, v)]
    ctx.write_blocks(pool, to_dev(np.arange(n, dtype=np.int32)), *rows)
    return pool


@pytest.mark.parametrize("fmt", ["bf16", "f16"])
@pytest.mark.parametrize("D,Hq,Hkv,seqs", ROW_GROUPS[:2])
def test_rows_decode_small_weights_and_query_range(ctx, D, Hq, Hkv, seqs, fmt):
    """One key of weight 1 and value 0 before a tail of weights near 2^-26 whose values are the
    output, and a query whose deciding element is 2^-44 of its largest (which meets zeros): both
    are far below fp16's smallest step, none of f32's.  Against f64: 2^-8 of the value (the
    output's bf16 rounding is 2^-9, weights of 16 bits and f32 sums far less)."""
    import torch

    L = 496
    k, v = np.zeros((L, Hkv, D)), np.ones((L, Hkv, D))
    k[0, :, 0] = 1.0
    k[2::2, :, 1] = 2.0**15
    v[0] = 0.0
    v[1::2, :, D // 2:] = 0.0  # the second half of the dims tells the even keys from the odd
    q = np.zeros((seqs, Hq, D))
    q[:, :, 0] = 18.0 * 2.0**-20
    q[:, :, 1] = 2.0**-34 * 133 / 128
    q[:, :, 2] = 2.0**10
    pool = one_pool(ctx, FMTS[fmt], D, Hkv, k, v)
    lens = np.full(seqs, L, np.int32)
    tables = np.tile(np.arange(L // BT, dtype=np.int32), (seqs, 1))
    out = torch.zeros(seqs * Hq * D, dtype=torch.int16, device="cuda")
    desc = ctx.decode_desc(to_dev(lens), to_dev(tables), Hq, L)
    before = ctx.route_calls()["rows_decode"]
    ctx.paged_decode(pool, desc, to_dev(oracle.f32_to_bf16(q.astype(np.float32).ravel())), out, 2.0**20)
    torch.cuda.synchronize()
    assert ctx.route_calls()["rows_decode"] == before + 1
    w = np.exp((k[:, 0] @ q[0, 0]) * 2.0**20 - 18.0)
    ref = (w / w.sum()) @ v[:, 0]
    got = oracle.bf16_to_f32(from_dev_bf16(out)).reshape(-1, D)
    assert 0 < ref.min() < ref.max() < 1e-4
    assert (np.abs(got - ref) <= ref * 2.0**-8).all(), (got[0, [0, -1]], ref[[0, -1]])
    assert ctx.device_errors() == 0, ctx.last_error()


@pytest.mark.parametrize("fmt", ["bf16", "f16"])
@pytest.mark.parametrize("D,Hq,Hkv,seqs", ROW_GROUPS[2:])
def test_rows_decode_error_is_no_larger_than_the_vector_kernels(ctx, opts, D, Hq, Hkv, seqs, fmt):
    """Groups of eight and four at head_dim 128: the distance from f64 over ragged short contexts,
    on the packed-row kernel and on the vector kernel (forced) that it stands in for."""
    from test_gpu_decode import run_decode

    lens = np.random.default_rng(5).integers(50, 501, seqs).astype(np.int32)
    batch = workloads.paged_batch(lens, BT, 0.10, 111)
    pool, q = build_case(ctx, batch, Hq, Hkv, FMTS[fmt], 112, head_dim=D)
    opool = oracle.Pool.from_raw(FMTS[fmt], BT, Hkv, D, batch.n_blocks, pool.raw())
    qf = oracle.bf16_to_f32(q).reshape(seqs, Hkv, Hq // Hkv, D).astype(np.float64)
    ref = np.empty_like(qf)
    for b, n in enumerate(lens):
        k, v = (x.reshape(n, Hkv, D).astype(np.float64) for x in opool.gather_f32(batch.tables[b], 0, n)[1:])
        s = np.einsum("hgd,nhd->hgn", qf[b], k) * 0.088
        w = np.exp(s - s.max(-1, keepdims=True))
        ref[b] = np.einsum("hgn,nhd->hgd", w / w.sum(-1, keepdims=True), v)
    err = {}
    for kernel in ("auto", "split"):
        opts(llm_hip.OPT_DECODE_KERNEL, kernel)
        before = ctx.route_calls()["rows_decode"]
        out = oracle.bf16_to_f32(run_decode(ctx, pool, batch, q, Hq, 0, 0.088)).reshape(ref.shape)
        assert ctx.route_calls()["rows_decode"] - before == (kernel == "auto")
        err[kernel] = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    print(err)
    assert err["auto"] <= err["split"], err


@pytest.mark.parametrize("fmt", ["bf16", "f16"])
@pytest.mark.parametrize("D,Hq,Hkv,seqs,L", [(*g, 304) for g in ROW_GROUPS] + [(*g, 4000) for g in ROW_GROUPS[:2]])
def test_rows_decode_infinite_values(ctx, opts, D, Hq, Hkv, seqs, L, fmt):
    """An infinite value row element gives that infinity in its dim, two of opposite signs NaN, and
    the other dims their sums, as from the reference-order kernel, in the last of several splits
    too (where the vector kernels' merge gives NaN)."""
    import torch

    rng = np.random.default_rng(7)
    k, v = (oracle.bf16_to_f32(oracle.f32_to_bf16(rng.standard_normal(L * Hkv * D).astype(np.float32)))
            .reshape(L, Hkv, D) for _ in range(2))
    v[70, :, 5], v[L - 9, :, 9], v[30, :, 11], v[L - 14, :, 11] = np.inf, -np.inf, np.inf, -np.inf
    pool = one_pool(ctx, FMTS[fmt], D, Hkv, k, v)
    lens = np.full(seqs, L, np.int32)
    tables = np.tile(np.arange(L // BT, dtype=np.int32), (seqs, 1))
    q = to_dev(oracle.f32_to_bf16(rng.standard_normal(seqs * Hq * D).astype(np.float32)))
    desc = ctx.decode_desc(to_dev(lens), to_dev(tables), Hq, L)
    outs = []
    for option in (None, (llm_hip.OPT_FORCE_GENERIC, 1) if D == 256 or Hq == 12 else (llm_hip.OPT_DECODE_KERNEL, 1)):
        if option:
            opts(*option)
        before = ctx.route_calls()["rows_decode"]
        out = torch.zeros(seqs, Hq, D, dtype=torch.bfloat16, device="cuda")
        ctx.paged_decode(pool, desc, q, out.view(torch.int16), 0.05)
        torch.cuda.synchronize()
        assert ctx.route_calls()["rows_decode"] - before == (option is None)
        outs.append(out.float().cpu())
    rows, other = outs
    assert (rows[..., 5] == math.inf).all() and (rows[..., 9] == -math.inf).all() and rows[..., 11].isnan().all()
    finite = [d for d in range(D) if d not in (5, 9, 11)]
    assert (rows[..., finite] - other[..., finite]).abs().max() <= 2e-2
    if D == 256 or Hq == 12:
        assert torch.equal(rows.isnan(), other.isnan()) and torch.equal(rows.isinf(), other.isinf())
    assert ctx.device_errors() == 0, ctx.last_error()


@pytest.mark.parametrize("D,Hq,Hkv,chunk,prefix,route", [
    (128, 16, 8, [8, 3], [2100, 40], "rows_prefill"),      # one sequence split, one not
    (128, 16, 8, [8, 3], [7000, 1600], "rows_prefill"),    # 28 splits, merged in groups, and 7
    (256, 8, 4, [5], [900], "rows_prefill"),
    (256, 8, 4, [5], [4000], "rows_prefill"),              # 32 splits (int8: as many)
    (256, 8, 4, [2], [3190], "rows_prefill"),              # 25 splits: a group of one
    (128, 32, 4, [300, 20], [1500, 1700], "cut_prefill"),
    (256, 16, 2, [150, 90], [1500, 30], "cut_prefill"),    # one sequence cut, one not
])
@pytest.mark.parametrize("fmt", ["bf16", "int8"])
def test_prefill_merges_in_its_launch_over_changing_inputs(ctx, D, Hq, Hkv, chunk, prefix, route, fmt):
    """Splits and pieces merged by the last workgroup to arrive: two pools in turn, a query each,
    back to back on one stream, so that the scratch always holds another call's partials; then the
    same calls in the opposite order.  Every output has the same bits both times, and the first
    ones meet the whole items of a captured call."""
    import torch

    from helpers import assert_parity

    if D == 256 and fmt == "int8":
        route = "rows_prefill"
    cases = [prefill_call(ctx, FMTS[fmt], D, Hq, Hkv, chunk, prefix, seed) for seed in (121, 131)]
    g = torch.Generator(device="cuda")
    g.manual_seed(122)
    q = torch.randn(60, cases[0][2].numel(), generator=g, device="cuda").to(torch.bfloat16).view(torch.int16)
    there, back = torch.zeros_like(q), torch.zeros_like(q)
    before = ctx.route_calls()[route]
    for out, order in ((there, range(len(q))), (back, reversed(range(len(q))))):
        for i in order:
            _, pool, _, _, desc = cases[i % 2]
            ctx.paged_prefill(pool, desc, q[i], out[i], 0.088)
    torch.cuda.synchronize()
    assert ctx.route_calls()[route] == before + 2 * len(q)
    assert torch.equal(there, back), int((there != back).sum())
    stream = torch.cuda.Stream()
    whole = torch.zeros_like(q[:2])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        for i in range(2):
            ctx.paged_prefill(cases[i][1], cases[i][4], q[i], whole[i], 0.088, stream=torch.cuda.current_stream())
    graph.replay()
    torch.cuda.synchronize()
    assert_parity(from_dev_bf16(there[:2]), oracle.bf16_to_f32(from_dev_bf16(whole)))
    assert ctx.device_errors() == 0, ctx.last_error()
    ctx.release_stream(stream)


@pytest.mark.parametrize("D,Hq,Hkv,fmt", [(128, 32, 4, "bf16"), (128, 6, 2, "f16"), (256, 16, 2, "bf16")])
@pytest.mark.parametrize("chunk,prefix", [([64] * 8, [256] * 8), ([300, 0, 130], [1900, 10, 900])])
def test_prefill_table_wider_than_the_contexts(ctx, opts, D, Hq, Hkv, fmt, chunk, prefix):
    """Block-table rows of 2048 blocks: whether items are cut, and how heads are packed where they
    are not, follows the contexts, so the bits are those of the exact table."""
    import torch

    opts(llm_hip.OPT_PREFILL_HEADS_PER_WG, 2)  # the tile kernels
    outs = []
    for width in (None, 2048):
        _, pool, q, out, desc = prefill_call(ctx, FMTS[fmt], D, Hq, Hkv, chunk, prefix, 141, table_blocks=width)
        before = ctx.route_calls()["cut_prefill"]
        ctx.paged_prefill(pool, desc, q, out, 0.088)
        torch.cuda.synchronize()
        assert ctx.route_calls()["cut_prefill"] - before == (width is not None or max(prefix) > 1000)
        outs.append(out)
    assert torch.equal(*outs)
    assert ctx.device_errors() == 0, ctx.last_error()


@pytest.mark.parametrize("fmt", ["bf16", "int8"])
@pytest.mark.parametrize("D,Hq,Hkv", [(128, 32, 4), (128, 12, 4), (256, 8, 4)])
def test_rows_decode_bound_far_above_the_lengths(ctx, D, Hq, Hkv, fmt):
    """A step called with the model's longest context as its bound (as a captured graph is), with and
    without a hint of the tokens, one long sequence among short and empty ones: as the oracle."""
    import torch

    from helpers import assert_parity

    lens = np.array(EDGES + [5000], np.int32)
    batch = workloads.paged_batch(lens, BT, 0.10, 161)
    pool, q = build_case(ctx, batch, Hq, Hkv, FMTS[fmt], 162, head_dim=D)
    tables = np.full((lens.size, 2048), -1, np.int32)
    tables[:, :batch.tables.shape[1]] = batch.tables
    ref = oracle_decode(pool, batch, FMTS[fmt], Hq, Hkv, 0, q, 0.088, head_dim=D)
    for hint in (0, int(lens.sum())):
        out = torch.full((q.size,), 0x7FC0, dtype=torch.int16, device="cuda")
        desc = ctx.decode_desc(to_dev(lens), to_dev(tables), Hq, 32768, total_tokens_hint=hint)
        before = ctx.route_calls()["rows_decode"]
        ctx.paged_decode(pool, desc, to_dev(q), out, 0.088)
        torch.cuda.synchronize()
        assert ctx.route_calls()["rows_decode"] == before + 1
        assert_parity(from_dev_bf16(out), ref, what=f"hint {hint}")
    assert ctx.device_errors() == 0, ctx.last_error()

