"""What the performance of this framework is measured on.

A case is one call that a serving program makes for one attention layer: a decode
step, a decode step that also appends the new token or projects the output, a prefill
chunk, the write of a prompt's blocks, or the host-side trait call.  Shapes are the
ones that the repository's workloads and tests use: Qwen3-like layers (16 or 32 query
heads over 8 or 4 kv heads, head_dim 128), Qwen3.6 full-attention layers (16 over 2,
head_dim 256, gated) and the 8-over-4 head_dim-256 layers of the tests.

Every case draws its pool from the seed alone: all blocks of the pool hold rows, the
block tables are a permutation of them, and sequences end inside their last block.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "kir-ai_amd"))

import llm_hip  # noqa: E402

BT = 16
FORMATS = {"bf16": llm_hip.KV_BF16, "f16": llm_hip.KV_F16, "int8": llm_hip.KV_INT8, "fp8": llm_hip.KV_FP8_E4M3}
ELEM = {"bf16": 2, "f16": 2, "int8": 1, "fp8": 1}
CHUNK = 2048  # blocks per generated piece

_context = []


def _ctx():
    """A serving program keeps one context for the process."""
    if not _context:
        _context.append(llm_hip.Context(0))
    return _context[0]


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one request, one token: the smallest call, where launches and latency count
        dict(name="decode_single", kind="decode", fmt="bf16", D=128, Hq=16, Hkv=8, B=1, len_lo=512, len_hi=512,
             lens_seed=1, window=0, gate=False),
        # a serving batch of ragged contexts, the benchmark's headline step
        dict(name="decode_ragged", kind="decode", fmt="bf16", D=128, Hq=16, Hkv=8, B=32, len_lo=256, len_hi=4096,
             lens_seed=2, window=0, gate=False),
        # append then attend in one call, gated, over the fp16 blocks of a Qwen3.6 layer
        dict(name="decode_append_gated", kind="append", fmt="f16", D=256, Hq=16, Hkv=2, B=12, len_lo=256, len_hi=4096,
             lens_seed=3, window=0, gate=True),
        # long contexts over int8 blocks: the largest traffic
        dict(name="decode_int8_long", kind="decode", fmt="int8", D=128, Hq=32, Hkv=8, B=64, len_lo=8192, len_hi=8192,
             lens_seed=4, window=0, gate=False),
        # the Qwen3.6 layer over quantised blocks
        dict(name="decode_fp8_d256", kind="decode", fmt="fp8", D=256, Hq=16, Hkv=2, B=16, len_lo=256, len_hi=4096,
             lens_seed=5, window=0, gate=True),
        # sliding window deep into long contexts, with the output projection
        dict(name="decode_window_project", kind="project", fmt="bf16", D=128, Hq=16, Hkv=8, B=4, len_lo=32768,
             len_hi=32768, lens_seed=6, window=4096, gate=False, rows=1024),
        # one request's prompt in the short chunks of the reference's driver, over a cached prefix
        dict(name="prefill_chunk8", kind="prefill", fmt="bf16", D=128, Hq=16, Hkv=8, B=1, prefix_lo=4099,
             prefix_hi=4099, chunk_lo=8, chunk_hi=8, lens_seed=7, window=0, gate=False),
        # a batch of prompt chunks over cached prefixes: the dense path
        dict(name="prefill_batch", kind="prefill", fmt="bf16", D=128, Hq=32, Hkv=4, B=8, prefix_lo=1536,
             prefix_hi=1536, chunk_lo=512, chunk_hi=512, lens_seed=8, window=0, gate=False),
        # a few ragged chunks of the gated Qwen3.6 layer
        dict(name="prefill_d256", kind="prefill", fmt="bf16", D=256, Hq=16, Hkv=2, B=3, prefix_lo=200, prefix_hi=1700,
             chunk_lo=100, chunk_hi=600, lens_seed=9, window=0, gate=True),
        # a prompt chunk of the same layer over int8 blocks
        dict(name="prefill_d256_int8", kind="prefill", fmt="int8", D=256, Hq=16, Hkv=2, B=2, prefix_lo=1024,
             prefix_hi=1024, chunk_lo=250, chunk_hi=250, lens_seed=10, window=0, gate=False),
        # quantise-on-write of a prompt chunk's blocks for that layer
        dict(name="write_int8_d256", kind="write", fmt="int8", D=256, Hkv=2, blocks=256),
        # the reference's synchronous per-layer call: host rows in, host rows out
        dict(name="trait_mix", kind="trait", fmt="bf16", D=128, Hq=16, Hkv=8, tokens=512, rows=500),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _fit(lo, hi, B, limit):
    """The length range cut so that a batch of the longest fits `limit` tokens."""
    hi = max(1, min(hi, limit // B))
    return min(lo, hi), hi


def draw(rng):
    kind = rng.choice(["decode", "decode", "append", "project", "prefill", "prefill", "write", "trait"])
    shapes = [(128, 16, 8), (128, 32, 8), (128, 32, 4), (256, 16, 2), (256, 16, 2), (256, 8, 4)]
    D, Hq, Hkv = rng.choice(shapes)
    fmt = rng.choice(["bf16", "bf16", "f16", "int8", "fp8"])
    seed = rng.randrange(1 << 30)
    if kind == "write":
        return dict(kind=kind, fmt=fmt, D=D, Hkv=Hkv, blocks=_log_int(rng, 1, 1024))
    if kind == "trait":
        tokens = 16 * _log_int(rng, 1, 256)
        return dict(kind=kind, fmt=rng.choice(["bf16", "int8"]), D=128, Hq=rng.choice([16, 32]), Hkv=8, tokens=tokens,
                    rows=rng.randint(max(1, tokens // 2), tokens))
    window = rng.choice([0, 0, 0, _log_int(rng, 64, 4096)])
    gate = D == 256 and rng.random() < 0.5
    if kind == "prefill":
        B = _log_int(rng, 1, 8)
        chunk = _log_int(rng, 8, 1024)
        p_hi = _log_int(rng, 16, 4096)
        chunk = max(1, min(chunk, 4096 // B))
        if D == 256 and fmt not in ("bf16", "f16"):
            chunk, p_hi = max(1, min(chunk, 512 // B)), min(p_hi, 1024)
        elif chunk * B > 512:
            p_hi = min(p_hi, 1024)
        return dict(kind=kind, fmt=fmt, D=D, Hq=Hq, Hkv=Hkv, B=B, prefix_lo=rng.choice([0, p_hi // 2, p_hi]),
                    prefix_hi=p_hi, chunk_lo=max(1, chunk // rng.choice([1, 2, 4])), chunk_hi=chunk, lens_seed=seed,
                    window=window, gate=gate)
    B = _log_int(rng, 1, 48)
    hi = _log_int(rng, 64, 16384)
    if kind == "append" and fmt == "fp8":
        fmt = "bf16"
    limit = (1 << (24 if kind == "append" else 28)) // (Hkv * D)
    if D == 256 and (fmt not in ("bf16", "f16") or Hq != 16):
        hi, limit = min(hi, 4096), min(limit, 32768)
    lo, hi = _fit(rng.choice([1, hi // 8 + 1, hi]), hi, B, limit)
    case = dict(kind=kind, fmt=fmt, D=D, Hq=Hq, Hkv=Hkv, B=B, len_lo=lo, len_hi=hi, lens_seed=seed, window=window,
                gate=gate)
    if kind == "project":
        case["rows"] = 128 * rng.randint(4, 32)
    return case


# ---------------------------------------------------------------------------
# geometry (from the case alone)
# ---------------------------------------------------------------------------
def _ints(seed, lo, hi, n, top=True):
    """n lengths in [lo, hi], the longest equal to hi."""
    v = np.random.Generator(np.random.PCG64(seed)).integers(lo, hi + 1, size=n)
    if top and n:
        v[n // 2] = hi
    return v.astype(np.int64)


def _lens(case):
    """Context lengths (the new tokens included) and the new tokens of each sequence."""
    if case["kind"] == "prefill":
        chunk = _ints(case["lens_seed"], case["chunk_lo"], case["chunk_hi"], case["B"])
        prefix = _ints(case["lens_seed"] + 1, case["prefix_lo"], case["prefix_hi"], case["B"])
        return prefix + chunk, chunk
    lens = _ints(case["lens_seed"], case["len_lo"], case["len_hi"], case["B"])
    return lens, np.ones_like(lens)


def _first_rows(case):
    """First attended position of each sequence's first query row."""
    lens, new = _lens(case)
    first = lens - new
    return np.maximum(0, first - case["window"] + 1) if case["window"] else np.zeros_like(first)


def _tables(case):
    """Block tables: a permutation of a pool with a tenth of its blocks free; blocks
    before the window are not resident."""
    lens, _ = _lens(case)
    lo = _first_rows(case) // BT
    nblk = (lens + BT - 1) // BT
    need = int((nblk - lo).sum())
    n_pool = need + need // 10 + 1
    perm = np.random.Generator(np.random.PCG64(case["lens_seed"] + 2)).permutation(n_pool)
    tables = np.full((lens.size, int(nblk.max())), -1, np.int32)
    cur = 0
    for b in range(lens.size):
        k = int(nblk[b] - lo[b])
        tables[b, lo[b]:nblk[b]] = perm[cur:cur + k]
        cur += k
    return tables, n_pool


# ---------------------------------------------------------------------------
# inputs (from the seed)
# ---------------------------------------------------------------------------
def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + salt) & 0x7FFFFFFFFFFFFFFF)
    return g


def _gains(case, seed, salt, heads):
    """Channels of projected keys and queries differ in scale."""
    return torch.exp(0.3 * torch.randn((heads, case["D"]), generator=_gen(seed, salt), device="cuda"))


def _rows(case, seed, salt, n, heads, gain=False):
    x = torch.randn((n, heads, case["D"]), generator=_gen(seed, salt), device="cuda")
    if gain:
        x *= _gains(case, seed, salt + 7, heads)
    return x.to(torch.bfloat16)


def _pieces(case, seed, n_blocks):
    """(first block, K rows, V rows) of the pool's blocks, [n][16][Hkv][D] bf16."""
    shape = (BT, case["Hkv"], case["D"])
    gk, gv = _gen(seed, 1), _gen(seed, 2)
    gain = _gains(case, seed, 3, case["Hkv"])
    for s in range(0, n_blocks, CHUNK):
        n = min(CHUNK, n_blocks - s)
        k = (torch.randn((n, *shape), generator=gk, device="cuda") * gain).to(torch.bfloat16)
        v = torch.randn((n, *shape), generator=gv, device="cuda").to(torch.bfloat16)
        yield s, k, v


class _View:
    """A pool's memory as a tensor (a program reads its own cache this way), which keeps the
    pool alive: the tensors made from it hold this object."""

    def __init__(self, pool, ptr, nbytes):
        self.pool = pool
        self.__cuda_array_interface__ = dict(shape=(nbytes,), typestr="|u1", data=(ptr, False), version=2)


def _pool_tensors(pool, fmt):
    i = pool.info
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "int8": torch.int8, "fp8": torch.uint8}[fmt]
    k = torch.as_tensor(_View(pool, i.d_k, i.k_bytes), device="cuda").view(dt).view(-1, i.kv_heads, BT, i.head_dim)
    v = torch.as_tensor(_View(pool, i.d_v, i.k_bytes), device="cuda").view(dt).view(-1, i.kv_heads, i.head_dim, BT)
    out = [k, v]
    if i.scale_bytes:
        s = torch.as_tensor(_View(pool, i.d_k_scales, 2 * i.scale_bytes), device="cuda")
        out.append(s.view(torch.float16 if fmt == "int8" else torch.float32))
    return out


def _new_token_slots(case):
    lens, _ = _lens(case)
    tables, _ = _tables(case)
    pos = lens - 1
    return tables[np.arange(lens.size), pos // BT].astype(np.int64), pos % BT


def prepare(case, seed):
    ctx = _ctx()
    kind, D, Hkv = case["kind"], case["D"], case["Hkv"]
    if kind == "trait":
        return _prepare_trait(ctx, case, seed)
    fmt = FORMATS[case["fmt"]]
    if kind == "write":
        n = case["blocks"]
        pool = ctx.pool(fmt, BT, Hkv, D, n)
        k, v = zip(*((k, v) for _, k, v in _pieces(case, seed, n)))
        ids = torch.randperm(n, generator=_gen(seed, 9), device="cuda").to(torch.int32)
        return dict(case=case, ctx=ctx, pool=pool, ids=ids, k=torch.cat(k), v=torch.cat(v),
                    view=_pool_tensors(pool, case["fmt"]))
    lens, new = _lens(case)
    tables, n_pool = _tables(case)
    pool = ctx.pool(fmt, BT, Hkv, D, n_pool)
    for s, k, v in _pieces(case, seed, n_pool):
        ctx.write_blocks(pool, torch.arange(s, s + k.shape[0], dtype=torch.int32, device="cuda"), k, v)
    T = int(new.sum())
    st = dict(case=case, ctx=ctx, pool=pool, scale=1.0 / math.sqrt(D), q=_rows(case, seed, 11, T, case["Hq"], True))
    st["gate"] = _rows(case, seed, 12, T, case["Hq"]) if case["gate"] else None
    st["tables"] = torch.from_numpy(tables).cuda()
    st["lens"] = torch.from_numpy(lens.astype(np.int32)).cuda()
    if kind == "prefill":
        starts = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
        st["starts"] = torch.from_numpy(starts).cuda()
        st["desc"] = ctx.prefill_desc(st["starts"], st["lens"], st["tables"], case["Hq"], int(new.max()),
                                      case["window"], total_q_rows=T, gate=st["gate"])
    else:
        st["desc"] = ctx.decode_desc(st["lens"], st["tables"], case["Hq"], int(lens.max()), case["window"],
                                     total_tokens_hint=int((lens - _first_rows(case)).sum()), gate=st["gate"])
    if kind == "append":
        st["k_new"] = _rows(case, seed, 13, T, Hkv)
        st["v_new"] = _rows(case, seed, 14, T, Hkv)
        st["view"] = _pool_tensors(pool, case["fmt"])
    if kind == "project":
        st["w"] = _proj_weight(case, seed)
        st["out"] = torch.empty((T, case["rows"]), dtype=torch.float32, device="cuda")
    else:
        st["out"] = torch.empty_like(st["q"])
    return st


def _proj_weight(case, seed):
    cols = case["Hq"] * case["D"]
    w = torch.randn((case["rows"], cols), generator=_gen(seed, 15), device="cuda")
    return (w / math.sqrt(cols)).to(torch.bfloat16)


def _trait_rows(case, seed):
    n, width = case["tokens"], case["Hkv"] * case["D"]
    rng = np.random.default_rng(seed)
    k = rng.standard_normal((n, width), dtype=np.float32)
    v = rng.standard_normal((n, width), dtype=np.float32)
    q = rng.standard_normal(case["Hq"] * case["D"], dtype=np.float32)
    return k, v, q


def _prepare_trait(ctx, case, seed):
    k, v, q = _trait_rows(case, seed)
    cache = llm_hip.LayerKvCache.from_rows(ctx, case["tokens"], case["Hkv"], case["D"], k, v, revision=case["tokens"],
                                           tokens_seen=case["tokens"], fmt=FORMATS[case["fmt"]])
    return dict(case=case, ctx=ctx, cache=cache, backend=llm_hip.HipNativeMatvecBackend(ctx), q=q,
                out=np.zeros_like(q), scale=1.0 / math.sqrt(case["D"]))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind == "decode":
        ctx.paged_decode(st["pool"], st["desc"], st["q"], st["out"], st["scale"])
        return st["out"]
    if kind == "append":
        ctx.paged_decode_append(st["pool"], st["desc"], st["k_new"], st["v_new"], st["q"], st["out"], st["scale"])
        return [st["out"], *st["view"]]
    if kind == "project":
        ctx.paged_decode_output_projection(st["pool"], st["desc"], st["q"], st["w"], case["rows"], st["out"],
                                           st["scale"])
        return st["out"]
    if kind == "prefill":
        ctx.paged_prefill(st["pool"], st["desc"], st["q"], st["out"], st["scale"])
        return st["out"]
    if kind == "write":
        ctx.write_blocks(st["pool"], st["ids"], st["k"], st["v"])
        return list(st["view"])
    st["backend"].full_attention_cache_mix_f32_in_place(st["cache"], st["q"], case["rows"], case["Hq"], case["Hkv"],
                                                        case["D"], st["scale"], st["out"])
    return st["out"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _scale_bytes(case, tokens, blocks):
    if case["fmt"] == "int8":
        return tokens * case["Hkv"] * 4
    return blocks * case["Hkv"] * 8 if case["fmt"] == "fp8" else 0


def work(case):
    D, Hkv, e = case["D"], case["Hkv"], ELEM[case["fmt"]]
    if case["kind"] == "write":
        tokens = case["blocks"] * BT
        moved = tokens * Hkv * D * 2 * (2 + e) + case["blocks"] * 4 + _scale_bytes(case, tokens, case["blocks"])
        return {"bytes": moved, "flops": 0}
    Hq = case["Hq"]
    if case["kind"] == "trait":
        tokens = case["rows"]
        moved = tokens * Hkv * D * e * 2 + _scale_bytes(case, tokens, -(-tokens // BT)) + 2 * Hq * D * 4
        return {"bytes": moved, "flops": 4 * D * Hq * tokens}
    lens, new = _lens(case)
    lo = _first_rows(case)
    tokens = int((lens - lo).sum())
    blocks = int(((lens + BT - 1) // BT - lo // BT).sum())
    T = int(new.sum())
    moved = tokens * Hkv * D * e * 2 + _scale_bytes(case, tokens, blocks) + blocks * 4 + lens.size * 4
    moved += T * Hq * D * 2 * (3 if case["gate"] else 2)
    pairs = 0
    for n, c in zip(lens.tolist(), new.tolist()):
        pos = np.arange(n - c, n, dtype=np.int64)
        first = np.maximum(0, pos - case["window"] + 1) if case["window"] else np.zeros_like(pos)
        pairs += int((pos - first + 1).sum())
    flops = 4 * D * Hq * pairs
    if case["kind"] == "append":
        moved += T * Hkv * D * 2 * (2 + e)
    if case["kind"] == "project":
        moved += case["rows"] * Hq * D * 2 + T * case["rows"] * 4 - T * Hq * D * 2
        flops += 2 * T * case["rows"] * Hq * D
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """Written blocks are codes and rounded elements: the same bytes.  Attention multiplies
    16-bit softmax weights (and 16-bit elements) and rounds its output to bf16."""
    if case["kind"] == "write":
        return "exact"
    return {"rel": 1e-2}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _stored(case, k):
    """Rows [n][16][Hkv][D] bf16 as the pool's format holds them, in f64."""
    if case["fmt"] == "bf16":
        return k.double()
    if case["fmt"] == "f16":
        return k.half().double()
    x = k.float()
    if case["fmt"] == "int8":
        s = (x.abs().amax(-1, keepdim=True).double() / 127.0).float().half().float()
        t = torch.where(s > 0, (x.double() / s.double()).float(), torch.zeros_like(x)).double()
        return (t.sign() * (t.abs() + 0.5).floor()).clamp(-127, 127) * s.double()
    s = (x.abs().amax((1, 3), keepdim=True).double() / 448.0).float()
    t = torch.where(s > 0, (x.double() / s.double()).float(), torch.zeros_like(x))
    c = t.clamp(-448, 448).cpu().to(torch.float8_e4m3fn).to(x.device).float()
    return c.double() * s.double()


def _attend(q, k, v, pos, window, scale):
    """q [T][Hq][D], k and v [n][Hkv][D] in f64; row t attends positions up to pos[t]."""
    T, Hq, D = q.shape
    n, Hkv, _ = k.shape
    G = Hq // Hkv
    out = torch.empty_like(q)
    key = torch.arange(n, device=q.device)
    keep = key[None, :] <= pos[:, None]
    if window:
        keep &= key[None, :] > pos[:, None] - window
    for h in range(Hkv):
        kh, vh = k[:, h].contiguous(), v[:, h].contiguous()
        for g in range(G):
            s = (q[:, h * G + g] @ kh.t()) * scale
            p = torch.softmax(s.masked_fill(~keep, -math.inf), dim=1)
            out[:, h * G + g] = p @ vh
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "write":
        return None
    D, Hq, Hkv = case["D"], case["Hq"], case["Hkv"]
    scale = 1.0 / math.sqrt(D)
    if kind == "trait":
        k, v, q = (torch.from_numpy(a).cuda() for a in _trait_rows(case, seed))
        n = case["rows"]
        if case["fmt"] == "bf16":
            k, v = (a[:n].view(n, Hkv, D).to(torch.bfloat16).double() for a in (k, v))
        else:  # quantised from the f32 rows, one scale per token and head
            k, v = (_stored(case, a[:n].view(n, 1, Hkv, D))[:, 0] for a in (k, v))
        out = _attend(q.double().view(1, Hq, D), k, v, torch.tensor([n - 1], device="cuda"), 0, scale)
        return out.view(-1).cpu().numpy()
    lens, new = _lens(case)
    tables, n_pool = _tables(case)
    ks, vs = zip(*((k, v) for _, k, v in _pieces(case, seed, n_pool)))
    K, V = torch.cat(ks), torch.cat(vs)
    del ks, vs
    T = int(new.sum())
    q = _rows(case, seed, 11, T, Hq, True).double()
    if kind == "append":
        blk, off = (torch.from_numpy(a).cuda() for a in _new_token_slots(case))
        K[blk, off] = _rows(case, seed, 13, T, Hkv)
        V[blk, off] = _rows(case, seed, 14, T, Hkv)
    outs, row, first = [], 0, _first_rows(case)
    for b in range(lens.size):
        n, c = int(lens[b]), int(new[b])
        j0 = int(first[b]) // BT
        ids = torch.from_numpy(tables[b, j0:(n + BT - 1) // BT].astype(np.int64)).cuda()
        k = _stored(case, K[ids]).view(-1, Hkv, D)[: n - j0 * BT]
        v = _stored(case, V[ids]).view(-1, Hkv, D)[: n - j0 * BT]
        pos = torch.arange(n - c, n, device="cuda") - j0 * BT
        outs.append(_attend(q[row:row + c], k, v, pos, case["window"], scale))
        row += c
    out = torch.cat(outs)
    if case["gate"]:
        out = out * torch.sigmoid(_rows(case, seed, 12, T, Hq).double())
    if kind == "project":
        return out.view(T, Hq * D) @ _proj_weight(case, seed).double().t()
    if kind == "append":
        if case["fmt"] not in ("bf16", "f16"):
            return [out, None, None, None]
        return [out, _stored(case, K).transpose(1, 2).contiguous(), _stored(case, V).permute(0, 2, 3, 1).contiguous()]
    return out
