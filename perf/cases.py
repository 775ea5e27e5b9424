"""Performance cases of the paged Q8_0 KV-cache path, through its public calls.

A case is a dict of plain values; `kind` names the call it stands for:

  decode        one layer's decode (or causal verify, q_len > 1) of a batch,
                this step's K/V rows appended in the launch (Pool.decode)
  prefill       one layer's chunked prefill: the chunks' K/V rows appended,
                then their causal attention (Pool.append, Pool.prefill)
  append        quantize-and-append of K/V rows into pages (append_q8)
  flash_decode  the drop-in for contiguous Q8_0 rows (flash_decode_q8)
  move          export of a sequence's K and V rows and their import into
                other pages (gather_q8, import_q8)
  spill         a token range of every layer as one R4KV page on the device
                (Pool.spill into its staging buffer)
  restore       an R4KV page in host memory back into a pool (Pool.restore)
  serve         a serving step: prefill chunks and decode rows through every
                layer, then the step's rollback (Serve)

K and V are bf16 N(0, 1) rows with 1% of each head's channels eight times
larger, queries N(0, 1), softmax scale 1/sqrt(head_dim) (flash_decode: none).
"""
from __future__ import annotations

import importlib.util
import math
import os
import random
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
BLOCK = 32  # values of a Q8_0 block: one f16 scale, then 32 int8 codes
DEV = "cuda"


def _rkv():
    name = "remora_lab_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            name, os.path.join(ROOT, "remora-lab_amd", "__init__.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


def listed():
    return [
        # one short request alone on the GPU: launches and latency only
        dict(name="decode_one_short", kind="decode", batch=1, ctx_lo=300, ctx_hi=300, spread=0,
             q_len=1, q_heads=8, kv_heads=2, head_dim=128, page=16, q="f32", out="f32"),
        # a batch of chat requests of mixed lengths
        dict(name="decode_16_mixed", kind="decode", batch=16, ctx_lo=4096, ctx_hi=16384, spread=1,
             q_len=1, q_heads=16, kv_heads=2, head_dim=256, page=64, q="bf16", out="f32"),
        # one request over a very long document
        dict(name="decode_one_262k", kind="decode", batch=1, ctx_lo=262144, ctx_hi=262144, spread=0,
             q_len=1, q_heads=16, kv_heads=2, head_dim=256, page=64, q="bf16", out="f32"),
        # a full GPU of long requests: the headline decode step
        dict(name="decode_64x32k", kind="decode", batch=64, ctx_lo=32767, ctx_hi=32767, spread=0,
             q_len=1, q_heads=16, kv_heads=2, head_dim=256, page=64, q="bf16", out="f32"),
        # speculative decoding: four draft rows per request, verified at once
        dict(name="verify_32x32k", kind="decode", batch=32, ctx_lo=32768, ctx_hi=32768, spread=0,
             q_len=4, q_heads=16, kv_heads=2, head_dim=256, page=64, q="bf16", out="f32"),
        # chunked prefill of eight requests deep in their prompts
        dict(name="prefill_8x512", kind="prefill", batch=8, ctx_lo=8192, ctx_hi=8192, rows_lo=512,
             rows_hi=512, spread=0, q_heads=16, kv_heads=2, head_dim=256, page=64, q="bf16",
             out="f32"),
        # prompts of odd lengths arriving together, some just starting, on the
        # reference's default heads
        dict(name="prefill_6_mixed", kind="prefill", batch=6, ctx_lo=0, ctx_hi=3000, rows_lo=17,
             rows_hi=701, spread=2, q_heads=24, kv_heads=4, head_dim=256, page=32, q="bf16",
             out="bf16"),
        # the rows of a long prompt written to the cache
        dict(name="append_64k", kind="append", rows=65536, seqs=16, kv_heads=2, head_dim=256,
             page=64, src="bf16", rule=0),
        # the shader's call at its default parameters
        dict(name="flash_decode_1k", kind="flash_decode", ctx=1024, q_heads=24, kv_heads=4,
             head_dim=256),
        # a request's cache exported and taken over by other pages
        dict(name="move_32k", kind="move", ctx=32768, kv_heads=2, head_dim=256, page=64),
        # a prefix of 4096 tokens over all layers leaving for another tier
        dict(name="spill_4k_48", kind="spill", first=0, tokens=4096, layers=48, kv_heads=2,
             head_dim=256, page=64),
        # a whole serving step: 8 chunks of 512 tokens and 56 decode rows
        dict(name="serve_64", kind="serve", decodes=56, chunks=8, rows=512, ctx_lo=512,
             ctx_hi=32768, spread=3, layers=4, q_heads=16, kv_heads=2, head_dim=256, page=64),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _heads(rng):
    kv = rng.choice([1, 2, 2, 4, 4, 8])
    return kv, kv * rng.choice([1, 2, 3, 4, 6, 8, 8])


def draw(rng):
    kind = rng.choice(["decode"] * 5 + ["prefill"] * 4 + ["append"] * 2 +
                      ["flash_decode", "move", "spill", "restore", "serve"])
    kv, qh = _heads(rng)
    d = rng.choice([128, 256, 256])
    page = rng.choice([16, 32, 64, 64, 128])
    c = dict(kind=kind, kv_heads=kv, head_dim=d)
    row = kv * d  # K (or V) values of one token
    if kind == "decode":
        q_len = rng.choice([1, 1, 1, 2, 3, 4])
        while q_len * (qh // kv) > 32:
            q_len -= 1
        batch = _log(rng, 1, 128)
        hi = _log(rng, 64, max(64, min(262144, (1 << 30) // (row * batch))))
        lo = _log(rng, max(1, hi // 8), hi)
        c.update(batch=batch, ctx_lo=lo, ctx_hi=hi, spread=rng.randrange(1 << 20), q_len=q_len,
                 q_heads=qh, page=page, q=rng.choice(["bf16", "bf16", "f32"]),
                 out=rng.choice(["f32", "bf16"]))
    elif kind == "prefill":
        batch = rng.choice([1, 1, 2, 3, 5, 8])
        rows = _log(rng, 8, 2048 if batch < 3 else 600)
        # rows * (context + rows) * heads * dim bounds the pass by the largest listed one
        room = (1 << 37) // (batch * rows * qh * d) - rows
        ctx = rng.choice([0, 1]) * _log(rng, 16, max(16, min(32768, room)))
        c.update(batch=batch, ctx_lo=ctx // 3, ctx_hi=ctx, rows_lo=max(1, rows // 3), rows_hi=rows,
                 spread=rng.randrange(1 << 20), q_heads=qh, page=page,
                 q=rng.choice(["bf16", "bf16", "bf16", "f32"]), out=rng.choice(["f32", "bf16"]))
    elif kind == "append":
        c.update(rows=_log(rng, 1, (1 << 25) // row), seqs=rng.choice([1, 3, 8, 32, 64]), page=page,
                 src=rng.choice(["bf16", "bf16", "f32"]), rule=rng.choice([0, 0, 1]))
    elif kind == "flash_decode":
        c.update(ctx=_log(rng, 16, 65536), q_heads=qh)
    elif kind == "move":
        c.update(ctx=_log(rng, 50, min(131072, (1 << 26) // row)), page=page)
    elif kind in ("spill", "restore"):
        layers = rng.choice([1, 4, 16, 48])
        c.update(first=rng.choice([0, 0, rng.randrange(1, 200)]),
                 tokens=_log(rng, 32, min(8192, (3 << 25) // (row * layers))), layers=layers, page=page)
    else:
        c.update(decodes=rng.randrange(1, 40), chunks=rng.randrange(0, 5), rows=_log(rng, 16, 256),
                 ctx_lo=64, ctx_hi=_log(rng, 256, 8192), spread=rng.randrange(1 << 20),
                 layers=rng.choice([1, 2, 4]), kv_heads=rng.choice([2, 4]), q_heads=16, page=page)
    return c


# ---- sizes ----------------------------------------------------------------------------

def _spread(case, n, lo, hi, salt=0):
    """n lengths between lo and hi, spread over their logarithm."""
    rng = random.Random(case["spread"] * 2 + salt)
    return [_log(rng, lo, hi) if lo > 0 else (rng.randrange(0, hi + 1) if hi > 0 else 0)
            for _ in range(n)]


def _lens(case):
    """Tokens cached before the pass, one number per sequence."""
    n = case["decodes"] + case["chunks"] if case["kind"] == "serve" else case["batch"]
    return _spread(case, n, case["ctx_lo"], case["ctx_hi"])


def _rows(case):
    """Chunk rows of each prefill entry."""
    if case["kind"] == "serve":
        return [case["rows"]] * case["chunks"]
    return _spread(case, case["batch"], case["rows_lo"], case["rows_hi"], 1)


def _pages(tokens, page):
    return (tokens + page - 1) // page


# ---- inputs ---------------------------------------------------------------------------

def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + salt) % (1 << 60))
    return g


def _kv(case, seed, salt, n):
    """K and V rows [n][kv_heads][head_dim] of one sequence (or of a chunk)."""
    g = _gen(seed, salt)
    shape = (n, case["kv_heads"], case["head_dim"])
    loud = _gen(seed, 7)  # the same channels in every row of a case
    mult = torch.ones(shape[1:], device=DEV)
    mult[torch.rand(shape[1:], generator=loud, device=DEV) < 0.01] = 8.0
    out = []
    for _ in range(2):
        out.append((torch.randn(shape, generator=g, device=DEV) * mult).to(torch.bfloat16))
    return out


def _query(case, seed, rows):
    q = torch.randn((rows, case["q_heads"], case["head_dim"]), generator=_gen(seed, 11), device=DEV)
    return q.to(DTYPES[case.get("q", "bf16")])


def _i32(values):
    return torch.tensor(list(values), dtype=torch.int32, device=DEV)


class _Memory:
    """Device memory of a pool, for torch to look at; holds the pool, which owns it."""

    def __init__(self, pool, n):
        self.pool = pool
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "|u1",
                                         "data": (pool.layer_pages(0), False), "version": 2}


def _pool(rkv, case, lens, layers=1):
    """A pool that holds `lens` tokens per sequence, its tables uploaded, and its page bytes."""
    page = case["page"]
    need = [_pages(n, page) for n in lens]
    pool = rkv.Pool(rkv.Ctx(0), layers, case["kv_heads"], case["head_dim"], page,
                    max(1, math.ceil(sum(need) * 1.1)), len(lens), max(need + [1]), seed=5)
    for s, n in enumerate(lens):
        pool.alloc.reserve(s, n)
    pool.sync_tables()
    bytes_ = layers * rkv.page_bytes(pool.geometry) * pool.geometry.num_pages
    view = torch.as_tensor(_Memory(pool, bytes_), device=DEV)
    view.pool = pool  # an output may outlive its state: the pool lives as long as this tensor
    view.zero_()
    return pool, view


def _fill(pool, case, seed, s, n, layer=0, salt=1000):
    k, v = _kv(case, seed, salt + s, n)
    if n:
        pool.append(layer, torch.full((n,), s, dtype=torch.int32, device=DEV),
                    torch.arange(n, dtype=torch.int32, device=DEV), k, v)


def _prepare_decode(rkv, case, seed):
    lens, b, ql = _lens(case), case["batch"], case["q_len"]
    pool, view = _pool(rkv, case, [n + ql for n in lens])
    for s, n in enumerate(lens):
        _fill(pool, case, seed, s, n)
    seqs = _i32(range(b))
    k, v = _kv(case, seed, 1, b * ql)
    app = rkv.append_args(seqs.repeat_interleave(ql),
                          _i32(n + j for n in lens for j in range(ql)), k, v)
    q = _query(case, seed, b * ql).reshape(b, ql, case["q_heads"], case["head_dim"])
    out = torch.empty(q.shape, dtype=DTYPES[case["out"]], device=DEV)
    scale, most = 1 / math.sqrt(case["head_dim"]), max(lens) + ql
    a = rkv.decode_args(q, out, seqs, scale, most, q_len=ql, append=app)
    ws = torch.empty(max(4, rkv.decode_workspace_bytes(pool.geometry, a)), dtype=torch.uint8, device=DEV)
    a = rkv.decode_args(q, out, seqs, scale, most, q_len=ql, workspace=ws, append=app)
    return dict(pool=pool, args=a, out=out, pages=view)


def _run_decode(s):
    s["pool"].decode(0, s["args"])
    return {"out": s["out"], "pages": s["pages"]}


def _prepare_prefill(rkv, case, seed):
    ctx, rows = _lens(case), _rows(case)
    pool, view = _pool(rkv, case, [c + n for c, n in zip(ctx, rows)])
    for s, n in enumerate(ctx):
        _fill(pool, case, seed, s, n)
    total, seqs = sum(rows), list(range(case["batch"]))
    k, v = _kv(case, seed, 1, total)
    q = _query(case, seed, total)
    out = torch.empty(q.shape, dtype=DTYPES[case["out"]], device=DEV)
    scale = 1 / math.sqrt(case["head_dim"])
    a = rkv.prefill_args(seqs, ctx, rows, q, out, scale)
    ws = torch.empty(max(1, pool.prefill_workspace_bytes(a)), dtype=torch.uint8, device=DEV)
    a = rkv.prefill_args(seqs, ctx, rows, q, out, scale, workspace=ws)
    return dict(pool=pool, args=a, out=out, pages=view, k=k, v=v,
                seqs=_i32(s for s, n in enumerate(rows) for _ in range(n)),
                positions=_i32(c + i for c, n in zip(ctx, rows) for i in range(n)))


def _run_prefill(s):
    s["pool"].append(0, s["seqs"], s["positions"], s["k"], s["v"])
    s["pool"].prefill(0, s["args"])
    return {"out": s["out"], "pages": s["pages"]}


def _tables(case, lens, seed):
    """Block tables of `lens` tokens per sequence over shuffled pages, and their number."""
    need = [_pages(n, case["page"]) for n in lens]
    total = max(1, math.ceil(sum(need) * 1.1))
    order = torch.randperm(total, generator=_gen(seed, 3), device=DEV).to(torch.int32)
    bt, at = torch.full((len(lens), max(need + [1])), -1, dtype=torch.int32, device=DEV), 0
    for s, n in enumerate(need):
        bt[s, :n] = order[at:at + n]
        at += n
    return bt, total


def _append_lens(case):
    each = case["rows"] // case["seqs"]
    return [each + (s < case["rows"] % case["seqs"]) for s in range(case["seqs"])]


def _prepare_append(rkv, case, seed):
    lens = _append_lens(case)
    bt, total = _tables(case, lens, 0)
    g = rkv.geometry(case["kv_heads"], case["head_dim"], case["page"], total)
    k, v = _kv(case, seed, 1, case["rows"])
    return dict(rkv=rkv, ctx=rkv.Ctx(0), g=g, bt=bt, rule=case["rule"],
                k=k.to(DTYPES[case["src"]]), v=v.to(DTYPES[case["src"]]),
                pages=torch.zeros(total * rkv.page_bytes(g), dtype=torch.uint8, device=DEV),
                seqs=_i32(s for s, n in enumerate(lens) for _ in range(n)),
                positions=_i32(i for n in lens for i in range(n)))


def _run_append(s):
    s["rkv"].append_q8(s["ctx"], s["g"], s["pages"], s["bt"], s["seqs"], s["positions"], s["k"],
                       s["v"], rule=s["rule"])
    return s["pages"]


def _prepare_flash(rkv, case, seed):
    n, kv, d = case["ctx"], case["kv_heads"], case["head_dim"]
    words = [_words(x.transpose(0, 1).contiguous()) for x in _kv(case, seed, 1, n)]
    q = torch.randn((case["q_heads"], d), generator=_gen(seed, 11), device=DEV) / math.sqrt(d)
    p = rkv.FlashDecodeParams(case["q_heads"], kv, n, 1024, d)
    scratch = torch.empty(rkv.flash_decode_scratch_bytes(p), dtype=torch.uint8, device=DEV)
    return dict(rkv=rkv, ctx=rkv.Ctx(0), p=p, k=words[0], v=words[1], q=q,
                out=torch.empty_like(q), scratch=scratch)


def _run_flash(s):
    s["rkv"].flash_decode_q8(s["ctx"], s["p"], s["k"], s["v"], s["q"], s["out"], s["scratch"])
    return s["out"]


def _prepare_move(rkv, case, seed):
    n, page = case["ctx"], case["page"]
    (bt, total), (to, _) = _tables(case, [n], 0), _tables(case, [n], 1)
    g = rkv.geometry(case["kv_heads"], case["head_dim"], page, total)
    ctx = rkv.Ctx(0)
    pages = torch.zeros(total * rkv.page_bytes(g), dtype=torch.uint8, device=DEV)
    k, v = _kv(case, seed, 1, n)
    rkv.append_q8(ctx, g, pages, bt, torch.zeros(n, dtype=torch.int32, device=DEV),
                  torch.arange(n, dtype=torch.int32, device=DEV), k, v)
    rows = [torch.zeros(case["kv_heads"] * n * rkv.row_bytes(case["head_dim"]), dtype=torch.uint8,
                        device=DEV) for _ in range(2)]
    return dict(rkv=rkv, ctx=ctx, g=g, n=n, bt=bt[0], to=to[0], pages=pages,
                other=torch.zeros_like(pages), rows=rows)


def _run_move(s):
    rkv, g = s["rkv"], s["g"]
    for kind in (rkv.K, rkv.V):
        rkv.gather_q8(s["ctx"], g, s["pages"], s["bt"], s["n"], kind, s["rows"][kind])
        rkv.import_q8(s["ctx"], g, s["other"], s["to"], s["n"], kind, s["rows"][kind])
    return {"k": s["rows"][0], "v": s["rows"][1], "pages": s["other"]}


def _prepare_tier(rkv, case, seed):
    """A pool with the range written in every layer (spill), or with its page
    in host memory (restore)."""
    first, n, layers = case["first"], case["tokens"], case["layers"]
    pool, view = _pool(rkv, case, [first + n], layers)
    for layer in range(layers):
        _fill(pool, case, seed, 0, first + n, layer, salt=1000 + 64 * layer)
    size = pool.r4kv_page_bytes(n, 0, layers - 1)
    ident = rkv.R4kvHeader(prefix_digest=0xC0FFEE, token_start=first, token_count=n, pos_start=first,
                           layer_lo=0, layer_hi=layers - 1, k_fmt=rkv.FMT_Q8, v_fmt=rkv.FMT_Q8,
                           epoch=1, generation=1, payload_len=0, sketch_offset=0, flags=0)
    s = dict(pool=pool, pages=view, first=first, n=n, layers=layers, ident=ident,
             staging=torch.zeros(size, dtype=torch.uint8, device=DEV))
    if case["kind"] == "restore":
        s["page"] = torch.empty(size, dtype=torch.uint8, pin_memory=True)
        pool.spill(0, first, n, 0, layers - 1, ident, s["staging"], s["page"])
        torch.cuda.synchronize()
        s["expect"] = rkv.R4kvExpect(prefix_digest=0xC0FFEE, token_start=first, pos_start=first,
                                     layer_lo=0, layer_hi=layers - 1, k_fmt=rkv.FMT_Q8,
                                     v_fmt=rkv.FMT_Q8, check_generation=0, generation_min=0,
                                     generation_max=0)
        view.zero_()
    return s


def _run_spill(s):
    s["pool"].spill(0, s["first"], s["n"], 0, s["layers"] - 1, s["ident"], s["staging"], s["staging"])
    return s["staging"]


def _run_restore(s):
    s["pool"].restore(0, s["page"], s["expect"], s["staging"])
    return s["pages"]


def _prepare_serve(rkv, case, seed):
    lens, rows, page, layers = _lens(case), _rows(case), case["page"], case["layers"]
    nd, nc = case["decodes"], case["chunks"]
    more = [1] * nd + rows
    need = [_pages(n + m, page) for n, m in zip(lens, more)]
    sv = rkv.Serve(rkv.Ctx(0), layers, case["kv_heads"], case["head_dim"], page,
                   math.ceil(sum(need) * 1.1) + len(need), len(lens), max(need) + 1,
                   q_heads=case["q_heads"], max_decode=len(lens), max_prefill_rows=max(1, sum(rows)),
                   seed=5)
    sv.begin_step(decode=[(i, 1) for i in range(len(lens))])
    for i, n in enumerate(lens):
        sv.alloc.reserve(sv.slot(i), n)
    sv.sync_tables()
    for i, n in enumerate(lens):
        for layer in range(layers):
            k, v = _kv(case, seed, 1000 + 1024 * layer + i, n)
            sv.pool_append(layer, torch.full((n,), sv.slot(i), dtype=torch.int32, device=DEV),
                           torch.arange(n, dtype=torch.int32, device=DEV), k, v)
    heads, d = case["q_heads"], case["head_dim"]
    qd, qp = _query(case, seed, nd), _query(case, seed + 1, sum(rows))
    kd, vd = _kv(case, seed, 1, nd)
    kp, vp = _kv(case, seed, 2, sum(rows))
    out = [[torch.empty((n, heads, d), device=DEV) for n in (sum(rows), nd)] for _ in range(layers)]
    return dict(sv=sv, layers=layers, scale=1 / math.sqrt(d), lens=lens, out=out,
                prefill=[(nd + i, n) for i, n in enumerate(rows)], decode=[(i, 1) for i in range(nd)],
                qd=qd, kd=kd, vd=vd, qp=qp, kp=kp, vp=vp)


def _run_serve(s):
    sv = s["sv"]
    sv.begin_step(prefill=s["prefill"], decode=s["decode"])
    for layer in range(s["layers"]):
        sv.prefill(layer, s["qp"], s["kp"], s["vp"], s["out"][layer][0], s["scale"])
        sv.decode(layer, s["qd"], s["kd"], s["vd"], s["out"][layer][1], s["scale"])
    for i, n in enumerate(s["lens"]):
        sv.truncate(i, n)
    return s["out"]


_PREPARE = dict(decode=_prepare_decode, prefill=_prepare_prefill, append=_prepare_append,
                flash_decode=_prepare_flash, move=_prepare_move, spill=_prepare_tier,
                restore=_prepare_tier, serve=_prepare_serve)
_RUN = dict(decode=_run_decode, prefill=_run_prefill, append=_run_append, flash_decode=_run_flash,
            move=_run_move, spill=_run_spill, restore=_run_restore, serve=_run_serve)


def prepare(case, seed):
    state = _PREPARE[case["kind"]](_rkv(), case, seed)
    state["run"] = _RUN[case["kind"]]
    return state


def run(state):
    return state["run"](state)


# ---- what a pass cannot do without ----------------------------------------------------

def work(case):
    kv, d, kind = case["kv_heads"], case["head_dim"], case["kind"]
    row = kv * (d // BLOCK) * 34      # Q8_0 bytes of one token's K (or V)
    src = {"f32": 4, "bf16": 2}
    size = src[case.get("q", "bf16")] + src[case.get("out", "f32")]  # a query value and its output
    if kind == "decode":
        ql, b = case["q_len"], case["batch"]
        tokens = sum(n + ql for n in _lens(case))
        seen = sum(n + j + 1 for n in _lens(case) for j in range(ql))
        new = b * ql * 2 * kv * d * 2
        return {"bytes": tokens * 2 * row + b * ql * case["q_heads"] * d * size + new,
                "flops": 4.0 * d * case["q_heads"] * seen}
    if kind == "prefill":
        pairs = list(zip(_lens(case), _rows(case)))
        total = sum(n for _, n in pairs)
        seen = sum(n * c + n * (n + 1) // 2 for c, n in pairs)
        return {"bytes": sum(c + n for c, n in pairs) * 2 * row + total * case["q_heads"] * d * size +
                total * 2 * kv * d * 2, "flops": 4.0 * d * case["q_heads"] * seen}
    if kind == "append":
        return {"bytes": case["rows"] * 2 * (kv * d * src[case["src"]] + row), "flops": 0}
    if kind == "flash_decode":
        return {"bytes": case["ctx"] * 2 * row + case["q_heads"] * d * 8,
                "flops": 4.0 * d * case["q_heads"] * case["ctx"]}
    if kind == "move":
        return {"bytes": case["ctx"] * 2 * row * 4, "flops": 0}
    if kind in ("spill", "restore"):
        return {"bytes": case["tokens"] * case["layers"] * 2 * row * 2, "flops": 0}
    lens, rows, layers = _lens(case), _rows(case), case["layers"]
    nd = case["decodes"]
    total = nd + sum(rows)
    seen = sum(n + 1 for n in lens[:nd]) + sum(n * c + n * (n + 1) // 2
                                               for c, n in zip(lens[nd:], rows))
    return {"bytes": layers * ((sum(lens) + total) * 2 * row + total * case["q_heads"] * d * size +
                               total * 2 * kv * d * 2),
            "flops": layers * 4.0 * d * case["q_heads"] * seen}


def tolerance(case):
    """f32 outputs: f32 sums in another order.  bf16 outputs: one rounding of
    the result to 8 bits, which falls to the other side now and then.  Page
    and row bytes are the same."""
    if case["kind"] in ("append", "move", "spill", "restore"):
        return "exact"
    return {"rel": 4e-6 if case.get("out", "f32") == "f32" else 1e-3,
            "max": 1e-4 if case.get("out", "f32") == "f32" else 1e-2}


# ---- the same results in 64 bits ------------------------------------------------------

def _quantize(x):
    """(codes, f16 scales) of the canonical Q8_0 rule over the last dim's blocks."""
    x = x.float().reshape(*x.shape[:-1], x.shape[-1] // BLOCK, BLOCK)
    d = x.abs().amax(-1, keepdim=True)
    d = d / torch.full_like(d, 127.0)  # (a divisor given as a number is multiplied by its reciprocal)
    inv = torch.where(d == 0, torch.zeros_like(d), torch.ones_like(d) / d)
    y = x * inv
    codes = torch.trunc(y.double() + torch.copysign(torch.full_like(y, 0.5), y).double())
    return codes.clamp(-127, 127), d.to(torch.float16)


def _stored(x):
    """What the cache holds of x, in 64 bits."""
    codes, d = _quantize(x)
    return (codes * d.double()).reshape(x.shape)


def _words(x):
    """Q8_0 rows (per block the f16 scale, then 32 codes) as 32-bit words."""
    codes, d = _quantize(x)
    rows = torch.cat([d.view(torch.uint8), codes.to(torch.int8).view(torch.uint8)], -1)
    return rows.reshape(-1).view(torch.int32)


def _attend(q, k, v, limits, scale):
    """Rows q [n][heads][d] over k, v [tokens][kv_heads][d]; row i sees limits[i] tokens."""
    n, heads, d = q.shape
    kv = k.shape[1]
    g = heads // kv
    out = torch.zeros((n, heads, d), dtype=torch.float64, device=DEV)
    at = torch.arange(k.shape[0], device=DEV)
    step = max(1, (1 << 27) // max(1, g * k.shape[0]))
    for h in range(kv):
        kh, vh = k[:, h].t().contiguous(), v[:, h].contiguous()
        for a in range(0, n, step):
            qh = q[a:a + step, h * g:(h + 1) * g].double()
            s = (qh.reshape(-1, d) @ kh * scale).reshape(qh.shape[0], g, -1)
            s.masked_fill_((at >= limits[a:a + step, None])[:, None], -math.inf)
            p = torch.softmax(s, -1)
            out[a:a + step, h * g:(h + 1) * g] = (p.reshape(-1, p.shape[-1]) @ vh).reshape(qh.shape)
    return out


def _joined(case, seed, salt, n, new):
    """K and V as cached after `new` (K, V) rows follow a sequence's first n."""
    return [torch.cat([_stored(a), _stored(b)]) for a, b in zip(_kv(case, seed, salt, n), new)]


def exact(case, seed):
    kind, scale = case["kind"], 1 / math.sqrt(case["head_dim"])
    if kind == "decode":
        ql, b = case["q_len"], case["batch"]
        k, v = _kv(case, seed, 1, b * ql)
        q = _query(case, seed, b * ql)
        out = []
        for s, n in enumerate(_lens(case)):
            at = slice(s * ql, s * ql + ql)
            kk, vv = _joined(case, seed, 1000 + s, n, (k[at], v[at]))
            out.append(_attend(q[at], kk, vv, n + 1 + torch.arange(ql, device=DEV), scale))
        return {"out": torch.stack(out), "pages": None}
    if kind == "prefill":
        rows = _rows(case)
        k, v = _kv(case, seed, 1, sum(rows))
        q, out, a = _query(case, seed, sum(rows)), [], 0
        for s, (c, n) in enumerate(zip(_lens(case), rows)):
            kk, vv = _joined(case, seed, 1000 + s, c, (k[a:a + n], v[a:a + n]))
            out.append(_attend(q[a:a + n], kk, vv, c + 1 + torch.arange(n, device=DEV), scale))
            a += n
        return {"out": torch.cat(out), "pages": None}
    if kind == "flash_decode":
        d = case["head_dim"]
        q = torch.randn((case["q_heads"], d), generator=_gen(seed, 11), device=DEV) / math.sqrt(d)
        k, v = (_stored(x) for x in _kv(case, seed, 1, case["ctx"]))
        return _attend(q[None], k, v, torch.tensor([case["ctx"]], device=DEV), 1.0)[0]
    if kind == "serve":
        rows, lens, nd, out = _rows(case), _lens(case), case["decodes"], []
        kd, vd = _kv(case, seed, 1, nd)
        kp, vp = _kv(case, seed, 2, sum(rows))
        qd, qp = _query(case, seed, nd), _query(case, seed + 1, sum(rows))
        for layer in range(case["layers"]):
            pre, dec, a = [], [], 0
            for i, n in enumerate(lens):
                salt = 1000 + 1024 * layer + i
                if i < nd:
                    kk, vv = _joined(case, seed, salt, n, (kd[i:i + 1], vd[i:i + 1]))
                    dec.append(_attend(qd[i:i + 1], kk, vv, torch.tensor([n + 1], device=DEV), scale))
                    continue
                m = rows[i - nd]
                kk, vv = _joined(case, seed, salt, n, (kp[a:a + m], vp[a:a + m]))
                pre.append(_attend(qp[a:a + m], kk, vv, n + 1 + torch.arange(m, device=DEV), scale))
                a += m
            empty = torch.zeros((0, case["q_heads"], case["head_dim"]), dtype=torch.float64, device=DEV)
            out.append([torch.cat(pre or [empty]), torch.cat(dec or [empty])])
        return out
    return None  # bytes
