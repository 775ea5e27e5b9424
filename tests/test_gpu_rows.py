"""Export, import, the drop-in decode's import and the R4KV spill at the edges
of the tiles that their kernels move whole: part-filled tiles, odd row
counts, output and input pointers of any alignment, several tiles per
workgroup.  Bit-exact, except the drop-in's attention (f32 sums)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    return torch


@pytest.mark.parametrize("D,PT", [(128, 16), (128, 64), (256, 16), (256, 32), (256, 128)])
def test_gather_import_edges(rkv, rko, ctx, D, PT):
    torch = _torch()
    rng = np.random.default_rng(D + PT)
    Hkv, RB = 3, rkv.row_bytes(D)
    for L, shift in [(1, 0), (15, 8), (16, 4), (17, 0), (31, 1), (32, 16), (33, 8), (2 * PT + 5, 0),
                     (3 * PT, 3)]:
        npg = (L + PT - 1) // PT
        g = rkv.geometry(Hkv, D, PT, npg + 3)
        bt = rng.permutation(npg + 3)[:npg].astype(np.int32)
        btd = torch.from_numpy(bt).cuda()
        before = rng.integers(0, 256, (npg + 3) * rkv.page_bytes(g), dtype=np.uint8)
        rows = rng.integers(0, 256, Hkv * L * RB, dtype=np.uint8)
        src = torch.zeros(rows.size + 64, dtype=torch.uint8, device="cuda")
        src[shift:shift + rows.size] = torch.from_numpy(rows).cuda()
        for kind in (0, 1):
            pages = torch.from_numpy(before).cuda()
            rkv.import_q8(ctx, g, pages, btd, L, kind, src[shift:])
            out = torch.full((rows.size + 64,), 7, dtype=torch.uint8, device="cuda")
            rkv.gather_q8(ctx, g, pages, btd, L, kind, out[shift:])
            ctx.sync()
            got = out.cpu().numpy()
            assert np.array_equal(got[shift:shift + rows.size], rows), (L, shift, kind)
            assert (got[:shift] == 7).all() and (got[shift + rows.size:] == 7).all(), (L, shift, kind)
            lay = rko.layout(Hkv, D, PT, npg + 3)
            assert np.array_equal(rko.paged_gather(lay, pages.cpu().numpy(), bt, L, kind).reshape(-1), rows)
            # exactly the L rows' bytes may change: the other kind and the slots
            # past L read back as before
            full = npg * PT
            for k in (0, 1):
                a = rko.paged_gather(lay, pages.cpu().numpy(), bt, full, k).reshape(Hkv, full, RB)
                b = rko.paged_gather(lay, before, bt, full, k).reshape(Hkv, full, RB)
                kept = slice(L, full) if k == kind else slice(0, full)
                assert np.array_equal(a[:, kept], b[:, kept]), (L, shift, kind, k)


@pytest.mark.parametrize("D", [128, 256])
@pytest.mark.parametrize("L", [0, 1, 31, 64, 65, 96, 97, 200, 256, 300])
def test_flash_decode_lengths(rkv, rko, ctx, D, L):
    torch = _torch()
    rng = np.random.default_rng(L + D)
    Hq, Hkv = 6, 2
    k, v = (rng.standard_normal((Hkv, L, D)).astype(np.float32) for _ in range(2))
    q = (rng.standard_normal((Hq, D)) / np.sqrt(D)).astype(np.float32)
    kr, vr = (np.frombuffer(b"".join(rko.q8_encode(x[h].reshape(-1)).tobytes() for h in range(Hkv)),
                            np.uint8).copy() for x in (k, v))
    p = rkv.FlashDecodeParams(Hq, Hkv, L, 1024, D)
    scratch = torch.full((rkv.flash_decode_scratch_bytes(p),), 0xFF, dtype=torch.uint8, device="cuda")
    out = torch.full((Hq, D), float("nan"), device="cuda")
    qd = torch.from_numpy(q).cuda()
    kd, vd = (torch.from_numpy(x).cuda() if L else None for x in (kr, vr))
    for _ in range(2):  # the second call finds its own scratch of the first
        rkv.flash_decode_q8(ctx, p, kd, vd, qd, out, scratch)
    ctx.sync()
    got = out.cpu().numpy()
    if L == 0:
        assert (got == 0).all()
        return
    blocks = [x.reshape(Hkv, L, D // 32, 34) for x in (kr, vr)]
    kq, vq = ((b[..., 2:].view(np.int8).astype(np.float64) *
               b[..., :2].copy().view(np.float16).astype(np.float64)).reshape(Hkv, L, D) for b in blocks)
    for h in range(Hq):
        s = kq[h // 3] @ q[h].astype(np.float64)
        w = np.exp(s - s.max())
        want = w @ vq[h // 3] / w.sum()
        # f32 sums of up to 300 terms: well inside 1e-5 of the row's largest value
        assert np.abs(got[h] - want).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("L", [200, 1000])
def test_flash_decode_captured(rkv, rko, ctx, L):
    """The drop-in in a HIP graph: each replay, with other rows and queries in
    the same buffers, gives an eager call's bits."""
    torch = _torch()
    Hq, Hkv, D = 6, 2, 128
    p = rkv.FlashDecodeParams(Hq, Hkv, L, 1024, D)
    scratch, other = (torch.full((rkv.flash_decode_scratch_bytes(p),), 0xFF, dtype=torch.uint8, device="cuda")
                      for _ in range(2))
    out, want = torch.empty((Hq, D), device="cuda"), torch.empty((Hq, D), device="cuda")
    k, v = (torch.empty(Hkv * L * rkv.row_bytes(D), dtype=torch.uint8, device="cuda") for _ in range(2))
    q = torch.empty((Hq, D), device="cuda")

    def fill(seed):
        rng = np.random.default_rng(seed)
        for t in (k, v):
            t.copy_(torch.from_numpy(rko.q8_encode(rng.standard_normal(Hkv * L * D).astype(np.float32)).copy()
                                     .view(np.uint8).reshape(-1)))
        q.copy_(torch.from_numpy((rng.standard_normal((Hq, D)) / np.sqrt(D)).astype(np.float32)))
        torch.cuda.synchronize()

    fill(0)
    side = torch.cuda.Stream()
    rkv.flash_decode_q8(ctx, p, k, v, q, out, scratch, stream=side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        rkv.flash_decode_q8(ctx, p, k, v, q, out, scratch, stream=side)
    for rep in range(4):
        fill(rep + 1)
        out.fill_(float("nan"))
        rkv.flash_decode_q8(ctx, p, k, v, q, want, other)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), rep
    del graph


@pytest.mark.parametrize("D,PT,Hkv,layers,first,count", [
    (128, 16, 4, 30, 7, 300),    # 3 tiles a workgroup, both edges part-filled
    (128, 64, 1, 1, 33, 62),     # odd rows: runs at odd multiples of 8 bytes
    (256, 64, 2, 48, 0, 640),    # whole tiles, 3 a workgroup
    (256, 32, 2, 3, 31, 34),     # one row, a tile, one row
    (256, 16, 3, 2, 5, 9),       # inside one tile
    (256, 128, 8, 2, 0, 1),
    (128, 32, 2, 2, 40, 0),      # no tokens: header and CRC of nothing
    (256, 64, 2, 48, 3, 4100),   # 15 tiles a workgroup, both edges part-filled
    (128, 16, 16, 56, 5, 1100),  # more streams than workgroups at once: 64 tiles each, the most
])
def test_spill_edges(rkv, ctx, D, PT, Hkv, layers, first, count):
    torch = _torch()
    n, RB = first + max(count, 1) + 3, rkv.row_bytes(D)
    pages = (n + PT - 1) // PT
    pool = rkv.Pool(ctx, layers, Hkv, D, PT, pages + 2, 1, pages, seed=3)
    pool.alloc.reserve(0, n)
    pool.sync_tables()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(D + count)
    pos = torch.arange(n, dtype=torch.int32, device="cuda")
    for layer in range(layers):
        k, v = (torch.randn((n, Hkv, D), generator=gen, device="cuda") for _ in range(2))
        pool.append(layer, torch.zeros_like(pos), pos, k, v)
    size = pool.r4kv_page_bytes(count, 0, layers - 1)
    ident = rkv.R4kvHeader(prefix_digest=11, pos_start=first, epoch=1, generation=2)
    staging = torch.full((size + 32,), 0xA5, dtype=torch.uint8, device="cuda")
    for _ in range(2):  # the second spill finds the state the first left
        pool.spill(0, first, count, 0, layers - 1, ident, staging, staging)
    ctx.sync()
    page = staging.cpu().numpy()
    assert (page[size:] == 0xA5).all()
    h, body = rkv.r4kv_unpack_host(page[:size])  # header, length and CRC
    assert (h.token_start, h.token_count, h.layer_hi) == (first, count, layers - 1)
    body = np.frombuffer(body, np.uint8).reshape(layers, 2, Hkv, count, RB)
    rows = torch.empty(Hkv * n * RB, dtype=torch.uint8, device="cuda")
    for layer in range(layers):
        for kind in (0, 1):
            pool.gather(layer, 0, kind, rows)
            ctx.sync()
            want = rows.cpu().numpy().reshape(Hkv, n, RB)[:, first:first + count]
            assert np.array_equal(body[layer, kind], want), (layer, kind)
    pool.close()


def test_spill_after_overlapping_replays(rkv, ctx):
    """Captured spills of one pool, replayed one at a time, give whole pages.
    Replayed on two streams at once they may spoil each other's CRC word (a
    restore refuses such a page), but no later spill's."""
    torch = _torch()
    layers, Hkv, D, PT, n = 8, 2, 256, 64, 2000
    W = -(-n // PT)
    pool = rkv.Pool(ctx, layers, Hkv, D, PT, W, 1, W, seed=9)
    pool.alloc.reserve(0, n)
    pool.sync_tables()
    pos = torch.arange(n, dtype=torch.int32, device="cuda")
    for layer in range(layers):
        k, v = (torch.randn((n, Hkv, D), device="cuda") for _ in range(2))
        pool.append(layer, torch.zeros_like(pos), pos, k, v)
    ident = rkv.R4kvHeader(prefix_digest=3, pos_start=0, epoch=1, generation=1)
    size = [pool.r4kv_page_bytes(c, 0, layers - 1) for c in (n, n - 33)]
    staging = [torch.zeros(x, dtype=torch.uint8, device="cuda") for x in size]
    streams = [torch.cuda.Stream() for _ in range(2)]

    def spill(i, stream=None):
        pool.spill(0, 0, n - 33 * i, 0, layers - 1, ident, staging[i], staging[i], stream=stream)

    def whole(i):
        rkv.r4kv_unpack_host(staging[i].cpu().numpy())  # raises unless header and CRC hold

    graphs = []
    for i, s in enumerate(streams):
        spill(i, s)
        torch.cuda.synchronize()
        whole(i)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            spill(i, s)
        graphs.append(g)
    for i in (0, 1, 0):
        staging[i].zero_()
        torch.cuda.synchronize()
        graphs[i].replay()
        torch.cuda.synchronize()
        whole(i)
    for _ in range(20):
        for g, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                g.replay()
    torch.cuda.synchronize()
    for i in (0, 1):
        staging[i].zero_()
        spill(i)
        ctx.sync()
        whole(i)
    del graphs
    pool.close()


@pytest.mark.parametrize("D,PT,rows", [(128, 16, 8200), (256, 16, 8200), (256, 64, 8301), (256, 32, 300), (128, 64, 37)])
def test_append_of_ragged_sequences(rkv, rko, ctx, D, PT, rows):
    """Runs of rows that start and end at every slot modulo 4, in 32-row
    workgroups (whole shifted quads, several sequences in one, a part-filled
    last one, a last chunk of row blocks that is not full) and 8-row ones."""
    torch = _torch()
    rng = np.random.default_rng(rows + D + PT)
    Hkv, sid, pos, ends = 8, [], [], []
    while len(sid) < rows:
        start = int(rng.integers(0, 70))
        n = min(int(rng.choice([1, 3, 30, 61, 130, 515])), rows - len(sid))
        sid += [len(ends)] * n
        pos += range(start, start + n)
        ends.append(start + n)
    W = max(-(-e // PT) for e in ends)
    need = sum(-(-e // PT) for e in ends)
    bt = np.full((len(ends), W), -1, np.int32)
    order, at = rng.permutation(need).astype(np.int32), 0
    for s, e in enumerate(ends):
        n = -(-e // PT)
        bt[s, :n] = order[at:at + n]
        at += n
    sid, pos = np.array(sid, np.int32), np.array(pos, np.int32)
    k, v = (rng.standard_normal((rows, Hkv, D)).astype(np.float32) for _ in range(2))
    g = rkv.geometry(Hkv, D, PT, need)
    before = rng.integers(0, 256, need * rkv.page_bytes(g), dtype=np.uint8)
    pages = torch.from_numpy(before).cuda()
    rkv.append_q8(ctx, g, pages, *(torch.from_numpy(x).cuda() for x in (bt, sid, pos, k, v)))
    ctx.sync()
    want = before.copy()
    rko.paged_append(rko.layout(Hkv, D, PT, need), want, bt, sid, pos, k, v)
    assert np.array_equal(pages.cpu().numpy(), want)
