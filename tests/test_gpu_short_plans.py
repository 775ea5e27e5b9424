"""Device-chosen partitions of batches that do not fill the machine: the
shortest partition is 1, 2 or 4 tiles by batch size and rows, and up to eight
tiles stay one partition that needs no workspace.  Lengths at the edges of
tiles and of those rules against the oracle."""
import math

import numpy as np
import pytest

from tests.test_gpu_parity import Scene, _bind_ctx, _run_decode, assert_close  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hkv,D,PT,lens,q_len", [
    (8, 2, 128, 16, [300], 1),                            # one-tile partitions
    (4, 1, 128, 16, [1], 1),
    (16, 2, 256, 64, [97], 1),                            # whole: three tiles and a token
    (16, 2, 256, 64, [96], 1),
    (16, 2, 256, 32, [2048], 1),                          # 128 one-tile partitions
    (16, 2, 256, 32, [2080], 1),                          # past them: two tiles each
    (16, 4, 256, 16, [33, 500, 1, 64, 65], 1),
    (32, 1, 256, 64, [161, 129, 128], 1),                 # whole: 32 rows of one token
    (32, 4, 128, 32, [130, 257, 31], 4),                  # 32 rows: four-tile partitions
    (48, 8, 128, 16, [161, 90, 158, 33, 129] * 8, 3),     # one partition of up to six tiles
    (48, 8, 128, 16, [289, 90, 257, 33, 129] * 8, 3),     # past them: four-tile partitions
])
def test_short_plans(rkv, rko, ctx, Hq, Hkv, D, PT, lens, q_len):
    print(f"short plan Hq={Hq} Hkv={Hkv} D={D} PT={PT} lens={lens[:6]} q_len={q_len}", flush=True)
    sc = Scene(rkv, rko, Hkv, D, PT, [max(L, q_len) for L in lens], seed=sum(lens))
    rng = np.random.default_rng(len(lens))
    q = rng.standard_normal((len(lens), q_len, Hq, D)).astype(np.float32)
    scale = 1.0 / math.sqrt(D)
    got, _ = _run_decode(rkv, ctx, sc, q, scale, q_len=q_len, partition_tokens=0)
    one = max(32, PT) * max(1, math.ceil(max(sc.lens) / max(32, PT)))
    whole, _ = _run_decode(rkv, ctx, sc, q, scale, q_len=q_len, partition_tokens=min(one, 64 * PT))
    # split against unsplit: f32 sums in another order
    assert np.abs(got - whole).max() <= 1e-5 * max(1.0, np.abs(whole).max())
    for b in range(len(lens)):
        for j in range(q_len):
            n = np.array([sc.lens[b] - q_len + j + 1], np.int32)
            want = rko.paged_decode(sc.lay, sc.pages, sc.bt[b:b + 1], n, np.zeros(1, np.int32), q[b:b + 1, j:j + 1],
                                    scale, 1024)
            assert_close(got[b:b + 1, j:j + 1], want, what=f"entry {b} row {j}")


def test_short_calls_need_no_workspace(rkv, rko, ctx):
    """Up to 256 tokens a call runs whole without a workspace, with a small and
    with a large one; above that a workspace of the largest call of a loop
    holds every smaller one."""
    import torch
    Hq, Hkv, D, PT = 16, 2, 256, 32
    sc = Scene(rkv, rko, Hkv, D, PT, [256, 200, 9], seed=4)
    q = torch.randn((3, 1, Hq, D), device="cuda")
    ids = torch.arange(3, dtype=torch.int32, device="cuda")
    outs = []
    for ws in (None, torch.empty(64, dtype=torch.uint8, device="cuda"),
               torch.empty(1 << 22, dtype=torch.uint8, device="cuda")):
        out = torch.empty_like(q)
        a = rkv.decode_args(q, out, ids, 1 / math.sqrt(D), 256, workspace=ws)
        rkv.decode_q8(ctx, sc.g, sc.pages_d, sc.bt_d, sc.lens_d, a)
        ctx.sync()
        outs.append(out.cpu().numpy())
    assert np.array_equal(outs[0], outs[1])
    assert np.abs(outs[0] - outs[2]).max() <= 1e-5  # split: f32 sums in another order
    need = {}
    for b in (1, 2, 3, 8, 64):
        for n in (257, 300, 2048, 2080, 4096, 40000):
            qq = torch.empty((b, 1, Hq, D), device="cuda")
            a = rkv.decode_args(qq, qq, torch.zeros(b, dtype=torch.int32, device="cuda"), 1.0, n)
            need[b, n] = rkv.decode_workspace_bytes(sc.g, a)
    for (b, n), x in need.items():
        assert all(x <= y for (c, m), y in need.items() if c >= b and m >= n), (b, n)


@pytest.mark.parametrize("Hq,Hkv,D,lens,q_len", [
    (8, 2, 128, [256], 1),
    (16, 2, 256, [256, 200, 9], 1),
    (16, 2, 256, [97, 256, 130, 255], 4),   # 32 rows
])
def test_short_calls_leave_a_workspace_alone(rkv, rko, ctx, Hq, Hkv, D, lens, q_len):
    """Up to 256 tokens a call writes none of a workspace that it is given, so
    calls that overlap may share one, and its bits are those of a call without
    one and of the no-alloc call."""
    import torch
    sc = Scene(rkv, rko, Hkv, D, 32, lens, seed=sum(lens))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(D)
    q = torch.randn((len(lens), q_len, Hq, D), generator=gen, device="cuda")
    ids = torch.arange(len(lens), dtype=torch.int32, device="cuda")
    ws = torch.full((1 << 22,), 0xA5, dtype=torch.uint8, device="cuda")
    outs = []
    for call, given in ((rkv.decode_q8, ws), (rkv.decode_q8, None), (rkv.decode_q8_noalloc, None)):
        out = torch.full_like(q, float("nan"))
        call(ctx, sc.g, sc.pages_d, sc.bt_d, sc.lens_d,
             rkv.decode_args(q, out, ids, 1 / math.sqrt(D), 256, q_len=q_len, workspace=given))
        ctx.sync()
        outs.append(out)
    assert bool((ws == 0xA5).all())
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
