"""Export and import at the edges of the tiles that their kernels move whole:
part-filled tiles, odd row counts, pointers of any alignment.  Bit-exact."""
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
