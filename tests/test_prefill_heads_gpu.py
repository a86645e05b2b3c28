"""Attention over portions at head size 256, four query heads of a kv head beside each other: the same
bits as the kernel that takes every head by itself."""
import pytest
import torch

from test_kernels_gpu import BF16, DEV, ops  # noqa: F401

pytestmark = pytest.mark.gpu


# portions of less than a tile, whole tiles and one row more, behind histories that end inside a page
# or a tile; pages of 16 and of more than a key tile; a window; a sink.  What no request holds is NaN:
# places behind a request's end, pages that the window gave back and the pool's first page, which
# stands in for them
@pytest.mark.parametrize("H,G,ps", [(16, 1, 16), (8, 2, 64), (4, 1, 32)])
@pytest.mark.parametrize("window", [0, 1, 50, 2048])
@pytest.mark.parametrize("sink", [False, True])
def test_same_bits_as_a_head_by_itself(ops, H, G, ps, window, sink):  # noqa: F811
    D, held, new = 256, [0, 31, 700, 33, 5], [65, 1, 96, 32, 300]
    g = torch.Generator().manual_seed(H + ps)
    T, n_pages = sum(new), sum((a + b + ps - 1) // ps for a, b in zip(held, new))
    q = torch.randn(T, H * D, generator=g).to(BF16).to(DEV)
    k = torch.full((n_pages + 1, G, ps, D), float("nan"), dtype=BF16)
    vt = torch.full((n_pages + 1, G, D, ps), float("nan"), dtype=BF16)
    order, at = torch.randperm(n_pages, generator=g) + 1, 0
    bt = torch.full((len(new), max((a + b + ps - 1) // ps for a, b in zip(held, new))), -1,
                    dtype=torch.int32)
    pos, seg, tiles, row = [], [], [], 0
    for i, (a, b) in enumerate(zip(held, new)):
        need = (a + b + ps - 1) // ps
        bt[i, :need] = order[at:at + need].int()
        if window:                          # pages that lie before every row's window are given back
            bt[i, :max(a - window + 1, 0) // ps] = -1
        at += need
        for p in range(need):
            n = min(ps, a + b - p * ps)
            if bt[i, p] >= 0:
                k[bt[i, p], :, :n] = torch.randn(G, n, D, generator=g).to(BF16)
                vt[bt[i, p], :, :, :n] = torch.randn(G, D, n, generator=g).to(BF16)
        pos += range(a, a + b)
        seg += [i] * b
        tiles += [(i, row + t, min(32, b - t), 0) for t in range(0, b, 32)]
        row += b
    k, vt = k.to(DEV), vt.to(DEV)
    ints = [torch.tensor(x, dtype=torch.int32, device=DEV) for x in (pos, seg)]
    mods = ops.ScoreMods(0.0, None, torch.randn(H, generator=g).to(DEV)) if sink else ops.ScoreMods()
    outs = [ops.paged_attention(q, H, G, D, k, vt, *ints, bt.to(DEV), ps, D ** -0.5, window=window,
                                q_tiles=torch.tensor(tiles, dtype=torch.int32, device=DEV),
                                single_rows=False, max_position=max(pos), kernel="prefill",
                                prefill_variant=variant, mods=mods) for variant in (0, 1)]
    a, b = (o.float() for o in outs)
    assert torch.isfinite(a).all()
    assert torch.equal(a, b), ((a != b).float().mean().item(), ((a - b).abs().max()).item())
