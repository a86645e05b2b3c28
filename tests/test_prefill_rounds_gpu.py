"""Portions whose key tiles are shared through LDS, behind histories of every length around the kernel's
rounds (three buffers of two tiles of 32 keys): no whole round, one, several, and each remainder; pages of
less and more than a tile, more of them than a wave keeps numbers of; a window.  Against the plain kernel,
within the same bound as the other tests of these kernels (two units of the stored type's rounding)."""
import pytest
import torch

from test_kernels_gpu import BF16, BF16_ULP, DEV, close, ops  # noqa: F401

pytestmark = pytest.mark.gpu

HELD = [0, 1, 63, 64, 127, 128, 191, 192, 193, 255, 256, 320, 383, 384, 449, 575, 576, 577, 640, 767, 768, 2200]


@pytest.mark.parametrize("H,G,D", [(8, 2, 64), (4, 1, 128)])
@pytest.mark.parametrize("ps", [16, 48, 64])
@pytest.mark.parametrize("n_new", [1, 33, 100])
@pytest.mark.parametrize("window", [0, 300])
def test_histories_around_the_rounds_of_buffers(ops, H, G, D, ps, n_new, window):  # noqa: F811
    g = torch.Generator().manual_seed(D + ps + n_new)
    need = [(a + n_new + ps - 1) // ps for a in HELD]
    T, n_pages = n_new * len(HELD), sum(need)
    q = torch.randn(T, H * D, generator=g).to(BF16).to(DEV)
    k = torch.full((n_pages + 1, G, ps, D), float("nan"), dtype=BF16)
    vt = torch.full((n_pages + 1, G, D, ps), float("nan"), dtype=BF16)
    order, at = torch.randperm(n_pages, generator=g) + 1, 0        # (the pool's first page is nobody's)
    bt = torch.full((len(HELD), max(need)), -1, dtype=torch.int32)
    pos, seg, tiles = [], [], []
    for i, a in enumerate(HELD):
        bt[i, :need[i]] = order[at:at + need[i]].int()
        at += need[i]
        for p in range(need[i]):
            n = min(ps, a + n_new - p * ps)
            k[bt[i, p], :, :n] = torch.randn(G, n, D, generator=g).to(BF16)
            vt[bt[i, p], :, :, :n] = torch.randn(G, D, n, generator=g).to(BF16)
        pos += range(a, a + n_new)
        seg += [i] * n_new
        nt = (n_new + 31) // 32
        tiles += [(i, i * n_new + 32 * t, min(32, n_new - 32 * t), t | nt << 16) for t in range(nt)]
    ints = [torch.tensor(x, dtype=torch.int32, device=DEV) for x in (pos, seg)]
    args = (q, H, G, D, k.to(DEV), vt.to(DEV), *ints, bt.to(DEV), ps, D ** -0.5)
    got = ops.paged_attention(*args, window=window, q_tiles=torch.tensor(tiles, dtype=torch.int32, device=DEV),
                              max_position=max(pos), kernel="prefill", prefill_variant=2)
    want = ops.paged_attention(*args, window=window, kernel="rows")
    close(got.float(), want.float().cpu().double(), 2 * BF16_ULP, "tiles shared through LDS")


@pytest.mark.parametrize("D,ps", [(64, (1 << 24) + (1 << 19)), (128, (1 << 23) + (1 << 17)), (256, (1 << 22) + (1 << 16))])
def test_pages_of_more_than_two_gibibytes(ops, D, ps):  # noqa: F811
    """A kv head's part of a page so large that the last places of its values lie behind 2 GiB."""
    assert (D - 1) * ps * 2 > 1 << 31
    g = torch.Generator().manual_seed(D)
    T, H, held = 40, 4, 70
    q, k, v = (torch.randn(n, D, generator=g).to(BF16) for n in (T * H, held + T, held + T))
    k_pool = torch.full((1, 1, ps, D), float("nan"), dtype=BF16, device=DEV)
    vt_pool = torch.full((1, 1, D, ps), float("nan"), dtype=BF16, device=DEV)
    k_pool[0, 0, :held + T] = k.to(DEV)
    vt_pool[0, 0, :, :held + T] = v.T.to(DEV)
    ints = [torch.tensor(x, dtype=torch.int32, device=DEV)
            for x in (range(held, held + T), [0] * T, [[0]], [(0, 0, 32, 0 | 2 << 16), (0, 32, T - 32, 1 | 2 << 16)])]
    got = ops.paged_attention(q.view(T, H * D).to(DEV), H, 1, D, k_pool, vt_pool, *ints[:3], ps, D ** -0.5,
                              q_tiles=ints[3], max_position=held + T - 1, kernel="prefill",
                              prefill_variant=0 if D == 256 else 2)
    s = q.view(T, H, D).double() @ k.double().T * D ** -0.5
    s.masked_fill_(torch.arange(held + T) > (held + torch.arange(T))[:, None, None], float("-inf"))
    close(got.float(), (s.softmax(2) @ v.double()).view(T, H * D), 2 * BF16_ULP, "large pages")
