"""The store of values where a wave turns eight rows over and stores a column's 16 bytes: portions that begin
at every place of an eight, rows of several requests in one eight, page and head sizes around the limits;
the pools' bits against the kernel's own input, places of nobody untouched.  (Queries and keys: the tests of
the kernel beside the plain one.)"""
import pytest
import torch

from kappai_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV, BF16 = "cuda:0", torch.bfloat16


@pytest.mark.parametrize("H,G,d", [(4, 2, 16), (3, 1, 32), (4, 2, 64), (5, 5, 128), (2, 1, 256), (1, 3, 64)])
@pytest.mark.parametrize("ps", [4, 8, 16, 24])
@pytest.mark.parametrize("held,new", [([0], [64]), ([8, 3, 0], [24, 17, 40]), ([5, 16, 7], [1, 1, 1]),
                                      ([0, 8, 16], [8, 8, 9])])
@pytest.mark.parametrize("parts", [0, 2])
def test_values_lie_where_their_positions_say(H, G, d, ps, held, new, parts):
    g = torch.Generator().manual_seed(d + ps)
    need = [(a + b + ps - 1) // ps for a, b in zip(held, new)]
    T, pages = sum(new), sum(need) + 1
    order, at, pos, seg = torch.randperm(pages, generator=g), 0, [], []
    bt = torch.full((len(new), max(need)), -1, dtype=torch.int32)
    for i, n in enumerate(need):
        bt[i, :n] = order[at:at + n].int()
        at += n
        pos += range(held[i], held[i] + new[i])
        seg += [i] * new[i]
    x = torch.randn(max(parts, 1), T, (H + 2 * G) * d, generator=g)
    total = x[0] + x[1] if parts else x[0].to(BF16).float()
    k = torch.full((pages, G, ps, d), 7.0, dtype=BF16, device=DEV)
    v = torch.full((pages, G, d, ps), 7.0, dtype=BF16, device=DEV)
    ints = [torch.tensor(t, dtype=torch.int32, device=DEV) for t in (pos, seg)]
    tab = torch.ones(max(pos) + 1, d // 2, device=DEV)
    ops.qk_norm_rope_store((x if parts else x[0].to(BF16)).contiguous().to(DEV), H, G, d, None, None, 1e-5, tab, tab,
                           0, 0, k, v, *ints, bt.to(DEV), ps)
    want_k, want_v = torch.full_like(k, 7.0).cpu(), torch.full_like(v, 7.0).cpu()
    rows = total.to(BF16).view(T, H + 2 * G, d)
    for t in range(T):
        page = int(bt[seg[t], pos[t] // ps])
        want_k[page, :, pos[t] % ps] = rows[t, H:H + G]
        want_v[page, :, :, pos[t] % ps] = rows[t, H + G:]
    assert torch.equal(v.cpu(), want_v) and torch.equal(k.cpu(), want_k)
