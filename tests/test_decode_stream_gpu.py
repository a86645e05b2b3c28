"""The decode attention's stream of keys (parts of 32, page ids 64 at a time) and the decoded rows that the
tiled kernels take beside portions, against the plain kernel on the same pools."""
import math

import pytest
import torch

from test_kernels_gpu import BF16, BF16_ULP, DEV, F32, close, ops, paged_case, rand  # noqa: F401

pytestmark = pytest.mark.gpu


def on_gpu(case):
    return {k: (v.to(DEV) if torch.is_tensor(v) else v) for k, v in case.items()}


def stored(c, H, G, d, ps):
    """The new rows' keys and values put into the pools (whose free slots are NaN)."""
    kv = c["qkv"].view(c["T"], H + 2 * G, d)
    for t in range(c["T"]):
        p = int(c["row_pos"][t])
        page = int(c["bt"][int(c["row_seg"][t]), p // ps])
        c["k_pool"][page, :, p % ps] = kv[t, H:H + G]
        c["v_pool"][page, :, :, p % ps] = kv[t, H + G:]
    return c


def compare(ops, c, H, G, d, ps, window, mods=None, **kw):  # noqa: F811
    args = (c["qkv"], H, G, d, c["k_pool"], c["v_pool"], c["row_pos"], c["row_seg"], c["bt"], ps,
            1.0 / math.sqrt(d))
    want = ops.paged_attention(*args, window=window, kernel="rows", mods=mods)
    got = ops.paged_attention(*args, window=window, max_position=c["max_pos"], mods=mods, **kw)
    # both round weights and results to bfloat16: twice what one is allowed against exact numbers
    close(got.float(), want.double(), 4 * BF16_ULP, kw)


# the 64th page and the pages beside it, a part that ends inside a page, one key; a window whose first key
# lies inside a part; page sizes that are no power of two
@pytest.mark.parametrize("H,G,d,ps,window", [(8, 2, 64, 16, 0), (4, 1, 64, 48, 0), (4, 4, 128, 16, 0),
                                             (16, 1, 256, 16, 0), (6, 3, 48, 32, 0), (8, 2, 64, 16, 1100),
                                             (2, 1, 16, 16, 37)])
@pytest.mark.parametrize("kernel", ["decode-split", "decode-block"])
def test_stream_of_keys(ops, H, G, d, ps, window, kernel):  # noqa: F811
    held = [0, 30, 31, 64 * ps - 2, 64 * ps - 1, 64 * ps, 64 * ps + 33, 65 * ps, 1007, 2079]
    c = on_gpu(stored(paged_case(21, BF16, H, G, d, ps, held, [1] * len(held)), H, G, d, ps))
    compare(ops, c, H, G, d, ps, window, single_rows=True, kernel=kernel)


# decoded rows of one key to 1,500 beside portions, one of which ends in a tile of one row
@pytest.mark.parametrize("H,G,d,variant", [(4, 2, 64, 1), (16, 1, 64, 1), (32, 1, 64, 1), (6, 3, 48, 1),
                                           (8, 2, 64, 2), (16, 1, 64, 2), (4, 1, 128, 2), (16, 1, 128, 2),
                                           (2, 2, 16, 1), (8, 1, 128, 1), (4, 1, 256, 1)])
@pytest.mark.parametrize("window", [0, 100])
def test_lone_rows_among_tiles(ops, H, G, d, variant, window):  # noqa: F811
    held, new = [0, 31, 500, 0, 1499, 64, 200], [1, 1, 1, 65, 1, 33, 1]
    c = on_gpu(stored(paged_case(22, BF16, H, G, d, 16, held, new), H, G, d, 16))
    compare(ops, c, H, G, d, 16, window, q_tiles=c["q_tiles"], kernel="prefill", prefill_variant=variant)


@pytest.mark.parametrize("variant", [1, 2])
def test_lone_rows_with_a_sink(ops, variant):  # noqa: F811
    H, G, d = 8, 2, 64
    c = on_gpu(stored(paged_case(23, BF16, H, G, d, 16, [0, 300, 40], [1, 40, 1]), H, G, d, 16))
    sink = rand((H,), F32, 24).to(DEV)
    compare(ops, c, H, G, d, 16, 0, mods=ops.ScoreMods(sink=sink), q_tiles=c["q_tiles"], kernel="prefill",
            prefill_variant=variant)


def pools_for(held, G, d, ps, seed, missing=()):
    """Pools of random keys and values in which every row has pages of its own, NaN where it holds nothing;
    ``missing``: (row, page of the row) that its table does not name."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    pages = [p // ps + 1 for p in held]
    shape = (sum(pages) + 1, G, ps, d)
    k = torch.randn(shape, generator=gen, device=DEV).to(BF16)
    v = torch.randn(shape, generator=gen, device=DEV).to(BF16).transpose(2, 3).contiguous()
    order = torch.randperm(sum(pages), generator=gen, device=DEV) + 1      # (page 0 is nobody's)
    bt = torch.full((len(held), max(pages) + 2), -1, dtype=torch.int32, device=DEV)
    at = 0
    for r, (p, n) in enumerate(zip(held, pages)):
        bt[r, :n] = order[at:at + n]
        last = int(order[at + n - 1])
        k[last, :, p % ps + 1:] = float("nan")
        v[last, :, :, p % ps + 1:] = float("nan")
        at += n
    k[0], v[0] = float("nan"), float("nan")
    for r, page in missing:
        bt[r, page] = -1
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)  # noqa: E731
    return k, v, bt, i32(held), torch.arange(len(held), dtype=torch.int32, device=DEV)


# a wave walks the whole of every row (as many rows and kv heads as there are blocks to split keys over): one part
# of 32 keys to fifteen, which is none to three rounds of the parts under way and every rest; pages of 64 by 64
@pytest.mark.parametrize("H,G,d,ps", [(64, 64, 64, 16), (128, 64, 128, 16), (64, 64, 16, 16), (64, 64, 32, 32),
                                      (64, 64, 48, 16), (64, 64, 192, 16), (64, 64, 256, 16), (64, 64, 80, 48)])
def test_every_number_of_parts(ops, H, G, d, ps):  # noqa: F811
    held = [32 * n + o for n in range(15) for o in (0, 1, 13, 31)] + [64 * ps + o for o in (-1, 0, 33, 127)]
    k, v, bt, pos, seg = pools_for(held, G, d, ps, 41)
    assert ops.decode_splits(32, len(held), G, max(held) + 1)[1] == 1
    q = rand((len(held), H * d), BF16, 42).to(DEV)
    args = (q, H, G, d, k, v, pos, seg, bt, ps, 1.0 / math.sqrt(d))
    want = ops.paged_attention(*args, kernel="rows")
    for kernel in ("decode-split", "decode-block"):
        got = ops.paged_attention(*args, single_rows=True, max_position=max(held), kernel=kernel)
        close(got.float(), want.float().cpu().double(), 4 * BF16_ULP, kernel)


# pages that a window has passed, in the part of the first key that it sees; a page among those that a row sees,
# whose keys and values read as zero
@pytest.mark.parametrize("window", [0, 45])
@pytest.mark.parametrize("kernel", ["decode-split", "decode-block"])
def test_pages_that_are_not_there(ops, window, kernel):  # noqa: F811
    H, G, d, ps = 4, 2, 64, 16
    held = [200, 77, 95, 300]
    gone = [(0, 11), (1, 4), (3, 18)] + ([(r, p) for r, n in enumerate(held)
                                         for p in range((n + 1 - window) // ps)] if window else [(2, 0)])
    k, v, bt, pos, seg = pools_for(held, G, d, ps, 43, gone)
    q = rand((len(held), H * d), BF16, 44)
    got = ops.paged_attention(q.to(DEV), H, G, d, k, v, pos, seg, bt, ps, 0.2, window=window, single_rows=True,
                              max_position=max(held), kernel=kernel)
    want = torch.zeros(len(held), H, d, dtype=torch.float64)
    kc, vc, tables = k.cpu().double(), v.cpu().double().transpose(2, 3), bt.cpu()
    for r, n in enumerate(held):
        keys = range(max(0, n + 1 - window) if window else 0, n + 1)
        for h in range(H):
            page = [int(tables[r, i // ps]) for i in keys]
            kk = torch.stack([kc[p, h // 2, i % ps] if p >= 0 else torch.zeros(d).double()
                              for p, i in zip(page, keys)])
            vv = torch.stack([vc[p, h // 2, i % ps] if p >= 0 else torch.zeros(d).double()
                              for p, i in zip(page, keys)])
            want[r, h] = torch.softmax(kk @ q.double().view(-1, H, d)[r, h] * 0.2, 0) @ vv
    # (weights and results are rounded to bfloat16)
    close(got.float(), want.view(len(held), -1), 2 * BF16_ULP, kernel)


# Two maps whose difference is the result (head size 16, the second map uniform over all keys): what bfloat16
# results leave of it when exact maps are rounded is the floor; shares of a row's keys over waves and blocks may
# add the rounding of their weights, less than half as much again.
@pytest.mark.parametrize("window", [0, 70, 200])
@pytest.mark.parametrize("d,T", [(16, 360), (48, 330), (16, 1500)])
def test_difference_of_two_maps(ops, window, d, T):  # noqa: F811
    ps, lam, needle, portion = 16, 0.9, 100, 40
    x = 0.05 * rand((T, 2, d), F32, 45)
    x[needle] = 3.0
    x[needle, :, ::2] += 4.0
    x[needle + 1:] += 0.35                       # every later query looks for that key
    x = x.to(BF16)
    val = rand((T, 2, d), BF16, 46)
    keys, vals = torch.zeros(T, 4, d, dtype=BF16), torch.zeros(T, 4, d, dtype=BF16)
    keys[:, ::2], vals[:, ::2], vals[:, 1::2] = x, val, val
    n_pages = T // ps + 1
    k = torch.full((n_pages, 4, ps, d), float("nan"), dtype=BF16)
    v = torch.full((n_pages, 4, d, ps), float("nan"), dtype=BF16)
    for t in range(T):
        k[t // ps, :, t % ps], v[t // ps, :, :, t % ps] = keys[t], vals[t]
    pos = list(range(T - 30, T)) + [needle + (window or 150) + i for i in range(-2, 3)]
    n = len(pos)
    exact = torch.zeros(n, 4, d, dtype=torch.float64)
    for r, p in enumerate(pos):
        seen = slice(max(0, p + 1 - window) if window else 0, p + 1)
        for h in range(4):
            exact[r, h] = torch.softmax(keys[seen, h].double() @ keys[p, h].double(), 0) @ vals[seen, h].double()

    def result(maps):
        o = maps[:, ::2] - lam * maps[:, 1::2]
        return o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5)
    want = result(exact)
    floor = float((result(exact.to(BF16).double()) - want).abs().max())
    on = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)  # noqa: E731
    q = torch.cat([keys[pos], torch.zeros(portion, 4, d, dtype=BF16)]).view(n + portion, -1).to(DEV)
    bt = torch.arange(n_pages, dtype=torch.int32, device=DEV).repeat(64 * n + 1, 1)
    tiles = [(r, r, 1, 1 << 16) for r in range(n)] + [(n, n, 32, 2 << 16), (n, n + 32, 8, 1 | 2 << 16)]
    common = dict(window=window, max_position=T - 1)
    args = lambda rows: (q[rows], 4, 4, d, k.to(DEV), v.to(DEV), on(pos + list(range(portion)))[rows],  # noqa: E731
                         on(list(range(n)) + [n] * portion)[rows], bt, ps, 1.0)
    every = torch.arange(n + portion, device=DEV)
    many = torch.arange(n, device=DEV).repeat(6)       # rows enough that the shares are planned
    got = {"beside a portion": ops.paged_attention(*args(every), q_tiles=on(tiles), kernel="prefill", **common)[:n],
           "split": ops.paged_attention(*args(many), single_rows=True, kernel="decode-split", **common)[:n],
           "block": ops.paged_attention(*args(every[:n]), single_rows=True, kernel="decode-block", **common)}
    for what, ctx in got.items():
        err = float((result(ctx.cpu().double().view(n, 4, d)) - want).abs().max())
        assert err <= 1.5 * floor + 1e-4, (what, err, floor)


# shares that come from the rows' own lengths and are no whole number of the smallest ones: the kernel and the merge
# behind it settle on the same
@pytest.mark.parametrize("d,G,keys", [(64, 8, 2600), (128, 8, 1700), (48, 8, 2600), (256, 4, 900)])
@pytest.mark.parametrize("softcap", [0.0, 20.0])
def test_planned_shares(ops, d, G, keys, softcap):  # noqa: F811
    H, ps, T = 2 * G, 16, 64
    held = [keys - 1 - (r * 7) % 50 for r in range(T)]
    k, v, bt, pos, seg = pools_for(held, G, d, ps, 47)
    q = rand((T, H * d), BF16, 48).to(DEV)
    mods = ops.ScoreMods(softcap=softcap) if softcap else None
    args = (q, H, G, d, k, v, pos, seg, bt, ps, 1.0 / math.sqrt(d))
    want = ops.paged_attention(*args, kernel="rows", mods=mods)
    got = ops.paged_attention(*args, single_rows=True, max_position=max(held), kernel="decode-split", mods=mods)
    close(got.float(), want.float().cpu().double(), 4 * BF16_ULP, (d, softcap))
