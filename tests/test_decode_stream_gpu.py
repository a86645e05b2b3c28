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
