"""The decode attention that keeps a row's keys in one block: with the norm, the rotation and the store
in its prologue against the two kernels, and the rule that chooses between blocks and splits."""
import math

import pytest
import torch

from test_decode_stream_gpu import compare, on_gpu, stored
from test_kernels_gpu import (BF16, BF16_ULP, DEV, F32, close, ops, paged_case, rand,  # noqa: F401
                              rope_tables)

pytestmark = pytest.mark.gpu


# fewer parts of 32 keys than waves, one to a wave, one more; the last key the first of a part and the
# last of a page; windows that start inside a part
@pytest.mark.parametrize("H,G,ps,window", [(8, 4, 16, 0), (32, 8, 16, 0), (16, 1, 16, 0), (3, 3, 32, 0),
                                           (8, 2, 16, 37), (8, 2, 16, 300)])
@pytest.mark.parametrize("store", [True, False])
def test_prologue_in_a_block(ops, H, G, ps, window, store):  # noqa: F811
    d = 64
    held = [0, 31, 32, 255, 256, 287, 511, 495]
    if window:
        held[-1] = 1500
    for some in (held[:4], held[4:]):
        c = on_gpu(paged_case(31, BF16, H, G, d, ps, some, [1] * len(some)))
        if not store:                    # the layer whose keys are read has stored this step's already
            c = on_gpu(stored(c, H, G, d, ps))
        assert ops.decode_block_takes_qk(d, c["max_pos"], window)
        qn, kn = (1 + rand((d,), F32, 30, 0.2)).to(DEV), (1 + rand((d,), F32, 31, 0.2)).to(DEV)
        cos, sin = (t.to(DEV) for t in rope_tables(max(some) + 1, d))
        k1, v1, k2, v2 = (c[n].clone() for n in ("k_pool", "v_pool") * 2)
        q = ops.qk_norm_rope_store(c["qkv"].clone(), H, G, d, qn, kn, 1e-5, cos, sin, d, 1, k1, v1,
                                   c["row_pos"], c["row_seg"], c["bt"], ps, store_kv=store)
        args = (c["row_pos"], c["row_seg"], c["bt"], ps, 1 / math.sqrt(d))
        kw = dict(window=window, single_rows=True, max_position=c["max_pos"])
        want = ops.paged_attention(q, H, G, d, k1, v1, *args, kernel="rows", **kw)
        got = ops.paged_attention(c["qkv"], H, G, d, k2, v2, *args, kernel="decode",
                                  qk=ops.QkPrologue(qn, kn, 1e-5, cos, sin, store_kv=store), **kw)
        flat = lambda t: torch.nan_to_num(t.float().cpu(), nan=-7.0)  # noqa: E731
        assert torch.equal(flat(v1), flat(v2)), "v pages"
        close(flat(k2), flat(k1).double(), BF16_ULP, "k pages")
        # (weights are rounded to bfloat16 and a key may differ in its last bit: two roundings)
        close(got.float(), want.float().cpu().double(), 2 * BF16_ULP, "attention")


# (a long row among short ones is the whole step's time in one block: from 192 blocks on 2,048 keys of 64 and 1,024 of
# 128, however many the blocks)
@pytest.mark.parametrize("rows,G,d,keys", [(1, 8, 64, 512), (8, 8, 64, 1024), (24, 8, 64, 2048),
                                           (64, 8, 64, 2048), (1, 8, 128, 512), (64, 4, 128, 1024),
                                           (16, 4, 128, 512), (64, 1, 48, 512), (64, 8, 256, 512),
                                           (16, 8, 256, 256), (15, 8, 192, 128), (1, 1, 256, 128)])
def test_most_keys_of_a_block(ops, rows, G, d, keys):  # noqa: F811
    form = lambda n: ops.decode_form(2 * G, G, d, n - 1, n_rows=rows)  # noqa: E731
    assert form(keys + 1) == "decode-split"
    assert keys == 0 or form(keys) == "decode-block"
    if keys > 512:
        assert ops.decode_form(2 * G, G, d, keys - 1, n_rows=rows, scored=True) == "decode-split"


def test_few_waves_a_block(ops):  # noqa: F811
    """Sixteen query heads of 256 on a kv head leave a block three waves: only with blocks for every CU."""
    form = lambda rows, n: ops.decode_form(16, 1, 256, n - 1, n_rows=rows)  # noqa: E731
    assert form(8, 40) == form(255, 40) == form(256, 513) == "decode-split"
    assert form(256, 512) == "decode-block"


@pytest.mark.parametrize("H,G,d,held", [(4, 2, 64, [0, 1023, 700, 33] * 8), (32, 16, 64, [2047, 5, 1024] * 4),
                                        (8, 8, 64, [4095, 0, 3000, 64] * 8)])
def test_many_rows_in_blocks(ops, H, G, d, held):  # noqa: F811
    assert max(held) > 2047 or ops.decode_form(H, G, d, max(held), n_rows=len(held)) == "decode-block"
    c = on_gpu(stored(paged_case(33, BF16, H, G, d, 16, held, [1] * len(held)), H, G, d, 16))
    compare(ops, c, H, G, d, 16, 0, single_rows=True, kernel="decode-block")
