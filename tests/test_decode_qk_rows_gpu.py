"""Decode steps of 5 to 16 rows whose attention kernel normalises, rotates and stores: the same comparison
as for a few rows (the two kernels, their pools and outputs), at the most rows the rule sends that way, over
requests of one length and of mixed lengths, in one block and split."""
import pytest

import test_kernels_gpu as kernels
from test_kernels_gpu import ops  # noqa: F401

pytestmark = pytest.mark.gpu


def test_where_the_rule_lies(ops):  # noqa: F811
    assert [ops.decode_qk_rows(d, 16) for d in (64, 128, 48, 256)] == [16, 4, 0, 0]
    assert ops.decode_qk_rows(64, 8) == 0
    # (keys over blocks: not many pairs over very long contexts; kept in one block: up to a block a CU)
    assert [ops.decode_split_takes_qk(n, 8, p) for n, p in ((4, 99999), (10, 99999), (11, 32767), (11, 32768))] == \
        [True, True, True, False]
    assert ops.decode_split_takes_qk(4, 32, 99999) and ops.decode_split_takes_qk(16, 8, 99999, 4096)
    assert [ops.decode_block_takes_qk(64, 400, 0, n) for n in (16, 256, 257)] == [True, True, False]


@pytest.mark.parametrize("H,G", [(32, 8), (16, 8), (4, 1)])
@pytest.mark.parametrize("held", [[200] * 16, [1500] * 5, [1023, 1024] * 8, [40 + i * i * 13 for i in range(16)]])
def test_the_most_rows(ops, H, G, held):  # noqa: F811
    for kernel in ("decode-split",) + (("auto",) if max(held) < 512 else ()):           # (auto: in one block)
        kernels.test_decode_attention_with_norm_rotation_and_store_inside(
            ops, (H, G, 64, 16, held, True, True, 0, True), kernel=kernel)
