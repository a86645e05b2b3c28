"""The forms of the block kernel that its rule chooses by size: products on both sides of every line
of the rule, against float64."""
import pytest
import torch

from test_kernels_gpu import BF16, DEV, F32, close, ops, rand  # noqa: F401

pytestmark = pytest.mark.gpu


# K ranges of 640 (two LDS buffers), 768 (four), 257 blocks of 128 x 128 (two a CU again), 140 and 139
# blocks of 256 x 256, and 272 of them (the second round mostly idle) against 392
@pytest.mark.parametrize("M,N,K,S", [(130, 264, 640, 1), (130, 264, 768, 1), (417, 520, 1536, 2),
                                     (129, 16512, 768, 1), (257, 17920, 128, 1),
                                     (200, 35584, 128, 1), (1000, 17408, 128, 1),
                                     (1759, 14336, 128, 1)])
def test_block_products_on_both_sides_of_the_rule(ops, M, N, K, S):  # noqa: F811
    x, w = rand((M, K), BF16, 71), rand((N, K), BF16, 72)
    want = x.double() @ w.double().T
    for matrix in (w.to(DEV), ops.InFragments.of(w.to(DEV))):
        if matrix is None:
            continue                     # (no whole pieces of 16 rows)
        if S == 1:
            got = ops.linear(x.to(DEV), matrix, out_dtype=F32)
        else:
            planes = ops.linear(x.to(DEV), matrix, partial_sums=True, split_k=S)
            assert planes.shape[0] == S
            got = planes.sum(0)
        # float32 sums of K exact products: K roundings of 2^-24 at the very most
        close(got, want, K * 2.0 ** -24, (M, N, K, S))
