"""How many ranges of K a product of many rows is cut into, and what its sums are handed on as."""
import numpy as np
import pytest
import torch

from kappai_amd.kernels import ops

# products over fragment order that are fastest over one range and over rows of W over two or more
ONE_RANGE = [(1600, 1024, 1024), (2100, 2048, 8192), (2880, 2048, 8192), (3300, 2048, 8192), (2880, 2048, 10752),
             (4200, 1024, 4608), (1700, 1024, 1024)]


@pytest.mark.parametrize("M,N,K", ONE_RANGE + [(1040, 1024, 1024), (3200, 1536, 6912), (600, 2048, 1024)])
def test_sums_that_were_float_stay_float(M, N, K):
    assert ops.sums_in_f32(M, N, K)


@pytest.mark.parametrize("M,N,K", [(2048, 1024, 1024), (4200, 2048, 2048), (2048, 6144, 2048), (200, 16384, 2048)])
def test_one_range_in_bfloat16(M, N, K):
    assert ops.split_k_for(M, N, K) == 1 and not ops.sums_in_f32(M, N, K)


def test_several_ranges_are_float():
    for M, N, K in ((300, 1024, 4608), (100, 2048, 2048), (8, 2048, 8192), (40, 1024, 4608), (575, 2048, 2048)):
        assert ops.split_k_for(M, N, K) > 1 and ops.sums_in_f32(M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", ONE_RANGE[:3])
def test_float_sums_over_one_range(M, N, K):
    """Against float64, by themselves and in the norm that takes them; bfloat16 would be off by 2^-9."""
    from test_kernels_gpu import BF16, DEV, F32, close, rand, ref
    x, w = rand((M, K), BF16, 91), rand((N, K), BF16, 92, 0.05)
    got = ops.linear(x.to(DEV), ops.InFragments.of(w.to(DEV)), partial_sums=True)
    assert got.dtype == F32 and tuple(got.shape) == (ops.split_k_for(M, N, K), M, N)
    close(got.sum(0), x.double() @ w.double().T, (K + 1) * 2.0 ** -24, "the sums")
    resid, wn = rand((M, N), F32, 93, 2.0), 1 + rand((N,), F32, 94, 0.1)
    on_gpu = resid.to(DEV).clone()
    ops.add_rmsnorm(on_gpu, got, wn.to(DEV), 1e-5, BF16)
    want = resid.clone()
    ref.add_rmsnorm(want, got.cpu(), wn, 1e-5, F32)
    close(on_gpu, want, 1e-6, "the stream")


@pytest.mark.parametrize("M,N,K,ranges", [(1400, 2040, 8192, 4), (2880, 2040, 8192, 2), (3072, 1000, 4096, 1),
                                          (417, 1032, 1024, 4)])
def test_rows_of_w_take_the_ranges_of_their_own_kernels(M, N, K, ranges):
    """A matrix whose rows are no multiple of 16 lies as rows and goes through kernels of its own."""
    assert ops.split_k_for(M, N, K) == ranges and ops.sums_in_f32(M, N, K) == (ranges > 1)


# the largest operands that the block products over fragment order take: 2^31 elements less one row
@pytest.mark.parametrize("rows,stride,K,ranges", [(4095, 524280, 524160, 1), (2097151, 1024, 1024, 2),
                                                  (131071, 16384, 10752, 3), (200, 8, 128, 1)])
@pytest.mark.parametrize("block", [256, 192, 128])
def test_loads_of_the_largest_operands(rows, stride, K, ranges, block):
    """The 32-bit offsets of A's loads in gemm_bf16_direct and gemm_bf16_staged (row times stride in bytes, what is
    left of 2^32 where a row past the end runs over) against the bytes that the buffer is given: a row that is there
    is read where it lies and whole; no load, of whatever row, ends outside the operand."""
    stride = max(stride, K)
    assert rows * stride < 2 ** 31
    K_range = K // ranges
    size = (rows - 1) * stride * 2 + K_range * 2                # of the buffer, from the range's first column on
    assert size < 2 ** 32
    blocks = (rows + block - 1) // block
    row = np.unique(np.r_[0:block, rows - 1, np.arange((blocks - 1) * block, blocks * block)]).astype(np.int64)
    chunk = np.arange(0, 128, 16)
    lane = ((row[:, None] * stride * 2) % 2 ** 32 + chunk).astype(np.int64)
    for tile in (0, K_range // 64 - 1):
        end = lane + tile * 128 + 16
        there = row < rows
        assert (end[there] <= size).all()
        assert (lane[there] == row[there][:, None] * stride * 2 + chunk).all()
        read = lane + tile * 128 < size                         # (what reaches the end is not read)
        assert (end[read] <= rows * stride * 2).all()
