"""The block products over a matrix in fragment order (256 x 256 and 256 x 192 blocks with W's pieces in
registers, 256 x 128 down to 64 x 64 with both operands in LDS), at sizes that end inside a block
and at the shortest runs of K, against the same product over the matrix's rows (bit for bit: every form adds
16 of K after 16) and against float64."""
import ctypes

import pytest
import torch

from test_block_shapes import FEW, WHOLE
from test_kernels_gpu import BF16, DEV, F32, close, ops, rand  # noqa: F401

pytestmark = pytest.mark.gpu
FORMS = {"256x256": 7, "256x192": 11, "256x128": 14, "192x128": 13, "128x128": 10, "64x128": 15, "128x64": 16, "64x64": 17}
ROWS = 8                       # the kernel for rows, 128 x 128 blocks


# one row beside whole blocks, a single piece of 16 columns in the last block, K of two, three and five
# pairs of 64 (fewer tiles than are under way at once), an odd number of ranges, a row stride
@pytest.mark.parametrize("M,N,K,S", [(129, 144, 128, 1), (193, 272, 384, 3), (257, 208, 640, 1),
                                     (384, 1040, 1280, 2), (513, 400, 256, 2), (65, 2064, 1024, 1)])
@pytest.mark.parametrize("form", list(FORMS))
def test_blocks_over_fragment_order(ops, M, N, K, S, form):  # noqa: F811
    wide = rand((M, K + 40), BF16, 81).to(DEV)
    x, w, b = wide[:, :K], rand((N, K), BF16, 82).to(DEV), rand((N,), F32, 83).to(DEV)
    kept = ops.InFragments.of(w)
    want = x.double() @ w.double().T
    for out_dtype, bias in ((F32, None), (F32, b), (BF16, b)):
        got = ops.linear(x, kept, bias, out_dtype=out_dtype, force_kernel=FORMS[form])
        assert torch.equal(got, ops.linear(x, w, bias, out_dtype=out_dtype, force_kernel=ROWS))
        if out_dtype == F32:       # float32 sums of K exact products: K roundings of 2^-24 at the most
            close(got, want + (0 if bias is None else bias.double()), (K + 1) * 2.0 ** -24, form)
    if S > 1:
        planes = ops.linear(x, kept, partial_sums=True, split_k=S, force_kernel=FORMS[form])
        assert planes.shape == (S, M, N)
        assert torch.equal(planes, ops.linear(x, w, partial_sums=True, split_k=S, force_kernel=ROWS))


@pytest.mark.parametrize("M,F,K", [(129, 16, 128), (193, 144, 256), (257, 112, 384), (520, 1040, 640)])
@pytest.mark.parametrize("form", list(FORMS))
def test_gated_blocks_over_fragment_order(ops, M, F, K, form):  # noqa: F811
    x = rand((M, K), BF16, 84).to(DEV)
    w = ops.interleave_gate_up(rand((F, K), BF16, 85, 0.2).to(DEV), rand((F, K), BF16, 86, 0.2).to(DEV))
    got = ops.linear_swiglu(x, ops.InFragments.of(w), force_kernel=FORMS[form])
    assert torch.equal(got, ops.linear_swiglu(x, w, force_kernel=ROWS))


# the rule's own choices, one product or more for every form (test_block_shapes.py has which)
@pytest.mark.parametrize("M,N,K", list(WHOLE))
def test_the_rule_takes_every_form(ops, M, N, K):  # noqa: F811
    x, w = rand((M, K), BF16, 87).to(DEV), rand((N, K), BF16, 88).to(DEV)
    assert torch.equal(ops.linear(x, ops.InFragments.of(w)), ops.linear(x, w, force_kernel=ROWS))


# 25 to 128 rows: blocks where the rule names some, else the kernel with 32 x 32 tiles, which adds in another order
@pytest.mark.parametrize("sizes", [s for s in FEW if s[0] <= 128])
def test_what_25_to_128_rows_take(ops, sizes):  # noqa: F811
    M, n, K, S, elem, gated = sizes
    x, w = rand((M, K), BF16, 93).to(DEV), ops.InFragments.of(rand((n, K), BF16, 94, 0.05).to(DEV))

    def product(force):
        if gated:
            return ops.linear_swiglu(x, w, force_kernel=force)
        how = dict(partial_sums=True, split_k=S) if S > 1 else dict(out_dtype=F32 if elem == 4 else BF16)
        return ops.linear(x, w, force_kernel=force, **how)
    blocks, tiles = product(FORMS["64x64"]), product(18)
    assert torch.equal(product(0), tiles if FEW[sizes] == "rows32" else blocks)
    if K // S > 256:                      # (float sums of one run of 256 may agree, and rounded ones do mostly)
        assert gated or elem == 2 or not torch.equal(tiles, blocks)


# blocks that end behind the last row and the last column, and columns between the rows of the result: nothing is
# written there, in one plane and in three, and what lies behind x and between its rows reaches no result
@pytest.mark.parametrize("M,N,K,S", [(200, 272, 384, 1), (129, 144, 768, 3), (385, 400, 256, 1)])
@pytest.mark.parametrize("form", list(FORMS))
def test_nothing_is_written_behind_the_result(ops, M, N, K, S, form):  # noqa: F811
    mark, ldc = -123.5, N + 24
    wide = torch.full((M + 200, K + 8), float("nan"), dtype=BF16, device=DEV)
    wide[:M, :K] = rand((M, K), BF16, 89).to(DEV)
    x, w = wide[:M, :K], rand((N, K), BF16, 90).to(DEV)
    if S == 1:
        want = ops.linear(x.contiguous(), w, force_kernel=ROWS, out_dtype=F32)[None]
    else:
        want = ops.linear(x.contiguous(), w, partial_sums=True, split_k=S, force_kernel=ROWS)
    out = torch.full((S * M + 300, ldc), mark, dtype=F32, device=DEV)
    i, none = ctypes.c_int, ctypes.c_void_p(0)
    at = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    frag = ops.fragment_order(w)
    status = ops.library("gemm").kappai_gemm_bf16(
        at(x), none, at(frag), none, at(out), i(M), i(N), i(K), i(x.stride(0)), i(ldc), i(1), i(FORMS[form]), i(S),
        i(0), none, i(0), ctypes.c_float(0), none, i(0), none, none, i(0), none,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert status == 0
    assert torch.equal(out[:S * M, :N].view(S, M, N), want)
    assert (out[:, N:] == mark).all() and (out[S * M:] == mark).all()


@pytest.mark.parametrize("M,F,K", [(129, 144, 256), (385, 208, 384)])
@pytest.mark.parametrize("form", list(FORMS))
def test_nothing_is_written_behind_the_gated_result(ops, M, F, K, form):  # noqa: F811
    mark, ldc = -123.5, F + 24
    x = rand((M, K), BF16, 84).to(DEV)
    w = ops.interleave_gate_up(rand((F, K), BF16, 85, 0.2).to(DEV), rand((F, K), BF16, 86, 0.2).to(DEV))
    out = torch.full((M + 300, ldc), mark, dtype=BF16, device=DEV)
    i, none = ctypes.c_int, ctypes.c_void_p(0)
    at = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    frag = ops.fragment_order(w)
    status = ops.library("gemm").kappai_gemm_bf16_swiglu(
        at(x), none, at(frag), at(out), i(M), i(F), i(K), i(K), i(ldc), i(FORMS[form]), i(0), none, i(0),
        ctypes.c_float(0), i(0), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert status == 0
    assert torch.equal(out[:M, :F], ops.linear_swiglu(x, w, force_kernel=ROWS))
    assert (out[:, F:] == mark).all() and (out[M:] == mark).all()


# more row tiles than a group of neighbours takes, groups that are not all of one size, a number of blocks that is
# no multiple of eight: every block of every range has its place
@pytest.mark.parametrize("M,N,K,S", [(1900, 384, 256, 2), (2180, 656, 384, 3), (4500, 144, 128, 1),
                                     (1100, 2576, 256, 1)])
@pytest.mark.parametrize("form", list(FORMS))
def test_every_block_has_its_place(ops, M, N, K, S, form):  # noqa: F811
    x, w = rand((M, K), BF16, 91).to(DEV), rand((N, K), BF16, 92).to(DEV)
    kept = ops.InFragments.of(w)
    how = dict(partial_sums=True, split_k=S) if S > 1 else dict(out_dtype=F32)
    assert torch.equal(ops.linear(x, kept, force_kernel=FORMS[form], **how),
                       ops.linear(x, w, force_kernel=ROWS, **how))
