"""Float32 products of few rows that norm the stream themselves and that add into it, against the norm's kernel, the
product and the sum one behind the other: bit for bit, at sizes around a turn of 512 values, a block's columns and
both forms of the product."""
import ctypes

import pytest
import torch

from test_kernels_gpu import DEV, F32, ops, rand  # noqa: F401

pytestmark = pytest.mark.gpu
I = ctypes.c_int


def p(t):
    return ctypes.c_void_p(0 if t is None else t.data_ptr())


def stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("K", [128, 512, 640, 1024, 1536, 2048])
@pytest.mark.parametrize("N", [3, 1000, 2048, 2050, 3080])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
def test_a_product_that_norms_its_rows(ops, M, N, K):  # noqa: F811
    lib = ops.library("gemm")
    x, w = rand((M, K), F32, 1, 3.0).to(DEV), rand((N, K), F32, 2).to(DEV)
    norm_w, bias, eps = rand((K,), F32, 3).to(DEV), rand((N,), F32, 4).to(DEV), 1e-5
    out = torch.full((M, N), -7.0, device=DEV)
    args = [p(x), p(norm_w), ctypes.c_float(eps), p(w), p(bias), p(out), I(M), I(N), I(K), I(N)]
    fits = M * -(-K // 512) <= 16
    assert bool(lib.kappai_gemm_f32_norms(I(M), I(K))) == fits
    status = lib.kappai_gemm_f32_normed(*args, I(0), stream())
    assert (status == 0) == fits
    if not fits:
        return
    rows = ops.add_rmsnorm(x.clone(), None, norm_w, eps, F32)
    assert torch.equal(out, ops.linear(rows, w, bias))
    F = N // 2
    if F and lib.kappai_gemm_f32_gates(I(M), I(F), I(K)):
        wide = w[:2 * F].contiguous()
        gated = torch.full((M, F), -7.0, device=DEV)
        assert lib.kappai_gemm_f32_normed(p(x), p(norm_w), ctypes.c_float(eps), p(wide), p(None), p(gated), I(M),
                                          I(F), I(K), I(F), I(1), stream()) == 0
        assert torch.equal(gated, ops.linear_swiglu_f32(rows, wide))


@pytest.mark.parametrize("M,N,K", [(1, 5, 7), (3, 1024, 4608), (8, 2048, 1024), (8, 2050, 300), (9, 1024, 640),
                                   (17, 100, 128), (64, 1024, 2304)])
def test_a_product_into_the_stream(ops, M, N, K):  # noqa: F811
    lib = ops.library("gemm")
    wide = rand((M, K + 4), F32, 5).to(DEV)
    x, w, bias = wide[:, :K], rand((N, K), F32, 6).to(DEV), rand((N,), F32, 7).to(DEV)
    resid = rand((M, N), F32, 8).to(DEV)
    want = resid + ops.linear(x, w, bias)
    assert lib.kappai_gemm_f32_add(p(x), p(w), p(bias), p(resid), I(M), I(N), I(K), I(K + 4), I(N), stream()) == 0
    assert torch.equal(resid, want)
    assert lib.kappai_gemm_f32_add(p(x), p(w), p(bias), p(resid), I(65), I(N), I(K), I(K + 4), I(N), stream()) != 0


# (a sum of squares that is rounded in another order shows in one row of a hundred)
@pytest.mark.parametrize("M,K", [(8, 512), (8, 1024), (5, 1536), (4, 2048)])
def test_many_rows_have_the_norms_bits(ops, M, K):  # noqa: F811
    lib = ops.library("gemm")
    w, norm_w = rand((64, K), F32, 9).to(DEV), rand((K,), F32, 10).to(DEV)
    xs = rand((200, M, K), F32, 11).to(DEV)
    for x in xs:
        out = torch.empty((M, 64), device=DEV)
        assert lib.kappai_gemm_f32_normed(p(x), p(norm_w), ctypes.c_float(1e-6), p(w), p(None), p(out), I(M), I(64),
                                          I(K), I(64), I(0), stream()) == 0
        assert torch.equal(out, ops.linear(ops.add_rmsnorm(x.clone(), None, norm_w, 1e-6, F32), w))
