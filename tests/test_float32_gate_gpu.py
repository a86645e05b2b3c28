"""The float32 product that applies the gate itself: the bits of the product and the gate behind it."""
import pytest
import torch

from test_kernels_gpu import DEV, F32, close, ops, rand  # noqa: F401

pytestmark = pytest.mark.gpu


# edges of the 16-, 32- and 64-row kernels and of blocks of 128, results that are no multiple of 8 or of
# 64, K that is no multiple of 4 or of a chunk, 8 and 32 runs
@pytest.mark.parametrize("M,F,K", [(1, 1032, 128), (8, 1025, 2049), (3, 4608, 1024), (9, 8, 100), (16, 333, 2176),
                                   (17, 5, 7), (32, 64, 4), (33, 100, 516), (64, 1030, 2200),
                                   (65, 16380, 130), (128, 16384, 128), (380, 4611, 72), (825, 4608, 256)])
@pytest.mark.parametrize("bias", [False, True])
def test_gate_inside(ops, M, F, K, bias):  # noqa: F811
    x, w = rand((M, K), F32, 41).to(DEV), rand((2 * F, K), F32, 42, 0.3).to(DEV)
    b = rand((2 * F,), F32, 43).to(DEV) if bias else None
    assert ops.linear_swiglu_f32_takes(x, w)
    got = ops.linear_swiglu_f32(x, w, b)
    assert torch.equal(got, ops.swiglu(ops.linear(x, w, b)))
    wide = torch.zeros((M, K + 3), device=DEV)              # rows further apart, off 16 bytes
    wide[:, 1:K + 1] = x
    assert torch.equal(ops.linear_swiglu_f32(wide[:, 1:K + 1], w, b), got)
    gu = x.double() @ w.double().T + (0 if b is None else b.double())
    close(got, gu[:, F:] * gu[:, :F] / (1 + torch.exp(-gu[:, :F])), 6e-6, "against 64 bits")


def test_no_finite_gates(ops):  # noqa: F811
    x = torch.tensor([[float("inf"), 1, 1, 1], [float("nan"), 1, 1, 1], [-200.0, 0, 0, 0]], device=DEV).repeat(4, 1)
    w = torch.ones((16, 4), device=DEV)
    got, want = ops.linear_swiglu_f32(x, w), ops.swiglu(ops.linear(x, w))
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))


def test_what_it_does_not_take(ops):  # noqa: F811
    x = torch.zeros((8, 64), device=DEV)
    for rows, w in ((x, torch.zeros((2048, 64), device=DEV)), (x[:, :3], torch.zeros((4096, 3), device=DEV)),
                    (torch.zeros((65, 64), device=DEV), torch.zeros((64, 64), device=DEV))):
        assert not ops.linear_swiglu_f32_takes(rows, w)
        with pytest.raises(ValueError):
            ops.linear_swiglu_f32(rows, w)
