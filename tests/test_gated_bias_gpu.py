"""The gated products whose epilogues add biases before the gate, in every kernel a number of rows can
take, against float64; and a biased product cut into K ranges."""
import pytest
import torch

from test_kernels_gpu import BF16, BF16_ULP, DEV, F32, close, ops, rand  # noqa: F401

pytestmark = pytest.mark.gpu


# F of whole 32-column tiles, of an odd number of 16s, and enough for 256 x 256 blocks; K of whole
# runs and with a rest
@pytest.mark.parametrize("F,K", [(64, 256), (48, 136), (9216, 128)])
@pytest.mark.parametrize("M", [1, 5, 8, 16, 17, 40, 64, 65, 128, 129, 300, 520])
def test_linear_swiglu_with_biases(ops, M, F, K):  # noqa: F811
    x = rand((M, K), BF16, 81)
    wg, wu = rand((F, K), BF16, 82, K ** -0.5), rand((F, K), BF16, 83, K ** -0.5)
    bg, bu = rand((F,), F32, 84), rand((F,), F32, 85)
    g = x.double() @ wg.double().T + bg.double()
    u = x.double() @ wu.double().T + bu.double()
    want = torch.nn.functional.silu(g) * u
    w = ops.interleave_gate_up(wg, wu).to(DEV)
    b = ops.interleave_gate_up(bg[:, None], bu[:, None]).reshape(-1).to(DEV)
    kept = ops.InFragments.of(w)
    # three roundings to bfloat16 behind each other, each by at most half of BF16_ULP of the value it
    # rounds: of g (|g silu'(g)| is at most 1.28 |silu(g)| above zero and 0.27 below), of u and of the
    # result: (1.28 + 1 + 1) / 2 = 1.64 of BF16_ULP of the largest result where that is above zero's
    # 0.27 |u|.  3 leaves room for products of two of them, the float32 sums and the exponential
    for matrix in (w, kept) if kept is not None else (w,):
        close(ops.linear_swiglu(x.to(DEV), matrix, bias=b).float(), want, 3 * BF16_ULP, (M, F, K))


@pytest.mark.parametrize("M,F,K", [(1, 9216, 1024), (3, 48, 136), (8, 320, 1024), (16, 64, 2048)])
def test_linear_swiglu_with_biases_on_scaled_rows(ops, M, F, K):  # noqa: F811
    """Rows whose norm the product still has to scale by, in fragment order from eight rows on, as a
    result in fragment order too."""
    x = rand((M, 96), BF16, 87)
    w1, wn = rand((K, 96), BF16, 88, 0.1), 1 + rand((K,), F32, 89, 0.1)
    wg, wu = rand((F, K), BF16, 90, K ** -0.5), rand((F, K), BF16, 91, K ** -0.5)
    bg, bu = rand((F,), F32, 92), rand((F,), F32, 93)
    w = ops.interleave_gate_up(wg, wu).to(DEV)
    b = ops.interleave_gate_up(bg[:, None], bu[:, None]).reshape(-1).to(DEV)
    resid = rand((M, K), F32, 94, 2.0).to(DEV)
    rows = ops.linear(x.to(DEV), w1.to(DEV), add_into=ops.AddInto(resid, wn.to(DEV), 1e-5))
    assert isinstance(rows, ops.ScaledRows)
    xn = resid.cpu().double()
    xn = xn / torch.sqrt((xn * xn).mean(dim=1, keepdim=True) + 1e-5) * wn.double()
    g, u = xn @ wg.double().T + bg.double(), xn @ wu.double().T + bu.double()
    want = torch.nn.functional.silu(g) * u
    # as above, and the rows' own rounding to bfloat16 (half of BF16_ULP of each, through sums of K)
    got = ops.linear_swiglu(rows, w, bias=b)
    close(got.float(), want, 4 * BF16_ULP, "scaled rows")
    frag = ops.linear_swiglu(rows, w, bias=b, out_fragment=True)
    if M >= 8:
        assert isinstance(frag, ops.FragmentRows)
        frag = frag.materialize()
    assert torch.equal(frag, got)


@pytest.mark.parametrize("M", [2, 12, 30, 100, 600])
def test_biased_products_in_k_ranges(ops, M):  # noqa: F811
    x, w, b = rand((M, 4608), BF16, 86), rand((1024, 4608), BF16, 87, 0.05), rand((1024,), F32, 88)
    parts = ops.linear(x.to(DEV), ops.InFragments.of(w.to(DEV)), b.to(DEV), partial_sums=True)
    assert parts.dim() == 3 and parts.dtype == F32
    close(parts.sum(0), x.double() @ w.double().T + b.double(), 2e-5, M)
