"""Kernels that ask for all they read before they compute, at the sizes where their rounds of loads end: the
per-head product over odd inputs, outputs and rows, and the gated unit's step over parts of 64 and 128
channels, against float64 within bounds of their float sums and one unit of the stored type."""
import pytest
import torch

from kappai_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16 = torch.bfloat16
EPS = 2.0 ** -24


def _gen(*key):
    return torch.Generator(device=DEV).manual_seed(sum((i + 1) * 7919 ** i * int(k) for i, k in enumerate(key)) % (1 << 31))


@pytest.mark.parametrize("T", [1, 16, 17, 70])
@pytest.mark.parametrize("n_out,n_in", [(1, 8), (40, 64), (224, 136), (65, 224), (64, 264), (130, 520)])
@pytest.mark.parametrize("gated", [False, True])
def test_headwise_linear(T, n_out, n_in, gated):
    g = _gen(T, n_out, n_in, gated)
    H = 3
    # heads side by side in rows of their own, NaN behind every head's input and behind W
    x = torch.full((T, H * (n_in + 8)), float("nan"), device=DEV, dtype=BF16)
    heads = x.view(T, H, n_in + 8)[:, :, :n_in]
    heads.copy_(torch.randn(T, H, n_in, generator=g, device=DEV))
    w = torch.full((H + 1, n_out, n_in), float("nan"), device=DEV, dtype=BF16)[:H]
    w.copy_(torch.randn(H, n_out, n_in, generator=g, device=DEV))
    gate = torch.randn(T, H * n_out, generator=g, device=DEV).to(BF16) if gated else None
    got = ops.headwise_linear(x, n_in + 8, w, out_dtype=torch.float32, gate=gate).view(T, H, n_out).double().cpu()
    a, b = heads.double().cpu(), w.double().cpu()
    want = torch.stack([a[:, h] @ b[h].T for h in range(H)], 1)
    size = torch.stack([a[:, h].abs() @ b[h].abs().T for h in range(H)], 1)
    if gated:
        s = torch.sigmoid(gate.double().cpu()).view(T, H, n_out)
        want, size = want * s, size * s
    # (the sigmoid: an exponential of 2 units, a sum and a division)
    assert ((got - want).abs() <= size * (n_in + 8) * EPS).all().item()


@pytest.mark.parametrize("T", [1024, 1025])
@pytest.mark.parametrize("n_out,n_in", [(64, 64), (63, 40), (65, 64)])
@pytest.mark.parametrize("out_dtype", [torch.float32, BF16])
def test_headwise_linear_gates_around_a_wave_a_simd(T, n_out, n_in, out_dtype):
    """16 heads: 1,024 waves and 1,040 where 64 columns hold the outputs, twice as many else.  Gates stand in
    rows with NaN behind them; the rows on either side of the rule are the same to the bit."""
    g = _gen(T, n_out, n_in)
    H = 16
    x = torch.randn(1025, H * n_in, generator=g, device=DEV).to(BF16)[:T]
    w = torch.randn(H, n_out, n_in, generator=g, device=DEV).to(BF16)
    rows = torch.full((1025, H * n_out + 5), float("nan"), device=DEV, dtype=BF16)
    gate = rows[:T, :H * n_out]
    gate.copy_(torch.randn(T, H * n_out, generator=g, device=DEV) * 3)
    got = ops.headwise_linear(x, n_in, w, out_dtype=out_dtype, gate=gate)
    few = torch.cat([ops.headwise_linear(x[i:i + 200], n_in, w, out_dtype=out_dtype, gate=gate[i:i + 200])
                     for i in range(0, T, 200)])
    assert torch.equal(got, few)
    s = torch.sigmoid(gate.double().cpu()).view(T, H, n_out)
    a, b = x.double().cpu().view(T, H, n_in), w.double().cpu()
    want = torch.stack([a[:, h] @ b[h].T for h in range(H)], 1) * s
    size = torch.stack([a[:, h].abs() @ b[h].abs().T for h in range(H)], 1) * s
    bound = size * (n_in + 8) * EPS
    if out_dtype == BF16:
        bound = bound + want.abs() * 2.0 ** -8
    assert ((got.view(T, H, n_out).double().cpu() - want).abs() <= bound).all().item()


@pytest.mark.parametrize("part", [64, 128, 96])
@pytest.mark.parametrize("n", [1, 2, 4, 5])
@pytest.mark.parametrize("T", [1, 3])
def test_gated_unit_step(part, n, T):
    """Beside float64 stands what the convolution's value is stored as; where float and float64 round it to
    neighbours, the next sums differ by a unit of bfloat16 of that value (2^-7)."""
    g = _gen(part, n, T)
    blocks = 3
    W = blocks * part
    r = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    proj = r(T, 2 * W + 8).to(BF16)
    taps, bias, gate_bias, state = r(W, n), r(W), r(2 * W), r(T + 2, W)
    conv = r(T + 2, n - 1, W)
    gate_w = (r(blocks, 2 * part, part) * 0.1).to(BF16)
    lam = torch.rand(W, generator=g, device=DEV) * 2 + 0.05
    pos = torch.tensor([2, 0, 9], device=DEV, dtype=torch.int32)[:T].contiguous()
    slot = torch.tensor([3, 1, 2], device=DEV, dtype=torch.int32)[:T].contiguous() % (T + 2)
    state0, conv0 = state.clone(), conv.clone()
    got = ops.gated_unit_step(proj[:, :2 * W], taps, bias, conv, gate_w, gate_bias, lam, 8.0, state, pos, slot)
    for t in range(T):
        s, p = int(slot[t]), int(pos[t])
        x, y = proj[t, :W].double(), proj[t, W:2 * W].double()
        hist = torch.cat([conv0[s].double(), x[None]])                   # oldest first
        for j in range(n - 1):
            if n - 1 - j > p:
                hist[j] = 0
        u = ((hist.T * taps.double()).sum(1) + bias.double()).to(torch.float32).to(BF16).double()
        sums = torch.einsum("bop,bp->bo", gate_w.double().cpu(), u.view(blocks, part).cpu()).to(DEV)
        sums = sums + gate_bias.double().view(blocks, 2 * part)
        rg, ig = sums[:, :part].reshape(W), sums[:, part:].reshape(W)
        la = -8.0 * torch.sigmoid(rg) * lam.double()
        want = torch.exp(la) * (state0[s].double() if p > 0 else 0) + \
            torch.sqrt(-torch.expm1(2 * la)) * torch.sigmoid(ig) * u
        # a unit of bfloat16 in one value of u moves a gate's sum by 2^-7 0.1 of it; many do not at once
        scale = want.abs() + u.abs() + state0[s].double().abs()
        assert ((state[s].double() - want).abs() <= 0.02 * scale + 1e-4).all().item()
        assert ((state[s].double() - want).norm() <= 2e-3 * want.norm()).item()
        gelu = 0.5 * y * (1 + torch.tanh(0.7978845608028654 * (y + 0.044715 * y ** 3)))
        assert ((got[t].double() - want * gelu).norm() <= 4e-3 * (want * gelu).norm()).item()
        if n > 1:
            kept = torch.cat([hist[1:-1], x[None]]).float() if n > 2 else x[None].float()
            assert torch.equal(conv[s], kept)
