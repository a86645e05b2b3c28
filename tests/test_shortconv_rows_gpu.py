"""Outputs and state of the short convolution in one kernel, against the form that takes the projection as float
sums and writes the state in a kernel of its own (one sum of the same values: the same bits), for segments
that begin at every place of a wave's run of four rows, single rows, and states that hold NaN where they do
not count."""
import pytest
import torch

from kappai_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV, F32, BF16 = "cuda:0", torch.float32, torch.bfloat16


@pytest.mark.parametrize("L", [2, 3, 4])
@pytest.mark.parametrize("D", [8, 504, 520, 1032])
@pytest.mark.parametrize("lens", [[1, 1, 1, 2], [3, 1, 1, 5, 4, 8, 2, 1, 6, 130, 1], [7], [2, 1027]])
def test_same_bits_as_outputs_and_state_apart(L, D, lens):
    g = torch.Generator().manual_seed(D + L + len(lens))
    S, T = len(lens), sum(lens)
    proj = torch.randn(T, 3 * D, generator=g).to(BF16).to(DEV)
    taps, bias = torch.randn(D, L, generator=g).to(DEV), torch.randn(D, generator=g).to(DEV)
    slots = torch.randperm(S + 2, generator=g)[:S]
    pos0 = torch.tensor([0 if i % 3 == 1 else 5 for i in range(S)])
    state = torch.randn(S + 2, D, L - 1, generator=g)
    state[slots[pos0 == 0]] = float("nan")
    meta = [t.int().to(DEV) for t in (torch.repeat_interleave(torch.arange(S), torch.tensor(lens)),
                                      torch.tensor([0] + lens).cumsum(0), pos0, slots)]
    for b in (bias, None):
        got_state, want_state = state.to(DEV), state.to(DEV)
        got = ops.shortconv(proj, taps, b, got_state, *meta)
        want = ops.shortconv(proj.float().unsqueeze(0).contiguous(), taps, b, want_state, *meta)
        assert torch.isfinite(got.float()).all()
        assert torch.equal(got, want)
        assert torch.equal(got_state.nan_to_num(7.0), want_state.nan_to_num(7.0))
        assert torch.isfinite(got_state[slots.to(DEV)]).all()
