"""The dense gated feed-forward over every kind of rows and weights it takes, with and without biases,
against float64: on the CPU with the kernels' stand-ins, on the GPU with the kernels."""
import pytest
import torch

import emulated_ops

F32, BF16 = torch.float32, torch.bfloat16
GPU = pytest.mark.gpu


# widths of which the gate can and cannot be part of the product
@pytest.mark.parametrize("W,Fh", [(40, 48), (64, 64), (36, 48), (40, 24)])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("weights,rows", [(F32, F32), (BF16, BF16), (BF16, F32)])
@pytest.mark.parametrize("view", [False, True])
@pytest.mark.parametrize("where", ["cpu", pytest.param("cuda:0", marks=GPU)])
def test_feed_forward_takes_any_rows(monkeypatch, where, W, Fh, bias, weights, rows, view):
    from kappai_amd.parts import SwiGLU
    if where == "cpu":
        emulated_ops.install(monkeypatch)
    g = torch.Generator().manual_seed(W + Fh)
    ffn = SwiGLU("f.", W, Fh, weights, bias=bias)
    w = {s.name: (torch.randn(s.shape, generator=g) * 0.2).to(weights)
         for s in ffn.tensor_specs()}
    ffn.bind({n: t.to(where) for n, t in w.items()})
    # (a matrix kept in fragment order takes bfloat16 rows that start on 16 bytes only)
    refused = view and rows == BF16 and not torch.is_tensor(ffn.gate_up.weight)
    for T in (1, 5, 20, 70):
        x = torch.randn(T, W, generator=g).to(rows)
        on = x.to(where)
        if view:                          # rows that do not start on 16 bytes
            wide = torch.zeros((T, W + 3), dtype=rows, device=where)
            wide[:, 3:] = on
            on = wide[:, 3:]
        if refused:
            with pytest.raises(ValueError, match="16-byte aligned"):
                ffn.forward(on, None)
            continue
        y = ffn.forward(on, None)
        y = (y if y.dim() == 2 else y.sum(0)).cpu().double()
        d = {n: t.double() for n, t in w.items()}

        def product(v, n):
            out = v @ d[f"f.{n}.weight"].T
            return out + d[f"f.{n}.bias"] if bias else out
        act = torch.nn.functional.silu(product(x.double(), "w1")) * product(x.double(), "w3")
        want = product(act, "w2")
        # bfloat16: the rows where they are not, both sums, the gated product and the result are
        # rounded, each by at most 2^-9 of its value
        tol = 1e-5 if weights == F32 else 2e-2
        assert float((y - want).abs().max() / want.abs().max()) < tol, T
