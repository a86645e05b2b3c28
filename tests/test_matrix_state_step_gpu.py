"""Steps of single rows of the recurrences with a matrix per head: the one kernel against the kernels it stands
for (what enters the recurrence, the walk, the norm with its gate), bit for bit, results and states."""
import pytest
import torch

from test_kernels_gpu import BF16, DEV, F32, ops, rand  # noqa: F401

pytestmark = pytest.mark.gpu

FORMS = {
    "gated": dict(sign=-1.0, scale=0.25, rate=True, bias=True, z=True),
    "fixed": dict(sign=1.0, scale=1.0, rate=True, bias=False, z=False, decay="fixed", silu_inputs=True),
    "delta": dict(sign=1.0, scale=0.25, rate=True, bias=True, z=True, beta=True, unit_qk=True),
    "bonus": dict(sign=1.0, scale=1.0, rate=False, bias=True, z=True, decay="double_exp", bonus=True),
}


# key sizes at both ends of 2 to 16 lanes a column and ones that are no power of two, value sizes that end inside a
# wave and take more than one group of columns, q and k shared by heads
@pytest.mark.parametrize("form,H,G,d,dv", [
    ("gated", 3, 3, 12, 5), ("gated", 8, 8, 64, 64), ("gated", 2, 2, 128, 127), ("gated", 1, 1, 68, 128),
    ("gated", 2, 2, 16, 508), ("fixed", 8, 8, 64, 64), ("fixed", 3, 3, 20, 33), ("delta", 16, 4, 64, 64),
    ("delta", 4, 2, 128, 128), ("delta", 3, 1, 16, 7), ("bonus", 16, 16, 64, 64), ("bonus", 5, 5, 100, 100)])
@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("rows", [1, 7])
def test_one_kernel_has_the_bits_of_three(ops, form, H, G, d, dv, dtype, rows):  # noqa: F811
    f = dict(FORMS[form])
    n, odd = 2 * G * d + 2 * H * dv, 0 if d % 8 == 0 else 3        # (rows that start on no 16 bytes, too)
    proj = rand((rows, n + odd), dtype, 1).to(DEV)
    q, k = proj[:, :G * d], proj[:, G * d:2 * G * d]
    v, g = proj[:, 2 * G * d:2 * G * d + H * dv], proj[:, 2 * G * d + H * dv:n]
    z = rand((rows, H * d), dtype, 2).to(DEV) if f.pop("z") else None
    rate = rand((H,), F32, 3).abs().clamp(0.05, 0.95).to(DEV) if f.pop("rate") else None
    bias = rand((H * d,), F32, 4).to(DEV) if f.pop("bias") else None
    if f.get("beta"):
        f["beta"] = rand((rows, H + 1), dtype, 5).to(DEV)[:, 1:] if H > 1 else rand((rows, 1), dtype, 5).to(DEV)
    if f.get("bonus"):
        f["bonus"] = rand((H, d), F32, 6).to(DEV)
    sign, scale = f.pop("sign"), f.pop("scale")
    state = rand((rows + 2, H, dv, d), F32, 7).to(DEV)
    i32 = dict(dtype=torch.int32, device=DEV)
    start, slot = torch.arange(rows + 1, **i32), torch.arange(rows, 0, -1, **i32)
    pos0 = (torch.arange(rows, **i32) % 3 != 1).to(torch.int32) * 9       # (some rows begin a request)
    kind = ops.GATE_SILU if "beta" in f or "bonus" in f else ops.GATE_SIGMOID
    assert ops.matrix_state_step_takes(q, state)
    for weight in (rand((dv,), F32, 8).to(DEV), rand((H, dv), F32, 9).to(DEV)):
        norm = ops.GatedNorm(weight, 1e-5, g, kind, H, dv)
        before, after = state.clone(), state.clone()
        args = (q, k, v, z, H, G, d, dv, rate, bias, sign, scale)
        o = ops.matrix_state_recurrence(*args, before, start, pos0, slot, **f)
        want = ops.head_norm_gate(o, weight, 1e-5, g, kind, H, dv, dtype)
        got = ops.matrix_state_step(*args, after, pos0, slot, norm=norm, **f)
        assert torch.equal(got, want) and torch.equal(after, before)
    plain = state.clone()
    assert torch.equal(ops.matrix_state_step(*args, plain, pos0, slot, **f), o)
    assert torch.equal(plain, before)


def test_what_the_kernel_does_not_take(ops):  # noqa: F811
    q = rand((2, 64), BF16, 1).to(DEV)
    for d, dv in ((8, 16), (30, 16), (132, 16), (16, 512), (128, 129)):
        assert not ops.matrix_state_step_takes(q, torch.zeros((3, 2, dv, d), device=DEV)), (d, dv)
    assert not ops.matrix_state_step_takes(q.cpu(), torch.zeros((3, 2, 16, 32)))
