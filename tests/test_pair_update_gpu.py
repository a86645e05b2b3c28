"""Two sublayers' results summed by one kernel: sides of either type and as float planes against the sum of the planes,
the widening and the sum one behind the other (bit for bit), into the stream with the next norm's rows, and a norm on
two terms of different types."""
import pytest
import torch

from test_kernels_gpu import BF16, DEV, F32, close, ops, rand  # noqa: F401

pytestmark = pytest.mark.gpu
SIDES = {"bf16": (BF16, 1), "f32": (F32, 1), "planes": (F32, 3)}


def side(kind, T, D, seed):
    dtype, parts = SIDES[kind]
    y = rand((T, D) if parts == 1 else (parts, T, D), dtype, seed).to(DEV)
    return y, y.float() if parts == 1 else y[0] + y[1] + y[2]


@pytest.mark.parametrize("T,D", [(1, 8), (3, 1024), (16, 260), (17, 1024), (40, 2100)])
@pytest.mark.parametrize("a", list(SIDES))
@pytest.mark.parametrize("b", list(SIDES))
@pytest.mark.parametrize("normed", [False, True])
def test_two_sides(ops, T, D, a, b, normed):  # noqa: F811
    (ya, fa), (yb, fb) = side(a, T, D, 1), side(b, T, D, 2)
    wa, wb = (rand((D,), F32, 3).to(DEV), rand((D,), F32, 4).to(DEV)) if normed else (None, None)
    want = ops.pair_norm_sum(fa, fb, 0.5, 0.75, wa, wb, 1e-5)
    assert torch.equal(ops.pair_norm_sum(ya, yb, 0.5, 0.75, wa, wb, 1e-5), want)
    resid, norm_w = rand((T, D), F32, 5).to(DEV), rand((D,), F32, 6).to(DEV)
    for nw in (None, norm_w):
        stream = resid.clone()
        got = ops.pair_norm_sum(ya, yb, 0.5, 0.75, wa, wb, 1e-5, add_into=ops.AddInto(stream, nw, 1e-5))
        if T > 16:
            assert torch.equal(got, want) and torch.equal(stream, resid)
            continue
        assert torch.equal(stream, resid + want) and got.resid is stream
        if nw is None:
            assert type(got) is ops.Added
        else:
            assert torch.equal(got.data, (stream * nw).bfloat16())
            # (D squares, each added once: no more roundings than that)
            close(got.ss[0, :T], stream.double().pow(2).sum(-1), (D + 1) * 2.0 ** -24, "sum of squares")


@pytest.mark.parametrize("T,D", [(2, 1024), (5, 1028), (3, 2056)])
@pytest.mark.parametrize("a", list(SIDES))
@pytest.mark.parametrize("b", ["bf16", "f32"])
def test_a_norm_on_two_terms(ops, T, D, a, b):  # noqa: F811
    (ya, fa), (yb, fb) = side(a, T, D, 7), side(b, T, D, 8)
    w, resid = rand((D,), F32, 9).to(DEV), rand((T, D), F32, 10).to(DEV)
    one, two = resid.clone(), resid.clone()
    rows = ops.output_norm_add(one, ya, w, 1e-5, rows_dtype=BF16, scale_a=0.5, b=yb, scale_b=0.25)
    want = ops.output_norm_add(two, fa, w, 1e-5, rows_dtype=BF16, scale_a=0.5, b=fb, scale_b=0.25)
    assert torch.equal(rows, want) and torch.equal(one, two)


@pytest.mark.parametrize("D", [1, 255, 1024, 1025, 2048])
@pytest.mark.parametrize("a,b", [(F32, BF16), (BF16, F32), (F32, F32)])
@pytest.mark.parametrize("normed", [False, True])
def test_two_sides_as_the_kernel_for_any_row(ops, D, a, b, normed):  # noqa: F811
    """Up to four planes with everything asked for at once, against the same planes and zeros as a fifth."""
    T, planes = 3, 4
    x = [rand((planes, T, D) if t == F32 else (T, D), t, 12 + i).to(DEV) for i, t in enumerate((a, b))]
    more = [torch.cat([y, torch.zeros_like(y[:1])]) if y.dim() == 3 else y for y in x]
    ws = [rand((D,), F32, 14 + i).to(DEV) if normed else None for i in range(2)]
    got, want = (ops.pair_norm_sum(*s, 0.5, 0.75, *ws, 1e-5) for s in (x, more))
    assert torch.equal(got, want)
    norm_w, resid = rand((D,), F32, 16).to(DEV), rand((T, D), F32, 17).to(DEV)
    out = []
    for s in (x, more):
        stream = resid.clone()
        y = ops.pair_norm_sum(*s, 0.5, 0.75, *ws, 1e-5, add_into=ops.AddInto(stream, norm_w, 1e-5))
        out.append((stream, y.data, y.ss[0, :T]))
    assert all(torch.equal(p, q) for p, q in zip(*out))


@pytest.mark.parametrize("a,b", [("planes", "bf16"), ("bf16", "planes"), ("f32", "bf16"), ("bf16", "bf16")])
def test_a_norm_from_outside_gets_terms_of_one_type(ops, a, b):  # noqa: F811
    """The two sides of a mixer behind which a norm stands that says nothing of planes or types: [T, D] in one type;
    the framework's own norm gets them as they were made, with the same stream."""
    from kappai_amd.parts import Hidden, Mixer, RMSNorm
    from kappai_amd.parts.block import OutputNormBlock
    from kappai_amd.parts.parallel import ParallelMixer
    T, D, seen = 3, 256, []
    (ya, fa), (yb, fb) = side(a, T, D, 21), side(b, T, D, 22)

    class Side(Mixer):
        def __init__(self, y):
            self.y = y

        def forward(self, x, batch, cache, shared_cache=False):
            return self.y.clone()

    class Outside(RMSNorm):
        def norm_output(self, resid, y, rows_dtype=None, add=True):
            seen.append((y.a, y.b))
            return super().norm_output(resid, y, rows_dtype, add)

    streams = []
    for cls in (RMSNorm, Outside):
        norm = cls("n", D, 1e-5, BF16)
        norm.weight = rand((D,), F32, 23).to(DEV)
        resid = rand((T, D), F32, 24).to(DEV)
        block = OutputNormBlock(ParallelMixer(Side(ya), Side(yb), 0.5, 0.25), norm)
        out = block.forward(Hidden(resid, None, resid.bfloat16()), None, None)
        streams.append((out.resid, out.rows))
    assert all(torch.equal(x, y) for x, y in zip(*streams))
    (got_a, got_b), = seen
    assert got_a.dtype == got_b.dtype and torch.equal(got_a.float(), fa) and torch.equal(got_b.float(), fb)
