"""The products of 1 to 24 rows over a matrix in fragment order, whose loads carry no conditions: K that
leaves waves with few pieces or none, column groups behind the last, rows behind M, the sums of squares of
narrow and wide norms, and memory full of NaN on every side of what they may read.  Results against float64
within the bound of a float sum of K products, gamma_K = K 2^-24 of the sum of magnitudes."""
import ctypes

import pytest
import torch

from kappai_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16 = torch.bfloat16
NAN = float("nan")


def _gen(*key):
    return torch.Generator(device=DEV).manual_seed(sum((i + 1) * 7919 ** i * int(k) for i, k in enumerate(key)) % (1 << 31))


def _rows(M, K, g):
    """[M, K] rows with NaN before, behind and between them."""
    big = torch.full((M + 2, K + 24), NAN, device=DEV, dtype=BF16)
    big[1:M + 1, 8:K + 8] = torch.randn(M, K, generator=g, device=DEV).to(BF16)
    return big[1:M + 1, 8:K + 8]


def _matrix(N, K, g):
    """A matrix in fragment order between matrices of NaN, and its rows."""
    w = torch.randn(N, K, generator=g, device=DEV).to(BF16)
    big = torch.full((N + 32, K), NAN, device=DEV, dtype=BF16)
    big[16:16 + N] = ops.fragment_order(w)
    return ops.InFragments(big[16:16 + N]), w


def _sums(x, w):
    """In float64 (on the CPU, where a product of a view is any product): the sums and their bound."""
    a, b = x.double().cpu(), w.double().cpu()
    return (a @ b.T).to(DEV), (a.abs() @ b.abs().T).to(DEV) * x.shape[1] * 2.0 ** -24


@pytest.mark.parametrize("M", [1, 4, 5, 16, 17, 24])
@pytest.mark.parametrize("K,N", [(32, 16), (64, 80), (96, 48), (288, 1040), (1056, 144), (2304, 64), (4608, 32)])
def test_plain(M, K, N):
    g = _gen(M, K, N)
    x = _rows(M, K, g)
    W, w = _matrix(N, K, g)
    want, bound = _sums(x, w)
    got = ops.linear(x, W, out_dtype=torch.float32)
    assert ((got.double() - want).abs() <= bound).all().item()
    parts = ops.linear(x, W, partial_sums=True, split_k=3 if K >= 288 else 1)
    if parts.dim() == 3:
        assert ((parts.double().sum(0) - want).abs() <= bound).all().item()


@pytest.mark.parametrize("M", [1, 3, 8, 16])
@pytest.mark.parametrize("K,N", [(32, 32), (64, 64), (96, 96), (1088, 96), (2304, 160), (4608, 64), (4640, 64)])
def test_into_the_stream(M, K, N):
    """(K = 4640: halves that are no whole pieces)"""
    g = _gen(M, K, N, 1)
    x = _rows(M, K, g)
    W, w = _matrix(N, K, g)
    want, bound = _sums(x, w)
    resid = torch.randn(M, N, generator=g, device=DEV)
    before = resid.double()
    norm = torch.rand(N, generator=g, device=DEV) + 0.5
    got = ops.linear(x, W, add_into=ops.AddInto(resid, norm, 1e-5))
    assert isinstance(got, ops.ScaledRows)
    assert ((resid.double() - before - want).abs() <= bound + resid.double().abs() * 2.0 ** -24).all().item()
    squares = got.ss[:, :M].double().sum(0)
    exact = (resid.double() ** 2).sum(1)
    assert ((squares - exact).abs() <= exact * N * 2.0 ** -24).all().item()


@pytest.mark.parametrize("M", [1, 5, 12, 16])
@pytest.mark.parametrize("D", [64, 1024, 4160])
def test_rows_still_to_be_scaled(M, D):
    """The product behind a folded norm: D / 8 parts of the sums of squares, one load of a wave or several."""
    g = _gen(M, D, 2)
    W0, _ = _matrix(D, 64, g)
    resid = torch.randn(M, D, generator=g, device=DEV)
    norm = torch.rand(D, generator=g, device=DEV) + 0.5
    scaled = ops.linear(_rows(M, 64, g), W0, add_into=ops.AddInto(resid, norm, 1e-5))
    W, w = _matrix(96, D, g)
    got = ops.linear(scaled, W, out_dtype=torch.float32)
    x = (resid * norm).to(BF16)                      # what the product before handed on
    want, bound = _sums(x, w)
    rms = (resid.double() ** 2).mean(1, keepdim=True).add(1e-5).sqrt()
    # the sum, the sum of squares (half its error), and the square root, division and product
    assert ((got.double() - want / rms).abs() <= (bound + want.abs() * (D / 2 + 4) * 2.0 ** -24) / rms).all().item()


@pytest.mark.parametrize("M", [1, 7, 16, 20, 48])
@pytest.mark.parametrize("D,L", [(32, 2), (64, 3), (1024, 3), (1536, 4), (96, 7)])
def test_conv_step(M, D, L):
    """The conv layer's step in one kernel against the same from float64 sums, the gates rounded as it
    rounds them.  A gate may differ by its sum's error and, beside a rounding boundary, by one unit of
    bfloat16 (2^-7 of it); what stands before the new value was stored in float and is the same."""
    g = _gen(M, D, L)
    x = _rows(M, D, g)
    W, w = _matrix(3 * D, D, g)
    taps = torch.randn(D, L, generator=g, device=DEV)
    bias = torch.randn(D, generator=g, device=DEV)
    slots = torch.randperm(M + 3, generator=g, device=DEV)[:M].to(torch.int32)
    pos = torch.arange(M, device=DEV, dtype=torch.int32)
    state = torch.randn(M + 3, D, L - 1, generator=g, device=DEV)
    before = state.clone()
    got = ops.linear_shortconv_step(x, W, None, taps, bias, state, pos, slots)
    sums, bounds = _sums(x, w)
    b, c, u = (t.to(BF16).double() for t in sums.float().split(D, 1))
    unit = 2.0 ** -7
    db, dc, du = (t + unit * v.abs() for t, v in zip(bounds.split(D, 1), (b, c, u)))
    old = before[slots.long()].double()
    old[pos == 0] = 0
    window = torch.cat([old, (b * u)[:, :, None]], 2)
    d_new = b.abs() * du + u.abs() * db + db * du + 2.0 ** -24 * (b * u).abs()
    terms = window * taps.double()
    s = terms.sum(2) + bias.double()
    ds = d_new * taps[:, -1].double().abs() + (L + 1) * 2.0 ** -23 * (terms.abs().sum(2) + bias.double().abs())
    slack = c.abs() * ds + dc * (s.abs() + ds)
    assert ((got.double() - c * s).abs() <= slack + unit * ((c * s).abs() + slack)).all().item()
    after = state[slots.long()].double()
    assert torch.equal(after[:, :, :-1], window[:, :, 1:-1])
    assert ((after[:, :, -1] - window[:, :, -1]).abs() <= d_new).all().item()
    rest = torch.ones(M + 3, dtype=torch.bool, device=DEV)
    rest[slots.long()] = False
    assert torch.equal(state[rest], before[rest])


@pytest.mark.parametrize("in_fragments", [True, False])
def test_into_a_stream_of_more_than_two_gibibytes(in_fragments):
    """Sixteen rows of a stream so far apart that the last lies behind 2 GiB: each is added to where it stands."""
    from kappai_amd.kernels.lib import library
    M, N, K, ldr = 16, 64, 64, 36_000_000
    assert (M - 1) * ldr * 4 > 1 << 31
    g = _gen(M, N, K, 9)
    x = _rows(M, K, g)
    W, w = _matrix(N, K, g)
    want, bound = _sums(x, w)
    flat = torch.empty((M - 1) * ldr + N, device=DEV)
    resid = flat.as_strided((M, N), (ldr, 1))
    resid.copy_(torch.randn(M, N, generator=g, device=DEV) * 10)
    before = resid.double()
    norm = torch.rand(N, generator=g, device=DEV) + 0.5
    rows = torch.empty(M, N, device=DEV, dtype=BF16)
    ss = torch.empty(N // 8, 16, device=DEV)
    vp, ci, cf = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    rc = library("gemm").kappai_gemm_bf16(
        vp(x.data_ptr()), vp(0 if in_fragments else w.data_ptr()), vp(W.data_ptr() if in_fragments else 0), vp(0),
        vp(0), ci(M), ci(N), ci(K), ci(x.stride(0)), ci(N), ci(1), ci(0), ci(1), ci(0), vp(0), ci(0), cf(0.0),
        vp(resid.data_ptr()), ci(ldr), vp(norm.data_ptr()), vp(rows.data_ptr()), ci(0), vp(ss.data_ptr()),
        vp(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    assert ((resid.double() - before - want).abs() <= bound + resid.double().abs() * 2.0 ** -24).all().item()
    assert torch.equal(rows, (resid * norm).to(BF16))


def test_conv_step_of_very_many_channels():
    """So many channels that their taps take more than 4 GiB: the last sixteen of them, on a matrix that is zero
    for all others."""
    D, K, L = 220_000_000, 8, 5
    assert D * L * 4 > 1 << 32
    g = _gen(D, 5)
    w = torch.zeros(3, D, K, device=DEV, dtype=BF16)
    taps, conv_bias, bias = (torch.empty(*n, device=DEV) for n in ((D, L), (D,), (3, D)))
    state = torch.empty(1, D, L - 1, device=DEV)
    for t in (w[:, -16:], taps[-16:], conv_bias[-16:], bias[:, -16:], state[:, -16:]):
        t.copy_(torch.randn(t.shape, generator=g, device=DEV))
    x = torch.randn(1, K, generator=g, device=DEV).to(BF16)
    old = state[0, -16:].double()
    got = ops.linear_shortconv_step(x, w.view(3 * D, K), bias.view(-1), taps, conv_bias, state,
                                    torch.ones(1, dtype=torch.int32, device=DEV),
                                    torch.zeros(1, dtype=torch.int32, device=DEV))
    b, c, u = ((w[i, -16:].double() * x.double()).sum(1) + bias[i, -16:].double() for i in range(3))
    b, c, u = (v.float().to(BF16).double() for v in (b, c, u))
    window = torch.cat([old, (b * u)[:, None]], 1)
    terms = window * taps[-16:].double()
    want = c * (terms.sum(1) + conv_bias[-16:].double())
    # (a gate may round the other way: 2^-7 of it; the result's own rounding beside that)
    slack = c.abs() * (4 * 2.0 ** -7 * (terms.abs().sum(1) + conv_bias[-16:].double().abs()))
    assert ((got[0, -16:].double() - want).abs() <= slack).all().item()


def test_rows_of_x_more_than_two_gibibytes_apart():
    """Rows of x so far apart that offsets within them take more than 31 bits: the kernels over fragment order that
    carry conditions give the bits of those without, whose rows lie side by side."""
    K = 64
    g = _gen(K, 11)
    for M, apart in ((16, 67_200_000), (24, 44_800_000)):
        assert M * apart * 2 > 1 << 31
        far = torch.empty((M - 1) * apart + K, device=DEV, dtype=BF16).as_strided((M, K), (apart, 1))
        x = torch.randn(M, K, generator=g, device=DEV).to(BF16)
        far.copy_(x)
        W, _ = _matrix(96, K, g)
        taps, state = torch.randn(32, 3, generator=g, device=DEV), torch.randn(M, 32, 2, generator=g, device=DEV)
        rows = torch.arange(M, device=DEV, dtype=torch.int32)

        def results(x):
            st = state.clone()
            out = [ops.linear(x, W, out_dtype=torch.float32), ops.linear_swiglu(x, W),
                   ops.linear_shortconv_step(x, W, None, taps, None, st, rows, rows), st]
            if M <= 16:
                resid, norm = torch.ones(M, 96, device=DEV), torch.linspace(0.5, 1.5, 96, device=DEV)
                scaled = ops.linear(x, W, add_into=ops.AddInto(resid, norm, 1e-5))
                out += [resid, scaled.data[:M] if not scaled.fragment else scaled.data, scaled.ss[:, :M]]
            return out

        for got, want in zip(results(far), results(x)):
            assert torch.equal(got, want)
        del far


@pytest.mark.parametrize("K,N", [(64, 32), (1024, 1024), (2304, 48), (4096, 16), (4608, 1024), (10752, 64)])
def test_into_the_stream_halves_of_k_share_a_fragment_up_to_8_rows(K, N):
    """Nine rows take two fragments of x for one of W, eight one: the same bits."""
    g = _gen(K, N, 18)
    x = _rows(9, K, g)
    W, _ = _matrix(N, K, g)
    norm, resid = torch.rand(N, generator=g, device=DEV) + 0.5, torch.randn(9, N, generator=g, device=DEV)
    out = []
    for rows in (9, 8, 3, 1):
        stream = resid[:rows].clone()
        got = ops.linear(x[:rows], W, add_into=ops.AddInto(stream, norm, 1e-5))
        out.append((stream, got.ss[:, :rows]))
    for stream, ss in out[1:]:
        n = stream.shape[0]
        assert torch.equal(stream, out[0][0][:n]) and torch.equal(ss, out[0][1][:, :n])


@pytest.mark.parametrize("K,N", [(1024, 64), (4096, 16), (4608, 1024), (10752, 64)])
def test_into_the_stream_from_rows_in_fragment_order(K, N):
    """Rows in fragment order ([K / 32][4][16 row slots][8]) give the bits of plain rows, up to 8 rows and beyond, and
    what lies in the slots of rows that are not there reaches nothing."""
    g = _gen(K, N, 19)
    W, _ = _matrix(N, K, g)
    norm, resid = torch.rand(N, generator=g, device=DEV) + 0.5, torch.randn(16, N, generator=g, device=DEV)
    every = _rows(16, K, g)
    for M in (1, 3, 8, 9, 16):
        x = every[:M].contiguous()
        slots = torch.full((16, K), float("nan"), dtype=torch.bfloat16, device=DEV)
        slots[:M] = x
        data = slots.view(16, K // 32, 4, 8).permute(1, 2, 0, 3).contiguous().view(16, K)
        one, two = resid[:M].clone(), resid[:M].clone()
        want = ops.linear(x, W, add_into=ops.AddInto(one, norm, 1e-5))
        got = ops.linear(ops.FragmentRows(data, M, two), W, add_into=ops.AddInto(two, norm, 1e-5))
        assert torch.equal(ops.FragmentRows(data, M, two).materialize(), x)
        assert torch.equal(one, two) and torch.equal(want.ss[:, :M], got.ss[:, :M]) and torch.isfinite(one).all()
        kept = [(ops.FragmentRows(r.data, M, one).materialize() if r.fragment else r.data) for r in (want, got)]
        assert torch.equal(*kept)
