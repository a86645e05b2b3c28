"""The norm kernels that have a form for each number of partial sums, against float64: the residual is the planes
added in order, so its bits are known; the norm's error is that of a sum of squares of at most 8 values a thread,
6 exchanges and 16 waves, one square root, one division and two products (34 roundings of 2^-24)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV, F32, BF16 = "cuda", torch.float32, torch.bfloat16
NORM = 34 * 2.0 ** -24


def rand(seed, *shape, scale=1.0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale


def bounded(got, want, slack, dtype, what):
    slack = slack + (2.0 ** -8 * want.abs() if dtype == BF16 else 0.0)
    over = (got.double().cpu() - want).abs() - slack
    assert bool((over <= 0).all()), (what, float(over.max()))


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("D", [8, 504, 512, 2048, 2056, 8192])
@pytest.mark.parametrize("parts", [0, 1, 2, 3, 4, 5, 8])
def test_residual_and_norm_of_partial_sums(parts, D, dtype):
    from kappai_amd.kernels import ops
    T = 5
    resid, w = rand(1, T, D, scale=2.0), 1 + rand(2, D, scale=0.2)
    planes = rand(3, parts, T, D) if parts else None
    dev = resid.to(DEV)
    out = ops.add_rmsnorm(dev, None if planes is None else planes.to(DEV), w.to(DEV), 1e-5, dtype)
    x = resid.clone()
    for p in range(parts):
        x += planes[p]
    assert torch.equal(dev.cpu(), x)
    want = x.double() / torch.sqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5) * w.double()
    bounded(out, want, NORM * want.abs(), dtype, "norm")
    if planes is not None:                  # rows picked, the stream left alone
        rows = torch.tensor([4, 0], dtype=torch.int32)
        dev = resid.to(DEV)
        some = ops.add_rmsnorm(dev, planes.to(DEV), w.to(DEV), 1e-5, dtype, rows=rows.to(DEV), write_resid=False)
        assert torch.equal(some, out[rows.long().to(DEV)]) and torch.equal(dev.cpu(), resid)


@pytest.mark.parametrize("add", [False, True])
@pytest.mark.parametrize("second", [False, True])
@pytest.mark.parametrize("D", [8, 504, 1024, 2048, 2056])
@pytest.mark.parametrize("parts", [0, 1, 2, 3, 4, 5, 9])
def test_norm_of_a_result_of_partial_sums(parts, D, second, add):
    """parts 0: one plane in bfloat16.  2,048 values are the last width of the kernel that keeps them in registers."""
    from kappai_amd.kernels import ops
    T, dtype = 3, F32 if parts else BF16
    a = rand(1, max(parts, 1), T, D).to(dtype)
    b = rand(2, T, D).to(dtype) if second else None
    w, resid = 1 + rand(3, D, scale=0.2), rand(4, T, D)
    dev = resid.to(DEV)
    rows = ops.output_norm_add(dev, (a if parts > 1 else a[0]).to(DEV), w.to(DEV), 1e-5, rows_dtype=BF16, scale_a=0.7,
                               b=None if b is None else b.to(DEV), scale_b=1.3, add=add)
    y = a[0].float().clone()
    for p in range(1, parts):
        y += a[p]
    y *= torch.tensor(0.7)
    if second:
        y = (torch.tensor(1.3).double() * b.double() + y.double()).float()
    n = y.double() / torch.sqrt((y.double() ** 2).mean(1, keepdim=True) + 1e-5) * w.double()
    want = n + resid.double() if add else n
    bounded(dev, want, NORM * n.abs() + 2.0 ** -24 * want.abs(), F32, "stream")
    assert torch.equal(rows.cpu(), dev.cpu().to(BF16))


@pytest.mark.parametrize("fragment", [0, 1])
def test_planes_more_than_sixteen_gigabytes_apart(fragment):
    """Two planes 2^32 + 64 values apart (16 rows picked of a projection of a million rows) give the bits of two
    planes side by side, in fragment order too."""
    import ctypes
    from kappai_amd.kernels.lib import library
    T, D, apart = 16, 2048, (1 << 32) + 64
    resid, w, planes = rand(1, T, D).to(DEV), (1 + rand(2, D, scale=0.2)).to(DEV), rand(3, 2, T, D).to(DEV)
    far = torch.empty(apart + T * D, device=DEV)
    far[:T * D], far[apart:] = planes[0].flatten(), planes[1].flatten()

    def norm(delta, distance):
        x, out = resid.clone(), torch.empty(T, D, device=DEV, dtype=BF16)
        vp, ci = ctypes.c_void_p, ctypes.c_int
        rc = library("elementwise").kappai_add_rmsnorm(
            vp(x.data_ptr()), vp(delta.data_ptr()), ci(1), ci(2), ctypes.c_long(distance), vp(w.data_ptr()),
            vp(out.data_ptr()), vp(0), ci(T), ci(D), ctypes.c_float(1e-5), ci(1), ci(1), ci(fragment),
            vp(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        return x, out

    for got, want in zip(norm(far, apart), norm(planes, T * D)):
        assert torch.equal(got, want)
