"""The 32-bit kernels at the sizes where their tiles, runs and places end: products against float64,
and a row's bits whatever it is computed with; attention against the plain statement of it."""
import math

import pytest
import torch

import emulated_ops as ref
from test_kernels_gpu import DEV, F32, close, ops, paged_case, rand  # noqa: F401

pytestmark = pytest.mark.gpu


# K of one chunk, of the two numbers of runs and with chunks left over, and no whole chunks; N around
# the widths that blocks own
@pytest.mark.parametrize("N,K", [(5, 128), (40, 2048), (2047, 2176), (2064, 4608), (33, 2050),
                                 (130, 8192), (9216, 1024), (40, 1), (33, 3), (700, 4), (2064, 7),
                                 (40, 20), (2064, 36), (33, 65), (70, 129), (2064, 140),
                                 (40, 2181)])
def test_a_rows_product_has_the_same_bits_in_every_batch(ops, N, K):  # noqa: F811
    x, w, b = rand((300, K), F32, 61), rand((N, K), F32, 62), rand((N,), F32, 63)
    want = x.double() @ w.double().T + b.double()
    x, w, b = x.to(DEV), w.to(DEV), b.to(DEV)
    whole = ops.linear(x, w, b)
    close(whole, want, 3e-6, "all rows")
    for M in (1, 8, 9, 16, 17, 32, 33, 64, 65, 129):
        assert torch.equal(ops.linear(x[:M].contiguous(), w, b), whole[:M]), M
    # rows that are not aligned to 16 bytes take element-wise loads, in the same order
    off = torch.empty((8, K + 1), dtype=F32, device=DEV)
    off[:, 1:] = x[:8]
    assert torch.equal(ops.linear(off[:, 1:], w, b), whole[:8])


# enough rows and columns for blocks of 128 x 128 (from 769 blocks of 64 x 64 on), ragged and whole, in
# each form of the loads
@pytest.mark.parametrize("M,N,K", [(330, 9217, 256), (330, 9217, 130), (321, 9300, 132),
                                   (512, 8192, 128), (330, 9217, 2177)])
def test_large_blocks_give_the_same_bits(ops, M, N, K):  # noqa: F811
    rounds = lambda b: (-(-M // b) * -(-N // b) + 255) // 256  # noqa: E731
    assert rounds(128) * 32 <= rounds(64) * 9, "the rule takes smaller blocks here"
    x, w, b = rand((M, K), F32, 65), rand((N, K), F32, 66), rand((N,), F32, 67)
    got = ops.linear(x.to(DEV), w.to(DEV), b.to(DEV))
    close(got, x.double() @ w.double().T + b.double(), 3e-6, (M, N, K))
    for m in (1, 64, 65, 200):
        few = ops.linear(x[M - m:].to(DEV), w.to(DEV), b.to(DEV))
        assert torch.equal(few, got[M - m:]), m
    for n in (5, 64, 1000):               # the last columns as a matrix of their own
        few = ops.linear(x.to(DEV), w[N - n:].to(DEV), b[N - n:].to(DEV))
        assert torch.equal(few, got[:, N - n:]), n


@pytest.mark.parametrize("M", [1, 8, 20, 40, 65, 700])
def test_a_product_over_nothing_is_its_bias(ops, M):  # noqa: F811
    b = rand((9000,), F32, 64).to(DEV)
    got = ops.linear(torch.empty((M, 0), device=DEV), torch.empty((9000, 0), device=DEV), b)
    assert torch.equal(got, b.expand(M, -1))


ATTENTION = [
    # H, G, d, page, held before, new rows, window
    (16, 8, 64, 16, [0, 5, 300], [37, 1, 70], 0),
    (2, 2, 16, 16, [0, 127, 128, 1000], [17, 1, 1, 16], 0),
    (3, 1, 32, 8, [3, 0], [6, 33], 0),
    (6, 1, 48, 4, [0, 19, 40], [9, 5, 1], 11),
    (24, 1, 80, 16, [60, 2], [3, 20], 0),
    (40, 2, 96, 16, [0, 90], [12, 2], 50),
    (4, 4, 112, 16, [30, 0], [40, 1], 0),
    (8, 2, 128, 32, [200, 0], [5, 66], 64),
]


@pytest.mark.parametrize("case", ATTENTION)
def test_attention_float32(ops, case):  # noqa: F811
    H, G, d, ps, before, new, window = case
    c = paged_case(21, F32, H, G, d, ps, before, new)
    held = {k: (v.to(DEV) if torch.is_tensor(v) else v) for k, v in c.items()}
    cos = torch.zeros((max(a + n for a, n in zip(before, new)) + 1, 1), device=DEV)
    ops.qk_norm_rope_store(held["qkv"], H, G, d, None, None, 1e-5, cos, cos, 0, 0, held["k_pool"],
                           held["v_pool"], held["row_pos"], held["row_seg"], held["bt"], ps)

    def run(rows):
        q = held["qkv"][rows]
        return ops.paged_attention(q, H, G, d, held["k_pool"], held["v_pool"],
                                   held["row_pos"][rows], held["row_seg"][rows], held["bt"], ps,
                                   d ** -0.5, window=window)

    T = c["row_pos"].shape[0]
    got = run(torch.arange(T, device=DEV))
    want = ref.paged_attention(held["qkv"].cpu(), H, G, d, held["k_pool"].cpu(),
                               held["v_pool"].cpu(), c["row_pos"], c["row_seg"], c["bt"], ps,
                               d ** -0.5, window=window)
    close(got, want, 6e-6, "attention")
    for t in (0, T // 2, T - 1):           # a row alone: the same bits
        assert torch.equal(run(torch.tensor([t], device=DEV))[0], got[t]), t


@pytest.mark.parametrize("bad", [math.inf, math.nan])
def test_a_later_rows_odd_value_stays_with_the_rows_that_see_it(ops, bad):  # noqa: F811
    H, G, d, ps = 4, 2, 32, 16
    c = paged_case(22, F32, H, G, d, ps, [0], [20])
    held = {k: (v.to(DEV) if torch.is_tensor(v) else v) for k, v in c.items()}
    held["qkv"][13, (H + G) * d + 5] = bad          # a value of row 13, kv head 0
    cos = torch.zeros((21, 1), device=DEV)
    ops.qk_norm_rope_store(held["qkv"], H, G, d, None, None, 1e-5, cos, cos, 0, 0, held["k_pool"],
                           held["v_pool"], held["row_pos"], held["row_seg"], held["bt"], ps)
    out = ops.paged_attention(held["qkv"], H, G, d, held["k_pool"], held["v_pool"],
                              held["row_pos"], held["row_seg"], held["bt"], ps, d ** -0.5).cpu()
    assert torch.isfinite(out[:13]).all() and not torch.isfinite(out[13:, 5]).any()
    rest = torch.ones(H * d, dtype=torch.bool)
    rest[[5, d + 5]] = False                        # the two heads on kv head 0
    assert torch.isfinite(out[:, rest]).all()


def test_rows_far_apart_read_their_own_pages_only(ops):  # noqa: F811
    """Neighbouring rows of a segment whose positions do not follow one another: no page between them
    is needed, so the table may name none; a row before the first position has no key at all."""
    H, G, d, ps, window = 4, 2, 32, 8, 11
    pos = [5, 6, 100, 101, 3, 160, 159]
    g = torch.Generator().manual_seed(23)
    needed = sorted({k // ps for p in pos for k in range(max(p - window + 1, 0), p + 1)})
    bt = torch.full((1, 21), -1, dtype=torch.int32)
    bt[0, needed] = torch.randperm(len(needed), generator=g).int()
    k = torch.randn(len(needed), G, ps, d, generator=g)
    v = torch.randn(len(needed), G, d, ps, generator=g)
    q = torch.randn(len(pos), H * d, generator=g)
    rows = torch.tensor(pos, dtype=torch.int32), torch.zeros(len(pos), dtype=torch.int32)
    want = ref.paged_attention(q, H, G, d, k, v, *rows, bt, ps, d ** -0.5, window=window)

    def run(q, pos):
        seg = torch.zeros(len(pos), dtype=torch.int32, device=DEV)
        return ops.paged_attention(q.to(DEV), H, G, d, k.to(DEV), v.to(DEV),
                                   torch.tensor(pos, dtype=torch.int32, device=DEV), seg,
                                   bt.to(DEV), ps, d ** -0.5, window=window)
    got = run(q, pos)
    close(got, want, 6e-6, "rows far apart")
    for t in range(len(pos)):
        assert torch.equal(run(q[t:t + 1], pos[t:t + 1])[0], got[t]), t
    before = run(torch.cat([q[:1], q[:1]]), [-1, 0])
    assert not torch.isfinite(before[0]).any()
    assert torch.equal(before[1], run(q[:1], [0])[0])


@pytest.mark.parametrize("d", [64, 80])
@pytest.mark.parametrize("n_new", [1, 16, 21])
@pytest.mark.parametrize("window", [0, 150])
def test_attention_around_whole_rounds_of_its_waves(ops, d, n_new, window):  # noqa: F811
    """A wave takes every eighth (heads above 64: fourth) step of 16 keys, two sets of registers in turn, its pages
    two steps ahead: contexts on both sides of none, one, two and three of a wave's steps, the pages in front of a
    window given back, NaN in every place that no request holds, single rows beside one another."""
    H, G, ps, scale = 4, 2, 16, d ** -0.5
    per_round = 16 * (8 if d <= 64 else 4)
    held = sorted({max(0, per_round * r + e - n_new) for r in range(4) for e in (-16, -1, 0, 1, 17)})
    g = torch.Generator().manual_seed(d + n_new)
    need = [(a + n_new + ps - 1) // ps for a in held]
    k = torch.full((sum(need) + 1, G, ps, d), math.nan)
    v = torch.full((sum(need) + 1, G, d, ps), math.nan)
    bt = torch.full((len(held), max(need)), -1, dtype=torch.int32)
    order, at, pos, seg = torch.randperm(sum(need), generator=g).int() + 1, 0, [], []
    for i, a in enumerate(held):
        first = max(a - window + 1, 0) // ps if window else 0          # the first page that some row needs
        for p in range(first, need[i]):
            n = min(ps, a + n_new - p * ps)
            bt[i, p] = order[at + p]
            k[bt[i, p], :, :n] = torch.randn(G, n, d, generator=g)
            v[bt[i, p], :, :, :n] = torch.randn(G, d, n, generator=g)
        at += need[i]
        pos += range(a, a + n_new)
        seg += [i] * n_new
    q = torch.randn(len(pos), H * d, generator=g)
    rows = [torch.tensor(x, dtype=torch.int32) for x in (pos, seg)]
    got = ops.paged_attention(q.to(DEV), H, G, d, k.to(DEV), v.to(DEV), *(x.to(DEV) for x in rows), bt.to(DEV), ps,
                              scale, window=window)
    want = ref.paged_attention(q, H, G, d, k, v, *rows, bt, ps, scale, window=window)
    close(got, want, 6e-6, "attention")


@pytest.mark.parametrize("M,N,K", [(70, 130, 256), (330, 9216, 128)])
def test_blocks_over_operands_of_four_gibibytes_give_the_same_bits(ops, M, N, K):  # noqa: F811
    """Rows of x so far apart that 32 bits do not address them: tiles through registers and not straight into LDS."""
    apart = (1 << 30) // M + 4 & ~3
    far = torch.empty((M - 1) * apart + K, device=DEV).as_strided((M, K), (apart, 1))
    x, w = rand((M, K), F32, 71).to(DEV), rand((N, K), F32, 72).to(DEV)
    far.copy_(x)
    assert M * apart >= 1 << 30 and apart % 4 == 0
    assert torch.equal(ops.linear(far, w), ops.linear(x, w))
    if ops.linear_swiglu_f32_takes(x, w):
        assert torch.equal(ops.linear_swiglu_f32(far, w), ops.linear_swiglu_f32(x, w))


# up to 4 rows and 1,024 columns a block owns four columns and four runs stand side by side; both sides of either
@pytest.mark.parametrize("N", [3, 1023, 1024, 1025])
@pytest.mark.parametrize("K", [20, 130, 1024, 2181, 4608, 5000])
def test_four_columns_a_block(ops, N, K):  # noqa: F811
    x, w, b = (rand(shape, F32, 65 + i).to(DEV) for i, shape in enumerate([(9, K), (N, K), (N,)]))
    whole = ops.linear(x, w, b)
    for M in (1, 2, 3, 4, 5):
        assert torch.equal(ops.linear(x[:M].contiguous(), w, b), whole[:M]), M
