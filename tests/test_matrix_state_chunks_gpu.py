"""The gated sum and the delta rule in chunks of 16 tokens on the matrix cores, against float64 and
against the walk along the tokens."""
import pytest
import torch

from test_kernels_gpu import BF16, DEV, F32, ops  # noqa: F401

F64 = torch.float64


def exact(q, k, v, a, beta, S):
    """One sequence in float64: q, k [T, H, d], v [T, H, dv], a [T, H, d], beta [T, H] or None,
    S [H, d, dv]; returns o [T, H, dv] and the state behind the last token."""
    out = []
    for t in range(q.shape[0]):
        S = a[t][:, :, None] * S
        u = v[t]
        if beta is not None:
            u = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
        S = S + k[t][:, :, None] * u[:, None, :]
        out.append((S * q[t][:, :, None]).sum(1))
    return torch.stack(out), S


@pytest.mark.parametrize("segments,longest,chunked", [
    (1, 1, False), (1, 25, False), (1, 26, True), (64, 1, False), (61, 145, False), (61, 146, True)])
def test_when_chunks_are_taken(segments, longest, chunked):
    from types import SimpleNamespace

    from kappai_amd.kernels import ops as real_ops
    from kappai_amd.parts.linear_attention import _chunk_rows
    batch = SimpleNamespace(seg_slot=torch.zeros(segments), max_segment_rows=longest)
    assert _chunk_rows(batch) == (real_ops.MATRIX_STATE_CHUNK_ROWS if chunked else 0)
    assert _chunk_rows(batch, F32) == 0


# key sizes below, at and beyond a tile of 64 and of 128, columns that end inside 16; segments of less
# than a chunk, of whole chunks (more and fewer than are asked for ahead) and one token more
@pytest.mark.gpu
@pytest.mark.parametrize("H,Hk,d,dv", [(2, 2, 64, 64), (4, 2, 64, 72), (2, 1, 128, 128), (3, 3, 4, 5),
                                       (2, 2, 24, 16), (1, 1, 72, 33)])
@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("strong", [False, True])
@pytest.mark.parametrize("dtype", [F32, BF16])
def test_chunks_against_the_walk(ops, H, Hk, d, dv, delta, strong, dtype):  # noqa: F811
    lens, pos0 = [33, 1, 16, 15, 130, 64], [0, 7, 5, 0, 3, 0]
    T, S = sum(lens), len(lens)
    g = torch.Generator().manual_seed(H * 1000 + d + dv)
    q, k, v = (torch.randn(T, n, generator=g).to(dtype) for n in (Hk * d, Hk * d, H * dv))
    # decays near one (a few per cent a token), or anything down to exp(-80) and below
    z = torch.randn(T, H * d, generator=g) * (30.0 if strong else 1.0) - (0.0 if strong else 3.0)
    z, b = z.to(dtype), torch.randn(T, H, generator=g).to(dtype)
    rate = torch.rand(H, generator=g) + 0.1
    slots = [5, 0, 3, 1, 6, 2]
    state = torch.randn(8, H, dv, d, generator=g)
    for i, p in enumerate(pos0):
        if p == 0:
            state[slots[i]] = float("nan")
    start = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    ints = [start.to(DEV)] + [torch.tensor(x, dtype=torch.int32, device=DEV) for x in (pos0, slots)]

    def run(chunk_rows):
        st = state.to(DEV)
        o = ops.matrix_state_recurrence(
            q.to(DEV), k.to(DEV), v.to(DEV), z.to(DEV), H, Hk, d, dv, rate.to(DEV), None, 1.0,
            d ** -0.5, st, *ints, beta=b.to(DEV) if delta else None, unit_qk=delta,
            chunk_rows=chunk_rows)
        return o.cpu(), st.cpu()

    qd, kd = (x.to(F64).reshape(T, Hk, d) for x in (q, k))
    if delta:
        qd, kd = (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (qd, kd))
    qd, kd = ((x * s).repeat_interleave(H // Hk, 1) for x, s in ((qd, d ** -0.5), (kd, 1.0)))
    a = torch.exp(-rate.to(F64)[:, None] * torch.nn.functional.softplus(z.to(F64).reshape(T, H, d),
                                                                     threshold=1e9))
    (o, st), (o_walk, st_walk) = run(ops.MATRIX_STATE_CHUNK_ROWS), run(0)
    untouched = [i for i in range(8) if i not in slots]
    assert torch.equal(st[untouched], state[untouched])
    errs = torch.zeros(2, 2, dtype=F64)
    for i in range(S):
        t = slice(int(start[i]), int(start[i + 1]))
        S0 = state[slots[i]].to(F64).transpose(1, 2) if pos0[i] else torch.zeros(H, d, dv, dtype=F64)
        want, last = exact(qd[t], kd[t], v[t].to(F64).reshape(-1, H, dv), a[t],
                           torch.sigmoid(b[t].to(F64)) if delta else None, S0)
        for n, (oo, ss) in enumerate(((o, st), (o_walk, st_walk))):
            e_o = (oo[t].reshape(-1, H, dv).to(F64) - want).abs().max() / want.abs().max()
            e_s = (ss[slots[i]].to(F64).transpose(1, 2) - last).abs().max() / last.abs().max()
            errs[n] = torch.maximum(errs[n], torch.stack([e_o, e_s]))
    # float32 sums over d and up to 130 tokens: as the walk's own test has it
    assert torch.isfinite(o).all() and (errs[0] < 2e-5).all(), errs


@pytest.mark.gpu
def test_empty_and_refused(ops):  # noqa: F811
    """A segment without tokens keeps its state; sizes the form does not take walk the tokens."""
    for d in (16, 18, 132):
        T, H, dv = 40, 1, 8
        g = torch.Generator().manual_seed(d)
        q, k, v, z = (torch.randn(T, n, generator=g).to(DEV) for n in (d, d, dv, d))
        start = torch.tensor([0, 0, 40], dtype=torch.int32, device=DEV)
        pos = torch.tensor([3, 0], dtype=torch.int32, device=DEV)
        slot = torch.tensor([1, 0], dtype=torch.int32, device=DEV)
        outs = []
        for rows in (0, ops.MATRIX_STATE_CHUNK_ROWS):
            st = torch.ones(2, H, dv, d, device=DEV)
            outs.append((ops.matrix_state_recurrence(
                q, k, v, z, H, H, d, dv, torch.ones(1, device=DEV), None, 1.0, 1.0, st, start, pos,
                slot, chunk_rows=rows), st))
            assert torch.equal(st[1], torch.ones_like(st[1]))
        (o, s), (o2, s2) = outs
        assert (o - o2).abs().max() <= 2e-5 * o.abs().max() and (s - s2).abs().max() <= 2e-5 * s.abs().max()
        if d != 16:
            assert torch.equal(o, o2) and torch.equal(s, s2)


@pytest.mark.gpu
@pytest.mark.parametrize("H,Hk,d,dv", [(2, 1, 64, 24), (2, 2, 128, 16)])
@pytest.mark.parametrize("what", ["v", "k", "q", "z", "beta"])
@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_value_that_is_no_number_stays_with_its_token_and_those_behind_it(  # noqa: F811
        ops, H, Hk, d, dv, what, delta, bad):
    """The tokens before it, other segments and (for a value) other columns keep their bits; what is
    finite on the walk is finite in chunks."""
    if what == "beta" and not delta:
        return
    at, lens = 21, [40, 5]               # the sixth token of the second chunk
    T = sum(lens)
    g = torch.Generator().manual_seed(d + dv)
    x = {n: torch.randn(T, c, generator=g) for n, c in
         (("q", Hk * d), ("k", Hk * d), ("v", H * dv), ("z", H * d), ("beta", H))}
    state = torch.randn(2, H, dv, d, generator=g)
    ints = [torch.tensor(t, dtype=torch.int32, device=DEV) for t in ([0, 40, 45], [3, 0], [1, 0])]

    def run(x, chunk_rows):
        st, on = state.to(DEV), {n: t.to(DEV) for n, t in x.items()}
        o = ops.matrix_state_recurrence(
            on["q"], on["k"], on["v"], on["z"], H, Hk, d, dv, torch.ones(H, device=DEV), None, 1.0,
            d ** -0.5, st, *ints, beta=on["beta"] if delta else None, unit_qk=delta,
            chunk_rows=chunk_rows)
        return o.cpu(), st.cpu()

    rows = ops.MATRIX_STATE_CHUNK_ROWS
    clean, clean_state = run(x, rows)
    x[what] = x[what].clone()
    x[what][at, 1] = bad
    (o, st), (walk, walk_state) = run(x, rows), run(x, 0)
    assert torch.equal(o[:at], clean[:at]) and torch.equal(o[40:], clean[40:])
    assert torch.equal(st[0], clean_state[0])
    if what == "v":
        rest = torch.arange(H * dv) != 1
        assert torch.equal(o[:, rest], clean[:, rest])
        assert not torch.isfinite(o[at:40, 1]).any()
    assert torch.equal(torch.isfinite(o), torch.isfinite(walk))
    assert torch.equal(torch.isfinite(st), torch.isfinite(walk_state))


@pytest.mark.gpu
@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("d,dv", [(64, 40), (128, 16)])
def test_slabs_of_scratch(ops, monkeypatch, d, dv, delta):  # noqa: F811
    """A scratch of any size gives the same bits; where there is no memory for one the tokens are
    walked."""
    lens, pos0, H = [70, 1, 16, 33, 15, 200], [0, 9, 3, 0, 4, 0], 2
    T, g = sum(lens), torch.Generator().manual_seed(d)
    q, k, v, z = (torch.randn(T, H * n, generator=g).to(DEV) for n in (d, d, dv, d))
    b = torch.randn(T, H, generator=g).to(DEV) if delta else None
    start = [0] + list(torch.tensor(lens).cumsum(0))
    ints = [torch.tensor(t, dtype=torch.int32, device=DEV) for t in (start, pos0, [5, 0, 3, 1, 4, 2])]
    state = torch.randn(6, H, dv, d, generator=g)

    def run(chunk_rows=ops.MATRIX_STATE_CHUNK_ROWS):
        st = state.to(DEV)
        return ops.matrix_state_recurrence(
            q, k, v, z, H, H, d, dv, torch.ones(H, device=DEV), None, 1.0, d ** -0.5, st, *ints,
            beta=b, unit_qk=delta, chunk_rows=chunk_rows), st

    whole, walked = run(), run(0)
    assert not torch.equal(whole[0], walked[0])
    slots = T // 16 + len(lens)
    one = (33 * d + 256 + (16 * d if delta else 0) + (dv + 15) // 16 * 256) * H
    empty, taken = torch.empty, []

    def spy(*size, **kw):
        taken.append(size[0])
        return empty(*size, **kw)
    for chunks in (0, 1, 2, 5, slots - 1, slots, slots + 1):
        monkeypatch.setattr(ops, "MATRIX_STATE_SCRATCH_FLOATS", chunks * one + one // 2)
        monkeypatch.setattr(ops.torch, "empty", spy)
        o, st = run()
        monkeypatch.setattr(ops.torch, "empty", empty)
        assert one * min(max(chunks, 1), slots) in taken
        taken.clear()
        assert torch.equal(o, whole[0]) and torch.equal(st, whole[1]), chunks

    def no_room(*size, **kw):
        if isinstance(size[0], int):
            raise torch.cuda.OutOfMemoryError("no room for the scratch")
        return empty(*size, **kw)
    monkeypatch.setattr(ops.torch, "empty", no_room)
    o, st = run()
    monkeypatch.setattr(ops.torch, "empty", empty)
    assert torch.equal(o, walked[0]) and torch.equal(st, walked[1])
