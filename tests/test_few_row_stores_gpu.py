"""What stands between projections and paged attention, up to 32 rows with a block for every 256 places of a row and
beyond with a block a row: the same queries, keys and values bit for bit, at places that are no whole blocks."""
import pytest
import torch

from test_kernels_gpu import BF16, DEV, F32, ops, rand  # noqa: F401

pytestmark = pytest.mark.gpu
I32, PS, ROWS = torch.int32, 16, 33


def ints(values):
    return torch.tensor(values, dtype=I32, device=DEV)


def around_the_rule(G, D, dtype, store):
    """``store(rows, pools..., positions...)`` for 33 rows at once and for 1 and 32 of them."""
    pos = torch.arange(ROWS) * 7 % 60
    seg = torch.arange(ROWS) % 3
    tables = ints([[1, 2, 3, 4], [5, 6, 7, 8], [9, 10, 11, 12]])
    got = []
    for cuts in ([0, ROWS], [0, 1, ROWS]):
        kp, vp = torch.zeros((13, G, PS, D), dtype=dtype, device=DEV), torch.zeros((13, G, D, PS), dtype=dtype,
                                                                                  device=DEV)
        q = [store(slice(a, b), kp, vp, ints(pos[a:b].tolist()), ints(seg[a:b].tolist()), tables)
             for a, b in zip(cuts, cuts[1:])]
        got.append((torch.cat(q), kp, vp))
    return got


def alike(got, rank=0, D=0):
    (q0, k0, v0), (q1, k1, v1) = got
    if rank:                                     # (places that are left for another kernel)
        q0, q1 = q0.view(ROWS, -1, D)[..., rank:], q1.view(ROWS, -1, D)[..., rank:]
    assert torch.equal(q0, q1) and torch.equal(k0, k1) and torch.equal(v0, v1) and k0.any().item()


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("H,G,d,dv,D", [(1, 1, 8, 8, 16), (8, 2, 80, 64, 128), (6, 3, 48, 40, 48), (16, 2, 64, 64, 64)])
def test_projection_norm_store(ops, dtype, H, G, d, dv, D):  # noqa: F811
    proj = rand((ROWS, H * d + G * (d + dv)), dtype, 1).to(DEV)
    qw, kw = rand((H * d,), F32, 2).to(DEV), rand((G * d,), F32, 3).to(DEV)
    alike(around_the_rule(G, D, dtype, lambda at, kp, vp, pos, seg, tables: ops.projection_norm_store(
        proj[at], H, G, d, dv, D, qw, kw, 1e-5, 0.1, 16, kp, vp, pos, seg, tables, PS)))


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("keys", [False, True])
@pytest.mark.parametrize("H,G,d,D", [(1, 1, 8, 16), (8, 2, 80, 128), (6, 3, 48, 48)])
def test_rotate_widen_store(ops, dtype, mode, keys, H, G, d, D):  # noqa: F811
    proj = rand((ROWS, H * d + G * d * (1 if keys else 2)), dtype, 4).to(DEV)
    cos, sin = rand((64, 4), F32, 5).to(DEV), rand((64, 4), F32, 6).to(DEV)
    alike(around_the_rule(G, D, dtype, lambda at, kp, vp, pos, seg, tables: ops.rotate_widen_store(
        proj[at], H, G, d, d, D, cos, sin, 8, mode, keys, kp, vp, pos, seg, tables, PS)))


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("H,d,rot,r,D", [(1, 8, 8, 8, 16), (16, 64, 32, 256, 320), (5, 32, 16, 96, 112), (2, 8, 0, 16, 16)])
def test_latent_store(ops, dtype, H, d, rot, r, D):  # noqa: F811
    q, kv = rand((ROWS, H * (d + rot)), dtype, 7).to(DEV), rand((ROWS, r + rot), dtype, 8).to(DEV)
    cos, sin = rand((64, 4), F32, 9).to(DEV), rand((64, 4), F32, 10).to(DEV)
    w = rand((r,), F32, 11).to(DEV)
    dims = min(8, rot)
    alike(around_the_rule(1, D, dtype, lambda at, kp, vp, pos, seg, tables: ops.latent_store(
        q[at], kv[at], H, d, rot, r, D, w, 1e-5, cos if dims else None, sin if dims else None, dims,
        1 if dims else 0, kp, vp, pos, seg, tables, PS)), r, D)
