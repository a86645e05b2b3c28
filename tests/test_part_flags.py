"""What a mixer announces it takes and does, in subclasses of the framework's own: one that brings a ``forward`` of its
own is called as that ``forward`` was written, with plain rows and without ``into``."""
import pytest

from kappai_amd.parts.block import PreNormBlock
from kappai_amd.parts.gated_unit import RealGatedUnit
from kappai_amd.parts.linear_attention import FixedDecayAttention
from kappai_amd.parts.parallel import ParallelMixer
from kappai_amd.parts.scored_attention import ScoredAttention

FLAGS = {RealGatedUnit: ("takes_deferred_rows", "adds_residual"), FixedDecayAttention: ("takes_deferred_rows",),
         ScoredAttention: ("takes_deferred_rows",), ParallelMixer: ("takes_deferred_rows", "adds_residual")}


def made(cls):
    """An instance without what its constructor would need (a pair of mixers that announce everything)."""
    m = cls.__new__(cls)
    if issubclass(cls, ParallelMixer):
        m.left = m.right = RealGatedUnit.__new__(RealGatedUnit)
        m.summed = True
    return m


class Norm:
    can_defer = True

    def fold(self):
        return None, 1e-5

    def add_norm(self, resid, delta, defer=False):
        return defer


@pytest.mark.parametrize("cls", list(FLAGS))
def test_a_subclass_with_a_forward_of_its_own(cls):
    def forward(self, x, batch, cache, shared_cache=False):
        return 2 * cls.forward(self, x, batch, cache, shared_cache)

    changed = made(type("Changed", (cls,), {"forward": forward}))
    kept = made(type("Kept", (cls,), {"weight_bytes": lambda self: 0}))
    said = made(type("Said", (cls,), {"forward": forward, **{f: True for f in FLAGS[cls]}}))
    for flag in FLAGS[cls]:
        assert [getattr(m, flag) for m in (made(cls), kept, said, changed)] == [True, True, True, False]
    # and the block calls it so
    norm = Norm()
    assert PreNormBlock._into(changed, None, norm, kept) is None
    assert (PreNormBlock._into(kept, None, norm, kept) is not None) == ("adds_residual" in FLAGS[cls])
    assert PreNormBlock._normed(norm, None, None, changed) is not True
    assert PreNormBlock._normed(norm, None, None, kept) is True
