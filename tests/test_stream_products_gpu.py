"""Float32 decode steps of few rows on the C side of a step, where products add into the residual stream and norm it
themselves: the same logits as the host's parts give, at sizes that those products do not take."""
import numpy as np
import pytest
import torch

from test_c_walk_gpu import DEV, replay

pytestmark = pytest.mark.gpu


def one_by_one(vocab, rows, prompt=9, steps=3):
    """A prompt for each of ``rows`` requests, then steps of one token each, all logits wanted."""
    rng = np.random.default_rng(rows)
    tok = lambda n: [int(t) for t in rng.integers(0, vocab, size=n)]  # noqa: E731
    out = [{"step": 0, "entries": [{"id": f"r{i}", "tokens": tok(prompt + i), "want": [prompt + i - 1]}
                                   for i in range(rows)], "end": []}]
    for s in range(steps):
        out.append({"step": s + 1, "entries": [{"id": f"r{i}", "tokens": tok(1), "want": [0]} for i in range(rows)],
                    "end": [f"r{i}" for i in range(rows)] if s == steps - 1 else []})
    return out


def from_both_sides(model, steps, tmp_path):
    got, runner = replay(model, steps, 512, tmp_path / "c", True, False)
    assert runner._cplan is not None
    want, _ = replay(model, steps, 512, tmp_path / "host", False, False)
    for a, b in zip(got, want):
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("rows", [1, 4])
@pytest.mark.parametrize("hidden", [1, 3, 4, 5])
def test_a_feed_forward_of_few_columns(tmp_path, hidden, rows):
    """The last product of a layer with an inner width below four, which the product into the stream does not take, and
    from there on."""
    from kappai_amd.config import config_from_dict
    from kappai_amd.models import load_model
    from kappai_amd.weights import write_random_model
    from tiny import TINY_A
    raw = dict(TINY_A, hidden_size=128, intermediate_size=hidden)
    write_random_model(tmp_path / "m", config_from_dict(raw), seed=3, std=0.1, norm_jitter=0.1)
    model = load_model(tmp_path / "m", "float32", DEV)
    from_both_sides(model, one_by_one(raw["vocab_size"], rows), tmp_path)
