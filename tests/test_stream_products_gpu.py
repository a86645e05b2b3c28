"""Float32 decode steps of few rows on the C side of a step, where products add into the residual stream and norm it
themselves: the same logits as the host's parts give, at sizes that those products do not take."""
from dataclasses import dataclass

import numpy as np
import pytest
import torch

from test_c_walk_gpu import DEV, define_toy_block, replay, toy_block_library

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


def define_two_readers():
    """An architecture of blocks from outside that give one norm's rows to a mixer and a feed-forward, both of which
    may add into the stream (``toy_two_readers_run`` of tests/toy_parts/layer_norm_block.hip)."""
    from ctypes import Structure

    from kappai_amd.config import ModelConfig, register_architecture
    from kappai_amd.models import Model
    from kappai_amd.parts import BLOCKS, OutputHead, TokenEmbedding, make_part, register_part
    from kappai_amd.parts.cdesc import RUNNER_BLOCK, NormPartDesc, PartDesc
    define_toy_block()
    if "toy_two_readers" in BLOCKS:
        return

    class TwoReadersDesc(Structure):
        _fields_ = [("norm", NormPartDesc), ("mixer", PartDesc), ("feed_forward", PartDesc)]

    class TwoReaders(BLOCKS["toy_parallel"]):
        def forward(self, h, batch, cache, shared_cache=False):
            return super().forward(h, batch, cache, shared_cache)

        def c_call(self, plan, view, shared_cache=False):
            lib = toy_block_library()
            lib.toy_two_readers_run.restype = None         # only its address is used
            plan.register_runner("block.toy_two_readers", RUNNER_BLOCK, lib.toy_two_readers_run, TwoReadersDesc)
            return plan.call("block.toy_two_readers", TwoReadersDesc(
                self.norm.c_norm(plan), self.mixer.c_part(plan, view, shared_cache),
                self.feed_forward.c_part(plan, None, False)))

    register_part("block", "toy_two_readers", TwoReaders)

    @dataclass
    class Config(ModelConfig):
        width: int = 0
        vocab_size: int = 0
        max_position_embeddings: int = 512

        @classmethod
        def from_dict(cls, raw):
            return cls(architecture="ToyTwoReadersForCausalLM", width=raw["width"], vocab_size=raw["vocab_size"])

        def to_dict(self):
            return {"architectures": ["ToyTwoReadersForCausalLM"], "width": self.width, "vocab_size": self.vocab_size}

    def build(cfg, dtype):
        W = cfg.width
        how = dict(width=W, dtype=dtype)
        rot = make_part("position_encoding", "rotary", head_dim=32, theta=100.0)

        def norm(name):
            return make_part("norm", "rmsnorm", name=name, eps=1e-5, **how)

        def block(i, mixer):
            return make_part("block", "toy_two_readers", norm=norm(f"b{i}.n"), mixer=mixer,
                             feed_forward=make_part("feed_forward", "swiglu", prefix=f"b{i}.ff.", hidden=96, **how))
        layers = [block(0, make_part("mixer", "conv", prefix="b0.c.", kernel_size=3, bias=True, **how)),
                  block(1, make_part("mixer", "attention", prefix="b1.a.", num_heads=4, num_kv_heads=2, head_dim=32,
                                     position=rot, qk_norm_eps=1e-5, **how)),
                  block(2, make_part("mixer", "conv", prefix="b2.c.", kernel_size=3, bias=True, **how))]
        emb = TokenEmbedding("emb", cfg.vocab_size, W)
        return Model(cfg, dtype, emb, layers, norm("final"), OutputHead("head", cfg.vocab_size, W, tied_to=emb))

    register_architecture("ToyTwoReadersForCausalLM", Config, build)


@pytest.mark.parametrize("rows", [1, 3])
def test_rows_that_two_parts_read(tmp_path, rows):
    """The rows of one norm, read by a second part after the first has added into the stream: they are the rows that
    were normed, whatever has joined the stream since."""
    from kappai_amd.config import config_from_dict
    from kappai_amd.models import load_model
    from kappai_amd.weights import write_random_model
    define_two_readers()
    raw = {"architectures": ["ToyTwoReadersForCausalLM"], "width": 128, "vocab_size": 211}
    write_random_model(tmp_path / "m", config_from_dict(raw), seed=5, std=0.1, norm_jitter=0.1)
    from_both_sides(load_model(tmp_path / "m", "float32", DEV), one_by_one(raw["vocab_size"], rows), tmp_path)


def define_stream_map():
    """An architecture whose feed-forwards read the stream itself (``toy_stream_map_run`` of
    tests/toy_parts/layer_norm_block.hip)."""
    from kappai_amd.config import ModelConfig, register_architecture
    from kappai_amd.models import Model
    from kappai_amd.parts import (FEED_FORWARDS, FeedForward, Linear, OutputHead, TokenEmbedding, make_part,
                                  register_part)
    from kappai_amd.parts.cdesc import RUNNER_PART, LinearDesc
    if "toy_stream_map" in FEED_FORWARDS:
        return

    class StreamMap(FeedForward):
        adds_residual = True           # (for the stream that comes with ``into``)

        def __init__(self, prefix, width):
            self.map = Linear([prefix + "map"], width, [width])

        def tensor_specs(self):
            return self.map.tensor_specs()

        def bind(self, tensors):
            self.map.bind(tensors)

        def weight_bytes(self):
            return self.map.weight_bytes()

        def forward(self, x, batch, into=None):
            return self.map.forward(into.resid)

        def c_part(self, plan, view=None, shared_cache=False):
            lib = toy_block_library()
            lib.toy_stream_map_run.restype = None         # only its address is used
            plan.register_runner("feed_forward.toy_stream_map", RUNNER_PART, lib.toy_stream_map_run, LinearDesc)
            return plan.part("feed_forward.toy_stream_map", plan.linear(self.map), adds_residual=True)

    register_part("feed_forward", "toy_stream_map", StreamMap)

    @dataclass
    class Config(ModelConfig):
        width: int = 0
        vocab_size: int = 0
        max_position_embeddings: int = 512

        @classmethod
        def from_dict(cls, raw):
            return cls(architecture="ToyStreamMapForCausalLM", width=raw["width"], vocab_size=raw["vocab_size"])

        def to_dict(self):
            return {"architectures": ["ToyStreamMapForCausalLM"], "width": self.width, "vocab_size": self.vocab_size}

    def build(cfg, dtype):
        how = dict(width=cfg.width, dtype=dtype)

        def norm(name):
            return make_part("norm", "rmsnorm", name=name, eps=1e-5, **how)
        layers = [make_part("block", "pre_norm", mixer_norm=norm(f"b{i}.n1"),
                            mixer=make_part("mixer", "conv", prefix=f"b{i}.c.", kernel_size=3, bias=True, **how),
                            ffn_norm=norm(f"b{i}.n2"),
                            feed_forward=make_part("feed_forward", "toy_stream_map", prefix=f"b{i}.", width=cfg.width))
                  for i in range(2)]
        emb = TokenEmbedding("emb", cfg.vocab_size, cfg.width)
        return Model(cfg, dtype, emb, layers, norm("final"), OutputHead("head", cfg.vocab_size, cfg.width, tied_to=emb))

    register_architecture("ToyStreamMapForCausalLM", Config, build)


@pytest.mark.parametrize("rows", [1, 3, 8])
def test_a_product_of_the_stream_into_the_stream(tmp_path, rows):
    """Rows that lie in the stream which their product would join: the product may not write them while its other
    blocks still read them, so it goes another way (width 1,024: a block for every CU reads all of them)."""
    from kappai_amd.config import config_from_dict
    from kappai_amd.models import load_model
    from kappai_amd.weights import write_random_model
    define_stream_map()
    raw = {"architectures": ["ToyStreamMapForCausalLM"], "width": 1024, "vocab_size": 211}
    write_random_model(tmp_path / "m", config_from_dict(raw), seed=5, std=0.03, norm_jitter=0.1)
    from_both_sides(load_model(tmp_path / "m", "float32", DEV), one_by_one(raw["vocab_size"], rows), tmp_path)
