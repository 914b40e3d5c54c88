"""A block that goes on with some rows alone (``forward_rows``) computes for them what the whole block computes."""

from types import SimpleNamespace

import pytest
import torch

from twins import TwinKernels
from simple_inference_amd.parts import BiasedDelta, BuildEnv, NormedSum, ResidualStream, ScaledSum
from simple_inference_amd.parts.block import GatedPreNormBlock, PreNormBlock
from simple_inference_amd.parts.norm import RMSNorm

TOKENS, HIDDEN = 40, 24


class RowTwins(TwinKernels):
    def take_rows(self, x, rows):
        return x[rows.long()]


def rnd(*shape, seed, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


class Mixer:
    """Returns what it is given, whatever it is asked for."""

    def __init__(self, result):
        self.result = result

    def forward(self, h, ctx, cache):
        return self.result()


class Half:
    by_row = True

    def forward(self, h, ctx):
        return h * 0.5


class Gate:
    by_row = True
    bias = None

    def logits(self, h):
        return h * 2.0


def norm(env):
    n = RMSNorm({"size": HIDDEN, "eps": 1e-5}, env)
    n.bind({"weight": 1.0 + 0.1 * rnd(HIDDEN, seed=9, dtype=torch.float32)})
    return n


RESULTS = {
    "a tensor": lambda k: rnd(TOKENS, HIDDEN, seed=1),
    "two terms": lambda k: ScaledSum([(rnd(TOKENS, HIDDEN, seed=1), 0.7), (rnd(TOKENS, HIDDEN, seed=2), 1.2)], k),
    "three terms": lambda k: ScaledSum([(rnd(TOKENS, HIDDEN, seed=i), 0.3 * i) for i in (1, 2, 3)], k),
    "normed terms": lambda k: NormedSum([(rnd(TOKENS, HIDDEN, seed=i), 0.3 * i, rnd(HIDDEN, seed=i, dtype=torch.float32), 1e-5)
                                         for i in (1, 2)], k),
    "a bias": lambda k: BiasedDelta(rnd(TOKENS, HIDDEN, seed=1), rnd(HIDDEN, seed=4, dtype=torch.float32), k),
}


@pytest.mark.parametrize("block,result", [("prenorm", r) for r in RESULTS] + [("scaled", r) for r in RESULTS if r != "a bias"]
                         + [("gated", "a tensor"), ("gated", "a bias")])
def test_what_a_mixer_leaves_to_the_residual_is_taken_there_by_rows_too(block, result):
    """A sum, or a bias behind a gate, goes into the float32 residual unrounded: the same bits as in the whole block."""
    k = RowTwins()
    env = BuildEnv(k, torch.device("cpu"), torch.bfloat16, 64)
    parts = dict(mixer=Mixer(lambda: RESULTS[result](k)), mixer_norm=norm(env), feed_forward=Half(), feed_forward_norm=norm(env))
    if block == "gated":
        made = GatedPreNormBlock(mixer_gate=Gate(), feed_forward_gate=Gate(), **parts)
    else:
        made = PreNormBlock(residual_scale=0.4 if block == "scaled" else None, **parts)
    ctx, last = SimpleNamespace(kernels=k), norm(env)
    rows = torch.tensor([39, 3, 3, 17], dtype=torch.int32)
    start = rnd(TOKENS, HIDDEN, seed=5, dtype=torch.float32)
    whole, alone = ResidualStream(start.clone()), ResidualStream(start.clone())
    made.forward(whole, ctx, None)
    want = last.forward(whole, rows=rows)
    assert made.forward_rows(alone, ctx, None, rows)
    assert torch.equal(last.forward(alone), want)


@pytest.mark.parametrize("kind", [PreNormBlock, GatedPreNormBlock])
def test_a_block_whose_forward_is_wrapped_is_run_by_it(kind):
    """Somebody who put a forward of their own in place of a block's, by a class or on the block, sees every step."""
    k = RowTwins()
    env = BuildEnv(k, torch.device("cpu"), torch.bfloat16, 64)
    parts = dict(mixer=Mixer(lambda: rnd(TOKENS, HIDDEN, seed=1)), mixer_norm=norm(env), feed_forward=Half(), feed_forward_norm=norm(env))
    if kind is GatedPreNormBlock:
        parts.update(mixer_gate=Gate(), feed_forward_gate=Gate())
    rows, ctx = torch.tensor([3], dtype=torch.int32), SimpleNamespace(kernels=k)
    by_rows = lambda block: block.forward_rows(ResidualStream(rnd(TOKENS, HIDDEN, seed=5, dtype=torch.float32)), ctx, None, rows)
    assert by_rows(kind(**parts))
    wrapped = kind(**parts)
    wrapped.forward = lambda *args: kind.forward(wrapped, *args)
    assert not by_rows(wrapped)
    assert not by_rows(type("Other", (kind,), {"forward": lambda self, *args: kind.forward(self, *args)})(**parts))


class RowsMixer(Mixer):
    def forward(self, h, ctx, cache):
        rows = getattr(ctx, "only_rows", None)
        return self.result() if rows is None else ctx.kernels.take_rows(self.result(), rows)

    def gives_only_rows(self):
        return True


@pytest.mark.parametrize("kind,name", [(PreNormBlock, n) for n in ("mixer", "feed_forward", "feed_forward_norm")]
                         + [(GatedPreNormBlock, n) for n in ("mixer", "feed_forward", "feed_forward_norm", "mixer_gate", "feed_forward_gate")])
def test_a_part_that_somebody_wraps_is_still_run_for_all_tokens(kind, name):
    """Somebody who put a computation of their own in front of a part's, on the part, is handed every token's rows."""
    k = RowTwins()
    env = BuildEnv(k, torch.device("cpu"), torch.bfloat16, 64)
    parts = dict(mixer=RowsMixer(lambda: rnd(TOKENS, HIDDEN, seed=1)), mixer_norm=norm(env), feed_forward=Half(),
                 feed_forward_norm=norm(env))
    if kind is GatedPreNormBlock:
        parts.update(mixer_gate=Gate(), feed_forward_gate=Gate())
    made, ctx, seen = kind(**parts), SimpleNamespace(kernels=k), []
    method = "logits" if name.endswith("gate") else "forward"
    own = getattr(parts[name], method)
    setattr(parts[name], method, lambda *args, **more: seen.append(own(*args, **more)) or seen[-1])
    stream = ResidualStream(rnd(TOKENS, HIDDEN, seed=5, dtype=torch.float32))
    if not made.forward_rows(stream, ctx, None, torch.tensor([3], dtype=torch.int32)):
        made.forward(stream, ctx, None)
    assert [len(t) for t in seen] == [TOKENS]
