"""A model's last layer goes on with the rows alone that are read: the same logits, the same keys, values and states."""

import pytest
import torch

import famepel_models as fm
import lunerax_models as lx
import melerax_models as ml
import mogisun_models as mg
import tadinex_models as tx
from helpers import TINIES, random_tokens, rel_err, write_tiny_model
from simple_inference_amd import Engine, EngineConfig
from simple_inference_amd.engine import StepEntry
from simple_inference_amd.parts.attention import Attention
from simple_inference_amd.parts.block import GatedPreNormBlock, PreNormBlock
from simple_inference_amd.parts.model import DecoderModel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    at = lambda name: tmp_path_factory.mktemp("last_" + name)
    out = {"llama-" + n: write_tiny_model(at("llama_" + n), t, seed=51) for n, t in TINIES.items()}
    for label, M in (("mogisun", mg), ("tadinex", tx), ("famepel", fm), ("lunerax", lx), ("melerax", ml)):
        for name in M.CONFIGS:
            config = M.CONFIGS[name]
            out[f"{label}-{name}"] = M.write_model(at(f"{label}_{name}"), M.all_experts(config) if hasattr(M, "all_experts") else config,
                                                   seed=5)
    return out


def steps(folder, dtype):
    """(logits, keys, values and states, the last block, what its ``forward_rows`` said, the rows of each ``rows_alone``).  Portions of
    two prompts that want nothing; a step of a decoded token, a prompt's end, a whole prompt with several places and one with
    its last place; portions beside decoded tokens; decoded tokens of all of them."""
    engine = Engine.from_folder(folder, EngineConfig(device="cuda:0", dtype=dtype, max_seq_len=512, block_size=16, max_running=5,
                                                     chunk_tokens=512, eos_id=-1, use_graphs=False))
    vocab, out, said, alone = engine.model.vocab_size, [], [], []
    block, kernels = engine.model.layers[engine.model.order[-1]].block, engine.kernels
    if hasattr(block, "forward_rows"):
        rows_of, block.forward_rows = block.forward_rows, lambda *args: said.append(rows_of(*args)) or said[-1]
    rows_alone = kernels.rows_alone
    kernels.rows_alone = lambda *args: alone.append(len(args[0])) or rows_alone(*args)
    toks = lambda n, seed: random_tokens(vocab, n, seed=seed)
    for r in range(1, 5):
        engine.cache.admit(r, 400, 512)
    run = lambda entries: engine.runner.run(entries)
    try:
        assert run([StepEntry(1, toks(40, 1)), StepEntry(2, toks(23, 2))]) is None
        out.append(run([StepEntry(1, toks(1, 3), [0]), StepEntry(2, toks(170, 4), [169]), StepEntry(3, toks(33, 5), [32, 3, 7]),
                        StepEntry(4, toks(18, 6), [17])]).clone())
        assert run([StepEntry(4, toks(200, 7))]) is None
        out.append(run([StepEntry(1, toks(150, 8), [149]), StepEntry(4, toks(1, 9), [0])]).clone())
        out.append(run([StepEntry(2, toks(1, 15), [0]), StepEntry(3, toks(90, 16), [89]), StepEntry(4, toks(1, 17), []),
                        StepEntry(1, toks(60, 18), [59])]).clone())
        out.append(run([StepEntry(r, toks(1, 10 + r), [0]) for r in range(1, 5)]).clone())
    finally:
        kernels.rows_alone = rows_alone
    kept = [t for g in engine.cache.groups for t in (g.k, g.v)] + list(engine.cache.slots.tensors)
    return out, kept, block, said, alone


MODELS = ([f"llama-{n}" for n in TINIES] + [f"mogisun-{n}" for n in mg.CONFIGS] + [f"tadinex-{n}" for n in tx.CONFIGS]
          + [f"lunerax-{n}" for n in lx.CONFIGS] + [f"melerax-{n}" for n in ml.CONFIGS] + [f"famepel-{next(iter(fm.CONFIGS))}"])


@pytest.mark.parametrize("alone_from", [0, 10 ** 9])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", MODELS)
def test_the_rows_that_are_read_alone_give_the_same_logits(folders, name, dtype, alone_from, monkeypatch):
    """Keys, values and states have the same bits, and in float32, where a row's sums do not depend on the others, so have
    the logits; bfloat16: the few rows take another product and another attention kernel, which agree within rounding
    (the tolerance of the engine's tests).  Pre-norm blocks with a feed-forward and nothing behind it go by rows in the five
    steps of 32 tokens and more; others say that they do not, or are not asked (sandwich blocks)."""
    monkeypatch.setattr(Attention, "ALONE_FROM", alone_from)
    monkeypatch.setattr(Attention, "ALONE_BESIDE", alone_from)
    got, got_kept, block, said, alone = steps(folders[name], dtype)
    monkeypatch.setattr(DecoderModel, "_few_rows_read", staticmethod(lambda ctx: False))
    want, want_kept, _, none, _ = steps(folders[name], dtype)
    by_rows = (isinstance(block, (PreNormBlock, GatedPreNormBlock)) and block.feed_forward is not None
               and getattr(block, "token_input", None) is None)
    assert said == ([by_rows] * 5 if hasattr(block, "forward_rows") else []) and none == []
    plain = by_rows and type(block.mixer) is Attention and not block.mixer.row_form and not block.mixer.out_gate
    assert alone == ([2, 3] if plain and alone_from == 0 else [])
    for g, w in zip(got_kept, want_kept):
        assert torch.equal(g, w)
    for g, w in zip(got, want):
        assert torch.equal(g, w) if dtype == "float32" else rel_err(g, w) <= 2.5e-2
