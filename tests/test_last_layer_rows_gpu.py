"""A model's last layer goes on with the rows alone that are read: the same logits, the same keys, values and states."""

import pytest
import torch

import famepel_models as fm
import mogisun_models as mg
import tadinex_models as tx
from helpers import TINIES, random_tokens, rel_err, write_tiny_model
from simple_inference_amd import Engine, EngineConfig
from simple_inference_amd.engine import StepEntry
from simple_inference_amd.parts.model import DecoderModel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    at = lambda name: tmp_path_factory.mktemp("last_" + name)
    out = {"llama-" + n: write_tiny_model(at("llama_" + n), t, seed=51) for n, t in TINIES.items()}
    for label, M in (("mogisun", mg), ("tadinex", tx), ("famepel", fm)):
        for name in M.CONFIGS:
            out[f"{label}-{name}"] = M.write_model(at(f"{label}_{name}"), M.all_experts(M.CONFIGS[name]), seed=5)
    return out


def steps(folder, dtype):
    """Logits of: portions of two prompts that want nothing; a step of a decoded token, a prompt's end, a whole prompt with
    several places and one with its last place; decoded tokens of all of them."""
    engine = Engine.from_folder(folder, EngineConfig(device="cuda:0", dtype=dtype, max_seq_len=512, block_size=16, max_running=5,
                                                     chunk_tokens=512, eos_id=-1, use_graphs=False))
    vocab, out = engine.model.vocab_size, []
    toks = lambda n, seed: random_tokens(vocab, n, seed=seed)
    for r in range(1, 5):
        engine.cache.admit(r, 400, 512)
    run = lambda entries: engine.runner.run(entries)
    assert run([StepEntry(1, toks(40, 1)), StepEntry(2, toks(23, 2))]) is None
    out.append(run([StepEntry(1, toks(1, 3), [0]), StepEntry(2, toks(170, 4), [169]), StepEntry(3, toks(33, 5), [32, 3, 7]),
                    StepEntry(4, toks(18, 6), [17])]).clone())
    assert run([StepEntry(4, toks(200, 7))]) is None
    out.append(run([StepEntry(1, toks(150, 8), [149]), StepEntry(4, toks(1, 9), [0])]).clone())
    out.append(run([StepEntry(r, toks(1, 10 + r), [0]) for r in range(1, 5)]).clone())
    return out


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["llama-a", "llama-b"] + [f"mogisun-{n}" for n in mg.CONFIGS] + [f"tadinex-{n}" for n in tx.CONFIGS]
                         + [f"famepel-{n}" for n in fm.CONFIGS])
def test_the_rows_that_are_read_alone_give_the_same_logits(folders, name, dtype, monkeypatch):
    """float32: a row's sums do not depend on the others, so the logits are equal up to the order of a head's norm (2e-6 of
    their size); bfloat16: the few rows take another product and another attention kernel, which agree within rounding
    (the tolerance of the engine's tests)."""
    got = steps(folders[name], dtype)
    monkeypatch.setattr(DecoderModel, "_few_rows_read", staticmethod(lambda ctx: False))
    want = steps(folders[name], dtype)
    for g, w in zip(got, want):
        assert rel_err(g, w) <= (2e-6 if dtype == "float32" else 2.5e-2)
