"""GPU parity of generation from whole windows in one launch (csrc/window.hip).

Every shape family of the kernel (width, head width, windows of up to 32 and 64
rows, both connectivities, weights staged in LDS or not), the operator switches,
prompts shorter and longer than the context, and the vocabularies around the
sampler's one and four tokens a lane: the tokens against the oracle's sliding
window (src/gpt/gpu.rs:2006-2053), and the decode state the launch leaves.
"""
import numpy as np
import pytest

import grokking_abmod_amd as G
import oracle_lib as O
from conftest import assert_close
from trajectory import check_trajectory, largest_values

pytestmark = pytest.mark.gpu


def _last(model):
    return lambda window: model.logits(window, len(window), last_only=True)[0]


CASES = [
    # the command line's default model, and each width and head width
    dict(width=32, heads=4, context=32, vocab_size=28), dict(width=32, heads=2, context=1, vocab_size=5),
    dict(width=64, heads=8, context=7, vocab_size=64, connectivity=1), dict(width=64, heads=4, context=16),
    dict(width=64, heads=2, context=33, vocab_size=65), dict(width=128, heads=8, context=31, connectivity=1),
    dict(width=128, heads=4, context=32, vocab_size=256), dict(width=128, heads=2, context=64),
    dict(width=32, heads=4, context=64, connectivity=1), dict(width=64, heads=4, context=50, connectivity=1),
    dict(width=128, heads=4, context=40, connectivity=1), dict(width=128, heads=2, context=17, layers=1),
    # weights past a CU's LDS, odd and one-layer stacks, operators off
    dict(width=128, heads=4, context=20, layers=12, vocab_size=99), dict(width=64, heads=4, context=20, layers=3,
         attention_mesh_depth=1, ffn_mesh_depth=9, connectivity=1),
    dict(width=32, heads=4, context=24, rope=0), dict(width=64, heads=8, context=24, qk_norm=0),
    dict(width=32, heads=2, context=24, xsa=0), dict(width=32, heads=4, context=24, embedding=1),
]


@pytest.mark.parametrize("wide", ["0", "1"])  # mesh values times log2(e), in their own units
@pytest.mark.parametrize("temperature", [0.0, 0.7])
@pytest.mark.parametrize("cfg", CASES, ids=["-".join(f"{k[:3]}{v}" for k, v in c.items()) for c in CASES])
def test_window_generation_matches_the_oracle(cfg, temperature, wide, monkeypatch):
    monkeypatch.setenv("MG_FORCE_WIDE", wide)
    kw = dict(dict(vocab_size=40, layers=2), **cfg)
    g, o = G.GptConfig(**kw), O.config(**kw)
    params = O.initialize(o, 7)
    n = kw["context"] + 3 if kw["context"] in (7, 31) else min(5, kw["context"])
    prompts = G.random_prompts(kw["vocab_size"], 3, n, 7)
    count = min(2 * kw["context"] + 10, 80)
    with G.MeshGpt(0, g, 7, max_batch=3) as model:
        got = model.generate_tokens(prompts, count, temperature, 7)
        last = model.last_logits(3)
        for b in (0, 2):
            check_trajectory(o, params, prompts[b], got[b], temperature, 7 + b, _last(model), cached=False)
        window = got[:, :-1][:, -kw["context"]:]
        assert_close(last, model.logits(window.reshape(-1), window.shape[1], last_only=True), what="last logits")
        alone = model.generate_tokens(prompts[:1], count, temperature, 7)
        assert np.array_equal(alone[0], got[0])


def test_decode_continues_a_window_generation(monkeypatch):
    """A generation that ends inside the context leaves the cache, lengths and
    sampler states that further decode steps need."""
    cfg = G.GptConfig(vocab_size=28, context=32, width=32, heads=4, layers=2)
    prompts = G.random_prompts(28, 2, 5, 7)
    with G.MeshGpt(0, cfg, 7, max_batch=2) as model:
        model.prefill(prompts, 0.7, 7, reserve=40)
        whole = model.generate_tokens(prompts, 20, 0.7, 7)
        model.generate_tokens(prompts, 8, 0.7, 7)
        model.decode(12)
        assert np.array_equal(model.read_tokens(2), whole)
    monkeypatch.setenv("MG_DISABLE_WINDOW", "1")
    with G.MeshGpt(0, cfg, 7, max_batch=2) as model:
        assert np.array_equal(model.generate_tokens(prompts, 20, 0.7, 7), whole)


@pytest.mark.parametrize("temperature", [0.0, 0.7])
@pytest.mark.parametrize("count", [20, 60])
@pytest.mark.parametrize("cfg", [dict(width=32, heads=4, context=32), dict(width=128, heads=2, context=40)],
                         ids=["W32", "W128"])
def test_a_generation_in_several_launches(cfg, count, temperature, monkeypatch):
    """Launches of 7 tokens give one launch's tokens, logits and state, inside the
    context (from which decode goes on) and past it."""
    prompts = G.random_prompts(40, 3, 5, 7)
    got = []
    for steps in ("0", "7"):
        monkeypatch.setenv("MG_WINDOW_STEPS", steps)
        monkeypatch.setenv("MG_DISABLE_PERSISTENT", "1")
        with G.MeshGpt(0, G.GptConfig(vocab_size=40, layers=2, **cfg), 7, max_batch=3) as model:
            model.prefill(prompts, temperature, 7, reserve=70)
            tokens = model.generate_tokens(prompts, count, temperature, 7)
            last = model.last_logits(3)
            if count == 20:
                model.decode(6)
            got.append((tokens, last, model.read_tokens(3), model.last_logits(3)))
    assert all(np.array_equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("cfg,count", [(dict(width=32, heads=4, context=32), 40),
                                       (dict(width=128, heads=4, context=64, attention_mesh_depth=9), 75)],
                         ids=["windows", "decode-then-windows"])
def test_more_sequences_than_workgroups_run_at_once(cfg, count):
    """A sequence's tokens are its own in a batch that takes three rounds, from
    windows alone and from the cached decode up to the context."""
    kw = dict(vocab_size=40, layers=2, **cfg)
    g, o = G.GptConfig(**kw), O.config(**kw)
    params = O.initialize(o, 7)
    prompts = G.random_prompts(40, 600, 5, 7)
    with G.MeshGpt(0, g, 7, max_batch=600) as model:
        got = model.generate_tokens(prompts, count, 0.7, 7)
        for b in (0, 255, 256, 599):
            check_trajectory(o, params, prompts[b], got[b], 0.7, 7 + b, _last(model), cached=False)


@pytest.mark.parametrize("W,H", [(32, 4), (64, 4), (128, 4)])
def test_a_mesh_may_reach_the_largest_values(W, H):
    """As the register-tile kernels' test of the same name: windows past the context."""
    kw = dict(vocab_size=16, context=20, width=W, heads=H, layers=1, attention_mesh_depth=2, ffn_mesh_depth=2,
              embedding=1)
    o = O.config(**kw)
    params = O.initialize(o, 7)
    largest_values(params, W, O.group_offsets(o)[3])
    prompts = G.random_prompts(16, 2, 21, 7)
    with G.MeshGpt(0, G.GptConfig(**kw), 7, max_batch=2) as model:
        model.set_parameters(params)
        got = model.generate_tokens(prompts, 6, 0.0, 7)
        last = model.last_logits(2)
    ref = [O.logits(o, params, got[b, -21:-1], 20)[-1] for b in range(2)]
    assert_close(last, ref, what="last logits")


def test_window_generation_reports_nonfinite_logits():
    cfg = dict(vocab_size=28, context=16, width=32, heads=4, layers=1)
    o = O.config(**cfg)
    params = O.initialize(o, 7)
    start = O.group_offsets(o)[3]
    params[start:start + 2 * 32 * 4] = 3e38
    with G.MeshGpt(0, G.GptConfig(**cfg), 7) as model:
        model.set_parameters(params)
        with pytest.raises(G.MeshGptError) as err:
            model.generate_tokens(G.random_prompts(28, 1, 4, 7), 30, 0.7, 7)
        assert err.value.status == G.MG_NONFINITE
