"""The sampled pick over more than 64 kept entries: the workgroup's parallel sums where they are certain
to give the pick of the sums in index order, and the fold in order elsewhere, against the C oracle's
sample_next (double sums in index order) on the same logits and draws. Whole numbers: exact."""
import ctypes

import numpy as np
import pytest

import kd

pytestmark = pytest.mark.gpu


def engine(kdb, vocab, embedding, positions=24, dim=8):
    rng = np.random.default_rng(vocab)
    g = kd.Gpt(kdb, vocab, positions, 1, 2, dim)
    for name, shape in kd.gpt2_parameter_shapes(vocab, positions, 1, dim):
        w = rng.normal(0, 0.5, shape)
        if name == "token_embedding.weight":
            w = embedding(rng, shape)
        elif ".ln" in name or name.startswith("ln"):
            w = np.full(shape, float(name.endswith("weight")))
        g.load(name, w.astype(np.float32))
    return g


def oracle_pick(oracle, logits, temperature, top_k, u):
    token = ctypes.c_int64()
    assert oracle.oracle_sample_topk(logits.ctypes.data_as(ctypes.c_void_p), logits.size, temperature, top_k, u,
                                     ctypes.byref(token)) == 0, oracle.oracle_last_error()
    return token.value


def check(oracle, g, prompt, draws, temperature, top_k):
    g.set_sampling(temperature, top_k)
    g.set_uniforms(draws)
    g.prefill(prompt)
    picks = [g.sequence()[-1]]
    assert picks[0] == oracle_pick(oracle, g.logits(), temperature, top_k, draws[0])
    for i, u in enumerate(draws[1:]):
        picks.extend(g.decode(1))
        assert picks[-1] == oracle_pick(oracle, g.logits(), temperature, top_k, u), i
    assert g.draws_used() == len(draws)
    return picks


# shares of 4 entries a lane (few lanes hold any) to the 64 of the largest vocabulary, kept lists in LDS
# (k up to 4096) and in memory, a flat and a peaked distribution
@pytest.mark.parametrize("vocab,temperature,top_k",
                         [(70, 1.0, 0), (1025, 1.0, 0), (4097, 0.7, 0), (50257, 1.0, 0), (50257, 0.05, 0), (65536, 1.0, 65536),
                          (200, 1.0, 65), (3000, 0.9, 1000), (50257, 1.0, 4096), (50257, 1.0, 6000)])
def test_picks_over_many_entries(kdb, oracle, vocab, temperature, top_k):
    g = engine(kdb, vocab, lambda rng, shape: rng.normal(0, 0.5, shape))
    rng = np.random.default_rng(top_k + 1)
    draws = np.concatenate([rng.uniform(0, 1, 12), [0.0, np.nextafter(1.0, 0.0), 1e-12, 1 - 1e-12]])
    picks = check(oracle, g, rng.integers(0, vocab, 6), draws, temperature, top_k)
    assert len(set(picks)) > 3


@pytest.mark.parametrize("vocab", [96, 1000, 50257])
def test_draws_on_the_boundaries_of_equal_weights(kdb, oracle, vocab):
    """Every logit alike, and draws at multiples of 1 / vocab: the point lies on a running sum, so that the
    pick hangs on the roundings of the sums in order."""
    g = engine(kdb, vocab, lambda rng, shape: np.zeros(shape))
    steps = np.linspace(1, vocab - 1, 14).astype(np.int64)
    check(oracle, g, np.zeros(4, np.int64), steps / vocab, 1.0, 0)
