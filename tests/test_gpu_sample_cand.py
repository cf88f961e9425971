"""The sampler's top-k candidates (k <= 256, 8192 logits and more) against the
oracle's sample_token: the edges of that route, ties that overflow its cut,
workgroups with fewer than k finite logits, and the step graph's replays."""
import numpy as np
import pytest

from test_gpu_sample import check, device_draws, oracle_draws  # noqa: F401

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("V", [8191, 8192, 8193, 32000, 128256, 262144])
def test_edges(hip, orc, V):
    print(f"[case] candidates V={V}", flush=True)
    x = (3.0 * np.random.default_rng(V).standard_normal(V)).astype(F)
    for i, cfg in enumerate([(0.8, 40, 0.95), (1.0, 1, 1.0), (1.3, 256, 0.9), (1.0, 255, 1.0), (1.0, 257, 1.0), (0.7, 2, 0.5)]):
        check(hip, orc, x, cfg, seed=50 + i, n=4)


def test_ties_and_nonfinite(hip, orc):
    print("[case] candidates: ties, -inf, few finite, NaN, +inf", flush=True)
    rng = np.random.default_rng(4)
    V = 20000
    ties = rng.integers(-3, 4, V).astype(F)  # thousands of equal values at the cut
    flat = np.full(V, 0.5, F)
    few = np.full(V, -np.inf, F)
    few[rng.choice(V, 30, replace=False)] = rng.standard_normal(30)
    some = np.full(V, -np.inf, F)
    some[6000:6300] = rng.standard_normal(300)
    wide = (rng.standard_normal(V) * 1e30).astype(F)
    neg = (-np.abs(rng.standard_normal(V)) - 1000).astype(F)
    nan = rng.standard_normal(V).astype(F)
    nan[777] = np.nan
    inf = rng.standard_normal(V).astype(F)
    inf[19999] = np.inf
    for j, x in enumerate((ties, flat, few, some, wide, neg, nan, inf)):
        for i, cfg in enumerate([(1.0, 40, 1.0), (0.8, 200, 0.6), (1.0, 1, 1.0), (0.5, 31, 0.9)]):
            print(f"[case] input {j} cfg {cfg}", flush=True)
            check(hip, orc, x, cfg, seed=70 + i, n=3)


def test_graph_replays(hip, orc):
    """Sampled generate (the step graph): each token is the oracle's draw from that step's logits."""
    cfg = hip.LlamaConfig(32000, 64, 128, 1, 4, 4, max_seq_len=64, tie_word_embeddings=False)
    m = hip.LlamaModel.new_random(cfg, 1, init_on_device=True)
    rng = hip.Rng.with_seed(9)
    sc = hip.SamplingConfig(temperature=0.9, top_k=40, top_p=0.95, max_tokens=24)
    toks, lg = m.generate([5, 6, 7], sc, rng, want_logits=True)
    st = 9
    for t, row in zip(toks, lg):
        want, st = orc.sample_token(np.asarray(row, F), 0.9, 40, 0.95, st)
        assert int(t) == want
    assert rng.state == st
    m.free()
