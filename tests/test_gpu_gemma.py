"""Gemma-2 text encoder on the GPU (sana_gemma_* C ABI) against the oracle.

The oracle (oracle/gemma_oracle.py) restates the Gemma-2 forward that the
reference runs through llama.cpp and is pinned against transformers'
Gemma2Model (tests/test_oracle_gemma.py).  The HIP path (fp16 GEMM operands,
fp32 accumulation, residual, norms and softmax) is held to a relative L2 of
2e-3 on the hidden states, the per-forward bar of the DiT.
"""
import os
import sys

import numpy as np
import pytest

from conftest import rel_l2
from gguf_writer import GGML_F16, write_gguf

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import gemma_oracle as G  # noqa: E402

pytestmark = pytest.mark.gpu
TOL = 2e-3

CONFIGS = {
    "gqa_window": dict(vocab=300, hidden=256, layers=2, heads=4, kv_heads=2, head_dim=64, ffn=512, sliding_window=8,
                       rms_eps=1e-6, rope_theta=10000.0, softcap=50.0, query_scale=1 / 8),
    "mqa_softcap": dict(vocab=200, hidden=192, layers=3, heads=2, kv_heads=1, head_dim=128, ffn=320,
                        sliding_window=0, rms_eps=1e-6, rope_theta=10000.0, softcap=2.0, query_scale=128 ** -0.5),
    # the Gemma-2 2B layer shapes, two layers and a small vocabulary
    "gemma2_2b_2layers": dict(G.GEMMA2_2B, vocab=1024, layers=2),
}


def build(cfg, seed=5, scale=0.05):
    import sana_dit
    w = G.random_weights(cfg, seed=seed, scale=scale)
    dev = sana_dit.Gemma(cfg)
    for name, arr in w.items():
        dev.set_weight(name, arr)
    dev.check_weights()
    return w, dev


@pytest.mark.parametrize("name,T", [("gqa_window", 37), ("gqa_window", 64), ("mqa_softcap", 19),
                                    ("gemma2_2b_2layers", 438)])
def test_encode_vs_oracle(name, T):
    cfg = CONFIGS[name]
    w, dev = build(cfg)
    try:
        tokens = np.random.default_rng(T).integers(0, cfg["vocab"], size=T)
        print(f"{name} T={T}: oracle forward on the host ...", flush=True)
        ref = G.forward(w, cfg, tokens)
        got = dev.encode(tokens)
        err = rel_l2(got, ref)
        print(f"{name} T={T}: hidden rel_l2 {err:.3e}")
        assert got.shape == (T, cfg["hidden"])
        assert np.isfinite(got).all()
        assert err < TOL
        assert np.array_equal(dev.encode(tokens), got)
    finally:
        dev.close()


@pytest.mark.parametrize("name,Ta,Tb", [("gqa_window", 37, 64), ("gqa_window", 20, 20), ("mqa_softcap", 5, 19),
                                         ("gemma2_2b_2layers", 438, 300), ("gemma2_2b_2layers", 150, 100)])
def test_encode_pair_equals_two_encodes(name, Ta, Tb):
    """Both sequences in one pass share the per-token kernels; every row must
    equal the separate encode of its own sequence bit for bit (attention stays
    within a sequence, RoPE positions restart at 0), and match the oracle."""
    cfg = CONFIGS[name]
    w, dev = build(cfg)
    try:
        rng = np.random.default_rng(Ta * 1000 + Tb)
        a = rng.integers(0, cfg["vocab"], size=Ta)
        b = rng.integers(0, cfg["vocab"], size=Tb)
        ha, hb = dev.encode_pair(a, b)
        assert np.array_equal(ha, dev.encode(a))
        assert np.array_equal(hb, dev.encode(b))
        assert rel_l2(hb, G.forward(w, cfg, b)) < TOL
        ha2, hb2 = dev.encode_pair(a, b)   # graph replay
        assert np.array_equal(ha2, ha) and np.array_equal(hb2, hb)
        hb3, ha3 = dev.encode_pair(b, a)   # the other order: its own graph
        assert np.array_equal(ha3, ha) and np.array_equal(hb3, hb)
    finally:
        dev.close()


def test_graph_replays_and_weight_reload():
    """The encoder runs as one cached graph per token count: interleaved
    lengths replay their own graphs with new tokens, and a weight set after a
    capture (which drops the graphs) is used by the next encode."""
    cfg = CONFIGS["gqa_window"]
    w, dev = build(cfg)
    try:
        rng = np.random.default_rng(11)
        for T in (23, 40, 23, 40, 23):
            tokens = rng.integers(0, cfg["vocab"], size=T)
            assert rel_l2(dev.encode(tokens), G.forward(w, cfg, tokens)) < TOL
        name = "blk.1.ffn_down.weight"
        w[name] = (w[name] * -1.5).astype(np.float32)
        dev.set_weight(name, w[name])
        tokens = rng.integers(0, cfg["vocab"], size=23)
        assert rel_l2(dev.encode(tokens), G.forward(w, cfg, tokens)) < TOL
    finally:
        dev.close()


def test_prefix_positions_are_causal():
    """Causal attention: the hidden states of a prefix do not depend on the
    tokens after it (the reference pads prompts at the end for this reason)."""
    cfg = CONFIGS["gqa_window"]
    w, dev = build(cfg)
    try:
        tokens = np.random.default_rng(3).integers(0, cfg["vocab"], size=40)
        a = dev.encode(tokens)
        b = dev.encode(np.concatenate([tokens[:25], np.zeros(15, np.int64)]))
        assert rel_l2(b[:25], a[:25]) < 1e-6
    finally:
        dev.close()


def test_load_gguf(tmp_path):
    cfg = CONFIGS["gqa_window"]
    w = G.random_weights(cfg, seed=5, scale=0.05)
    path = str(tmp_path / "gemma.gguf")
    write_gguf(path, w, ggml_type=GGML_F16)
    import sana_dit
    dev = sana_dit.Gemma(cfg)
    try:
        dev.load_gguf(path)
        dev.check_weights()
        tokens = np.random.default_rng(9).integers(0, cfg["vocab"], size=21)
        w16 = {k: v.astype(np.float16).astype(np.float32) for k, v in w.items()}
        assert rel_l2(dev.encode(tokens), G.forward(w16, cfg, tokens)) < TOL
    finally:
        dev.close()


def test_rejects_bad_input():
    import sana_dit
    with pytest.raises(sana_dit.SanaError):
        sana_dit.Gemma(dict(CONFIGS["gqa_window"], heads=3))       # heads % kv_heads
    with pytest.raises(sana_dit.SanaError):
        sana_dit.Gemma(dict(CONFIGS["gqa_window"], head_dim=48))   # head dim % 64
    cfg = CONFIGS["gqa_window"]
    w, dev = build(cfg)
    try:
        with pytest.raises(sana_dit.SanaError) as e:
            dev.encode(np.array([1, cfg["vocab"]]))
        assert e.value.code == sana_dit.SANA_ERR_INVALID_ARGUMENT
        with pytest.raises(sana_dit.SanaError) as e:
            dev.encode_pair(np.array([1, 2]), np.array([3, -1]))
        assert e.value.code == sana_dit.SANA_ERR_INVALID_ARGUMENT
        with pytest.raises(sana_dit.SanaError) as e:
            dev.encode_pair(np.array([1, 2]), np.array([], np.int64))
        assert e.value.code == sana_dit.SANA_ERR_INVALID_ARGUMENT
        with pytest.raises(sana_dit.SanaError) as e:
            dev.set_weight("blk.0.attn_q.weight", np.zeros((3, 3), np.float32))
        assert e.value.code == sana_dit.SANA_ERR_SHAPE
    finally:
        dev.close()


EDGE = dict(vocab=50, hidden=192, layers=2, heads=4, kv_heads=2, head_dim=64, ffn=128, sliding_window=0, rms_eps=1e-6,
            rope_theta=10000.0, softcap=50.0, query_scale=1 / 8)


@pytest.mark.parametrize("d", [64, 128, 192, 256])
@pytest.mark.parametrize("T,window", [(1, 0), (31, 0), (32, 5), (33, 40), (65, 64), (97, 33), (130, 1), (161, 0),
                                      (300, 100)])
def test_attention_edges_vs_oracle(d, T, window):
    """Query and key blocks of 32, windows that start inside, at and outside a
    block, single rows; head dim 192 takes the product path."""
    cfg = dict(EDGE, head_dim=d, sliding_window=window, query_scale=d ** -0.5)
    w, dev = build(cfg, scale=0.1)
    try:
        tokens = np.random.default_rng(T + d).integers(0, cfg["vocab"], size=T)
        got = dev.encode(tokens)
        assert rel_l2(got, G.forward(w, cfg, tokens)) < TOL
        other = np.random.default_rng(T).integers(0, cfg["vocab"], size=max(1, T // 2))
        a, b = dev.encode_pair(other, tokens)
        assert np.array_equal(b, got) and np.array_equal(a, dev.encode(other))
    finally:
        dev.close()


@pytest.mark.parametrize("hidden,ffn", [(64, 64), (1088, 128), (2112, 8192), (3136, 64), (4096, 64)])
def test_norm_widths_vs_oracle(hidden, ffn):
    """Row widths of one to four 1024-channel runs, one, two and four split-K partials."""
    cfg = dict(EDGE, hidden=hidden, ffn=ffn, heads=16 if ffn > 64 else 4)
    w, dev = build(cfg, scale=0.03)
    try:
        tokens = np.random.default_rng(hidden).integers(0, cfg["vocab"], size=21)
        assert rel_l2(dev.encode(tokens), G.forward(w, cfg, tokens)) < TOL
    finally:
        dev.close()


@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("cap", [0.02, 0.7, 1e19, 1e25])
def test_softcap_ranges_vs_oracle(d, cap):
    """Scores far past the soft cap, around it (both branches of tanh) and far below
    it; the last cap takes the product path."""
    cfg = dict(EDGE, head_dim=d, softcap=cap, query_scale=d ** -0.5)
    w, dev = build(cfg, scale=0.1)
    try:
        tokens = np.random.default_rng(d).integers(0, cfg["vocab"], size=97)
        assert rel_l2(dev.encode(tokens), G.forward(w, cfg, tokens)) < TOL
    finally:
        dev.close()
