"""Spans of 2 to 7 tokens run token by token whatever came before them, and key
shares of batched spans deep in the context."""
import os

import numpy as np
import pytest

from chatnet_amd import QWEN2_0_5B, HipLlamaModel, _native, synth
from gpu_util import announce, run_with_failing_malloc
from test_gpu_model import LOGIT_TOL, SPAN_SMALL, span_case

pytestmark = pytest.mark.gpu


def per_token(cfg, ck, toks, pos=0, first=None):
    os.environ["CHATNET_SPAN_BATCH"] = "0"
    try:
        with HipLlamaModel(cfg, ck) as m:
            if first is not None:
                m.forward(first, 0)
            return m.forward(toks, pos).copy()
    finally:
        del os.environ["CHATNET_SPAN_BATCH"]


@pytest.mark.parametrize("n,n_next", [(3, 7), (7, 3), (40, 5)])
@pytest.mark.parametrize("mix", ["q4_0", "q8_0"])
def test_short_spans_match_oracle(mix, n, n_next):
    announce(f"short spans {mix}, {n} + {n_next} tokens")
    span_case(SPAN_SMALL, 61, n, n_next=n_next, mix=mix)


def test_short_span_of_a_qwen2_layer():
    announce("short span: qwen2-0.5b layer, 6 + 3 tokens")
    cfg = QWEN2_0_5B.replace(n_layers=1, vocab_size=2048, context_length=64)
    ck = synth.llama_checkpoint(cfg, seed=62, mix="q8_0", with_output=False, embedding=8)
    span_case(cfg, 62, 6, n_next=3, ck=ck)


@pytest.mark.parametrize("mix,n", [("q4_0", 2), ("q4_0", 3), ("q4_k", 7), ("q6_k", 5), ("legacy_blocks", 7), ("f16", 6), ("f32", 3), ("iq_a", 4)])
@pytest.mark.parametrize("before", [0, 12])
def test_short_spans_are_the_single_tokens(mix, n, before):
    """The bits of one call per token: fp32 attention and activations, whether or
    not a longer span has packed matrices before."""
    announce(f"short span {mix}, {before} + {n} tokens")
    ck = synth.llama_checkpoint(SPAN_SMALL, seed=63, mix=mix)
    toks = synth.tokens(63, "prompt", before + n, SPAN_SMALL.vocab_size)
    with HipLlamaModel(SPAN_SMALL, ck) as m:
        if before:
            m.forward(toks[:before], 0)
        g = m.forward(toks[before:], before).copy()
    with HipLlamaModel(SPAN_SMALL, ck) as m:
        if before:
            m.forward(toks[:before], 0)
        for i in range(before, before + n):
            h = m.forward(toks[i:i + 1], i)
        assert np.array_equal(g, h)


def test_short_span_with_activations_past_fp16():
    """SwiGLU outputs past 65504 (norm weights of 3000) stay finite, the single
    tokens' bits."""
    announce("short span, activations past fp16")
    ck = synth.llama_checkpoint(SPAN_SMALL, seed=66, mix="q4_0")
    t = ck["blk.0.ffn_norm.weight"]
    ck["blk.0.ffn_norm.weight"] = synth.SynthTensor(t.type, t.dims, (t.data.view(np.float32) * 3000).view(np.uint8))
    toks = synth.tokens(66, "prompt", 5, SPAN_SMALL.vocab_size)
    with HipLlamaModel(SPAN_SMALL, ck) as m:
        g = m.forward(toks, 0).copy()
    with HipLlamaModel(SPAN_SMALL, ck) as m:
        for i in range(5):
            h = m.forward(toks[i:i + 1], i)
        assert np.all(np.isfinite(g)) and np.array_equal(g, h)


# Keys shared out over workgroups: both head sizes and cache types, groups of 1, 2
# and 7 heads, two shares to sixteen, a share past a token's own keys.  The token by
# token side deals its blocks out to 4- and 8-wave workgroups (8 for all but 4/4).
@pytest.mark.parametrize("heads,kv,hd,f16", [(14, 2, 64, False), (4, 4, 64, True), (4, 2, 128, False), (2, 1, 128, True)])
@pytest.mark.parametrize("pos,n", [(377, 8), (250, 10), (630, 100), (2030, 12)])
def test_spans_deep_in_the_context_share_their_keys(heads, kv, hd, f16, pos, n):
    announce(f"shared keys: {heads}/{kv} heads of {hd}, f16 cache {f16}, {n} tokens at {pos}")
    cfg = SPAN_SMALL.replace(n_layers=2, dim=heads * hd, hidden_dim=512, n_heads=heads, n_kv_heads=kv, head_dim=hd,
                             vocab_size=512, context_length=2048, kv_dtype=_native.KV_F16 if f16 else _native.KV_F32)
    ck = synth.llama_checkpoint(cfg, seed=65, mix="q4_0")
    toks = synth.tokens(65, "prompt", pos + n, cfg.vocab_size)
    with HipLlamaModel(cfg, ck) as m:
        m.forward(toks[:pos], 0)
        g = m.forward(toks[pos:], pos).copy()
    h = per_token(cfg, ck, toks[pos:], pos, toks[:pos])
    # each schedule's bound against the oracle, twice that for an fp16 cache
    assert float(np.max(np.abs(g - h))) <= 2 * LOGIT_TOL * (2 if f16 else 1)


# The O projection merges the splits' partials: from fp32 records (Q4_1, IQ4_XS),
# packed units (IQ3_S), F16 and F32 rows.  (The digit types' staging drops a NaN.)
@pytest.mark.parametrize("seq", [20, 300, 1000])
@pytest.mark.parametrize("mix", ["legacy_blocks", "iq_a", "iq_b", "f16", "f32"])
def test_a_nan_key_reaches_the_logits_from_any_split(mix, seq):
    """A token whose embedding is NaN leaves a NaN key and value at its position;
    whichever split of the decode attention holds it, later logits are NaN."""
    announce(f"NaN key, {mix}, {seq} tokens")
    cfg = SPAN_SMALL.replace(n_layers=1)
    ck = synth.llama_checkpoint(cfg, seed=67, mix=mix)
    emb = ck["token_embd.weight"]
    rows = emb.data.view(np.float32).reshape(cfg.vocab_size, cfg.dim).copy()
    bad = 7
    rows[bad] = np.nan
    ck["token_embd.weight"] = synth.SynthTensor(emb.type, emb.dims, rows.reshape(-1).view(np.uint8))
    toks = synth.tokens(67, "prompt", seq, cfg.vocab_size)
    toks[toks == bad] = bad + 1
    for at in {0, 9, seq // 2, seq - 2}:
        t = toks.copy()
        t[at] = bad
        with HipLlamaModel(cfg, ck) as m:
            m.forward(t[:-1], 0)
            assert np.all(np.isnan(m.forward(t[-1:], seq - 1))), at


SHARED_KEYS_WITHOUT_MEMORY = """
import os
import numpy as np
from chatnet_amd import HipLlamaModel, TINY_TEST, synth
cfg = TINY_TEST.replace(n_layers=2, dim=256, hidden_dim=512, n_heads=2, n_kv_heads=1, head_dim=128, context_length=2048)
ck = synth.llama_checkpoint(cfg, seed=68, mix="q4_0")
toks = synth.tokens(68, "prompt", 1512, cfg.vocab_size)
def run(limit):
    print("[gpu-case] shared keys, allocation limit", limit, flush=True)
    with HipLlamaModel(cfg, ck) as m:
        m.forward(toks[:12], 0)  # the span buffers and the GEMMs' partials
        os.environ["CHATNET_SPAN_BATCH"] = "0"
        m.forward(toks[12:1500], 12)
        del os.environ["CHATNET_SPAN_BATCH"]
        malloc_limit(limit)
        g = m.forward(toks[1500:], 1500).copy()
        malloc_limit(2 ** 62)
        return g
a, b = run(2 ** 62), run(1024)
assert np.all(np.isfinite(b)) and np.max(np.abs(a - b)) <= 1e-4, np.max(np.abs(a - b))
assert not np.array_equal(a, b)  # one share a row sums in another order
"""


def test_spans_without_memory_for_key_shares(tmp_path):
    """A span whose keys would be shared runs without shares where their partial
    results have no memory."""
    run_with_failing_malloc(tmp_path, SHARED_KEYS_WITHOUT_MEMORY)
