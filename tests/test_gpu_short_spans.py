"""Spans of 3 to 7 tokens: batched for models of the 19-bit types (Q4_0, Q8_0,
Q3_K .. Q6_K) when no matrix would have to be packed for them, token by token
otherwise, both against the oracle."""
import os

import numpy as np
import pytest

from chatnet_amd import QWEN2_0_5B, HipLlamaModel, synth
from gpu_util import announce
from test_gpu_model import SPAN_SMALL, span_case

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
def test_short_spans_run_batched_and_match_oracle(mix, n, n_next):
    announce(f"short spans {mix}, {n} + {n_next} tokens")
    span_case(SPAN_SMALL, 61, n, n_next=n_next, mix=mix, check_batched=True)


def test_short_span_of_a_qwen2_layer():
    announce("short span: qwen2-0.5b layer, 6 + 3 tokens")
    cfg = QWEN2_0_5B.replace(n_layers=1, vocab_size=2048, context_length=64)
    ck = synth.llama_checkpoint(cfg, seed=62, mix="q8_0", with_output=False, embedding=8)
    span_case(cfg, 62, 6, n_next=3, ck=ck, check_batched=True)


@pytest.mark.parametrize("mix,n", [("q4_0", 2), ("q6_k", 5), ("legacy_blocks", 7), ("f16", 6), ("f32", 3), ("iq_a", 4)])
def test_short_spans_that_stay_token_by_token(mix, n):
    """Two tokens, a type read as packed units with none made yet (Q6_K), float and
    finer types: the same bits as the token by token schedule."""
    announce(f"short span {mix}, {n} tokens, token by token")
    ck = synth.llama_checkpoint(SPAN_SMALL, seed=63, mix=mix)
    toks = synth.tokens(63, "prompt", n, SPAN_SMALL.vocab_size)
    with HipLlamaModel(SPAN_SMALL, ck) as m:
        g = m.forward(toks, 0).copy()
    assert np.array_equal(g, per_token(SPAN_SMALL, ck, toks))


def test_short_span_after_a_long_one_uses_the_packs():
    """Q6_K matrices packed by a 12-token span serve the 4-token span after it."""
    announce("short span after a packed one, q6_k 12 + 4")
    ck = synth.llama_checkpoint(SPAN_SMALL, seed=64, mix="q6_k")
    toks = synth.tokens(64, "prompt", 16, SPAN_SMALL.vocab_size)
    with HipLlamaModel(SPAN_SMALL, ck) as m:
        m.forward(toks[:12], 0)
        g = m.forward(toks[12:], 12).copy()
    h = per_token(SPAN_SMALL, ck, toks[12:], 12, toks[:12])
    assert not np.array_equal(g, h)
    assert float(np.max(np.abs(g - h))) <= 1e-3
