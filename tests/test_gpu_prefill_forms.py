"""GPU: every form that a prefill launch can take (cq_state_set_prefill_form)
against the decode step run once per prompt token, at ragged shapes.  Left to
their own rules the launches take one form per shape, so the other prefill
tests reach only some of them."""
import functools

import numpy as np
import pytest

import cuqwen_amd as cq
from tests.conftest import tiny_config

pytestmark = pytest.mark.gpu
# the two paths round in different places: 1e-2 of the largest value as in the
# other prefill tests; a row of a quantized cache may differ by a code (int8:
# 1/127 of its maximum, E4M3: 0.08), and E4M3 codes move the logits (3e-2)
LOGITS = {cq.KV_FP16: 1e-2, cq.KV_INT8: 1e-2, cq.KV_FP8: 3e-2}
ROWS = {cq.KV_FP16: 1e-2, cq.KV_INT8: 2e-2, cq.KV_FP8: 0.08}


def _rel(a, b):
    a, b = a.astype(np.float64), b.astype(np.float64)
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-6)


def _prompt(cfg, n):
    return [int(cq.lib.cq_synth_uniform(8, 0, i, cfg.vocab_size)) for i in range(n)]


def _config(shape, quant, layers):
    d, inter, heads, kv_heads, hd = shape
    return tiny_config(quant, dim=d, intermediate_size=inter, n_heads=heads, n_kv_heads=kv_heads, head_dim=hd,
                       n_layers=layers, max_seq_len=4096)


def _results(cfg, st, n, pos0):
    rows = [st.kv_read(cfg.n_layers - 1, h, kind, pos0 + n)[pos0:] for h in range(cfg.n_kv_heads) for kind in (0, 1)]
    return st.logits(), rows


@functools.lru_cache(maxsize=None)
def _decoded(shape, quant, layers, kv, n, pos0):
    """Logits after the last token and the last layer's new cache rows, one decode step per token."""
    cfg = _config(shape, quant, layers)
    w = cq.synth_weights(cfg, 41)
    st = cq.State(cfg, w, kv_dtype=kv)
    if pos0:
        st.fill_kv(pos0, 5)
    for i, t in enumerate(_prompt(cfg, n)):
        st.forward(t, pos0 + i, [])
    out = _results(cfg, st, n, pos0)
    st.free()
    w.free()
    return out


def _check(shape, quant, layers, kv, n, pos0, **form):
    print(shape, quant, kv, n, pos0, form, flush=True)
    cfg = _config(shape, quant, layers)
    w = cq.synth_weights(cfg, 41)
    st = cq.State(cfg, w, kv_dtype=kv)
    if pos0:
        st.fill_kv(pos0, 5)
    st.set_prefill_form(**form)
    st.prefill(_prompt(cfg, n), pos0)
    logits, rows = _results(cfg, st, n, pos0)
    st.free()
    w.free()
    ref_logits, ref_rows = _decoded(shape, quant, layers, kv, n, pos0)
    assert _rel(logits, ref_logits) <= LOGITS[kv], kv
    for i, (a, b) in enumerate(zip(rows, ref_rows)):
        assert _rel(a, b) <= ROWS[kv], (kv, i)


# K of 5, 9, 8 and 22 steps of 128 (odd ones: unequal halves of the stream's
# blocks), rows that do not fill a block, 70 tokens at position 5: token tiles
# and the groups of four positions of V ragged at both ends.  Split 1 of the
# large tile is the fused epilogue (quantized rows included), of the stream the
# fused SwiGLU.
@pytest.mark.parametrize("tokens,split", [(16, 1), (16, 3), (32, 1), (32, 3), (64, 1), (64, 4), (128, 1), (128, 3)])
@pytest.mark.parametrize("shape", [(640, 1152, 10, 2, 64), (1024, 2816, 8, 4, 128)])
@pytest.mark.parametrize("quant", [0, 1, 2])
def test_gemm_forms(quant, shape, tokens, split):
    for kv in (cq.KV_FP16, cq.KV_INT8, cq.KV_FP8):
        _check(shape, quant, 3, kv, 70, 5, gemm_tokens=tokens, gemm_split=split)


# 75 tokens of a group of seven are 525 rows: two or more blocks, the last one
# ragged.  After 2900 positions a block takes up to 47 steps, or as few as one
# in 40 ranges; at position 0 the first blocks have fewer tiles than ranges.
@pytest.mark.parametrize("rows", [64, 128, 256])
@pytest.mark.parametrize("splits,pos0", [(1, 2900), (3, 2900), (40, 2900), (1, 0), (3, 0)])
@pytest.mark.parametrize("heads,kv_heads,hd", [(14, 2, 64), (7, 1, 128)])
def test_attention_forms(heads, kv_heads, hd, splits, pos0, rows):
    for kv in (cq.KV_FP16, cq.KV_INT8):
        _check((512, 512, heads, kv_heads, hd), 2, 2, kv, 75, pos0, attn_rows=rows, attn_splits=splits)


def test_form_arguments():
    cfg = tiny_config(2)   # K of 256: two steps, too few for the stream
    w = cq.synth_weights(cfg, 3)
    st = cq.State(cfg, w)
    for bad in ((8, 1, 0, 1), (16, 0, 0, 1), (128, 33, 0, 1), (0, 1, 32, 1), (0, 1, 64, 0), (0, 1, 64, 65)):
        with pytest.raises(cq.CuQwenError):
            st.set_prefill_form(*bad)
    st.set_prefill_form(16, 1)
    with pytest.raises(cq.CuQwenError, match="weight stream"):
        st.prefill([1, 2, 3], 0)
    st.set_prefill_form()
    st.prefill([1, 2, 3], 0)
    st.free()
    w.free()
