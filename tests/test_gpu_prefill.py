"""GPU batched prefill (cq_prefill) against the host oracle run token by
token, which is the reference's own prefill loop (src/main.cu:87-92: one
qwen_forward per prompt token, no penalty history)."""
import numpy as np
import pytest

import cuqwen_amd as cq
from oracle import oracle as orc
from tests.conftest import tiny_config

pytestmark = pytest.mark.gpu
TOL = 1e-2


def _gap(logits):
    l = np.sort(logits.astype(np.float64))
    return l[-1] - l[-2]


def _rel(a, b):
    a, b = a.astype(np.float64), b.astype(np.float64)
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-6)


def _prompt(cfg, n, seed):
    return [int(cq.lib.cq_synth_uniform(seed, 0, i, cfg.vocab_size)) for i in range(n)]


def _check_kv(cfg, st, ref_kv, n, layers=None):
    for layer in (layers if layers is not None else range(cfg.n_layers)):
        for h in range(cfg.n_kv_heads):
            for kind in (0, 1):
                g = st.kv_read(layer, h, kind, n)
                assert _rel(g, ref_kv(layer, h, kind, n)) <= TOL, (layer, h, kind)


def _oracle_prompt(om, prompt, pos0):
    tok = None
    for i, t in enumerate(prompt):
        tok = om.forward(t, pos0 + i, [])
    return tok


@pytest.mark.parametrize("quant", [0, 1, 2])
@pytest.mark.parametrize("segments", [[70], [1], [30, 45], [17, 1, 64]])
def test_prefill_tiny_matches_oracle(quant, segments):
    """Ragged lengths (not multiples of the 16-token attention or 64-token GEMM
    tiles), a one-token prompt, and prompts continued at pos0 > 0."""
    cfg = tiny_config(quant)
    w = cq.synth_weights(cfg, 21)
    om = orc.Model.synth(cfg, 21, cfg.max_seq_len)
    st = cq.State(cfg, w)
    pos = 0
    for si, n in enumerate(segments):
        prompt = _prompt(cfg, n, 100 + si)
        ot = _oracle_prompt(om, prompt, pos)
        gt = st.prefill(prompt, pos)
        ol = om.logits()
        assert _rel(st.logits(), ol) <= TOL
        if _gap(ol) > 1e-2:
            assert gt == ot
        pos += n
    _check_kv(cfg, st, om.kv, pos)
    # decoding continues from the prefilled cache like the oracle
    tok = ot
    for i in range(6):
        a, b = om.forward(tok, pos + i, []), st.forward(tok, pos + i, [])
        assert _rel(st.logits(), om.logits()) <= TOL
        if _gap(om.logits()) > 1e-2:
            assert a == b
        tok = a
    st.free()
    w.free()


@pytest.mark.parametrize("heads,kv_heads,hd", [(16, 1, 64), (12, 1, 128), (10, 1, 64), (24, 2, 64)])
@pytest.mark.parametrize("quant", [0, 2])
def test_prefill_large_gqa_groups_match_oracle(quant, heads, kv_heads, hd):
    """GQA groups of 9-16 query heads per kv head (more rows of a token than
    a 16-row slice has, or not a multiple of it) against the oracle run token
    by token: logits, top-1 and the KV cache, then decode continues."""
    cfg = tiny_config(quant, n_heads=heads, n_kv_heads=kv_heads, head_dim=hd, dim=1024)
    w = cq.synth_weights(cfg, 23)
    om = orc.Model.synth(cfg, 23, cfg.max_seq_len)
    st = cq.State(cfg, w)
    prompt = _prompt(cfg, 83, 7)
    ot = _oracle_prompt(om, prompt, 0)
    gt = st.prefill(prompt, 0)
    assert _rel(st.logits(), om.logits()) <= TOL
    if _gap(om.logits()) > 1e-2:
        assert gt == ot
    _check_kv(cfg, st, om.kv, len(prompt))
    a, b = om.forward(ot, len(prompt), []), st.forward(ot, len(prompt), [])
    assert _rel(st.logits(), om.logits()) <= TOL
    st.free()
    w.free()


@pytest.mark.parametrize("n", [2100, 2049])
def test_prefill_crosses_chunks(n):
    """A prompt longer than 2048 tokens is several passes of at most 2048
    (2049: the last pass holds only the last token)."""
    cfg = tiny_config(2, max_seq_len=4096)
    w = cq.synth_weights(cfg, 5)
    om = orc.Model.synth(cfg, 5, cfg.max_seq_len)
    st = cq.State(cfg, w)
    prompt = _prompt(cfg, n, 9)
    ot = _oracle_prompt(om, prompt, 0)
    gt = st.prefill(prompt, 0)
    assert _rel(st.logits(), om.logits()) <= TOL
    if _gap(om.logits()) > 1e-2:
        assert gt == ot
    _check_kv(cfg, st, om.kv, n)
    st.free()
    w.free()


def _gpu_reference(cfg, w, prompt, pos0, n_ctx):
    """The same prompt through the GPU decode step one token at a time."""
    st = cq.State(cfg, w)
    if n_ctx:
        st.fill_kv(n_ctx, 77)
    tok = None
    for i, t in enumerate(prompt):
        tok = st.forward(t, pos0 + i, [])
    return st, tok


@pytest.mark.parametrize("model,quant,layers,n,n_ctx", [
    ("7B", "int4", 2, 130, 2000), ("0.5B", "int8", 24, 1024, 0), ("14B", "int4", 2, 64, 100),
    ("7B", "fp16", 2, 80, 0), ("1.5B", "int4", 3, 200, 4000), ("7B", "int8", 2, 33, 32768 - 40),
    ("7B", "int4", 2, 2100, 10)])
def test_prefill_matches_decode_real_shapes(model, quant, layers, n, n_ctx):
    """BASELINE model shapes: batched prefill equals the decode step run once
    per prompt token (logits within 1e-2, same top-1 where the top-2 gap
    exceeds 1e-2, same KV cache within 1e-2), in the forms that the launches
    pick for these shapes (tests/test_gpu_prefill_forms.py: every form)."""
    cfg = cq.preset(model, quant).replace(n_layers=layers)
    w = cq.synth_weights(cfg, 0x5157454E)
    prompt = _prompt(cfg, n, 31)
    ref, rt = _gpu_reference(cfg, w, prompt, n_ctx, n_ctx)
    st = cq.State(cfg, w)
    if n_ctx:
        st.fill_kv(n_ctx, 77)
    gt = st.prefill(prompt, n_ctx)
    rl = ref.logits()
    assert _rel(st.logits(), rl) <= TOL
    if _gap(rl) > 1e-2:
        assert gt == rt
    _check_kv(cfg, st, lambda l, h, k, m: ref.kv_read(l, h, k, m), n_ctx + n, layers=[0, layers - 1])
    st.free()
    ref.free()
    w.free()


# query rows (n * group) around the 32-row waves and the 64 / 128 / 256-row
# blocks (256 only at contexts of a few tiles: tests/test_gpu_prefill_forms.py
# has each block size over long ones), contexts around the 32-key tiles and long
# enough for split key ranges (2 tokens at 3001: more ranges than a block has
# waves), every cache format, both head sizes, groups that do not divide a wave
@pytest.mark.parametrize("heads,kv_heads,hd,n,pos0", [
    (14, 2, 64, 9, 0), (14, 2, 64, 37, 31), (14, 2, 64, 5, 1000), (16, 16, 64, 33, 0), (28, 4, 128, 2, 3001),
    (28, 4, 128, 10, 0), (28, 4, 128, 37, 95), (12, 1, 128, 11, 700), (16, 1, 128, 17, 33), (5, 5, 128, 64, 32)])
@pytest.mark.parametrize("kv", [cq.KV_FP16, cq.KV_INT8, cq.KV_FP8])
def test_prefill_attention_edges_match_decode(heads, kv_heads, hd, n, pos0, kv):
    cfg = tiny_config(2, n_heads=heads, n_kv_heads=kv_heads, head_dim=hd, dim=512, max_seq_len=4096)
    w = cq.synth_weights(cfg, 11)
    prompt = _prompt(cfg, n, 3)
    st, ref = cq.State(cfg, w, kv_dtype=kv), cq.State(cfg, w, kv_dtype=kv)
    if pos0:
        st.fill_kv(pos0, 5)
        ref.fill_kv(pos0, 5)
    st.prefill(prompt, pos0)
    for i, t in enumerate(prompt):
        ref.forward(t, pos0 + i, [])
    assert _rel(st.logits(), ref.logits()) <= TOL
    # layer 1's rows come from layer 0's attention of every token; a quantized
    # row may differ by a code (int8: 1/127 of its maximum, E4M3: 0.08)
    tol = {cq.KV_FP16: TOL, cq.KV_INT8: 2e-2, cq.KV_FP8: 0.08}[kv]
    for h in range(kv_heads):
        for kind in (0, 1):
            a, b = (x.kv_read(1, h, kind, pos0 + n)[pos0:] for x in (st, ref))
            assert _rel(a, b) <= tol, (h, kind)
    st.free()
    ref.free()
    w.free()


# tokens around the 16-token slices and the stream's 16 / 32 / 64-token tiles;
# K of 5, 9 (odd numbers of 128-wide steps: unequal K groups, scales of a row's
# end fetched with its last four), 8 and 22 steps, row counts that do not fill
# a 128-row block
@pytest.mark.parametrize("n", [2, 15, 16, 17, 33, 64, 65, 130])
@pytest.mark.parametrize("shape", [(640, 1152, 10, 2, 64), (1024, 2816, 8, 4, 128)])
@pytest.mark.parametrize("quant", [0, 1, 2])
def test_prefill_few_tokens_match_decode(quant, shape, n):
    d, inter, heads, kv_heads, hd = shape
    cfg = tiny_config(quant, dim=d, intermediate_size=inter, n_heads=heads, n_kv_heads=kv_heads, head_dim=hd, n_layers=3)
    w = cq.synth_weights(cfg, 41)
    prompt = _prompt(cfg, n, 8)
    for kv in (cq.KV_FP16, cq.KV_INT8):
        st, ref = cq.State(cfg, w, kv_dtype=kv), cq.State(cfg, w, kv_dtype=kv)
        st.prefill(prompt, 0)
        for i, t in enumerate(prompt):
            ref.forward(t, i, [])
        assert _rel(st.logits(), ref.logits()) <= TOL
        # an int8 row may differ by a code, 1/127 of its maximum
        tol = TOL if kv == cq.KV_FP16 else 2e-2
        for h in range(kv_heads):
            for kind in (0, 1):
                assert _rel(st.kv_read(2, h, kind, n), ref.kv_read(2, h, kind, n)) <= tol, (h, kind)
        st.free()
        ref.free()
    w.free()


# the unsplit QKV epilogue (enough row and token blocks that a split does not
# pay) stores V by aligned groups of four positions: ragged ends and starts
@pytest.mark.parametrize("n,pos0", [(1025, 0), (1051, 3), (1027, 6)])
def test_prefill_unsplit_qkv_cache_rows(n, pos0):
    cfg = tiny_config(2, n_heads=56, n_kv_heads=8, head_dim=64, dim=512, max_seq_len=2048, n_layers=1)
    w = cq.synth_weights(cfg, 17)
    prompt = _prompt(cfg, n, 5)
    st, ref = cq.State(cfg, w), cq.State(cfg, w)
    if pos0:
        st.fill_kv(pos0, 5)
        ref.fill_kv(pos0, 5)
    st.prefill(prompt, pos0)
    for i in range(0, n, 63):   # layer 0's rows depend on their own token alone
        ref.forward(prompt[i], pos0 + i, [])
    ref.forward(prompt[-1], pos0 + n - 1, [])
    rows = [pos0 + i for i in range(0, n, 63)] + [pos0 + n - 1]
    for h in range(8):
        for kind in (0, 1):
            a, b = st.kv_read(0, h, kind, pos0 + n + 8), ref.kv_read(0, h, kind, pos0 + n + 8)
            assert _rel(a[rows], b[rows]) <= TOL, (h, kind)
            assert np.array_equal(a[:pos0], b[:pos0]) and not a[pos0 + n:].any()
    st.free()
    w.free()
    ref.free()


@pytest.mark.parametrize("hd,n,pos0", [(64, 40, 0), (128, 3, 600), (128, 33, 5)])
def test_prefill_ignores_stale_cache(hd, n, pos0):
    """Whatever the cache holds past the context (NaN here) stays out of the
    result, bit for bit."""
    cfg = tiny_config(0, n_heads=4, n_kv_heads=2, head_dim=hd, max_seq_len=1024)
    w = cq.synth_weights(cfg, 12)
    prompt = _prompt(cfg, n, 4)
    out = []
    for stale in (False, True):
        st = cq.State(cfg, w)
        if stale:
            bad = np.full((1024, hd), np.nan, dtype=np.float16)
            for layer in range(cfg.n_layers):
                for h in range(2):
                    for kind in (0, 1):
                        st.kv_write(layer, h, kind, bad)
        if pos0:
            st.fill_kv(pos0, 6)
        st.prefill(prompt, pos0)
        out.append(st.logits())
        st.free()
    assert np.isfinite(out[0]).all() and np.array_equal(out[0], out[1])
    w.free()


def test_prefill_config2_shapes_match_oracle():
    """BASELINE config 2's model (Qwen2.5-0.5B INT8, tied lm_head) with 3 of
    the 24 layers, a 300-token synthetic prompt, against the oracle token by
    token (the full 1024-token prompt is compared GPU-to-GPU above)."""
    cfg = cq.preset("0.5B", "int8").replace(n_layers=3)
    w = cq.synth_weights(cfg, 0x5157454E)
    om = orc.Model.synth(cfg, 0x5157454E, 1024)
    st = cq.State(cfg, w)
    prompt = _prompt(cfg, 300, 42)
    ot = _oracle_prompt(om, prompt, 0)
    gt = st.prefill(prompt, 0)
    assert _rel(st.logits(), om.logits()) <= TOL
    if _gap(om.logits()) > 1e-2:
        assert gt == ot
    _check_kv(cfg, st, om.kv, 300, layers=[0, 2])
    st.free()
    w.free()


def test_prefill_errors():
    cfg = tiny_config(1)
    w = cq.synth_weights(cfg, 3)
    st = cq.State(cfg, w)
    with pytest.raises(cq.CuQwenError, match="max_seq_len"):
        st.prefill([1] * 10, cfg.max_seq_len - 5)
    with pytest.raises(cq.CuQwenError, match="vocabulary"):
        st.prefill([1, cfg.vocab_size], 0)
    with pytest.raises(cq.CuQwenError, match="no tokens"):
        st.prefill([], 0)
    st.free()
    w.free()
