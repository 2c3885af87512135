"""-m gpu: Qwen3-Embedding / Qwen3-Reranker entry point (aha_hip_embed) against the oracle restatement
(oracle/qwen3.py embed_one / rerank; reference: qwen3_embedding/mod.rs:50-64, qwen3_reranker/mod.rs:23-31)."""
import numpy as np
import pytest
import torch

from aha_amd.configs import tiny_qwen3
from aha_amd.weights import qwen3_text_weights
from oracle import qwen3 as oq
from oracle.numerics import Numerics

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pair(gpu):
    from aha_amd.model import HipInferenceModel
    cfg = tiny_qwen3(layers=3, hidden=512, heads=4, kv_heads=2, inter=1024, vocab=4096)
    w = qwen3_text_weights(cfg, seed=0)
    m = HipInferenceModel(cfg, w)
    o = oq.OracleQwen3(cfg, w, Numerics("bf16", matmul_f64=True))
    yield cfg, m, o
    m.close()


def seqs_for(cfg, lens, seed):
    g = np.random.default_rng(seed)
    return [[int(x) for x in g.integers(0, cfg.vocab_size, size=n)] for n in lens]


def test_embed_matches_oracle(pair):
    """Both sides hold the pooled hidden state in bf16 and normalise in f32; the hidden state itself differs by f32
    accumulation order upstream (same tolerance class as the logits tests): per element <= 0.04 of the vector's rms,
    cosine to the oracle embedding >= 0.9995, unit norm to 1e-5."""
    cfg, m, o = pair
    for ids in seqs_for(cfg, [1, 7, 64, 65, 300], 1):
        got = m.embed_one(ids)
        ref = oq.embed_one(o, ids).numpy()
        assert got.shape == ref.shape == (cfg.hidden_size,)
        assert abs(float(np.linalg.norm(got)) - 1.0) < 1e-5
        rms = float(np.sqrt((ref ** 2).mean()))
        assert float(np.abs(got - ref).max()) <= 0.04 * rms
        assert float(got @ ref) >= 0.9995
        assert m.cache_len() == 0   # clear_kv_cache after every embedding (qwen3_embedding/mod.rs:58)


def test_embed_is_prefix_independent_and_deterministic(pair):
    """The cache is cleared before and after: embedding B after A equals embedding B alone, bit for bit."""
    cfg, m, o = pair
    a, b = seqs_for(cfg, [40, 90], 2)
    m.forward_initial(a, 0)   # leave a dirty cache on purpose
    e1 = m.embed_one(b)
    m.embed_one(a)
    e2 = m.embed_one(b)
    np.testing.assert_array_equal(e1, e2)


def test_rerank_matches_oracle(pair):
    cfg, m, o = pair
    q, *docs = seqs_for(cfg, [12, 30, 5, 77], 3)
    got = m.rerank(q, docs)
    ref = oq.rerank(o, q, docs).numpy()
    assert got.shape == ref.shape == (3,)
    assert float(np.abs(got - ref).max()) < 2e-3
    assert abs(float(m.rerank(q, [q])[0]) - 1.0) < 1e-5   # a document identical to the query scores 1


def test_embed_errors(pair):
    from aha_amd._lib import AhaHipError
    cfg, m, o = pair
    with pytest.raises(AhaHipError, match="empty"):
        m.embed_one([])
    with pytest.raises(ValueError, match="cannot be empty"):
        m.embed_multi([])
    with pytest.raises(AhaHipError, match="out of range"):
        m.embed_one([cfg.vocab_size])


def test_documents_without_ids_are_refused(pair):
    """aha_hip_embed_multi with a null id array, whatever the lengths say, as aha_hip_embed refuses it; nothing is written."""
    import ctypes as C
    from aha_amd._lib import lib
    cfg, m, _ = pair
    out = np.full((3, cfg.hidden_size), 7, dtype=np.float32)
    fp, up = C.POINTER(C.c_float), C.POINTER(C.c_uint64)
    for lens in ([5, 9, 2], [1, 4, 4], [0, 0, 0]):
        n = np.array(lens, dtype=np.uint64)
        one = lib().aha_hip_embed(m.handle, None, lens[0], out.ctypes.data_as(fp))
        assert lib().aha_hip_embed_multi(m.handle, None, n.ctypes.data_as(up), 3, out.ctypes.data_as(fp)) == one == -1
    assert (out == 7).all() and m.cache_len() == 0


@pytest.mark.parametrize("heads, kv_heads", [(4, 2), (16, 8)])
def test_documents_together(gpu, heads, kv_heads):
    """embed_multi's joint prefill, document lengths around a cache page (64) and around the rows that one prefill takes (4096), with one-token documents
    between: each vector within the bound of test_embed_matches_oracle of what the document gives alone, both being within half of it of the exact one."""
    from aha_amd._lib import AhaHipError
    from aha_amd.model import HipInferenceModel
    cfg = tiny_qwen3(layers=2, hidden=256, heads=heads, kv_heads=kv_heads, inter=512, vocab=2048)
    m = HipInferenceModel(cfg, qwen3_text_weights(cfg, seed=1))
    try:
        for lens in ([2, 3], [63, 1, 64, 65, 300, 2, 129], [2000, 2100, 7], [4097, 5, 4095, 1, 1], [90] * 70):
            docs = seqs_for(cfg, lens, len(lens))
            got = m.embed_multi(docs)
            ref = np.stack([m.embed_one(x) for x in docs])
            assert got.shape == ref.shape and m.cache_len() == 0
            rms = np.sqrt((ref ** 2).mean(1))
            assert float((np.abs(got - ref).max(1) / rms).max()) <= 0.04
            assert float((got * ref).sum(1).min()) >= 0.9995
        for bad in ([[1, 2], [3, 4], []], [[1, 2], [3, cfg.vocab_size], [5, 6]]):
            with pytest.raises(AhaHipError, match="empty|out of range"):
                m.embed_multi(bad)
    finally:
        m.close()


def test_documents_on_pages_of_others(gpu):
    """Keys and values that are not numbers, left by an earlier call on the pages that a document now fills in part: its vector is what it was on fresh ones."""
    from aha_amd.model import HipInferenceModel
    cfg = tiny_qwen3(layers=2, hidden=256, heads=4, kv_heads=2, inter=512, vocab=2048)
    w = qwen3_text_weights(cfg, seed=1)
    w["model.embed_tokens.weight"][7] = float("nan")
    m = HipInferenceModel(cfg, w)
    docs = [[t if t != 7 else 8 for t in d] for d in seqs_for(cfg, [3, 70, 33, 128, 5], 6)]
    first = m.embed_multi(docs)
    assert np.isfinite(first).all()
    assert np.isnan(m.embed_multi([[7] * 320, [7] * 320])).all()
    np.testing.assert_array_equal(m.embed_multi(docs), first)
    m.close()


@pytest.mark.parametrize("how", ["environment", "hook"])
def test_documents_one_by_one_in_a_form_that_was_asked_for(gpu, how):
    """AHA_ATTN_FORM (read once per process: a child) and aha_hip_debug_attn_form name the attention kernel of every prefill: no joint one, the vectors of
    embed_one bit for bit."""
    import os
    import subprocess
    import sys
    code = """
import numpy as np
from aha_amd._lib import lib
from aha_amd.model import HipInferenceModel
from tests.test_embedding_gpu import qwen3_text_weights, seqs_for, tiny_qwen3
cfg = tiny_qwen3(layers=2, hidden=256, heads=4, kv_heads=2, inter=512, vocab=2048)
m = HipInferenceModel(cfg, qwen3_text_weights(cfg, seed=1))
docs = seqs_for(cfg, [300, 129, 200], 5)
if %r == "hook":
    lib().aha_hip_debug_attn_form(64)
np.testing.assert_array_equal(m.embed_multi(docs), np.stack([m.embed_one(x) for x in docs]))
m.close()
""" % how
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, PYTHONPATH=root)
    env.pop("AHA_ATTN_FORM", None)
    if how == "environment":
        env["AHA_ATTN_FORM"] = "64"
    r = subprocess.run([sys.executable, "-c", code], cwd=root, env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]


def test_documents_in_little_memory(gpu):
    """Whatever memory is left: documents that fit one by one are embedded together or one by one, never refused (the joint prefill's scratch, larger
    than a single document's, may leave no room for the cache slab that both need)."""
    from aha_amd._lib import AhaHipError, check, lib
    from aha_amd.model import HipInferenceModel
    cfg = tiny_qwen3(layers=2, hidden=256, heads=4, kv_heads=2, inter=512, vocab=2048)
    w = qwen3_text_weights(cfg, seed=1)
    docs = seqs_for(cfg, [900] * 4 + [30], 5)
    outcomes = set()
    for limit in range(8 << 20, 120 << 20, 4 << 20):
        alone, together = [], []
        for out, call in ((alone, lambda m: np.stack([m.embed_one(x) for x in docs])), (together, lambda m: m.embed_multi(docs))):
            m = HipInferenceModel(cfg, w)
            check(lib().aha_hip_debug_memory_limit(m.handle, limit))
            try:
                out.append(call(m))
            except AhaHipError as e:
                assert "hipMalloc" in str(e)
            m.close()
        assert len(alone) <= len(together), limit
        outcomes.add((len(alone), len(together)))
        if alone:
            assert float((alone[0] * together[0]).sum(1).min()) >= 0.9995
    assert outcomes == {(0, 0), (1, 1)}   # the limits range from too little for a document to room for all


def test_a_document_that_repeats_the_query_scores_one(gpu):
    """Among other documents too, at widths where the kernels follow the number of rows (K >= 768: few rows alone, tiles together); equal documents of
    one call get equal vectors."""
    from aha_amd.model import HipInferenceModel
    cfg = tiny_qwen3(layers=4, hidden=1024, heads=8, kv_heads=2, inter=3072, vocab=2048)
    m = HipInferenceModel(cfg, qwen3_text_weights(cfg, seed=2))
    q, a, b = seqs_for(cfg, [19, 230, 77], 9)
    s = m.rerank(q, [a, q, b, q])
    assert abs(float(s[1]) - 1) < 1e-5 and s[1] == s[3] and s[0] < 0.999 and s[2] < 0.999
    v = m.embed_multi([b, q, a, b, q])
    np.testing.assert_array_equal(v[0], v[3])
    np.testing.assert_array_equal(v[1], v[4])
    with pytest.raises(ValueError, match="cannot be empty"):
        m.rerank(q, [])
    m.close()
