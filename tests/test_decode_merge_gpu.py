"""-m gpu: decode attention whose split-KV partials are merged by the o_proj matvec (attn_decode_defer_kernel + gemv_merge_kernel), against the form
that launches norm, attention and combine by themselves."""
import numpy as np
import pytest

from aha_amd.configs import tiny_qwen3
from aha_amd.weights import qwen3_text_weights
from tests.test_model_gpu import LOGIT_RMS_STD, LOGIT_TOL_STD, ids_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,lens", [
    (4, 2, [126, 127, 128, 255, 1022, 3070]),       # 1 -> 2 splits, whole pages, 8 splits and the last length merged this way
    (6, 2, [190, 700]),                             # 768 columns: no whole chunk groups for the matvec
    (1, 1, [320]),                                  # one head, 128 columns
    (16, 1, [449]),                                 # sixteen query heads in one block, 2048 columns
    (32, 8, [128, 1534, 1535, 1536]),               # 4096 columns: 4 splits, the first length beyond them
])
def test_partials_merged_by_the_projection(gpu, monkeypatch, heads, kv_heads, lens):
    """Two layers, three steps from each length on; the bound is that of the two decode forms' own test (test_model_gpu.py): the same arithmetic per
    token, another merge order."""
    from aha_amd.model import HipInferenceModel
    cfg = tiny_qwen3(layers=2, hidden=512, heads=heads, kv_heads=kv_heads, inter=512, vocab=1024)
    w = qwen3_text_weights(cfg, seed=4)
    monkeypatch.setenv("AHA_DECODE_FUSED", "1")
    merged = HipInferenceModel(cfg, w)
    monkeypatch.setenv("AHA_DECODE_FUSED", "0")
    plain = HipInferenceModel(cfg, w)
    for S in lens:
        ids = ids_for(cfg, S, 7 + S)
        merged.clear_cache(); plain.clear_cache()
        _, tok = plain.forward_initial(ids, 0)
        merged.forward_initial(ids, 0)
        for step in range(3):
            a, am = plain.forward_step(tok, S + step)
            b, _ = merged.forward_step(tok, S + step)
            std = float(a.std())
            assert np.isfinite(b).all()
            assert float(np.abs(a - b).max()) <= LOGIT_TOL_STD * std and float(np.sqrt(((a - b) ** 2).mean())) <= LOGIT_RMS_STD * std, (S, step)
            tok = am
    merged.close(); plain.close()


@pytest.mark.parametrize("scrambled", [False, True])
@pytest.mark.parametrize("lens", [[1, 2, 62, 63, 64, 65], [127, 128, 191, 256, 319, 320], [381, 382, 383, 500], [1021, 1022, 1023, 1500], [2047, 12286]])
def test_projection_in_slices(gpu, monkeypatch, lens, scrambled):
    """attn_oproj_kernel (up to six pages), oproj_slice_kernel (9 to 16 splits, 17 to 192 pages) and gemv_row_slices_kernel at the widths they are built for,
    across the lengths where one takes over from another, pages at one distance from each other and not; the bound as above."""
    from aha_amd.model import HipInferenceModel
    cfg = tiny_qwen3(layers=3, hidden=1024, heads=16, kv_heads=8, inter=1536, vocab=1024)
    w = qwen3_text_weights(cfg, seed=14)
    monkeypatch.setenv("AHA_DECODE_FUSED", "1")
    sliced = HipInferenceModel(cfg, w)
    monkeypatch.setenv("AHA_DECODE_FUSED", "0")
    plain = HipInferenceModel(cfg, w)
    sliced.debug_scramble_pages(scrambled)
    for S in lens:
        ids = ids_for(cfg, S, 9 + S)
        sliced.clear_cache(); plain.clear_cache()
        _, tok = plain.forward_initial(ids, 0)
        sliced.forward_initial(ids, 0)
        for step in range(4):
            a, am = plain.forward_step(tok, S + step)
            b, _ = sliced.forward_step(tok, S + step)
            std = float(a.std())
            assert np.isfinite(b).all()
            assert float(np.abs(a - b).max()) <= LOGIT_TOL_STD * std and float(np.sqrt(((a - b) ** 2).mean())) <= LOGIT_RMS_STD * std, (S, step)
            tok = am
    sliced.close(); plain.close()


@pytest.mark.parametrize("positions, launches", [(20, 3), (500, 4), (1200, 4)])
def test_profile_of_the_projection_in_slices(gpu, positions, launches):
    """Bytes and launches are booked where they run: o_proj's weights with the attention where one launch does both (20 positions), with the matvecs elsewhere."""
    from aha_amd.model import HipInferenceModel
    H, nq, nkv, I, V, layers = 1024, 2048, 1024, 1536, 1024, 3
    cfg = tiny_qwen3(layers=layers, hidden=H, heads=16, kv_heads=8, inter=I, vocab=V)
    m = HipInferenceModel(cfg, qwen3_text_weights(cfg, seed=14))
    m.forward_initial(ids_for(cfg, positions, 3), 0)
    m.set_profiling(True)
    m.forward_step(5, positions)
    m.set_profiling(False)
    gemv, attn = m.get_profile("gemv"), m.get_profile("attn_decode")
    m.close()
    o = nq * H
    weights = layers * ((nq + 2 * nkv) * H + 3 * I * H + (0 if launches == 3 else o)) + V * H
    cache = layers * (positions + 1) * 2 * nkv
    assert gemv["launches"] == layers * launches + 1 and attn["launches"] == layers
    assert 2 * weights <= gemv["bytes"] <= 1.02 * 2 * weights and 2 * weights <= gemv["flops"] <= 1.02 * 2 * weights
    both = 2 * (cache + (layers * o if launches == 3 else 0))
    assert both <= attn["bytes"] <= 1.02 * both + layers * (17 * nq * 4 + 8 * H * 4)   # (the splits' partials, the slices' sums)


@pytest.mark.parametrize("hidden, vocab", [(256, 64), (256, 5000), (1024, 70001)])
def test_between_two_steps(gpu, hidden, vocab):
    """The launch between two steps of the greedy loop (arg-max, state, embedding row, rope table) against the same tokens fed one by one: the kernels
    in between are the same, so tokens and the last logits agree exactly; fewer and more partials than threads, two calls in a row."""
    from aha_amd.configs import tiny_qwen3
    from aha_amd.model import HipInferenceModel
    from aha_amd.weights import qwen3_text_weights
    cfg = tiny_qwen3(layers=2, hidden=hidden, heads=4, kv_heads=2, inter=512, vocab=vocab)
    m = HipInferenceModel(cfg, qwen3_text_weights(cfg, seed=2))
    try:
        prompt = [int(t) for t in np.random.default_rng(vocab).integers(0, vocab, 61)]
        _, first = m.forward_initial(prompt, 0)
        got = m.decode_greedy(first, 61, 5)
        got += m.decode_greedy(got[-1], 66, 4)
        last = m.last_logits()
        m.clear_cache()
        _, tok = m.forward_initial(prompt, 0)
        ref = []
        for i in range(9):
            logits, tok = m.forward_step(tok, 61 + i)
            ref.append(int(tok))
        assert got == ref
        np.testing.assert_array_equal(last, logits)
    finally:
        m.close()


def test_three_launch_form_keeps_its_splits(gpu):
    """AHA_DECODE_FUSED=0 has a combine launch of its own and splits the cache as AHA_ATTN_PAGES_PER_BLOCK says (four pages when unset; read once per
    process: children), whatever the merging form would choose: the same logits, bit for bit, with the variable at its default and unset."""
    import os
    import subprocess
    import sys
    code = """
import hashlib
from aha_amd.configs import tiny_qwen3
from aha_amd.model import HipInferenceModel
from aha_amd.weights import qwen3_text_weights
from tests.test_model_gpu import ids_for
cfg = tiny_qwen3(layers=2, hidden=512, heads=4, kv_heads=2, inter=512, vocab=1024)
m = HipInferenceModel(cfg, qwen3_text_weights(cfg, seed=4))
h = hashlib.sha256()
for S in (190, 2200, 3000):
    m.clear_cache()
    _, tok = m.forward_initial(ids_for(cfg, S, S), 0)
    for i in range(2):
        logits, tok = m.forward_step(tok, S + i)
        h.update(logits.tobytes())
m.close()
print("LOGITS", h.hexdigest())
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    seen = []
    for extra in ({}, {"AHA_ATTN_PAGES_PER_BLOCK": "4"}):
        env = dict({k: v for k, v in os.environ.items() if k != "AHA_ATTN_PAGES_PER_BLOCK"}, PYTHONPATH=root, AHA_DECODE_FUSED="0", **extra)
        r = subprocess.run([sys.executable, "-c", code], cwd=root, env=env, capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        seen.append([ln for ln in r.stdout.splitlines() if ln.startswith("LOGITS")][0])
    assert seen[0] == seen[1]


def test_timelines_of_the_projection_in_slices(gpu):
    """AHA_GEMV_TRACE and AHA_ATTN_TRACE (read once per process: a child): the attention and gate + up leave their stamps in every form; o_proj has a line where
    it is a traced launch (500 positions) and none, not that of the step before, where it is not (20 and 1200)."""
    import os
    import subprocess
    import sys
    code = """
import sys
from aha_amd.configs import tiny_qwen3
from aha_amd.model import HipInferenceModel
from aha_amd.weights import qwen3_text_weights
from tests.test_model_gpu import ids_for
cfg = tiny_qwen3(layers=3, hidden=1024, heads=16, kv_heads=8, inter=1536, vocab=1024)
m = HipInferenceModel(cfg, qwen3_text_weights(cfg, seed=4))
for S in (500, 20, 500, 1200):
    m.clear_cache()
    _, tok = m.forward_initial(ids_for(cfg, S, S), 0)
    print("positions", S, file=sys.stderr, flush=True)
    m.forward_step(tok, S)
    print("end", file=sys.stderr, flush=True)
m.close()
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", code], cwd=root, env=dict(os.environ, PYTHONPATH=root, AHA_GEMV_TRACE="1", AHA_ATTN_TRACE="1"), capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    for part in r.stderr.split("positions ")[1:]:
        S = int(part.split()[0])
        part = part.split("\nend")[0].splitlines()
        assert [ln.split()[2] for ln in part if ln.startswith("[gemv trace]")] == ["qkv"] + ["o_proj"] * (S == 500) + ["gate_up", "down"], S
        assert [ln.split()[3] for ln in part if ln.startswith("[attn trace]")] == ["0:"] + ["1:"] * (S > 20), S
