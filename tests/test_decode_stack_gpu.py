"""-m gpu: a decode step whose layers run as one launch (kernels_decode_stack.hip) against the separate launches, and what happens when it gives up waiting."""
import threading

import numpy as np
import pytest

from aha_amd.configs import tiny_qwen3
from aha_amd.weights import qwen3_text_weights
from tests.test_model_gpu import LOGIT_RMS_STD, LOGIT_TOL_STD, ids_for

pytestmark = pytest.mark.gpu


def models(monkeypatch, n=1, layers=3, vocab=1024):
    """A model of separate launches and n of one launch, the sizes it is written for."""
    from aha_amd.model import HipInferenceModel
    cfg = tiny_qwen3(layers=layers, hidden=1024, heads=16, kv_heads=8, inter=3072, vocab=vocab)
    w = qwen3_text_weights(cfg, seed=14)
    monkeypatch.setenv("AHA_DECODE_STACK", "0")
    plain = HipInferenceModel(cfg, w)
    monkeypatch.setenv("AHA_DECODE_STACK", "1")
    return cfg, plain, [HipInferenceModel(cfg, w) for _ in range(n)]


def close_to(a, b, what):
    """The bound of two decode forms' own test (test_model_gpu.py): the same arithmetic per token, sums in another order."""
    std = float(a.std())
    assert np.isfinite(b).all(), what
    assert float(np.abs(a - b).max()) <= LOGIT_TOL_STD * std and float(np.sqrt(((a - b) ** 2).mean())) <= LOGIT_RMS_STD * std, what


@pytest.mark.parametrize("scrambled", [False, True])
@pytest.mark.parametrize("lens", [[1, 2, 62, 63, 64, 65], [127, 128, 700], [1983, 1984, 2046, 2047, 2048, 2110], [4095, 4159, 6300], [32764]])
def test_one_launch_against_separate_ones(gpu, monkeypatch, lens, scrambled):
    """No page behind the new token, pages' edges, the last length with a page per block at most (2048), two and three pages a block, the last length that is taken
    (32768 positions; the steps behind it are separate launches again)."""
    cfg, plain, (m,) = models(monkeypatch)
    m.debug_scramble_pages(scrambled)
    for S in lens:
        ids = ids_for(cfg, S, 9 + S)
        m.clear_cache(); plain.clear_cache()
        _, tok = plain.forward_initial(ids, 0)
        m.forward_initial(ids, 0)
        before = m.debug_decode_stack()[0]
        for step in range(6 if S > 32000 else 4):
            a, am = plain.forward_step(tok, S + step)
            b, _ = m.forward_step(tok, S + step)
            close_to(a, b, (S, step))
            tok = am
        assert m.debug_decode_stack() == (before + 4, 0), S
    assert plain.debug_decode_stack()[0] == 0
    m.close(); plain.close()


def test_tags_that_come_again(gpu, monkeypatch):
    """A step with more splits than every block joins for itself, behind as many with fewer as bring its first layer the low half of the tag that the last such step's
    last layer had: 21846 steps of three layers are 65538."""
    cfg, plain, (m,) = models(monkeypatch, vocab=256)
    short, long = ids_for(cfg, 3, 1), ids_for(cfg, 200, 2)
    _, tok = plain.forward_initial(long, 0)
    want, _ = plain.forward_step(tok, 200)
    m.forward_initial(ids_for(cfg, 200, 3), 0)
    m.forward_step(5, 200)
    start = m.debug_decode_stack()[0]
    left = 21845
    while left:
        m.clear_cache()
        _, t = m.forward_initial(short, 0)
        m.decode_greedy(t, len(short), min(left, 110))
        left = start + 21845 - m.debug_decode_stack()[0]
        assert left >= 0
    m.clear_cache()
    m.forward_initial(long, 0)
    got, _ = m.forward_step(tok, 200)
    assert m.debug_decode_stack() == (start + 21846, 0)
    close_to(want, got, "a tag that came again")
    m.close(); plain.close()


def test_waits_that_end(gpu, monkeypatch):
    """Waves that may not ask even once give up, the launch ends, and the step is run as separate launches: a single step, steps of the device's loop (from the first
    one, and behind steps that went well), a step whose logits are fetched or sampled from later, one that nobody asks for.  After three of them the model stays with
    separate launches."""
    cfg, plain, ms = models(monkeypatch, 6)
    S = 70
    ids = ids_for(cfg, S, 5)
    _, tok = plain.forward_initial(ids, 0)
    ref, _ = plain.forward_step(tok, S)
    want_vals, want_idx = plain.sample_candidates([], 1.0, 1.0, 5)[:2]
    plain.clear_cache()
    plain.forward_initial(ids, 0)
    want = plain.decode_greedy(tok, S, 12)
    last = plain.last_logits()
    for m in ms:
        m.forward_initial(ids, 0)

    ms[0].debug_decode_stack(0)
    got, _ = ms[0].forward_step(tok, S)
    np.testing.assert_array_equal(got, ref)     # (the launches of the other model)
    assert ms[0].debug_decode_stack() == (1, 1)

    ms[1].debug_decode_stack(0)
    assert ms[1].decode_greedy(tok, S, 12) == want
    np.testing.assert_array_equal(ms[1].last_logits(), last)
    assert ms[1].debug_decode_stack()[1] == 1

    assert ms[2].decode_greedy(tok, S, 4) == want[:4]
    ms[2].debug_decode_stack(0)
    assert ms[2].decode_greedy(want[3], S + 4, 8) == want[4:]
    close_to(last, ms[2].last_logits(), "behind steps that went well")
    assert ms[2].debug_decode_stack()[1] == 1

    ms[3].debug_decode_stack(0)
    ms[3].forward_step_enqueue(tok, S)
    np.testing.assert_array_equal(ms[3].last_logits(), ref)

    ms[4].debug_decode_stack(0)
    ms[4].forward_step_enqueue(tok, S)
    vals, idx = ms[4].sample_candidates([], 1.0, 1.0, 5)[:2]
    np.testing.assert_array_equal(idx, want_idx)
    np.testing.assert_array_equal(vals, want_vals)

    ms[5].debug_decode_stack(0)
    ms[5].forward_step_enqueue(tok, S)
    ms[5].clear_cache()
    ms[5].forward_initial(ids, 0)
    for step in range(3):
        ms[5].forward_step(tok, S + step)
    assert ms[5].debug_decode_stack() == (3, 3)
    for m in [plain] + ms:
        m.close()


def test_two_models_at_once(gpu, monkeypatch):
    """Two threads with a model each: one has the right to the one launch at a time, the other runs separate ones; nobody waits in vain.  Both are fed the same
    tokens as a model alone (greedy tokens of random weights hang on the order of sums), under the bound of the two forms."""
    cfg, plain, ms = models(monkeypatch, 2)
    prompts, fed = [ids_for(cfg, 50, 1), ids_for(cfg, 90, 2)], ids_for(cfg, 40, 3)
    want, got = [], [[], []]
    for p in prompts:
        plain.clear_cache()
        plain.forward_initial(p, 0)
        want.append([plain.forward_step(t, len(p) + i)[0] for i, t in enumerate(fed)])

    def run(i):
        ms[i].forward_initial(prompts[i], 0)
        got[i] = [ms[i].forward_step(t, len(prompts[i]) + k)[0] for k, t in enumerate(fed)]
        ms[i].clear_cache()
        _, tok = ms[i].forward_initial(prompts[i], 0)
        assert len(ms[i].decode_greedy(tok, len(prompts[i]), 60)) == 60
    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(2):
        assert len(got[i]) == len(fed)
        for k in range(len(fed)):
            close_to(want[i][k], got[i][k], (i, k))
    assert [m.debug_decode_stack()[1] for m in ms] == [0, 0] and max(m.debug_decode_stack()[0] for m in ms) > 0
    for m in [plain] + ms:
        m.close()


def pre_norm_models(monkeypatch, n=1, layers=7):
    """The layer list of the state-space / latent-attention / experts design at the sizes kernels_prenorm_stack.hip is written for: a model of separate launches and n
    of runs of sublayers.  Seven layers: runs of four, seven and one of two; attention in the third and the last."""
    from aha_amd import configs, configs_layered
    from aha_amd.model import HipInferenceModel
    from aha_amd.weights_layered import vamatar_weights
    t = configs.qwen3_0_6b()
    t.vocab_size = 2048
    cfg = configs_layered.vamatar_like(t, layers=layers)
    w = vamatar_weights(cfg, seed=3, device="cuda:0")
    monkeypatch.setenv("AHA_DECODE_STACK", "0")
    plain = HipInferenceModel(cfg, w)
    monkeypatch.setenv("AHA_DECODE_STACK", "1")
    return cfg, plain, [HipInferenceModel(cfg, w) for _ in range(n)]


@pytest.mark.parametrize("S", [1, 2, 3, 4, 70])
def test_runs_of_sublayers_against_separate_launches(gpu, monkeypatch, S):
    """Step by step from prompts with fewer tokens than taps on, past the turn of the histories (8): sums in f32 in another order, and features rounded to bf16 behind
    them, so a share of an ulp of theirs: a quarter of the bound of the stacks whose residual stream is bf16.  Then the same tokens by the device's loop."""
    cfg, plain, (m,) = pre_norm_models(monkeypatch)
    ids = ids_for(cfg, S + 20, 11)
    plain.forward_initial(ids[:S], 0)
    m.forward_initial(ids[:S], 0)
    before = m.debug_decode_stack()[0]
    for i in range(20):
        a, _ = plain.forward_step(ids[S + i], S + i)
        b, _ = m.forward_step(ids[S + i], S + i)
        std = float(a.std())
        assert np.isfinite(b).all() and float(np.abs(a - b).max()) <= LOGIT_TOL_STD * std and float(np.sqrt(((a - b) ** 2).mean())) <= LOGIT_RMS_STD / 4 * std, (S, i)
    assert m.debug_decode_stack() == (before + 20 * 2, 0)      # (a lone sublayer behind the last attention is separate launches)
    first = int(np.argmax(b))
    got = m.decode_greedy(first, S + 20, 12)
    last = m.last_logits()
    m.clear_cache()
    m.forward_initial(ids[:S], 0)
    for i in range(20):
        m.forward_step(ids[S + i], S + i)
    ref, tok = [], first
    for i in range(12):
        logits, tok = m.forward_step(tok, S + 20 + i)
        ref.append(int(tok))
    assert got == ref
    np.testing.assert_array_equal(last, logits)
    m.close(); plain.close()


def test_runs_that_give_up(gpu, monkeypatch):
    """A step and the device's loop with waves that may not ask even once: run again as separate launches, from the states and histories in front of the step.  Further
    sequences keep their states in place and never use the runs."""
    cfg, plain, ms = pre_norm_models(monkeypatch, 2)
    S = 30
    ids = ids_for(cfg, S + 3, 12)
    plain.forward_initial(ids[:S], 0)
    refs = [plain.forward_step(ids[S + i], S + i)[0] for i in range(3)]
    want = plain.decode_greedy(7, S + 3, 10)
    last = plain.last_logits()
    for m in ms:
        m.forward_initial(ids[:S], 0)
    ms[0].debug_decode_stack(0)
    for i in range(3):
        np.testing.assert_array_equal(ms[0].forward_step(ids[S + i], S + i)[0], refs[i])
    assert ms[0].debug_decode_stack() == (6, 3)
    assert ms[0].decode_greedy(7, S + 3, 10) == want
    np.testing.assert_array_equal(ms[0].last_logits(), last)

    for i in range(3):
        ms[1].forward_step(ids[S + i], S + i)
    ms[1].debug_decode_stack(0)
    assert len(ms[1].decode_greedy(7, S + 3, 10)) == 10
    assert ms[1].debug_decode_stack()[1] == 1
    close_to(last, ms[1].last_logits(), "behind steps that went well")

    steps = ms[1].debug_decode_stack(100000)[0]
    q = ms[1].seq_open()
    ms[1].forward_batch([(q, ids[:S], [S - 1])], want_logits=True)
    got, _ = ms[1].forward_batch([(q, [ids[S]], [0])], want_logits=True)
    close_to(refs[0], got[0], "a further sequence")
    assert ms[1].debug_decode_stack() == (steps, 1)
    ms[1].seq_close(q)
    for m in [plain] + ms:
        m.close()


def wide_models(monkeypatch, layers=2):
    from aha_amd.model import HipInferenceModel
    cfg = tiny_qwen3(layers=layers, hidden=4096, heads=32, kv_heads=8, inter=1024, vocab=512)
    w = qwen3_text_weights(cfg, seed=15)
    monkeypatch.setenv("AHA_DECODE_STACK", "0")
    plain = HipInferenceModel(cfg, w)
    monkeypatch.setenv("AHA_DECODE_STACK", "1")
    return cfg, plain, HipInferenceModel(cfg, w)


@pytest.mark.parametrize("scrambled", [False, True])
def test_attention_half_in_one_launch(gpu, monkeypatch, scrambled):
    """4096 columns: a layer's q k v, attention and o_proj in one launch (kernels_decode_attn.hip) give the bits of three.  No page behind the new token, pages' edges, one,
    three and four splits, units with two pages (up to 24 pages); splits of a page a wave, seven to sixteen of them, a page and two pages a block (33 and on); the last length that is
    taken (64 pages) and the first that is not."""
    cfg, plain, m = wide_models(monkeypatch)
    m.debug_scramble_pages(scrambled)
    for S in [1, 63, 64, 65, 255, 256, 257, 319, 320, 384, 448, 700, 1023, 1024, 1025, 1471, 1534, 1599, 1791, 2046, 2048, 2111, 3000, 4094]:
        ids = ids_for(cfg, S, 9 + S)
        m.clear_cache(); plain.clear_cache()
        _, tok = plain.forward_initial(ids, 0)
        m.forward_initial(ids, 0)
        before = m.debug_decode_stack()[0]
        for step in range(3):
            a, am = plain.forward_step(tok, S + step)
            b, _ = m.forward_step(tok, S + step)
            np.testing.assert_array_equal(a, b, err_msg=str((S, step)))
            tok = am
        assert m.debug_decode_stack() == (before + 2 * (2 if S == 4094 else 3), 0), S
    assert plain.debug_decode_stack()[0] == 0
    m.close(); plain.close()


def test_attention_half_that_gives_up(gpu, monkeypatch):
    """The same with waves that may not ask even once, in a single step and in the device's loop: run again as separate launches."""
    cfg, plain, m = wide_models(monkeypatch)
    ids = ids_for(cfg, 300, 4)
    _, tok = plain.forward_initial(ids, 0)
    m.forward_initial(ids, 0)
    ref, first = plain.forward_step(tok, 300)
    m.debug_decode_stack(0)
    np.testing.assert_array_equal(m.forward_step(tok, 300)[0], ref)
    assert m.debug_decode_stack() == (2, 1)
    m.debug_decode_stack(100000)
    want = plain.decode_greedy(first, 301, 12)
    assert m.decode_greedy(first, 301, 4) == want[:4]
    m.debug_decode_stack(0)
    assert m.decode_greedy(want[3], 305, 8) == want[4:]
    np.testing.assert_array_equal(m.last_logits(), plain.last_logits())
    assert m.debug_decode_stack()[1] == 2
    m.close(); plain.close()


@pytest.mark.parametrize("design, dtype", [("dense", "bfloat16"), ("post-norm", "bfloat16"), ("post-norm", "float32"), ("state-space", "bfloat16"), ("state-space", "float32")])
def test_device_loop_without_an_arg_max(gpu, design, dtype):
    """No logit is a number: the loop's steps, queued ahead of the host, embed a token that there is, and every token is reported as none (0xffffffff)."""
    from aha_amd.model import HipInferenceModel
    if design == "dense":
        cfg = tiny_qwen3(layers=2, hidden=256, heads=4, kv_heads=2, inter=512, vocab=512)
        w, norm = qwen3_text_weights(cfg, seed=1), "model.norm.weight"
    elif design == "post-norm":
        from tests import test_dosovik_gpu as t
        cfg = t.config([t.layer(), t.layer()], dtype=dtype)
        w, norm = t.dosovik_weights(cfg, seed=1), "final.norm"
    else:
        from tests import test_vamatar_gpu as t
        cfg = t.config([t.ssm(), t.att()], dtype=dtype)
        w, norm = t.vamatar_weights(cfg, seed=1), "final.norm"
    assert norm in w
    w[norm][:] = float("nan")
    m = HipInferenceModel(cfg, w)
    m.forward_initial([3, 1, 2], 0)
    assert m.decode_greedy(5, 3, 9) == [0xffffffff] * 9
    assert not np.isfinite(m.last_logits()).any()
    m.close()


def test_a_loop_that_ended_with_an_error_leaves_nothing(gpu, monkeypatch):
    """The device loop returns an error (one that an earlier call of the host's thread left) with steps queued that give up: the prompt behind it is a prompt, not a
    step to run again."""
    import ctypes
    cfg, plain, (m,) = models(monkeypatch)
    ids, other = ids_for(cfg, 70, 5), ids_for(cfg, 90, 6)
    _, tok = m.forward_initial(ids, 0)
    m.debug_decode_stack(0)
    assert ctypes.CDLL("libamdhip64.so").hipSetDevice(1000) != 0
    with pytest.raises(RuntimeError):
        m.decode_greedy(tok, 70, 12)
    m.debug_decode_stack(100000)
    m.clear_cache()
    want, tok = plain.forward_initial(other, 0)
    got, _ = m.forward_initial(other, 0)
    np.testing.assert_array_equal(got, want)
    close_to(plain.forward_step(tok, 90)[0], m.forward_step(tok, 90)[0], "the step behind")
    m.close(); plain.close()


def test_a_batch_that_ended_with_an_error_leaves_nothing(gpu, monkeypatch):
    """The same for a step of the state-space design: the next portion of a further sequence, whose states are updated in place, runs once."""
    import ctypes
    cfg, plain, (m,) = pre_norm_models(monkeypatch)
    ids = ids_for(cfg, 40, 7)
    seqs = {}
    for x in (plain, m):
        seqs[x] = x.seq_open()
        x.forward_batch([(seqs[x], ids[:20], [])])
    m.forward_initial(ids[:5], 0)
    m.debug_decode_stack(0)
    assert ctypes.CDLL("libamdhip64.so").hipSetDevice(1000) != 0
    with pytest.raises(RuntimeError):
        m.forward_step(ids[5], 5)
    m.debug_decode_stack(100000)
    want, got = (x.forward_batch([(seqs[x], ids[20:30], [9])])[0] for x in (plain, m))
    np.testing.assert_array_equal(got, want)
    m.close(); plain.close()


@pytest.mark.parametrize("hidden, heads, inter", [(1024, 16, 3072), (4096, 32, 1024)])
@pytest.mark.parametrize("polls", [0, 1, 3, 10, 40])
def test_what_gave_up_leaves_numbers(gpu, monkeypatch, polls, hidden, heads, inter):
    """Scores of hundreds, among them a new token's far below zero: a step that gives up joins splits that are not there, and what it and the steps queued behind
    it append lies on the pages that the step run again reads (with weight zero, which NaN survives).  Both one-launch forms of the dense stack."""
    from aha_amd.model import HipInferenceModel
    cfg = tiny_qwen3(layers=3, hidden=hidden, heads=heads, kv_heads=8, inter=inter, vocab=1024)
    w = qwen3_text_weights(cfg, seed=14)
    for k in w:
        if k.endswith(("q_norm.weight", "k_norm.weight")):
            w[k] = w[k] * 20
    monkeypatch.setenv("AHA_DECODE_STACK", "0")
    plain = HipInferenceModel(cfg, w)
    monkeypatch.setenv("AHA_DECODE_STACK", "1")
    launches = 3 if hidden == 4096 else 1
    for S in (70, 130, 200):
        m = HipInferenceModel(cfg, w)
        ids = ids_for(cfg, S, S)
        for _ in range(2):      # (the second time the exchange has values of the first)
            plain.clear_cache(); m.clear_cache()
            _, tok = plain.forward_initial(ids, 0)
            m.forward_initial(ids, 0)
            n, gone = m.debug_decode_stack(polls)
            want, got = plain.decode_greedy(tok, S, 8), m.decode_greedy(tok, S, 8)
            assert np.isfinite(m.last_logits()).all(), S
            after = m.debug_decode_stack()
            if hidden == 4096 or after == (n + 4 * launches, gone + 1):   # (the same bits in any case; or none of its four queued steps counted)
                assert got == want, S
                np.testing.assert_array_equal(m.last_logits(), plain.last_logits())
        m.close()
    plain.close()


def test_two_models_give_the_bits_of_one(gpu, monkeypatch):
    """Beside another model, its prompts and its steps, one that nobody has waited for among them, a model's steps take the form that they take alone: its logits and
    tokens are those of a model alone."""
    cfg, plain, (alone, *ms) = models(monkeypatch, 3)
    plain.close()
    prompts, fed = [ids_for(cfg, 50, 1), ids_for(cfg, 90, 2)], ids_for(cfg, 40, 3)

    def run(m, i):
        out = []
        for _ in range(3):
            m.clear_cache()
            _, tok = m.forward_initial(prompts[i], 0)
            out += [m.forward_step(t, len(prompts[i]) + k)[0] for k, t in enumerate(fed)]
            out.append(np.array(m.decode_greedy(tok, len(prompts[i]) + len(fed), 60)))
        m.forward_step_enqueue(5, len(prompts[i]) + len(fed) + 60)
        return out
    want, got = [run(alone, i) for i in range(2)], [None, None]
    steps = alone.debug_decode_stack()[0] // 2     # (and waits for it)
    ms[0].forward_initial(prompts[0], 0)
    ms[0].forward_step_enqueue(7, 50)

    def thread(i):
        got[i] = run(ms[i], i)
    threads = [threading.Thread(target=thread, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(2):
        assert len(got[i]) == len(want[i])
        for k, (a, b) in enumerate(zip(want[i], got[i])):
            np.testing.assert_array_equal(a, b, err_msg=str((i, k)))
    assert [m.debug_decode_stack() for m in ms] == [(steps + 1, 0), (steps, 0)]
    for m in [alone] + ms:
        m.close()


def test_a_model_that_gave_up_tries_again(gpu, monkeypatch):
    """Three steps that gave up: 16384 steps as separate launches, then one launch again; a fourth that gives up: as many again."""
    cfg, plain, (m,) = models(monkeypatch, vocab=256)
    plain.close()
    ids = ids_for(cfg, 30, 1)

    def steps(n):
        while n:
            m.clear_cache()
            _, tok = m.forward_initial(ids, 0)
            n -= len(m.decode_greedy(tok, len(ids), min(n, 500)))
    m.forward_initial(ids, 0)
    m.debug_decode_stack(0)
    for i in range(3):
        m.forward_step(5, len(ids) + i)
    assert m.debug_decode_stack(100000) == (3, 3)
    steps(16384)
    assert m.debug_decode_stack() == (3, 3)
    steps(5)
    assert m.debug_decode_stack(0) == (8, 3)
    m.clear_cache()
    m.forward_initial(ids, 0)
    m.forward_step(5, len(ids))
    assert m.debug_decode_stack(100000) == (9, 4)
    steps(700)
    assert m.debug_decode_stack() == (9, 4)
    m.close()


def test_profile_of_the_launches_that_run(gpu, monkeypatch):
    """A profiled step is the step without a profile: the same bits, the one-launch forms booked as classes of their own with the bytes of what they read."""
    def profiled(m, step, classes):
        m.set_profiling(True)
        step()
        m.set_profiling(False)
        return [m.get_profile(c) for c in classes]

    def near(p, elements, launches):
        assert p["launches"] == launches and 2 * elements <= p["bytes"] <= 1.02 * 2 * elements, p

    S, cache = 300, 301 * 2 * 1024                       # (of a layer)
    for make, layers, H, nq, inter, vocab in ((models, 3, 1024, 2048, 3072, 1024), (wide_models, 2, 4096, 4096, 1024, 512)):
        cfg, plain, m = make(monkeypatch)
        m = m[0] if isinstance(m, list) else m
        plain.close()
        ids = ids_for(cfg, S, 2)
        m.forward_initial(ids, 0)
        want, _ = m.forward_step(5, S)
        m.clear_cache()
        m.forward_initial(ids, 0)
        got = []
        stack, attn, gemv, separate = profiled(m, lambda: got.append(m.forward_step(5, S)[0]), ("decode_stack", "decode_attn", "gemv", "attn_decode"))
        np.testing.assert_array_equal(got[0], want)
        half, ff = H * (2 * nq + 2 * 1024), 3 * H * inter
        assert separate["launches"] == 0
        if make is models:
            near(stack, layers * (half + ff + cache), 1)
            near(gemv, vocab * H, 1)
            assert attn["launches"] == 0
        else:
            near(attn, layers * (half + cache), layers)
            near(gemv, layers * ff + vocab * H, 2 * layers + 1)
            assert stack["launches"] == 0
        m.close()

    cfg, plain, (m,) = pre_norm_models(monkeypatch)
    plain.close()
    ids = ids_for(cfg, 30, 2)
    m.forward_initial(ids, 0)
    (runs,) = profiled(m, lambda: m.forward_step(5, 30), ("decode_run",))
    assert runs["launches"] == 2 and runs["bytes"] > 0
    m.close()


@pytest.mark.parametrize("S, pages", [(700, (0, 1, 5, 10)), (2100, (0, 1, 31, 32)), (4159, (0, 32, 63, 64)), (6330, (2, 34, 66, 98)), (6300, (1, 33, 65, 97)),
                                      (32700, (30, 62, 94, 126)), (32700, (30, 286, 478, 510))])
def test_every_page_counts_once(gpu, monkeypatch, S, pages):
    """Four keys, one on each of four pages, take the whole weight of the new token's attention in every layer, a quarter each, and their values differ: without one
    of these pages, or with one twice, the logits are others.  A block's first, second and later pages, the first and the last page.  How: half of the columns of the
    residual stream never change; keys read those alone, queries the same in reverse order, values the rest; the dims that rotate visibly have no weight."""
    import dataclasses
    import torch
    from aha_amd.model import HipInferenceModel
    cfg = dataclasses.replace(tiny_qwen3(layers=3, hidden=1024, heads=16, kv_heads=8, inter=3072, vocab=1024), rope_theta=1e12)
    w = qwen3_text_weights(cfg, seed=21)
    emb, mid = w["model.embed_tokens.weight"], 512
    emb[1:5, :mid] = emb[1, :mid].clone()                  # tokens 1 to 4: the same key, four values
    emb[0, :mid] = emb[1, :mid].flip(0)                    # token 0: the query of that key
    for i in range(cfg.num_hidden_layers):
        p = f"model.layers.{i}."
        k = w[p + "self_attn.k_proj.weight"]
        k[:, mid:] = 0
        heads = k.view(8, 1, 128, 1024).expand(8, 2, 128, 1024).reshape(2048, 1024)
        w[p + "self_attn.q_proj.weight"] = torch.cat([heads[:, :mid].flip(1), heads[:, mid:]], 1).contiguous()
        w[p + "self_attn.v_proj.weight"][:, :mid] = 0
        w[p + "self_attn.o_proj.weight"][:mid] = 0
        w[p + "mlp.down_proj.weight"][:mid] = 0
        for n in ("q_norm", "k_norm"):                     # pairs 32 to 63 of the rotation: an angle of 0.03 at most; scores of 51 for the four, 6.4 of spread for others
            g = torch.zeros(128)
            g[32:64] = g[96:128] = 3.0
            w[p + f"self_attn.{n}.weight"] = g.bfloat16()
        w[p + "input_layernorm.weight"][:] = 1
    monkeypatch.setenv("AHA_DECODE_STACK", "0")
    plain = HipInferenceModel(cfg, w)
    monkeypatch.setenv("AHA_DECODE_STACK", "1")
    m = HipInferenceModel(cfg, w)
    ids = [5 + t % 1019 for t in ids_for(cfg, S, S + pages[1])]
    places = [p * 64 + (0, 63, 17, 40)[j] for j, p in enumerate(pages)]
    assert places[-1] < S
    for j, at in enumerate(places):
        ids[at] = 1 + j

    def step(x, ids):
        x.clear_cache()
        x.forward_initial(ids, 0, want_logits=False)
        return x.forward_step(0, S)[0]
    want = step(plain, ids)
    close_to(want, step(m, ids), (S, pages))
    assert m.debug_decode_stack() == (1, 0)
    for j, at in enumerate(places):                        # (what the test can see: without one of the four the logits are far outside the bound)
        other = step(plain, ids[:at] + [77 + j] + ids[at + 1:])
        assert float(np.sqrt(((want - other) ** 2).mean())) > 10 * LOGIT_RMS_STD * float(want.std()), (S, at)
    m.close(); plain.close()


@pytest.mark.parametrize("K", [512, 1024, 3072])
@pytest.mark.parametrize("what", ["normal", "wide", "cancelling"])
def test_dot_products_of_pairs(gpu, K, what):
    """The stack's dot products (two exact products at a time) against 64 bits: as close as a chain of fma over the same columns for weights and activations as a model
    has them and for sums that cancel to a hundredth (12 draws: 0.992 to 1.005 times).  Numbers over 24 octaves: the unit drops, downwards, what lies far below the
    largest of its three addends, 2 u at most, where two fma round to the nearest twice, u each: the same worst case, and sqrt(2) times the rms if every step did so
    (12 draws: 0.96 to 1.09)."""
    import ctypes
    import torch
    from aha_amd._lib import check, lib
    g = torch.Generator(device=gpu).manual_seed(K)
    N = 8192
    W, x = torch.randn(N, K, generator=g, device=gpu) * 0.02, torch.randn(K, generator=g, device=gpu)
    if what == "wide":
        W *= torch.exp2(torch.randint(-12, 12, (N, K), generator=g, device=gpu).float())
    if what == "cancelling":
        x[K // 2:] = x[:K // 2]
        W[:, K // 2:] = -W[:, :K // 2] + 0.01 * W[:, K // 2:]
    W, x = W.bfloat16(), x.bfloat16()
    exact, size = W.double() @ x.double(), W.double().abs() @ x.double().abs()
    off = []
    for chain in (0, 1):
        y = torch.empty(N, device=gpu)
        check(lib().aha_hip_debug_dot_bf16(W.data_ptr(), x.data_ptr(), y.data_ptr(), N, K, chain, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        torch.cuda.synchronize()
        off.append(float((((y.double() - exact) / size) ** 2).mean().sqrt()))
    # (rms over 8192 sums: drawn anew they differ by 1 %)
    assert off[0] <= (2 ** 0.5 if what == "wide" else 1.02) * off[1] and off[0] < 2 ** -24, off


def test_a_step_that_nobody_asked_for_holds_nobody_up(gpu, monkeypatch):
    """A model's queued step has run and is not asked for: the next step of another one, also where it would make way (4096 columns), takes the one launch."""
    import torch
    _, plain, (first,) = models(monkeypatch)
    cfg, plain2, wide = wide_models(monkeypatch)
    plain.close(); plain2.close()
    ids = ids_for(cfg, 40, 1)
    wide.forward_initial(ids, 0)
    first.forward_initial(ids, 0)
    first.forward_step_enqueue(3, 40)
    torch.cuda.synchronize()
    wide.forward_step(3, 40)
    assert wide.debug_decode_stack() == (2, 0)
    wide.close(); first.close()
