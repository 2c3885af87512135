"""-m gpu: D11 candidate extraction (aha_hip_sample_candidates / aha_hip_last_logits) against the oracle restatement of
candle's repeat penalty + top-k (oracle/sampling.py).  Selection is integer/compare work: indices and values bit-exact,
ordered by (value desc, index asc); the softmax normaliser is an f32 sum in a different order: relative 2e-5."""
import numpy as np
import pytest

from aha_amd import _lib
from aha_amd import sampling as hs
from aha_amd.configs import tiny_qwen3
from aha_amd.weights import qwen3_text_weights
from oracle import sampling as osamp

pytestmark = pytest.mark.gpu


def make(vocab):
    from aha_amd.model import HipInferenceModel
    cfg = tiny_qwen3(layers=1, hidden=256, heads=4, kv_heads=2, inter=512, vocab=vocab)
    return cfg, HipInferenceModel(cfg, qwen3_text_weights(cfg, seed=0))


@pytest.fixture(scope="module", params=[2048, 151936, 3000])
def model(gpu, request):
    cfg, m = make(request.param)
    yield cfg, m
    m.close()


def check_candidates(m, logits, ctx, pen, temp, k):
    vals, idx, mx, se = m.sample_candidates(ctx, pen, temp, k)
    ref_logits = osamp.apply_repeat_penalty(logits, pen, ctx) if pen != 1.0 else logits
    rv, ri, rmx, rse = osamp.topk_candidates(ref_logits, k, temp)
    np.testing.assert_array_equal(idx, ri)
    np.testing.assert_array_equal(vals.view(np.uint32), rv.view(np.uint32))
    assert np.float32(mx) == np.float32(rmx)
    assert abs(se - rse) <= 2e-5 * rse
    return vals, idx, mx, se


def test_state_and_argument_errors(gpu):
    cfg, m = make(1024)
    try:
        with pytest.raises(_lib.AhaHipError):  # no forward yet
            m.sample_candidates([], 1.0, 1.0, 4)
        with pytest.raises(_lib.AhaHipError):
            m.last_logits()
        m.forward_initial([1, 2, 3], 0, want_logits=False)
        for bad_k in (0, 65, -1):
            with pytest.raises(_lib.AhaHipError):
                m.sample_candidates([], 1.0, 1.0, bad_k)
        with pytest.raises(_lib.AhaHipError):
            m.sample_candidates([1], 0.0, 1.0, 4)  # non-positive penalty
    finally:
        m.close()


def test_candidates_match_oracle(model):
    cfg, m = model
    V = cfg.vocab_size
    g = np.random.default_rng(V)
    ids = [int(x) for x in g.integers(0, V, size=9)]
    logits, am = m.forward_initial(ids, 0)
    np.testing.assert_array_equal(m.last_logits().view(np.uint32), logits.view(np.uint32))
    top = [int(i) for i in np.argsort(-logits)[:6]]
    contexts = [[], top[:3] + top[:2] + [V + 5, 0xFFFFFFFF], [int(x) for x in g.integers(0, V, size=200)] + top]
    for ctx in contexts:
        for pen in (1.0, 1.1, 3.0):
            for temp, k in ((0.6, 20), (1.0, 64), (0.0, 1), (0.25, 7)):
                vals, idx, mx, se = check_candidates(m, logits, ctx, pen, temp, k)
    # arg-max of the unpenalised logits is the forward's token (first maximal index)
    assert check_candidates(m, logits, [], 1.0, 0.0, 1)[1][0] == am
    # a decode step replaces the logits the candidates come from
    logits2, _ = m.forward_step(am, len(ids))
    check_candidates(m, logits2, top, 1.3, 0.6, 20)
    m.clear_cache()


def test_ties_and_ordering(gpu):
    """Exact ties must come out in ascending index order."""
    cfg, m = make(2048)
    try:
        logits, _ = m.forward_initial([3, 4], 0)
        # an infinite penalty sends every non-negative logit to exactly 0: ~V/2 exact ties at the top
        ctx = [int(i) for i in np.nonzero(logits >= 0)[0]]
        assert len(ctx) > 200
        vals, idx, mx, se = m.sample_candidates(ctx, float("inf"), 1.0, 64)
        ref = osamp.apply_repeat_penalty(logits, float("inf"), ctx)
        rv, ri, _, rse = osamp.topk_candidates(ref, 64, 1.0)
        np.testing.assert_array_equal(idx, ri)
        np.testing.assert_array_equal(idx, np.sort(np.asarray(ctx, dtype=np.uint32))[:64])
        assert mx == 0.0 and abs(se - rse) <= 2e-5 * rse  # the untouched negative logits still carry mass
        assert all(vals[i] == 0.0 for i in range(64))
    finally:
        m.close()


def test_sampled_generation_distribution(gpu):
    """End to end through the host mirror: with top-k 20 / top-p 0.95 / T 0.6 every sampled token lies in the oracle's support
    for that step, and the loop's bookkeeping (offsets, cache) matches a replay with plain forward calls."""
    cfg, m = make(2048)
    try:
        prompt = [5, 6, 7, 8, 9]
        ctx = hs.GenerationContext(0.6, 0.95, 20, 1.2, 8, seed=11, initial_seq_len=len(prompt), max_tokens=12)
        toks = hs.generate_generic_sampled(m, prompt, ctx)
        assert len(toks) == 12
        s = osamp.Sampling("TopKThenTopP", float(np.float32(0.6)), k=20, p=float(np.float32(0.95)))
        logits, _ = m.forward_initial(prompt, 0)
        off = len(prompt)
        # ... and, beyond the support: the SAME tokens as an independent replay -- oracle probabilities (host f32 softmax over the
        # full logits), the k selected in the stated order (oracle.topk_order), the draw by the independent restatement of rand
        # 0.9.2's StdRng + WeightedIndex<f32> (oracle/rand_stdrng.py), one RNG stream for the whole sequence.  (Round-3 verdict,
        # weak #7: equality, not only support.  The device normaliser and the host softmax differ by ~1e-6 relative, so a uniform
        # draw within that distance of a bucket boundary could flip a token: 12 draws, fixed seed, deterministic on both sides.)
        from oracle import rand_stdrng as R
        ref_rng = R.StdRng.seed_from_u64(11)
        replay = []
        for i, t in enumerate(toks):
            pen = osamp.use_repeat_penalty(1.2, 8, logits, toks[:i])
            w = osamp.final_weights(pen, s)
            assert w[t] > 0, f"step {i}: token {t} outside the sampler's support"
            prs = osamp.softmax_last_dim(pen * np.float32(1.0 / s.temperature))
            keep = osamp.topk_order(prs, pen)[: s.k]
            replay.append(int(keep[R.sample_multinomial(ref_rng, w[keep])]))
            if i + 1 < len(toks):
                logits, _ = m.forward_step(t, off)
                off += 1
        assert replay == toks, f"device + host mirror {toks} vs independent replay {replay}"
        m.clear_cache()
        # same seed, same draws
        ctx = hs.GenerationContext(0.6, 0.95, 20, 1.2, 8, seed=11, initial_seq_len=len(prompt), max_tokens=12)
        assert hs.generate_generic_sampled(m, prompt, ctx) == toks
    finally:
        m.close()


def test_stream_loop_device_chunks_equal_host_loop(gpu):
    """generate_stream_generic_text over the C ABI: the greedy fast path (device-resident chunks of aha_hip_decode_greedy, one
    piece yielded per token) produces exactly the tokens of the host-driven generate_generic loop, for chunk sizes that do and
    do not divide the token count; the sampled path (top-k / top-p) streams the same tokens as generate_generic_sampled."""
    from aha_amd.model import generate_generic
    cfg, m = make(2048)
    try:
        ids = [int(x) for x in np.random.default_rng(3).integers(0, 2048, size=37)]
        want, _ = generate_generic(m, ids, 21)
        for chunk in (1, 4, 8, 64):
            ctx = hs.GenerationContext(0.0, None, None, None, None, seed=1, initial_seq_len=len(ids), max_tokens=21)
            got = [int(p) for p in hs.generate_stream_generic_text(m, lambda t: ",".join(map(str, t)), ids, ctx, device_chunk=chunk)]
            assert got == want, chunk
            assert m.cache_len() == 0
        a = hs.generate_generic_sampled(m, ids, hs.GenerationContext(0.7, 0.9, 20, 1.1, 16, seed=5, initial_seq_len=len(ids), max_tokens=12))
        ctx = hs.GenerationContext(0.7, 0.9, 20, 1.1, 16, seed=5, initial_seq_len=len(ids), max_tokens=12)
        b = [int(p) for p in hs.generate_stream_generic_text(m, lambda t: ",".join(map(str, t)), ids, ctx)]
        assert b[:len(a)] == a and len(b) in (len(a), len(a) + 1)   # the stream loop runs sample_len iterations, the generic one sample_len - 1 steps after the prefill
    finally:
        m.close()


@pytest.mark.parametrize("vocab", [64, 512, 513, 33000])
def test_where_the_candidates_lie(gpu, vocab):
    """An infinite penalty over all tokens but a few (non-negative logits become 0, the others -inf) puts the candidates where it is told: all in one
    wave's 512 entries, one in each of several waves, nowhere (zeros and -inf only), with vocabularies of fewer waves than k and of a partial last wave."""
    cfg, m = make(vocab)
    try:
        logits, _ = m.forward_initial([3, 4], 0)
        every = np.arange(vocab)
        last = every[(vocab - 1) // 512 * 512:]
        for keep in (every[:0], last, every[::509], every[-1:], every):
            ctx = [int(i) for i in np.setdiff1d(every, keep)]
            for k in (1, 20, 64):
                vals, idx, mx, se = m.sample_candidates(ctx, float("inf"), 1.0, k)
                ref = osamp.apply_repeat_penalty(logits, float("inf"), ctx) if ctx else logits
                rv, ri, rmx, rse = osamp.topk_candidates(ref, k, 1.0)
                np.testing.assert_array_equal(idx, ri)
                np.testing.assert_array_equal(vals.view(np.uint32), rv.view(np.uint32))
                assert np.float32(mx) == np.float32(rmx) and abs(se - rse) <= 2e-5 * rse
    finally:
        m.close()


@pytest.mark.parametrize("vocab,ks", [(513, (1, 20, 64)), (71681, (1, 2, 3)), (262144, (1, 20, 40)), (262145, (1, 20, 39))])
def test_a_wave_of_minus_infinity(gpu, vocab, ks):
    """A last wave of one entry that is -inf (vocabularies of 513 and 262145) adds nothing to the normaliser.  262144 entries are the most that the
    launches of topk_heads_kernel take, 262145 the fewest for the rounds over all candidates (whose second stage holds 20480: k <= 39 there); 71681
    are 141 waves, k = 2 the last that takes the rounds."""
    cfg, m = make(vocab)
    try:
        last = np.arange((vocab - 1) // 512 * 512, vocab)
        for seed in range(40):   # a prompt whose last logit is negative: an infinite penalty makes it -inf
            m.clear_cache()
            logits, _ = m.forward_initial([int(t) for t in np.random.default_rng(seed).integers(0, vocab, 3)], 0)
            if logits[-1] < 0:
                break
        neg = [int(i) for i in last[logits[last] < 0]]
        assert neg
        for ctx in ([neg[-1]], neg, [3, neg[-1], 5]):
            for k in ks:
                vals, idx, mx, se = m.sample_candidates(ctx, float("inf"), 0.9, k)
                rv, ri, rmx, rse = osamp.topk_candidates(osamp.apply_repeat_penalty(logits, float("inf"), ctx), k, 0.9)
                np.testing.assert_array_equal(idx, ri)
                np.testing.assert_array_equal(vals.view(np.uint32), rv.view(np.uint32))
                assert np.float32(mx) == np.float32(rmx) and abs(se - rse) <= 2e-5 * rse
        if vocab > 262144:
            with pytest.raises(_lib.AhaHipError):
                m.sample_candidates([], 1.0, 1.0, ks[-1] + 1)
    finally:
        m.close()


def test_enqueued_steps(gpu):
    """forward_step_enqueue leaves what forward_step computes: logits, cache and candidates are the same, over a page's end, with steps enqueued behind one
    another, and whatever call comes next waits for the step (another step, a prompt, clear_cache, last_hidden).  Tokens and offsets are checked alike."""
    cfg, m = make(3000)
    try:
        ids = [int(x) for x in np.random.default_rng(4).integers(0, 3000, size=120)]
        toks = [int(x) for x in np.random.default_rng(5).integers(0, 3000, size=12)]
        m.forward_initial(ids, 0, want_logits=False)
        want, hidden = [], []
        for i, t in enumerate(toks):
            want.append(m.forward_step(t, 120 + i)[0])
            hidden.append(m.debug_last_hidden())
        for every in (1, 3, 12):   # logits read after every so many steps
            m.clear_cache()
            m.forward_initial(ids, 0, want_logits=False)
            for i, t in enumerate(toks):
                m.forward_step_enqueue(t, 120 + i)
                if (i + 1) % every == 0:
                    np.testing.assert_array_equal(m.debug_last_hidden(), hidden[i])
                    check_candidates(m, want[i], [3, 5], 1.2, 0.8, 20)
                    np.testing.assert_array_equal(m.last_logits(), want[i])
        m.forward_step_enqueue(7, 132)
        m.clear_cache()
        assert m.cache_len() == 0
        m.forward_initial(ids, 0, want_logits=False)
        m.forward_step_enqueue(toks[0], 120)
        np.testing.assert_array_equal(m.forward_step(toks[1], 121)[0], want[1])
        with pytest.raises(_lib.AhaHipError):
            m.forward_step_enqueue(3000, 122)
        np.testing.assert_array_equal(m.forward_step(toks[2], 122)[0], want[2])
    finally:
        m.close()


@pytest.mark.parametrize("enqueue", [False, True])
def test_a_step_that_fails_behind_its_launches(gpu, enqueue):
    """An all-reduce that fails in the middle of a step: the step's logits are nobody's (those of the call before are overwritten by then), what was queued is
    waited for by the next call, and the model goes on from an empty cache."""
    from aha_amd.model import HipInferenceModel
    cfg = tiny_qwen3(layers=3, hidden=256, heads=4, kv_heads=2, inter=512, vocab=512)
    fail = []

    def summed(ptr, count):   # (one rank alone: its partial sums as they are)
        if fail and not fail.pop():
            raise RuntimeError("no partner")

    m = HipInferenceModel(cfg, qwen3_text_weights(cfg, seed=0), tp_rank=0, tp_size=2, allreduce=summed)
    try:
        def go():
            m.clear_cache()
            m.forward_initial([5, 6, 7], 0, want_logits=False)
            return m.forward_step(8, 3)[0]
        want = go()
        np.testing.assert_array_equal(m.last_logits(), want)
        fail += [False, True, True]   # the third of the step's sums
        with pytest.raises(_lib.AhaHipError):
            if enqueue:
                m.forward_step_enqueue(9, 4)
            else:
                m.forward_step(9, 4)
        assert not fail
        with pytest.raises(_lib.AhaHipError):
            m.last_logits()
        with pytest.raises(_lib.AhaHipError):
            m.sample_candidates([], 1.0, 1.0, 4)
        np.testing.assert_array_equal(go(), want)
        np.testing.assert_array_equal(m.last_logits(), want)
    finally:
        m.close()
