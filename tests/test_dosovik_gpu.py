"""Dosovik (csrc/layered.hip) on the GPU against the plain restatement of its equations (oracle/dosovik.py, float64): every mechanism through
the C ABI, prompts against decoding, portions, batches, pages and slots used again, greedy generation.  Tests make their own configurations and
weights; where random weights would hide a fault, one query / key pair is scaled so that its score stands out.

Tolerances: f32 mode -- rounding only (2e-5 of the logits' spread); bf16 mode -- matrix inputs rounded to bf16 (2^-9 relative) through a few
layers: rms 2 % of the logits' spread, and between two ways through the same layers 1.5 %."""
import numpy as np
import pytest
import torch

from aha_amd import _lib
from aha_amd.configs_layered import DosovikConfig, LayerConfig
from aha_amd.model import HipContext, HipInferenceModel, generate_generic
from aha_amd.weights_layered import dosovik_weights
from oracle import dosovik as od

pytestmark = pytest.mark.gpu

TOL = {"float32": 2e-5, "bfloat16": 2e-2}
TOL_SAME = {"float32": 2e-5, "bfloat16": 1.5e-2}


def layer(heads=6, kv_heads=2, dim=48, vdim=40, chunk=48, rope_dims=32, base=10000.0, scale=0.17, v_mix=True, ff=136):
    return LayerConfig(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, chunk=chunk, rope_dims=rope_dims, rope_base=base, scale=scale, v_mix=v_mix, ff=ff)


def config(layers, width=136, vocab=322, taps=3, alpha=1.7, scale=5.5, eps=1e-5, dtype="float32", eos=()):
    return DosovikConfig(hidden_size=width, vocab_size=vocab, layers=layers, embed_scale=scale, post_norm_alpha=alpha, conv_taps=taps, rms_norm_eps=eps,
                         eos_token_ids=list(eos), compute_dtype=dtype)


def tokens(n, vocab, seed=0):
    return torch.randint(0, vocab, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


def reference(cfg, w, ids):
    return od.forward(cfg.to_json(), {k: v.double() for k, v in w.items()}, ids).numpy()


def err(got, want):
    """rms over the vocabulary of the difference, mean taken off, over the spread of all wanted logits; the largest row"""
    d = np.atleast_2d(got) - np.atleast_2d(want)
    d = d - d.mean(-1, keepdims=True)
    return float(np.sqrt((d * d).mean(-1)).max() / want.std())


@pytest.fixture(scope="module")
def ctx(gpu):
    c = HipContext(0)
    yield c
    c.close()


class Model:
    def __init__(self, ctx, cfg, w):
        self.m = HipInferenceModel(cfg, w, ctx=ctx)

    def __enter__(self):
        return self.m

    def __exit__(self, *_):
        self.m.close()


def all_logits(m, ids, cuts=None):
    """logits of every position; cuts: portion lengths (their sum is len(ids))"""
    s = m.seq_open()
    out, at = [], 0
    for n in cuts or [len(ids)]:
        lg, _ = m.forward_batch([(s, ids[at:at + n], list(range(n)))])
        out.append(lg)
        at += n
    assert at == len(ids) and m.seq_len(s) == at
    m.seq_close(s)
    return np.concatenate(out)


VARIANTS = {
    # name: (layers, other config fields)
    "chunk smaller than a page": ([layer(chunk=20), layer(chunk=20)], {}),
    "chunk of one and of two": ([layer(chunk=1), layer(chunk=2)], {}),
    "chunks of several pages, differing": ([layer(chunk=192), layer(chunk=70), layer(chunk=128)], {}),
    "one head per kv head": ([layer(heads=3, kv_heads=3, dim=64, vdim=64)] * 2, {}),
    "one kv head": ([layer(heads=8, kv_heads=1, dim=32, vdim=32, rope_dims=32)] * 2, {}),
    "more than 16 heads per kv head": ([layer(heads=20, kv_heads=1, dim=32, vdim=16, rope_dims=16)] * 2, {}),
    "eight kv heads (xcd order)": ([layer(heads=16, kv_heads=8, dim=32, vdim=24, rope_dims=8)] * 2, {}),
    "wide heads": ([layer(heads=2, kv_heads=1, dim=160, vdim=200, rope_dims=100), layer(heads=4, kv_heads=2, dim=128, vdim=100, rope_dims=128)], {}),
    "very wide heads": ([layer(heads=2, kv_heads=1, dim=272, vdim=20, rope_dims=272)] * 2, {}),
    "odd sizes": ([layer(heads=5, kv_heads=5, dim=18, vdim=7, rope_dims=6, ff=77)] * 2, dict(width=99, vocab=103)),
    "values wider than keys": ([layer(dim=24, vdim=120, rope_dims=24)] * 2, {}),
    "full rotation, other base": ([layer(rope_dims=48, base=500.0), layer(rope_dims=16, base=31.0)], {}),
    "no rotation": ([layer(rope_dims=0)] * 2, {}),
    "no feed-forward in some layers": ([layer(ff=0), layer(), layer(ff=0)], {}),
    "no feed-forward at all": ([layer(ff=0), layer(ff=0)], {}),
    "value mixing starts late, skips": ([layer(v_mix=False), layer(), layer(v_mix=False), layer(), layer()], {}),
    "no value mixing": ([layer(v_mix=False)] * 2, {}),
    "one tap": ([layer()] * 2, dict(taps=1)),
    "two taps": ([layer()] * 2, dict(taps=2)),
    "six taps": ([layer()] * 2, dict(taps=6)),
    "large eps, alpha 1, embedding scale 1": ([layer(scale=0.4)] * 2, dict(eps=0.3, alpha=1.0, scale=1.0)),
    "rows of whole load groups": ([layer(heads=8, kv_heads=2, dim=64, vdim=64, ff=2048), layer(heads=16, kv_heads=4, dim=64, vdim=128, ff=1024, v_mix=False)], dict(width=1024)),
    "wide feed-forward of whole load groups": ([layer(heads=8, kv_heads=2, dim=64, vdim=64, ff=5120)], dict(width=1024)),
    "feed-forward of whole rounds of 32 x 64 tiles": ([layer(heads=8, kv_heads=2, dim=64, vdim=64, ff=9600)], dict(width=1024)),
    "wide rows": ([layer(heads=4, kv_heads=2, ff=2600)], dict(width=2100)),
}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", list(VARIANTS))
def test_prompt_and_decoding_follow_the_equations(ctx, name, dtype):
    """Whole prompt, and the same tokens half as a prompt and half one by one, against the restatement at every position."""
    layers, kw = VARIANTS[name]
    cfg = config(layers, dtype=dtype, **kw)
    w = dosovik_weights(cfg, seed=len(name))
    n = 70 if "rows" in name else 150
    ids = tokens(n, cfg.vocab_size, 1)
    want = reference(cfg, w, ids)
    with Model(ctx, cfg, w) as m:
        whole = all_logits(m, ids)
        half = all_logits(m, ids, [n // 2] + [1] * (n - n // 2))
    assert err(whole, want) <= TOL[dtype], name
    assert err(half, want) <= TOL[dtype], name
    assert err(half, whole) <= TOL_SAME[dtype], name


F32_HEADS = [   # heads, kv heads, dims, chunk, rotated dims: groups of 1, 2, 3 (no divisor of 16), 16 and 32 heads; chunks around 16 keys and a page
    (16, 8, 128, 150, 128), (4, 4, 64, 20, 64), (6, 2, 128, 1, 40), (16, 1, 64, 192, 0), (32, 1, 64, 33, 8), (4, 2, 128, 64, 64),
]


@pytest.mark.parametrize("heads,kv_heads,dim,chunk,rope_dims", F32_HEADS)
def test_32_bit_heads_of_whole_pieces(ctx, heads, kv_heads, dim, chunk, rope_dims):
    """attn_chunk_f32_kernel and qkv_post_f32_kernel: a prompt whose last tile is partly full, then token by token."""
    cfg = config([layer(heads=heads, kv_heads=kv_heads, dim=dim, vdim=dim, chunk=chunk, rope_dims=rope_dims)] * 2)
    w = dosovik_weights(cfg, seed=7)
    ids = tokens(211, cfg.vocab_size, 3)
    want = reference(cfg, w, ids)
    with Model(ctx, cfg, w) as m:
        assert err(all_logits(m, ids), want) <= TOL["float32"]
        assert err(all_logits(m, ids, [1, 130, 63] + [1] * 17), want) <= TOL["float32"]


@pytest.mark.parametrize("heads,kv_heads,dim,chunk,rope_dims,v_mix", [(8, 8, 128, 700, 128, True), (16, 8, 128, 600, 64, True), (12, 4, 64, 50, 0, False), (8, 2, 128, 300, 128, True),
                                                                      (16, 4, 64, 16, 32, True), (10, 2, 128, 300, 128, True), (32, 32, 128, 300, 128, False), (48, 24, 128, 300, 128, False)])
def test_32_bit_decoding_in_one_launch(ctx, heads, kv_heads, dim, chunk, rope_dims, v_mix):
    """One token each of sequences that end around 16 keys, a page and a round of 128 or 256 keys, the first token among them; groups of 1 to 4 heads, five
    heads, 8192 columns of q and k and more of them in the launches they had."""
    cfg = config([layer(heads=heads, kv_heads=kv_heads, dim=dim, vdim=dim, chunk=chunk, rope_dims=rope_dims, v_mix=v_mix)] * 2)
    w = dosovik_weights(cfg, seed=17)
    ids = tokens(560, cfg.vocab_size, 18)
    want = reference(cfg, w, ids)
    at = [0, 1, 15, 16, 17, 63, 64, 127, 128, 255, 256, 257, 513, 559]
    with Model(ctx, cfg, w) as m:
        seqs = [m.seq_open() for _ in at]
        for s, p in zip(seqs, at):
            if p:
                m.forward_batch([(s, ids[:p], [])])
        got, _ = m.forward_batch([(s, ids[p:p + 1], [0]) for s, p in zip(seqs, at)])
        assert err(got, want[at]) <= TOL["float32"]
        for k in range(3):   # on from the keys and values that the launch appended, alone
            one, _ = m.forward_batch([(seqs[4], ids[18 + k:19 + k], [0])])
            assert err(one, want[18 + k:19 + k]) <= TOL["float32"]


@pytest.mark.parametrize("rows,ff,vocab", [(8, 2624, 24600), (16, 2624, 322), (20, 2624, 24600), (32, 2624, 322), (33, 2624, 322), (65, 2624, 322), (97, 2624, 322),
                                           (150, 2624, 322), (300, 2624, 322), (500, 2624, 322), (257, 4160, 322)])
def test_32_bit_products_of_every_tile(ctx, rows, ff, vocab):
    """gemm_f32_kernel and gemm_f32_few_kernel: every tile and row count that launch_gemm_f32 chooses between, K of five chunks (no multiple of the chunks of a
    stage), columns that are no multiple of the eight column tiles that the XCDs take in turn; against 64 bits."""
    cfg = config([layer(heads=4, kv_heads=2, dim=64, vdim=64, chunk=600, rope_dims=64, ff=ff)], width=320, vocab=vocab)
    w = dosovik_weights(cfg, seed=11)
    ids = tokens(rows, vocab, 12)
    want = reference(cfg, w, ids)
    with Model(ctx, cfg, w) as m:
        assert err(all_logits(m, ids), want) <= TOL["float32"]


@pytest.mark.parametrize("width,ff", [(1024, 1536), (1030, 1599), (832, 4100), (2048, 12288)])
@pytest.mark.parametrize("rows", [2, 7, 8, 9, 16, 17])
def test_polynorm_between_few_row_products(ctx, width, ff, rows):
    """2 to 16 rows at once, 17 by the launch of its own; part blocks, pad columns and rows that a fragment does not fill.  Each row against the restatement."""
    cfg = config([layer(heads=4, kv_heads=2, dim=64, vdim=64, ff=ff)] * 2, width=width, dtype="bfloat16")
    w = dosovik_weights(cfg, seed=31)
    ids = [tokens(3, cfg.vocab_size, seed=40 + i) for i in range(rows)]
    with Model(ctx, cfg, w) as m:
        seqs = [m.seq_open() for _ in range(rows)]
        m.forward_batch([(s, x[:2], []) for s, x in zip(seqs, ids)])
        got, _ = m.forward_batch([(s, x[2:], [0]) for s, x in zip(seqs, ids)])
    want = np.stack([reference(cfg, w, x)[-1] for x in ids])
    assert err(got, want) <= TOL["bfloat16"]


# PolyNorm inside the two products around it: (width, ff, rows, weight rows per block of the up product, of the down product).  Every block width of either product
# with one group of eight rows and with two (from 64 MB on, csrc/kernels_gemm.hip gemm_takes_poly), pad columns among them.
POLY = [(1030, 1599, 2, 16, 16), (1024, 6208, 7, 32, 16), (832, 4100, 8, 24, 16), (768, 8256, 8, 48, 16), (4130, 1536, 8, 16, 24), (6210, 1536, 5, 16, 32), (4096, 12288, 9, 48, 16), (4096, 8192, 16, 32, 16),
        (8190, 4096, 16, 16, 32), (6100, 5504, 13, 24, 24)]


@pytest.mark.parametrize("width,ff,rows,up,down", POLY)
def test_polynorm_inside_every_form_of_the_products(ctx, width, ff, rows, up, down):
    """The launch has to be the fused pair, of the block widths named; each row against the restatement."""
    assert {_lib.lib().aha_hip_debug_poly_plan(rows, -(-width // 256) * 256, -(-ff // 64) * 64, ws) for ws in (0, 32 << 20, 96 << 20)} == {up | down << 8}
    cfg = config([layer(heads=2, kv_heads=1, dim=64, vdim=64, ff=ff)], width=width, vocab=130, taps=3 if width < 2048 else 1, dtype="bfloat16")
    w = dosovik_weights(cfg, seed=33)
    ids = [tokens(2, cfg.vocab_size, seed=60 + i) for i in range(rows)]
    with Model(ctx, cfg, w) as m:
        seqs = [m.seq_open() for _ in range(rows)]
        m.forward_batch([(s, x[:1], []) for s, x in zip(seqs, ids)])
        got, _ = m.forward_batch([(s, x[1:], [0]) for s, x in zip(seqs, ids)])
    want = np.stack([reference(cfg, w, x)[-1] for x in ids])
    assert err(got, want) <= TOL["bfloat16"]


@pytest.mark.parametrize("dim", [64, 128])
def test_32_bit_rows_do_not_see_a_later_row_that_is_not_finite(ctx, dim):
    cfg = config([layer(heads=8, kv_heads=4, dim=dim, vdim=dim, chunk=100, rope_dims=dim)] * 2)
    w = dosovik_weights(cfg, seed=8)
    last = cfg.vocab_size - 1
    w["embed"][last] = float("inf")
    ids = [t % last for t in tokens(75, cfg.vocab_size, 4)]
    want = reference(cfg, w, ids)
    with Model(ctx, cfg, w) as m:
        got = all_logits(m, ids + [last])
        assert err(got[:-1], want) <= TOL["float32"] and not np.isfinite(got[-1]).all()
        assert err(all_logits(m, ids), want) <= TOL["float32"]   # (in pages that hold that row)


@pytest.mark.parametrize("heads,kv_heads,chunk", [(16, 8, 8192), (14, 2, 192), (8, 8, 20), (32, 8, 64), (1, 1, 100), (16, 2, 192)])
def test_decoding_with_whole_heads_of_128(ctx, heads, kv_heads, chunk):
    """attn_chunk_decode_kernel's LEAN form (eight query heads per kv head: the other one), two sequences token by token and one alone, several pages per
    unit and units without any, chunk edges on the way."""
    cfg = config([layer(heads=heads, kv_heads=kv_heads, dim=128, vdim=128, chunk=chunk, rope_dims=128, scale=0.09)] * 3, dtype="bfloat16")
    w = dosovik_weights(cfg, seed=9)
    a, b = tokens(420, cfg.vocab_size, 5), tokens(90, cfg.vocab_size, 6)
    want_a, want_b = reference(cfg, w, a), reference(cfg, w, b)
    with Model(ctx, cfg, w) as m:
        assert err(all_logits(m, a, [380] + [1] * 40), want_a) <= TOL["bfloat16"]
        s, t = m.seq_open(), m.seq_open()
        m.forward_batch([(s, a[:395], [394]), (t, b[:57], [56])])
        got = [m.forward_batch([(s, [a[395 + i]], [0]), (t, [b[57 + i]], [0])])[0] for i in range(25)]
        m.seq_close(s)
        m.seq_close(t)
    assert err(np.stack([g[0] for g in got]), want_a[395:420]) <= TOL["bfloat16"]
    assert err(np.stack([g[1] for g in got]), want_b[57:82]) <= TOL["bfloat16"]


def neutral(cfg, seed):
    """Weights under which every mechanism but the projections is switched off: no convolution, unit norms, no biases, no mixing, act = N(z)."""
    w = dosovik_weights(cfg, seed=seed)
    for n, t in w.items():
        if "canon" in n or n.endswith((".b", "norm1", "norm2", "vmix")) or n == "final.norm":
            w[n] = torch.zeros_like(t)
        elif n.endswith((".q.norm", ".k.norm")):
            w[n] = torch.ones_like(t)
        elif n.endswith("mlp.act"):
            w[n] = torch.tensor([1.0, 0.0, 0.0, 0.0]).bfloat16()
    return w


NEUTRAL = dict(chunk=1000, rope_dims=0, scale=0.3)
MECHANISMS = {
    # name: (layer fields, config fields, weights taken from the random set)
    "nothing": ({}, {}, ()),
    "mixer convolution": ({}, {}, ("canon1",)),
    "feed-forward convolution": ({}, {}, ("canon2",)),
    "zero-centred norms": ({}, {}, ("norm1", "norm2", "final.norm")),
    "post-norm alpha": ({}, dict(alpha=3.25), ()),
    "embedding scale": ({}, dict(scale=0.75), (".b",)),     # (without biases the normed stack does not see it)
    "eps": ({}, dict(eps=0.5), ()),
    "biases": ({}, {}, (".b",)),
    "query and key norm weights": ({}, {}, (".q.norm", ".k.norm")),
    "rotation": (dict(rope_dims=48, base=50.0), {}, ()),
    "rotation of a part": (dict(rope_dims=16, base=50.0), {}, ()),
    "chunks": (dict(chunk=13), {}, ()),
    "score scale": (dict(scale=0.05), {}, ()),
    "value mixing": ({}, {}, ("vmix",)),
    "second power": ({}, {}, {"mlp.act": (0.0, 1.0, 0.0, 0.0)}),
    "third power": ({}, {}, {"mlp.act": (0.0, 0.0, 1.0, 0.0)}),
    "constant": ({}, {}, {"mlp.act": (1.0, 0.0, 0.0, 2.5)}),
}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", list(MECHANISMS))
def test_one_mechanism_at_a_time(ctx, name, dtype):
    """Everything else neutral; the mechanism's effect on the logits is large against the tolerance, so that leaving it out would show."""
    lk, ck, ws = MECHANISMS[name]
    base = config([layer(**NEUTRAL)] * 2, dtype=dtype)
    cfg = config([layer(**{**NEUTRAL, **lk})] * 2, dtype=dtype, **ck)
    w0 = neutral(base, 30)
    w, full = dict(w0), dosovik_weights(base, seed=30)
    for n in w:
        if isinstance(ws, dict):
            for end, v in ws.items():
                if n.endswith(end):
                    w[n] = torch.tensor(v).bfloat16()
        elif n.endswith(tuple(ws)) and ws:
            w[n] = full[n]
    ids = tokens(80, cfg.vocab_size, 31)
    want = reference(cfg, w, ids)
    with Model(ctx, cfg, w) as m:
        assert err(all_logits(m, ids), want) <= TOL[dtype]
        assert err(all_logits(m, ids, [30, 2, 8] + [1] * 40), want) <= TOL[dtype]
    if name != "nothing":
        assert err(reference(base, w if ck else w0, ids), want) > 3 * TOL[dtype]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_residual_stream_after_every_layer(ctx, dtype):
    cfg = config([layer(), layer(ff=0), layer(chunk=64)], dtype=dtype)
    w = dosovik_weights(cfg, seed=3)
    ids = tokens(90, cfg.vocab_size, 3)
    ref = []
    od.forward(cfg.to_json(), {k: v.double() for k, v in w.items()}, ids, ref)
    with Model(ctx, cfg, w) as m:
        m.debug_keep_residual()
        s = m.seq_open()
        m.forward_batch([(s, ids[:-1], [])])
        got = [m.debug_residual(i) for i in range(3)]
        m.forward_batch([(s, ids[-1:], [])])
        last = [m.debug_residual(i) for i in range(3)]
    for i in range(3):
        full = np.concatenate([got[i], last[i]])
        assert np.abs(full - ref[i].numpy()).max() <= (2e-5 if dtype == "float32" else 0.08), i


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("cuts", [[2] * 65, [1] * 130, [3, 61, 2, 2, 62], [64, 64, 2], [63, 2, 65], [1, 129], [7] * 18 + [4]])
def test_portions_do_not_change_the_logits(ctx, dtype, cuts):
    cfg = config([layer(chunk=50), layer(chunk=64), layer(chunk=100, ff=0)], taps=4, dtype=dtype)
    w = dosovik_weights(cfg, seed=5)
    ids = tokens(130, cfg.vocab_size, 5)
    want = reference(cfg, w, ids)
    with Model(ctx, cfg, w) as m:
        assert err(all_logits(m, ids, cuts), want) <= TOL[dtype]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_unequal_requests_in_one_batch_against_each_alone(ctx, dtype):
    """Prompts of different lengths (one token to several pages) in one step, decoded together, the shorter ones ending earlier; pages handed out
    in a scrambled order, slots and pages of finished requests used again by the next batch."""
    cfg = config([layer(chunk=40), layer(chunk=128)], dtype=dtype)
    w = dosovik_weights(cfg, seed=7)
    lens = [1, 130, 64, 65, 2, 17, 200]
    with Model(ctx, cfg, w) as m:
        m.debug_scramble_pages(True)
        for rnd in range(2):
            ids = [tokens(n + 12, cfg.vocab_size, 10 * rnd + i) for i, n in enumerate(lens)]
            alone = [all_logits(m, x) for x in ids]
            seqs = [m.seq_open() for _ in ids]
            lg, _ = m.forward_batch([(s, x[:n], list(range(n))) for s, x, n in zip(seqs, ids, lens)])
            at, got = 0, []
            for n in lens:
                got.append([lg[at:at + n]])
                at += n
            live = list(range(len(lens)))
            for step in range(12):
                lg, am = m.forward_batch([(seqs[i], [ids[i][lens[i] + step]], [0]) for i in live], want_argmax=True)
                assert (am == lg.argmax(-1)).all()
                for k, i in enumerate(live):
                    got[i].append(lg[k:k + 1])
                for i in [i for i in live if i % 3 == step % 3 and step > 5]:
                    m.seq_close(seqs[i])
                    live.remove(i)
                if not live:
                    break
            for i in live:
                m.seq_close(seqs[i])
            for i, g in enumerate(got):
                g = np.concatenate(g)
                assert err(g, alone[i][:len(g)]) <= TOL_SAME[dtype], (rnd, i)
                assert err(g, reference(cfg, w, ids[i])[:len(g)]) <= TOL[dtype], (rnd, i)


def test_portions_of_different_sizes_and_single_tokens_share_a_step(ctx):
    """One step with a first prompt, a continued one and a single decoded token."""
    cfg = config([layer(chunk=33), layer(chunk=64)], dtype="bfloat16")
    w = dosovik_weights(cfg, seed=8)
    a, b, c = (tokens(n, cfg.vocab_size, n) for n in (90, 140, 61))
    with Model(ctx, cfg, w) as m:
        sa, sb, sc = (m.seq_open() for _ in range(3))
        m.forward_batch([(sb, b[:65], []), (sc, c[:60], [])])
        lg, _ = m.forward_batch([(sa, a, [89]), (sb, b[65:], [0, 74]), (sc, c[60:], [0])])
    want = np.stack([reference(cfg, w, a)[89], reference(cfg, w, b)[65], reference(cfg, w, b)[139], reference(cfg, w, c)[60]])
    assert err(lg, want) <= TOL["bfloat16"]


def spotlight(cfg, w, key_pos, n, layer_index=0):
    """Weights and ids under which one token's key answers one query: token A's key row and token B's query row point the same way with a large
    score, so that B's output changes visibly if (and only if) A's position is visible.  One layer, no rotation, no convolution (one tap)."""
    mx = f"l{layer_index}.mix."
    l = cfg.layers[layer_index]
    A, B, rest = 0, 1, 2
    ids = [rest + (i * 7) % (cfg.vocab_size - 2) for i in range(n)]
    ids[key_pos] = A
    emb = torch.randn(cfg.vocab_size, cfg.hidden_size, generator=torch.Generator().manual_seed(99)) * 0.3
    emb[:, :2] = 0
    emb[A, 0] = 20.0
    emb[B, 1] = 20.0
    w["embed"] = emb.bfloat16()
    wq, wk = w[mx + "q"].float() * 0.1, w[mx + "k"].float() * 0.1
    for h in range(l.heads):
        wq[h * l.dim, 1] = 40.0
    for g in range(l.kv_heads):
        wk[g * l.dim, 0] = 40.0
    wv = w[mx + "v"].float()
    wv[:, 0] *= 5
    w[mx + "q"], w[mx + "k"], w[mx + "v"] = wq.bfloat16(), wk.bfloat16(), wv.bfloat16()
    w["l0.canon1"] = torch.zeros_like(w["l0.canon1"])
    return ids, A, B


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("chunk,query", [(48, 95), (48, 96), (64, 63), (64, 64), (64, 127), (64, 128), (100, 99), (100, 100), (192, 191), (192, 192)])
@pytest.mark.parametrize("how", ["prompt", "decoded"])
def test_one_key_at_an_edge(ctx, dtype, chunk, query, how):
    """A key that stands out, at the first position of the query's chunk (visible) and at the position just before it (not visible), queries at a
    chunk's last and first positions: the output moves with the first and not with the second, in prompts and in decoding."""
    cfg = config([layer(heads=4, kv_heads=2, dim=32, vdim=32, chunk=chunk, rope_dims=0, scale=0.25, v_mix=False, ff=64)], taps=1, dtype=dtype)
    lo = query // chunk * chunk
    outs = {}
    for where, kp in (("in", lo), ("out", lo - 1), ("none", None)):
        if kp is not None and (kp < 0 or kp == query):
            continue
        w = dosovik_weights(cfg, seed=11)
        ids, A, B = spotlight(cfg, w, kp if kp is not None else 0, query + 1)
        if kp is None:
            ids[0] = 5
        ids[query] = B
        want = reference(cfg, w, ids)
        with Model(ctx, cfg, w) as m:
            got = all_logits(m, ids) if how == "prompt" else all_logits(m, ids, [query, 1])
        assert err(got, want) <= TOL[dtype]
        outs[where] = (got[query], want[query])
    spread = outs["none"][1].std()
    if "in" in outs:      # the planted key is seen ...
        assert np.abs(outs["in"][0] - outs["none"][0]).max() > 0.2 * spread
    if "out" in outs:     # ... and its neighbour on the other side of the edge is not: the same logits to rounding
        assert np.abs(outs["out"][0] - outs["none"][0]).max() < (1e-3 if dtype == "float32" else 0.05) * spread


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_far_key_among_thousands(ctx, dtype):
    """One visible key 1400 positions back inside a chunk of 2048 (22 pages, several decode splits), the same key moved to page borders."""
    cfg = config([layer(heads=4, kv_heads=2, dim=64, vdim=48, chunk=2048, rope_dims=0, scale=0.125, v_mix=False, ff=64)], taps=1, dtype=dtype)
    n = 1500
    outs = []
    for kp in (0, 63, 64, 99, n - 2):
        w = dosovik_weights(cfg, seed=12)
        ids, A, B = spotlight(cfg, w, kp, n)
        ids[-1] = B
        with Model(ctx, cfg, w) as m:
            s = m.seq_open()
            m.forward_batch([(s, ids[:-1], [])])
            dec, _ = m.forward_batch([(s, ids[-1:], [0])])
            t = m.seq_open()
            pro, _ = m.forward_batch([(t, ids, [n - 1])])
        x = reference(cfg, w, ids)[-1:]
        assert err(dec, x) <= TOL[dtype] and err(pro, x) <= TOL[dtype], kp
        outs.append(dec[0])
    spread = outs[0].std()
    for o in outs[1:]:
        assert np.abs(o - outs[0]).max() < 0.3 * spread     # wherever the key is, it is found


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_the_sink_takes_its_share(ctx, dtype):
    """Scores far below and far above zero: with the sink the first drive the attention output to (near) zero, the second ignore the sink.  The
    planted mistake -- a softmax without the added one -- lives in the restatement and must differ from the device."""
    for qb in (-6.0, 6.0):
        cfg = config([layer(heads=4, kv_heads=2, dim=32, vdim=32, chunk=64, rope_dims=0, scale=0.2, v_mix=False, ff=0)], taps=1, dtype=dtype)
        w = dosovik_weights(cfg, seed=13)
        w["l0.mix.q.b"] = torch.full_like(w["l0.mix.q.b"], qb)
        w["l0.mix.k.b"] = torch.full_like(w["l0.mix.k.b"], 6.0)
        ids = tokens(80, cfg.vocab_size, 13)
        want = reference(cfg, w, ids)
        keep = od.softmax_sink
        try:
            od.softmax_sink = lambda s: torch.softmax(s, -1)
            wrong = reference(cfg, w, ids)
        finally:
            od.softmax_sink = keep
        with Model(ctx, cfg, w) as m:
            got = all_logits(m, ids, [40] + [1] * 40)
        assert err(got, want) <= TOL[dtype]
        if qb < 0:
            assert err(got, wrong) > 5 * TOL[dtype]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_first_tokens_of_a_sequence(ctx, dtype):
    cfg = config([layer()] * 2, taps=5, dtype=dtype)
    w = dosovik_weights(cfg, seed=14)
    ids = tokens(9, cfg.vocab_size, 14)
    want = reference(cfg, w, ids)
    with Model(ctx, cfg, w) as m:
        for n in range(1, 9):
            assert err(all_logits(m, ids[:n], [1] * n), want[:n]) <= TOL[dtype]
            assert err(all_logits(m, ids[:n]), want[:n]) <= TOL[dtype]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_decoding_gives_passed_pages_back(ctx, dtype):
    """400 decoded tokens with chunks of 64 and 96: pages in front of both chunks return to the pool, the logits keep following the equations."""
    cfg = config([layer(chunk=64), layer(chunk=96)], dtype=dtype)
    w = dosovik_weights(cfg, seed=15)
    ids = tokens(420, cfg.vocab_size, 15)
    want = reference(cfg, w, ids)
    with Model(ctx, cfg, w) as m:
        s = m.seq_open()
        m.forward_batch([(s, ids[:20], [])])
        rows, most = [], 0
        for t in ids[20:]:
            lg, _ = m.forward_batch([(s, [t], [0])])
            rows.append(lg)
            most = max(most, m.seq_pages(s))
        assert most <= 3
        assert err(np.concatenate(rows), want[20:]) <= TOL[dtype]
        m.seq_close(s)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_greedy_generation_by_every_loop(ctx, dtype):
    """generate_generic step by step, its device-resident loop, and the batch loop: the same tokens as stepping the restatement (margins of the
    arg-max above the rounding, so the sequence is determined)."""
    from aha_amd.scheduler import Request, generate_batch
    cfg = config([layer(chunk=32), layer(chunk=64)], dtype=dtype)
    w = dosovik_weights(cfg, seed=16)
    w["head"] = (w["head"].float() * 8).bfloat16()
    prompts = [tokens(n, cfg.vocab_size, 20 + n) for n in (5, 50, 33)]
    want = []
    for p in prompts:
        ids, margin = list(p), []
        for _ in range(40):
            lg = reference(cfg, w, ids)[-1]
            top = np.sort(lg)[-2:]
            margin.append((top[1] - top[0]) / lg.std())
            ids.append(int(lg.argmax()))
        safe = next((i for i, x in enumerate(margin) if x < (1e-3 if dtype == "float32" else 0.08)), 40)
        want.append(ids[len(p):len(p) + safe])
    assert sum(len(x) for x in want) > 10
    with Model(ctx, cfg, w) as m:
        outs = generate_batch(m, [Request(p, max_tokens=40) for p in prompts])
        for p, x, o in zip(prompts, want, outs):
            a, _ = generate_generic(m, p, 40)
            b, _ = generate_generic(m, p, 40, device_loop=True)
            assert a[:len(x)] == x and b[:len(x)] == x and o[:len(x)] == x
            if dtype == "float32":
                assert a == b
        assert m.cache_len() == 0


def test_device_loop_stops_at_a_stop_token_and_continues_cleanly(ctx):
    """The loop runs ahead of the host; after a stop token the state must be that of the last kept token."""
    cfg = config([layer(chunk=32), layer(chunk=64)], dtype="bfloat16")
    w = dosovik_weights(cfg, seed=17)
    p = tokens(30, cfg.vocab_size, 17)
    with Model(ctx, cfg, w) as m:
        free, _ = generate_generic(m, p, 30, device_loop=True)
    stop = free[12]
    first = free.index(stop)
    if first < 2:
        pytest.skip("the generated sequence repeats its first tokens")
    cfg2 = config([layer(chunk=32), layer(chunk=64)], dtype="bfloat16", eos=[stop])
    with Model(ctx, cfg2, w) as m:
        _, t0 = m.forward_initial(p, 0, want_logits=False)
        out = m.decode_greedy(t0, len(p), 29)
        assert [t0] + out == free[:first + 1]
        assert m.cache_len() == len(p) + len(out)
        lg, _ = m.forward_step(out[-1], m.cache_len())
        ids = p + [t0] + out
        fresh = m.seq_open()
        ref, _ = m.forward_batch([(fresh, ids, [len(ids) - 1])])
        assert err(lg, ref) <= TOL_SAME["bfloat16"]


def test_sampling_on_batch_rows(ctx):
    """sample_candidates works on the row of the batch that select_logits picked."""
    cfg = config([layer()] * 2, dtype="bfloat16")
    w = dosovik_weights(cfg, seed=18)
    with Model(ctx, cfg, w) as m:
        seqs = [m.seq_open() for _ in range(3)]
        lg, am = m.forward_batch([(s, tokens(10 + i, cfg.vocab_size, i), [9 + i]) for i, s in enumerate(seqs)], want_argmax=True)
        for i in range(3):
            m.select_logits(i)
            vals, idx, mx, _ = m.sample_candidates([], 1.0, 1.0, 5)
            order = np.argsort(-lg[i], kind="stable")[:5]
            assert idx.tolist() == order.tolist() and idx[0] == am[i] and abs(mx - lg[i].max()) < 1e-6
            assert np.array_equal(m.last_logits(), lg[i])
        with pytest.raises(Exception):
            m.select_logits(3)


def test_sampled_batch_equals_sampled_alone(ctx):
    from aha_amd.sampling import GenerationContext, generate_generic_sampled
    from aha_amd.scheduler import Request, generate_batch
    cfg = config([layer(chunk=32), layer(chunk=64)], dtype="float32")
    w = dosovik_weights(cfg, seed=19)
    prompts = [tokens(n, cfg.vocab_size, 30 + n) for n in (4, 40)]

    def gctx(i, n):
        return GenerationContext(0.8, 0.9, 20, 1.1, 64, 100 + i, n, 12)
    with Model(ctx, cfg, w) as m:
        alone = [generate_generic_sampled(m, p, gctx(i, len(p))) for i, p in enumerate(prompts)]
        both = generate_batch(m, [Request(p, max_tokens=12, ctx=gctx(i, len(p))) for i, p in enumerate(prompts)])
    assert both == alone


def test_errors_are_refused(ctx):
    cfg = config([layer()] * 2, dtype="bfloat16")
    w = dosovik_weights(cfg, seed=20)
    from aha_amd._lib import AhaHipError
    with Model(ctx, cfg, w) as m:
        s = m.seq_open()
        for bad in ([(s + 5, [1], [])], [(s, [], [])], [(s, [cfg.vocab_size], [])], [(s, [1], [1])], [(s, [1], []), (s, [2], [])], []):
            with pytest.raises(AhaHipError):
                m.forward_batch(bad)
        assert m.seq_len(s) == 0
        with pytest.raises(AhaHipError):
            m.forward_initial([1, 2], 3)
        m.seq_close(s)
        with pytest.raises(AhaHipError):
            m.seq_close(s)
    bad = dict(w)
    del bad["l1.mix.k.norm"]
    with pytest.raises(AhaHipError):
        HipInferenceModel(cfg, bad, ctx=ctx)
    bad = dict(w)
    bad["l0.mix.o"] = bad["l0.mix.o"][:, :-1].contiguous()
    with pytest.raises(AhaHipError):
        HipInferenceModel(cfg, bad, ctx=ctx)


def test_checkpoint_directory_and_trace_runner(ctx, tmp_path):
    """save_checkpoint -> the native loader -> bin/trace_run as a child process, step by step."""
    import json
    import os
    import subprocess
    import sys
    from aha_amd.checkpoint import save_checkpoint
    cfg = config([layer(chunk=24), layer(ff=0, v_mix=False), layer(chunk=64)], dtype="float32")
    w = dosovik_weights(cfg, seed=21)
    save_checkpoint(str(tmp_path / "m"), cfg, w)
    a, b = tokens(40, cfg.vocab_size, 1), tokens(70, cfg.vocab_size, 2)
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": a[:38], "want": [0, 37]}, {"id": "b", "tokens": b[:69], "want": []}], "end": []},
             {"step": 1, "entries": [{"id": "a", "tokens": a[38:39], "want": []}, {"id": "b", "tokens": b[69:], "want": [0]}], "end": ["b"]},
             {"step": 2, "entries": [{"id": "a", "tokens": a[39:], "want": [0]}], "end": ["a"]}]
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    for dtype in ("float32", "bfloat16"):
        out = tmp_path / dtype
        out.mkdir()
        r = subprocess.run([sys.executable, os.path.join(root, "bin", "trace_run"), "--model", str(tmp_path / "m"), "--dtype", dtype, "--out", str(out),
                            "--max-tokens", "200"], input="".join(json.dumps(s) + "\n" for s in steps), capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        assert [x for x in r.stdout.splitlines() if x.startswith("done")] == ["done 0", "done 1", "done 2"]
        ra, rb = reference(cfg, w, a), reference(cfg, w, b)
        got = [np.fromfile(out / f"{i}.f32", dtype="<f4").reshape(-1, cfg.vocab_size) for i in range(3)]
        for g, x in zip(got, (ra[[0, 37]], rb[[69]], ra[[39]])):
            assert g.shape == x.shape and err(g, x) <= TOL[dtype]
