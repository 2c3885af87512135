"""Vamatar (csrc/layered_prenorm.hip) on the GPU against the plain restatement of its equations (oracle/vamatar.py, float64): every mechanism
through the C ABI, prompts against decoding, portions, batches, pages and slots used again, greedy generation.  Tests make their own
configurations and weights; where random weights would hide a fault, one query / key pair is scaled so that its score stands out.

Tolerances: f32 mode -- rounding only (4e-5 of the logits' spread); bf16 mode -- matrix inputs rounded to bf16 (2^-9 relative) through a few
layers: rms 3 % of the logits' spread, and between two ways through the same layers 2.5 %.  Sequences with routed experts are drawn so that no
router's choice is close: rounding may pick another expert there, which is no fault."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from aha_amd.configs_layered import GatedConfig, LatentConfig, Mamba2Config, MoeConfig, PreNormLayer, VamatarConfig
from aha_amd.model import HipContext, HipInferenceModel, generate_generic
from aha_amd.weights_layered import vamatar_weights
from oracle import vamatar as ov

pytestmark = pytest.mark.gpu

TOL = {"float32": 4e-5, "bfloat16": 3e-2}
TOL_SAME = {"float32": 4e-5, "bfloat16": 2.5e-2}


def ssm(heads=6, vdim=24, state=40, groups=2, norm_groups=3, conv=4, mlp=GatedConfig(88)):
    return PreNormLayer(Mamba2Config(heads=heads, vdim=vdim, state=state, groups=groups, norm_groups=norm_groups, conv=conv), mlp)


def att(heads=5, dim=40, rot_dim=16, vdim=24, kv_rank=56, window=50, rope_base=3000.0, scale=0.14, kv_from=None, mlp=GatedConfig(72)):
    return PreNormLayer(LatentConfig(heads=heads, dim=dim, rot_dim=rot_dim, vdim=vdim, kv_rank=kv_rank, window=window, rope_base=rope_base, scale=scale, kv_from=kv_from), mlp)


def config(layers, width=104, vocab=210, scale=2.5, eps=1e-5, cap=20.0, dtype="float32", eos=()):
    return VamatarConfig(hidden_size=width, vocab_size=vocab, layers=layers, embed_scale=scale, norm_eps=eps, logit_softcap=cap, eos_token_ids=list(eos), compute_dtype=dtype)


def tokens(n, vocab, seed=0):
    return torch.randint(0, vocab, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


def close_calls(cfg, w, ids, margin):
    """-> (the restatement's logits, the positions where some router's last chosen and first unchosen logit differ by less than `margin` of the
    row's spread)"""
    seen = []
    keep = ov.route

    def watched(h, wr, top):
        z = h @ wr.T
        if top < z.shape[1]:
            s = z.sort(-1, descending=True).values
            seen.append((s[:, top - 1] - s[:, top]) / z.std())
        return keep(h, wr, top)
    try:
        ov.route = watched
        ref = ov.forward(cfg.to_json(), {k: v.double() for k, v in w.items()}, ids).numpy()
    finally:
        ov.route = keep
    low = torch.stack(seen).min(0).values if seen else torch.full((len(ids),), 9.0)
    bad = (low < margin).nonzero().flatten().tolist()
    return ref, bad


def reference(cfg, w, ids):
    return ov.forward(cfg.to_json(), {k: v.double() for k, v in w.items()}, ids).numpy()


def row_err(got, want):
    """per row: rms over the vocabulary of the difference, mean taken off, over the spread of all wanted logits"""
    d = np.atleast_2d(got) - np.atleast_2d(want)
    d = d - d.mean(-1, keepdims=True)
    return np.sqrt((d * d).mean(-1)) / want.std()


def err(got, want):
    return float(row_err(got, want).max())


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


def clear_ids(cfg, w, n, seed, margin):
    """token ids (an n-long sequence) without a close call of any router, found by replacing the offending tokens"""
    ids = tokens(n, cfg.vocab_size, seed)
    g = torch.Generator().manual_seed(seed + 1000)
    for _ in range(60):
        ref, bad = close_calls(cfg, w, ids, margin)
        if not bad:
            return ids, ref
        for b in bad[:max(1, len(bad) // 2)]:
            ids[b] = int(torch.randint(0, cfg.vocab_size, (1,), generator=g))
    return ids, ref


VARIANTS = {
    # name: (layers, other config fields)
    "one state-space layer": ([ssm()], {}),
    "one attention layer": ([att()], {}),
    "one head": ([ssm(heads=1, vdim=40, state=24, groups=1, norm_groups=1, conv=2)] * 2, {}),
    "state of one": ([ssm(heads=4, vdim=12, state=1, groups=1, norm_groups=1, conv=2)] * 2, {}),
    "groups as heads, parts unlike groups": ([ssm(heads=4, vdim=16, state=32, groups=4, norm_groups=1), ssm(heads=4, vdim=16, state=64, groups=1, norm_groups=2)], {}),
    "parts across heads": ([ssm(heads=6, vdim=10, state=16, groups=3, norm_groups=4)] * 2, {}),
    "wide state": ([ssm(heads=4, vdim=32, state=200, groups=2, norm_groups=2)] * 2, {}),
    "very wide state": ([ssm(heads=2, vdim=16, state=300, groups=1, norm_groups=2)] * 2, {}),
    "wide values": ([ssm(heads=2, vdim=136, state=96, groups=1, norm_groups=2)] * 2, {}),
    "many heads": ([ssm(heads=64, vdim=32, state=128, groups=8, norm_groups=8)], {}),
    "one tap": ([ssm(conv=1)] * 2, {}),
    "three taps, seven taps": ([ssm(conv=3), ssm(conv=7)], {}),
    "window smaller than a page": ([att(window=20), att(window=33)], {}),
    "window of one and of two": ([att(window=1), att(window=2)], {}),
    "windows of several pages": ([att(window=128), att(window=65), att(window=70)], {}),
    "window beyond the sequence, none": ([att(window=5000), att(window=0)], {}),
    "one attention head": ([att(heads=1, dim=64, rot_dim=32, vdim=64, kv_rank=128)] * 2, {}),
    "seventeen heads": ([att(heads=17, dim=16, rot_dim=8, vdim=8, kv_rank=24)] * 2, {}),
    "eight heads (xcd order)": ([att(heads=8, dim=64, rot_dim=32, vdim=64, kv_rank=112)] * 2, {}),
    "wide heads": ([att(heads=2, dim=128, rot_dim=64, vdim=128, kv_rank=256), att(heads=3, dim=190, rot_dim=60, vdim=200, kv_rank=192)], {}),
    "very wide heads": ([att(heads=2, dim=300, rot_dim=20, vdim=280, kv_rank=72)] * 2, {}),
    "rotation wider than the rest": ([att(heads=3, dim=8, rot_dim=80, vdim=100, kv_rank=40)] * 2, {}),
    "wide latent": ([att(heads=4, dim=32, rot_dim=32, vdim=32, kv_rank=520), att(heads=4, dim=32, rot_dim=2, vdim=32, kv_rank=1000)], {}),
    "rank 512": ([att(heads=16, dim=128, rot_dim=64, vdim=128, kv_rank=512, window=100)], {}),
    "one cache for several layers": ([att(window=40), ssm(), att(kv_from=0, window=90, heads=3, dim=20, vdim=50), att(window=30, kv_rank=24), att(kv_from=0, window=7, scale=0.3),
                                      att(kv_from=3, kv_rank=24, heads=9)], {}),
    "mixed order": ([ssm(), att(), ssm(conv=2), ssm(), att(window=70, kv_from=1)], {}),
    "odd sizes": ([ssm(heads=3, vdim=7, state=9, groups=3, norm_groups=7, mlp=GatedConfig(33)), att(heads=3, dim=5, rot_dim=6, vdim=7, kv_rank=11, mlp=GatedConfig(19))], dict(width=51, vocab=97)),
    "no feed-forward in some layers": ([ssm(mlp=None), att(), att(mlp=None), ssm(mlp=None)], {}),
    "experts, one per token": ([ssm(mlp=MoeConfig(40, 8, 1, 56)), att(mlp=MoeConfig(24, 5, 1, 16))], {}),
    "experts, three per token": ([ssm(mlp=MoeConfig(40, 8, 3, 56)), att(mlp=MoeConfig(24, 5, 2, 16))], {}),
    "every expert, no shared one": ([att(mlp=MoeConfig(17, 4, 4)), ssm(mlp=MoeConfig(64, 1, 1))], {}),
    "more than 64 experts": ([ssm(mlp=MoeConfig(16, 150, 2, 30))], {}),
    "large eps, no cap, embedding scale 1": ([ssm(), att()], dict(eps=0.3, cap=0.0, scale=1.0)),
    "small cap": ([ssm(), att()], dict(cap=1.5)),
    "rows of whole load groups": ([ssm(heads=16, vdim=64, state=128, groups=2, norm_groups=2, mlp=GatedConfig(2048)), att(heads=8, dim=64, rot_dim=64, vdim=64, kv_rank=512, mlp=MoeConfig(512, 4, 2, 1024))],
                                  dict(width=1024)),
    "wide rows": ([ssm(mlp=GatedConfig(2600)), att(mlp=MoeConfig(200, 4, 1, 300))], dict(width=2100)),
}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", list(VARIANTS))
def test_prompt_and_decoding_follow_the_equations(ctx, name, dtype):
    """Whole prompt, and the same tokens half as a prompt and half one by one, against the restatement at every position."""
    layers, kw = VARIANTS[name]
    cfg = config(layers, dtype=dtype, **kw)
    w = vamatar_weights(cfg, seed=len(name))
    n = 70 if "rows" in name or "512" in name else 150
    ids, want = clear_ids(cfg, w, n, 1, 1e-4 if dtype == "float32" else 0.03)
    with Model(ctx, cfg, w) as m:
        whole = all_logits(m, ids)
        half = all_logits(m, ids, [n // 2] + [1] * (n - n // 2))
    assert np.isfinite(whole).all() and np.isfinite(half).all()
    assert err(whole, want) <= TOL[dtype], name
    assert err(half, want) <= TOL[dtype], name
    assert err(half, whole) <= TOL_SAME[dtype], name


SHORT_ROWS = {   # name: (layers, width): the sizes of gemv_row_body.h -- K of 1024 (norms, 1021 of them real), 2048 (parts of 256), 3072 (experts' down) -- and neighbours
    "whole load groups": ([ssm(heads=32, vdim=64, state=128, groups=8, norm_groups=8, mlp=MoeConfig(ff=768, experts=32, top=2, shared_ff=1536)),
                           att(heads=16, dim=128, rot_dim=64, vdim=128, kv_rank=256, mlp=GatedConfig(3072))], 1024),
    "pad columns, four choices of 64": ([ssm(heads=32, vdim=64, state=64, groups=2, norm_groups=8, mlp=MoeConfig(ff=509, experts=64, top=4, shared_ff=1020)),
                                         ssm(heads=32, vdim=64, state=40, groups=4, norm_groups=4, mlp=GatedConfig(1500))], 1021),
    "one choice of 70": ([ssm(heads=16, vdim=64, state=64, groups=2, norm_groups=4, mlp=MoeConfig(ff=1024, experts=70, top=1, shared_ff=2048))], 1024),
}


@pytest.mark.parametrize("name", list(SHORT_ROWS))
def test_one_token_steps_on_short_rows(ctx, name):
    layers, width = SHORT_ROWS[name]
    cfg = config(layers, width=width, dtype="bfloat16")
    w = vamatar_weights(cfg, seed=len(name))
    ids, want = clear_ids(cfg, w, 40, 1, 0.03)
    with Model(ctx, cfg, w) as m:
        assert err(all_logits(m, ids, [12] + [1] * 28), want) <= TOL["bfloat16"]


def test_a_token_that_is_not_finite_among_64_experts(ctx):
    """All 64 router logits of its row are NaN: its own logits are not finite, the steps of another sequence around it keep their bits."""
    cfg = config([ssm(heads=32, vdim=64, state=64, groups=2, norm_groups=8, mlp=MoeConfig(ff=512, experts=64, top=4, shared_ff=1024))], width=1024, dtype="bfloat16")
    w = vamatar_weights(cfg, seed=3)
    w["embed"][7] = float("nan")
    ids = [i + (i == 7) for i in tokens(9, cfg.vocab_size, 2)]
    with Model(ctx, cfg, w) as m:
        want = all_logits(m, ids, [5, 1, 1, 1, 1])
        s, bad = m.seq_open(), m.seq_open()
        got = [m.forward_batch([(s, ids[:5], list(range(5)))])[0]]
        m.forward_batch([(bad, ids[:5], [4])])
        for i in range(5, 9):
            lost, _ = m.forward_batch([(bad, [7], [0])])
            assert not np.isfinite(lost).any()
            got.append(m.forward_batch([(s, [ids[i]], [0])])[0])
    assert np.isfinite(want).all() and (np.concatenate(got) == want).all()


# ---- every mechanism, by leaving it out or getting it wrong in the restatement ------------------------------------------------------------
def mistakes():
    """name -> (function of the restatement, its mistaken version)"""
    m = {}

    def on(name, fn, make):
        m[name] = (fn, make(getattr(ov, fn)))
    on("norm without bias", "layer_norm", lambda f: lambda x, w, b, e: f(x, w, b * 0, e))
    on("norm without the mean", "layer_norm", lambda f: lambda x, w, b, e: ov.rms(x, e) * w + b)
    on("norm without eps", "layer_norm", lambda f: lambda x, w, b, e: f(x, w, b, 0.0))
    on("convolution without bias", "short_conv", lambda f: lambda u, w, b: f(u, w, b * 0))
    on("convolution turned round", "short_conv", lambda f: lambda u, w, b: f(u, w.flip(1), b))
    on("convolution of the current token only", "short_conv", lambda f: lambda u, w, b: f(u, w[:, -1:], b))
    on("step sizes without softplus", "softplus", lambda f: lambda z: z.clamp(min=0))
    on("state without decay", "ssm_scan", lambda f: lambda x, B, C, dt, A, D: f(x, B, C, dt, A * 0, D))
    on("state that does not reach the next token", "ssm_scan", lambda f: lambda x, B, C, dt, A, D: f(x, B, C, dt, A * 1e4, D))
    on("state without the direct path", "ssm_scan", lambda f: lambda x, B, C, dt, A, D: f(x, B, C, dt, A, D * 0))
    on("state fed without the step size", "ssm_scan", lambda f: lambda x, B, C, dt, A, D: f(x, B / dt.mean(), C, dt, A, D))
    on("heads dealt to groups in turn", "ssm_scan", lambda f: lambda x, B, C, dt, A, D: f(x, B.flip(1), C.flip(1), dt, A, D))
    on("gate after the norm", "gated_group_norm", lambda f: lambda y, z, w, n, e: ov.rms(y.reshape(len(y), n, -1), e).reshape(y.shape) * w * ov.silu(z))
    on("no gate", "gated_group_norm", lambda f: lambda y, z, w, n, e: ov.rms(y.reshape(len(y), n, -1), e).reshape(y.shape) * w)
    on("norm over all parts at once", "gated_group_norm", lambda f: lambda y, z, w, n, e: f(y, z, w, 1, e))
    on("no rotation", "rope", lambda f: lambda x, pos, base: f(x, pos * 0, base))
    on("rotation of the next position for queries and keys alike is no mistake", "rope", lambda f: lambda x, pos, base: f(x, pos + 1, base))
    on("rotation of neighbouring pairs", "rope", lambda f: lambda x, pos, base: f(torch.cat([x[..., 0::2], x[..., 1::2]], -1), pos, base))
    on("other rotation base", "rope", lambda f: lambda x, pos, base: f(x, pos, base / 50))
    on("window one wider", "window_visible", lambda f: lambda S, n: f(S, n + 1))
    on("window one narrower", "window_visible", lambda f: lambda S, n: f(S, n - 1))
    on("latent without its norm", "latent_kv", lambda f: lambda h, w, p, mx, e, pos: (h @ w[p + "dkv"].T[:, :mx["kv_rank"]], f(h, w, p, mx, e, pos)[1]))
    on("key part without rotation", "latent_kv", lambda f: lambda h, w, p, mx, e, pos: f(h, w, p, mx, e, pos * 0))
    on("score scale", "latent_mixer", lambda f: lambda h, w, p, mx, kv, pos: f(h, w, p, dict(mx, scale=mx["scale"] * 0.5), kv, pos))
    on("expert outputs weighted instead of inputs", "moe_ff", lambda f: _weighted_outputs)
    on("scores renormalized", "route", lambda f: lambda h, wr, top: (lambda i, v: (i, v / v.sum(-1, keepdim=True)))(*f(h, wr, top)))
    on("softmax scores", "route", lambda f: lambda h, wr, top: (lambda i, v: (i, torch.softmax(h @ wr.T, -1).gather(1, i)))(*f(h, wr, top)))
    on("no shared expert", "moe_ff", lambda f: lambda h, w, p, ml: f(h, w, p, dict(ml, shared=None)))
    on("one expert too few", "route", lambda f: lambda h, wr, top: f(h, wr, top - 1))
    on("no soft cap", "softcap", lambda f: lambda z, cap: z)
    on("gelu-like gate", "gated_ff", lambda f: lambda h, w, p: (torch.nn.functional.gelu(h @ w[p + "gate"].T) * (h @ w[p + "up"].T)) @ w[p + "down"].T)
    return m


def _weighted_outputs(h, w, p, ml):
    idx, sc = ov.route(h, w[p + "router"], ml["router"]["top"])
    out = ov.gated_ff(h, w, p + "shared.")
    for e in range(ml["router"]["experts"]):
        for t, k in (idx == e).nonzero().tolist():
            out[t] += sc[t, k] * ov.gated_ff(h[t:t + 1], w, f"{p}e{e}.")[0]
    return out


MECH = [ssm(heads=4, vdim=16, state=24, groups=2, norm_groups=4, mlp=MoeConfig(40, 6, 2, 40)), att(window=9, scale=0.3, mlp=GatedConfig(64)), att(window=6, kv_from=1, scale=0.3, mlp=None)]


@pytest.fixture(scope="module", params=["float32", "bfloat16"])
def mechanisms(request, ctx):
    cfg = config(MECH, eps=0.05, cap=3.0, dtype=request.param)
    w = vamatar_weights(cfg, seed=41)
    ids, want = clear_ids(cfg, w, 90, 42, 0.03)
    with Model(ctx, cfg, w) as m:
        got = [all_logits(m, ids), all_logits(m, ids, [30, 2, 8] + [1] * 50)]
    return cfg, w, ids, want, got


@pytest.mark.parametrize("name", list(mistakes()))
def test_one_mistake_at_a_time(mechanisms, name):
    """The device agrees with the restatement, and with no version of it in which one mechanism is left out or wrong."""
    cfg, w, ids, want, got = mechanisms
    tol = TOL[cfg.compute_dtype]
    fn, wrong = mistakes()[name]
    keep = getattr(ov, fn)
    try:
        setattr(ov, fn, wrong)
        bad = reference(cfg, w, ids)
    finally:
        setattr(ov, fn, keep)
    for g in got:
        assert err(g, want) <= tol
        if "no mistake" in name:
            assert err(g, bad) <= tol
        else:
            assert err(g, bad) > 2.5 * tol, name


def test_embedding_scale_reaches_the_stream(ctx):
    layers = [ssm(), att()]
    w = vamatar_weights(config(layers), seed=43)
    ids = tokens(40, 210, 43)
    for scale in (0.25, 7.0):
        cfg = config(layers, scale=scale)
        with Model(ctx, cfg, w) as m:
            assert err(all_logits(m, ids), reference(cfg, w, ids)) <= TOL["float32"]
    assert err(reference(config(layers, scale=0.25), w, ids), reference(config(layers, scale=7.0), w, ids)) > 0.1


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_residual_stream_after_every_layer(ctx, dtype):
    cfg = config([ssm(), att(mlp=None), ssm(mlp=MoeConfig(32, 4, 2, 32)), att(kv_from=1, mlp=None)], dtype=dtype)
    w = vamatar_weights(cfg, seed=3)
    ids, _ = clear_ids(cfg, w, 90, 3, 0.03)
    ref = []
    ov.forward(cfg.to_json(), {k: v.double() for k, v in w.items()}, ids, ref)
    with Model(ctx, cfg, w) as m:
        m.debug_keep_residual()
        s = m.seq_open()
        m.forward_batch([(s, ids[:-1], [])])
        got = [m.debug_residual(i) for i in range(4)]
        m.forward_batch([(s, ids[-1:], [])])
        last = [m.debug_residual(i) for i in range(4)]
    for i in range(4):
        full = np.concatenate([got[i], last[i]])
        d = full - ref[i].numpy()
        assert np.sqrt((d * d).mean(-1)).max() <= (1e-5 if dtype == "float32" else 4e-2) * ref[i].std(), i


# ---- portions, batches, slots ----------------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("cuts", [[2] * 65, [1] * 130, [3, 61, 2, 2, 62], [64, 64, 2], [63, 2, 65], [1, 129], [7] * 18 + [4]])
def test_portions_do_not_change_the_logits(ctx, dtype, cuts):
    cfg = config([ssm(conv=5), att(window=50), att(window=100, kv_from=1, mlp=None), ssm(conv=2, mlp=MoeConfig(32, 6, 1, 24))], dtype=dtype)
    w = vamatar_weights(cfg, seed=5)
    ids, want = clear_ids(cfg, w, 130, 5, 0.03)
    with Model(ctx, cfg, w) as m:
        assert err(all_logits(m, ids, cuts), want) <= TOL[dtype]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_unequal_requests_in_one_batch_against_each_alone(ctx, dtype):
    """Prompts of different lengths (one token to several pages) in one step, decoded together, the shorter ones ending earlier; pages handed out
    in a scrambled order, slots, states and pages of finished requests used again by the next batch."""
    cfg = config([ssm(), att(window=40), ssm(mlp=MoeConfig(40, 6, 2, 24)), att(window=128)], dtype=dtype)
    w = vamatar_weights(cfg, seed=7)
    lens = [1, 130, 64, 65, 2, 17, 200]
    with Model(ctx, cfg, w) as m:
        m.debug_scramble_pages(True)
        for rnd in range(2):
            drawn = [clear_ids(cfg, w, n + 12, 10 * rnd + i, 0.03) for i, n in enumerate(lens)]
            ids = [d[0] for d in drawn]
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
                assert err(g, drawn[i][1][:len(g)]) <= TOL[dtype], (rnd, i)


SEGMENTED = {   # (state-space layer, prompts of one step)
    "whole heads per block": (dict(heads=64, vdim=64, state=100, groups=4, norm_groups=4), [520, 65]),
    "half heads": (dict(heads=40, vdim=32, state=64, groups=2, norm_groups=2), [900, 1, 330]),
    "wide state": (dict(heads=9, vdim=60, state=250, groups=3, norm_groups=1), [300, 641]),
    "few heads": (dict(heads=2, vdim=16, state=16, groups=1, norm_groups=1), [257, 130, 1200]),
}


@pytest.mark.parametrize("name", list(SEGMENTED))
def test_long_prompts_of_the_recurrence_run_in_segments(ctx, name):
    """Prompts cut into segments that run beside each other, from nothing and from a carried state, unequal ones in a step; slowly decaying
    states, so that the first segment reaches the last."""
    kw, lens = SEGMENTED[name]
    cfg = config([ssm(mlp=None, **kw)] * 2, dtype="bfloat16")
    w = vamatar_weights(cfg, seed=29)
    for i in range(2):
        w[f"l{i}.mix.A_log"] = torch.full_like(w[f"l{i}.mix.A_log"], -4.0)
    ids = [tokens(n + 290, cfg.vocab_size, n) for n in lens]
    with Model(ctx, cfg, w) as m:
        seqs = [m.seq_open() for _ in ids]
        a, _ = m.forward_batch([(s, x[:n], list(range(n))) for s, x, n in zip(seqs, ids, lens)])
        b, _ = m.forward_batch([(s, x[n:], list(range(290))) for s, x, n in zip(seqs, ids, lens)])
        one, _ = m.forward_batch([(s, [5], [0]) for s in seqs])
        pieces = [all_logits(m, x, [64] * (len(x) // 64) + [len(x) % 64] * (len(x) % 64 > 0)) for x in ids]   # one chunk, one segment a step
    at = 0
    for i, n in enumerate(lens):
        got, want = np.concatenate([a[at:at + n], b[i * 290:(i + 1) * 290]]), reference(cfg, w, ids[i] + [5])
        assert err(got, pieces[i]) <= 0.01
        # (a row whose recurrence nearly cancels shows more of its bf16 inputs' rounding than the others: the rows' errors together)
        assert np.sqrt((row_err(got, want[:-1]) ** 2).mean()) <= 0.01
        assert err(one[i], want[-1]) <= TOL["bfloat16"]
        at += n


@pytest.mark.parametrize("ff,experts", [(2040, 2), (200, 3)])
def test_many_tokens_per_expert(ctx, ff, experts):
    """Tiles of 256 slots in one piece and in two, whole and partial.  Every expert is chosen, so that no choice is close."""
    cfg = config([att(heads=1, window=20, mlp=MoeConfig(ff, experts, experts, 64))], width=1800, dtype="bfloat16")
    w = vamatar_weights(cfg, seed=31)
    ids = tokens(3300, cfg.vocab_size, 31)
    rows = list(range(0, 3300, 7)) + [3299]
    want = reference(cfg, w, ids)[rows]
    with Model(ctx, cfg, w) as m:
        s = m.seq_open()
        got, _ = m.forward_batch([(s, ids, rows)])
    assert err(got, want) <= TOL["bfloat16"]


def test_portions_of_different_sizes_and_single_tokens_share_a_step(ctx):
    """One step with a first prompt, a continued one and a single decoded token."""
    cfg = config([ssm(), att(window=33), att(window=90, kv_from=1)], dtype="bfloat16")
    w = vamatar_weights(cfg, seed=8)
    a, b, c = (tokens(n, cfg.vocab_size, n) for n in (90, 140, 61))
    with Model(ctx, cfg, w) as m:
        sa, sb, sc = (m.seq_open() for _ in range(3))
        m.forward_batch([(sb, b[:65], []), (sc, c[:60], [])])
        lg, _ = m.forward_batch([(sa, a, [89]), (sb, b[65:], [0, 74]), (sc, c[60:], [0])])
    want = np.stack([reference(cfg, w, a)[89], reference(cfg, w, b)[65], reference(cfg, w, b)[139], reference(cfg, w, c)[60]])
    assert err(lg, want) <= TOL["bfloat16"]


@pytest.mark.parametrize("wide", [{}, dict(heads=16, vdim=60, state=70, groups=4, norm_groups=2)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_more_sequences_than_the_first_slots_keep_their_states(ctx, dtype, wide):
    """Slots are added while others hold states and histories; many sequences decode in one step (the batched forms of every kernel)."""
    cfg = config([ssm(**wide), att(window=30), ssm(mlp=MoeConfig(24, 40, 2, 24))], dtype=dtype)
    w = vamatar_weights(cfg, seed=9)
    drawn = [clear_ids(cfg, w, 14 + i % 5, 100 + i, 0.08) for i in range(37)]
    with Model(ctx, cfg, w) as m:
        seqs, got = [], []
        for ids, _ in drawn:      # one after the other: every later slot is opened while the earlier ones hold state
            s = m.seq_open()
            m.forward_batch([(s, ids[:6], [])])
            seqs.append(s)
        for step in range(6, 14):
            lg, _ = m.forward_batch([(s, ids[step:step + 1], [0]) for s, (ids, _) in zip(seqs, drawn)])
            got.append(lg)
    got = np.stack(got)
    for i, (_, want) in enumerate(drawn):
        assert row_err(got[:, i], want[6:14]).max() <= TOL[dtype], i


@pytest.mark.parametrize("state,n", [(64, 4), (60, 7), (64, 8), (90, 6)])
def test_step_of_states_on_both_sides_of_the_caches(ctx, state, n):
    """128 heads x 64 values in blocks of 64 columns: 8 to 17 MB of states per layer (16 MB: past the caches)"""
    cfg = config([ssm(heads=128, vdim=64, state=state, groups=8, norm_groups=8)] * 2, dtype="bfloat16")
    w = vamatar_weights(cfg, seed=state)
    ids = [tokens(9, cfg.vocab_size, 50 + i) for i in range(n)]
    with Model(ctx, cfg, w) as m:
        seqs = [m.seq_open() for _ in ids]
        m.forward_batch([(s, x[:5], []) for s, x in zip(seqs, ids)])
        got = np.stack([m.forward_batch([(s, x[i:i + 1], [0]) for s, x in zip(seqs, ids)])[0] for i in range(5, 9)], 1)
    for i, x in enumerate(ids):
        assert err(got[i], reference(cfg, w, x)[5:]) <= TOL["bfloat16"], i


def test_a_slot_used_again_starts_from_nothing(ctx):
    cfg = config([ssm(), att(window=30), ssm()], dtype="bfloat16")
    w = vamatar_weights(cfg, seed=10)
    a, b = tokens(70, 210, 1), tokens(40, 210, 2)
    with Model(ctx, cfg, w) as m:
        first = all_logits(m, b)
        all_logits(m, a)
        assert np.array_equal(all_logits(m, b), first)
        one = all_logits(m, b, [1] * 40)
        all_logits(m, a, [60] + [1] * 10)
        assert np.array_equal(all_logits(m, b, [1] * 40), one)
        m.forward_initial(a, 0)           # sequence 0 and its rotating states
        m.clear_cache()
        x, _ = m.forward_initial(b, 0)
        assert err(x, first[-1:]) <= 1e-6


# ---- keys far away and at edges -----------------------------------------------------------------------------------------------------------------
def spotlight(cfg, w, key_pos, n):
    """Weights and ids under which one token's key answers one query: token A's latent and token B's query meet in one dimension with a large
    score, so that B's output changes visibly if (and only if) A's position is visible.  One attention layer, plain norms."""
    x = cfg.layers[0].mixer
    A, B = 0, 1
    ids = [2 + (i * 7) % (cfg.vocab_size - 2) for i in range(n)]
    if key_pos is not None:
        ids[key_pos] = A
    emb = torch.randn(cfg.vocab_size, cfg.hidden_size, generator=torch.Generator().manual_seed(99)) * 0.3
    emb[:, :2] = 0
    emb[A, 0] = 20.0
    emb[B, 1] = 20.0
    w["embed"] = emb.bfloat16()
    w["l0.norm1"], w["l0.norm1.b"] = torch.ones_like(w["l0.norm1"]), torch.zeros_like(w["l0.norm1.b"])
    dkv, uk, q, uv = (w["l0.mix." + k].float() for k in ("dkv", "uk", "q", "uv"))
    dkv[0] = 0
    dkv[0, 0] = 8.0
    w["l0.mix.dkv.norm"] = torch.ones_like(w["l0.mix.dkv.norm"])
    q, uk = q * 0.1, uk * 0.1
    for h in range(x.heads):
        uk[h * x.dim] = 0
        uk[h * x.dim, 0] = 2.0
        q[h * (x.dim + x.rot_dim)] = 0
        q[h * (x.dim + x.rot_dim), 1] = 4.0
    uv[:, 0] *= 3
    for k, t in (("dkv", dkv), ("uk", uk), ("q", q), ("uv", uv)):
        w["l0.mix." + k] = t.bfloat16()
    return ids, B


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("window,query", [(7, 40), (48, 47), (48, 48), (64, 63), (64, 64), (64, 127), (64, 128), (65, 128), (65, 129), (100, 163), (100, 164), (128, 191), (128, 192), (33, 64)])
@pytest.mark.parametrize("how", ["prompt", "decoded", "portion of two"])
def test_one_key_at_an_edge(ctx, dtype, window, query, how):
    """A key that stands out, at the oldest visible position of the query's window and at the position before it: the output moves with the first
    and not with the second, in prompts, portions and decoding, wherever pages, tiles and portions end."""
    cfg = config([att(heads=3, dim=32, rot_dim=16, vdim=32, kv_rank=64, window=window, scale=0.2, mlp=None)], dtype=dtype, cap=0.0)
    lo = max(0, query - window + 1)
    outs = {}
    for where, kp in (("in", lo), ("out", lo - 1), ("none", None)):
        if kp is not None and (kp < 0 or kp == query):
            continue
        w = vamatar_weights(cfg, seed=11)
        ids, B = spotlight(cfg, w, kp, query + 1)
        ids[query] = B
        want = reference(cfg, w, ids)
        with Model(ctx, cfg, w) as m:
            got = all_logits(m, ids, {"prompt": None, "decoded": [query, 1], "portion of two": [query - 1, 2]}[how])
        assert err(got, want) <= TOL[dtype]
        outs[where] = (got[query], want[query])
    spread = outs["none"][1].std()
    if "in" in outs:      # the planted key is seen ...
        assert np.abs(outs["in"][0] - outs["none"][0]).max() > 0.2 * spread
    if "out" in outs:     # ... and its neighbour on the other side of the edge is not: the same logits to rounding
        assert np.abs(outs["out"][0] - outs["none"][0]).max() < (1e-3 if dtype == "float32" else 0.05) * spread


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_far_key_among_thousands(ctx, dtype):
    """One visible key up to 1500 positions back inside a window of 2048 (many tiles, several decode splits), the same key moved to page borders."""
    cfg = config([att(heads=4, dim=64, rot_dim=32, vdim=48, kv_rank=128, window=2048, scale=0.1, mlp=None)], dtype=dtype, cap=0.0)
    n = 1500
    outs = []
    for kp in (0, 31, 32, 63, 64, 99, n - 2):
        w = vamatar_weights(cfg, seed=12)
        ids, B = spotlight(cfg, w, kp, n)
        ids[-1] = B
        with Model(ctx, cfg, w) as m:
            s = m.seq_open()
            m.forward_batch([(s, ids[:-1], [])])
            dec, _ = m.forward_batch([(s, ids[-1:], [0])])
            t = m.seq_open()
            pro, _ = m.forward_batch([(t, ids, [n - 1])])
            # with a neighbour: the batched form (joined latents, then the values of all sequences)
            many = [m.seq_open() for _ in range(6)]
            m.forward_batch([(x, ids[:-1], []) for x in many])
            bat, _ = m.forward_batch([(x, ids[-1:], [0]) for x in many])
        x = reference(cfg, w, ids)[-1:]
        assert err(dec, x) <= TOL[dtype] and err(pro, x) <= TOL[dtype] and err(bat, np.repeat(x, 6, 0)) <= TOL[dtype], kp
        outs.append(dec[0])
    spread = outs[0].std()
    for o in outs[1:]:
        assert np.abs(o - outs[0]).max() < 0.3 * spread     # wherever the key is, it is found


@pytest.mark.parametrize("rank,rot,window", [(256, 64, 0), (256, 20, 100), (512, 64, 0), (500, 32, 96), (128, 64, 33), (288, 64, 0)])
def test_decoding_where_tiles_end(ctx, rank, rot, window):
    """A wave per tile of 32 positions (ranks padded to 128, 256 and 512, key parts to 32 and 64; 288: four waves per tile): contexts that end in front of,
    at and behind a tile, a round of four waves and a page, the sequences one by one and in one step, with a head group that is not full."""
    cfg = config([att(heads=17, dim=32, rot_dim=rot, vdim=32, kv_rank=rank, window=window, scale=0.3, mlp=None)], dtype="bfloat16", cap=0.0)
    w = vamatar_weights(cfg, seed=14)
    ids = tokens(420, cfg.vocab_size, seed=15)
    want = reference(cfg, w, ids)
    at = [1, 31, 32, 33, 63, 64, 127, 128, 129, 256, 419]
    with Model(ctx, cfg, w) as m:
        seqs = [m.seq_open() for _ in at]
        for s, p in zip(seqs, at):
            m.forward_batch([(s, ids[:p], [])])
            t = m.seq_open()
            m.forward_batch([(t, ids[:p], [])])
            one, _ = m.forward_batch([(t, ids[p:p + 1], [0])])
            assert err(one, want[p:p + 1]) <= TOL["bfloat16"], p
            m.seq_close(t)
        got, _ = m.forward_batch([(s, ids[p:p + 1], [0]) for s, p in zip(seqs, at)])
    assert err(got, want[at]) <= TOL["bfloat16"]


@pytest.mark.parametrize("groups,state,conv,rows", [(256, 8, 4, 257), (512, 4, 7, 254)])
def test_steps_in_parts(ctx, groups, state, conv, rows):
    """launch_ssm_step: groups x sequences beyond the grid's 65535 go in parts (255 sequences at 256 groups, 127 at 512); a second part of two sequences and a
    full one, whose logits come from what the step before left of state and history; against the restatement."""
    cfg = config([ssm(heads=groups, vdim=8, state=state, groups=groups, norm_groups=8, conv=conv, mlp=None)], width=64, vocab=64, dtype="bfloat16", cap=0.0)
    w = vamatar_weights(cfg, seed=21)
    ids = [tokens(4, cfg.vocab_size, seed=70 + i) for i in range(rows)]
    want = [reference(cfg, w, x) for x in ids]
    with Model(ctx, cfg, w) as m:
        seqs = [m.seq_open() for _ in ids]
        m.forward_batch([(s, x[:2], []) for s, x in zip(seqs, ids)])
        for at in (2, 3):
            got, _ = m.forward_batch([(s, x[at:at + 1], [0]) for s, x in zip(seqs, ids)])
            assert err(got, np.stack([r[at] for r in want])) <= TOL["bfloat16"]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 128, 200])
def test_a_token_far_back_in_the_state(ctx, dtype, n):
    """States that hardly decay: the first token's share of the output `n` tokens later, through chunk borders, portions and decoding, is the
    restatement's; the same with the first token replaced moves the logits."""
    cfg = config([ssm(heads=4, vdim=16, state=16, groups=1, norm_groups=1, conv=4, mlp=None)], dtype=dtype, cap=0.0)
    w = vamatar_weights(cfg, seed=23)
    w["l0.mix.A_log"] = torch.full_like(w["l0.mix.A_log"], -9.0)
    w["l0.mix.dt_bias"] = torch.full_like(w["l0.mix.dt_bias"], -4.0)
    dt_rows = w["l0.mix.in"].float()
    dt_rows[-4:] = 0
    dt_rows[-4:, 0] = 2.0       # the first dimension of a token's normed row opens its step
    w["l0.mix.in"] = dt_rows.bfloat16()
    w["l0.norm1"], w["l0.norm1.b"] = torch.ones_like(w["l0.norm1"]), torch.zeros_like(w["l0.norm1.b"])
    emb = w["embed"].float()
    emb[:, 0] = -1.0
    emb[0, 0], emb[1, 0] = 3.0, 3.0
    w["embed"] = emb.bfloat16()
    ids = [0] + [2 + (i * 11) % 200 for i in range(n)]
    other = [1] + ids[1:]
    want, moved = reference(cfg, w, ids), reference(cfg, w, other)
    assert np.abs(want[-1] - moved[-1]).max() > 0.3 * want.std()
    with Model(ctx, cfg, w) as m:
        for cuts in (None, [1] * (n + 1), [1, n], [n, 1]):
            assert err(all_logits(m, ids, cuts), want) <= TOL[dtype], cuts


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_first_tokens_of_a_sequence(ctx, dtype):
    cfg = config([ssm(conv=5), att()], dtype=dtype)
    w = vamatar_weights(cfg, seed=14)
    ids = tokens(9, cfg.vocab_size, 14)
    want = reference(cfg, w, ids)
    with Model(ctx, cfg, w) as m:
        for n in range(1, 9):
            assert err(all_logits(m, ids[:n], [1] * n), want[:n]) <= TOL[dtype]
            assert err(all_logits(m, ids[:n]), want[:n]) <= TOL[dtype]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_decoding_gives_passed_pages_back(ctx, dtype):
    """400 decoded tokens with windows of 64 and 96: pages in front of both return to the pool, the logits keep following the equations."""
    cfg = config([ssm(), att(window=64), att(window=96, kv_from=1, mlp=None)], dtype=dtype)
    w = vamatar_weights(cfg, seed=15)
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
        # a long portion behind passed pages
        more = tokens(100, cfg.vocab_size, 16)
        lg, _ = m.forward_batch([(s, more, list(range(100)))])
        assert err(lg, reference(cfg, w, ids + more)[420:]) <= TOL[dtype]
        m.seq_close(s)


# ---- generation ------------------------------------------------------------------------------------------------------------------------------------
GEN = [ssm(), att(window=32), ssm(mlp=MoeConfig(32, 4, 1, 32)), att(window=20, kv_from=1)]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_greedy_generation_by_every_loop(ctx, dtype):
    """generate_generic step by step, its device-resident loop, and the batch loop: the same tokens as stepping the restatement (as far as the
    margins of the arg-max and of the routers are above the rounding)."""
    from aha_amd.scheduler import Request, generate_batch
    cfg = config(GEN, dtype=dtype, cap=0.0)
    w = vamatar_weights(cfg, seed=16)
    prompts = [tokens(n, cfg.vocab_size, 20 + n) for n in (5, 50, 33)]
    want = []
    for p in prompts:
        ids, safe = list(p), 40
        for i in range(40):
            ref, bad = close_calls(cfg, w, ids, 1e-4 if dtype == "float32" else 0.02)
            top = np.sort(ref[-1])[-2:]
            if bad or (top[1] - top[0]) / ref[-1].std() < (1e-3 if dtype == "float32" else 0.12):
                safe = i
                break
            ids.append(int(ref[-1].argmax()))
        want.append(ids[len(p):len(p) + safe])
    assert sum(len(x) for x in want) > (40 if dtype == "float32" else 3)
    with Model(ctx, cfg, w) as m:
        outs = generate_batch(m, [Request(p, max_tokens=40) for p in prompts])
        for p, x, o in zip(prompts, want, outs):
            a, _ = generate_generic(m, p, 40)
            b, _ = generate_generic(m, p, 40, device_loop=True)
            assert a[:len(x)] == x and b[:len(x)] == x and o[:len(x)] == x
            assert a == b
        assert m.cache_len() == 0


def test_device_loop_stops_at_a_stop_token_and_continues_cleanly(ctx):
    """The loop runs ahead of the host; after a stop token the recurrent state must be that of the last kept token."""
    w = vamatar_weights(config(GEN), seed=17)
    p = tokens(30, 210, 17)
    with Model(ctx, config(GEN, dtype="bfloat16"), w) as m:
        free, _ = generate_generic(m, p, 30, device_loop=True)
    stop = free[12]
    first = free.index(stop)
    if first < 2:
        pytest.skip("the generated sequence repeats its first tokens")
    with Model(ctx, config(GEN, dtype="bfloat16", eos=[stop]), w) as m:
        _, t0 = m.forward_initial(p, 0, want_logits=False)
        out = m.decode_greedy(t0, len(p), 29)
        assert [t0] + out == free[:first + 1]
        assert m.cache_len() == len(p) + len(out)
        lg, _ = m.forward_step(out[-1], m.cache_len())
        ids = p + [t0] + out
        fresh = m.seq_open()
        m.forward_batch([(fresh, p, [])])
        for t in ids[len(p):]:
            ref, _ = m.forward_batch([(fresh, [t], [0])])
        assert err(lg, ref) <= 1e-6


def test_sampled_batch_equals_sampled_alone(ctx):
    from aha_amd.sampling import GenerationContext, generate_generic_sampled
    from aha_amd.scheduler import Request, generate_batch
    cfg = config(GEN, dtype="float32")
    w = vamatar_weights(cfg, seed=19)
    prompts = [tokens(n, cfg.vocab_size, 30 + n) for n in (4, 40)]

    def gctx(i, n):
        return GenerationContext(0.8, 0.9, 20, 1.1, 64, 100 + i, n, 12)
    with Model(ctx, cfg, w) as m:
        alone = [generate_generic_sampled(m, p, gctx(i, len(p))) for i, p in enumerate(prompts)]
        both = generate_batch(m, [Request(p, max_tokens=12, ctx=gctx(i, len(p))) for i, p in enumerate(prompts)])
    assert both == alone


def test_errors_are_refused(ctx):
    cfg = config([ssm(), att()], dtype="bfloat16")
    w = vamatar_weights(cfg, seed=20)
    from aha_amd._lib import AhaHipError
    with Model(ctx, cfg, w) as m:
        s = m.seq_open()
        for bad in ([(s + 5, [1], [])], [(s, [], [])], [(s, [cfg.vocab_size], [])], [(s, [1], [1])], [(s, [1], []), (s, [2], [])], []):
            with pytest.raises(AhaHipError):
                m.forward_batch(bad)
        assert m.seq_len(s) == 0
        m.seq_close(s)
    for name in ("l0.mix.conv.b", "l1.mix.dkv.norm", "l1.norm2.b", "final.norm.b"):
        with pytest.raises(AhaHipError):
            HipInferenceModel(cfg, {k: v for k, v in w.items() if k != name}, ctx=ctx)
    bad = dict(w)
    bad["l1.mix.o"] = bad["l1.mix.o"][:, :-1].contiguous()
    with pytest.raises(AhaHipError):
        HipInferenceModel(cfg, bad, ctx=ctx)
    for layers in ([att(kv_from=0)], [ssm(), att(kv_from=0)], [att(), att(kv_from=0, kv_rank=40)], [att(), att(kv_from=0), att(kv_from=1)], [ssm(heads=5, groups=2)],
                   [ssm(norm_groups=5)], [att(rot_dim=7)], [ssm(mlp=MoeConfig(8, 4, 5, 8))]):
        with pytest.raises(AhaHipError):
            HipInferenceModel(config(layers), w, ctx=ctx)


def test_checkpoint_directory_and_trace_runner(ctx, tmp_path):
    """save_checkpoint -> the native loader -> bin/trace_run as a child process, step by step."""
    from aha_amd.checkpoint import save_checkpoint
    cfg = config([ssm(), att(window=24, mlp=None), ssm(mlp=MoeConfig(32, 4, 1, 24)), att(window=64, kv_from=1)], dtype="float32")
    w = vamatar_weights(cfg, seed=21)
    save_checkpoint(str(tmp_path / "m"), cfg, w)
    (a, ra), (b, rb) = clear_ids(cfg, w, 40, 1, 0.03), clear_ids(cfg, w, 70, 2, 0.03)
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
        got = [np.fromfile(out / f"{i}.f32", dtype="<f4").reshape(-1, cfg.vocab_size) for i in range(3)]
        for g, x in zip(got, (ra[[0, 37]], rb[[69]], ra[[39]])):
            assert g.shape == x.shape and err(g, x) <= TOL[dtype]
