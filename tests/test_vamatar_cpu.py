"""Vamatar without a GPU: the restatement's mechanisms against hand-made cases (one function each), the config reader, the checkpoint round
trip, struct layouts, the scheduler's entry point on a stand-in model."""
import ctypes
import json
import math
import os

import numpy as np
import pytest
import torch

from aha_amd import _lib
from aha_amd.checkpoint import config_from_desc, open_weights, parse_config, save_checkpoint
from aha_amd.configs import qwen3_0_6b
from aha_amd.configs_layered import GatedConfig, LatentConfig, Mamba2Config, MoeConfig, PreNormLayer, VamatarConfig, vamatar_like
from aha_amd.model import make_desc
from aha_amd.weights_layered import vamatar_weights
from oracle import vamatar as ov

D = torch.float64


def t(*v):
    return torch.tensor(v, dtype=D)


def cfg_small(**kw):
    a = Mamba2Config(heads=6, vdim=5, state=7, groups=3, norm_groups=2, conv=3)
    b = LatentConfig(heads=3, dim=6, rot_dim=4, vdim=5, kv_rank=9, window=11, rope_base=77.0, scale=0.31)
    c = LatentConfig(heads=2, dim=3, rot_dim=4, vdim=8, kv_rank=9, window=4, rope_base=77.0, scale=0.2, kv_from=1)
    d = LatentConfig(heads=1, dim=3, rot_dim=2, vdim=2, kv_rank=5, window=0, rope_base=1e4, scale=0.5)
    return VamatarConfig(hidden_size=20, vocab_size=31, layers=[PreNormLayer(a, GatedConfig(18)), PreNormLayer(b, MoeConfig(12, 5, 2, 14)), PreNormLayer(c, None),
                                                                PreNormLayer(d, MoeConfig(8, 3, 1))],
                         embed_scale=2.5, norm_eps=1e-4, logit_softcap=kw.pop("cap", 12.0), **kw)


# ---- the mechanisms ------------------------------------------------------------------------------------------------------------------
def test_layer_norm_takes_the_mean_off_and_adds_the_bias():
    x = t(1, 5, 1, 5)[None]
    assert torch.allclose(ov.layer_norm(x, t(1, 1, 2, 2), t(0, 10, 0, 10), 0.0), t(-1, 11, -2, 12)[None])
    assert torch.allclose(ov.layer_norm(x, t(1, 1, 1, 1), t(0, 0, 0, 0), 12.0), t(-0.5, 0.5, -0.5, 0.5)[None])   # eps inside the root


def test_rms_and_softplus():
    assert torch.allclose(ov.rms(t(3, -4, 0, 0)[None], 2.75), t(1, -4 / 3, 0, 0)[None])
    z = t(-800, -1, 0, 1, 800)
    assert torch.allclose(ov.softplus(z), t(0, math.log1p(math.exp(-1)), math.log(2), math.log1p(math.e), 800))


def test_short_convolution_is_causal_per_channel_with_bias():
    u = torch.arange(1.0, 11.0, dtype=D).reshape(5, 2)
    w = torch.tensor([[100.0, 10.0, 1.0], [0.0, 0.0, 2.0]], dtype=D)
    y = ov.short_conv(u, w, t(0.5, -1))
    assert y[:, 0].tolist() == [1.5, 13.5, 135.5, 357.5, 579.5]
    assert y[:, 1].tolist() == [2 * v - 1 for v in (2, 4, 6, 8, 10)]


def test_state_space_recurrence_by_hand():
    """one head, one column: S_t = e^(A dt) S + dt B x, y = S . C + D x; heads read their group's B and C"""
    x, B, C, dt = torch.zeros(2, 2, 1, dtype=D), torch.zeros(2, 2, 2, dtype=D), torch.zeros(2, 2, 2, dtype=D), torch.zeros(2, 2, dtype=D)
    x[:, 0, 0], B[:, 0], C[:, 0], dt[:, 0] = t(2, 3), torch.stack([t(1, 4), t(5, 0)]), torch.stack([t(1, 1), t(10, 1)]), t(0.5, 0.25)
    y = ov.ssm_scan(x, B, C, dt, t(-math.log(16.0), -1.0), t(7, 0))
    s0 = 0.5 * t(1, 4) * 2
    s1 = s0 * 0.5 + 0.25 * t(5, 0) * 3                                  # 16^-0.25 = 0.5
    assert torch.allclose(y[:, 0, 0], torch.stack([s0.sum() + 14, (s1 * t(10, 1)).sum() + 21]))
    assert y[:, 1].abs().max() == 0                                     # the second head has group 1's zeros
    four = ov.ssm_scan(x[:, :1].expand(2, 4, 1), B, C, dt[:, :1].expand(2, 4), torch.full((4,), -math.log(16.0), dtype=D), torch.full((4,), 7.0, dtype=D))
    assert torch.allclose(four[:, 0], y[:, 0]) and torch.allclose(four[:, 1], y[:, 0])      # heads 0, 1: group 0
    assert torch.allclose(four[:, 2], 7 * x[:, 0]) and torch.allclose(four[:, 3], 7 * x[:, 0])


def test_gate_comes_before_the_norm_of_every_part():
    y, z = t(3, 4, 1, 1)[None], t(0, 1e3, 1e3, 1e3)[None]
    g = ov.gated_group_norm(y, z, t(1, 1, 1, 5), 2, 0.0)                # silu(0) = 0: the first part is (0, 4000)
    assert torch.allclose(g, t(0, math.sqrt(2), 1, 5)[None])


def test_rotation_pairs_and_angles():
    x = torch.zeros(2, 1, 4, dtype=D)
    x[:, 0, 1] = 1.0                                                    # pair (1, 3), frequency base^(-2 / 4)
    y = ov.rope(x, torch.tensor([0, 3]), 16.0)
    a = 3 * 16.0 ** -0.5
    assert torch.allclose(y[0], x[0]) and torch.allclose(y[1, 0], t(0, math.cos(a), 0, math.sin(a)))


def test_window_mask():
    m = ov.window_visible(5, 2)
    assert [r.nonzero().flatten().tolist() for r in m] == [[0], [0, 1], [1, 2], [2, 3], [3, 4]]
    assert ov.window_visible(4, 0).sum() == 10


def test_latent_attention_by_hand():
    """two heads over one latent: scores from the unrotated and the shared rotated part, values from the latent"""
    g = torch.Generator().manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g, dtype=D)
    mx = dict(heads=2, dim=3, rot_dim=2, vdim=4, kv_rank=5, scale=0.7, mask={"size": 2}, rot={"base": 9.0, "dims": 2})
    w = {"q": r(10, 6), "dkv": r(7, 6), "dkv.norm": r(5), "uk": r(6, 5), "uv": r(8, 5), "o": torch.eye(8, dtype=D)}
    h, pos = r(3, 6), torch.arange(3)
    c, kr = ov.latent_kv(h, w, "", mx, 1e-5, pos)
    lat = h @ w["dkv"][:5].T
    assert torch.allclose(c, lat / torch.sqrt((lat ** 2).mean(-1, keepdim=True) + 1e-5) * w["dkv.norm"])
    assert torch.allclose(kr[0], h[0] @ w["dkv"][5:].T)
    out = ov.latent_mixer(h, w, "", mx, (c, kr), pos)
    q = h[2] @ w["q"][5:].T                                             # head 1 of the last token sees tokens 1 and 2
    qr = ov.rope(q[None, 3:], torch.tensor([2]), 9.0)[0]
    s = torch.stack([(q[:3] @ (w["uk"][3:] @ c[j]) + qr @ kr[j]) * 0.7 for j in (1, 2)])
    p = s.exp() / s.exp().sum()
    assert torch.allclose(out[2, 4:], p[0] * (w["uv"][4:] @ c[1]) + p[1] * (w["uv"][4:] @ c[2]))


def test_routing_picks_the_largest_scores_and_weights_the_input():
    h, wr = t(1, 2)[None], torch.tensor([[1.0, 0.0], [0.0, 1.0], [-1.0, 0.0]], dtype=D)
    i, s = ov.route(h, wr, 2)
    assert i.tolist() == [[1, 0]] and torch.allclose(s, torch.sigmoid(t(2, 1))[None])      # not renormalized
    w = {"router": wr}
    for e in range(3):
        w.update({f"e{e}.gate": (e + 1.0) * torch.eye(2, dtype=D), f"e{e}.up": torch.eye(2, dtype=D), f"e{e}.down": torch.eye(2, dtype=D)})
    got = ov.moe_ff(h, w, "", {"router": {"experts": 3, "top": 2}})
    want = 0
    for e, sc in ((1, torch.sigmoid(t(2))), (0, torch.sigmoid(t(1)))):
        x = sc * h
        g = (e + 1) * x
        want = want + g * torch.sigmoid(g) * x
    assert torch.allclose(got, want)


def largest_logits(z, top):
    """The choice of any number of experts (wave_topk): a logit that is not a number, or -inf, is never larger than another; the lowest index among equals,
    the last expert when nothing is left."""
    left, out = z.copy(), []
    for _ in range(top):
        m = np.fmax.reduce(left, initial=np.float32(-np.inf))
        i = int(np.flatnonzero(left == m)[0]) if m > -np.inf else len(z) - 1
        left[i] = -np.inf
        out.append((i, 1 / (1 + np.exp(-m, dtype=np.float32))))
    return out


@pytest.mark.parametrize("experts,top", [(1, 1), (2, 2), (63, 1), (63, 6), (63, 63), (64, 1), (64, 6), (64, 63)])
def test_one_logit_per_lane_chooses_the_same_experts(hip_lib, experts, top):
    """csrc/expert_choice.h: finite logits, ties, infinities, NaN in some, in all but one and in every place, with and without spare lanes"""
    rng = np.random.default_rng(experts * 100 + top)
    rows = [rng.standard_normal(experts), rng.integers(0, 3, experts).astype(float), np.full(experts, np.nan), np.full(experts, -np.inf), np.full(experts, np.inf)]
    some = rng.standard_normal(experts)
    some[rng.random(experts) < 0.5] = np.nan
    one = np.full(experts, np.nan)
    one[experts // 2] = -3
    mixed = rng.standard_normal(experts)
    mixed[::3], mixed[1::5], mixed[-1] = -np.inf, np.nan, np.inf
    for z in rows + [some, one, mixed]:
        z = z.astype(np.float32)
        sel, weight = np.full(top, -77, np.int32), np.full(top, -77, np.float32)
        assert hip_lib.aha_hip_debug_expert_choice(z.ctypes.data, experts, top, sel.ctypes.data, weight.ctypes.data) == 0
        with np.errstate(over="ignore"):
            want = largest_logits(z, top)
        assert sel.tolist() == [i for i, _ in want], z
        assert np.allclose(weight, [w for _, w in want], rtol=1e-6, atol=0), z


def test_one_cache_serves_the_layers_that_name_it():
    cfg = cfg_small()
    w = {k: v.double() for k, v in vamatar_weights(cfg, seed=1).items()}
    assert "l2.mix.dkv" not in w and "l3.mix.dkv" in w
    ids = [3, 1, 4, 1, 5, 9, 2, 6]
    a = ov.forward(cfg.to_json(), w, ids)
    w["l1.mix.dkv"] = w["l1.mix.dkv"].flip(0)
    for k in ("l1.mix.o", "l1.mlp.shared.down", *(f"l1.mlp.e{e}.down" for e in range(5))):
        w[k] = w[k] * 0                                                 # layer 1 adds nothing itself
    b = ov.forward(cfg.to_json(), w, ids)
    w["l1.mix.dkv"] = w["l1.mix.dkv"].flip(0)
    assert not torch.allclose(b, ov.forward(cfg.to_json(), w, ids)) and a.shape == (8, 31)


def test_softcap_bounds_the_logits():
    assert torch.allclose(ov.softcap(t(0, 1e9, -1e9), 5.0), t(0, 5, -5)) and torch.allclose(ov.softcap(t(1, 2), None), t(1, 2))


# ---- config reader and checkpoint ------------------------------------------------------------------------------------------------------
def same_layers(a, b):
    for x, y in zip(a.layers, b.layers):
        assert type(x.mixer) is type(y.mixer) and x.mlp == y.mlp
        for k, v in vars(y.mixer).items():
            assert getattr(x.mixer, k) == (float(np.float32(v)) if k == "scale" else v), k
    assert len(a.layers) == len(b.layers)


def test_config_reader_takes_every_field_from_the_file(hip_lib, tmp_path):
    cfg = cfg_small()
    (tmp_path / "config.json").write_text(json.dumps(cfg.to_json()))
    d = parse_config(str(tmp_path))                # no generation_config.json: no stop tokens
    assert d.arch == _lib.AHA_ARCH_VAMATAR and d.n_stop_tokens == 0
    back = config_from_desc(d)
    assert (back.hidden_size, back.vocab_size) == (20, 31)
    for f in ("embed_scale", "norm_eps", "logit_softcap"):
        assert getattr(back, f) == float(np.float32(getattr(cfg, f)))
    same_layers(back, cfg)
    same_layers(config_from_desc(make_desc(cfg)), cfg)
    (tmp_path / "generation_config.json").write_text('{"eos_token_id": [4, 9]}')
    assert config_from_desc(parse_config(str(tmp_path))).eos_token_ids == [4, 9]
    j = cfg_small(cap=0.0).to_json()
    assert "logit_softcap" not in j and "mask" not in j["layers"][3]["mixer"]
    (tmp_path / "config.json").write_text(json.dumps(dict(j, logit_softcap=None)))
    assert config_from_desc(parse_config(str(tmp_path))).logit_softcap == 0.0


@pytest.mark.parametrize("path,value", [
    (("width",), None), (("vocab",), 3.5), (("embedding",), None), (("norm", "eps"), None), (("logit_softcap",), "x"), (("layers",), []),
    (("layers", 0, "type"), "attention"), (("layers", 0, "mixer", "state"), None), (("layers", 0, "mixer", "conv"), None), (("layers", 0, "mixer", "norm_groups"), "2"),
    (("layers", 1, "mixer", "rot", "base"), None), (("layers", 1, "mixer", "rot", "dims"), 2), (("layers", 1, "mixer", "mask", "size"), 0),
    (("layers", 1, "mixer", "scale"), None), (("layers", 2, "mixer", "kv_from"), "1"), (("layers", 0, "mlp", "kind"), "sparse"), (("layers", 0, "mlp", "ff"), None),
    (("layers", 1, "mlp", "router"), None), (("layers", 1, "mlp", "router", "top"), None), (("layers", 1, "mlp", "expert"), None), (("layers", 1, "mlp", "shared", "ff"), None)])
def test_config_reader_refuses(hip_lib, tmp_path, path, value):
    j = json.loads(json.dumps(cfg_small().to_json()))
    o = j
    for k in path[:-1]:
        o = o[k]
    if value is None:
        del o[path[-1]]
    else:
        o[path[-1]] = value
    (tmp_path / "config.json").write_text(json.dumps(j))
    with pytest.raises(_lib.AhaHipError):
        parse_config(str(tmp_path))


def test_checkpoint_round_trip(hip_lib, tmp_path):
    cfg = cfg_small(eos_token_ids=[3])
    w = vamatar_weights(cfg, seed=2)
    save_checkpoint(str(tmp_path), cfg, w, shards=2)
    got = open_weights(str(tmp_path))
    assert set(got) == set(w)
    for n, x in w.items():
        assert got[n][0] == _lib.AHA_BF16 and got[n][1] == tuple(x.shape) and got[n][2] == x.contiguous().view(torch.uint8).numpy().tobytes()
    assert config_from_desc(parse_config(str(tmp_path))).eos_token_ids == [3]


def test_model_struct_mirrors_the_header():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    src = open(os.path.join(root, "include", "aha_hip.h")).read()
    for name, value in (("AHA_ARCH_VAMATAR", _lib.AHA_ARCH_VAMATAR), ("AHA_MIXER_MAMBA2", _lib.AHA_MIXER_MAMBA2), ("AHA_MIXER_LATENT", _lib.AHA_MIXER_LATENT),
                        ("AHA_MLP_GATED", _lib.AHA_MLP_GATED), ("AHA_MLP_MOE", _lib.AHA_MLP_MOE)):
        assert f"{name} = {value}" in src, name
    body = src[:src.index("} aha_layer_desc;")]
    body = body[body.rindex("{"):]
    at = [body.find(f" {n}") for n, _ in _lib.LayerDesc._fields_]
    assert all(x > 0 for x in at) and ctypes.sizeof(_lib.LayerDesc) % 8 == 0


def test_like_sizes():
    b = qwen3_0_6b()
    c = vamatar_like(b, layers=8)
    kinds = [type(x.mixer) for x in c.layers]
    assert kinds.count(LatentConfig) == 2 and kinds.count(Mamba2Config) == 6 and c.layers[0].mlp.ff == b.intermediate_size
    m = c.layers[1].mlp
    assert m.top * m.ff + m.shared_ff == b.intermediate_size


# ---- the batch scheduler --------------------------------------------------------------------------------------------------------------
def test_the_scheduler_serves_the_restatement():
    """generate_batch over a model whose step runs the restatement: greedy tokens of every request as alone, sequences given back"""
    from aha_amd.scheduler import Request, generate_batch
    cfg = cfg_small()
    j, w = cfg.to_json(), {k: v.double() for k, v in vamatar_weights(cfg, seed=3).items()}

    class Plain:
        seqs = {}

        def stop_token_ids(self):
            return []

        def seq_open(self):
            s = max(self.seqs, default=0) + 1
            self.seqs[s] = []
            return s

        def seq_close(self, s):
            del self.seqs[s]

        def forward_batch(self, entries, want_logits=True, want_argmax=False):
            out = []
            for s, toks, want in entries:
                n = len(self.seqs[s])
                self.seqs[s] = self.seqs[s] + list(toks)
                out += [int(ov.forward(j, w, self.seqs[s])[n + i].argmax()) for i in want]
            return None, np.array(out, dtype=np.uint32)

    def alone(p, n):
        ids = list(p)
        for _ in range(n):
            ids.append(int(ov.forward(j, w, ids)[-1].argmax()))
        return ids[len(p):]
    prompts = [[1, 2, 3], [7], [9, 8] * 4]
    m = Plain()
    assert generate_batch(m, [Request(p, n) for p, n in zip(prompts, (4, 1, 6))]) == [alone(p, n) for p, n in zip(prompts, (4, 1, 6))] and not m.seqs
