"""-m gpu: pieces of a batched step -- the arg-max of many rows in one pass, experts with any small number of slots."""
import numpy as np
import pytest
import torch

from aha_amd import weights_layered
from aha_amd.configs_layered import GatedConfig, LatentConfig, MoeConfig, PreNormLayer, VamatarConfig
from aha_amd.model import HipInferenceModel
from oracle import vamatar as V

pytestmark = pytest.mark.gpu


def moe_model(gpu, experts, top, ff, shared, hidden=256, vocab=5000):
    att = LatentConfig(heads=2, dim=32, rot_dim=16, vdim=32, kv_rank=64, window=64, rope_base=1e4, scale=48 ** -0.5)
    cfg = VamatarConfig(hidden_size=hidden, vocab_size=vocab, layers=[PreNormLayer(att, MoeConfig(ff=ff, experts=experts, top=top, shared_ff=shared)),
                                                                     PreNormLayer(att, GatedConfig(128))], embed_scale=16.0)
    w = weights_layered.vamatar_weights(cfg, seed=3)
    return cfg, w, HipInferenceModel(cfg, {k: v.to(gpu) for k, v in w.items()})


@pytest.mark.parametrize("experts,top,ff,shared,hidden,rows", [(*c, 256, r) for c in [(1, 1, 96, 0), (3, 2, 200, 64), (64, 3, 72, 0)]
                                                               for r in (2, 7, 8, 9, 16, 17, 31, 33, 70)] + [(48, 3, 200, 0, 512, r) for r in (33, 200, 380)])
def test_experts_with_few_slots(gpu, experts, top, ff, shared, hidden, rows):
    """1 to 70 slots per expert (8, 16 and 32 activation rows per tile, one tile and several, an expert without slots), widths that end inside a
    block of 16 weight rows, and of 48 (48 experts x 11 blocks: both products, about 2, 12 and 24 slots per expert): `rows` sequences of one token each, every one against the restatement in 64 bits; the bound is the layer-list
    decoders' (3 % of the logits' spread in bf16).  Left out are rows whose best unchosen expert is closer to the chosen ones than bf16 rounding of
    the stream can move a router logit (0.02 of the logits' spread)."""
    cfg, w, m = moe_model(gpu, experts, top, ff, shared, hidden)
    w64, c = {k: v.double() for k, v in w.items()}, cfg.to_json()
    ids = torch.randint(0, cfg.vocab_size, (rows,), generator=torch.Generator().manual_seed(rows)).tolist()
    seqs = [m.seq_open() for _ in ids]
    lg, _ = m.forward_batch([(s, [i], [0]) for s, i in zip(seqs, ids)])
    seen, z = [], []
    for i in ids:
        h = V.layer_norm(w64["embed"][[i]] * cfg.embed_scale, w64["l0.norm1"], w64["l0.norm1.b"], c["norm"]["eps"])
        mx, pos = c["layers"][0]["mixer"], torch.arange(1)
        x = w64["embed"][[i]] * cfg.embed_scale + V.latent_mixer(h, w64, "l0.mix.", mx, V.latent_kv(h, w64, "l0.mix.", mx, c["norm"]["eps"], pos), pos)
        z.append((V.layer_norm(x, w64["l0.norm2"], w64["l0.norm2.b"], c["norm"]["eps"]) @ w64["l0.mlp.router"].T)[0])
        seen.append(V.forward(c, w64, [i])[0].numpy())
    ref, z = np.stack(seen), torch.stack(z)
    near = torch.zeros(rows, dtype=torch.bool)
    if top < experts:
        best = torch.sort(z, -1, descending=True).values
        near = best[:, top - 1] - best[:, top] < 0.02 * z.std()
    keep = ~near.numpy()
    assert keep.sum() >= rows // 2
    err = np.sqrt(((lg - ref) ** 2).mean(1)) / ref.std()
    assert err[keep].max() < 0.03, (err, near)
    for s in seqs:
        m.seq_close(s)
    m.close()


@pytest.mark.parametrize("n", [2, 3, 33])
def test_argmax_of_many_rows(gpu, n):
    """Every wanted row's first maximal index, from the same logits that the step returns."""
    cfg, _, m = moe_model(gpu, 3, 2, 64, 0, vocab=9001)
    s = m.seq_open()
    lg, am = m.forward_batch([(s, list(range(1, n + 1)), list(range(n)))], want_argmax=True)
    assert (am == lg.argmax(1)).all()
    m.seq_close(s)
    m.close()


@pytest.mark.parametrize("rows", [1, 8, 9, 17, 33, 64, 65, 96, 131])
@pytest.mark.parametrize("dim,vdim,chunk", [(32, 64, 0), (21, 40, 50), (64, 136, 1000), (20, 300, 7)])
def test_32_bit_mode_by_row_count(gpu, rows, dim, vdim, chunk):
    """The 32-bit mode's products (few rows by 8 / 16 / 32 / 64, tiles of 32 rows with a short last one) and its attention (pages dealt to four
    waves, head dims with and without whole groups of four, every width class of the values, chunks that leave waves without a page): a prompt of
    `rows` tokens and one more token behind it, within the layer-list decoders' bound for 32 bits (2e-5 of the logits' spread)."""
    from aha_amd.configs_layered import DosovikConfig, LayerConfig
    from oracle import dosovik as D
    lay = LayerConfig(heads=4, kv_heads=2, dim=dim, vdim=vdim, chunk=chunk, rope_dims=16, rope_base=1e4, scale=dim ** -0.5, ff=200)
    cfg = DosovikConfig(hidden_size=200, vocab_size=1000, layers=[lay, lay], embed_scale=14.0, post_norm_alpha=1.3, compute_dtype="float32")
    w = weights_layered.dosovik_weights(cfg, seed=5)
    m = HipInferenceModel(cfg, {k: v.to(gpu) for k, v in w.items()})
    ids = torch.randint(0, 1000, (rows + 1,), generator=torch.Generator().manual_seed(rows)).tolist()
    js = cfg.to_json()
    for l in js["layers"]:
        l["mixer"]["mask"]["size"] = l["mixer"]["mask"]["size"] or 1 << 20
    ref = D.forward(js, {k: v.double() for k, v in w.items()}, ids).numpy()
    s = m.seq_open()
    got = np.concatenate([m.forward_batch([(s, ids[:rows], list(range(rows)))])[0], m.forward_batch([(s, ids[rows:], [0])])[0]])
    assert np.abs(got - ref).max() < 2e-5 * ref.std() * 4 and np.sqrt(((got - ref) ** 2).mean()) < 2e-5 * ref.std()
    m.seq_close(s)
    m.close()


@pytest.mark.parametrize("rows", [1, 9, 17])
def test_32_bit_head_in_wide_blocks(gpu, rows):
    """A vocabulary whose head makes 515 blocks of 48 weight rows, the last one short, for 8, 16 and 32 activation rows; the bound of the test above."""
    from aha_amd.configs_layered import DosovikConfig, LayerConfig
    from oracle import dosovik as D
    lay = LayerConfig(heads=4, kv_heads=2, dim=32, vdim=32, chunk=1 << 20, rope_dims=16, rope_base=1e4, scale=32 ** -0.5, ff=200)
    cfg = DosovikConfig(hidden_size=200, vocab_size=24700, layers=[lay], embed_scale=14.0, post_norm_alpha=1.3, compute_dtype="float32")
    w = weights_layered.dosovik_weights(cfg, seed=6)
    m = HipInferenceModel(cfg, {k: v.to(gpu) for k, v in w.items()})
    ids = torch.randint(0, 24700, (rows,), generator=torch.Generator().manual_seed(rows)).tolist()
    ref = D.forward(cfg.to_json(), {k: v.double() for k, v in w.items()}, ids).numpy()
    s = m.seq_open()
    got, _ = m.forward_batch([(s, ids, list(range(rows)))])
    assert np.abs(got - ref).max() < 2e-5 * ref.std() * 4 and np.sqrt(((got - ref) ** 2).mean()) < 2e-5 * ref.std()
    m.seq_close(s)
    m.close()
