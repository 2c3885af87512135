"""-m gpu: pieces of a batched step -- the arg-max of many rows in one pass."""
import pytest
import torch

from aha_amd import weights_layered
from aha_amd.configs_layered import GatedConfig, LatentConfig, MoeConfig, PreNormLayer, VamatarConfig
from aha_amd.model import HipInferenceModel

pytestmark = pytest.mark.gpu


def moe_model(gpu, experts, top, ff, shared, hidden=256, vocab=5000):
    att = LatentConfig(heads=2, dim=32, rot_dim=16, vdim=32, kv_rank=64, window=64, rope_base=1e4, scale=48 ** -0.5)
    cfg = VamatarConfig(hidden_size=hidden, vocab_size=vocab, layers=[PreNormLayer(att, MoeConfig(ff=ff, experts=experts, top=top, shared_ff=shared)),
                                                                     PreNormLayer(att, GatedConfig(128))], embed_scale=16.0)
    w = weights_layered.vamatar_weights(cfg, seed=3)
    return cfg, w, HipInferenceModel(cfg, {k: v.to(gpu) for k, v in w.items()})


@pytest.mark.parametrize("n", [2, 3, 33])
def test_argmax_of_many_rows(gpu, n):
    """Every wanted row's first maximal index, from the same logits that the step returns."""
    cfg, _, m = moe_model(gpu, 3, 2, 64, 0, vocab=9001)
    s = m.seq_open()
    lg, am = m.forward_batch([(s, list(range(1, n + 1)), list(range(n)))], want_argmax=True)
    assert (am == lg.argmax(1)).all()
    m.seq_close(s)
    m.close()
