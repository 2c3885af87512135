"""What this framework is timed on: requests as a serving program sends them, through the public entry points (process_images, forward_initial,
forward_step, decode_greedy, generate_generic_sampled, embed_multi, forward_batch), at the sizes of the repository's own model configurations.

Every pass is a whole request (or a whole batch of requests): the cache is empty before it and prompt, decoding and logits are part of it, so a
pass can be repeated on the same state.  Weights are random, with two structures that trained weights have and random ones lack, because without
them outputs would hang on the order of sums: a token's successor stands out among the logits (greedy and sampled tokens are the same for every
correct implementation), and a token's experts stand out among the router's scores.

`exact` restates the models in 64 bits with plain torch operations on whole sequences, without caches."""
from __future__ import annotations

import math

import numpy as np
import torch

DEV = "cuda:0"
TEXT_IDS = 151642       # ids below the special tokens (an even number of them)


# ---- the cases ----------------------------------------------------------------------------------------------------------------------------------

def listed():
    return [
        # one short question, sampled with temperature / top-k / top-p by the host loop: one launch chain and one host round trip per token
        {"name": "chat_0.6b_sampled", "kind": "text", "prompt": 19, "new": 12, "sampled": True},
        # a document of 2 k tokens continued by 256 tokens in the device-resident greedy loop
        {"name": "text_0.6b_2k", "kind": "text", "prompt": 2048, "new": 256, "sampled": False},
        # text embeddings of a handful of documents of unequal lengths (retrieval, reranking): prompts only, no logits
        {"name": "embed_0.6b_docs", "kind": "embed", "docs": 8, "prompt": 300},
        # two thumbnails and one sentence to the 8B vision-language model, a short answer
        {"name": "vl_8b_thumbs", "kind": "vl", "images": 2, "height": 256, "width": 320, "prompt": 37, "new": 8},
        # the headline request: one 1024 x 1024 image and 512 text tokens, time to the first token's logits
        {"name": "vl_8b_1024_prefill", "kind": "vl", "images": 1, "height": 1024, "width": 1024, "prompt": 512, "new": 1},
        # a photo of no convenient size (resized on the way in) and a question, an answer of 64 tokens
        {"name": "vl_8b_photo_answer", "kind": "vl", "images": 1, "height": 720, "width": 1090, "prompt": 61, "new": 64},
        # a large image and a long text: 8 k tokens
        {"name": "vl_8b_2048_long", "kind": "vl", "images": 1, "height": 2048, "width": 2048, "prompt": 4096, "new": 1},
        # transcription of 30 s of sound from raw samples
        {"name": "asr_0.6b_30s", "kind": "asr", "samples": 480000, "new": 48},
        # eight requests of unequal lengths served together by the post-norm layer list
        {"name": "dosovik_8b_batch8", "kind": "layers", "arch": "dosovik", "size": "8b", "layers": 12, "dtype": "bfloat16", "batch": 8, "prompt": 260, "new": 32},
        # thirty-two short requests served together by the state-space / latent-attention / experts layer list
        {"name": "vamatar_8b_batch32", "kind": "layers", "arch": "vamatar", "size": "8b", "layers": 12, "dtype": "bfloat16", "batch": 32, "prompt": 90, "new": 24},
        # one long prompt of the same design at the small size, continued token by token
        {"name": "vamatar_0.6b_7k", "kind": "layers", "arch": "vamatar", "size": "0.6b", "layers": 28, "dtype": "bfloat16", "batch": 1, "prompt": 7001, "new": 48},
        # 32-bit computation (what a comparison against another framework runs), two sequences
        {"name": "dosovik_0.6b_f32", "kind": "layers", "arch": "dosovik", "size": "0.6b", "layers": 8, "dtype": "float32", "batch": 2, "prompt": 150, "new": 6},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["text", "embed", "vl", "vl", "asr", "layers", "layers", "layers"])
    if kind == "text":
        return {"kind": kind, "prompt": log(4, 3000), "new": log(4, 200), "sampled": rng.random() < 0.4}
    if kind == "embed":
        return {"kind": kind, "docs": rng.randint(1, 10), "prompt": log(12, 700)}
    if kind == "vl":
        n = rng.randint(1, 3)
        return {"kind": kind, "images": n, "height": log(200, 1500 // n), "width": log(200, 1500 // n), "prompt": log(5, 3000), "new": log(1, 40)}
    if kind == "asr":
        return {"kind": kind, "samples": log(8000, 960000), "new": log(2, 60)}
    size, dtype = rng.choice([("8b", "bfloat16"), ("0.6b", "bfloat16"), ("0.6b", "float32")])
    f32 = dtype == "float32"
    batch = rng.choice([1, 2, 3, 5, 8, 13, 16, 24, 32])
    return {"kind": kind, "arch": rng.choice(["dosovik", "vamatar"]), "size": size, "layers": 12 if size == "8b" else rng.choice([4, 8] if f32 else [8, 28]),
            "dtype": dtype, "batch": min(batch, 5) if f32 else batch, "prompt": log(3, 200 if f32 else max(12, 6000 // batch)), "new": log(2, 8 if f32 else 40)}


# ---- inputs -------------------------------------------------------------------------------------------------------------------------------------

def _config(case):
    from aha_amd import configs, configs_layered
    kind = case["kind"]
    if kind in ("text", "embed"):
        return configs.qwen3_0_6b()
    if kind == "vl":
        return configs.qwen3vl_8b()
    if kind == "asr":
        return configs.qwen3_asr_0_6b()
    t = configs.qwen3vl_8b_text() if case["size"] == "8b" else configs.qwen3_0_6b()
    t.vocab_size = 32768
    make = configs_layered.dosovik_like if case["arch"] == "dosovik" else configs_layered.vamatar_like
    cfg = make(t, layers=case["layers"])
    cfg.compute_dtype = case["dtype"]
    return cfg


def _successors(n, seed):
    """A permutation of range(n) that is one cycle: the token that follows each token."""
    order = torch.randperm(n, generator=torch.Generator().manual_seed(seed))
    after = torch.empty(n, dtype=torch.int64)
    after[order] = torch.roll(order, -1)
    return after


def _tied(w, embed, norm, seed):
    """Tied embedding and head: tokens 2i and 2i + 1 follow each other (their rows differ by the signs that the final norm puts on the stream)."""
    e = w[embed].float()
    sign = (torch.randint(0, 2, (e.shape[1],), generator=torch.Generator().manual_seed(seed)).float() * 2 - 1).to(e.device)
    e[1:TEXT_IDS:2] = e[0:TEXT_IDS:2] * sign
    w[embed], w[norm] = (e * 32).bfloat16(), sign.bfloat16()
    return torch.arange(e.shape[0]) ^ 1


def _weights(case, cfg, seed):
    """(weights on the GPU, the token that follows each token)"""
    from aha_amd import weights, weights_layered
    kind = case["kind"]
    if kind in ("text", "embed"):
        w = weights.qwen3_text_weights(cfg, seed=seed, device=DEV)
        return w, _tied(w, "model.embed_tokens.weight", "model.norm.weight", seed)
    if kind == "asr":
        w = weights.qwen3_asr_weights(cfg, seed=seed, device=DEV)
        return w, _tied(w, "thinker.model.embed_tokens.weight", "thinker.model.norm.weight", seed)
    if kind == "vl":
        w = weights.qwen3vl_weights(cfg, seed=seed, device=DEV)
        after = _successors(TEXT_IDS, seed)
        e = w["model.language_model.embed_tokens.weight"]
        w["lm_head.weight"][after.to(DEV)] = e[:TEXT_IDS]
        w["model.language_model.embed_tokens.weight"] = e * 128      # a power of two: exact
        return w, after
    w = (weights_layered.dosovik_weights if case["arch"] == "dosovik" else weights_layered.vamatar_weights)(cfg, seed=seed, device=DEV)
    for name in w:      # sublayers that add less than a unit each, so that the token's own row is still seen behind the last of them
        if name.endswith((".mix.o", ".down")):
            w[name] *= 0.5
    routers = [n for n in w if n.endswith(".router")]
    if routers:         # every token belongs to `top` experts of each layer
        H, E, top = cfg.hidden_size, w[routers[0]].shape[0], next(l.mlp.top for l in cfg.layers if hasattr(l.mlp, "top"))
        gen = torch.Generator(device=DEV).manual_seed(seed + 1)
        d = torch.randn(E, H, generator=gen, device=DEV)
        d /= d.norm(dim=1, keepdim=True)
        for i, n in enumerate(routers):
            w[n] = (0.25 * torch.roll(d, 7 * i + 1, 0)).to(w[n].dtype)
        own = torch.rand(cfg.vocab_size, E, generator=gen, device=DEV).topk(top, dim=1).indices
        e = w["embed"].float()
        w["embed"] = (e + 0.4 * e.norm(dim=1, keepdim=True) * d[own].sum(1)).to(w["embed"].dtype)
    after = _successors(cfg.vocab_size, seed)
    w["head"][after.to(DEV)] = w["embed"] if cfg.embed_scale == 1 else (w["embed"].float() * (cfg.embed_scale * cfg.hidden_size ** -0.5)).to(w["head"].dtype)
    return w, after


def _lengths(n, mean, rng):
    """n unequal lengths around `mean`, from a quarter of it to twice it"""
    return [max(1, int(round(mean * x))) for x in np.exp(rng.uniform(math.log(0.25), math.log(2.0), n))] if n > 1 else [mean]


def _inputs(case, cfg, seed):
    """Token ids of every request, and what else it brings (images: u8 tensors on the GPU; sound: f32 samples on the host)."""
    rng = np.random.default_rng([seed, 5])
    kind = case["kind"]

    def text(n, hi=TEXT_IDS):
        return rng.integers(0, hi, n).tolist()
    if kind == "text":
        return {"ids": [text(case["prompt"])]}
    if kind == "embed":
        return {"ids": [text(n) for n in _lengths(case["docs"], case["prompt"], rng)]}
    if kind == "layers":
        return {"ids": [text(n, cfg.vocab_size) for n in _lengths(case["batch"], case["prompt"], rng)]}
    if kind == "asr":
        from aha_amd.audio_host import audio_prompt_ids
        t = np.arange(case["samples"]) / 16000.0       # a voiced sound that comes and goes, and noise
        wave = 0.25 * np.sin(2 * np.pi * 3 * t) * np.sin(2 * np.pi * rng.uniform(90, 250) * t) + rng.normal(0, 0.05, case["samples"])
        return {"ids": [audio_prompt_ids(cfg, case["samples"], text(9), text(5))], "wave": np.clip(wave, -1, 1).astype(np.float32)}
    from aha_amd.vision_host import img_smart_resize
    gen = torch.Generator(device=DEV).manual_seed(seed + 2)
    images, ids, grids = [], text(4), []
    for _ in range(case["images"]):
        h, w = case["height"], case["width"]
        smooth = torch.nn.functional.interpolate(torch.rand(1, 3, 9, 9, generator=gen, device=DEV), (h, w), mode="bicubic")[0]   # areas, edges and grain
        img = (smooth * 220 + torch.randn(3, h, w, generator=gen, device=DEV) * 6).clamp(0, 255).to(torch.uint8)
        images.append(img.permute(1, 2, 0).contiguous())
        th, tw = img_smart_resize(h, w)
        grids.append((th // 16, tw // 16))
        ids = ids + [cfg.vision_start_token_id] + [cfg.image_token_id] * (th * tw // 1024) + [cfg.vision_end_token_id]
    return {"ids": [ids + text(case["prompt"])], "images": images, "grids": grids}


def prepare(case, seed):
    from aha_amd.model import HipInferenceModel
    cfg = _config(case)
    w, _ = _weights(case, cfg, seed)
    s = dict(_inputs(case, cfg, seed), case=case, cfg=cfg)
    torch.cuda.synchronize()
    s["model"] = HipInferenceModel(cfg, w, kv_reserve_tokens=sum(len(i) for i in s["ids"]) + 64 * (len(s["ids"]) + 4))
    return s


# ---- a pass -------------------------------------------------------------------------------------------------------------------------------------

def run(s):
    case, m, ids = s["case"], s["model"], s["ids"]
    kind = case["kind"]
    if kind == "embed":
        return {"embeddings": m.embed_multi(ids)}
    if kind == "layers" and case["batch"] > 1:
        return _run_batch(m, ids, case["new"])
    if case.get("sampled"):
        from aha_amd.sampling import GenerationContext, generate_generic_sampled
        ctx = GenerationContext(temperature=0.7, top_p=0.8, top_k=20, repeat_penalty=1.05, repeat_last_n=64, seed=299792458, initial_seq_len=len(ids[0]),
                                max_tokens=case["new"])
        tokens = generate_generic_sampled(m, ids[0], ctx)
        return {"tokens": np.asarray(tokens, dtype=np.int64), "last": m.last_logits()}
    data = None
    if kind == "vl":
        from aha_amd.vision_host import process_images
        data = process_images(s["images"], s["cfg"])
    elif kind == "asr":
        from aha_amd.model import MultiModalData
        data = MultiModalData(audio_samples=s["wave"])
    m.clear_cache()
    first, tok = m.forward_initial(ids[0], 0, data)
    tokens = [tok]
    if case["new"] > 1:
        tokens += m.decode_greedy(tok, len(ids[0]), case["new"] - 1)
    return {"tokens": np.asarray(tokens, dtype=np.int64), "first": first, "last": m.last_logits()}


def _run_batch(m, ids, new):
    """Requests that start and end together: one ragged prompt step, then a step per token."""
    seqs = [m.seq_open() for _ in ids]
    try:
        first, am = m.forward_batch([(q, i, [len(i) - 1]) for q, i in zip(seqs, ids)], want_logits=True, want_argmax=True)
        tokens, last = [am], first
        for step in range(1, new):
            last, am = m.forward_batch([(q, [int(t)], [0]) for q, t in zip(seqs, am)], want_logits=step == new - 1, want_argmax=True)
            tokens.append(am)
    finally:
        for q in seqs:
            m.seq_close(q)
    return {"tokens": np.stack(tokens, 1).astype(np.int64), "first": first, "last": last}


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------------------------------

def _sizes(case, cfg):
    """(lengths of the prompts, [h, w] patch grids) as _inputs makes them for any seed (unequal lengths: their mean)"""
    kind = case["kind"]
    if kind == "asr":
        from aha_amd.audio_host import get_feat_extract_output_lengths
        return [get_feat_extract_output_lengths(case["samples"] // 160) + 16], []
    if kind == "vl":
        from aha_amd.vision_host import img_smart_resize
        th, tw = img_smart_resize(case["height"], case["width"])
        return [4 + case["images"] * (th * tw // 1024 + 2) + case["prompt"]], [(th // 16, tw // 16)] * case["images"]
    n = case.get("docs", case.get("batch", 1))
    return [case["prompt"] if n == 1 else max(1, round(0.84 * case["prompt"]))] * n, []


def work(case):
    """Weights once for the prompt step and once for every decoding step, cached keys and values (or states) once per step, logits; two operations
    per weight and token and for attention's two products over the visible keys."""
    cfg = _config(case)
    lens, grids = _sizes(case, cfg)
    kind, new = case["kind"], case.get("new", 1)
    rows, B = sum(lens), len(lens)
    esz = 4 if case.get("dtype") == "float32" else 2
    nbytes = flops = 0.0
    if kind == "layers":
        H = cfg.hidden_size
        head = cfg.vocab_size * H
        for l in cfg.layers:
            x = getattr(l, "mixer", l)
            if hasattr(x, "state"):
                inner = x.heads * x.vdim
                mix = H * (2 * inner + 2 * x.groups * x.state + x.heads) + H * inner
                cache = lambda n, x=x: 2 * 4 * x.heads * x.vdim * x.state          # noqa: E731  the state, read and written
                pair, vis = 0, lambda n: 0                                          # noqa: E731
                extra = 6 * x.heads * x.vdim * x.state                               # per token
            elif hasattr(x, "kv_rank"):
                mix = H * (x.heads * (x.dim + x.rot_dim) + x.kv_rank + x.rot_dim) + x.kv_rank * x.heads * (x.dim + x.vdim) + H * x.heads * x.vdim
                cache = lambda n, x=x: esz * (x.kv_rank + x.rot_dim) * min(n, x.window or n)   # noqa: E731
                pair, vis = 2 * x.heads * (x.dim + x.rot_dim + x.vdim), lambda n, x=x: min(n, x.window or n)   # noqa: E731
                extra = 0
            else:
                mix = H * (x.heads * x.dim + x.kv_heads * (x.dim + x.vdim)) + H * x.heads * x.vdim
                cache = lambda n, x=x: esz * x.kv_heads * (x.dim + x.vdim) * min(n, x.chunk)   # noqa: E731
                pair, vis = 2 * x.heads * (x.dim + x.vdim), lambda n, x=x: min(n, x.chunk)     # noqa: E731
                extra = 0
            ml = l.mlp if hasattr(l, "mlp") else None
            if ml is None:
                ff_tok = 2 * H * getattr(l, "ff", 0)
                ff_read = lambda t: ff_tok                                           # noqa: E731
            elif hasattr(ml, "experts"):
                ff_tok = 3 * H * (ml.top * ml.ff + ml.shared_ff) + H * ml.experts
                ff_read = lambda t, ml=ml: 3 * H * (ml.experts * (1 - (1 - ml.top / ml.experts) ** t) * ml.ff + ml.shared_ff) + H * ml.experts  # noqa: E731
            else:
                ff_tok = 3 * H * ml.ff
                ff_read = lambda t, ml=ml: 3 * H * ml.ff                             # noqa: E731
            nbytes += esz * (mix + ff_read(rows)) + (new - 1) * esz * (mix + ff_read(B)) + sum(cache(n) for n in lens)
            nbytes += sum(cache(n + new // 2) for n in lens) * (new - 1)
            tok = rows + B * (new - 1)
            flops += tok * (2 * (mix + ff_tok) + extra)
            flops += pair * sum((n * vis(n) - vis(n) ** 2 / 2) + (new - 1) * vis(n + new // 2) for n in lens)
        nbytes += new * (esz * head + 4 * B * cfg.vocab_size)
        flops += 2.0 * new * B * head
        return {"bytes": nbytes, "flops": flops}
    t = cfg.text if hasattr(cfg, "text") else cfg
    H, d = t.hidden_size, t.head_dim
    layer = H * (t.num_attention_heads + 2 * t.num_key_value_heads) * d + t.num_attention_heads * d * H + 3 * H * t.intermediate_size
    stack, head = layer * t.num_hidden_layers, t.vocab_size * H
    if kind == "embed":
        for n in lens:
            flops += 2.0 * n * stack + 2.0 * t.num_hidden_layers * t.num_attention_heads * d * n * n
            nbytes += 2.0 * stack
        return {"bytes": nbytes, "flops": flops}
    n = lens[0]
    kv = 2 * 2 * t.num_key_value_heads * d * t.num_hidden_layers
    nbytes += new * (2.0 * (stack + head) + 4 * t.vocab_size) + n * kv + (new - 1) * (n + new / 2) * kv
    flops += 2.0 * stack * (n + new - 1) + 2.0 * head * new
    flops += 2.0 * t.num_hidden_layers * t.num_attention_heads * d * (n * n + 2 * (new - 1) * (n + new / 2))
    for h, w in grids:
        v = cfg.vision
        block = 4 * v.hidden_size ** 2 + 2 * v.hidden_size * v.intermediate_size
        merge = (4 * v.hidden_size) ** 2 + 4 * v.hidden_size * v.out_hidden_size
        vit = v.depth * block + v.patch_dim * v.hidden_size
        flops += 2.0 * h * w * (vit + merge) + 4.0 * v.depth * v.hidden_size * (h * w) ** 2
        nbytes += 2.0 * (vit + 4 * merge) / len(grids) + 3 * case["height"] * case["width"]
    if kind == "asr":
        a = cfg.audio
        frames, A = case["samples"] // 160, a.downsample_hidden_size
        enc = a.encoder_layers * (4 * a.d_model ** 2 + 2 * a.d_model * a.encoder_ffn_dim)
        flops += 2.0 * enc * n + 4.0 * a.encoder_layers * a.d_model * n * n + 2.0 * frames * 9 * A * (64 / 2 + A * 32 / 4 + A * 16 / 8) + 2.0 * n * 16 * A * a.d_model
        nbytes += 2.0 * (enc + 18 * A * A + 16 * A * a.d_model) + 4 * case["samples"]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what the present implementation is off from `exact`, and no more than 3 %: 1.2e-6 in 32 bits; in bf16 0.4 % (12 layers with
    an f32 residual stream), 0.5 to 0.9 % (the same with a recurrence), 1.3 % (28 layers whose residual stream is bf16), 2.9 % (36 such layers).
    Tokens stand out by many standard deviations: none may differ."""
    if case.get("dtype") == "float32":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.0}
    if case.get("arch") == "dosovik":
        return {"rel": 0.016, "max": 0.15, "differ": 0.0}
    return {"rel": 0.03, "max": 0.25, "differ": 0.0}


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------------------------------------

def _lin(x, w, b=None):
    y = x @ w.double().reshape(w.shape[0], -1).T
    return y if b is None else y + b.double()


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _ln(x, w, b, eps):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w.double() + b.double()


def _rot(x, cos, sin):
    """The last axis of x (S, heads, d) rotated, dimension i with i + d / 2; cos, sin (S, d / 2)"""
    a, b = x.chunk(2, -1)
    c, s = cos[:, None], sin[:, None]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _angles(pos, d, base):
    f = base ** (-torch.arange(0, d, 2, dtype=torch.float64, device=DEV) / d)
    return torch.as_tensor(pos, dtype=torch.float64, device=DEV)[:, None] * f


def _attend(q, k, v, scale, low=None, causal=True, sink=False):
    """q (S, H, d), k (S, G, d), v (S, G, dv) -> (S, H * dv); low (S): the first key that a row sees"""
    S, H, d = q.shape
    G = k.shape[1]
    kt, vt = k.permute(1, 2, 0).contiguous(), v.transpose(0, 1).contiguous()
    step = max(1, int(2.5e8 // (H * S)))
    out = []
    for a in range(0, S, step):
        b = min(S, a + step)
        qq = q[a:b].reshape(b - a, G, H // G, d).permute(1, 2, 0, 3).reshape(G, -1, d)
        s = (torch.matmul(qq, kt) * scale).reshape(G, H // G, b - a, S)
        if causal:
            i, j = torch.arange(a, b, device=DEV)[:, None], torch.arange(S, device=DEV)[None]
            hide = j > i
            if low is not None:
                hide = hide | (j < low[a:b, None])
            s.masked_fill_(hide, -math.inf)
        m = s.amax(-1, keepdim=True)
        if sink:
            m = m.clamp(min=0.0)
        s.sub_(m).exp_()
        z = s.sum(-1, keepdim=True) + (torch.exp(-m) if sink else 0.0)
        o = torch.matmul(s.div_(z).reshape(G, -1, S), vt).reshape(G, H // G, b - a, -1)
        out.append(o.permute(2, 0, 1, 3).reshape(b - a, -1))
    return torch.cat(out, 0)


def _qwen3(w, t, prefix, x, angles, deep=None, rows=None):
    """The decoder stack on embedded rows x (S, H) -> final-norm rows"""
    cos, sin = angles.cos(), angles.sin()
    S, eps = x.shape[0], t.rms_norm_eps
    for i in range(t.num_hidden_layers):
        p = f"{prefix}layers.{i}."
        h = _rms(x, eps) * w[p + "input_layernorm.weight"].double()
        q, k, v = (_lin(h, w[f"{p}self_attn.{n}_proj.weight"]).reshape(S, -1, t.head_dim) for n in "qkv")
        q, k = (_rot(_rms(y, eps) * w[f"{p}self_attn.{n}_norm.weight"].double(), cos, sin) for y, n in ((q, "q"), (k, "k")))
        x = x + _lin(_attend(q, k, v, t.head_dim ** -0.5), w[p + "self_attn.o_proj.weight"])
        h = _rms(x, eps) * w[p + "post_attention_layernorm.weight"].double()
        x = x + _lin(torch.nn.functional.silu(_lin(h, w[p + "mlp.gate_proj.weight"])) * _lin(h, w[p + "mlp.up_proj.weight"]), w[p + "mlp.down_proj.weight"])
        if deep is not None and i < len(deep):
            x[rows] += deep[i]
    return _rms(x, eps) * w[prefix + "norm.weight"].double()


def _catmull_rom(n_in, n_out):
    """(n_out, n_in): rows of normalised weights"""
    ratio = n_in / n_out
    width = max(ratio, 1.0)
    m = np.zeros((n_out, n_in))
    for o in range(n_out):
        c = (o + 0.5) * ratio
        lo, hi = max(0, math.floor(c - 2 * width)), min(n_in, math.ceil(c + 2 * width))
        a = np.abs((np.arange(lo, hi) - (c - 0.5)) / width)
        k = np.where(a < 1, 1.5 * a ** 3 - 2.5 * a ** 2 + 1, np.where(a < 2, -0.5 * a ** 3 + 2.5 * a ** 2 - 4 * a + 2, 0.0))
        m[o, lo:hi] = k / k.sum()
    return torch.from_numpy(m).to(DEV)


def _blocks(a, h, w):
    """(h, w, ...) -> (h * w, ...) in windows of 2 x 2"""
    return a.reshape(h // 2, 2, w // 2, 2, *a.shape[2:]).transpose(1, 2).reshape(h * w, *a.shape[2:])


def _vision(w, v, image, grid):
    """One u8 image -> (its rows for the text stack, the rows added behind the first text layers)"""
    gh, gw = grid
    img = image.double()
    if img.shape[:2] != (gh * 16, gw * 16):
        img = torch.einsum("oh,hwc->owc", _catmull_rom(img.shape[0], gh * 16), img)
        img = torch.einsum("pw,owc->opc", _catmull_rom(img.shape[1], gw * 16), img).clamp(0, 255).add(0.5).floor()
    px = (img / 255 - 0.5) / 0.5
    px = _blocks(px.reshape(gh, 16, gw, 16, 3).transpose(1, 2), gh, gw).permute(0, 3, 1, 2)          # (N, 3, 16, 16)
    p = "model.visual."
    N, D, d = gh * gw, v.hidden_size, v.head_dim
    x = _lin(px[:, :, None].expand(N, 3, 2, 16, 16).reshape(N, -1), w[p + "patch_embed.proj.weight"], w[p + "patch_embed.proj.bias"])
    G = int(math.isqrt(v.num_position_embeddings))
    table = w[p + "pos_embed.weight"].double().reshape(G, G, D)

    def line(n):
        m = torch.zeros(n, G, dtype=torch.float64, device=DEV)
        at = torch.arange(n, dtype=torch.float64, device=DEV) * ((G - 1) / (n - 1) if n > 1 else 0.0)
        lo = at.floor().long().clamp(max=G - 1)
        m[torch.arange(n), lo] += 1 - (at - lo)
        m[torch.arange(n), (lo + 1).clamp(max=G - 1)] += at - lo
        return m
    x = x + _blocks(torch.einsum("yg,ghd,xh->yxd", line(gh), table, line(gw)), gh, gw)
    yy, xx = torch.meshgrid(torch.arange(gh), torch.arange(gw), indexing="ij")
    ang = torch.cat([_angles(_blocks(a, gh, gw), d // 2, 10000.0) for a in (yy, xx)], 1)
    cos, sin = ang.cos(), ang.sin()

    def merger(q, x, behind):
        M = 4 * D
        y = x.reshape(-1, M) if behind else x
        y = _ln(y, w[q + "norm.weight"], w[q + "norm.bias"], 1e-6).reshape(-1, M)
        y = torch.nn.functional.gelu(_lin(y, w[q + "linear_fc1.weight"], w[q + "linear_fc1.bias"]))
        return _lin(y, w[q + "linear_fc2.weight"], w[q + "linear_fc2.bias"])
    deep = []
    for i in range(v.depth):
        q = f"{p}blocks.{i}."
        h = _ln(x, w[q + "norm1.weight"], w[q + "norm1.bias"], 1e-6)
        a, b, c = _lin(h, w[q + "attn.qkv.weight"], w[q + "attn.qkv.bias"]).reshape(N, 3, -1, d).unbind(1)
        o = _attend(_rot(a, cos, sin), _rot(b, cos, sin), c, d ** -0.5, causal=False)
        x = x + _lin(o, w[q + "attn.proj.weight"], w[q + "attn.proj.bias"])
        h = _ln(x, w[q + "norm2.weight"], w[q + "norm2.bias"], 1e-6)
        h = torch.nn.functional.gelu(_lin(h, w[q + "mlp.linear_fc1.weight"], w[q + "mlp.linear_fc1.bias"]), approximate="tanh")
        x = x + _lin(h, w[q + "mlp.linear_fc2.weight"], w[q + "mlp.linear_fc2.bias"])
        if i in v.deepstack_visual_indexes:
            deep.append(merger(f"{p}deepstack_merger_list.{len(deep)}.", x, True))
    return merger(p + "merger.", x, False), deep


def _rope_index(ids, cfg, grids):
    """(3, S) positions: text counts up; an image's tokens share one time and have their row and column"""
    pos, at, g = [], 0, iter(grids)
    i = 0
    while i < len(ids):
        if ids[i] == cfg.image_token_id:
            h, w = (x // 2 for x in next(g))
            y, x = np.divmod(np.arange(h * w), w)
            pos.append(np.stack([np.full(h * w, at), at + y, at + x]))
            at += max(h, w)
            i += h * w
        else:
            pos.append(np.full((3, 1), at))
            at += 1
            i += 1
    return np.concatenate(pos, 1)


def _mel(wave):
    """Log-mel features (128, frames) of 16 kHz samples: 400-sample symmetric Hann windows every 160, Slaney mel triangles, 8 dB-decades of range"""
    x = wave.astype(np.float64)
    y = np.concatenate([x[1:201][::-1], x])
    y = np.concatenate([y, y[len(x) - 200:len(x)][::-1]])        # the right edge is cut at the unpadded index, as the frontend's definition has it
    frames = (len(y) - 400) // 160                                # the last frame is dropped
    idx = np.arange(400)[None] + 160 * np.arange(frames)[:, None]
    win = 0.5 - 0.5 * np.cos(2 * np.pi * np.arange(400) / 399)
    power = np.abs(np.fft.rfft(y[idx] * win, axis=1)) ** 2
    top = 15 + math.log(8.0) * 27 / math.log(6.4)
    m = np.linspace(0.0, top, 130)
    hz = np.where(m < 15, m * 200 / 3, 1000 * np.exp(math.log(6.4) / 27 * (m - 15)))
    fft = np.linspace(0, 8000, 201)
    up = (fft[:, None] - hz[None, :-2]) / (hz[1:-1] - hz[:-2])
    down = (hz[None, 2:] - fft[:, None]) / (hz[2:] - hz[1:-1])
    bank = np.maximum(np.minimum(up, down), 0) * (2 / (hz[2:] - hz[:-2]))
    lg = np.log10(np.maximum(power @ bank, 1e-10)).T
    return (np.maximum(lg, lg.max() - 8) + 4) * 0.25


def _sound(w, a, feats):
    p = "thinker.audio_tower."
    C = a.n_window * 2
    F = feats.shape[1]
    x = torch.nn.functional.pad(torch.from_numpy(feats).to(DEV), (0, -F % C)).reshape(128, -1, C).transpose(0, 1)[:, None]
    gelu = torch.nn.functional.gelu

    def out(n):
        for _ in range(3):
            n = (n - 1) // 2 + 1
        return n
    for n in ("conv2d1", "conv2d2", "conv2d3"):                  # 3 x 3, stride 2, as a product over gathered columns
        k, b = w[p + n + ".weight"], w[p + n + ".bias"]
        hh, ww = (x.shape[2] - 1) // 2 + 1, (x.shape[3] - 1) // 2 + 1
        cols = torch.nn.functional.unfold(x, 3, padding=1, stride=2)
        x = gelu((k.double().reshape(k.shape[0], -1) @ cols + b.double()[:, None]).reshape(x.shape[0], -1, hh, ww), approximate="tanh")
    n_tok = (F // C) * out(C) + (out(F % C) if F % C else 0)
    B, ch, f, t = x.shape
    x = _lin(x.permute(0, 3, 1, 2).reshape(B, t, ch * f), w[p + "conv_out.weight"])
    ang = _angles(range(t), a.d_model, 10000.0)
    x = (x + torch.cat([ang.sin(), ang.cos()], 1)).reshape(B * t, -1)[:n_tok]
    for i in range(a.encoder_layers):
        q = f"{p}layers.{i}."
        h = _ln(x, w[q + "self_attn_layer_norm.weight"], w[q + "self_attn_layer_norm.bias"], 1e-5)
        s = [_lin(h, w[f"{q}self_attn.{n}_proj.weight"], w[f"{q}self_attn.{n}_proj.bias"]).reshape(n_tok, -1, a.head_dim) for n in "qkv"]
        x = x + _lin(_attend(*s, a.head_dim ** -0.5, causal=False), w[q + "self_attn.out_proj.weight"], w[q + "self_attn.out_proj.bias"])
        h = _ln(x, w[q + "final_layer_norm.weight"], w[q + "final_layer_norm.bias"], 1e-5)
        x = x + _lin(gelu(_lin(h, w[q + "fc1.weight"], w[q + "fc1.bias"])), w[q + "fc2.weight"], w[q + "fc2.bias"])
    x = _ln(x, w[p + "ln_post.weight"], w[p + "ln_post.bias"], 1e-5)
    return _lin(gelu(_lin(x, w[p + "proj1.weight"], w[p + "proj1.bias"])), w[p + "proj2.weight"], w[p + "proj2.bias"])


def _spans(lens):
    at = np.cumsum([0] + list(lens))
    return list(zip(at[:-1].tolist(), at[1:].tolist()))


def _taps(u, w):
    """Causal per-channel convolution of one sequence; the last tap meets the current token"""
    w = w.double()
    out = torch.zeros_like(u)
    for j in range(w.shape[1]):
        back = w.shape[1] - 1 - j
        if back < u.shape[0]:
            out[back:] += w[:, j] * u[: u.shape[0] - back]
    return out


def _dosovik(w, cfg, ids, lens):
    """Rows of several sequences behind one another -> final-norm rows"""
    eps, alpha = cfg.rms_norm_eps, cfg.post_norm_alpha
    x = w["embed"][ids].double() * cfg.embed_scale
    spans = _spans(lens)

    def canon(h, k):
        return torch.cat([h[a:b] + _taps(h[a:b], k) for a, b in spans])

    def norm(y, k):
        return _rms(y, eps) * (1 + k.double())
    first = None
    for i, l in enumerate(cfg.layers):
        p, m = f"l{i}.", f"l{i}.mix."
        h = canon(x, w[p + "canon1"])
        q, k, v = (_lin(h, w[m + n], w[m + n + ".b"]) for n in "qkv")
        q = (_rms(q, eps) * w[m + "q.norm"].double()).reshape(-1, l.heads, l.dim)
        k = (_rms(k, eps) * w[m + "k.norm"].double()).reshape(-1, l.kv_heads, l.dim)
        if l.v_mix:
            first = v if first is None else first
            lam = w[m + "vmix"].double()
            v = v if first is v else (1 - lam) * v + lam * first
        v = v.reshape(-1, l.kv_heads, l.vdim)
        o = []
        for a, b in spans:
            ang = _angles(range(b - a), l.rope_dims, l.rope_base)
            qq, kk = (torch.cat([_rot(y[a:b, :, :l.rope_dims], ang.cos(), ang.sin()), y[a:b, :, l.rope_dims:]], -1) for y in (q, k))
            low = torch.arange(b - a, device=DEV) // l.chunk * l.chunk
            o.append(_attend(qq, kk, v[a:b], l.scale, low, sink=True))
        x = norm(alpha * x + _lin(torch.cat(o), w[m + "o"]), w[p + "norm1"])
        if l.ff:
            z = _lin(canon(x, w[p + "canon2"]), w[p + "mlp.up"])
            c = w[p + "mlp.act"].double()
            z = c[0] * _rms(z, eps) + c[1] * _rms(z ** 2, eps) + c[2] * _rms(z ** 3, eps) + c[3]
            x = norm(alpha * x + _lin(z, w[p + "mlp.down"]), w[p + "norm2"])
    return norm(x, w["final.norm"])


def _recurrence(x, B, C, dt, A, step=64):
    """One sequence: x (S, H, P), B, C (S, G, N), dt (S, H), A (H) -> (S, H, P), `step` tokens at a time"""
    S, H, P = x.shape
    rep = H // B.shape[1]
    state = torch.zeros(H, B.shape[2], P, dtype=torch.float64, device=DEV)
    out = []
    for a in range(0, S, step):
        xx, d = x[a:a + step].transpose(0, 1), dt[a:a + step].T                                       # (H, n, P), (H, n)
        b, c = (y[a:a + step].transpose(0, 1).repeat_interleave(rep, 0) for y in (B, C))               # (H, n, N)
        run = torch.cumsum(A[:, None] * d, 1)
        n = d.shape[1]
        keep = torch.ones(n, n, dtype=torch.bool, device=DEV).tril()
        decay = torch.exp((run[:, :, None] - run[:, None, :]).masked_fill(~keep, -math.inf))
        y = torch.matmul(torch.matmul(c, b.transpose(1, 2)) * decay * d[:, None, :], xx) + torch.exp(run)[:, :, None] * torch.matmul(c, state)
        state = torch.exp(run[:, -1])[:, None, None] * state + torch.matmul((b * (torch.exp(run[:, -1:] - run) * d)[:, :, None]).transpose(1, 2), xx)
        out.append(y.transpose(0, 1))
    return torch.cat(out)


def _vamatar(w, cfg, ids, lens):
    eps, silu = cfg.norm_eps, torch.nn.functional.silu
    x = w["embed"][ids].double() * cfg.embed_scale
    spans = _spans(lens)

    def ff(h, p):
        return _lin(silu(_lin(h, w[p + "gate"])) * _lin(h, w[p + "up"]), w[p + "down"])
    cached = {}
    for i, l in enumerate(cfg.layers):
        p, m, t = f"l{i}.", f"l{i}.mix.", l.mixer
        h = _ln(x, w[p + "norm1"], w[p + "norm1.b"], eps)
        if hasattr(t, "state"):
            inner, gn = t.heads * t.vdim, t.groups * t.state
            z, u, dt = torch.split(_lin(h, w[m + "in"]), [inner, inner + 2 * gn, t.heads], -1)
            u = silu(torch.cat([_taps(u[a:b], w[m + "conv"]) for a, b in spans]) + w[m + "conv.b"].double())
            xs, B, C = torch.split(u, [inner, gn, gn], -1)
            xs, B, C = xs.reshape(-1, t.heads, t.vdim), B.reshape(-1, t.groups, t.state), C.reshape(-1, t.groups, t.state)
            dt, A = torch.nn.functional.softplus(dt + w[m + "dt_bias"].double()), -torch.exp(w[m + "A_log"].double())
            y = torch.cat([_recurrence(xs[a:b], B[a:b], C[a:b], dt[a:b], A) for a, b in spans]) + w[m + "D"].double()[:, None] * xs
            g = y.reshape(-1, inner) * silu(z)
            o = _rms(g.reshape(g.shape[0], t.norm_groups, -1), eps).reshape(g.shape) * w[m + "norm"].double()
        else:
            if t.kv_from is None:
                c, kr = torch.split(_lin(h, w[m + "dkv"]), [t.kv_rank, t.rot_dim], -1)
                ang = torch.cat([_angles(range(b - a), t.rot_dim, t.rope_base) for a, b in spans])
                cached[i] = _rms(c, eps) * w[m + "dkv.norm"].double(), _rot(kr[:, None], ang.cos(), ang.sin())
            c, kr = cached[i if t.kv_from is None else t.kv_from]
            ang = torch.cat([_angles(range(b - a), t.rot_dim, t.rope_base) for a, b in spans])
            q = _lin(h, w[m + "q"]).reshape(-1, t.heads, t.dim + t.rot_dim)
            q = torch.cat([q[..., :t.dim], _rot(q[..., t.dim:], ang.cos(), ang.sin())], -1)
            k = torch.cat([_lin(c, w[m + "uk"]).reshape(-1, t.heads, t.dim), kr.expand(-1, t.heads, -1)], -1)
            v = _lin(c, w[m + "uv"]).reshape(-1, t.heads, t.vdim)
            o = []
            for a, b in spans:
                low = (torch.arange(b - a, device=DEV) - (t.window - 1)).clamp(min=0) if t.window else None
                o.append(_attend(q[a:b], k[a:b], v[a:b], t.scale, low))
            o = torch.cat(o)
        x = x + _lin(o, w[m + "o"])
        if l.mlp is None:
            continue
        h = _ln(x, w[p + "norm2"], w[p + "norm2.b"], eps)
        if not hasattr(l.mlp, "experts"):
            x = x + ff(h, p + "mlp.")
            continue
        score, own = torch.sigmoid(_lin(h, w[p + "mlp.router"])).topk(l.mlp.top, -1)
        y = ff(h, p + "mlp.shared.") if l.mlp.shared_ff else torch.zeros_like(h)
        for e in range(l.mlp.experts):
            at, k = (own == e).nonzero(as_tuple=True)
            if len(at):
                y[at] += ff(score[at, k][:, None] * h[at], f"{p}mlp.e{e}.")
        x = x + y
    return _ln(x, w["final.norm"], w["final.norm.b"], eps)


def exact(case, seed):
    cfg = _config(case)
    w, after = _weights(case, cfg, seed)
    s = _inputs(case, cfg, seed)
    kind, new = case["kind"], case.get("new", 1)
    seqs = []
    for ids in s["ids"]:        # every request with the tokens that follow it; the last of them is not fed back
        ids = list(ids)
        for _ in range(new - 1):
            ids.append(int(after[ids[-1]]))
        seqs.append(ids)
    if kind == "layers":
        lens = [len(i) for i in seqs]
        ids = torch.tensor([t for i in seqs for t in i], device=DEV)
        h = (_dosovik if case["arch"] == "dosovik" else _vamatar)(w, cfg, ids, lens)
        want = torch.tensor([[a + len(p) - 1 + k for k in range(new)] for (a, _), p in zip(_spans(lens), s["ids"])], device=DEV)
        lg = _lin(h[want.reshape(-1)], w["head"])
        cap = getattr(cfg, "logit_softcap", 0.0)
        lg = (cap * torch.tanh(lg / cap) if cap else lg).reshape(len(seqs), new, -1)
        r = {"tokens": lg.argmax(-1), "first": lg[:, 0], "last": lg[:, -1]}
        return {k: v[0] for k, v in r.items()} if len(seqs) == 1 else r
    t = cfg.text if hasattr(cfg, "text") else cfg
    prefix = {"text": "model.", "embed": "model.", "asr": "thinker.model.", "vl": "model.language_model."}[kind]
    if kind == "embed":
        out = []
        for ids in seqs:
            h = _qwen3(w, t, prefix, w[prefix + "embed_tokens.weight"][torch.tensor(ids, device=DEV)].double(), _angles(range(len(ids)), t.head_dim, t.rope_theta))[-1]
            out.append(h / torch.sqrt((h * h).sum() + 1e-6))
        return {"embeddings": torch.stack(out)}
    ids = seqs[0]
    at = torch.tensor(ids, device=DEV)
    x = w[prefix + "embed_tokens.weight"][at].double()
    angles, deep, rows = _angles(range(len(ids)), t.head_dim, t.rope_theta), None, None
    if kind == "asr":
        x[at == cfg.audio_token_id] = _sound(w, cfg.audio, _mel(s["wave"]))
    if kind == "vl":
        seen = [_vision(w, cfg.vision, im, g) for im, g in zip(s["images"], s["grids"])]
        rows = at == cfg.image_token_id
        x[rows] = torch.cat([a for a, _ in seen])
        deep = [torch.cat(d) for d in zip(*(d for _, d in seen))]
        three = [_angles(p, t.head_dim, t.rope_theta) for p in _rope_index(ids, cfg, s["grids"])]
        angles = three[0].clone()
        for axis in (1, 2):
            angles[:, axis:t.mrope_section[axis] * 3:3] = three[axis][:, axis:t.mrope_section[axis] * 3:3]
    h = _qwen3(w, t, prefix, x, angles, deep, rows)
    n = len(s["ids"][0])
    lg = _lin(h[n - 1:], w["lm_head.weight" if kind == "vl" else prefix + "embed_tokens.weight"])
    r = {"tokens": lg.argmax(-1), "first": lg[0], "last": lg[-1]}
    if case.get("sampled"):
        del r["first"]
    return r
