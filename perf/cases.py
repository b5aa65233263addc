"""The framework's work, as its users have it done, for timing and for checks of its results.

Five families, each through the engine that serves it:

* ``sd``: Stable Diffusion 2.1 text to image (``StableDiffusionEngine.generate``), the headline workload: one prompt at a time
  for latency, a batch for throughput, 512 x 512 and the sizes around it.  A request has 4 denoising steps here instead of 50:
  every step is the same work, beside one text encoding and one image decoding.
* ``vit``: image classification (``ImageClassifierEngine``, ViT-base/16), uint8 images in, logits out.
* ``t5``: caption embeddings (``TextEmbeddingEngine``, T5-v1.1-large), texts in, one vector each out.
* ``mistral``: an LLM served with continuous batching (``LLMEngine``): the layers, heads and vocabulary of Mistral-7B, 8 of its
  32 layers, so that weights are made quickly.  Requests are fed by ``open_request`` / ``extend`` / ``close_request``, the way
  traces are replayed and texts scored: a packed prefill of all prompts, then decode steps with given tokens.
* ``pugozen``: a layer-list decoder (delta rule, retention, attention beside a delta rule) on the same engine, the small size of
  its benchmark.

Weights and inputs are random, made from the seed.  Every family has a plain fp64 form of its model here (``exact``), which also
says which tensors a checkpoint has: one description for both.
"""
from __future__ import annotations

import functools
import math
import re
import zlib

import torch

GELU = torch.nn.functional.gelu
SILU = torch.nn.functional.silu

WORDS = ("a photo of an astronaut riding horse on mars dramatic lighting red dust highly detailed portrait old castle river "
         "sunset mountain dragon flower garden robot city night sky blue gold").split()
SD_STEPS = 4
MISTRAL_LAYERS = 8
# layers, width, heads, kv heads, head size, recurrence heads, query / key heads of the delta rule, key and value size, rank of
# thin products, feed-forward, vocabulary
PUGOZEN = ("DPRPDPRP", 2048, 16, 4, 128, 16, 8, 128, 128, 128, 8448, 32768)
VOCAB = 32768                       # of both LLMs


def listed():
    return [
        # one image at a time: what a request waits for
        {"name": "sd_1", "kind": "sd", "batch": 1, "height": 512, "width": 512},
        # a replica's batch of requests
        {"name": "sd_8", "kind": "sd", "batch": 8, "height": 512, "width": 512},
        # one image, and a full batch, of a classification service
        {"name": "vit_1", "kind": "vit", "batch": 1},
        {"name": "vit_32", "kind": "vit", "batch": 32},
        # one prompt of a search box, and a batch of captions padded to the service's length
        {"name": "t5_1", "kind": "t5", "batch": 1, "length": 32},
        {"name": "t5_32", "kind": "t5", "batch": 32, "length": 128},
        # one chat: a short prompt, then token by token
        {"name": "mistral_chat", "kind": "mistral", "batch": 1, "prompt": 100, "gen": 32},
        # a full batch of requests, as the throughput benchmark has them
        {"name": "mistral_batch", "kind": "mistral", "batch": 64, "prompt": 128, "gen": 32},
        # one long document
        {"name": "mistral_long", "kind": "mistral", "batch": 1, "prompt": 8000, "gen": 0},
        # the same three of a decoder with recurrent layers
        {"name": "pugozen_chat", "kind": "pugozen", "batch": 1, "prompt": 100, "gen": 32},
        {"name": "pugozen_batch", "kind": "pugozen", "batch": 64, "prompt": 128, "gen": 32},
        {"name": "pugozen_long", "kind": "pugozen", "batch": 7, "prompt": 1100, "gen": 0},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["sd", "vit", "t5", "mistral", "mistral", "pugozen", "pugozen"])
    if kind == "sd":
        h, w = 64 * rng.randint(4, 12), 64 * rng.randint(4, 12)
        return {"kind": kind, "batch": _log(rng, 1, max(1, min(8, 8 * 512 * 512 // (h * w)))), "height": h, "width": w}
    if kind == "vit":
        return {"kind": kind, "batch": _log(rng, 1, 64)}
    if kind == "t5":
        length = _log(rng, 8, 512)
        return {"kind": kind, "batch": _log(rng, 1, min(64, 8192 // length)), "length": length}
    if rng.random() < 0.5:          # prompts only
        batch = _log(rng, 1, 32)
        return {"kind": kind, "batch": batch, "prompt": _log(rng, 16, 8000 // batch), "gen": 0}
    batch = _log(rng, 1, 64)
    return {"kind": kind, "batch": batch, "prompt": _log(rng, 16, min(2000, 8192 // batch)), "gen": _log(rng, 8, 32)}


# ---------------------------------------------------------------------------------------------- weights
class Asked:
    """Stands in for a model's weights on the meta device: notes every tensor that the model asks for."""

    def __init__(self):
        self.tensors = {}

    def __call__(self, name, *shape, std=None, mean=0.0):
        self.tensors.setdefault(name, (shape, shape[-1] ** -0.5 if std is None else std, mean))
        return torch.empty(shape, dtype=torch.float64, device="meta")


class Given:
    """The weights of a model, each in 64 bits when the model asks for it."""

    def __init__(self, tensors):
        self.tensors = tensors

    def __call__(self, name, *shape, std=None, mean=0.0):
        return self.tensors[name].double()


@functools.lru_cache(maxsize=None)
def _tensors(model):
    """{name: (shape, standard deviation, mean)} of every tensor of ``model``'s checkpoint, with a small input."""
    p, ids = Asked(), torch.zeros(1, 3, dtype=torch.long, device="meta")
    if model == "clip":
        _clip(p, ids)
    elif model == "unet":
        z = torch.empty(1, 8, 8, 4, dtype=torch.float64, device="meta")
        _unet(p, z, 1.0, torch.empty(1, 3, 1024, dtype=torch.float64, device="meta"))
    elif model == "vae":
        _vae(p, torch.empty(1, 2, 2, 4, dtype=torch.float64, device="meta"))
    elif model == "vit":
        _vit(p, torch.empty(1, 224, 224, 3, dtype=torch.float64, device="meta"))
    elif model == "t5":
        _t5(p, ids, [3])
    else:
        {"mistral": _mistral, "pugozen": _pugozen}[model](p, ids, 0)
    return p.tensors


def _weights(model, seed):
    """Random bf16 tensors under the names of a checkpoint."""
    g = torch.Generator(device="cuda")
    g.manual_seed(zlib.crc32(model.encode()) + int(seed))
    out = {}
    for name, (shape, std, mean) in _tensors(model).items():
        t = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std)
        out[name] = (t.add_(mean) if mean else t).to(torch.bfloat16)
    return out


def _load(module, model, seed):
    from shai_amd.weights import load_into
    with torch.no_grad():
        load_into(module, _weights(model, seed), module.convert_hf_state_dict, strict=True)


def _numel(model):
    return sum(math.prod(shape) for shape, _, _ in _tensors(model).values())


# ---------------------------------------------------------------------------------------------- inputs
def _texts(n, seed, least, most):
    g = torch.Generator().manual_seed(int(seed))
    out = []
    for _ in range(n):
        k = int(torch.randint(least, most + 1, (1,), generator=g))
        out.append(" ".join(WORDS[i] for i in torch.randint(len(WORDS), (k,), generator=g).tolist()))
    return out


def _word_ids(text, vocab, first=256):
    """Ids of a text's words without a checkpoint's tokenizer: a checksum's place among the ordinary ids."""
    return [first + zlib.crc32(w.encode()) % (vocab - first) for w in re.findall(r"\w+|[^\w\s]", text.lower())]


def _ids(n, length, seed):
    g = torch.Generator().manual_seed(int(seed))
    return torch.randint(10, VOCAB - 10, (n, length), generator=g)


def _images(batch, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return torch.randint(0, 256, (batch, 224, 224, 3), generator=g, device="cuda", dtype=torch.uint8)


# ---------------------------------------------------------------------------------------------- the framework
def prepare(case, seed):
    """The engine a service holds, with its weights, warmed up the way a service does it before it takes requests, and the inputs
    of one pass."""
    kind, state = case["kind"], {"case": case, "seed": int(seed)}
    if kind == "sd":
        from shai_amd.engines.diffusion import SDConfig, StableDiffusionEngine
        eng = StableDiffusionEngine(SDConfig.sd21(height=case["height"], width=case["width"]), device="cuda")
        _load(eng.text_encoder, "clip", seed)
        _load(eng.unet, "unet", seed)
        _load(eng.vae, "vae", seed)
        eng.unet.build_temb_bank()
        state["prompts"] = _texts(case["batch"], seed, 6, 40)
        eng.generate([""] * case["batch"], 1, seed=0, output="tensor")
    elif kind == "vit":
        from shai_amd.engines.encoders import ImageClassifierEngine
        eng = ImageClassifierEngine(device="cuda")
        _load(eng.model, "vit", seed)
        state["images"] = _images(case["batch"], seed)
        eng.logits_u8(torch.zeros_like(state["images"]))
    elif kind == "t5":
        from shai_amd.engines.encoders import TextEmbeddingEngine
        eng = TextEmbeddingEngine(device="cuda")
        _load(eng.model, "t5", seed)
        state["texts"] = _texts(case["batch"], seed, max(1, case["length"] // 3), case["length"] + 4)
        eng.embed([""] * case["batch"], case["length"])
    else:
        from shai_amd.engines.llm import LLMEngine
        if kind == "mistral":
            from shai_amd.models.llama import LlamaConfig
            cfg = LlamaConfig.mistral_7b()
            cfg.num_hidden_layers = MISTRAL_LAYERS
        else:
            from shai_amd.models.pugozen import PugozenConfig
            cfg = PugozenConfig.uniform(*PUGOZEN)
        length = case["prompt"] + case["gen"]
        eng = LLMEngine(cfg, device="cuda", max_num_seqs=case["batch"], max_model_len=length,
                        num_kv_blocks=case["batch"] * (-(-length // 64)) + 8, enable_prefix_caching=False)
        _load(eng.model, kind, seed)
        state["engine"] = eng
        state["tokens"] = _ids(case["batch"], length, seed + 1).tolist()
        run(state)
        state["tokens"] = _ids(case["batch"], length, seed).tolist()
    state["engine"] = eng
    return state


def run(state):
    case, eng = state["case"], state["engine"]
    kind = case["kind"]
    if kind == "sd":
        return eng.generate(state["prompts"], SD_STEPS, seed=state["seed"], output="tensor")
    if kind == "vit":
        return eng.logits_u8(state["images"])
    if kind == "t5":
        return eng.embed(state["texts"], case["length"])
    n, tokens = case["prompt"], state["tokens"]
    requests = [eng.open_request() for _ in tokens]
    logits = [eng.extend([(r, t[:n], [n - 1]) for r, t in zip(requests, tokens)])]
    for j in range(n, n + case["gen"]):
        logits.append(eng.extend([(r, [t[j]], [0]) for r, t in zip(requests, tokens)]))
    for r in requests:
        eng.close_request(r)
    return logits


# ---------------------------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind == "sd":
        from torch.utils.flop_counter import FlopCounterMode
        B, h, w = case["batch"], case["height"] // 8, case["width"] // 8
        make = lambda *s: torch.empty(*s, dtype=torch.float64, device="meta")  # noqa: E731
        counts = []
        for once in (lambda p: _clip(p, torch.zeros(2 * B, 77, dtype=torch.long, device="meta")),
                     lambda p: _unet(p, make(2 * B, h, w, 4), 1.0, make(2 * B, 77, 1024)),
                     lambda p: _vae(p, make(B, h, w, 4))):
            with FlopCounterMode(display=False) as f:
                once(Asked())
            counts.append(f.get_total_flops())
        nbytes = 2 * (_numel("clip") + SD_STEPS * _numel("unet") + _numel("vae")) + 2 * B * 64 * h * w * 3
        return {"bytes": nbytes, "flops": counts[0] + SD_STEPS * counts[1] + counts[2]}
    if kind == "vit":
        B, T, D, L = case["batch"], 197, 768, 12
        flops = B * (2 * T * 768 * D + L * (2 * T * 12 * D * D + 4 * T * T * D))
        return {"bytes": 2 * _numel("vit") + B * 224 * 224 * 3 + 2 * B * 1000, "flops": flops}
    if kind == "t5":
        B, T, D, L = case["batch"], case["length"], 1024, 24
        flops = B * L * (2 * T * (4 * D * D + 3 * D * 2816) + 4 * T * T * D)
        return {"bytes": 2 * (_numel("t5") - 32128 * D) + 4 * B * D, "flops": flops}
    B, P, G = case["batch"], case["prompt"], case["gen"]
    weights = _numel(kind) - 2 * VOCAB * (4096 if kind == "mistral" else 2048)
    head = VOCAB * (4096 if kind == "mistral" else 2048)
    pairs = P * (P + 1) // 2 + sum(P + j + 1 for j in range(G))
    late = sum(P + j + 1 for j in range(G))                 # cached tokens that the decode steps read
    if kind == "mistral":
        attention, cache, state = 4 * 32 * 128 * MISTRAL_LAYERS, 2 * 8 * 128 * 2 * MISTRAL_LAYERS, 0
    else:
        attention, cache, state = 4 * 16 * 128 * 4, 2 * 4 * 128 * 2 * 4, 8 * 16 * 128 * 128
    flops = B * (2 * (P + G) * weights + 2 * (1 + G) * head + attention * pairs + (P + G) * 6 * state)
    nbytes = (1 + G) * (2 * (weights + head) + 4 * B * VOCAB) + B * ((P + G) * cache + late * cache) + B * G * 8 * state
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """bf16 models: about four times their distance from the fp64 form (relative: 0.006 to 0.011, images 0.015)."""
    return {"rel": 0.03, "max": 0.2}


# ---------------------------------------------------------------------------------------------- the same in 64 bits
def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "sd":
            return _sd_exact(case, seed)
        p = Given(_weights(kind, seed))
        if kind == "vit":
            return _vit(p, _images(case["batch"], seed).double() / 127.5 - 1)
        if kind == "t5":
            L = case["length"]
            rows = [_word_ids(t, 32128) + [1] for t in _texts(case["batch"], seed, max(1, L // 3), L + 4)]
            rows = [r if len(r) <= L else r[:L - 1] + [1] for r in rows]
            ids = torch.tensor([r + [0] * (L - len(r)) for r in rows], device="cuda")
            return _t5(p, ids, [len(r) for r in rows]).cpu().numpy()
        ids = _ids(case["batch"], case["prompt"] + case["gen"], seed).cuda()
        logits = {"mistral": _mistral, "pugozen": _pugozen}[kind](p, ids, case["prompt"] - 1)
        return [logits[:, j] for j in range(case["gen"] + 1)]


def _sd_exact(case, seed):
    B, h, w = case["batch"], case["height"] // 8, case["width"] // 8
    rows = [[49406] + _word_ids(t, 49406) + [49407] for t in [""] * B + _texts(B, seed, 6, 40)]
    ids = torch.tensor([r + [0] * (77 - len(r)) for r in rows], device="cuda")
    ctx = _clip(Given(_weights("clip", seed)), ids)
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    x = torch.randn(B, h, w, 4, generator=g, device="cuda", dtype=torch.float32).to(torch.bfloat16).double()
    alphas = torch.cumprod(1 - torch.linspace(0.00085 ** 0.5, 0.012 ** 0.5, 1000, dtype=torch.float64) ** 2, 0).tolist()
    unet, ratio = Given(_weights("unet", seed)), 1000 // SD_STEPS
    for t in range(1 + ratio * (SD_STEPS - 1), 0, -ratio):
        at, before = alphas[t], alphas[max(t - ratio, 0)]
        u, c = _unet(unet, torch.cat([x, x]), float(t), ctx).chunk(2)
        v = u + 7.5 * (c - u)
        clean, noise = at ** 0.5 * x - (1 - at) ** 0.5 * v, at ** 0.5 * v + (1 - at) ** 0.5 * x
        x = before ** 0.5 * clean + (1 - before) ** 0.5 * noise
    del unet
    return _vae(Given(_weights("vae", seed)), x)


def _linear(p, name, x, n, bias=True, **kw):
    y = x @ p(name + ".weight", n, x.shape[-1], **kw).T
    return y + p(name + ".bias", n, std=0.02) if bias else y


def _conv(p, name, x, n, k=3, stride=1, std=None):
    """x [B, H, W, C], padded to keep its size at stride 1."""
    C = x.shape[-1]
    w = p(name + ".weight", n, C, k, k, std=(C * k * k) ** -0.5 if std is None else std)
    q = k // 2
    x = torch.nn.functional.pad(x, (0, 0, q, q, q, q))
    H, W = (x.shape[1] - k) // stride + 1, (x.shape[2] - k) // stride + 1
    y = 0
    for i in range(k):
        for j in range(k):
            part = x[:, i:i + (H - 1) * stride + 1:stride, j:j + (W - 1) * stride + 1:stride]
            y = y + part @ w[:, :, i, j].T
    return y + p(name + ".bias", n, std=0.02)


def _gain(p, name, n):
    return p(name + ".weight", n, std=0.1, mean=1.0)


def _layer_norm(p, name, x, eps):
    x = x - x.mean(-1, keepdim=True)
    x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    return x * _gain(p, name, x.shape[-1]) + p(name + ".bias", x.shape[-1], std=0.02)


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _group_norm(p, name, x, eps):
    B, C = x.shape[0], x.shape[-1]
    g = x.reshape(B, -1, 32, C // 32)
    g = g - g.mean((1, 3), keepdim=True)
    g = g * torch.rsqrt((g * g).mean((1, 3), keepdim=True) + eps)
    return g.reshape(x.shape) * _gain(p, name, C) + p(name + ".bias", C, std=0.02)


def _attend(q, k, v, heads, scale, causal=False, bias=None, lens=None, factor=None, sink=None):
    """q [B, S, heads * d], k and v [B, S', kv heads * d]: softmax attention, batch rows one by one.  ``factor``: of a head's
    scores; ``sink``: exp(sink) in a head's denominator."""
    B, S, d = q.shape[0], q.shape[1], q.shape[-1] // heads
    G = k.shape[-1] // d
    out = []
    for b in range(B):
        qb = q[b].view(S, heads, d).transpose(0, 1)
        kb, vb = (t[b].view(t.shape[1], G, d).transpose(0, 1).repeat_interleave(heads // G, 0) for t in (k, v))
        s = (qb @ kb.transpose(1, 2)) * scale
        if factor is not None:
            s = s * factor[:, None, None]
        if bias is not None:
            s = s + bias
        if causal:
            s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device=s.device).triu(1), -math.inf)
        if lens is not None:
            s[:, :, lens[b]:] = -math.inf
        if sink is not None:
            s = torch.cat([s, sink[:, None, None].expand(heads, S, 1)], -1)
        e = torch.softmax(s, -1)
        out.append((e[..., :kb.shape[1]] @ vb).transpose(0, 1).reshape(S, heads * d))
    return torch.stack(out)


def _clip(p, ids):
    x = p("text_model.embeddings.token_embedding.weight", 49408, 1024, std=0.02)[ids]
    x = x + p("text_model.embeddings.position_embedding.weight", 77, 1024, std=0.02)[:ids.shape[1]]
    for i in range(23):
        n = f"text_model.encoder.layers.{i}."
        h = _layer_norm(p, n + "layer_norm1", x, 1e-5)
        q, k, v = (_linear(p, f"{n}self_attn.{c}_proj", h, 1024) for c in "qkv")
        x = x + _linear(p, n + "self_attn.out_proj", _attend(q, k, v, 16, 0.125, causal=True), 1024)
        h = _layer_norm(p, n + "layer_norm2", x, 1e-5)
        x = x + _linear(p, n + "mlp.fc2", GELU(_linear(p, n + "mlp.fc1", h, 4096)), 1024)
    return _layer_norm(p, "text_model.final_layer_norm", x, 1e-5)


def _resnet(p, name, x, n, temb=None, eps=1e-5):
    h = _conv(p, name + ".conv1", SILU(_group_norm(p, name + ".norm1", x, eps)), n)
    if temb is not None:
        h = h + _linear(p, name + ".time_emb_proj", temb, n)[:, None, None, :]
    # a block's last convolution is small, as training starts it near zero: rounding does not pile up from block to block
    h = _conv(p, name + ".conv2", SILU(_group_norm(p, name + ".norm2", h, eps)), n, std=0.3 * (9 * n) ** -0.5)
    return h + (x if x.shape[-1] == n else _conv(p, name + ".conv_shortcut", x, n, 1))


def _spatial(p, name, x, ctx):
    """A transformer block over an image's places, with cross-attention to the text."""
    B, H, W, C = x.shape
    h = _linear(p, name + ".proj_in", _group_norm(p, name + ".norm", x, 1e-6).reshape(B, H * W, C), C)
    b = name + ".transformer_blocks.0."
    for i, source in ((1, None), (2, ctx)):
        g = _layer_norm(p, f"{b}norm{i}", h, 1e-5)
        s = g if source is None else source
        q, k, v = (_linear(p, f"{b}attn{i}.to_{c}", t, C, bias=False) for c, t in (("q", g), ("k", s), ("v", s)))
        h = h + _linear(p, f"{b}attn{i}.to_out.0", _attend(q, k, v, C // 64, 0.125), C)
    value, gate = _linear(p, b + "ff.net.0.proj", _layer_norm(p, b + "norm3", h, 1e-5), 8 * C).chunk(2, -1)
    h = h + _linear(p, b + "ff.net.2", value * GELU(gate), C)
    return x + _linear(p, name + ".proj_out", h, C).view(B, H, W, C)


def _twice(x):
    return x.repeat_interleave(2, 1).repeat_interleave(2, 2)


def _unet(p, x, t, ctx):
    f = torch.exp(-math.log(10000.0) * torch.arange(160, dtype=torch.float64, device=x.device) / 160) * t
    f = torch.cat([torch.cos(f), torch.sin(f)])[None].expand(x.shape[0], -1)
    temb = SILU(_linear(p, "time_embedding.linear_2", SILU(_linear(p, "time_embedding.linear_1", f, 1280)), 1280))
    x = _conv(p, "conv_in", x, 320)
    skips, sizes = [x], (320, 640, 1280, 1280)
    for i, n in enumerate(sizes):
        for j in range(2):
            x = _resnet(p, f"down_blocks.{i}.resnets.{j}", x, n, temb)
            if i < 3:
                x = _spatial(p, f"down_blocks.{i}.attentions.{j}", x, ctx)
            skips.append(x)
        if i < 3:
            x = _conv(p, f"down_blocks.{i}.downsamplers.0.conv", x, n, stride=2)
            skips.append(x)
    x = _resnet(p, "mid_block.resnets.0", x, 1280, temb)
    x = _spatial(p, "mid_block.attentions.0", x, ctx)
    x = _resnet(p, "mid_block.resnets.1", x, 1280, temb)
    for i, n in enumerate(reversed(sizes)):
        for j in range(3):
            x = _resnet(p, f"up_blocks.{i}.resnets.{j}", torch.cat([x, skips.pop()], -1), n, temb)
            if i > 0:
                x = _spatial(p, f"up_blocks.{i}.attentions.{j}", x, ctx)
        if i < 3:
            x = _conv(p, f"up_blocks.{i}.upsamplers.0.conv", _twice(x), n)
    # small outputs: with independent random weights the two halves of the guidance are as far apart as two models' outputs, and
    # 7.5 times their rounding would be the image
    return _conv(p, "conv_out", SILU(_group_norm(p, "conv_norm_out", x, 1e-5)), 4, std=0.25 * 2880 ** -0.5)


def _vae(p, z):
    x = _conv(p, "decoder.conv_in", _conv(p, "post_quant_conv", z / 0.18215, 4, 1), 512)
    x = _resnet(p, "decoder.mid_block.resnets.0", x, 512, eps=1e-6)
    a, (B, H, W, C) = "decoder.mid_block.attentions.0.", x.shape
    h = _group_norm(p, a + "group_norm", x, 1e-6).reshape(B, H * W, C)
    q, k, v = (_linear(p, a + "to_" + c, h, C) for c in "qkv")
    x = x + _linear(p, a + "to_out.0", _attend(q, k, v, 1, C ** -0.5), C).view(x.shape)
    x = _resnet(p, "decoder.mid_block.resnets.1", x, 512, eps=1e-6)
    for i, n in enumerate((512, 512, 256, 128)):
        for j in range(3):
            x = _resnet(p, f"decoder.up_blocks.{i}.resnets.{j}", x, n, eps=1e-6)
        if i < 3:
            x = _conv(p, f"decoder.up_blocks.{i}.upsamplers.0.conv", _twice(x), n)
    return _conv(p, "decoder.conv_out", SILU(_group_norm(p, "decoder.conv_norm_out", x, 1e-6)), 3)


def _vit(p, x):
    """x [B, 224, 224, 3] in -1 .. 1."""
    B = x.shape[0]
    w = p("vit.embeddings.patch_embeddings.projection.weight", 768, 3, 16, 16, std=768 ** -0.5)
    x = x.view(B, 14, 16, 14, 16, 3).permute(0, 1, 3, 5, 2, 4).reshape(B, 196, 768) @ w.view(768, 768).T
    x = x + p("vit.embeddings.patch_embeddings.projection.bias", 768, std=0.02)
    x = torch.cat([p("vit.embeddings.cls_token", 1, 1, 768, std=1.0).expand(B, 1, 768), x], 1)
    x = x + p("vit.embeddings.position_embeddings", 1, 197, 768, std=0.3)
    for i in range(12):
        n = f"vit.encoder.layer.{i}."
        h = _layer_norm(p, n + "layernorm_before", x, 1e-12)
        q, k, v = (_linear(p, f"{n}attention.attention.{c}", h, 768) for c in ("query", "key", "value"))
        x = x + _linear(p, n + "attention.output.dense", _attend(q, k, v, 12, 0.125), 768)
        h = _layer_norm(p, n + "layernorm_after", x, 1e-12)
        x = x + _linear(p, n + "output.dense", GELU(_linear(p, n + "intermediate.dense", h, 3072)), 768)
    return _linear(p, "classifier", _layer_norm(p, "vit.layernorm", x[:, 0], 1e-12), 1000)


def _t5(p, ids, lens):
    """Mean over all places of the encoder's last hidden state."""
    x, S = p("shared.weight", 32128, 1024, std=1.0)[ids], ids.shape[1]
    rel = torch.arange(S, device=ids.device)[None, :] - torch.arange(S, device=ids.device)[:, None]
    far = 8 + (torch.log(rel.abs().clamp(min=1).float() / 8) / math.log(16) * 8).long()
    bucket = torch.where(rel.abs() < 8, rel.abs(), far.clamp(max=15)) + (rel > 0).long() * 16
    bias = p("encoder.block.0.layer.0.SelfAttention.relative_attention_bias.weight", 32, 16, std=1.0)[bucket].permute(2, 0, 1)
    for i in range(24):
        n = f"encoder.block.{i}.layer."
        h = _rms(x, 1e-6) * _gain(p, n + "0.layer_norm", 1024)
        q = _linear(p, n + "0.SelfAttention.q", h, 1024, bias=False, std=2.0 ** -8)
        k, v = (_linear(p, n + "0.SelfAttention." + c, h, 1024, bias=False) for c in "kv")
        x = x + _linear(p, n + "0.SelfAttention.o", _attend(q, k, v, 16, 1.0, bias=bias, lens=lens), 1024, bias=False)
        h = _rms(x, 1e-6) * _gain(p, n + "1.layer_norm", 1024)
        gate, up = (_linear(p, n + "1.DenseReluDense." + c, h, 2816, bias=False) for c in ("wi_0", "wi_1"))
        x = x + _linear(p, n + "1.DenseReluDense.wo", GELU(gate, approximate="tanh") * up, 1024, bias=False)
    return (_rms(x, 1e-6) * _gain(p, "encoder.final_layer_norm", 1024)).mean(1)


def _rotate(x, dims, base):
    """x [B, S, heads, d]: dimension i < dims / 2 turns with i + dims / 2."""
    half = dims // 2
    a = torch.arange(x.shape[1], dtype=torch.float64, device=x.device)[:, None] \
        * base ** (-torch.arange(half, dtype=torch.float64, device=x.device) / half)
    c, s = torch.cos(a)[:, None, :], torch.sin(a)[:, None, :]
    u, v = x[..., :half], x[..., half:dims]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., dims:]], -1)


def _mistral(p, ids, first):
    """Logits of places ``first`` and later."""
    B, S = ids.shape
    x = p("model.embed_tokens.weight", VOCAB, 4096, std=1.0)[ids]
    for i in range(MISTRAL_LAYERS):
        n = f"model.layers.{i}."
        h = _rms(x, 1e-5) * _gain(p, n + "input_layernorm", 4096)
        q, k, v = (_linear(p, f"{n}self_attn.{c}_proj", h, m * 128, bias=False) for c, m in (("q", 32), ("k", 8), ("v", 8)))
        q, k = (_rotate(t.view(B, S, -1, 128), 128, 1e6).reshape(t.shape) for t in (q, k))
        x = x + _linear(p, n + "self_attn.o_proj", _attend(q, k, v, 32, 128 ** -0.5, causal=True), 4096, bias=False)
        h = _rms(x, 1e-5) * _gain(p, n + "post_attention_layernorm", 4096)
        gate, up = (_linear(p, f"{n}mlp.{c}_proj", h, 14336, bias=False) for c in ("gate", "up"))
        x = x + _linear(p, n + "mlp.down_proj", SILU(gate) * up, 4096, bias=False)
    return _linear(p, "lm_head", _rms(x[:, first:], 1e-5) * _gain(p, "model.norm", 4096), VOCAB, bias=False)


def _pugozen(p, ids, first):
    """Logits of places ``first`` and later."""
    kinds, D, H, G, d, R, K, dk, dv, rank, ff, _ = PUGOZEN
    eps, (B, S) = 1e-6, ids.shape
    gain = lambda name, n: p(name, n, std=0.3, mean=1.0)                                                         # noqa: E731
    mat = lambda name, x, n, **kw: x @ p(name, n, x.shape[-1], **kw).T                                          # noqa: E731

    def scan(q, k, v, decay, beta=None):
        """q, k [B, S, R, dk], v [B, S, R, dv], decay [B, S, R, dk], beta [B, S, R] (None: keys are added, not corrected)."""
        state, out = torch.zeros(B, R, dk, dv, dtype=q.dtype, device=q.device), []
        for t in range(S):
            state = state * decay[:, t, :, :, None]
            u = v[:, t]
            if beta is not None:
                u = beta[:, t, :, None] * (u - (k[:, t, :, None, :] @ state)[:, :, 0])
            state = state + k[:, t, :, :, None] * u[:, :, None, :]
            out.append((q[:, t, :, None, :] @ state)[:, :, 0])
        return torch.stack(out, 1)

    def delta(n, h, heads, channels):
        def conv(name, c):
            x, taps, y = mat(n + name, h, c), p(n + name + ".conv", c, 4), 0
            for j in range(4):
                y = y + torch.nn.functional.pad(x, (0, 0, 3 - j, 0))[:, :S] * taps[:, j]
            return SILU(y)
        unit = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)                                 # noqa: E731
        q, k = (unit(conv(c, heads * dk).view(B, S, heads, dk)).repeat_interleave(R // heads, 2) for c in "qk")
        v, beta = conv("v", R * dv).view(B, S, R, dv), torch.sigmoid(mat(n + "b", h, R, std=2 * D ** -0.5))
        rate = torch.exp(p(n + "A_log", R, std=1.5))
        soft = torch.nn.functional.softplus
        if channels:
            z = mat(n + "a2", mat(n + "a1", h, rank), R * dk, std=1.0) + p(n + "dt_bias", R * dk, std=2.0, mean=-3.0)
            decay = torch.exp(-rate[:, None] * soft(z).view(B, S, R, dk))
            gate = torch.sigmoid(mat(n + "g2", mat(n + "g1", h, rank), R * dv))
        else:
            decay = torch.exp(-rate * soft(mat(n + "a", h, R) + p(n + "dt_bias", R, std=2.0, mean=-3.0)))[..., None].expand(q.shape)
            gate = SILU(mat(n + "g", h, R * dv))
        o = _rms(scan(q * dk ** -0.5, k, v, decay, beta), eps) * gain(n + "norm", dv)
        return mat(n + "o", o.reshape(B, S, R * dv) * gate, D)

    def retention(n, h):
        q, k = (_rotate(mat(n + c, h, R * dk).view(B, S, R, dk), dk, 10000.0) for c in "qk")
        decay = torch.tensor([1.0 - 2.0 ** -(5.0 + 5.0 * i / R) for i in range(R)], dtype=q.dtype, device=q.device)
        o = scan(q, k * dk ** -0.5, mat(n + "v", h, R * dv).view(B, S, R, dv), decay[:, None].expand(q.shape))
        return mat(n + "o", _rms(o, eps).reshape(B, S, R * dv) * SILU(mat(n + "g", h, R * dv)), D)

    def attention(n, h):
        q, k = mat(n + "q", h, H * d), mat(n + "k", h, G * d)
        turn = lambda x, c: _rotate(_rms(x.view(B, S, -1, d), eps) * gain(n + c + ".norm", d), d // 2, 10000.0).reshape(x.shape)  # noqa: E731
        o = _attend(turn(q, "q"), turn(k, "k"), k, H, d ** -0.5, causal=True, factor=gain(n + "temp", H),
                    sink=p(n + "sink", H, std=1.5))
        return mat(n + "o", o, D)

    x = p("embed", VOCAB, D, std=0.5)[ids]
    for i, kind in enumerate(kinds):
        n = f"l{i}.mix."
        h = _rms(x, eps) * gain(f"l{i}.norm1", D)
        y = mat(f"l{i}.mlp.down", torch.relu(mat(f"l{i}.mlp.up", h, ff)) ** 2, D)
        if kind == "D":
            y = y + delta(n, h, K, False)
        elif kind == "R":
            y = y + retention(n, h)
        else:
            y = y + 0.7 * attention(n + "left.", h) + 0.7 * delta(n + "right.", h, R, True)
        x = x + y
    return mat("head", _rms(x[:, first:], eps) * gain("final.norm", D), VOCAB)
