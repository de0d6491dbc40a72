"""What the engine's speed is measured on: requests served from their tokens to their last logits.

A case is a small batch of requests on one model: when they arrive, how long their prompts and replies are, in what
portions the prompts are fed. One pass serves all of them through the engine's step function, as a program with an
`Engine` and a `Sampler` does it: prompt portions and decoded tokens in one batch, a pick after every step whose
logits are wanted, the next token fed from the device, a pick read by the host one step late, every request released
at its end. The replies' tokens are given (a vector on the device that stands where the picked ids would): a near tie
that falls the other way would otherwise make two correct runs incomparable. The outputs are the logits behind every
request's last token, which depend on all that was computed and cached before.

A program loads its model once and serves many requests with it, so an engine is kept per model and data type, its
random weights drawn from the model's own seed; a state is a new set of requests.

Models: the LFM2-1.2B and -350M shapes, and the Rekezen and Vebusun designs at the 350M size, all as the benchmark
runs them. Tolerances are four times what was measured against 64 bits (`exact`).
"""
import itertools
import json
import math
import os
import shutil
import tempfile
import zlib

import torch

from imparo_amd import Engine, StepEntry
from imparo_amd.config import plan_from_config
from imparo_amd.engine import DeviceToken
from imparo_amd.engine.model import declared_tensors
from imparo_amd.sampling import Sampler
from imparo_amd.weights import WEIGHTS_FILE, save_file

STEP_TOKENS = 8192              # the most tokens of one step (the engine's default)
POOL_TOKENS = 65536             # the most tokens that live requests hold


# ------------------------------------------------------------------ models
def _lfm2(hidden, heads, block_ff_dim):
    return dict(architectures=["Lfm2ForCausalLM"], model_type="lfm2", vocab_size=65536, hidden_size=hidden,
                num_hidden_layers=16, num_attention_heads=heads, num_key_value_heads=8,
                layer_types=["full_attention" if i in (2, 5, 8, 10, 12, 14) else "conv" for i in range(16)],
                block_auto_adjust_ff_dim=True, block_ff_dim=block_ff_dim, block_multiple_of=256,
                block_ffn_dim_multiplier=1.0, conv_L_cache=3, conv_bias=False, rope_theta=1000000.0,
                tie_embedding=True, norm_eps=1e-5, max_position_embeddings=128000)


def _rekezen(width, heads, kv_heads, ff):
    def mixer(i):
        m = dict(heads=heads, kv_heads=kv_heads, dim=64, vdim=64, scale=0.125, softcap=30.0,
                 rot=dict(dims=64, base=1000000.0, scaling=dict(factor=8.0, original=8192, fast=32.0, slow=1.0)))
        return dict(m, kv_from=i - 1) if i % 2 else m
    mlp = dict(kind="moe", expert=dict(ff=ff, limit=7.0), router=dict(experts=8, top=4), shared=dict(ff=ff, limit=7.0))
    return dict(architecture="Rekezen", vocab=65536, width=width, norm=dict(eps=1e-5), streams=4, logit_scale=1.0,
                embedding=dict(bigram=dict(buckets=65536, mul_prev=31337, mul_cur=1009)),
                layers=[dict(type="attention", mixer=mixer(i), mlp=mlp) for i in range(16)])


def _vebusun(width, heads, ff):
    wide = width // 128
    delta = dict(type="channel_delta", mixer=dict(heads=wide, kv_heads=wide // 2, dim=128, vdim=128, conv=4))
    pair = dict(type="parallel", mixer=dict(
        left=dict(heads=heads, kv_heads=8, dim=64, vdim=64, scale=0.125, softcap=30.0, mask=dict(size=4096, keep_first=64),
                  rot=dict(dims=64, base=1000000.0)),
        right=dict(heads=wide, dim=128, vdim=128, decay=[1.0 - 2.0 ** (-5 - 5 * i / (wide - 1)) for i in range(wide)]),
        left_scale=0.8, right_scale=0.6))
    run = [delta, pair, delta, delta]
    return dict(architecture="Vebusun", vocab=65536, width=width, norm=dict(eps=1e-5), residual_mult=0.5,
                embedding=dict(scale=1.0), layers=[dict(run[i % 4], mlp=dict(kind="dense", ff=ff)) for i in range(16)])


MODELS = {"lfm2-1.2b": _lfm2(2048, 32, 12288), "lfm2-350m": _lfm2(1024, 16, 6656),
          "rekezen-350m": _rekezen(1024, 16, 8, 768), "vebusun-350m": _vebusun(1024, 16, 3072)}


def _weight(model, name, decl, init):
    """A weight on the GPU in bfloat16, drawn from its name: the distributions of the random-weights mode, but for a
    stream that is built up as a trained model's is: embeddings of 0.1, which give logits a spread of 3 to 5, and
    the matrices that add to the stream drawn smaller by the root of how many there are, so that no layer outweighs
    what came before it."""
    g = torch.Generator(device="cuda").manual_seed(zlib.crc32(f"{model}:{name}".encode()))
    shape = tuple(decl.shape)
    if init in ("norm", "share"):
        t = 1.0 + (torch.rand(shape, generator=g, device="cuda") * 0.2 - 0.1)
        t = t / shape[0] if init == "share" else t
    elif init == "mixing":
        t = torch.eye(*shape, device="cuda") + 0.05 * torch.randn(shape, generator=g, device="cuda")
    else:
        spread = {"conv": 0.1, "wide": 0.5}.get(init, 0.02)
        if name in ("embed", "bigram", "model.embed_tokens.weight"):
            spread = 0.1
        elif name.endswith((".o", ".down", ".out_proj.weight", ".w2.weight")):
            spread = 0.02 / math.sqrt(32)
        t = torch.randn(shape, generator=g, device="cuda") * spread
    return t.to(torch.bfloat16)


_engines = {}
_numbers = {}
_state_ids = itertools.count()


def _declared(model):
    return declared_tensors(plan_from_config(MODELS[model])[1])


def _engine(model, dtype):
    """The program's engine for a model: built from a model folder at first use, kept after."""
    if (model, dtype) not in _engines:
        folder = tempfile.mkdtemp(prefix="perf_model_")
        try:
            with open(os.path.join(folder, "config.json"), "w", encoding="utf-8") as f:
                json.dump(MODELS[model], f)
            save_file({name: _weight(model, name, decl, init).cpu() for name, (decl, init) in _declared(model).items()},
                      os.path.join(folder, WEIGHTS_FILE))
            engine = Engine(folder, dtype=dtype, max_tokens=POOL_TOKENS, max_requests=64, max_step_tokens=STEP_TOKENS)
        finally:
            shutil.rmtree(folder)
        _engines[model, dtype] = engine, Sampler(engine.device)
    return _engines[model, dtype]


# ------------------------------------------------------------------ cases
def _case(model, requests, prompt, reply, portion=2048, ragged=False, every=0, temperature=0.0, dtype="bfloat16"):
    """`requests` of `prompt` tokens (`ragged`: from that many down to half) and a reply of `reply` tokens each, one
    arriving every `every` steps (0: all at once), prompts fed in portions of `portion` tokens."""
    return dict(model=model, dtype=dtype, requests=requests, prompt=prompt, ragged=ragged, reply=reply, portion=portion,
                every=every, temperature=temperature)


def listed():
    return [
        # one short question at a time on a small model: every launch counts
        dict(_case("lfm2-350m", 1, 37, 24), name="question"),
        # a few people chatting: decode at batch 8 over short contexts, weights read once a step
        dict(_case("lfm2-1.2b", 8, 300, 64, ragged=True), name="chat"),
        # the same over 4,096-token contexts, as after a long document (the benchmark's headline batch and context)
        dict(_case("lfm2-1.2b", 8, 4096, 64), name="chat_long"),
        # many at once, sampled with a temperature: decode at batch 64
        dict(_case("lfm2-1.2b", 64, 450, 24, ragged=True, temperature=0.8), name="many"),
        # the time to the first token of a short, an ordinary and a long prompt
        dict(_case("lfm2-1.2b", 1, 128, 0), name="prompt_128"),
        dict(_case("lfm2-1.2b", 1, 2048, 0), name="prompt_2048"),
        dict(_case("lfm2-1.2b", 1, 16001, 0, portion=8192), name="prompt_16001"),
        # a server under load: 512-token portions of late prompts beside the tokens of those that came before
        dict(_case("lfm2-1.2b", 12, 1500, 40, portion=512, ragged=True, every=3), name="serving"),
        # the float32 engine, which results are checked with
        dict(_case("lfm2-350m", 2, 333, 8, dtype="float32"), name="float32"),
        # a mixture of experts over attention: a prompt, and decode at batch 8
        dict(_case("rekezen-350m", 1, 2048, 0), name="experts_prompt"),
        dict(_case("rekezen-350m", 8, 200, 32, ragged=True), name="experts_chat"),
        # recurrences beside attention: prompts in one batch, then decode
        dict(_case("vebusun-350m", 4, 1024, 24, ragged=True), name="recurrent"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["prompt", "prompt", "chat", "chat", "chat", "serving", "float32", "other_prompt", "other_chat"])
    lfm2 = rng.choice(["lfm2-1.2b", "lfm2-1.2b", "lfm2-350m"])
    other = rng.choice(["rekezen-350m", "vebusun-350m"])
    if kind == "prompt":
        return _case(lfm2, 1, _log_int(rng, 16, 16384), 0, portion=rng.choice([512, 2048, 8192]))
    if kind == "chat":
        requests = _log_int(rng, 1, 64)
        return _case(lfm2, requests, _log_int(rng, 16, min(4096, 28000 // requests)), rng.randint(8, 24 if requests > 16 else 64),
                     ragged=rng.random() < 0.7, temperature=rng.choice([0.0, 0.0, 0.8]))
    if kind == "serving":
        return _case(lfm2, rng.randint(4, 14), _log_int(rng, 200, 2000), rng.randint(16, 48), portion=rng.choice([256, 512, 1024]),
                     ragged=True, every=rng.randint(1, 5))
    if kind == "float32":
        return _case("lfm2-350m", rng.randint(1, 2), _log_int(rng, 16, 400), rng.randint(1, 8), ragged=True, dtype="float32")
    if kind == "other_prompt":
        return _case(other, 1, _log_int(rng, 64, 4096), 0)
    return _case(other, rng.randint(1, 16), _log_int(rng, 16, 512), rng.randint(8, 40), ragged=True)


def _prompt_lengths(case):
    n, p = case["requests"], case["prompt"]
    return [max(1, p * (2 * n - i) // (2 * n)) if case["ragged"] else p for i in range(n)]


def _steps(case):
    """The pass as steps: each a list of (request, first token, behind the last token, whether its logits are wanted).
    A step takes every request that has come in, its next portion or its next token, up to STEP_TOKENS tokens."""
    prompts = _prompt_lengths(case)
    done = [0] * len(prompts)
    steps = []
    while any(d < p + case["reply"] for d, p in zip(done, prompts)):
        step, room = [], STEP_TOKENS
        for i, p in enumerate(prompts):
            if done[i] >= p + case["reply"] or (i * case["every"] > len(steps)):
                continue
            n = min(case["portion"], p - done[i]) if done[i] < p else 1
            if n > room:
                continue
            room -= n
            step.append((i, done[i], done[i] + n, done[i] + n >= p))
            done[i] += n
        steps.append(step)
    return steps


def _tokens(case, seed):
    """The tokens of every request, prompt and reply, uniform over the vocabulary: [requests][tokens] on the host."""
    g = torch.Generator().manual_seed(seed)
    return [torch.randint(0, 65536, (p + case["reply"],), generator=g).tolist() for p in _prompt_lengths(case)]


def prepare(case, seed):
    engine, sampler = _engine(case["model"], case["dtype"])
    tokens = _tokens(case, seed)
    prompts = _prompt_lengths(case)
    replies = torch.tensor([t for ids, p in zip(tokens, prompts) for t in ids[p:]] or [0], dtype=torch.int32, device=engine.device)
    tag = next(_state_ids)
    steps, last = [], {}
    for step in _steps(case):
        entries, wanted = [], 0
        for i, lo, hi, want in step:
            ids = [DeviceToken(replies, i * case["reply"] + lo - prompts[i])] if lo >= prompts[i] else tokens[i][lo:hi]
            entries.append(StepEntry((tag, i), ids, [hi - lo - 1] if want else []))
            if want:
                last[i] = (len(steps), wanted)
                wanted += 1
        ends = [i for i, lo, hi, _ in step if hi == prompts[i] + case["reply"]]
        g = torch.Generator().manual_seed(seed + len(steps))
        steps.append(dict(entries=entries, ends=ends, rows=[last[i][1] for i in ends], temperatures=[case["temperature"]] * wanted,
                          uniforms=torch.rand(wanted, generator=g).tolist()))
    return dict(engine=engine, sampler=sampler, steps=steps, tag=tag, requests=case["requests"])


def run(state):
    engine, sampler = state["engine"], state["sampler"]
    outputs = [None] * state["requests"]
    pending = None
    for step in state["steps"]:
        logits = engine.step(step["entries"])
        if logits is None:
            continue
        picked = sampler.pick_async(logits, step["temperatures"], step["uniforms"])
        if step["ends"]:
            kept = logits.clone()                # (the engine's next step writes its logits where these lie)
            for i, row in zip(step["ends"], step["rows"]):
                outputs[i] = kept[row]
                engine.release((state["tag"], i))
        if pending is not None:
            pending.tokens()                     # the step before's ids, read while this one runs
        pending = picked
    pending.tokens()
    return torch.stack(outputs)


# ------------------------------------------------------------------ what a pass cannot do without
def _sizes(model):
    """Matrix parameters of the layers that every token meets, of one expert, of the head; bytes of keys and values a
    token a layer's cache and of one request's fixed state; flops a query-key pair; experts and how many a token takes."""
    if model not in _numbers:
        cfg, every, expert = MODELS[model], 0, 0
        experts, top = 1, 0
        for name, (decl, _) in _declared(model).items():
            if decl.role != "matrix" or name in ("embed", "bigram", "head", "model.embed_tokens.weight"):
                continue
            if ".mlp.e" in name:
                expert += math.prod(decl.shape)
            else:
                every += math.prod(decl.shape)
        if model.startswith("lfm2"):
            width, heads = cfg["hidden_size"], cfg["num_attention_heads"]
            attention = owners = sum(t == "full_attention" for t in cfg["layer_types"])
            state = (16 - attention) * 2 * width * 4
        else:
            width, layers = cfg["width"], cfg["layers"]
            mixers = [m for m in (l["mixer"].get("left", l["mixer"]) for l in layers) if "scale" in m]
            heads, attention, owners = 16, len(mixers), sum("kv_from" not in m for m in mixers)
            state = 0 if model.startswith("rekezen") else 16 * width * 128 * 4
            if layers[0]["mlp"]["kind"] == "moe":
                experts, top = layers[0]["mlp"]["router"]["experts"], layers[0]["mlp"]["router"]["top"]
        _numbers[model] = dict(every=every, expert=expert // experts, head=65536 * width, width=width, kv=owners * 2 * 8 * 64,
                               pair=attention * 4 * heads * 64, state=state, experts=experts, top=top)
    return _numbers[model]


def work(case):
    """Every step reads the weights its tokens meet once (an expert nobody chose is not read), the head where logits
    are wanted, the cache of its requests; it writes its tokens' keys and values and the wanted logits."""
    n, prompts = _sizes(case["model"]), _prompt_lengths(case)
    e = 4 if case["dtype"] == "float32" else 2
    data, flops = 0.0, 0.0
    for step in _steps(case):
        tokens = sum(hi - lo for _, lo, hi, _ in step)
        wanted = sum(want for *_, want in step)
        met = n["experts"] * (1.0 - (1.0 - n["top"] / n["experts"]) ** tokens)
        data += e * (n["every"] + met * n["expert"] + (n["head"] if wanted else 0) + tokens * (n["width"] + n["kv"]))
        data += sum(e * lo * n["kv"] + 2 * n["state"] for _, lo, _, _ in step) + wanted * 65536 * 4
        flops += 2.0 * tokens * (n["every"] + n["top"] * n["expert"]) + 2.0 * wanted * n["head"]
        flops += n["pair"] * sum((hi * (hi + 1) - lo * (lo + 1)) / 2 for _, lo, hi, _ in step)
    return {"bytes": data, "flops": flops}


def tolerance(case):
    # float32: against 64 bits 4e-6 to 6e-6 (the rotation's frequencies are float32). bfloat16: 2e-3 to 1.2e-2 (the
    # rounding of what products read, over sixteen layers), a single logit up to 0.055 of their spread
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 0.03, "max": 0.25}


# ------------------------------------------------------------------ the same in 64 bits
# Sequences side by side, padded at their ends (nothing looks ahead): x is [requests, tokens, width].
def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _turn(x, freq, magnitude=1.0, neighbours=False):
    """Rotates x [B, T, heads, dim] by position over its first 2 * len(freq) numbers, i with i + len(freq) or 2i with 2i + 1."""
    half = freq.numel()
    a = (torch.arange(x.shape[1], device=x.device, dtype=x.dtype)[:, None] * freq)[None, :, None, :]
    c, s = torch.cos(a) * magnitude, torch.sin(a) * magnitude
    u, v = (x[..., 0:2 * half:2], x[..., 1:2 * half:2]) if neighbours else (x[..., :half], x[..., half:2 * half])
    turned = [u * c - v * s, v * c + u * s]
    turned = torch.stack(turned, -1).flatten(-2) if neighbours else torch.cat(turned, -1)
    return torch.cat([turned, x[..., 2 * half:]], -1)


def _freq(dims, base):
    return base ** (-torch.arange(0, dims, 2, device="cuda", dtype=torch.float64) / dims)


def _yarn(dims, base, s):
    """Frequencies rescaled after YaRN, and the factor on sine and cosine."""
    at = lambda turns: dims * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(at(s["fast"])), 0), min(math.ceil(at(s["slow"])), dims - 1)
    ramp = ((torch.arange(dims // 2, device="cuda", dtype=torch.float64) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    f = _freq(dims, base)
    return f / s["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(s["factor"]) + 1.0


def _attend(q, k, v, scale, softcap=None, window=None, keep_first=0, sink=None):
    """Causal attention, a request, a head and 4,096 queries at a time: scores capped, keys in a window or among the
    first ones, a sink a head in the denominator."""
    B, T, H, _ = q.shape
    per = H // k.shape[2]
    out = torch.empty(B, T, H, v.shape[-1], device=q.device, dtype=q.dtype)
    for b in range(B):
        for h in range(H):
            for lo in range(0, T, 4096):
                hi = min(T, lo + 4096)
                s = (q[b, lo:hi, h] @ k[b, :hi, h // per].t()) * scale
                if softcap is not None:
                    s = softcap * torch.tanh(s / softcap)
                i, j = torch.arange(lo, hi, device=q.device)[:, None], torch.arange(hi, device=q.device)
                seen = (j <= i) if window is None else (j <= i) & ((i - j < window) | (j < keep_first))
                s = s.masked_fill_(~seen, -math.inf)
                if sink is not None:
                    s = torch.cat([s, sink[h].expand(hi - lo, 1)], 1)
                out[b, lo:hi, h] = torch.softmax(s, -1)[:, :hi] @ v[b, :hi, h // per]
    return out


def _conv(u, taps, bias=None):
    """A causal conv a channel: u [B, T, C], taps [C, n], the last tap the current token's."""
    T, n = u.shape[1], taps.shape[1]
    padded = torch.nn.functional.pad(u, (0, 0, n - 1, 0))
    y = sum(padded[:, j:j + T] * taps[:, j] for j in range(n))
    return y if bias is None else y + bias


def _silu(z):
    return z * torch.sigmoid(z)


def _mixture(h, chosen, weights, experts, expert):
    y = torch.zeros_like(h)
    for e in range(experts):
        t, j = (chosen == e).nonzero(as_tuple=True)
        y.index_put_((t,), weights[t, j][:, None] * expert(e, h[t]), accumulate=True)
    return y


def _lfm2_exact(cfg, w, tokens):
    eps, H = cfg["norm_eps"], cfg["num_attention_heads"]
    B, T = tokens.shape
    x = w("model.embed_tokens.weight")[tokens]
    freq = _freq(64, cfg["rope_theta"])
    for i, kind in enumerate(cfg["layer_types"]):
        p = f"model.layers.{i}."
        h = _rms(x, eps) * w(p + "operator_norm.weight")
        if kind == "conv":
            b, c, u = (h @ w(p + "conv.in_proj.weight").t()).chunk(3, -1)
            y = (c * _conv(b * u, w(p + "conv.conv.weight")[:, 0])) @ w(p + "conv.out_proj.weight").t()
        else:
            a = p + "self_attn."
            q, k, v = ((h @ w(f"{a}{n}_proj.weight").t()).view(B, T, -1, 64) for n in "qkv")
            q = _turn(_rms(q, eps) * w(a + "q_layernorm.weight"), freq)
            k = _turn(_rms(k, eps) * w(a + "k_layernorm.weight"), freq)
            y = _attend(q, k, v, 0.125).reshape(B, T, H * 64) @ w(a + "out_proj.weight").t()
        x = x + y
        h = _rms(x, eps) * w(p + "ffn_norm.weight")
        f = p + "feed_forward."
        x = x + (_silu(h @ w(f + "w1.weight").t()) * (h @ w(f + "w3.weight").t())) @ w(f + "w2.weight").t()
    return _rms(x, eps) * w("model.embedding_norm.weight"), w("model.embed_tokens.weight")


def _rekezen_exact(cfg, w, tokens):
    eps = cfg["norm"]["eps"]
    B, T = tokens.shape

    def norm(x, name):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], w(name), w(name + ".b"), eps)

    def unit(h, p, limit):
        g, u = (h @ w(p + ".gate").t()).clamp(max=limit), (h @ w(p + ".up").t()).clamp(-limit, limit)
        return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w(p + ".down").t()

    bigram = cfg["embedding"]["bigram"]
    pairs = (tokens[:, :-1] * bigram["mul_prev"] + tokens[:, 1:] * bigram["mul_cur"]) % bigram["buckets"]
    pairs = torch.nn.functional.pad(pairs, (1, 0), value=bigram["buckets"])
    X = (w("embed")[tokens] + w("bigram")[pairs])[None].repeat(cfg["streams"], 1, 1, 1)
    kept = {}
    for i, layer in enumerate(cfg["layers"]):
        L, mx, mlp = f"l{i}", layer["mixer"], layer["mlp"]
        freq, magnitude = _yarn(mx["rot"]["dims"], mx["rot"]["base"], mx["rot"]["scaling"])

        def heads(h, n):
            z = _rms(h @ w(f"{L}.mix.{n}").t(), eps) * w(f"{L}.mix.{n}.norm")
            return _turn(z.view(B, T, -1, mx["dim"]), freq, magnitude)

        def mixer(h):
            if "kv_from" not in mx:
                kept[i] = heads(h, "k"), (h @ w(f"{L}.mix.v").t()).view(B, T, -1, mx["vdim"])
            o = _attend(heads(h, "q"), *kept[mx.get("kv_from", i)], mx["scale"], mx["softcap"])
            return (o * torch.sigmoid(h @ w(f"{L}.mix.g").t())[..., None]).flatten(2) @ w(f"{L}.mix.o").t()

        def feed_forward(h):
            h = h.view(B * T, -1)
            best, chosen = torch.topk(h @ w(f"{L}.mlp.router").t() + w(f"{L}.mlp.router.b"), mlp["router"]["top"], -1)
            y = _mixture(h, chosen, torch.softmax(best, -1), mlp["router"]["experts"],
                         lambda e, z: unit(z, f"{L}.mlp.e{e}", mlp["expert"]["limit"]))
            return (y + unit(h, f"{L}.mlp.shared", mlp["shared"]["limit"])).view(B, T, -1)

        for k, sublayer in ((1, mixer), (2, feed_forward)):
            y = sublayer(norm(torch.einsum("s,sbte->bte", w(f"{L}.hc{k}.in"), X), f"{L}.norm{k}"))
            X = torch.einsum("st,sbne->tbne", w(f"{L}.hc{k}.mix"), X) + w(f"{L}.hc{k}.out")[:, None, None, None] * y
    return norm(X.sum(0), "final.norm"), w("embed")


def _vebusun_exact(cfg, w, tokens):
    eps = cfg["norm"]["eps"]
    B, T = tokens.shape

    def linear(h, name):
        return h @ w(name).t()

    def norm(x, name):
        return torch.tanh(w(name + ".alpha") * x) * w(name) + w(name + ".b")

    def channel_delta(h, P, mx):
        H, Hk, d, V = mx["heads"], mx["kv_heads"], mx["dim"], mx["vdim"]
        q, k, v = (_silu(_conv(linear(h, f"{P}.{n}"), w(f"{P}.{n}.conv"))).view(B, T, -1, s) for n, s in (("q", d), ("k", d), ("v", V)))
        q, k = ((z * torch.rsqrt((z * z).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // Hk, 2) for z in (q, k))
        q = q * d ** -0.5
        beta = torch.sigmoid(linear(h, P + ".b"))
        step = torch.nn.functional.softplus(linear(linear(h, P + ".a1"), P + ".a2") + w(P + ".dt_bias")).view(B, T, H, d)
        decay = torch.exp(-torch.exp(w(P + ".A_log"))[:, None] * step)
        S, o = h.new_zeros(B, H, d, V), torch.empty_like(v)
        for t in range(T):
            S = decay[:, t, :, :, None] * S
            u = beta[:, t, :, None] * (v[:, t] - (S * k[:, t, :, :, None]).sum(2))
            S = S + k[:, t, :, :, None] * u[:, :, None, :]
            o[:, t] = (S * q[:, t, :, :, None]).sum(2)
        o = (_rms(o, eps) * w(P + ".norm")).flatten(2)
        return linear(o * torch.sigmoid(linear(linear(h, P + ".g1"), P + ".g2")), P + ".o")

    def attention(h, P, mx):
        q, k, v = (linear(h, f"{P}.{n}").view(B, T, -1, 64) for n in "qkv")
        freq = _freq(mx["rot"]["dims"], mx["rot"]["base"])
        q, k = (_turn(_rms(z, eps) * w(f"{P}.{n}.norm"), freq) for z, n in ((q, "q"), (k, "k")))
        o = _attend(q, k, v, mx["scale"], mx["softcap"], mx["mask"]["size"], mx["mask"]["keep_first"], w(P + ".sink"))
        return linear(o.flatten(2), P + ".o")

    def lightning(h, P, mx):
        q, k, v = (_silu(linear(h, f"{P}.{n}")).view(B, T, mx["heads"], -1) for n in "qkv")
        decay = torch.tensor(mx["decay"], device=h.device, dtype=h.dtype)[:, None, None]
        S, o = h.new_zeros(B, mx["heads"], mx["dim"], mx["vdim"]), torch.empty_like(v)
        for t in range(T):
            S = decay * S + k[:, t, :, :, None] * v[:, t, :, None, :]
            o[:, t] = (S * q[:, t, :, :, None]).sum(2)
        return linear(_rms(o.flatten(2), eps) * w(P + ".norm") * torch.sigmoid(linear(h, P + ".g")), P + ".o")

    x = w("embed")[tokens] * cfg["embedding"]["scale"]
    for i, layer in enumerate(cfg["layers"]):
        L, mx = f"l{i}", layer["mixer"]
        h, P = norm(x, L + ".norm1"), L + ".mix"
        if layer["type"] == "parallel":
            y = mx["left_scale"] * attention(h, P + ".left", mx["left"]) + mx["right_scale"] * lightning(h, P + ".right", mx["right"])
        else:
            y = channel_delta(h, P, mx)
        x = x + cfg["residual_mult"] * y
        h, P = norm(x, L + ".norm2"), L + ".mlp"
        x = x + cfg["residual_mult"] * linear(_silu(linear(h, P + ".gate")) * linear(h, P + ".up"), P + ".down")
    return norm(x, "final.norm"), w("head")


def exact(case, seed):
    model = case["model"]
    declared = _declared(model)
    tokens = _tokens(case, seed)
    lengths = [len(t) for t in tokens]
    padded = torch.tensor([t + [0] * (max(lengths) - len(t)) for t in tokens], device="cuda")
    forward = {"lfm2": _lfm2_exact, "reke": _rekezen_exact, "vebu": _vebusun_exact}[model[:4]]
    with torch.no_grad():
        h, head = forward(MODELS[model], lambda name: _weight(model, name, *declared[name]).double(), padded)
        return torch.stack([h[i, n - 1] @ head.t() for i, n in enumerate(lengths)])
