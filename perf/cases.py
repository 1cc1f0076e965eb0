"""Cases of performance: what a user of the library has it do, with the sizes, inputs, necessary work and exact results of each.

A case is a request: prompts of given lengths in one step, then ``new`` tokens a sequence, one step each.  ``entry`` says which
public entry point runs it:

* ``step``: the model's step function over a cache that the program keeps, as a serving loop calls it: slots are taken, the
  prompts go through one step, the given tokens follow one step each, the slots are given back.  The tokens are given and not
  chosen, because in bfloat16 two correct implementations choose different tokens sooner or later, and from there on their
  logits have nothing in common.
* ``generate``: the whole greedy generation of the 32-bit model, prompts in, tokens and logits out.

``sizes`` names layer sizes given below.  Models have the full depth where three of them fit the card, and fewer layers of
the full size elsewhere.  Weights are random, as ``from_config`` draws them.  Routed experts are in no case: in bfloat16 the
choice between two experts of nearly the same score is an accident, and outputs of two correct implementations cannot be compared.
"""
import math
import random
import zlib

import torch

from pytorch_transformers_amd import AutoModelForCausalLM, FalconConfig, PavodraConfig
from pytorch_transformers_amd.config import VerelornConfig

STD = 0.02
DEVICE = "cuda:0"

# Falcon: sizes of one layer, of the three published models ("7b", "11b", "40b"), of a model with biases, ALiBi and norms in
# sequence whose width and vocabulary are no multiples of 64 ("odd"), and of a model for trials ("tiny").
FALCON = {
    "7b": dict(vocab_size=65024, hidden_size=4544, num_attention_heads=71, multi_query=True, new_decoder_architecture=False,
               parallel_attn=True, bias=False, alibi=False, ffn_hidden_size=18176, rope_theta=10000.0, tie_word_embeddings=True),
    "11b": dict(vocab_size=65024, hidden_size=4096, num_attention_heads=32, num_kv_heads=8, new_decoder_architecture=True,
                num_ln_in_parallel_attn=1, parallel_attn=True, bias=False, alibi=False, ffn_hidden_size=16384,
                rope_theta=500042.0, tie_word_embeddings=False),
    "40b": dict(vocab_size=65024, hidden_size=8192, num_attention_heads=128, num_kv_heads=8, new_decoder_architecture=True,
                num_ln_in_parallel_attn=2, parallel_attn=True, bias=False, alibi=False, ffn_hidden_size=32768,
                rope_theta=10000.0, tie_word_embeddings=False),
    "odd": dict(vocab_size=50001, hidden_size=1040, num_attention_heads=13, multi_query=False, new_decoder_architecture=False,
                parallel_attn=False, bias=True, alibi=True, ffn_hidden_size=4160, tie_word_embeddings=True),
    "tiny": dict(vocab_size=512, hidden_size=64, num_attention_heads=4, num_kv_heads=2, new_decoder_architecture=True,
                 num_ln_in_parallel_attn=2, parallel_attn=True, bias=False, alibi=False, ffn_hidden_size=256,
                 rope_theta=10000.0, tie_word_embeddings=True),
}
EPS = 1e-5
VOCAB_2K = 32768


def pavodra_config(layers):
    mlp = {"kind": "dense", "ff": 8192}
    kinds = [
        {"type": "latent_attention", "mixer": {"heads": 16, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512,
                                               "scale": 192 ** -0.5, "rot": {"base": 10000.0, "dims": 64}}, "mlp": mlp},
        {"type": "mingru", "mixer": {"width": 2048}, "mlp": mlp},
        {"type": "mamba2", "mixer": {"heads": 64, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}, "mlp": mlp},
    ]
    return PavodraConfig(vocab=VOCAB_2K, width=2048, layers=[kinds[i % 3] for i in range(layers)], norm={"eps": 1e-6},
                         residual_mult=0.3, logit_scale=1.0, initializer_range=STD)


def verelorn_config(layers):
    dense = {"kind": "dense", "ff": 5504}
    lat = {"heads": 16, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "q_rank": 1536, "scale": 192 ** -0.5,
           "rot": {"base": 10000.0, "dims": 64}}
    delta = {"heads": 16, "kv_heads": 8, "dim": 128, "vdim": 128, "conv": 4, "a_rank": 128, "g_rank": 128}
    attn = {"heads": 16, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
            "rot": {"base": 500000.0, "dims": 128, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}
    kinds = [{"type": "latent_attention", "mixer": lat, "mlp": dense}, {"type": "channel_delta", "mixer": delta, "mlp": dense},
             {"type": "attention", "mixer": attn, "mlp": dense}]
    out = [dict(kinds[i % 3]) for i in range(layers)]
    for i in range(3, layers, 6):  # every second latent layer reads the latents of the layer three before it
        out[i] = {"type": "latent_attention", "mixer": dict(lat, kv_from=i - 3), "mlp": dense}
    return VerelornConfig(vocab=VOCAB_2K, width=2048, streams=4, layers=out, norm={"eps": 1e-6}, canon={"taps": 4},
                          initializer_range=STD)


def config_of(case):
    if case["sizes"] in FALCON:
        return FalconConfig(num_hidden_layers=case["layers"], layer_norm_epsilon=EPS, max_position_embeddings=8192,
                            initializer_range=STD, **FALCON[case["sizes"]])
    return pavodra_config(case["layers"]) if case["sizes"] == "pavodra2k" else verelorn_config(case["layers"])


def _case(name, sizes, layers, dtype, entry, batch, lo, hi, new):
    """``batch`` prompts of ``lo`` to ``hi`` tokens, then ``new`` tokens each."""
    c = dict(sizes=sizes, layers=layers, dtype=dtype, entry=entry, batch=batch, lo=lo, hi=hi, new=new)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a first trial of the library, a test or a replay: two short prompts through a tiny 32-bit model; launches and host work
        _case("tiny f32 generate", "tiny", 2, "float32", "generate", 2, 5, 11, 6),
        # one user's question to a 32-bit model, short prompt, an answer token by token: every weight is read once a token
        _case("7b-size f32 answer", "7b", 4, "float32", "generate", 1, 60, 60, 16),
        # the same model over a batch of unequal prompts (comparing a model's logits with another implementation's)
        _case("7b-size f32 prompts", "7b", 4, "float32", "generate", 4, 90, 700, 2),
        # a chat with one user: the latency of a token
        _case("7b one sequence", "7b", 32, "bfloat16", "step", 1, 37, 37, 24),
        # a small service: eight conversations of unequal length
        _case("7b batch 8", "7b", 32, "bfloat16", "step", 8, 20, 130, 24),
        # a busy service: 64 short requests at once
        _case("7b batch 64", "7b", 32, "bfloat16", "step", 64, 8, 60, 16),
        # the prompt of the headline figure: 2,048 tokens, the last place's logits
        _case("7b prompt 2048", "7b", 32, "bfloat16", "step", 1, 2048, 2048, 0),
        # documents of very unequal length read in one step, with the first tokens of the answers
        _case("11b-size documents", "11b", 8, "bfloat16", "step", 16, 128, 4096, 4),
        # grouped heads and two norms at the widest layers: a batch of 32
        _case("40b-size batch 32", "40b", 4, "bfloat16", "step", 32, 64, 256, 16),
        # a small model of the older arrangement (ALiBi, biases, norms in sequence), sizes that fill no tile
        _case("odd sizes batch 5", "odd", 24, "bfloat16", "step", 5, 17, 301, 24),
        # a hybrid of latent attention and two recurrences: eight conversations
        _case("pavodra batch 8", "pavodra2k", 6, "bfloat16", "step", 8, 64, 700, 16),
        # several residual streams, delta rule, latent attention: two long prompts and the first tokens of the answers
        _case("verelorn prompts", "verelorn2k", 6, "bfloat16", "step", 2, 1500, 1900, 8),
    ]


# what drawn cases are drawn from: sizes, layers, type, entry, most sequences, most tokens of prompts together, longest prompt, most new tokens
RANGES = [
    ("tiny", 2, "float32", "generate", 8, 200, 100, 12),
    ("7b", 4, "float32", "generate", 8, 1500, 1000, 16),
    ("7b", 32, "bfloat16", "step", 96, 2048, 2048, 24),
    ("11b", 8, "bfloat16", "step", 32, 24000, 4096, 8),
    ("40b", 4, "bfloat16", "step", 64, 6000, 1500, 16),
    ("odd", 24, "bfloat16", "step", 24, 3000, 1200, 24),
    ("pavodra2k", 6, "bfloat16", "step", 24, 4000, 2048, 16),
    ("verelorn2k", 6, "bfloat16", "step", 16, 3800, 2048, 16),
]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    sizes, layers, dtype, entry, most, tokens, longest, new = rng.choice(RANGES)
    batch = _log_int(rng, 1, most)
    hi = _log_int(rng, 8, max(8, min(longest, 2 * tokens // (batch + 1))))
    lo = rng.randint(max(1, hi // 16), hi)
    return _case(None, sizes, layers, dtype, entry, batch, lo, hi, rng.randint(1 if entry == "generate" else 0, new))


def lengths(case):
    """The prompts' lengths: the shortest, the longest, and others between them, the same for every seed."""
    rng = random.Random(case["lo"] * 1000003 + case["hi"] * 101 + case["batch"])
    lens = [rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]
    lens[0] = case["hi"]
    if case["batch"] > 1:
        lens[-1] = case["lo"]
    return lens


def _vocab(case):
    return FALCON[case["sizes"]]["vocab_size"] if case["sizes"] in FALCON else VOCAB_2K


def requests(case, seed):
    """(prompts, tokens that follow them): lists of token ids, uniform over the vocabulary."""
    rng = random.Random(seed * 7919 + 13)
    vocab = _vocab(case)
    prompts = [[rng.randrange(vocab) for _ in range(n)] for n in lengths(case)]
    follow = [[[rng.randrange(vocab)] for _ in prompts] for _ in range(case["new"])]
    return prompts, follow


def prepare(case, seed):
    """The model, the prompts, and for ``step`` the cache that the program keeps and the tokens that it will feed."""
    model = AutoModelForCausalLM.from_config(config_of(case), seed=seed, dtype=case["dtype"], device=DEVICE)
    prompts, follow = requests(case, seed)
    state = {"model": model, "prompts": prompts, "follow": follow, "entry": case["entry"], "new": case["new"]}
    if case["entry"] == "step":
        page = model.page_size
        state["cache"] = model.new_cache(sum((len(p) + case["new"] + page - 1) // page * page for p in prompts),
                                         max_slots=case["batch"])
    return state


def run(state):
    model, prompts = state["model"], state["prompts"]
    if state["entry"] == "generate":
        out = model.generate(prompts, max_new_tokens=state["new"], do_sample=False, eos_token_id=None,
                             return_dict_in_generate=True, output_logits=True)
        return {"tokens": torch.tensor([s[-state["new"]:] for s in out.sequences]),
                "logits": torch.stack([torch.stack(list(rows)) for rows in out.logits])}
    cache = state["cache"]
    slots = [cache.alloc() for _ in prompts]
    logits = [model.step(cache, slots, prompts, "last")]
    for tokens in state["follow"]:
        logits.append(model.step(cache, slots, tokens, "last"))
    for slot in slots:
        cache.free(slot)
    return logits


def tolerance(case):
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-4, "differ": 0.0}  # against 64 bits: 4.2e-6 at the 7b sizes
    return {"rel": 0.03, "max": 0.3}  # against 64 bits: 6e-3 to 1.4e-2 by depth


# ---- the work that a pass cannot do without -----------------------------------------------------------------------------
def _sizes(case):
    """(matrix elements of all layers, of the head, per position and head pairs of attention: flops a (query, key) pair over all
    layers, cache elements a token over all layers, elements of state a sequence over all layers)"""
    L = case["layers"]
    if case["sizes"] in FALCON:
        c = FALCON[case["sizes"]]
        H, F, nh = c["hidden_size"], c["ffn_hidden_size"], c["num_attention_heads"]
        d = H // nh
        nkv = c["num_kv_heads"] if c["new_decoder_architecture"] else (1 if c["multi_query"] else nh)
        return (L * ((nh + 2 * nkv) * d * H + H * H + 2 * H * F), c["vocab_size"] * H, 4.0 * d * nh * L, 2 * nkv * d * L, 0)
    W, mats, pair, kept, state = 2048, 0, 0.0, 0, 0
    for i, layer in enumerate(config_of(case).layers):
        m, kind = layer["mixer"], layer["type"]
        if kind == "latent_attention":
            q_in = m.get("q_rank", W)
            mats += (W * m["q_rank"] if "q_rank" in m else 0) + q_in * m["heads"] * (m["dim"] + m["rot_dim"])
            mats += (m["kv_rank"] + m["rot_dim"]) * W if m.get("kv_from") is None else 0
            mats += m["kv_rank"] * m["heads"] * (m["dim"] + m["vdim"]) + m["heads"] * m["vdim"] * W
            pair += 2.0 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
            kept += m["kv_rank"] + m["rot_dim"] if m.get("kv_from") is None else 0
        elif kind == "mingru":
            mats += 4 * W * m["width"]
            state += m["width"]
        elif kind == "mamba2":
            inner = m["heads"] * m["vdim"]
            mats += W * (2 * inner + 2 * m["groups"] * m["state"] + m["heads"]) + inner * W
            state += m["heads"] * m["vdim"] * m["state"]
        elif kind == "channel_delta":
            qk, inner = m["kv_heads"] * m["dim"], m["heads"] * m["vdim"]
            mats += W * (2 * qk + inner + m["heads"] + m["a_rank"] + m["g_rank"]) + m["a_rank"] * m["heads"] * m["dim"]
            mats += m["g_rank"] * inner + inner * W
            state += m["heads"] * m["dim"] * m["vdim"]
        else:
            mats += W * m["dim"] * (3 * m["heads"] + m["kv_heads"])
            pair += 4.0 * m["heads"] * m["dim"]
            kept += 2 * m["kv_heads"] * m["dim"]
        mats += (3 if case["sizes"] == "verelorn2k" else 2) * W * layer["mlp"]["ff"]
    return mats, VOCAB_2K * W, pair, kept, state


def work(case):
    mats, head, pair, kept, state = _sizes(case)
    elem = 4 if case["dtype"] == "float32" else 2
    lens, B, new = lengths(case), case["batch"], case["new"]
    steps = new - 1 if case["entry"] == "generate" else new  # the prompts' step gives the first of generate's tokens
    T = sum(lens)
    nbytes = (1 + steps) * (mats + head) * elem  # every matrix once a step
    nbytes += (1 + steps) * B * _vocab(case) * 4  # the logits
    nbytes += T * kept * elem + sum(sum(n + k for n in lens) for k in range(1, steps + 1)) * kept * elem  # keys and values: written once, read a step
    nbytes += (1 + 2 * steps) * B * state * 4  # states: left by the prompts, read and written by each step
    flops = 2.0 * (T + steps * B) * mats + 2.0 * (1 + steps) * B * head
    flops += pair * sum((n + steps) * (n + steps + 1) / 2.0 for n in lens)
    flops += 8.0 * state * (T + steps * B)
    return {"bytes": float(nbytes), "flops": float(flops)}


# ---- the same in 64 bits, from the models' equations ----------------------------------------------------------------------
F64 = torch.float64


class _Weights:
    """Tensors by name, as ``from_config`` draws them: a generator per name, values rounded to bfloat16."""

    def __init__(self, seed):
        self.seed = seed

    def __call__(self, name, shape, kind="normal"):
        g = torch.Generator(device=DEVICE)
        g.manual_seed((int(self.seed) * 0x9E3779B1 + zlib.crc32(name.encode("utf-8"))) % (2 ** 63))
        t = torch.empty(shape, dtype=torch.float32, device=DEVICE).normal_(0.0, STD, generator=g)
        if kind == "one":
            t.add_(1.0)
        elif kind == "eye":
            t.add_(torch.eye(shape[0], dtype=torch.float32, device=DEVICE))
        return t.to(torch.bfloat16).to(F64)


def _spans(lens):
    at, out = 0, []
    for n in lens:
        out.append((at, at + n))
        at += n
    return out


def _attend(q, k, v, scale, bias=None, sink=None):
    """q [T, heads, d], k and v [T, kv heads, .]: causal softmax attention, [T, heads * dv].  ``bias`` [heads, T] is added to the
    scores, ``sink`` [heads] is one more term of each head's sum."""
    T, H, d = q.shape
    G = k.shape[1]
    per = H // G
    out = torch.empty((T, H, v.shape[2]), dtype=F64, device=q.device)
    masked = torch.ones((T, T), dtype=torch.bool, device=q.device).triu(1)
    for h in range(H):
        s = q[:, h].contiguous() @ k[:, h // per].t().contiguous() * scale
        if bias is not None:
            s = s + bias[h][None, :]
        s.masked_fill_(masked, float("-inf"))
        if sink is not None:
            s = torch.cat([s, sink[h].expand(T, 1)], 1)
        a = torch.softmax(s, -1)[:, :T]
        out[:, h] = a @ v[:, h // per].contiguous()
    return out.reshape(T, -1)


def _layer_norm(x, w, b):
    mean = x.mean(-1, keepdim=True)
    return (x - mean) / torch.sqrt(((x - mean) ** 2).mean(-1, keepdim=True) + EPS) * w + b


def _turn(x, pos, freq, pairs):
    """Rotation of the last axis of [T, heads, d] by pos * freq: in pairs (i, i + d/2) or (2i, 2i + 1).  Angles are 32-bit products,
    as the published models define them."""
    ang = (pos.float()[:, None] * freq.float()[None, :]).to(F64)
    c, s = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
    if pairs == "half":
        a, b = x[..., :x.shape[-1] // 2], x[..., x.shape[-1] // 2:]
        return torch.cat([a * c - b * s, b * c + a * s], -1)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)


def _freq(base, dims):
    return 1.0 / (base ** (torch.arange(0, dims, 2, dtype=torch.int64, device=DEVICE).float() / dims))


def _alibi(heads, n, d):
    """[heads, n]: bfloat16(slope) * position rounded to bfloat16, over sqrt(d)."""
    n2 = 2 ** math.floor(math.log2(heads))
    base = torch.tensor(2 ** (-(2 ** -(math.log2(n2) - 3))), dtype=torch.float32)
    slopes = torch.pow(base, torch.arange(1, 1 + n2, dtype=torch.int32))
    if n2 != heads:
        extra = torch.tensor(2 ** (-(2 ** -(math.log2(2 * n2) - 3))), dtype=torch.float32)
        slopes = torch.cat([slopes, torch.pow(extra, torch.arange(1, 1 + 2 * min(n2, heads - n2), 2, dtype=torch.int32))])
    return ((slopes[:, None].bfloat16() * torch.arange(n)[None, :]).to(F64) / math.sqrt(d)).to(DEVICE)


def _falcon(case, w, ids, lens):
    c = FALCON[case["sizes"]]
    H, F, nh, V = c["hidden_size"], c["ffn_hidden_size"], c["num_attention_heads"], c["vocab_size"]
    d = H // nh
    grouped, multi = c["new_decoder_architecture"], c["multi_query"] if "multi_query" in c else False
    nkv = c["num_kv_heads"] if grouped else (1 if multi else nh)
    table = w("transformer.word_embeddings.weight", (V, H))
    x = table[ids]
    pos = torch.cat([torch.arange(n, device=DEVICE) for n in lens])

    def norm(v, name):
        return _layer_norm(v, w(name + ".weight", (H,), "one"), w(name + ".bias", (H,), "zero"))

    def lin(v, name, rows, cols):
        y = v @ w(name + ".weight", (rows, cols)).t()
        return y + w(name + ".bias", (rows,), "zero") if c["bias"] else y

    def mlp(v, p):
        u = lin(v, p + "mlp.dense_h_to_4h", F, H)
        return lin(0.5 * u * (1.0 + torch.erf(u / math.sqrt(2.0))), p + "mlp.dense_4h_to_h", H, F)

    for i in range(case["layers"]):
        p = "transformer.h.%d." % i
        two = grouped and c["num_ln_in_parallel_attn"] == 2
        a = norm(x, p + ("ln_attn" if two else "input_layernorm"))
        fused = lin(a, p + "self_attention.query_key_value", (nh + 2 * nkv) * d, H)
        if grouped:
            f = fused.view(-1, nkv, nh // nkv + 2, d)
            q, k, v = f[:, :, :-2].reshape(-1, nh, d), f[:, :, -2], f[:, :, -1]
        elif multi:
            f = fused.view(-1, nh + 2, d)
            q, k, v = f[:, :-2], f[:, -2:-1], f[:, -1:]
        else:
            f = fused.view(-1, nh, 3, d)
            q, k, v = f[:, :, 0], f[:, :, 1], f[:, :, 2]
        if not c["alibi"]:
            freq = _freq(c["rope_theta"], d)
            q, k = _turn(q, pos, freq, "half"), _turn(k, pos, freq, "half")
        o = torch.cat([_attend(q[b:e], k[b:e], v[b:e], d ** -0.5, _alibi(nh, e - b, d) if c["alibi"] else None)
                       for b, e in _spans(lens)])
        o = lin(o, p + "self_attention.dense", H, H)
        if c["parallel_attn"]:
            x = x + (mlp(norm(x, p + "ln_mlp") if two else a, p) + o)
        else:
            x = x + o
            x = x + mlp(norm(x, p + "post_attention_layernorm"), p)
    head = table if c["tie_word_embeddings"] else w("lm_head.weight", (V, H))
    return norm(x, "transformer.ln_f"), head


def _rms(x, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _softplus(x):
    return torch.logaddexp(x, torch.zeros_like(x))


def _conv(x, taps, lens):
    """Causal convolution of every channel of [T, C] along its own sequence; taps [C, K], the last one the token's own."""
    K = taps.shape[1]
    out = []
    for b, e in _spans(lens):
        padded = torch.cat([torch.zeros((K - 1, x.shape[1]), dtype=F64, device=x.device), x[b:e]])
        out.append(sum(padded[j:j + e - b] * taps[:, j] for j in range(K)))
    return torch.cat(out)


def _latent(w, p, m, x, pos, lens, kept):
    """Attention over latents; ``kept`` is the (latents, rotated key parts) of the layer that it reads, or None: its own."""
    H, d, dr, dv, R, W = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], x.shape[1]
    freq = _freq(m["rot"]["base"], dr)
    if "q_rank" in m:
        c = _rms(x @ w(p + ".dq", (m["q_rank"], W)).t()) * w(p + ".dq.norm", (m["q_rank"],), "one")
        q = c @ w(p + ".uq", (H * (d + dr), m["q_rank"])).t()
    else:
        q = x @ w(p + ".q", (H * (d + dr), W)).t()
    q = q.view(-1, H, d + dr)
    q = torch.cat([q[..., :d], _turn(q[..., d:], pos, freq, "interleaved")], -1)
    if kept is None:
        down = x @ w(p + ".dkv", (R + dr, W)).t()
        kept = (_rms(down[:, :R]) * w(p + ".dkv.norm", (R,), "one"), _turn(down[:, None, R:], pos, freq, "interleaved"))
    c, r = kept
    k = torch.cat([(c @ w(p + ".uk", (H * d, R)).t()).view(-1, H, d), r.expand(-1, H, -1)], -1)
    v = (c @ w(p + ".uv", (H * dv, R)).t()).view(-1, H, dv)
    o = torch.cat([_attend(q[b:e], k[b:e], v[b:e], m["scale"]) for b, e in _spans(lens)])
    return o @ w(p + ".o", (W, H * dv)).t(), kept


def _pavodra(case, w, ids, lens):
    cfg = config_of(case)
    W = cfg.width
    pos = torch.cat([torch.arange(n, device=DEVICE) for n in lens])
    table = w("embed", (cfg.vocab, W))

    def norm(v, name):
        return _rms(v) * (1.0 + w(name, (W,), "zero"))

    def mingru(p, m, x):
        C = m["width"]
        z = torch.sigmoid(x @ w(p + ".z", (C, W)).t() + w(p + ".z.b", (C,), "zero"))
        u = x @ w(p + ".x", (C, W)).t() + w(p + ".x.b", (C,), "zero")
        u = torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
        s_all = torch.empty_like(u)
        for b, e in _spans(lens):
            s = torch.zeros(C, dtype=F64, device=x.device)
            for t in range(b, e):
                s = torch.lerp(s, u[t], z[t])
                s_all[t] = s
        return (s_all * _silu(x @ w(p + ".g", (C, W)).t())) @ w(p + ".o", (W, C)).t()

    def mamba2(p, m, x):
        Hn, P, N, G, K = m["heads"], m["vdim"], m["state"], m["groups"], m["conv"]
        inner, chans = Hn * P, Hn * P + 2 * G * N
        proj = x @ w(p + ".in", (inner + chans + Hn, W)).t()
        z, xbc, dt = proj[:, :inner], proj[:, inner:inner + chans], proj[:, inner + chans:]
        xbc = _silu(_conv(xbc, w(p + ".conv", (chans, K)), lens) + w(p + ".conv.b", (chans,), "zero"))
        xs = xbc[:, :inner].reshape(-1, Hn, P)
        B = xbc[:, inner:inner + G * N].reshape(-1, G, N).repeat_interleave(Hn // G, 1)
        C = xbc[:, inner + G * N:].reshape(-1, G, N).repeat_interleave(Hn // G, 1)
        dt = _softplus(dt + w(p + ".dt_bias", (Hn,), "zero"))
        decay = torch.exp(-torch.exp(w(p + ".A_log", (Hn,), "zero")) * dt)
        y = torch.empty_like(xs)
        for b, e in _spans(lens):
            S = torch.zeros((Hn, N, P), dtype=F64, device=x.device)
            for t in range(b, e):
                S = torch.baddbmm(S * decay[t, :, None, None], B[t, :, :, None], (xs[t] * dt[t, :, None])[:, None, :])
                y[t] = torch.bmm(C[t, :, None, :], S)[:, 0]
        y = y + w(p + ".D", (Hn,), "one")[:, None] * xs
        y = y.reshape(-1, inner) * _silu(z)
        y = _rms(y.view(-1, m["norm_groups"], inner // m["norm_groups"])).reshape(-1, inner) * w(p + ".norm", (inner,), "one")
        return y @ w(p + ".o", (W, inner)).t()

    x = table[ids]
    outs = [x]
    for i, layer in enumerate(cfg.layers):
        p, m, kind, ff = "l%d" % i, layer["mixer"], layer["type"], layer["mlp"]["ff"]
        if kind == "latent_attention":
            y = _latent(w, p + ".mix", m, x, pos, lens, None)[0]
        else:
            y = (mingru if kind == "mingru" else mamba2)(p + ".mix", m, x)
        x = x + cfg.residual_mult * norm(y, p + ".norm1")
        u = torch.relu(x @ w(p + ".mlp.up", (ff, W)).t()) ** 2 @ w(p + ".mlp.down", (W, ff)).t()
        x = x + cfg.residual_mult * norm(u, p + ".norm2")
        outs.append(x)
        a = w(p + ".dwa", (i + 2,), "one")
        x = sum(a[j] * outs[j] for j in range(i + 2))
    return norm(x, "final.norm"), table


def _verelorn(case, w, ids, lens):
    cfg = config_of(case)
    W, S, taps = cfg.width, cfg.streams, cfg.taps
    pos = torch.cat([torch.arange(n, device=DEVICE) for n in lens])

    def norm(v, name):
        return _rms(v) * (1.0 + w(name, (W,), "zero"))

    def attention(p, m, x):
        H, G, d, rot = m["heads"], m["kv_heads"], m["dim"], m["rot"]
        freq = _freq(rot["base"], rot["dims"]).to(F64)
        sc, wave = rot["scaling"], 2.0 * math.pi / freq
        s = (sc["original"] / wave - sc["low"]) / (sc["high"] - sc["low"])
        mid = (1.0 - s) * freq / sc["factor"] + s * freq
        freq = torch.where(wave > sc["original"] / sc["low"], freq / sc["factor"], torch.where(wave < sc["original"] / sc["high"], freq, mid))
        q = (x @ w(p + ".q", (H * d, W)).t() + w(p + ".q.b", (H * d,), "zero")).view(-1, H, d)
        k = (x @ w(p + ".k", (G * d, W)).t() + w(p + ".k.b", (G * d,), "zero")).view(-1, G, d)
        qr, kr, sink = _turn(q, pos, freq, "half"), _turn(k, pos, freq, "half"), w(p + ".sink", (H,), "zero")
        o = torch.cat([_attend(qr[b:e], kr[b:e], k[b:e], m["scale"], sink=sink) for b, e in _spans(lens)])
        return (o * torch.sigmoid(x @ w(p + ".g", (H * d, W)).t())) @ w(p + ".o", (W, H * d)).t()

    def delta(p, m, x):
        H, G, d, dv, K = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["conv"]
        q, k, v = (_silu(_conv(x @ w("%s.%s" % (p, t), (n, W)).t(), w("%s.%s.conv" % (p, t), (n, K)), lens))
                   for t, n in (("q", G * d), ("k", G * d), ("v", H * dv)))
        q, k, v = q.view(-1, G, d), k.view(-1, G, d), v.view(-1, H, dv)
        q = (q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * d ** -0.5).repeat_interleave(H // G, 1)
        k = (k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
        beta = torch.sigmoid(x @ w(p + ".b", (H, W)).t())
        a = x @ w(p + ".a1", (m["a_rank"], W)).t() @ w(p + ".a2", (H * d, m["a_rank"])).t() + w(p + ".dt_bias", (H * d,), "zero")
        g = torch.exp(-torch.exp(w(p + ".A_log", (H,), "zero"))[:, None] * _softplus(a.view(-1, H, d)))
        o = torch.empty_like(v)
        for b, e in _spans(lens):
            st = torch.zeros((H, d, dv), dtype=F64, device=x.device)
            for t in range(b, e):
                st = st * g[t, :, :, None]
                u = beta[t, :, None, None] * (v[t, :, None, :] - torch.bmm(k[t, :, None, :], st))
                st = torch.baddbmm(st, k[t, :, :, None], u)
                o[t] = torch.bmm(q[t, :, None, :], st)[:, 0]
        o = (_rms(o) * w(p + ".norm", (dv,), "one")).reshape(-1, H * dv)
        gate = torch.sigmoid(x @ w(p + ".g1", (m["g_rank"], W)).t() @ w(p + ".g2", (H * dv, m["g_rank"])).t())
        return (o * gate) @ w(p + ".o", (W, H * dv)).t()

    def read(xs, name):
        a = w(name, (S,), "one")
        return sum(a[s] * xs[s] for s in range(S))

    def write(xs, name, y):
        mix, out = w(name + ".mix", (S, S), "eye"), w(name + ".out", (S,), "one")
        return [sum(mix[s, t] * xs[s] for s in range(S)) + out[t] * y for t in range(S)]

    xs = [norm(w("embed", (cfg.vocab, W))[ids], "embed.norm")] * S
    kept = {}
    for i, layer in enumerate(cfg.layers):
        p, m, kind, ff = "l%d" % i, layer["mixer"], layer["type"], layer["mlp"]["ff"]
        h = norm(read(xs, p + ".hc1.in"), p + ".norm1")
        h = h + _conv(h, w(p + ".canon1", (W, taps)), lens)
        if kind == "latent_attention":
            y, kept[i] = _latent(w, p + ".mix", m, h, pos, lens, kept.get(m.get("kv_from")))
        else:
            y = (attention if kind == "attention" else delta)(p + ".mix", m, h)
        xs = write(xs, p + ".hc1", y)
        h = norm(read(xs, p + ".hc2.in"), p + ".norm2")
        g = h @ w(p + ".mlp.gate", (ff, W)).t()
        g = 0.5 * g * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (g + 0.044715 * g ** 3)))
        xs = write(xs, p + ".hc2", (g * (h @ w(p + ".mlp.up", (ff, W)).t())) @ w(p + ".mlp.down", (W, ff)).t())
    return norm(sum(xs), "final.norm"), w("head", (cfg.vocab, W))


def exact(case, seed):
    model = _falcon if case["sizes"] in FALCON else _pavodra if case["sizes"] == "pavodra2k" else _verelorn
    prompts, follow = requests(case, seed)
    w = _Weights(seed)

    def last(sequences, count):
        """The logits of every sequence's last ``count`` places, a list of [sequences, vocabulary] from the first of them on."""
        lens = [len(s) for s in sequences]
        with torch.no_grad():
            h, head = model(case, w, torch.tensor([t for s in sequences for t in s], device=DEVICE), lens)
            ends = [e for _, e in _spans(lens)]
            return [h[torch.tensor([e - count + j for e in ends], device=DEVICE)] @ head.t() for j in range(count)]

    if case["entry"] == "step":
        return last([p + [row[i][0] for row in follow] for i, p in enumerate(prompts)], case["new"] + 1)
    tokens, logits = [[] for _ in prompts], []
    for _ in range(case["new"]):
        logits.append(last([p + t for p, t in zip(prompts, tokens)], 1)[0])
        for t, best in zip(tokens, logits[-1].argmax(-1).tolist()):
            t.append(best)
    return {"tokens": torch.tensor(tokens), "logits": torch.stack(logits, 1)}
