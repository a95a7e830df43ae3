"""What users of this library have it do, as cases that can be timed.

A case is a model (an architecture, the layer sizes of a published Qwen3 dense model, a number of layers, a type) and one of the
two things a step is: ``prompt`` (all prompts of a batch go through in one step, the logits of every last token come back) or
``decode`` (one step of the answer: every sequence brings one token and gets the logits for the next).  Both run through
``Model.random`` and ``Model.step``; a decode step runs as a captured graph, which is the library's default.

Lengths follow from the case alone; token ids and weights from the seed.  The three designs beside Qwen3 are the ones whose
parts differ most: Zidepel (hyper-connections, gated linear attention), Dagezen (latent attention, talking heads, time mixing,
a state-space mixer) and Kisepel (chunked attention beside the delta rule, linear attention with a fixed decay, experts).  Their
experts are chosen by token id or not there at all: a router's choice between two near-equal experts turns with the last bit of
its input, and the outputs of two correct runs could then not be compared.
"""
import math
import random

import torch

# Layer sizes of the published Qwen3 dense models (width, heads, feed-forward, tied output matrix); all have 8 key heads of 128.
SIZES = {"0.6b": (1024, 16, 3072, True), "1.7b": (2048, 16, 6144, True), "4b": (2560, 32, 9728, True),
         "8b": (4096, 32, 12288, False), "32b": (5120, 64, 25600, False)}
KV_HEADS, DIM = 8, 128
ROOM = 2048                      # tokens a sequence of a decode case may grow by before it starts anew
ANSWERED = 5                     # tokens of the answer that are out before a decode case's first pass


def _case(name, design, size, layers, dtype, phase, batch, low, high):
    return {"name": name, "design": design, "size": size, "layers": layers, "dtype": dtype, "phase": phase,
            "batch": batch, "low": low, "high": high}


def listed():
    return [
        # one user's chat with a small model: the latency of a token, where launches count
        _case("chat_small", "qwen3", "0.6b", 28, "bfloat16", "decode", 1, 1024, 1024),
        # a few users of a stretch of the 8B model after long prompts: weights stream from memory (more layers than 8 of this width
        # carry bfloat16's roundings on to more than what a tolerance may allow)
        _case("chat_8b", "qwen3", "8b", 8, "bfloat16", "decode", 8, 2048, 2048),
        # a full batch of unequal sequences: the cache weighs as much as the weights
        _case("serve_8b", "qwen3", "8b", 8, "bfloat16", "decode", 64, 1100, 2040),
        # one prompt of 2,048 tokens: matrix products
        _case("prompt_8b", "qwen3", "8b", 6, "bfloat16", "prompt", 1, 2048, 2048),
        # a batch of unequal prompts through a small model: ragged rows, small products
        _case("prompts_small", "qwen3", "0.6b", 28, "bfloat16", "prompt", 16, 16, 1024),
        # a long document at the largest layer sizes: attention over many keys
        _case("document_32b", "qwen3", "32b", 3, "bfloat16", "prompt", 1, 8192, 8192),
        # the float32 path, as used to check a checkpoint: a few unequal prompts
        _case("check_float32", "qwen3", "0.6b", 28, "float32", "prompt", 3, 33, 400),
        # the other designs: prompts (scans over the tokens, attention of other kinds) and decode steps (states)
        _case("zidepel_prompts", "zidepel", "8b", 4, "bfloat16", "prompt", 3, 500, 1500),
        _case("dagezen_prompt", "dagezen", "8b", 4, "bfloat16", "prompt", 1, 2048, 2048),
        _case("dagezen_decode", "dagezen", "8b", 4, "bfloat16", "decode", 8, 1100, 1500),
        _case("kisepel_prompts", "kisepel", "8b", 4, "bfloat16", "prompt", 4, 300, 1800),
        _case("kisepel_decode", "kisepel", "8b", 4, "bfloat16", "decode", 32, 1024, 1024),
    ]


def _spread(rng, low, high):
    """A whole number from ``low`` to ``high``, spread over the logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    design = rng.choice(("qwen3", "qwen3", "qwen3", "float32", "zidepel", "dagezen", "kisepel"))
    phase = rng.choice(("prompt", "decode"))
    if design == "float32":
        return _drawn("qwen3", "0.6b", rng.randint(2, 28), "float32", phase, _spread(rng, 1, 12), _spread(rng, 16, 100), rng)
    if design == "qwen3":
        size = rng.choice(("0.6b", "1.7b", "4b", "8b"))
        layers = rng.randint(4, 6 if size in ("4b", "8b") else 16)
        if phase == "decode":
            return _drawn("qwen3", size, layers, "bfloat16", phase, _spread(rng, 1, 64), _spread(rng, 64, 1100), rng)
        batch = _spread(rng, 1, 16)
        return _drawn("qwen3", size, layers, "bfloat16", phase, batch, _spread(rng, 16, 2048 // batch), rng)
    size, layers = rng.choice((("0.6b", 4), ("0.6b", 8), ("8b", 4)))
    if phase == "decode":
        return _drawn(design, size, layers, "bfloat16", phase, _spread(rng, 1, 40), _spread(rng, 64, 800), rng)
    batch = _spread(rng, 1, 8)
    return _drawn(design, size, layers, "bfloat16", phase, batch, _spread(rng, 16, 2048 // batch), rng)


def _drawn(design, size, layers, dtype, phase, batch, low, rng):
    case = _case("", design, size, layers, dtype, phase, batch, low, low + rng.randint(0, low))
    del case["name"]
    return case


# ---------------------------------------------------------------- the models
def _vocab(case):
    return 151936 if case["design"] == "qwen3" else 32768


def _limit(case):
    return case["high"] + (ROOM + ANSWERED if case["phase"] == "decode" else 0)


def config(case):
    """config.json of the case's model."""
    width, heads, ff, tied = SIZES[case["size"]]
    vocab, n = _vocab(case), case["layers"]
    scale = DIM ** -0.5
    if case["design"] == "qwen3":
        return {"architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "vocab_size": vocab, "hidden_size": width,
                "intermediate_size": ff, "num_hidden_layers": n, "num_attention_heads": heads, "num_key_value_heads": KV_HEADS,
                "head_dim": DIM, "rope_theta": 1000000.0, "rms_norm_eps": 1e-6, "tie_word_embeddings": tied,
                "max_position_embeddings": _limit(case)}
    base = {"vocab": vocab, "width": width, "norm": {"eps": 1e-5}}
    grouped = {"heads": heads, "kv_heads": KV_HEADS, "dim": DIM, "vdim": DIM, "scale": scale}
    ssm = {"heads": heads, "vdim": DIM, "state": DIM, "groups": KV_HEADS, "conv": 4, "norm_groups": KV_HEADS}
    few = max(1, heads // 4)
    if case["design"] == "zidepel":
        att = {"type": "attention", "mlp": {"kind": "dense", "ff": ff * 3 // 2},
               "mixer": dict(grouped, softcap=30.0, q_temp={"coef": 0.1, "every": 512})}
        gla = {"type": "gla", "mlp": None, "mixer": {"heads": heads, "dim": DIM, "vdim": DIM, "tau": 16.0, "rank": 16}}
        return dict(base, architecture="Zidepel", max_positions=_limit(case), streams=4, layers=[(att, att, gla, att)[i % 4] for i in range(n)])
    if case["design"] == "dagezen":
        mlp = {"kind": "dense", "ff": ff * 3 // 2, "limit": 7.0}
        lat = {"type": "latent_attention", "mlp": mlp,
               "mixer": {"heads": heads, "dim": DIM, "rot_dim": DIM // 2, "vdim": DIM, "kv_rank": 4 * DIM, "scale": (DIM * 1.5) ** -0.5,
                         "rot": {"dims": DIM // 2, "base": 1e6}}}
        par = {"type": "parallel", "mlp": mlp,
               "mixer": {"left": dict(grouped, mask={"size": 1024}), "right": {"heads": few, "dim": DIM, "rank": 64},
                         "left_scale": 0.7, "right_scale": 0.7}}
        return dict(base, architecture="Dagezen", postln_alpha=1.5, logit_softcap=30.0,
                    layers=[(lat, par, {"type": "mamba2", "mlp": None, "mixer": ssm}, par)[i % 4] for i in range(n)])
    moe = {"kind": "moe", "expert": {"ff": ff // 2}, "shared": {"ff": ff // 4}, "router": {"experts": 8, "top": 2}}
    par = {"type": "parallel", "mlp": moe,
           "mixer": {"left": dict(grouped, mask={"size": 1024}, rot={"dims": DIM, "base": 1e6, "scaling": {"factor": 4.0}}),
                     "right": {"heads": few, "kv_heads": few, "dim": DIM, "vdim": DIM, "conv": 4, "rank": DIM}}}
    lin = {"type": "lightning", "mlp": None,
           "mixer": {"heads": heads, "dim": DIM, "vdim": DIM, "decay": [1.0 - 2.0 ** -(3 + 5 * i / max(1, heads - 1)) for i in range(heads)]}}
    return dict(base, architecture="Kisepel", embedding={"scale": 8.0}, logit_scale=0.5,
                layers=[({"type": "mamba2", "mlp": moe, "mixer": ssm}, par, lin, par)[i % 4] for i in range(n)])


def lengths(case):
    r = random.Random(repr((case["batch"], case["low"], case["high"])))
    return [r.randint(case["low"], case["high"]) for _ in range(case["batch"])]


def _tokens(case, seed):
    """Every sequence's prompt, and the ids that are fed to it one a step while it is answered."""
    g = torch.Generator().manual_seed(seed)
    prompts = [torch.randint(0, _vocab(case), (n,), generator=g).tolist() for n in lengths(case)]
    answer = torch.randint(0, _vocab(case), (ROOM + ANSWERED, case["batch"]), generator=g).tolist()
    return prompts, answer


class _State:
    pass


def _start(s):
    """The prompts and the answer's first tokens (the step's graph is captured among them)."""
    s.slots = [s.model.cache.acquire() for _ in s.prompts]
    s.model.step([(slot, p, "last") for slot, p in zip(s.slots, s.prompts)])
    s.fed = 0
    for _ in range(ANSWERED - 1):
        _feed(s)


def _feed(s):
    ids = s.answer[s.fed]
    s.fed += 1
    return s.model.step([(slot, (t,), "last") for slot, t in zip(s.slots, ids)])


def prepare(case, seed):
    from rust_inference_amd import Model
    s = _State()
    s.case = case
    s.prompts, s.answer = _tokens(case, seed)
    s.model = Model.random(config(case), seed=seed, dtype=case["dtype"], max_batch=case["batch"], max_seq_len=_limit(case))
    if case["phase"] == "decode":
        _start(s)
    return s


def run(s):
    """One step.  A decode case's sequences go on from pass to pass and start anew when they are full."""
    if s.case["phase"] == "decode":
        if s.fed == len(s.answer):
            for slot in s.slots:
                s.model.cache.release(slot)
            _start(s)
        return _feed(s)
    slots = [s.model.cache.acquire() for _ in s.prompts]
    logits = s.model.step([(slot, p, "last") for slot, p in zip(slots, s.prompts)])
    for slot in slots:
        s.model.cache.release(slot)
    return logits


# ---------------------------------------------------------------- the work of a pass
def work(case):
    """The weights in use and the cache are read once, logits and new cache entries written once; products, scores and states."""
    width, heads, ff, _ = SIZES[case["size"]]
    decode, wide = case["phase"] == "decode", 4 if case["dtype"] == "float32" else 2
    lens, b = lengths(case), case["batch"]
    tokens = b if decode else sum(lens)
    before = [n + ANSWERED - 1 if decode else 0 for n in lens]              # keys in the cache before the step
    new = [1 if decode else n for n in lens]
    hd, kd, few = heads * DIM, KV_HEADS * DIM, max(1, heads // 4) * DIM
    pairs = lambda most: float(sum(min(p + i + 1, most) for p, n in zip(before, new) for i in range(n)))
    seen = lambda most: float(sum(min(p, most) for p in before))
    cached = (sum(before) > 0)

    # a layer: matrix elements in use for a token; elements held that the step reads; flops beside the products; bytes of cache
    def attention(window=1 << 40, values=kd):
        return ((2 * hd + kd + values) * width,) * 2 + (4.0 * hd * pairs(window), wide * 2 * kd * (seen(window) + tokens))

    def recurrent(elements, state, ops_a_token):
        return elements, elements, ops_a_token * tokens, 4.0 * state * b * (2 if cached else 1)

    def dense(n):
        return n * width * (ff * 3 // 2 if case["design"] != "qwen3" else ff), n * width * (ff * 3 // 2 if case["design"] != "qwen3" else ff), 0.0, 0.0

    def experts():
        one, shared = 3 * width * (ff // 2), 3 * width * (ff // 4)
        return 2 * one + shared, min(8, 2 * tokens) * one + shared, 0.0, 0.0

    inner = heads * DIM
    ssm = recurrent((3 * inner + 2 * KV_HEADS * DIM + heads) * width, inner * DIM, 5.0 * inner * DIM)
    if case["design"] == "qwen3":
        kinds = [[attention(), dense(3)]]
    elif case["design"] == "zidepel":
        kinds = [[attention(), dense(2)], [attention(), dense(2)], [recurrent(5 * hd * width, hd * DIM, 5.0 * hd * DIM)], [attention(), dense(2)]]
    elif case["design"] == "dagezen":
        rank = 4 * DIM
        lat = (hd * 3 // 2 * width + (rank + DIM // 2) * width + 2 * hd * rank + hd * width,) * 2 \
            + (2.0 * hd * 2.5 * pairs(1 << 40), wide * (rank + DIM // 2) * (seen(1 << 40) + tokens))
        left = attention(1024, 0)
        left = (left[0] + hd * width, left[1] + hd * width, left[2] + 2.0 * heads * heads * pairs(1024), left[3])
        par = [left, recurrent(5 * few * width, few * DIM, 6.0 * few * DIM), dense(3)]
        kinds = [[lat, dense(3)], par, [ssm], par]
    else:
        par = [attention(), recurrent((4 * few + 3 * DIM) * width, few * DIM, 7.0 * few * DIM), experts()]
        kinds = [[ssm, experts()], par, [recurrent(5 * hd * width, hd * DIM, 4.0 * hd * DIM)], par]
    head = _vocab(case) * width
    nbytes, flops = wide * head + 4.0 * b * _vocab(case) + wide * tokens * width, 2.0 * head * b
    for i in range(case["layers"]):
        for use, held, ops, cache in kinds[i % len(kinds)]:
            nbytes += wide * held + cache
            flops += 2.0 * use * tokens + ops
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Relative error of the logits.  Against 64-bit results the float32 path shows 2e-6; the bfloat16 path 0.4 to 0.8 per cent at the
    small sizes and 1 to 2 per cent over 3 to 8 layers at the larger, and two correct runs are up to 1.4 times as far from each other."""
    return {"rel": 1e-5} if case["dtype"] == "float32" else {"rel": 0.03}


# ---------------------------------------------------------------- the same in 64 bits, plainly
def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, w, b, eps):
    x = x - x.mean(-1, keepdim=True)
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w + b


def _silu(z):
    return z * torch.sigmoid(z)


def _turn(x, dims, base, factor=1.0, pairs=False):
    """x [B, T, heads, dim]: the first ``dims`` elements of every head turn by position * base^(-2i / dims) / factor, neighbours
    (``pairs``) or halves together."""
    half = dims // 2
    freq = base ** (-2.0 * torch.arange(half, dtype=torch.float64, device=x.device) / dims) / factor
    a = torch.arange(x.shape[1], dtype=torch.float64, device=x.device)[:, None] * freq
    c, s = a.cos()[:, None], a.sin()[:, None]
    u, v = (x[..., :dims:2], x[..., 1:dims:2]) if pairs else (x[..., :half], x[..., half:dims])
    y = (u * c - v * s, v * c + u * s)
    return torch.cat([torch.stack(y, -1).flatten(-2) if pairs else torch.cat(y, -1), x[..., dims:]], -1)


def _attend(q, k, v, scale, seen=None, cap=None, more=None, sink=None, mix=None):
    """q [B, T, H, d], k and v [B, T, G, .]: causal attention; ``seen(i, j)``, ``more(scores, i - j)`` and ``mix`` change the rest."""
    t, share = q.shape[1], q.shape[2] // k.shape[2]
    at = torch.arange(t, device=q.device)
    gap = at[:, None] - at
    hidden = gap < 0 if seen is None else (gap < 0) | ~seen(at[:, None], at)
    out = []
    for i in range(q.shape[0]):
        kh, vh = (z[i].transpose(0, 1).repeat_interleave(share, 0) for z in (k, v))
        s = (q[i].transpose(0, 1) @ kh.transpose(1, 2)).mul_(scale)
        if cap:
            s = cap * torch.tanh(s / cap)
        if more is not None:
            s = more(s, gap.clamp(min=0).double())
        s.masked_fill_(hidden, -math.inf)
        if sink is None:
            s = torch.softmax(s, -1)
        else:
            s = torch.softmax(torch.cat([s, sink[:, None, None].expand(-1, t, 1)], -1), -1)[..., :t]
        if mix is not None:
            s = (mix @ s.flatten(1)).view(s.shape)
        out.append((s @ vh).transpose(0, 1))
    return torch.stack(out).flatten(2)


def _conv(x, taps, bias=None):
    """x [B, T, channels] through a causal convolution a channel, the last tap the current token's."""
    n = taps.shape[1]
    line = torch.nn.functional.pad(x, (0, 0, n - 1, 0))
    out = sum(line[:, j:j + x.shape[1]] * taps[:, j] for j in range(n))
    return out if bias is None else out + bias


def _walk(q, k, v, decay, beta=None, bonus=None):
    """The state S [dim, vdim] of every head, token after token: decayed per key channel, then written with k v^T (``beta``: the delta
    rule's k beta (v - S^T k)^T), read with q; ``bonus``: read before the write, which counts times that."""
    b, t, h, d = q.shape
    s = torch.zeros(b, h, d, v.shape[-1], dtype=torch.float64, device=q.device)
    out = torch.empty(b, t, h, v.shape[-1], dtype=torch.float64, device=q.device)
    for i in range(t):
        ki, vi = k[:, i, :, :, None], v[:, i, :, None]
        if bonus is not None:
            kv = ki * vi
            out[:, i] = ((s + bonus[:, :, None] * kv) * q[:, i, :, :, None]).sum(2)
            s = s * decay[:, i, :, :, None] + kv
            continue
        s *= decay[:, i, :, :, None]
        if beta is None:
            s += ki * vi
        else:
            s += ki * (beta[:, i, :, None, None] * (vi - (s * ki).sum(2, keepdim=True)))
        out[:, i] = (s * q[:, i, :, :, None]).sum(2)
    return out


class _Plain:
    """A design's forward in float64, all sequences padded behind their ends (every part is causal)."""

    def __init__(self, case, weights, ids):
        self.cfg, self.case, self.weights, self.ids = config(case), case, weights, ids

    def w(self, name):
        return self.weights[name].double()

    def lin(self, x, name):
        return x @ self.w(name).T

    def heads(self, x, name, dim=DIM):
        return self.lin(x, name).unflatten(-1, (-1, dim))

    # -- Qwen3
    def qwen3(self):
        eps, x = 1e-6, self.w("model.embed_tokens.weight")[self.ids]
        for i in range(self.case["layers"]):
            p = f"model.layers.{i}."
            h, a = _rms(x, eps) * self.w(p + "input_layernorm.weight"), p + "self_attn."
            q, k = (_turn(_rms(self.heads(h, f"{a}{n}_proj.weight"), eps) * self.w(f"{a}{n}_norm.weight"), DIM, 1e6) for n in "qk")
            x = x + self.lin(_attend(q, k, self.heads(h, a + "v_proj.weight"), DIM ** -0.5), a + "o_proj.weight")
            h, m = _rms(x, eps) * self.w(p + "post_attention_layernorm.weight"), p + "mlp."
            x = x + self.lin(_silu(self.lin(h, m + "gate_proj.weight")) * self.lin(h, m + "up_proj.weight"), m + "down_proj.weight")
        return _rms(x, eps) * self.w("model.norm.weight"), "model.embed_tokens.weight" if SIZES[self.case["size"]][3] else "lm_head.weight"

    # -- Zidepel
    def zidepel(self):
        ln = lambda x, n: _layer_norm(x, self.w(n), self.w(n + ".b"), 1e-5)
        x = ln(self.w("embed")[self.ids] + self.w("pos")[:self.ids.shape[1]], "embed.norm")
        xs = x[None].repeat(4, 1, 1, 1)

        def through(p, branch):
            y = branch(torch.einsum("s,sbtd->btd", self.w(p + "in"), xs))
            return torch.einsum("sr,sbtd->rbtd", self.w(p + "mix"), xs) + self.w(p + "out")[:, None, None, None] * y

        for i, layer in enumerate(self.cfg["layers"]):
            p = f"l{i}."
            mixer = self.gla if layer["type"] == "gla" else self.tempered
            xs = through(p + "hc1.", lambda u: mixer(ln(u, p + "norm1"), p + "mix."))
            if layer["mlp"]:
                xs = through(p + "hc2.", lambda u: self.lin(self.lin(ln(u, p + "norm2"), p + "mlp.up").clamp(min=0).square(), p + "mlp.down"))
        return ln(xs.sum(0), "final.norm"), "head"

    def tempered(self, h, p):
        q, k = (_rms(self.heads(h, p + n), 1e-5) * self.w(f"{p}{n}.norm") for n in "qk")
        at = torch.arange(h.shape[1], device=h.device)
        q = q * (1.0 + 0.1 * torch.log((at + 1).div(512, rounding_mode="floor") + 1.0).double())[:, None, None]
        return self.lin(_attend(q, k, self.heads(h, p + "v"), DIM ** -0.5, cap=30.0), p + "o")

    def gla(self, h, p):
        z = self.lin(self.lin(h, p + "a1"), p + "a2") + self.w(p + "a2.b")
        decay = torch.exp(torch.nn.functional.logsigmoid(z) / 16.0).unflatten(-1, (-1, DIM))
        o = _walk(self.heads(h, p + "q") * DIM ** -0.5, self.heads(h, p + "k"), self.heads(h, p + "v"), decay)
        return self.lin((_rms(o, 1e-5) * self.w(p + "norm")).flatten(2) * _silu(self.lin(h, p + "g")), p + "o")

    # -- Dagezen
    def dagezen(self):
        ln = lambda x, n: _layer_norm(x, self.w(n), self.w(n + ".b"), 1e-5)
        x = self.w("embed")[self.ids]
        for i, layer in enumerate(self.cfg["layers"]):
            p = f"l{i}."
            mixer = {"latent_attention": self.latent, "mamba2": self.ssm, "parallel": self.talking_and_time}[layer["type"]]
            x = ln(1.5 * x + mixer(x, p + "mix."), p + "norm1")
            if layer["mlp"]:
                m = p + "mlp."
                g = (self.lin(x, m + "gate") + self.w(m + "gate.b")).clamp(max=7.0)
                u = (self.lin(x, m + "up") + self.w(m + "up.b")).clamp(-7.0, 7.0)
                x = ln(1.5 * x + self.lin(g * torch.sigmoid(1.702 * g) * (u + 1.0), m + "down") + self.w(m + "down.b"), p + "norm2")
        return ln(x, "final.norm"), "embed"

    def latent(self, h, p):
        rank, rot = 4 * DIM, DIM // 2
        q, both = self.heads(h, p + "q", DIM + rot), self.lin(h, p + "dkv")
        q = torch.cat([q[..., :DIM], _turn(q[..., DIM:], rot, 1e6, pairs=True)], -1)
        c = _rms(both[..., :rank], 1e-5) * self.w(p + "dkv.norm")
        turned = _turn(both[..., None, rank:], rot, 1e6, pairs=True)
        k = torch.cat([self.heads(c, p + "uk"), turned.expand(-1, -1, q.shape[2], -1)], -1)
        o = _attend(q, k, self.heads(c, p + "uv"), (DIM * 1.5) ** -0.5, sink=self.w(p + "sink"))
        return self.lin((o.unflatten(-1, (-1, DIM)) * torch.sigmoid(self.lin(h, p + "g"))[..., None]).flatten(2), p + "o")

    def talking_and_time(self, h, p):
        l, r = p + "left.", p + "right."
        raw = self.lin(h, l + "k")
        q, k = _rms(self.lin(h, l + "q"), 1e-5) * self.w(l + "q.norm"), _rms(raw, 1e-5) * self.w(l + "k.norm")
        slope, bend = self.w(l + "r1")[:, None, None], self.w(l + "r2")[:, None, None]
        q, k, v = (z.unflatten(-1, (-1, DIM)) for z in (q, k, raw))
        left = _attend(q, k, v, DIM ** -0.5, seen=lambda i, j: i - j < 1024, more=lambda s, gap: s - slope * torch.log1p(bend * gap), mix=self.w(l + "talk"))
        left = self.lin(left * torch.sigmoid(self.lin(h, l + "g")), l + "o")
        step = torch.nn.functional.pad(h, (0, 0, 1, 0))[:, :-1] - h
        mixed = {n: h + step * self.w(r + "mu." + n) for n in "rkvgw"}
        decay = torch.exp(-torch.exp(self.lin(torch.tanh(self.lin(mixed["w"], r + "w1")), r + "w2") + self.w(r + "w0"))).unflatten(-1, (-1, DIM))
        o = _walk(*(self.heads(mixed[n], r + n) for n in "rkv"), decay, bonus=self.w(r + "u"))
        right = self.lin(_rms(o, 1e-5).flatten(2) * self.w(r + "norm") * _silu(self.lin(mixed["g"], r + "g")), r + "o")
        return 0.7 * left + 0.7 * right

    def ssm(self, h, p):
        proj = self.lin(h, p + "in")
        inner = self.w(p + "D").shape[0] * DIM
        z, xbc, dt = proj.split([inner, inner + 2 * KV_HEADS * DIM, inner // DIM], -1)
        xbc = _silu(_conv(xbc, self.w(p + "conv"), self.w(p + "conv.b")))
        x, b, c = (y.unflatten(-1, (-1, DIM)) for y in xbc.split([inner, KV_HEADS * DIM, KV_HEADS * DIM], -1))
        dt = torch.nn.functional.softplus(dt + self.w(p + "dt_bias"), threshold=1e9)
        share = x.shape[2] // KV_HEADS
        b, c = (y.repeat_interleave(share, 2) for y in (b, c))
        y = _walk(c, b * dt[..., None], x, torch.exp(-self.w(p + "A_log").exp() * dt)[..., None]) + self.w(p + "D")[:, None] * x
        y = (y.flatten(2) * _silu(z)).unflatten(-1, (KV_HEADS, -1))
        return self.lin(_rms(y, 1e-5).flatten(2) * self.w(p + "norm"), p + "o")

    # -- Kisepel
    def kisepel(self):
        first = lambda x, n: _rms(x, 1e-5) * (1.0 + self.w(n))
        x = self.w("embed")[self.ids] * 8.0
        for i, layer in enumerate(self.cfg["layers"]):
            p = f"l{i}."
            h = first(x, p + "norm1")
            y = {"mamba2": self.ssm, "parallel": self.chunks_and_delta, "lightning": self.lightning}[layer["type"]](h, p + "mix.")
            x = x + y + (self.experts(h, p + "mlp.") if layer["mlp"] else 0.0)
        return first(x, "final.norm") * 0.5, "embed"

    def gated(self, h, p):
        return self.lin(_silu(self.lin(h, p + "gate")) * self.lin(h, p + "up"), p + "down")

    def experts(self, h, p):
        flat, chosen = h.flatten(0, 1), self.weights[p + "table"].long()[self.ids].flatten(0, 1)[:, :2]
        out = self.gated(flat, p + "shared.")
        for e in range(8):
            rows = (chosen == e).any(-1).nonzero()[:, 0]
            out[rows] += 0.5 * self.gated(flat[rows], f"{p}e{e}.")
        return out.view(h.shape)

    def lightning(self, h, p):
        q, k, v = (_silu(self.heads(h, p + n)) for n in "qkv")
        heads = q.shape[2]
        decay = torch.tensor([1.0 - 2.0 ** -(3 + 5 * i / max(1, heads - 1)) for i in range(heads)], dtype=torch.float64, device=h.device)
        o = _walk(q, k, v, decay[None, None, :, None].expand(q.shape[0], q.shape[1], heads, 1)).flatten(2)
        return self.lin(_rms(o, 1e-5) * self.w(p + "norm") * torch.sigmoid(self.lin(h, p + "g")), p + "o")

    def chunks_and_delta(self, h, p):
        l, r = p + "left.", p + "right."
        q, k = (_turn(_rms(self.heads(h, l + n), 1e-5) * self.w(f"{l}{n}.norm"), DIM, 1e6, 4.0) for n in "qk")
        left = self.lin(_attend(q, k, self.heads(h, l + "v"), DIM ** -0.5, seen=lambda i, j: i // 1024 == j // 1024), l + "o")
        q, k, v = (_silu(_conv(self.lin(h, r + n), self.w(f"{r}{n}.conv"))).unflatten(-1, (-1, DIM)) for n in "qkv")
        q, k = (z * torch.rsqrt(z.square().sum(-1, keepdim=True) + 1e-6) for z in (q, k))
        z = self.lin(self.lin(h, r + "a1"), r + "a2") + self.w(r + "dt_bias")
        decay = torch.exp(-self.w(r + "A_log").exp()[:, None] * torch.nn.functional.softplus(z, threshold=1e9).unflatten(-1, (-1, DIM)))
        o = _walk(q * DIM ** -0.5, k, v, decay, beta=torch.sigmoid(self.lin(h, r + "b")))
        gate = torch.sigmoid(self.lin(self.lin(h, r + "g1"), r + "g2"))
        right = self.lin((_rms(o, 1e-5) * self.w(r + "norm")).flatten(2) * gate, r + "o")
        return 0.5 * (_rms(left, 1e-5) * self.w(p + "left.out") + _rms(right, 1e-5) * self.w(p + "right.out"))


def exact(case, seed):
    """The logits of a state's first pass.  The weights are the ones ``Model.random`` makes from this configuration and seed."""
    from rust_inference_amd.config import config_from_dict
    from rust_inference_amd.parts.model import expected_tensors
    from rust_inference_amd.weights import random_tensors
    device = "cuda" if torch.cuda.is_available() else "cpu"
    arch, cfg = config_from_dict(config(case))
    weights = random_tensors(expected_tensors(arch.build_spec(cfg), for_writing=True), seed, torch.bfloat16, device=device)
    prompts, answer = _tokens(case, seed)
    if case["phase"] == "decode":
        prompts = [p + [answer[i][n] for i in range(ANSWERED)] for n, p in enumerate(prompts)]
    longest = max(len(p) for p in prompts)
    rows = []
    together = max(1, 16384 // longest)                       # sequences side by side: what the scans' launches cost is shared
    for at in range(0, len(prompts), together):
        part = prompts[at:at + together]
        ids = torch.tensor([p + [0] * (longest - len(p)) for p in part], device=device)
        plain = _Plain(case, weights, ids)
        x, head = getattr(plain, case["design"])()
        last = torch.tensor([len(p) - 1 for p in part], device=device)
        logits = x[torch.arange(len(part), device=device), last] @ plain.w(head).T
        rows.append(30.0 * torch.tanh(logits / 30.0) if case["design"] == "dagezen" else logits)
    return torch.cat(rows)
