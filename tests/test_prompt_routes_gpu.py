"""Which kernels a prompt's parts choose, and that what they choose agrees with the plain functions: parts alone, at sizes that
reach the kernels of long prompts; the same of products of a few rows with large matrices.

Like tests/test_kernels_gpu.py these run without a GPU when the environment says RI_TEST_KERNELS=emulated
(tests/test_kernels_emulated.py starts that run): the CPU build of the same sources."""
import math
import os

import numpy as np
import pytest
import torch

from helpers import rel_to_max
from plain import dagezen_plain as P

EMULATED = os.environ.get("RI_TEST_KERNELS") == "emulated"
pytestmark = [] if EMULATED else pytest.mark.gpu
DEV = "cpu" if EMULATED else "cuda:0"
PAGE = 32


@pytest.fixture(scope="module")
def ops():
    if EMULATED:
        import emulated
        return emulated.ops()
    from rust_inference_amd.kernels import ops
    return ops


def runtime_of(dtype, invariant=False):
    from rust_inference_amd.parts import Runtime
    if not EMULATED:
        return Runtime(DEV, dtype, invariant)
    made = Runtime.__new__(Runtime)                          # (a runtime refuses to be made for the CPU)
    made.device, made.dtype, made.invariant, made._mm_out_dtype = torch.device(DEV), dtype, invariant, None
    return made


@pytest.fixture(scope="module")
def rt(ops):
    return runtime_of(torch.bfloat16)


def t(a, dtype=torch.float32):
    return torch.tensor(np.asarray(a), dtype=dtype, device=DEV)


def f64(x):
    return x.detach().to("cpu", torch.float64).numpy()


def calls_of(monkeypatch, ops, name):
    """What is given to ``ops.<name>`` from now on, call by call."""
    real, seen = getattr(ops, name), []

    def recorded(*args, **kw):
        seen.append((args, kw))
        return real(*args, **kw)
    monkeypatch.setattr(ops, name, recorded)
    return seen


def random_weights(part, rng, std=0.1):
    return {name: torch.tensor(std * rng.normal(size=spec.shape) + (spec.kind == "gain")).to(torch.bfloat16)
            for name, spec in part.tensors().items()}


class Sequences:
    """Sequences that take tokens step by step, their pages in shuffled order: a step's context and the store of one cache entry."""

    def __init__(self, need, most, rng):
        from rust_inference_amd.cache import KVView
        held = -(-most // PAGE)
        order = rng.permutation(held * 8)
        self.table, self.done = order.reshape(8, held), [0] * 8
        pages = (held * 8, need.kv_heads)
        k, v = torch.zeros(pages + (PAGE, need.head_dim)), torch.zeros(pages + (need.value_dim, PAGE))
        self.store = KVView(0, k.to(DEV, torch.bfloat16), v.to(DEV, torch.bfloat16), PAGE, None)

    def step(self, counts):
        """``counts[s]`` tokens of sequence ``s`` (0: none): the context, the page table, (sequence, first, last) of each."""
        from rust_inference_amd.parts.context import StepContext
        seqs = [s for s, n in enumerate(counts) if n]
        new, starts = [counts[s] for s in seqs], [self.done[s] for s in seqs]
        for s in seqs:
            self.done[s] += counts[s]
        i32 = lambda a: t(a, torch.int32)
        pos = [p for n, at in zip(new, starts) for p in range(at, at + n)]
        ctx = StepContext(T=sum(new), B=len(seqs), new_counts=new, slot_list=seqs, starts=starts, tokens=i32(np.zeros(sum(new))),
                          tok_seq=i32(np.repeat(np.arange(len(seqs)), new)), tok_pos=i32(pos), slots=i32(seqs),
                          cu_seqlens=i32(np.concatenate([[0], np.cumsum(new)])), len_after=i32([self.done[s] for s in seqs]),
                          max_new=max(new), max_len=max(a + n for a, n in zip(starts, new)))
        return ctx, i32(self.table[seqs]), [(s, a, a + n) for s, a, n in zip(seqs, starts, new)]


# ---------------------------------------------------------------- latent attention
LATENT_STEPS = [[37, 100, 3, 0, 64], [90, 1, 40, 33], [0, 130], [1, 1, 1, 1, 1]]


@pytest.mark.parametrize("heads, dim, vdim, rank, extras, expanded", [
    (8, 64, 64, 72, True, 3), (2, 128, 128, 64, False, 3),
    (4, 64, 64, 100, True, 0),           # (rows of 164 elements: neither the rows side by side nor the turned part would be aligned)
    (3, 64, 64, 72, True, 0)])           # (queries in rows of 523)
def test_latent_attention_of_prompts(ops, rt, monkeypatch, heads, dim, vdim, rank, extras, expanded):
    """Fresh prompts of unequal lengths, prompts that go on in the middle of a page and at its border beside a single token, a
    sequence by itself, and single tokens: against 64 bits on the whole sequences, whether the heads' keys and values are made
    first or the attention runs on the latents.  The bound is the one for parts in bfloat16: weights, latents and results of
    eight bits."""
    from rust_inference_amd.parts import PartSpec, build_part
    rng = np.random.default_rng(heads + rank)
    rot, hidden, scale, eps = 64, 96, 0.11, 1e-5
    part = build_part("mixer", PartSpec("latent_attention", {
        "hidden": hidden, "heads": heads, "dim": dim, "rot_dim": rot, "vdim": vdim, "kv_rank": rank, "scale": scale, "prefix": "a.",
        "eps": eps, "sinks": extras, "gate": extras, "position": PartSpec("rotate_pairs", {"head_dim": rot, "dims": rot, "base": 1e4})}))
    w = random_weights(part, rng)
    part.bind(w, rt)
    w64 = {name: f64(x) for name, x in w.items()}
    if not extras:                                           # (the plain function has both: a gate of 1 and a sink of nothing)
        w64["a.sink"], w64["a.g"] = np.full(heads, -np.inf), None
    m = {"heads": heads, "dim": dim, "rot_dim": rot, "vdim": vdim, "kv_rank": rank, "scale": scale, "rot": {"dims": rot, "base": 1e4}}
    seqs = Sequences(part.cache_need(), 240, rng)
    x = {s: t(rng.normal(size=(240, hidden)), torch.bfloat16) for s in range(5)}
    made = calls_of(monkeypatch, ops, "latent_prompt")
    got = {s: [] for s in range(5)}
    for counts in LATENT_STEPS:
        ctx, table, own = seqs.step(counts)
        out = part.forward(torch.cat([x[s][a:b] for s, a, b in own]), ctx, seqs.store, table)
        rows = f64(ops.as_rows(out) if out.dim() == 2 else out.sum(0))
        for s, a, b in own:
            got[s].append(rows[:b - a])
            rows = rows[b - a:]
    assert len(made) == expanded
    for s in range(5):
        have = np.concatenate(got[s])
        want = latent_mixer(f64(x[s][:len(have)]), w64, m, eps)
        assert rel_to_max(have, want) < 2e-2, f"sequence {s}"


def latent_mixer(h, w, m, eps):
    if w["a.g"] is None:
        w = dict(w, **{"a.g": np.zeros((m["heads"], h.shape[1])), "a.o": 2.0 * w["a.o"]})
    return P.latent_mixer(h, w, "a.", m, eps, {})


# ---------------------------------------------------------------- products in tiles
def placeless(rows, columns, stride=None, dtype=torch.bfloat16):
    """A matrix that is nowhere in memory, for rules that look at sizes alone."""
    return torch.empty((rows, columns if stride is None else stride), dtype=dtype, device="meta")[:, :columns]


def test_products_in_tiles_only_where_the_kernel_takes_them(ops, rt):
    """Matrices and rows on both sides of what the kernel can address; what is beyond stays with the library's product."""
    from rust_inference_amd.parts.runtime import Runtime
    tile = lambda m, n, k, out=torch.bfloat16, act=None, x=None, w=None, ldo=None: Runtime._tile(
        rt, placeless(m, k, x), placeless(n, k, w), out, act, **({} if ldo is None else {"ldo": ldo}))
    for gate in ("silu_gate", "clamped_gate"):
        assert tile(2048, 2 * 65536, 16384 - 64, act=gate) is not None          # (65,536 + 256 rows of w from a workgroup's first)
        assert tile(2048, 2 * 65536, 16384, act=gate) is None
        assert tile(2048, 2 * 65536, 8192, w=16384, act=gate) is None
    assert tile(4096, 8192, 4096, torch.float32, x=(1 << 22) - 8) is not None and tile(4096, 8192, 4096, torch.float32, x=1 << 22) is None
    assert tile(4096, 8192, 4096, torch.float32, w=(1 << 22) - 8) is not None and tile(4096, 8192, 4096, torch.float32, w=1 << 22) is None
    assert tile(4096, (1 << 22) - 8, 4096, torch.float32) is not None and tile(4096, 1 << 22, 4096, torch.float32) is None
    assert tile(4096, 8192, 4096, torch.float32, ldo=(1 << 22) - 8) is not None and tile(4096, 8192, 4096, torch.float32, ldo=1 << 22) is None


def test_latent_prompts_only_where_the_kernel_takes_them(ops, rt):
    """Steps on both sides of what one launch can hold: rows by their padded pages, runs of 128 tokens; beyond, the latents."""
    from rust_inference_amd.parts import PartSpec, build_part
    part = build_part("mixer", PartSpec("latent_attention", {"hidden": 64, "heads": 1, "dim": 64, "rot_dim": 64, "vdim": 64, "kv_rank": 64, "scale": 0.1,
                                                             "prefix": "a.", "sinks": False, "gate": False}))
    part.bind(random_weights(part, np.random.default_rng(0)), rt)

    class Step:
        def __init__(self, new, starts):
            self.new_counts, self.starts, self.T, self.B = new, starts, sum(new), len(new)
    pays = lambda new, starts: part._expand_pays(Step(new, starts), placeless(1, part.w_in.n), type("Store", (), {"page_size": PAGE}))
    most = part.EXPAND_BYTES // (2 * (part.dim + part.vdim))          # rows that the keys and values of one head may have
    assert pays([most // 2], [most // 2]) and not pays([most // 2], [most // 2 + 1])
    assert pays([32] * 52758, [0] * 52758) and not pays([32] * 52759, [0] * 52759)           # 31 B / 128 + B of 65,535 and 65,536
    part.EXPAND_BYTES >>= 7
    assert pays([33] * (most >> 13), [0] * (most >> 13)) and not pays([33] * ((most >> 13) + 1), [0] * ((most >> 13) + 1))


@pytest.fixture
def small_machine(ops, monkeypatch):
    """The rule of the products in tiles on a machine of two compute units, from 128 rows on; the kernel runs on the real one."""
    from rust_inference_amd.parts import runtime
    runtime._tiles_plan.cache_clear()
    monkeypatch.setattr(runtime, "_compute_units", lambda: 2)
    monkeypatch.setattr(runtime, "TILES_MIN_ROWS", 128)
    yield calls_of(monkeypatch, ops, "gemm_tiles_bf16")
    runtime._tiles_plan.cache_clear()


def activation_of(call):
    args, kw = call
    return args[4] if len(args) > 4 else kw.get("activation")


def sigmoid(z):
    return 1.0 / (1.0 + np.exp(-z))


class Forms:
    """The gated forms and the squared ReLU in 64 bits."""

    @staticmethod
    def clamped(g, u, limit):
        g, u = np.minimum(g, limit), np.clip(u, -limit, limit)
        return g * sigmoid(1.702 * g) * (u + 1.0)

    silu = staticmethod(lambda g, u: g * sigmoid(g) * u)
    relu2 = staticmethod(lambda z: np.maximum(z, 0.0) ** 2)


@pytest.mark.parametrize("rows, tiles", [(250, True), (100, False)])
@pytest.mark.parametrize("kind", ["swiglu", "relu2", "gelu_tanh", "clamped", "clamped with biases"])
def test_feed_forward_of_prompts(ops, rt, monkeypatch, small_machine, kind, rows, tiles):
    """A feed-forward whose products go in tiles, the activation in the first of them, and one of too few rows, where the activation
    is a kernel of its own: both against 64 bits (gate and up exchanged, a bias or a clamp left out would be of order one)."""
    from rust_inference_amd.parts import PartSpec, build_part
    rng = np.random.default_rng(rows + len(kind))
    hidden, inter, limit = 256, 192, 0.9
    name, args = {"swiglu": ("swiglu", {}), "relu2": ("dense", {"activation": "relu2"}), "gelu_tanh": ("dense", {"activation": "gelu_tanh"}),
                  "clamped": ("glu_clamped", {"limit": limit, "biases": False}), "clamped with biases": ("glu_clamped", {"limit": limit})}[kind]
    part = build_part("feed_forward", PartSpec(name, {"hidden": hidden, "inter": inter, "prefix": "m.", **args}))
    w = random_weights(part, rng)
    part.bind(w, rt)
    w = {key[2:].replace("_proj.weight", ""): f64(x) for key, x in w.items()}
    x = t(rng.normal(size=(rows, hidden)), torch.bfloat16)
    out = part.forward(x, None)
    out = f64(out if out.dim() == 2 else out.sum(0))
    if getattr(part, "out_bias", None) is not None:
        out = out + f64(part.out_bias)
    h = f64(x)
    up = h @ w["up"].T + w.get("up.b", 0.0)
    if "gate" in w:
        gate = h @ w["gate"].T + w.get("gate.b", 0.0)
        act = Forms.silu(gate, up) if kind == "swiglu" else Forms.clamped(gate, up, limit)
    else:
        act = Forms.relu2(up) if kind == "relu2" else 0.5 * up * (1.0 + np.tanh(np.sqrt(2 / np.pi) * (up + 0.044715 * up ** 3)))
    assert rel_to_max(out, act @ w["down"].T + w.get("down.b", 0.0)) < 2e-2
    fused = {"swiglu": "silu_gate", "relu2": "relu2", "gelu_tanh": None}.get(kind, "clamped_gate")
    want = ([fused] if fused else []) + [None] if tiles else []
    assert [activation_of(call) for call in small_machine] == want


@pytest.mark.parametrize("kind", ["silu", "clamped", "relu2", "gelu_erf"])
def test_experts_of_prompts(ops, rt, monkeypatch, small_machine, kind):
    """Experts whose rows lie side by side, two of them with enough for tiles and one without: the activation in the product, and beside
    it, against 64 bits; the stretches of the two matrices are an expert's own."""
    from rust_inference_amd.parts import PartSpec, build_part
    rng = np.random.default_rng(len(kind))
    hidden, inter, vocab, tokens, limit = 256, 192, 40, 508, 0.8
    args = {"silu": {"limit": None}, "clamped": {"limit": limit}}.get(kind, {"limit": None, "gated": False, "activation": kind})
    part = build_part("feed_forward", PartSpec("routed_experts", {"hidden": hidden, "inter": inter, "experts": 3, "top": 1, "prefix": "m.", "scores": "table",
                                                                  "vocab": vocab, "shared_gate": False, **args}))
    w = random_weights(part, rng)
    w["m.table"] = torch.tensor([[0 if i < 20 else 1 if i < 38 else 2] for i in range(vocab)], dtype=torch.int32)
    part.bind(w, rt)
    ids = np.concatenate([rng.integers(0, 20, 250), rng.integers(20, 38, 240), rng.integers(38, 40, 18)])
    rng.shuffle(ids)
    x = t(rng.normal(size=(tokens, hidden)), torch.bfloat16)
    ctx = type("Step", (), {"tokens": t(ids, torch.int32), "T": tokens, "is_decode": False})
    if EMULATED:                                             # (the host's wait for the row counts needs a GPU)
        def sort(x, chosen):
            dest, offsets = ops.experts_sort(chosen, part.outs)
            return ops.experts_gather(x, dest, part.top), dest, offsets, type("There", (), {"synchronize": staticmethod(lambda: None)})
        monkeypatch.setattr(part, "sort", sort)
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    out = part.forward(x, ctx)
    out = f64(out if out.dim() == 2 else out.sum(0))
    h, want, w = f64(x), np.zeros((tokens, hidden)), {key[2:]: f64(v) for key, v in w.items()}
    erf = np.vectorize(math.erf)
    for e in range(3):
        mine = w["table"][ids, 0] == e
        up = h[mine] @ w[f"e{e}.up"].T
        if kind in ("silu", "clamped"):
            gate = h[mine] @ w[f"e{e}.gate"].T
            act = Forms.silu(gate, up) if kind == "silu" else Forms.clamped(gate, up, limit)
        else:
            act = Forms.relu2(up) if kind == "relu2" else 0.5 * up * (1.0 + erf(up / np.sqrt(2.0)))
        want[mine] = act @ w[f"e{e}.down"].T
    assert rel_to_max(out, want) < 2e-2
    fused = {"silu": ["silu_gate"], "clamped": ["clamped_gate"], "relu2": ["relu2"], "gelu_erf": []}[kind]
    assert [activation_of(call) for call in small_machine] == (fused + [None]) * 2


@pytest.mark.parametrize("kind", ["silu", "clamped", "relu2"])
def test_experts_of_prompts_in_one_launch(ops, rt, monkeypatch, kind):
    """From four experts on, two a token, one that nobody takes: two products for all of them, against 64 bits."""
    from rust_inference_amd.parts import PartSpec, build_part
    rng = np.random.default_rng(len(kind))
    hidden, inter, vocab, tokens, limit, experts = 256, 192, 40, 300, 0.8, 5
    args = {"silu": {"limit": None}, "clamped": {"limit": limit}}.get(kind, {"limit": None, "gated": False, "activation": kind})
    part = build_part("feed_forward", PartSpec("routed_experts", {"hidden": hidden, "inter": inter, "experts": experts, "top": 2, "prefix": "m.",
                                                                  "scores": "table", "vocab": vocab, "shared_gate": False, **args}))
    w = random_weights(part, rng)
    w["m.table"] = torch.tensor([[i % 2, 2 if i < 30 else 4] for i in range(vocab)], dtype=torch.int32)
    part.bind(w, rt)
    ids = rng.integers(0, vocab, tokens)
    x = t(rng.normal(size=(tokens, hidden)), torch.bfloat16)
    ctx = type("Step", (), {"tokens": t(ids, torch.int32), "T": tokens, "is_decode": False})
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    calls = calls_of(monkeypatch, ops, "gemm_tiles_groups")
    out = f64(part.forward(x, ctx))
    h, want, w = f64(x), np.zeros((tokens, hidden)), {key[2:]: f64(v) for key, v in w.items()}
    for e in range(experts):
        mine = (w["table"][ids] == e).any(1)
        up = h[mine] @ w[f"e{e}.up"].T
        act = Forms.relu2(up)
        if kind != "relu2":
            gate = h[mine] @ w[f"e{e}.gate"].T
            act = Forms.silu(gate, up) if kind == "silu" else Forms.clamped(gate, up, limit)
        want[mine] += 0.5 * (act @ w[f"e{e}.down"].T)
    assert rel_to_max(out, want) < 2e-2
    assert len(calls) == 2


@pytest.mark.parametrize("m", [1, 3, 20])
@pytest.mark.parametrize("mode", ["bfloat16", "invariant", "float32"])
def test_weights_of_one_size_in_the_storage_they_come_in(ops, mode, m):
    """Weights that go together, some stored in bfloat16 and some in float32: the bits of each alone; the float32 path keeps every one in
    its own storage, bfloat16 has them side by side."""
    rt = runtime_of(torch.float32 if mode == "float32" else torch.bfloat16, mode == "invariant")
    rng = np.random.default_rng(m)
    n, k, stored = 48, 264, (torch.bfloat16, torch.float32, torch.bfloat16, torch.float32)
    ws = [t(rng.normal(size=(n, k)) / np.sqrt(k), kind) for kind in stored]
    x = t(rng.normal(size=(4, m, k)), rt.dtype)
    together = rt.stack(ws)
    assert [pw.w.dtype for pw in together.each] == (list(stored) if mode == "float32" else [torch.bfloat16] * 4)
    assert (together.w is not None) == (mode == "bfloat16") and (together.packed is None or mode == "bfloat16")
    for got, one, w in zip(rt.linear_each(x, together), x, ws):
        assert torch.equal(got, ops.as_rows(rt.linear_packed(one.contiguous(), rt.pack(rt.place_matrix(w)))))
    from rust_inference_amd.errors import ShapeError
    with pytest.raises(ShapeError):
        rt.stack([ws[0], ws[1][:1]])
    if mode != "invariant":                                  # (rows of no multiple of 8 are the library's, each matrix from an address of its own)
        odd = [w[:, :13].contiguous() for w in ws]
        assert rt.stack(odd).w is None
        for got, one, w in zip(rt.linear_each(x[:, :, :13].contiguous(), rt.stack(odd)), x, odd):
            assert rel_to_max(f64(got), f64(one)[:, :13] @ f64(w).T) < 1e-2


@pytest.mark.parametrize("lie", ["side by side", "rows of longer ones", "x off a line", "w off a line", "w transposed", "x transposed", "results off a line",
                                 "results in rows of 252"])
def test_rows_and_matrices_that_lie_as_the_tiles_want_them(ops, rt, small_machine, lie):
    """Products into given rows: stretches of longer rows go in tiles; what lies off a multiple of sixteen bytes or across stays with the
    library, with the same result."""
    rng = np.random.default_rng(len(lie))
    m, n, k = 256, 256, 192
    put = lambda rows, columns, off=0, pad=0: torch.zeros(rows * (columns + pad) + off, dtype=torch.bfloat16, device=DEV)[off:].view(rows, columns + pad)[:, :columns]
    x, w, out = put(m, k), put(n, k), put(m, n)
    if lie == "rows of longer ones":
        x, w, out = put(m, k, 8, 16), put(n, k, 16, 8), put(m, n, 8, 24)
    elif lie == "x off a line":
        x = put(m, k, 4)
    elif lie == "w off a line":
        w = put(n, k, 4)
    elif lie == "w transposed":
        w = put(k, n).t()
    elif lie == "x transposed":
        x = put(k, m).t()
    elif lie == "results off a line":
        out = put(m, n, 4)
    elif lie == "results in rows of 252":
        out = put(m + 4, 252)[4:].as_strided((m, n - 8), (252, 1))
        w, n = put(n - 8, k), n - 8
    x.copy_(t(rng.normal(size=(m, k))))
    w.copy_(t(rng.normal(size=(n, k))))
    rt.rows_into(out, x, w)
    assert rel_to_max(f64(out), f64(x) @ f64(w).T) < 4e-3
    assert len(small_machine) == (lie in ("side by side", "rows of longer ones"))


def test_the_rule_of_the_products_in_tiles(monkeypatch):
    """On 256 compute units, at sizes measured beside the rule: full rounds, an activation that rides along, and what is left to the library."""
    from rust_inference_amd.parts import runtime
    from rust_inference_amd.kernels.ops import TILES
    monkeypatch.setattr(runtime, "_compute_units", lambda: 256)
    runtime._tiles_plan.cache_clear()
    plan = runtime._tiles_plan
    large, wide, tall = TILES.index((256, 256)), TILES.index((128, 256)), TILES.index((256, 128))
    assert plan(2048, 4096, 4096, False, None) in (wide, tall) and plan(1536, 5120, 5120, True, None) in (wide, tall)       # one round
    assert plan(2048, 3400, 4096, False, None) is None                                  # (0.83 of one round)
    assert plan(8192, 5120, 8192, False, None) == large and plan(5120, 8192, 4096, False, None) == large                    # three rounds, 0.8 to 0.93
    assert plan(8192, 12288, 4096, False, None) is None and plan(8192, 12288, 4096, True, None) == large                    # full: float32 results alone
    for act in ("silu_gate", "clamped_gate"):
        assert plan(2048, 24576, 4096, False, act) == large and plan(759, 24576, 4096, False, act) is not None
        assert plan(759, 6144, 1024, False, act) is not None and plan(759, 6144, 4096, False, act) is None                  # 0.45 for short rows, else 0.62
        assert plan(2048, 24576 + 8, 4096, False, act) is None                          # (halves that are no multiple of 8)
    assert plan(759, 6144, 1024, False, "relu2") is None and plan(2048, 18432, 4096, False, "relu2") == tall              # 0.1 more without a gate
    for m, n, k in ((511, 4096, 4096), (2048, 4096, 4096 + 32), (2048, 4096, 128), (2048, 4096 + 4, 4096)):
        assert plan(m, n, k, False, None) is None and plan(m, n, k, False, "relu2") is None
    runtime._tiles_plan.cache_clear()


def test_the_rule_of_products_in_groups(monkeypatch):
    """Four to 64 groups of sizes that the kernel takes; the smaller tile where its rounds are the shorter."""
    from rust_inference_amd.parts import runtime
    monkeypatch.setattr(runtime, "_compute_units", lambda: 256)
    runtime._groups_tile.cache_clear()
    tile = lambda m, groups, n, k, ldw=None, gated=False: runtime._groups_tile(m, groups, n, k, ldw or k, gated)
    assert tile(9842, 8, 6144, 4096, gated=True) == 0 and tile(9842, 8, 4096, 6144, 8 * 6144) == 0
    assert tile(512, 8, 6144, 4096, gated=True) == 1 and tile(512, 64, 64, 192) == 1
    assert tile(9842, 3, 6144, 4096) is None and tile(9842, 65, 6144, 4096) is None
    assert tile(9842, 8, 6144, 4128) is None and tile(9842, 8, 6148, 4096) is None and tile(9842, 8, 6144, 128) is None
    assert tile(9842, 8, 6144, 4096, 1 << 22) is None
    runtime._groups_tile.cache_clear()


# ---------------------------------------------------------------- steps of a few rows
# float32 sums of the library's product of bfloat16; on the CPU torch rounds them to bfloat16 first (half a unit in the eighth bit)
LIBRARY_F32 = 2.0 ** -8 if EMULATED else 1e-5


def output_head(rt, monkeypatch, vocab, dim, rng):
    from rust_inference_amd.parts import PartSpec, build_part
    head = build_part("head", PartSpec("linear", {"vocab": vocab, "dim": dim, "name": "head", "tied": False}))
    w = torch.tensor(rng.normal(size=(vocab, dim)) / np.sqrt(dim)).to(torch.bfloat16)
    head.bind({"head": w}, rt)
    if EMULATED:
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    return head, f64(w)


@pytest.mark.parametrize("rows", [3, 20, 64])
def test_output_matrix_without_room_for_a_second_copy(ops, monkeypatch, rows):
    """The library's product then, and no second attempt; the invariant mode has no other product and says what is missing."""
    rng = np.random.default_rng(rows)
    x = t(rng.normal(size=(rows, 64)), torch.bfloat16)
    for invariant in (False, True):
        rt = runtime_of(torch.bfloat16, invariant)
        head, w = output_head(rt, monkeypatch, 256 * 64, 64, rng)
        monkeypatch.setattr(type(rt), "many_waves", staticmethod(lambda n, k, m, few: 8 if m > 16 else None))
        tried = []

        def full(*args, **kw):
            tried.append(args)
            raise torch.OutOfMemoryError("no room")
        monkeypatch.setattr(rt, "pack", full)
        if invariant:
            with pytest.raises(torch.OutOfMemoryError):
                head.forward(x)
            continue
        for _ in range(2):
            assert rel_to_max(f64(head.forward(x)), f64(x) @ w.T) < LIBRARY_F32
        assert len(tried) == 1


# (results, K) -> row tiles a workgroup on a machine of one compute unit: bfloat16 and float32 results at 17, 48, 49 and 64 rows, an output matrix at 9, 16
# and those; 0: three or four up to 48 rows, then the library
MANY_TILES = {(288, 72): ((20, 20, 0, 0), (20, 20, 20, 20), (6, 6, 20, 20, 20, 20)), (250, 72): ((8, 8, 0, 0), (8, 8, 8, 8), (0, 8, 8, 8, 8, 8)),
              (250, 2056): ((8, 8, 8, 8), (8, 8, 8, 8), (0, 8, 8, 8, 8, 8)), (380, 72): ((8, 12, 0, 0), (8, 12, 12, 12), (0, 8, 8, 12, 12, 12)),
              (620, 72): ((20, 20, 0, 0), (20, 20, 20, 20), (20,) * 6), (410, 72): ((0, 8, 0, 0), (0, 8, 8, 8), (0, 0, 0, 8, 8, 8))}


@pytest.mark.parametrize("rows", [9, 16, 17, 48, 49, 64, 65])
@pytest.mark.parametrize("n, k", list(MANY_TILES))
def test_products_of_many_row_tiles_are_sent_to_the_form_that_is_chosen(ops, rt, monkeypatch, n, k, rows):
    """A plain matrix and an output matrix at the edges of the rows that each form takes: what the kernel is given, and float64.  Where the rule
    has no form of many row tiles, a plain matrix has three or four from 17 to 48 rows, an output matrix four from 9 rows on, and others the rest."""
    from rust_inference_amd.parts import runtime
    runtime._wide_many_waves.cache_clear()
    monkeypatch.setattr(runtime, "_compute_units", lambda: 1)
    monkeypatch.setattr(runtime, "MID_MAX_BYTES", 0)           # (matrices of these sizes are the packed kernel's otherwise)
    rng = np.random.default_rng(n + rows)
    head, w = output_head(rt, monkeypatch, n, k, rng)
    x = t(rng.normal(size=(rows, k)), torch.bfloat16)
    want = f64(x) @ w.T
    half, whole, logits = ({9: 0, 16: 0, 17: a[-4], 48: a[-3], 49: a[-2], 64: a[-1]}.get(rows, 0) for a in MANY_TILES[n, k])
    logits = {9: MANY_TILES[n, k][2][0], 16: MANY_TILES[n, k][2][1]}.get(rows, logits)
    wide = calls_of(monkeypatch, ops, "gemm_wide_packed_bf16")

    plain = rt.pack(t(w, torch.bfloat16), always=True)
    for dtype, bound, many in ((torch.bfloat16, 1e-2, half), (torch.float32, LIBRARY_F32, whole)):
        wide.clear()
        assert rel_to_max(f64(rt.linear_packed(x, plain, out_dtype=dtype)), want) < bound
        given = [kw["waves"] for _, kw in wide]
        assert given == ([many] if many else [runtime._wide_whole_waves(n, rows)] if 17 <= rows <= 48 else [])
        assert many or not given or given[0] in (3, 4)
    wide.clear()
    made = head.forward(x)
    assert made.dtype == torch.float32 and rel_to_max(f64(made), want) < LIBRARY_F32
    assert [kw["waves"] for _, kw in wide] == ([logits] if logits else [4] if rows <= 48 else [])
    assert (head.packed is not None) == bool(wide)
    runtime._wide_many_waves.cache_clear()
