"""The kernels of the Dagezen design alone, each against the plain function of its mechanism
(tests/plain/dagezen_plain.py), at sizes that are no power of two and differ from one another.

Like tests/test_kernels_gpu.py these run without a GPU when the environment says RI_TEST_KERNELS=emulated
(tests/test_kernels_emulated.py starts that run): the CPU build of the same sources between guard pages."""
import math
import os

import numpy as np
import pytest
import torch

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


@pytest.fixture(autouse=True)
def _guarded_buffers_go_back():
    yield
    if EMULATED:
        import gc
        import emulated
        gc.collect()
        emulated.free_all()


def guarded(x):
    if EMULATED:
        import emulated
        return emulated.tensor(x.contiguous(), "a test's operand")
    return x


def t(a, dtype=torch.float32):
    return guarded(torch.tensor(np.asarray(a), dtype=dtype, device=DEV))


def f64(x):
    return x.detach().to("cpu", torch.float64).numpy()


def close(got, want, rel, what=""):
    want = np.asarray(want, dtype=np.float64)
    err = np.abs(f64(got) - want).max() / max(np.abs(want).max(), 1e-30)
    assert err <= rel, f"{what}: error {err:.3e} of the largest value exceeds {rel:.0e}"


F32 = 5e-6


class Steps:
    """Sequences of unequal lengths cut into steps, with pages handed out in shuffled order: what a kernel gets of a
    step's layout (``tok_seq``, ``tok_pos``, ``cu_seqlens``, ``slots``, the page table)."""

    def __init__(self, lengths, slots, rng, pages=64):
        self.lengths, self.slots, self.done = list(lengths), list(slots), [0] * len(lengths)
        order = rng.permutation(pages)
        width = max(-(-n // PAGE) for n in lengths)
        self.table = np.full((len(lengths), width), -1, dtype=np.int32)
        at = 0
        for s, n in enumerate(lengths):
            for p in range(-(-n // PAGE)):
                self.table[s, p] = order[at]
                at += 1
        self.pages = pages

    def step(self, counts):
        """The next ``counts[s]`` tokens of every sequence (0: the sequence sits this step out)."""
        seqs = [s for s, c in enumerate(counts) if c > 0]
        tok_seq, tok_pos, cu, rows = [], [], [0], []
        for i, s in enumerate(seqs):
            for j in range(counts[s]):
                tok_seq.append(i)
                tok_pos.append(self.done[s] + j)
                rows.append((s, self.done[s] + j))
            cu.append(len(tok_seq))
            self.done[s] += counts[s]
        return dict(seqs=seqs, rows=rows, tok_seq=t(tok_seq, torch.int32), tok_pos=t(tok_pos, torch.int32),
                    cu=t(cu, torch.int32), slots=t([self.slots[s] for s in seqs], torch.int32),
                    table=t(self.table[seqs], torch.int32))


CUTS = [[(7, 3), (1, 1), (1, 0), (30, 36), (2, 1), (1, 1), (1, 1)]]      # (tokens of sequence 0, of sequence 1) step by step


# ---------------------------------------------------------------- the norm behind the sum, activations, the cap
@pytest.mark.parametrize("act", [None, torch.bfloat16])
@pytest.mark.parametrize("parts, dim", [(1, 70), (3, 256)])
def test_scaled_sum_norm(ops, act, parts, dim):
    rng = np.random.default_rng(1)
    rows, alpha, eps = 5, 2.5, 1e-5
    r, y = rng.standard_normal((rows, dim)), rng.standard_normal((parts, rows, dim))
    yb, g, b = rng.standard_normal(dim), 1 + 0.1 * rng.standard_normal(dim), 0.1 * rng.standard_normal(dim)
    res = t(r)
    got = ops.scaled_sum_norm(res, t(y if parts > 1 else y[0]), t(yb), alpha, t(g), t(b), eps, ops.NORM_LAYER, act)
    want = P.layer_norm(alpha * r + y.sum(0) + yb, g, b, eps)
    close(res, want, F32, "the residual")
    if act is not None:
        close(got, want, 8e-3, "its copy")
    res = t(r)
    ops.scaled_sum_norm(res, t(y[0]), None, alpha, t(g), None, eps, ops.NORM_RMS, None)
    close(res, P.rms_unit(alpha * r + y[0], eps) * g, F32, "rms")


def test_clamped_gate_with_biases_and_the_experts_plain_activation_and_the_cap(ops):
    rng = np.random.default_rng(2)
    rows, ff, limit = 6, 37, 1.5
    gu, bg, bu = 2 * rng.standard_normal((rows, 2 * ff)), rng.standard_normal(ff), rng.standard_normal(ff)
    g = np.minimum(gu[:, :ff] + bg, limit)
    u = np.clip(gu[:, ff:] + bu, -limit, limit)
    close(ops.glu_clamped_bias(t(gu), t(bg), t(bu), limit), g * P.sigmoid(1.702 * g) * (u + 1), F32, "clamped gate")
    wide = 2 * rng.standard_normal((3, 2 * 48))                       # bfloat16 rows of a multiple of 8: eight elements a thread
    gb, ub = rng.standard_normal(48), rng.standard_normal(48)
    rounded = f64(t(wide, torch.bfloat16))
    g8, u8 = np.minimum(rounded[:, :48] + gb, limit), np.clip(rounded[:, 48:] + ub, -limit, limit)
    close(ops.glu_clamped_bias(t(wide, torch.bfloat16), t(gb), t(ub), limit), g8 * P.sigmoid(1.702 * g8) * (u8 + 1), 8e-3,
          "clamped gate, bfloat16")
    experts = 5
    up, dense = rng.standard_normal((rows, experts * ff)), rng.random((rows, experts)) * (rng.random((rows, experts)) < 0.5)
    want = (P.gelu_erf(up).reshape(rows, experts, ff) * dense[:, :, None]).reshape(rows, -1)
    close(ops.experts_activate_plain(t(up), t(dense), ff, "gelu_erf"), want, F32, "experts without a gate")
    close(ops.gelu_erf(t(up)), P.gelu_erf(up), F32, "exact gelu")
    x = 40 * rng.standard_normal((3, 50))
    close(ops.softcap_rows(t(x), 15.0), 15.0 * np.tanh(x / 15.0), F32, "cap")


# ---------------------------------------------------------------- attention over a cached latent
@pytest.mark.parametrize("heads, dim, rot, vdim, rank", [(3, 20, 6, 12, 28), (2, 8, 16, 24, 72)])
def test_latent_attention_through_every_cut(ops, heads, dim, rot, vdim, rank):
    rng = np.random.default_rng(3)
    width, eps, scale = 40, 1e-5, 0.3
    m = {"heads": heads, "dim": dim, "rot_dim": rot, "vdim": vdim, "kv_rank": rank, "scale": scale,
         "rot": {"dims": rot, "base": 100.0}}
    w = {"q": rng.standard_normal((heads * (dim + rot), width)) / 6, "dkv": rng.standard_normal((rank + rot, width)) / 6,
         "dkv.norm": 1 + 0.1 * rng.standard_normal(rank), "uk": rng.standard_normal((heads * dim, rank)) / 5,
         "uv": rng.standard_normal((heads * vdim, rank)) / 5, "sink": rng.standard_normal(heads),
         "g": rng.standard_normal((heads, width)) / 6, "o": np.eye(heads * vdim)}
    inv_freq = t(100.0 ** (-2.0 * np.arange(rot // 2) / rot))
    w_uk = t(w["uk"].reshape(heads, dim, rank))
    w_uv = t(np.ascontiguousarray(w["uv"].reshape(heads, vdim, rank).transpose(0, 2, 1)))
    lengths = [43, 43]
    h = [rng.standard_normal((n, width)) for n in lengths]
    steps = Steps(lengths, [0, 1], rng)
    k_pages = guarded(torch.zeros((steps.pages, 1, PAGE, rank + rot), device=DEV))
    v_pages = guarded(torch.zeros((steps.pages, 1, rank, PAGE), device=DEV))
    states = [{}, {}]
    for counts in CUTS[0]:
        st = steps.step(counts)
        x = np.stack([h[s][p] for s, p in st["rows"]])
        proj = t(np.concatenate([x @ w["q"].T, x @ w["dkv"].T, x @ w["g"].T], 1))
        qw = heads * (dim + rot)
        ops.latent_prepare(proj, 0, qw, t(w["dkv.norm"]), eps, inv_freq, st["tok_pos"], st["tok_seq"], st["table"], k_pages,
                           v_pages, heads, dim, rot, rank)
        q = ops.head_products(proj, 0, dim + rot, w_uk, heads, dim, rank, extra=rot)
        o = ops.attention(q, k_pages, v_pages, st["tok_pos"], st["tok_seq"], st["table"], heads, 1, rank + rot, None, scale,
                          sinks=t(w["sink"]))
        got = ops.head_products(o, 0, rank, w_uv, heads, rank, vdim, gates=proj, g_off=qw + rank + rot)
        want, at = [], 0
        for s in st["seqs"]:
            n = sum(1 for r in st["rows"] if r[0] == s)
            want.append(P.latent_mixer(x[at:at + n], w, "", m, eps, states[s]))
            at += n
        close(got, np.concatenate(want), 2e-5, f"latent attention, step {counts}")


# ---------------------------------------------------------------- the windowed attention whose heads talk
@pytest.mark.skipif(EMULATED, reason="a thousand tokens; on an emulated machine of one unit the small tests take this form")
@pytest.mark.parametrize("heads, kv_heads, dim, window, first", [(32, 8, 32, 100, 1000), (16, 2, 32, None, 2000), (24, 8, 32, 64, 1000),
                                                                 (32, 8, 64, None, 1000), (32, 8, 128, 100, 1000), (32, 8, 128, None, 1000)])
def test_talking_attention_of_a_full_machine(ops, heads, kv_heads, dim, window, first):
    """Enough tiles that a wavefront of the first walk takes four heads, 512 wavefronts and more (and groups of three, which it cannot), with the
    table of distances and with a logarithm a score; against the general kernel."""
    counts = [first, 45, 3]
    assert heads % (4 * kv_heads) or sum(-(-n // 16) for n in counts) * heads // 4 >= 2 * 256
    rng = np.random.default_rng(heads)
    pages = -(-first // 32)
    k_pages, v_pages = ((torch.randn(shape, device=DEV) * 0.6).to(torch.bfloat16) for shape in
                        ((pages + 3, kv_heads, PAGE, dim), (pages + 3, kv_heads, dim, PAGE)))
    table = np.zeros((3, pages), dtype=np.int32)
    table[0], table[1, :2], table[2, 0] = np.arange(pages), [pages, pages + 1], pages + 2
    seq, pos = t([s for s, n in enumerate(counts) for _ in range(n)], torch.int32), t([i for n in counts for i in range(n)], torch.int32)
    proj = (torch.randn((sum(counts), heads * dim), device=DEV) * 0.6).to(torch.bfloat16)
    args = (heads, kv_heads, dim, window, 0.2, t(rng.random(heads)), t(rng.random(heads) * 3), t(np.eye(heads) + 0.2 * rng.standard_normal((heads, heads))))
    want = ops.talking_attention(proj, 0, k_pages, v_pages, pos, seq, t(table, torch.int32), *args)
    got = ops.talking_attention_mfma(proj, 0, k_pages, v_pages, pos, t(np.concatenate([[0], np.cumsum(counts)]), torch.int32), counts,
                                     t(table, torch.int32), *args, first)
    close(got, f64(want), 1.5e-2, "matrix cores against the general kernels")


@pytest.mark.parametrize("heads, kv_heads, dim, window, shares", [(4, 2, 12, 9, 1), (3, 3, 20, 33, 2), (6, 1, 8, 70, 1), (20, 2, 16, None, 3)])
def test_talking_attention_through_every_cut(ops, heads, kv_heads, dim, window, shares):
    rng = np.random.default_rng(4)
    width, eps, scale = 36, 1e-5, 0.4
    m = {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": dim, "scale": scale, "mask": {"size": window or 10 ** 6}}
    w = {"q": rng.standard_normal((heads * dim, width)) / 3, "k": rng.standard_normal((kv_heads * dim, width)) / 3,
         "q.norm": 1 + 0.1 * rng.standard_normal(heads * dim), "k.norm": 1 + 0.1 * rng.standard_normal(kv_heads * dim),
         "r1": rng.random(heads), "r2": rng.random(heads) * 3, "talk": np.eye(heads) + 0.3 * rng.standard_normal((heads, heads)),
         "g": rng.standard_normal((heads * dim, width)) / 6, "o": np.eye(heads * dim)}
    lengths = [43, 43]
    h = [rng.standard_normal((n, width)) for n in lengths]
    steps = Steps(lengths, [1, 0], rng)
    k_pages = guarded(torch.zeros((steps.pages, kv_heads, PAGE, dim), device=DEV))
    v_pages = guarded(torch.zeros((steps.pages, kv_heads, dim, PAGE), device=DEV))
    states = [{}, {}]
    for counts in CUTS[0]:
        st = steps.step(counts)
        x = np.stack([h[s][p] for s, p in st["rows"]])
        proj = t(np.concatenate([x @ w["q"].T, x @ w["k"].T, x @ w["g"].T], 1))
        qw, kw = heads * dim, kv_heads * dim
        ops.whole_norm_kv_write(proj, 0, qw, t(w["q.norm"]), t(w["k.norm"]), eps, st["tok_pos"], st["tok_seq"], st["table"],
                                k_pages, v_pages, heads, kv_heads, dim)
        o = ops.talking_attention(proj, 0, k_pages, v_pages, st["tok_pos"], st["tok_seq"], st["table"], heads, kv_heads, dim,
                                  window, scale, t(w["r1"]), t(w["r2"]), t(w["talk"]), shares)
        got = guarded(torch.zeros((len(x), qw + 3), device=DEV))
        ops.gate_rows(got, 3, o, proj, qw + kw, 0.5, ops.GATE_SIGMOID)
        want, at = [], 0
        for s in st["seqs"]:
            n = sum(1 for r in st["rows"] if r[0] == s)
            want.append(P.talking_mixer(x[at:at + n], w, "", m, eps, states[s]))
            at += n
        close(got[:, 3:], 0.5 * np.concatenate(want), 2e-5, f"talking attention, step {counts}")


@pytest.mark.parametrize("dtype, rel", [(torch.float32, F32), (torch.bfloat16, 8e-3)])
@pytest.mark.parametrize("heads, kv_heads, dim, stray", [(18, 9, 128, 0), (9, 3, 8, 0), (32, 16, 32, 0), (16, 4, 256, 0), (3, 1, 40, 4), (2, 1, 6, 0)])
def test_whole_norm_and_both_writes(ops, dtype, rel, heads, kv_heads, dim, stray):
    """Pieces of sixteen bytes and single elements (rows that they do not divide), prompts and single tokens, pages begun and left inside:
    keys normed over the row, values the keys as projected, the columns beside them and the pages' other places as they were."""
    rng = np.random.default_rng(heads)
    before, new = [0, 5, 31, 40, 24], [33, 1, 2, 24, 9]
    seq, pos = [b for b, n in enumerate(new) for _ in range(n)], [before[b] + i for b, n in enumerate(new) for i in range(n)]
    tokens, qw, kw, gap = len(seq), heads * dim, kv_heads * dim, 8 + stray
    rows = t(rng.standard_normal((tokens, gap + qw + kw + 8 + stray)), dtype)
    q_gain, k_gain = 1 + 0.1 * rng.standard_normal(qw), 1 + 0.1 * rng.standard_normal(kw)
    table = rng.permutation(10).reshape(5, 2)
    x = f64(rows)
    q, k = x[:, gap:gap + qw], x[:, gap + qw:gap + qw + kw]
    norm = lambda v, g: v / np.sqrt((v * v).mean(1, keepdims=True) + 1e-5) * g
    for bounds in ({}, dict(cu_seqlens=t(np.concatenate([[0], np.cumsum(new)]), torch.int32), max_new=max(new))):
        k_pages, v_pages = (t(np.full((10, kv_heads) + shape, 7.0), dtype) for shape in ((PAGE, dim), (dim, PAGE)))
        proj = guarded(rows.clone())
        ops.whole_norm_kv_write(proj, gap, gap + qw, t(q_gain), t(k_gain), 1e-5, t(pos, torch.int32), t(seq, torch.int32), t(table, torch.int32),
                                k_pages, v_pages, heads, kv_heads, dim, **bounds)
        got = f64(proj)
        close(t(got[:, gap:gap + qw]), norm(q, q_gain), rel, "queries")
        got[:, gap:gap + qw] = q
        assert np.array_equal(got, x)
        want_k, want_v, kn = np.full(k_pages.shape, 7.0), np.full(v_pages.shape, 7.0), norm(k, k_gain)
        for i, (b, p) in enumerate(zip(seq, pos)):
            want_k[table[b, p // PAGE], :, p % PAGE] = kn[i].reshape(kv_heads, dim)
            want_v[table[b, p // PAGE], :, :, p % PAGE] = k[i].reshape(kv_heads, dim)
        close(k_pages, want_k, rel, "keys")
        assert np.array_equal(f64(v_pages), want_v)


def test_a_key_at_the_windows_edge_counts_and_the_next_one_does_not(ops):
    """One loud key: at distance window - 1 it takes the softmax, at distance window it is not seen."""
    heads, dim, window, n = 2, 8, 37, 80
    k_pages = guarded(torch.zeros((4, 1, PAGE, dim), device=DEV))
    v_pages = guarded(torch.zeros((4, 1, dim, PAGE), device=DEV))
    for edge, seen in ((window - 1, True), (window, False)):
        loud = n - 1 - edge
        k_pages.zero_(), v_pages.zero_()
        k_pages[loud // PAGE, 0, loud % PAGE, :] = 30.0
        v_pages[loud // PAGE, 0, 0, loud % PAGE] = 1.0
        q = t(np.ones((1, heads * dim)))
        o = ops.talking_attention(q, 0, k_pages, v_pages, t([n - 1], torch.int32), t([0], torch.int32),
                                  t([[0, 1, 2, 3]], torch.int32), heads, 1, dim, window, 1.0, None, None, None, 1 if seen else 2)
        assert (f64(o)[0, 0] > 0.99) == seen


# ---------------------------------------------------------------- time mixing
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("seqs, width", [(1, 70), (5, 256), (9, 300)])
def test_single_tokens_are_mixed_and_kept_in_one_launch(ops, seqs, width, dtype):
    """The bits of the mixes and then the move, slots in any order, the others' rows left alone."""
    rng = np.random.default_rng(seqs)
    slots = t(rng.permutation(seqs + 2)[:seqs], torch.int32)
    kept = t(rng.normal(size=(seqs + 2, width)))
    x, mu = t(rng.normal(size=(seqs, width))), t(rng.uniform(size=(5, width)))
    seq, cu = t(np.arange(seqs), torch.int32), t(np.arange(seqs + 1), torch.int32)
    apart, together = kept.clone(), kept.clone()
    want = ops.shift_mix(x, apart, mu, seq, cu, slots, dtype)
    ops.shift_keep(apart, x, cu, slots)
    assert torch.equal(ops.shift_mix(x, together, mu, seq, cu, slots, dtype, keep=True), want)
    assert torch.equal(together, apart)


@pytest.mark.parametrize("columns", [True, False])
@pytest.mark.parametrize("heads, dim", [(3, 12), (2, 40), (1, 70), (1, 130)])
def test_time_mixing_through_every_cut(ops, heads, dim, columns):
    rng = np.random.default_rng(5)
    width, eps, rank = 30, 1e-5, 5
    hw = heads * dim
    m = {"heads": heads, "dim": dim}
    w = {x: rng.standard_normal((hw, width)) / 3 for x in "rkvg"}
    w.update({"mu." + s: rng.random(width) for s in "rkvgw"})
    w.update({"w1": rng.standard_normal((rank, width)) / 3, "w2": rng.standard_normal((hw, rank)), "w0": rng.standard_normal(hw) - 1,
              "u": rng.standard_normal((heads, dim)), "norm": 1 + 0.1 * rng.standard_normal(hw), "o": np.eye(hw)})
    lengths = [43, 43]
    h = [rng.standard_normal((n, width)) for n in lengths]
    steps = Steps(lengths, [2, 0], rng)
    state = guarded(torch.zeros((3, heads, dim, dim), device=DEV))
    kept = guarded(torch.zeros((3, width), device=DEV))
    mu = t(np.stack([w["mu." + s] for s in "rkvgw"]))
    states = [{}, {}]
    for counts in CUTS[0]:
        st = steps.step(counts)
        x = np.stack([h[s][p] for s, p in st["rows"]])
        x32 = t(x)
        mixes = ops.shift_mix(x32, kept, mu, st["tok_seq"], st["cu"], st["slots"], torch.float32)
        ops.shift_keep(kept, x32, st["cu"], st["slots"])
        mx = f64(mixes)
        r, k, v, g = (t(mx[i] @ w[s].T) for i, s in enumerate("rkvg"))
        z = t(np.tanh(mx[4] @ w["w1"].T) @ w["w2"].T)
        out = guarded(torch.zeros((len(x), hw + 2), device=DEV))
        ops.timemix_scan(out, 2, 0.7, r, k, v, g, z, t(w["w0"]), t(w["u"].reshape(-1)), t(w["norm"]), eps, state, st["cu"],
                         st["slots"], heads, dim, columns)
        want, at = [], 0
        for s in st["seqs"]:
            n = sum(1 for r_ in st["rows"] if r_[0] == s)
            want.append(P.time_mixer(x[at:at + n], w, "", m, eps, states[s]))
            at += n
        close(out[:, 2:], 0.7 * np.concatenate(want), 3e-5, f"time mixing, step {counts}")
    close(ops.tanh_rows(t(x), torch.float32), np.tanh(x), F32, "tanh")


# ---------------------------------------------------------------- the state-space mixer
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lengths, channels", [([1, 2, 3, 5, 505], 1536), ([600, 2, 1, 8], 1540), ([771], 1028)])
def test_convolution_of_four_taps_by_blocks_of_tokens(ops, lengths, channels, dtype):
    """The form of many tokens (eight a thread, four channels side by side) against a call a sequence and piece, which is
    below its first size: sequences that begin inside a block, shorter than the taps, a last block that is not full, and one that
    goes on where it stopped.  The sums are the same sums in the same order: the same bits."""
    rng = np.random.default_rng(channels)
    seqs, tokens = len(lengths), sum(lengths)
    assert ops.causal_conv_blocks(tokens, seqs, channels) and not ops.causal_conv_blocks(100, 1, channels)
    proj = t(rng.standard_normal((tokens, channels + 8)), dtype)
    w, bias = t(rng.standard_normal((channels, 4)) / 2), t(rng.standard_normal(channels))
    tails = t(rng.standard_normal((seqs + 1, 3, channels)))
    order = [int(x) for x in rng.permutation(seqs + 1)[:seqs]]
    cu = np.cumsum([0, *lengths])
    kept = tails.clone()
    got = ops.causal_conv_silu(proj, 4, channels, w, bias, kept, t(np.repeat(np.arange(seqs), lengths), torch.int32),
                               t(cu, torch.int32), t(order, torch.int32))
    for s in range(seqs):
        for at in range(cu[s], cu[s + 1], 100):
            end = min(at + 100, cu[s + 1])
            want = ops.causal_conv_silu(proj[at:end].contiguous(), 4, channels, w, bias, tails, t([0] * (end - at), torch.int32),
                                        t([0, end - at], torch.int32), t([order[s]], torch.int32))
            assert torch.equal(got[at:end], want), f"sequence {s}, tokens {at}..{end}"
    assert torch.equal(kept, tails)


def test_convolution_of_single_tokens_keeps_an_element_a_thread(ops):
    """Steps whose rows mostly take their tails go by blocks from four times as many results on."""
    blocks = lambda tokens, seqs, channels=6144: ops.causal_conv_blocks(tokens, seqs, channels)
    assert blocks(128, 1) and blocks(128, 64) and blocks(512, 512) and blocks(600, 301)
    assert not blocks(127, 1) and not blocks(128, 128) and not blocks(128, 65) and not blocks(256, 256) and not blocks(600, 600, 1536)


@pytest.mark.parametrize("columns", [True, False])
@pytest.mark.parametrize("heads, vdim, n, groups, taps, parts", [(4, 12, 10, 2, 3, 2), (2, 20, 40, 1, 1, 5), (3, 8, 70, 3, 5, 1),
                                                                 (1, 70, 130, 1, 2, 1)])
def test_state_space_mixer_through_every_cut(ops, heads, vdim, n, groups, taps, parts, columns):
    rng = np.random.default_rng(6)
    width, eps = 30, 1e-5
    inner = heads * vdim
    channels = inner + 2 * groups * n
    m = {"heads": heads, "vdim": vdim, "state": n, "groups": groups, "conv": taps, "norm_groups": parts}
    w = {"in": rng.standard_normal((inner + channels + heads, width)) / 3, "conv": rng.standard_normal((channels, taps)) / 2,
         "conv.b": rng.standard_normal(channels) / 3, "dt_bias": rng.standard_normal(heads), "A_log": rng.standard_normal(heads),
         "D": rng.standard_normal(heads), "norm": 1 + 0.1 * rng.standard_normal(inner), "o": np.eye(inner)}
    lengths = [43, 43]
    h = [rng.standard_normal((k, width)) for k in lengths]
    steps = Steps(lengths, [1, 2], rng)
    state = guarded(torch.zeros((3, heads, n, vdim), device=DEV))
    tails = guarded(torch.zeros((3, max(taps - 1, 1), channels), device=DEV))
    states = [{}, {}]
    for counts in CUTS[0]:
        st = steps.step(counts)
        x = np.stack([h[s][p] for s, p in st["rows"]])
        proj = t(x @ w["in"].T)
        xbc = ops.causal_conv_silu(proj, inner, channels, t(w["conv"]), t(w["conv.b"]), tails, st["tok_seq"], st["cu"], st["slots"])
        y = ops.ssd_scan(xbc, inner, inner + groups * n, proj, 0, inner + channels, t(w["dt_bias"]), t(w["A_log"]), t(w["D"]),
                         state, st["cu"], st["slots"], heads, groups, n, vdim, columns)
        got = ops.group_rms_norm(y, t(w["norm"]), eps, parts, torch.float32)
        want, at = [], 0
        for s in st["seqs"]:
            k = sum(1 for r in st["rows"] if r[0] == s)
            want.append(P.mamba2_mixer(x[at:at + k], w, "", m, eps, states[s]))
            at += k
        close(got, np.concatenate(want), 3e-5, f"state-space mixer, step {counts}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads, groups, n, vdim, lens", [(2, 1, 64, 32, (200,)), (3, 3, 12, 20, (64, 1, 130)), (2, 1, 128, 128, (65, 63)),
                                                          (4, 2, 100, 36, (2, 191, 128)), (2, 2, 4, 8, (129,))])
def test_state_space_walk_in_chunks(ops, dtype, heads, groups, n, vdim, lens):
    """States that are not zero, at slots in another order, lengths on and beside a chunk's edge, steps that hardly decay and such that
    forget all within a few tokens; against the recurrence in 64 bits, whose distance is no larger than the walk's, and against the walk."""
    rng = np.random.default_rng(heads * 17 + n)
    T, inner = sum(lens), heads * vdim
    channels, b_off, c_off = inner + 2 * groups * n + 4, inner + 4, inner + 4 + groups * n
    xbc, proj = t(rng.normal(size=(T, channels))), t(rng.normal(size=(T, 3 + inner + heads)), dtype)
    dt_bias, a_log, skip = t(rng.normal(size=heads) * 2), t(np.linspace(-6, 3, heads)), t(rng.normal(size=heads))
    slots = [2, 0, 3][:len(lens)]
    start = t(rng.normal(size=(4, heads, n, vdim)))
    x, p, want_state = f64(xbc), f64(proj), f64(start).copy()
    want = np.zeros((T, inner))
    cu = np.concatenate([[0], np.cumsum(lens)])
    for s, slot in enumerate(slots):
        for i in range(cu[s], cu[s + 1]):
            for h in range(heads):
                raw = p[i, 3 + inner + h] + f64(dt_bias)[h]
                dt = raw if raw > 20 else np.log1p(np.exp(raw))
                B, C = (x[i, o + h * groups // heads * n:][:n] for o in (b_off, c_off))
                xv, z = x[i, h * vdim:(h + 1) * vdim], p[i, 3 + h * vdim:3 + (h + 1) * vdim]
                S = want_state[slot, h]
                S[:] = np.exp(-np.exp(f64(a_log)[h]) * dt) * S + dt * np.outer(B, xv)
                want[i, h * vdim:(h + 1) * vdim] = (S.T @ C + f64(skip)[h] * xv) * z / (1 + np.exp(-z))
    args = (xbc, b_off, c_off, proj, 3, 3 + inner, dt_bias, a_log, skip)
    more = (t(cu, torch.int32), t(slots, torch.int32), heads, groups, n, vdim)
    assert ops.ssd_chunks_fit(n, vdim, channels, (b_off, c_off))
    chunked, walked = guarded(start.clone()), guarded(start.clone())
    got, walk = ops.ssd_scan_chunked(*args, chunked, *more, max(lens)), ops.ssd_scan(*args, walked, *more)
    close(got, want, 1e-5, "outputs")
    close(chunked, want_state, 1e-5, "state")
    assert np.array_equal(f64(chunked[1]), f64(start[1]))     # a slot that no sequence of the step has
    close(got, f64(walk), 1e-5, "chunks against the walk")
    error = lambda y: np.linalg.norm(f64(y) - want) / np.linalg.norm(want)
    assert error(got) <= 1.5 * error(walk) + 1e-7


@pytest.mark.parametrize("lens", [(70,), (33, 1, 130)])
def test_state_space_chunks_of_decays_of_every_size(ops, lens):
    """Heads whose exponents are moderate on some tokens and beyond every sum of moderate ones on the others (A = e^25, e^30, e^35), and heads
    that forget all with every token (A past float32, and infinite): the bounds of the test above."""
    rng = np.random.default_rng(len(lens))
    a_logs, n, vdim, T = [25.0, 30.0, 35.0, 89.0, np.inf], 8, 12, sum(lens)
    heads, groups = len(a_logs), 1
    inner = heads * vdim
    channels, b_off, c_off = inner + 2 * n, inner, inner + n
    raw = np.stack([(rng.normal(size=T) - (a * (rng.random(T) < 0.8) if a < 80 else 0)) for a in a_logs], 1)
    xbc, proj = t(rng.normal(size=(T, channels))), t(np.concatenate([rng.normal(size=(T, inner)), raw], 1))
    a_log, start = t(a_logs), t(rng.normal(size=(4, heads, n, vdim)))
    slots, cu = [2, 0, 3][:len(lens)], np.concatenate([[0], np.cumsum(lens)])
    x, p, want_state, want = f64(xbc), f64(proj), f64(start).copy(), np.zeros((T, inner))
    with np.errstate(over="ignore"):
        A = np.exp(np.array(a_logs, dtype=np.float32)).astype(np.float64)          # (float32's range: past it a decay is 0)
    for s, slot in enumerate(slots):
        for i in range(cu[s], cu[s + 1]):
            for h in range(heads):
                dt, xv, z = np.log1p(np.exp(p[i, inner + h])), x[i, h * vdim:(h + 1) * vdim], p[i, h * vdim:(h + 1) * vdim]
                S = want_state[slot, h]
                S[:] = np.exp(-A[h] * dt) * S + dt * np.outer(x[i, b_off:b_off + n], xv)
                want[i, h * vdim:(h + 1) * vdim] = S.T @ x[i, c_off:] * z / (1 + np.exp(-z))
    args = (xbc, b_off, c_off, proj, 0, inner, None, a_log, None)
    more = (t(cu, torch.int32), t(slots, torch.int32), heads, groups, n, vdim)
    chunked, walked = guarded(start.clone()), guarded(start.clone())
    got, walk = ops.ssd_scan_chunked(*args, chunked, *more, max(lens)), ops.ssd_scan(*args, walked, *more)
    for h in range(heads):                                    # (a head by itself: steps differ by many powers of ten)
        of = slice(h * vdim, (h + 1) * vdim)
        close(got[:, of], want[:, of], 1e-5, f"outputs, A = e^{a_logs[h]}")
        close(chunked[:, h], want_state[:, h], 1e-5, f"state, A = e^{a_logs[h]}")
        close(got[:, of], f64(walk[:, of]), 1e-5, f"chunks against the walk, A = e^{a_logs[h]}")


@pytest.mark.parametrize("n, vdim, bias", [(128, 64, 1.0), (128, 32, -3.0), (64, 64, -3.0)])
def test_state_space_chunks_err_no_more_than_the_walk(ops, n, vdim, bias):
    """Distance from 64 bits (2-norm), for steps that forget fast and slowly: of the outputs and the states that of the walk, up to a tenth
    for what differs by chance (a sum over 128 rows in one chain has twice as much)."""
    rng = np.random.default_rng(n + vdim)
    heads, groups, T = 8, 2, 200
    inner, gn = heads * vdim, groups * n
    xbc, proj = t(rng.normal(size=(T, inner + 2 * gn))), t(rng.normal(size=(T, inner + heads)), torch.bfloat16)
    dt_bias, a_log, start = t(rng.normal(size=heads) + bias), t(np.log(rng.uniform(1, 16, heads))), t(rng.normal(size=(1, heads, n, vdim)))
    x, p = f64(xbc), f64(proj)
    dt = np.log1p(np.exp(p[:, inner:] + f64(dt_bias)))
    B, C = (np.repeat(x[:, o:o + gn].reshape(T, groups, n), heads // groups, 1) for o in (inner, inner + gn))
    decay, xv, S, want = np.exp(-np.exp(f64(a_log)) * dt), x[:, :inner].reshape(T, heads, vdim), f64(start)[0].copy(), []
    for i in range(T):
        S = decay[i][:, None, None] * S + (dt[i][:, None] * B[i])[:, :, None] * xv[i][:, None, :]
        want.append(np.einsum("hn,hnv->hv", C[i], S).reshape(-1) * p[i, :inner] / (1 + np.exp(-p[i, :inner])))
    args = (xbc, inner, inner + gn, proj, 0, inner, dt_bias, a_log, None)
    more = (t([0, T], torch.int32), t([0], torch.int32), heads, groups, n, vdim)
    chunked, walked = guarded(start.clone()), guarded(start.clone())
    got, walk = ops.ssd_scan_chunked(*args, chunked, *more, T), ops.ssd_scan(*args, walked, *more)
    error = lambda y, w: np.linalg.norm(f64(y) - w) / np.linalg.norm(w)
    assert error(got, np.stack(want)) <= 1.1 * error(walk, np.stack(want)) and error(chunked[0], S) <= 1.1 * error(walked[0], S)


def test_state_space_chunks_leave_a_state_off_their_loads_boundary_to_the_walk(ops):
    whole = guarded(torch.zeros(1 + 2 * 8 * 12, device=DEV))
    fit = lambda state: ops.ssd_chunks_fit(8, 12, 40, (24, 32), state)
    assert fit(whole[:-1].view(1, 2, 8, 12)) and not fit(whole[1:].view(1, 2, 8, 12))


def test_state_space_chunks_where_the_walk_waits_for_its_tokens(ops, monkeypatch):
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    pay = ops.ssd_chunks_pay
    assert pay([2048], 32, 128, 128) and pay([512], 32, 128, 128) and pay([300, 1800, 1500, 1300], 32, 128, 128) and pay([500] * 8, 32, 64, 64)
    assert not pay([256], 32, 128, 128) and not pay([500] * 8, 32, 128, 128) and not pay([1000] * 32, 32, 128, 128)
    assert not pay([1] * 40 + [200], 32, 128, 128) and not pay([128] * 32, 32, 64, 64) and not pay([64], 32, 64, 64)


# ---------------------------------------------------------------- the products per head through the library
@pytest.mark.parametrize("heads, k, n, extra, gated", [(3, 24, 40, 6, False), (5, 40, 12, 0, True), (2, 16, 16, 10, True)])
def test_batched_head_products_are_the_products_per_head(ops, heads, k, n, extra, gated):
    """bfloat16 rows with the heads somewhere inside a wider row, columns in front and behind: the batched product with the
    copied elements and a gate a head against the sums written out in float64, and beside the kernel that does it alone."""
    rng = np.random.default_rng(heads)
    tokens, x_off, x_head = 37, 5, k + extra + 3
    stride = x_off + heads * x_head + heads + 4
    x = t(rng.standard_normal((tokens, stride)), torch.bfloat16)
    w = t(rng.standard_normal((heads, k, n)) / 4, torch.bfloat16)
    g_off = x_off + heads * x_head + 2
    got = ops.head_products_batched(x, x_off, x_head, w, heads, k, n, extra=extra, gates=x if gated else None, g_off=g_off)
    alone = ops.head_products(x, x_off, x_head, w, heads, k, n, extra=extra, gates=x if gated else None, g_off=g_off)
    xs, ws = f64(x), f64(w)
    want = np.zeros((tokens, heads, n + extra))
    for h in range(heads):
        rows = xs[:, x_off + h * x_head: x_off + (h + 1) * x_head]
        want[:, h, :n] = rows[:, :k] @ ws[h]
        want[:, h, n:] = rows[:, k:k + extra]
        if gated:
            want[:, h] *= (1 / (1 + np.exp(-xs[:, g_off + h])))[:, None]
    want = want.reshape(tokens, -1)
    assert got.dtype == torch.bfloat16 and tuple(got.shape) == want.shape
    close(got, want, 1.2e-2, "batched products per head")          # two roundings to bfloat16 with a gate, one without
    close(alone, want, 6e-3, "products per head")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens, k, n, extra", [(1, 128, 8, 0), (17, 132, 136, 5), (16, 516, 128, 0), (3, 1020, 8, 2), (33, 160, 264, 64)])
def test_products_per_head_with_bfloat16_matrices(ops, dtype, tokens, k, n, extra):
    """Tiles of 16 tokens and 128 columns, slices of the rows that leave wavefronts without one, and their remainders, in float32."""
    rng = np.random.default_rng(k)
    heads, x_off = 2, 3
    x = t(rng.standard_normal((tokens, x_off + heads * (k + extra) + heads)), dtype)
    w = t(rng.standard_normal((heads, k, n)), torch.bfloat16)
    gated = k > 140
    got = ops.head_products(x, x_off, k + extra, w, heads, k, n, extra=extra, gates=x if gated else None, g_off=x_off + heads * (k + extra),
                            scale=0.5, out_dtype=torch.float32)
    xs = f64(x)[:, x_off:x_off + heads * (k + extra)].reshape(tokens, heads, k + extra)
    want = 0.5 * np.concatenate([np.einsum("thk,hkn->thn", xs[:, :, :k], f64(w)), xs[:, :, k:]], 2)
    if gated:
        want *= (1 / (1 + np.exp(-f64(x)[:, -heads:])))[:, :, None]
    close(got, want.reshape(tokens, -1), F32, "products per head")


def test_products_per_head_err_no_more_than_a_column_at_a_time(ops):
    """Heads of 128 x 512, 2-norm against 64 bits: 5.3e-8 with a thread a column, whose slices of the rows are 32 long; eight slices of sixteen
    rows added in order have 5.5e-8, two by two 4.9e-8 (each for these sizes, whatever the numbers, to about a hundredth)."""
    rng = np.random.default_rng(3)
    tokens, heads, k, n = 8, 2 if EMULATED else 32, 128, 512
    x, w = t(rng.standard_normal((tokens, heads * k)), torch.bfloat16), t(rng.standard_normal((heads, k, n)), torch.bfloat16)
    got = f64(ops.head_products(x, 0, k, w, heads, k, n, out_dtype=torch.float32))
    want = np.einsum("thk,hkn->thn", f64(x).reshape(tokens, heads, k), f64(w)).reshape(tokens, -1)
    error = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert error <= 5.2e-8, error


# ---------------------------------------------------------------- the latent attention on the matrix cores
@pytest.mark.parametrize("heads", [3, 20])
def test_latent_attention_on_the_matrix_cores_is_the_general_kernel(ops, heads):
    """bfloat16, key rows of 160 and value rows of 128: tokens at the start of a sequence, at a page's border and inside a
    page, of two sequences whose pages lie in shuffled order, with sinks; against the general kernel on the same pages."""
    rng = np.random.default_rng(11)
    dk, rank, pages = 160, 128, 12
    k_pages = guarded((torch.randn((pages, 1, PAGE, dk), device=DEV) * 0.5).to(torch.bfloat16))
    v_pages = guarded(k_pages[:, :, :, :rank].transpose(2, 3).contiguous())
    table = t([[5, 2, 9, 0], [7, 1, 3, 11]], torch.int32)
    tok_seq, tok_pos = t([0, 0, 0, 1, 1, 1, 1], torch.int32), t([0, 31, 32, 5, 63, 64, 100], torch.int32)
    q = guarded((torch.randn((7, heads * dk), device=DEV) * 0.5).to(torch.bfloat16))
    sinks = t(rng.standard_normal(heads))
    for sink in (sinks, None):
        want = ops.attention(q, k_pages, v_pages, tok_pos, tok_seq, table, heads, 1, dk, None, 0.11, sinks=sink)
        got = ops.latent_attention_mfma(q, k_pages, v_pages, tok_pos, tok_seq, table, heads, 0.11, sink)
        close(got, f64(want), 1.2e-2, "matrix cores against the general kernel")
        for bound in (101, 128, 1024):                    # chunks of one page, of one page with more room than pages, of eight
            got = ops.latent_attention_mfma(q, k_pages, v_pages, tok_pos, tok_seq, table, heads, 0.11, sink, bound)
            close(got, f64(want), 1.2e-2, f"in chunks, sequences of up to {bound}")


@pytest.mark.parametrize("heads, dk, rank", [(3, 160, 128), (20, 288, 256), (16, 576, 512)])
def test_latent_attention_of_single_tokens_in_quarters(ops, heads, dk, rank, monkeypatch):
    """A workgroup's wavefronts on a quarter of the key rows and of the value rows each: whole walks, chunks of a page and of several, more
    chunks than pages; against a wavefront that walks all of them, up to the order of float32 sums and their rounding to bfloat16."""
    pages, ends = 9, [0, 31, 32, 100, 69]
    k_pages = guarded((torch.randn((pages, 1, PAGE, dk), device=DEV) * 0.3).to(torch.bfloat16))
    v_pages = guarded(k_pages[:, :, :, :rank].transpose(2, 3).contiguous())
    table = t([[8, -1, -1, -1], [0, -1, -1, -1], [3, 1, -1, -1], [7, 5, 2, 4], [6, 3, 0, -1]], torch.int32)
    pos, seq = t(ends, torch.int32), t(range(5), torch.int32)
    q = guarded((torch.randn((5, heads * dk), device=DEV) * 0.3).to(torch.bfloat16))
    sinks = t(np.linspace(-1, 1, heads))
    want = f64(ops.latent_attention_mfma(q, k_pages, v_pages, pos, seq, table, heads, 0.11, sinks))
    for fill in (1, 5 * -(-heads // 16) * 2, 512):
        monkeypatch.setattr(ops, "LATENT_DECODE_FILL", fill)
        for bound in (101, 2048):
            got = ops.latent_attention_mfma(q, k_pages, v_pages, pos, seq, table, heads, 0.11, sinks, bound)
            close(got, want, 8e-3, f"{fill} workgroups, sequences of up to {bound}")


@pytest.mark.parametrize("heads, dk, rank", [(16, 160, 128), (16, 576, 512)])
def test_latent_attention_of_single_tokens_keeps_its_weights_whole(ops, heads, dk, rank):
    """2-norm against 64 bits: what a rounding to bfloat16 of the result has, 2^-9 / sqrt(3) of a power of two that is 0.7 of the value on average,
    1.65e-3.  Weights rounded to bfloat16 as well make it 1.9e-3 to 2.1e-3."""
    torch.manual_seed(dk)
    pages, ends = 12, [95, 200, 70]
    k_pages = guarded(torch.randn((pages, 1, PAGE, dk), device=DEV).to(torch.bfloat16))
    v_pages = guarded(k_pages[:, :, :, :rank].transpose(2, 3).contiguous())
    table = t([[0, 1, 2, 0, 0, 0, 0], [3, 4, 5, 6, 7, 8, 9], [10, 11, 2, 0, 0, 0, 0]], torch.int32)
    q = guarded(torch.randn((3, heads * dk), device=DEV).to(torch.bfloat16))
    scale, want = 1.2 * dk ** -0.5, []
    for b, end in enumerate(ends):
        keys = f64(k_pages[table[b].long()]).reshape(-1, dk)[:end + 1]
        s = np.exp(f64(q[b]).reshape(heads, dk) @ keys.T * scale)
        want.append((s @ keys[:, :rank] / s.sum(1, keepdims=True)).reshape(-1))
    got = f64(ops.latent_attention_mfma(q, k_pages, v_pages, t(ends, torch.int32), t(range(3), torch.int32), table, heads, scale, None, 256))
    error = np.linalg.norm(got - np.stack(want)) / np.linalg.norm(want)
    assert error <= 1.75e-3, error


@pytest.mark.parametrize("heads, dk, rank", [(3, 160, 128), (20, 288, 256), (40, 160, 128), (130, 160, 128), (16, 576, 512)])
def test_latent_attention_with_shared_pages_gives_the_same_bits(ops, heads, dk, rank, monkeypatch):
    """Eight (token, tile of heads) pairs a workgroup: workgroups whose tokens are of two and three sequences, of more tiles than
    pairs, a last one that is not full; against a wavefront that fetches its pages itself."""
    rng = np.random.default_rng(heads + dk)
    new, lens = [9, 1, 2, 5], [40, 1, 34, 5]
    pages = sum(-(-n // PAGE) for n in lens) + 2
    k_pages = guarded((torch.randn((pages, 1, PAGE, dk), device=DEV) * 0.5).to(torch.bfloat16))
    v_pages = guarded(k_pages[:, :, :, :rank].transpose(2, 3).contiguous())
    order = iter(rng.permutation(pages))
    table = t([[next(order) if i < -(-n // PAGE) else -1 for i in range(2)] for n in lens], torch.int32)
    tok_seq = t([s for s, n in enumerate(new) for _ in range(n)], torch.int32)
    tok_pos = t([lens[s] - n + i for s, n in enumerate(new) for i in range(n)], torch.int32)
    q = guarded((torch.randn((sum(new), heads * dk), device=DEV) * 0.5).to(torch.bfloat16))
    sinks = t(rng.standard_normal(heads))
    got = []
    for least in (1 << 30, 0):
        monkeypatch.setattr(ops, "LATENT_SHARED_FROM", least)
        got.append(f64(ops.latent_attention_mfma(q, k_pages, v_pages, tok_pos, tok_seq, table, heads, 0.11, sinks)))
    assert np.isfinite(got[0]).all() and np.array_equal(*got)


@pytest.mark.parametrize("heads, dk, rank", [(20, 160, 128), (130, 160, 128), (40, 288, 256), (16, 576, 512)])
def test_latent_attention_with_shared_pages_a_sequence_a_workgroup(ops, heads, dk, rank, monkeypatch):
    """The sequences' bounds given: workgroups of one sequence alone, more sequences than a wavefront has lanes, single tokens among
    them; the same bits as a wavefront that fetches its pages itself."""
    rng = np.random.default_rng(heads)
    new = [1] * 30 + [9, 2, 1, 5] + [1] * 33 + [3] if dk == 160 and heads == 20 else [9, 1, 1, 5]
    before = [int(n) for n in rng.integers(0, 60, len(new))]
    width = -(-max(a + n for a, n in zip(before, new)) // PAGE)
    pages = sum(-(-(a + n) // PAGE) for a, n in zip(before, new)) + 2
    k_pages = guarded((torch.randn((pages, 1, PAGE, dk), device=DEV) * 0.5).to(torch.bfloat16))
    v_pages = guarded(k_pages[:, :, :, :rank].transpose(2, 3).contiguous())
    order = iter(rng.permutation(pages))
    table = t([[next(order) if i < -(-(a + n) // PAGE) else -1 for i in range(width)] for a, n in zip(before, new)], torch.int32)
    tok_seq = t([s for s, n in enumerate(new) for _ in range(n)], torch.int32)
    tok_pos = t([before[s] + i for s, n in enumerate(new) for i in range(n)], torch.int32)
    q = guarded((torch.randn((sum(new), heads * dk), device=DEV) * 0.5).to(torch.bfloat16))
    cu, sinks, got = t(np.concatenate([[0], np.cumsum(new)]), torch.int32), t(rng.standard_normal(heads)), []
    for keys in (1, 1 << 30):                                 # shared from one key on, and apart
        monkeypatch.setattr(ops, "LATENT_SHARED", {dk: (1 << 20, keys)})
        assert (ops.latent_attention_shared(new, before, heads, dk) > 0) == (keys == 1)
        got.append(f64(ops.latent_attention_mfma(q, k_pages, v_pages, tok_pos, tok_seq, table, heads, 0.11, sinks, new_counts=new,
                                                 starts=before, cu_seqlens=cu)))
    assert np.isfinite(got[0]).all() and np.array_equal(*got)


@pytest.mark.parametrize("order", [[3, 0, 2, 1, 4], [4, 3, 2, 1, 0]])
def test_latent_attention_with_shared_pages_takes_the_tokens_in_any_order(ops, order, monkeypatch):
    """The tokens of a sequence need not come by their positions: every one sees its own keys, the same bits as by position."""
    torch.manual_seed(1)
    heads, dk, rank, before, n = 16, 160, 128, 61, 5
    pages = -(-(before + n) // PAGE)
    k_pages = guarded((torch.randn((pages, 1, PAGE, dk), device=DEV) * 0.5).to(torch.bfloat16))
    v_pages = guarded(k_pages[:, :, :, :rank].transpose(2, 3).contiguous())
    table, seq = t([list(range(pages))], torch.int32), t([0] * n, torch.int32)
    q = (torch.randn((n, heads * dk), device=DEV) * 0.5).to(torch.bfloat16)
    monkeypatch.setattr(ops, "LATENT_SHARED_FROM", 0)
    want = f64(ops.latent_attention_mfma(guarded(q), k_pages, v_pages, t(before + np.arange(n), torch.int32), seq, table, heads, 0.11, None))
    got = f64(ops.latent_attention_mfma(guarded(q[order].contiguous()), k_pages, v_pages, t(before + np.array(order), torch.int32), seq, table,
                                        heads, 0.11, None))
    assert np.isfinite(want).all() and np.array_equal(got, want[order])


def test_latent_attention_shares_pages_where_that_is_less_to_wait_for(ops, monkeypatch):
    """Small prompts fetch for themselves; long ones and steps that fill the machine share, in workgroups of one sequence each."""
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    plan = ops.latent_attention_shared
    assert plan([2048], [0], 32, 576) == 512 and plan([16], [2000], 32, 576) == 4 and plan([20] * 32, [0] * 32, 32, 576) == 160
    assert plan([2048] + [1] * 64, [0] + [4000] * 64, 32, 576) == 512 + 64
    assert plan([128], [0], 32, 576) == plan([17] * 10, [0] * 10, 32, 576) == plan([512], [8000], 32, 288) == plan([300], [0], 20, 160) == 0
    assert plan([2048], [0], 32, 288) == 512 and plan([2048] + [1] * 64, [0] + [2000] * 64, 32, 288) == 0 and plan([16], [8000], 32, 160) == 4


@pytest.mark.parametrize("heads, kv_heads, dim, window", [(8, 2, 32, 40), (16, 16, 32, None), (8, 1, 64, 33), (32, 8, 128, 40), (8, 2, 64, None)])
def test_talking_attention_on_the_matrix_cores_is_the_general_kernel(ops, heads, kv_heads, dim, window):
    """bfloat16: two sequences whose pages lie in shuffled order, one that goes on from 37 cached tokens with 21 new ones
    (two tiles, the second partial) and one that starts with 50; with the distance bias and the mixing matrix, and without;
    against the general kernels on the same pages."""
    rng = np.random.default_rng(12)
    pages = 10
    k_pages = guarded((torch.randn((pages, kv_heads, PAGE, dim), device=DEV) * 0.6).to(torch.bfloat16))
    v_pages = guarded((torch.randn((pages, kv_heads, dim, PAGE), device=DEV) * 0.6).to(torch.bfloat16))
    table = t([[5, 2, 9], [7, 1, 3]], torch.int32)
    counts, starts = [21, 50], [37, 0]
    tok_seq = t([0] * 21 + [1] * 50, torch.int32)
    tok_pos = t(list(range(37, 58)) + list(range(50)), torch.int32)
    cu = t([0, 21, 71], torch.int32)
    proj = guarded((torch.randn((71, heads * dim + 16), device=DEV) * 0.6).to(torch.bfloat16))
    r1, r2 = t(rng.random(heads)), t(rng.random(heads) * 3)
    talk = t(np.eye(heads) + 0.3 * rng.standard_normal((heads, heads)))
    for a, b, c in ((r1, r2, talk), (None, None, None)):
        want = ops.talking_attention(proj, 8, k_pages, v_pages, tok_pos, tok_seq, table, heads, kv_heads, dim, window, 0.2, a, b, c)
        got = ops.talking_attention_mfma(proj, 8, k_pages, v_pages, tok_pos, cu, counts, table, heads, kv_heads, dim, window, 0.2,
                                         a, b, c)
        close(got, f64(want), 1.5e-2, "matrix cores against the general kernels")


@pytest.mark.parametrize("heads, kv_heads, dim, window", [(8, 2, 32, 40), (16, 16, 32, None), (4, 2, 128, 33), (16, 1, 64, 32), (24, 12, 128, 1),
                                                          (64, 8, 32, None)])
def test_single_tokens_of_talking_heads_are_the_general_kernel(ops, heads, kv_heads, dim, window, monkeypatch):
    """bfloat16: sequences that end at the first and last key of a page, pages behind the window given back (-1 in the table), bounds on
    the length above the real one; a page a workgroup, several and all of them; with the distance bias and the mixing matrix and
    without; against the general kernels on the same pages in float32."""
    rng = np.random.default_rng(heads)
    pages, ends = 12, [0, 31, 32, 95, 65]
    k_pages = guarded((torch.randn((pages, kv_heads, PAGE, dim), device=DEV) * 0.6).to(torch.bfloat16))
    v_pages = guarded((torch.randn((pages, kv_heads, dim, PAGE), device=DEV) * 0.6).to(torch.bfloat16))
    table = np.full((5, 4), -1, dtype=np.int32)
    free = iter(rng.permutation(pages))
    for b, end in enumerate(ends):
        for page in range(max(0, end - window + 1) // 32 if window else 0, end // 32 + 1):
            table[b, page] = next(free)
    table, pos, seq = t(table, torch.int32), t(ends, torch.int32), t(range(5), torch.int32)
    proj = guarded((torch.randn((5, heads * dim + 16), device=DEV) * 0.6).to(torch.bfloat16))
    r1, r2 = t(rng.random(heads)), t(rng.random(heads) * 3)
    talk = t(np.eye(heads) + 0.3 * rng.standard_normal((heads, heads)))
    assert ops.talking_decode_fits(torch.bfloat16, 5, 128, window, heads, kv_heads, dim, PAGE)
    for fill, longest in ((512, 128), (5 * -(-kv_heads * dim // 1024) * 2, 96), (1, 4096)):
        monkeypatch.setattr(ops, "TALKING_DECODE_FILL", fill)
        for a, b, c in ((r1, r2, talk), (None, None, None)):
            want = [ops.talking_attention(proj[i:i + 1].float(), 8, k_pages.float(), v_pages.float(), pos[i:i + 1], seq[i:i + 1], table,
                                          heads, kv_heads, dim, window, 0.2, a, b, c) for i in range(5)] if heads * dim <= 3072 else \
                   [ops.talking_attention(proj[i:i + 1], 8, k_pages, v_pages, pos[i:i + 1], seq[i:i + 1], table, heads, kv_heads, dim, window,
                                          0.2, a, b, c, 2) for i in range(5)]
            got = ops.talking_decode(proj, 8, k_pages, v_pages, pos, seq, table, heads, kv_heads, dim, window, 0.2, a, b, c, longest)
            close(got, np.concatenate([f64(w) for w in want]), F32, f"{fill} workgroups")


@pytest.mark.parametrize("fill", [1, 1 << 20])
def test_single_tokens_of_talking_heads_in_a_bounded_workspace(ops, fill, monkeypatch):
    """What a step keeps between its launches is bounded however many tokens and keys it has; a token, two and several a pair of launches,
    whole and in shares of the pages: the same bits as all tokens in one."""
    for tokens, pages, heads in ((64, 512, 32), (512, 64, 64), (1, 4, 8), (40, 8000, 32)):
        assert ops.talking_decode_piece(tokens, pages, heads) * pages * heads * 34 * 4 <= max(1 << 26, pages * heads * 136)
    assert ops.talking_decode_piece(64, 32, 32) == 64 and ops.talking_decode_fits(torch.bfloat16, 64, 65536, None, 32, 8, 128, PAGE)
    monkeypatch.setattr(ops, "TALKING_DECODE_FILL", fill)
    heads, kv_heads, dim, n = 8, 4, 32, 5
    k_pages, v_pages = (guarded((torch.randn(shape, device=DEV) * 0.6).to(torch.bfloat16)) for shape in
                        ((12, kv_heads, PAGE, dim), (12, kv_heads, dim, PAGE)))
    table, pos, seq = t(np.arange(15).reshape(5, 3) % 12, torch.int32), t([0, 31, 32, 95, 65], torch.int32), t(range(n), torch.int32)
    proj = guarded((torch.randn((n, heads * dim + 16), device=DEV) * 0.6).to(torch.bfloat16))
    args = (heads, kv_heads, dim, None, 0.2, t(np.arange(heads) / 9.0), t(np.arange(heads) / 4.0), t(np.eye(heads) + 0.1), 96)
    whole = f64(ops.talking_decode(proj, 8, k_pages, v_pages, pos, seq, table, *args))
    for piece in (1, 2, 3):
        monkeypatch.setattr(ops, "TALKING_DECODE_SCORES", piece * 3 * heads * 136)
        assert np.array_equal(f64(ops.talking_decode(proj, 8, k_pages, v_pages, pos, seq, table, *args)), whole), f"{piece} tokens at a time"


@pytest.mark.parametrize("dim, window, table", [(32, 40, True), (64, 45, False), (128, None, False)])
def test_talking_attention_whole_and_in_shares(ops, dim, window, table, monkeypatch):
    """Tiles that are walked whole, whose result is bfloat16 at once, and in two, three and four shares of their pages, whose float32 sums
    are added first, some of them without a page; the bias from the table of distances and as a logarithm a score.  Each against the
    general kernel, and the shares against the whole: a sum of fewer than 128 weighted values (their magnitudes' sum is under 30) in another
    order, then a rounding to bfloat16."""
    torch.manual_seed(dim)
    rng = np.random.default_rng(dim)
    heads, kv_heads, counts, starts, lens = 8, 2, [33, 70], [21, 0], [54, 70]
    k_pages = guarded((torch.randn((10, kv_heads, PAGE, dim), device=DEV) * 0.6).to(torch.bfloat16))
    v_pages = guarded((torch.randn((10, kv_heads, dim, PAGE), device=DEV) * 0.6).to(torch.bfloat16))
    pages = t([[5, 2, 9], [7, 1, 3]], torch.int32)
    tok_seq = t([0] * 33 + [1] * 70, torch.int32)
    tok_pos = t(list(range(21, 54)) + list(range(70)), torch.int32)
    cu = t([0, 33, 103], torch.int32)
    proj = guarded((torch.randn((103, heads * dim), device=DEV) * 0.6).to(torch.bfloat16))
    r1, r2 = t(rng.random(heads)), t(rng.random(heads) * 3)
    talk = t(np.eye(heads) + 0.3 * rng.standard_normal((heads, heads)))
    want = f64(ops.talking_attention(proj, 0, k_pages, v_pages, tok_pos, tok_seq, pages, heads, kv_heads, dim, window, 0.2, r1, r2, talk))
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    monkeypatch.setattr(ops, "TALKING_TABLE_WINDOW", 16384 if table else 0)
    whole = None
    for shares in (1, 2, 3, 4):
        monkeypatch.setattr(ops, "TALKING_MAX_SHARES", shares)
        for longest in (max(lens), None):
            assert ops.talking_attention_mfma_shares(8, longest, window) == (min(shares, 3) if longest and window is None else
                                                                            min(shares, 2) if longest else shares)
            got = ops.talking_attention_mfma(proj, 0, k_pages, v_pages, tok_pos, cu, counts, pages, heads, kv_heads, dim, window, 0.2,
                                             r1, r2, talk, longest)
            close(got, want, 1.5e-2, f"{shares} shares against the general kernel")
            got = f64(got)
            whole = got if whole is None else whole
            assert (np.abs(got - whole) <= 2.0 ** -7 * np.abs(whole) + 128 * 2.0 ** -24 * 30).all(), f"{shares} shares against one"


def test_talking_attention_cuts_no_page_between_shares(ops, monkeypatch):
    """As many shares as leave no compute unit idle, none of them without a page: prompts of a page or two are walked whole or in two."""
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    shares = ops.talking_attention_mfma_shares
    assert [shares(1, n, 1024) for n in (16, 32, 33, 100, 2016)] == [1, 1, 2, 4, 4]
    assert shares(64, 17, 1024) == 1 and shares(128, 2048, 1024) == 2 and shares(128, 2048, None) == 2 and shares(129, 2064, 1024) == 1
    assert shares(1, 5000, 16) == 1 and shares(1, 5000, 17) == 2 and shares(1, None, 1024) == 4


# ---------------------------------------------------------------- the walks over states of 65 to 128 rows
@pytest.mark.parametrize("kind", ["ssd", "timemix", "gla"])
def test_walks_take_a_state_that_starts_anywhere(ops, kind):
    """A state that is a part of a larger buffer, four bytes behind the boundary of 16-byte loads: the same bits, and nothing beside it
    is touched."""
    rng = np.random.default_rng(5)
    heads, n, T = 2, 68, 3
    start = rng.standard_normal(heads * n * n)
    cu, slots = t([0, 1, 2, 3], torch.int32), t([0, 0, 0], torch.int32)[:1]
    row = rng.standard_normal((T, 4 * heads * n))
    zero = t(np.zeros(heads * n))

    def run(offset):
        whole = guarded(torch.full((offset + heads * n * n + 3,), 7.0, device=DEV))
        state = whole[offset:offset + heads * n * n].view(1, heads, n, n)
        state.copy_(torch.tensor(start, dtype=torch.float32).view(1, heads, n, n))
        outs = []
        for k in range(T):                                    # (single tokens: four columns a lane)
            one, c1 = row[k:k + 1], t([0, 1], torch.int32)
            a, b, v, z = (one[:, i * heads * n:(i + 1) * heads * n] for i in range(4))
            if kind == "ssd":
                proj = t(np.concatenate([z, one[:, :heads]], 1))
                outs.append(ops.ssd_scan(t(np.concatenate([v, b, a], 1)), heads * n, 2 * heads * n, proj, 0, heads * n, None, t(np.zeros(heads)),
                                         None, state, c1, slots, heads, heads, n, n))
            elif kind == "timemix":
                o = guarded(torch.zeros((1, heads * n), device=DEV))
                ops.timemix_scan(o, 0, 1.0, t(a), t(b), t(v), t(z), t(z), zero, zero, t(np.ones(heads * n)), 1e-5, state, c1, slots, heads, n)
                outs.append(o)
            else:
                outs.append(ops.gla_scan(t(np.concatenate([a, b, v], 1)), 0, heads * n, 2 * heads * n, t(z), None, 2.0, 1.0, state, c1, slots,
                                         heads, n, n))
        assert (whole[:offset] == 7).all() and (whole[offset + heads * n * n:] == 7).all()
        return np.concatenate([f64(x) for x in outs]), f64(state)

    at, off = run(0), run(1)
    assert np.isfinite(at[0]).all() and np.array_equal(at[0], off[0]) and np.array_equal(at[1], off[1])


@pytest.mark.parametrize("kind", ["ssd", "timemix", "gla"])
@pytest.mark.parametrize("rows, cols, heads, many", [(65, 65, 2, False), (100, 33, 2, False), (128, 40, 1, False), (128, 128, 33, True)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_walks_in_tiles_of_four_rows(ops, kind, rows, cols, heads, many, dtype):
    """Sequences that end inside a block of eight tokens, at its end and past 64 and 128 tokens, whole against the sums in 64 bits and
    cut anywhere against whole (the same bits).  A sum runs over `rows` products and as many steps of the state as its decay
    lets through (under ten here): (rows / 4 + 5 + 2 x 10) roundings of half a unit, against the largest result."""
    if kind == "timemix":
        cols = rows
    lens = [150, 64, 17, 9, 1] if many or not EMULATED else [70, 8, 1]
    if many and EMULATED:
        pytest.skip("thousands of columns: minutes when emulated")
    if many:
        lens = lens * 2                                       # more columns than the wavefronts of one or two a lane
    rng = np.random.default_rng(rows + cols)
    total, slots = sum(lens), rng.permutation(len(lens))
    width, wv = heads * rows, heads * cols
    a, b = (rng.standard_normal((total, heads, rows)) for _ in range(2))           # read by the results, written into the state
    v = rng.standard_normal((total, heads, cols))
    rounded = lambda x: f64(t(x, dtype)) if kind != "ssd" else f64(t(x))
    a, b, v = rounded(a), rounded(b), rounded(v)
    s0 = f64(t(rng.standard_normal((len(lens), heads, rows, cols))))
    raw = f64(t(rng.standard_normal((total, heads)), dtype))
    z = f64(t(rng.standard_normal((total, heads, rows)) - (1 if kind == "timemix" else 0)))
    u = f64(t(rng.standard_normal((heads, rows))))
    if kind == "ssd":
        dt = np.logaddexp(0.0, raw)
        decay, b64 = np.exp(-dt)[..., None] * np.ones(rows), b * dt[..., None]
        gate = f64(t(rng.standard_normal((total, heads, cols)), dtype))
    elif kind == "timemix":
        decay, b64 = np.exp(-np.exp(z)), b
    else:
        decay, b64 = (1.0 / (1.0 + np.exp(-z))) ** 0.5, b
    want, at = np.zeros((total, heads, cols)), 0
    end = np.zeros_like(s0)
    for i, n in enumerate(lens):
        s = s0[slots[i]].copy()
        for k in range(at, at + n):
            kv = b64[k][:, :, None] * v[k][:, None, :]
            if kind == "timemix":
                want[k] = np.einsum("hrc,hr->hc", s + u[:, :, None] * kv, a[k])
                s = decay[k][:, :, None] * s + kv
            else:
                s = decay[k][:, :, None] * s + kv
                want[k] = np.einsum("hrc,hr->hc", s, a[k])
        end[slots[i]] = s
        at += n
    if kind == "ssd":
        want *= gate / (1.0 + np.exp(-gate))

    def run(pieces):
        """Every sequence's tokens in the given number of steps."""
        state = t(s0)
        got, done = np.zeros_like(want), [0] * len(lens)
        starts = np.concatenate([[0], np.cumsum(lens)])
        for p in range(pieces):
            take = [(i, starts[i] + done[i], starts[i] + (n * (p + 1)) // pieces) for i, n in enumerate(lens)]
            take = [(i, x, y) for i, x, y in take if y > x]
            rows_of = np.concatenate([np.arange(x, y) for _, x, y in take])
            for i, x, y in take:
                done[i] += y - x
            cu = t(np.concatenate([[0], np.cumsum([y - x for _, x, y in take])]), torch.int32)
            sl = t([slots[i] for i, _, _ in take], torch.int32)
            m = len(rows_of)
            if kind == "ssd":
                xbc = t(np.concatenate([v[rows_of].reshape(m, -1), b[rows_of].reshape(m, -1), a[rows_of].reshape(m, -1)], 1))
                proj = t(np.concatenate([gate[rows_of].reshape(m, -1), raw[rows_of]], 1), dtype)
                zero = t(np.zeros(heads))
                o = ops.ssd_scan(xbc, wv, wv + width, proj, 0, wv, zero, zero, None, state, cu, sl, heads, heads, rows, cols)
            elif kind == "timemix":
                out = guarded(torch.zeros((m, width), dtype=dtype, device=DEV))
                gates = t(np.full((m, width), 30.0), dtype)                        # silu(30) = 30
                r_, k_, v_ = (t(x[rows_of].reshape(m, -1), dtype) for x in (a, b, v))
                ops.timemix_scan(out, 0, 1.0, r_, k_, v_, gates, t(z[rows_of].reshape(m, -1)), t(np.zeros(width)), t(u.reshape(-1)),
                                 t(np.ones(width)), 0.0, state, cu, sl, heads, rows)
                o = out
            else:
                proj = t(np.concatenate([x[rows_of].reshape(m, -1) for x in (a, b, v)], 1), dtype)
                o = ops.gla_scan(proj, 0, width, 2 * width, t(z[rows_of].reshape(m, -1)), None, 2.0, 1.0, state, cu, sl, heads, rows, cols)
            got[rows_of] = f64(o).reshape(m, heads, cols)
        return got, f64(state)

    if kind == "timemix":
        want = want / np.sqrt((want * want).mean(-1, keepdims=True)) * 30.0
    whole, state = run(1)
    bound = (rows / 4 + 25) * 2.0 ** -24 * 4                  # (four: the largest result beside the largest term of its sum)
    assert np.abs(state - end).max() <= bound * np.abs(end).max()
    if kind == "timemix" and dtype == torch.bfloat16:
        bound = 2.0 ** -8                                     # the normed heads are written in bfloat16
    assert np.abs(whole - want).max() <= bound * np.abs(want).max()
    cut, cut_state = run(3)
    assert np.array_equal(cut, whole) and np.array_equal(cut_state, state)


# ---------------------------------------------------------------- the latent attention of prompts, keys and values of all heads made
@pytest.mark.parametrize("dim, rot, vdim, rank, heads, counts, starts", [
    (64, 64, 64, 128, 3, [1, 129, 40, 33], [0, 0, 31, 64]), (64, 64, 64, 64, 2, [5, 1, 130], [100, 63, 7]),
    (128, 64, 128, 512, 2, [70, 3], [0, 33]), (128, 64, 128, 64, 1, [32, 256], [32, 0])])
def test_latent_attention_of_prompts_with_every_heads_keys(ops, dim, rot, vdim, rank, heads, counts, starts):
    """Pages in shuffled order laid side by side; sequences of a token, of a run of 128 and one more, in the middle of a page, at its
    border, with keys before them; sinks and gates, and without; against 64 bits on the same keys and values.  The weights are rounded to
    bfloat16 (2^-9 of each) and the result once more: 2^-8 of the largest."""
    rng = np.random.default_rng(dim + len(counts))
    seqs, key_dim, ends = len(counts), rank + rot, [s + n for s, n in zip(starts, counts)]
    held = [-(-e // PAGE) for e in ends]
    order, width = rng.permutation(sum(held) + 2), max(held) + 1
    table, at = np.zeros((seqs, width), np.int32), 0
    for s, n in enumerate(held):
        table[s, :n], at = order[at:at + n], at + n
    k_pages = guarded((torch.randn((sum(held) + 2, 1, PAGE, key_dim), device=DEV) * 0.6).to(torch.bfloat16))
    rows = ops.latent_gather(k_pages, t(ends, torch.int32), t(table, torch.int32), sum(held))
    want_rows, pages = [], f64(k_pages)[:, 0]
    for s, e in enumerate(ends):
        own = np.concatenate([pages[table[s, j]] for j in range(held[s])])
        own[e:] = 0
        want_rows.append(own)
    assert np.array_equal(f64(rows), np.concatenate(want_rows))
    c = f64(rows)[:, :rank]
    uk, uv = rng.normal(size=(heads * dim, rank)) / np.sqrt(rank), rng.normal(size=(heads * vdim, rank)) / np.sqrt(rank)
    keys, values = t(c @ uk.T, torch.bfloat16), t(uv @ c.T, torch.bfloat16)
    qw, tokens = heads * (dim + rot), sum(counts)
    q = guarded((torch.randn((tokens, qw + 16 + (-heads) % 8 + heads), device=DEV) * 1.5).to(torch.bfloat16))
    sinks, g_off, scale = rng.normal(size=heads), qw + 16, 0.3
    cu = np.concatenate([[0], np.cumsum(counts)])
    pos = t([p for s, n in enumerate(counts) for p in range(starts[s], starts[s] + n)], torch.int32)
    k64, v64, q64 = f64(keys), f64(values), f64(q)
    for sink, gate in ((True, True), (False, False)):
        got = ops.latent_prompt(q, heads, dim, rot, vdim, keys, rows, values, scale, t(sinks) if sink else None, g_off if gate else None,
                                t(cu, torch.int32), pos, t(ends, torch.int32))
        want, first = np.zeros((tokens, heads, vdim)), 0
        for s in range(seqs):
            for h in range(heads):
                k = np.concatenate([k64[first:first + ends[s], h * dim:(h + 1) * dim], f64(rows)[first:first + ends[s], rank:]], 1)
                sc = scale * q64[cu[s]:cu[s + 1], h * (dim + rot):(h + 1) * (dim + rot)] @ k.T
                sc[np.arange(ends[s])[None, :] > np.arange(starts[s], ends[s])[:, None]] = -np.inf
                top = sc.max(1, keepdims=True)
                w = np.exp(sc - top)
                den = w.sum(1, keepdims=True) + (np.exp(np.float32(sinks[h]) - top) if sink else 0)
                o = (w / den) @ v64[h * vdim:(h + 1) * vdim, first:first + ends[s]].T
                want[cu[s]:cu[s + 1], h] = o / (1 + np.exp(-q64[cu[s]:cu[s + 1], g_off + h, None])) if gate else o
            first += held[s] * PAGE
        close(got, want.reshape(tokens, -1), 2.0 ** -8, f"latent prompt, sinks {sink}, gates {gate}")
