"""Each HIP kernel alone against its plain reference, at other sizes than the tiny models use.
Where random inputs would hide a fault, the inputs are made so that it shows.

The same tests run without a GPU when the environment says RI_TEST_KERNELS=emulated: then the kernels are the
CPU build of the same sources (tests/emulated.py), every operand lies between guard pages, and a kernel that
touches memory outside a buffer ends the run with a report.  tests/test_kernels_emulated.py starts that run."""
import os

import numpy as np
import pytest
import torch

from plain import qwen3_plain as P

EMULATED = os.environ.get("RI_TEST_KERNELS") == "emulated"
pytestmark = [] if EMULATED else pytest.mark.gpu
DEV = "cpu" if EMULATED else "cuda:0"


@pytest.fixture(scope="module")
def ops():
    if EMULATED:
        import emulated
        return emulated.ops()
    from rust_inference_amd.kernels import ops
    return ops


@pytest.fixture(autouse=True)
def _guarded_buffers_go_back():
    """Emulated: what a test laid between guard pages is unmapped when it ends (a later touch of it would fault)."""
    yield
    if EMULATED:
        import gc
        import emulated
        gc.collect()
        emulated.free_all()


def guarded(x):
    """On the GPU the tensor itself; emulated, a copy between guard pages."""
    if EMULATED:
        import emulated
        return emulated.tensor(x.contiguous(), "a test's operand")
    return x


def t(a, dtype=torch.float32):
    return guarded(torch.tensor(np.asarray(a), dtype=dtype, device=DEV))


def f64(x):
    return x.detach().to("cpu", torch.float64).numpy()


# What a kernel that hands out bfloat16 is held to, from what the comparisons below measured on an MI355X (every
# comparison can write what it measures into the file RI_TEST_ERROR_REPORT names): a bfloat16 result is rounded once
# at the end, half a unit of its last place, which is up to 3.9e-3 of its own size; the attention kernels, the norms
# with rotation and the products with bfloat16 out measure 2.2e-3 to 3.8e-3 of the largest value, and are held to
# twice that.  Where the result went through two such roundings (the fused decode attention reads the key it has just
# rounded; a linked gate|up product rounds its normed input and its result) 4.2e-3 to 4.7e-3 was measured.  Where the
# wanted result is one value row picked out by a score that stands out, rounding hardly shows: 2.8e-4 measured.
BF16_OUT = 7.5e-3
BF16_TWICE = 9.5e-3
BF16_ONE_KEY = 6e-4


def close(got, want, rel, what=""):
    want = np.asarray(want, dtype=np.float64)
    err = np.abs(f64(got) - want).max() / max(np.abs(want).max(), 1e-30)
    report = os.environ.get("RI_TEST_ERROR_REPORT")          # a file that collects what every comparison measured
    if report:
        with open(report, "a") as f:
            f.write(f"{os.environ.get('PYTEST_CURRENT_TEST', '?')}\t{what}\t{err:.3e}\t{rel:.0e}\n")
    assert err <= rel, f"{what}: error {err:.3e} of the largest value exceeds {rel:.0e}"


def test_the_extension_is_loaded_from_the_tree(ops):
    from rust_inference_amd.kernels import load_library
    lib = load_library()
    assert lib.ri_abi_version() >= 1


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embedding(ops, dtype):
    rng = np.random.default_rng(0)
    table = t(rng.normal(size=(1000, 200)), dtype)               # a vocabulary and a width that are no power of two
    ids = [999, 0, 2, 2, 517]
    got = ops.embed_gather(table, t(ids, torch.int32))
    assert got.dtype == torch.float32 and np.array_equal(f64(got), P.embedding(f64(table), ids))


@pytest.mark.parametrize("dim", [104, 4096, 5000])
@pytest.mark.parametrize("pending_dtype", [None, torch.float32, torch.bfloat16])
def test_add_rmsnorm(ops, dim, pending_dtype):
    rng = np.random.default_rng(dim)
    res = t(rng.normal(size=(7, dim)) * 3)
    pend = None if pending_dtype is None else t(rng.normal(size=(7, dim)), pending_dtype)
    gain = t(1 + 0.1 * rng.normal(size=dim))
    total = f64(res) + (0 if pend is None else f64(pend))
    want = P.rms_norm(total, f64(gain), 1e-5)
    before = guarded(res.clone())
    out = ops.add_rmsnorm(res, pend, gain, 1e-5, torch.float32)
    close(out, want, 2e-6, "norm")
    close(res, total, 1e-7, "residual written back")
    # rows: the same sums for a few rows, nothing written back
    res2 = guarded(before.clone())
    rows = t([5, 0, 5], torch.int32)
    out2 = ops.add_rmsnorm(res2, pend, gain, 1e-5, torch.bfloat16, rows)
    assert torch.equal(res2, before) and out2.dtype == torch.bfloat16
    close(out2, P.bf16_round(want[[5, 0, 5]].astype(np.float32)), 5e-3, "gathered rows")
    close(ops.add_rows(guarded(before.clone()), pend, rows), total[[5, 0, 5]], 1e-7, "add_rows")


def test_add_rmsnorm_adds_the_parts_of_a_split_product(ops):
    rng = np.random.default_rng(11)
    res, parts = t(rng.normal(size=(6, 4096))), t(rng.normal(size=(3, 6, 4096)))
    gain = t(1 + 0.1 * rng.normal(size=4096))
    total = f64(res) + f64(parts).sum(0)
    out = ops.add_rmsnorm(res, parts, gain, 1e-6, torch.float32)
    close(out, P.rms_norm(total, f64(gain), 1e-6), 2e-6, "norm over parts")
    close(res, total, 2e-7, "residual over parts")
    rows = t([4, 1], torch.int32)
    res2 = t(rng.normal(size=(6, 104)))
    p2 = t(rng.normal(size=(2, 6, 104)))
    g2 = t(np.ones(104))
    want = P.rms_norm((f64(res2) + f64(p2).sum(0))[[4, 1]], np.ones(104), 1e-6)
    close(ops.add_rmsnorm(res2, p2, g2, 1e-6, torch.float32, rows), want, 2e-6, "gathered rows over parts")


@pytest.mark.parametrize("n_parts", [2, 4, 5, 8, 9])
@pytest.mark.parametrize("dim", [72, 1000, 4096, 5120])
def test_the_norm_adds_any_number_of_parts_in_their_order(ops, n_parts, dim):
    """The parts are fetched four at a time; the sum is residual + part 0 + part 1 + ... in float32, bit for bit,
    whatever their number, and a row shorter than the threads' reach is not read beyond its end."""
    rng = np.random.default_rng(n_parts * dim)
    res = t(rng.normal(size=(5, dim)))
    parts = t(rng.normal(size=(n_parts, 5, dim)))
    gain = t(1 + 0.1 * rng.normal(size=dim))
    want_sum = guarded(res.clone())
    for q in range(n_parts):
        want_sum += parts[q]
    got = guarded(res.clone())
    out = ops.add_rmsnorm(got, parts, gain, 1e-6, torch.float32)
    assert torch.equal(got, want_sum)
    close(out, P.rms_norm(f64(want_sum), f64(gain), 1e-6), 2e-6, "norm over parts")


@pytest.mark.parametrize("pending_dtype", [torch.float32, torch.bfloat16])
def test_add_rows_in_place_and_bias(ops, pending_dtype):
    rng = np.random.default_rng(12)
    res, pend = t(rng.normal(size=(7, 104))), t(rng.normal(size=(7, 104)), pending_dtype)
    want = f64(res) + f64(pend)
    got = ops.add_rows(res, pend, in_place=True)
    assert got.data_ptr() == res.data_ptr()
    close(res, want, 1e-7, "the sum is written into the residual itself")
    bias = t(rng.normal(size=104))
    x = t(rng.normal(size=(5, 104)), pending_dtype)
    want = f64(x) + f64(bias)
    close(ops.add_bias(x, bias), want, 1e-7 if pending_dtype == torch.float32 else 5e-3, "bias")


@pytest.mark.parametrize("m, dim, partials, tiled", [(1, 104, 1, False), (5, 4096, 256, False), (16, 584, 37, True),
                                                      (40, 4096, 4096, True)])
def test_a_norm_left_to_a_product_can_be_finished_alone(ops, m, dim, partials, tiled):
    """xg = bfloat16(r * gain) and partial sums of r^2 per row: the normed rows are xg / sqrt(sum / dim + eps)."""
    rng = np.random.default_rng(m + dim)
    r, gain = rng.normal(size=(m, dim)), 1 + 0.1 * rng.normal(size=dim)
    xg = t(r * gain, torch.bfloat16)
    ssq = rng.dirichlet(np.ones(partials), size=m) * (r * r).sum(1, keepdims=True)      # any split of the sums
    if tiled:
        data = ops.TiledRows.empty(m, dim, DEV)
        data.data.zero_()
        padded = torch.zeros((data.data.shape[0] * 16, data.data.shape[1] * 32), dtype=torch.bfloat16, device=DEV)
        padded[:m, :dim] = xg
        data.data.copy_(padded.view(-1, 16, data.data.shape[1], 4, 8).permute(0, 2, 3, 1, 4).reshape(data.data.shape))
        assert torch.equal(data.rows(), xg)
        src = data
    else:
        src = xg
    got = ops.finish_norm(ops.NormedLater(src, t(ssq), 1e-6, dim))
    want = f64(xg) / np.sqrt((r * r).sum(1, keepdims=True) / dim + 1e-6)
    close(got, want, 5e-3, "finished norm")


def test_add_rmsnorm_fused_equals_unfused_bit_for_bit(ops):
    # src/ops/norm.rs:84-98
    a, r = t([[0.5, -1.0, 2.0, 0.25]]), t([[1.0, 1.0, -1.0, 0.0]])
    w = t([1.0, 0.5, 2.0, 1.0])
    res = guarded(r.clone())
    fused = ops.add_rmsnorm(res, a, w, 1e-6, torch.float32)
    plain_sum = (a + r).contiguous()
    assert torch.equal(res, plain_sum)
    assert torch.equal(fused, ops.add_rmsnorm(guarded(plain_sum.clone()), None, w, 1e-6, torch.float32))


def paged(rng, lens, hkv, dh, page_size=32, dtype=torch.float32, spare=3):
    """Keys and values of several sequences laid into pages in a shuffled physical order."""
    pages_per = [-(-n // page_size) for n in lens]
    num_pages = sum(pages_per) + spare
    order = list(rng.permutation(num_pages))
    width = max(pages_per) + 1
    table = np.full((len(lens), width), -1, dtype=np.int32)
    k = [rng.normal(size=(n, hkv, dh)) for n in lens]
    v = [rng.normal(size=(n, hkv, dh)) for n in lens]
    kp = np.zeros((num_pages, hkv, page_size, dh))
    vp = np.zeros((num_pages, hkv, dh, page_size))                 # values lie transposed inside a page
    for b, n in enumerate(lens):
        for lp in range(pages_per[b]):
            table[b, lp] = order.pop()
        for pos in range(n):
            kp[table[b, pos // page_size], :, pos % page_size] = k[b][pos]
            vp[table[b, pos // page_size], :, :, pos % page_size] = v[b][pos]
    return k, v, t(kp, dtype), t(vp, dtype), t(table, torch.int32)


@pytest.mark.parametrize("paged_values", [False, True])
@pytest.mark.parametrize("dtype, rel", [(torch.float32, 3e-6), (torch.bfloat16, BF16_OUT)])
@pytest.mark.parametrize("heads, kv_heads, dh", [(6, 2, 48), (4, 4, 128), (9, 1, 16), (2, 1, 256), (5, 5, 64), (8, 2, 32),
                                                 (4, 2, 8), (6, 3, 24), (3, 1, 40), (2, 2, 2), (2, 1, 328), (4, 2, 512)])
def test_qk_norm_rope_kv_write(ops, dtype, rel, heads, kv_heads, dh, paged_values):
    rng = np.random.default_rng(heads * dh)
    lens_before, new = [37, 0, 63, 30], [3, 2, 5, 70]            # writes cross page boundaries; one spans four pages
    lens = [a + b for a, b in zip(lens_before, new)]
    _, _, kp, vp, table = paged(rng, lens, kv_heads, dh, dtype=dtype)
    kp.zero_(); vp.zero_()
    tokens = sum(new)
    qkv = rng.normal(size=(tokens, (heads + 2 * kv_heads) * dh)) * 2
    qkv_t = t(qkv, dtype)
    qkv = f64(qkv_t)
    tok_seq = [b for b, n in enumerate(new) for _ in range(n)]
    tok_pos = [lens_before[b] + i for b, n in enumerate(new) for i in range(n)]
    qg, kg = 1 + 0.2 * rng.normal(size=dh), 1 + 0.2 * rng.normal(size=dh)
    theta, eps = 50000.0, 1e-5
    inv_freq = t(P.rope_inv_freq(dh, theta))
    # with the sequences' bounds the 16-byte kernels and the page-wise value writer run (where the head size fits)
    extra = dict(cu_seqlens=t(np.concatenate([[0], np.cumsum(new)]), torch.int32), max_new=max(new)) if paged_values else {}
    ops.qk_norm_rope_kv_write(qkv_t, t(qg), t(kg), eps, inv_freq, t(tok_pos, torch.int32), t(tok_seq, torch.int32),
                              table, kp, vp, heads, kv_heads, dh, **extra)
    ang = P.rope_angles(tok_pos, dh, theta)
    q = qkv[:, :heads * dh].reshape(tokens, heads, dh)
    k = qkv[:, heads * dh:(heads + kv_heads) * dh].reshape(tokens, kv_heads, dh)
    v = qkv[:, (heads + kv_heads) * dh:].reshape(tokens, kv_heads, dh)
    q_want = P.apply_rope(P.rms_norm(q, f64(t(qg)), eps), ang)
    k_want = P.apply_rope(P.rms_norm(k, f64(t(kg)), eps), ang)
    close(qkv_t[:, :heads * dh].reshape(tokens, heads, dh), q_want, rel, "q in place")
    tab = table.cpu().numpy()
    for i in range(tokens):
        page, off = tab[tok_seq[i], tok_pos[i] // 32], tok_pos[i] % 32
        close(kp[page, :, off], k_want[i], rel, f"k of token {i}")
        assert np.array_equal(f64(vp[page, :, :, off]), v[i]), "v is a copy"
    # nothing else was written: as many rows are non-zero as tokens
    assert int((kp.float().abs().sum(-1) > 0).sum()) == tokens * kv_heads
    assert int((vp.float().abs().sum(-2) > 0).sum()) == tokens * kv_heads
    # without gains and rotation the kernel only moves k and v
    qkv2 = t(qkv, dtype)
    ops.qk_norm_rope_kv_write(qkv2, None, None, eps, None, t(tok_pos, torch.int32), t(tok_seq, torch.int32),
                              table, kp, vp, heads, kv_heads, dh, **extra)
    assert np.array_equal(f64(qkv2), qkv)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads, kv_heads, dh", [(2, 1, 16), (3, 3, 128), (6, 2, 256)])
def test_values_turned_by_groups_of_eight_positions(ops, dtype, heads, kv_heads, dh):
    """Steps that begin and end on and beside a group's and a page's edge: the values as they are, and no other place touched."""
    before, new = [0, 8, 7, 9, 24, 31, 0, 33, 40], [32, 8, 1, 6, 8, 2, 9, 31, 64]
    rng = np.random.default_rng(dh)
    _, _, kp, vp, table = paged(rng, [a + n for a, n in zip(before, new)], kv_heads, dh, dtype=dtype)
    want = f64(vp).copy()
    qkv = t(rng.normal(size=(sum(new), (heads + 2 * kv_heads) * dh)), dtype)
    seq, pos = [b for b, n in enumerate(new) for _ in range(n)], [before[b] + i for b, n in enumerate(new) for i in range(n)]
    for i, (b, p) in enumerate(zip(seq, pos)):
        want[table[b, p // 32].item(), :, :, p % 32] = f64(qkv[i, (heads + kv_heads) * dh:]).reshape(kv_heads, dh)
    ops.qk_norm_rope_kv_write(qkv, None, None, 1e-5, None, t(pos, torch.int32), t(seq, torch.int32), table, kp, vp, heads, kv_heads, dh,
                              cu_seqlens=t(np.concatenate([[0], np.cumsum(new)]), torch.int32), max_new=max(new))
    assert np.array_equal(f64(vp), want)


@pytest.mark.skipif(EMULATED, reason="eight million workgroups, almost all of them empty")
def test_values_in_a_launch_of_their_own_past_what_one_holds(ops):
    """A bound on the new tokens far above the real ones, whose workgroups are more than the launch with the queries is to hold."""
    rng = np.random.default_rng(5)
    heads, kv_heads, dh, new = 16, 2, 128, [37, 3]
    qkv, out = t(rng.normal(size=(40, (heads + 2 * kv_heads) * dh)), torch.bfloat16), []
    pos, seq, cu = t(list(range(37)) + [0, 1, 2], torch.int32), t([0] * 37 + [1] * 3, torch.int32), t([0, 37, 40], torch.int32)
    for most in (37, 1 << 27):
        _, _, kp, vp, table = paged(np.random.default_rng(6), new, kv_heads, dh, dtype=torch.bfloat16)
        rows = qkv.clone()
        ops.qk_norm_rope_kv_write(rows, None, None, 1e-5, None, pos, seq, table, kp, vp, heads, kv_heads, dh, cu_seqlens=cu, max_new=most)
        whole, wk, wv = qkv[:, :(heads + kv_heads) * dh].contiguous(), kp.clone(), vp.clone()
        ops.whole_norm_kv_write(whole, 0, heads * dh, t(np.ones(heads * dh)), t(np.ones(kv_heads * dh)), 1e-5, pos, seq, table, wk, wv, heads, kv_heads, dh,
                                cu_seqlens=cu, max_new=most)
        out.append([f64(x) for x in (rows, kp, vp, whole, wk, wv)])
    assert all(np.array_equal(a, b) for a, b in zip(*out)) and (out[0][2] != 0).any()


@pytest.mark.parametrize("dtype, rel", [(torch.float32, 3e-6), (torch.bfloat16, BF16_OUT)])
@pytest.mark.parametrize("dh, rot", [(64, 16), (48, 24), (40, 8), (7, 4), (9, 0), (130, 128), (512, 64)])
def test_rotation_over_part_of_the_head(ops, dtype, rel, dh, rot):
    """The first `rot` elements of a head are rotated in pairs (i, i + rot/2) by frequencies of their own, the rest
    is normed only; `rot` 0: no rotation at all, which an odd head size allows."""
    rng = np.random.default_rng(dh + rot)
    heads, kv_heads, new = 3, 1, [5, 40]
    _, _, kp, vp, table = paged(rng, new, kv_heads, dh, dtype=dtype)
    kp.zero_(); vp.zero_()
    tokens = sum(new)
    qkv_t = t(rng.normal(size=(tokens, (heads + 2 * kv_heads) * dh)) * 2, dtype)
    qkv = f64(qkv_t)
    tok_seq = [b for b, n in enumerate(new) for _ in range(n)]
    tok_pos = [i for n in new for i in range(n)]
    qg, kg = 1 + 0.2 * rng.normal(size=dh), 1 + 0.2 * rng.normal(size=dh)
    inv = (1.0 / 10000.0 ** (np.arange(rot // 2) * 2.0 / max(rot, 1))).astype(np.float32) if rot else None
    ops.qk_norm_rope_kv_write(qkv_t, t(qg), t(kg), 1e-5, None if inv is None else t(inv), t(tok_pos, torch.int32),
                              t(tok_seq, torch.int32), table, kp, vp, heads, kv_heads, dh)

    def want(x, gain):
        y = P.rms_norm(x, f64(t(gain)), 1e-5)
        if rot:
            ang = (np.asarray(tok_pos, dtype=np.float32)[:, None] * inv[None, :]).astype(np.float32).astype(np.float64)
            y = np.concatenate([P.apply_rope(y[..., :rot], ang), y[..., rot:]], -1)
        return y
    q = qkv[:, :heads * dh].reshape(tokens, heads, dh)
    k = qkv[:, heads * dh:(heads + kv_heads) * dh].reshape(tokens, kv_heads, dh)
    close(qkv_t[:, :heads * dh].reshape(tokens, heads, dh), want(q, qg), rel, "q")
    tab = table.cpu().numpy()
    k_want = want(k, kg)
    for i in range(tokens):
        close(kp[tab[tok_seq[i], tok_pos[i] // 32], :, tok_pos[i] % 32], k_want[i], rel, f"k of token {i}")
    with pytest.raises(Exception, match="frequencies"):
        ops.qk_norm_rope_kv_write(qkv_t, t(qg), t(kg), 1e-5, t(np.ones(dh // 2 + 1, dtype=np.float32)), t(tok_pos, torch.int32),
                                  t(tok_seq, torch.int32), table, kp, vp, heads, kv_heads, dh)


def attention_case(ops, rng, lens, new, heads, kv_heads, dh, dtype, window=None, boost=None, kernel="generic", paired=False):
    k, v, kp, vp, table = paged(rng, lens, kv_heads, dh, dtype=dtype, spare=12)
    tokens = sum(new)
    width = (heads + 2 * kv_heads) * dh
    qkv = np.zeros((tokens, width))
    qkv[:, :heads * dh] = rng.normal(size=(tokens, heads * dh))
    tok_seq = [b for b, n in enumerate(new) for _ in range(n)]
    tok_pos = [lens[b] - n + i for b, n in enumerate(new) for i in range(n)]
    if boost is not None:
        boost(qkv, k, kp, table)
    qkv_t = t(qkv, dtype)
    pos_t, seq_t = t(tok_pos, torch.int32), t(tok_seq, torch.int32)
    cu = t(np.concatenate([[0], np.cumsum(new)]), torch.int32)
    scale = 1.0 / np.sqrt(dh)
    if kernel == "generic":
        out = ops.attention(qkv_t, kp, vp, pos_t, seq_t, table, heads, kv_heads, dh, window, scale)
    elif kernel == "prefill":
        out = ops.attention_prefill_bf16(qkv_t, kp, vp, cu, pos_t, table, len(lens), max(new), heads, kv_heads, dh,
                                         window, scale, **({} if paired is False else dict(new_counts=new, paired=paired)))
    else:
        assert all(n == 1 for n in new)
        # a bound on the length well above the real one: it sizes grid and workspace, never the result
        out = ops.attention_decode_bf16(qkv_t, kp, vp, cu, pos_t, table, len(lens), max(lens) + 300, heads,
                                        kv_heads, dh, window, scale)
    q = f64(qkv_t)[:, :heads * dh].reshape(tokens, heads, dh)
    want = np.zeros((tokens, heads, dh))
    i = 0
    for b, n in enumerate(new):
        kb = np.stack([f64(kp[table[b, p // 32].item(), :, p % 32]) for p in range(lens[b])])
        vb = np.stack([f64(vp[table[b, p // 32].item(), :, :, p % 32]) for p in range(lens[b])])
        want[i:i + n] = P.attention(q[i:i + n], kb, vb, window=window)
        i += n
    return out.reshape(tokens, heads, dh), want


@pytest.mark.parametrize("dtype, rel", [(torch.float32, 3e-6), (torch.bfloat16, BF16_OUT)])
@pytest.mark.parametrize("heads, kv_heads, dh", [(4, 2, 16), (6, 2, 48), (8, 1, 128), (3, 3, 64), (9, 1, 32),
                                                 # any head size: the reference's own attention test runs 8
                                                 # (src/attention.rs:189-219); odd ones; beyond 256
                                                 (4, 2, 8), (6, 2, 24), (2, 1, 40), (3, 1, 7), (2, 2, 1), (2, 1, 328), (2, 1, 512)])
def test_attention_prompts_pieces_and_single_tokens(ops, dtype, rel, heads, kv_heads, dh):
    rng = np.random.default_rng(heads + dh)
    # a whole prompt, a piece of five tokens at the end of 300, one token at 257 (a tile's first key), one at 1
    out, want = attention_case(ops, rng, [70, 300, 257, 1], [70, 5, 1, 1], heads, kv_heads, dh, dtype)
    close(out, want, rel, "attention")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads, kv_heads, dh, vd, form", [(8, 4, 128, 128, "plain"), (10, 2, 24, 40, "window"), (8, 1, 64, 200, "chunk"),
                                                           (8, 8, 16, 16, "kept"), (24, 2, 32, 128, "plain")])
def test_attention_rows_of_queries_share_their_loads(ops, dtype, heads, kv_heads, dh, vd, form):
    """Runs of tokens (whole prompts, the ends of longer sequences, single tokens among them) as rows that share keys: the same
    bits as a workgroup for every token and head, whatever the mask."""
    lens, new = ([11, 270, 257], [11, 7, 1]) if EMULATED else ([200, 700, 257, 3, 90], [200, 60, 1, 3, 90])
    rng = np.random.default_rng(heads + dh)
    _, _, kp, _, table = paged(rng, lens, kv_heads, dh, dtype=dtype, spare=12)
    vp = t(rng.normal(size=(kp.shape[0], kv_heads, vd, 32)), dtype)
    qkv = t(rng.normal(size=(sum(new), heads * dh + 8)), dtype)
    seq = t([b for b, n in enumerate(new) for _ in range(n)], torch.int32)
    pos = t([lens[b] - n + i for b, n in enumerate(new) for i in range(n)], torch.int32)
    more = {"plain": dict(softcap=20.0), "window": dict(slopes=t(rng.uniform(0.01, 0.1, heads))), "chunk": dict(chunk=50),
            "kept": dict(keep_first=5, sinks=t(rng.normal(size=heads)))}[form]
    window = {"window": 37, "kept": 270}.get(form)
    alone, shared = (f64(ops.attention(qkv, kp, vp, pos, seq, table, heads, kv_heads, dh, window, dh ** -0.5, most_new=most, **more))
                     for most in (1, max(new)))
    assert np.isfinite(alone).all() and np.array_equal(alone, shared)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", [dict(window=37), dict(chunk=50), dict(window=37, keep_first=5), dict(window=300, keep_first=40)])
@pytest.mark.parametrize("dh", [64, 48])
def test_attention_rows_of_queries_leave_pages_given_back_alone(ops, dtype, form, dh, monkeypatch):
    """Steps that go on behind a window or a chunk: the pages that no query can see any more are out of the tables (-1, as the cache
    leaves them), and the first visible key lies in the middle of a tile of 256 and of its page.  The same bits as a workgroup for
    every token and head, which reads the keys it sees alone.  (float32 heads of 64 take the matrix cores each time.)"""
    before, new = ([380, 301, 90, 0, 611], [10, 7, 1, 12, 5]) if EMULATED else ([380, 701, 90, 0, 1200], [10, 70, 1, 200, 33])
    heads, kv_heads, page = 8, 2, 32
    rng = np.random.default_rng(len(form) + sum(form.values()))
    _, _, kp, vp, table = paged(rng, [a + n for a, n in zip(before, new)], kv_heads, dh, dtype=dtype)
    window, chunk, keep = form.get("window"), form.get("chunk"), form.get("keep_first", 0)
    for b, length in enumerate(before):
        first = length - length % chunk if chunk else max(0, length - window + 1)
        table[b, -(-keep // page):max(first // page, -(-keep // page))] = -1
    qkv = t(rng.normal(size=(sum(new), heads * dh)), dtype)
    seq = t([b for b, n in enumerate(new) for _ in range(n)], torch.int32)
    pos = t([before[b] + i for b, n in enumerate(new) for i in range(n)], torch.int32)
    monkeypatch.setattr(ops, "ATTENTION_ROWS_BYTES", 0)
    runs = dict(new_counts=new, starts=before, cu_seqlens=t(np.concatenate([[0], np.cumsum(new)]), torch.int32))
    alone, shared, runs = (f64(ops.attention(qkv, kp, vp, pos, seq, table, heads, kv_heads, dh, window, dh ** -0.5, keep_first=keep,
                                             chunk=chunk, **how)) for how in ({}, dict(most_new=max(new)), runs))
    assert np.isfinite(alone).all() and np.array_equal(alone, shared) and np.array_equal(alone, runs)


@pytest.mark.parametrize("heads, kv_heads, dh, vd", [(4, 4, 16, 24), (8, 2, 32, 160), (16, 1, 16, 16)])
def test_attention_rows_of_queries_beside_single_tokens(ops, heads, kv_heads, dh, vd, monkeypatch):
    """A step of single tokens, short pieces and prompts, more sequences than a wavefront has lanes: the prompts' runs share their
    loads, every other token keeps a workgroup a head.  The same bits as without the sequences' bounds."""
    new = [1] * 5 + [40, 3, 1, 4, 17] + [1] * 57 + [9, 1, 16, 2]
    rng = np.random.default_rng(heads)
    before = [int(n) for n in rng.integers(0, 40 if EMULATED else 700, len(new))]
    _, _, kp, _, table = paged(rng, [a + n for a, n in zip(before, new)], kv_heads, dh)
    vp = t(rng.normal(size=(kp.shape[0], kv_heads, vd, 32)))
    qkv = t(rng.normal(size=(sum(new), heads * dh)))
    seq = t([b for b, n in enumerate(new) for _ in range(n)], torch.int32)
    pos = t([before[b] + i for b, n in enumerate(new) for i in range(n)], torch.int32)
    cu = t(np.concatenate([[0], np.cumsum(new)]), torch.int32)
    monkeypatch.setattr(ops, "ATTENTION_ROWS_BYTES", 0)
    least, tokens, runs = ops.attention_rows_plan(new, before, heads, kv_heads, 4 * dh, None)
    per = 16 // (heads // kv_heads)
    many = [n for n in new if n >= least]
    assert least == max(4, 8 * kv_heads // heads) and tokens == sum(many) < sum(new) and runs == sum(-(-n // per) for n in many)
    got = ops.attention(qkv, kp, vp, pos, seq, table, heads, kv_heads, dh, None, 0.3, new_counts=new, starts=before, cu_seqlens=cu)
    want = ops.attention(qkv, kp, vp, pos, seq, table, heads, kv_heads, dh, None, 0.3)
    assert torch.isfinite(want).all() and torch.equal(got, want)


@pytest.mark.parametrize("heads, kv_heads, dh, form", [(4, 2, 64, dict(softcap=15.0)), (3, 1, 128, dict(window=20, keep_first=5)),
                                                       (16, 1, 64, dict(chunk=24)), (2, 2, 128, dict())])
def test_attention_float32_on_the_matrix_cores(ops, heads, kv_heads, dh, form):
    """Tiles of sixteen keys and sixteen rows and their remainders, every mask, with sinks and slopes, against 64 bits; whatever lies
    behind a sequence's last key does not count; the same bits in runs, as tokens lie and one by one, and in pieces."""
    before, new = [0, 0, 0, 15, 16, 63, 40, 0], [1, 15, 33, 1, 17, 2, 30, 16]
    rng = np.random.default_rng(dh + heads)
    k, v, kp, vp, table = paged(rng, [a + n for a, n in zip(before, new)], kv_heads, dh)
    for b, (a, n) in enumerate(zip(before, new)):
        if (a + n) % 32:
            page = table[b, (a + n) // 32].item()
            kp[page, :, (a + n) % 32:], vp[page, :, :, (a + n) % 32:] = float("nan"), float("nan")
    q = rng.normal(size=(sum(new), heads * dh)).astype(np.float32)
    slopes, sinks = (rng.uniform(0.01, 0.1, heads).astype(np.float32), rng.normal(size=heads).astype(np.float32))
    window, chunk, keep, cap = (form.get(n) for n in ("window", "chunk", "keep_first", "softcap"))
    more = dict(softcap=cap, slopes=t(slopes), keep_first=keep or 0, sinks=t(sinks), chunk=chunk)

    def run(pieces, **how):
        """Every sequence's new tokens from its piece of them on."""
        rows = [sum(new[:b]) + i for b, (lo, hi) in enumerate(pieces) for i in range(lo, hi)]
        pos = t([before[b] + i for b, (lo, hi) in enumerate(pieces) for i in range(lo, hi)], torch.int32)
        seq = t([b for b, (lo, hi) in enumerate(pieces) for _ in range(lo, hi)], torch.int32)
        if how.pop("runs", False):
            n = [hi - lo for lo, hi in pieces]
            how = dict(new_counts=n, starts=[a + lo for a, (lo, hi) in zip(before, pieces)], cu_seqlens=t(np.concatenate([[0], np.cumsum(n)]), torch.int32))
        return rows, f64(ops.attention(t(q[rows]), kp, vp, pos, seq, table, heads, kv_heads, dh, window, dh ** -0.5, **how, **more))

    whole = [(0, n) for n in new]
    got = run(whole, runs=True)[1]
    assert np.array_equal(got, run(whole)[1]) and np.array_equal(got, run(whole, most_new=max(new))[1])
    for pieces in ([(0, n // 2) for n in new], [(n // 2, n) for n in new]):
        rows, part = run(pieces, runs=True)
        assert np.array_equal(part, got[rows])
    row = 0
    for b, (a, n) in enumerate(zip(before, new)):
        kb = np.stack([f64(kp[table[b, j // 32].item(), :, j % 32]) for j in range(a + n)])
        vb = np.stack([f64(vp[table[b, j // 32].item(), :, :, j % 32]) for j in range(a + n)])
        for i in range(n):
            at, j = a + i, np.arange(a + i + 1)
            lo = at - at % chunk if chunk else max(0, at - window + 1) if window else 0
            for h in range(heads):
                s = kb[:at + 1, h * kv_heads // heads] @ q[row, h * dh:(h + 1) * dh].astype(np.float64) * dh ** -0.5
                s = (cap * np.tanh(s / cap) if cap else s) - slopes[h].astype(np.float64) * (at - j)
                p = np.where((j >= lo) | (j < (keep or 0)), np.exp(s), 0.0)
                want = p @ vb[:at + 1, h * kv_heads // heads] / (p.sum() + np.exp(np.float64(sinks[h])))
                close(t(got[row, h * dh:(h + 1) * dh]), want, 3e-6, f"sequence {b}, token {i}, head {h}")
            row += 1


@pytest.mark.parametrize("dh, form", [(64, dict(window=37)), (128, dict(chunk=50)), (64, dict(window=37, keep_first=5)), (128, dict(window=100, keep_first=40))])
def test_attention_float32_on_the_matrix_cores_leaves_pages_given_back_alone(ops, dh, form):
    """Behind a window or a chunk a table holds -1; in runs, as tokens lie and one by one, against the general kernel, which takes the same
    pages where they start off a 16-byte boundary.  float32 sums in another order."""
    before, new = [180, 101, 90, 0, 211], [10, 7, 1, 12, 5]
    heads, kv_heads, page = 8, 2, 32
    rng = np.random.default_rng(dh + sum(form.values()))
    _, _, kp, vp, table = paged(rng, [a + n for a, n in zip(before, new)], kv_heads, dh)
    window, chunk, keep = form.get("window"), form.get("chunk"), form.get("keep_first", 0)
    for b, length in enumerate(before):
        first = length - length % chunk if chunk else max(0, length - window + 1)
        table[b, -(-keep // page):max(first // page, -(-keep // page))] = -1
    assert (table[:, :3] == -1).any()
    qkv = t(rng.normal(size=(sum(new), heads * dh)))
    seq, pos = t([b for b, n in enumerate(new) for _ in range(n)], torch.int32), t([before[b] + i for b, n in enumerate(new) for i in range(n)], torch.int32)
    runs = dict(new_counts=new, starts=before, cu_seqlens=t(np.concatenate([[0], np.cumsum(new)]), torch.int32))

    def off(x):
        """The same numbers four bytes behind a boundary."""
        whole = t(np.zeros(x.numel() + 1))
        whole[1:] = x.reshape(-1)
        return whole[1:].view(x.shape)

    run = lambda k, v, how: f64(ops.attention(qkv, k, v, pos, seq, table, heads, kv_heads, dh, window, dh ** -0.5, keep_first=keep, chunk=chunk, **how))
    want = run(off(kp), off(vp), {})
    assert np.array_equal(want, run(off(kp), off(vp), runs)) and np.isfinite(want).all()
    for how in ({}, dict(most_new=max(new)), runs):
        close(t(run(kp, vp, how)), want, 3e-6, str(list(how)))


def test_attention_shares_loads_where_that_is_less_to_wait_for(ops, monkeypatch):
    """Prompts enough to fill the machine do; one of 130 tokens, many of four and steps of single tokens do not, nor do single tokens
    that stand beside a prompt."""
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    plan = lambda new, starts, heads=16, kv_heads=8, reach=None: ops.attention_rows_plan(new, starts, heads, kv_heads, 512, reach)[1:]
    assert plan([326, 33, 400], [0] * 3) == (759, 41 + 5 + 50) and plan([2000], [0]) == (2000, 250)
    assert plan([1] * 64 + [300], [2000] * 64 + [0]) == (300, 38) and plan([130], [2000]) == (130, 17)
    assert plan([130], [0]) == plan([4] * 200, [0] * 200) == plan([1] * 300, [1000] * 300) == plan([1] * 300 + [4], [1000] * 301) == (0, 0)
    assert plan([200], [3000], reach=512) == (200, 25) and plan([2000], [0], 32, 1) == (0, 0)      # (32 heads a kv head: too many rows)
    assert ops.attention_rows_plan([1000], [0], 16, 8, 48, None)[1:] == (1000, 125)               # (small rows: what a key costs beside its bytes)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_attention_finds_one_far_key_among_hundreds(ops, dtype):
    """One key far back gets a score that stands out: the output must be its value, wherever it lies."""
    rng = np.random.default_rng(9)
    heads, kv_heads, dh = 4, 2, 64
    for far in (0, 31, 32, 255, 256, 511, 640):
        def boost(qkv, k, kp, table, far=far):
            # sequence 0's single query, head 1 (kv head 0): q = 8 * k_far / |k_far| * sqrt(dh)
            kf = f64(kp[table[0, far // 32].item(), 0, far % 32])
            qkv[0, dh:2 * dh] = 40.0 * kf / np.linalg.norm(kf) ** 2 * np.sqrt(dh)
        out, want = attention_case(ops, rng, [700], [1], heads, kv_heads, dh, dtype, boost=boost)
        close(out, want, 3e-6 if dtype == torch.float32 else BF16_ONE_KEY, f"far key {far}")
        # and the plain result really is that one value (the test is not vacuous)
        assert np.abs(want[0, 1]).max() > 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("window", [1, 32, 33, 100, 256, 300])
def test_attention_window_edges(ops, dtype, window):
    rng = np.random.default_rng(window)
    out, want = attention_case(ops, rng, [290, 40], [34, 40], 4, 2, 32, dtype, window=window)
    close(out, want, 3e-6 if dtype == torch.float32 else BF16_OUT, f"window {window}")


MFMA_SHAPES = [(4, 1, 32), (8, 2, 32), (6, 2, 64), (3, 3, 64), (32, 8, 128), (16, 1, 128), (5, 5, 128)]


@pytest.mark.parametrize("heads, kv_heads, dh", MFMA_SHAPES)
def test_mfma_prefill_attention(ops, heads, kv_heads, dh):
    rng = np.random.default_rng(heads * 7 + dh)
    # whole prompts of unequal lengths (one shorter than a tile, one of one token), and pieces that
    # continue sequences already in the cache, all in one call
    out, want = attention_case(ops, rng, [70, 300, 257, 1, 45, 131], [70, 5, 1, 1, 45, 99], heads, kv_heads, dh,
                               torch.bfloat16, kernel="prefill")
    close(out, want, BF16_OUT, "prefill attention on the matrix cores")


@pytest.mark.parametrize("heads", [20, 32])
def test_prompt_attention_with_two_tiles_a_wavefront(ops, heads):
    """More query heads a key head than one tile of sixteen columns holds: two tiles whatever the step's size."""
    out, want = attention_case(ops, np.random.default_rng(heads), [33, 100, 1], [33, 5, 1], heads, 1, 128, torch.bfloat16, kernel="prefill")
    close(out, want, BF16_OUT, "prefill attention, two tiles a wavefront")


@pytest.mark.parametrize("heads, window", [(16, None), (13, 50), (16, 20)])
def test_prompt_attention_with_two_tiles_on_a_small_machine(ops, heads, window):
    """Heads of 128 whose queries one tile would hold: two where a machine of one unit is filled (on a larger one, one)."""
    if ops.compute_units() == 1:
        assert ops.attention_prefill_tiles([110], heads, 1, 128) == 2 and ops.attention_prefill_tiles([110, 97], heads, 1, 128) == 2
    for lens, new in (([130], [110]), ([110, 160], [110, 97])):
        out, want = attention_case(ops, np.random.default_rng(heads), lens, new, heads, 1, 128, torch.bfloat16, window=window, kernel="prefill")
        close(out, want, BF16_OUT, "prefill attention, two tiles a wavefront")


def test_prompt_attention_tiles_follow_the_tokens_of_the_long_prompts(ops):
    """Heads of 128 on 256 compute units, as measured beside the rule: two tiles a wavefront for long prompts, for very long ones also
    where single tokens stand beside them; one for short prompts and for steps that two would not fill."""
    if not EMULATED and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("measured on 256 compute units")
    tiles = ops.attention_prefill_tiles
    ragged = [200 + i * 824 // 11 for i in range(12)]
    assert tiles([8192], 16, 8, 128) == 2 and tiles([8192] + [1] * 40, 16, 8, 128) == 2 and tiles([4096, 4096] + [1] * 200, 32, 8, 128) == 2
    assert tiles([3072], 32, 8, 128) == 2 and tiles([300, 900, 1500, 1800], 32, 8, 128) == 2
    assert tiles([500, 1500, 900], 32, 8, 128) == 1 and tiles(ragged, 16, 8, 128) == 1 and tiles([2048], 32, 8, 128) == 1
    assert tiles([3000] + [1] * 63, 32, 8, 128) == 1 and tiles([1024] * 8 + [1] * 8, 16, 8, 128) == 1 and tiles([1] * 1000, 16, 8, 128) == 1


@pytest.mark.parametrize("heads, kv_heads, dh, vdim", [(16, 1, 128, 128), (32, 2, 64, 64), (15, 1, 32, 32), (16, 1, 24, 40)])
def test_prompt_attention_of_a_prompt_among_single_tokens(ops, heads, kv_heads, dh, vdim):
    """Steps whose grid would be empty for the most part go run by run: prompts of one workgroup's tokens, one more and many, first, last
    and between single tokens; the same bits as every sequence by itself."""
    rng = np.random.default_rng(dh)
    new = [1] * 5 + [33] + [1] * 2 + [4, 5] + [1] * 4 + [17]
    before = [int(x) for x in rng.integers(0, 70, len(new))]
    pages = [-(-(a + n) // 32) for a, n in zip(before, new)]
    table = np.full((len(new), max(pages)), -1, dtype=np.int32)
    order = iter(rng.permutation(sum(pages)))
    for b, n in enumerate(pages):
        table[b, :n] = [next(order) for _ in range(n)]
    kp, vp = (t(rng.normal(size=(sum(pages), kv_heads) + shape), torch.bfloat16) for shape in ((32, dh), (vdim, 32)))
    qkv, at = t(rng.normal(size=(sum(new), heads * dh)), torch.bfloat16), np.concatenate([[0], np.cumsum(new)])
    pos = [a + i for a, n in zip(before, new) for i in range(n)]

    def run(seqs):
        n, rows = [new[b] for b in seqs], [i for b in seqs for i in range(at[b], at[b + 1])]
        args = (t(f64(qkv)[rows], torch.bfloat16), kp, vp, t(np.concatenate([[0], np.cumsum(n)]), torch.int32), t([pos[i] for i in rows], torch.int32),
                t(table[seqs], torch.int32), len(n), max(n), heads, kv_heads)
        if dh == vdim:
            return f64(ops.attention_prefill_bf16(*args, dh, None, dh ** -0.5, new_counts=n))
        return f64(ops.attention_prefill_padded(*args, None, dh ** -0.5))

    together = run(list(range(len(new))))
    for b in range(len(new)):
        assert np.array_equal(together[at[b]:at[b + 1]], run([b])), f"sequence {b} of {new[b]} tokens"


@pytest.mark.skipif(EMULATED, reason="eight thousand tokens")
@pytest.mark.parametrize("cap", [None, 20.0])
def test_prompt_attention_of_a_long_prompt_is_its_pieces(ops, cap):
    """A prompt long enough for two tiles a wavefront, and its last tokens in a step of their own, with one: the same bits."""
    rng = np.random.default_rng(3)
    n, last, heads, kv_heads, dh = 8000, 75, 16, 8, 128
    kp, vp = (torch.randn(shape, device=DEV).to(torch.bfloat16) for shape in ((250, kv_heads, 32, dh), (250, kv_heads, dh, 32)))
    table = t(rng.permutation(250)[None], torch.int32)
    qkv = torch.randn((n, heads * dh), device=DEV).to(torch.bfloat16)
    run = lambda first: ops.attention_prefill_bf16(qkv[first:], kp, vp, t([0, n - first], torch.int32), t(np.arange(first, n), torch.int32), table,
                                                   1, n - first, heads, kv_heads, dh, None, dh ** -0.5, cap)
    assert torch.equal(run(0)[n - last:], run(n - last))


@pytest.mark.parametrize("heads, kv_heads, dh", MFMA_SHAPES)
def test_mfma_decode_attention(ops, heads, kv_heads, dh):
    rng = np.random.default_rng(heads * 11 + dh)
    # lengths at and around page and chunk edges: 1, 32, 33, 256, 257, 512, 700
    lens = [1, 32, 33, 256, 257, 512, 700, 5]
    out, want = attention_case(ops, rng, lens, [1] * len(lens), heads, kv_heads, dh, torch.bfloat16, kernel="decode")
    close(out, want, BF16_OUT, "decode attention on the matrix cores")


@pytest.mark.parametrize("window", [None, 4500])
def test_mfma_decode_attention_over_thousands_of_keys(ops, window):
    """Past 16 chunks of 256 keys the chunks are joined in runs: sequences on both sides of that edge in one
    call, and in the longest a key that stands out, placed in the first run, in a middle one and in the last."""
    heads, kv_heads, dh = 4, 2, 64
    lens = [4096, 4097, 6000, 700]
    for far in (0, 2500, 5999):
        rng = np.random.default_rng(31 + far)

        def boost(qkv, k, kp, table, far=far):
            kf = f64(kp[table[2, far // 32].item(), 0, far % 32])          # sequence 2, kv head 0: query head 1
            qkv[2, dh:2 * dh] = 40.0 * kf / np.linalg.norm(kf) ** 2 * np.sqrt(dh)
        out, want = attention_case(ops, rng, lens, [1] * len(lens), heads, kv_heads, dh, torch.bfloat16,
                                   window=window, boost=boost, kernel="decode")
        close(out, want, BF16_OUT, f"far key {far}, window {window}")


def test_mfma_decode_attention_joins_more_chunks_than_a_run_fetches_at_once(ops):
    """One kv head and 40,000 keys: 157 chunks, too few workgroups to stream, joined in eight runs of 20 chunks,
    which a run fetches sixteen at a time.  A key that stands out among the first sixteen chunks of a run, among
    its last four, and in the sequence's last chunk; beside it a sequence of 20 chunks (runs of three)."""
    heads, kv_heads, dh = 2, 1, 32
    lens = [40000, 5000]
    assert not ops.decode_attention_streams(len(lens), kv_heads, max(lens) + 300)
    for far in (100, 256 * 18 + 7, 39990):
        rng = np.random.default_rng(61 + far)

        def boost(qkv, k, kp, table, far=far):
            kf = f64(kp[table[0, far // 32].item(), 0, far % 32])          # sequence 0, query head 1
            qkv[0, dh:2 * dh] = 40.0 * kf / np.linalg.norm(kf) ** 2 * np.sqrt(dh)
        out, want = attention_case(ops, rng, lens, [1] * len(lens), heads, kv_heads, dh, torch.bfloat16, boost=boost,
                                   kernel="decode")
        close(out, want, BF16_OUT, f"far key {far}")
        assert np.abs(want[0, 1]).max() > 0


@pytest.mark.parametrize("heads, kv_heads, dh, window", [(16, 8, 32, None), (16, 8, 32, 100), (16, 8, 32, 300),
                                                         (32, 8, 128, None), (32, 8, 128, 300), (8, 8, 64, None)])
def test_mfma_decode_attention_streams_over_many_sequences(ops, heads, kv_heads, dh, window):
    """From 512 (sequence, kv head) pairs on a workgroup walks a sequence's pages in one run and writes the
    output itself: 64 sequences with lengths at and around page and chunk edges, one of them with a key that
    stands out early in a long sequence."""
    rng = np.random.default_rng(77)
    lens = [1, 32, 33, 256, 257, 512, 700, 5, 1025, 2048, 2049, 31] + [int(n) for n in rng.integers(1, 1500, 52)]
    assert ops.decode_attention_streams(len(lens), kv_heads, max(lens) + 300)

    def boost(qkv, k, kp, table):
        head = 3 * (heads // kv_heads)                                 # sequence 9, kv head 3: its first query head
        kf = f64(kp[table[9, 40 // 32].item(), 3, 40 % 32])
        qkv[9, head * dh:(head + 1) * dh] = 40.0 * kf / np.linalg.norm(kf) ** 2 * np.sqrt(dh)
    out, want = attention_case(ops, rng, lens, [1] * len(lens), heads, kv_heads, dh, torch.bfloat16, window=window,
                               boost=boost, kernel="decode")
    close(out, want, BF16_OUT, f"streaming decode attention, window {window}")


WIDE_LENS = [1, 32, 33, 256, 257, 512, 700, 5, 1025, 1200, 1199, 31, 64, 1024, 300, 97,
             2, 63, 65, 100, 129, 255, 258, 400, 511, 513, 640, 767, 769, 900, 1000, 1100]


@pytest.mark.parametrize("heads, kv_heads, dh, window", [(16, 8, 32, None), (16, 8, 32, 100), (32, 8, 128, None),
                                                         (16, 8, 128, 300), (8, 8, 64, None)])
def test_mfma_decode_attention_streams_short_sequences_with_eight_wavefronts(ops, heads, kv_heads, dh, window):
    """Thirty-two sequences of eight kv heads and up to 1,200 keys: a run for every compute unit and none a second, and
    no sequence longer than sixteen chunks, is walked in one run by workgroups of eight wavefronts; some of the
    sequences have fewer pages than wavefronts."""
    if ops.compute_units() != 256:
        pytest.skip("the rule is written for the machine's size")
    rng = np.random.default_rng(78)
    assert ops.decode_attention_runs(len(WIDE_LENS), kv_heads, max(WIDE_LENS) + 300) == 1
    assert ops.decode_attention_runs(len(WIDE_LENS) - 7, kv_heads, max(WIDE_LENS) + 300) == 0
    assert ops.decode_attention_runs(len(WIDE_LENS), kv_heads, 4097) == 0
    assert ops.decode_attention_runs(len(WIDE_LENS) + 1, kv_heads, max(WIDE_LENS) + 300) == 0

    def boost(qkv, k, kp, table):
        head = 3 * (heads // kv_heads)                                 # sequence 9, kv head 3: its first query head
        kf = f64(kp[table[9, 40 // 32].item(), 3, 40 % 32])
        qkv[9, head * dh:(head + 1) * dh] = 40.0 * kf / np.linalg.norm(kf) ** 2 * np.sqrt(dh)
    out, want = attention_case(ops, rng, WIDE_LENS, [1] * len(WIDE_LENS), heads, kv_heads, dh, torch.bfloat16,
                               window=window, boost=boost, kernel="decode")
    close(out, want, BF16_OUT, f"eight wavefronts a run, window {window}")


@pytest.mark.parametrize("heads, kv_heads, dh, window", [(16, 8, 32, None), (16, 8, 32, 40), (32, 8, 128, None),
                                                         (16, 8, 128, 40), (128, 8, 64, None)])
def test_fused_decode_attention_streams_short_sequences_with_eight_wavefronts(ops, heads, kv_heads, dh, window):
    """The same from the raw projection (two query heads a wavefront to norm where a kv head has sixteen)."""
    if ops.compute_units() != 256:
        pytest.skip("the rule is written for the machine's size")
    assert ops.decode_attention_runs(len(WIDE_LENS), kv_heads, max(WIDE_LENS) + 301) == 1
    fused_decode_case(ops, heads, kv_heads, dh, window, WIDE_LENS, steps=2 if dh == 32 else 1, repeats=2 if dh == 32 else 1)


@pytest.mark.parametrize("window", [None, 4500])
def test_mfma_decode_attention_streams_long_sequences_in_runs(ops, window):
    """Long sequences with 64 (sequence, kv head) pairs and more are cut into 16 runs of whole chunks each, by
    their own lengths, and the runs are joined in order: sequences of every size in one call (most of a short
    one's runs are empty), and in the longest a key that stands out in the first run and in a late one."""
    heads, kv_heads, dh = 8, 8, 32
    lens = [16400, 700, 1, 4097, 257, 33, 9000, 2048]
    assert ops.decode_attention_streams(len(lens), kv_heads, max(lens) + 300)
    for far in (3, 15000):
        rng = np.random.default_rng(41 + far)

        def boost(qkv, k, kp, table, far=far):
            kf = f64(kp[table[0, far // 32].item(), 5, far % 32])          # sequence 0, kv head 5 = query head 5
            qkv[0, 5 * dh:6 * dh] = 40.0 * kf / np.linalg.norm(kf) ** 2 * np.sqrt(dh)
        out, want = attention_case(ops, rng, lens, [1] * len(lens), heads, kv_heads, dh, torch.bfloat16,
                                   window=window, boost=boost, kernel="decode")
        close(out, want, BF16_OUT, f"far key {far}, window {window}")


def test_mfma_decode_attention_streams_one_very_long_sequence(ops):
    """Two sequences, one of 66,000 keys: 33 runs each, joined in eight groups side by side; the short
    sequence's runs are empty but the first.  A key that stands out in the first run, in a middle one, in the
    last."""
    heads, kv_heads, dh = 8, 8, 32
    lens = [66000, 300]
    assert ops.decode_attention_streams(len(lens), kv_heads, max(lens) + 300)
    for far in (100, 33000, 65990):
        rng = np.random.default_rng(51 + far)

        def boost(qkv, k, kp, table, far=far):
            kf = f64(kp[table[0, far // 32].item(), 2, far % 32])          # sequence 0, kv head 2 = query head 2
            qkv[0, 2 * dh:3 * dh] = 40.0 * kf / np.linalg.norm(kf) ** 2 * np.sqrt(dh)
        out, want = attention_case(ops, rng, lens, [1] * len(lens), heads, kv_heads, dh, torch.bfloat16, boost=boost,
                                   kernel="decode")
        close(out, want, BF16_OUT, f"far key {far}")
        assert np.abs(want[0, 2]).max() > 0


@pytest.mark.parametrize("kernel", ["prefill", "decode"])
def test_mfma_attention_finds_one_far_key(ops, kernel):
    rng = np.random.default_rng(19)
    heads, kv_heads, dh = 8, 2, 128
    for far in (0, 3, 4, 31, 32, 255, 256, 511, 640, 699):
        def boost(qkv, k, kp, table, far=far):
            kf = f64(kp[table[0, far // 32].item(), 1, far % 32])          # kv head 1: query heads 4..7
            qkv[0, 6 * dh:7 * dh] = 40.0 * kf / np.linalg.norm(kf) ** 2 * np.sqrt(dh)
        out, want = attention_case(ops, rng, [700], [1], heads, kv_heads, dh, torch.bfloat16, boost=boost,
                                   kernel=kernel)
        close(out, want, BF16_ONE_KEY, f"far key {far}")
        vfar = f64(out[0, 6])
        assert np.abs(vfar - want[0, 6]).max() < 0.05


@pytest.mark.parametrize("kernel", ["prefill", "decode"])
@pytest.mark.parametrize("window", [1, 32, 33, 100, 256, 300])
def test_mfma_attention_window_edges(ops, kernel, window):
    rng = np.random.default_rng(window + 5)
    new = [1, 1] if kernel == "decode" else [34, 40]
    out, want = attention_case(ops, rng, [290, 40], new, 4, 2, 64, torch.bfloat16, window=window, kernel=kernel)
    close(out, want, BF16_OUT, f"window {window}")


@pytest.mark.parametrize("heads, kv_heads, dh", MFMA_SHAPES)
@pytest.mark.parametrize("window", [None, 40])
def test_fused_decode_attention(ops, heads, kv_heads, dh, window):
    """Norm, rotation, cache write and attention from the raw projection, against the plain parts; twice in
    a row on the same buffers, then one token further."""
    fused_decode_case(ops, heads, kv_heads, dh, window, [1, 32, 33, 256, 257, 512, 700, 5])


@pytest.mark.parametrize("heads, kv_heads, dh, window", [(16, 8, 32, None), (16, 8, 32, 40), (32, 8, 128, None),
                                                         (32, 8, 128, 40), (16, 8, 64, None)])
def test_fused_decode_attention_streams_over_many_sequences(ops, heads, kv_heads, dh, window):
    """The same from 512 (sequence, kv head) pairs on, where a workgroup walks a sequence's pages in one run,
    and the one whose run ends at the new token stores its key and value before any page is read."""
    rng = np.random.default_rng(3)
    lens = [1, 32, 33, 256, 257, 512, 700, 5, 31, 64, 65, 1000] + [int(n) for n in rng.integers(1, 600, 52)]
    assert ops.decode_attention_streams(len(lens), kv_heads, max(lens) + 301)
    fused_decode_case(ops, heads, kv_heads, dh, window, lens, steps=2 if dh == 32 else 1, repeats=2 if dh == 32 else 1)


@pytest.mark.parametrize("seqs, kv_heads", [(100, 8), (256, 2), (257, 2), (97, 7)])
def test_streams_that_share_a_compute_unit_take_every_sequence_once(ops, seqs, kv_heads):
    """Where two streams and more fall to a compute unit, the longest go out beside the shortest: rounds of
    workgroups that are not all full, equal lengths, and one sequence more than are ranked."""
    if ops.compute_units() not in (256, 1):
        pytest.skip("the sizes are for the machine's")
    rng = np.random.default_rng(seqs)
    lens = [40] * (seqs // 2) + [int(n) for n in rng.integers(1, 90, seqs - seqs // 2)]
    assert ops.decode_attention_runs(seqs, kv_heads, max(lens) + 300) == 1
    fused_decode_case(ops, 2 * kv_heads, kv_heads, 32, None, lens, steps=1, repeats=1)
    out, want = attention_case(ops, rng, lens, [1] * seqs, 2 * kv_heads, kv_heads, 32, torch.bfloat16, kernel="decode")
    close(out, want, BF16_OUT, f"{seqs} sequences of {kv_heads} heads")


@pytest.mark.parametrize("window", [None, 40])
def test_streams_that_share_a_compute_unit_and_their_ranks(ops, window):
    """Lengths that all differ, that are one for a half of the sequences and the rest longer or shorter, and that a window makes one; more
    sequences than a wavefront has lanes, the last length of all the longest."""
    if ops.compute_units() not in (256, 1):
        pytest.skip("the sizes are for the machine's")
    seqs, kv_heads = 130, 4
    assert ops.decode_attention_ranks(seqs, kv_heads, 400)
    for lens in ([1 + (37 * i) % 131 for i in range(seqs - 1)] + [200], [64] * 65 + [63] * 32 + [65] * 33, [48 + i % 2 for i in range(seqs)]):
        out, want = attention_case(ops, np.random.default_rng(1), lens, [1] * seqs, kv_heads, kv_heads, 32, torch.bfloat16, window,
                                   kernel="decode")
        close(out, want, BF16_OUT, f"{lens[:4]} ...")


def test_streams_are_ranked_where_their_walks_are_longer_than_the_look(ops):
    """Several streams a compute unit whose bound is more than one chunk of keys, up to 256 of them."""
    if ops.compute_units() != 256:
        pytest.skip("the sizes are for the machine's")
    ranks = ops.decode_attention_ranks
    assert ranks(64, 8, 257) and ranks(256, 8, 2000) and ranks(100, 8, 2000)
    assert not (ranks(256, 8, 256) or ranks(64, 8, 100) or ranks(32, 8, 2000) or ranks(257, 8, 2000) or ranks(1, 8, 100000))


@pytest.mark.parametrize("heads, kv_heads, dh", [(8, 8, 32), (32, 8, 128)])
def test_fused_decode_attention_streams_long_sequences_in_runs(ops, heads, kv_heads, dh):
    """And with long sequences cut into 16 runs each: the last run that is not empty holds the new token."""
    lens = [16400, 700, 1, 4097, 257, 33, 8191, 8192]
    assert ops.decode_attention_streams(len(lens), kv_heads, max(lens) + 301)
    fused_decode_case(ops, heads, kv_heads, dh, None, lens, steps=1, repeats=1)


def fused_decode_case(ops, heads, kv_heads, dh, window, lens, steps=2, repeats=2):
    """`lens`: the sequences' lengths after the first step."""
    rng = np.random.default_rng(heads * 13 + dh)
    B = len(lens)
    k, v, kp, vp, table = paged(rng, [n + 1 for n in lens], kv_heads, dh, dtype=torch.bfloat16, spare=12)
    width = (heads + 2 * kv_heads) * dh
    qg, kg = t(1 + 0.2 * rng.normal(size=dh)), t(1 + 0.2 * rng.normal(size=dh))
    theta, eps = 50000.0, 1e-5
    inv_freq = t(P.rope_inv_freq(dh, theta))
    for step in range(steps):
        cur = [n + step for n in lens]
        pos = [n - 1 for n in cur]
        raw = t(rng.normal(size=(B, width)) * 2, torch.bfloat16)
        raw64 = f64(raw)
        for repeat in range(repeats):
            out = ops.attention_decode_fused_bf16(raw, qg, kg, eps, inv_freq, kp, vp, t(pos, torch.int32), table, B,
                                                  max(cur) + 300, heads, kv_heads, dh, window, 1.0 / np.sqrt(dh))
            assert torch.equal(raw, t(raw64, torch.bfloat16)), "the projection is read, not changed"
            q = raw64[:, :heads * dh].reshape(B, heads, dh)
            kn = raw64[:, heads * dh:(heads + kv_heads) * dh].reshape(B, kv_heads, dh)
            vn = raw64[:, (heads + kv_heads) * dh:].reshape(B, kv_heads, dh)
            ang = P.rope_angles(pos, dh, theta)
            q = P.bf16_round(P.apply_rope(P.rms_norm(q, f64(qg), eps), ang).astype(np.float32)).astype(np.float64)
            kn = P.apply_rope(P.rms_norm(kn, f64(kg), eps), ang)
            tab = table.cpu().numpy()
            for b in range(B):
                page, off = tab[b, pos[b] // 32], pos[b] % 32
                close(kp[page, :, off], kn[b], BF16_OUT, "the new key in its page")
                assert np.array_equal(f64(vp[page, :, :, off]), vn[b]), "the new value in its page"
                kb = np.stack([f64(kp[tab[b, p // 32], :, p % 32]) for p in range(cur[b])])
                vb = np.stack([f64(vp[tab[b, p // 32], :, :, p % 32]) for p in range(cur[b])])
                want = P.attention(q[b:b + 1], kb, vb, window=window)
                close(out[b].reshape(1, heads, dh), want, BF16_TWICE, f"sequence {b}, step {step}, repeat {repeat}")


def test_mfma_and_generic_attention_agree(ops):
    """The same call through all three kernels: decode against prefill against generic."""
    outs = []
    for kernel in ("generic", "prefill", "decode"):
        rng = np.random.default_rng(23)
        out, want = attention_case(ops, rng, [400, 77, 1], [1, 1, 1], 8, 2, 128, torch.bfloat16, kernel=kernel)
        outs.append(f64(out))
    assert np.abs(outs[0] - outs[1]).max() < 2e-2 and np.abs(outs[1] - outs[2]).max() < 2e-2


@pytest.mark.parametrize("w_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 9, 130])
def test_gemm_f32(ops, w_dtype, m):
    # sizes of the reference's own linear test (src/cpu/linear.rs:634-647): n = 37, k = 70
    rng = np.random.default_rng(m)
    x, w = t(rng.normal(size=(m, 70))), t(rng.normal(size=(37, 70)), w_dtype)
    close(ops.gemm_f32(x, w), f64(x) @ f64(w).T, 2e-6, "gemm_f32")


def test_gemm_f32_rows_do_not_depend_on_the_batch(ops):
    rng = np.random.default_rng(1)
    x, w = t(rng.normal(size=(100, 333))), t(rng.normal(size=(129, 333)))
    whole = ops.gemm_f32(x, w)
    assert torch.equal(whole[17:18], ops.gemm_f32(x[17:18].contiguous(), w))
    assert torch.equal(whole[60:], ops.gemm_f32(x[60:].contiguous(), w))


@pytest.mark.parametrize("m,n,k", [(1, 37, 72), (33, 129, 192), (65, 130, 64), (65, 16500, 72), (33, 4100, 136),
                                   (33, 129, 256), (65, 130, 128), (70, 40, 512), (33, 4100, 256)])
def test_gemm_f32_on_the_matrix_cores(ops, m, n, k):
    """bfloat16 weights: edges of the tiles of 32 and 64 rows, 32 to 128 columns and stages of 64 k, whole turns of stages among them (no part
    of one is masked then), values over many orders of magnitude.  An additions' chain of k / 32 steps and 32 products a step: (k / 32 + 32) half units of 2^-24 of the sum of
    magnitudes at most."""
    if EMULATED and n > 1000:
        pytest.skip("the larger tiles run on the emulated machine of one unit, at small sizes")
    rng = np.random.default_rng(m + n + k)
    x, w = t(rng.normal(size=(m, k)) * 10.0 ** rng.uniform(-6, 6, size=(m, k))), t(rng.normal(size=(n, k)), torch.bfloat16)
    got = f64(ops.gemm_f32(x, w))
    bound = (k / 32 + 32) * 2.0 ** -24 * (np.abs(f64(x)) @ np.abs(f64(w)).T)
    assert (np.abs(got - f64(x) @ f64(w).T) <= bound).all()
    some = ops.gemm_f32(x[m // 2:].contiguous(), w)
    assert np.array_equal(got[m // 2:], f64(some)), "a row's sums depend on the other rows"


@pytest.mark.parametrize("m,n,k", [(385, 4096, 200), (1153, 4096, 64), (1200, 4096, 392), (31, 4096, 328), (385, 4096, 256), (1153, 4096, 1024),
                                   (31, 4096, 512)])
def test_gemm_f32_tiles_of_a_full_machine(ops, m, n, k):
    """The tiles of 64 x 128 that a whole machine chooses, their edges and stages, whole and not, and the smallest ones' four stages;
    the bound of the test above."""
    rng = np.random.default_rng(m + n + k)
    x, w = t(rng.normal(size=(m, k))), t(rng.normal(size=(n, k)), torch.bfloat16)
    got = f64(ops.gemm_f32(x, w))
    bound = (k / 32 + 32) * 2.0 ** -24 * (np.abs(f64(x)) @ np.abs(f64(w)).T)
    assert (np.abs(got - f64(x) @ f64(w).T) <= bound).all()
    assert np.array_equal(got[m - 30:], f64(ops.gemm_f32(x[m - 30:].contiguous(), w))), "a row's sums depend on the other rows"


@pytest.mark.parametrize("tile", range(3, 7))
@pytest.mark.parametrize("m,n,k", [(1, 8, 64), (130, 164, 128), (67, 60, 192), (128, 160, 448)])
def test_gemm_f32_in_tiles_copied_as_they_are(ops, m, n, k, tile):
    """Edges of the tiles whose x is split out of LDS, fewer stages of 64 k than buffers and more: the bits of the smallest tile, also
    where an infinity leaves the matrix cores' sums without a value.  (That tile against 64 bits: above.)"""
    rng = np.random.default_rng(m + n + k)
    x, w = t(rng.normal(size=(m, k)) * 10.0 ** rng.uniform(-6, 6, size=(m, k))), t(rng.normal(size=(n, k)), torch.bfloat16)
    x[m // 2, k - 1] = float("inf")
    assert np.array_equal(f64(ops.gemm_f32(x, w, tile)), f64(ops.gemm_f32(x, w, 2)), equal_nan=True)


@pytest.mark.parametrize("m, n", [(5, 48), (70, 72)])
def test_gemm_f32_where_the_first_parts_cancel(ops, m, n):
    """Pairs of k with opposite weights and x that agree in their first eight bits: what is left are the lower parts' products, whose sum is
    rounded once for each of the S = K / 32 steps of the second part.  A rounding errs by some 2.5e-8 of the partial sum, which after s steps is
    sqrt(s / S) of the result (2-norm): sqrt(S / 2) 2.5e-8 = 1.0e-7 at K = 1,024, and more within the steps (1.75e-7 measured); the third
    part's additions in the same sum make it sqrt(2) as much (2.65e-7 measured)."""
    rng = np.random.default_rng(m)
    k = 1024
    top = rng.normal(size=(m, k // 2)).astype(np.float32).view(np.uint32) & np.uint32(0xFFFF0000)
    x = np.repeat(top, 2, 1) | rng.integers(0, 1 << 16, (m, k), dtype=np.uint32)
    w = np.repeat(rng.normal(size=(n, k // 2)), 2, 1) * np.where(np.arange(k) % 2, -1.0, 1.0)
    x, w = t(x.view(np.float32)), t(w, torch.bfloat16)
    want = f64(x) @ f64(w).T
    error = np.linalg.norm(f64(ops.gemm_f32(x, w)) - want) / np.linalg.norm(want)
    assert error <= 2.2e-7, error


@pytest.mark.parametrize("top", [-100, -112, -118, -126, -135])
def test_gemm_f32_of_the_smallest_numbers(ops, top):
    """x down to the smallest float32, subnormal numbers among them: no bit of it is lost.  The bound of the test above, and half the
    smallest float32 for every one of the products and additions that may end among the subnormal numbers."""
    rng = np.random.default_rng(-top)
    m, n, k = 33, 40, 136
    x = t(np.ldexp(rng.choice([-1.0, 1.0], (m, k)) * rng.uniform(1, 2, (m, k)), rng.integers(top - 8, top + 1, (m, k))))
    w = t(rng.normal(size=(n, k)), torch.bfloat16)
    got = f64(ops.gemm_f32(x, w))
    bound = (k / 32 + 32) * 2.0 ** -24 * (np.abs(f64(x)) @ np.abs(f64(w)).T) + 3 * 2 * k * 2.0 ** -150
    assert (np.abs(got - f64(x) @ f64(w).T) <= bound).all()


def test_gemm_f32_infinities_and_nan(ops):
    """Numbers that have no parts: the row of x and the column of the weights they stand in become what multiply-adds make of them."""
    rng = np.random.default_rng(3)
    x, w = t(rng.normal(size=(40, 136))), t(rng.normal(size=(50, 136)), torch.bfloat16)
    clean = f64(ops.gemm_f32(x, w))
    x[3, 7], x[4, 9], x[5, 0], w[6, 11] = float("inf"), float("nan"), 3.4e38, float("-inf")
    got, want = f64(ops.gemm_f32(x, w)), f64(x) @ f64(w).T
    rows, cols = [i for i in range(40) if i not in (3, 4, 5)], [j for j in range(50) if j != 6]
    assert np.array_equal(got[np.ix_(rows, cols)], clean[np.ix_(rows, cols)])
    assert np.array_equal(got[3, cols], want[3, cols]) and np.isnan(got[4]).all()
    assert np.array_equal(np.isnan(got[:, 6]), np.isnan(want[:, 6])) and not np.isfinite(got[:, 6]).any()
    big = np.abs(want[5, cols]) < 3e38
    assert np.allclose(got[5, cols][big], want[5, cols][big], rtol=1e-5)


def test_gemm_f32_is_true_32_bit(ops):
    """Values that a reduced-precision matrix mode (tf32, bf16 inputs) would round away."""
    x = t([[1.0, 2.0 ** -12, 0.0, 0.0]]).repeat(1, 16)
    w = t([[1.0, 1.0, 0.0, 0.0]]).repeat(1, 16)
    assert ops.gemm_f32(x, w).item() == 16.0 * (1.0 + 2.0 ** -12)


@pytest.mark.parametrize("k", [8, 504, 512, 520, 1024, 1032, 1536, 2568, 3072, 3584, 4088, 4096, 4104, 4616, 5120, 5128])
def test_gemv_of_one_row_whole(ops, k):
    """One row of x and rows of w that a wavefront asks for whole, one to ten pieces of 512, and the first size past them: the bits of that row
    beside another, rows past the edge, a weight that is no number behind the row's end left alone."""
    rng = np.random.default_rng(k)
    x = t(rng.normal(size=(2, k)), torch.bfloat16)
    for n in (1, 4, 37):
        w = t(rng.normal(size=(n, k)), torch.bfloat16)
        for out_dtype in (torch.float32, torch.bfloat16):
            got = ops.gemv_bf16(x[:1].contiguous(), w, out_dtype)
            assert torch.equal(got, ops.gemv_bf16(x, w, out_dtype)[:1])
        close(got, f64(x[:1]) @ f64(w).T, 5e-3, "one row")
        pair = torch.cat([w, w.flip(0)])
        assert torch.equal(ops.gemv_bf16(x[:1].contiguous(), pair, swiglu=True), ops.gemv_bf16(x, pair, swiglu=True)[:1])
    w[-1, -1] = float("inf")
    got = ops.gemv_bf16(x[:1].contiguous(), w, torch.float32)
    assert torch.isfinite(got[0, :-1]).all() and torch.equal(got, ops.gemv_bf16(x, w, torch.float32)[:1])


@pytest.mark.parametrize("k, n", [(1024, 37), (1024, 1032), (2560, 96), (4104, 40), (5120, 8)])
@pytest.mark.parametrize("n_in", [1, 256, 300, 1281])
def test_linked_product_of_one_row_whole(ops, k, n, n_in):
    """The norm before it from any number of partial sums of squares, and the stream's sum and the next norm's preparation after it."""
    rng = np.random.default_rng(n + n_in)
    xg, ssq = t(rng.normal(size=(1, k)), torch.bfloat16), t(rng.uniform(0.5, 1.5, size=(1, n_in)) * k / n_in)
    w, residual, gain = t(rng.normal(size=(n, k)) / np.sqrt(k), torch.bfloat16), t(rng.normal(size=(1, n))), t(rng.normal(size=(n,)))
    y = f64(xg) @ f64(w).T / np.sqrt(f64(ssq).sum() / k + 1e-6)
    later = ops.NormedLater(xg, ssq, 1e-6, k)
    close(ops.linked_product(later, w, n, False, torch.float32), y, 2e-6, "normed")
    total = residual.clone()
    made = ops.linked_product(later, w, n, False, residual=total, next_gain=gain, next_eps=1e-6)
    want = f64(residual) + y
    close(total, want, 2e-6, "the stream")
    close(made.xg, want * f64(gain), 5e-3, "the next rows")
    close(made.ssq.sum(1), (want ** 2).sum(1), 1e-5, "sums of squares")


@pytest.mark.parametrize("m", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [584, 2560, 1544, 2048, 9728])      # steps of 512: one and a bit, five, three and a bit, four, nineteen
def test_gemv_bf16(ops, m, out_dtype, k):
    rng = np.random.default_rng(m)
    x, w = t(rng.normal(size=(m, k)), torch.bfloat16), t(rng.normal(size=(37, k)), torch.bfloat16)
    want = f64(x) @ f64(w).T
    close(ops.gemv_bf16(x, w, out_dtype), want, 2e-6 if out_dtype == torch.float32 else 5e-3, "gemv")
    wgu = t(rng.normal(size=(2 * 45, k)) * 0.1, torch.bfloat16)
    y = f64(x) @ f64(wgu).T
    close(ops.gemv_bf16(x, wgu, out_dtype, swiglu=True), P.silu(y[:, :45]) * y[:, 45:],
          3e-6 if out_dtype == torch.float32 else 5e-3, "gemv with swiglu")
    # a row's result does not depend on the other rows
    if m > 1:
        assert torch.equal(ops.gemv_bf16(x, w, out_dtype)[m - 1:], ops.gemv_bf16(x[m - 1:].contiguous(), w, out_dtype))


@pytest.mark.parametrize("m", [1, 3, 8, 16])
@pytest.mark.parametrize("n, k", [(37, 584), (100, 96), (4096, 4096), (50, 12288), (320, 104),
                                  (96, 2560), (48, 9728)])       # K whose share of a wavefront is no whole round of 8 steps
def test_gemm_skinny_packed_bf16(ops, m, n, k):
    rng = np.random.default_rng(m + n)
    x, w = t(rng.normal(size=(m, k)), torch.bfloat16), t(rng.normal(size=(n, k)), torch.bfloat16)
    want = f64(x) @ f64(w).T
    packed = ops.pack_for_mfma(w)
    close(ops.gemm_skinny_packed_bf16(x, packed, n, torch.float32), want, 3e-6, "packed skinny product")
    # a row's result does not depend on the other rows
    if m > 1:
        assert torch.equal(ops.gemm_skinny_packed_bf16(x, packed, n, torch.float32)[m - 1:],
                           ops.gemm_skinny_packed_bf16(x[m - 1:].contiguous(), packed, n, torch.float32))
    wgu = t(rng.normal(size=(2 * n, k)) * (4.0 / np.sqrt(k)), torch.bfloat16)
    y = f64(x) @ f64(wgu).T
    close(ops.gemm_skinny_packed_bf16(x, ops.pack_for_mfma(wgu, swiglu=True), n, torch.bfloat16, swiglu=True),
          P.silu(y[:, :n]) * y[:, n:], 5e-3, "packed, with swiglu")
    for parts in (2, 3):                                   # K cut in pieces: the pieces add up to the product
        got = ops.gemm_skinny_packed_bf16(x, packed, n, torch.float32, parts=parts)
        assert got.shape == (parts, m, n)
        close(got.sum(0), want, 3e-6, f"{parts} parts of K")


@pytest.mark.parametrize("m", [1, 2, 8, 9, 16])
@pytest.mark.parametrize("n, k", [(37, 72), (512, 1024), (1000, 264), (48, 8192)])
def test_packed_products_of_one_size_in_one_launch(ops, m, n, k):
    """The bits of a launch each, over both numbers of wavefronts, edges of the row tiles and of K."""
    rng = np.random.default_rng(m + n)
    x = t(rng.normal(size=(3, m, k)), torch.bfloat16)
    packed = torch.stack([ops.pack_for_mfma(t(rng.normal(size=(n, k)), torch.bfloat16)) for _ in range(3)])
    for out_dtype in (torch.float32, torch.bfloat16):
        got = ops.gemm_skinny_batch(x, packed, n, out_dtype)
        for i in range(3):
            assert torch.equal(got[i], ops.gemm_skinny_packed_bf16(x[i], packed[i], n, out_dtype))


@pytest.mark.parametrize("m", [1, 16, 17, 33, 40, 49, 64])
@pytest.mark.parametrize("n, k", [(37, 72), (1000, 1024), (584, 12288), (4096, 4096), (70, 264)])
def test_wide_packed_product(ops, m, n, k):
    """The product for steps of 17 to 64 tokens: whole, in parts of K that add up, with the activation, from and
    into rows in the matrix cores' order; and a row's result does not depend on how many rows there are."""
    rng = np.random.default_rng(m + n + k)
    x, w = t(rng.normal(size=(m, k)), torch.bfloat16), t(rng.normal(size=(n, k)), torch.bfloat16)
    want = f64(x) @ f64(w).T
    packed = ops.pack_for_mfma(w)
    whole = ops.gemm_wide_packed_bf16(x, packed, n, torch.float32)
    close(whole, want, 3e-6, "wide product")
    close(ops.gemm_wide_packed_bf16(x, packed, n, torch.bfloat16), want, 5e-3, "wide product, bfloat16 out")
    for parts in (2, 3, ops.wide_product_plan(n, k, rows=m)[1]):
        got = ops.gemm_wide_packed_bf16(x, packed, n, torch.float32, parts=parts)
        assert got.shape == ((parts, m, n) if parts > 1 else (m, n))
        if parts > 1:
            close(got.sum(0), want, 3e-6, f"{parts} parts of K")
            close(ops.sum_parts(got, torch.float32), want, 3e-6, "parts added by the kernel")
            assert torch.equal(ops.sum_parts(got, torch.bfloat16, tiled_out=True).rows(), ops.sum_parts(got, torch.bfloat16))
    wgu = t(rng.normal(size=(2 * n, k)) * (4.0 / np.sqrt(k)), torch.bfloat16)
    y = f64(x) @ f64(wgu).T
    pgu = ops.pack_for_mfma(wgu, swiglu=True)
    close(ops.gemm_wide_packed_bf16(x, pgu, n, torch.bfloat16, swiglu=True), P.silu(y[:, :n]) * y[:, n:], 5e-3,
          "wide, with swiglu")
    raw = ops.gemm_wide_packed_bf16(x, pgu, n, torch.float32, swiglu=True, parts=2)        # the activation after the parts
    assert raw.shape == (2, m, 2 * n)
    close(ops.sum_parts(raw, torch.float32, swiglu=True), P.silu(y[:, :n]) * y[:, n:], 5e-6, "swiglu over parts")
    assert torch.equal(ops.gemm_wide_packed_bf16(x, packed, n, torch.float32, depth=1), whole)    # the same sums either way
    # three row tiles a workgroup instead of four: the same sums again, whole, in parts and with the activation
    assert torch.equal(ops.gemm_wide_packed_bf16(x, packed, n, torch.float32, waves=3), whole)
    assert torch.equal(ops.gemm_wide_packed_bf16(x, packed, n, torch.float32, parts=3, waves=3, depth=1),
                       ops.gemm_wide_packed_bf16(x, packed, n, torch.float32, parts=3))
    assert torch.equal(ops.gemm_wide_packed_bf16(x, pgu, n, torch.bfloat16, swiglu=True, waves=3, tiled_out=True).rows(),
                       ops.gemm_wide_packed_bf16(x, pgu, n, torch.bfloat16, swiglu=True))
    # five to eight wavefronts a workgroup (matrices of more than a thousand pairs of row tiles): the same bits
    gated = ops.gemm_wide_packed_bf16(x, pgu, n, torch.bfloat16, swiglu=True, depth=1)
    for many in (5, 6, 7, 8):
        assert torch.equal(ops.gemm_wide_packed_bf16(x, pgu, n, torch.bfloat16, swiglu=True, depth=1, waves=many), gated)
    assert torch.equal(ops.gemm_wide_packed_bf16(x, pgu, n, torch.bfloat16, swiglu=True, depth=1, waves=7, tiled_out=True).rows(), gated)
    with pytest.raises(Exception, match="wavefronts"):
        ops.gemm_wide_packed_bf16(x, packed, n, torch.float32, waves=5)
    waves, parts = ops.wide_product_plan(n, k, True)
    assert 3 <= waves <= 8 and parts == 1                   # the activation is never left to a second kernel
    assert ops.wide_product_plan(16 * 4 * ops.compute_units() + 16, k, True) == (5, 1)
    assert ops.wide_product_plan(16 * 7 * ops.compute_units(), k, True) == (7, 1)
    # rows in the matrix cores' order on either side: the same bits
    tiled = ops.sum_parts(x.float()[None].contiguous(), torch.bfloat16, tiled_out=True)
    assert torch.equal(tiled.rows(), x)
    assert torch.equal(ops.gemm_wide_packed_bf16(tiled, packed, n, torch.float32), whole)
    assert torch.equal(ops.gemm_wide_packed_bf16(x, packed, n, torch.bfloat16, tiled_out=True).rows(),
                       ops.gemm_wide_packed_bf16(x, packed, n, torch.bfloat16))
    if m > 1:
        assert torch.equal(whole[m - 1:], ops.gemm_wide_packed_bf16(x[m - 1:].contiguous(), packed, n, torch.float32))


@pytest.mark.parametrize("m", [1, 16, 17, 33, 49, 64])
@pytest.mark.parametrize("n, k", [(37, 72), (1000, 1024), (5137, 264), (320, 136)])
def test_product_with_many_row_tiles_a_workgroup(ops, m, n, k):
    """Six, eight and twelve row tiles a workgroup and ten pairs of them, x in half slices: edges of the groups, of a pair, of the slices and of
    four sums a store; the same bits as four row tiles, from rows in either order."""
    rng = np.random.default_rng(m + n + k)
    x, w = t(rng.normal(size=(m, k)), torch.bfloat16), t(rng.normal(size=(n, k)), torch.bfloat16)
    packed = ops.pack_for_mfma(w)
    tiled = ops.sum_parts(x.float()[None].contiguous(), torch.bfloat16, tiled_out=True)
    whole = ops.gemm_wide_packed_bf16(x, packed, n, torch.float32, depth=1)
    close(whole, f64(x) @ f64(w).T, 3e-6, "wide product")
    rounded = ops.gemm_wide_packed_bf16(x, packed, n, torch.bfloat16, depth=1)
    for waves in (6, 8, 12, 20):
        for rows in (x, tiled):
            assert torch.equal(ops.gemm_wide_packed_bf16(rows, packed, n, torch.float32, depth=1, waves=waves), whole)
            assert torch.equal(ops.gemm_wide_packed_bf16(rows, packed, n, torch.bfloat16, depth=1, waves=waves), rounded)
        if waves < 20:
            assert torch.equal(ops.gemm_wide_packed_bf16(x, packed, n, torch.bfloat16, depth=1, waves=waves, tiled_out=True).rows(), rounded)
        with pytest.raises(Exception, match="wavefronts"):
            ops.gemm_wide_packed_bf16(x, packed, n, torch.float32, parts=2, depth=1, waves=waves)
    with pytest.raises(Exception, match="wavefronts"):
        ops.gemm_wide_packed_bf16(x, packed, n, torch.bfloat16, depth=1, waves=20, tiled_out=True)


@pytest.mark.parametrize("m", [65, 80, 81, 100, 113, 128, 129, 150, 200, 256])
@pytest.mark.parametrize("n, k", [(37, 72), (1000, 1024), (584, 12288), (4096, 4096), (70, 264), (16, 520)])
def test_wide_packed_product_of_65_to_256_rows(ops, m, n, k):
    """Five to eight tiles of x, two row tiles of the matrix a wavefront (an odd number of row tiles leaves the last
    wavefront one), past 128 rows in two passes (129 rows: five tiles and four): whole and in parts of K that add up,
    with three and four wavefronts a workgroup; a row's sums are those of the kernel for up to 64 rows, bit for bit."""
    rng = np.random.default_rng(m + n + k)
    x, w = t(rng.normal(size=(m, k)), torch.bfloat16), t(rng.normal(size=(n, k)), torch.bfloat16)
    want = f64(x) @ f64(w).T
    packed = ops.pack_for_mfma(w)
    whole = ops.gemm_wide_packed_bf16(x, packed, n, torch.float32)
    assert whole.shape == (m, n)
    close(whole, want, 3e-6, "wide product of more than 64 rows")
    waves, planned = ops.wide_product_plan(n, k, rows=m)
    assert waves in (3, 4) and planned >= 1
    for parts in (2, 3, planned):
        got = ops.gemm_wide_packed_bf16(x, packed, n, torch.float32, parts=parts, waves=waves)
        assert got.shape == ((parts, m, n) if parts > 1 else (m, n))
        if parts > 1:
            close(got.sum(0), want, 3e-6, f"{parts} parts of K")
        assert torch.equal(got, ops.gemm_wide_packed_bf16(x, packed, n, torch.float32, parts=parts, waves=7 - waves))
        first = ops.gemm_wide_packed_bf16(x[:64].contiguous(), packed, n, torch.float32, parts=parts, depth=1)
        last = ops.gemm_wide_packed_bf16(x[m - 1:].contiguous(), packed, n, torch.float32, parts=parts, depth=1)
        assert torch.equal(got[..., :64, :], first) and torch.equal(got[..., m - 1:, :], last)
    if m <= 128:        # with the activation, five to eight wavefronts a workgroup: the bits of the kernel for 64 rows
        wgu = t(rng.normal(size=(2 * n, k)) * (4.0 / np.sqrt(k)), torch.bfloat16)
        y = f64(x) @ f64(wgu).T
        pgu = ops.pack_for_mfma(wgu, swiglu=True)
        gated = ops.gemm_wide_packed_bf16(x, pgu, n, torch.bfloat16, swiglu=True, waves=5)
        close(gated, P.silu(y[:, :n]) * y[:, n:], 5e-3, "more than 64 rows with the activation")
        for many in (6, 7, 8):
            assert torch.equal(ops.gemm_wide_packed_bf16(x, pgu, n, torch.bfloat16, swiglu=True, waves=many), gated)
        assert torch.equal(gated[:64], ops.gemm_wide_packed_bf16(x[:64].contiguous(), pgu, n, torch.bfloat16, swiglu=True, depth=1))
        with pytest.raises(Exception, match="wavefronts"):
            ops.gemm_wide_packed_bf16(x, pgu, n, torch.bfloat16, swiglu=True, waves=4)
    with pytest.raises(Exception, match="64"):
        ops.gemm_wide_packed_bf16(x, packed, n, torch.bfloat16)
    with pytest.raises(Exception, match="256"):
        ops.gemm_wide_packed_bf16(t(rng.normal(size=(257, k)), torch.bfloat16), packed, n, torch.float32)


@pytest.mark.parametrize("packed, m", [(False, 1), (False, 2), (False, 5), (True, 1), (True, 3), (True, 16)])
@pytest.mark.parametrize("hidden, k, inter", [(104, 72, 56), (4096, 4096, 1000), (584, 12288, 37)])
def test_products_linked_to_norms(ops, packed, m, hidden, k, inter):
    """A branch's last product adds into the residual stream and prepares the next RMSNorm; the
    product after it finishes that norm.  Checked against add, norm and products done one by one."""
    rng = np.random.default_rng(m + hidden)
    eps = 1e-5
    x = t(rng.normal(size=(m, k)), torch.bfloat16)
    w_out = t(rng.normal(size=(hidden, k)) / np.sqrt(k), torch.bfloat16)
    r0 = t(rng.normal(size=(m, hidden)) * 3)
    gain = t(1 + 0.3 * rng.normal(size=hidden))
    w_next = t(rng.normal(size=(inter, hidden)), torch.bfloat16)
    w_gu = t(rng.normal(size=(2 * inter, hidden)) * (4.0 / np.sqrt(hidden)), torch.bfloat16)
    prep = (lambda w, **kw: ops.pack_for_mfma(w, **kw)) if packed else (lambda w, **kw: w)

    r1 = f64(r0) + f64(x) @ f64(w_out).T
    residual = guarded(r0.clone())
    later = ops.linked_product(x, prep(w_out), hidden, packed, residual=residual, next_gain=gain, next_eps=eps)
    close(residual, r1, 3e-6, "residual after the linked product")
    close(later.xg, f64(residual) * f64(gain), 4e-3, "rows times gain")       # one rounding to bfloat16
    close(later.ssq.sum(1), (f64(residual) ** 2).sum(1), 1e-5, "sums of squares")
    assert later.dim == hidden and later.eps == eps
    # a second call leaves the same partial sums: they do not depend on scheduling
    again = ops.linked_product(x, prep(w_out), hidden, packed, residual=guarded(r0.clone()), next_gain=gain, next_eps=eps)
    assert torch.equal(again.ssq, later.ssq) and torch.equal(again.xg, later.xg)

    normed = P.rms_norm(f64(residual), f64(gain), eps)
    close(ops.linked_product(later, prep(w_next), inter, packed, torch.float32), normed @ f64(w_next).T, 6e-3,
          "product that finishes the norm")
    y = normed @ f64(w_gu).T
    close(ops.linked_product(later, prep(w_gu, swiglu=True) if packed else w_gu, inter, packed, torch.bfloat16,
                             swiglu=True), P.silu(y[:, :inter]) * y[:, inter:], BF16_TWICE, "the same with swiglu")
    # both sides at once: the next branch's product reads prepared rows and prepares the following norm
    w_back = t(rng.normal(size=(hidden, hidden)) / np.sqrt(hidden), torch.bfloat16)
    r2 = f64(residual) + normed @ f64(w_back).T
    chained = ops.linked_product(later, prep(w_back), hidden, packed, residual=residual, next_gain=gain, next_eps=eps)
    close(residual, r2, 6e-3, "residual after two linked products")
    close(chained.ssq.sum(1), (f64(residual) ** 2).sum(1), 1e-5, "sums of squares, second link")


@pytest.mark.parametrize("m", [1, 17, 32, 33, 41, 48, 50, 64])
@pytest.mark.parametrize("n, k", [(37, 72), (1000, 1024), (584, 12288)])
def test_packed_product_of_17_to_64_rows(ops, m, n, k):
    rng = np.random.default_rng(m + n)
    x = t(rng.normal(size=(m, k)), torch.bfloat16)
    w = t(rng.normal(size=(n, k)) / np.sqrt(k), torch.bfloat16)
    gu = t(rng.normal(size=(2 * n, k)) * (4.0 / np.sqrt(k)), torch.bfloat16)
    pw, pgu = ops.pack_for_mfma(w), ops.pack_for_mfma(gu, swiglu=True)
    out = ops.gemm_mid_packed_bf16(x, pw, n, torch.float32)
    close(out, f64(x) @ f64(w).T, 2e-5, "packed product, 17 to 64 rows")
    y = f64(x) @ f64(gu).T
    close(ops.gemm_mid_packed_bf16(x, pgu, n, torch.bfloat16, swiglu=True), P.silu(y[:, :n]) * y[:, n:], BF16_OUT,
          "the same with swiglu")
    # a row's result is the same whatever the number of rows, and the same as the kernel for up to 16 rows gives
    first = min(m, 16)
    assert torch.equal(out[:first], ops.gemm_skinny_packed_bf16(x[:first].contiguous(), pw, n, torch.float32))
    with pytest.raises(Exception, match="1 to 64"):
        ops.gemm_mid_packed_bf16(t(rng.normal(size=(65, k)), torch.bfloat16), pw, n)


@pytest.mark.parametrize("m", [1, 16, 17, 40, 64])
@pytest.mark.parametrize("dim, n", [(104, 56), (4096, 1000), (584, 40)])
def test_every_maker_of_rows_can_tile_them(ops, m, dim, n):
    """The norm, the decode attention and the product for 17 to 64 rows write their rows in the matrix cores'
    order on request, bit for bit the rows they write plainly; the products read them so."""
    rng = np.random.default_rng(5 * m + dim)
    residual = t(rng.normal(size=(m, dim)) * 2)
    pending = t(rng.normal(size=(m, dim)), torch.bfloat16)
    gain = t(1 + 0.2 * rng.normal(size=dim))
    plain = ops.add_rmsnorm(guarded(residual.clone()), pending, gain, 1e-5, torch.bfloat16)
    r2 = guarded(residual.clone())
    tiled = ops.add_rmsnorm(r2, pending, gain, 1e-5, torch.bfloat16, tiled=True)
    assert isinstance(tiled, ops.TiledRows) and tiled.shape == (m, dim) and torch.equal(tiled.rows(), plain)
    close(r2, f64(residual) + f64(pending), 1e-6, "the sum is written back either way")
    # into the products: the one for 17 to 64 rows takes fewer too
    pw = ops.pack_for_mfma(t(rng.normal(size=(n, dim)) / np.sqrt(dim), torch.bfloat16))
    pgu = ops.pack_for_mfma(t(rng.normal(size=(2 * n, dim)) * (4.0 / np.sqrt(dim)), torch.bfloat16), swiglu=True)
    want = ops.gemm_mid_packed_bf16(plain, pw, n)
    assert torch.equal(ops.gemm_mid_packed_bf16(tiled, pw, n), want)
    out_tiled = ops.gemm_mid_packed_bf16(tiled, pw, n, tiled_out=True)
    assert isinstance(out_tiled, ops.TiledRows) and torch.equal(out_tiled.rows(), want)
    assert torch.equal(ops.gemm_mid_packed_bf16(tiled, pgu, n, swiglu=True, tiled_out=True).rows(),
                       ops.gemm_mid_packed_bf16(plain, pgu, n, swiglu=True))
    if m <= 16:
        assert torch.equal(ops.gemm_skinny_packed_bf16(tiled, pw, n), want)
    with pytest.raises(Exception, match="64"):
        ops.add_rmsnorm(t(rng.normal(size=(65, dim))), None, gain, 1e-5, torch.bfloat16, tiled=True)


def test_streaming_attention_walks_a_run_of_more_pages_than_it_holds_table_entries_for(ops):
    """A wavefront of the streaming kernel fetches the page table's entries for 256 of its pages at a time; a run
    of more than 1,024 pages (32,768 keys) goes round that loop again.  64 sequences of one kv head each side of
    that length, eight kv heads (512 runs: one a sequence and kv head), against the generic kernel on the same
    pages; the sequences are of unequal length and one key far back in one of them gets a score that stands out."""
    heads, kv_heads, dh, B = 8, 8, 32, 64
    gen = torch.Generator(device=DEV).manual_seed(3)
    lens = [33_000 + 37 * b for b in range(B)]
    lens[5] = 40_000
    pages_per = [-(-n // 32) for n in lens]
    width = max(pages_per)
    num_pages = sum(pages_per)
    assert ops.decode_attention_runs(B, kv_heads, max(lens)) == 1
    kp = torch.randn((num_pages, kv_heads, 32, dh), device=DEV, generator=gen).to(torch.bfloat16)
    vp = torch.randn((num_pages, kv_heads, dh, 32), device=DEV, generator=gen).to(torch.bfloat16)
    order = torch.randperm(num_pages, device=DEV, generator=gen).to(torch.int32)
    table = torch.zeros((B, width), dtype=torch.int32, device=DEV)
    at = 0
    for b, n in enumerate(pages_per):
        table[b, :n] = order[at:at + n]
        at += n
    qkv = torch.randn((B, (heads + 2 * kv_heads) * dh), device=DEV, generator=gen).to(torch.bfloat16)
    # Queries that are a multiple of one far key, so that the output is that key's value: a key among a
    # wavefront's first 256 pages (position 9,000 of sequence 5) and keys among its later ones (pages from 1,024
    # on: position 39,990 of sequence 5, a key of sequence 9's last pages and one of sequence 20's page 1,024)
    for b, far, head in ((5, 9_000, 2), (5, 39_990, 3), (9, lens[9] - 100, 1), (20, 32_768 + 10, 4)):
        key = kp[table[b, far // 32].item(), head, far % 32].float()
        qkv[b, head * dh:(head + 1) * dh] = (8.0 * key / key.norm() * dh ** 0.25).to(torch.bfloat16)
    pos = t([n - 1 for n in lens], torch.int32)
    cu = t(np.arange(B + 1), torch.int32)
    seq = t(np.arange(B), torch.int32)
    got = ops.attention_decode_bf16(qkv, kp, vp, cu, pos, table, B, max(lens), heads, kv_heads, dh, None, dh ** -0.5)
    want = ops.attention(qkv, kp, vp, pos, seq, table, heads, kv_heads, dh, None, dh ** -0.5)
    close(got, f64(want), BF16_OUT, "a run of more than 1,024 pages")
    for b, head in ((5, 2), (5, 3), (9, 1), (20, 4)):       # and these rows are not drowned by the others' size
        row = slice(head * dh, (head + 1) * dh)
        assert want[b, row].float().abs().max() > 0.5
        close(got[b, row], f64(want[b, row]), BF16_OUT, f"sequence {b}, head {head}")


@pytest.mark.parametrize("fused", [False, True])
def test_decode_attention_writes_tiled_rows(ops, fused):
    rng = np.random.default_rng(77)
    heads, kv_heads, dh = 8, 2, 64
    lens = [int(x) for x in rng.integers(1, 600, size=20)]
    B = len(lens)
    k, v, kp, vp, table = paged(rng, [n + 1 for n in lens], kv_heads, dh, dtype=torch.bfloat16, spare=12)
    pos = t([n - 1 for n in lens], torch.int32)
    outs = []
    for tiles in (False, True):
        if fused:
            raw = t(np.random.default_rng(78).normal(size=(B, (heads + 2 * kv_heads) * dh)) * 2, torch.bfloat16)
            gains = t(np.ones(dh))
            out = ops.attention_decode_fused_bf16(raw, gains, gains, 1e-5, t(P.rope_inv_freq(dh, 1e4)), kp, vp, pos, table,
                                                  B, max(lens) + 50, heads, kv_heads, dh, None, dh ** -0.5, tiled_out=tiles)
        else:
            qkv = t(np.random.default_rng(79).normal(size=(B, (heads + 2 * kv_heads) * dh)), torch.bfloat16)
            cu = t(np.arange(B + 1), torch.int32)
            out = ops.attention_decode_bf16(qkv, kp, vp, cu, pos, table, B, max(lens) + 50, heads, kv_heads, dh, None,
                                            dh ** -0.5, tiled_out=tiles)
        assert isinstance(out, ops.TiledRows) == tiles
        outs.append(ops.as_rows(out))
    assert torch.equal(outs[0], outs[1]) and outs[0].shape == (B, heads * dh)


@pytest.mark.parametrize("m", [1, 3, 8, 13, 16])
@pytest.mark.parametrize("hidden, k, inter", [(104, 72, 56), (4096, 4096, 1000), (584, 12288, 40)])
def test_rows_in_the_matrix_cores_order(ops, m, hidden, k, inter):
    """A packed product can leave its result in the order the next packed product loads as an operand, and take
    its input in it: every such chain gives, bit for bit, what the same chain gives through plain rows."""
    rng = np.random.default_rng(3 * m + hidden)
    eps = 1e-5
    x = t(rng.normal(size=(m, k)), torch.bfloat16)
    pw_a = ops.pack_for_mfma(t(rng.normal(size=(hidden, k)) / np.sqrt(k), torch.bfloat16))
    pw_gu = ops.pack_for_mfma(t(rng.normal(size=(2 * inter, hidden)) * (4.0 / np.sqrt(hidden)), torch.bfloat16), swiglu=True)
    pw_b = ops.pack_for_mfma(t(rng.normal(size=(hidden, inter)) / np.sqrt(inter), torch.bfloat16))
    gain = t(1 + 0.3 * rng.normal(size=hidden))
    r0 = t(rng.normal(size=(m, hidden)) * 3)

    # the layout itself: rows() undoes it
    plain = ops.gemm_skinny_packed_bf16(x, pw_a, hidden)
    tiled = ops.gemm_skinny_packed_bf16(x, pw_a, hidden, tiled_out=True)
    assert isinstance(tiled, ops.TiledRows) and tiled.shape == (m, hidden)
    assert torch.equal(tiled.rows(), plain)
    # read back as an operand: with the activation, plain, and with K cut into parts
    pw_c = ops.pack_for_mfma(t(rng.normal(size=(inter, hidden)) / np.sqrt(hidden), torch.bfloat16))
    assert torch.equal(ops.gemm_skinny_packed_bf16(tiled, pw_gu, inter, torch.bfloat16, swiglu=True),
                       ops.gemm_skinny_packed_bf16(plain, pw_gu, inter, torch.bfloat16, swiglu=True))
    assert torch.equal(ops.gemm_skinny_packed_bf16(tiled, pw_c, inter), ops.gemm_skinny_packed_bf16(plain, pw_c, inter))
    assert torch.equal(ops.gemm_skinny_packed_bf16(tiled, pw_c, inter, torch.float32, parts=2),
                       ops.gemm_skinny_packed_bf16(plain, pw_c, inter, torch.float32, parts=2))
    # a layer's chain of links: norm left to the products, rows handed on in either layout
    outs = []
    for tiles in (False, True):
        residual = guarded(r0.clone())
        later = ops.linked_product(x, pw_a, hidden, True, residual=residual, next_gain=gain, next_eps=eps,
                                   tiled_out=tiles)
        assert isinstance(later.xg, ops.TiledRows) == tiles
        act = ops.linked_product(later, pw_gu, inter, True, torch.bfloat16, swiglu=True, tiled_out=tiles)
        later2 = ops.linked_product(act, pw_b, hidden, True, residual=residual, next_gain=gain, next_eps=eps,
                                    tiled_out=tiles)
        outs.append((residual, ops.as_rows(later.xg), ops.as_rows(act), ops.as_rows(later2.xg), later.ssq, later2.ssq))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    with pytest.raises(Exception, match="tiled"):
        ops.gemm_skinny_packed_bf16(x, pw_a, hidden, torch.float32, tiled_out=True)


@pytest.mark.parametrize("dtype, rel", [(torch.float32, 1e-6), (torch.bfloat16, 5e-3)])
def test_swiglu(ops, dtype, rel):
    assert f64(ops.swiglu(t([[0.0, 2.0, 3.0, 3.0]])))[0, 0] == 0.0                 # src/ops/elementwise.rs:59-70
    close(ops.swiglu(t([[0.0, 2.0, 3.0, 3.0]])), [[0.0, 6.0 / (1.0 + np.exp(-2.0))]], 1e-6)
    rng = np.random.default_rng(3)
    for inter in (333, 232, 1000):                 # odd, and multiples of 8 (the 16-byte form)
        y = t(rng.normal(size=(5, 2 * inter)) * 3, dtype)
        close(ops.swiglu(y), P.silu(f64(y)[:, :inter]) * f64(y)[:, inter:], rel, f"swiglu, {inter}")
        tiled = ops.swiglu(y, tiled_out=True)      # the matrix cores' order where the kernel can (16-byte form, bfloat16)
        if dtype == torch.bfloat16 and inter % 8 == 0:
            assert isinstance(tiled, ops.TiledRows) and torch.equal(tiled.rows(), ops.swiglu(y))
        else:
            assert torch.equal(tiled, ops.swiglu(y))


def test_argmax(ops):
    assert ops.argmax(t([[1.0, 3.0, 3.0], [-1.0, 0.0, -5.0]])).tolist() == [1, 1]   # src/ops/reduce.rs:75-78
    rng = np.random.default_rng(4)
    x = rng.normal(size=(5, 151937)).astype(np.float32)
    x[1, 70000] = x[1, 150000] = 9.0            # equal maxima far apart: the lower index wins
    x[2, 151936] = 10.0                         # the last element
    x[3, 0] = 10.0
    x[4, :] = -np.inf
    assert ops.argmax(t(x)).tolist() == [int(np.argmax(x[0])), 70000, 151936, 0, 0]


def test_kernels_refuse_what_they_cannot_do(ops):
    from rust_inference_amd.errors import KernelError, ShapeError
    if not EMULATED:
        with pytest.raises(KernelError, match="GPU only"):
            ops.swiglu(torch.zeros(2, 4))
    with pytest.raises(KernelError, match="1 to 8"):
        ops.gemv_bf16(torch.zeros(9, 16, dtype=torch.bfloat16, device=DEV), torch.zeros(4, 16, dtype=torch.bfloat16, device=DEV))
    with pytest.raises(KernelError, match="between 1 and 1024"):
        ops.attention(torch.zeros(1, 3 * 1032, device=DEV), torch.zeros(1, 1, 32, 1032, device=DEV),
                      torch.zeros(1, 1, 1032, 32, device=DEV), t([0], torch.int32), t([0], torch.int32),
                      t([[0]], torch.int32), 1, 1, 1032, None, 1.0)
    with pytest.raises(ShapeError, match="contiguous"):
        ops.swiglu(torch.zeros(4, 8, device=DEV)[:, ::2])


def test_kernels_agree_with_their_plain_cpp_twins(ops):
    """Each kernel family beside its scalar C++ twin (csrc/plain), float32: norm with the add, q/k norm and rotation,
    attention over pages, the product, the activation, argmax."""
    from rust_inference_amd.kernels import plain as N
    rng = np.random.default_rng(21)
    res, pend, gain = rng.normal(size=(5, 104)), rng.normal(size=(5, 104)), 1 + 0.1 * rng.normal(size=104)
    r_t = t(res)
    out = ops.add_rmsnorm(r_t, t(pend), t(gain), 1e-5, torch.float32)
    total, want = N.add_rms_norm(res, pend, gain, 1e-5)
    assert np.array_equal(r_t.cpu().numpy(), total)
    close(out, want, 1e-6, "add + norm")
    x, w = rng.normal(size=(7, 200)), rng.normal(size=(33, 200))
    close(ops.gemm_f32(t(x), t(w)), N.linear(x, w), 2e-6, "product")
    y = rng.normal(size=(4, 2 * 40)) * 3
    close(ops.swiglu(t(y)), N.swiglu(y), 1e-6, "swiglu")
    logits = rng.normal(size=(3, 1000)).astype(np.float32)
    logits[1, 5] = logits[1, 700] = 9.0
    assert ops.argmax(t(logits)).tolist() == [N.argmax(r) for r in logits]
    heads, kv_heads, dh, lens = 6, 2, 24, [40, 70]
    _, _, kp, vp, table = paged(rng, lens, kv_heads, dh)
    kp.zero_(); vp.zero_()
    tokens = sum(lens)
    qkv = rng.normal(size=(tokens, (heads + 2 * kv_heads) * dh))
    tok_seq = [b for b, n in enumerate(lens) for _ in range(n)]
    tok_pos = [i for n in lens for i in range(n)]
    qg, kg = 1 + 0.2 * rng.normal(size=dh), 1 + 0.2 * rng.normal(size=dh)
    inv = N.rope_inv_freq(dh, 1e4)
    qkv_t = t(qkv)
    ops.qk_norm_rope_kv_write(qkv_t, t(qg), t(kg), 1e-6, t(inv), t(tok_pos, torch.int32), t(tok_seq, torch.int32),
                              table, kp, vp, heads, kv_heads, dh)
    q = qkv.astype(np.float32)[:, :heads * dh].reshape(tokens, heads, dh)
    q_want = N.rope(N.rms_norm(q, qg, 1e-6), tok_pos, inv)
    close(qkv_t[:, :heads * dh].reshape(tokens, heads, dh), q_want, 3e-6, "q norm and rotation")
    got = ops.attention(qkv_t, kp, vp, t(tok_pos, torch.int32), t(tok_seq, torch.int32), table, heads, kv_heads, dh, None,
                        1 / np.sqrt(dh))
    want = N.attention(qkv_t.cpu().numpy()[:, :heads * dh].reshape(tokens, heads, dh), kp.cpu().numpy(), vp.cpu().numpy(),
                       tok_pos, tok_seq, table.cpu().numpy(), None, 1 / np.sqrt(dh))
    close(got.reshape(tokens, heads, dh), want, 3e-6, "attention over the pages the kernel wrote")


@pytest.mark.parametrize("act", [None, "float32", "relu2", "silu_gate", "clamped_gate"])
@pytest.mark.parametrize("m, n, k", [(1, 8, 192), (129, 264, 256), (257, 128, 320), (300, 520, 192), (70, 1032, 448)])
def test_product_in_tiles(ops, act, m, n, k):
    """Products of prompts in tiles: edges of a tile in rows and columns, the fewest stages of K, stages of either number; every
    activation on the sums; matrices that are a slice of longer rows; the same bits from every tile and from any number of rows."""
    rng = np.random.default_rng(m + n + k)
    gated = act in ("silu_gate", "clamped_gate")
    x = t(rng.normal(size=(m, k)), torch.bfloat16)
    wide = t(rng.normal(size=((2 if gated else 1) * n, k + 64)) * (3.0 / np.sqrt(k)), torch.bfloat16)
    w = wide[:, 64:] if m % 2 else wide[:, :k].contiguous()
    y = f64(x) @ f64(w).T
    g, u = y[:, :n], y[:, n:]
    bg, bu, limit = rng.normal(size=n), rng.normal(size=n), 2.5
    kw, want = {}, y
    if act == "relu2":
        want = np.maximum(y, 0) ** 2
    if act == "silu_gate":
        want = P.silu(g) * u
    if act == "clamped_gate":
        kw = dict(b_gate=t(bg), b_up=t(bu), limit=limit)
        g, u = np.minimum(g + np.float32(bg), limit), np.clip(u + np.float32(bu), -limit, limit)
        want = g / (1 + np.exp(-1.702 * g)) * (u + 1)
    out_dtype, name = (torch.float32, None) if act == "float32" else (torch.bfloat16, act)
    got = ops.gemm_tiles_bf16(x, w, 0, out_dtype, name, **kw)
    # bfloat16 results: half a unit in their last place, 2^-9 at the most; float32: sums of k products of eight bits each
    close(got, want, 3e-6 if act == "float32" else 4e-3, f"tiles, {act}")
    for tile in (1,) if gated else (1, 2):
        assert torch.equal(ops.gemm_tiles_bf16(x, w, tile, out_dtype, name, **kw), got)
    assert torch.equal(ops.gemm_tiles_bf16(x[m - 1:].contiguous(), w, 1, out_dtype, name, **kw), got[m - 1:])
    taller = torch.full((m + 2, n), 7.0, dtype=out_dtype, device=x.device)
    ops.gemm_tiles_bf16(x, w, 1, out_dtype, name, out=taller[1:m + 1], **kw)         # nothing beside its own rows
    assert torch.equal(taller[1:m + 1], got) and bool((taller[0] == 7).all()) and bool((taller[m + 1] == 7).all())
    with pytest.raises(Exception, match="gemm_tiles_bf16"):
        ops.gemm_tiles_bf16(x[:, :128].contiguous(), w[:, :128].contiguous(), 0, out_dtype, name, **kw)
    if gated:
        with pytest.raises(Exception, match="tile"):
            ops.gemm_tiles_bf16(x, w, 2, out_dtype, name, **kw)


@pytest.mark.parametrize("act", [None, "float32", "silu_gate"])
def test_product_in_tiles_over_rounds(ops, act):
    """Workgroups that take one tile after another, the last round partly filled: what runs ahead into the next tile is that tile's."""
    rng = np.random.default_rng(5)
    room = max(8, ops.compute_units() // 8 * 8)
    m, n, k = 256 * (room * 5 // 8) - 126, 272, 192          # 1.25 rounds of 256 x 256 and more, edges in rows and columns
    x = t(rng.normal(size=(m, k)), torch.bfloat16)
    w = t(rng.normal(size=(n, k)) * (3.0 / np.sqrt(k)), torch.bfloat16)
    out_dtype, name = (torch.float32, None) if act == "float32" else (torch.bfloat16, act)
    y = x.float() @ w.float().t()
    want = torch.nn.functional.silu(y[:, :n // 2]) * y[:, n // 2:] if act == "silu_gate" else y
    for tile in ((0, 1) if act == "silu_gate" else (0, 1, 2)):
        got = ops.gemm_tiles_bf16(x, w, tile, out_dtype, name)
        error = (got.float() - want).abs().amax(1) / want.abs().amax()
        assert float(error.max()) < (1e-5 if act == "float32" else 8e-3), (tile, int(error.argmax()))


@pytest.mark.parametrize("counts, n, k", [((0, 1, 130, 0, 256, 300, 0), 72, 192), ((257,), 264, 256), ((0, 0, 5), 8, 192), ((3,) * 64, 136, 320)])
@pytest.mark.parametrize("act", [None, "silu_gate", "clamped_gate", "relu2"])
def test_product_of_groups_of_rows(ops, act, counts, n, k):
    """Rows in groups with a matrix each, edges of the tiles and empty groups: the bits of a product a group, the matrices by rows and by columns;
    rows past the last group's stay out of it."""
    rng = np.random.default_rng(n + k)
    groups, starts = len(counts), np.concatenate([[0], np.cumsum(counts)])
    gated = act in ("silu_gate", "clamped_gate")
    x = t(rng.normal(size=(starts[-1] + 3, k)), torch.bfloat16)
    rows = (2 if gated else 1) * n
    w = t(rng.normal(size=(groups * rows, k)) * (3.0 / np.sqrt(k)), torch.bfloat16)
    by_columns = w.view(groups, rows, k).transpose(0, 1).reshape(rows, groups * k).contiguous()
    at = t(starts, torch.int32)
    for tile in (0, 1):
        for matrix, columns in ((w, False), (by_columns, True)):
            got = ops.gemm_tiles_groups(x, matrix, at, groups, n, tile, act, 0.8, by_columns=columns,
                                        out=t(np.full((len(x), n), 77.0), torch.bfloat16))
            assert (got[int(starts[-1]):] == 77.0).all(), (tile, columns)
            for i in range(groups):
                a, b = int(starts[i]), int(starts[i + 1])
                if b > a:
                    want = ops.gemm_tiles_bf16(x[a:b], w[i * rows:(i + 1) * rows], tile, torch.bfloat16, act, limit=0.8)
                    assert torch.equal(got[a:b], want), (tile, columns, i)


@pytest.mark.parametrize("given, held", [((0, 13, 50, 70), (0, 13, 30, 30)), ((0, 20, 5, 30), (0, 20, 20, 30)),
                                         ((-5, 10, 2 ** 31 - 1, 0), (0, 10, 30, 30)), ((50, 2, 60, 3), (30, 30, 30, 30))])
def test_groups_that_begin_outside_the_rows_are_held_to_them(ops, given, held):
    """Starts past the rows, before them and that descend: no row outside is read or written, none twice."""
    rng = np.random.default_rng(len(set(given)))
    n, k, groups = 72, 192, 3
    x, w = t(rng.normal(size=(30, k)), torch.bfloat16), t(rng.normal(size=(groups * n, k)) * (3.0 / np.sqrt(k)), torch.bfloat16)
    got = ops.gemm_tiles_groups(x, w, t(given, torch.int32), groups, n, 1, out=t(np.full((30, n), 77.0), torch.bfloat16))
    for i in range(groups):
        a, b = held[i], held[i + 1]
        if b > a:
            close(got[a:b], f64(x[a:b]) @ f64(w[i * n:(i + 1) * n]).T, BF16_OUT, f"group {i}")
    assert (got[:held[0]] == 77.0).all() and (got[held[-1]:] == 77.0).all()


def test_groups_of_rows_that_take_several_rounds(ops):
    """More tiles than places: workgroups go from one group's tiles to the next one's."""
    rng = np.random.default_rng(9)
    room = max(8, ops.compute_units() // 8 * 8)
    counts, k = (300, 0, 20, 513, 256), 192
    n, starts = 8 * (room * 8 + 9), np.concatenate([[0], np.cumsum(counts)])     # (columns for a quarter of a round, seven tiles of rows)
    x = t(rng.normal(size=(starts[-1], k)), torch.bfloat16)
    w = t(rng.normal(size=(len(counts) * n, k)) * (3.0 / np.sqrt(k)), torch.bfloat16)
    got = ops.gemm_tiles_groups(x, w, t(starts, torch.int32), len(counts), n, 0)
    for i in range(len(counts)):
        a, b = int(starts[i]), int(starts[i + 1])
        want = x[a:b].float() @ w[i * n:(i + 1) * n].float().t()
        if b > a:
            assert float((got[a:b].float() - want).abs().max() / want.abs().max()) < 8e-3, i


PAIR_FORMS = {"plain": {}, "window": {"window": 40}, "a page's window": {"window": 32}, "kept": {"window": 45, "keep_first": 37}, "kept pair": {"window": 70, "keep_first": 64},
              "chunk": {"chunk": 96}, "cap": {"softcap": 3.0}, "slopes": {"slopes": 0.05}, "sinks": {"sinks": True}}


@pytest.mark.parametrize("form", list(PAIR_FORMS))
@pytest.mark.parametrize("heads, kv_heads, dh", [(16, 1, 128), (20, 1, 128), (5, 5, 64), (17, 1, 64), (6, 2, 32), (20, 1, 32), (64, 1, 32), (40, 1, 64)])
def test_prompt_attention_in_pairs_of_pages(ops, heads, kv_heads, dh, form):
    """Two pages a turn against one: whole prompts and pieces, sequences that end in either page of a pair, windows and kept tokens whose first
    and last pages are of either number, pages that nobody sees not mapped; one tile of columns, two and four.  The two are up to a rounding of the weights
    (2^-9 of each) and of the result away from one another.  And the same bits alone, in one step with others and in pieces."""
    rng = np.random.default_rng(heads + dh)
    lens, new = [70, 300, 257, 1, 45, 131, 64], [70, 5, 1, 1, 45, 99, 64]
    kw = dict(PAIR_FORMS[form])
    reach = kw.get("window"), kw.get("chunk"), kw.get("keep_first", 0)
    held = [-(-n // 32) for n in lens]
    kp, vp = ((torch.randn(shape, device=DEV) * 0.8).to(torch.bfloat16) for shape in ((sum(held), kv_heads, 32, dh), (sum(held), kv_heads, dh, 32)))
    if EMULATED:
        kp, vp = (guarded(x) for x in (kp, vp))
    order = rng.permutation(sum(held))
    table, at = np.full((len(lens), max(held)), -1, np.int32), 0
    for b, n in enumerate(held):
        first = lens[b] - new[b]
        first = first - first % reach[1] if reach[1] else max(0, first - reach[0] + 1) if reach[0] else 0
        for p in range(n):
            if p >= first // 32 or p * 32 < reach[2]:
                table[b, p] = order[at + p]
        at += n
    if "slopes" in kw:
        kw["slopes"] = t(np.linspace(0.01, kw["slopes"], heads))
    if "sinks" in kw:
        kw["sinks"] = t(rng.normal(size=heads))
    window, cap = kw.pop("window", None), kw.pop("softcap", None)
    qkv = (torch.randn((sum(new), heads * dh), device=DEV) * 0.8).to(torch.bfloat16)
    pos = [p for b, n in enumerate(new) for p in range(lens[b] - n, lens[b])]

    def run(first, seqs, paired):                            # sequences `seqs`, their tokens from `first` of them on
        rows = [i for b in seqs for i in range(sum(new[:b]) + min(first, new[b] - 1), sum(new[:b + 1]))]
        counts = [new[b] - min(first, new[b] - 1) for b in seqs]
        index = torch.tensor(rows, device=qkv.device)
        q = guarded(qkv[index].contiguous()) if EMULATED else qkv[index].contiguous()
        return rows, f64(ops.attention_prefill_bf16(q, kp, vp, t(np.concatenate([[0], np.cumsum(counts)]), torch.int32),
                                                    t([pos[i] for i in rows], torch.int32), t(table[seqs], torch.int32), len(seqs), max(counts), heads,
                                                    kv_heads, dh, window, dh ** -0.5, cap, new_counts=counts, paired=paired, **kw))
    every = list(range(len(lens)))
    _, want = run(0, every, False)
    _, got = run(0, every, True)
    scale = np.abs(want).max()
    assert np.isfinite(got).all() and np.abs(got - want).max() <= 2.0 ** -8 * scale, np.abs(got - want).max() / scale
    for b in every:
        rows, alone = run(0, [b], True)
        assert np.array_equal(alone, got[rows])
    for first in (1, 33, 64):
        rows, pieces = run(first, every, True)
        assert np.array_equal(pieces, got[rows])


@pytest.mark.parametrize("window", [None, 50])
@pytest.mark.parametrize("heads, kv_heads, dh", MFMA_SHAPES + [(20, 1, 32), (64, 1, 32), (40, 1, 64)])
def test_prompt_attention_in_pairs_against_64_bits(ops, heads, kv_heads, dh, window):
    """Whole prompts and pieces of unequal lengths in pairs of pages against 64 bits, every number of tiles."""
    out, want = attention_case(ops, np.random.default_rng(heads * 3 + dh), [70, 300, 257, 1, 45, 131], [70, 5, 1, 1, 45, 99], heads, kv_heads, dh,
                               torch.bfloat16, window=window, kernel="prefill", paired=True)
    close(out, want, BF16_OUT, "prefill attention in pairs of pages")


def test_prompts_take_pairs_of_pages_by_themselves(ops):
    """A step's rule: prompts that bring enough tokens go in pairs of pages, the same bits as when told so; shorter ones a page a turn."""
    for lens, new in (([450, 460], [440, 460]), ([450, 90], [330, 90])):
        both = [f64(attention_case(ops, np.random.default_rng(7), lens, new, 4, 2, 32, torch.bfloat16, kernel="prefill", paired=p)[0])
                for p in (None, sum(new) >= 400 * len(new))]
        assert (ops.attention_prefill_pairs(new, 4, 2, 32) > 0) == (sum(new) >= 400 * len(new)) and np.array_equal(*both)


def test_prompts_of_more_tokens_than_a_launch_of_pairs_holds(ops):
    """A launch has 65,535 workgroups of a sequence's tokens: where pairs of pages take fewer tokens a workgroup than a page a turn, the
    longest prompts go a page a turn."""
    pairs = ops.attention_prefill_pairs
    assert pairs([2048], 16, 8, 128) > 0 and pairs([4 * 65535], 16, 1, 64) == 1 and pairs([4 * 65535 + 1], 16, 1, 64) == 0
    assert pairs([4 * 65535], 24, 1, 32) == 2 and pairs([4 * 65535 + 1], 24, 1, 32) == 0 and pairs([64 * 65535 + 1], 1, 1, 128) > 0
    if EMULATED:                                             # (too many tokens for the CPU)
        return
    n, last, heads, dh, pages = 4 * 65535 + 1, 40, 16, 32, 8193
    kp, vp = (torch.randn(shape, device=DEV).to(torch.bfloat16) for shape in ((pages, 1, 32, dh), (pages, 1, dh, 32)))
    qkv, table = torch.randn((n, heads * dh), device=DEV).to(torch.bfloat16), t(np.arange(pages)[None], torch.int32)

    def run(first, paired):
        return ops.attention_prefill_bf16(qkv[first:], kp, vp, t([0, n - first], torch.int32), torch.arange(first, n, dtype=torch.int32, device=DEV),
                                          table, 1, n - first, heads, 1, dh, None, dh ** -0.5, paired=paired)
    assert torch.equal(run(0, None)[n - last:], run(n - last, False))


def test_pairs_of_pages_where_they_pay(ops):
    """On 256 compute units, as measured beside the rule: prompts of hundreds of tokens on average whose tokens see hundreds of keys; windows
    and chunks shorter than that go a page a turn, unless that would take larger tiles."""
    if not EMULATED and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("measured on 256 compute units")
    pairs = ops.attention_prefill_pairs
    for heads in (16, 32, 64):
        for new in ([2048], [8192], [700] * 6):
            assert pairs(new, heads, 8, 128) > 0 and pairs(new, heads, 8, 128, 512) > 0
            assert pairs(new, heads, 8, 128, 128) == 0 and pairs(new, heads, 8, 128, 511) == 0
    for group in (9, 10, 17, 18, 21):                        # (pairs' tiles would leave almost half of their columns empty)
        assert pairs([1500] * 3, 4 * group, 4, 32) == 0 and pairs([500] * 8, 4 * group, 4, 32) == 0
        assert (pairs([1500] * 3, 4 * group, 4, 64) == 0) == (group < 16) and pairs([6000], 4 * group, 4, 64) > 0
    assert pairs([1500] * 3, 12 * 4, 4, 32) > 0 and pairs([1500] * 3, 22 * 4, 4, 32) > 0 and pairs([2000], 20, 1, 32) > 0
    assert pairs([300] * 16, 16, 8, 128) == 0 and pairs([8192] + [1] * 40, 16, 8, 128) == 0
    assert pairs([8192], 32, 8, 64, 128) == 1 and ops.attention_prefill_tiles([8192], 32, 8, 64) == 4 and pairs([2048], 32, 8, 64, 128) == 0
