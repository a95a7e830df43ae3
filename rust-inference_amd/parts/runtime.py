"""What parts need from their surroundings at run time: the device, the compute
dtype, and the matrix product that fits both."""
from __future__ import annotations

import functools
import math

import torch

from ..errors import KernelError, ShapeError
from ..kernels import ops


@functools.lru_cache(maxsize=None)
def _wide_plan(n: int, k: int, swiglu: bool, rows: int = 64) -> tuple[int, int]:
    """``ops.wide_product_plan``, asked once per matrix size and tile of 16 rows."""
    return ops.wide_product_plan(n, k, swiglu, rows)

# Which product kernel runs, by the number of rows of x (bfloat16; the measurements behind every constant
# here are written up with the design notes, under "Which product kernel serves which step"):
#   1 row      one wavefront per weight row (ops.gemv_bf16).
#   2-16 rows  the matrix-core kernel on weights packed into MFMA tiles ahead of time, where a part asked for the
#              packed copy (the rule is _packed_pays below); it hands its rows to the next packed product in the
#              operand's order (ops.TiledRows) and does the norms around it.
#   17-64      the wide kernel (tiles of x shared through LDS) where the reader adds stretches of K or the
#              gate|up pairs fill the machine; the packed kernel with two or four tiles of x on small matrices
#              and up to 32 rows of tiled x; else the library.
#   65-128     the wide kernel with two row tiles a wavefront for matrices of long rows whose reader adds stretches
#              of K (`down`; up to 256 rows for the longest), and for the largest gate|up pairs; else the library.
#   512 and more  the product in tiles (ops.gemm_tiles_bf16) where its tiles fill the machine or the activation rides in it
#              (the rule is _tiles_plan below).
#   else       the vendor library (the reference hands every product to one: src/cuda/mod.rs:186-232).
GEMV_MAX_ROWS = 1
SKINNY_MAX_ROWS = 16
MID_MAX_ROWS = 64
MID_MAX_BYTES = 20_000_000       # up to this size the packed kernel beats the library at 17 to 64 plain rows
MID_TILED_ROWS = 32              # and up to this many rows when the rows come tiled,
MID_TILED_BYTES = 64_000_000     # on matrices up to this size (7168 x 5120 draws level with the library, 10240 x 5120 loses: 28 us to 20)
WIDE_MIN_K = 4096                # rows shorter than this leave the wide kernel's stretches too little to do
WIDE_MIN_ROWS = 17
PAIRS_MAX_ROWS = 128             # 65 to 128 rows: the wide kernel with two row tiles a wavefront, where the library does badly:
PAIRS_MIN_K = 8192               # matrices of long rows (and at least twice as long as there are rows: `down`)
PAIRS_MORE_ROWS = 256            # and in two passes up to this many rows where the rows have PACKED_LONG_K elements and more
SMALL_ONLY_ROWS = 64             # a matrix packed for small steps alone stays on the wide kernel up to this many rows
# (5,120 x 8,192 at 32 / 48 / 64 rows: 20 / 24 / 29 us against the library's 19 to 34 / 30 / 23; 5,120 x 5,120: 15 / 18 / 21 against 19 / 20 / 19;
# with three stretches of 80 groups of four wavefronts 24 and 18 us at 64 rows: a step of 49 to 64 sequences 1 to 1.6% shorter at those sizes)
WIDE_GATED_FILL = 0.75            # gate|up goes to the wide kernel where its workgroups fill this share of the rounds,
WIDE_GATED_ROWS = 48             # and up to this many rows whatever they fill, if the packed kernel of 17 to 64 rows is no match:
WIDE_GATED_BYTES = 64_000_000    # pairs larger than this (smaller ones, up to 32 tiled rows, are that kernel's)
# 17 to 48 rows (to 64 where _wide_many_waves below says so) against a plain matrix of many rows (all experts' gates and ups side by side: 4 row tiles a compute unit and
# more): the wide kernel, K whole.  98,304 x 4,096 at 17 / 32 / 48 / 64 rows: 136 / 143 / 163 / 183 us against the library's 180 / 180 / 172 / 177;
# 24,576 x 1,024: 13 / 15 / 17 / 20 against 32 / 32 / 18 / 18; 24,576 x 4,096 37 / 41 / 49 / 58 against 52 / 51 / 51 / 51; with fewer row
# tiles level (12,288 x 4,096 at 32 rows 23 against 24).  Weights not in the caches, at 17 / 32 / 48 rows, the wide kernel : the library: 16,384 x 1,024
# 8.9 / 9.6 / 10.6 : 12.9 / 12.8 / 13.3, x 5,120 30 / 32 / 36 : 35 / 35 / 37; 32,768 x 4,096 50 / 53 / 55 : 66 / 66 / 67; 49,152 x 2,048 37 / 40 / 45 : 50 / 49 / 49;
# 151,936 x 2,048 108 / 120 / 139 : 151 / 153 / 150.  At 48 rows some sizes are the library's: 20,480 x 4,096 33 / 37 / 43 : 41 / 40 / 41, 24,576 x 2,560
# 25 / 28 / 32 : 28 / 27 / 29, 65,536 x 768 22 / 26 / 29 : 25 / 25 / 26 (no rule of tiles and K tells them from the others).
WIDE_PLAIN_TILES = 4
WIDE_PLAIN_ROWS = 48
SPLIT_K = 4096                   # pieces of a long K (PACKED_LONG_K and more) whose sums the next norm adds
# Which matrices get a packed copy for 2 to 16 rows (the gate|up matrix always does: its activation rides in
# the kernel): up to 40 MB always; up to PACKED_MAX_BYTES unless the last round of workgroups (one per 16 rows)
# would leave most compute units idle; rows of PACKED_LONG_K elements and more always, cut into parts.
PACKED_MAX_BYTES = 101_000_000
PACKED_LONG_K = 16384


@functools.lru_cache(maxsize=None)
def _compute_units() -> int:
    return ops.compute_units()


# Row tiles a workgroup of the wide kernel with K whole: 3 or 4 (whole slices of x), or many in half slices, one a wavefront or (20) two.  A
# compute unit fetches some 30 GB/s whatever it fetches, so the form is the one with which it fetches the fewest rows: of x (those that there are;
# the rest of a tile comes from a kilobyte of zeros) for every round of workgroups, and of the matrix.  Many row tiles where their share of the
# rows that three or four fetch is no more than below: in a single round (few large workgroups have a slow beginning and end), in several.  The limits are
# where 1,800 sizes of 16,384 to 160,000 rows by 512 to 8,192 at 9 to 64 rows of x, weights from memory, stop gaining; 1,023 of them take many row tiles, 0.88 of
# the time (at most 1.02 against three or four, 1.08 against the library).  us, many : three or four: 18,432 x 4,096 in sixes at 32 / 48 rows 34.5 : 35.9 / 32.3 : 42.5, at 17 (0.87
# of the rows) 32.6 : 30.5; 73,728 x 4,096 in 20s at 17 / 32 93 : 104 / 95 : 111; 98,304 x 4,096 in twelves at 32 / 48 136 : 140 / 142 : 160; 151,936 in 20s,
# float32 sums, at 9 / 16 / 32 / 48 / 64: x 4,096 188 / 193 / 204 / 215 / 221 : 203 / 212 / 237 / 265 / 287, x 1,024 51 / 53 / 58 / 63 / 66 : 52 / 56 / 64 / 72 / 80.
WIDE_MANY = {6: (0.80, 0.88), 8: (0.83, 0.90), 12: (0.80, 0.86), 20: (0.92, 0.92)}
# A single round not for up to 16 rows of x (24,576 x 4,096: 43.5 : 35.6) nor, but for 20s, for rows shorter than WIDE_MANY_MIN_K.  Eights whose rows are
# a power of two of 1,024 to 4,096 elements lose whatever they fetch, below 4,096 always (65,536 x 2,048 at 17 / 32 / 48 rows 60 / 62 / 60 : 46 / 51 / 57; 20s of
# it 46 / 49 / 50), at 4,096 past this share (65,536 at 17 rows, 0.90: 96 : 90).
WIDE_MANY_MIN_K = 2048
WIDE_EVEN_EIGHTS = 0.84
# Past WIDE_PLAIN_ROWS the library takes the step otherwise.  With float32 results it is behind nearly everywhere (at 64 rows 151,936 x 4,096 221 : 267,
# x 1,024 66 : 81; ahead at 50,304 x 5,120 105 : 100), with bfloat16 results ahead for short rows (57,344 x 1,024 32 : 26) and, but for the fewest rows fetched,
# for rows past 4,096 (26,624 x 5,120 in eights 59 : 54, 122,880 x 5,120 in twelves 248 : 220; 81,920 x 5,120 in 20s 137 : 171).
WIDE_LIBRARY_K = 4096
WIDE_LIBRARY_SHARE = 0.70


def _wide_rows(n: int, m: int, waves: int) -> tuple[int, int]:
    """Rounds of workgroups of that many row tiles, and the rows (of x and of the matrix) that a compute unit fetches in them."""
    rounds = -(-n // (16 * waves * _compute_units()))
    return rounds, rounds * (m + 16 * waves)


def _wide_whole_waves(n: int, m: int) -> int:
    """Three or four row tiles a workgroup of the wide kernel with K whole: whichever has a compute unit fetch fewer rows (of
    x in whole tiles for every round of workgroups, and of the matrix)."""
    tiled = -(-m // 16) * 16
    return 3 if _wide_rows(n, tiled, 3)[1] < _wide_rows(n, tiled, 4)[1] else 4


@functools.lru_cache(maxsize=4096)
def _wide_many_waves(n: int, k: int, m: int, wide_out: bool = False, few: int | None = None) -> int | None:
    """Many row tiles a workgroup of the wide kernel with K whole (of WIDE_MANY), where they pay: against ``few`` (three or four by the rule
    above), past WIDE_PLAIN_ROWS against the library's product with float32 (``wide_out``) or bfloat16 results."""
    beside = _wide_rows(n, m, few or _wide_whole_waves(n, m))[1]
    even = 1024 <= k <= 4096 and k & (k - 1) == 0
    best = None
    for waves, limits in WIDE_MANY.items():
        rounds, rows = _wide_rows(n, m, waves)
        limit = limits[rounds > 1]
        if rounds == 1 and (m <= SKINNY_MAX_ROWS or (waves < 20 and k < WIDE_MANY_MIN_K)):
            continue
        if waves == 8 and even:
            limit = min(limit, WIDE_EVEN_EIGHTS if k == 4096 else 0.0)
        if m > WIDE_PLAIN_ROWS and not wide_out:
            if k < WIDE_MANY_MIN_K or (k > WIDE_LIBRARY_K and waves < 12):
                continue
            limit = min(limit, WIDE_LIBRARY_SHARE) if k > WIDE_LIBRARY_K else limit
        if rows <= limit * beside and (best is None or rows < best[0]):
            best = (rows, waves)
    return best[1] if best else None


def _packed_pays(n: int, k: int) -> bool:
    if k >= PACKED_LONG_K or n * k * 2 <= 40_000_000:
        return True
    tiles = -(-n // 16)
    cus = _compute_units()
    last_round = tiles % cus
    return n * k * 2 <= PACKED_MAX_BYTES and not (tiles > cus and 0 < last_round < cus // 2)


# Which tile of the product in tiles, if any.  Its time goes in rounds of tiles (one a compute unit), 256 x 256 at 1.35 PFLOP/s, the smaller
# ones 0.87 of that; the library's product into bfloat16 makes 1.4 where its own rounds are full, into float32 1.22 (its epilogue), and 0.9 to 1.05
# where half a round is left after two or more.  So, by the share of the rounds that is filled (us, tiles : library; rows; columns x K):
#   one round of the smaller tiles from 0.88 on, either result: 2,048; 4,096 x 4,096 56 : 62, x 12,288 168 : 188; 7,640; 1,024 x 2,048 29 : 33, x 3,072
#     41 : 46; 1,536; 5,120 x 5,120 69 : 79 (at 0.83 level, at 0.62 to 0.66 47 : 50 and 111 : 107);
#   three and more rounds of 256 x 256, 0.8 to 0.93: 8,192; 5,120 x 8,192 499 : 667, x 25,600 1,606 : 2,088; 5,120; 8,192 x 4,096 265 : 367; 6,144; 12,288 x 4,096 458 : 582
#     (at 0.75 253 : 239); float32 results also above, and in any number of rounds: 4,096; 8,192 x 4,096 210 : 227, 8,192; 12,288 x 4,096 604 : 656, 1,280 105 : 115
#     (bfloat16 195 : 186, 582 : 562, 99 : 100);
#   with the activation in it, which saves a kernel that reads and writes the results again: 2,048; 24,576 x 4,096 288 : 284 + 29, 7,640; 6,144 x 1,024 74 : 79 + 25,
#     8,192; 51,200 x 5,120 3,072 : 3,119 + 212; from 0.62 on (the smaller tiles' share counted 0.87; 759; 24,576 x 4,096, 0.64: 159 : 147 + 13, 300, 0.59: 87 : 70 + 8),
#     rows of up to 2,048 from 0.45 (759; 6,144 x 1,024: 14 : 15 + 5).  Without a gate less is saved: 0.1 more.
TILES_MIN_ROWS = 512
TILES_ONE_ROUND, TILES_FULL, TILES_MOST = 0.88, 0.93, 0.80
TILES_FUSED, TILES_FUSED_SHORT, TILES_SHORT_K, TILES_SMALLER = 0.62, 0.45, 2048, 0.87


@functools.lru_cache(maxsize=4096)
def _tiles_plan(m: int, n: int, k: int, wide_out: bool, activation: str | None) -> int | None:
    """The tile (of ``ops.TILES``) with which ``m`` rows go through a matrix of ``n`` rows of ``k``; None: not in tiles.  ``wide_out``: float32
    results; ``activation``: what may ride in the product."""
    gated = activation in ("silu_gate", "clamped_gate")
    if m < TILES_MIN_ROWS or k < ops.TILES_MIN_K or k % 64 or n % (16 if gated else 8):
        return None
    cus = _compute_units()

    def rounds_and_fill(tile):
        rows, cols = ops.TILES[tile]
        rounds = -(-(-(-m // rows) * -(-n // cols)) // cus)
        return rounds, m * n / (rounds * cus * rows * cols)
    rounds, fill = rounds_and_fill(0)
    smaller = max((1,) if gated else (2, 1), key=lambda tile: rounds_and_fill(tile)[1])
    small_rounds, small_fill = rounds_and_fill(smaller)
    if activation is not None:
        worth = max(fill, TILES_SMALLER * small_fill)
        least = (TILES_FUSED_SHORT if k <= TILES_SHORT_K else TILES_FUSED) + (0.0 if gated else 0.1)
        return None if worth < least else 0 if fill >= TILES_SMALLER * small_fill else smaller
    if small_rounds == 1 and small_fill >= TILES_ONE_ROUND:
        return smaller
    if (rounds >= 3 and TILES_MOST <= fill < TILES_FULL) or (wide_out and fill >= TILES_FULL):
        return 0
    return None


# The same for rows in groups, a matrix each, in one launch (ops.gemm_tiles_groups), from four groups on (fewer fill the machine one by one).
# us, in one launch : the library's product and the activation a group; rows in eight groups: 9,842; gate and up 6,144 x 4,096 756 : 870, down 4,096 x 6,144
# 414 : 551; 2,048; the same 222 : 431 and 138 : 239; 512; 187 : 229 and 113 : 178; gate and up 1,536 x 1,024, down 1,024 x 1,536, 4,096 rows 30 : 113 and 34 : 71,
# 512 18 : 90 and 20 : 60; in 64 groups, 1,024 rows 81 : 754 and 36 : 437.  Whole mixtures of 4 to 64 experts of drawn sizes, even and skewed, 256 to 5,900 tokens: 0.02
# (launches of the host) to 0.93 of an expert a launch.  The host does not know how the rows are shared out: half a tile a group more than
# they fill, for the choice of the tile.  A round of the smaller takes 0.53 to 0.75 of the larger's time where tiles are full (9,842 rows, 15 : 8 rounds 866 : 756 us, 5 : 3 rounds 493 : 414).
GROUPS_LEAST = 4
GROUPS_SMALLER = 0.68


@functools.lru_cache(maxsize=4096)
def _groups_tile(m: int, groups: int, n: int, k: int, ldw: int, gated: bool) -> int | None:
    """The tile (of ``ops.TILES``) for ``m`` rows in ``groups`` groups through matrices of ``n`` results of ``k``; None: not in one launch."""
    if not GROUPS_LEAST <= groups <= ops.TILES_GROUPS_MOST or k < ops.TILES_MIN_K or k % 64 or n % 8:
        return None
    if not ops.gemm_tiles_fits(m, n, k, ldw, n, "silu_gate" if gated else None):
        return None

    def time(tile):
        rows, cols = ops.TILES[tile]
        tiles = groups * max(1.0, m / (groups * rows) + 0.5) * -(-n // (cols // 2 if gated else cols))
        return math.ceil(tiles / _compute_units()) * (GROUPS_SMALLER if tile else 1.0)
    return 1 if time(1) < time(0) else 0


# Products of one size that a part makes together (four of time mixing), all known: in one launch while the larger tile makes up to two rounds, after
# which one product fills the machine by itself.  us, in one launch : the library's four; 512 / 1,000 / 2,048 / 4,096 / 8,192 rows; 1,024 x 4,096 44 / 47 / 61 / 101 /
# 196 : 58 / 73 / 108 / 160 / 262; 512 x 1,024 16 / 17 / 18 / 22 / 34 : 33 / 35 / 38 / 44 / 56; 2,048 x 4,096 56 / 62 / 102 / 198 / 397 : 84 / 109 / 164 / 247 / 394.
TOGETHER_ROUNDS = 2


@functools.lru_cache(maxsize=4096)
def _together_tile(count: int, m: int, n: int, k: int) -> int | None:
    """The tile for ``count`` products of ``m`` rows with matrices of ``n`` rows of ``k`` in one launch; None: one after the other."""
    if m < TILES_MIN_ROWS or _groups_tile(count * m, count, n, k, k, False) is None:
        return None

    def rounds(tile):
        rows, cols = ops.TILES[tile]
        return -(-count * -(-m // rows) * -(-n // cols) // _compute_units())
    if rounds(0) > TOGETHER_ROUNDS:
        return None
    return 1 if rounds(1) * GROUPS_SMALLER < rounds(0) else 0


@functools.lru_cache(maxsize=4096)
def _tiles_fit(m: int, n: int, ldx: int, ldw: int, ldo: int, activation: str | None) -> bool:
    """``ops.gemm_tiles_fits``, asked once per size."""
    return ops.gemm_tiles_fits(m, n, ldx, ldw, ldo, activation)


class PackedWeight:
    """A bfloat16 weight as the library product wants it (row-major) and, for decode-size products,
    packed into MFMA tiles."""

    def __init__(self, w: torch.Tensor, packed: torch.Tensor | None, swiglu: bool):
        self.w, self.packed, self.swiglu = w, packed, swiglu
        self.n = w.shape[0] // 2 if swiglu else w.shape[0]
        self.k = w.shape[1]
        # a long K is cut into pieces of 4096 whose float32 sums the next norm adds up: more workgroups
        # stream the weights (768 instead of 256 for 4096 x 12288), and the sum is never rounded to 16 bits
        self.parts = self.k // SPLIT_K if (not swiglu and self.k >= PACKED_LONG_K) else 1
        # 2 to 16 rows into the residual stream go to the wide kernel (set by Runtime.pack: see there)
        self.small_wide = False
        self.small_only = False      # the packed copy was made for that alone: larger steps stay where they were


class StackedWeights:
    """Weights of one size whose products go together, each as a ``PackedWeight``; where one launch may take them all, row-major
    ``w [count, n, k]`` and the packed copies likewise, whose memory the single ones share (else None)."""

    def __init__(self, each: list[PackedWeight], w: torch.Tensor | None = None, packed: torch.Tensor | None = None):
        self.each, self.w, self.packed = each, w, packed
        self.n, self.k = each[0].n, each[0].k


class Runtime:
    """``dtype`` is the compute dtype: bfloat16 (16-bit activations and cache,
    float32 statistics and residual stream) or float32 (everything in true 32-bit;
    weights stay as stored and are widened exactly inside the kernels).

    ``invariant`` (bfloat16 only; float32 is so by itself): every step runs the same form of every kernel whatever
    its size, so that a request's logits are the same bits alone and in any batch, whole and token by token, as a
    graph and launched from the host.  The bfloat16 path otherwise chooses the product kernel by the number of rows,
    the attention kernel by the number of sequences and leaves small steps' norms to the products, and each form
    rounds at other places.  Here every product is the packed kernel for 17 to 64 rows in slices of 64 rows
    (a row's sums in it do not depend on the other rows), every norm the plain kernel, the q/k norm, rotation
    and cache write the kernel of one wavefront per token and head, and the attention the prompt kernel for
    single tokens too (a token's sums run over its sequence's pages in order whatever shares its tile), or the
    generic kernel, whose key tiles start at fixed positions, where that one does not take the sizes.  It is
    several times slower on prompts; it is for runs that must reproduce bit for bit."""

    def __init__(self, device="cuda:0", dtype=torch.bfloat16, invariant: bool = False):
        if dtype not in (torch.bfloat16, torch.float32):
            raise ShapeError(f"compute dtype {dtype} is neither bfloat16 nor float32")
        self.device = torch.device(device)
        if self.device.type != "cuda":
            raise KernelError(f"this library computes on the GPU only, not on {self.device}")
        self.dtype = dtype
        self.invariant = bool(invariant) and dtype == torch.bfloat16
        self._mm_out_dtype = None

    # ---- weights
    def place_matrix(self, w: torch.Tensor) -> torch.Tensor:
        """A linear or embedding weight on the device: bfloat16 for bfloat16 compute,
        as stored for float32 compute."""
        w = w.to(self.device, non_blocking=False)
        if self.dtype == torch.bfloat16 and w.dtype != torch.bfloat16:
            w = w.to(torch.bfloat16)
        return w.contiguous()

    def place_gain(self, g: torch.Tensor) -> torch.Tensor:
        """Norm gains are used in float32 whatever they are stored in
        (the reference: src/models/qwen3.rs:184, src/models/cuda.rs:45)."""
        return g.to(self.device).to(torch.float32).contiguous()

    # ---- products
    @staticmethod
    def many_waves(n: int, k: int, m: int, few: int) -> int | None:
        """``_wide_many_waves`` for parts that call the wide kernel themselves, for float32 sums, with ``few`` row tiles otherwise."""
        return _wide_many_waves(n, k, m, True, few)

    def linear(self, x: torch.Tensor, w: torch.Tensor, out_dtype=None) -> torch.Tensor:
        """``x @ w.T`` with float32 accumulation; no bias anywhere in this family
        (the reference: src/ops/linear.rs:7-19)."""
        out_dtype = out_dtype or self.dtype
        if x.shape[1] != w.shape[1]:
            raise ShapeError(f"linear: x has {x.shape[1]} columns, the weight {w.shape[1]}")
        if self.dtype == torch.float32:
            return ops.gemm_f32(x, w)
        m, k = x.shape
        if m <= GEMV_MAX_ROWS and k % 8 == 0:
            if isinstance(x, ops.NormedLater):
                return ops.linked_product(x, w, w.shape[0], False, out_dtype)
            return ops.gemv_bf16(ops.as_rows(x), w, out_dtype)
        tile = self._tile(x, w, out_dtype)
        if tile is not None:
            return ops.gemm_tiles_bf16(self.normed_now(x), w, tile, out_dtype)
        return self._library_mm(self.normed_now(x), w, out_dtype)

    @staticmethod
    def normed_now(x):
        """The rows of a ``NormedLater`` for a product that cannot do the norm itself."""
        if not isinstance(x, ops.NormedLater):
            return ops.as_rows(x)
        return ops.finish_norm(x)

    def pack(self, w: torch.Tensor, swiglu: bool = False, always: bool = False, parts_ok: bool = False) -> PackedWeight:
        """A placed weight, with a packed copy where the packed kernel is the faster one for 2 to 16
        rows (bfloat16 compute only), or wherever it can be used when the caller says ``always``.
        ``parts_ok``: the product's reader adds stretches of K (the residual stream's next norm).  Then a matrix
        that the packed kernel serves badly at 2 to 16 rows, one whose row tiles leave most compute units idle in
        their last round (5,120 rows) or whose long rows it cuts into parts itself (K of 16,384 and more), goes to
        the wide kernel there, which shares the rows of x through LDS and plans its stretches for the machine
        (5,120 x 5,120 at 8 rows: 11 us against the library's 19; 5,120 x 25,600: 41 against 51)."""
        n, k = w.shape
        if self.invariant and k % 8:
            raise ShapeError(f"the invariant mode's product takes rows of a multiple of 8 elements, not {k}")
        pays = always or swiglu or self.invariant or _packed_pays(n, k)
        small_wide = (parts_ok and not swiglu and not self.invariant and k >= WIDE_MIN_K
                      and (not pays or k >= PACKED_LONG_K))
        if self.dtype != torch.bfloat16 or k % 8 or not (pays or small_wide):
            return PackedWeight(w, None, swiglu)
        pw = PackedWeight(w, ops.pack_for_mfma(w, swiglu), swiglu)
        pw.small_wide, pw.small_only = small_wide, small_wide and not pays
        return pw

    @staticmethod
    def _mid_pays(pw: PackedWeight, m: int, tiled: bool) -> bool:
        """Whether the packed kernel for 17 to 64 rows beats the library's product (and, for gate|up, its
        activation kernel) on this matrix."""
        size = pw.w.shape[0] * pw.k * 2
        if size <= MID_MAX_BYTES:
            return True
        return tiled and m <= MID_TILED_ROWS and size <= MID_TILED_BYTES

    @staticmethod
    def _wide_gated(pw: PackedWeight, m: int) -> bool:
        """Whether the wide kernel takes a gate|up pair at 17 to 64 rows: up to WIDE_GATED_ROWS rows whenever the
        pair is too large for the packed kernel of those rows (which takes twice as long for twice the rows);
        beyond, where its workgroups (of three or four wavefronts, K whole) fill the compute units evenly; else a
        quarter of the machine idles and the library with its activation kernel is as fast."""
        if pw.packed is None:
            return False
        size = pw.w.shape[0] * pw.k * 2
        if m <= WIDE_GATED_ROWS and (size > WIDE_GATED_BYTES or (m > MID_TILED_ROWS and size > MID_MAX_BYTES)):
            return True
        waves, parts = _wide_plan(pw.n, pw.k, True)
        groups = -(-(-(-pw.n // 16)) // waves) * parts
        cus = _compute_units()
        return groups / (-(-groups // cus) * cus) >= WIDE_GATED_FILL

    def takes_tiled(self, pw: PackedWeight, m: int, parts_ok: bool = False) -> bool:
        """Whether the product of ``m`` rows with this weight (called with this ``parts_ok``) runs on a packed
        kernel: whoever makes its rows then makes them as ``ops.TiledRows``."""
        if self.dtype != torch.bfloat16 or pw.packed is None or pw.k % 8 or self.invariant:
            return False
        if pw.small_only:                                        # a packed copy made for small steps into the stream alone:
            return parts_ok and 2 < m <= SMALL_ONLY_ROWS         # the wide kernel takes those, nothing else of it
        if GEMV_MAX_ROWS < m <= SKINNY_MAX_ROWS:
            return True
        if WIDE_MIN_ROWS <= m <= MID_MAX_ROWS and (self._wide_gated(pw, m) if pw.swiglu
                                                   else parts_ok and pw.k >= WIDE_MIN_K):
            return True                                          # the wide kernel (where the reader adds its parts)
        return SKINNY_MAX_ROWS < m <= MID_MAX_ROWS and self._mid_pays(pw, m, True)

    def linear_packed(self, x, pw: PackedWeight, out_dtype=None, parts_ok: bool = False, link=None,
                      tiled_out: bool = False):
        """``x @ w.T`` (or ``silu(x @ gate.T) * (x @ up.T)`` for a fused gate|up weight) with the kernel
        that fits the number of rows.  With ``parts_ok`` the result may be ``[parts, M, N]`` float32, the
        sums over pieces of K, for a consumer that adds them (the residual stream's next norm).

        ``x`` may be a ``NormedLater`` or ``TiledRows``.  With ``tiled_out`` the caller takes the result as
        ``TiledRows`` where the packed kernel makes it (2 to 16 rows): the layout the next packed product
        reads fastest.  With ``link`` (the residual stream's offer to the last product of
        a branch) a kernel that can adds the result into the stream and prepares the next norm; the
        return value is then ``(NormedLater, norm)`` for the stream instead of a tensor."""
        out_dtype = out_dtype or self.dtype
        m = x.shape[0]
        if self.invariant:
            # one kernel for every step: a row's sums in it depend on the row and the matrix alone
            x = self.normed_now(x)
            outs = [ops.gemm_mid_packed_bf16(x[i:i + MID_MAX_ROWS], pw.packed, pw.n, out_dtype, swiglu=pw.swiglu)
                    for i in range(0, m, MID_MAX_ROWS)]
            return outs[0] if len(outs) == 1 else torch.cat(outs, 0)
        if self.dtype == torch.bfloat16 and pw.k % 8 == 0:
            later = isinstance(x, ops.NormedLater)
            mine = None
            if (max(GEMV_MAX_ROWS, 2 if pw.small_only else 0) < m <= SKINNY_MAX_ROWS and pw.small_wide and parts_ok):
                # (the parts beat a link to the next norm, as they do for the packed kernel's own; two rows of a
                # matrix that had no packed copy stay with the kernel of one wavefront a row, which takes the link)
                x = self.normed_now(x) if later else x
                waves, parts = _wide_plan(pw.n, pw.k, False, -(-m // 16) * 16)
                return ops.gemm_wide_packed_bf16(x, pw.packed, pw.n, torch.float32, parts=parts, depth=1, waves=waves)
            if (SKINNY_MAX_ROWS // 2 < m <= SKINNY_MAX_ROWS and pw.swiglu and pw.packed is not None and not later
                    and pw.k >= WIDE_MIN_K):
                # 9 to 16 rows of a gate|up pair whose input is plain rows (the norm before it was a kernel of its
                # own): the packed kernel loads every row of x once per 16 rows of weights there (its form that
                # serves two steps with one load takes 8 rows), the wide one shares them through LDS (16 rows at
                # Qwen3-8B, 14B and 32B sizes: 33, 64 and 86 us against 35, 67 and 95)
                waves, _ = _wide_plan(pw.n, pw.k, True)
                return ops.gemm_wide_packed_bf16(x, pw.packed, pw.n, out_dtype, swiglu=True, depth=1, waves=waves,
                                                 tiled_out=tiled_out and out_dtype == torch.bfloat16)
            if m <= GEMV_MAX_ROWS or (m <= 2 and (pw.packed is None or pw.small_only)):
                mine = (pw.w, False)
            elif m <= SKINNY_MAX_ROWS and pw.packed is not None and not pw.small_only:
                mine = (pw.packed, True)
            if mine is not None:
                in_parts = mine[1] and parts_ok and pw.parts > 1        # very long rows: parts beat the link
                tiles = mine[1] and tiled_out and out_dtype == torch.bfloat16
                if link is not None and not pw.swiglu and not in_parts and link.residual.shape == (m, pw.n):
                    made = ops.linked_product(x, mine[0], pw.n, mine[1], residual=link.residual,
                                              next_gain=link.gain, next_eps=link.eps,
                                              tiled_out=mine[1] and link.tiled)
                    return (made, link.norm)
                if in_parts:
                    x = self.normed_now(x) if later else x
                    return ops.gemm_skinny_packed_bf16(x, pw.packed, pw.n, torch.float32, parts=pw.parts)
                if later:
                    return ops.linked_product(x, mine[0], pw.n, mine[1], out_dtype, swiglu=pw.swiglu, tiled_out=tiles)
                if not mine[1]:
                    return ops.gemv_bf16(ops.as_rows(x), pw.w, out_dtype, swiglu=pw.swiglu)
                return ops.gemm_skinny_packed_bf16(x, pw.packed, pw.n, out_dtype, swiglu=pw.swiglu, tiled_out=tiles)
            if (WIDE_MIN_ROWS <= m <= MID_MAX_ROWS and pw.packed is not None and parts_ok and not pw.swiglu
                    and pw.k >= WIDE_MIN_K and not (pw.small_only and m > SMALL_ONLY_ROWS)):
                # 17 to 64 rows into the residual stream: K in stretches, every stretch a workgroup that shares the tiles of x
                # through LDS; the stream's next norm adds the stretches' sums
                x = self.normed_now(x) if later else x
                waves, parts = _wide_plan(pw.n, pw.k, False, -(-m // 16) * 16)
                return ops.gemm_wide_packed_bf16(x, pw.packed, pw.n, torch.float32, parts=parts, depth=1, waves=waves)
            if (MID_MAX_ROWS < m <= (PAIRS_MORE_ROWS if pw.k >= PACKED_LONG_K else PAIRS_MAX_ROWS) and pw.packed is not None
                    and parts_ok and not pw.swiglu and pw.k >= PAIRS_MIN_K and pw.k >= 2 * pw.n):
                # 65 to 128 rows against a matrix of long rows whose result goes into the residual stream (`down`):
                # the wide kernel with two row tiles a wavefront, K in stretches that the stream's next norm adds
                # (the longest rows up to 256 rows of x, in two passes over the weights)
                x = self.normed_now(x) if later else x
                x = x.rows() if isinstance(x, ops.TiledRows) else x
                waves, parts = _wide_plan(pw.n, pw.k, False, -(-m // 16) * 16)
                return ops.gemm_wide_packed_bf16(x, pw.packed, pw.n, torch.float32, parts=parts, depth=1, waves=waves)
            if MID_MAX_ROWS < m <= PAIRS_MAX_ROWS and pw.swiglu and pw.packed is not None:
                # 65 to 128 rows of the largest gate|up pairs (those that take five to eight wavefronts a workgroup)
                waves, _ = _wide_plan(pw.n, pw.k, True)
                if waves > 4:
                    x = self.normed_now(x) if later else x
                    x = x.rows() if isinstance(x, ops.TiledRows) else x
                    return ops.gemm_wide_packed_bf16(x, pw.packed, pw.n, out_dtype, swiglu=True, depth=1, waves=waves)
            if WIDE_MIN_ROWS <= m <= MID_MAX_ROWS and pw.swiglu and self._wide_gated(pw, m):
                x = self.normed_now(x) if later else x
                waves, _ = _wide_plan(pw.n, pw.k, True)
                return ops.gemm_wide_packed_bf16(x, pw.packed, pw.n, out_dtype, swiglu=True, depth=1, waves=waves,
                                                 tiled_out=tiled_out and out_dtype == torch.bfloat16)
            if (SKINNY_MAX_ROWS < m <= MID_MAX_ROWS and pw.packed is not None
                    and self._mid_pays(pw, m, isinstance(x, ops.TiledRows))):
                x = self.normed_now(x) if later else x
                return ops.gemm_mid_packed_bf16(x, pw.packed, pw.n, out_dtype, swiglu=pw.swiglu,
                                                tiled_out=tiled_out and out_dtype == torch.bfloat16)
            if (WIDE_MIN_ROWS <= m <= MID_MAX_ROWS and pw.packed is not None and not pw.swiglu and not pw.small_only
                    and pw.n >= 16 * WIDE_PLAIN_TILES * _compute_units()):
                many = _wide_many_waves(pw.n, pw.k, m, out_dtype == torch.float32)
                if many or m <= WIDE_PLAIN_ROWS:
                    x = self.normed_now(x) if later else x
                    return ops.gemm_wide_packed_bf16(x, pw.packed, pw.n, out_dtype, depth=1,
                                                     waves=many or _wide_whole_waves(pw.n, m))
        if pw.swiglu:
            tile = self._tile(x, pw.w, self.dtype, "silu_gate")
            if tile is not None:
                return ops.gemm_tiles_bf16(self.normed_now(x), pw.w, tile, self.dtype, "silu_gate")
            return ops.swiglu(self.linear(x, pw.w), tiled_out=tiled_out)
        return self.linear(x, pw.w, out_dtype)

    def stack(self, weights: list[torch.Tensor]) -> StackedWeights:
        """Weights of one size, for ``linear_each``: side by side for bfloat16 compute (moved there one by one); where no launch takes them
        together (float32, the invariant mode, rows of no multiple of 8) each as it is placed."""
        if any(w.shape != weights[0].shape for w in weights):
            raise ShapeError(f"weights of {[list(w.shape) for w in weights]} are not of one size")
        if self.dtype != torch.bfloat16 or self.invariant or weights[0].shape[1] % 8:
            return StackedWeights([self.pack(self.place_matrix(w)) for w in weights])
        w = torch.empty((len(weights), *weights[0].shape), dtype=self.dtype, device=self.device)
        each, packed = [], None
        for i, one in enumerate(weights):
            w[i].copy_(self.place_matrix(one))
            pw = self.pack(w[i])
            if pw.packed is not None:                    # (by size: all have one or none has)
                if packed is None:
                    packed = torch.empty((len(weights), *pw.packed.shape), dtype=pw.packed.dtype, device=pw.packed.device)
                packed[i].copy_(pw.packed)
                pw.packed = packed[i]
            each.append(pw)
        return StackedWeights(each, w, packed)

    def linear_each(self, x: torch.Tensor, weights: StackedWeights) -> list[torch.Tensor]:
        """``x[i] @ w[i].T`` of ``x [count, m, k]`` in the compute dtype: 2 to 16 rows in one launch of the packed kernel, prompts in one of the
        product in tiles (_together_tile), else one after the other."""
        count, m, k = x.shape
        if self.dtype == torch.bfloat16 and not self.invariant:
            if GEMV_MAX_ROWS < m <= SKINNY_MAX_ROWS and weights.packed is not None:
                return list(ops.gemm_skinny_batch(x, weights.packed, weights.n).unbind(0))
            tile = _together_tile(count, m, weights.n, k)
            if tile is not None:
                starts = torch.arange(0, count * m + 1, m, dtype=torch.int32, device=x.device)
                out = ops.gemm_tiles_groups(x.view(count * m, k), weights.w.view(count * weights.n, k), starts, count, weights.n, tile)
                return list(out.view(count, m, weights.n).unbind(0))
        return [ops.as_rows(self.linear_packed(x[i], pw)) for i, pw in enumerate(weights.each)]

    def linear_activated(self, x, pw: PackedWeight, activation: str, after, b_gate=None, b_up=None, limit: float = 0.0):
        """``after(x @ w.T)``, with the activation (of ``ops.TILES_ACTIVATIONS``; ``after`` does the same) in the product where that goes in
        tiles; the result in the compute dtype."""
        tile = self._tile(x, pw.w, self.dtype, activation)
        if tile is None:
            return after(ops.as_rows(self.linear_packed(x, pw)))
        return ops.gemm_tiles_bf16(self.normed_now(x), pw.w, tile, self.dtype, activation, b_gate, b_up, limit)

    def rows_activated(self, x, w: torch.Tensor, activation: str, after, limit: float = 0.0):
        """``linear_activated`` for rows and a stretch of a larger matrix (an expert's), without biases."""
        tile = self._tile(x, w, self.dtype, activation)
        if tile is None:
            return after(torch.mm(x, w.t()))
        return ops.gemm_tiles_bf16(x, w, tile, self.dtype, activation, limit=limit)

    def rows_into(self, out, x, w: torch.Tensor) -> None:
        """``out <- x @ w.T``; rows of any of the three may be stretches of longer ones."""
        tile = self._tile(x, w, out.dtype, ldo=out.stride(0)) if out.data_ptr() % 16 == 0 and out.stride(0) % 8 == 0 else None
        if tile is None:
            torch.mm(x, w.t(), out=out)
        else:
            ops.gemm_tiles_bf16(x, w, tile, out=out)

    def groups_tile(self, m: int, groups: int, n: int, k: int, ldw: int, gated: bool = False) -> int | None:
        """``_groups_tile`` for this type; None also where every step runs the same kernels."""
        return None if self.dtype != torch.bfloat16 or self.invariant else _groups_tile(m, groups, n, k, ldw, gated)

    def _tile(self, x, w: torch.Tensor, out_dtype, activation=None, ldo: int | None = None) -> int | None:
        """The tile for ``x @ w.T`` as these operands lie (results in rows of ``ldo``, else side by side); None: the library's product."""
        if self.dtype != torch.bfloat16 or self.invariant or x.shape[0] < TILES_MIN_ROWS:
            return None
        tile = _tiles_plan(x.shape[0], w.shape[0], w.shape[1], out_dtype == torch.float32, activation)
        if tile is None or w.stride(1) != 1 or w.stride(0) % 8 or w.data_ptr() % 16:
            return None
        if isinstance(x, torch.Tensor) and (x.stride(1) != 1 or x.stride(0) % 8 or x.stride(0) < x.shape[1] or x.data_ptr() % 16):
            return None                                          # the library's product takes any strides
        n = w.shape[0] // 2 if activation in ("silu_gate", "clamped_gate") else w.shape[0]
        ldx = x.stride(0) if isinstance(x, torch.Tensor) else x.shape[1]
        return tile if _tiles_fit(x.shape[0], n, ldx, w.stride(0), ldo or n, activation) else None

    def _library_mm(self, x, w, out_dtype):
        # The reference hands every product to a vendor library (src/cuda/mod.rs:186-232);
        # so does this path, for the shapes its own kernels do not cover.
        if out_dtype == torch.float32:
            if self._mm_out_dtype is None:
                try:
                    torch.mm(x[:1], w[:1].t(), out_dtype=torch.float32)
                    self._mm_out_dtype = True
                except (TypeError, RuntimeError):
                    self._mm_out_dtype = False
            if self._mm_out_dtype:
                return torch.mm(x, w.t(), out_dtype=torch.float32)
            return torch.mm(x, w.t()).to(torch.float32)
        return torch.mm(x, w.t())
