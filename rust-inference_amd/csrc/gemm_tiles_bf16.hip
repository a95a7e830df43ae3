// Products of prompts: out[M, N] = x[M, K] . w[N, K]^T, bfloat16 in, float32 sums, in tiles of up to 256 x 256 results; with the
// feed-forward's activation on the sums, before they are rounded.
//
// A workgroup of four wavefronts works on a tile, K in stages of 64 through two LDS buffers that copies from memory fill without passing
// through registers.  What bounds it at large sizes is power: 256 x 256 takes 2,440 cycles a stage where its products alone are 2,048, at
// 1.75 GHz (8,192 rows; 10,240 x 5,120: 563 us, 1.53 PFLOP/s, the library 577); the smaller tiles are bound by LDS (a stage of 128 x 256
// is 96 KB read and 48 KB written for 1,024 cycles of products: 1,400).  Therefore:
//  - the largest tile that four wavefronts can hold: 256 sums a lane, one wavefront a SIMD, which has to hide everything by itself;
//  - so a stage's memory instructions stand between its products one by one (a run of them, some sixty cycles, is a gap of the matrix
//    cores: 2,700 cycles a stage), the fragments of a half of K read while the other half is multiplied, and the buffer given back as soon
//    as the second half's are read (at 0.28 of a stage, 0.25 in the smaller tiles), so that the copies, one every few products from there on,
//    have 1.2 stages (the first) to 0.6 (the last) to arrive;
//  - workgroups stay and take tile after tile, and the copies run ahead into the next tile, so that a tile begins with its operands there
//    (a launch a tile: 3,800 cycles before the first product and 7,400 after the last, of 50,000 at K = 1,024);
//  - the rows of w go into a fragment in an order that leaves a lane eight neighbouring bfloat16 results, and two lanes exchange halves, so
//    that stores write whole lines without LDS, which the next tile's operands fill.
// A 16-byte piece of a row of a stage (128 bytes) lies at its place exchanged by the row's number, so that a fragment's reads meet all banks.
// Tried and no faster: 32 x 32 x 16 products; stages of 32 in four or five buffers (a copy of half a line a row: 3,000 cycles); a last
// round cut along K, its float32 sums through memory (256 KB a tile there and back: 16 us, and a launch; only K of 12,288 gains from it).
#include "gemm_tiles.h"

template <int TM, int TN, int ACT, typename TO>
static void launch_tiles_bf16(GtArgs a, hipStream_t s) {
    const int bm = 32 * TM, bn = ACT == GT_SILU_GATE || ACT == GT_CLAMPED_GATE ? 16 * TN : 32 * TN;
    a.m_tiles = (a.M + bm - 1) / bm;
    a.n_tiles = (a.N + bn - 1) / bn;
    a.band = 1024 / bm;                                       // the 32 tiles of an L2 cache are about square
    const long tiles = (long)a.m_tiles * a.n_tiles, room = ri_compute_units() / 8 * 8;
    const long grid = tiles < room ? (tiles + 7) / 8 * 8 : room > 8 ? room : 8;
    gemm_tiles_bf16_kernel<TM, TN, ACT, TO><<<(unsigned)grid, 256, 0, s>>>(a);
}

template <int ACT, typename TO>
static void launch_tiles_form(int tile, const GtArgs& a, hipStream_t s) {
    if (tile == RI_TILE_256_256) return launch_tiles_bf16<8, 8, ACT, TO>(a, s);
    if constexpr (ACT == GT_PLAIN || ACT == GT_RELU2)
        if (tile == RI_TILE_256_128) return launch_tiles_bf16<8, 4, ACT, TO>(a, s);
    launch_tiles_bf16<4, 8, ACT, TO>(a, s);
}

// (a tile's rows are reached by 32-bit offsets in bytes, those of up from those of its gate too)
extern "C" int ri_gemm_tiles_bf16_fits(int m, int n, int ldx, int ldw, int ldo, int gated) {
    return ldx < (1 << 22) && ldo < (1 << 22) && ((long)(gated ? n : 0) + 256) * ldw < (1L << 30) && (long)m * n < (1L << 46);
}

extern "C" int ri_gemm_tiles_bf16(void* out, int out_dtype, int ldo, const void* x, int ldx, const void* w, int ldw, int m, int n, int k,
                                  int act, const float* b_gate, const float* b_up, float limit, int tile, void* stream) {
    const bool gated = act == GT_SILU_GATE || act == GT_CLAMPED_GATE;
    RI_REQUIRE(m > 0 && n > 0 && n % 8 == 0 && k >= 192 && k % 64 == 0, "gemm_tiles_bf16: m %d, n %d, k %d", m, n, k);
    RI_REQUIRE(out_dtype == RI_BF16 || (out_dtype == RI_F32 && act == GT_PLAIN), "gemm_tiles_bf16: out dtype %d, activation %d", out_dtype, act);
    RI_REQUIRE(act >= GT_PLAIN && act <= GT_RELU2 && (act != GT_CLAMPED_GATE || limit > 0.f), "gemm_tiles_bf16: activation %d, limit %g", act, (double)limit);
    RI_REQUIRE(tile == RI_TILE_256_256 || tile == RI_TILE_128_256 || (tile == RI_TILE_256_128 && !gated), "gemm_tiles_bf16: tile %d", tile);
    RI_REQUIRE(ldx >= k && ldw >= k && ldo >= n && (ldx | ldw | ldo) % 8 == 0, "gemm_tiles_bf16: rows of %d, %d and %d", ldx, ldw, ldo);
    RI_REQUIRE(((uintptr_t)out | (uintptr_t)x | (uintptr_t)w) % 16 == 0, "gemm_tiles_bf16: an operand is off a multiple of 16 bytes");
    RI_REQUIRE(ri_gemm_tiles_bf16_fits(m, n, ldx, ldw, ldo, gated),
               "gemm_tiles_bf16: %d rows of %d, %d rows of %d exceed one launch", m, ldx, n, ldw);
    const GtArgs a = {out, (const bf16_t*)x, (const bf16_t*)w, b_gate, b_up, limit, m, n, k, ldx, ldw, ldo, 0, 0, 0, nullptr, 0, 0};
    hipStream_t s = (hipStream_t)stream;
    if (out_dtype == RI_F32) launch_tiles_form<GT_PLAIN, float>(tile, a, s);
    else if (act == GT_PLAIN) launch_tiles_form<GT_PLAIN, bf16_t>(tile, a, s);
    else if (act == GT_SILU_GATE) launch_tiles_form<GT_SILU_GATE, bf16_t>(tile, a, s);
    else if (act == GT_CLAMPED_GATE) launch_tiles_form<GT_CLAMPED_GATE, bf16_t>(tile, a, s);
    else launch_tiles_form<GT_RELU2, bf16_t>(tile, a, s);
    RI_LAUNCH_CHECK("gemm_tiles_bf16");
    return 0;
}
