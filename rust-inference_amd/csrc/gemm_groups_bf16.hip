// Products of a prompt's rows that lie in groups, each with a matrix of its own (the experts of a mixture): the tiles of gemm_tiles_bf16.hip,
// all groups' in one launch.
//
// A launch an expert is a round of tiles an expert, and its last tiles fill a part of the machine: of eight experts with some 1,230 rows each
// (4,921 tokens, two experts a token; 6,144 x 4,096 gates and ups, 4,096 x 6,144 downs) gates and ups are 240 tiles a launch of 256 places, downs
// 80, which the library cuts into smaller ones (69 to 72 us each, 0.86 PFLOP/s).  Workgroups that stay go from one group's tiles to the next one's
// here, so only the last round of all is partly filled: gates and ups with the activation 756 us (8 launches 772, the
// library's and an activation kernel 870), downs 414 (8 of the library's 551; 398 where an expert's matrix lies in one piece and not, as the mixture's
// does, in rows 98,304 bytes apart); inside the model 729 and 419.  Where a group's rows begin is read from memory, where the sort has left it: the
// host need not know.
#include "gemm_tiles.h"

template <int TM, int TN, int ACT>
static void launch_tiles_groups(GtArgs a, hipStream_t s) {
    const int bm = 32 * TM, bn = ACT == GT_SILU_GATE || ACT == GT_CLAMPED_GATE ? 16 * TN : 32 * TN;
    a.n_tiles = (a.N + bn - 1) / bn;
    a.band = 1024 / bm;
    const long most = ((long)a.M / bm + a.groups) * a.n_tiles, room = ri_compute_units() / 8 * 8;    // tiles, however the rows are shared out
    const long grid = most < room ? (most + 7) / 8 * 8 : room > 8 ? room : 8;
    gemm_tiles_bf16_kernel<TM, TN, ACT, bf16_t, true><<<(unsigned)grid, 256, 0, s>>>(a);
}

template <int ACT>
static void launch_groups_form(int tile, const GtArgs& a, hipStream_t s) {
    if (tile == RI_TILE_256_256) launch_tiles_groups<8, 8, ACT>(a, s);
    else launch_tiles_groups<4, 8, ACT>(a, s);
}

extern "C" int ri_gemm_tiles_groups_bf16(void* out, int ldo, const void* x, int ldx, const void* w, int ldw, long w_group, const int32_t* starts,
                                         int groups, int m, int n, int k, int act, float limit, int tile, void* stream) {
    const bool gated = act == GT_SILU_GATE || act == GT_CLAMPED_GATE;
    RI_REQUIRE(groups > 0 && groups <= RI_WAVE && starts, "gemm_tiles_groups_bf16: %d groups", groups);
    RI_REQUIRE(m > 0 && n > 0 && n % 8 == 0 && k >= 192 && k % 64 == 0, "gemm_tiles_groups_bf16: m %d, n %d, k %d", m, n, k);
    RI_REQUIRE(act >= GT_PLAIN && act <= GT_RELU2 && (act != GT_CLAMPED_GATE || limit > 0.f), "gemm_tiles_groups_bf16: activation %d, limit %g", act,
               (double)limit);
    RI_REQUIRE(tile == RI_TILE_256_256 || tile == RI_TILE_128_256, "gemm_tiles_groups_bf16: tile %d", tile);
    RI_REQUIRE(ldx >= k && ldw >= k && ldo >= n && (ldx | ldw | ldo) % 8 == 0 && w_group > 0 && w_group % 8 == 0,
               "gemm_tiles_groups_bf16: rows of %d, %d and %d, matrices %ld apart", ldx, ldw, ldo, w_group);
    RI_REQUIRE(((uintptr_t)out | (uintptr_t)x | (uintptr_t)w) % 16 == 0, "gemm_tiles_groups_bf16: an operand is off a multiple of 16 bytes");
    // (the tiles of all groups are counted in 32 bits)
    RI_REQUIRE(ri_gemm_tiles_bf16_fits(m, n, ldx, ldw, ldo, gated) && ((long)m / 128 + groups) * ((n + 127) / 128) < (1L << 30),
               "gemm_tiles_groups_bf16: %d rows of %d, %d rows of %d exceed one launch", m, ldx, n, ldw);
    const GtArgs a = {out, (const bf16_t*)x, (const bf16_t*)w, nullptr, nullptr, limit, m, n, k, ldx, ldw, ldo, 0, 0, 0, starts, groups, w_group};
    hipStream_t s = (hipStream_t)stream;
    if (act == GT_PLAIN) launch_groups_form<GT_PLAIN>(tile, a, s);
    else if (act == GT_SILU_GATE) launch_groups_form<GT_SILU_GATE>(tile, a, s);
    else if (act == GT_CLAMPED_GATE) launch_groups_form<GT_CLAMPED_GATE>(tile, a, s);
    else launch_groups_form<GT_RELU2>(tile, a, s);
    RI_LAUNCH_CHECK("gemm_tiles_groups_bf16");
    return 0;
}
