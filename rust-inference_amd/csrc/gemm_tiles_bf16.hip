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
#include "api.h"
#include "common.h"
#include "matrix_async.h"

#include <type_traits>

// GT_SILU_GATE: silu(gate) * up, GT_CLAMPED_GATE: g sigmoid(1.702 g) (u + 1) with g = min(gate + b_gate, limit), u = clamp(up + b_up, -limit,
// limit), both of w = [gate; up] with N results; GT_RELU2: max(v, 0)^2.
enum { GT_PLAIN = 0, GT_SILU_GATE = 1, GT_CLAMPED_GATE = 2, GT_RELU2 = 3 };

struct GtArgs {
    void* out;
    const bf16_t* x;
    const bf16_t* w;
    const float* b_gate;
    const float* b_up;
    float limit;
    int M, N, K, ldx, ldw, ldo, m_tiles, n_tiles, band;
};

// (One unit in the last place of float32 or two; what is stored has eight bits.)
__device__ __forceinline__ float gt_sigmoid(float z) { return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * -1.44269504f)); }

template <int ACT>
__device__ __forceinline__ float gt_act(float z, float u, float bg, float bu, float limit) {
    if (ACT == GT_SILU_GATE) return z * gt_sigmoid(z) * u;
    if (ACT == GT_CLAMPED_GATE) {
        z = fminf(z + bg, limit);
        return z * gt_sigmoid(1.702f * z) * (fminf(fmaxf(u + bu, -limit), limit) + 1.f);
    }
    if (ACT == GT_RELU2) return fmaxf(z, 0.f) * fmaxf(z, 0.f);
    return z;
}

// TM x TN fragments of 16 rows of x and of w a wavefront, two by two wavefronts.  The grid is a multiple of eight.
template <int TM, int TN, int ACT, typename TO>
__global__ void __launch_bounds__(256, 1)
gemm_tiles_bf16_kernel(const GtArgs a) {
    constexpr bool GATED = ACT == GT_SILU_GATE || ACT == GT_CLAMPED_GATE, HALF = sizeof(TO) == 2;
    constexpr int BM = 32 * TM, BN = 32 * TN, COLS = GATED ? 8 * TN : 16 * TN, STAGE = (BM + BN) * 8;
    constexpr int P = TM * TN, FR = TM + TN;                  // products half a stage, fragments and copies a stage
    constexpr bool LARGE = P == 64;
    constexpr int RP = LARGE ? 2 : 1, DP = LARGE ? 5 : 3, FREE = RP * FR + 4, EARLY = (P - FREE + DP - 1) / DP;
    // a fragment is read every RP products; from product FREE on the buffer is free, a copy goes out every DP, EARLY in the first half
    static_assert(FREE <= P && EARLY + P / DP >= FR, "a stage's copies go out within a stage");
    __shared__ uint4 lds[2 * STAGE];
    const int M = a.M, N = a.N;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const int wm = wave & 1, wn = wave >> 1, nk = a.K / 64;

    // This workgroup's tile of a round, in bands of rows of x that are walked column by column.  Workgroups go to the eight L2 caches in turn:
    // those of one cache take neighbours.
    struct Tile { int m0, n0; };
    auto tile_of = [&](int round, Tile& t) -> bool {
        const int before = round * (int)gridDim.x, left = min(a.m_tiles * a.n_tiles - before, (int)gridDim.x);
        const int per = (left + 7) / 8, at = blockIdx.x >> 3, id = (blockIdx.x & 7) * per + at;
        if (left <= 0 || at >= per || id >= left) return false;
        const int i = before + id, band = i / (a.band * a.n_tiles), first = band * a.band, rows = min(a.band, a.m_tiles - first);
        const int in = i - first * a.n_tiles;
        t.m0 = (first + in % rows) * BM;
        t.n0 = in / rows * (GATED ? BN / 2 : BN);
        return true;
    };
    Tile here;
    if (!tile_of(0, here)) return;

    // A copy of a wavefront fills eight rows of a stage: lane l row l / 8, place l % 8.  Rows past the edge are the last row again.
    uint32_t xo[TM], wo[TN];
    auto offsets = [&](const Tile& t) {
        const int row = lane >> 3, slot = lane & 7;
#pragma unroll
        for (int j = 0; j < TM; ++j)
            xo[j] = (uint32_t)min(wave * 8 * TM + j * 8 + row, M - 1 - t.m0) * (uint32_t)a.ldx * 2u + (slot ^ row) * 16;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int at = wave * 8 * TN + j * 8 + row, piece = slot ^ (HALF ? (row & 3) | (j & 1) << 2 : row);
            int from;
            if (GATED) {                                      // a wavefront's rows of w: half of the gate, the same half of up
                const int part = at / (16 * TN), in = at % (16 * TN);
                from = min(part * COLS + in % COLS, N - 1 - t.n0) + (in >= COLS ? N : 0);
            } else from = min(at, N - 1 - t.n0);
            wo[j] = (uint32_t)from * (uint32_t)a.ldw * 2u + piece * 16;
        }
    };
    offsets(here);
    const bf16_t* xa = a.x + (size_t)here.m0 * a.ldx;
    const bf16_t* wa = a.w + (size_t)here.n0 * a.ldw;
    const ma_lds_t x_at = ma_lds(lds + wave * 8 * TM * 8), w_at = ma_lds(lds + (BM + wave * 8 * TN) * 8);
    auto copy = [&](int e, int buf, size_t k) {
        if (e < TN) ma_copy16(w_at + buf * STAGE * 16 + e * 1024, wo[e], wa + k);
        else ma_copy16(x_at + buf * STAGE * 16 + (e - TN) * 1024, xo[e - TN], xa + k);
    };
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int e = 0; e < FR; ++e) copy(e, s, s * 64);

    ma_floatx4 acc[TM][TN];
    const uint4* xr = lds + (wm * 16 * TM + r) * 8;
    const uint4* wr = lds + (BM + wn * 16 * TN + (HALF ? 8 * (r >> 2) + (r & 3) : r)) * 8;
    const int slot0 = g ^ (r & 7), slot1 = (4 + g) ^ (r & 7);
    ma_bf16x8 xf[2][TM], wf[2][TN];
    auto read = [&](int e, int to, int buf) {
        const int s = buf * STAGE + (to ? slot1 : slot0);
        if (e < TN) wf[to][e] = *reinterpret_cast<const ma_bf16x8*>(wr + (HALF ? (e >> 1) * 256 + (e & 1) * 32 : e * 128) + s);
        else xf[to][e - TN] = *reinterpret_cast<const ma_bf16x8*>(xr + (e - TN) * 128 + s);
    };
    ma_wait_copies<FR>();
    ma_meet();
#pragma unroll
    for (int e = 0; e < FR; ++e) read(e, 0, 0);

    int buf = 0;
    auto first_half = [&](auto first, size_t k) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            if constexpr (decltype(first)::value) ma_product_first(acc[p / TN][p % TN], wf[0][p % TN], xf[0][p / TN]);
            else ma_product(acc[p / TN][p % TN], wf[0][p % TN], xf[0][p / TN]);
            if (p % RP == 0 && p / RP < FR) read(p / RP, 1, buf);
            if (p == FREE - 1) {
                ma_wait_lds();
                ma_meet();
            }
            if (p >= FREE && (p - FREE) % DP == 0) copy((p - FREE) / DP, buf, k);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto second_half = [&](size_t k) {
        ma_meet();
#pragma unroll
        for (int p = 0; p < P; ++p) {
            ma_product(acc[p / TN][p % TN], wf[1][p % TN], xf[1][p / TN]);
            if (p % RP == 0 && p / RP < FR) read(p / RP, 0, buf ^ 1);
            if (p % DP == DP - 1 && EARLY + p / DP < FR) copy(EARLY + p / DP, buf, k);
            __builtin_amdgcn_sched_barrier(0);
        }
        buf ^= 1;
    };
    // A tile's stores may still be under way when the next tile's second stage has to be there; they were issued after its copies.
    constexpr int STORES = TM * COLS / (HALF ? 32 : 16), PENDING = EARLY + STORES > 63 ? 63 : EARLY + STORES;
    bool stored = false;
    for (int round = 0;;) {
        first_half(std::true_type(), 128);
        if (stored) ma_wait_copies<PENDING>();
        else ma_wait_copies<EARLY>();
        second_half(128);
        size_t k = 192;
#pragma nounroll
        for (int s = 3; s < nk; ++s) {
            first_half(std::false_type(), k);
            ma_wait_copies<EARLY>();
            second_half(k);
            k += 64;
        }
        Tile next = here;                                     // (none: the copies fetch this one's first stages, for nobody)
        const bool more = tile_of(++round, next);
        if (more) {
            offsets(next);
            xa = a.x + (size_t)next.m0 * a.ldx;
            wa = a.w + (size_t)next.n0 * a.ldw;
        }
#pragma nounroll
        for (k = 0; k < 128; k += 64) {
            first_half(std::false_type(), k);
            ma_wait_copies<EARLY>();
            second_half(k);
        }
        ma_wait_products();
        const int m0 = here.m0 + wm * 16 * TM, n0 = here.n0 + wn * COLS, rows = M - m0, cols = N - n0;
        const bool whole = rows >= 16 * TM && cols >= COLS;
        TO* o = (TO*)a.out + (size_t)m0 * a.ldo + n0;
        uint32_t ldo = a.ldo;
        ma_opaque(ldo);                                       // (or the rows' places are kept through the products, for want of registers in memory)
        constexpr int PIECES = COLS / (HALF ? 32 : 16);      // a lane's 16-byte pieces of a row
        static_assert(PIECES % 2 == 0 && (!GATED || PIECES == 2), "stores go two by two");
        float bg[2][8], bu[2][8];
        if (ACT == GT_CLAMPED_GATE) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int n = min(n0 + 32 * h + 8 * g + e, N - 1);
                    bg[h][e] = a.b_gate ? a.b_gate[n] : 0.f;
                    bu[h][e] = a.b_up ? a.b_up[n] : 0.f;
                }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int q = 0; q < PIECES; q += 2) {
                uint32_t v[2][4];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if (HALF) {
                        float f[8];
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            const float z = ma_taken(acc[i][2 * (q + h) + e / 4][e % 4]);
                            float u = 0.f;
                            if (GATED) u = ma_taken(acc[i][(TN / 2 + 2 * (q + h) + e / 4) % TN][e % 4]);
                            f[e] = gt_act<ACT>(z, u, bg[h][e], bu[h][e], a.limit);
                        }
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[h][e] = pack_bf16x2(f[2 * e], f[2 * e + 1]);
                    } else
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[h][e] = __float_as_uint(ma_taken(acc[i][q + h][e]));
                }
                // both rows of eight get the two places side by side, so that a store writes whole lines
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t lo = v[0][e], hi = v[1][e];
                    v[0][e] = ma_upper_from(lo, hi);
                    v[1][e] = ma_lower_from(lo, hi);
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int row = 16 * i + 8 * h + (r & 7), col = (q + (r >> 3)) * (HALF ? 32 : 16) + g * (HALF ? 8 : 4);
                    if (whole || (row < rows && col < cols))
                        *reinterpret_cast<uint4*>(o + ((uint32_t)row * ldo + col)) = make_uint4(v[h][0], v[h][1], v[h][2], v[h][3]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (!more) break;
        stored = whole;
        here = next;
    }
    ma_wait_copies<0>();
}

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
    const GtArgs a = {out, (const bf16_t*)x, (const bf16_t*)w, b_gate, b_up, limit, m, n, k, ldx, ldw, ldo, 0, 0, 0};
    hipStream_t s = (hipStream_t)stream;
    if (out_dtype == RI_F32) launch_tiles_form<GT_PLAIN, float>(tile, a, s);
    else if (act == GT_PLAIN) launch_tiles_form<GT_PLAIN, bf16_t>(tile, a, s);
    else if (act == GT_SILU_GATE) launch_tiles_form<GT_SILU_GATE, bf16_t>(tile, a, s);
    else if (act == GT_CLAMPED_GATE) launch_tiles_form<GT_CLAMPED_GATE, bf16_t>(tile, a, s);
    else launch_tiles_form<GT_RELU2, bf16_t>(tile, a, s);
    RI_LAUNCH_CHECK("gemm_tiles_bf16");
    return 0;
}
