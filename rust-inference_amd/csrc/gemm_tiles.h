// The kernel of a prompt's products in tiles (gemm_tiles_bf16.hip has the reasons), with one matrix for all rows or one a group of rows.
#pragma once
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
    // in groups: group i has the rows starts[i] to starts[i + 1] of x and out, and its matrix i * w_group elements after w
    const int32_t* starts;
    int groups;
    long w_group;
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

// TM x TN fragments of 16 rows of x and of w a wavefront, two by two wavefronts.  The grid is a multiple of eight.  GROUPED: up to 64
// groups of rows, each with a matrix of its own; their tiles are one sequence.
template <int TM, int TN, int ACT, typename TO, bool GROUPED = false>
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

    // The groups, a lane each: its rows, and the tiles of the groups up to it.  Where a group ends is the largest of the starts up to there
    // within x, so whatever the starts hold, groups lie side by side inside x and out.
    int first_row = 0, its_rows = 0, its_tiles = 0, upto = 0, all_tiles = a.m_tiles * a.n_tiles;
    if (GROUPED) {
        const int begin = min(max(a.starts[0], 0), M);
        int end = max(min(a.starts[min(lane + 1, a.groups)], M), begin);
#pragma unroll
        for (int d = 1; d < RI_WAVE; d *= 2) end = max(end, __shfl(end, max(lane - d, 0), RI_WAVE));
        const int before_it = __shfl(end, max(lane - 1, 0), RI_WAVE);
        first_row = lane ? before_it : begin;
        its_rows = end - first_row;                           // (none past the last group)
        upto = its_tiles = (its_rows + BM - 1) / BM * a.n_tiles;
#pragma unroll
        for (int d = 1; d < RI_WAVE; d *= 2) {
            const int before = __shfl(upto, max(lane - d, 0), RI_WAVE);
            upto += lane >= d ? before : 0;
        }
        all_tiles = __builtin_amdgcn_readfirstlane(__shfl(upto, RI_WAVE - 1, RI_WAVE));
    }

    // This workgroup's tile of a round, in bands of rows of x that are walked column by column.  Workgroups go to the eight L2 caches in turn:
    // those of one cache take neighbours.
    struct Tile { int m0, n0, end, group; };                 // (end: of the group's rows)
    auto tile_of = [&](int round, Tile& t) -> bool {
        const int before = round * (int)gridDim.x, left = min(all_tiles - before, (int)gridDim.x);
        const int per = (left + 7) / 8, at = blockIdx.x >> 3, id = (blockIdx.x & 7) * per + at;
        if (left <= 0 || at >= per || id >= left) return false;
        int i = before + id, m_tiles = a.m_tiles, start = 0;
        t.end = M;
        t.group = 0;
        if (GROUPED) {
            t.group = __builtin_ctzll(__ballot(upto > i));    // (i < all_tiles: there is one)
            i -= __builtin_amdgcn_readfirstlane(__shfl(upto - its_tiles, t.group, RI_WAVE));
            start = __builtin_amdgcn_readfirstlane(__shfl(first_row, t.group, RI_WAVE));
            const int its = __builtin_amdgcn_readfirstlane(__shfl(its_rows, t.group, RI_WAVE));
            m_tiles = (its + BM - 1) / BM;
            t.end = start + its;
        }
        const int band = i / (a.band * a.n_tiles), first = band * a.band, rows = min(a.band, m_tiles - first);
        const int in = i - first * a.n_tiles;
        t.m0 = start + (first + in % rows) * BM;
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
            xo[j] = (uint32_t)min(wave * 8 * TM + j * 8 + row, t.end - 1 - t.m0) * (uint32_t)a.ldx * 2u + (slot ^ row) * 16;
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
    const bf16_t* wa = a.w + (size_t)here.n0 * a.ldw + (GROUPED ? here.group * a.w_group : 0);
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
            wa = a.w + (size_t)next.n0 * a.ldw + (GROUPED ? next.group * a.w_group : 0);
        }
#pragma nounroll
        for (k = 0; k < 128; k += 64) {
            first_half(std::false_type(), k);
            ma_wait_copies<EARLY>();
            second_half(k);
        }
        ma_wait_products();
        const int m0 = here.m0 + wm * 16 * TM, n0 = here.n0 + wn * COLS, rows = here.end - m0, cols = N - n0;
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
