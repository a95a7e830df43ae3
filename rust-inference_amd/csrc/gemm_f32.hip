// out[M, N] = x[M, K] . w[N, K]^T for float32 x, with the accuracy of 32-bit arithmetic.  w may be stored as bfloat16
// and is widened exactly.  The sum over k of every output element is built the same way however many rows a call
// has, so a row's result does not depend on the other rows.
//
// bfloat16 weights (a checkpoint's usual form) run on the matrix cores without loss: a float32 has 24 bits, three
// bfloat16 of eight each (a published method: Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype
// For Higher-Precision Computations", 2019).  Here x = a + (b + c) 2^-16 exactly, for every float32: the parts are cut off, not
// rounded, and b and c are kept 2^16 times as large, so that the last bit of the smallest float32, 2^-149, is still one of bfloat16's
// (2^-133; the matrix cores take subnormal numbers as they are).  Every product of a part and a weight is exact in float32 above
// the subnormal numbers, and the sums of the three parts are float32 sums of their own, added at the end: what is rounded is the
// additions alone, as in a chain of multiply-adds, and there are fewer of them.  (The lower two in one sum would be twice as many
// additions at the size of the second part's: where the first parts cancel, K = 1,024, 2.65e-7 instead of 1.75e-7.)  Relative error against
// 64 bits (2-norm, normal x and weights): at K = 1,024 1.9e-7 where the chain of multiply-adds has 5.7e-7, at 3,072
// 3.4e-7 : 9.9e-7.  The three products run at a third of the bfloat16 rate, ten times the vector units' multiply-adds.
// An infinity, a NaN or a number past 2^119 has no such parts, but leaves an infinity or NaN in every sum it enters: such an
// output is computed again by the chain.
//
// Other forms (float32 weights, rows that 16-byte loads do not divide): float32 multiply-adds on the vector units, every
// output one sum over k = 0..K-1.
#include "api.h"
#include "common.h"
#include "matrix_async.h"

#include <type_traits>

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 f32_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32_floatx4;

__device__ __forceinline__ f32_bf16x8 as_bf16x8(uint4 v) { return *reinterpret_cast<const f32_bf16x8*>(&v); }

// Two floats' upper halves in one word, the first in the low half.
__device__ __forceinline__ uint32_t upper_halves(float a, float b) {
    return (__float_as_uint(a) >> 16) | (__float_as_uint(b) & 0xFFFF0000u);
}
__device__ __forceinline__ float below_upper(float a) { return a - __uint_as_float(__float_as_uint(a) & 0xFFFF0000u); }

#define F32_LOWER 65536.f     // the second and third part are so much larger than what they stand for

// Eight floats as three times eight bfloat16 whose sum they are, the first and 1 / F32_LOWER of the others.
__device__ __forceinline__ void split8(const float4 lo, const float4 hi, uint4& a, uint4& b, uint4& c) {
    float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    uint32_t p[3][4];
#pragma unroll
    for (int part = 0; part < 3; ++part) {
#pragma unroll
        for (int i = 0; i < 4; ++i)                           // (the last part's cut off halves are not needed: one byte exchange for two)
            p[part][i] = part < 2 ? upper_halves(v[2 * i], v[2 * i + 1])
                                  : __builtin_amdgcn_perm(__float_as_uint(v[2 * i + 1]), __float_as_uint(v[2 * i]), 0x07060302u);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = part == 0 ? below_upper(v[i]) * F32_LOWER : below_upper(v[i]);
    }
    a = make_uint4(p[0][0], p[0][1], p[0][2], p[0][3]);
    b = make_uint4(p[1][0], p[1][1], p[1][2], p[1][3]);
    c = make_uint4(p[2][0], p[2][1], p[2][2], p[2][3]);
}

// A thread's outputs (rows m + 16 i, columns n + 16 j + 0..3) that are no finite numbers, once more by the chain of multiply-adds.
template <int MT, int NT>
__device__ __forceinline__ void chain_again(float* out, const float* x, const bf16_t* w, int m, int n, int M, int N, int K) {
#pragma nounroll
    for (int at = 0; at < MT * NT * 4; ++at) {
        const int mm = m + at / (4 * NT) * 16, nn = n + at / 4 % NT * 16 + at % 4;
        if (mm >= M || nn >= N || fabsf(out[(size_t)mm * N + nn]) < INFINITY) continue;
        float sum = 0.f;
        for (int k = 0; k < K; ++k) sum = fmaf(x[(size_t)mm * K + k], bf16_to_f32(w[(size_t)nn * K + k]), sum);
        out[(size_t)mm * N + nn] = sum;
    }
}

// Tiles of 16 MT rows of x and 16 NT rows of weights a wavefront, WM by WN wavefronts a workgroup, K in stages of 64 through two LDS
// buffers; x is split once, on its way into LDS.  A row of a stage is 128 bytes, its 16-byte pieces exchanged by the row's number so
// that reads of a fragment's sixteen rows meet every bank equally.  What bounds a tile is its chain of stages, each the
// split (half as many cycles of the vector units as the matrix cores take for it), LDS both ways and a barrier: 0.4 us for 32 x 32, 0.8 for
// 64 x 128 with eight wavefronts (0.95 with four).
#define FT_BK 64
// A thread's share of a stage on its way through registers: 16 bytes of bfloat16 (8 k) of rows row + THREADS / 8 i.
template <int XN, int WR, int THREADS>
struct TileStage {
    float4 lo[XN], hi[XN];
    uint4 w[WR];
    __device__ __forceinline__ void fetch(const float* const (&xp)[XN], const bf16_t* const (&wp)[WR], int k) {
#pragma unroll
        for (int i = 0; i < XN; ++i) {
            lo[i] = *reinterpret_cast<const float4*>(xp[i] + k);
            hi[i] = *reinterpret_cast<const float4*>(xp[i] + k + 4);
        }
#pragma unroll
        for (int i = 0; i < WR; ++i) w[i] = *reinterpret_cast<const uint4*>(wp[i] + k);
    }
    __device__ __forceinline__ void store(uint4* xs, uint4* ws, int slot, int plane, uint32_t keep) const {
#pragma unroll
        for (int i = 0; i < XN; ++i) {
            uint4 a, b, c;
            split8(lo[i], hi[i], a, b, c);
            xs[slot + THREADS * i] = make_uint4(a.x & keep, a.y & keep, a.z & keep, a.w & keep);
            xs[plane + slot + THREADS * i] = make_uint4(b.x & keep, b.y & keep, b.z & keep, b.w & keep);
            xs[2 * plane + slot + THREADS * i] = make_uint4(c.x & keep, c.y & keep, c.z & keep, c.w & keep);
        }
#pragma unroll
        for (int i = 0; i < WR; ++i) ws[slot + THREADS * i] = w[i];
    }
};

template <int MT, int NT>
__device__ __forceinline__ void multiply_stage(f32_floatx4 (&acc)[MT][NT][3], const uint4* xs, const uint4* ws, int plane, int wm,
                                               int wn, int r, int g) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        const int at = (ks * 4 + g) ^ (r & 7);
        f32_bf16x8 wf[NT], xf[MT][3];
#pragma unroll
        for (int j = 0; j < NT; ++j) wf[j] = as_bf16x8(ws[(wn + 16 * j + r) * 8 + at]);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < 3; ++q) xf[i][q] = as_bf16x8(xs[q * plane + (wm + 16 * i + r) * 8 + at]);
#pragma unroll
        for (int q = 2; q >= 0; --q)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], xf[i][q], acc[i][j][q], 0, 0, 0);
    }
}

template <int MT, int NT, int WM, int WN, int DEEP, bool FULL>
__global__ void __launch_bounds__(64 * WM * WN, 2)
gemm_f32_tile_kernel(float* __restrict__ out, const float* __restrict__ x, const bf16_t* __restrict__ w, int M, int N, int K,
                     int m_tiles, int n_tiles) {
    constexpr int BM = 16 * MT * WM, BN = 16 * NT * WN, THREADS = 64 * WM * WN, XN = BM * 8 / THREADS, WR = BN * 8 / THREADS, STEP = THREADS / 8;
    __shared__ uint4 xs[2][3 * BM * 8];
    __shared__ uint4 ws[2][BN * 8];
    // workgroups that read the same weights are a multiple of eight apart, so that they meet in one L2 cache
    const int group = blockIdx.x / (8 * m_tiles), within = blockIdx.x % (8 * m_tiles);
    const int nt = group * 8 + within % 8, m0 = within / 8 * BM, n0 = nt * BN;
    if (nt >= n_tiles) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
    const int wm = wave % WM * 16 * MT, wn = wave / WM * 16 * NT;
    const int piece = tid & 7, row = tid >> 3;              // of a stage: 16 bytes of bfloat16 (8 k) of rows row + STEP i
    const float* xp[XN];
    const bf16_t* wp[WR];
#pragma unroll
    for (int i = 0; i < XN; ++i) xp[i] = x + (size_t)min(m0 + row + STEP * i, M - 1) * K;
#pragma unroll
    for (int i = 0; i < WR; ++i) wp[i] = w + (size_t)min(n0 + row + STEP * i, N - 1) * K;
    const int slot = row * 8 + (piece ^ (row & 7));         // (STEP rows on, a multiple of eight, the exchange is the same)
    f32_floatx4 acc[MT][NT][3];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int p = 0; p < 3; ++p) acc[i][j][p] = f32_floatx4{0.f, 0.f, 0.f, 0.f};
    // DEEP stages are under way in registers while another is multiplied: a stage of a small tile is multiplied in a fraction of the
    // time that its loads take.
    TileStage<XN, WR, THREADS> ahead[DEEP];
    const int stages = (K + FT_BK - 1) / FT_BK;
#pragma unroll
    for (int d = 0; d < DEEP; ++d) ahead[d].fetch(xp, wp, min(d * FT_BK + 8 * piece, K - 8));
    ahead[0].store(xs[0], ws[0], slot, BM * 8, FULL || 8 * piece < K ? ~0u : 0u);
    __syncthreads();
    for (int s = 0; s < stages; s += DEEP) {
        const int k = s * FT_BK + 8 * piece;                // (beyond K: x counts as zeros where it is stored)
#pragma unroll
        for (int d = 0; d < DEEP; ++d) {
            ahead[d].fetch(xp, wp, min(k + (d + DEEP) * FT_BK, K - 8));
            multiply_stage<MT, NT>(acc, xs[d & 1], ws[d & 1], BM * 8, wm, wn, r, g);
            ahead[(d + 1) % DEEP].store(xs[(d + 1) & 1], ws[(d + 1) & 1], slot, BM * 8, FULL || k + (d + 1) * FT_BK < K ? ~0u : 0u);
            __syncthreads();
        }
    }
    const bool four = N % 4 == 0;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int m = m0 + wm + 16 * i + r, n = n0 + wn + 16 * j + 4 * g;
            if (m >= M || n >= N) continue;
            float sum[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sum[e] = acc[i][j][0][e] + (acc[i][j][1][e] + acc[i][j][2][e]) * (1.f / F32_LOWER);
                bad |= !(fabsf(sum[e]) < INFINITY);
            }
            float* o = out + (size_t)m * N + n;
            if (four) *reinterpret_cast<float4*>(o) = make_float4(sum[0], sum[1], sum[2], sum[3]);
            else
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) o[e] = sum[e];
        }
    if (bad) chain_again<MT, NT>(out, x, w, m0 + wm + r, n0 + wn + 4 * g, M, N, K);
}

template <int MT, int NT, int WM, int WN, int DEEP>
static void launch_tiles(float* out, const float* x, const bf16_t* w, int m, int n, int k, hipStream_t s) {
    constexpr int BM = 16 * MT * WM, BN = 16 * NT * WN;
    const int m_tiles = (m + BM - 1) / BM, n_tiles = (n + BN - 1) / BN;
    const int grid = (n_tiles + 7) / 8 * 8 * m_tiles;
    if (k % (DEEP * FT_BK) == 0) gemm_f32_tile_kernel<MT, NT, WM, WN, DEEP, true><<<grid, 64 * WM * WN, 0, s>>>(out, x, w, m, n, k, m_tiles, n_tiles);
    else gemm_f32_tile_kernel<MT, NT, WM, WN, DEEP, false><<<grid, 64 * WM * WN, 0, s>>>(out, x, w, m, n, k, m_tiles, n_tiles);
}

// ---- large tiles: x as it is into LDS, split where its fragments are read

// Two floats' share of the split above, in steps of three or four instructions that fit between products.
struct SplitPair {
    float t0, t1;
    __device__ __forceinline__ void step(int u, float& v0, float& v1, uint32_t& a, uint32_t& b, uint32_t& c) {
        if (u == 0 || u == 2) {
            (u == 0 ? a : b) = __builtin_amdgcn_perm(__float_as_uint(v1), __float_as_uint(v0), 0x07060302u);
            t0 = __uint_as_float(__float_as_uint(v0) & 0xFFFF0000u);
            t1 = __uint_as_float(__float_as_uint(v1) & 0xFFFF0000u);
        } else if (u == 1) {
            v0 = (v0 - t0) * F32_LOWER;
            v1 = (v1 - t1) * F32_LOWER;
        } else {
            v0 -= t0;
            v1 -= t1;
            c = __builtin_amdgcn_perm(__float_as_uint(v1), __float_as_uint(v0), 0x07060302u);
        }
    }
};

// Tiles of 16 MT WAVES rows of x and 16 NT of w: a wavefront has 16 MT rows and all columns, so that no row is split twice and none of its parts
// written.  K in stages of 64 through SLOTS buffers, filled by copies that do not pass through registers and go out SLOTS - LAG stages ahead: two
// (three buffers), three (five) or four (six).
// The split, the reads and the copies stand between the products, three or four instructions each.  What bounds a large tile is then the matrix
// cores at the clock that they leave (128 x 160: 1,920 cycles of products a stage, 1.19 us; 759 rows, 6,144 x 1,024: 48 -> 33 us; 128 x 128,
// 4,096 x 1,024: 30 -> 23), the smallest the instructions it issues, half of them the split (64 x 64: 0.46 us a stage; 1,024 x 3,072: 31 -> 27).
// The order of every sum is the one of the tiles above, to the bit.
template <int MT, int NT, int WAVES, int SLOTS>
__global__ void __launch_bounds__(64 * WAVES, WAVES / 4)
gemm_f32_copied_kernel(float* __restrict__ out, const float* __restrict__ x, const bf16_t* __restrict__ w, int M, int N, int K,
                       int m_tiles, int n_tiles) {
    constexpr int BM = 16 * MT * WAVES, BN = 16 * NT, XC = 4 * MT, WC = 2 * NT / WAVES, FR = XC + WC, STAGE = BM * 16 + BN * 8;
    constexpr int EACH = 3 * MT, P = EACH * NT, LAG = SLOTS > 4 ? 2 : 1, MEET = EACH * (3 - LAG) - 1, SPLITS = 16 * MT, READ0 = P <= 24 ? 0 : P / 3,
                  GAP = (P - 1 - READ0) / FR;
    static_assert(2 * NT % WAVES == 0 && GAP >= 1 && SLOTS > 2 && (SLOTS - 2) * FR <= 63, "a stage's copies go out within half a stage");
    __shared__ uint4 lds[SLOTS * STAGE];
    const int group = blockIdx.x / (8 * m_tiles), within = blockIdx.x % (8 * m_tiles);
    const int nt = group * 8 + within % 8, m0 = within / 8 * BM, n0 = nt * BN;
    if (nt >= n_tiles) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const int stages = K / 64;

    // A copy of a wavefront fills four rows of x or eight of w.  Rows past the edge are the last row again.
    uint32_t xo[XC], wo[WC];
#pragma unroll
    for (int j = 0; j < XC; ++j) {
        const int row = 4 * j + (lane >> 4);
        xo[j] = (uint32_t)min(wave * 16 * MT + row, M - 1 - m0) * (uint32_t)K * 4u + ((lane & 15) ^ (row & 15)) * 16;
    }
#pragma unroll
    for (int j = 0; j < WC; ++j) {
        const int row = lane >> 3;
        wo[j] = (uint32_t)min(wave * 8 * WC + 8 * j + row, N - 1 - n0) * (uint32_t)K * 2u + ((lane & 7) ^ row) * 16;
    }
    const float* xa = x + (size_t)m0 * K;
    const bf16_t* wa = w + (size_t)n0 * K;
    const ma_lds_t x_at = ma_lds(lds + wave * 16 * MT * 16), w_at = ma_lds(lds + BM * 16 + wave * 64 * WC);
    auto copy = [&](int e, int buf, size_t k) {
        if (e < WC) ma_copy16(w_at + buf * STAGE * 16 + e * 1024, wo[e], wa + k);
        else ma_copy16(x_at + buf * STAGE * 16 + (e - WC) * 1024, xo[e - WC], xa + k);
    };
#pragma unroll
    for (int s = 0; s < SLOTS - LAG; ++s)
#pragma unroll
        for (int e = 0; e < FR; ++e) copy(e, s, (size_t)min(s, stages - 1) * 64);

    ma_floatx4 acc[MT][NT][3];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int q = 0; q < 3; ++q) acc[i][j][q] = ma_floatx4{0.f, 0.f, 0.f, 0.f};
    const float4* xr = reinterpret_cast<const float4*>(lds) + (wave * 16 * MT + r) * 16;
    const uint4* wr = lds + BM * 16 + r * 8;
    float raw[2][MT][8];
    uint32_t xf[2][MT][3][4];
    ma_bf16x8 wf[NT];
    SplitPair pair;
    auto read_x = [&](int to, int buf) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float4 v = xr[buf * STAGE + i * 256 + ((to * 8 + 2 * g + h) ^ r)];
                raw[to][i][4 * h] = v.x, raw[to][i][4 * h + 1] = v.y, raw[to][i][4 * h + 2] = v.z, raw[to][i][4 * h + 3] = v.w;
            }
    };
    auto read_w = [&](int j, int to, int buf) { wf[j] = *reinterpret_cast<const ma_bf16x8*>(wr + buf * STAGE + j * 128 + ((to * 4 + g) ^ (r & 7))); };
    auto split = [&](int t, int to) {
        const int i = t / 16, at = t % 16 / 4;
        pair.step(t % 4, raw[to][i][2 * at], raw[to][i][2 * at + 1], xf[to][i][0][at], xf[to][i][1][at], xf[to][i][2][at]);
    };
    ma_wait_copies<(SLOTS - LAG - 1) * FR>();
    ma_meet();
    read_x(0, 0);
    read_x(1, 0);
#pragma unroll
    for (int j = 0; j < NT; ++j) read_w(j, 0, 0);
#pragma unroll
    for (int t = 0; t < SPLITS; ++t) split(t, 0);

    // Products of half a stage; under them the next half's x is split in steps, that of the half after it read (a wavefront's own copies), and
    // the next half's fragments of w, each where this half's has been used.
    auto half = [&](auto which, int buf, int next, int free, size_t k) {
        constexpr int H = decltype(which)::value, READ = H ? 0 : READ0;
        ma_wait_written();
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int j = p / EACH, i = p % EACH / 3, q = 2 - p % 3;
            ma_product(acc[i][j][q], wf[j], *reinterpret_cast<const ma_bf16x8*>(xf[H][i][q]));
            if (p == READ) {
                if (!H) ma_wait_copies<(SLOTS - LAG - 2) * FR>();
                read_x(H, next);
            }
            if (H && p == MEET) {
                if (LAG == 1) ma_wait_lds();
                ma_meet();
#pragma unroll
                for (int before = 0; before < j; ++before) read_w(before, 0, next);
            }
            if (p % EACH == EACH - 1 && (!H || p >= MEET)) read_w(j, 1 - H, H ? next : buf);
            if (!H && p > READ && (p - READ) % GAP == 0 && (p - READ) / GAP <= FR) copy((p - READ) / GAP - 1, free, k);
#pragma unroll
            for (int c = 0; c < (SPLITS + P - 2) / (P - 1); ++c) {
                const int t = p * SPLITS / (P - 1) + c;
                if (p < P - 1 && t < (p + 1) * SPLITS / (P - 1)) split(t, 1 - H);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int buf = 0, free = SLOTS - LAG;
#pragma nounroll
    for (int s = 0; s < stages; ++s) {
        const int next = buf + 1 == SLOTS ? 0 : buf + 1;
        half(std::integral_constant<int, 0>(), buf, next, free, (size_t)min(s - LAG + SLOTS, stages - 1) * 64);
        half(std::integral_constant<int, 1>(), buf, next, free, 0);
        buf = next;
        free = free + 1 == SLOTS ? 0 : free + 1;
    }
    ma_wait_products();
    bool bad = false;
    const int m = m0 + wave * 16 * MT + r, n = n0 + 4 * g;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            float sum[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                sum[e] = ma_taken(acc[i][j][0][e]) + (ma_taken(acc[i][j][1][e]) + ma_taken(acc[i][j][2][e])) * (1.f / F32_LOWER);
            if (m + 16 * i >= M || n + 16 * j >= N) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e) bad |= !(fabsf(sum[e]) < INFINITY);
            *reinterpret_cast<float4*>(out + (size_t)(m + 16 * i) * N + n + 16 * j) = make_float4(sum[0], sum[1], sum[2], sum[3]);
        }
    ma_wait_copies<0>();
    if (bad) chain_again<MT, NT>(out, x, w, m, n, M, N, K);
}

template <int MT, int NT, int WAVES, int SLOTS>
static void launch_copied(float* out, const float* x, const bf16_t* w, int m, int n, int k, hipStream_t s) {
    constexpr int BM = 16 * MT * WAVES;
    const int m_tiles = (m + BM - 1) / BM, n_tiles = (n + 16 * NT - 1) / (16 * NT);
    gemm_f32_copied_kernel<MT, NT, WAVES, SLOTS><<<(n_tiles + 7) / 8 * 8 * m_tiles, 64 * WAVES, 0, s>>>(out, x, w, m, n, k, m_tiles, n_tiles);
}

#define GT_M 64
#define GT_N 64
#define GT_K 16

template <typename TW>
__global__ void __launch_bounds__(256)
gemm_f32_kernel(float* __restrict__ out, const float* __restrict__ x, const TW* __restrict__ w, int M, int N, int K) {
    __shared__ float xs[GT_K][GT_M + 4];
    __shared__ float ws[GT_K][GT_N + 4];
    const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
    const int m0 = blockIdx.y * GT_M, n0 = blockIdx.x * GT_N;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += GT_K) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = tid + i * 256, r = e / GT_K, kk = e % GT_K;
            const int k = k0 + kk;
            xs[kk][r] = (m0 + r < M && k < K) ? x[(size_t)(m0 + r) * K + k] : 0.f;
            ws[kk][r] = (n0 + r < N && k < K) ? to_f32(w[(size_t)(n0 + r) * K + k]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < GT_K; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) { a[i] = xs[kk][ty * 4 + i]; b[i] = ws[kk][tx * 4 + i]; }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int m = m0 + ty * 4 + i, n = n0 + tx * 4 + j;
            if (m < M && n < N) out[(size_t)m * N + n] = acc[i][j];
        }
}

extern "C" int ri_gemm_f32(float* out, const float* x, const void* w, int w_dtype, int m, int n, int k, int tile, void* stream) {
    RI_REQUIRE(m > 0 && n > 0 && k > 0, "gemm_f32: m %d, n %d, k %d", m, n, k);
    RI_REQUIRE(w_dtype == RI_F32 || w_dtype == RI_BF16, "gemm_f32: weight dtype %d", w_dtype);
    dim3 grid((n + GT_N - 1) / GT_N, (m + GT_M - 1) / GT_M);
    RI_REQUIRE(grid.y <= 65535, "gemm_f32: %d rows exceed one launch", m);
    hipStream_t s = (hipStream_t)stream;
    const bool aligned = k % 8 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0 && (uintptr_t)out % 16 == 0;
    if (w_dtype == RI_F32)
        gemm_f32_kernel<float><<<grid, 256, 0, s>>>(out, x, (const float*)w, m, n, k);
    else if (!aligned)
        gemm_f32_kernel<bf16_t><<<grid, 256, 0, s>>>(out, x, (const bf16_t*)w, m, n, k);
    else {
        // The order of a row's sums is the same in every tile.  Without copies (K off a multiple of 64) 64 x 128 from three quarters of the
        // machine on (one workgroup a compute unit), else 32 x 64 as soon as 32 x 32 would need a second round.  us for 32 x 32 / 32 x 64 /
        // 64 x 128 (rows; columns x K): 759; 6,144 x 1,024 72 / 47 / 49, 4,096 x 1,024 47 / 31 / 30, 1,024 x 3,072 36 / 31 / 46; 1,200; 6,144 x
        // 1,024 115 / 77 / 63; 400; 4,096 x 1,024 27 / 21 / 18; 200; 4,096 x 1,024 17 / 12.5 / 17; 1,000; 12,288 x 4,096 844 / 453 / 320; 33;
        // 4,096 x 1,024 8.5 / 9.4 / 16 (the vector units' form: 759; 1,024 x 3,072 363).
        // Up to 32 rows half of a tile of 64 would be padding: 151,936 x 1,024 at one row 77 / 57 / 75.
        const auto tiles = [&](int rows, int cols) { return (long)((m + rows - 1) / rows) * ((n + cols - 1) / cols); };
        const bf16_t* wb = (const bf16_t*)w;
        RI_REQUIRE(tiles(32, 32) + 8 * ((m + 31) / 32) < (1L << 31), "gemm_f32: %d x %d exceed one launch", m, n);
        const bool copied = k % 64 == 0 && n % 4 == 0 && k < (1 << 22);
        RI_REQUIRE(tile >= -1 && tile <= (copied ? 6 : 2), "gemm_f32: tile %d for %d columns, K %d", tile, n, k);
        const long units = ri_compute_units();
        if (tile < 0) {
            tile = m > 32 && 4 * tiles(64, 128) >= 3 * units ? 0 : tiles(32, 32) > units ? 1 : 2;
            if (copied && m > 32) {
                // With copies what a tile takes is its rounds times (a beginning and an end + its stages), in us; the smaller tiles above share
                // a compute unit instead.  Measured, in the order 128 x 160 / 128 x 128 / 64 x 128 / 64 x 64 and the best of those above: 759; 6,144 x
                // 1,024 33 / 43 / 42 / 51, 47; 759; 4,096 x 1,024 29 / 23 / 28 / 31, 30; 759; 1,024 x 3,072 63 / 49 / 34 / 27, 31; 1,200; 6,144 x
                // 1,024 58 / 49 / 60 / 84, 62; 1,200; 1,024 x 3,072 63 / 48 / 34 / 51, 42; 400; 4,096 x 1,024 26 / 20 / 15 / 21, 18; 400; 1,024 x
                // 3,072 63 / 48 / 33 / 26, 23; 100; 6,144 x 1,024 25 / 19 / 14 / 11.2, 13; 50; 6,144 x 1,024 25 / 18 / 13 / 10.5, 9.6; 1,000;
                // 12,288 x 4,096 274 / 248 / 293 / 407, 312; 2,400; 6,144 x 1,024 91 / 100 / 119 / 153, 121.
                static const struct { int rows, cols; double ends, stage; } form[4] = {{128, 160, 13, 1.19}, {128, 128, 9, 0.9}, {64, 128, 5, 0.61}, {64, 64, 4, 0.46}};
                const double stages = k / 64, load = tiles(32, 64) / (double)units;
                double best = tile == 2 ? 1.5 + 0.37 * stages : tile == 1 ? 2. + stages * (0.25 + 0.25 * (load > 0.8 ? load : 0.8)) : 1e30;
                for (int i = 0; i < 4; ++i) {
                    // (the eight L2 caches' columns are dealt out as the kernel does)
                    const long own = (((n + form[i].cols - 1) / form[i].cols + 7) / 8) * (long)((m + form[i].rows - 1) / form[i].rows), room = units > 8 ? units / 8 : 1;
                    const double takes = (own + room - 1) / room * (form[i].ends + form[i].stage * stages);
                    if (takes < best) best = takes, tile = 3 + i;
                }
            }
        }
        switch (tile) {
        case 0: launch_tiles<2, 2, 2, 4, 2>(out, x, wb, m, n, k, s); break;
        case 1: launch_tiles<1, 2, 2, 2, 2>(out, x, wb, m, n, k, s); break;
        case 2: launch_tiles<1, 1, 2, 2, 4>(out, x, wb, m, n, k, s); break;
        case 3: launch_copied<2, 10, 4, 3>(out, x, wb, m, n, k, s); break;
        case 4: launch_copied<1, 8, 8, 3>(out, x, wb, m, n, k, s); break;
        case 5: launch_copied<1, 8, 4, 5>(out, x, wb, m, n, k, s); break;
        case 6: launch_copied<1, 4, 4, 6>(out, x, wb, m, n, k, s); break;
        }
    }
    RI_LAUNCH_CHECK("gemm_f32");
    return 0;
}
