// The windowed attention whose heads talk, on the matrix cores, for prompts in bfloat16.
//
// The mixing of the heads' weights needs every head's finished softmax, so the keys are walked twice, as in the general
// kernels (talking_attention.hip), with tiles of 16 tokens of a sequence as the 16 columns of the matrix cores' tiles:
//   talking_stats_mfma:  a wavefront per (tile of tokens, head, or four heads of a key head): S^T = K Q^T page by page, the distance bias, the window's
//                        mask, and each column's running maximum and sum;
//   talking_mix_mfma:    a workgroup of eight wavefronts per tile of tokens, each wavefront on an eighth of the heads:
//                        for a page it makes its heads' weights exp(s - m) / l from the first walk's numbers and leaves
//                        them in LDS (float32); after a barrier it mixes, for each of its heads, the weights of all
//                        heads (w'_h = sum_g T[h, g] w_g, on the vector units), rounds the mix to bfloat16 and adds
//                        O^T += V^T W'^T with the values of the head's own key head.
// The key rows of a half page are permuted (row r of the first half is key 8 (r / 4) + r % 4, of the second that plus
// 4), so that a lane's eight scores are eight neighbouring keys, which is how the value product wants its weights.
// Scores, the logarithm, maxima, sums, the weights before and after the mix and the accumulators are float32.  A token's
// sums run over its sequence's pages in order, or over equal parts of them that are added: into how many depends on the step's tiles
// and its longest sequence, so that in bfloat16 the rest of a step may move a token's result by the rounding of its float32 sums.
//
// The distance bias of a windowed head is a number a distance: a table of window + 16 entries a head is made first, by the
// same logarithm, and both walks read eight neighbouring entries of it for their eight keys (a logarithm a score was half
// of what the walks took).  The second walk of a step with fewer tiles than compute units cuts every tile's pages into
// shares, whose float32 results are added.  2,048 tokens, 32 heads of 128 over 8, a window of 1,024, us: first walk 283 ->
// 136, second 950 -> 394 with the adding, and 101 and 246 since a key head's loads serve all of its heads in a wavefront.
#include "api.h"
#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 tm_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float tm_floatx4;

union TmFrag {
    tm_bf16x8 v;
    uint4 u;
    uint32_t w[4];
};

#define TM_PAGE 32
#define TM_TILE 16           // tokens of a tile
#define TM_WAVES 8           // wavefronts of the second walk's workgroup

// Which tile of which sequence a workgroup takes: tiles are counted sequence after sequence.  Returns false past the last.
__device__ __forceinline__ bool tile_of(int index, const int32_t* __restrict__ cu_seqlens, int seqs, int& seq, int& first,
                                        int& count) {
    for (int s = 0; s < seqs; ++s) {
        const int n = cu_seqlens[s + 1] - cu_seqlens[s];
        const int tiles = (n + TM_TILE - 1) / TM_TILE;
        if (index < tiles) {
            seq = s;
            first = cu_seqlens[s] + index * TM_TILE;
            count = min(TM_TILE, cu_seqlens[s + 1] - first);
            return true;
        }
        index -= tiles;
    }
    return false;
}

// table[h][8 + gap] = r1_h log(1 + r2_h gap) for gaps -8 .. window + 7 (those outside 0 .. window - 1 are read and not used).
__global__ void __launch_bounds__(256)
talking_bias_kernel(float* __restrict__ table, const float* __restrict__ r1, const float* __restrict__ r2, int heads, int window) {
    const int e = blockIdx.x * 256 + threadIdx.x, span = window + 16;
    if (e >= heads * span) return;
    const int h = e / span;
    table[e] = r1[h] * log1pf(r2[h] * (float)max(e % span - 8, 0));
}

struct __attribute__((packed, aligned(4))) TmEight { float v[8]; };

// A lane's fragments of a page's keys (both half pages).
template <int KS>
__device__ __forceinline__ void talking_keys(TmFrag (&k0)[KS], TmFrag (&k1)[KS], const bf16_t* __restrict__ kp) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        k0[ks].u = *reinterpret_cast<const uint4*>(kp + ks * 32);
        k1[ks].u = *reinterpret_cast<const uint4*>(kp + 4 * 32 * KS + ks * 32);
    }
}
// The biases of the gaps from the last of the lane's eight keys up to the first's; `bias` is the head's row of the table of distances, its
// entry for a gap of 0.
__device__ __forceinline__ TmEight talking_gaps(const float* __restrict__ bias, int qpos, int key0, int window) {
    return *reinterpret_cast<const TmEight*>(bias + min(max(qpos - key0 - 7, -8), window));
}

// The eight scores of a lane (column = token, keys key0 .. key0 + 7) of a head for one page: raw products times the scale,
// minus the distance bias, minus infinity where the token does not see the key.
template <int KS, bool TABLE>
__device__ __forceinline__ void talking_scores(float (&s)[8], const TmFrag (&qf)[KS], const TmFrag (&k0)[KS], const TmFrag (&k1)[KS],
                                               const TmEight& by_gap, float scale, float b1, float b2, bool biased, int qpos, int lo, int key0) {
    tm_floatx4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0[ks].v, qf[ks].v, s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1[ks].v, qf[ks].v, s1, 0, 0, 0);
    }
    const float raw[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int key = key0 + e;
        float v = raw[e] * scale;
        if (TABLE) v -= by_gap.v[7 - e];
        else if (biased) v -= b1 * log1pf(b2 * (float)max(qpos - key, 0));
        s[e] = (key > qpos || key < lo) ? -INFINITY : v;
    }
}

// HG: query heads of one key head that a wavefront takes: a page's keys are loaded once for all of them, the next page's while
// these are weighed.  A wavefront a head is bound by the caches (every key row 32 times over): 2,048 tokens, 32 heads over 8 of 128, a
// window of 1,024 133 us, 101 with four heads.
template <int KS, int HG, bool TABLE>
__global__ void __launch_bounds__(64)
talking_stats_mfma_kernel(float* __restrict__ stats, const bf16_t* __restrict__ q, int q_stride, int q_off,
                          const bf16_t* __restrict__ k_pages, const int32_t* __restrict__ tok_pos,
                          const int32_t* __restrict__ cu_seqlens, int seqs, const int32_t* __restrict__ page_table,
                          int table_width, int heads, int kv_heads, int window, float scale, const float* __restrict__ r1,
                          const float* __restrict__ r2, const float* __restrict__ bias) {
    constexpr int DIM = 32 * KS;
    int seq, first, count;
    if (!tile_of(blockIdx.x, cu_seqlens, seqs, seq, first, count)) return;
    const int h0 = blockIdx.y * HG, lane = threadIdx.x;
    const int col = lane & 15, g = lane >> 4;
    const int t = first + min(col, count - 1);                 // a column pulled back inside the tile: loads are issued anyway
    const int qpos = tok_pos[t];
    const int lo = window > 0 ? max(0, qpos - window + 1) : 0;
    const int kvh = h0 / (heads / kv_heads);
    const int32_t* table = page_table + (size_t)seq * table_width;
    const bool biased = r1 != nullptr;
    TmFrag qf[HG][KS], k0[KS], k1[KS];
    float b1[HG], b2[HG], m[HG], l[HG];
#pragma unroll
    for (int i = 0; i < HG; ++i) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            qf[i][ks].u = *reinterpret_cast<const uint4*>(q + (size_t)t * q_stride + q_off + (size_t)(h0 + i) * DIM + ks * 32 + 8 * g);
        b1[i] = biased ? r1[h0 + i] : 0.f;
        b2[i] = biased ? r2[h0 + i] : 0.f;
        m[i] = -INFINITY;
        l[i] = 0.f;
    }
    const int pos_first = tok_pos[first], pos_last = pos_first + count - 1;
    const int lo_first = window > 0 ? max(0, pos_first - window + 1) : 0;
    const int key_row = 8 * (col >> 2) + (col & 3);
    const auto keys_of = [&](int page) { return k_pages + (((long)table[page] * kv_heads + kvh) * TM_PAGE + key_row) * (long)DIM + 8 * g; };
    const int page_last = pos_last / TM_PAGE;
    talking_keys<KS>(k0, k1, keys_of(lo_first / TM_PAGE));
    for (int page = lo_first / TM_PAGE; page <= page_last; ++page) {
        const int key0 = page * TM_PAGE + 8 * g;
        const bf16_t* next = keys_of(min(page + 1, page_last));
        TmEight gaps[HG];
        float s[HG][8];
#pragma unroll
        for (int i = 0; i < HG; ++i)
            if (TABLE) gaps[i] = talking_gaps(bias + (size_t)(h0 + i) * (window + 16) + 8, qpos, key0, window);
#pragma unroll
        for (int i = 0; i < HG; ++i) talking_scores<KS, TABLE>(s[i], qf[i], k0, k1, gaps[i], scale, b1[i], b2[i], biased, qpos, lo, key0);
        __builtin_amdgcn_sched_barrier(0);
        talking_keys<KS>(k0, k1, next);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < HG; ++i) {
            float mx = fmaxf(fmaxf(fmaxf(s[i][0], s[i][1]), fmaxf(s[i][2], s[i][3])), fmaxf(fmaxf(s[i][4], s[i][5]), fmaxf(s[i][6], s[i][7])));
            mx = fmaxf(mx, __shfl_xor(mx, 16, RI_WAVE));
            mx = fmaxf(mx, __shfl_xor(mx, 32, RI_WAVE));
            const float m_new = fmaxf(m[i], mx);
            const float m_safe = m_new == -INFINITY ? 0.f : m_new;  // a column that has seen no key yet
            float sum = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) sum += expf(s[i][e] - m_safe);
            l[i] = l[i] * expf(m[i] - m_safe) + sum;                 // the factor is 0 while m is -inf
            m[i] = m_new;
        }
    }
#pragma unroll
    for (int i = 0; i < HG; ++i) {
        l[i] += __shfl_xor(l[i], 16, RI_WAVE);
        l[i] += __shfl_xor(l[i], 32, RI_WAVE);
        if (g == 0 && col < count) {
            stats[((size_t)t * heads + h0 + i) * 2] = m[i];
            stats[((size_t)t * heads + h0 + i) * 2 + 1] = l[i];
        }
    }
}

#define TM_ROW (TM_PAGE + 4)  // of a token's weights in LDS: sixteen tokens' pieces meet every bank equally
// ONE: a wavefront's heads read one key head, whose keys and values a page it then loads once instead of once a head.  What bounds a page
// is a chain of trips to memory (keys, queries a head, values) and the mix between them, two wavefronts a SIMD.  Both walks, 32 heads over 8
// of 128, a window of 1,024, us keys and values a head and tokens' rows of 32 in LDS : this: 2,048 tokens 511 : 327 (this walk 370 : 221 in a
// model's step), 1,024 259 : 195, 256 76 : 59, 17 40 : 33; 16 heads 223 : 166, 119 : 97, 41 : 33, 22 : 18.
template <int KS, int HPW, bool TABLE, bool ONE>
__global__ void __launch_bounds__(64 * TM_WAVES)
talking_mix_mfma_kernel(bf16_t* __restrict__ out, float* __restrict__ parts, size_t part_stride, const float* __restrict__ stats, const bf16_t* __restrict__ q, int q_stride,
                        int q_off, const bf16_t* __restrict__ k_pages, const bf16_t* __restrict__ v_pages,
                        const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ cu_seqlens, int seqs,
                        const int32_t* __restrict__ page_table, int table_width, int kv_heads, int window, float scale,
                        const float* __restrict__ r1, const float* __restrict__ r2, const float* __restrict__ talk,
                        const float* __restrict__ bias) {
    constexpr int DIM = 32 * KS, VT = DIM / 16, HEADS = HPW * TM_WAVES;
    extern __shared__ float lds[];
    float* ps = lds;                                           // [HEADS][TM_TILE][TM_ROW] the heads' weights of a page
    float* tk = ps + HEADS * TM_TILE * TM_ROW;                 // [HEADS][HEADS] the mixing matrix, transposed
    int seq, first, count;
    if (!tile_of(blockIdx.x, cu_seqlens, seqs, seq, first, count)) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 15, g = lane >> 4;
    const int t = first + min(col, count - 1);
    const int qpos = tok_pos[t];
    const int lo = window > 0 ? max(0, qpos - window + 1) : 0;
    const int share = HEADS / kv_heads;
    const int32_t* table = page_table + (size_t)seq * table_width;
    for (int e = threadIdx.x; e < HEADS * HEADS; e += 64 * TM_WAVES) tk[e % HEADS * HEADS + e / HEADS] = talk ? talk[e] : (e / HEADS == e % HEADS ? 1.f : 0.f);
    const bool biased = r1 != nullptr;
    float ms[HPW], inv_l[HPW], b1[HPW], b2[HPW];
#pragma unroll
    for (int i = 0; i < HPW; ++i) {
        const int h = wave * HPW + i;
        ms[i] = stats[((size_t)t * HEADS + h) * 2];
        inv_l[i] = 1.0f / stats[((size_t)t * HEADS + h) * 2 + 1];
        b1[i] = biased ? r1[h] : 0.f;
        b2[i] = biased ? r2[h] : 0.f;
    }
    tm_floatx4 o[HPW][VT];
#pragma unroll
    for (int i = 0; i < HPW; ++i)
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) o[i][vt] = tm_floatx4{0.f, 0.f, 0.f, 0.f};
    const int pos_first = tok_pos[first], pos_last = pos_first + count - 1;
    const int lo_first = window > 0 ? max(0, pos_first - window + 1) : 0;
    const int key_row = 8 * (col >> 2) + (col & 3);
    // (a share of the pages: workgroup y of gridDim.y)
    const int page0 = lo_first / TM_PAGE, pages = pos_last / TM_PAGE + 1 - page0;
    const int page_first = page0 + (int)((long)pages * blockIdx.y / gridDim.y), page_end = page0 + (int)((long)pages * (blockIdx.y + 1) / gridDim.y);
    __syncthreads();
    for (int page = page_first; page < page_end; ++page) {
        const long phys = table[page];
        // this wavefront's heads: their weights of the page, into LDS
        // (queries are fetched again a page, a head ahead where the sums leave registers for it)
        constexpr bool AHEAD = HPW * VT < 32;
        TmFrag k0[KS], k1[KS], qf[AHEAD ? 2 : 1][KS];
        TmEight gaps[AHEAD ? 2 : 1];
        const auto fetch = [&](int i) {
            const int h = wave * HPW + i;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                qf[AHEAD ? i & 1 : 0][ks].u = *reinterpret_cast<const uint4*>(q + (size_t)t * q_stride + q_off + (size_t)h * DIM + ks * 32 + 8 * g);
            if (TABLE) gaps[AHEAD ? i & 1 : 0] = talking_gaps(bias + (size_t)h * (window + 16) + 8, qpos, page * TM_PAGE + 8 * g, window);
        };
        const auto keys_of = [&](int h) { return k_pages + ((phys * kv_heads + h / share) * TM_PAGE + key_row) * (long)DIM + 8 * g; };
        if (ONE) talking_keys<KS>(k0, k1, keys_of(wave * HPW));
        if (AHEAD) fetch(0);
#pragma unroll
        for (int i = 0; i < HPW; ++i) {
            const int h = wave * HPW + i;
            if (!ONE) talking_keys<KS>(k0, k1, keys_of(h));
            if (!AHEAD) fetch(i);
            else if (i + 1 < HPW) fetch(i + 1);
            __builtin_amdgcn_sched_barrier(0);
            float s[8];
            talking_scores<KS, TABLE>(s, qf[AHEAD ? i & 1 : 0], k0, k1, gaps[AHEAD ? i & 1 : 0], scale, b1[i], b2[i], biased, qpos, lo, page * TM_PAGE + 8 * g);
            float4 lo4, hi4;
            lo4.x = expf(s[0] - ms[i]) * inv_l[i]; lo4.y = expf(s[1] - ms[i]) * inv_l[i];
            lo4.z = expf(s[2] - ms[i]) * inv_l[i]; lo4.w = expf(s[3] - ms[i]) * inv_l[i];
            hi4.x = expf(s[4] - ms[i]) * inv_l[i]; hi4.y = expf(s[5] - ms[i]) * inv_l[i];
            hi4.z = expf(s[6] - ms[i]) * inv_l[i]; hi4.w = expf(s[7] - ms[i]) * inv_l[i];
            float* pp = ps + (h * TM_TILE + col) * TM_ROW + 8 * g;
            *reinterpret_cast<float4*>(pp) = lo4;
            *reinterpret_cast<float4*>(pp + 4) = hi4;
            __builtin_amdgcn_sched_barrier(0);                 // (a head at a time: the registers are the sums')
        }
        const auto values_of = [&](TmFrag (&vf)[VT], int h) {
            const bf16_t* vp = v_pages + ((phys * kv_heads + h / share) * (long)DIM + col) * TM_PAGE + 8 * g;
#pragma unroll
            for (int vt = 0; vt < VT; ++vt) vf[vt].u = *reinterpret_cast<const uint4*>(vp + (long)vt * 16 * TM_PAGE);
        };
        TmFrag vf[VT];
        if (ONE && AHEAD) values_of(vf, wave * HPW);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        // the mix for this wavefront's heads, then their value products; a head's values are asked for together (left to itself
        // the compiler waits for every single load)
        TmFrag p[HPW];
        float mixed[HPW][8];
#pragma unroll
        for (int i = 0; i < HPW; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) mixed[i][e] = 0.f;
        for (int gh = 0; gh < HEADS; ++gh) {
            const float* pp = ps + (gh * TM_TILE + col) * TM_ROW + 8 * g;
            const float4 a = *reinterpret_cast<const float4*>(pp), b = *reinterpret_cast<const float4*>(pp + 4);
            const float w8[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < HPW; ++i) {
                const float c = tk[gh * HEADS + wave * HPW + i];
#pragma unroll
                for (int e = 0; e < 8; ++e) mixed[i][e] += c * w8[e];
            }
        }
#pragma unroll
        for (int i = 0; i < HPW; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) p[i].w[e] = pack_bf16x2(mixed[i][2 * e], mixed[i][2 * e + 1]);
#pragma unroll
        for (int i = 0; i < HPW; ++i) {
            if (!ONE || (!AHEAD && i == 0)) values_of(vf, wave * HPW + i);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int vt = 0; vt < VT; ++vt)
                o[i][vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[vt].v, p[i].v, o[i][vt], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();                                       // before the next page's weights overwrite these
    }
    if (col < count) {
#pragma unroll
        for (int i = 0; i < HPW; ++i) {
            if (parts) {
                float* fp = parts + blockIdx.y * part_stride + (size_t)t * HEADS * DIM + (size_t)(wave * HPW + i) * DIM + 4 * g;
#pragma unroll
                for (int vt = 0; vt < VT; ++vt) *reinterpret_cast<tm_floatx4*>(fp + vt * 16) = o[i][vt];
                continue;
            }
            bf16_t* op = out + (size_t)t * HEADS * DIM + (size_t)(wave * HPW + i) * DIM + 4 * g;
#pragma unroll
            for (int vt = 0; vt < VT; ++vt) {
                uint2 w;
                w.x = pack_bf16x2(o[i][vt][0], o[i][vt][1]);
                w.y = pack_bf16x2(o[i][vt][2], o[i][vt][3]);
                *reinterpret_cast<uint2*>(op + vt * 16) = w;
            }
        }
    }
}

extern "C" int ri_talking_attention_mfma_fits(int heads, int kv_heads, int dim, int page_size) {
    return page_size == TM_PAGE && (dim == 32 || dim == 64 || dim == 128) && heads % TM_WAVES == 0 && heads / TM_WAVES <= 4 &&
           kv_heads >= 1 && heads % kv_heads == 0;
}

// out [tokens, heads * dim] bfloat16; stats: float32 workspace [tokens][heads][2]; bias: float32 workspace [heads][window + 16], used where
// there is a window and a bias (NULL: the logarithm a score); parts: with shares > 1, float32 [shares][tokens][heads * dim], whose sum is the
// result (out is then not written); tiles: an upper bound on the tiles of
// 16 tokens that the sequences' new tokens make (every sequence's count rounded up).
extern "C" int ri_talking_attention_mfma(void* out, float* stats, const void* q, int q_stride, int q_off, const void* k_pages,
                                         const void* v_pages, const int32_t* tok_pos, const int32_t* cu_seqlens, int seqs,
                                         const int32_t* page_table, int table_width, int tiles, int heads, int kv_heads, int dim,
                                         int page_size, int window, float scale, const float* r1, const float* r2,
                                         const float* talk, float* bias, float* parts, int shares, int tokens, void* stream) {
    RI_REQUIRE(shares >= 1 && shares <= 65535 && tokens > 0 && (shares == 1 || (parts && (uintptr_t)parts % 16 == 0)),
               "talking_attention_mfma: %d shares of %d tokens", shares, tokens);
    RI_REQUIRE(seqs > 0 && tiles > 0 && ri_talking_attention_mfma_fits(heads, kv_heads, dim, page_size),
               "talking_attention_mfma: %d sequences, %d heads over %d of %d, pages of %d", seqs, heads, kv_heads, dim, page_size);
    RI_REQUIRE(q_off >= 0 && q_off + heads * dim <= q_stride && q_stride % 8 == 0 && q_off % 8 == 0 && (uintptr_t)q % 16 == 0 &&
               (uintptr_t)k_pages % 16 == 0 && (uintptr_t)v_pages % 16 == 0 && (uintptr_t)out % 8 == 0,
               "talking_attention_mfma: column %d of rows of %d, or a buffer that is not aligned", q_off, q_stride);
    RI_REQUIRE((r1 == nullptr) == (r2 == nullptr) && window >= 0 && table_width > 0 && stats, "talking_attention_mfma: arguments");
    const size_t lds = ((size_t)heads * TM_TILE * TM_ROW + (size_t)heads * heads) * sizeof(float);
    RI_REQUIRE(lds <= 80 * 1024, "talking_attention_mfma: %d heads need %zu bytes of LDS", heads, lds);
    hipStream_t s = (hipStream_t)stream;
    const int hpw = heads / TM_WAVES;
    const bool table = bias && r1 && window > 0;
    if (table) {
        RI_REQUIRE((long)heads * (window + 16) < (1L << 30), "talking_attention_mfma: a window of %d", window);
        talking_bias_kernel<<<(heads * (window + 16) + 255) / 256, 256, 0, s>>>(bias, r1, r2, heads, window);
    }
    if (shares == 1) parts = nullptr;
    // (four heads a wavefront from as many wavefronts on as half of the machine's SIMDs; a wavefront's heads read one key head)
    const int of_kv = heads / kv_heads;
    const bool four = of_kv % 4 == 0 && (long)tiles * heads / 4 >= 2L * ri_compute_units();
#define RI_STATS(KS, HG, T)                                                                                             \
    talking_stats_mfma_kernel<KS, HG, T><<<dim3(tiles, heads / HG), 64, 0, s>>>(stats, (const bf16_t*)q, q_stride, q_off, \
                                                                     (const bf16_t*)k_pages, tok_pos, cu_seqlens, seqs, \
                                                                     page_table, table_width, heads, kv_heads, window, scale, r1, r2, bias)
#define RI_MIX(KS, HPW, T, ONE)                                                                                         \
    do {                                                                                                                \
        if (lds > 64 * 1024)                                                                                            \
            hipFuncSetAttribute((const void*)talking_mix_mfma_kernel<KS, HPW, T, ONE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
        talking_mix_mfma_kernel<KS, HPW, T, ONE><<<dim3(tiles, shares), 64 * TM_WAVES, lds, s>>>(                       \
            (bf16_t*)out, parts, (size_t)tokens * heads * dim, stats, (const bf16_t*)q, q_stride, q_off, (const bf16_t*)k_pages, \
            (const bf16_t*)v_pages, tok_pos, cu_seqlens, seqs, page_table, table_width, kv_heads, window, scale, r1, r2, talk, bias); \
    } while (0)
#define RI_MIX_OF(KS, HPW, T) do { if (of_kv % HPW == 0) RI_MIX(KS, HPW, T, true); else RI_MIX(KS, HPW, T, false); } while (0)
#define RI_BY_TABLE(KS, T)                                                                                              \
    do {                                                                                                                \
        if (four) RI_STATS(KS, 4, T); else RI_STATS(KS, 1, T);                                                          \
        if (hpw == 1) RI_MIX(KS, 1, T, true); else if (hpw == 2) RI_MIX_OF(KS, 2, T); else if (hpw == 3) RI_MIX_OF(KS, 3, T); else RI_MIX_OF(KS, 4, T); \
    } while (0)
#define RI_BY_HEADS(KS) do { if (table) RI_BY_TABLE(KS, true); else RI_BY_TABLE(KS, false); } while (0)
    if (dim == 32) RI_BY_HEADS(1); else if (dim == 64) RI_BY_HEADS(2); else RI_BY_HEADS(4);
#undef RI_BY_HEADS
#undef RI_BY_TABLE
#undef RI_MIX_OF
#undef RI_MIX
#undef RI_STATS
    RI_LAUNCH_CHECK("talking_attention_mfma");
    return 0;
}
