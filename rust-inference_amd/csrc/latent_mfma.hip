// Attention over a cached latent on the matrix cores, for prompts in bfloat16.
//
// The cache entry is one key/value head: key rows [c | rotated part] of DK = 32 KS elements, value rows c of 16 VT
// elements (the first 16 VT of a key row, kept a second time transposed inside a page for the value product).  All query
// heads read it, so a wavefront takes 16 query heads of one token as the 16 columns of its tiles and walks the token's
// pages: scores S^T = K Q^T (KS products a half page), the softmax's running maximum and sum per column, and
// O^T += V^T P^T (VT products a page).  The key rows of a half page are permuted (row r of the first half is key
// 8 (r / 4) + r % 4, of the second that plus 4), so that a lane's eight scores are eight neighbouring keys, which is
// how the value product wants its weights: no exchange between lanes.  A sink per head joins the sum once at the end.
// Scores, maxima, sums and the accumulators are float32; the weights are rounded to bfloat16 for the value product, as
// in this library's other matrix-core attention (of single tokens what that leaves of them is a second product's).  A token's sums run over its pages in order, whatever else the step holds.
// A step of few single tokens cuts a token's pages into chunks that workgroups walk side by side; each leaves its maximum, its sum
// and its sums of values, and a second kernel joins them in the chunks' order.
#include "api.h"
#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 lm_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float lm_floatx4;

union LmFrag {
    lm_bf16x8 v;
    uint4 u;
    uint32_t w[4];
};

#define LM_PAGE 32
#define LM_WAVES 4
#define LM_MAX_CHUNKS 64

template <int KS, int VT>
__global__ void __launch_bounds__(64 * LM_WAVES)
latent_attention_mfma_kernel(bf16_t* __restrict__ out, const bf16_t* __restrict__ q, int q_stride,
                             const bf16_t* __restrict__ k_pages, const bf16_t* __restrict__ v_pages,
                             const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ tok_seq,
                             const int32_t* __restrict__ page_table, int table_width, int tokens, int heads, int tiles,
                             float scale_log2, const float* __restrict__ sinks) {
    constexpr int DK = 32 * KS, RANK = 16 * VT;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int pair = blockIdx.x * LM_WAVES + wave;            // (token, tile of 16 heads)
    if (pair >= tokens * tiles) return;
    // (long prompts first: the workgroups launched last are the short ones)
    const int t = tokens - 1 - pair / tiles, tile = pair % tiles;
    const int col = lane & 15, g = lane >> 4;
    const int head = tile * 16 + col;
    const int hq = head < heads ? head : heads - 1;           // a column pulled back inside the heads: loads are issued anyway
    const int qpos = tok_pos[t];
    const int32_t* table = page_table + (size_t)tok_seq[t] * table_width;

    LmFrag qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
        qf[ks].u = *reinterpret_cast<const uint4*>(q + (size_t)t * q_stride + (size_t)hq * DK + ks * 32 + 8 * g);
    lm_floatx4 o[VT];
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) o[vt] = lm_floatx4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    const int key_row = 8 * (col >> 2) + (col & 3);           // the key this lane's operand row holds in the first half page

    for (int page = 0; page <= qpos / LM_PAGE; ++page) {
        const long phys = table[page];
        const bf16_t* kp = k_pages + phys * LM_PAGE * (long)DK + (long)key_row * DK + 8 * g;
        lm_floatx4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            LmFrag k0, k1;
            k0.u = *reinterpret_cast<const uint4*>(kp + ks * 32);
            k1.u = *reinterpret_cast<const uint4*>(kp + 4 * DK + ks * 32);
            s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0.v, qf[ks].v, s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1.v, qf[ks].v, s1, 0, 0, 0);
        }
        float s[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
        const int key0 = page * LM_PAGE + 8 * g;
        if (key0 + 7 > qpos) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (key0 + e > qpos) s[e] = -INFINITY;
        }
        float mx = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
        mx = fmaxf(mx, __shfl_xor(mx, 16, RI_WAVE));
        mx = fmaxf(mx, __shfl_xor(mx, 32, RI_WAVE));
        const float m_new = fmaxf(m, mx * scale_log2);        // the scale is positive; key 0 is seen by every token: finite
        LmFrag p;
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float a = exp2f(fmaf(s[2 * e], scale_log2, -m_new));
            const float b = exp2f(fmaf(s[2 * e + 1], scale_log2, -m_new));
            p.w[e] = pack_bf16x2(a, b);
            sum += a + b;
        }
        const float corr = exp2f(m - m_new);                  // 0 at the first page (m = -inf)
        l = l * corr + sum;
        m = m_new;
        const bf16_t* vp = v_pages + phys * (long)RANK * LM_PAGE + (long)col * LM_PAGE + 8 * g;
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
            LmFrag vf;
            vf.u = *reinterpret_cast<const uint4*>(vp + (long)vt * 16 * LM_PAGE);
            o[vt] *= corr;
            o[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, p.v, o[vt], 0, 0, 0);
        }
    }
    l += __shfl_xor(l, 16, RI_WAVE);                          // a column's sum over its four lanes
    l += __shfl_xor(l, 32, RI_WAVE);
    if (sinks) l += exp2f(sinks[hq] * 1.4426950408889634f - m);
    const float inv = 1.0f / l;
    if (head < heads) {
        bf16_t* op = out + ((size_t)t * heads + head) * RANK + 4 * g;
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
            uint2 w;
            w.x = pack_bf16x2(o[vt][0] * inv, o[vt][1] * inv);
            w.y = pack_bf16x2(o[vt][2] * inv, o[vt][3] * inv);
            *reinterpret_cast<uint2*>(op + vt * 16) = w;
        }
    }
}

// Single tokens: the four wavefronts of a workgroup share a (token, tile of 16 heads, chunk of pages).  Each makes the scores' products
// over its quarter of the key rows' elements, the quarters meet lane by lane in LDS (one barrier a page: two buffers take turns), and
// each goes on with all scores and a quarter of the value rows.  What bounds the kernel above on a step of few tokens is a wavefront's
// wait for the 68 loads a page that its registers cannot hold at once; a quarter's 18 are all asked for together, the next page's
// keys before the values are used.  With fewer, longer chunks fewer weights are the 1 of a chunk's largest score, which bfloat16 holds
// whole: what the rounding leaves of the weights goes through the matrix cores as well.  Error (2-norm) against 64 bits, 32 heads, keys of
// 576 / 16 heads, keys of 288, a wavefront a chunk 1.93e-3 / 1.90e-3, in quarters with the weights rounded 1.96e-3 / 1.91e-3, so 1.66e-3 / 1.66e-3
// (the result's own rounding); 48.8 : 50.3 us for 40 tokens at 1,500 keys.  32 heads, keys of 576, us with the join, a wavefront a chunk : this: one token at 1,000 keys 21.5 :
// 11.9, 8 at 1,400 42.4 : 16.6, 40 at 1,500 165 : 47, 128 at 1,000 571 : 81, 300 at 1,000 590 : 216; 16 heads, keys of 160: 8.2 : 7.4,
// 11.5 : 8.7, 21.9 : 16.4, 27.8 : 19.1.
template <int KS, int VT>
__global__ void __launch_bounds__(64 * LM_WAVES)
latent_attention_quarters_kernel(bf16_t* __restrict__ out, const bf16_t* __restrict__ q, int q_stride,
                                 const bf16_t* __restrict__ k_pages, const bf16_t* __restrict__ v_pages,
                                 const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ tok_seq,
                                 const int32_t* __restrict__ page_table, int table_width, int tokens, int heads, int tiles,
                                 float scale_log2, const float* __restrict__ sinks, float* __restrict__ partial, int chunks,
                                 int chunk_pages) {
    constexpr int DK = 32 * KS, RANK = 16 * VT, KW = (KS + LM_WAVES - 1) / LM_WAVES, VW = VT / LM_WAVES;
    __shared__ lm_floatx4 scores[2][LM_WAVES][2][RI_WAVE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), unit = blockIdx.x;
    const int pair = unit / chunks, chunk = unit % chunks;
    const int t = tokens - 1 - pair / tiles, tile = pair % tiles;
    const int col = lane & 15, g = lane >> 4;
    const int head = tile * 16 + col;
    const int hq = head < heads ? head : heads - 1;
    const int qpos = tok_pos[t];
    const int32_t* table = page_table + (size_t)tok_seq[t] * table_width;
    const int k0 = KS * wave / LM_WAVES, k1 = KS * (wave + 1) / LM_WAVES;        // this wavefront's steps over the key rows

    LmFrag qf[KW], kf[KW][2], vf[VW];
#pragma unroll
    for (int i = 0; i < KW; ++i)
        qf[i].u = *reinterpret_cast<const uint4*>(q + (size_t)t * q_stride + (size_t)hq * DK + min(k0 + i, KS - 1) * 32 + 8 * g);
    lm_floatx4 o[VW];
#pragma unroll
    for (int vt = 0; vt < VW; ++vt) o[vt] = lm_floatx4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    const int key_row = 8 * (col >> 2) + (col & 3);           // (the kernel above's order of keys)
    const int page_end = chunks > 1 ? min(qpos / LM_PAGE + 1, (chunk + 1) * chunk_pages) : qpos / LM_PAGE + 1;
    const int page_begin = chunks > 1 ? chunk * chunk_pages : 0;
    auto fetch_keys = [&](long phys) {
        const bf16_t* kp = k_pages + phys * LM_PAGE * (long)DK + (long)key_row * DK + 8 * g;
#pragma unroll
        for (int i = 0; i < KW; ++i) {
            kf[i][0].u = *reinterpret_cast<const uint4*>(kp + min(k0 + i, KS - 1) * 32);
            kf[i][1].u = *reinterpret_cast<const uint4*>(kp + 4 * DK + min(k0 + i, KS - 1) * 32);
        }
    };
    long phys = 0;
    if (page_begin < page_end) fetch_keys(phys = table[page_begin]);
    for (int page = page_begin, buf = 0; page < page_end; ++page, buf ^= 1) {    // (the same for the whole workgroup)
        const bf16_t* vp = v_pages + phys * (long)RANK * LM_PAGE + (long)(wave * VW * 16 + col) * LM_PAGE + 8 * g;
        phys = table[min(page + 1, page_end - 1)];
#pragma unroll
        for (int vt = 0; vt < VW; ++vt) vf[vt].u = *reinterpret_cast<const uint4*>(vp + (long)vt * 16 * LM_PAGE);
        lm_floatx4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < KW; ++i)
            if (k0 + i < k1) {                                // (the same for the whole wavefront)
                s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[i][0].v, qf[i].v, s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[i][1].v, qf[i].v, s1, 0, 0, 0);
            }
        fetch_keys(phys);
        scores[buf][wave][0][lane] = s0;
        scores[buf][wave][1][lane] = s1;
        __syncthreads();
        s0 = scores[buf][0][0][lane];
        s1 = scores[buf][0][1][lane];
#pragma unroll
        for (int w = 1; w < LM_WAVES; ++w) {
            s0 += scores[buf][w][0][lane];
            s1 += scores[buf][w][1][lane];
        }
        float s[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
        const int key0 = page * LM_PAGE + 8 * g;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (key0 + e > qpos) s[e] = -INFINITY;
        float mx = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
        mx = fmaxf(mx, __shfl_xor(mx, 16, RI_WAVE));
        mx = fmaxf(mx, __shfl_xor(mx, 32, RI_WAVE));
        const float m_new = fmaxf(m, mx * scale_log2);        // the scale is positive; every page of the walk has a key that is seen
        LmFrag p, rest;                                       // the weights in bfloat16, and what that leaves of them
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float a = exp2f(fmaf(s[2 * e], scale_log2, -m_new));
            const float b = exp2f(fmaf(s[2 * e + 1], scale_log2, -m_new));
            p.w[e] = pack_bf16x2(a, b);
            rest.w[e] = pack_bf16x2(a - __uint_as_float(p.w[e] << 16), b - __uint_as_float(p.w[e] & 0xFFFF0000u));
            sum += a + b;
        }
        const float corr = exp2f(m - m_new);
        l = l * corr + sum;
        m = m_new;
#pragma unroll
        for (int vt = 0; vt < VW; ++vt) {
            o[vt] *= corr;
            o[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[vt].v, p.v, o[vt], 0, 0, 0);
            o[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[vt].v, rest.v, o[vt], 0, 0, 0);
        }
    }
    l += __shfl_xor(l, 16, RI_WAVE);
    l += __shfl_xor(l, 32, RI_WAVE);
    if (head >= heads) return;
    if (chunks > 1) {
        float* pp = partial + (((size_t)t * heads + head) * chunks + chunk) * (RANK + 2);
        if (g == 0 && wave == 0) { pp[0] = m; pp[1] = l; }
#pragma unroll
        for (int vt = 0; vt < VW; ++vt)
#pragma unroll
            for (int i = 0; i < 4; ++i) pp[2 + (wave * VW + vt) * 16 + 4 * g + i] = o[vt][i];
        return;
    }
    if (sinks) l += exp2f(sinks[hq] * 1.4426950408889634f - m);
    const float inv = 1.0f / l;
    bf16_t* op = out + ((size_t)t * heads + head) * RANK + wave * VW * 16 + 4 * g;
#pragma unroll
    for (int vt = 0; vt < VW; ++vt) {
        uint2 w;
        w.x = pack_bf16x2(o[vt][0] * inv, o[vt][1] * inv);
        w.y = pack_bf16x2(o[vt][2] * inv, o[vt][3] * inv);
        *reinterpret_cast<uint2*>(op + vt * 16) = w;
    }
}

// Prompts: a workgroup of eight wavefronts takes eight (token, tile of 16 heads) pairs of neighbouring tokens (of one sequence, where
// cu_seqlens says which are), which walk the same pages, and brings every page into LDS once for all of them.  What bounds the kernel above on a prompt is the caches: every wavefront
// fetches every page for itself, 69 KB for 68 MFMAs.  Here a page crosses once for eight wavefronts, and what is left is the wait for
// the next half page and for the two barriers a page (83% of the wavefronts' cycles; LDS is busy a fifth of the time, the matrix cores a
// ninth).  A page's key and value halves take turns: while the scores are made from the keys the values are on their way into registers,
// and the other way round.  Pieces of 16 bytes are exchanged by the row's number so that a fragment's sixteen rows meet every
// bank equally.  A token's sums are the other kernel's.  2,048 tokens, 32 heads, keys of 576: 1,400 us with a page a wavefront, 525.
#define LP_WAVES 8
template <int KS, int VT>
__global__ void __launch_bounds__(64 * LP_WAVES)
latent_attention_shared_kernel(bf16_t* __restrict__ out, const bf16_t* __restrict__ q, int q_stride,
                               const bf16_t* __restrict__ k_pages, const bf16_t* __restrict__ v_pages,
                               const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ tok_seq,
                               const int32_t* __restrict__ page_table, int table_width, int tokens, int heads, int tiles,
                               float scale_log2, const float* __restrict__ sinks, const int32_t* __restrict__ cu_seqlens, int seqs) {
    constexpr int DK = 32 * KS, RANK = 16 * VT, THREADS = 64 * LP_WAVES;
    constexpr int KP = DK / 8, KPIECES = LM_PAGE * KP;        // 16-byte pieces of a key row and of a page's keys
    constexpr int VP = LM_PAGE / 8, VPIECES = RANK * VP;      // ... of a value channel's row and of a page's values
    constexpr int KN = (KPIECES + THREADS - 1) / THREADS, VN = (VPIECES + THREADS - 1) / THREADS;
    __shared__ uint4 ks_[KPIECES], vs_[VPIECES];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 15, g = lane >> 4;
    // (long prompts first: the workgroups launched last are the short ones; pairs count back from the last token's)
    Run run = {0, tokens, (int)blockIdx.x * LP_WAVES, 0};
    run.count = min(LP_WAVES, tokens * tiles - run.first);
    if (cu_seqlens && !run_of(blockIdx.x, cu_seqlens, seqs, 1, LP_WAVES, tiles, run)) return;
    const bool there = wave < run.count;
    const int mine = run.first + min(wave, run.count - 1), last = run.start + run.tokens - 1;
    const int t = last - mine / tiles, tile = mine % tiles;
    const int head = tile * 16 + col, hq = head < heads ? head : heads - 1;
    const int qpos = tok_pos[t], seq = tok_seq[t];
    // where the tokens of a workgroup are of several sequences, these go one after the other
    const int t_last = last - run.first / tiles, t_first = last - (run.first + run.count - 1) / tiles;

    LmFrag qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
        qf[ks].u = *reinterpret_cast<const uint4*>(q + (size_t)t * q_stride + (size_t)hq * DK + ks * 32 + 8 * g);
    lm_floatx4 o[VT];
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) o[vt] = lm_floatx4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    const int key_row = 8 * (col >> 2) + (col & 3);
    uint4 kn[KN], vn[VN];
    auto fetch_keys = [&](long phys) {
        const uint4* from = reinterpret_cast<const uint4*>(k_pages + phys * LM_PAGE * (long)DK);
#pragma unroll
        for (int i = 0; i < KN; ++i) kn[i] = from[min(tid + i * THREADS, KPIECES - 1)];
    };
    auto fetch_values = [&](long phys) {
        const uint4* from = reinterpret_cast<const uint4*>(v_pages + phys * LM_PAGE * (long)RANK);
#pragma unroll
        for (int i = 0; i < VN; ++i) vn[i] = from[min(tid + i * THREADS, VPIECES - 1)];
    };
    // (a fragment's key rows are 0 .. 3 of every eight, or 4 .. 7; pieces stay within eight, or four where eight do not divide a row)
    auto key_at = [](int row, int piece) { return row * KP + (piece ^ (((row >> 1 & 1) | (row >> 3 & 3) << 1) & (KP % 8 == 0 ? 7 : 3))); };
    auto value_at = [](int row, int piece) { return row * VP + (piece ^ (row >> 2 & 3)); };

    for (int from = t_last; from >= t_first;) {               // (uniform: the tokens' sequences and positions are memory's)
        const int s_now = tok_seq[from];
        int to = from, far = tok_pos[from];                   // (the tokens of a sequence may come in any order)
        while (to > t_first && tok_seq[to - 1] == s_now) far = max(far, tok_pos[--to]);
        const bool active = there && t <= from && t >= to;
        const int32_t* table = page_table + (size_t)s_now * table_width;
        const int pages = far / LM_PAGE + 1;
        fetch_keys(table[0]);
        for (int page = 0; page < pages; ++page) {
            const long phys = table[page], next = table[min(page + 1, pages - 1)];
#pragma unroll
            for (int i = 0; i < KN; ++i) {
                const int e = tid + i * THREADS;
                if (KPIECES % THREADS == 0 || e < KPIECES) ks_[key_at(e / KP, e % KP)] = kn[i];
            }
            fetch_values(phys);
            __syncthreads();                                  // the keys are in place, and the page before's values have been read
            const bool sees = active && page * LM_PAGE <= qpos;          // (the same for the whole wavefront)
            LmFrag p;
            float corr = 1.f;
            if (sees) {
                lm_floatx4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    LmFrag k0, k1;
                    k0.u = ks_[key_at(key_row, ks * 4 + g)];
                    k1.u = ks_[key_at(key_row + 4, ks * 4 + g)];
                    s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0.v, qf[ks].v, s0, 0, 0, 0);
                    s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1.v, qf[ks].v, s1, 0, 0, 0);
                }
                float s[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
                const int key0 = page * LM_PAGE + 8 * g;
                if (key0 + 7 > qpos) {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (key0 + e > qpos) s[e] = -INFINITY;
                }
                float mx = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
                mx = fmaxf(mx, __shfl_xor(mx, 16, RI_WAVE));
                mx = fmaxf(mx, __shfl_xor(mx, 32, RI_WAVE));
                const float m_new = fmaxf(m, mx * scale_log2);        // the scale is positive; key 0 is seen by every token: finite
                float sum = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float a = exp2f(fmaf(s[2 * e], scale_log2, -m_new));
                    const float b = exp2f(fmaf(s[2 * e + 1], scale_log2, -m_new));
                    p.w[e] = pack_bf16x2(a, b);
                    sum += a + b;
                }
                corr = exp2f(m - m_new);                      // 0 at the first page (m = -inf)
                l = l * corr + sum;
                m = m_new;
            }
#pragma unroll
            for (int i = 0; i < VN; ++i) {
                const int e = tid + i * THREADS;
                if (VPIECES % THREADS == 0 || e < VPIECES) vs_[value_at(e / VP, e % VP)] = vn[i];
            }
            fetch_keys(next);
            __syncthreads();                                  // the values are in place, and the keys have been read
            if (sees) {
#pragma unroll
                for (int vt = 0; vt < VT; ++vt) {
                    LmFrag vf;
                    vf.u = vs_[value_at(vt * 16 + col, g)];
                    o[vt] *= corr;
                    o[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, p.v, o[vt], 0, 0, 0);
                }
            }
        }
        from = to - 1;
    }
    if (!there) return;
    l += __shfl_xor(l, 16, RI_WAVE);                          // a column's sum over its four lanes
    l += __shfl_xor(l, 32, RI_WAVE);
    if (sinks) l += exp2f(sinks[hq] * 1.4426950408889634f - m);
    const float inv = 1.0f / l;
    if (head < heads) {
        bf16_t* op = out + ((size_t)t * heads + head) * RANK + 4 * g;
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
            uint2 w;
            w.x = pack_bf16x2(o[vt][0] * inv, o[vt][1] * inv);
            w.y = pack_bf16x2(o[vt][2] * inv, o[vt][3] * inv);
            *reinterpret_cast<uint2*>(op + vt * 16) = w;
        }
    }
}

// The chunks of a token's pages, joined: the largest maximum, every chunk's sums scaled to it, the sink, the division.
__global__ void __launch_bounds__(256)
latent_attention_join_kernel(bf16_t* __restrict__ out, const float* __restrict__ partial, const float* __restrict__ sinks,
                             int heads, int chunks, int rank) {
    __shared__ float ms[LM_MAX_CHUNKS], ws[LM_MAX_CHUNKS], ls[LM_MAX_CHUNKS];
    const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const float* pp = partial + ((size_t)t * heads + h) * chunks * (rank + 2);
    if (tid < chunks) {
        ms[tid] = pp[(size_t)tid * (rank + 2)];
        ls[tid] = pp[(size_t)tid * (rank + 2) + 1];
    }
    __syncthreads();
    float m = -INFINITY;
    for (int c = 0; c < chunks; ++c) m = fmaxf(m, ms[c]);
    if (tid < chunks) ws[tid] = exp2f(ms[tid] - m);           // a chunk's factor, once
    __syncthreads();
    float l = 0.f;
    for (int c = 0; c < chunks; ++c) l += ls[c] * ws[c];
    if (sinks) l += exp2f(sinks[h] * 1.4426950408889634f - m);
    const float inv = 1.0f / l;
    for (int d = tid; d < rank; d += 256) {
        const float* col = pp + 2 + d;
        float a = 0.f;
        int c = 0;
        for (; c + 8 <= chunks; c += 8) {                     // eight loads asked for before the first is used
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = col[(size_t)(c + i) * (rank + 2)];
#pragma unroll
            for (int i = 0; i < 8; ++i) a += v[i] * ws[c + i];
        }
        for (; c < chunks; ++c) a += col[(size_t)c * (rank + 2)] * ws[c];
        out[((size_t)t * heads + h) * rank + d] = f32_to_bf16(a * inv);
    }
}

extern "C" int ri_latent_attention_mfma_fits(int key_dim, int rank, int page_size) {
    return page_size == LM_PAGE && ((key_dim == 576 && rank == 512) || (key_dim == 288 && rank == 256) || (key_dim == 160 && rank == 128));
}

// out [tokens, heads * rank] bfloat16: causal attention of every new token's heads (q [tokens, >= heads * key_dim], the
// heads side by side) over its sequence's one key/value head of key rows of key_dim and value rows of rank.
// shared_pages: neighbouring tokens share the pages they fetch (the results are the same bits): in as many workgroups of eight
// (token, tile of 16 heads) pairs as it says, each of one sequence, where cu_seqlens [seqs + 1] is given; else 1, a workgroup's tokens
// the step's neighbours, of one sequence for the most part.  quarters: for single tokens, a workgroup a (token, tile, chunk).
extern "C" int ri_latent_attention_mfma(void* out, const void* q, int q_stride, const void* k_pages, const void* v_pages,
                                        const int32_t* tok_pos, const int32_t* tok_seq, const int32_t* page_table,
                                        int table_width, int tokens, int heads, int key_dim, int rank, int page_size, float scale,
                                        const float* sinks, float* partial, int chunks, int chunk_pages, int shared_pages,
                                        const int32_t* cu_seqlens, int seqs, int quarters, void* stream) {
    RI_REQUIRE(tokens > 0 && heads > 0 && ri_latent_attention_mfma_fits(key_dim, rank, page_size),
               "latent_attention_mfma: %d tokens, %d heads, keys of %d, values of %d, pages of %d", tokens, heads, key_dim, rank, page_size);
    RI_REQUIRE(q_stride >= heads * key_dim && q_stride % 8 == 0 && (uintptr_t)q % 16 == 0 && (uintptr_t)k_pages % 16 == 0 &&
               (uintptr_t)v_pages % 16 == 0 && (uintptr_t)out % 8 == 0, "latent_attention_mfma: rows of %d for %d heads of %d, or a buffer that is not aligned",
               q_stride, heads, key_dim);
    RI_REQUIRE(scale > 0.f && table_width > 0, "latent_attention_mfma: scale %g", (double)scale);
    RI_REQUIRE(chunks >= 1 && chunks <= LM_MAX_CHUNKS && (chunks == 1 || (quarters && partial && chunk_pages >= 1)) && heads <= 65535,
               "latent_attention_mfma: %d chunks of %d pages", chunks, chunk_pages);
    const int tiles = (heads + 15) / 16;
    const long pairs = (long)tokens * tiles * chunks;
    RI_REQUIRE((pairs + LM_WAVES - 1) / LM_WAVES <= 2147483647L, "latent_attention_mfma: %ld tiles exceed one launch", pairs);
    const unsigned blocks = (unsigned)((pairs + LM_WAVES - 1) / LM_WAVES);
    const float scale_log2 = scale * 1.4426950408889634f;
    hipStream_t s = (hipStream_t)stream;
#define RI_GO(KS, VT)                                                                                                   \
    latent_attention_mfma_kernel<KS, VT><<<blocks, 64 * LM_WAVES, 0, s>>>((bf16_t*)out, (const bf16_t*)q, q_stride,     \
                                                                          (const bf16_t*)k_pages, (const bf16_t*)v_pages, \
                                                                          tok_pos, tok_seq, page_table, table_width, tokens, \
                                                                          heads, tiles, scale_log2, sinks)
    if (quarters) {
        RI_REQUIRE(pairs <= 2147483647L, "latent_attention_mfma: %ld tiles exceed one launch", pairs);
#define RI_QUARTERS(KS, VT)                                                                                             \
    latent_attention_quarters_kernel<KS, VT><<<(unsigned)pairs, 64 * LM_WAVES, 0, s>>>(                                 \
        (bf16_t*)out, (const bf16_t*)q, q_stride, (const bf16_t*)k_pages, (const bf16_t*)v_pages, tok_pos, tok_seq, page_table, table_width, \
        tokens, heads, tiles, scale_log2, sinks, partial, chunks, chunk_pages)
        if (key_dim == 576) RI_QUARTERS(18, 32); else if (key_dim == 288) RI_QUARTERS(9, 16); else RI_QUARTERS(5, 8);
#undef RI_QUARTERS
    } else if (shared_pages) {
        RI_REQUIRE(pairs <= 2147483647L - LP_WAVES && (!cu_seqlens || seqs > 0), "latent_attention_mfma: %ld pairs of %d sequences", pairs, seqs);
        const unsigned groups = cu_seqlens ? (unsigned)shared_pages : (unsigned)((pairs + LP_WAVES - 1) / LP_WAVES);
#define RI_SHARED(KS, VT)                                                                                               \
    latent_attention_shared_kernel<KS, VT><<<groups, 64 * LP_WAVES, 0, s>>>((bf16_t*)out, (const bf16_t*)q, q_stride,   \
                                                                            (const bf16_t*)k_pages, (const bf16_t*)v_pages, tok_pos, \
                                                                            tok_seq, page_table, table_width, tokens, heads, tiles, \
                                                                            scale_log2, sinks, cu_seqlens, seqs)
        if (key_dim == 576) RI_SHARED(18, 32); else if (key_dim == 288) RI_SHARED(9, 16); else RI_SHARED(5, 8);
#undef RI_SHARED
    } else if (key_dim == 576) RI_GO(18, 32); else if (key_dim == 288) RI_GO(9, 16); else RI_GO(5, 8);
#undef RI_GO
    if (chunks > 1)
        latent_attention_join_kernel<<<dim3(tokens, heads), 256, 0, s>>>((bf16_t*)out, partial, sinks, heads, chunks, rank);
    RI_LAUNCH_CHECK("latent_attention_mfma");
    return 0;
}
