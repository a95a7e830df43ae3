// The windowed attention whose heads talk (talking_attention.hip) for steps of single tokens in bfloat16, in two launches that both
// fill the machine:
//   talking_scores:  a wavefront per (page of 32 keys, key head, token): the scores of the key head's query heads on the matrix
//                    cores, with the distance bias and the window's mask, as float32 into a workspace, and each head's maximum and
//                    sum over the page;
//   talking_apply:   a workgroup per (token, share of the pages, 1,024 channels of values): from the pages' maxima and sums each
//                    head's own, then page by page the weights exp(s - m) / l, their mix w'_h = sum_g T[h, g] w_g, and the
//                    products with the values; the shares' float32 results are added by the caller.
// A score is made once (the general kernels make it once a walk), no workgroup walks more than its few pages, and the values of a
// page are asked for before the weights that they meet are made.  Scores, logarithm, softmax, mix and accumulators are float32.
// What bounds it: the trips to memory one after the other, some four a launch.  32 heads over 8 of 128, a window of 1,024, us with the
// sum of the shares, the general kernels : these: one token at 64 keys 47 : 17, at 2,000 84 : 20; 8 at 1,400 89 : 28 (scores 9.7,
// apply 15.8); 40 at 1,500 212 : 59; 128 at 1,500 1,292 : 154.  8 heads over 8 of 64: 25 : 12, 44 : 15, 44 : 18, 91 : 37, 476 : 82.
#include "api.h"
#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 td_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float td_floatx4;

#define TD_PAGE 32
#define TD_HEADS 64          // heads at most
#define TD_SLOTS 4           // value channels a thread accumulates: 256 * TD_SLOTS a workgroup

__device__ __forceinline__ td_bf16x8 td_load8(const bf16_t* p) { return *reinterpret_cast<const td_bf16x8*>(p); }

// scores [token][page][head][32], sums [token][page][head][2]; page 0 is the first that the token sees.
template <int STEPS>                                          // head_dim / 32
__global__ void __launch_bounds__(64)
talking_scores_kernel(float* __restrict__ scores, float* __restrict__ sums, const bf16_t* __restrict__ q, int q_stride, int q_off,
                      const bf16_t* __restrict__ k_pages, const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ tok_seq,
                      const int32_t* __restrict__ page_table, int table_width, int pages, int heads, int kv_heads, int window,
                      float scale, const float* __restrict__ r1, const float* __restrict__ r2) {
    constexpr int DIM = 32 * STEPS;
    const int t = blockIdx.z, kvh = blockIdx.y, lane = threadIdx.x, r = lane & 15, g = lane >> 4;
    const int qpos = tok_pos[t], lo = window > 0 ? max(0, qpos - window + 1) : 0, page = lo / TD_PAGE + blockIdx.x;
    if (page > qpos / TD_PAGE || (int)blockIdx.x >= pages) return;
    const int group = heads / kv_heads, h = kvh * group + min(r, group - 1);
    const bf16_t* kr = k_pages + ((long)page_table[(size_t)tok_seq[t] * table_width + page] * kv_heads + kvh) * TD_PAGE * DIM + (long)r * DIM + 8 * g;
    const bf16_t* qr = q + (size_t)t * q_stride + q_off + (size_t)h * DIM + 8 * g;
    td_bf16x8 kf[2][STEPS], qf[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        kf[0][s] = td_load8(kr + 32 * s);
        kf[1][s] = td_load8(kr + 16 * DIM + 32 * s);
        qf[s] = td_load8(qr + 32 * s);
    }
    const float b1 = r1 ? r1[h] : 0.f, b2 = r1 ? r2[h] : 0.f;
    float s[2][4], m = -INFINITY, l = 0.f;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        td_floatx4 dot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < STEPS; ++k) dot = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[u][k], qf[k], dot, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int j = page * TD_PAGE + 16 * u + 4 * g + i;
            const bool seen = j >= lo && j <= qpos;
            float v = dot[i] * scale;
            if (r1) v -= b1 * log1pf(b2 * (float)max(qpos - j, 0));
            s[u][i] = seen ? v : -INFINITY;
            m = fmaxf(m, s[u][i]);
        }
    }
    m = fmaxf(m, __shfl_xor(m, 16, RI_WAVE));
    m = fmaxf(m, __shfl_xor(m, 32, RI_WAVE));
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int j = page * TD_PAGE + 16 * u + 4 * g + i;
            l += j >= lo && j <= qpos ? expf(s[u][i] - m) : 0.f;
        }
    l += __shfl_xor(l, 16, RI_WAVE);
    l += __shfl_xor(l, 32, RI_WAVE);
    if (r >= group) return;
    const size_t at = ((size_t)t * pages + blockIdx.x) * heads + h;
#pragma unroll
    for (int u = 0; u < 2; ++u)
        *reinterpret_cast<float4*>(scores + at * TD_PAGE + 16 * u + 4 * g) = make_float4(s[u][0], s[u][1], s[u][2], s[u][3]);
    if (g == 0) *reinterpret_cast<float2*>(sums + at * 2) = make_float2(m, l);
}

// GROUP: query heads of a key head.
template <int GROUP>
__global__ void __launch_bounds__(256)
talking_apply_kernel(float* __restrict__ out, size_t share_stride, const float* __restrict__ scores, const float* __restrict__ sums,
                     const bf16_t* __restrict__ v_pages, const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ tok_seq,
                     const int32_t* __restrict__ page_table, int table_width, int pages, int kv_heads, int dim, int window,
                     const float* __restrict__ talk) {
    __shared__ float ps[TD_HEADS][TD_PAGE + 1];               // a page's weights
    __shared__ __attribute__((aligned(16))) float mixed[TD_HEADS][TD_PAGE + 4];
    __shared__ float tk[TD_HEADS][TD_HEADS + 1];              // the mixing matrix
    __shared__ float ms[TD_HEADS], ls[TD_HEADS];
    const int t = blockIdx.x, tid = threadIdx.x, heads = kv_heads * GROUP;
    const int qpos = tok_pos[t], lo = window > 0 ? max(0, qpos - window + 1) : 0;
    const int first = lo / TD_PAGE, count = min(qpos / TD_PAGE - first + 1, pages);
    const int32_t* table = page_table + (size_t)tok_seq[t] * table_width + first;
    const int channels = kv_heads * dim, c0 = blockIdx.z * 256 * TD_SLOTS;
    const int h0 = c0 / dim * GROUP, h1 = min(heads, (c0 + 256 * TD_SLOTS + dim - 1) / dim * GROUP);      // the heads of this workgroup's channels
    if (talk)
        for (int e = tid; e < heads * heads; e += 256) tk[e / heads][e % heads] = talk[e];
    // every head's maximum and sum, eight threads a head
    for (int h_from = 0; h_from < heads; h_from += 32) {
        const int h = min(h_from + tid / 8, heads - 1);
        const float2* at = reinterpret_cast<const float2*>(sums) + (size_t)t * pages * heads + h;
        float m = -INFINITY, l = 0.f;
        for (int p = tid % 8; p < count; p += 8) m = fmaxf(m, at[(size_t)p * heads].x);
#pragma unroll
        for (int d = 1; d < 8; d *= 2) m = fmaxf(m, __shfl_xor(m, d, RI_WAVE));
        for (int p = tid % 8; p < count; p += 8) {
            const float2 v = at[(size_t)p * heads];
            l += v.y * expf(v.x - m);
        }
#pragma unroll
        for (int d = 1; d < 8; d *= 2) l += __shfl_xor(l, d, RI_WAVE);
        if (tid % 8 == 0 && h_from + tid / 8 < heads) { ms[h] = m; ls[h] = 1.0f / l; }
    }
    float acc[TD_SLOTS][GROUP] = {};
    for (int p = blockIdx.y; p < count; p += gridDim.y) {
        // the values of the page's 32 keys: each channel's lie side by side
        const bf16_t* vp = v_pages + (long)table[p] * kv_heads * dim * TD_PAGE;
        uint4 v[TD_SLOTS][4];
#pragma unroll
        for (int i = 0; i < TD_SLOTS; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                v[i][k] = *reinterpret_cast<const uint4*>(vp + (long)min(c0 + tid + 256 * i, channels - 1) * TD_PAGE + 8 * k);
        __syncthreads();                                      // maxima, sums and matrix are there; the last page's weights are read
        const float* sp = scores + ((size_t)t * pages + p) * heads * TD_PAGE;
        for (int e = tid; e < heads * TD_PAGE; e += 256) ps[e / TD_PAGE][e % TD_PAGE] = expf(sp[e] - ms[e / TD_PAGE]) * ls[e / TD_PAGE];
        __syncthreads();
        for (int h = h0 + tid / TD_PAGE; h < h1; h += 256 / TD_PAGE) {
            const int j = tid % TD_PAGE;
            float w = 0.f;
            if (talk) {
#pragma unroll 8
                for (int g = 0; g < heads; ++g) w += tk[h][g] * ps[g][j];
            } else {
                w = ps[h][j];
            }
            mixed[h][j] = w;
        }
        __syncthreads();
        const int base = (first + p) * TD_PAGE;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (base + 8 * k > qpos || base + 8 * k + 7 < lo) continue;      // (the same for the whole workgroup: none of the eight keys is seen)
#pragma unroll
            for (int i = 0; i < TD_SLOTS; ++i) {
                const int kvh = min(c0 + tid + 256 * i, channels - 1) / dim;
                const uint32_t w[4] = {v[i][k].x, v[i][k].y, v[i][k].z, v[i][k].w};
#pragma unroll
                for (int hh = 0; hh < GROUP; ++hh) {
                    const float4 a = *reinterpret_cast<const float4*>(&mixed[kvh * GROUP + hh][8 * k]);
                    const float4 b = *reinterpret_cast<const float4*>(&mixed[kvh * GROUP + hh][8 * k + 4]);
                    const float m8[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {             // (a key that is not seen has the weight 0)
                        acc[i][hh] += m8[2 * e] * __uint_as_float(w[e] << 16);
                        acc[i][hh] += m8[2 * e + 1] * __uint_as_float(w[e] & 0xFFFF0000u);
                    }
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < TD_SLOTS; ++i) {
        const int oc = c0 + tid + 256 * i;
        if (oc >= channels) continue;
#pragma unroll
        for (int hh = 0; hh < GROUP; ++hh)
            out[blockIdx.y * share_stride + (size_t)t * heads * dim + (size_t)(oc / dim * GROUP + hh) * dim + oc % dim] = acc[i][hh];
    }
}

extern "C" int ri_talking_decode_fits(int heads, int kv_heads, int dim, int page_size) {
    const int group = kv_heads > 0 ? heads / kv_heads : 0;
    return heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && heads <= TD_HEADS && page_size == TD_PAGE &&
           (group == 1 || group == 2 || group == 4 || group == 8 || group == 16) && (dim == 32 || dim == 64 || dim == 128);
}

// pages: as many as any token sees at most; scores float32 [tokens][pages][heads][32], sums [tokens][pages][heads][2], out [shares]
// [tokens][heads * dim].
extern "C" int ri_talking_decode(float* out, int shares, float* scores, float* sums, int pages, const void* q, int q_stride, int q_off,
                                 const void* k_pages, const void* v_pages, const int32_t* tok_pos, const int32_t* tok_seq,
                                 const int32_t* page_table, int table_width, int tokens, int heads, int kv_heads, int dim, int page_size,
                                 int window, float scale, const float* r1, const float* r2, const float* talk, void* stream) {
    RI_REQUIRE(ri_talking_decode_fits(heads, kv_heads, dim, page_size), "talking_decode: %d heads over %d of %d, pages of %d", heads, kv_heads,
               dim, page_size);
    RI_REQUIRE(tokens > 0 && tokens <= 65535 && pages > 0 && shares > 0 && shares <= 65535 && table_width > 0 && window >= 0,
               "talking_decode: %d tokens, %d pages in %d shares", tokens, pages, shares);
    RI_REQUIRE(q_off >= 0 && q_off + heads * dim <= q_stride && q_off % 8 == 0 && q_stride % 8 == 0,
               "talking_decode: columns %d of rows of %d", q_off, q_stride);
    RI_REQUIRE((((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages | (uintptr_t)scores | (uintptr_t)sums) & 15) == 0,
               "talking_decode: queries, pages and workspace start on 16-byte boundaries");
    RI_REQUIRE((r1 == nullptr) == (r2 == nullptr), "talking_decode: the distance bias has two numbers a head");
    hipStream_t s = (hipStream_t)stream;
#define RI_SCORES(STEPS)                                                                                                     \
    talking_scores_kernel<STEPS><<<dim3(pages, kv_heads, tokens), 64, 0, s>>>(scores, sums, (const bf16_t*)q, q_stride, q_off, \
        (const bf16_t*)k_pages, tok_pos, tok_seq, page_table, table_width, pages, heads, kv_heads, window, scale, r1, r2)
    if (dim == 32) RI_SCORES(1); else if (dim == 64) RI_SCORES(2); else RI_SCORES(4);
#undef RI_SCORES
    RI_LAUNCH_CHECK("talking_decode");
    const int blocks = (kv_heads * dim + 256 * TD_SLOTS - 1) / (256 * TD_SLOTS);
#define RI_APPLY(GROUP)                                                                                                      \
    talking_apply_kernel<GROUP><<<dim3(tokens, shares, blocks), 256, 0, s>>>(out, (size_t)tokens * heads * dim, scores, sums, \
        (const bf16_t*)v_pages, tok_pos, tok_seq, page_table, table_width, pages, kv_heads, dim, window, talk)
    switch (heads / kv_heads) {
        case 1: RI_APPLY(1); break;
        case 2: RI_APPLY(2); break;
        case 4: RI_APPLY(4); break;
        case 8: RI_APPLY(8); break;
        default: RI_APPLY(16);
    }
#undef RI_APPLY
    RI_LAUNCH_CHECK("talking_decode");
    return 0;
}
