// Attention over a cached latent: what lies around the attention kernel.
//
// A token's keys and values of all heads are products of one latent vector c (kv_rank numbers) with per-head matrices,
// plus one rotated key part shared by the heads.  Only c and that part are cached, and the attention runs on them
// directly: with k_h = U_h c the score q_h . k_h is (U_h^T q_h) . c, and sum_j w_j (V_h c_j) is V_h (sum_j w_j c_j).  So
// the cache holds, per token, one key row [c | rotated part] and one value row c for a single key/value head, the
// queries become [U_h^T q_h | rotated q_h] (kv_rank + rot numbers a head), and the heads' results (kv_rank numbers) go
// through V_h afterwards.
//
//   latent_prepare:  c = rms_norm(first kv_rank outputs of the down projection) * gain; the last rot outputs and the
//                    last rot elements of every query head turn in neighbouring pairs (2i, 2i + 1) by p * f_i; c and
//                    the turned key part go to the key page, c to the value page (transposed inside a page);
//   head_products:   out[t, h, :] = gate[t, h] * x[t, h, :] W_h for matrices W_h [K, N] of a stack [H, K, N], with the
//                    elements of x behind K copied behind N (the rotated part of a query rides along); the gate is the
//                    sigmoid of one number per token and head, or absent.
//
// Norm statistics, angles, sines and cosines, the gate's sigmoid and every sum are float32.
#include "api.h"
#include "common.h"

template <typename TA, typename TC>
__global__ void __launch_bounds__(256)
latent_prepare_kernel(TA* __restrict__ proj, int stride, int q_off, int kv_off, const float* __restrict__ gain, float eps,
                      const float* __restrict__ inv_freq, const int32_t* __restrict__ tok_pos,
                      const int32_t* __restrict__ tok_seq, const int32_t* __restrict__ page_table, int table_width,
                      TC* __restrict__ k_pages, TC* __restrict__ v_pages, int page_size, int heads, int dim, int rot, int rank) {
    __shared__ float scratch[16];
    const int t = blockIdx.x, tid = threadIdx.x;
    const int pos = tok_pos[t];
    TA* row = proj + (size_t)t * stride;
    const long page = page_table[(size_t)tok_seq[t] * table_width + pos / page_size];
    const int slot = pos % page_size;
    TC* krow = k_pages + (page * page_size + slot) * (long)(rank + rot);
    TC* vcol = v_pages + page * (long)rank * page_size + slot;
    float ss = 0.f;
    for (int r = tid; r < rank; r += 256) {
        const float v = to_f32(row[kv_off + r]);
        ss += v * v;
    }
    const float inv = 1.0f / sqrtf(block_sum(ss, scratch) / (float)rank + eps);
    for (int r = tid; r < rank; r += 256) {
        const float c = to_f32(row[kv_off + r]) * inv * gain[r];
        from_f32(krow + r, c);
        from_f32(vcol + (long)r * page_size, c);
    }
    const int half = rot / 2;
    // the shared key part (one "head") and every query head's last rot elements
    for (int e = tid; e < (heads + 1) * half; e += 256) {
        const int h = e / half, i = e % half;
        const float a = (float)pos * inv_freq[i];
        const float cs = cosf(a), sn = sinf(a);
        if (h == heads) {
            const float u = to_f32(row[kv_off + rank + 2 * i]), v = to_f32(row[kv_off + rank + 2 * i + 1]);
            from_f32(krow + rank + 2 * i, u * cs - v * sn);
            from_f32(krow + rank + 2 * i + 1, v * cs + u * sn);
        } else {
            TA* qp = row + q_off + (size_t)h * (dim + rot) + dim + 2 * i;
            const float u = to_f32(qp[0]), v = to_f32(qp[1]);
            from_f32(qp, u * cs - v * sn);
            from_f32(qp + 1, v * cs + u * sn);
        }
    }
}

extern "C" int ri_latent_prepare(void* proj, int act_dtype, int stride, int q_off, int kv_off, const float* gain, float eps,
                                 const float* inv_freq, const int32_t* tok_pos, const int32_t* tok_seq,
                                 const int32_t* page_table, int table_width, void* k_pages, void* v_pages, int cache_dtype,
                                 int page_size, int tokens, int heads, int dim, int rot, int rank, void* stream) {
    RI_REQUIRE(tokens > 0 && heads > 0 && dim >= 0 && rank > 0 && rot >= 0 && rot % 2 == 0,
               "latent_prepare: %d tokens, %d heads of %d + %d, latent %d", tokens, heads, dim, rot, rank);
    RI_REQUIRE(q_off >= 0 && kv_off >= 0 && q_off + heads * (dim + rot) <= stride && kv_off + rank + rot <= stride,
               "latent_prepare: columns %d and %d of rows of %d", q_off, kv_off, stride);
    RI_REQUIRE(act_dtype == cache_dtype && (act_dtype == RI_F32 || act_dtype == RI_BF16), "latent_prepare: dtypes %d and %d",
               act_dtype, cache_dtype);
    RI_REQUIRE(rot == 0 || inv_freq, "latent_prepare: a rotation needs its frequencies");
    RI_REQUIRE(page_size > 0 && table_width > 0, "latent_prepare: page geometry");
    hipStream_t s = (hipStream_t)stream;
    if (act_dtype == RI_F32)
        latent_prepare_kernel<float, float><<<tokens, 256, 0, s>>>((float*)proj, stride, q_off, kv_off, gain, eps, inv_freq,
                                                                  tok_pos, tok_seq, page_table, table_width, (float*)k_pages,
                                                                  (float*)v_pages, page_size, heads, dim, rot, rank);
    else
        latent_prepare_kernel<bf16_t, bf16_t><<<tokens, 256, 0, s>>>((bf16_t*)proj, stride, q_off, kv_off, gain, eps, inv_freq,
                                                                    tok_pos, tok_seq, page_table, table_width, (bf16_t*)k_pages,
                                                                    (bf16_t*)v_pages, page_size, heads, dim, rot, rank);
    RI_LAUNCH_CHECK("latent_prepare");
    return 0;
}

// ------------------------------------------------------------------ a product per head
#define HP_TOKENS 8          // tokens of a workgroup: a matrix element is loaded once for all of them
#define HP_COLS 64           // result columns of a workgroup
#define HP_SLICES 4          // slices of K that the four wavefronts of a workgroup take: a lane sums its slice's rows in order,
                             // the slices meet through LDS in order

template <typename TX, typename TW, typename TO>
__global__ void __launch_bounds__(HP_COLS * HP_SLICES)
head_products_kernel(TO* __restrict__ out, int out_stride, int out_off, int out_head, const TX* __restrict__ x, int x_stride,
                     int x_off, int x_head, const TW* __restrict__ w, const TX* __restrict__ gates, int g_stride, int g_off,
                     float scale, int tokens, int k, int n, int extra) {
    extern __shared__ float lds[];
    float* xs = lds;                                          // [HP_TOKENS][k + extra]
    const int width = k + extra;
    float* red = xs + HP_TOKENS * width;                      // [HP_SLICES][HP_TOKENS][HP_COLS]
    const int h = blockIdx.y, t0 = blockIdx.x * HP_TOKENS, tid = threadIdx.x;
    const int lane = tid % HP_COLS, slice = tid / HP_COLS;
    const int c = blockIdx.z * HP_COLS + lane;
    for (int e = tid; e < HP_TOKENS * width; e += HP_COLS * HP_SLICES) {
        const int tt = e / width, col = e % width, t = t0 + tt;
        xs[e] = t < tokens ? to_f32(x[(size_t)t * x_stride + x_off + (size_t)h * x_head + col]) : 0.f;
    }
    __syncthreads();
    float acc[HP_TOKENS];
#pragma unroll
    for (int tt = 0; tt < HP_TOKENS; ++tt) acc[tt] = 0.f;
    if (c < n) {
        const TW* wc = w + (size_t)h * k * n + c;
        const int per = (k + HP_SLICES - 1) / HP_SLICES;      // rows of a slice
        const int r0 = slice * per, r1 = min(k, r0 + per);
        int r = r0;
        for (; r + 8 <= r1; r += 8) {                         // eight loads asked for before the first is used
            float wv[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) wv[i] = to_f32(wc[(size_t)(r + i) * n]);
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int tt = 0; tt < HP_TOKENS; ++tt) acc[tt] += xs[tt * width + r + i] * wv[i];
        }
        for (; r < r1; ++r) {
            const float wv = to_f32(wc[(size_t)r * n]);
#pragma unroll
            for (int tt = 0; tt < HP_TOKENS; ++tt) acc[tt] += xs[tt * width + r] * wv;
        }
    } else if (c < n + extra && slice == 0) {
#pragma unroll
        for (int tt = 0; tt < HP_TOKENS; ++tt) acc[tt] = xs[tt * width + k + (c - n)];
    }
#pragma unroll
    for (int tt = 0; tt < HP_TOKENS; ++tt) red[(slice * HP_TOKENS + tt) * HP_COLS + lane] = acc[tt];
    __syncthreads();
    if (slice == 0 && c < n + extra) {
#pragma unroll
        for (int tt = 0; tt < HP_TOKENS; ++tt) {
            const int t = t0 + tt;
            if (t >= tokens) break;
            float v = red[tt * HP_COLS + lane];
            for (int sl = 1; sl < HP_SLICES; ++sl) v += red[(sl * HP_TOKENS + tt) * HP_COLS + lane];
            float g = scale;
            if (gates) g *= 1.f / (1.f + expf(-to_f32(gates[(size_t)t * g_stride + g_off + h])));
            from_f32(out + (size_t)t * out_stride + out_off + (size_t)h * out_head + c, v * g);
        }
    }
}

// bfloat16 matrices whose rows 16-byte pieces divide: tiles of 16 tokens by 128 columns, the eight wavefronts of a workgroup on a slice of K
// each, on the matrix cores' float32 product (16x16x4; the matrix elements are widened, so every product and sum is a 32-bit one).  Lane
// (g, r) reads eight neighbouring columns of row k + g at once, one of each of eight products, up to sixteen such loads asked for
// together; the slices meet through LDS two by two, so a result's sum depends on K alone.  What bounds it is two trips to memory and
// the sum; the kernel above made sixteen, two bytes a lane.  32 heads, us the kernel above : this: 512 x 128, one token
// 16.7 : 9.8, 32 19.3 : 11.8, 120 42 : 18; 128 x 512 6.3 : 5.6, 9.2 : 7.0, 28 : 24 (with cold caches, as in a model's step, 8 tokens
// 37 : 12.7 and 12.0 : 7.0).
#define HM_TOKENS 16
#define HM_COLS 128
#define HM_WAVES 8
#define HM_DEEP 16           // loads of a wavefront that are under way together
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float hm_floatx4;

template <typename TX, typename TO>
__global__ void __launch_bounds__(64 * HM_WAVES)
head_products_matrix_kernel(TO* __restrict__ out, int out_stride, int out_off, int out_head, const TX* __restrict__ x, int x_stride,
                            int x_off, int x_head, const bf16_t* __restrict__ w, const TX* __restrict__ gates, int g_stride, int g_off,
                            float scale, int tokens, int k, int n, int extra) {
    extern __shared__ float4 lds4[];
    float* xs = reinterpret_cast<float*>(lds4);               // [HM_TOKENS][k + 4], then the slices' sums [HM_WAVES][HM_TOKENS][HM_COLS]
    const int h = blockIdx.y, t0 = blockIdx.x * HM_TOKENS, tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), c0 = blockIdx.z * HM_COLS, pitch = k + 4;
    const int steps = (k / 4 + HM_WAVES - 1) / HM_WAVES, s0 = min(wave * steps, k / 4), s1 = min(s0 + steps, k / 4);
    const bf16_t* wp = w + (size_t)h * k * n + min(c0 + 8 * r, n - 8);
    uint4 wv[HM_DEEP];
    auto fetch = [&](int from) {
#pragma unroll
        for (int i = 0; i < HM_DEEP; ++i) wv[i] = *reinterpret_cast<const uint4*>(wp + (size_t)(4 * min(from + i, k / 4 - 1) + g) * n);
    };
    fetch(s0);
    for (int e = tid; e < HM_TOKENS * k; e += 64 * HM_WAVES) {
        const int tt = e / k, col = e % k, t = t0 + tt;
        xs[tt * pitch + col] = t < tokens ? to_f32(x[(size_t)t * x_stride + x_off + (size_t)h * x_head + col]) : 0.f;
    }
    __syncthreads();
    hm_floatx4 acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = hm_floatx4{0.f, 0.f, 0.f, 0.f};
    for (int s = s0; s < s1; s += HM_DEEP) {
#pragma unroll
        for (int i = 0; i < HM_DEEP; ++i) {
            if (s + i >= s1) break;                           // (the same for the whole wavefront)
            const float xv = xs[r * pitch + 4 * (s + i) + g];
            const uint32_t p[4] = {wv[i].x, wv[i].y, wv[i].z, wv[i].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[2 * j] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv, __uint_as_float(p[j] << 16), acc[2 * j], 0, 0, 0);
                acc[2 * j + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv, __uint_as_float(p[j] & 0xFFFF0000u), acc[2 * j + 1], 0, 0, 0);
            }
        }
        if (s + HM_DEEP < s1) fetch(s + HM_DEEP);
    }
    __syncthreads();                                          // the rows have been read
#pragma unroll
    for (int i = 0; i < 4; ++i) {                             // token 4 g + i, columns 8 r ..+8
        float4* to = lds4 + ((wave * HM_TOKENS + 4 * g + i) * HM_COLS + 8 * r) / 4;
        to[0] = make_float4(acc[0][i], acc[1][i], acc[2][i], acc[3][i]);
        to[1] = make_float4(acc[4][i], acc[5][i], acc[6][i], acc[7][i]);
    }
    __syncthreads();
    for (int e = tid; e < HM_TOKENS * HM_COLS; e += 64 * HM_WAVES) {
        const int tt = e / HM_COLS, c = c0 + e % HM_COLS, t = t0 + tt;
        if (t >= tokens || c >= n) continue;
        float v[HM_WAVES];
#pragma unroll
        for (int s = 0; s < HM_WAVES; ++s) v[s] = xs[s * HM_TOKENS * HM_COLS + e];
#pragma unroll
        for (int step = 1; step < HM_WAVES; step *= 2) // (in order they err more at 128 x 512 than the kernel above: 2-norm against 64 bits 5.5e-8 : 5.3e-8, so 4.9e-8)
#pragma unroll
            for (int s = 0; s < HM_WAVES; s += 2 * step) v[s] += v[s + step];
        float f = scale;
        if (gates) f *= 1.f / (1.f + expf(-to_f32(gates[(size_t)t * g_stride + g_off + h])));
        from_f32(out + (size_t)t * out_stride + out_off + (size_t)h * out_head + c, v[0] * f);
    }
    if (blockIdx.z == 0)
        for (int e = tid; e < HM_TOKENS * extra; e += 64 * HM_WAVES) {
            const int c = e % extra, t = t0 + e / extra;
            if (t >= tokens) break;
            float f = scale;
            if (gates) f *= 1.f / (1.f + expf(-to_f32(gates[(size_t)t * g_stride + g_off + h])));
            from_f32(out + (size_t)t * out_stride + out_off + (size_t)h * out_head + n + c,
                     to_f32(x[(size_t)t * x_stride + x_off + (size_t)h * x_head + k + c]) * f);
        }
}

extern "C" int ri_head_products(void* out, int out_dtype, int out_stride, int out_off, int out_head, const void* x, int x_dtype,
                                int x_stride, int x_off, int x_head, const void* w, int w_dtype, const void* gates, int g_stride,
                                int g_off, float scale, int tokens, int heads, int k, int n, int extra, void* stream) {
    // k = n = 0: no product, the copied elements alone (with the head's gate and the scale); w is not read
    RI_REQUIRE(tokens > 0 && heads > 0 && heads <= 65535 && extra >= 0 && ((k > 0 && n > 0) || (k == 0 && n == 0 && extra > 0)),
               "head_products: %d tokens, %d heads of %d x %d (+%d)", tokens, heads, k, n, extra);
    RI_REQUIRE(x_off >= 0 && x_head >= k + extra && x_off + (long)(heads - 1) * x_head + k + extra <= x_stride,
               "head_products: heads of %d at column %d of rows of %d", x_head, x_off, x_stride);
    RI_REQUIRE(out_off >= 0 && out_head >= n + extra && out_off + (long)(heads - 1) * out_head + n + extra <= out_stride,
               "head_products: results of %d at column %d of rows of %d", out_head, out_off, out_stride);
    RI_REQUIRE(!gates || (g_off >= 0 && g_off + heads <= g_stride), "head_products: gates at column %d of rows of %d", g_off, g_stride);
    RI_REQUIRE((x_dtype == RI_F32 || x_dtype == RI_BF16) && (w_dtype == RI_F32 || w_dtype == RI_BF16) &&
               (out_dtype == RI_F32 || out_dtype == RI_BF16), "head_products: dtypes %d, %d, %d", x_dtype, w_dtype, out_dtype);
    const size_t lds = ((size_t)HP_TOKENS * (k + extra) + (size_t)HP_SLICES * HP_TOKENS * HP_COLS) * sizeof(float);
    RI_REQUIRE(lds <= 64 * 1024, "head_products: heads of %d exceed the kernel's 1792", k + extra);
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid((tokens + HP_TOKENS - 1) / HP_TOKENS, heads, (n + extra + HP_COLS - 1) / HP_COLS);
    RI_REQUIRE(grid.z <= 65535, "head_products: results of %d", n + extra);
    // Sizes and alignment alone decide, so that a token's result does not depend on the step.  Fewer than 128 rows are too few for eight
    // slices (16 heads of 64 x 128, us the other : this: 8 tokens 4.8 : 5.1, 64 5.0 : 5.5); up to 1,020 fit the kernel's LDS.
    const size_t sums = sizeof(float) * HM_WAVES * HM_TOKENS * HM_COLS, rows = sizeof(float) * HM_TOKENS * ((size_t)k + 4);
    if (k >= 128 && w_dtype == RI_BF16 && k % 4 == 0 && n % 8 == 0 && rows <= 64 * 1024 && (uintptr_t)w % 16 == 0 &&
        !(x_dtype == RI_F32 && out_dtype != RI_F32)) {
        const dim3 tiles((tokens + HM_TOKENS - 1) / HM_TOKENS, heads, (n + HM_COLS - 1) / HM_COLS);
#define RI_MATRIX(TX, TO)                                                                                               \
    head_products_matrix_kernel<TX, TO><<<tiles, 64 * HM_WAVES, rows > sums ? rows : sums, s>>>(                        \
        (TO*)out, out_stride, out_off, out_head, (const TX*)x, x_stride, x_off, x_head, (const bf16_t*)w, (const TX*)gates, g_stride, g_off, \
        scale, tokens, k, n, extra)
        if (x_dtype == RI_F32) RI_MATRIX(float, float);
        else if (out_dtype == RI_F32) RI_MATRIX(bf16_t, float);
        else RI_MATRIX(bf16_t, bf16_t);
#undef RI_MATRIX
        RI_LAUNCH_CHECK("head_products");
        return 0;
    }
#define RI_GO(TX, TW, TO)                                                                                               \
    head_products_kernel<TX, TW, TO><<<grid, HP_COLS * HP_SLICES, lds, s>>>((TO*)out, out_stride, out_off, out_head, (const TX*)x, x_stride, \
                                                            x_off, x_head, (const TW*)w, (const TX*)gates, g_stride, g_off, \
                                                            scale, tokens, k, n, extra)
    if (x_dtype == RI_F32) {
        RI_REQUIRE(out_dtype == RI_F32, "head_products: float32 rows give float32 results");
        if (w_dtype == RI_F32) RI_GO(float, float, float); else RI_GO(float, bf16_t, float);
    } else {
        RI_REQUIRE(w_dtype == RI_BF16, "head_products: bfloat16 rows take bfloat16 matrices");
        if (out_dtype == RI_F32) RI_GO(bf16_t, bf16_t, float); else RI_GO(bf16_t, bf16_t, bf16_t);
    }
#undef RI_GO
    RI_LAUNCH_CHECK("head_products");
    return 0;
}
