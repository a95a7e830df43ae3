// Recurrences whose decay is one number a head and token over prompts, in chunks of 64 tokens instead of token by token:
//     S_t = d_t S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t,
// linear attention with a fixed decay (d_t = d_h; q = silu(.) * q_scale, k = silu(.), v = silu(.)) and the state-space mixer
// (ssd.hip: d_t = exp(-exp(A_log_h) dt_t), q = C, k = B, v = dt x; y = o + D x, times silu(z)).
// The tokens of a chunk need not wait for one another.  With D(i, j) = d_(j+1) ... d_i, for a chunk of n tokens from the state S0,
//     o_i   = sum_{j <= i} D(i, j) (q_i . k_j) v_j  +  D(i, -1) S0^T q_i,
//     S_end = D(n - 1, -1) S0 + sum_j D(n - 1, j) k_j v_j^T,
// so a step is three launches: every chunk's own sum U = sum_j D(n - 1, j) k_j v_j^T (all chunks side by side), the
// walk from chunk to chunk, S0 of the next = D S0 + U, which leaves every chunk's S0 where its U was and the last
// state in the sequence's slot (a few loads and stores an element), and every chunk's outputs (all chunks side by side).
// Only products of decays from an earlier token to a later one appear, never their inverses: the powers d^m, m >= 0, of a fixed decay, and
// those tokens' own decays multiplied in 64 bits and rounded once (a difference of exponents summed from the chunk's start would lose a
// small one behind a large one, and is NaN where a decay is 0).  Everything else is float32: the activations, the scores q . k, the state
// and all sums; the products run on the matrix cores' float32 product (16x16x4), whose products and sums are 32-bit ones.  A sum goes by
// blocks of sixteen steps, the blocks two by two, a score's four products at a time two by two: one chain of 128 steps errs twice as much as
// the walk's sums over its lanes.  Relative error against 64 bits, 2-norm, x 1e-8, outputs and states: state-space mixer, 32 heads, steps
// that forget fast and slowly, 128 x 128: the walk 10.5 5.2, 11.1 6.7, in one chain 21.7 4.9, 20.9 6.6, so 10.5 4.9, 11.0 6.7; 64 x 64 10.0
// 4.9, 10.4 7.2 : 16.0 4.8, 14.9 7.2 : 10.1 4.8, 10.3 7.1; fixed decay, 128 x 128 11.8 41 : 17.0 12.4 : 9.1 11.3.
// A workgroup of eight wavefronts takes one (chunk, sequence, head), a wavefront sixteen columns of the results (sixteen rows of a
// chunk's own sum): what only its columns need comes straight from memory, once, and what all need (q and k, the scores, v) passes
// through LDS.  What bounds it: the products, some 230 of 32 cycles a wavefront and chunk, and two trips to memory.  32 heads
// of 128 x 128, us the walk : in chunks: one prompt of 2,048 tokens 671 : 131 (fixed decay; 182 on the vector units, 124 with one chain a
// sum), 287 : 134 (state-space mixer); eight of 500 620 : 248, 257 : 277; four of 300 to 1,800 490 : 372 (state-space mixer).
// Head sizes: multiples of 4 up to 128.
#include "api.h"
#include "common.h"

#define DC_TOK 64                // tokens of a chunk
#define DC_MAX 128               // largest key or value head
#define DC_STRIDE (DC_MAX + 4)   // of the rows of q and k, and of v, in LDS
#define DC_ASTRIDE (DC_TOK + 4)
#define DC_THREADS 512           // of the workgroups that work on a chunk: a wavefront for sixteen of 128 columns
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float dc_floatx4;

__device__ __forceinline__ float dc_silu(float v) { return v / (1.0f + expf(-v)); }

__device__ __forceinline__ float4 dc_ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 dc_ld4(const bf16_t* p) {
    const uint2 w = *reinterpret_cast<const uint2*>(p);
    return make_float4(__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xFFFF0000u), __uint_as_float(w.y << 16),
                       __uint_as_float(w.y & 0xFFFF0000u));
}

// The workspace's entry of chunk c of sequence b, which starts at token t0 of the step: sequences' entries do not
// meet, since a sequence of len tokens has at most len / 64 + 1 chunks.
__device__ __forceinline__ size_t dc_entry(int t0, int b, int c) { return (size_t)(t0 / DC_TOK + b + c); }

// Where a head's q, k and v come from, and its decays.  `Made` is the workgroup's, in LDS: what its decays are read from.
template <typename TA>
struct DcFixed {
    struct Made {
        float powers[DC_TOK + 1];
    };
    const TA* proj;
    int row, q_off, k_off, v_off;
    const float* head_decay;
    float q_scale;
    __device__ __forceinline__ float4 q4(int t, int h, int dim, int k) const {
        const float4 v = dc_ld4(proj + (size_t)t * row + q_off + h * dim + k);
        return make_float4(dc_silu(v.x) * q_scale, dc_silu(v.y) * q_scale, dc_silu(v.z) * q_scale, dc_silu(v.w) * q_scale);
    }
    __device__ __forceinline__ float4 k4(int t, int h, int dim, int k) const {
        const float4 v = dc_ld4(proj + (size_t)t * row + k_off + h * dim + k);
        return make_float4(dc_silu(v.x), dc_silu(v.y), dc_silu(v.z), dc_silu(v.w));
    }
    __device__ __forceinline__ float4 v4(int t, int, int h, int vdim, int c, const Made&) const {
        const float4 v = dc_ld4(proj + (size_t)t * row + v_off + h * vdim + c);
        return make_float4(dc_silu(v.x), dc_silu(v.y), dc_silu(v.z), dc_silu(v.w));
    }
    __device__ __forceinline__ float k1(int t, int h, int dim, int k) const { return dc_silu(to_f32(proj[(size_t)t * row + k_off + h * dim + k])); }
    __device__ __forceinline__ float v1(int t, int, int h, int vdim, int c, const Made&) const {
        return dc_silu(to_f32(proj[(size_t)t * row + v_off + h * vdim + c]));
    }
    __device__ __forceinline__ void make(Made& made, int, int, int h) const {
        const int m = threadIdx.x;                           // (d^0 = 1 also for d = 0)
        if (m <= DC_TOK) made.powers[m] = m == 0 ? 1.0f : powf(head_decay[h], (float)m);
        __syncthreads();
    }
    __device__ __forceinline__ float between(const Made& made, int i, int j) const { return made.powers[i - j]; }
    __device__ __forceinline__ float from_start(const Made& made, int i) const { return made.powers[i + 1]; }
    __device__ __forceinline__ float finish(float o, int, int, int, int) const { return o; }
};

template <typename TA>
struct DcSteps {
    // Products of decays, of 64 bits until they are whole, by blocks of sixteen tokens: near[j][i % 16] from j + 1 to i of j's block,
    // behind[j] from j + 1 to its block's end, upto[i] from its block's start to i, of whole blocks, and from the chunk's start to i.
    struct Made {
        double behind[DC_TOK], upto[DC_TOK], blocks[DC_TOK / 16];
        float near[DC_TOK][16], start[DC_TOK], dt[DC_TOK];
    };
    const float* xbc;
    int channels, b_off, c_off;
    const TA* proj;
    int stride, z_off, dt_off;
    const float *dt_bias, *a_log, *d_skip;
    int share;                                               // heads that read one B and C
    __device__ __forceinline__ float4 q4(int t, int h, int dim, int k) const {
        return dc_ld4(xbc + (size_t)t * channels + c_off + h / share * dim + k);
    }
    __device__ __forceinline__ float4 k4(int t, int h, int dim, int k) const {
        return dc_ld4(xbc + (size_t)t * channels + b_off + h / share * dim + k);
    }
    __device__ __forceinline__ float4 v4(int t, int j, int h, int vdim, int c, const Made& made) const {
        const float4 v = dc_ld4(xbc + (size_t)t * channels + h * vdim + c);
        const float dt = made.dt[j];
        return make_float4(dt * v.x, dt * v.y, dt * v.z, dt * v.w);
    }
    __device__ __forceinline__ float k1(int t, int h, int dim, int k) const { return xbc[(size_t)t * channels + b_off + h / share * dim + k]; }
    __device__ __forceinline__ float v1(int t, int j, int h, int vdim, int c, const Made& made) const {
        return made.dt[j] * xbc[(size_t)t * channels + h * vdim + c];
    }
    __device__ __forceinline__ void make(Made& made, int first, int n, int h) const {
        const int i = threadIdx.x, first_of = i / 16 * 16;
        if (i < DC_TOK) {
            const float raw = to_f32(proj[(size_t)(first + min(i, n - 1)) * stride + dt_off + h]) + (dt_bias ? dt_bias[h] : 0.f);
            made.dt[i] = raw > 20.f ? raw : log1pf(expf(raw));           // softplus: beyond 20 it is its argument to the last bit
            made.upto[i] = exp((double)-expf(a_log[h]) * (double)made.dt[i]);
        }
        __syncthreads();
        double upto = 1.0, behind = 1.0;
        if (i < DC_TOK) {
            double d[16];
#pragma unroll
            for (int m = 0; m < 16; ++m) d[m] = made.upto[first_of + m];
#pragma unroll
            for (int m = 0; m < 16; ++m) {
                if (first_of + m <= i) upto *= d[m];
                else behind *= d[m];
                made.near[i][m] = (float)behind;
            }
        }
        __syncthreads();                                     // the tokens' own decays have been read
        if (i < DC_TOK) {
            made.upto[i] = upto;
            made.behind[i] = behind;
            if (i % 16 == 15) made.blocks[i / 16] = upto;
        }
        __syncthreads();
        if (i < DC_TOK) {
            for (int b = 0; b < i / 16; ++b) upto *= made.blocks[b];
            made.start[i] = (float)upto;
        }
        __syncthreads();
    }
    // from token j to token i, j <= i
    __device__ __forceinline__ float between(const Made& made, int i, int j) const {
        if (i / 16 == j / 16) return made.near[j][i % 16];
        double d = made.behind[j] * made.upto[i];
        for (int b = j / 16 + 1; b < i / 16; ++b) d *= made.blocks[b];
        return (float)d;
    }
    __device__ __forceinline__ float from_start(const Made& made, int i) const { return made.start[i]; }
    __device__ __forceinline__ float finish(float o, int t, int h, int vdim, int c) const {
        if (d_skip) o += d_skip[h] * xbc[(size_t)t * channels + h * vdim + c];
        const float z = to_f32(proj[(size_t)t * stride + z_off + h * vdim + c]);
        return o * (z / (1.f + expf(-z)));
    }
};

// The products of sixteen steps of a sum, four a matrix instruction: one after the other, or each added to nothing and the four results
// two by two (APART).
template <bool APART, typename A, typename B>
__device__ __forceinline__ dc_floatx4 dc_block(const A& a, const B& b) {
    const dc_floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    dc_floatx4 x[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], APART || e == 0 ? zero : x[e - 1], 0, 0, 0);
    return APART ? (x[0] + x[1]) + (x[2] + x[3]) : x[3];
}

// The sum of up to N such blocks (a power of two; `block(q)` of those there are), two by two.
template <int N, typename F>
__device__ __forceinline__ dc_floatx4 dc_tree(int from, int count, const F& block) {
    if constexpr (N == 1) return from < count ? block(from) : dc_floatx4{0.f, 0.f, 0.f, 0.f};
    else {
        const dc_floatx4 first = dc_tree<N / 2>(from, count, block);
        return first + dc_tree<N / 2>(from + N / 2, count, block);
    }
}

// U[entry, h] = sum_j D(n - 1, j) k_j v_j^T   [dim, vdim]; wholes[entry, h] = D(n - 1, -1)
template <typename SRC>
__global__ void __launch_bounds__(DC_THREADS, 6)
decay_chunk_sums_kernel(float* __restrict__ U, float* __restrict__ wholes, SRC src, const int32_t* __restrict__ cu_seqlens, int heads,
                        int dim, int vdim) {
    __shared__ __align__(16) float Vs[DC_TOK * DC_STRIDE];
    __shared__ typename SRC::Made made;
    const int c = blockIdx.x, b = blockIdx.y, h = blockIdx.z, tid = threadIdx.x;
    const int lane = tid & 63, r = lane & 15, g = lane >> 4, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t0 = cu_seqlens[b], t1 = cu_seqlens[b + 1];
    const int first = t0 + c * DC_TOK;
    if (first >= t1) return;
    const int n = min(DC_TOK, t1 - first);
    const int k = 16 * wave + r, kk = min(k, dim - 1);       // this lane's row of the result
    float kv[4][4];                                          // its keys of tokens 16 b + 4 g + e
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) kv[q][e] = src.k1(first + min(16 * q + 4 * g + e, n - 1), h, dim, kk);
    src.make(made, first, n, h);
    const int wide = (vdim + 15) / 16 * 16;
    for (int e = tid; e < DC_TOK * wide / 4; e += DC_THREADS) {
        const int j = e / (wide / 4), at = e % (wide / 4) * 4;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (j < n && at < vdim) v = src.v4(first + j, j, h, vdim, at, made);
        *reinterpret_cast<float4*>(Vs + j * DC_STRIDE + at) = v;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int j = 16 * q + 4 * g + e;
            kv[q][e] = j < n && k < dim ? kv[q][e] * src.between(made, n - 1, min(j, n - 1)) : 0.f;
        }
    const size_t entry = dc_entry(t0, b, c) * heads + h;
    if (tid == 0) wholes[entry] = src.from_start(made, n - 1);
    __syncthreads();
    if (16 * wave >= dim) return;
    float* Uc = U + entry * dim * vdim;
    for (int ct = 0; ct < wide / 16; ++ct) {
        const dc_floatx4 acc = dc_tree<4>(0, 4, [&](int q) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = Vs[(16 * q + 4 * g + e) * DC_STRIDE + 16 * ct + r];
            return dc_block<false>(kv[q], v);
        });
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (16 * wave + 4 * g + e < dim && 16 * ct + r < vdim) Uc[(size_t)(16 * wave + 4 * g + e) * vdim + 16 * ct + r] = acc[e];
    }
}

// From chunk to chunk: every chunk's entry gets the state it starts from, the slot the state after the last token.
__global__ void __launch_bounds__(256)
decay_chunk_carry_kernel(float* __restrict__ U, const float* __restrict__ wholes, float* __restrict__ state,
                         const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ slots, int heads, int dim, int vdim) {
    const int b = blockIdx.y, h = blockIdx.z;
    const int e = (blockIdx.x * 256 + threadIdx.x) * 4, size = dim * vdim;
    const int t0 = cu_seqlens[b], len = cu_seqlens[b + 1] - t0;
    if (e >= size || len <= 0) return;
    float* Sp = state + ((size_t)slots[b] * heads + h) * size + e;
    float4 s = *reinterpret_cast<const float4*>(Sp);
    const int chunks = (len + DC_TOK - 1) / DC_TOK;
    const size_t entry = dc_entry(t0, b, 0) * heads + h;
    float* Up = U + entry * size + e;
    const size_t step = (size_t)heads * size;
    float4 u = *reinterpret_cast<const float4*>(Up);
    for (int c = 0; c < chunks; ++c) {
        // the next chunk's sum is asked for before this one's place is written (the last chunk asks for its own again)
        const float4 next = *reinterpret_cast<const float4*>(Up + (size_t)min(c + 1, chunks - 1) * step);
        *reinterpret_cast<float4*>(Up + (size_t)c * step) = s;
        const float f = wholes[entry + (size_t)c * heads];
        s.x = f * s.x + u.x;
        s.y = f * s.y + u.y;
        s.z = f * s.z + u.z;
        s.w = f * s.w + u.w;
        u = next;
    }
    *reinterpret_cast<float4*>(Sp) = s;
}

// o_i = sum_{j <= i} D(i, j) (q_i . k_j) v_j + D(i, -1) S0^T q_i for the tokens of one chunk.
template <typename SRC>
__global__ void __launch_bounds__(DC_THREADS, 4)
decay_chunk_out_kernel(float* __restrict__ out, const float* __restrict__ U, SRC src, const int32_t* __restrict__ cu_seqlens, int heads,
                       int dim, int vdim) {
    __shared__ __align__(16) float Qs[DC_TOK * DC_STRIDE];
    __shared__ __align__(16) float Ks[DC_TOK * DC_STRIDE];   // the keys, later the scores times the decays [64][DC_ASTRIDE]
    __shared__ typename SRC::Made made;
    float* As = Ks;
    const int c = blockIdx.x, b = blockIdx.y, h = blockIdx.z, tid = threadIdx.x;
    const int lane = tid & 63, r = lane & 15, g = lane >> 4, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t0 = cu_seqlens[b], t1 = cu_seqlens[b + 1];
    const int first = t0 + c * DC_TOK;
    if (first >= t1) return;
    const int n = min(DC_TOK, t1 - first), wide = (dim + 15) / 16 * 16;
    for (int e = tid; e < DC_TOK * wide / 4; e += DC_THREADS) {
        const int j = e / (wide / 4), at = e % (wide / 4) * 4;
        float4 qv = make_float4(0.f, 0.f, 0.f, 0.f), kv = qv;
        if (j < n && at < dim) {
            qv = src.q4(first + j, h, dim, at);
            kv = src.k4(first + j, h, dim, at);
        }
        *reinterpret_cast<float4*>(Qs + j * DC_STRIDE + at) = qv;
        *reinterpret_cast<float4*>(Ks + j * DC_STRIDE + at) = kv;
    }
    src.make(made, first, n, h);
    __syncthreads();
    // this wavefront's columns of the values and of the state, on their way while the scores are made
    const int col = 16 * wave + r, cc = min(col, vdim - 1);
    const float* S0 = U + (dc_entry(t0, b, c) * heads + h) * dim * vdim;
    float v[4][4], sv[DC_MAX / 16][4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int j = 16 * q + 4 * g + e;
            const float x = src.v1(first + min(j, n - 1), min(j, n - 1), h, vdim, cc, made);
            v[q][e] = j < n ? x : 0.f;
        }
#pragma unroll
    for (int q = 0; q < DC_MAX / 16; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = 16 * q + 4 * g + e;
            const float x = S0[(size_t)min(k, dim - 1) * vdim + cc];
            sv[q][e] = k < dim ? x : 0.f;
        }
    // scores: the tiles of 16 x 16 on and below the diagonal, ten of a whole chunk
    dc_floatx4 score[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int tile = wave + 8 * u, ti = tile < 1 ? 0 : tile < 3 ? 1 : tile < 6 ? 2 : 3, tj = tile - ti * (ti + 1) / 2;
        if (tile >= 10) break;
        score[u] = dc_tree<DC_MAX / 16>(0, 16 * ti < n ? wide / 16 : 0, [&](int q) {
            const dc_floatx4 qa = *reinterpret_cast<const dc_floatx4*>(Qs + (16 * ti + r) * DC_STRIDE + 16 * q + 4 * g);
            const dc_floatx4 kb = *reinterpret_cast<const dc_floatx4*>(Ks + (16 * tj + r) * DC_STRIDE + 16 * q + 4 * g);
            return dc_block<true>(qa, kb);
        });
    }
    __syncthreads();                                         // the keys have been read: the scores take their place
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int tile = wave + 8 * u, ti = tile < 1 ? 0 : tile < 3 ? 1 : tile < 6 ? 2 : 3, tj = tile - ti * (ti + 1) / 2;
        if (tile >= 10) break;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = 16 * ti + 4 * g + e, j = 16 * tj + r;
            As[i * DC_ASTRIDE + j] = j <= i && i < n ? score[u][e] * src.between(made, i, min(j, i)) : 0.f;
        }
    }
    __syncthreads();
    if (16 * wave >= vdim) return;
#pragma unroll 1
    for (int t = 0; t < 4; ++t) {
        if (16 * t >= n) break;                              // (the same for the whole workgroup)
        const dc_floatx4 from_state = dc_tree<DC_MAX / 16>(0, wide / 16, [&](int q) {
            return dc_block<false>(*reinterpret_cast<const dc_floatx4*>(Qs + (16 * t + r) * DC_STRIDE + 16 * q + 4 * g), sv[q]);
        });
        const dc_floatx4 sum = dc_tree<4>(0, t + 1, [&](int q) {
            return dc_block<false>(*reinterpret_cast<const dc_floatx4*>(As + (16 * t + r) * DC_ASTRIDE + 16 * q + 4 * g), v[q]);
        });
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = 16 * t + 4 * g + e;
            if (i < n && col < vdim)
                out[(size_t)(first + i) * heads * vdim + h * vdim + col] =
                    src.finish(sum[e] + src.from_start(made, i) * from_state[e], first + i, h, vdim, col);
        }
    }
}

template <typename SRC>
static void launch_chunks(float* out, float* workspace, const SRC& src, float* state, const int32_t* cu_seqlens, const int32_t* slots,
                          int seqs, int tokens, int max_new, int heads, int dim, int vdim, hipStream_t s) {
    const dim3 grid((max_new + DC_TOK - 1) / DC_TOK, seqs, heads);
    float* wholes = workspace + ((size_t)tokens / DC_TOK + seqs) * heads * dim * vdim;
    decay_chunk_sums_kernel<SRC><<<grid, DC_THREADS, 0, s>>>(workspace, wholes, src, cu_seqlens, heads, dim, vdim);
    decay_chunk_carry_kernel<<<dim3((dim * vdim / 4 + 255) / 256, seqs, heads), 256, 0, s>>>(workspace, wholes, state, cu_seqlens, slots,
                                                                                             heads, dim, vdim);
    decay_chunk_out_kernel<SRC><<<grid, DC_THREADS, 0, s>>>(out, workspace, src, cu_seqlens, heads, dim, vdim);
}

extern "C" int ri_decay_chunks_fit(int dim, int vdim) {
    return dim >= 4 && vdim >= 4 && dim <= DC_MAX && vdim <= DC_MAX && dim % 4 == 0 && vdim % 4 == 0;
}

// How many floats of workspace a step of `tokens` tokens in `seqs` sequences needs.
extern "C" long ri_decay_chunks_workspace(int seqs, int tokens, int heads, int dim, int vdim) {
    return ((long)tokens / DC_TOK + seqs) * heads * (dim * vdim + 1L);
}

extern "C" int ri_decay_scan_chunked(float* out, const void* proj, int act_dtype, int row, int q_off, int k_off, int v_off,
                                     const float* head_decay, float q_scale, float* state, const int32_t* cu_seqlens,
                                     const int32_t* slots, int seqs, int tokens, int max_new, int heads, int dim, int vdim,
                                     float* workspace, long workspace_floats, void* stream) {
    RI_REQUIRE(out && proj && head_decay && state && cu_seqlens && slots && workspace, "decay_scan_chunked: a null pointer");
    RI_REQUIRE(act_dtype == RI_F32 || act_dtype == RI_BF16, "decay_scan_chunked: dtype %d", act_dtype);
    RI_REQUIRE(ri_decay_chunks_fit(dim, vdim), "decay_scan_chunked: heads of %d x %d (multiples of 4 up to %d)", dim, vdim, DC_MAX);
    RI_REQUIRE(seqs >= 1 && tokens >= seqs && heads >= 1 && heads <= 65535 && seqs <= 65535 && max_new >= 1 && max_new <= tokens,
               "decay_scan_chunked: %d tokens in %d sequences of at most %d, %d heads", tokens, seqs, max_new, heads);
    RI_REQUIRE(row % 4 == 0 && q_off % 4 == 0 && k_off % 4 == 0 && v_off % 4 == 0 && q_off >= 0 && k_off >= 0 && v_off >= 0 &&
               q_off + heads * dim <= row && k_off + heads * dim <= row && v_off + heads * vdim <= row,
               "decay_scan_chunked: columns %d, %d, %d of rows of %d (multiples of 4)", q_off, k_off, v_off, row);
    RI_REQUIRE(workspace_floats >= ri_decay_chunks_workspace(seqs, tokens, heads, dim, vdim),
               "decay_scan_chunked: a workspace of %ld floats", workspace_floats);
    hipStream_t s = (hipStream_t)stream;
#define RI_DC_GO(T)                                                                                                  \
    launch_chunks(out, workspace, DcFixed<T>{(const T*)proj, row, q_off, k_off, v_off, head_decay, q_scale}, state, cu_seqlens, slots, seqs, \
                  tokens, max_new, heads, dim, vdim, s)
    if (act_dtype == RI_F32) RI_DC_GO(float); else RI_DC_GO(bf16_t);
#undef RI_DC_GO
    RI_LAUNCH_CHECK("decay_scan_chunked");
    return 0;
}

extern "C" int ri_ssd_scan_chunked(float* out, const float* xbc, int channels, int b_off, int c_off, const void* proj, int act_dtype,
                                   int stride, int z_off, int dt_off, const float* dt_bias, const float* a_log, const float* d_skip,
                                   float* state, const int32_t* cu_seqlens, const int32_t* slots, int seqs, int tokens, int max_new,
                                   int heads, int groups, int n, int vdim, float* workspace, long workspace_floats, void* stream) {
    RI_REQUIRE(out && xbc && proj && a_log && state && cu_seqlens && slots && workspace, "ssd_scan_chunked: a null pointer");
    RI_REQUIRE(act_dtype == RI_F32 || act_dtype == RI_BF16, "ssd_scan_chunked: dtype %d", act_dtype);
    RI_REQUIRE(ri_decay_chunks_fit(n, vdim), "ssd_scan_chunked: states of %d x %d (multiples of 4 up to %d)", n, vdim, DC_MAX);
    RI_REQUIRE(seqs >= 1 && tokens >= seqs && heads >= 1 && heads <= 65535 && seqs <= 65535 && max_new >= 1 && max_new <= tokens &&
               groups >= 1 && heads % groups == 0, "ssd_scan_chunked: %d tokens in %d sequences of at most %d, %d heads in %d groups", tokens,
               seqs, max_new, heads, groups);
    RI_REQUIRE(channels % 4 == 0 && b_off % 4 == 0 && c_off % 4 == 0 && b_off >= 0 && c_off >= 0 && b_off + groups * n <= channels &&
               c_off + groups * n <= channels && heads * vdim <= channels && (uintptr_t)xbc % 16 == 0 && (uintptr_t)state % 16 == 0 &&
               (uintptr_t)workspace % 16 == 0, "ssd_scan_chunked: columns %d and %d of %d channels, or a buffer that is not aligned", b_off,
               c_off, channels);
    RI_REQUIRE(z_off >= 0 && dt_off >= 0 && z_off + heads * vdim <= stride && dt_off + heads <= stride,
               "ssd_scan_chunked: columns %d and %d of rows of %d", z_off, dt_off, stride);
    RI_REQUIRE(workspace_floats >= ri_decay_chunks_workspace(seqs, tokens, heads, n, vdim), "ssd_scan_chunked: a workspace of %ld floats",
               workspace_floats);
    hipStream_t s = (hipStream_t)stream;
#define RI_DC_GO(T)                                                                                                  \
    launch_chunks(out, workspace, DcSteps<T>{xbc, channels, b_off, c_off, (const T*)proj, stride, z_off, dt_off, dt_bias, a_log, d_skip, \
                                             heads / groups}, state, cu_seqlens, slots, seqs, tokens, max_new, heads, n, vdim, s)
    if (act_dtype == RI_F32) RI_DC_GO(float); else RI_DC_GO(bf16_t);
#undef RI_DC_GO
    RI_LAUNCH_CHECK("ssd_scan_chunked");
    return 0;
}
