// A state-space mixer with a scalar decay per head (the structured state-space duality form), on a float32 state per
// sequence and head.
//
//   causal_conv_silu:  every channel's causal convolution over the tokens of its sequence, bias, silu; the inputs before
//                      a step's first token come from the sequence's kept tail (its last taps - 1 inputs, oldest first,
//                      zeros at a sequence's start); the taps are added oldest first, the current token's last;
//   conv_tails:        moves every sequence's tail on by the step's tokens (a launch of its own: the first tokens of a
//                      step read the tail that the last ones would write);
//   ssd_scan:          per head h (which reads B and C of group h / (heads / groups)), with dt = softplus(dt_raw + dt_bias_h):
//                          S_t = exp(-exp(A_log_h) dt) S_(t-1) + dt B_t x_t^T,      y_t = S_t^T C_t + D_h x_t,
//                      then y times silu(z), float32;
//   group_rms_norm:    a row in equal parts, each divided by its own root mean square, times a gain an element.
//
// The step size with its softplus, the decay with both exponentials, the state, every sum of the recurrence, the gate and
// the norm are float32.  A workgroup of ssd_scan owns one (sequence, head): a thread holds some rows of one column of
// the state in registers and the slices of rows meet through LDS in a fixed order, so a token's sums do not depend on
// how the tokens were cut into steps.  The same kernels walk a prompt and take a single step; prompts whose walk is a chain of many
// tokens with little beside it go in chunks instead (decay_chunks.hip), whose sums differ from the walk's by rounding.
#include "api.h"
#include "common.h"
#include "walk.h"

#define SSD_MAX_TAPS 16

template <typename TA>
__global__ void __launch_bounds__(256)
causal_conv_silu_kernel(float* __restrict__ out, const TA* __restrict__ proj, int stride, int col0, const float* __restrict__ taps_w,
                        const float* __restrict__ bias, const float* __restrict__ tails, int taps,
                        const int32_t* __restrict__ tok_seq, const int32_t* __restrict__ cu_seqlens,
                        const int32_t* __restrict__ slots, int channels) {
    const int t = blockIdx.x, ch = blockIdx.y * 256 + threadIdx.x;
    if (ch >= channels) return;
    const int seq = tok_seq[t];
    const int first = cu_seqlens[seq];
    const int i = t - first;                                  // the token's place in this step
    const float* tail = tails + (size_t)slots[seq] * (taps - 1) * channels;
    float sum = 0.f;
    for (int a = 0; a < taps; ++a) {                          // oldest first
        const int src = i - (taps - 1 - a);
        const float in = src >= 0 ? to_f32(proj[(size_t)(first + src) * stride + col0 + ch])
                                  : tail[(size_t)(taps - 1 + src) * channels + ch];
        sum += in * taps_w[(size_t)ch * taps + a];
    }
    if (bias) sum += bias[ch];
    out[(size_t)t * channels + ch] = sum / (1.f + expf(-sum));
}

// Four taps, four channels and eight tokens a thread: a row is read once for the four tokens that use it (11 loads of four
// channels, all asked for together, where the kernel above makes 32 of one), and the taps once for eight tokens.  The sums are the
// same, in the same order.  A row whose tap lies before its sequence's tokens of the step takes the tail instead, in a pass
// of its own for the threads that have such a row.  Bound by memory: 6,144 channels of 4,928 and 2,048 tokens, 225 and 85 us an
// element a thread, 43.8 and 20.6 so (4.1 and 3.7 TB/s).
#define CONV_TOKENS 8
#define CONV_BLOCK_FROM (3L << 18)  // tokens * channels
typedef float conv_f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t conv_u16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ conv_f32x4 conv_four(const float* p) { return *reinterpret_cast<const conv_f32x4*>(p); }
__device__ __forceinline__ conv_f32x4 conv_four(const bf16_t* p) {
    const conv_u16x4 v = *reinterpret_cast<const conv_u16x4*>(p);
    conv_f32x4 f;
#pragma unroll
    for (int c = 0; c < 4; ++c) f[c] = to_f32((bf16_t)v[c]);
    return f;
}

template <typename TA>
__global__ void __launch_bounds__(256)
causal_conv_silu_block_kernel(float* __restrict__ out, const TA* __restrict__ proj, int stride, int col0, const float* __restrict__ taps_w,
                              const float* __restrict__ bias, const float* __restrict__ tails, const int32_t* __restrict__ tok_seq,
                              const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ slots, int tokens, int channels) {
    const int t0 = blockIdx.x * CONV_TOKENS, ch = (blockIdx.y * 256 + threadIdx.x) * 4;
    if (ch >= channels) return;
    conv_f32x4 row[CONV_TOKENS + 3], w[4], b = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < CONV_TOKENS + 3; ++r)                 // (rows before the first and past the last: read again, not used)
        row[r] = conv_four(proj + (size_t)min(max(t0 - 3 + r, 0), tokens - 1) * stride + col0 + ch);
#pragma unroll
    for (int c = 0; c < 4; ++c) w[c] = conv_four(taps_w + (size_t)(ch + c) * 4);
    if (bias) b = conv_four(bias + ch);
#pragma unroll
    for (int d = 0; d < CONV_TOKENS; ++d) {
        const int t = t0 + d;
        if (t >= tokens) return;
        const int seq = tok_seq[t], i = t - cu_seqlens[seq];  // the token's place in this step
        conv_f32x4 in[4] = {row[d], row[d + 1], row[d + 2], row[d + 3]}, y;
        if (i < 3) {
            const float* tail = tails + (size_t)slots[seq] * 3 * channels + ch;
#pragma unroll
            for (int a = 0; a < 3; ++a)
                if (i + a < 3) in[a] = conv_four(tail + (size_t)(i + a) * channels);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float sum = 0.f;
#pragma unroll
            for (int a = 0; a < 4; ++a) sum += in[a][c] * w[c][a];  // oldest first
            if (bias) sum += b[c];
            y[c] = sum / (1.f + expf(-sum));
        }
        *reinterpret_cast<conv_f32x4*>(out + (size_t)t * channels + ch) = y;
    }
}

template <typename TA>
__global__ void __launch_bounds__(256)
conv_tails_kernel(float* __restrict__ tails, const TA* __restrict__ proj, int stride, int col0, int taps,
                  const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ slots, int channels) {
    const int seq = blockIdx.x, ch = blockIdx.y * 256 + threadIdx.x;
    if (ch >= channels) return;
    const int first = cu_seqlens[seq], n = cu_seqlens[seq + 1] - first;
    if (n == 0) return;
    float* tail = tails + (size_t)slots[seq] * (taps - 1) * channels;
    float keep[SSD_MAX_TAPS];
    for (int idx = 0; idx < taps - 1; ++idx) {
        const int src = n - (taps - 1) + idx;                 // the step's token that lands at this place, if any
        keep[idx] = src >= 0 ? to_f32(proj[(size_t)(first + src) * stride + col0 + ch])
                             : tail[(size_t)(idx + n) * channels + ch];
    }
    for (int idx = 0; idx < taps - 1; ++idx) tail[(size_t)idx * channels + ch] = keep[idx];
}

// Whether a step takes the block form: from as many results on as fill the machine with 32 a thread; below, its chain of eight tokens is
// what a launch takes (us with the tails' launch, an element a thread : blocks; 1,536 channels of 256 / 512 / 1,024 tokens 6.4 : 7.9, 8.8 :
// 8.4, 12.7 : 8.6; 6,144 channels of 64 / 128 / 256 / 2,048 tokens 6.4 : 8.1, 9.2 : 8.2, 12.9 : 8.7, 86.0 : 22.9).  Where sequences bring
// fewer than two tokens on average most rows take their tails, four loads a row in a pass of their own: four times as many
// results (6,144 channels of 128 / 256 / 512 sequences of one token 11.1 : 15.9, 18.3 : 21.4, 34.2 : 26.9; of two tokens 20.3 : 15.8 at 128).
extern "C" int ri_causal_conv_blocks(int tokens, int seqs, int channels) {
    return (long)tokens * channels >= (tokens >= 2L * seqs ? 1 : 4) * CONV_BLOCK_FROM;
}

extern "C" int ri_causal_conv_silu(float* out, const void* proj, int act_dtype, int stride, int col0, const float* taps_w,
                                   const float* bias, float* tails, int taps, const int32_t* tok_seq, const int32_t* cu_seqlens,
                                   const int32_t* slots, int tokens, int seqs, int channels, int update_tails, void* stream) {
    RI_REQUIRE(tokens > 0 && seqs > 0 && channels > 0 && taps >= 1 && taps <= SSD_MAX_TAPS,
               "causal_conv_silu: %d tokens, %d channels, %d taps (up to %d)", tokens, channels, taps, SSD_MAX_TAPS);
    RI_REQUIRE(col0 >= 0 && col0 + channels <= stride, "causal_conv_silu: columns %d..%d of rows of %d", col0, col0 + channels, stride);
    RI_REQUIRE(act_dtype == RI_F32 || act_dtype == RI_BF16, "causal_conv_silu: dtype %d", act_dtype);
    RI_REQUIRE(taps == 1 || tails, "causal_conv_silu: a convolution of %d taps keeps a tail", taps);
    hipStream_t s = (hipStream_t)stream;
    const int cy = (channels + 255) / 256;
    // (a thread's four channels of the block form have to start on the boundary of their loads)
    const bool four = taps == 4 && ri_causal_conv_blocks(tokens, seqs, channels) && channels % 4 == 0 && stride % 4 == 0 && col0 % 4 == 0 &&
                      (((uintptr_t)out | (uintptr_t)taps_w | (uintptr_t)bias | (uintptr_t)tails) & 15) == 0 &&
                      ((uintptr_t)proj & (act_dtype == RI_F32 ? 15 : 7)) == 0;
    if (!update_tails && four) {
        const dim3 grid((tokens + CONV_TOKENS - 1) / CONV_TOKENS, (channels / 4 + 255) / 256);
        if (act_dtype == RI_F32)
            causal_conv_silu_block_kernel<float><<<grid, 256, 0, s>>>(out, (const float*)proj, stride, col0, taps_w, bias, tails, tok_seq,
                                                                     cu_seqlens, slots, tokens, channels);
        else
            causal_conv_silu_block_kernel<bf16_t><<<grid, 256, 0, s>>>(out, (const bf16_t*)proj, stride, col0, taps_w, bias, tails, tok_seq,
                                                                      cu_seqlens, slots, tokens, channels);
    } else if (!update_tails) {
        if (act_dtype == RI_F32)
            causal_conv_silu_kernel<float><<<dim3(tokens, cy), 256, 0, s>>>(out, (const float*)proj, stride, col0, taps_w, bias, tails,
                                                                           taps, tok_seq, cu_seqlens, slots, channels);
        else
            causal_conv_silu_kernel<bf16_t><<<dim3(tokens, cy), 256, 0, s>>>(out, (const bf16_t*)proj, stride, col0, taps_w, bias,
                                                                            tails, taps, tok_seq, cu_seqlens, slots, channels);
    } else if (taps > 1) {
        if (act_dtype == RI_F32)
            conv_tails_kernel<float><<<dim3(seqs, cy), 256, 0, s>>>(tails, (const float*)proj, stride, col0, taps, cu_seqlens, slots, channels);
        else
            conv_tails_kernel<bf16_t><<<dim3(seqs, cy), 256, 0, s>>>(tails, (const bf16_t*)proj, stride, col0, taps, cu_seqlens, slots, channels);
    }
    RI_LAUNCH_CHECK("causal_conv_silu");
    return 0;
}

// ------------------------------------------------------------------ the walk
// blockDim.x = vdim * slices; thread (slice, c) holds the rows slice * RPT .. + RPT - 1 (of the state's N) of column c.
template <typename TA, int RPT>
__global__ void __launch_bounds__(1024)
ssd_scan_kernel(float* __restrict__ out, const float* __restrict__ xbc, int channels, int b_off, int c_off,
                const TA* __restrict__ proj, int stride, int z_off, int dt_off, const float* __restrict__ dt_bias,
                const float* __restrict__ a_log, const float* __restrict__ d_skip, float* __restrict__ state,
                const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ slots, int heads, int groups, int n,
                int vdim, int slices) {
    extern __shared__ float lds[];
    float* bs = lds;                       // [n] B
    float* cs = bs + n;                    // [n] C
    float* xs = cs + n;                    // [vdim] x
    float* red = xs + vdim;                // [slices][vdim]
    const int seq = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const int c = tid % vdim, slice = tid / vdim;
    const int row0 = slice * RPT;
    const int group = h / (heads / groups);
    const int inner = heads * vdim;
    float* sp = state + (((size_t)slots[seq] * heads + h) * n) * vdim;
    float st[RPT];
#pragma unroll
    for (int i = 0; i < RPT; ++i) st[i] = row0 + i < n ? sp[(size_t)(row0 + i) * vdim + c] : 0.f;
    const float neg_a = -expf(a_log[h]), skip = d_skip ? d_skip[h] : 0.f, bias = dt_bias ? dt_bias[h] : 0.f;
    const int t0 = cu_seqlens[seq], t1 = cu_seqlens[seq + 1];
    for (int t = t0; t < t1; ++t) {
        const float* row = xbc + (size_t)t * channels;
        __syncthreads();
        for (int e = tid; e < n; e += blockDim.x) {
            bs[e] = row[b_off + group * n + e];
            cs[e] = row[c_off + group * n + e];
        }
        if (tid < vdim) xs[tid] = row[h * vdim + tid];
        __syncthreads();
        const float raw = to_f32(proj[(size_t)t * stride + dt_off + h]) + bias;
        const float dt = raw > 20.f ? raw : log1pf(expf(raw));           // softplus: beyond 20 it is its argument to the last bit
        const float decay = expf(neg_a * dt);
        const float dx = dt * xs[c];
        float part = 0.f;
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const int r = row0 + i;
            if (r < n) {
                st[i] = decay * st[i] + bs[r] * dx;
                part += st[i] * cs[r];
            }
        }
        red[slice * vdim + c] = part;
        __syncthreads();
        if (tid < vdim) {
            float y = 0.f;
            for (int s = 0; s < slices; ++s) y += red[s * vdim + tid];
            y += skip * xs[tid];
            const float z = to_f32(proj[(size_t)t * stride + z_off + h * vdim + tid]);
            out[(size_t)t * inner + h * vdim + tid] = y * (z / (1.f + expf(-z)));
        }
    }
#pragma unroll
    for (int i = 0; i < RPT; ++i)
        if (row0 + i < n) sp[(size_t)(row0 + i) * vdim + c] = st[i];
}

extern "C" int ri_ssd_scan(float* out, const float* xbc, int channels, int b_off, int c_off, const void* proj, int act_dtype,
                           int stride, int z_off, int dt_off, const float* dt_bias, const float* a_log, const float* d_skip,
                           float* state, const int32_t* cu_seqlens, const int32_t* slots, int seqs, int heads, int groups,
                           int n, int vdim, void* stream) {
    RI_REQUIRE(seqs > 0 && heads > 0 && heads <= 65535 && groups > 0 && heads % groups == 0 && n >= 1 && vdim >= 1 && vdim <= 256 &&
               n <= 1024, "ssd_scan: %d sequences, %d heads in %d groups, state %d x %d", seqs, heads, groups, n, vdim);
    RI_REQUIRE(b_off >= 0 && c_off >= 0 && b_off + groups * n <= channels && c_off + groups * n <= channels && heads * vdim <= channels,
               "ssd_scan: columns %d and %d of %d channels", b_off, c_off, channels);
    RI_REQUIRE(z_off >= 0 && dt_off >= 0 && z_off + heads * vdim <= stride && dt_off + heads <= stride,
               "ssd_scan: columns %d and %d of rows of %d", z_off, dt_off, stride);
    RI_REQUIRE(act_dtype == RI_F32 || act_dtype == RI_BF16, "ssd_scan: dtype %d", act_dtype);
    int slices = (n + 31) / 32;
    while (slices * 2 * vdim <= 256) slices *= 2;
    if (slices > n) slices = n;
    while (slices > 1 && slices * vdim > 1024) slices /= 2;
    const int rpt = (n + slices - 1) / slices;
    RI_REQUIRE(slices * vdim <= 1024 && rpt <= 64, "ssd_scan: a state of %d x %d does not fit a workgroup", n, vdim);
    const dim3 grid(seqs, heads);
    const int threads = slices * vdim;
    const size_t lds = ((size_t)2 * n + vdim + (size_t)slices * vdim) * sizeof(float);
    hipStream_t s = (hipStream_t)stream;
#define RI_GO(TA, RPT)                                                                                                  \
    ssd_scan_kernel<TA, RPT><<<grid, threads, lds, s>>>(out, xbc, channels, b_off, c_off, (const TA*)proj, stride, z_off, \
                                                        dt_off, dt_bias, a_log, d_skip, state, cu_seqlens, slots, heads, \
                                                        groups, n, vdim, slices)
#define RI_BY_ROWS(TA)                                                                                                  \
    if (rpt <= 8) RI_GO(TA, 8); else if (rpt <= 16) RI_GO(TA, 16); else if (rpt <= 32) RI_GO(TA, 32); else RI_GO(TA, 64)
    if (act_dtype == RI_F32) { RI_BY_ROWS(float); } else { RI_BY_ROWS(bf16_t); }
#undef RI_BY_ROWS
#undef RI_GO
    RI_LAUNCH_CHECK("ssd_scan");
    return 0;
}

// ------------------------------------------------------------------ the walk, a wavefront on 16 columns
// States of up to 64 rows: a wavefront owns 16 columns of one (sequence, head), its lanes four slices of the rows of a
// column each, the rows in registers; a token's sum over the rows is the lane's own sum (four partial sums, so that no
// addition waits for the one before) and two exchanges between the lanes of a column.  A workgroup is four wavefronts
// on columns of their own, which share the tokens staged in LDS in blocks of SSD_BLOCK (B, C, x, the step size and decay, z), the next block's loads asked
// for before the block in work is computed.  The order of a token's additions is fixed by the sizes alone.
#define SSD_BLOCK 8
#define SSD_WAVES 4          // wavefronts of a workgroup: they share the staged tokens, each on columns of its own

template <typename TA, int RPL>                               // RPL: rows a lane holds, a multiple of 4
__global__ void __launch_bounds__(64 * SSD_WAVES)
ssd_scan_cols_kernel(float* __restrict__ out, const float* __restrict__ xbc, int channels, int b_off, int c_off,
                     const TA* __restrict__ proj, int stride, int z_off, int dt_off, const float* __restrict__ dt_bias,
                     const float* __restrict__ a_log, const float* __restrict__ d_skip, float* __restrict__ state,
                     const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ slots, int heads, int groups, int n,
                     int vdim) {
    // SL: slices of rows; COLS: columns of a wavefront; NC: of the workgroup; TPP: tokens whose x and z one pass of the workgroup's threads fetches
    constexpr int SL = 4, ROWS = SL * RPL, COLS = 64 / SL, NC = COLS * SSD_WAVES, THREADS = 64 * SSD_WAVES, TPP = THREADS / NC,
                  PASSES = SSD_BLOCK / TPP;
    __shared__ __attribute__((aligned(16))) float bs[2][SSD_BLOCK][ROWS];
    __shared__ __attribute__((aligned(16))) float cs[2][SSD_BLOCK][ROWS];
    __shared__ float xs[2][SSD_BLOCK][NC];
    __shared__ float zs[2][SSD_BLOCK][NC];
    __shared__ float dts[2][SSD_BLOCK], decays[2][SSD_BLOCK];
    const int seq = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane % COLS, slice = lane / COLS, row0 = slice * RPL;
    const int wcol = wave * COLS + col;                       // the lane's column among the workgroup's
    const int c = blockIdx.z * NC + wcol;
    const bool has_col = c < vdim;
    const int cc = has_col ? c : vdim - 1;                    // a column pulled back inside the head: loads are issued anyway
    const int group = h / (heads / groups), inner = heads * vdim;
    float* sp = state + (((size_t)slots[seq] * heads + h) * n) * vdim + cc;
    float st[RPL];
#pragma unroll
    for (int i = 0; i < RPL; ++i) st[i] = row0 + i < n ? sp[(size_t)(row0 + i) * vdim] : 0.f;
    const float neg_a = -expf(a_log[h]), skip = d_skip ? d_skip[h] : 0.f, bias = dt_bias ? dt_bias[h] : 0.f;
    const int t0 = cu_seqlens[seq], t1 = cu_seqlens[seq + 1];
    constexpr int PER = (2 * SSD_BLOCK * ROWS + THREADS - 1) / THREADS;     // B and C elements of a block a thread stages
    const int vcol = min((int)blockIdx.z * NC + tid % NC, vdim - 1), vtok = tid / NC;      // the thread's place in a pass over x and z

    float pre_bc[PER], pre_x[PASSES], pre_z[PASSES], pre_raw = 0.f;
    auto fetch = [&](int tb) {                                // a block's loads, into registers
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = tid + i * THREADS;                  // (which, token, row)
            const int r = e % ROWS, tt = (e / ROWS) % SSD_BLOCK, which = e / (ROWS * SSD_BLOCK);
            const int t = min(tb + tt, t1 - 1);
            pre_bc[i] = (r < n && which < 2) ? xbc[(size_t)t * channels + (which ? c_off : b_off) + group * n + r] : 0.f;
        }
#pragma unroll
        for (int ps = 0; ps < PASSES; ++ps) {                 // x and z of the block's tokens for this wavefront's columns
            const int t = min(tb + ps * TPP + vtok, t1 - 1);
            pre_x[ps] = xbc[(size_t)t * channels + h * vdim + vcol];
            pre_z[ps] = to_f32(proj[(size_t)t * stride + z_off + h * vdim + vcol]);
        }
        if (tid < SSD_BLOCK) pre_raw = to_f32(proj[(size_t)min(tb + tid, t1 - 1) * stride + dt_off + h]);
    };
    auto stage = [&](int buf) {                               // ... and from there into LDS
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = tid + i * THREADS;
            const int r = e % ROWS, tt = (e / ROWS) % SSD_BLOCK, which = e / (ROWS * SSD_BLOCK);
            if (which == 0) bs[buf][tt][r] = pre_bc[i];
            else if (which == 1) cs[buf][tt][r] = pre_bc[i];
        }
#pragma unroll
        for (int ps = 0; ps < PASSES; ++ps) {
            xs[buf][ps * TPP + vtok][tid % NC] = pre_x[ps];
            zs[buf][ps * TPP + vtok][tid % NC] = pre_z[ps];
        }
        if (tid < SSD_BLOCK) {
            const float raw = pre_raw + bias;
            const float dt = raw > 20.f ? raw : log1pf(expf(raw));       // softplus: beyond 20 it is its argument to the last bit
            dts[buf][tid] = dt;
            decays[buf][tid] = expf(neg_a * dt);
        }
    };
    if (t0 < t1) {
        fetch(t0);
        stage(0);
    }
    __syncthreads();
    int buf = 0;
    for (int tb = t0; tb < t1; tb += SSD_BLOCK, buf ^= 1) {
        const bool more = tb + SSD_BLOCK < t1;
        if (more) {
            fetch(tb + SSD_BLOCK);
        }
        const int count = min(SSD_BLOCK, t1 - tb);
        float part[SSD_BLOCK];                                // the lane's share of each token's sum: the exchanges wait for the block's end,
#pragma unroll                                                // so that no token waits for the one before it
        for (int tt = 0; tt < SSD_BLOCK; ++tt) {
            part[tt] = 0.f;
            if (tt < count) {
                const float decay = decays[buf][tt];
                const float dx = dts[buf][tt] * xs[buf][tt][wcol];
                float y0 = 0.f, y1 = 0.f, y2 = 0.f, y3 = 0.f;
#pragma unroll
                for (int i = 0; i < RPL; i += 4) {
                    const float4 b4 = *reinterpret_cast<const float4*>(&bs[buf][tt][row0 + i]);
                    const float4 c4 = *reinterpret_cast<const float4*>(&cs[buf][tt][row0 + i]);
                    st[i] = decay * st[i] + b4.x * dx;             y0 += st[i] * c4.x;
                    st[i + 1] = decay * st[i + 1] + b4.y * dx;     y1 += st[i + 1] * c4.y;
                    st[i + 2] = decay * st[i + 2] + b4.z * dx;     y2 += st[i + 2] * c4.z;
                    st[i + 3] = decay * st[i + 3] + b4.w * dx;     y3 += st[i + 3] * c4.w;
                }
                part[tt] = (y0 + y1) + (y2 + y3);
            }
        }
#pragma unroll
        for (int tt = 0; tt < SSD_BLOCK; ++tt) {
            float y = part[tt];
            y += __shfl_xor(y, 16, RI_WAVE);                  // the slices of a column
            y += __shfl_xor(y, 32, RI_WAVE);
            if (tt < count && has_col && slice == 0) {
                y += skip * xs[buf][tt][wcol];
                const float z = zs[buf][tt][wcol];
                out[(size_t)(tb + tt) * inner + h * vdim + c] = y * (z / (1.f + expf(-z)));
            }
        }
        if (more) stage(buf ^ 1);
        __syncthreads();
    }
    if (has_col) {
#pragma unroll
        for (int i = 0; i < RPL; ++i)
            if (row0 + i < n) sp[(size_t)(row0 + i) * vdim] = st[i];
    }
}

// States of 65 to 128 rows: the walk of walk.h.  2,048 tokens of one sequence, 32 heads of 128 x 128: 1,130 us with a lane on 16
// rows of a column (its reads of B and C from LDS for one column each), 310 with tiles of four rows.
template <typename TA, int CPL, bool VEC>
__global__ void __launch_bounds__(256)
ssd_walk_kernel(float* __restrict__ out, const float* __restrict__ xbc, int channels, int b_off, int c_off,
                const TA* __restrict__ proj, int stride, int z_off, int dt_off, const float* __restrict__ dt_bias,
                const float* __restrict__ a_log, const float* __restrict__ d_skip, float* __restrict__ state,
                const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ slots, int heads, int groups, int n,
                int vdim) {
    constexpr int NC = 8 * CPL;
    __shared__ float4 bs[2][WALK_BLOCK][WALK_ROWS / 4], cs[2][WALK_BLOCK][WALK_ROWS / 4];
    __shared__ __attribute__((aligned(16))) float xs[2][WALK_BLOCK][NC];
    __shared__ float zs[2][WALK_BLOCK][NC];
    __shared__ float dts[2][64], decays[2][64];               // 64 tokens' step sizes and decays, and the next 64's
    const int seq = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int slice = lane & 31, row0 = 4 * slice, wcol = wave * 2 * CPL + (lane >> 5) * CPL, first_col = blockIdx.z * NC;
    const int group = h / (heads / groups), inner = heads * vdim;
    float* sp = state + (((size_t)slots[seq] * heads + h) * n) * vdim;
    float st[4][CPL];
    walk_load<CPL>(st, sp, row0, n, first_col + wcol, vdim);
    const float neg_a = -expf(a_log[h]), skip = d_skip ? d_skip[h] : 0.f, bias = dt_bias ? dt_bias[h] : 0.f;
    const int t0 = cu_seqlens[seq], t1 = cu_seqlens[seq + 1];
    if (t0 >= t1) return;                                     // (the whole workgroup; the state stays)
    const int btok = tid / 32, brow = 4 * (tid & 31);         // the thread's piece of B and C, and its element of x and z
    const int vtok = tid / NC % WALK_BLOCK, vcol = min(first_col + tid % NC, vdim - 1);
    struct Ahead { float4 b, c; float x, z; };
    auto fetch = [&](Ahead& a, int tb) {                      // (always issued, from a token pulled back inside the sequence)
        const float* row = xbc + (size_t)min(tb + btok, t1 - 1) * channels + group * n;
        a.b = walk_rows<VEC>(row + b_off, brow, n);
        a.c = walk_rows<VEC>(row + c_off, brow, n);
        const int t = min(tb + vtok, t1 - 1);
        a.x = xbc[(size_t)t * channels + h * vdim + vcol];
        a.z = to_f32(proj[(size_t)t * stride + z_off + h * vdim + vcol]);
    };
    auto stage = [&](const Ahead& a, int tb, int buf) {
        const bool in = tb + btok < t1;
        bs[buf][btok][tid & 31] = walk_keep(a.b, brow, n, in, 0.f);
        cs[buf][btok][tid & 31] = walk_keep(a.c, brow, n, in, 0.f);
        if (tid < WALK_BLOCK * NC) {
            xs[buf][vtok][tid % NC] = tb + vtok < t1 ? a.x : 0.f;
            zs[buf][vtok][tid % NC] = a.z;
        }
    };
    // the step sizes of 64 tokens at once, a lane a token: softplus and the decay's exponential take a wavefront what one token's do
    auto raw_of = [&](int first) { return to_f32(proj[(size_t)min(first + lane, t1 - 1) * stride + dt_off + h]); };
    auto put_steps = [&](float raw, int first) {
        raw += bias;
        const float dt = raw > 20.f ? raw : log1pf(expf(raw));           // softplus: beyond 20 it is its argument to the last bit
        const bool in = first + lane < t1;
        dts[(first - t0) >> 6 & 1][lane] = in ? dt : 0.f;
        decays[(first - t0) >> 6 & 1][lane] = in ? expf(neg_a * dt) : 1.f;
    };
    auto block = [&](int tb, int buf, float raw) {
        const int at = (tb - t0) & 63, half = (tb - t0) >> 6 & 1;
        float part[WALK_BLOCK * CPL];
#pragma unroll
        for (int tt = 0; tt < WALK_BLOCK; ++tt) {
            const float dt = dts[half][at + tt], decay = decays[half][at + tt];
            const float4 b = bs[buf][tt][slice], c = cs[buf][tt][slice];
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const float dx = dt * xs[buf][tt][wcol + j];
                st[0][j] = decay * st[0][j] + b.x * dx;
                st[1][j] = decay * st[1][j] + b.y * dx;
                st[2][j] = decay * st[2][j] + b.z * dx;
                st[3][j] = decay * st[3][j] + b.w * dx;
                part[tt * CPL + j] = (st[0][j] * c.x + st[1][j] * c.y) + (st[2][j] * c.z + st[3][j] * c.w);
            }
        }
        const float sum = walk_sum<CPL>(part, lane);
        const int mine = walk_mine<CPL>(lane), tt = mine / CPL, col = wcol + mine % CPL;
        if (mine < WALK_BLOCK * CPL && tb + tt < t1 && first_col + col < vdim) {
            const float y = sum + skip * xs[buf][tt][col], z = zs[buf][tt][col];
            out[(size_t)(tb + tt) * inner + h * vdim + first_col + col] = y * (z / (1.f + expf(-z)));
        }
        if (at == 64 - WALK_BLOCK && wave == 0) put_steps(raw, tb + WALK_BLOCK);
    };
    // two blocks are on their way in registers while a third is computed: a block is computed in less than memory's latency
    Ahead even, odd;
    fetch(even, t0);
    fetch(odd, t0 + WALK_BLOCK);
    if (wave == 0) put_steps(raw_of(t0), t0);
    stage(even, t0, 0);
    __syncthreads();
    for (int tb = t0; tb < t1; tb += 2 * WALK_BLOCK) {        // (blocks come in pairs)
        const float raw = raw_of(t0 + (((tb - t0) >> 6) + 1) * 64);
        fetch(even, tb + 2 * WALK_BLOCK);
        block(tb, 0, raw);
        stage(odd, tb + WALK_BLOCK, 1);
        __syncthreads();
        if (tb + WALK_BLOCK >= t1) break;                     // (a step of single tokens is one block)
        fetch(odd, tb + 3 * WALK_BLOCK);
        block(tb + WALK_BLOCK, 1, raw);
        stage(even, tb + 2 * WALK_BLOCK, 0);
        __syncthreads();
    }
    walk_store<CPL>(st, sp, row0, n, first_col + wcol, vdim);
}

extern "C" int ri_ssd_scan_cols_fits(int n, int vdim) { return n >= 1 && n <= 128 && vdim >= 1; }

extern "C" int ri_ssd_scan_cols(float* out, const float* xbc, int channels, int b_off, int c_off, const void* proj, int act_dtype,
                                int stride, int z_off, int dt_off, const float* dt_bias, const float* a_log, const float* d_skip,
                                float* state, const int32_t* cu_seqlens, const int32_t* slots, int tokens, int seqs, int heads, int groups,
                                int n, int vdim, void* stream) {
    RI_REQUIRE(tokens >= 0 && seqs > 0 && heads > 0 && heads <= 65535 && groups > 0 && heads % groups == 0 && ri_ssd_scan_cols_fits(n, vdim),
               "ssd_scan_cols: %d sequences, %d heads in %d groups, state %d x %d", seqs, heads, groups, n, vdim);
    RI_REQUIRE(b_off >= 0 && c_off >= 0 && b_off + groups * n <= channels && c_off + groups * n <= channels && heads * vdim <= channels,
               "ssd_scan_cols: columns %d and %d of %d channels", b_off, c_off, channels);
    RI_REQUIRE(z_off >= 0 && dt_off >= 0 && z_off + heads * vdim <= stride && dt_off + heads <= stride,
               "ssd_scan_cols: columns %d and %d of rows of %d", z_off, dt_off, stride);
    RI_REQUIRE(act_dtype == RI_F32 || act_dtype == RI_BF16, "ssd_scan_cols: dtype %d", act_dtype);
    hipStream_t s = (hipStream_t)stream;
    if (n > 64) {
        const int cpl = walk_columns((long)seqs * heads * vdim, tokens == seqs);
        const dim3 grid(seqs, heads, (vdim + 8 * cpl - 1) / (8 * cpl));
        RI_REQUIRE(grid.z <= 65535, "ssd_scan_cols: heads of %d channels", vdim);
        const bool vec = n % 4 == 0 && (channels | b_off | c_off) % 4 == 0 && (uintptr_t)xbc % 16 == 0;
#define RI_GO(TA, CPL, VEC)                                                                                             \
    ssd_walk_kernel<TA, CPL, VEC><<<grid, 256, 0, s>>>(out, xbc, channels, b_off, c_off, (const TA*)proj, stride, z_off, dt_off, \
                                                       dt_bias, a_log, d_skip, state, cu_seqlens, slots, heads, groups, n, vdim)
#define RI_BY_COLUMNS(TA, VEC) if (cpl == 1) RI_GO(TA, 1, VEC); else if (cpl == 2) RI_GO(TA, 2, VEC); else RI_GO(TA, 4, VEC)
        if (act_dtype == RI_F32) { if (vec) { RI_BY_COLUMNS(float, true); } else { RI_BY_COLUMNS(float, false); } }
        else                     { if (vec) { RI_BY_COLUMNS(bf16_t, true); } else { RI_BY_COLUMNS(bf16_t, false); } }
#undef RI_BY_COLUMNS
#undef RI_GO
        RI_LAUNCH_CHECK("ssd_scan_cols");
        return 0;
    }
    const int cols = 16 * SSD_WAVES;
    const dim3 grid(seqs, heads, (vdim + cols - 1) / cols);
    RI_REQUIRE(grid.z <= 65535, "ssd_scan_cols: heads of %d channels", vdim);
#define RI_GO(TA, RPL)                                                                                                  \
    ssd_scan_cols_kernel<TA, RPL><<<grid, 64 * SSD_WAVES, 0, s>>>(out, xbc, channels, b_off, c_off, (const TA*)proj, stride, z_off,  \
                                                      dt_off, dt_bias, a_log, d_skip, state, cu_seqlens, slots, heads,   \
                                                      groups, n, vdim)
#define RI_BY_ROWS(TA)                                                                                                  \
    if (n <= 16) RI_GO(TA, 4); else if (n <= 32) RI_GO(TA, 8); else RI_GO(TA, 16)
    if (act_dtype == RI_F32) { RI_BY_ROWS(float); } else { RI_BY_ROWS(bf16_t); }
#undef RI_BY_ROWS
#undef RI_GO
    RI_LAUNCH_CHECK("ssd_scan_cols");
    return 0;
}

// ------------------------------------------------------------------ the norm in parts
template <typename TO>
__global__ void __launch_bounds__(256)
group_rms_norm_kernel(TO* __restrict__ out, const float* __restrict__ x, const float* __restrict__ gain, float eps, int width,
                      int part) {
    __shared__ float scratch[16];
    const size_t at = (size_t)blockIdx.x * width + (size_t)blockIdx.y * part;
    float ss = 0.f;
    for (int d = threadIdx.x; d < part; d += 256) ss += x[at + d] * x[at + d];
    const float inv = 1.0f / sqrtf(block_sum(ss, scratch) / (float)part + eps);
    for (int d = threadIdx.x; d < part; d += 256)
        from_f32(out + at + d, x[at + d] * inv * (gain ? gain[blockIdx.y * part + d] : 1.f));
}

extern "C" int ri_group_rms_norm(void* out, int out_dtype, const float* x, const float* gain, float eps, int rows, int width,
                                 int parts, void* stream) {
    RI_REQUIRE(rows > 0 && width > 0 && parts >= 1 && parts <= 65535 && width % parts == 0, "group_rms_norm: %d rows of %d in %d parts",
               rows, width, parts);
    RI_REQUIRE(out_dtype == RI_F32 || out_dtype == RI_BF16, "group_rms_norm: dtype %d", out_dtype);
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid(rows, parts);
    if (out_dtype == RI_F32) group_rms_norm_kernel<float><<<grid, 256, 0, s>>>((float*)out, x, gain, eps, width, width / parts);
    else group_rms_norm_kernel<bf16_t><<<grid, 256, 0, s>>>((bf16_t*)out, x, gain, eps, width, width / parts);
    RI_LAUNCH_CHECK("group_rms_norm");
    return 0;
}
