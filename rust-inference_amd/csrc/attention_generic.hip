// Causal grouped-query attention over the paged cache for any number of new tokens per sequence:
// the form every other attention kernel here is checked against, and the one the float32 path runs (heads of 64 and 128 in a form of
// their own on the matrix cores, at the end).
// One workgroup per (token, query head); keys in tiles of 256 that start at multiples of 256, so the
// order of every sum depends on the key's position alone, never on how tokens were cut into steps.
//
// score_j = (q . k_j) * scale, then, with a cap c > 0, score_j <- c tanh(score_j / c), then, with a slope per
// query head, score_j <- score_j - slope_h (p - j); the query at position p
// sees keys lo..p with lo = 0, p - window + 1 or the start of the chunk of positions that p lies in, and with keep_first > 0 also the keys 0..keep_first-1 that lie
// before lo (the first tokens of a sequence stay visible behind the window); with a sink per query head the
// softmax's denominator also holds exp(sink_h), which has no key and no value;
// online softmax with running maximum m, running sum l and factor exp(m_old - m_new)
// (the reference: src/attention.rs:117-149; its GPU form src/cuda/kernels.cu:345-405).
//
// Any head size from 1 to 1,024 (the reference asks only that it be even, and only because of its rotation:
// src/models/config.rs:98-100; its own attention test runs head size 8, src/attention.rs:189-219): keys are
// read 16 bytes at a time where a key row starts on a 16-byte boundary (head sizes that are multiples of 4
// in float32, of 8 in bfloat16) and element by element otherwise; a thread accumulates up to four channels.
// The value heads may have another size (v_dim) than the query and key heads.
#include "api.h"
#include "common.h"

#define ATT_TILE 256

template <typename TC> struct Vec;
template <> struct Vec<float> {
    static constexpr int N = 4;
    __device__ static void load(const float* p, float* o) {
        const float4 v = *reinterpret_cast<const float4*>(p);
        o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
    }
};
template <> struct Vec<bf16_t> {
    static constexpr int N = 8;
    __device__ static void load(const bf16_t* p, float* o) {
        const uint4 v = *reinterpret_cast<const uint4*>(p);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o[2 * i] = __uint_as_float(w[i] << 16);
            o[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
        }
    }
};

#define ATT_ACCS 4                              // channels of a value head a thread accumulates
#define ATT_MAX_HEAD_DIM (ATT_ACCS * ATT_TILE)

template <typename TA, typename TC, bool VEC>
__global__ void __launch_bounds__(ATT_TILE)
attention_generic_kernel(TA* __restrict__ out, const TA* __restrict__ q, int q_stride, const TC* __restrict__ k_pages,
                         const TC* __restrict__ v_pages, const int32_t* __restrict__ tok_pos,
                         const int32_t* __restrict__ tok_seq, const int32_t* __restrict__ page_table, int table_width,
                         int heads, int kv_heads, int head_dim, int v_dim, int page_size, Reach reach, float scale,
                         float softcap, const float* __restrict__ slopes, int keep_first,
                         const float* __restrict__ sinks, const int32_t* __restrict__ cu_seqlens, int rows_from) {
    // (sequences of so many new tokens are the other kernel's, below)
    if (cu_seqlens && cu_seqlens[tok_seq[blockIdx.x] + 1] - cu_seqlens[tok_seq[blockIdx.x]] >= rows_from) return;
    extern __shared__ float qs[];                 // head_dim floats: the query
    __shared__ float ps[ATT_TILE];                // this tile's weights
    __shared__ long rowoff[ATT_TILE];             // element offset of each key's column in the value pool
    __shared__ float scratch[16];

    const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const int kvh = h / (heads / kv_heads);       // consecutive query heads share a kv head
    const int qpos = tok_pos[t];
    const int lo = reach.first(qpos);
    const float slope = slopes ? slopes[h] : 0.f;
    const int32_t* table = page_table + (size_t)tok_seq[t] * table_width;

    for (int d = tid; d < head_dim; d += ATT_TILE) qs[d] = to_f32(q[(size_t)t * q_stride + (size_t)h * head_dim + d]);
    __syncthreads();

    float m = -INFINITY, l = 0.f, acc = 0.f, acc2 = 0.f;      // channels tid and tid + 256
    float acc3 = 0.f, acc4 = 0.f;                              // and tid + 512, tid + 768 (value heads above 512)
    const int kept = min(keep_first, lo);         // keys 0..kept-1 are seen although they lie behind the window
    const int lo_tile = lo / ATT_TILE, kept_tiles = (kept + ATT_TILE - 1) / ATT_TILE;
    for (int tile = 0; tile <= qpos / ATT_TILE; ++tile) {
        if (tile >= kept_tiles && tile < lo_tile) { tile = lo_tile - 1; continue; }      // (the same for the whole workgroup)
        const int j = tile * ATT_TILE + tid;
        const bool valid = (j >= lo || j < kept) && j <= qpos;
        float s = -INFINITY;
        if (valid) {
            const long page_head = ((long)table[j / page_size] * kv_heads + kvh) * page_size;
            const long head_base = page_head * head_dim;
            rowoff[tid] = page_head * v_dim + j % page_size;       // the key's column in the transposed value page
            const TC* kr = k_pages + head_base + (long)(j % page_size) * head_dim;
            float dot = 0.f;
            if (VEC) {
                for (int d = 0; d < head_dim; d += Vec<TC>::N) {
                    float kv[Vec<TC>::N];
                    Vec<TC>::load(kr + d, kv);
#pragma unroll
                    for (int e = 0; e < Vec<TC>::N; ++e) dot += qs[d + e] * kv[e];
                }
            } else {
                for (int d = 0; d < head_dim; ++d) dot += qs[d] * to_f32(kr[d]);      // the same order of additions
            }
            s = dot * scale;
            if (softcap > 0.f) s = softcap * tanhf(s / softcap);
            if (slopes) s -= slope * (float)(qpos - j);
        }
        const float m_new = fmaxf(m, block_max(s, scratch));
        const float p = valid ? expf(s - m_new) : 0.f;
        ps[tid] = p;
        const float tile_sum = block_sum(p, scratch);      // its barriers also publish ps and rowoff
        const float corr = expf(m - m_new);                // 0 on the first tile (m = -inf)
        l = l * corr + tile_sum;
        m = m_new;
        if (tid < v_dim) {
            acc *= corr;
            acc2 *= corr;
            acc3 *= corr;
            acc4 *= corr;
            const int base = tile * ATT_TILE;
            const int last = min(qpos, base + ATT_TILE - 1) - base;
            const bool second = tid + ATT_TILE < v_dim, third = tid + 2 * ATT_TILE < v_dim, fourth = tid + 3 * ATT_TILE < v_dim;
            if (VEC && page_size % 8 == 0) {
                // eight neighbouring keys of a channel lie side by side in a value page: one 16-byte load (two in
                // float32) instead of eight elements; a key that is not seen has the weight 0
                for (int j0 = 0; j0 <= last; j0 += 8) {
                    const int a = base + j0, b = min(a + 7, qpos);
                    if (b < lo && a >= kept) continue;                         // none of the eight is seen
                    const TC* vp = v_pages + ((long)table[a / page_size] * kv_heads + kvh) * page_size * (long)v_dim +
                                   a % page_size + (long)tid * page_size;
                    float vv[8];
                    Vec<TC>::load(vp, vv);
                    if (Vec<TC>::N == 4) Vec<TC>::load(vp + 4, vv + 4);
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc += ps[j0 + e] * vv[e];
                    if (second) {
                        Vec<TC>::load(vp + (long)ATT_TILE * page_size, vv);
                        if (Vec<TC>::N == 4) Vec<TC>::load(vp + (long)ATT_TILE * page_size + 4, vv + 4);
#pragma unroll
                        for (int e = 0; e < 8; ++e) acc2 += ps[j0 + e] * vv[e];
                    }
                    if (third) {
                        Vec<TC>::load(vp + 2L * ATT_TILE * page_size, vv);
                        if (Vec<TC>::N == 4) Vec<TC>::load(vp + 2L * ATT_TILE * page_size + 4, vv + 4);
#pragma unroll
                        for (int e = 0; e < 8; ++e) acc3 += ps[j0 + e] * vv[e];
                    }
                    if (fourth) {
                        Vec<TC>::load(vp + 3L * ATT_TILE * page_size, vv);
                        if (Vec<TC>::N == 4) Vec<TC>::load(vp + 3L * ATT_TILE * page_size + 4, vv + 4);
#pragma unroll
                        for (int e = 0; e < 8; ++e) acc4 += ps[j0 + e] * vv[e];
                    }
                }
            } else
            for (int jj = 0; jj <= last; ++jj) {
                if (base + jj < lo && base + jj >= kept) continue;         // not seen: no weight, and no offset either
                acc += ps[jj] * to_f32(v_pages[rowoff[jj] + (long)tid * page_size]);
                if (second) acc2 += ps[jj] * to_f32(v_pages[rowoff[jj] + (long)(tid + ATT_TILE) * page_size]);
                if (third) acc3 += ps[jj] * to_f32(v_pages[rowoff[jj] + (long)(tid + 2 * ATT_TILE) * page_size]);
                if (fourth) acc4 += ps[jj] * to_f32(v_pages[rowoff[jj] + (long)(tid + 3 * ATT_TILE) * page_size]);
            }
        }
        __syncthreads();                                   // before the next tile overwrites ps and rowoff
    }
    if (sinks) l += expf(sinks[h] - m);                    // the sink: a term of the denominator alone
    if (tid < v_dim) from_f32(out + ((size_t)t * heads + h) * v_dim + tid, acc / l);
    if (tid + ATT_TILE < v_dim) from_f32(out + ((size_t)t * heads + h) * v_dim + tid + ATT_TILE, acc2 / l);
    if (tid + 2 * ATT_TILE < v_dim) from_f32(out + ((size_t)t * heads + h) * v_dim + tid + 2 * ATT_TILE, acc3 / l);
    if (tid + 3 * ATT_TILE < v_dim) from_f32(out + ((size_t)t * heads + h) * v_dim + tid + 3 * ATT_TILE, acc4 / l);
}

// The same for runs of tokens: a workgroup takes up to `per` neighbouring tokens (of one sequence, where cu_seqlens says which are)
// and the query heads of one kv head, up to 16 rows of queries that share every key and value it loads; every row's sums are the other kernel's, addition by addition, so that a
// token's result is the same bits in either.  What bounds the kernel above is that a key row is loaded again for every
// token and head; here sixteen rows share a load, and what is left is the loads' spread (a lane a key row, a lane a value
// channel: 64 cache lines a load).  759 tokens of three sequences, 16 heads over 8 of 128, float32: 222 us a layer with the
// kernel above, 133 with this one, 94 with the longest walks first (before such heads went to the matrix cores, below).
// head_dim and the value rows in 16-byte pieces, v_dim <= 512 / SHARES: the rows' weighted sums go to SHARES groups of threads,
// two channels a thread, so that a weight read from LDS serves two of them; a query read from LDS serves two keys likewise.
#define ATT_ROWS 16
template <typename T, int SHARES>
__global__ void __launch_bounds__(ATT_TILE)
attention_rows_kernel(T* __restrict__ out, const T* __restrict__ q, int q_stride, const T* __restrict__ k_pages,
                      const T* __restrict__ v_pages, const int32_t* __restrict__ tok_pos,
                      const int32_t* __restrict__ tok_seq, const int32_t* __restrict__ page_table, int table_width, int tokens,
                      int per, int heads, int kv_heads, int head_dim, int v_dim, int page_size, Reach reach, float scale,
                      float softcap, const float* __restrict__ slopes, int keep_first, const float* __restrict__ sinks,
                      const int32_t* __restrict__ cu_seqlens, int seqs, int rows_from) {
    constexpr int MINE = ATT_ROWS / SHARES;                 // rows whose weighted sums a thread holds
    extern __shared__ float4 qs4[];                         // ATT_ROWS rows of head_dim floats: the queries
    float* qs = reinterpret_cast<float*>(qs4);
    __shared__ float4 ps4[ATT_ROWS][ATT_TILE / 4];          // this tile's weights
    __shared__ float part[2][ATT_ROWS][ATT_TILE / RI_WAVE];
    __shared__ float state[3][ATT_ROWS];                    // every row's running maximum, sum and this tile's factor
    const int tid = threadIdx.x, lane = tid & (RI_WAVE - 1), wave = tid / RI_WAVE;
    // The last tokens first, a run's key heads side by side: a workgroup walks 256 keys in some 36 us whatever it does with them, the machine
    // holds two a compute unit, and a run of two tiles that goes out last is waited for alone.  Three prompts of 130 to 378 tokens, 16
    // heads over 8 of 128: 146 us in the order of the tokens, 94 so; 300 / 200 / 250 130 : 88, one of 2,000 1,095 : 904, 16 of 200 278 : 260.
    const int place = blockIdx.x + gridDim.x * blockIdx.y, at_run = gridDim.x - 1 - place / kv_heads;
    const int kvh = place % kv_heads, group = heads / kv_heads, h0 = kvh * group;
    int begin = at_run * per, end = min(begin + per, tokens);
    if (cu_seqlens) {
        Run run;
        if (!run_of(at_run, cu_seqlens, seqs, rows_from, per, 1, run)) return;
        begin = run.start + run.first;
        end = begin + run.count;
    }
    const int share = tid / (ATT_TILE / SHARES), d = tid % (ATT_TILE / SHARES);
    const int row0 = (wave >> 1) * (ATT_ROWS / 2), at = tid & 127;               // scores: half of the rows, two keys of a tile
    // the tokens of one sequence at a time, as far as their positions follow one another
    for (int t0 = begin, t1; t0 < end; t0 = t1) {
        const int seq = tok_seq[t0], p0 = tok_pos[t0];
        for (t1 = t0 + 1; t1 < end && tok_seq[t1] == seq && tok_pos[t1] == p0 + (t1 - t0);) ++t1;
        const int rows = (t1 - t0) * group, last_pos = p0 + (t1 - 1 - t0);       // row r: token t0 + r / group, head h0 + r % group
        const int32_t* table = page_table + (size_t)seq * table_width;
        __syncthreads();
        for (int e = tid; e < ATT_ROWS * head_dim; e += ATT_TILE) {
            const int r = e / head_dim, c = e % head_dim;
            qs[e] = r < rows ? to_f32(q[(size_t)(t0 + r / group) * q_stride + (size_t)(h0 + r % group) * head_dim + c]) : 0.f;
        }
        if (tid < ATT_ROWS) { state[0][tid] = -INFINITY; state[1][tid] = 0.f; }
        __syncthreads();
        float acc[2][MINE] = {};                            // channels d and d + ATT_TILE / SHARES
        const int lo_first = reach.first(p0), lo_tile = lo_first / ATT_TILE;       // the first token sees the furthest back
        // A key that no row sees is not looked up: behind a window or chunk its page has been given back, and the table holds -1.
        // What the rows see between them: the keys before `kept` (the last row's, whose window ends furthest on) and those
        // from lo_first on.  (The rest of their pages is there: a page is given back once no later query sees any key of it.)
        const int kept = min(keep_first, reach.first(last_pos)), kept_tiles = (kept + ATT_TILE - 1) / ATT_TILE;
        for (int tile = 0; tile <= last_pos / ATT_TILE; ++tile) {
            if (tile >= kept_tiles && tile < lo_tile) { tile = lo_tile - 1; continue; }
            const int base = tile * ATT_TILE;
            float dot[2][ATT_ROWS / 2] = {};                // keys base + at and base + at + 128 with rows row0 ..+ 8
            const T* kr[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                int j = base + at + 128 * u;
                if (j > last_pos || (j < lo_first && j >= kept)) j = last_pos;     // (read as the last and not seen)
                kr[u] = k_pages + (((long)table[j / page_size] * kv_heads + kvh) * page_size + j % page_size) * (long)head_dim;
            }
            for (int c = 0; c < head_dim; c += Vec<T>::N) {
                float kv[2][Vec<T>::N];
                Vec<T>::load(kr[0] + c, kv[0]);
                Vec<T>::load(kr[1] + c, kv[1]);
#pragma unroll
                for (int i = 0; i < ATT_ROWS / 2; ++i)
#pragma unroll
                    for (int e = 0; e < Vec<T>::N; e += 4) {
                        const float4 qv = qs4[((row0 + i) * head_dim + c + e) / 4];
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            dot[u][i] += qv.x * kv[u][e]; dot[u][i] += qv.y * kv[u][e + 1];
                            dot[u][i] += qv.z * kv[u][e + 2]; dot[u][i] += qv.w * kv[u][e + 3];
                        }
                    }
            }
            uint32_t seen = 0;                               // bit 8 u + i: row row0 + i sees key u of this thread
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int i = 0; i < ATT_ROWS / 2; ++i) {
                    const int j = base + at + 128 * u, r = row0 + i, qpos = p0 + r / group, lo = reach.first(qpos);
                    const bool valid = r < rows && (j >= lo || j < min(keep_first, lo)) && j <= qpos;
                    float s = -INFINITY;
                    if (valid) {
                        s = dot[u][i] * scale;
                        if (softcap > 0.f) s = softcap * tanhf(s / softcap);
                        if (slopes) s -= slopes[h0 + r % group] * (float)(qpos - j);
                        seen |= 1u << (8 * u + i);
                    }
                    dot[u][i] = s;
                    const float top = wave_max(s);
                    if (lane == 0) part[0][r][(wave & 1) + 2 * u] = top;
                }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < ATT_ROWS / 2; ++i) {
                const int r = row0 + i;
                float m_new = state[0][r];
#pragma unroll
                for (int w = 0; w < ATT_TILE / RI_WAVE; ++w) m_new = fmaxf(m_new, part[0][r][w]);
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const float p = (seen >> (8 * u + i)) & 1 ? expf(dot[u][i] - m_new) : 0.f;
                    reinterpret_cast<float*>(ps4[r])[at + 128 * u] = p;
                    const float sum = wave_sum(p);
                    if (lane == 0) part[1][r][(wave & 1) + 2 * u] = sum;
                }
            }
            __syncthreads();
            if (tid < ATT_ROWS) {
                const float m = state[0][tid];
                float m_new = m, sum = 0.f;
#pragma unroll
                for (int w = 0; w < ATT_TILE / RI_WAVE; ++w) {
                    m_new = fmaxf(m_new, part[0][tid][w]);
                    sum += part[1][tid][w];
                }
                const float corr = m_new > -INFINITY ? expf(m - m_new) : 1.f;      // (a row that has seen no key yet stays as it is)
                state[1][tid] = state[1][tid] * corr + sum;
                state[0][tid] = m_new;
                state[2][tid] = corr;
            }
            __syncthreads();
            if (d < v_dim) {
                const bool two = d + ATT_TILE / SHARES < v_dim;
#pragma unroll
                for (int i = 0; i < MINE; ++i) {
                    acc[0][i] *= state[2][share * MINE + i];
                    acc[1][i] *= state[2][share * MINE + i];
                }
                const int last = min(last_pos, base + ATT_TILE - 1) - base;
                for (int j0 = 0; j0 <= last; j0 += 8) {
                    const int a = base + j0;
                    if (a + 7 < lo_first && a >= kept) continue;                   // (the same for the whole workgroup)
                    float vv[2][8];
                    const T* vp = v_pages + ((long)table[a / page_size] * kv_heads + kvh) * page_size * (long)v_dim + a % page_size +
                                  (long)d * page_size;
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        const T* vc = vp + (c && two ? (long)(ATT_TILE / SHARES) * page_size : 0);
                        Vec<T>::load(vc, vv[c]);
                        if (Vec<T>::N == 4) Vec<T>::load(vc + 4, vv[c] + 4);
                    }
#pragma unroll
                    for (int i = 0; i < MINE; ++i) {
                        // (the same for the whole share: none of the eight is seen by this row)
                        const int r = share * MINE + i, qpos = p0 + r / group, b = min(a + 7, qpos);
                        const int lo = reach.first(qpos);
                        if (r >= rows || a > qpos || (b < lo && a >= min(keep_first, lo))) continue;
                        const float4 pa = ps4[r][j0 / 4], pb = ps4[r][j0 / 4 + 1];
                        const float w[8] = {pa.x, pa.y, pa.z, pa.w, pb.x, pb.y, pb.z, pb.w};
#pragma unroll
                        for (int c = 0; c < 2; ++c)
#pragma unroll
                            for (int e = 0; e < 8; ++e) acc[c][i] += w[e] * vv[c][e];
                    }
                }
            }
            __syncthreads();                                 // before the next tile overwrites the weights
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int ch = d + c * (ATT_TILE / SHARES);
            if (ch >= v_dim) continue;
#pragma unroll
            for (int i = 0; i < MINE; ++i) {
                const int r = share * MINE + i;
                if (r >= rows) continue;
                float l = state[1][r];
                if (sinks) l += expf(sinks[h0 + r % group] - state[0][r]);
                from_f32(out + ((size_t)(t0 + r / group) * heads + h0 + r % group) * v_dim + ch, acc[c][i] / l);
            }
        }
    }
}

// float32 heads of 64 and 128 run on the matrix cores' float32 products (16x16x4): every product and sum is a 32-bit one, the dot
// product of a query and a key in two chains of head_dim / 2 (by blocks of sixteen channels), added at the end.  A workgroup takes
// sixteen rows of queries (neighbouring tokens of one sequence times the query heads of one kv head); its four wavefronts take
// the tiles of sixteen keys in turn, tile t the wavefront t % 4, each with its own running maximum, sum and weighted values, joined
// in the wavefronts' order at the end: a row's result depends on its own position and the keys alone, never on the rows
// beside it.  The scores are computed with the keys as rows and the queries as columns: lane (g, r) then holds keys 4 g ..+4 of query r,
// which is what the second product reads from it as its operand, and both products read keys and values 16 bytes a lane
// straight from their pages, whole 64-byte pieces of a row: nothing passes through LDS but the join.
// What bounds it: the products, 2,048 cycles a tile of keys, and for short prompts the depth of the longest walk.  759 tokens of
// three prompts (of 33 to 400), 16 heads over 8 of 128: 31 us a layer, by rows on the vector units 91; one prompt of 2,000 248 : 906,
// 12 of 200 68 : 201, 64 single tokens at 500 keys 47 : 74, one at 2,000 60 : 105, one at 50 13 : 13 (heads of 64 alike).
// Error against 64 bits over a whole model's logits 1.0e-6 : 1.1e-6.
#define ATT_M_WAVES 4
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float att_floatx4;

template <int D>
__global__ void __launch_bounds__(64 * ATT_M_WAVES)
attention_f32_matrix_kernel(float* __restrict__ out, const float* __restrict__ q, int q_stride, const float* __restrict__ k_pages,
                            const float* __restrict__ v_pages, const int32_t* __restrict__ tok_pos,
                            const int32_t* __restrict__ tok_seq, const int32_t* __restrict__ page_table, int table_width, int tokens,
                            int per, int heads, int kv_heads, int page_size, Reach reach, float scale, float softcap,
                            const float* __restrict__ slopes, int keep_first, const float* __restrict__ sinks,
                            const int32_t* __restrict__ cu_seqlens, int seqs) {
    constexpr int BLOCKS = D / 16, PITCH = D + 4;
    __shared__ float sums[ATT_M_WAVES][ATT_ROWS][PITCH];
    __shared__ float tops[ATT_M_WAVES][ATT_ROWS], totals[ATT_M_WAVES][ATT_ROWS];
    const int tid = threadIdx.x, lane = tid & (RI_WAVE - 1), r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid / RI_WAVE);
    // the longest walks first, a run's key heads side by side (as in the kernel above)
    const int place = blockIdx.x + gridDim.x * blockIdx.y, at_run = gridDim.x - 1 - place / kv_heads;
    const int kvh = place % kv_heads, group = heads / kv_heads, h0 = kvh * group;
    int begin = at_run * per, end = min(begin + per, tokens);
    if (cu_seqlens) {
        Run run;
        if (!run_of(at_run, cu_seqlens, seqs, 1, per, 1, run)) return;
        begin = run.start + run.first;
        end = begin + run.count;
    }
    // the tokens of one sequence at a time, as far as their positions follow one another
    for (int t0 = begin, t1; t0 < end; t0 = t1) {
        const int seq = tok_seq[t0], p0 = tok_pos[t0];
        // (a lane a token: one after the other each would be a trip to memory)
        const int ahead = min(t0 + 1 + lane, tokens - 1);
        const bool follows = t0 + 1 + lane < end && tok_seq[ahead] == seq && tok_pos[ahead] == p0 + 1 + lane;
        t1 = t0 + 1 + __builtin_ctzll(~__ballot(follows));   // (a run is shorter than a wavefront)
        const int rows = (t1 - t0) * group, last_pos = p0 + (t1 - 1 - t0);       // row r: token t0 + r / group, head h0 + r % group
        const int32_t* table = page_table + (size_t)seq * table_width;
        const int mine = min(r, rows - 1), qpos = p0 + mine / group, head = h0 + mine % group;   // (rows past the last are it again)
        const int lo = reach.first(qpos), kept = min(keep_first, lo);
        const float slope = slopes ? slopes[head] : 0.f;
        att_floatx4 qf[BLOCKS], acc[BLOCKS];
        const float* qp = q + (size_t)(t0 + mine / group) * q_stride + (size_t)head * D + 4 * g;
#pragma unroll
        for (int b = 0; b < BLOCKS; ++b) {
            qf[b] = att_floatx4{qp[16 * b], qp[16 * b + 1], qp[16 * b + 2], qp[16 * b + 3]};
            acc[b] = att_floatx4{0.f, 0.f, 0.f, 0.f};
        }
        float m = -INFINITY, l = 0.f;                       // l: of this lane's keys
        // the tiles that any row sees: those of the kept keys, and from the first token's first key on
        const int first_tile = reach.first(p0) / 16, kept_tiles = (min(keep_first, reach.first(last_pos)) + 15) / 16;
        const auto seen_from = [&](int tile) {              // this wavefront's first such tile from `tile` on
            return tile >= kept_tiles && tile < first_tile ? tile + (first_tile - tile + ATT_M_WAVES - 1) / ATT_M_WAVES * ATT_M_WAVES : tile;
        };
        const auto page_of = [&](int tile) { return ((long)table[tile * 16 / page_size] * kv_heads + kvh) * page_size * D; };
        const auto fetch_keys = [&](att_floatx4 (&kf)[BLOCKS], long page, int tile) {
            const float* kp = k_pages + page + (long)(tile * 16 % page_size + r) * D + 4 * g;
#pragma unroll
            for (int b = 0; b < BLOCKS; ++b) kf[b] = *reinterpret_cast<const att_floatx4*>(kp + 16 * b);
        };
        const int last_tile = last_pos / 16;
        att_floatx4 kf[BLOCKS], vf[BLOCKS];
        long page = 0;
        int tile = seen_from(wave);
        if (tile <= last_tile) fetch_keys(kf, page = page_of(tile), tile);
        // a tile's values are asked for before its scores are computed, the next tile's keys before the values are used
        for (int next; tile <= last_tile; tile = next) {
            const int base = tile * 16;
            next = seen_from(tile + ATT_M_WAVES);
            const long next_page = page_of(min(next, last_tile));
            const float* vp = v_pages + page + (long)r * page_size + base % page_size + 4 * g;
#pragma unroll
            for (int b = 0; b < BLOCKS; ++b) vf[b] = *reinterpret_cast<const att_floatx4*>(vp + (long)(16 * b) * page_size);
            __builtin_amdgcn_sched_barrier(0);
            att_floatx4 dot[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int b = 0; b < BLOCKS; b += 2)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    dot[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[b][i], qf[b][i], dot[0], 0, 0, 0);
                    dot[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[b + 1][i], qf[b + 1][i], dot[1], 0, 0, 0);
                }
            __builtin_amdgcn_sched_barrier(0);
            fetch_keys(kf, page = next_page, min(next, last_tile));
            __builtin_amdgcn_sched_barrier(0);
            float s[4], top = -INFINITY;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int j = base + 4 * g + i;
                s[i] = (dot[0][i] + dot[1][i]) * scale;
                if (softcap > 0.f) s[i] = softcap * tanhf(s[i] / softcap);
                if (slopes) s[i] -= slope * (float)(qpos - j);
                if (!((j >= lo || j < kept) && j <= qpos)) s[i] = -INFINITY;
                top = fmaxf(top, s[i]);
            }
            top = fmaxf(top, __shfl_xor(top, 16, RI_WAVE));
            top = fmaxf(top, __shfl_xor(top, 32, RI_WAVE));
            const float m_new = fmaxf(m, top), ref = m_new > -INFINITY ? m_new : 0.f;   // (nothing seen yet: any number will do)
            const float corr = expf(m - ref);
            float p[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] = expf(s[i] - ref);
            l = l * corr + ((p[0] + p[1]) + (p[2] + p[3]));
            m = m_new;
            if (base + 15 > last_pos) {                     // keys that no row has yet: whatever their places hold does not count
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int b = 0; b < BLOCKS; ++b) vf[b][i] = base + 4 * g + i <= last_pos ? vf[b][i] : 0.f;
            }
#pragma unroll
            for (int b = 0; b < BLOCKS; ++b) acc[b] *= corr;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int b = 0; b < BLOCKS; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[b][i], p[i], acc[b], 0, 0, 0);
        }
        l += __shfl_xor(l, 16, RI_WAVE);
        l += __shfl_xor(l, 32, RI_WAVE);
        __syncthreads();                                    // the last run's sums have been read
#pragma unroll
        for (int b = 0; b < BLOCKS; ++b) *reinterpret_cast<att_floatx4*>(&sums[wave][r][16 * b + 4 * g]) = acc[b];
        if (g == 0) { tops[wave][r] = m; totals[wave][r] = l; }
        __syncthreads();
        const int row = tid / 16, h = h0 + row % group;
        if (row >= rows) continue;
        float all = tops[0][row], total = 0.f, part[ATT_M_WAVES];
#pragma unroll
        for (int w = 1; w < ATT_M_WAVES; ++w) all = fmaxf(all, tops[w][row]);
#pragma unroll
        for (int w = 0; w < ATT_M_WAVES; ++w) {
            part[w] = tops[w][row] > -INFINITY ? expf(tops[w][row] - all) : 0.f;
            total += totals[w][row] * part[w];
        }
        if (sinks) total += expf(sinks[h] - all);           // the sink: a term of the denominator alone
        float* o = out + ((size_t)(t0 + row / group) * heads + h) * D;
#pragma unroll
        for (int c = 4 * (tid % 16); c < D; c += 64) {
            att_floatx4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < ATT_M_WAVES; ++w) sum += *reinterpret_cast<const att_floatx4*>(&sums[w][row][c]) * part[w];
#pragma unroll
            for (int i = 0; i < 4; ++i) o[c + i] = sum[i] / total;
        }
    }
}

template <typename T, bool VEC>
static void launch_attention(void* out, const void* q, int q_stride, const void* k_pages, const void* v_pages,
                             const int32_t* tok_pos, const int32_t* tok_seq, const int32_t* page_table,
                             int table_width, int tokens, int heads, int kv_heads, int head_dim, int v_dim,
                             int page_size, Reach reach, float scale, float softcap, const float* slopes, int keep_first,
                             const float* sinks, const int32_t* cu_seqlens, int rows_from, hipStream_t s) {
    attention_generic_kernel<T, T, VEC><<<dim3(tokens, heads), ATT_TILE, (size_t)head_dim * sizeof(float), s>>>(
        (T*)out, (const T*)q, q_stride, (const T*)k_pages, (const T*)v_pages, tok_pos, tok_seq, page_table,
        table_width, heads, kv_heads, head_dim, v_dim, page_size, reach, scale, softcap, slopes, keep_first, sinks, cu_seqlens,
        rows_from);
}

template <typename T, int SHARES>
static void launch_rows(void* out, const void* q, int q_stride, const void* k_pages, const void* v_pages, const int32_t* tok_pos,
                        const int32_t* tok_seq, const int32_t* page_table, int table_width, int tokens, int heads, int kv_heads,
                        int head_dim, int v_dim, int page_size, Reach reach, float scale, float softcap, const float* slopes,
                        int keep_first, const float* sinks, const int32_t* cu_seqlens, int seqs, int rows_from, int runs, hipStream_t s) {
    const int per = ATT_ROWS / (heads / kv_heads);
    attention_rows_kernel<T, SHARES><<<dim3(cu_seqlens ? runs : (tokens + per - 1) / per, kv_heads), ATT_TILE, (size_t)ATT_ROWS * head_dim * sizeof(float), s>>>(
        (T*)out, (const T*)q, q_stride, (const T*)k_pages, (const T*)v_pages, tok_pos, tok_seq, page_table, table_width, tokens, per,
        heads, kv_heads, head_dim, v_dim, page_size, reach, scale, softcap, slopes, keep_first, sinks, cu_seqlens, seqs, rows_from);
}

// Whether a step's sizes can run by rows of queries.
static bool attention_rows_fit(int heads, int kv_heads, int head_dim, int v_dim, int page_size, int element) {
    return heads / kv_heads <= ATT_ROWS && head_dim % (16 / element) == 0 && head_dim <= 256 && v_dim <= ATT_TILE && page_size % 8 == 0;
}

// Whether a step's sizes run on the matrix cores: a rule on types and sizes alone, so that a sequence's tokens have the same bits
// however they are cut into steps.
static bool attention_matrix_fits(int dtype, int heads, int kv_heads, int head_dim, int v_dim, int page_size) {
    return dtype == RI_F32 && heads / kv_heads <= ATT_ROWS && (head_dim == 64 || head_dim == 128) && v_dim == head_dim && page_size % 16 == 0;
}

// Which of the two other forms a step runs (their results are the same bits): with cu_seqlens, the sequences of rows_from and more new
// tokens by rows, `runs` runs of 16 / (heads / kv_heads) tokens in all and rows_tokens tokens, and the rest a workgroup a
// (token, head), in a launch that the others' workgroups leave at once; without, all by rows where a sequence brings four
// tokens and more (most_new) and the (token, head) pairs are past one round of resident workgroups, eight a compute unit.
extern "C" int ri_attention_kept(void* out, const void* q, int act_dtype, int q_stride, const void* k_pages,
                            const void* v_pages, int cache_dtype, const int32_t* tok_pos, const int32_t* tok_seq,
                            const int32_t* page_table, int table_width, int tokens, int heads, int kv_heads,
                            int head_dim, int v_dim, int page_size, int window, int chunk, float scale, float softcap,
                            const float* slopes, int keep_first, const float* sinks, int most_new, const int32_t* cu_seqlens,
                            int seqs, int rows_from, int rows_tokens, int runs, void* stream) {
    RI_REQUIRE(chunk >= 0 && (chunk == 0 || window <= 0), "attention: chunks of %d beside a window of %d", chunk, window);
    const Reach reach = {window, chunk};
    RI_REQUIRE(keep_first >= 0, "attention: %d first tokens kept", keep_first);
    RI_REQUIRE(tokens > 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0,
               "attention: tokens %d, heads %d, kv heads %d", tokens, heads, kv_heads);
    RI_REQUIRE(head_dim >= 1 && head_dim <= ATT_MAX_HEAD_DIM, "attention: head_dim %d must be between 1 and %d", head_dim,
               ATT_MAX_HEAD_DIM);
    RI_REQUIRE(v_dim >= 1 && v_dim <= ATT_MAX_HEAD_DIM, "attention: value head size %d must be between 1 and %d", v_dim,
               ATT_MAX_HEAD_DIM);
    RI_REQUIRE(heads <= 65535, "attention: %d heads exceed one launch", heads);
    RI_REQUIRE(q_stride >= heads * head_dim, "attention: q row stride %d for %d heads of %d", q_stride, heads, head_dim);
    RI_REQUIRE(act_dtype == cache_dtype && (act_dtype == RI_F32 || act_dtype == RI_BF16),
               "attention: activations (%d) and cache (%d) must share float32 or bfloat16", act_dtype, cache_dtype);
    RI_REQUIRE(page_size > 0 && table_width > 0, "attention: page geometry");
    hipStream_t s = (hipStream_t)stream;
    // a key row starts on a 16-byte boundary when the head size is a multiple of 4 (float32) or 8 (bfloat16):
    // the pools themselves are 256-byte aligned allocations
    const bool vec = head_dim % (act_dtype == RI_F32 ? 4 : 8) == 0 && (uintptr_t)k_pages % 16 == 0 && (uintptr_t)v_pages % 16 == 0;
#define RI_ATT_GO(T, V) launch_attention<T, V>(out, q, q_stride, k_pages, v_pages, tok_pos, tok_seq, page_table, \
                                               table_width, tokens, heads, kv_heads, head_dim, v_dim, page_size, reach, scale, \
                                               softcap, slopes, window > 0 ? keep_first : 0, sinks, cu_seqlens, rows_from, s)
    const bool by_rows = vec && attention_rows_fit(heads, kv_heads, head_dim, v_dim, page_size, act_dtype == RI_F32 ? 4 : 2) &&
                         (cu_seqlens ? runs > 0 : most_new >= 4 && (long)tokens * heads > 8L * ri_compute_units());
    RI_REQUIRE(!cu_seqlens || (seqs > 0 && rows_from > 0 && rows_tokens >= 0 && rows_tokens <= tokens && (runs > 0) == (rows_tokens > 0)),
               "attention: %d runs of %d tokens of %d sequences", runs, rows_tokens, seqs);
    if (vec && attention_matrix_fits(act_dtype, heads, kv_heads, head_dim, v_dim, page_size)) {
        // runs of neighbours of one sequence where all of them are known, else tokens as they lie, one by one where no sequence
        // is said to bring several
        const bool known = cu_seqlens && runs > 0 && rows_from == 1 && rows_tokens == tokens;
        const int per = known || cu_seqlens || most_new >= 4 ? ATT_ROWS / (heads / kv_heads) : 1;
        const dim3 matrix_grid(known ? runs : (tokens + per - 1) / per, kv_heads);
#define RI_ATT_MATRIX(D) attention_f32_matrix_kernel<D><<<matrix_grid, 64 * ATT_M_WAVES, 0, s>>>( \
            (float*)out, (const float*)q, q_stride, (const float*)k_pages, (const float*)v_pages, tok_pos, tok_seq, page_table, table_width, tokens, \
            per, heads, kv_heads, page_size, reach, scale, softcap, slopes, window > 0 ? keep_first : 0, sinks, known ? cu_seqlens : nullptr, seqs)
        if (head_dim == 64) RI_ATT_MATRIX(64); else RI_ATT_MATRIX(128);
#undef RI_ATT_MATRIX
        RI_LAUNCH_CHECK("attention");
        return 0;
    }
    if (by_rows) {
#define RI_ATT_ROWS(T, S) launch_rows<T, S>(out, q, q_stride, k_pages, v_pages, tok_pos, tok_seq, page_table, table_width, tokens, heads, \
                                            kv_heads, head_dim, v_dim, page_size, reach, scale, softcap, slopes, \
                                            window > 0 ? keep_first : 0, sinks, cu_seqlens, seqs, rows_from, runs, s)
        if (act_dtype == RI_F32) { if (v_dim <= 128) RI_ATT_ROWS(float, 4); else RI_ATT_ROWS(float, 2); }
        else                     { if (v_dim <= 128) RI_ATT_ROWS(bf16_t, 4); else RI_ATT_ROWS(bf16_t, 2); }
#undef RI_ATT_ROWS
    }
    if (!by_rows) cu_seqlens = nullptr;
    if (by_rows && !(cu_seqlens && rows_tokens < tokens)) {
        // (no token is left for the other form)
    } else if (act_dtype == RI_F32) { if (vec) RI_ATT_GO(float, true); else RI_ATT_GO(float, false); }
    else                     { if (vec) RI_ATT_GO(bf16_t, true); else RI_ATT_GO(bf16_t, false); }
#undef RI_ATT_GO
    RI_LAUNCH_CHECK("attention");
    return 0;
}

extern "C" int ri_attention(void* out, const void* q, int act_dtype, int q_stride, const void* k_pages,
                            const void* v_pages, int cache_dtype, const int32_t* tok_pos, const int32_t* tok_seq,
                            const int32_t* page_table, int table_width, int tokens, int heads, int kv_heads,
                            int head_dim, int v_dim, int page_size, int window, float scale, float softcap,
                            const float* slopes, void* stream) {
    return ri_attention_kept(out, q, act_dtype, q_stride, k_pages, v_pages, cache_dtype, tok_pos, tok_seq, page_table,
                             table_width, tokens, heads, kv_heads, head_dim, v_dim, page_size, window, 0, scale, softcap,
                             slopes, 0, nullptr, 1, nullptr, 0, 0, 0, 0, stream);
}
