// What the kernels that make queries, keys and values ready for the cache share: eight neighbours at once, and a
// prompt's values into their pages, eight positions or a page at a time.
#pragma once
#include "common.h"

template <typename T> struct Eight;
template <> struct Eight<float> {
    __device__ static void load(const float* p, float* o) {
        const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
        o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w; o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
    }
    __device__ static void store(float* p, const float* v) {
        *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
    }
};
template <> struct Eight<bf16_t> {
    __device__ static void load(const bf16_t* p, float* o) {
        const uint4 v = *reinterpret_cast<const uint4*>(p);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o[2 * i] = __uint_as_float(w[i] << 16);
            o[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
        }
    }
    __device__ static void store(bf16_t* p, const float* v) {
        *reinterpret_cast<uint4*>(p) = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]),
                                                  pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
    }
};

// Values into their pages, turned in registers: a thread takes 16 bytes of channels of eight neighbouring positions (those that
// start at a multiple of eight), eight loads all asked for together, and writes channel rows of eight positions, 16 bytes each
// (two in float32); neighbouring threads take the four such groups of 32 positions, so that a store covers whole lines.  What bounded
// the form through LDS below is the wait for its loads, a barrier and its few workgroups at work (three prompts of 500 to 1,500 tokens,
// 8 heads of 128, bfloat16: 13.8 us, 9.1 so).  A workgroup of 256 threads is number `part` of the values_turn_parts of one sequence's
// `piece`-th 32 positions that this step may touch.
#define QT_TOKENS 32
template <typename T>
static inline int values_turn_parts(int kv_heads, int vdim) { return (kv_heads * (vdim / (16 / (int)sizeof(T))) * 4 + 255) / 256; }
static inline int values_turn_pieces(int max_new) { return (max_new + QT_TOKENS - 2) / QT_TOKENS + 1; }

template <typename T>
__device__ __forceinline__ void values_turn(const T* __restrict__ rows, size_t row_len, size_t v_off, const int32_t* __restrict__ cu_seqlens,
                                            const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ page_table, int table_width,
                                            T* __restrict__ v_pages, int kv_heads, int vdim, int page_size,
                                            const float* __restrict__ bias, int piece, int seq, int part) {
    constexpr int E = 16 / (int)sizeof(T);                   // channels a thread takes
    const int t_begin = cu_seqlens[seq], n = cu_seqlens[seq + 1] - t_begin;
    if (n <= 0) return;
    const int start = tok_pos[t_begin];                      // the sequence's new tokens sit at start .. start + n - 1
    const int item = part * 256 + threadIdx.x, of_head = vdim / E, rest = item >> 2, kvh = rest / of_head, d = rest % of_head * E;
    const int first = (start / QT_TOKENS + piece) * QT_TOKENS + (item & 3) * 8;
    if (kvh >= kv_heads || first + 7 < start || first >= start + n) return;
    const T* from = rows + v_off + (size_t)kvh * vdim + d;
    uint4 in[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)                              // (positions that are not the step's: read as its first or last, not written)
        in[j] = *reinterpret_cast<const uint4*>(from + (size_t)(t_begin + min(max(first + j - start, 0), n - 1)) * row_len);
    const bool whole = first >= start && first + 8 <= start + n;
    const int page = page_table[(size_t)seq * table_width + first / page_size];
    T* to = v_pages + (((size_t)page * kv_heads + kvh) * vdim + d) * page_size + first % page_size;
#pragma unroll
    for (int c = 0; c < E; ++c, to += page_size) {
        T y[8];
        const float b = bias ? bias[(size_t)kvh * vdim + d + c] : 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t w[4] = {in[j].x, in[j].y, in[j].z, in[j].w};
            if constexpr (sizeof(T) == 4) y[j] = __uint_as_float(w[c]) + (bias ? b : 0.f);
            else {
                y[j] = (T)(w[c / 2] >> (c & 1) * 16);
                if (bias) from_f32(&y[j], to_f32(y[j]) + b);
            }
        }
        if (whole) {
            if constexpr (sizeof(T) == 4) Eight<T>::store(to, y);
            else
                *reinterpret_cast<uint4*>(to) = make_uint4(y[0] | (uint32_t)y[1] << 16, y[2] | (uint32_t)y[3] << 16, y[4] | (uint32_t)y[5] << 16,
                                                           y[6] | (uint32_t)y[7] << 16);
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (first + j >= start && first + j < start + n) to[j] = y[j];
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(256)
values_turn_kernel(const T* __restrict__ rows, size_t row_len, size_t v_off, const int32_t* __restrict__ cu_seqlens,
                   const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ page_table, int table_width,
                   T* __restrict__ v_pages, int kv_heads, int vdim, int page_size, const float* __restrict__ bias) {
    values_turn<T>(rows, row_len, v_off, cu_seqlens, tok_pos, page_table, table_width, v_pages, kv_heads, vdim, page_size, bias, blockIdx.x,
                   blockIdx.y, blockIdx.z);
}

// Through LDS, where 16-byte pieces do not divide the value heads or their rows, a page at a time: one workgroup per (32 positions touched by this step, sequence, kv
// head) reads the new tokens' value heads as rows, turns them through LDS and writes channel rows.
template <typename TA, typename TC>
__global__ void __launch_bounds__(256)
values_to_pages_kernel(const TA* __restrict__ qkv, size_t row_len, size_t v_off, const int32_t* __restrict__ cu_seqlens,
                       const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ page_table, int table_width,
                       TC* __restrict__ v_pages, int kv_heads, int vdim, int page_size, const float* __restrict__ bias) {
    extern __shared__ float tile[];                          // [QT_TOKENS][vdim + 1]
    const int b = blockIdx.y, kvh = blockIdx.z;
    const int t_begin = cu_seqlens[b], n = cu_seqlens[b + 1] - t_begin;
    if (n <= 0) return;
    const int start = tok_pos[t_begin];                      // the sequence's new tokens sit at start .. start + n - 1
    const int first = (start / QT_TOKENS + blockIdx.x) * QT_TOKENS;
    const int lo = max(first, start), hi = min(first + QT_TOKENS - 1, start + n - 1);
    if (lo > hi) return;
    const int stride = vdim + 1;
    const TA* from = qkv + v_off + (size_t)kvh * vdim;
    const float* add = bias ? bias + (size_t)kvh * vdim : nullptr;
    const bool whole = lo == first && hi == first + QT_TOKENS - 1;
    if (sizeof(TA) == 2 && whole && vdim % 8 == 0 && (row_len % 8) == 0 && (v_off % 8) == 0) {
        const int pieces = vdim / 8;
        for (int e = threadIdx.x; e < QT_TOKENS * pieces; e += blockDim.x) {
            const int tt = e / pieces, d = (e - tt * pieces) * 8;
            float v[8];
            Eight<TA>::load(from + (size_t)(t_begin + first - start + tt) * row_len + d, v);
#pragma unroll
            for (int j = 0; j < 8; ++j) tile[tt * stride + d + j] = v[j];
        }
    } else {
        for (int e = threadIdx.x; e < (hi - lo + 1) * vdim; e += blockDim.x) {
            const int tt = e / vdim, d = e - tt * vdim;
            tile[(lo - first + tt) * stride + d] = to_f32(from[(size_t)(t_begin + lo - start + tt) * row_len + d]);
        }
    }
    __syncthreads();
    const int page = page_table[(size_t)b * table_width + first / page_size];
    TC* base = v_pages + ((size_t)page * kv_heads + kvh) * page_size * vdim + first % page_size;
    if (whole && page_size % 8 == 0) {
        for (int e = threadIdx.x; e < vdim * (QT_TOKENS / 8); e += blockDim.x) {
            const int d = e / (QT_TOKENS / 8), t8 = (e - d * (QT_TOKENS / 8)) * 8;
            const float b = add ? add[d] : 0.f;
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = tile[(t8 + j) * stride + d] + b;
            Eight<TC>::store(base + (size_t)d * page_size + t8, v);
        }
    } else {
        for (int e = threadIdx.x; e < vdim * QT_TOKENS; e += blockDim.x) {
            const int d = e / QT_TOKENS, tt = e - d * QT_TOKENS;
            if (first + tt >= lo && first + tt <= hi) from_f32(base + (size_t)d * page_size + tt, tile[tt * stride + d] + (add ? add[d] : 0.f));
        }
    }
}

// A prompt's values into their pages (which hold a multiple of 32 positions).
template <typename T>
static void launch_values_to_pages(const T* rows, size_t row_len, size_t v_off, const int32_t* cu_seqlens, const int32_t* tok_pos,
                                   const int32_t* page_table, int table_width, T* v_pages, int seqs, int max_new, int kv_heads, int vdim,
                                   int page_size, const float* bias, hipStream_t s) {
    constexpr int E = 16 / (int)sizeof(T);
    const int parts = vdim % E == 0 ? values_turn_parts<T>(kv_heads, vdim) : 0;
    if (parts > 0 && parts <= 65535 && row_len % E == 0 && v_off % E == 0 && ((uintptr_t)rows | (uintptr_t)v_pages) % 16 == 0)
        values_turn_kernel<T><<<dim3(values_turn_pieces(max_new), seqs, parts), 256, 0, s>>>(
            rows, row_len, v_off, cu_seqlens, tok_pos, page_table, table_width, v_pages, kv_heads, vdim, page_size, bias);
    else
        values_to_pages_kernel<T, T><<<dim3(values_turn_pieces(max_new), seqs, kv_heads), 256, QT_TOKENS * (vdim + 1) * sizeof(float), s>>>(
            rows, row_len, v_off, cu_seqlens, tok_pos, page_table, table_width, v_pages, kv_heads, vdim, page_size, bias);
}
