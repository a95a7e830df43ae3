// What the recurrences that walk a prompt's tokens over a float32 state have in common (ssd.hip, timemix.hip, gla.hip), for
// states of 65 to 128 rows: a lane holds a tile of four rows by CPL columns, the 32 lanes of half a wavefront all rows of its
// columns, a workgroup of four wavefronts 8 CPL neighbouring columns.  Tokens are staged in LDS in blocks of eight, the next
// block's loads on their way while a block is computed.  What bounds a walk is its chain of tokens, so a token must cost
// a wavefront little: a row's inputs are read from LDS once for CPL columns (a lane that holds 16 rows of one column
// reads four times as much, and the LDS of a compute unit was what those walks waited for), and the sums over the rows
// meet for eight tokens at once, two sums in one exchange and the rest by lane shifts that ride in the additions.  Now vector
// instructions are issued 71 to 77% of the time where a launch fills the machine, and the LDS is busy 19 to 44%.  A block's
// missing tokens are staged so that they change nothing: no branch stands between the tokens.
// The order of every sum is fixed by the lanes' places, not by CPL: CPL is chosen by how many columns a launch has.
// States of up to 64 rows keep the forms of their own in ssd.hip, timemix.hip and gla.hip: half of the lanes here would hold no row.  Their
// single tokens and steps that fill the machine are faster so, their few long prompts would not be (32 heads of 64 x 64, us own form : this
// one, state-space / time mixing / gated linear attention: 32 single tokens 11 : 17, 17 : 22, 36 : 20; 32 prompts of 256 194 : 257, 361 : 350,
// 486 : 271; one of 2,048 911 : 241, 863 : 229, 455 : 231).
#pragma once
#include "common.h"

#define WALK_ROWS 128
#define WALK_BLOCK 8

// Columns a lane holds: as few as keep the wavefronts within eight a compute unit, two a SIMD (one hides the other's waits),
// at most four (less to read per column where the machine is full).  A step of single tokens moves the state and little else:
// four columns, 16 bytes of a row a lane.
static inline int walk_columns(long columns, bool single_tokens) {
    if (single_tokens) return 4;
    const long waves = 8L * ri_compute_units();
    return columns / 2 <= waves ? 1 : columns / 4 <= waves ? 2 : 4;
}

// Four neighbouring rows from `row` on of n; VEC: n and every row's address are multiples of four elements.  Loads are issued
// whatever the indices are; rows beyond n are zeros.
template <bool VEC>
__device__ __forceinline__ float4 walk_rows(const float* __restrict__ p, int row, int n) {
    if (VEC) return *reinterpret_cast<const float4*>(p + min(row, n - 4));
    return make_float4(p[min(row, n - 1)], p[min(row + 1, n - 1)], p[min(row + 2, n - 1)], p[min(row + 3, n - 1)]);
}
template <bool VEC>
__device__ __forceinline__ float4 walk_rows(const bf16_t* __restrict__ p, int row, int n) {
    if (VEC) {
        const uint2 w = *reinterpret_cast<const uint2*>(p + min(row, n - 4));
        return make_float4(__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xFFFF0000u), __uint_as_float(w.y << 16),
                           __uint_as_float(w.y & 0xFFFF0000u));
    }
    return make_float4(bf16_to_f32(p[min(row, n - 1)]), bf16_to_f32(p[min(row + 1, n - 1)]), bf16_to_f32(p[min(row + 2, n - 1)]),
                       bf16_to_f32(p[min(row + 3, n - 1)]));
}
// The rows that are there, and `fill` in the others' place (in all of them where the token is not there).
__device__ __forceinline__ float4 walk_keep(const float4 v, int row, int n, bool token, float fill) {
    return make_float4(token && row < n ? v.x : fill, token && row + 1 < n ? v.y : fill, token && row + 2 < n ? v.z : fill,
                       token && row + 3 < n ? v.w : fill);
}

// A lane's tile of the state, and back: 16 bytes of a row at a time where the state starts on the boundary of such loads.
template <int CPL>
__device__ __forceinline__ void walk_load(float (&st)[4][CPL], const float* sp, int row0, int n, int c0, int vdim) {
    if (CPL == 4 && vdim % 4 == 0 && (uintptr_t)sp % 16 == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 v = *reinterpret_cast<const float4*>(sp + (size_t)min(row0 + i, n - 1) * vdim + min(c0, vdim - 4));
            const bool in = row0 + i < n && c0 < vdim;
            st[i][0] = in ? v.x : 0.f; st[i][CPL > 1 ? 1 : 0] = in ? v.y : 0.f;
            st[i][CPL > 2 ? 2 : 0] = in ? v.z : 0.f; st[i][CPL > 3 ? 3 : 0] = in ? v.w : 0.f;
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
            const float v = sp[(size_t)min(row0 + i, n - 1) * vdim + min(c0 + j, vdim - 1)];
            st[i][j] = row0 + i < n && c0 + j < vdim ? v : 0.f;
        }
}
template <int CPL>
__device__ __forceinline__ void walk_store(const float (&st)[4][CPL], float* sp, int row0, int n, int c0, int vdim) {
    const bool four = CPL == 4 && vdim % 4 == 0 && (uintptr_t)sp % 16 == 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (row0 + i >= n) continue;
        float* to = sp + (size_t)(row0 + i) * vdim + c0;
        if (four) {
            if (c0 < vdim)
                *reinterpret_cast<float4*>(to) = make_float4(st[i][0], st[i][CPL > 1 ? 1 : 0], st[i][CPL > 2 ? 2 : 0], st[i][CPL > 3 ? 3 : 0]);
        } else {
#pragma unroll
            for (int j = 0; j < CPL; ++j)
                if (c0 + j < vdim) to[j] = st[i][j];
        }
    }
}

// The value of lane `lane ^ (1, 2)` of every four, or the mirror image inside every eight or sixteen lanes.
template <int CONTROL>
__device__ __forceinline__ float walk_shift(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CONTROL, 0xF, 0xF, true));
}

// part[tt * CPL + j]: the lane's share of token tt's sum in its column j.  Returns the whole sum of one of them, number
// walk_mine<CPL>(lane), where that is below WALK_BLOCK * CPL.
template <int CPL>
__device__ __forceinline__ int walk_mine(int lane) { return 2 * (lane & 15) + ((lane >> 4) & 1); }
template <int CPL>
__device__ __forceinline__ float walk_sum(const float (&part)[WALK_BLOCK * CPL], int lane) {
    float mine = 0.f;
#pragma unroll
    for (int i = 0; i < WALK_BLOCK * CPL / 2; ++i) {
        // even rows of 16 lanes go on with the first of two sums, odd rows with the second
        const auto both = __builtin_amdgcn_permlane16_swap(__float_as_uint(part[2 * i]), __float_as_uint(part[2 * i + 1]), false, false);
        float s = __uint_as_float(both[0]) + __uint_as_float(both[1]);
        s += walk_shift<0xB1>(s);
        s += walk_shift<0x4E>(s);
        s += walk_shift<0x141>(s);
        s += walk_shift<0x140>(s);
        mine = (lane & 15) == i ? s : mine;
    }
    return mine;
}
