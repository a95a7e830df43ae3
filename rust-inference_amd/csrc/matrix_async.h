// Pieces of matrix kernels whose instructions are put in order by hand: copies from memory straight into LDS, matrix products that add in
// place, and waits that count the copies in flight.  The compiler waits for every copy under way before it reads LDS at all, and moves sums
// of this size between register files; in a loop that keeps two stages in flight neither can be left to it.
#pragma once
#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 ma_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float ma_floatx4;

#ifdef RI_EMULATED
typedef char* ma_lds_t;
__device__ __forceinline__ ma_lds_t ma_lds(void* p) { return (char*)p; }
__device__ __forceinline__ void ma_copy16(ma_lds_t at, uint32_t off, const void* base) {
    memcpy(at + 16 * (threadIdx.x & 63), (const char*)base + off, 16);
}
__device__ __forceinline__ void ma_product(ma_floatx4& c, const ma_bf16x8 a, const ma_bf16x8 b) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ void ma_product_first(ma_floatx4& c, const ma_bf16x8 a, const ma_bf16x8 b) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, (ma_floatx4{0.f, 0.f, 0.f, 0.f}), 0, 0, 0);
}
__device__ __forceinline__ float ma_taken(const float& a) { return a; }
template <int N> __device__ __forceinline__ void ma_wait_copies() {}
__device__ __forceinline__ void ma_wait_lds() {}
__device__ __forceinline__ void ma_wait_products() {}
__device__ __forceinline__ void ma_wait_written() {}
__device__ __forceinline__ void ma_meet() { __syncthreads(); }
#else
typedef uint32_t ma_lds_t;                                    // an address within a workgroup's LDS
__device__ __forceinline__ ma_lds_t ma_lds(void* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)p; }
// Sixteen bytes a lane from base + off (off a lane's own) to LDS, lane l's at `at` + 16 l (`at` the wavefront's).
// (M0 holds the place; nothing else in these kernels uses that register, and the compiler, which sets it where it needs it, is told.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void ma_copy16(ma_lds_t at, uint32_t off, const void* base) {
    at = __builtin_amdgcn_readfirstlane(at);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(at), "v"(off), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop
// c += a . b (16 x 16 x 32), c in the accumulation registers; _first: c = a . b.
__device__ __forceinline__ void ma_product(ma_floatx4& c, const ma_bf16x8 a, const ma_bf16x8 b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void ma_product_first(ma_floatx4& c, const ma_bf16x8 a, const ma_bf16x8 b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
}
// An element of such a sum (after ma_wait_products).
__device__ __forceinline__ float ma_taken(const float& a) {
    float v;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
    return v;
}
// Until at most N of this wavefront's copies, loads and stores are under way; they end in the order in which they were issued.
template <int N> __device__ __forceinline__ void ma_wait_copies() {
    static_assert(N >= 0 && N <= 63, "the counter has six bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void ma_wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// Until the last product's sum may be read (more than the longest product takes).
__device__ __forceinline__ void ma_wait_products() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }
// Until a product may read what the vector instruction before has written (the compiler does not know these products for what they are).
__device__ __forceinline__ void ma_wait_written() { asm volatile("s_nop 3" ::: "memory"); }
// The workgroup's wavefronts meet; what each has to have waited for before, it has waited for itself.
__device__ __forceinline__ void ma_meet() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
#endif

// A value that the compiler is not to know anything about (the same for the whole wavefront).
__device__ __forceinline__ void ma_opaque(uint32_t& v) {
#ifndef RI_EMULATED
    asm volatile("" : "+s"(v));
#endif
}

// b in lanes 8 to 15 of every sixteen from the lane eight before; a in the others.
__device__ __forceinline__ uint32_t ma_upper_from(uint32_t a, uint32_t b) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)a, (int)b, 0x128, 0xF, 0xC, false);      // (turned by eight, banks 2 and 3)
}
// a in lanes 0 to 7 of every sixteen from the lane eight after; b in the others.
__device__ __forceinline__ uint32_t ma_lower_from(uint32_t a, uint32_t b) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)b, (int)a, 0x128, 0xF, 0x3, false);
}
