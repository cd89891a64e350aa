// mfma_util.h -- device helpers shared by the matrix-core GEMMs that
// dequantize in registers (gemm_f16.hip, gemm_wide.hip): global -> LDS
// buffer loads, inline LDS reads with explicit waits, the nibble / byte to
// binary16 dequantization.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace rce_qmm {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ half2v as_h2(uint32_t u) {
    half2v h;
    __builtin_memcpy(&h, &u, 4);
    return h;
}

// Buffer load of 16 bytes per lane straight into LDS at lds_wave + 16 * lane:
// byte voff (per lane) + soff (uniform) of the buffer described by r.
__device__ __forceinline__ void buf_load_lds16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff,
                                               unsigned char *lds_wave) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds_wave, 16, voff, soff, 0, 0);
}
// Raw byte buffer of n bytes (gfx9 descriptor word 3 for untyped access).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t byte_buffer(const void *base, uint32_t n) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)n, 0x00020000);
}

// LDS accesses of the pipelined loop are inline ds_read / ds_write: the
// compiler counts the global->LDS loads as writes to all of LDS and would
// wait for every load in flight before each LDS access (the whole
// pipeline).  Their completion is waited for explicitly instead
// (s_waitcnt lgkmcnt(0), then pin below).  OFF is the instruction's
// immediate byte offset.
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}
template <int OFF>
__device__ __forceinline__ half8 lds_read_frag(uint32_t a) {
    static_assert(OFF >= 0 && OFF < 65536, "ds offset");
    half8 v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF) : "memory");
    return v;
}
template <int OFF>
__device__ __forceinline__ uint32_t lds_read_u8(uint32_t a) {
    static_assert(OFF >= 0 && OFF < 65536, "ds offset");
    uint32_t v;
    asm volatile("ds_read_u8 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF) : "memory");
    return v;
}
template <int OFF>
__device__ __forceinline__ uint32_t lds_read_u16(uint32_t a) {
    static_assert(OFF >= 0 && OFF < 65536, "ds offset");
    uint32_t v;
    asm volatile("ds_read_u16 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF) : "memory");
    return v;
}
template <int OFF>
__device__ __forceinline__ uint32_t lds_read4(uint32_t a) {
    static_assert(OFF >= 0 && OFF < 65536, "ds offset");
    uint32_t v;
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF) : "memory");
    return v;
}
template <int OFF>
__device__ __forceinline__ u32x2 lds_read8(uint32_t a) {
    static_assert(OFF >= 0 && OFF < 65536, "ds offset");
    u32x2 v;
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF) : "memory");
    return v;
}
// After s_waitcnt lgkmcnt(0): an empty asm that "redefines" a register
// the reads above filled, so no use of it can move ahead of the wait.
template <class T>
__device__ __forceinline__ void pin(T &r) {
    asm volatile("" : "+v"(r));
}
// pin the low word of a pair only (the high word never written)
__device__ __forceinline__ void pin_lo(u32x2 &r) {
    uint32_t x = r.x;
    asm volatile("" : "+v"(x));
    r.x = x;
}

// s_waitcnt vmcnt(N) (gfx9 encoding; expcnt and lgkmcnt not waited for),
// then a barrier without the memory fence __syncthreads would add (that
// fence waits for every load in flight, the whole pipeline).
template <int N>
__device__ __forceinline__ void wait_vm_barrier() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
    __builtin_amdgcn_s_barrier();
}

// Four bytes of x (nibbles masked to 0..15, or Q8_0's int8 values offset to
// 0..255) as two f16 pairs in byte order: value = s * (n - OFF + 1024) + b
// (packed f16 fma, one rounding), with sb = f16 {s, b}.  Eight VALU ops;
// two calls make one MFMA fragment.
template <int OFF = 1024>
__device__ __forceinline__ void dequant4(uint32_t x, uint32_t sb, half2v &lo, half2v &hi) {
    const uint32_t K64 = 0x64646464u;
    const half2v m1024 = {(_Float16)(-(float)OFF), (_Float16)(-(float)OFF)};
    const half2v p = as_h2(sb);
    const half2v sc = __builtin_shufflevector(p, p, 0, 0), bias = __builtin_shufflevector(p, p, 1, 1);
    // byte pairs (n, 0x64): f16 bits 0x64nn = 1024 + n
    const uint32_t p0 = __builtin_amdgcn_perm(x, K64, 0x00050004u);
    const uint32_t p1 = __builtin_amdgcn_perm(x, K64, 0x00070006u);
    lo = __builtin_elementwise_fma(as_h2(p0) + m1024, sc, bias);
    hi = __builtin_elementwise_fma(as_h2(p1) + m1024, sc, bias);
}

__device__ __forceinline__ half8 join8(half2v a, half2v b, half2v c, half2v d) {
    return half8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}

template <int U>
using ic = std::integral_constant<int, U>;

// f(ic<I>{}) for I = 0 .. N - 1.
template <int N, int I = 0, class Fn>
__device__ __forceinline__ void static_for(Fn &&f) {
    if constexpr (I < N) {
        f(ic<I>{});
        static_for<N, I + 1>(f);
    }
}

}  // namespace
}  // namespace rce_qmm
