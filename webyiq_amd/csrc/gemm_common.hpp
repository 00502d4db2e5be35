// Shared parts of the prefill GEMM kernels (gemm_q4q8.hip, gemm_wave.hip): the
// launch parameters, the LDS chunk swizzles, the nibble expansion and the
// direct global -> LDS loads.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace wq {
namespace {

constexpr int kBK = 128;          // codes per K step (= bytes per int8 tile row)
constexpr int kXcds = 8;          // MI355X: 8 XCDs, workgroups dispatched round robin
constexpr int kLdsBytes = 160 * 1024;  // LDS per workgroup (gfx950)

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;

struct GemmParams {
    LinearArgs a;
    int tilesM, tilesN;
    int NE, NG;  // accumulation and weight groups per row
    // 128-token tiles: split K across workgroup pairs, workspace of per-tile
    // ready flags (one 64-byte line each) and partial sums
    int split;
    unsigned int* flags;  // [T] lines
    float* part;          // [T][128 * BN] partial sums of the first half
    // K split between waves: the launch's tiles, and whether ws, xs and dx are
    // 16-byte aligned
    int first, count, wide;
};

// Chunk swizzles: activation rows are 128 bytes (8 chunks), packed weight
// rows 64 bytes (4 chunks); chunk c of row r sits at position c ^ f(r).
__device__ __forceinline__ int swz_a(int r) { return (r ^ (r >> 3)) & 7; }
__device__ __forceinline__ int swz_b(int r) { return (r >> 1) & 3; }
// Packed weight rows of two K steps (128 bytes, 8 chunks: the even step's 4,
// then the odd step's): chunk c of row r at position c ^ swz_p(r), so that 16
// consecutive rows' 16-byte reads of one chunk cover 256 distinct bytes of
// banks.
__device__ __forceinline__ int swz_p(int r) { return (r >> 1) & 7; }

// f(std::integral_constant<int, I>) for I = B .. E-1, in order
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// 16 codes (8 packed bytes) -> 16 int8 in code order: the low nibbles of a
// word are codes 8i..8i+3, the high nibbles 8i+4..8i+7.
__device__ __forceinline__ v4i expand8(uint32_t w0, uint32_t w1) {
    return v4i{(int)(w0 & kNibbleMask), (int)((w0 >> 4) & kNibbleMask),
               (int)(w1 & kNibbleMask), (int)((w1 >> 4) & kNibbleMask)};
}

// End of a pipeline step: wait until at most n vector-memory operations of
// this wave are in flight and all its LDS operations are done, then barrier.
// The barrier carries no memory fence, so loads issued for later steps stay
// in flight across it.
template <int n>
__device__ __forceinline__ void step_barrier() {
    static_assert(n >= 0 && n < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4));
    asm volatile("s_barrier" ::: "memory");
}

// Direct global -> LDS loads of 16 (4) bytes per lane: lane l's bytes land at
// LDS address lds + 16 l (4 l); base and lds are wave-uniform, off per lane.
// Written as inline assembly so that the compiler's wait-count pass does not
// track them: it cannot tell the stages of the ring apart and would wait for
// every load in flight before the first LDS read of a step.  The waits these
// loads need are explicit (step_barrier); for loads the compiler does track,
// untracked loads issued in between only make its waits stricter.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void*)p);
}
__device__ __forceinline__ const void* uniform_ptr(const void* p) {
    const uint64_t v = (uint64_t)(uintptr_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const void*)(uintptr_t)(((uint64_t)hi << 32) | lo);
}
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma4(const void* base, uint32_t off, const void* lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 ::"v"(off), "s"(uniform_ptr(base)), "s"(lds_addr(lds)) : "memory", "m0");
}
// The same with the LDS destination given as a wave-uniform 32-bit LDS byte
// address (kept in scalar registers by the caller: no per-load conversion of
// a generic pointer).
__device__ __forceinline__ void dma16_at(const void* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 ::"v"(off), "s"(uniform_ptr(base)), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void dma4_at(const void* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 ::"v"(off), "s"(uniform_ptr(base)), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop

}  // namespace
}  // namespace wq
