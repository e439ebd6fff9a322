// What a tile GEMM launch computes, shared by the GEMM kernel files.
#pragma once

#include <type_traits>
#include <utility>

#include "common.h"

namespace bx {

// Up to three weights share the activation rows X (q / k / v): member i has
// N[i] output columns in Y[i], tiles_n[i] column tiles; a block's tile index
// runs over the members' column tiles in order.  EPI_STORE writes Y = f16(acc
// + bias); EPI_RESID adds f16(acc) to the FP32 residual H[M, N[0]]; EPI_SWIGLU
// computes gate (W[0]) and up (W[1]) columns of the same tile and writes Y[0] =
// f16(f16(silu(f16(gate))) * f16(up)).  EPI_RESID and EPI_SWIGLU give the bits of
// the separate linear, add, silu and mul kernels (weights on 16-byte
// boundaries); several members give those of their plain launches too, but for
// quantized weights whose K slices differ there (gemm_quant.hip), where they
// differ by the order of FP32 sums.
enum : int { EPI_STORE = 0, EPI_RESID = 1, EPI_SWIGLU = 2 };
struct TileJob {
    const void* W[3];
    uint16_t* Y[3];
    int N[3];
    int tiles_n[3];
    int members;
    int tiles_m;
    float* H;
};

// Tile t of T (tiles of M fastest within a weight column) for block b: the
// dispatcher deals blocks to the 8 XCDs round-robin, so XCD x receives
// blocks x, x+8, ...; those are given the x-th contiguous run of tiles.
__device__ __forceinline__ int xcd_tile(int b, int T) {
    const int x = b & 7, i = b >> 3, per = T >> 3, rem = T & 7;
    return (x < rem ? x * (per + 1) : rem * (per + 1) + (x - rem) * per) + i;
}

// The split-K workspace of the linear entry points (bx_linear_workspace_bytes):
// one arrival counter per tile or tile group (tagged_arrive), then FP32
// partial sums.
constexpr int kSplGroups = 4096;                 // counters
constexpr int64_t kSplFloats = 16ll << 20;       // partials: 64 MB
constexpr size_t kSplCntBytes = (size_t)kSplGroups * 8;

// Cache policy of the partials' buffer stores and loads: sc1, device scope.
constexpr int kSc1 = 16;

// f(std::integral_constant<int, i>) for i = 0 .. N - 1, unrolled.
template <class F, int... I>
__device__ __forceinline__ void static_for_(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_(f, std::make_integer_sequence<int, N>{});
}

// LDS-DMA copies issued from inline assembly: lane i's 16 (4) bytes land at
// the wave-uniform LDS address lds + 16 i (4 i).  The compiler's wait-count
// pass does not see them, so it does not make every LDS read wait for every
// copy in flight (it cannot tell the two apart); the kernels wait with
// wait_vm before the barrier that publishes the data.  M0 holds the LDS
// address; nothing else in these kernels uses it.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(uint32_t voff, const void* base, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(lds)
                 : "memory", "m0");
}
__device__ __forceinline__ void dma16p(const void* src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds)
                 : "memory", "m0");
}
__device__ __forceinline__ void dma4p(const void* src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(lds)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

// At most N vector-memory operations of this wavefront still in flight, and
// all of its LDS reads done; then every wavefront of the workgroup.
template <int N>
__device__ __forceinline__ void wait_vm_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

}  // namespace bx
