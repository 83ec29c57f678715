// Shared device helpers for the gfx950 attention kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rt_kernels.hpp"

namespace rt {

constexpr int kWave = 64;
constexpr float kLog2e = 1.4426950408889634f;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// bf16 bit pattern <-> f32.  Round to nearest even; NaN stays a quiet NaN.
__device__ __forceinline__ float bf16_bits_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float x) {
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x0040u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
// Two f32 -> packed bf16x2 (lo in bits 0..15).
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    return (uint32_t)f32_to_bf16_bits(lo) | ((uint32_t)f32_to_bf16_bits(hi) << 16);
}
__device__ __forceinline__ float bf16_lo(uint32_t packed) { return __uint_as_float(packed << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t packed) { return __uint_as_float(packed & 0xffff0000u); }

constexpr uint32_t kBufferFlags = 0x00020000u;  // dword 3 of a raw buffer descriptor: 32-bit data format, no swizzle

// 16 bytes per lane from a buffer straight into LDS: lane l lands at LDS byte address lds_block + 16 l (lds_block is
// wave-uniform and goes through M0); a lane whose offset lies past the end of the descriptor lands zeros.  Issued as
// inline assembly so that the compiler's counter bookkeeping does not make every later LDS read wait for it:
// completion is awaited explicitly (s_waitcnt vmcnt before the barrier that publishes the tile).  Loads the
// compiler does not know of can only make its own vmcnt waits longer, never shorter: the counter retires in order.
// (The statement counts as a writer of memory, which keeps the compiler from moving LDS reads across it.)
__device__ __forceinline__ void buffer_to_lds(const u32x4_t& rsrc, uint32_t lane_off, uint32_t tile_off, uint32_t lds_block) {
    const uint32_t m = __builtin_amdgcn_readfirstlane(lds_block);
    const uint32_t so = __builtin_amdgcn_readfirstlane(tile_off);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(m), "v"(lane_off), "s"(rsrc), "s"(so)
                 : "memory");
}
// the same past the caches (`nt`), for what no other workgroup reads
__device__ __forceinline__ void buffer_to_lds_past(const u32x4_t& rsrc, uint32_t lane_off, uint32_t tile_off, uint32_t lds_block) {
    const uint32_t m = __builtin_amdgcn_readfirstlane(lds_block);
    const uint32_t so = __builtin_amdgcn_readfirstlane(tile_off);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 :
                 : "s"(m), "v"(lane_off), "s"(rsrc), "s"(so)
                 : "memory");
}
// the same for the lanes of `on` alone (what the others would have brought stays as it is in LDS); no branch around it
__device__ __forceinline__ void buffer_to_lds_of(uint64_t on, const u32x4_t& rsrc, uint32_t lane_off, uint32_t tile_off, uint32_t lds_block) {
    const uint32_t m = __builtin_amdgcn_readfirstlane(lds_block);
    const uint32_t so = __builtin_amdgcn_readfirstlane(tile_off);
    uint64_t all;
    asm volatile("s_mov_b32 m0, %1\n\ts_and_saveexec_b64 %0, %5\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds\n\ts_mov_b64 exec, %0"
                 : "=&s"(all)
                 : "s"(m), "v"(lane_off), "s"(rsrc), "s"(so), "s"(on)
                 : "memory", "scc");
}
// the same, 4 bytes per lane: lane l lands at lds_block + 4 l
__device__ __forceinline__ void buffer_to_lds_b32(const u32x4_t& rsrc, uint32_t lane_off, uint32_t tile_off, uint32_t lds_block) {
    const uint32_t m = __builtin_amdgcn_readfirstlane(lds_block);
    const uint32_t so = __builtin_amdgcn_readfirstlane(tile_off);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                 :
                 : "s"(m), "v"(lane_off), "s"(rsrc), "s"(so)
                 : "memory");
}
// a raw buffer descriptor as four scalars: base, no stride, `bytes` addressable
__device__ __forceinline__ u32x4_t make_rsrc(const void* base, uint32_t bytes) {
    const uint64_t a = (uint64_t)(uintptr_t)base;
    return u32x4_t{(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu),
                   (uint32_t)__builtin_amdgcn_readfirstlane(bytes), kBufferFlags};
}

// A store of output that nothing of the launch reads again, past the caches (`nt`).  Stored plainly it stays in the L2s of the
// XCDs, 4 MB each, until the end of the launch, which then waits for what is left of it to be written back, and K and V
// meanwhile have that much less room.  us, plainly -> past the caches, bf16: padded batch of 16 x 16 heads, N=1024 D=64 30.1 ->
// 26.9; window 256, 4 x 16 heads, N=4096 D=64 45.9 -> 41.9; causal 2 x 32 / 8 heads, N=1501 D=128 46.8 -> 45.8.  (What the next
// kernel pays for it, and from which size on it is worth it, stands at out_goes_past; the persistent kernel, which takes calls that
// write 11 MB or more, stores this way always.)  For whole lines:
// the f32 kernels' pieces of 32 bytes a row took longer that way (train, 4 x 16 heads, N=1024 D=64 411 -> 418).
template <typename T>
__device__ __forceinline__ void store_past(void* dst, T v) { __builtin_nontemporal_store(v, (T*)dst); }

// x / d by the multiplier 2^32 / d + 1 (exact where x d < 2^32), or by one for the multiplier 0
__device__ __forceinline__ int div_magic(int x, uint32_t magic) { return magic ? (int)__umulhi((uint32_t)x, magic) : x; }

// Value held by the lane 32 positions away (the other half of the wave).
__device__ __forceinline__ float other_half(float x) { return __shfl_xor(x, 32, 64); }

__device__ __forceinline__ float quiet_nan() { return __uint_as_float(0x7fc00000u); }
__device__ __forceinline__ float neg_inf() { return __uint_as_float(0xff800000u); }

}  // namespace rt
