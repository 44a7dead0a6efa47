// fmha_device.h — device-side pieces shared by the gfx950 attention kernels:
// operand types, tile constants, LDS-DMA, waits, the XOR-swizzled tile reads
// and the MFMA they feed (the layouts are described in fmha_fwd_kernel.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fmha_fwd.h"

namespace fmha_gfx950 {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));

constexpr int kWaves = FMHA_KBLOCK / 64;  // 4
constexpr int kRowsPerWave = 32;
constexpr int kTileM = kWaves * kRowsPerWave;  // 128
constexpr int kTileN = FMHA_KN0;               // 64 keys per tile
constexpr int kRowBytes = 128;                 // 64 bf16 per K/V row in LDS
constexpr int kTileBytes = kTileN * kRowBytes; // 8 KiB
constexpr int kRing = 4;                       // stages per ring (K and V)
constexpr int kLoadsPerTile = 2;                   // 1 KiB DMA per load, per wave
constexpr float kGrowSum = 65536.0f;               // tile-sum bound of the speculative softmax
// Running-max seed, in the scaled (exp2) domain: below every finite scaled
// score, so a row's first visible key always re-frames it (its P overflows
// the bound).  The reference seeds -5000 raw-score units (pipeline.hpp:248-252),
// which drops rows whose every score lies below that; its CPU checker
// (cpu_ref.cpp:124-136) has no seed at all, and neither has this kernel.
constexpr float kMaxSeed = -3.402823466e38f;       // -FLT_MAX
constexpr uint32_t kBufferWord3 = 0x00020000u;     // raw dword buffer, gfx9 family
constexpr int kPartFloatsPerWave = 34 * 64;        // balanced form: one wave's partial result (O^T, m, l)
// Cache policy of the O stores: non-temporal (NT).  No block reads O back, and
// O kept out of the caches leaves them to K/V (dense B4 H16 S2048 and causal
// B1 H16 S8192 +1 %, short form dense B128 H16 S128 +2.5 %).
constexpr int kStoreStream = 2;

static_assert(kTileM == FMHA_KM0, "tile rows must match the grid contract");
static_assert(kWaves * kLoadsPerTile * 1024 == kTileBytes, "one tile = one DMA round of the block");

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t num_bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)num_bytes, (int)kBufferWord3);
}

typedef __attribute__((address_space(3))) char lds_char;

// 64 lanes x 16 bytes global -> LDS (buffer_load_dwordx4 ... lds); lane L
// lands at dst + 16*L.  dst must be wave-uniform.
__device__ __forceinline__ void lds_dma_16(__amdgpu_buffer_rsrc_t rsrc, lds_char* dst, int voffset) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)dst, 16, voffset, 0, 0, 0);
}
// The same with a wave-uniform byte offset in the scalar offset operand.
__device__ __forceinline__ void lds_dma_16(__amdgpu_buffer_rsrc_t rsrc, lds_char* dst, int voffset, int soffset) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)dst, 16, voffset, soffset,
                                             0, 0);
}
// Own-wave DMA completion before a tile barrier (the barrier then makes every
// wave's part of the tile visible).
template <int N>
__device__ __forceinline__ void vmcnt_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// s_waitcnt immediate for vmcnt(0) alone (gfx9 encoding: vmcnt [3:0] and
// [15:14], expcnt [6:4] and lgkmcnt [11:8] at their no-wait maxima)
constexpr int kWaitVmcnt0 = 0x0F70;
// s_waitcnt immediate for lgkmcnt(0) alone (vmcnt and expcnt at their maxima)
constexpr int kWaitLgkmcnt0 = 0xC07F;
// Workgroup barrier of the K/V ring, without __syncthreads()'s memory fence:
// that fence waits vmcnt(0), i.e. also for the prefetches still in flight.
// Before the barrier each wave has waited for its own DMA of the tile about
// to be read (vmcnt_wait) and, here, for all of its own LDS reads
// (lgkmcnt(0)): right after the barrier other waves refill the stages those
// reads came from, and s_barrier itself waits for no memory operation (the
// compiler may otherwise leave a read in flight across it when it sinks the
// consuming MFMA past the barrier).  The "memory" clobber keeps the compiler
// from moving LDS accesses across it.
__device__ __forceinline__ void ring_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// A copy of a wave-uniform value in a VGPR.  A VALU operand read from an SGPR
// costs gfx950 ~4.4 issue cycles per wave64 instruction against ~2.6-3.2 for
// VGPR operands (fma, mul, sub alike), so per-element operands are kept in VGPRs.
__device__ __forceinline__ float in_vgpr(float x) {
    float v;
    asm("v_mov_b32 %0, %1" : "=v"(v) : "s"(x));
    return v;
}

// XOR swizzle of the 16-byte chunk index inside a 128-byte K row (row & 15 is
// all it depends on).  Conflict-free ds_read_b128 for both 32- and 64-bank LDS.
__device__ __forceinline__ int k_swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }
// V rows: the tr_b16 read touches 4 consecutive rows x 4 chunks per 32 lanes.
__device__ __forceinline__ int v_swz(int row) { return (row & 3) << 1; }

__device__ __forceinline__ float wave_max_halves(float x) {
    auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
__device__ __forceinline__ float wave_sum_halves(float x) {
    auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
typedef __attribute__((address_space(3))) i32x2 lds_i32x2;
typedef __attribute__((address_space(3))) i32x4 lds_i32x4;

__device__ __forceinline__ bf16x8 lds_read_b128(const lds_char* p) { return *(const lds_bf16x8*)p; }
// 8 keys x 1 head-dim column of V for the GEMM1 A operand (two tr_b16 reads,
// rows key0..key0+3 and key0+8..key0+11).
__device__ __forceinline__ bf16x8 lds_read_vt(const lds_char* p) {
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)p);
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(p + 8 * kRowBytes));
    i16x4 both[2] = {lo, hi};
    return __builtin_bit_cast(bf16x8, both);
}

__device__ __forceinline__ f32x16 mfma(const bf16x8& a, const bf16x8& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

}  // namespace fmha_gfx950
