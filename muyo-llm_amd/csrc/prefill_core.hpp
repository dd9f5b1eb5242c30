// Device helpers shared by the batched-prefill kernels: the matrix-core operation they are built on
// and the split of an f32 value into two f16 planes.
//
// Matrix-core lane layout of v_mfma_f32_32x32x16_f16 (D = A.B, A 32x16, B 16x32), as used here:
// lane l supplies A[l % 32][8 * (l / 32) .. +8] and B[8 * (l / 32) .. +8][l % 32], and receives
// D[8 * (r / 4) + 4 * (l / 32) + r % 4][l % 32] in accumulator r (0..15).
#pragma once

#include "common.hpp"

namespace muyo
{
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef uint16_t ushort4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx16 Mfma(half8 a, half8 b, floatx16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

/// v = hi + lo to ~21 bits. hi is v with its 13 low mantissa bits cleared: 11 significant bits,
/// exact in f16. Rounding hi to f16 instead is not safe here: with contraction the compiler feeds
/// a product straight into v_fma_mix*_f16 (one rounding to f16) for one use and rounds it to f32
/// first (two roundings) for another, so the stored hi and the hi subtracted for lo can differ by
/// an f16 ulp near a tie. The bit mask works on the f32 value, and lo = v - hi is exact in f32
/// before its one rounding into f16. |v| must stay below 65536 (f16's range).
__device__ __forceinline__ float HiPart(float v) { return __uint_as_float(__float_as_uint(v) & 0xFFFFE000u); }

__device__ __forceinline__ _Float16 HiHalf(float v) { return static_cast<_Float16>(HiPart(v)); }

__device__ __forceinline__ _Float16 LoHalf(float v) { return static_cast<_Float16>(v - HiPart(v)); }

__device__ __forceinline__ void StoreSplit4(uint16_t* hi, uint16_t* lo, uint64_t at, float a, float b, float c,
                                            float d)
{
    const half4 h = {HiHalf(a), HiHalf(b), HiHalf(c), HiHalf(d)};
    const half4 l = {LoHalf(a), LoHalf(b), LoHalf(c), LoHalf(d)};
    *reinterpret_cast<half4*>(hi + at) = h;
    *reinterpret_cast<half4*>(lo + at) = l;
}

/// Requests 16 bytes per lane from base + offset bytes (base uniform across the wave) straight into
/// LDS: the wave's 64 pieces land in lane order in the 1 KB at LDS address to + more (`more` a
/// constant once the loops around are unrolled). The compiler does not see the load: it neither
/// counts it nor orders LDS reads after it (WaitAndMeet does), and keeps no wait states before it.
/// It needs one after m0 is written, and would need five after a vector instruction has written
/// its scalar base (v_readfirstlane, the return of a spilled scalar): the base goes through a
/// scalar move, which waits for either by itself and is the wait state of m0. (m0 is a register
/// in which the compiler keeps nothing across instructions.)
///
/// A wave issues a slab's loads one instruction at a time, so these count in a GEMM of few rows,
/// us, 17 rows of 4864 x 896: 24.3 with the LDS address added up before and an s_nop for m0's wait
/// state alone, 26.1 with an s_nop for the base's five, 24.8 with the move, 21.1 with the move and
/// the addition into m0.
__device__ __forceinline__ void LoadToLds(uint32_t to, uint32_t more, uint32_t offset, const void* base)
{
    uint64_t scalarBase;
    asm volatile("s_add_u32 m0, %1, %2\n\ts_mov_b64 %0, %4\n\tglobal_load_lds_dwordx4 %3, %0"
                 : "=&s"(scalarBase)
                 : "s"(to), "i"(more), "v"(offset), "s"(base)
                 : "scc");
}

/// Waits until at most kLeft of this wave's loads are in flight and its LDS reads are done, then
/// meets the other waves.
template <int kLeft>
__device__ __forceinline__ void WaitAndMeet()
{
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kLeft) : "memory");
}
}  // namespace muyo
