// Unpadded operand tiles in LDS (gfx950 only): where their 16-byte chunks lie, and the MFMA operand reads of k-outer rows.
#pragma once
#include "ksmm_mfma.h"

namespace ksmm {

// chunk swizzles (applied to the global address a lane fetches and by the operand reads)
// LDS has 64 banks of 4 bytes: a ds_read_b64 is served 32 lanes per clock and a ds_read_b128
// 16 lanes per clock, conflict-free when those lanes cover 256 bytes of distinct banks.
//  k-outer fp16 rows (CPR chunks of 16 bytes): the 32 lanes of a transpose load read 4 rows x
//  64 bytes -> XOR the 64-byte group index with row & 3 (rows of 128 bytes alternate bank
//  halves already: row / 2 & 1).
//  k-outer e4m3 rows: the 32 lanes of a transpose load read 8 rows x 32 bytes -> XOR the
//  32-byte group index with row & 7 (rows of 128 bytes: two rows per bank line, (row / 2) & 3;
//  rows of 64 bytes: four per bank line, (row / 4) & 1).
//  k-outer fp32: 2 rows x 128 bytes per ds_read_b32 wave -> XOR the 128-byte half with row & 1.
//  k-inner rows: 16 lanes read one chunk of 16 consecutive rows -> XOR the chunk so that the
//  rows sharing a 256-byte bank line differ (rows of 64, 128, >= 256 bytes).
template <typename CT, int CPR> __device__ __forceinline__ int swz_outer(int row)
{
    if (sizeof(CT) == 1) return CPR >= 16 ? 2 * (row & 7) : CPR == 8 ? 2 * ((row >> 1) & 3) : 2 * ((row >> 2) & 1);
    return sizeof(CT) == 2 ? (CPR >= 16 ? 4 * (row & 3) : 4 * ((row >> 1) & 1)) : 8 * (row & 1);
}
template <int CPR> __device__ __forceinline__ int swz_inner(int row)
{
    return CPR == 4 ? ((row >> 2) & 3) : CPR == 8 ? ((row >> 1) & 7) : (row & 15);
}

// k-outer operand (weights always, input for bs_last): S[k][idx], row of COLS elements.
// The address of a fragment is (per-lane byte offset, fixed for the kernel) + (stage base,
// uniform) + (k0 * row bytes, a compile-time constant that goes into the instruction's offset
// field): outer_off gives the first, outer_read takes the sum of the first two.
typedef __attribute__((address_space(3))) unsigned char *lds_bytes_t;
template <typename CT, int COLS> struct outer_frag;
template <int COLS> struct outer_frag<half_t, COLS> {
    __device__ static __forceinline__ uint32_t off(int idx0, int lane)
    {
        const int kq = lane >> 5, i16 = lane & 15, hs = (lane >> 4) & 1;
        const int row = 8 * kq + (i16 >> 2);  // + k0 (a multiple of 16): same row & 3
        const int chunk = (idx0 >> 3) + 2 * hs + ((i16 & 3) >> 1);
        return (uint32_t)(row * COLS * 2 + ((chunk ^ swz_outer<half_t, COLS / 8>(row)) << 4) + 8 * (i16 & 1));
    }
    __device__ static __forceinline__ half8_t read(uint32_t addr, int k0)
    {
        typedef short4_t __attribute__((address_space(3))) * lds_ptr;
        short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(lds_bytes_t)(uintptr_t)(addr + k0 * COLS * 2));
        short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(lds_bytes_t)(uintptr_t)(addr + (k0 + 4) * COLS * 2));
        typedef short short8_t __attribute__((ext_vector_type(8)));
        short8_t r = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        return __builtin_bit_cast(half8_t, r);
    }
};
template <int COLS> struct outer_frag<fp8_t, COLS> {
    // ds_read_b64_tr_b8: 16 lanes address 8 rows x 16 bytes (lanes 2i, 2i+1: the two halves of
    // row i) and lane j receives column j, i.e. 8 consecutive k of one index
    __device__ static __forceinline__ uint32_t off(int idx0, int lane)
    {
        const int kq = lane >> 5, l16 = lane & 15, hs = (lane >> 4) & 1;
        const int row = 8 * kq + (l16 >> 1);  // + k0 (a multiple of 16): same row & 7
        const int chunk = (idx0 >> 4) + hs;
        return (uint32_t)(row * COLS + ((chunk ^ swz_outer<fp8_t, COLS / 16>(row)) << 4) + 8 * (l16 & 1));
    }
    __device__ static __forceinline__ long read(uint32_t addr, int k0)
    {
        typedef int int2_t __attribute__((ext_vector_type(2)));
        typedef int2_t __attribute__((address_space(3))) * lds_ptr;
        const int2_t r = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_ptr)(lds_bytes_t)(uintptr_t)(addr + k0 * COLS));
        return __builtin_bit_cast(long, r);
    }
};
template <int COLS> struct outer_frag<float, COLS> {
    __device__ static __forceinline__ uint32_t off(int idx0, int lane)
    {
        const int row = lane >> 5, col = idx0 + (lane & 31);  // + k0 (even): same row & 1
        return (uint32_t)((row * COLS + ((((col >> 2) ^ (8 * (row & 1))) << 2) | (col & 3))) * 4);
    }
    __device__ static __forceinline__ float read(uint32_t addr, int k0)
    {
        typedef __attribute__((address_space(3))) float *lds_ptr;
        return *(lds_ptr)(lds_bytes_t)(uintptr_t)(addr + k0 * COLS * 4);
    }
};

}  // namespace ksmm
