// Operands that go from global memory straight into MFMA registers (gfx950 only): vectors at element alignment,
// and the 16-bit pairs an operand is put together from.
#pragma once
#include "ksmm_common.h"

namespace ksmm {

// N consecutive elements at element alignment (global memory takes unaligned vector accesses), kept
// as the dwords they arrive in: 16-bit elements in variables of their own would take a register each.
// (a uniform base and a 32-bit byte offset per lane: one address register instead of two)
template <typename T, int N> struct rawn {
    uint32_t v[(N * sizeof(T) + 3) / 4];
};
template <typename T, int N> __device__ __forceinline__ rawn<T, N> load_n(const T *base, uint32_t offset)
{
    rawn<T, N> r;
    __builtin_memcpy(&r, (const char *)base + offset, N * sizeof(T));
    return r;
}
template <typename T, int N> struct vecn {
    T v[N];
};

// the dword that holds 16-bit elements i and i + 1 (i even) of what was loaded; e4m3 is decoded
template <int N> __device__ __forceinline__ uint32_t pair16(const rawn<half_t, N> &r, int i) { return r.v[i >> 1]; }
template <int N> __device__ __forceinline__ uint32_t pair16(const rawn<fp8_t, N> &r, int i)
{
    return __builtin_bit_cast(uint32_t, (i & 2) ? fp8x2_hi_to_half2(r.v[i >> 2]) : fp8x2_to_half2(r.v[i >> 2]));
}
// (element i of a, element j of b) as one dword
template <typename T, int N> __device__ __forceinline__ uint32_t pick16(const rawn<T, N> &a, int i, const rawn<T, N> &b, int j)
{
    const uint32_t sel = ((i & 1) ? 0x0302u : 0x0100u) | ((j & 1) ? 0x07060000u : 0x05040000u);
    return __builtin_amdgcn_perm(pair16(b, j & ~1), pair16(a, i & ~1), sel);
}

template <typename T> struct op_type { typedef half_t type; };
template <> struct op_type<float> { typedef float type; };

}  // namespace ksmm
