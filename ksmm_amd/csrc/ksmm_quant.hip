// Quantisation of a layer's input to e4m3fn: one scale for the tensor, amax / 448, codes t / scale rounded
// to nearest even.  The scale stays on the device: the first factor's kernel reads it (Epi::x_scale), so
// nothing waits for the GPU.
//
// Two passes over the input, in one launch where it is small.  What bounds them: HBM (or the cache that the layer before left the input in),
// 2 + 2 + 1 bytes a value in fp16.  The same steps as tensor operations (to fp32, abs, max, compare, select,
// divide, to e4m3) move about 40 bytes a value, and reading the scale on the host waits for them: a ViT-B
// feed-forward block on 6304 rows took 324 us with them and takes 111, 30 of them here (6304 x 3072 fp16:
// 8 us for the maximum, 12.8 for the codes, 15 when they divided; 6304 x 768: 2.5 and 5.3).  Fewer workgroups with
// the loads ahead of the scale's reduction: the same time.
//
// Bit for bit what those operations give on this GPU: amax is the largest magnitude as an integer (a NaN is
// above infinity and stays), the division by 448 is the product with its rounded reciprocal, values are
// divided (or given the quotient's bits by residuals), and what rounds beyond 448 (scales that under- or overflowed, NaN) is the NaN code.
#include "ksmm_common.h"

namespace ksmm {

namespace {

constexpr int QUANT_BLOCKS = 1024, RUN = 16;  // workgroups of the first pass, values a thread takes at once

template <typename T> struct qvec {
    static constexpr int N = 16 / sizeof(T), LOADS = RUN / N;
};
typedef uint16_t ushort2_t __attribute__((ext_vector_type(2)));

// largest magnitude of the values of a word, as the bits of that type (fp16: two halves, kept apart)
template <typename T> __device__ __forceinline__ uint32_t max_bits(uint32_t m, uint32_t v);
template <> __device__ __forceinline__ uint32_t max_bits<float>(uint32_t m, uint32_t v) { return max(m, v & 0x7fffffffu); }
template <> __device__ __forceinline__ uint32_t max_bits<half_t>(uint32_t m, uint32_t v)
{
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(ushort2_t, m),
                                                                  __builtin_bit_cast(ushort2_t, v & 0x7fff7fffu)));
}

// the bits as those of the value in fp32
template <typename T> __device__ __forceinline__ uint32_t as_f32_bits(uint32_t m);
template <> __device__ __forceinline__ uint32_t as_f32_bits<float>(uint32_t m) { return m; }
template <> __device__ __forceinline__ uint32_t as_f32_bits<half_t>(uint32_t m)
{
    const uint16_t h = (uint16_t)max(m & 0xffffu, m >> 16);
    return __builtin_bit_cast(uint32_t, (float)__builtin_bit_cast(half_t, h));
}

// largest value over a workgroup of W waves
template <int W> __device__ __forceinline__ uint32_t block_max(uint32_t m, uint32_t *red)
{
#pragma unroll
    for (int s = 32; s; s >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, s, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < W; ++w) m = max(m, red[w]);
    return m;
}

// Largest magnitude (its bits in fp32) of the values that thread `me` of `stride` takes.
// ALIGNED: x starts on a 16-byte boundary (else single elements)
template <typename T, bool ALIGNED> __device__ __forceinline__ uint32_t max_of(const T *__restrict__ x, int64_t n, int64_t me, int64_t stride)
{
    constexpr int N = qvec<T>::N, U = 4;
    const int64_t vecs = ALIGNED ? n / N : 0;
    const uint4_t *xv = (const uint4_t *)x;
    uint32_t m = 0;
    int64_t i = me;
    for (; i + (U - 1) * stride < vecs; i += U * stride) {
        uint4_t v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = xv[i + u * stride];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) m = max_bits<T>(m, v[u][e]);
    }
    for (; i < vecs; i += stride) {
        const uint4_t v = xv[i];
#pragma unroll
        for (int e = 0; e < 4; ++e) m = max_bits<T>(m, v[e]);
    }
    m = as_f32_bits<T>(m);
    for (int64_t k = vecs * N + me; k < n; k += stride) {
        const float v = (float)x[k];
        m = max(m, __builtin_bit_cast(uint32_t, v) & 0x7fffffffu);
    }
    return m;
}

template <typename T, bool ALIGNED>
__global__ __launch_bounds__(256) void ks_amax_kernel(const T *__restrict__ x, uint32_t *__restrict__ part, int64_t n)
{
    __shared__ uint32_t red[4];
    const uint32_t m = block_max<4>(max_of<T, ALIGNED>(x, n, (int64_t)blockIdx.x * 256 + threadIdx.x, (int64_t)gridDim.x * 256), red);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// t / scale as an e4m3fn code in the low byte
__device__ __forceinline__ uint32_t quant_code(float t, float scale)
{
    const float v = t / scale;
    const uint32_t code = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(v, v, 0, false) & 0xffu;
    // 464 is halfway between 448, which is even, and the next step; NaN fails the comparison
    return fabsf(v) <= 464.f ? code : ((__builtin_bit_cast(uint32_t, v) >> 24) & 0x80u) | 0x7fu;
}

// t / scale correctly rounded, for r = 1 / scale correctly rounded: the first residual brings the quotient
// within one unit in the last place, the second to the nearest (Markstein's theorem; both residuals are exact
// in an fma).  The sign is t's, which a residual of zero would lose for t = -0.
__device__ __forceinline__ float quotient(float t, float scale, float r)
{
    float q = t * r;
    q = fmaf(fmaf(-q, scale, t), r, q);
    q = fmaf(fmaf(-q, scale, t), r, q);
    return copysignf(q, t);
}

// codes of the whole tensor for its largest magnitude (the bits of it); one run a thread at a time
template <typename T, bool ALIGNED>
__device__ __forceinline__ void quant_all(const T *__restrict__ x, uint8_t *__restrict__ q, uint32_t max_f32, float *__restrict__ scale_out,
                                          int64_t n, int64_t me, int64_t stride)
{
    constexpr int N = qvec<T>::N, LOADS = qvec<T>::LOADS;
    const float amax = __builtin_bit_cast(float, max_f32);
    const float scale = amax > 0.f ? amax * (1.0f / 448.0f) : 1.0f;
    if (me == 0) *scale_out = scale;
    const int64_t runs = ALIGNED ? n / RUN : 0;
    // A division is ten instructions, a quarter-rate one among them, and bounded the codes.  For ordinary scales
    // seven do: every quotient that is not rounded to zero has residuals above the subnormals, and none is
    // beyond 448 by more than its rounding, so nothing is tested.  0, infinite and NaN maxima divide.
    const bool ordinary = amax > 0.f && scale >= 0x1p-60f && scale <= 0x1p60f;
    const float r = 1.0f / scale;
    for (int64_t i = me; i < runs; i += stride) {
        uint4_t v[LOADS];
#pragma unroll
        for (int l = 0; l < LOADS; ++l) v[l] = ((const uint4_t *)x)[i * LOADS + l];
        uint4_t o = {0u, 0u, 0u, 0u};
        if (ordinary) {
#pragma unroll
            for (int e = 0; e < RUN; e += 4) {
                const T *t = (const T *)&v[e / N] + e % N;
                const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(quotient((float)t[0], scale, r), quotient((float)t[1], scale, r), 0, false);
                o[e / 4] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(quotient((float)t[2], scale, r), quotient((float)t[3], scale, r), lo, true);
            }
        } else {
#pragma unroll
            for (int e = 0; e < RUN; ++e) {
                const T *t = (const T *)&v[e / N];
                o[e / 4] |= quant_code((float)t[e % N], scale) << (8 * (e % 4));
            }
        }
        ((uint4_t *)q)[i] = o;
    }
    for (int64_t k = runs * RUN + me; k < n; k += stride) q[k] = (uint8_t)quant_code((float)x[k], scale);
}

template <typename T, bool ALIGNED>
__global__ __launch_bounds__(256) void ks_quant_kernel(const T *__restrict__ x, uint8_t *__restrict__ q,
                                                       const uint32_t *__restrict__ part, int parts, float *__restrict__ scale_out,
                                                       int64_t n)
{
    __shared__ uint32_t red[4];
    uint32_t m = 0;
    for (int i = threadIdx.x; i < parts; i += 256) m = max(m, part[i]);
    m = block_max<4>(m, red);
    quant_all<T, ALIGNED>(x, q, m, scale_out, n, (int64_t)blockIdx.x * 256 + threadIdx.x, (int64_t)gridDim.x * 256);
}

// Both passes of a small tensor in one launch: every workgroup looks for the maximum itself.  What bounds it up to
// 64 KB is the launch, then one CU's rate of loads from L2 (about 100 GB/s).
template <typename T>
__global__ __launch_bounds__(1024) void ks_quant_small_kernel(const T *__restrict__ x, uint8_t *__restrict__ q, float *__restrict__ scale_out,
                                                              int n)
{
    __shared__ uint32_t red[16];
    const uint32_t m = block_max<16>(max_of<T, true>(x, n, threadIdx.x, 1024), red);
    quant_all<T, true>(x, q, m, scale_out, n, blockIdx.x * 1024 + threadIdx.x, gridDim.x * 1024);
}

// Bytes up to which one launch is the faster.  Layers of (4,64,64,1) / (1,128,128,16), us a call with two launches and
// with one: fp16 64 KB 11.5 / 11.4 and 9.7 / 8.9, 256 KB 11.6 / 11.5 and 10.8 / 9.4, 384 KB 14.7 / 13.2 and 12.5 / 10.9,
// 512 KB 13.4 / 13.2 and 13.0 / 11.7, 768 KB 13.3 / 13.3 and 14.7 / 13.5; fp32 within 0.5 of these.
constexpr int64_t SMALL_BYTES = 384 << 10;

// e4m3fn codes as fp16 (exact), for the weights of a whole chain in one launch
struct DecodeArgs {
    struct {
        const uint8_t *codes;
        half_t *to;
        int64_t n;
        uint32_t first;  // the job's first workgroup
    } job[KSMM_MAX_FACTORS];
    int jobs;
};

__global__ __launch_bounds__(256) void ks_decode_kernel(DecodeArgs d)
{
    int k = 0;
    while (k + 1 < d.jobs && blockIdx.x >= d.job[k + 1].first) ++k;
    const uint8_t *codes = d.job[k].codes;
    half_t *to = d.job[k].to;
    const int64_t n = d.job[k].n, at = ((int64_t)(blockIdx.x - d.job[k].first) * 256 + threadIdx.x) * RUN;
    if (at >= n) return;
    if (at + RUN <= n) {
        uint4_t v;
        __builtin_memcpy(&v, codes + at, 16);  // (any alignment)
        uint4_t o[2];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            o[w >> 1][2 * (w & 1)] = __builtin_bit_cast(uint32_t, fp8x2_to_half2(v[w]));
            o[w >> 1][2 * (w & 1) + 1] = __builtin_bit_cast(uint32_t, fp8x2_hi_to_half2(v[w]));
        }
        ((uint4_t *)(to + at))[0] = o[0];
        ((uint4_t *)(to + at))[1] = o[1];
    } else {
        for (int64_t i = at; i < n; ++i) to[i] = fp8_to_half(codes[i]);
    }
}

template <typename T> int launch(const void *x, void *q, uint32_t *part, float *scale, int64_t n, hipStream_t s)
{
    const bool aligned = ((uintptr_t)x & 15) == 0;
    if (aligned && n * (int64_t)sizeof(T) <= SMALL_BYTES) {
        const int64_t blocks = (n + 1024 * RUN - 1) / (1024 * RUN);
        hipLaunchKernelGGL(ks_quant_small_kernel<T>, dim3((unsigned)blocks), dim3(1024), 0, s, (const T *)x, (uint8_t *)q, scale, (int)n);
        return hipGetLastError() == hipSuccess ? KSMM_OK : KSMM_ERR_LAUNCH;
    }
    // first pass: four vectors a thread, four workgroups a CU at most; second: one run a thread
    int64_t parts = (n + 256 * 4 * qvec<T>::N - 1) / (256 * 4 * qvec<T>::N), blocks = (n + 256 * RUN - 1) / (256 * RUN);
    if (parts > QUANT_BLOCKS) parts = QUANT_BLOCKS;
    if (blocks > 4096) blocks = 4096;
    const auto first = aligned ? &ks_amax_kernel<T, true> : &ks_amax_kernel<T, false>;
    const auto second = aligned ? &ks_quant_kernel<T, true> : &ks_quant_kernel<T, false>;
    hipLaunchKernelGGL(first, dim3((unsigned)parts), dim3(256), 0, s, (const T *)x, part, n);
    hipLaunchKernelGGL(second, dim3((unsigned)blocks), dim3(256), 0, s, (const T *)x, (uint8_t *)q, part, (int)parts, scale, n);
    return hipGetLastError() == hipSuccess ? KSMM_OK : KSMM_ERR_LAUNCH;
}

}  // namespace

int decode_run(const DecodeJob *jobs, int n, hipStream_t stream)
{
    DecodeArgs d;
    int64_t blocks = 0;
    d.jobs = n;
    for (int i = 0; i < n; ++i) {
        d.job[i].codes = (const uint8_t *)jobs[i].codes;
        d.job[i].to = (half_t *)jobs[i].to;
        d.job[i].n = jobs[i].n;
        d.job[i].first = (uint32_t)blocks;
        blocks += (jobs[i].n + 256 * RUN - 1) / (256 * RUN);
        if (blocks > 0x7fffffffLL) return KSMM_ERR_TOO_LARGE;
    }
    if (blocks < 1) return KSMM_OK;
    hipLaunchKernelGGL(ks_decode_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, d);
    return hipGetLastError() == hipSuccess ? KSMM_OK : KSMM_ERR_LAUNCH;
}

int64_t quantize_scratch_bytes() { return 4 * QUANT_BLOCKS; }

int quantize_run(const void *x, int x_dtype, void *codes, float *scale, void *scratch, int64_t n, hipStream_t stream)
{
    if (x_dtype == KSMM_F32) return launch<float>(x, codes, (uint32_t *)scratch, scale, n, stream);
    if (x_dtype == KSMM_F16) return launch<half_t>(x, codes, (uint32_t *)scratch, scale, n, stream);
    return KSMM_ERR_BAD_DTYPE;
}

}  // namespace ksmm
