// Backward pass of a layer's epilogue y = act(z), z = K x + bias:
//   dz = dy * act'(z)              (nothing is written without an activation: dz is dy)
//   dbias[f] = sum over the batch of dz[f, n]
// in one pass over dy and z.  The sums are fp32, one slice of partial sums per batch range, added in a
// fixed order (no atomics): the same bits on every run.
//
// What bounds it: HBM, 6 bytes a value in fp16.  The sums cost no traffic of their own; apart they are a
// pass over dz that reads it back.  Batch-size-first, a thread keeps the sums of one 16-byte vector of
// features and walks down the rows; batch-size-last, a wavefront walks along one feature's row.
// fp16, 25088 x 1536 with GELU: 44 us (5.3 TB/s).  With the bias added in the last factor's kernel a
// training step of a ViT-S feed-forward block on 25088 rows went from 489 to 447 us, one of the fp32 layer
// (6,64,64,1)+(1,768,192,2) on 6272 batch-size-last columns (bias only: 10 us here) from 266 to 242 (on one
// box each; such a step varies by a tenth between boxes and with the host).
#include "ksmm_common.h"

namespace ksmm {

namespace {

constexpr float INV_SQRT_2PI = 0.39894228040143268f;

// d gelu / dx = Phi(x) + x phi(x)
template <typename T> __device__ __forceinline__ float gelu_slope(float x);
template <> __device__ __forceinline__ float gelu_slope<float>(float x)
{
    return fmaf(x * INV_SQRT_2PI, expf(-0.5f * x * x), fmaf(0.5f, erff(x * 0.70710678118654752f), 0.5f));
}
// fp16: the series of gelu_erf, whose exponential is phi's as well: erff and expf would take longer than the loads.
// Largest error of the slope over all fp16 values 3.0e-7 (1.3e-7 with erff), next to the type's 5e-4
template <> __device__ __forceinline__ float gelu_slope<half_t>(float x)
{
    const float z = fabsf(x) * 0.84932180028801907f;
    const float t = __builtin_amdgcn_rcpf(fmaf(0.2727374808792225f, z, 1.0f));
    float poly = fmaf(0.5307027145f, t, -0.7265760135f);
    poly = fmaf(poly, t, 0.7107068705f);
    poly = fmaf(poly, t, -0.142248368f);
    poly = fmaf(poly, t, 0.127414796f);
    const float ex = __builtin_amdgcn_exp2f(-(z * z)), tail = (poly * t) * ex;
    return fmaf(x * INV_SQRT_2PI, ex, x >= 0.f ? 1.f - tail : tail);
}

// VEC elements as one load or store
template <typename T, int VEC> struct Vec {
    T v[VEC];
};
template <typename T, int VEC> __device__ __forceinline__ Vec<T, VEC> vload(const T *p)
{
    Vec<T, VEC> r;
    __builtin_memcpy(&r, __builtin_assume_aligned(p, sizeof(r)), sizeof(r));
    return r;
}
template <typename T, int VEC> __device__ __forceinline__ void vstore(T *p, const Vec<T, VEC> &r)
{
    __builtin_memcpy(__builtin_assume_aligned(p, sizeof(r)), &r, sizeof(r));
}

template <typename T, bool ACT> __device__ __forceinline__ float slope_times(float dy, T z)
{
    return ACT ? dy * gelu_slope<T>((float)z) : dy;
}

// Batch-size-first (rows x features).  lx lanes side by side take VEC features each, 256 / lx of them
// below each other walk down the rows, four at a time.  The sums go to a slice of part, or to dbias where
// there is one batch range; both are null when no bias gradient is wanted.
template <typename T, int VEC, bool ACT>
__global__ __launch_bounds__(256) void ks_act_bwd_bf_kernel(const T *__restrict__ dy, const T *__restrict__ z, T *__restrict__ dz,
                                                            float *__restrict__ part, T *__restrict__ dbias, int64_t batch,
                                                            int64_t features, int lx, int col_blocks, int64_t rows)
{
    __shared__ float red[256 * VEC];
    const int split = blockIdx.x / col_blocks, cb = blockIdx.x - split * col_blocks;
    const int tx = threadIdx.x % lx, ty = threadIdx.x / lx, ly = 256 / lx;
    const int64_t col = ((int64_t)cb * lx + tx) * VEC;
    const int64_t r_end = min(batch, (split + 1) * rows);
    float sum[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) sum[e] = 0.f;
    if (col < features) {  // (VEC divides the features)
        auto some = [&](int64_t r, auto count) {
            constexpr int U = decltype(count)::value;
            Vec<T, VEC> g[U], h[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                g[u] = vload<T, VEC>(dy + (r + u * ly) * features + col);
                if (ACT) h[u] = vload<T, VEC>(z + (r + u * ly) * features + col);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                Vec<T, VEC> o;
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const float v = slope_times<T, ACT>((float)g[u].v[e], ACT ? h[u].v[e] : T(0));
                    sum[e] += v;
                    o.v[e] = (T)v;
                }
                if (ACT) vstore<T, VEC>(dz + (r + u * ly) * features + col, o);
            }
        };
        int64_t r = split * rows + ty;
        for (; r + 3 * ly < r_end; r += 4 * ly) some(r, std::integral_constant<int, 4>());
        for (; r < r_end; r += ly) some(r, std::integral_constant<int, 1>());
    }
    if (!part && !dbias) return;
    // element e of all threads side by side: no two lanes of a wave share a bank
#pragma unroll
    for (int e = 0; e < VEC; ++e) red[e * 256 + threadIdx.x] = sum[e];
    __syncthreads();
    for (int i = threadIdx.x; i < lx * VEC; i += 256) {
        const int64_t at = (int64_t)cb * lx * VEC + i;
        if (at >= features) continue;
        const int e = i % VEC, x = i / VEC;
        float s = 0.f;
        for (int y = 0; y < ly; ++y) s += red[e * 256 + y * lx + x];
        if (dbias) dbias[at] = (T)s;
        else part[split * features + at] = s;
    }
}

// Batch-size-last (features x batch).  One wavefront per feature and batch range.  The vectors lie on
// the tensor's 16-byte grid, not on the row's: only the first and the last of a row can hold elements
// of its neighbours, and these two go element by element.
template <typename T, int VEC, bool ACT>
__global__ __launch_bounds__(256) void ks_act_bwd_bl_kernel(const T *__restrict__ dy, const T *__restrict__ z, T *__restrict__ dz,
                                                            float *__restrict__ part, T *__restrict__ dbias, int64_t batch,
                                                            int64_t features, int splits, int64_t cols)
{
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int64_t f = wave / splits, split = wave - f * splits;
    if (f >= features) return;
    const int64_t row0 = f * batch, row1 = row0 + batch;
    // in units of VEC, on the tensor's grid (cols: vectors per split)
    const int64_t v0 = row0 / VEC + split * cols, v1 = min((row1 + VEC - 1) / VEC, v0 + cols);
    float sum = 0.f;
    auto some = [&](int64_t v, auto count) {
        constexpr int U = decltype(count)::value;
        Vec<T, VEC> g[U], h[U];
        bool full[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t at = (v + 64 * u) * VEC;
            full[u] = at >= row0 && at + VEC <= row1;
            if (full[u]) {
                g[u] = vload<T, VEC>(dy + at);
                if (ACT) h[u] = vload<T, VEC>(z + at);
            } else {
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const bool in = at + e >= row0 && at + e < row1;
                    g[u].v[e] = in ? dy[at + e] : T(0);
                    if (ACT) h[u].v[e] = in ? z[at + e] : T(0);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t at = (v + 64 * u) * VEC;
            Vec<T, VEC> o;
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                const float d = slope_times<T, ACT>((float)g[u].v[e], ACT ? h[u].v[e] : T(0));
                sum += d;
                o.v[e] = (T)d;
            }
            if (!ACT) continue;
            if (full[u]) {
                vstore<T, VEC>(dz + at, o);
            } else {
#pragma unroll
                for (int e = 0; e < VEC; ++e)
                    if (at + e >= row0 && at + e < row1) dz[at + e] = o.v[e];
            }
        }
    };
    int64_t v = v0 + lane;
    for (; v + 192 < v1; v += 256) some(v, std::integral_constant<int, 4>());
    for (; v < v1; v += 64) some(v, std::integral_constant<int, 1>());
    if (!part && !dbias) return;
#pragma unroll
    for (int s = 32; s; s >>= 1) sum += __shfl_xor(sum, s, 64);
    if (lane) return;
    if (dbias) dbias[f] = (T)sum;
    else part[split * features + f] = sum;
}

struct ActBwd {
    int lx, col_blocks;  // batch-size-first
    int64_t splits, size;  // batch ranges; rows (batch-size-first) or vectors (batch-size-last) of each
};

ActBwd plan(int64_t batch, int64_t features, int vec, bool bs_last)
{
    ActBwd p;
    if (bs_last) {
        // enough waves for 32 a CU; eight vectors a lane, so that the 4-byte sums stay below the traffic
        const int64_t vecs = (batch + vec - 1) / vec + 1;  // a row touches one more than it fills
        p.lx = p.col_blocks = 0;
        p.splits = (8192 + features - 1) / features;
        if (p.splits > (vecs + 511) / 512) p.splits = (vecs + 511) / 512;
        p.size = (vecs + p.splits - 1) / p.splits;
        p.splits = (vecs + p.size - 1) / p.size;
        return p;
    }
    // the widest row of lanes that wastes the fewest of them
    const int64_t vecs = features / vec;
    p.lx = 64;
    for (int l = 32; l >= 8; l >>= 1)
        if ((vecs + l - 1) / l * l < (vecs + p.lx - 1) / p.lx * p.lx) p.lx = l;
    p.col_blocks = (int)((vecs + p.lx - 1) / p.lx);
    const int64_t ly = 256 / p.lx;
    // eight workgroups a CU, eight rows a thread
    p.splits = (2048 + p.col_blocks - 1) / p.col_blocks;
    const int64_t most = (batch + 8 * ly - 1) / (8 * ly);
    if (p.splits > most) p.splits = most;
    p.size = (batch + p.splits - 1) / p.splits;
    p.splits = (batch + p.size - 1) / p.size;
    return p;
}

// Elements per access: 16 bytes where the rows (batch-size-first) and addresses allow it, else a word,
// else one element.
int vec_of(uintptr_t addresses, int64_t features, int dtype, bool bs_last)
{
    const int size = (int)dtype_size(dtype);
    for (int bytes = 16; bytes > size; bytes = bytes == 16 ? 4 : size)
        if (addresses % bytes == 0 && (bs_last || features * size % bytes == 0)) return bytes / size;
    return 1;
}

template <typename T, int VEC, bool ACT>
int launch(const void *dy, const void *z, void *dz, float *part, void *dbias, int64_t batch, int64_t features, const ActBwd &p, bool bs_last,
           hipStream_t s)
{
    const int64_t blocks = bs_last ? (features * p.splits + 3) / 4 : p.splits * p.col_blocks;
    if (blocks > 0x7fffffffLL) return KSMM_ERR_TOO_LARGE;
    if (bs_last)
        hipLaunchKernelGGL((ks_act_bwd_bl_kernel<T, VEC, ACT>), dim3((unsigned)blocks), dim3(256), 0, s, (const T *)dy, (const T *)z,
                           (T *)dz, part, (T *)dbias, batch, features, (int)p.splits, p.size);
    else
        hipLaunchKernelGGL((ks_act_bwd_bf_kernel<T, VEC, ACT>), dim3((unsigned)blocks), dim3(256), 0, s, (const T *)dy, (const T *)z,
                           (T *)dz, part, (T *)dbias, batch, features, p.lx, p.col_blocks, p.size);
    return hipGetLastError() == hipSuccess ? KSMM_OK : KSMM_ERR_LAUNCH;
}

template <typename T, bool ACT>
int launch_vec(int vec, const void *dy, const void *z, void *dz, float *part, void *dbias, int64_t batch, int64_t features, const ActBwd &p,
               bool bs_last, hipStream_t s)
{
    constexpr int WIDE = 16 / sizeof(T), WORD = 4 / sizeof(T);
    if (vec == WIDE) return launch<T, WIDE, ACT>(dy, z, dz, part, dbias, batch, features, p, bs_last, s);
    if (vec == WORD) return launch<T, WORD, ACT>(dy, z, dz, part, dbias, batch, features, p, bs_last, s);
    return launch<T, 1, ACT>(dy, z, dz, part, dbias, batch, features, p, bs_last, s);
}

}  // namespace

int64_t act_bwd_partial_floats(int64_t batch, int64_t features, int dtype, int bs_last)
{
    int64_t most = 1;
    for (int bytes : {16, 4, 2}) {
        const int vec = bytes / (int)dtype_size(dtype);
        if (vec < 1 || (!bs_last && features % vec != 0)) continue;
        const int64_t n = plan(batch, features, vec, bs_last).splits;
        if (n > most) most = n;
    }
    return most * features;
}

int act_bwd_run(const void *dy, const void *z, void *dz, void *dbias, float *acc, int64_t batch, int64_t features, int dtype,
                int bs_last, int act, hipStream_t stream, FinishJob *rest)
{
    const bool on = act != KSMM_ACT_NONE;
    const uintptr_t at = (uintptr_t)dy | (on ? (uintptr_t)z | (uintptr_t)dz : 0);
    const int vec = vec_of(at, features, dtype, bs_last);
    const ActBwd p = plan(batch, features, vec, bs_last);
    float *part = dbias && p.splits > 1 ? acc : nullptr;
    void *one = p.splits == 1 ? dbias : nullptr;
    int rc;
    if (dtype == KSMM_F32)
        rc = on ? launch_vec<float, true>(vec, dy, z, dz, part, one, batch, features, p, bs_last, stream)
                : launch_vec<float, false>(vec, dy, z, dz, part, one, batch, features, p, bs_last, stream);
    else
        rc = on ? launch_vec<half_t, true>(vec, dy, z, dz, part, one, batch, features, p, bs_last, stream)
                : launch_vec<half_t, false>(vec, dy, z, dz, part, one, batch, features, p, bs_last, stream);
    *rest = FinishJob{acc, dbias, features, part ? (int)p.splits : 0, 1.f};
    return rc;
}

}  // namespace ksmm
