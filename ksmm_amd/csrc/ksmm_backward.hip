// Backward pass of one Kronecker-sparse factor y = K x (forward: ksmm_factor_forward).
//
//   dX = K^T dY   is itself a KS factor: pattern (a, c, b, d) with every b x c block transposed,
//                 so it runs on the forward kernels once the blocks are transposed (ks_block_transpose_kernel)
//   dW[a_i, b_i, c_i, d_i] = sum_n dY[a_i, b_i, d_i, n] * X[a_i, c_i, d_i, n]
//                 one (b x B) @ (B x c) product per (a_i, d_i) block, reduced over the batch.
//                 Batch-size-last: MFMA kernels below (operand rows are batch-contiguous, so both
//                 operands come straight from global memory in MFMA layout); batch-size-first:
//                 ksmm_wgrad_bf.hip; rows shorter than a 16-byte vector: an LDS-tiled FMA kernel.
//                 Every batch split writes its partial sums to a slice of its own in the
//                 workspace, and a finish kernel adds the slices in a fixed order, scales, converts
//                 and writes kernel format (a*d*c, b): the result is the same bit for bit from run
//                 to run (no atomics).
//
// The reference has no backward pass (src/ksmm_py/layer/kronecker_sparse/kernel.py:319-329 refers
// to an undefined symbol; forward_bmm.py:12-15 is `pass`); the definition above is the adjoint of
// its forward product (interface.py:108-113).
#include "ksmm_common.h"

namespace ksmm {

namespace {

// out block g (b x c, c contiguous)  <-  in block g (c x b, b contiguous); both in "kernel format"
// of their own pattern: in = (a*d*c, b) of (a,b,c,d), out = (a*d*b, c) of (a,c,b,d).  One launch takes
// the weights of a whole layer.  A workgroup moves a 64 x 64 square through LDS, so that both sides are
// whole lines; few elements, and blocks that leave most of their squares empty, are moved an element a thread (their
// lines stay in the cache): a square each would be a workgroup per block, however small.  What bounds it is the launch.
struct TransposeArgs {
    struct {
        const void *in;
        void *out;
        int b, c, b_tiles, c_tiles;  // b_tiles 0: element by element
        uint32_t total;              // elements
        uint32_t first;              // the job's first workgroup
    } job[KSMM_MAX_FACTORS];
    int jobs;
};

template <typename T> __global__ __launch_bounds__(256) void ks_block_transpose_kernel(TransposeArgs t)
{
    __shared__ T square[64][64 + 4 / sizeof(T)];
    int k = 0;
    while (k + 1 < t.jobs && blockIdx.x >= t.job[k + 1].first) ++k;
    const int b = t.job[k].b, c = t.job[k].c, bt = t.job[k].b_tiles, ct = t.job[k].c_tiles;
    const T *in = (const T *)t.job[k].in;
    T *out = (T *)t.job[k].out;
    uint32_t id = blockIdx.x - t.job[k].first;
    if (bt == 0) {
        const uint32_t total = t.job[k].total, size = (uint32_t)b * c;  // (at most 2^31)
        const uint32_t at = id * 256 + threadIdx.x, g = at / size, rem = at - g * size;
        const uint32_t bi = rem / c, ci = rem - bi * c;
        if (at < total) out[at] = in[(size_t)g * size + ci * b + bi];
        return;
    }
    const int b0 = (int)(id % bt) * 64;
    id /= bt;
    const int c0 = (int)(id % ct) * 64;
    const size_t block = (size_t)(id / ct) * b * c;
    const int x = threadIdx.x & 63, y = threadIdx.x >> 6;
    T v[16];  // (every load in flight before the first is waited for: none is behind a branch)
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = in[block + (size_t)min(c0 + y + 4 * i, c - 1) * b + min(b0 + x, b - 1)];
#pragma unroll
    for (int i = 0; i < 16; ++i) square[y + 4 * i][x] = v[i];
    __syncthreads();
    if (c0 + x < c)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (b0 + y + 4 * i < b) out[block + (size_t)(b0 + y + 4 * i) * c + c0 + x] = square[x][y + 4 * i];
}

// out[i] = scale * (sum of the slices); slices are n floats apart.  One launch takes all the sums of a
// layer's backward pass: weight gradients and the bias's.  A workgroup's G groups of 256 / G threads add a
// G-th of the slices each, in slice order, for V outputs a thread, and the G partial sums are added
// in group order: the association is fixed by (splits) alone, so the result has the same bits
// on every run.  What bounds it: the latency of a thread's loads, so eight are in flight, the last few
// slices among them, and many slices (a bias gradient's: few outputs) are shared by more groups; the launch
// itself where the slices are few.
struct FinishArgs {
    struct {
        const float *acc;
        void *out;
        int64_t n;
        int splits;
        float scale;
        uint32_t first;  // the job's first workgroup
    } job[KSMM_MAX_FACTORS + 1];
    int jobs;
};

template <int V> struct FinishVec {
    float v[V];
};
template <typename T, int G, int V>
__device__ __forceinline__ void finish_part(const float *__restrict__ acc, T *__restrict__ out, int64_t n, int splits, float scale,
                                            uint32_t block, float *part)
{
    constexpr int LANES = 256 / G;
    const int g = threadIdx.x / LANES, l = threadIdx.x % LANES;
    const int64_t i = ((int64_t)block * LANES + l) * V;
    const int per = (splits + G - 1) / G, k0 = g * per, k1 = min(k0 + per, splits);
    float s[V];
#pragma unroll
    for (int e = 0; e < V; ++e) s[e] = 0.f;
    if (i < n) {  // (V divides n)
        for (int k = k0; k < k1; k += 8) {
            FinishVec<V> v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (k + j < k1) __builtin_memcpy(&v[j], __builtin_assume_aligned(acc + (int64_t)(k + j) * n + i, 4 * V), 4 * V);
                else v[j] = FinishVec<V>{};
            }
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int e = 0; e < V; ++e) s[e] += v[j].v[e];
        }
    }
#pragma unroll
    for (int e = 0; e < V; ++e) part[(e * G + g) * LANES + l] = s[e];
    __syncthreads();
    if (g || i >= n) return;
#pragma unroll
    for (int e = 0; e < V; ++e) {
#pragma unroll
        for (int k = 1; k < G; ++k) s[e] += part[(e * G + k) * LANES + l];
        out[i + e] = (T)(s[e] * scale);
    }
}

// where the slices are shared by 16 groups: four have more than one round of loads each
__host__ __device__ inline bool finish_wide(int splits) { return splits > 32; }
// outputs per workgroup: a vector of four a thread where that divides n (slices stay aligned)
__host__ __device__ inline int finish_outputs(int64_t n, int splits) { return (finish_wide(splits) ? 16 : 64) * (n % 4 == 0 ? 4 : 1); }

template <typename T> __global__ __launch_bounds__(256) void ks_finish_kernel(FinishArgs f)
{
    __shared__ float part[4 * 256];
    int k = 0;
    while (k + 1 < f.jobs && blockIdx.x >= f.job[k + 1].first) ++k;
    const float *acc = f.job[k].acc;
    T *out = (T *)f.job[k].out;
    const int64_t n = f.job[k].n;
    const int splits = f.job[k].splits;
    const float scale = f.job[k].scale;
    const uint32_t block = blockIdx.x - f.job[k].first;
    if (n % 4 == 0) {
        if (finish_wide(splits)) finish_part<T, 16, 4>(acc, out, n, splits, scale, block, part);
        else finish_part<T, 4, 4>(acc, out, n, splits, scale, block, part);
    } else {
        if (finish_wide(splits)) finish_part<T, 16, 1>(acc, out, n, splits, scale, block, part);
        else finish_part<T, 4, 1>(acc, out, n, splits, scale, block, part);
    }
}

// One 16-byte vector; ANY: at element alignment.  fp16 vectors at odd elements come as aligned words
// that are shifted into place (a 2-byte aligned vector load takes about twice as long); no word is
// read that does not hold one of the elements.
template <bool NTL, bool ANY, typename V, typename T> __device__ __forceinline__ V wg_load(const T *p)
{
    if (ANY && sizeof(T) == 2) {
        const uintptr_t at = (uintptr_t)p;
        const uint32_t *w = (const uint32_t *)(at & ~(uintptr_t)3);
        const uint32_t odd = (uint32_t)at & 2;
        uint4_t v;
        __builtin_memcpy(&v, w, 16);
        const uint32_t last = w[odd ? 4 : 3];
        v = uint4_t{__builtin_amdgcn_alignbyte(v[1], v[0], odd), __builtin_amdgcn_alignbyte(v[2], v[1], odd),
                    __builtin_amdgcn_alignbyte(v[3], v[2], odd), __builtin_amdgcn_alignbyte(last, v[3], odd)};
        return __builtin_bit_cast(V, v);
    }
    if (ANY) {
        V v;
        __builtin_memcpy(&v, p, sizeof(V));
        return v;
    }
    return NTL ? __builtin_nontemporal_load((const V *)p) : *(const V *)p;
}

template <typename T> struct wg_vec;
template <> struct wg_vec<float> {
    static constexpr int N = 4, MFMAS = 4;  // elements per 16-byte load; MFMAs fed by one load pair
    typedef float4_t type;
    __device__ static __forceinline__ float4_t mfma(int e, float4_t a, float4_t b, float4_t c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
    }
};
template <> struct wg_vec<half_t> {
    static constexpr int N = 8, MFMAS = 2;
    typedef half8_t type;
    __device__ static __forceinline__ float4_t mfma(int e, half8_t a, half8_t b, float4_t c)
    {
        const half4_t ah = {a[4 * e], a[4 * e + 1], a[4 * e + 2], a[4 * e + 3]};
        const half4_t bh = {b[4 * e], b[4 * e + 1], b[4 * e + 2], b[4 * e + 3]};
        return __builtin_amdgcn_mfma_f32_16x16x16f16(ah, bh, c, 0, 0, 0);
    }
};

// Batch-size-last blocks of at most 16 MT x 16 MT.  One wavefront owns one block's gradient and a range of batch columns.  Lane
// (r = lane % 16, q = lane / 16) loads N consecutive batch elements of operand rows r + 16 i at column n + N*q; MFMA e
// multiplies element group e of every lane, i.e. its k-set is {n + N*q + e ...}: the same set for
// both operands, and the order of a sum's terms is free.  NTL: non-temporal loads, every operand row is read by one wave.
// ANY: rows of any length and alignment (a batch that the vector does not divide): vectors at element
// alignment, and the last one of a row pulled back to end with it, its first elements cleared where
// the vector before has them.
template <typename T, int MT, bool NTL, bool ANY>
__global__ __launch_bounds__(256) void ks_wgrad_bl_kernel(const T *__restrict__ dy, const T *__restrict__ x,
                                                          float *__restrict__ acc_out, int batch, int a, int b,
                                                          int c, int d, int splits, int cols_per_split, int64_t slice)
{
    typedef wg_vec<T> V;
    constexpr int STEP = 4 * V::N;  // batch columns per step (4 lane groups)
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int split = (int)(wave % splits);
    const int64_t g = wave / splits;
    if (g >= (int64_t)a * d) return;
    const int a_i = (int)(g / d), d_i = (int)(g - (int64_t)a_i * d);
    const int n_begin = split * cols_per_split, n_end = min(batch, n_begin + cols_per_split);
    if (n_begin >= n_end) return;
    const size_t row_stride = (size_t)d * batch;
    // rows behind b (or c) are clamped to the last valid one and dropped at the end
    const T *ap[MT], *bp[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        ap[i] = dy + ((size_t)a_i * b * d + d_i) * batch + (size_t)min(16 * i + r, b - 1) * row_stride;
        bp[i] = x + ((size_t)a_i * c * d + d_i) * batch + (size_t)min(16 * i + r, c - 1) * row_stride;
    }
    float4_t acc[MT][MT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    typedef typename V::type vec_t;
    // U sub-steps per iteration, all their loads issued before the first MFMA: a row is then read
    // in runs of U * 64 bytes, and the loads of the whole iteration are in flight together
    constexpr int U = 4;
    for (int n = n_begin; n < n_end; n += U * STEP) {
        vec_t av[U][MT], bv[U][MT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int col = n + u * STEP + V::N * q;
            const bool live = col < n_end;          // whole vectors: batch and the split are multiples of N
            const int lcol = ANY ? min(col, batch - V::N) : live ? col : n_begin;  // (a valid address; the value is zeroed)
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                av[u][i] = wg_load<NTL, ANY, vec_t>(ap[i] + lcol);
                bv[u][i] = wg_load<NTL, ANY, vec_t>(bp[i] + lcol);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int col = n + u * STEP + V::N * q;
            if (ANY ? col + V::N > n_end : col >= n_end) {
                // elements in front of `drop` are not this vector's (n_end is the batch where ANY gets here with col < n_end)
                const int drop = ANY && col < n_end ? col - min(col, batch - V::N) : V::N;
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int e = 0; e < V::N; ++e) {
                        av[u][i][e] = e < drop ? (T)0 : av[u][i][e];
                        bv[u][i][e] = e < drop ? (T)0 : bv[u][i][e];
                    }
            }
#pragma unroll
            for (int e = 0; e < V::MFMAS; ++e)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < MT; ++j) acc[i][j] = V::mfma(e, av[u][i], bv[u][j], acc[i][j]);
        }
    }
    // D: lane holds column (c index) r and rows (b index) 4*q .. 4*q + 3 of each 16 x 16 tile
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        const int k = 16 * j + r;
        if (k >= c) continue;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = 16 * i + 4 * q + e;
                if (m < b) acc_out[(size_t)split * slice + ((size_t)g * c + k) * b + m] = acc[i][j][e];
            }
    }
}

// Any layout, any batch: 16 x 16 threads compute a 16 x 16 tile of one block's gradient over a
// batch range, staging 16 x 16 element tiles of both operands in LDS (fp32 FMAs).
template <typename T, bool BS_LAST>
__global__ __launch_bounds__(256) void ks_wgrad_tiled_kernel(const T *__restrict__ dy, const T *__restrict__ x,
                                                             float *__restrict__ acc_out, int64_t batch, int a,
                                                             int b, int c, int d, int m_tiles, int n_tiles,
                                                             int splits, int64_t cols_per_split, int64_t slice)
{
    __shared__ float sa[16][17], sb[16][17];
    int64_t t = blockIdx.x;
    const int split = (int)(t % splits);
    t /= splits;
    const int nt = (int)(t % n_tiles);
    t /= n_tiles;
    const int mt = (int)(t % m_tiles);
    const int64_t g = t / m_tiles;
    const int a_i = (int)(g / d), d_i = (int)(g - (int64_t)a_i * d);
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int64_t in_size = (int64_t)a * c * d, out_size = (int64_t)a * b * d;
    const int64_t n_begin = split * cols_per_split, n_end = min(batch, n_begin + cols_per_split);
    // staging: thread (ty, tx) loads operand row ty, batch element n + tx (batch-size-last: tx runs
    // along the contiguous axis) or row tx, batch element n + ty (batch-size-first: features contiguous)
    const int lrow = BS_LAST ? ty : tx, lcol = BS_LAST ? tx : ty;
    const int m_ld = mt * 16 + lrow, c_ld = nt * 16 + lrow;
    const int64_t fa = ((int64_t)a_i * b + min(m_ld, b - 1)) * d + d_i;  // feature of dY
    const int64_t fb = ((int64_t)a_i * c + min(c_ld, c - 1)) * d + d_i;  // feature of X
    float acc = 0.f;
    for (int64_t n = n_begin; n < n_end; n += 16) {
        const int64_t nn = n + lcol;
        float va = 0.f, vb = 0.f;
        if (nn < n_end) {
            va = elem<T>::load(BS_LAST ? dy + fa * batch + nn : dy + nn * out_size + fa);
            vb = elem<T>::load(BS_LAST ? x + fb * batch + nn : x + nn * in_size + fb);
        }
        sa[lrow][lcol] = va;
        sb[lrow][lcol] = vb;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 16; ++k) acc += sa[tx][k] * sb[ty][k];
        __syncthreads();
    }
    const int m = mt * 16 + tx, cc = nt * 16 + ty;  // consecutive threads: consecutive b_i (contiguous in dW)
    if (m < b && cc < c) acc_out[(size_t)split * slice + ((size_t)g * c + cc) * b + m] = acc;
}

// Weight gradient of blocks beyond 16 x 16 on batch-size-last operands: a TM x TN tile of one block's
// gradient and a range of batch columns per workgroup (4 waves, 2 x 2, on 32x32 MFMA tiles).  Both operands have the batch
// axis contiguous, so a slab is 128 bytes (64 columns in fp16, 32 in fp32) of TM + TN rows: it goes through registers into LDS
// (16-byte chunks, the chunk index XORed with row / 2 so that the operand reads of 16 consecutive rows hit different
// banks), double-buffered, one barrier per slab.  fp32: a lane's chunk is four of the sum's elements, one for each of
// four MFMAs, the same four for both operands.  D = X-rows x dY-rows^T, so a lane holds one output feature m (contiguous in
// kernel format) and 16 inputs k.  Rows behind b (or c) repeat the last valid one and are dropped at the end.
// What bounds it: in fp32 the matrix cores (at half their rate); in fp16 the latency of a slab, two to five workgroups of 32
// to 64 KB on a CU.  With the sums of the slices, us / us before, where a wave per 64 x 64 tile loaded its operands itself
// (one batch of loads in flight, every row read once a tile; fp16 multiples of 128 had the 128 x 128 tile): 25088 columns
// fp16 (1,768,192,2) 123 / 41, (6,64,256,1) 60 / 28, (1,1536,384,2) 133 / 101; fp32 237 / 146; 6272 columns fp32
// (1,768,192,2) 83 / 49, (6,64,64,1) 33 / 16; 197 columns (6,64,256,1) 28 / 10; (3,200,768,3) fp16 at 9850 337 / 95.
// ANY as in the kernel above.
template <typename T, int TM, int TN, bool ANY>
__global__ __launch_bounds__(256, 2) void ks_wgrad_gemm_kernel(const T *__restrict__ dy, const T *__restrict__ x,
                                                               float *__restrict__ acc_out, int batch, int a, int b, int c,
                                                               int d, int m_tiles, int n_tiles, int splits, int cols, int64_t slice)
{
    constexpr int N = wg_vec<T>::N, TK = 8 * N, VA = TM / 32, VB = TN / 32, MT = TM / 64, NT = TN / 64;
    extern __shared__ __attribute__((aligned(16))) uint4_t wg_lds[];  // [2][TM + TN rows][8 chunks]
    // an XCD takes an eighth of the workgroups, the tiles of a split side by side: they share its rows in that L2
    const int tiles = a * d * m_tiles * n_tiles, per_xcd = (tiles * splits + 7) / 8;
    const int lid = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (lid >= tiles * splits) return;
    const int split = lid / tiles;
    int id = lid - split * tiles;
    const int mt = id % m_tiles;
    id /= m_tiles;
    const int nt = id % n_tiles, g = id / n_tiles;
    const int a_i = g / d, d_i = g - a_i * d;
    const int m0 = mt * TM, n0 = nt * TN;
    const int k_begin = split * cols, k_end = min(k_begin + cols, batch);
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, lq = lane >> 5;
    const int wave = tid >> 6, wm = wave >> 1, wn = wave & 1;
    // staging: vector v = tid + 256 * i is row v / 8, physical chunk v % 8, which holds the logical
    // chunk (v % 8) ^ ((row / 2) % 8): the same one for all vectors of a thread
    const int row0 = tid >> 3, lc = ((tid & 7) ^ ((row0 >> 1) & 7)) * N;
    const T *ga[VA], *gb[VB];
#pragma unroll
    for (int i = 0; i < VA; ++i) ga[i] = dy + ((size_t)(a_i * b + min(m0 + row0 + 32 * i, b - 1)) * d + d_i) * batch;
#pragma unroll
    for (int i = 0; i < VB; ++i) gb[i] = x + ((size_t)(a_i * c + min(n0 + row0 + 32 * i, c - 1)) * d + d_i) * batch;
    uint4_t ra[VA], rb[VB];
    // (whole vectors of a row that the batch ends in, or the one that ends with it: a valid address, and no branch around
    // the loads; what is not of this slab is cleared on the way to LDS)
    auto gload = [&](int k) {
        const int col = min(k + lc, batch - N);
#pragma unroll
        for (int i = 0; i < VA; ++i) ra[i] = wg_load<false, ANY, uint4_t>(ga[i] + col);
#pragma unroll
        for (int i = 0; i < VB; ++i) rb[i] = wg_load<false, ANY, uint4_t>(gb[i] + col);
    };
    auto lstore = [&](uint4_t *to, int k) {
        if (k + TK > k_end) {
            // elements before `from` are not of this vector, those from `until` on not of this split
            const int col = k + lc, back = col - min(col, batch - N), from = min(back, N), until = min(max(k_end - col, 0) + from, N);
            auto keep = [&](uint4_t &v) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint32_t mask = 0u;
                    if constexpr (N == 8) {
                        if (2 * e >= from && 2 * e < until) mask |= 0xffffu;
                        if (2 * e + 1 >= from && 2 * e + 1 < until) mask |= 0xffff0000u;
                    } else if (e >= from && e < until) {
                        mask = 0xffffffffu;
                    }
                    v[e] &= mask;
                }
            };
#pragma unroll
            for (int i = 0; i < VA; ++i) keep(ra[i]);
#pragma unroll
            for (int i = 0; i < VB; ++i) keep(rb[i]);
        }
#pragma unroll
        for (int i = 0; i < VA; ++i) to[tid + 256 * i] = ra[i];
#pragma unroll
        for (int i = 0; i < VB; ++i) to[TM * 8 + tid + 256 * i] = rb[i];
    };
    float16_t acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    uint4_t *now = wg_lds, *next = wg_lds + (TM + TN) * 8;
    gload(k_begin);
    lstore(now, k_begin);
    __syncthreads();
    for (int k = k_begin; k < k_end; k += TK) {
        gload(k + TK);  // (behind the last slab: of the last columns, and not used)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            uint4_t fx[NT], fy[MT];
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                const int r = wn * (TN / 2) + i * 32 + l32;
                fx[i] = now[TM * 8 + r * 8 + ((2 * ks + lq) ^ ((r >> 1) & 7))];
            }
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                const int r = wm * (TM / 2) + j * 32 + l32;
                fy[j] = now[r * 8 + ((2 * ks + lq) ^ ((r >> 1) & 7))];
            }
#pragma unroll
            for (int e = 0; e < (N == 4 ? 4 : 1); ++e)
#pragma unroll
                for (int i = 0; i < NT; ++i)
#pragma unroll
                    for (int j = 0; j < MT; ++j) {
                        if constexpr (N == 4)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(float, (uint32_t)fx[i][e]),
                                                                             __builtin_bit_cast(float, (uint32_t)fy[j][e]), acc[i][j], 0, 0, 0);
                        else
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, fx[i]),
                                                                               __builtin_bit_cast(half8_t, fy[j]), acc[i][j], 0, 0, 0);
                    }
        }
        if (k + TK < k_end) lstore(next, k + TK);
        __syncthreads();
        uint4_t *const was = now;
        now = next;
        next = was;
    }
    // D[k'][m]: lane l32 = output feature m, rows k' = 8 * (e / 4) + 4 * lq + e % 4
    float *out = acc_out + (size_t)split * slice + (size_t)g * c * b;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int kk = n0 + wn * (TN / 2) + i * 32 + 8 * (e >> 2) + 4 * lq + (e & 3);
                const int m = m0 + wm * (TM / 2) + j * 32 + l32;
                if (kk < c && m < b) out[(size_t)kk * b + m] = acc[i][j][e];
            }
}

// Batch ranges: every one is non-empty and writes a slice of a*b*c*d partial sums of its own.
struct WgradSplit {
    int64_t splits, cols;
};
// `want` of them, of whole `step`s and at least `least` columns, and beyond `fill` no more partial sums (written, then read)
// than the operands have bytes or 24 MB
WgradSplit wgrad_split(int64_t batch, int a, int b, int c, int d, int dtype, int64_t want, int64_t fill, int64_t least, int64_t step)
{
    const int64_t bytes = batch * a * (b + c) * d * (int64_t)dtype_size(dtype), slice = (int64_t)a * b * c * d;
    const int64_t by_traffic = (bytes > (24ll << 20) ? bytes : 24ll << 20) / (8 * slice), by_cols = (batch + least - 1) / least;
    int64_t splits = want < by_cols ? want : by_cols;
    const int64_t most = by_traffic > fill ? by_traffic : fill;
    if (splits > most) splits = most;
    if (splits < 1) splits = 1;
    int64_t cols = (batch + splits - 1) / splits;
    cols = (cols + step - 1) / step * step;
    return WgradSplit{(batch + cols - 1) / cols, cols};
}

// Blocks of 16 x 16 leave fifteen sixteenths of the GEMM tile empty, and in fp32, which waits for its matrix cores, those of 32 x 32 cost
// three quarters of it: on 8670 drawn problems of 17 .. 32 rows the wave's kernel takes 0.85 of the tile's time, from 16 MB of
// operands on 0.6 to 0.7 (1.00 below 4 MB): (16,32,32,4) on 10538 columns 61 us / 44, (6,20,16,32) on 12579 202 / 93.  In fp16 it takes
// 1.01.  Beyond, the tile is ahead of waves with tiles of 32, 48 and 64 (us with those / on it): fp16 (1,32,32,32) at 25088 columns
// 37.4 / 26.3, (1,48,48,16) fp32 63.0 / 48.7 and fp16 32.9 / 22.3.
bool wgrad_gemm_ok(int b, int c, int dtype)
{
    const int edge = dtype == KSMM_F32 ? 32 : 16;
    return b > edge || c > edge;
}

// An edge of 128 where that pads the block by no more than a tenth beyond what 64 does
int wgrad_gemm_edge(int n)
{
    const int wide = (n + 127) / 128 * 128, narrow = (n + 63) / 64 * 64;
    return 10 * wide <= 11 * narrow ? 128 : 64;
}
// as many workgroups as the CUs' LDS has room for at once, of at least two slabs each; one a CU whatever the partial sums cost
WgradSplit wgrad_gemm_split(int64_t batch, int a, int b, int c, int d, int dtype)
{
    const int tm = wgrad_gemm_edge(b), tn = wgrad_gemm_edge(c), slab = 128 / (int)dtype_size(dtype);
    const int64_t tiles = (int64_t)a * d * ((b + tm - 1) / tm) * ((c + tn - 1) / tn), room = 256 * (tm + tn == 256 ? 2 : tm + tn == 192 ? 3 : 4);
    return wgrad_split(batch, a, b, c, d, dtype, room / tiles, (256 + tiles - 1) / tiles, 2 * slab, slab);
}

// about 16 waves per CU; at least 4 loop iterations per wave, or one where that leaves SIMDs without a wave
WgradSplit wgrad_bl_split(int64_t batch, int a, int b, int c, int d, int dtype)
{
    const int step = 16 * (16 / (int)dtype_size(dtype));  // columns per loop iteration (four sub-steps)
    const int64_t tiles = (int64_t)a * d;
    const int64_t long_ones = (batch + 4 * step - 1) / (4 * step);
    if (long_ones * tiles >= 1024) return wgrad_split(batch, a, b, c, d, dtype, (4096 + tiles - 1) / tiles, (1024 + tiles - 1) / tiles, 4 * step, step);
    return wgrad_split(batch, a, b, c, d, dtype, (1024 + tiles - 1) / tiles, 1, step, step);
}

void wgrad_tiled_splits(int64_t batch, int64_t tiles, int64_t *splits_out, int64_t *cols_out)
{
    int64_t splits = (2048 + tiles - 1) / tiles;
    const int64_t max_splits = (batch + 255) / 256;
    if (splits > max_splits) splits = max_splits;
    if (splits < 1) splits = 1;
    int64_t cols = (batch + splits - 1) / splits;
    cols = (cols + 15) / 16 * 16;
    *splits_out = (batch + cols - 1) / cols;
    *cols_out = cols;
}

// Batch-size-last with at least one vector per row.  Against the tiled kernel at 6501 columns, which
// the vector does not divide: (1,768,192,2) fp16 310 -> 58 us, fp32 310 -> 82.
bool wgrad_mfma_ok(int64_t batch, int dtype, int bs_last) { return bs_last && batch >= 16 / (int)dtype_size(dtype); }

// rows of whole, aligned vectors
bool wgrad_aligned(const void *dy, const void *x, int64_t batch, int dtype)
{
    return batch % (16 / (int)dtype_size(dtype)) == 0 && ((((uintptr_t)dy | (uintptr_t)x) & 15) == 0);
}

template <typename T>
int launch_wgrad_bl(const void *dy, const void *x, float *acc, int64_t batch, int a, int b, int c, int d,
                    hipStream_t s, int *splits_used)
{
    const auto [splits, cols] = wgrad_bl_split(batch, a, b, c, d, elem<T>::dtype);
    const int64_t waves = (int64_t)a * d * splits, blocks = (waves + 3) / 4;
    if (blocks > 0x7fffffffLL) return KSMM_ERR_TOO_LARGE;
    *splits_used = (int)splits;
    const bool whole = wgrad_aligned(dy, x, batch, elem<T>::dtype);
    auto fn = whole ? &ks_wgrad_bl_kernel<T, 1, true, false> : &ks_wgrad_bl_kernel<T, 1, false, true>;
    if constexpr (sizeof(T) == 4)
        // (plain loads: 0.93 of the time of non-temporal ones)
        if (b > 16 || c > 16) fn = whole ? &ks_wgrad_bl_kernel<T, 2, false, false> : &ks_wgrad_bl_kernel<T, 2, false, true>;
    hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(256), 0, s, (const T *)dy, (const T *)x, acc, (int)batch, a, b, c, d,
                       (int)splits, (int)cols, (int64_t)a * b * c * d);
    return hipGetLastError() == hipSuccess ? KSMM_OK : KSMM_ERR_LAUNCH;
}

template <typename T>
int launch_wgrad_tiled(const void *dy, const void *x, float *acc, int64_t batch, int a, int b, int c, int d,
                       int bs_last, hipStream_t s, int *splits_used)
{
    const int m_tiles = (b + 15) / 16, n_tiles = (c + 15) / 16;
    const int64_t tiles = (int64_t)a * d * m_tiles * n_tiles;
    int64_t splits, cols;
    wgrad_tiled_splits(batch, tiles, &splits, &cols);
    const int64_t blocks = tiles * splits;
    if (blocks > 0x7fffffffLL) return KSMM_ERR_TOO_LARGE;
    *splits_used = (int)splits;
    const int64_t slice = (int64_t)a * b * c * d;
    if (bs_last)
        hipLaunchKernelGGL((ks_wgrad_tiled_kernel<T, true>), dim3((unsigned)blocks), dim3(256), 0, s, (const T *)dy,
                           (const T *)x, acc, batch, a, b, c, d, m_tiles, n_tiles, (int)splits, cols, slice);
    else
        hipLaunchKernelGGL((ks_wgrad_tiled_kernel<T, false>), dim3((unsigned)blocks), dim3(256), 0, s, (const T *)dy,
                           (const T *)x, acc, batch, a, b, c, d, m_tiles, n_tiles, (int)splits, cols, slice);
    return hipGetLastError() == hipSuccess ? KSMM_OK : KSMM_ERR_LAUNCH;
}

template <typename T, int TM, int TN>
int launch_wgrad_gemm_tile(const void *dy, const void *x, float *acc, int64_t batch, int a, int b, int c, int d,
                           hipStream_t s, int *splits_used)
{
    const int m_tiles = (b + TM - 1) / TM, n_tiles = (c + TN - 1) / TN;
    const int64_t tiles = (int64_t)a * d * m_tiles * n_tiles;
    const auto [splits, cols] = wgrad_gemm_split(batch, a, b, c, d, elem<T>::dtype);
    const int64_t blocks = (splits * tiles + 7) / 8 * 8;
    if (blocks > 0x7fffffffLL) return KSMM_ERR_TOO_LARGE;
    *splits_used = (int)splits;
    const auto fn = wgrad_aligned(dy, x, batch, elem<T>::dtype) ? &ks_wgrad_gemm_kernel<T, TM, TN, false> : &ks_wgrad_gemm_kernel<T, TM, TN, true>;
    const int lds = 2 * (TM + TN) * 128;
    hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(256), lds, s, (const T *)dy, (const T *)x, acc, (int)batch, a, b, c, d,
                       m_tiles, n_tiles, (int)splits, (int)cols, (int64_t)a * b * c * d);
    return hipGetLastError() == hipSuccess ? KSMM_OK : KSMM_ERR_LAUNCH;
}
template <typename T>
int launch_wgrad_gemm(const void *dy, const void *x, float *acc, int64_t batch, int a, int b, int c, int d,
                      hipStream_t s, int *splits_used)
{
    const int tm = wgrad_gemm_edge(b), tn = wgrad_gemm_edge(c);
    const auto fn = tm == 128 ? (tn == 128 ? launch_wgrad_gemm_tile<T, 128, 128> : launch_wgrad_gemm_tile<T, 128, 64>)
                              : (tn == 128 ? launch_wgrad_gemm_tile<T, 64, 128> : launch_wgrad_gemm_tile<T, 64, 64>);
    return fn(dy, x, acc, batch, a, b, c, d, s, splits_used);
}

// the batch-size-last kernels, and the one for rows shorter than a vector in either layout
template <typename T>
int wgrad_last(const void *dy, const void *x, float *acc, int64_t batch, int a, int b, int c, int d, int bs_last, hipStream_t s, int *splits)
{
    if (!wgrad_mfma_ok(batch, elem<T>::dtype, bs_last)) return launch_wgrad_tiled<T>(dy, x, acc, batch, a, b, c, d, bs_last, s, splits);
    return wgrad_gemm_ok(b, c, elem<T>::dtype) ? launch_wgrad_gemm<T>(dy, x, acc, batch, a, b, c, d, s, splits)
                               : launch_wgrad_bl<T>(dy, x, acc, batch, a, b, c, d, s, splits);
}

}  // namespace

// the b x c blocks of each job's w transposed: kernel format (a*d*b, c) of pattern (a, c, b, d)
int block_transpose_run(const TransposeJob *jobs, int n, int dtype, hipStream_t stream)
{
    TransposeArgs t;
    int64_t blocks = 0;
    t.jobs = n;
    for (int i = 0; i < n; ++i) {
        const TransposeJob &j = jobs[i];
        auto &o = t.job[i];
        o.in = j.w;
        o.out = j.wt;
        o.b = j.b;
        o.c = j.c;
        o.b_tiles = (j.b + 63) / 64;
        o.c_tiles = (j.c + 63) / 64;
        o.first = (uint32_t)blocks;
        const int64_t total = j.blocks * j.b * j.c, squares = j.blocks * o.b_tiles * o.c_tiles;
        o.total = (uint32_t)total;
        // Element by element: squares that are filled to an eighth or less, and few elements, whose time is the latency of
        // one workgroup.  dX of 16 rows in fp16, us with squares / by elements: (1,2,2,131072) 166 / 19, (64,16,16,64)
        // 14.7 / 10.6, (6,64,64,1) 6.5 / 5.6, (1,192,192,2) 9.5 / 8.4, (1,512,512,1) 8.5 / 8.3, but (1,512,512,2)
        // 11.7 / 12.5, (16,64,64,16) 8.9 / 10.3, (6,192,192,16) 19 / 28.
        if (total <= squares * 512 || total <= 1 << 18) o.b_tiles = 0;
        blocks += o.b_tiles ? squares : (total + 255) / 256;
        if (blocks > 0x7fffffffLL) return KSMM_ERR_TOO_LARGE;
    }
    if (n < 1) return KSMM_OK;
    if (dtype == KSMM_F32)
        hipLaunchKernelGGL((ks_block_transpose_kernel<float>), dim3((unsigned)blocks), dim3(256), 0, stream, t);
    else
        hipLaunchKernelGGL((ks_block_transpose_kernel<half_t>), dim3((unsigned)blocks), dim3(256), 0, stream, t);
    return hipGetLastError() == hipSuccess ? KSMM_OK : KSMM_ERR_LAUNCH;
}

// Floats of partial sums the weight gradient of this problem writes (slices of a*b*c*d, one per
// batch split), whichever kernel takes it: the largest of the kernels' needs.
int64_t wgrad_partial_floats(int64_t batch, int a, int b, int c, int d, int dtype, int bs_last)
{
    if (!bs_last && wgrad_bf_ok(a, b, c, d, dtype)) return wgrad_bf_partial_floats(batch, a, b, c, d, dtype);
    const int64_t n = (int64_t)a * b * c * d;
    int64_t cols, most = 1;
    if (wgrad_mfma_ok(batch, dtype, bs_last))
        most = (wgrad_gemm_ok(b, c, dtype) ? wgrad_gemm_split : wgrad_bl_split)(batch, a, b, c, d, dtype).splits;
    else
        wgrad_tiled_splits(batch, (int64_t)a * d * ((b + 15) / 16) * ((c + 15) / 16), &most, &cols);
    return most * n;
}

// out[i] (type `dtype`, i < n) of each job <- scale * the sum of its slices of n floats
int finish_run(const FinishJob *jobs, int n, int dtype, hipStream_t stream)
{
    FinishArgs f;
    int64_t blocks = 0;
    f.jobs = 0;
    for (int i = 0; i < n; ++i) {
        const FinishJob &j = jobs[i];
        if (j.splits < 1) continue;  // complete already
        auto &o = f.job[f.jobs++];
        o.acc = j.acc;
        o.out = j.out;
        o.n = j.n;
        o.splits = j.splits;
        o.scale = j.scale;
        o.first = (uint32_t)blocks;
        const int64_t per = finish_outputs(j.n, j.splits);
        blocks += (j.n + per - 1) / per;
        if (blocks > 0x7fffffffLL) return KSMM_ERR_TOO_LARGE;
    }
    if (f.jobs < 1) return KSMM_OK;
    if (dtype == KSMM_F32)
        hipLaunchKernelGGL((ks_finish_kernel<float>), dim3((unsigned)blocks), dim3(256), 0, stream, f);
    else
        hipLaunchKernelGGL((ks_finish_kernel<half_t>), dim3((unsigned)blocks), dim3(256), 0, stream, f);
    return hipGetLastError() == hipSuccess ? KSMM_OK : KSMM_ERR_LAUNCH;
}

// dw (kernel format, type `dtype`) <- scale * sum over the batch of dY x X^T per block; acc is an
// fp32 buffer of wgrad_partial_floats() elements.  dw is complete once *rest has been finished.
int wgrad_run(const void *dy, const void *x, void *dw, float *acc, int64_t batch, int a, int b, int c, int d,
              int dtype, int bs_last, float scale, hipStream_t stream, FinishJob *rest)
{
    const int64_t n = (int64_t)a * b * c * d;
    int rc, splits = 1;
    *rest = FinishJob{acc, dw, n, 0, scale};
    if (!bs_last && wgrad_bf_ok(a, b, c, d, dtype)) {
        rc = wgrad_bf_run(dy, x, dw, acc, batch, a, b, c, d, dtype, scale, stream, &splits);
        if (rc != KSMM_OK || splits == 1) return rc;
    } else if (dtype == KSMM_F32) {
        rc = wgrad_last<float>(dy, x, acc, batch, a, b, c, d, bs_last, stream, &splits);
    } else if (dtype == KSMM_F16) {
        rc = wgrad_last<half_t>(dy, x, acc, batch, a, b, c, d, bs_last, stream, &splits);
    } else {
        return KSMM_ERR_BAD_DTYPE;
    }
    rest->splits = splits;
    return rc;
}

}  // namespace ksmm
