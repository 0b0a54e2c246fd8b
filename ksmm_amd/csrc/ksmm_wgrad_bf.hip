// Weight gradient of a Kronecker-sparse factor on batch-size-first tensors:
//   dW[a_i, m, k, d_i] = sum_n dY[n, (a_i b + m) d + d_i] * X[n, (a_i c + k) d + d_i]
// one (b x B) @ (B x c) product per (a_i, d_i) block, reduced over the rows n.
//
// The rows are the contiguous axis of neither operand, while the MFMA wants the elements of its sum
// side by side.  A thread therefore loads one 16-byte vector (N features) of N rows, transposes the
// N x N square in registers (16-bit types: one v_perm per output register; fp32: a renaming) and
// writes N vectors of N rows each into LDS rows that belong to one feature.  The features are sorted
// by block there, so any d works; batches of any length are cut by a test on the row, and vectors
// need element alignment only.
//
// A wavefront owns a 16T x 16T tile of one block's gradient; the waves of a workgroup are the d_i
// that share the loaded cache lines (all of them for d <= 8, eight otherwise), times the tiles of a
// block or the neighbouring blocks, up to four waves (more only where d asks for them).
//
// What bounds it: at full batches the latency of a slab (load, transpose, two barriers, or one: two_slabs()), three
// or four slabs of 16 KB in flight per CU; four waves a workgroup, three workgroups a CU.  Eight-wave
// workgroups read less through L2 but leave one workgroup a CU: 83 us instead of 52 on the second
// shape below.  128 registers a wave (four waves a SIMD) spill: 74 us.
// (fp16 blocks of 48 and more with d up to 4 or 6 have ksmm_wgrad_wide.hip.)
// Against transposed copies of both operands in HBM and the batch-size-last kernel on them, fp16 at
// 25088 rows: (1,768,192,2) 156 -> 52 us, (6,64,256,1) 90 -> 35, (1,128,128,3) 38 -> 23,
// (1,1536,384,2) 213 -> 157 (180 on another box), (1,16,16,64) 70 -> 46; fp32: 323 -> 200, 193 -> 72, 108 -> 52, 1083 -> 680, 148 -> 52.
#include <algorithm>

#include "ksmm_common.h"
#include "ksmm_wgrad_wide.h"

namespace ksmm {

namespace {

struct WgradBf {
    int64_t batch;
    int a, b, c, d;
    int ta, td, wm, wn;              // waves: ta blocks a_i x td of d_i x wm x wn tiles of a block
    int m_groups, n_groups, d_groups, a_groups;
    int splits;
    int64_t rows;                    // rows per split, a multiple of the slab
    int64_t slice;                   // a * b * c * d
    float scale;
};

template <typename T> struct wbf;
template <> struct wbf<float> {
    static constexpr int N = 4, U = 2;  // elements per vector, vector squares per thread
    typedef float4_t vec_t;
    // element e of every row's vector, as one vector over the rows
    __device__ static __forceinline__ uint4_t column(const uint4_t (&v)[4], int e) { return uint4_t{v[0][e], v[1][e], v[2][e], v[3][e]}; }
    __device__ static __forceinline__ float4_t mfma(float4_t a, float4_t b, float4_t c)
    {
#pragma unroll
        for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
        return c;
    }
};
template <> struct wbf<half_t> {
    static constexpr int N = 8, U = 1;
    typedef half8_t vec_t;
    __device__ static __forceinline__ uint4_t column(const uint4_t (&v)[8], int e)
    {
        const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
        uint4_t r;
#pragma unroll
        for (int p = 0; p < 4; ++p) r[p] = __builtin_amdgcn_perm(v[2 * p + 1][e >> 1], v[2 * p][e >> 1], sel);
        return r;
    }
    __device__ static __forceinline__ float4_t mfma(half8_t a, half8_t b, float4_t c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

// LDS position (in 16-byte units) of chunk `ch` of feature row `row`; CH chunks per row.  256 bytes
// (all 64 banks) hold 16 / CH rows: their 16 units are permuted by an XOR with a hash of the 256-byte
// block that differs for the blocks of 16 consecutive rows (the operand reads) and for rows 8 apart
// (the writes of neighbouring lanes at d = 1).
template <int CH> __device__ __forceinline__ int lds_unit(int row, int ch)
{
    const int u = row * CH + ch, blk = u >> 4;
    int h;
    if (CH == 4) h = (((blk >> 3) & 3) << 2) | ((blk ^ (blk >> 2)) & 3);
    else if (CH == 8) h = (((blk >> 6) & 1) << 3) | ((blk ^ (blk >> 3)) & 7);
    else h = (blk ^ (blk >> 4)) & 15;
    return (blk << 4) | ((u ^ h) & 15);
}

// acc_out: one slice of partial sums per split; dw (used when there is one split): the result.
// TWO: two slabs in LDS, see two_slabs()
template <typename T, int TT, int CH, bool TWO>
__global__ __launch_bounds__(512) void ks_wgrad_bf_kernel(const T *__restrict__ dy, const T *__restrict__ x,
                                                          float *__restrict__ acc_out, T *__restrict__ dw, WgradBf g)
{
    typedef wbf<T> V;
    typedef typename V::vec_t vec_t;
    constexpr int N = V::N, U = V::U, SLAB = CH * N, EDGE = 16 * TT;
    extern __shared__ __attribute__((aligned(16))) uint4_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;

    // workgroup -> (split, tile).  Workgroups go round the eight XCDs: with eight splits and more all
    // tiles of a split run on one of them and share its rows in that L2.
    const int tiles = g.a_groups * g.d_groups * g.m_groups * g.n_groups;
    int split, t;
    if (g.splits >= 8) {
        const int j = blockIdx.x >> 3;
        split = (blockIdx.x & 7) + 8 * (j / tiles);
        t = j % tiles;
    } else {
        split = blockIdx.x % g.splits;
        t = blockIdx.x / g.splits;
    }
    if (split >= g.splits) return;
    const int ng = t % g.n_groups;
    t /= g.n_groups;
    const int mg = t % g.m_groups;
    t /= g.m_groups;
    const int d0 = min((t % g.d_groups) * g.td, g.d - g.td), a0 = (t / g.d_groups) * g.ta;
    const int m0 = mg * g.wm * EDGE, k0 = ng * g.wn * EDGE;
    const int64_t n_begin = split * g.rows, n_end = min(g.batch, n_begin + g.rows);

    // ---- what this thread loads: U squares of N rows x N features ----
    const int rows_a = g.ta * g.td * g.wm * EDGE, rows_b = g.ta * g.td * g.wn * EDGE;  // LDS rows
    const bool whole = g.td == g.d;  // features of the tile are contiguous
    auto groups_of = [&](int size, int edge) {
        return g.ta > 1 ? (g.ta * size * g.d + N - 1) / N : (edge * g.td + N - 1) / N;
    };
    const int fga = groups_of(g.b, g.wm * EDGE), fgb = groups_of(g.c, g.wn * EDGE);
    const T *src[U];
    int pitch[U], left[U];  // row length; rows left in the split
    uint32_t dst[U][N / 2];  // two LDS units (of 16 bytes) each
    const int dump = (rows_a + rows_b) * CH;  // where features outside the tile go
#pragma unroll
    for (int u = 0; u < U; ++u) {
        int id = tid + u * blockDim.x;
        const bool second = id >= fga * CH;
        if (second) id -= fga * CH;
        const int fgs = second ? fgb : fga, size = second ? g.c : g.b, first = second ? k0 : m0;
        const int edge = (second ? g.wn : g.wm) * EDGE;
        const int rg = id / fgs, fg = id - rg * fgs;
        const bool used = rg < CH;
        const int width = g.a * size * g.d;
        int f0, base = 0, m = 0, dl = 0;
        if (whole) {
            base = (a0 * size + first) * g.d;
            f0 = min(base + N * fg, width - N);
        } else {
            m = fg / (8 / N);
            dl = (fg % (8 / N)) * N;
            f0 = (a0 * size + min(first + m, size - 1)) * g.d + d0 + dl;
        }
        pitch[u] = width;
        src[u] = (second ? x : dy) + (used ? n_begin + rg * N : n_begin) * width + f0;
        left[u] = used ? (int)(n_end - n_begin) - rg * N : 0;
#pragma unroll
        for (int e = 0; e < N; ++e) {
            int row;
            bool in = used;
            if (whole) {
                const int rel = f0 + e - base;
                int al = 0, rest = rel;
                if (g.ta > 1) {
                    al = rel / (size * g.d);
                    rest = rel - al * size * g.d;
                }
                const int mm = rest / g.d;
                in = in && rel >= 0 && al < g.ta && mm < edge;
                row = (al * g.td + (rest - mm * g.d)) * edge + mm;
            } else {
                row = (dl + e) * edge + m;
            }
            const uint32_t at = in ? lds_unit<CH>(row + (second ? rows_a : 0), rg) : dump;
            dst[u][e / 2] = e & 1 ? dst[u][e / 2] | (at << 16) : at;
        }
    }
    uint4_t v[U][N];
    auto load = [&]() {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const T *p = src[u];
            if (left[u] >= N) {
#pragma unroll
                for (int j = 0; j < N; ++j, p += pitch[u]) __builtin_memcpy(&v[u][j], p, 16);
            } else {
#pragma unroll
                for (int j = 0; j < N; ++j, p += pitch[u]) {
                    v[u][j] = uint4_t{0u, 0u, 0u, 0u};
                    if (j < left[u]) __builtin_memcpy(&v[u][j], p, 16);
                }
            }
            src[u] += (int64_t)SLAB * pitch[u];
            left[u] -= SLAB;
        }
    };

    // ---- this wave's tile ----
    int w = tid >> 6;
    const int wn = w % g.wn;
    w /= g.wn;
    const int wm = w % g.wm;
    w /= g.wm;
    const int dl = w % g.td, al = w / g.td;
    const int ra = (al * g.td + dl) * g.wm * EDGE + wm * EDGE + r, rb = rows_a + (al * g.td + dl) * g.wn * EDGE + wn * EDGE + r;
    float4_t acc[TT][TT];
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

    auto store = [&](uint4_t *to) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < N; ++e)
                to[e & 1 ? dst[u][e / 2] >> 16 : dst[u][e / 2] & 0xffffu] = V::column(v[u], e);
    };
    auto multiply = [&](const uint4_t *from) {
#pragma unroll
        for (int ks = 0; ks < CH / 4; ++ks) {
            int ua = ra, ub = rb;
            asm volatile("" : "+v"(ua), "+v"(ub));  // the positions are recomputed per slab: held, they would cost a wave per SIMD
            vec_t fa[TT];
#pragma unroll
            for (int i = 0; i < TT; ++i) fa[i] = __builtin_bit_cast(vec_t, from[lds_unit<CH>(ua + 16 * i, 4 * ks + q)]);
#pragma unroll
            for (int j = 0; j < TT; ++j) {
                const vec_t fb = __builtin_bit_cast(vec_t, from[lds_unit<CH>(ub + 16 * j, 4 * ks + q)]);
#pragma unroll
                for (int i = 0; i < TT; ++i) acc[i][j] = V::mfma(fa[i], fb, acc[i][j]);
            }
        }
    };

    load();
    if constexpr (TWO) {
        // one barrier a slab: the next one goes to the other buffer while other waves still multiply
        uint4_t *now = lds, *next = lds + dump + 1;
        store(now);
        if (n_begin + SLAB < n_end) load();
        __syncthreads();
        for (int64_t n = n_begin; n < n_end; n += SLAB) {
            multiply(now);
            if (n + SLAB < n_end) {
                store(next);
                if (n + 2 * SLAB < n_end) load();
            }
            __syncthreads();
            uint4_t *const was = now;
            now = next;
            next = was;
        }
    } else {
        for (int64_t n = n_begin; n < n_end; n += SLAB) {
            __syncthreads();  // the slab in LDS is consumed
            store(lds);
            __syncthreads();
            if (n + SLAB < n_end) load();
            multiply(lds);
        }
    }

    // ---- D: lane holds column (input k) r and rows (output m) 4q .. 4q + 3 of each 16 x 16 tile ----
    if (a0 + al >= g.a) return;
    const size_t block = (size_t)(a0 + al) * g.d + d0 + dl;
    float *out = acc_out + (size_t)split * g.slice;
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j) {
            const int k = k0 + wn * EDGE + 16 * j + r, m = m0 + wm * EDGE + 16 * i + 4 * q;
            if (k >= g.c) continue;
            const size_t at = (block * g.c + k) * g.b + m;
            if (g.splits == 1) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (m + e < g.b) dw[at + e] = (T)(acc[i][j][e] * g.scale);
            } else if ((g.b & 3) == 0 && m < g.b) {
                *(float4_t *)(out + at) = acc[i][j];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (m + e < g.b) out[at + e] = acc[i][j][e];
            }
        }
}

int vec_of(int dtype) { return 16 / (int)dtype_size(dtype); }

// edge of a wave's tile in units of 16: the smallest that holds a block, else 64 (48 where that
// divides the block and 64 does not)
int edge_of(int b, int c)
{
    return (b <= 16 && c <= 16) ? 1 : (b <= 32 && c <= 32) ? 2 : (b % 64 && c % 64 && b % 48 == 0 && c % 48 == 0) ? 3 : 4;
}
int chunks_of(int edge) { return edge == 1 ? 16 : edge == 2 ? 8 : 4; }

WgradBf plan(int64_t batch, int a, int b, int c, int d, int dtype, float scale)
{
    WgradBf g;
    g.batch = batch;
    g.a = a;
    g.b = b;
    g.c = c;
    g.d = d;
    g.scale = scale;
    g.slice = (int64_t)a * b * c * d;
    const int t = edge_of(b, c), edge = 16 * t, slab = chunks_of(t) * vec_of(dtype);
    const int mt = (b + edge - 1) / edge, nt = (c + edge - 1) / edge;
    g.td = d <= 8 ? d : 8;
    g.d_groups = (d + g.td - 1) / g.td;
    const int most = g.td < 4 ? 4 / g.td : 1;
    // the split of a workgroup's waves over a block's tiles that loads the fewest features
    g.wm = g.wn = 1;
    int64_t best = -1;
    for (int wm = 1; wm <= most && wm <= mt; ++wm)
        for (int wn = 1; wm * wn <= most && wn <= nt; ++wn) {
            const int64_t mgs = (mt + wm - 1) / wm, ngs = (nt + wn - 1) / wn, cost = mgs * ngs * (wm + wn);
            if (best < 0 || cost < best) {
                best = cost;
                g.wm = wm;
                g.wn = wn;
            }
        }
    // blocks of one tile: neighbouring blocks (contiguous features) fill the workgroup
    g.ta = 1;
    if (mt == 1 && nt == 1 && d <= 8)
        while (g.ta < a && (g.ta + 1) * g.td <= 4) ++g.ta;
    g.m_groups = (mt + g.wm - 1) / g.wm;
    g.n_groups = (nt + g.wn - 1) / g.wn;
    g.a_groups = (a + g.ta - 1) / g.ta;
    const int64_t tiles = (int64_t)g.a_groups * g.d_groups * g.m_groups * g.n_groups;
    const int waves = g.ta * g.td * g.wm * g.wn;
    // Enough row ranges for 12 waves a CU (fp16 (1,768,192,2) at 25088 rows: 57 us with 8, 52 with 12 and
    // 16), each at least 128 rows (fp32 64) or half that where there are few of them ((1,128,128,3) fp16:
    // 1576 rows 12.5 us against 12.9, 196 rows 10.9 against 9.5), and no more partial sums than the
    // operands have bytes or 24 MB, so that the finish kernel stays below the reduction itself.
    int64_t splits = (3072 / waves + tiles - 1) / tiles;
    int64_t least = batch <= 1024 ? 8 * vec_of(dtype) : 16 * vec_of(dtype);
    if (least < slab) least = slab;
    const int64_t by_rows = (batch + least - 1) / least;
    const int64_t bytes = batch * a * (b + c) * d * (int64_t)dtype_size(dtype);
    const int64_t by_traffic = (bytes > (24ll << 20) ? bytes : 24ll << 20) / (8 * g.slice);
    if (splits > by_traffic) splits = by_traffic;
    if (splits > by_rows) splits = by_rows;
    if (splits < 1) splits = 1;
    if (splits > 8) splits = (splits + 7) / 8 * 8;
    g.rows = (batch + splits - 1) / splits;
    g.rows = (g.rows + slab - 1) / slab * slab;
    g.splits = (int)((batch + g.rows - 1) / g.rows);
    return g;
}

// Tiles of 64 x 64 leave registers for twelve waves a CU: one workgroup of the five to eight that d asks for.  Nobody
// multiplies while that one waits at the two barriers of a slab, and LDS has room for a second slab: one barrier.  us with one
// and with two, 25088 rows: fp16 (2,96,384,8) 196 / 156, (1,192,192,32) 712 / 547, (2,64,64,6) 36.0 / 35.0, (1,100,70,5) 45.2 / 43.3;
// fp32, 12544 rows: 393 / 372, 747 / 677, 49.2 / 49.0, 77.6 / 75.2.  Where several workgroups share a CU they fill each other's
// waits and the second slab costs some of them their place: (1,512,512,2) 70.6 / 75, (16,64,64,1) 34.6 / 36.5, 48 x 48 tiles
// (1,48,48,16) 27.2 / 29.2; from 0.9 to 1.1 elsewhere.
constexpr bool two_slabs(int edge, int waves) { return edge == 4 && waves > 4; }

template <typename T, int TT, bool TWO> int launch(const void *dy, const void *x, float *acc, void *dw, const WgradBf &g, hipStream_t s)
{
    constexpr int CH = TT == 1 ? 16 : TT == 2 ? 8 : 4;
    const int64_t tiles = (int64_t)g.a_groups * g.d_groups * g.m_groups * g.n_groups;
    const int64_t blocks = g.splits >= 8 ? (int64_t)((g.splits + 7) / 8 * 8) * tiles : g.splits * tiles;
    if (blocks > 0x7fffffffLL) return KSMM_ERR_TOO_LARGE;
    const int lds = (TWO ? 2 : 1) * (g.ta * g.td * (g.wm + g.wn) * 16 * TT * CH + 1) * 16;
    constexpr int MOST = (TWO ? 2 : 1) * (8 * 2 * 16 * TT * CH + 1) * 16;  // eight waves (the limit is set once a kernel)
    const int rc = ensure_dynamic_lds((const void *)ks_wgrad_bf_kernel<T, TT, CH, TWO>, MOST);
    if (rc != KSMM_OK) return rc;
    hipLaunchKernelGGL((ks_wgrad_bf_kernel<T, TT, CH, TWO>), dim3((unsigned)blocks), dim3(64 * g.ta * g.td * g.wm * g.wn), lds, s,
                       (const T *)dy, (const T *)x, acc, (T *)dw, g);
    return hipGetLastError() == hipSuccess ? KSMM_OK : KSMM_ERR_LAUNCH;
}

template <typename T> int launch_edge(int t, const void *dy, const void *x, float *acc, void *dw, const WgradBf &g, hipStream_t s)
{
    switch (t) {
    case 1: return launch<T, 1, false>(dy, x, acc, dw, g, s);
    case 2: return launch<T, 2, false>(dy, x, acc, dw, g, s);
    case 3: return launch<T, 3, false>(dy, x, acc, dw, g, s);
    default:
        return two_slabs(t, g.ta * g.td * g.wm * g.wn) ? launch<T, 4, true>(dy, x, acc, dw, g, s) : launch<T, 4, false>(dy, x, acc, dw, g, s);
    }
}

}  // namespace

// Rows of at least one 16-byte vector on both sides (shorter ones stay on the tiled kernel).
bool wgrad_bf_ok(int a, int b, int c, int d, int dtype)
{
    return (dtype == KSMM_F32 || dtype == KSMM_F16) && (int64_t)a * b * d >= vec_of(dtype) && (int64_t)a * c * d >= vec_of(dtype);
}

int64_t wgrad_bf_partial_floats(int64_t batch, int a, int b, int c, int d, int dtype)
{
    // (which of the two kernels runs depends on the tensors' alignment)
    const WgradBf g = plan(batch, a, b, c, d, dtype, 1.f);
    return std::max(g.splits > 1 ? g.splits * g.slice : 0, wgrad_wide_partial_floats(batch, a, b, c, d, dtype));
}

// dw is complete when *splits is 1; otherwise acc holds *splits slices of partial sums.
int wgrad_bf_run(const void *dy, const void *x, void *dw, float *acc, int64_t batch, int a, int b, int c, int d, int dtype,
                 float scale, hipStream_t stream, int *splits)
{
    const int rc = wgrad_wide_run(dy, x, dw, acc, batch, a, b, c, d, dtype, scale, stream, splits);
    if (rc != KSMM_ERR_BAD_ALGO) return rc;
    const WgradBf g = plan(batch, a, b, c, d, dtype, scale);
    *splits = g.splits;
    const int t = edge_of(b, c);
    return dtype == KSMM_F32 ? launch_edge<float>(t, dy, x, acc, dw, g, stream) : launch_edge<half_t>(t, dy, x, acc, dw, g, stream);
}

}  // namespace ksmm
