// Weight gradient of a Kronecker-sparse factor on batch-size-first fp16 tensors, blocks of 48 and more with d up to 4 or 6:
//   dW[a_i, m, k, d_i] = sum_n dY[n, (a_i b + m) d + d_i] * X[n, (a_i c + k) d + d_i]
// A slab of rows n is staged as it lies, one plane of [n][features] per d_i and operand: a thread loads 8 features of all d_i of a
// row, d vectors in a row, sorts them by d_i (one v_perm per word, nothing at d = 1) and writes a vector into each plane.  The
// n that a MFMA wants side by side come from transpose loads (ds_read_b64_tr_b16), as for the weights of the GEMM tiles, whose
// swizzle the planes have.  A wave owns 64 x 64 of one d_i; on blocks of few tiles the waves share a tile and each takes
// every KS-th part of a slab, summed in LDS at the end, so that a workgroup still writes one tile of partial sums.
//
// What bounds it: the rate at which rows reach a workgroup, 38 to 46 bytes a ns and CU, which takes every slab's loads two slabs
// early and without a branch around them (with one, each wait was a wait for all: (1,768,192,2) at 25088 rows 80 us), and on small
// blocks the launch of the sum over the splits.  One workgroup a CU reaches it, so there are few splits, and big tiles read less.
// fp16, us with the sum, the kernel of ksmm_wgrad_bf.hip / this one at 25088 rows: (1,1536,384,2) 168 / 100 (35 would take the
// bytes), (1,768,192,2) 61 / 46, (6,64,256,1) 40 / 26.5, (6,64,64,1) 23 / 15.7, (1,128,128,3) 23.4 / 22.1, (1,96,96,4) 25.0 / 21.5;
// (1,768,192,2) at 3000 rows 25.5 / 17.0, (6,64,64,1) at 1000 11.2 / 8.3; (12,64,64,6) at 9000 64.5 / 46.3.  Over 28 shapes 1.31 times as fast in the geometric mean.
// That kernel keeps fp32, which waits for its matrix cores, other d, blocks below 48 and what no 16-byte vector divides.
#include <algorithm>
#include <type_traits>

#include "ksmm_swizzle.h"
#include "ksmm_wgrad_wide.h"

namespace ksmm {

namespace {

struct WideArgs {
    int64_t batch, rows, slice;  // rows per split, a multiple of the slab; a * b * c * d
    int a, b, c;
    int m_tiles, n_tiles, tiles, splits;
    float scale;
};

template <int DD, int TM, int TN, int KS, int SLAB> struct WideCfg {
    static constexpr int WM = TM / 64, WN = TN / 64, THREADS = 64 * DD * WM * WN * KS;
    static constexpr int AC = TM / 8, BC = TN / 8;                      // units of 8 features x DD of a row
    static constexpr int AR = THREADS / AC, BR = THREADS / BC;          // rows that all threads load at once, and how often
    static constexpr int AN = (SLAB + AR - 1) / AR, BN = (SLAB + BR - 1) / BR;
    static constexpr int A_PLANE = SLAB * TM * 2, B_PLANE = SLAB * TN * 2, B_OFF = DD * A_PLANE, STAGE = DD * (A_PLANE + B_PLANE);
    static constexpr int STEPS = SLAB / 16 / KS;                        // of 16 n, per wave and slab
    static constexpr int SUM = DD * WM * WN * (KS - 1) * 64 * 64 * 4;
    static constexpr int LDS_BYTES = 2 * STAGE > SUM ? 2 * STAGE : SUM;
    static_assert(AR % 4 == 0 && BR % 4 == 0, "the swizzle repeats every four rows");
    static_assert(SLAB % (16 * KS) == 0 && LDS_BYTES <= 160 * 1024, "slab");
};

template <int DD, int TM, int TN, int KS, int SLAB, int OCC>
__global__ __launch_bounds__(64 * DD * (TM / 64) * (TN / 64) * KS, OCC) void ks_wgrad_wide_kernel(const half_t *__restrict__ dy,
                                                                                                 const half_t *__restrict__ x,
                                                                                                 float *__restrict__ acc_out,
                                                                                                 half_t *__restrict__ dw, WideArgs g)
{
    typedef WideCfg<DD, TM, TN, KS, SLAB> C;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;

    // the tiles of a split run side by side on one XCD and share its rows in that L2
    const int blocks = g.splits * g.tiles, per_xcd = (blocks + 7) / 8, lid = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (lid >= blocks) return;
    const int split = lid / g.tiles, t = lid % g.tiles;
    const int k0 = t % g.n_tiles * TN, m0 = t / g.n_tiles % g.m_tiles * TM, a_i = t / (g.n_tiles * g.m_tiles);
    const int64_t n_begin = split * g.rows, n_end = min(g.batch, n_begin + g.rows);

    // ---- staging: units of 8 features (behind b and c: the last ones again) ----
    const int arow = tid / C::AC, ach = tid % C::AC, brow = tid / C::BC, bch = tid % C::BC;
    const int aw = g.a * g.b * DD, bw = g.a * g.c * DD;
    const half_t *as = dy + n_begin * aw, *bs = x + n_begin * bw;  // uniform: the slab's first row
    const uint32_t aoff = (uint32_t)(arow * aw + (a_i * g.b + min(m0 + 8 * ach, g.b - 8)) * DD) * 2;
    const uint32_t boff = (uint32_t)(brow * bw + (a_i * g.c + min(k0 + 8 * bch, g.c - 8)) * DD) * 2;
    const int adst = arow * (TM * 2) + ((ach ^ swz_outer<half_t, C::AC>(arow)) << 4);
    const int bdst = C::B_OFF + brow * (TN * 2) + ((bch ^ swz_outer<half_t, C::BC>(brow)) << 4);
    typedef uint4_t regs_t[C::AN + C::BN][DD];
    regs_t v0, v1;
    // rows of the slab that starts at row n of the split, the first `left` of which are there.  Whole slabs are loaded without a
    // branch (a thread whose row is behind the slab repeats the last one): behind loads that may have been passed by, a wait for
    // earlier ones is a wait for all.
    auto load = [&](regs_t &v, int n, int left, auto whole) {
        auto rows = [&](int count, int at, int each, int row, const half_t *p, int width, uint32_t off) {
#pragma unroll
            for (int i = 0; i < count; ++i) {
                const bool in = (i + 1) * each <= SLAB;
                const char *const q = (const char *)(p + (int64_t)n * width + (in ? (int64_t)i * each * width : 0));
                const uint32_t o = in ? off : off + (uint32_t)((min(row + i * each, SLAB - 1) - row) * width) * 2;
                if (!decltype(whole)::value) {
#pragma unroll
                    for (int j = 0; j < DD; ++j) v[at + i][j] = uint4_t{0u, 0u, 0u, 0u};
                }
                if (decltype(whole)::value || row + i * each < left) {
#pragma unroll
                    for (int j = 0; j < DD; ++j) v[at + i][j] = *(const uint4_t *)(q + o + 16 * j);
                }
            }
        };
        rows(C::AN, 0, C::AR, arow, as, aw, aoff);
        rows(C::BN, C::AN, C::BR, brow, bs, bw, boff);
    };
    auto store = [&](const regs_t &v, unsigned char *to) {
        auto rows = [&](int n, int at, int each, int row, int dst, int pitch, int plane) {
#pragma unroll
            for (int i = 0; i < n; ++i) {
                if ((i + 1) * each > SLAB && row + i * each >= SLAB) continue;
#pragma unroll
                for (int dd = 0; dd < DD; ++dd) {
                    uint4_t o;
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        const int e0 = 2 * p * DD + dd, e1 = (2 * p + 1) * DD + dd, w0 = e0 >> 1, w1 = e1 >> 1;
                        o[p] = DD == 1 ? v[at + i][0][p]
                                       : __builtin_amdgcn_perm(v[at + i][w1 >> 2][w1 & 3], v[at + i][w0 >> 2][w0 & 3],
                                                               ((e0 & 1) ? 0x0302u : 0x0100u) | ((e1 & 1) ? 0x07060000u : 0x05040000u));
                    }
                    *(uint4_t *)(to + dst + i * each * pitch + dd * plane) = o;
                }
            }
        };
        rows(C::AN, 0, C::AR, arow, adst, TM * 2, C::A_PLANE);
        rows(C::BN, C::AN, C::BR, brow, bdst, TN * 2, C::B_PLANE);
    };

    // ---- this wave's tile ----
    int w = tid >> 6;
    const int dd = w % DD;
    w /= DD;
    const int ks = w % KS;
    w /= KS;
    const int wm = w % C::WM, wn = w / C::WM;
    float16_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    uint32_t at_a[2], at_b[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        at_a[i] = base + dd * C::A_PLANE + ks * C::STEPS * 16 * (TM * 2) + outer_frag<half_t, TM>::off(wm * 64 + 32 * i, lane);
        at_b[i] = base + C::B_OFF + dd * C::B_PLANE + ks * C::STEPS * 16 * (TN * 2) + outer_frag<half_t, TN>::off(wn * 64 + 32 * i, lane);
    }
    auto multiply = [&](int buf) {
#pragma unroll
        for (int s = 0; s < C::STEPS; ++s) {
            half8_t fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                fa[i] = outer_frag<half_t, TM>::read(at_a[i] + buf * C::STAGE, 16 * s);
                fb[i] = outer_frag<half_t, TN>::read(at_b[i] + buf * C::STAGE, 16 * s);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = frag<half_t>::mfma(fa[i], fb[j], acc[i][j]);
        }
    };

    // two slabs in flight in registers, two in LDS, one barrier a slab (behind the last whole one it is loaded again, not used)
    const int rows = (int)(n_end - n_begin), slabs = rows / SLAB;
    auto next = [&](regs_t &v, int s) { load(v, min(s, slabs - 1) * SLAB, SLAB, std::true_type()); };
    if (slabs) {
        next(v0, 0);
        next(v1, 1);
        store(v0, smem);
        next(v0, 2);
        __syncthreads();
        for (int s = 0; s < slabs; s += 2) {
            multiply(0);
            store(v1, smem + C::STAGE);
            next(v1, s + 3);
            __syncthreads();
            if (s + 1 < slabs) multiply(1);
            store(v0, smem);
            next(v0, s + 4);
            __syncthreads();
        }
    }
    if (slabs * SLAB < rows) {
        load(v0, slabs * SLAB, rows - slabs * SLAB, std::false_type());
        store(v0, smem);
        __syncthreads();
        multiply(0);
        if (KS > 1) __syncthreads();
    }

    if constexpr (KS > 1) {
        float *const sum = (float *)smem + (size_t)(((wn * C::WM + wm) * DD + dd) * (KS - 1)) * 4096;
        if (ks) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) sum[(ks - 1) * 4096 + ((i * 2 + j) * 16 + e) * 64 + lane] = acc[i][j][e];
        }
        __syncthreads();
        if (ks) return;
#pragma unroll 1
        for (int q = 0; q < KS - 1; ++q)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[i][j][e] += sum[q * 4096 + ((i * 2 + j) * 16 + e) * 64 + lane];
    }

    // lane: column (input k) lane % 32, rows (output m) 8 eg + 4 (lane / 32) .. + 3 of each 32 x 32 tile
    const size_t block = (size_t)a_i * DD + dd;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int k = k0 + wn * 64 + 32 * j + (lane & 31);
        if (k >= g.c) continue;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int eg = 0; eg < 4; ++eg) {
                const int m = m0 + wm * 64 + 32 * i + 8 * eg + 4 * (lane >> 5);
                if (m >= g.b) continue;  // (b is a multiple of 8)
                const size_t at = (block * g.c + k) * g.b + m;
                const float4_t r = {acc[i][j][4 * eg], acc[i][j][4 * eg + 1], acc[i][j][4 * eg + 2], acc[i][j][4 * eg + 3]};
                if (g.splits == 1)
                    *(half4_t *)(dw + at) = half4_t{(half_t)(r[0] * g.scale), (half_t)(r[1] * g.scale), (half_t)(r[2] * g.scale), (half_t)(r[3] * g.scale)};
                else
                    *(float4_t *)(acc_out + (size_t)split * g.slice + at) = r;
            }
    }
}

struct WideInst {
    int dd, tm, tn, ks, slab, threads, lds;
    const void *fn;
};
#define WIDE_INST(DD_, TM_, TN_, KS_, SLAB_, OCC_)                                                                         \
    {DD_, TM_, TN_, KS_, SLAB_, WideCfg<DD_, TM_, TN_, KS_, SLAB_>::THREADS, WideCfg<DD_, TM_, TN_, KS_, SLAB_>::LDS_BYTES, \
     (const void *)ks_wgrad_wide_kernel<DD_, TM_, TN_, KS_, SLAB_, OCC_>}
const WideInst wide_insts[] = {
    WIDE_INST(1, 64, 64, 4, 64, 2), WIDE_INST(1, 128, 64, 4, 64, 2), WIDE_INST(1, 64, 128, 4, 64, 2), WIDE_INST(1, 128, 128, 2, 64, 2),
    WIDE_INST(2, 64, 64, 4, 64, 2), WIDE_INST(2, 128, 64, 2, 64, 2), WIDE_INST(2, 64, 128, 2, 64, 2), WIDE_INST(2, 128, 128, 1, 32, 2),
    WIDE_INST(3, 64, 64, 2, 96, 2), WIDE_INST(3, 128, 64, 1, 48, 2), WIDE_INST(3, 64, 128, 1, 48, 2),
    WIDE_INST(4, 64, 64, 2, 64, 2),
    // (d = 8: 0.56 to 0.77 of the other kernel's speed, its rows fill half of a load)
    WIDE_INST(6, 64, 64, 1, 32, 2),
};

struct WidePlan {
    const WideInst *inst;  // null: not taken
    WideArgs g;
};

WidePlan wide_plan(int64_t batch, int a, int b, int c, int d, int dtype, float scale)
{
    WidePlan p{};
    // (32-bit offsets inside a slab; slabs of three and more d_i take longer to fill than few rows take on the other kernel:
    // (1,128,128,3) on 196 rows 9.7 us there and 10.5 here, (1,64,256,4) on 777 12.1 and 12.4, (1,96,96,6) on 1100 13.8 and 14.1)
    if (batch < (d > 4 ? 2048 : d > 2 ? 1024 : 0)) return p;
    if (dtype != KSMM_F16 || d > 6 || b % 8 || c % 8 || b < 48 || c < 48 || (int64_t)a * (b > c ? b : c) * d > 1 << 24) return p;
    const int64_t slice = (int64_t)a * b * c * d, by_rows = batch <= 1024 ? (batch + 63) / 64 : (batch + 127) / 128;
    // The tile and the splits: 1 .. 4 rounds of a workgroup a CU, whose rows arrive at 42 bytes a ns, and partial sums written and
    // read at 5 TB/s
    double least = 0.;
    int64_t splits = 1;
    for (const WideInst &t : wide_insts) {
        if (t.dd != d) continue;
        const int64_t mt = (b + t.tm - 1) / t.tm, nt = (c + t.tn - 1) / t.tn, tiles = a * mt * nt;
        if (tiles > 1 << 20) continue;
        for (int r = 1; r <= 4; ++r) {
            const int64_t n = std::max<int64_t>(1, std::min<int64_t>(256 * r / tiles, by_rows)), rounds = (n * tiles + 255) / 256;
            const double us = (double)rounds * ((batch + n - 1) / n) * (t.tm + t.tn) * d * 2 / 42e3 + (double)n * slice * 8 / 5e6;
            if (p.inst && us >= least) continue;
            least = us;
            splits = n;
            p.inst = &t;
            p.g.m_tiles = (int)mt;
            p.g.n_tiles = (int)nt;
            p.g.tiles = (int)tiles;
        }
    }
    if (!p.inst) return p;
    WideArgs &g = p.g;
    g.batch = batch;
    g.a = a;
    g.b = b;
    g.c = c;
    g.slice = slice;
    g.scale = scale;
    g.rows = ((batch + splits - 1) / splits + p.inst->slab - 1) / p.inst->slab * p.inst->slab;
    g.splits = (int)((batch + g.rows - 1) / g.rows);
    return p;
}

}  // namespace

int64_t wgrad_wide_partial_floats(int64_t batch, int a, int b, int c, int d, int dtype)
{
    const WidePlan p = wide_plan(batch, a, b, c, d, dtype, 1.f);
    return !p.inst ? -1 : p.g.splits > 1 ? p.g.splits * p.g.slice : 0;
}

int wgrad_wide_run(const void *dy, const void *x, void *dw, float *acc, int64_t batch, int a, int b, int c, int d, int dtype, float scale,
                   hipStream_t stream, int *splits)
{
    if ((((uintptr_t)dy | (uintptr_t)x) & 15) || ((uintptr_t)dw & 7)) return KSMM_ERR_BAD_ALGO;
    WidePlan p = wide_plan(batch, a, b, c, d, dtype, scale);
    if (!p.inst) return KSMM_ERR_BAD_ALGO;
    *splits = p.g.splits;
    const int64_t blocks = ((int64_t)p.g.splits * p.g.tiles + 7) / 8 * 8;
    if (blocks > 0x7fffffffLL) return KSMM_ERR_TOO_LARGE;
    const int rc = ensure_dynamic_lds(p.inst->fn, p.inst->lds);
    if (rc != KSMM_OK) return rc;
    void *args[] = {(void *)&dy, (void *)&x, (void *)&acc, (void *)&dw, &p.g};
    return hipLaunchKernel(p.inst->fn, dim3((unsigned)blocks), dim3(p.inst->threads), args, p.inst->lds, stream) == hipSuccess ? KSMM_OK
                                                                                                                            : KSMM_ERR_LAUNCH;
}

}  // namespace ksmm
