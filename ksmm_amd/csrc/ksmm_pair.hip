// Two factors in one launch for small batches: y = act(K1 (K0 x) + bias), either layout, all types.
//
// A layer of two factors on a few hundred rows is two launches of 4 to 7 us, each a chain of loads, sums and stores
// around a product that takes the matrix cores less than a microsecond.  Here a workgroup owns 16 NT batch columns and
// 64 MG outputs of DG neighbouring blocks d_i of the second factor, and computes the inputs these need itself: all outputs
// of the first factor that feed block a_i, into LDS as DG planes [d_i][column][c_i] in the type that the intermediate has in
// memory.  The first factor is so repeated by every workgroup of a batch tile: its weights are read from L2 again and
// its products done again, which small batches can afford and large ones cannot (pair_us).
//  * Operands come straight from global memory (ksmm_direct.h): a lane holds four consecutive outputs of a weight row, so
//    lane (r, q) ends up with 16 consecutive outputs of column r, whole vectors of a plane.
//  * The waves take 64-output tiles of the first factor in turn, then a share of c of one (64 outputs, d_i) each; their
//    first weights of the second factor are requested before the first factor is begun.
//  * The sums of a tile's waves meet in LDS in the lane order of the accumulators, as in the split-K kernel.
//
// What bounds it: a launch (2.0 us of a replay with an empty kernel), one latency for the first loads and 16 cycles per
// load instruction, whatever its width: hence four outputs a lane and not two (those: 10.3 for 9.4 us where c0 is 256).
// Eight waves of up to 256 registers: sixteen of 128 spill, 7.9 against 6.4 us.  us of a replay, two launches / this one:
// (6,64,64,1)+(1,768,192,2) + GELU, 196 rows: fp16 9.8 / 7.1, fp32 13.5 / 9.4, e4m3 10.1 / 6.5, feature-major 9.0 / 6.8,
// 10.1 / 9.6, 8.6 / 6.0; on weights and inputs that no cache holds fp16 9.9 / 7.7, fp32 15.6 / 10.8; (12,64,64,1)+(1,1536,384,2) 14.3 / 11.4, 18.9 / 17.5, 13.8 / 9.5.  A call costs the host 2 us less as well.
#include "ksmm_direct.h"
#include "ksmm_pair.h"

#include <type_traits>

namespace ksmm {

namespace {

struct PairArgs {
    int batch;
    int a0, b0, c0;  // d0 = 1
    int a1, b1, c1, d1;
    int m_tiles, d_groups, tiles;  // tiles = a1 * d_groups * m_tiles
    int mg, ks;
    int lds_parts;  // byte offset of the partial sums
    float scale0;
    const float *x_scale;
};

constexpr int PAIR_WAVES = 8, PAIR_LDS = 160 * 1024;

template <typename TX, typename TW, typename TY, bool LAST, int NT, int DG>
__global__ __launch_bounds__(64 * PAIR_WAVES) void ks_pair_kernel(const TX *__restrict__ x, const TW *__restrict__ w0,
                                                                      const TW *__restrict__ w1, TY *__restrict__ y, PairArgs s, Epi ep)
{
    typedef typename op_type<TX>::type op_t;
    constexpr bool F32 = sizeof(op_t) == 4;
    constexpr int KV = F32 ? 4 : 8, KSTEP = 4 * KV, TN = 16 * NT, WAVES = PAIR_WAVES;
    typedef op_t opv_t __attribute__((ext_vector_type(KV)));
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    op_t *const h = (op_t *)smem;
    float *const part = (float *)(smem + s.lds_parts);
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = blockIdx.x % s.tiles, nt = blockIdx.x / s.tiles;
    const int mt = t % s.m_tiles, ag = t / s.m_tiles, dg = ag % s.d_groups, a_i = ag / s.d_groups;
    const int m0 = mt * 64 * s.mg, n0 = nt * TN, d0 = dg * DG;
    const int ldh = s.c1 + KV;  // (16 bytes more: the rows of an operand read start on different banks)
    const int ncol = LAST ? min(n0 + NT * r, s.batch - NT) : 0;
    uint32_t xo0[LAST ? 1 : NT];
    if constexpr (LAST) {
        xo0[0] = ((uint32_t)(KV * q) * (uint32_t)s.batch + (uint32_t)ncol) * (uint32_t)sizeof(TX);
    } else {
#pragma unroll
        for (int j = 0; j < NT; ++j)
            xo0[j] = ((uint32_t)min(n0 + 16 * j + r, s.batch - 1) * (uint32_t)(s.a0 * s.c0) + (uint32_t)(KV * q)) * (uint32_t)sizeof(TX);
    }

    // VM consecutive outputs of a weight row a lane: MFMA tile i has the outputs VM r + i, lane (r, q) ends up with
    // 4 VM consecutive ones of a column
    auto multiply = [&](auto &wv, const opv_t (&xo)[NT], auto &acc) {
        constexpr int VM = sizeof(acc) / sizeof(acc[0]);
        if constexpr (F32) {
#pragma unroll
            for (int k = 0; k < KV; ++k)
#pragma unroll
                for (int i = 0; i < VM; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, wv[k].v[i]), xo[j][k], acc[i][j], 0, 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < VM; ++i) {
                uint4_t wo;
#pragma unroll
                for (int k = 0; k < KV; k += 2) wo[k / 2] = pick16(wv[k], i, wv[k + 1], i);
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, wo), xo[j], acc[i][j], 0, 0, 0);
            }
        }
    };
    auto clear = [](auto &acc) {
        for (auto &row : acc)
            for (auto &v : row) v = float4_t{0.f, 0.f, 0.f, 0.f};
    };

    // the wave's share of the second factor: 64 outputs of one d_i, every ks-th step of c
    const int g = wave % DG, rest = wave / DG, mgi = rest % s.mg, slice = rest / s.mg;
    const bool busy = slice < s.ks;
    const int steps1 = s.c1 / KSTEP;
    const TW *const w1p = w1 + (size_t)(a_i * s.d1 + d0 + g) * s.c1 * s.b1;
    // (a uniform address and one 32-bit byte offset per lane for all loads)
    const uint32_t m1 = (uint32_t)(min(m0 + 64 * mgi + 4 * r, s.b1 - 4) + KV * q * s.b1) * (uint32_t)sizeof(TW);
    const uint32_t k1 = (uint32_t)(s.b1 * sizeof(TW)), k0b = (uint32_t)(s.b0 * sizeof(TW)), kx = LAST ? (uint32_t)s.batch * (uint32_t)sizeof(TX) : (uint32_t)sizeof(TX);
    rawn<TW, 4> next1[KV];
    auto load1 = [&](int step) {
#pragma unroll
        for (int k = 0; k < KV; ++k)
            next1[k] = load_n<TW, 4>(w1p, m1 + (uint32_t)(step * KSTEP + k) * k1);
    };
    load1(busy ? slice : 0);

    // first factor: 64 outputs of a block at a time
    constexpr int P = NT == 1 ? 2 : 1;  // steps of a batch of loads, two batches in flight
    const int blocks = s.c1 * s.d1 / s.b0, per = (s.b0 + 63) / 64, steps0 = s.c0 / KSTEP;
    float scale0 = s.scale0;
    if constexpr (sizeof(TX) == 1)
        if (s.x_scale) scale0 *= *s.x_scale;
    struct Batch {
        rawn<TW, 4> w[P][KV];
        rawn<TX, LAST ? NT : KV> x[P][LAST ? KV : NT];
    };
#pragma unroll 1
    for (int task = wave; task < blocks * per; task += WAVES) {
        const int blk = task / per, mt0 = task % per * 64, block = a_i * blocks + blk;
        const TW *const w0p = w0 + (size_t)block * s.c0 * s.b0;
        const uint32_t m = (uint32_t)(min(mt0 + 4 * r, s.b0 - 4) + KV * q * s.b0) * (uint32_t)sizeof(TW);
        const TX *xp = LAST ? x + (size_t)block * s.c0 * s.batch : x + (size_t)block * s.c0;
        // (behind the last step they repeat it: a branch around loads would make every wait a full one)
        auto load = [&](Batch &f, int step) {
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int k0 = min(step + p, steps0 - 1) * KSTEP;
#pragma unroll
                for (int k = 0; k < KV; ++k) f.w[p][k] = load_n<TW, 4>(w0p, m + (uint32_t)(k0 + k) * k0b);
                if constexpr (LAST) {
#pragma unroll
                    for (int k = 0; k < KV; ++k)
                        f.x[p][k] = load_n<TX, NT>(xp, xo0[0] + (uint32_t)(k0 + k) * kx);
                } else {
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        f.x[p][j] = load_n<TX, KV>(xp, xo0[j] + (uint32_t)k0 * kx);
                }
            }
        };
        float4_t acc[4][NT];
        clear(acc);
        auto products = [&](const Batch &f, int step) {
#pragma unroll
            for (int p = 0; p < P; ++p) {
                if (step + p >= steps0) break;
                opv_t xo[NT];
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    if constexpr (F32) {
#pragma unroll
                        for (int k = 0; k < KV; ++k) xo[j][k] = __builtin_bit_cast(float, LAST ? f.x[p][LAST ? k : 0].v[LAST ? j : 0] : f.x[p][LAST ? 0 : j].v[LAST ? 0 : k]);
                    } else {
                        uint4_t o;
#pragma unroll
                        for (int k = 0; k < KV; k += 2) {
                            if constexpr (LAST)
                                o[k / 2] = pick16(f.x[p][k], j, f.x[p][k + 1], j);
                            else
                                o[k / 2] = pair16(f.x[p][j], k);
                        }
                        xo[j] = __builtin_bit_cast(half8_t, o);
                    }
                }
                multiply(f.w[p], xo, acc);
            }
        };
        Batch fa, fb;
        load(fa, 0);
        if (steps0 <= P) {
            products(fa, 0);
        } else {
#pragma unroll 1
            for (int step = 0; step < steps0; step += 2 * P) {
                load(fb, step + P);
                products(fa, step);
                if (step + P >= steps0) break;
                load(fa, step + 2 * P);
                products(fb, step + P);
            }
        }
        // lane (r, q): outputs 16 q .. 16 q + 15 of column r, four from each e
        if (mt0 + 16 * q < s.b0) {
            const int f0 = blk * s.b0 + mt0 + 16 * q;
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                op_t *const row = h + (16 * j + r) * ldh;
                if (DG != 3 && s.d1 == DG) {
                    constexpr int D = DG == 3 ? 1 : DG, N = 16 / D;
                    typedef op_t run_t __attribute__((ext_vector_type(N)));
#pragma unroll
                    for (int dd = 0; dd < D; ++dd) {
                        run_t v;
#pragma unroll
                        for (int k = 0; k < N; ++k) v[k] = (op_t)(acc[(k * D + dd) & 3][j][(k * D + dd) >> 2] * scale0);
                        *(run_t *)(row + dd * TN * ldh + f0 / D) = v;
                    }
                } else {
                    int c_i = f0 / s.d1, dd = f0 - c_i * s.d1 - d0;
#pragma unroll
                    for (int k = 0; k < 16; ++k) {
                        if (dd >= 0 && dd < DG) row[dd * TN * ldh + c_i] = (op_t)(acc[k & 3][j][k >> 2] * scale0);
                        if (++dd == s.d1 - d0) dd = -d0, ++c_i;
                    }
                }
            }
        }
    }
    __syncthreads();

    float4_t acc[4][NT];
    clear(acc);
    if (busy) {
        const op_t *const plane = h + g * TN * ldh;
#pragma unroll 1
        for (int step = slice; step < steps1; step += s.ks) {
            rawn<TW, 4> now[KV];
#pragma unroll
            for (int k = 0; k < KV; ++k) now[k] = next1[k];
            load1(min(step + s.ks, steps1 - 1));
            opv_t xo[NT];
#pragma unroll
            for (int j = 0; j < NT; ++j) xo[j] = *(const opv_t *)(plane + (16 * j + r) * ldh + step * KSTEP + KV * q);
            multiply(now, xo, acc);
        }
    }
    // partial sums: [slice][group of 64][d_i][tile][e][lane]
    if (s.lds_parts == 0) __syncthreads();  // (in the place of the planes)
    if (busy) {
        float *const mine = part + (size_t)((slice * s.mg + mgi) * DG + g) * (4 * NT * 256) + lane;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) mine[((i * NT + j) * 4 + e) * 64] = acc[i][j][e];
    }
    __syncthreads();
    auto total = [&](int mi, int gi, int i, int j, int e) {
        const float *p = part + (size_t)(mi * DG + gi) * (4 * NT * 256) + ((i * NT + j) * 4 + e) * 64 + lane;
        float v = 0.f;
        for (int k = 0; k < s.ks; ++k) v += p[(size_t)k * s.mg * DG * 4 * NT * 256];
        return v;
    };
    if constexpr (LAST) {
        for (int item = wave; item < s.mg * DG * 16; item += WAVES) {
            const int e = item & 3, i = item >> 2 & 3, gi = (item >> 4) % DG, mi = (item >> 4) / DG;
            const int m = m0 + 64 * mi + 4 * (4 * q + e) + i;
            float v[NT];
#pragma unroll
            for (int j = 0; j < NT; ++j) v[j] = total(mi, gi, i, j, e);
            if (m < s.b1) {
                const size_t feature = (size_t)(a_i * s.b1 + m) * s.d1 + d0 + gi;
                const float bv = epi_bias<TY>(ep, feature);
                struct {
                    TY v[NT];
                } o;
#pragma unroll
                for (int j = 0; j < NT; ++j) o.v[j] = (TY)epi_finish(ep, v[j], bv);
                __builtin_memcpy(y + feature * s.batch + ncol, &o, sizeof(o));
            }
        }
    } else {
        // runs of IL outputs of DG blocks: short ones where there are few, for all waves to have some
        auto finish = [&](auto run) {
            constexpr int IL = decltype(run)::value, IG = 4 / IL;
            for (int item = wave; item < s.mg * 4 * NT * IG; item += WAVES) {
                const int e = item & 3, ig = (item >> 2) % IG, j = (item >> 2) / IG % NT, mi = (item >> 2) / IG / NT;
                const int m = m0 + 64 * mi + 4 * (4 * q + e) + IL * ig, n = n0 + 16 * j + r;
                const size_t feature = (size_t)(a_i * s.b1 + m) * s.d1 + d0;
                if (m >= s.b1 || n >= s.batch) continue;
                float v[IL][DG];
#pragma unroll
                for (int i = 0; i < IL; ++i)
#pragma unroll
                    for (int gi = 0; gi < DG; ++gi) v[i][gi] = epi_bias<TY>(ep, feature + i * s.d1 + gi);
                struct {
                    TY v[IL * DG];
                } o;
#pragma unroll
                for (int i = 0; i < IL; ++i)
#pragma unroll
                    for (int gi = 0; gi < DG; ++gi) o.v[i * DG + gi] = (TY)epi_finish(ep, total(mi, gi, IL * ig + i, j, e), v[i][gi]);
                TY *const yp = y + (size_t)n * ((size_t)s.a1 * s.b1 * s.d1) + feature;
                if (s.d1 == DG) {
                    __builtin_memcpy(yp, &o, sizeof(o));
                } else {
#pragma unroll
                    for (int i = 0; i < IL; ++i) __builtin_memcpy(yp + (size_t)i * s.d1, &o.v[i * DG], DG * sizeof(TY));
                }
            }
        };
        if (s.mg * NT < 4)
            finish(std::integral_constant<int, 1>{});
        else
            finish(std::integral_constant<int, 4>{});
    }
}

const void *pair_fn(int combo, int last, int nt, int dg)
{
#define PAIR_DG(TX_, TW_, TY_, LAST_, NT_)                                                                               \
    {                                                                                                                    \
        (const void *)&ks_pair_kernel<TX_, TW_, TY_, LAST_, NT_, 1>, (const void *)&ks_pair_kernel<TX_, TW_, TY_, LAST_, NT_, 2>, \
            (const void *)&ks_pair_kernel<TX_, TW_, TY_, LAST_, NT_, 3>, (const void *)&ks_pair_kernel<TX_, TW_, TY_, LAST_, NT_, 4> \
    }
#define PAIR_NT(TX_, TW_, TY_, LAST_) {PAIR_DG(TX_, TW_, TY_, LAST_, 1), PAIR_DG(TX_, TW_, TY_, LAST_, 2)}
#define PAIR_SET(TX_, TW_, TY_) {PAIR_NT(TX_, TW_, TY_, false), PAIR_NT(TX_, TW_, TY_, true)}
    static const void *const fns[4][2][2][4] = {PAIR_SET(float, float, float), PAIR_SET(half_t, half_t, half_t),
                                                PAIR_SET(fp8_t, fp8_t, half_t), PAIR_SET(half_t, fp8_t, half_t)};
    return fns[combo][last ? 1 : 0][nt - 1][dg - 1];
}

// What a chain and a shape come to; false: not for this kernel
struct PairPlan {
    int combo, dg, ks, lds, parts_at;
    int64_t m_tiles, tiles, grid;
};
bool pair_plan(const ksmm_factor_desc *f, int n, int64_t batch, int x_dtype, int y_dtype, int bs_last, const PairShape &s, PairPlan *p)
{
    if (n != 2 || f[0].w_dtype != f[1].w_dtype || f[0].d != 1) return false;
    p->combo = combo_of(x_dtype, f[0].w_dtype, y_dtype);
    if (p->combo < 0) return false;
    const int kstep = p->combo == 0 ? 16 : 32, hs = p->combo == 0 ? 4 : 2;
    const int b0 = f[0].b, c0 = f[0].c, b1 = f[1].b, c1 = f[1].c, d1 = f[1].d;
    if (b0 % 16 || b1 % 16 || c0 % kstep || c1 % kstep || (int64_t)c1 * d1 % b0) return false;
    if ((s.nt != 1 && s.nt != 2) || s.mg < 1 || (bs_last && batch < s.nt)) return false;
    p->dg = d1 <= 4 ? d1 : d1 % 4 == 0 ? 4 : d1 % 3 == 0 ? 3 : d1 % 2 == 0 ? 2 : 1;
    if (s.mg * p->dg > PAIR_WAVES) return false;
    // 32-bit byte offsets inside a block of weights and inside the input
    const int64_t xs = (int64_t)dtype_size(x_dtype), ws = (int64_t)dtype_size(f[0].w_dtype), limit = 0xffffffffLL;
    if ((int64_t)f[0].a * c0 * batch * xs > limit || (int64_t)b0 * c0 * ws > limit || (int64_t)b1 * c1 * ws > limit) return false;
    p->ks = PAIR_WAVES / (s.mg * p->dg);
    if (p->ks > c1 / kstep) p->ks = c1 / kstep;
    const int64_t planes = (int64_t)p->dg * 16 * s.nt * (c1 + 16 / hs) * hs;
    const int parts = p->ks * s.mg * p->dg * s.nt * 4096;  // at most 64 KB
    if (planes > PAIR_LDS) return false;
    const bool apart = planes + parts <= PAIR_LDS;
    p->parts_at = apart ? (int)planes : 0;
    p->lds = (int)(apart ? planes + parts : planes > parts ? planes : parts);
    p->m_tiles = (b1 + 64 * s.mg - 1) / (64 * s.mg);
    p->tiles = (int64_t)f[1].a * (d1 / p->dg) * p->m_tiles;
    p->grid = p->tiles * ((batch + 16 * s.nt - 1) / (16 * s.nt));
    return p->grid <= 0x7fffffffLL;
}

}  // namespace

// Predicted time in microseconds (< 0: the kernel does not take the chain, or no shape of it gives a single round of
// workgroups: with more of them the first factor is repeated too often) and the shape that takes it.
//     t = f . (1, p, q, l, l g, p nt, g, q nt, nt mg dg, r nt, z r nt, p g, q g)
//   p, q  steps that a wave does one after the other in the first and the second factor
//   l     load instructions of a workgroup / 100: sixteen cycles each, whatever their width
//   g     workgroups / 256
//   r     tasks that a wave does one after the other in the first factor: each writes its outputs to the planes,
//   z     element by element (1) unless the planes hold all d_i and these are not three (0)
// with non-negative coefficients fitted to 49600 replays below 25 us (16280 chains of feed-forward projections of widths 192 .. 1024
// and of drawn pairs of factors, 1 .. 3000 rows or columns): within 0.87 .. 1.11 for nine in ten.
float pair_us(const ksmm_factor_desc *f, int n, int64_t batch, int x_dtype, int y_dtype, int bs_last, PairShape *best)
{
    constexpr int TERMS = 13;
    static const float coef[3][2][TERMS] = {
        {{2.452f, 0.f, 0.f, 0.812f, 0.018f, 0.211f, 2.739f, 0.548f, 0.161f, 0.716f, 0.333f, 0.f, 0.f},
         {2.309f, 0.f, 0.f, 0.625f, 0.107f, 0.214f, 1.721f, 0.612f, 0.267f, 0.571f, 0.425f, 0.f, 0.f}},  // fp32
        {{3.461f, 0.f, 0.f, 0.880f, 0.161f, 0.034f, 1.415f, 0.071f, 0.175f, 0.133f, 0.493f, 0.125f, 0.f},
         {3.592f, 0.012f, 0.063f, 0.583f, 0.112f, 0.f, 0.661f, 0.064f, 0.274f, 0.064f, 0.426f, 0.151f, 0.f}},  // fp16
        {{3.410f, 0.f, 0.f, 0.376f, 0.235f, 0.071f, 1.250f, 0.142f, 0.143f, 0.198f, 0.579f, 0.021f, 0.f},
         {3.412f, 0.053f, 0.f, 0.314f, 0.f, 0.011f, 0.404f, 0.102f, 0.277f, 0.196f, 0.500f, 0.213f, 0.101f}},  // e4m3
    };
    float us = -1.f;
    for (int nt = 1; nt <= 2; ++nt)
        for (int mg = 1; mg <= 2; ++mg) {
            const PairShape s{nt, mg};
            PairPlan p;
            if (!pair_plan(f, n, batch, x_dtype, y_dtype, bs_last, s, &p) || p.grid > 256) continue;
            const int kv = p.combo == 0 ? 4 : 8, steps0 = f[0].c / (4 * kv), steps1 = f[1].c / (4 * kv);
            const int tasks = f[1].c * f[1].d / f[0].b * ((f[0].b + 63) / 64), rounds = (tasks + PAIR_WAVES - 1) / PAIR_WAVES;
            const float first = (float)(rounds * steps0), second = (float)((steps1 + p.ks - 1) / p.ks);
            const float loads = (float)(tasks * steps0 * (kv + (bs_last ? kv : nt)) + mg * p.dg * steps1 * kv) / 100.f;
            const float g = (float)p.grid / 256.f, put = (float)(rounds * nt);
            const float v[TERMS] = {1.f, first, second, loads, loads * g, first * nt, g, second * nt, (float)(nt * mg * p.dg),
                                    put, p.dg != 3 && f[1].d == p.dg ? 0.f : put, first * g, second * g};
            const float *c = coef[p.combo < 2 ? p.combo : 2][bs_last ? 1 : 0];
            float t = 0.f;
            for (int i = 0; i < TERMS; ++i) t += c[i] * v[i];
            if (us < 0.f || t < us) us = t, *best = s;
        }
    return us;
}

int pair_run(const ksmm_factor_desc *f, int n, const void *x, void *y, int64_t batch, int x_dtype, int y_dtype, int bs_last,
             const PairShape &shape, hipStream_t stream, const ksmm_epilogue *ep, const float *x_scale)
{
    PairPlan p;
    if (!pair_plan(f, n, batch, x_dtype, y_dtype, bs_last, shape, &p)) return KSMM_ERR_BAD_ALGO;
    const void *fn = pair_fn(p.combo, bs_last, shape.nt, p.dg);
    const int rc = ensure_dynamic_lds(fn, PAIR_LDS);
    if (rc != KSMM_OK) return rc;
    PairArgs s{(int)batch, f[0].a, f[0].b, f[0].c, f[1].a, f[1].b, f[1].c, f[1].d, (int)p.m_tiles, f[1].d / p.dg, (int)p.tiles,
               shape.mg, p.ks, p.parts_at, f[0].scale, x_scale};
    Epi e{f[1].scale, ep ? ep->act : KSMM_ACT_NONE, ep ? ep->bias : nullptr, nullptr};
    const void *w0 = f[0].w, *w1 = f[1].w;
    void *args[] = {(void *)&x, (void *)&w0, (void *)&w1, (void *)&y, &s, &e};
    return hipLaunchKernel(fn, dim3((unsigned)p.grid), dim3(64 * PAIR_WAVES), args, p.lds, stream) == hipSuccess ? KSMM_OK : KSMM_ERR_LAUNCH;
}

}  // namespace ksmm
