// Split-K tiles for small and ragged batches: any b >= 4, any c, any d, any batch, both layouts.
//
// A layer called on a few hundred rows is bound by latency, not by bytes: the tiles tuned for
// full batches leave most of the chip idle there ((1,1536,384,2) on 196 rows is 8 workgroups of
// the 256 x 128 tile, each of which walks the whole of c).  This kernel cuts a problem into many
// small pieces instead and keeps each wave's chain of dependent loads short:
//  * a wave multiplies a (16 VM) x (16 NT) tile of DD neighbouring blocks over a share of c: the
//    waves of a workgroup take every KS-th step of 32 (fp32: 16) inputs, and their sums meet in
//    LDS, in the lane order of the accumulators (no bank conflicts, no transpose);
//  * operands come from global memory straight into MFMA registers.  A lane loads VM consecutive
//    outputs of a weight row (MFMA tile i holds rows m = VM r + i), so no LDS transpose is needed.
//    Inputs are NT consecutive columns (batch-size-last), a run of c (batch-size-first, d = 1) or
//    runs of DD neighbouring d_i (batch-size-first, d > 1: with DD = d a lane's inputs of a step are
//    one run of 8 d elements), which the registers then hold one operand per d_i from;
//  * the results of a lane are runs of NT columns or of VM x DD features and leave from registers;
//  * nothing needs an aligned row: vectors that would cross the end of a row start earlier
//    and repeat columns a neighbour has too (the same value is then written twice), so a
//    batch-size-last batch that no vector divides needs no padded copies.
#include "ksmm_direct.h"

namespace ksmm {

namespace {

struct SplitArgs {
    int batch, a, b, c, d;
    int m_tiles, n_tiles, d_groups, ks, tiles;  // tiles = a * d_groups * m_tiles
};

// most waves of a workgroup: the registers of one (sums, and two steps of operands in flight)
constexpr int split_waves(int vm, int nt, int dd) { return vm * nt * dd <= 4 ? 16 : vm * nt * dd <= 8 ? 8 : 4; }

// LAST: batch-size-last (DD = 1); else batch-size-first.  RUN: a lane's inputs of a step are one run
// of memory (batch-size-first, d = DD, c a multiple of KV)
template <typename TX, typename TW, typename TY, bool LAST, bool RUN, int VM, int NT, int DD>
__global__ __launch_bounds__(64 * split_waves(VM, NT, DD), 2) void ks_split_kernel(
    const TX *__restrict__ x, const TW *__restrict__ w, TY *__restrict__ y, SplitArgs s, Epi ep)
{
    epi_load<TX>(ep);
    typedef typename op_type<TX>::type op_t;
    constexpr bool F32 = sizeof(op_t) == 4;
    constexpr int KV = F32 ? 4 : 8, KSTEP = 4 * KV, TM = 16 * VM, TN = 16 * NT, TILES = VM * NT * DD;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    float *part = (float *)smem;  // [wave][tile][e][lane]
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int ki = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // batch tiles of one weight tile get ids that are equal mod 8: the XCD whose L2 holds the weights
    const int slot = blockIdx.x >> 3, nt = slot % s.n_tiles;
    const int t = (slot / s.n_tiles) * 8 + (blockIdx.x & 7);
    if (t >= s.tiles) return;
    const int mt = t % s.m_tiles, ag = t / s.m_tiles, dg = ag % s.d_groups, a_i = ag / s.d_groups;
    const int m0 = mt * TM, n0 = nt * TN, d0 = dg * DD;
    const int b = s.b, c = s.c, d = s.d;
    const TW *wp = w + (size_t)(a_i * d + d0) * c * b;
    const uint32_t wo0 = (uint32_t)min(m0 + VM * r, b - VM) * sizeof(TW), wk = (uint32_t)b * sizeof(TW);
    const uint32_t wd = wk * (uint32_t)c;  // bytes from the block of d_i to that of d_i + 1
    const int ncol = LAST ? min(n0 + NT * r, s.batch - NT) : 0;
    const TX *xp = LAST ? x + ((size_t)a_i * c * d + d0) * s.batch : x + (size_t)a_i * c * d + d0;
    uint32_t xo0[LAST ? 1 : NT];
    if constexpr (LAST) {
        xo0[0] = (uint32_t)ncol * sizeof(TX);
    } else {
#pragma unroll
        for (int j = 0; j < NT; ++j)
            xo0[j] = (uint32_t)min(n0 + 16 * j + r, s.batch - 1) * (uint32_t)(s.a * c * d) * (uint32_t)sizeof(TX);
    }
    const uint32_t xk = (uint32_t)d * (LAST ? (uint32_t)s.batch : 1u) * sizeof(TX);  // bytes from input k to k + 1

    struct Frag {
        rawn<TW, VM> wv[DD][KV];
        rawn<TX, LAST ? NT : RUN ? KV * DD : DD> xv[LAST || RUN ? 1 : NT][RUN ? NT : KV];  // RUN: [0][batch tile]
    };
    const int steps = (c + KSTEP - 1) / KSTEP;
    auto load = [&](Frag &f, int step) {
        const int k0 = step * KSTEP + KV * q;
        if constexpr (RUN) {
#pragma unroll
            for (int i = 0; i < NT; ++i)
                f.xv[0][i] = load_n<TX, KV * DD>(xp, xo0[i] + (uint32_t)min(k0, c - KV) * (uint32_t)(DD * sizeof(TX)));
        }
#pragma unroll
        for (int j = 0; j < KV; ++j) {
            const uint32_t k = (uint32_t)min(k0 + j, c - 1);
#pragma unroll
            for (int g = 0; g < DD; ++g) f.wv[g][j] = load_n<TW, VM>(wp, wo0 + k * wk + (uint32_t)g * wd);
            if constexpr (LAST) f.xv[0][j] = load_n<TX, NT>(xp, xo0[0] + k * xk);
            if constexpr (!LAST && !RUN) {
#pragma unroll
                for (int i = 0; i < NT; ++i) f.xv[i][j] = load_n<TX, DD>(xp, xo0[i] + k * xk);
            }
        }
    };
    float4_t acc[DD][VM][NT];
#pragma unroll
    for (int g = 0; g < DD; ++g)
#pragma unroll
        for (int i = 0; i < VM; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[g][i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const Frag &f, int step) {
        // inputs of this lane that exist: behind the last one both operands are cleared
        const bool tail = (step + 1) * KSTEP > c;
        const int left = c - step * KSTEP - KV * q;
#pragma unroll
        for (int g = 0; g < DD; ++g) {
            if constexpr (F32) {
#pragma unroll
                for (int k = 0; k < KV; ++k) {
                    float wo[VM], xo[NT];
#pragma unroll
                    for (int i = 0; i < VM; ++i) wo[i] = !tail || k < left ? __builtin_bit_cast(float, f.wv[g][k].v[i]) : 0.f;
#pragma unroll
                    for (int j = 0; j < NT; ++j) {
                        const uint32_t v = LAST ? f.xv[0][k].v[j] : RUN ? f.xv[0][RUN ? j : 0].v[k * DD + g] : f.xv[RUN ? 0 : j][k].v[g];
                        xo[j] = !tail || k < left ? __builtin_bit_cast(float, v) : 0.f;
                    }
#pragma unroll
                    for (int i = 0; i < VM; ++i)
#pragma unroll
                        for (int j = 0; j < NT; ++j)
                            acc[g][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wo[i], xo[j], acc[g][i][j], 0, 0, 0);
                }
            } else {
                uint4_t wo[VM], xo[NT];
#pragma unroll
                for (int k = 0; k < KV; k += 2) {
#pragma unroll
                    for (int i = 0; i < VM; ++i) wo[i][k / 2] = pick16(f.wv[g][k], i, f.wv[g][k + 1], i);
#pragma unroll
                    for (int j = 0; j < NT; ++j) {
                        if constexpr (LAST)
                            xo[j][k / 2] = pick16(f.xv[0][k], j, f.xv[0][k + 1], j);
                        else if constexpr (RUN)
                            xo[j][k / 2] = pick16(f.xv[0][j], k * DD + g, f.xv[0][j], (k + 1) * DD + g);
                        else
                            xo[j][k / 2] = pick16(f.xv[j][k], g, f.xv[j][k + 1], g);
                    }
                }
                if (tail) {
#pragma unroll
                    for (int k = 0; k < KV; k += 2) {
                        const uint32_t mask = k + 1 < left ? 0xffffffffu : k < left ? 0xffffu : 0u;
#pragma unroll
                        for (int i = 0; i < VM; ++i) wo[i][k / 2] &= mask;
#pragma unroll
                        for (int j = 0; j < NT; ++j) xo[j][k / 2] &= mask;
                    }
                }
#pragma unroll
                for (int i = 0; i < VM; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        acc[g][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, wo[i]),
                                                                              __builtin_bit_cast(half8_t, xo[j]),
                                                                              acc[g][i][j], 0, 0, 0);
            }
        }
    };
    // steps ki, ki + ks, ... (ks <= steps: every wave has one).  The loads of the next one are issued
    // before the products of this one (behind the last step they repeat it: a branch around loads
    // would make every wait a full one), except where two steps of operands would spill
    if constexpr (F32 || DD * VM < 16) {
        Frag cur, nxt;
        int step = ki;
        load(cur, step);
        if (s.ks < steps) {
            for (; step < steps; step += 2 * s.ks) {
                const int s1 = step + s.ks, s2 = s1 + s.ks;
                load(nxt, min(s1, steps - 1));
                multiply(cur, step);
                if (s1 >= steps) break;
                load(cur, min(s2, steps - 1));
                multiply(nxt, s1);
            }
        } else {
            multiply(cur, step);
        }
    } else {
        for (int step = ki; step < steps; step += s.ks) {
            Frag cur;
            load(cur, step);
            multiply(cur, step);
        }
    }
    // D of a 16 x 16 tile: lane (r, q) holds column r, rows 4 q .. 4 q + 3; row e of lane group q is
    // what lane 4 q + e loaded, i.e. outputs min(m0 + VM (4 q + e), b - VM) + i
    auto put = [&](int e, int j, const float (&v)[DD][VM]) {  // one run of a lane's results
        const int m = min(m0 + VM * (4 * q + e), b - VM);
        const int n = n0 + 16 * j + r;
        if (LAST || n < s.batch) {
            vecn<TY, VM * DD> o;
#pragma unroll
            for (int i = 0; i < VM; ++i)
#pragma unroll
                for (int g = 0; g < DD; ++g) {
                    const size_t feature = (size_t)(a_i * b + m + i) * d + d0 + g;
                    o.v[i * DD + g] = (TY)epi_finish(ep, v[g][i], epi_bias<TY>(ep, feature));
                }
            TY *yp = y + (size_t)n * ((size_t)s.a * b * d) + (size_t)(a_i * b + m) * d + d0;
            if (d == DD) {
                __builtin_memcpy(yp, &o, sizeof(o));
            } else {
#pragma unroll
                for (int i = 0; i < VM; ++i) __builtin_memcpy(yp + (size_t)i * d, &o.v[i * DD], DD * sizeof(TY));
            }
        }
    };
    auto put_last = [&](int e, int i, const float (&v)[NT]) {
        const int m = min(m0 + VM * (4 * q + e), b - VM) + i;
        const size_t feature = (size_t)(a_i * b + m) * d + d0;
        const float bv = epi_bias<TY>(ep, feature);
        vecn<TY, NT> o;
#pragma unroll
        for (int j = 0; j < NT; ++j) o.v[j] = (TY)epi_finish(ep, v[j], bv);
        __builtin_memcpy(y + feature * s.batch + ncol, &o, sizeof(o));
    };
    if (s.ks == 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if constexpr (LAST) {
#pragma unroll
                for (int i = 0; i < VM; ++i) {
                    float v[NT];
#pragma unroll
                    for (int j = 0; j < NT; ++j) v[j] = acc[0][i][j][e];
                    put_last(e, i, v);
                }
            } else {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    float v[DD][VM];
#pragma unroll
                    for (int g = 0; g < DD; ++g)
#pragma unroll
                        for (int i = 0; i < VM; ++i) v[g][i] = acc[g][i][j][e];
                    put(e, j, v);
                }
            }
        }
        return;
    }
    float *mine = part + (size_t)ki * TILES * 256 + lane;
#pragma unroll
    for (int g = 0; g < DD; ++g)
#pragma unroll
        for (int i = 0; i < VM; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) mine[(((g * VM + i) * NT + j) * 4 + e) * 64] = acc[g][i][j][e];
    __syncthreads();
    const float *sums = part + lane;
    auto total = [&](int tile, int e) {
        float v = 0.f;
        for (int k = 0; k < s.ks; ++k) v += sums[(size_t)k * TILES * 256 + (tile * 4 + e) * 64];
        return v;
    };
    // the runs of the tile are dealt to the waves
    if constexpr (LAST) {
        for (int item = ki; item < 4 * VM; item += s.ks) {
            const int e = item & 3, i = item >> 2;
            float v[NT];
#pragma unroll
            for (int j = 0; j < NT; ++j) v[j] = total(i * NT + j, e);
            put_last(e, i, v);
        }
    } else {
        for (int item = ki; item < 4 * NT; item += s.ks) {
            const int e = item & 3, j = item >> 2;
            float v[DD][VM];
#pragma unroll
            for (int g = 0; g < DD; ++g)
#pragma unroll
                for (int i = 0; i < VM; ++i) v[g][i] = total((g * VM + i) * NT + j, e);
            put(e, j, v);
        }
    }
}

struct SplitInst {
    int combo, last, run, vm, nt, dd;
    const void *fn;
};
#define SPLIT_INST(COMBO_, TX_, TW_, TY_, LAST_, RUN_, VM_, NT_, DD_) \
    {COMBO_, LAST_, RUN_, VM_, NT_, DD_, (const void *)&ks_split_kernel<TX_, TW_, TY_, LAST_, RUN_, VM_, NT_, DD_>}
#define SPLIT_FIRST(COMBO_, TX_, TW_, TY_, RUN_)                                                            \
    SPLIT_INST(COMBO_, TX_, TW_, TY_, false, RUN_, 4, 1, 1), SPLIT_INST(COMBO_, TX_, TW_, TY_, false, RUN_, 4, 2, 1), \
        SPLIT_INST(COMBO_, TX_, TW_, TY_, false, RUN_, 4, 4, 1), SPLIT_INST(COMBO_, TX_, TW_, TY_, false, RUN_, 4, 1, 2), \
        SPLIT_INST(COMBO_, TX_, TW_, TY_, false, RUN_, 4, 2, 2), SPLIT_INST(COMBO_, TX_, TW_, TY_, false, RUN_, 4, 1, 3), \
        SPLIT_INST(COMBO_, TX_, TW_, TY_, false, RUN_, 4, 1, 4), SPLIT_INST(COMBO_, TX_, TW_, TY_, false, RUN_, 2, 1, 6)
#define SPLIT_SET(COMBO_, TX_, TW_, TY_)                                                                            \
    SPLIT_INST(COMBO_, TX_, TW_, TY_, true, false, 4, 1, 1), SPLIT_INST(COMBO_, TX_, TW_, TY_, true, false, 4, 2, 1), \
        SPLIT_INST(COMBO_, TX_, TW_, TY_, true, false, 4, 4, 1), SPLIT_FIRST(COMBO_, TX_, TW_, TY_, false),           \
        SPLIT_FIRST(COMBO_, TX_, TW_, TY_, true), SPLIT_INST(COMBO_, TX_, TW_, TY_, false, false, 2, 1, 8)

const SplitInst split_insts[] = {
    SPLIT_SET(0, float, float, float),
    SPLIT_SET(1, half_t, half_t, half_t),
    SPLIT_SET(2, fp8_t, fp8_t, half_t),
    SPLIT_SET(3, half_t, fp8_t, half_t),
};
constexpr int N_SPLIT_INSTS = sizeof(split_insts) / sizeof(SplitInst);

bool split_fits(const SplitInst &t, const Problem &p, int combo)
{
    if (t.combo != combo || t.last != p.bs_last || p.b < 4) return false;
    if (t.last) return p.batch >= t.nt;
    if (p.d % t.dd) return false;
    return t.run == (p.d == t.dd && p.c % (combo == 0 ? 4 : 8) == 0);
}

}  // namespace

int split_inst_count() { return N_SPLIT_INSTS; }

uint32_t split_inst_id(int i)
{
    if (i < 0 || i >= N_SPLIT_INSTS) return 0;
    const SplitInst &t = split_insts[i];
    const int v[6] = {t.combo, t.last, t.run, t.vm, t.nt, t.dd};
    return inst_hash('P', v, 6);
}

// variant: instance | waves per workgroup << 8 (0: automatic), or -1 for the automatic instance
int split_run(const Problem &p, int variant, bool launch, ksmm_tile *tile)
{
    const int waves = variant < 0 ? 0 : (variant >> 8) & 0xff;
    if (variant >= 0) variant &= 0xff;
    const int combo = combo_of(p.x_dtype, p.w_dtype, p.y_dtype);
    if (combo < 0) return KSMM_ERR_BAD_DTYPE;
    // 32-bit byte offsets inside the weights of DD blocks and inside the input
    if ((int64_t)p.b * p.c * 8 * (int64_t)dtype_size(p.w_dtype) > 0xffffffffLL ||
        (int64_t)p.a * p.c * p.d * p.batch * (int64_t)dtype_size(p.x_dtype) > 0xffffffffLL)
        return KSMM_ERR_BAD_ALGO;
    int pick = -1;
    if (variant >= 0) {
        if (variant < N_SPLIT_INSTS && split_fits(split_insts[variant], p, combo)) pick = variant;
    } else {
        // as many neighbouring d_i as there are, then the widest batch tile that still gives every
        // CU two workgroups
        int64_t best = -1;
        for (int i = 0; i < N_SPLIT_INSTS; ++i) {
            const SplitInst &t = split_insts[i];
            if (!split_fits(t, p, combo)) continue;
            const int64_t grid = (int64_t)p.a * (p.d / t.dd) * ((p.b + 16 * t.vm - 1) / (16 * t.vm)) * ((p.batch + 16 * t.nt - 1) / (16 * t.nt));
            int64_t score = t.dd * 10 + t.nt;
            if (t.nt > 1 && (grid < 512 || p.batch <= 8 * t.nt)) score -= 10000;
            if (score > best || pick < 0) best = score, pick = i;
        }
    }
    if (pick < 0) return KSMM_ERR_BAD_ALGO;
    const SplitInst &t = split_insts[pick];
    const int tm = 16 * t.vm, tn = 16 * t.nt, tiles_w = t.vm * t.nt * t.dd;
    const int m_tiles = (p.b + tm - 1) / tm, kstep = combo == 0 ? 16 : 32, steps = (p.c + kstep - 1) / kstep;
    int ks = split_waves(t.vm, t.nt, t.dd);
    if (waves > ks) return KSMM_ERR_BAD_ALGO;
    if (waves) ks = waves;
    if (ks > steps) ks = steps;
    const int64_t d_groups = p.d / t.dd, tiles = (int64_t)p.a * d_groups * m_tiles;
    const int64_t n_tiles = (p.batch + tn - 1) / tn, grid = (tiles + 7) / 8 * 8 * n_tiles;
    if (grid > 0x7fffffffLL) return KSMM_ERR_TOO_LARGE;
    const int lds = ks > 1 ? ks * tiles_w * 1024 : 0;  // at most 64 KB
    if (tile) {
        tile->algo = KSMM_ALGO_TILE;
        tile->variant = (5 << 24) | (ks << 8) | pick;
        tile->tile_m = tm;
        tile->tile_n = tn;
        tile->tile_k = kstep;
        tile->tile_d = t.dd;
        tile->threads = 64 * ks;
        tile->lds_bytes = lds;
        tile->grid = grid;
    }
    if (!launch) return KSMM_OK;
    SplitArgs s{(int)p.batch, p.a, p.b, p.c, p.d, m_tiles, (int)n_tiles, (int)d_groups, ks, (int)tiles};
    Epi ep = epi_of(p);
    void *args[] = {(void *)&p.x, (void *)&p.w, (void *)&p.y, &s, &ep};
    return hipLaunchKernel(t.fn, dim3((unsigned)grid), dim3(64 * ks), args, lds, p.stream) == hipSuccess
               ? KSMM_OK
               : KSMM_ERR_LAUNCH;
}

}  // namespace ksmm
