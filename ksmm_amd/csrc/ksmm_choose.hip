// Which kernel instance takes a problem the measured table does not cover: small and medium
// batches, and batch-size-last batches off the vector.
//
// The table and the heuristics of the families were measured at full batches, where the tile with
// the fewest re-reads wins.  Below a few thousand rows that tile leaves most of the chip idle and
// walks c alone: over 2400 problems drawn from the layers' shapes (batches 1 .. 25088, all types,
// both layouts) the heuristics' choice took 1.4 to 2.2 times the time of the fastest instance in the
// geometric mean, and up to 12 times.  Here every instance that takes the problem is priced by a
// linear model of its time in microseconds,
//     t = f . (1, s, cu s, s w, cu s w, cu, by, by w, far)
//   s   steps of a workgroup's loop over c (wave and row kernels: size of a tile times the tiles of a wave
//       or workgroup; one thread per output and vector form: eighths of c)
//   cu  rounds of workgroups over the 256 CUs (split-K, wave and row kernels: of waves over the SIMDs)
//   w   share of a 64-byte line a batch-size-first tile does not use, as a factor
//   by  bytes of input, output and weights at 5 TB/s
//   far those beyond 125 MB, which the last-level cache does not keep for the next kernel
// with non-negative coefficients fitted per instance to its measured times, and the cheapest one is
// taken.  The table comes from `python -m ksmm_amd.prices`, which also says how good the choice is on
// problems that were held back from the fit (1.04 to 1.08 times the fastest instance in the geometric
// mean by type and layout); instances that it lists as having no price are not offered.  The generic kernels are priced for the comparison only: they are the choice at full batches
// of what has no other kernel, or of blocks of a few elements.
#include <math.h>
#include <string.h>

#include "ksmm_choose.h"

namespace ksmm {

namespace {

// tile sub-families have their own numbers
constexpr int FAM_SPLIT = 5, FAM_GENERIC = 13, FAM_WAVE = 14, FAM_ROWS = 15;
constexpr int COST_TERMS = 9;
struct CostRow {
    int family, combo, bs_last;
    uint32_t id;  // of the instance (generic family: the variant)
    float f[COST_TERMS];
};
const CostRow cost_rows[] = {
#include "ksmm_cost.inc"
};
constexpr int N_COST = (int)(sizeof(cost_rows) / sizeof(CostRow));

constexpr int N_SUBS = 6, MAX_INST = 128, MAX_ROWS = 1024;
struct CostIndex {  // rows by family and instance
    const CostRow *tile[N_SUBS][4][2][MAX_INST], *generic[4][2][2];
    const CostRow *wave[4][MAX_INST], *rows[4][MAX_ROWS];  // batch-size-last, batch-size-first
    int count[N_SUBS];
    CostIndex()
    {
        memset(this, 0, sizeof(*this));
        const int n[N_SUBS] = {ktile_inst_count(), ws_inst_count(), stream_inst_count(),
                               bf_inst_count(), gemm_inst_count(), split_inst_count()};
        uint32_t (*const id[N_SUBS])(int) = {ktile_inst_id, ws_inst_id, stream_inst_id,
                                             bf_inst_id, gemm_inst_id, split_inst_id};
        for (int s = 0; s < N_SUBS; ++s) count[s] = n[s] < MAX_INST ? n[s] : MAX_INST;
        for (int i = 0; i < N_COST; ++i) {
            const CostRow &r = cost_rows[i];
            if (r.family == FAM_GENERIC) generic[r.combo][r.bs_last][r.id & 1] = &r;
            if (r.family == FAM_WAVE)
                for (int k = 0; k < wave_inst_count(r.combo) && k < MAX_INST; ++k)
                    if (wave_inst_id(r.combo, k) == r.id) wave[r.combo][k] = &r;
            if (r.family == FAM_ROWS)
                for (int k = 0; k < rows_inst_count() && k < MAX_ROWS; ++k)
                    if (rows_inst_id(k) == r.id) rows[r.combo][k] = &r;
            if (r.family >= N_SUBS) continue;
            for (int k = 0; k < count[r.family]; ++k)
                if (id[r.family](k) == r.id) tile[r.family][r.combo][r.bs_last][k] = &r;
        }
    }
};
const CostIndex &cost_index()
{
    static const CostIndex index;
    return index;
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// batch-size-last rows that no 16-byte vector divides
bool ragged_rows(const Problem &p) { return p.bs_last && p.batch % (16 / (int64_t)dtype_size(p.x_dtype)) != 0; }

// The k-loop tiles on batch-size-last rows that no vector divides, against whole ones: 1.00 to 1.04 times the time in fp32
// and e4m3, up to 1.2 in fp16 (seven patterns at 6500 and 6501 columns: vectors off their alignment).  Against the
// split-K kernel, which alone took such rows before (us at 6501 / 25061 columns): (4,192,192,1) fp16 18 / 38 and 9 / 22,
// (1,256,256,3) fp16 24 / 46 and 12 / 26, (1,1536,384,2) fp16 47 / 184 and 36 / 112, fp32 166 / 560 and 143 / 507.
constexpr float RAGGED_H = 1.1f;
// and where they fill their last tile of outputs in part, by which they have to be ahead: the split-K kernel skips some of
// what is not there, and its price is up to 1.4 times too high on such blocks.  us on that kernel / on the tile: (12,48,192,6)
// fp16 at 997 columns 11.8 / 16.5 and (12,48,48,4) fp32 at 4531 23.0 / 25.3 stay where they are for it; (6,96,384,2) fp16 at
// 9259, 41.0 / 24.5, has its tile.
// What both factors give: on 8519 drawn ragged problems the choice takes 0.965 (fp32), 0.930 (fp16), 0.963 and 0.946 (e4m3, e4m3
// weights) of the time without these tiles in the geometric mean; on 127 of them, 1.5 percent, it is more than 3 percent slower,
// by 1.09 in their mean.  Prices of these tiles fitted to such rows instead gave 0.963, 0.923, 0.963 and 0.945 with 120 that are
// slower: the tiles' own prices are within 3 percent there, the error is that of the split-K prices (a factor of 1.2 to 1.4).
constexpr float RAGGED_PART = 1.3f;

float price(const CostRow &r, const Problem &p, const ksmm_tile &t)
{
    const double ex = (double)dtype_size(p.x_dtype), ew = (double)dtype_size(p.w_dtype), ey = (double)dtype_size(p.y_dtype);
    const double n = (double)p.batch, ad = (double)p.a * p.d;
    const int64_t blocks = r.family == FAM_ROWS ? ceil_div((int64_t)p.a * p.d, t.tile_d) : (int64_t)p.a * (p.d / t.tile_d);
    int64_t groups = blocks * ceil_div(p.b, t.tile_m) * ceil_div(p.batch, t.tile_n);
    double s = (double)ceil_div(p.c, t.tile_k);
    int64_t cu = ceil_div(groups, 256);
    if (r.family == FAM_SPLIT) {
        const int ks = t.threads / 64;
        s = (double)ceil_div((int64_t)s, ks);
        cu = ceil_div(groups * ks, 1024);
    } else if (r.family == FAM_WAVE || r.family == FAM_ROWS) {
        // workers (waves, or a row kernel's workgroups) walk over tiles of the whole of c
        const int64_t waves = t.grid * (t.threads / 64), workers = r.family == FAM_WAVE ? waves : t.grid;
        s = (double)t.tile_m * t.tile_n * t.tile_d * p.c / 65536. * (double)ceil_div(groups, workers);
        cu = ceil_div(waves, 1024);
    } else if (r.family == FAM_GENERIC) {  // one thread's loop over c; workgroups of 256
        s = (double)p.c / 8.;
        cu = ceil_div(t.grid, 256);
    }
    const double by = (n * ad * (p.c * ex + p.b * ey) + ad * p.b * p.c * ew) / 5e6;
    double w = 1.;
    if (!p.bs_last && t.tile_d < p.d) {
        const double line = p.d * ex < 64. ? p.d * ex : 64.;
        w = line / (t.tile_d * ex) > 1. ? line / (t.tile_d * ex) : 1.;
    }
    const double v[COST_TERMS] = {1., s, cu * s, s * w, cu * s * w, (double)cu, by, by * w, by > 25. ? by - 25. : 0.};
    double us = 0.;
    for (int i = 0; i < COST_TERMS; ++i) us += r.f[i] * v[i];
    if (t.algo == KSMM_ALGO_TILE && t.variant >> 24 == 0 && ragged_rows(p))
        us *= (p.x_dtype == KSMM_F16 && p.w_dtype == KSMM_F16 ? RAGGED_H : 1.f) * (p.b % t.tile_m ? RAGGED_PART : 1.f);
    return (float)us;
}

const CostRow *row_of(const Problem &p, int combo, int algo, int variant)
{
    const CostIndex &ix = cost_index();
    if (variant < 0) return nullptr;
    if (algo == KSMM_ALGO_GENERIC) return variant < 2 ? ix.generic[combo][p.bs_last][variant] : nullptr;
    if (algo == KSMM_ALGO_WAVE) {
        if (p.bs_last) return (variant & 0xff) < MAX_INST ? ix.wave[combo][variant & 0xff] : nullptr;
        return variant >= 1000 ? ix.rows[combo][(variant - 1000) & (MAX_ROWS - 1)] : nullptr;
    }
    if (algo != KSMM_ALGO_TILE) return nullptr;
    const int sub = variant >> 24, inst = variant & 0xff;
    return sub < N_SUBS && inst < MAX_INST ? ix.tile[sub][combo][p.bs_last][inst] : nullptr;
}

}  // namespace

float predicted_us(const Problem &p, const ksmm_tile &t)
{
    const int combo = combo_of(p.x_dtype, p.w_dtype, p.y_dtype);
    const CostRow *r = combo < 0 ? nullptr : row_of(p, combo, t.algo, t.variant);
    return r ? price(*r, p, t) : -1.f;
}

Choice cheapest_instance(const Problem &p, bool any_alignment)
{
    Choice best{KSMM_ALGO_AUTO, -1, -1.f}, split = best;
    const int combo = combo_of(p.x_dtype, p.w_dtype, p.y_dtype);
    if (combo < 0) return best;
    const bool ragged = ragged_rows(p);
    auto offer = [&](int algo, int variant) {
        ksmm_tile t;
        memset(&t, 0, sizeof(t));
        const int rc = algo == KSMM_ALGO_WAVE ? wave_run(p, variant, false, &t) : tile_run(p, variant, false, &t);
        if (rc != KSMM_OK) return;
        const CostRow *r = row_of(p, combo, t.algo, t.variant);
        if (!r || (t.threads & 63) || t.tile_d < 1) return;
        const float us = price(*r, p, t);
        if (best.us < 0.f || us < best.us) best = Choice{t.algo, t.variant, us};
        if (r->family == FAM_SPLIT && (split.us < 0.f || us < split.us)) split = Choice{t.algo, t.variant, us};
    };
    const CostIndex &ix = cost_index();
    if (!any_alignment) {
        offer(KSMM_ALGO_WAVE, -1);
        for (int sub = 0; sub < FAM_SPLIT; ++sub)
            for (int i = 0; i < ix.count[sub]; ++i)
                if (ix.tile[sub][combo][p.bs_last][i]) offer(KSMM_ALGO_TILE, (sub << 24) | (sub == 0 && ragged ? 1 << 8 : 0) | i);
    }
    for (int i = 0; any_alignment && i < ix.count[3]; ++i)
        if (bf_inst_whole(i) && ix.tile[3][combo][p.bs_last][i]) offer(KSMM_ALGO_TILE, (3 << 24) | i);
    for (int i = 0; i < ix.count[FAM_SPLIT]; ++i) {
        if (!ix.tile[FAM_SPLIT][combo][p.bs_last][i]) continue;
        for (int waves = 1; waves <= 16; waves *= 2) offer(KSMM_ALGO_TILE, (FAM_SPLIT << 24) | (waves << 8) | i);
    }
    // 16-bit and e4m3 rows that fill the split-K kernel's 16 in part are priced too high there: what is beyond 5 us shrinks with
    // them, to a quarter and less.  A whole-d tile has to be ahead of that: (16,256,256,3) e4m3 on one row, priced 9.0 and 8.0, takes
    // 5.0 on split-K and 8.5 on the tile.
    if (!p.bs_last && p.x_dtype != KSMM_F32 && p.batch < 16 && split.us > 5.f && best.algo == KSMM_ALGO_TILE && best.variant >> 24 == 3 &&
        bf_inst_whole(best.variant & 0xff) && 5.f + (split.us - 5.f) * (0.25f + 0.75f / 16.f * p.batch) < best.us)
        best = split;
    return best;
}

float copy_us(int64_t rows, int64_t cols_in, int64_t cols_out, int elem_bytes, bool transpose)
{
    // measured: 7.4 us for 19 + 19 MB transposed, 28 us for 77 + 77; 8.3 us for 10 + 10 MB re-pitched from memory
    // that no kernel has just read (3 TB/s), 68 us for 205 + 205, 280 us for 822 + 822 (5.9 TB/s)
    const float bytes = (float)((double)rows * (cols_in + cols_out) * elem_bytes);
    return 2.5f + (transpose ? bytes / 5.2e6f : fminf(bytes / 3e6f, 20.f + bytes / 5.9e6f));
}

}  // namespace ksmm
