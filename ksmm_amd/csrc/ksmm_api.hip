// C ABI of libksmm_hip.so: argument checks, kernel-family dispatch, factor chains.
#include <string.h>

#include <atomic>

#include "ksmm_choose.h"
#include "ksmm_pair.h"

using namespace ksmm;

namespace ksmm {

// (kernel, device) pairs whose dynamic-LDS limit has been raised: a fixed open-addressing set
// of atomics.  Insert-only and idempotent, so concurrent callers need no lock; it holds no
// caller-visible state (a lost race only repeats the attribute call).
int ensure_dynamic_lds(const void *fn, int bytes)
{
    if (bytes <= 64 * 1024) return KSMM_OK;
    constexpr unsigned SLOTS = 4096;  // far more than kernels x devices
    static std::atomic<uintptr_t> seen[SLOTS];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return KSMM_ERR_LAUNCH;
    const uintptr_t key = ((uintptr_t)fn << 8) ^ (uintptr_t)(dev + 1);
    unsigned h = (unsigned)((key * 0x9E3779B97F4A7C15ull) >> 40) % SLOTS;
    for (unsigned probe = 0; probe < SLOTS; ++probe, h = (h + 1) % SLOTS) {
        const uintptr_t cur = seen[h].load(std::memory_order_acquire);
        if (cur == key) return KSMM_OK;
        if (cur != 0) continue;
        // every instance declares its full ring; the limit never has to grow afterwards
        if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess)
            return KSMM_ERR_LAUNCH;
        uintptr_t expected = 0;
        seen[h].compare_exchange_strong(expected, key, std::memory_order_release);
        return KSMM_OK;
    }
    // table full (cannot happen with the instance counts of this library): set it every time
    return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess
               ? KSMM_OK
               : KSMM_ERR_LAUNCH;
}

}  // namespace ksmm

// Scratch memory of ksmm_chain_forward_static: one fixed device array per GPU (each GPU that
// runs the library holds its own copy until the process ends).  In host code the name is only
// a handle for hipGetSymbolAddress (static_scratch below), never a device address.
constexpr int64_t KSMM_STATIC_SCRATCH_BYTES = 32ll << 20;
static __device__ __align__(256) unsigned char scratch[KSMM_STATIC_SCRATCH_BYTES];

namespace {

bool dtype_known(int dt) { return dt == KSMM_F32 || dt == KSMM_F16 || dt == KSMM_FP8_E4M3; }

int check_shape(int64_t batch, int a, int b, int c, int d, int xd, int wd, int yd)
{
    if (a < 1 || b < 1 || c < 1 || d < 1) return KSMM_ERR_BAD_PATTERN;
    if (batch < 1) return KSMM_ERR_BAD_BATCH;
    if (!dtype_known(xd) || !dtype_known(wd) || !dtype_known(yd)) return KSMM_ERR_BAD_DTYPE;
    if (combo_of(xd, wd, yd) < 0) return KSMM_ERR_BAD_DTYPE;
    const int64_t lim = 0x7fffffffLL;
    // products are checked step by step so that they cannot wrap
    int64_t acd = (int64_t)a * c;
    if (acd > lim) return KSMM_ERR_TOO_LARGE;
    acd *= d;
    int64_t abd = (int64_t)a * b;
    if (abd > lim) return KSMM_ERR_TOO_LARGE;
    abd *= d;
    if (acd > lim || abd > lim) return KSMM_ERR_TOO_LARGE;
    if (acd * batch > lim || abd * batch > lim) return KSMM_ERR_TOO_LARGE;
    int64_t nnz = (int64_t)a * b;
    nnz *= c;
    if (nnz > lim) return KSMM_ERR_TOO_LARGE;
    nnz *= d;
    if (nnz > lim) return KSMM_ERR_TOO_LARGE;
    return KSMM_OK;
}

// Measured choices for known patterns (the counterpart of the reference's *.best tables,
// src/ksmm_py/layer/kronecker_sparse/kernel.py:151-239): rows sorted by key.
// A row names its kernel by family, stable instance id (inst_hash of the instance's parameters)
// and a family-specific launch parameter, never by a position in an instance table.
struct TunedRow {
    int a, b, c, d, combo, bs_last, algo;
    uint32_t id;
    int param;
};
const TunedRow tuned_rows[] = {
#include "ksmm_tuned.inc"
    {0, 0, 0, 0, 0, 0, 0, 0, 0},  // sentinel: keeps the array non-empty
};

// (family, variant) <-> (family, instance id, parameter).  Variant layouts are those of
// ksmm_factor_forward_algo; `param` keeps what is not the instance: tiles per wave and tile
// order (wave), workgroups per a_i (row kernels), workgroups per block (stream, weight-stationary).
bool describe_variant(int algo, int variant, int combo, int bs_last, uint32_t *id, int *param)
{
    *param = 0;
    if (algo == KSMM_ALGO_GENERIC) {
        const int v[1] = {variant};
        *id = inst_hash('X', v, 1);
        return variant == 0 || variant == 1;
    }
    if (algo == KSMM_ALGO_WAVE) {
        if (bs_last) {
            if (variant < 0) return false;
            *id = wave_inst_id(combo, variant & 0xff);
            *param = variant >> 8;
        } else {
            if (variant < 1000) return false;
            *id = rows_inst_id((variant - 1000) & 0x3ff);
            *param = (variant - 1000) >> 10;
        }
        return *id != 0;
    }
    if (algo == KSMM_ALGO_TILE) {
        if (variant < 0) return false;
        const int sub = (variant >> 24) & 15, inst = variant & 0xff;
        *param = (variant >> 8) & 0xffff;
        switch (sub) {
        case 0: *id = ktile_inst_id(inst); break;
        case 1: *id = ws_inst_id(inst); break;
        case 2: *id = stream_inst_id(inst); break;
        case 3: *id = bf_inst_id(inst); break;
        case 4: *id = gemm_inst_id(inst); break;
        case 5: *id = split_inst_id(inst); break;
        default: *id = 0;
        }
        return *id != 0;
    }
    return false;
}

template <typename F> int find_id(int n, uint32_t id, F id_of)
{
    for (int i = 0; i < n; ++i)
        if (id_of(i) == id) return i;
    return -1;
}

bool resolve_variant(int algo, uint32_t id, int param, int combo, int bs_last, int *variant)
{
    if (algo == KSMM_ALGO_GENERIC) {
        for (int v = 0; v <= 1; ++v) {
            const int a[1] = {v};
            if (inst_hash('X', a, 1) == id) return *variant = v, true;
        }
        return false;
    }
    if (algo == KSMM_ALGO_WAVE) {
        if (bs_last) {
            const int i = find_id(wave_inst_count(combo), id, [&](int k) { return wave_inst_id(combo, k); });
            return i >= 0 ? (*variant = i | (param << 8), true) : false;
        }
        const int i = find_id(rows_inst_count(), id, rows_inst_id);
        return i >= 0 ? (*variant = 1000 + (i | (param << 10)), true) : false;
    }
    if (algo == KSMM_ALGO_TILE) {
        int i, sub = 0;
        if ((i = find_id(ktile_inst_count(), id, ktile_inst_id)) >= 0) sub = 0;
        else if ((i = find_id(ws_inst_count(), id, ws_inst_id)) >= 0) sub = 1;
        else if ((i = find_id(stream_inst_count(), id, stream_inst_id)) >= 0) sub = 2;
        else if ((i = find_id(bf_inst_count(), id, bf_inst_id)) >= 0) sub = 3;
        else if ((i = find_id(gemm_inst_count(), id, gemm_inst_id)) >= 0) sub = 4;
        else if ((i = find_id(split_inst_count(), id, split_inst_id)) >= 0) sub = 5;
        else return false;
        *variant = (sub << 24) | ((param & 0xffff) << 8) | i;
        return true;
    }
    return false;
}
constexpr int N_TUNED = (int)(sizeof(tuned_rows) / sizeof(TunedRow)) - 1;
constexpr int64_t TUNED_MIN_BATCH = 8192;  // the table was measured at batch 25088

int cmp_key(const TunedRow &r, const Problem &p, int combo)
{
    const int k[6] = {p.a, p.b, p.c, p.d, combo, p.bs_last};
    const int q[6] = {r.a, r.b, r.c, r.d, r.combo, r.bs_last};
    for (int i = 0; i < 6; ++i)
        if (q[i] != k[i]) return q[i] < k[i] ? -1 : 1;
    return 0;
}

const TunedRow *tuned_lookup(const Problem &p)
{
    const int combo = combo_of(p.x_dtype, p.w_dtype, p.y_dtype);
    int lo = 0, hi = N_TUNED - 1;
    while (lo <= hi) {
        const int mid = (lo + hi) / 2, c = cmp_key(tuned_rows[mid], p, combo);
        if (c == 0) return &tuned_rows[mid];
        if (c < 0)
            lo = mid + 1;
        else
            hi = mid - 1;
    }
    return nullptr;
}

// Whether a measured row names an instance of the library for the problem
bool tuned_for(const Problem &p)
{
    const TunedRow *row = p.batch >= TUNED_MIN_BATCH ? tuned_lookup(p) : nullptr;
    int variant;
    return row && row->algo != KSMM_ALGO_AUTO && resolve_variant(row->algo, row->id, row->param, row->combo, row->bs_last, &variant);
}

// A family's kernel, or its own choice (variant < 0).
int family_run(const Problem &p, int algo, int variant, bool launch, ksmm_tile *tile)
{
    switch (algo) {
    case KSMM_ALGO_GENERIC: return generic_run(p, variant, launch, tile);
    case KSMM_ALGO_WAVE: return wave_run(p, variant, launch, tile);
    case KSMM_ALGO_TILE: return tile_run(p, variant, launch, tile);
    default: return KSMM_ERR_BAD_ALGO;
    }
}

// The choice measured at full batches: the tuned table (unless `table` is off, which is what the
// tuner compares against), then the heuristics: the table inside each family decides whether it
// takes the problem; the generic family always does.
int table_run(const Problem &p, bool table, bool launch, ksmm_tile *tile)
{
    if (table && p.batch >= TUNED_MIN_BATCH) {
        const TunedRow *row = tuned_lookup(p);
        int row_variant;
        if (row && row->algo != KSMM_ALGO_AUTO &&
            resolve_variant(row->algo, row->id, row->param, row->combo, row->bs_last, &row_variant)) {
            const int rc = family_run(p, row->algo, row_variant, launch, tile);
            if (rc != KSMM_ERR_BAD_ALGO) return rc;
        }
    }
    // Family order from sweeps at batch 25088: batch-size-first 16-bit mid-sized blocks
    // (64x64 .. 192x192) go to the stream kernels of the tile family; batch-size-last blocks
    // the wave family has an instance for (up to 96x96), and fp32, go to the wave family,
    // larger 16-bit blocks to the stream kernels again (inside the tile family), the rest to
    // the GEMM and k-loop tiles; shapes none of them takes run on the generic kernel.
    int rc = KSMM_ERR_BAD_ALGO;
    if (p.x_dtype == KSMM_F16 && !p.bs_last) rc = stream_run(p, -1, launch, tile);
    if (rc != KSMM_ERR_BAD_ALGO) return rc;
    rc = wave_run(p, -1, launch, tile);
    if (rc != KSMM_ERR_BAD_ALGO) return rc;
    rc = tile_run(p, -1, launch, tile);
    if (rc != KSMM_ERR_BAD_ALGO) return rc;
    return generic_run(p, -1, launch, tile);
}

// Rows of a batch-size-last workspace copy are padded to a multiple of 16 columns (the 16-byte
// vector of every type).
int64_t padded_batch(int64_t batch) { return (batch + 15) / 16 * 16; }

// A batch-size-first problem that only the generic kernel takes, while its batch-size-last
// twin has a real kernel: worth two transposes.  (The transposed copy has padded rows, so the
// twin runs at the padded batch.)
bool find_transposed(const Problem &p)
{
    if (p.bs_last) return false;
    ksmm_tile t;
    memset(&t, 0, sizeof(t));
    if (table_run(p, true, false, &t) != KSMM_OK || t.algo != KSMM_ALGO_GENERIC) return false;
    Problem q = p;
    q.bs_last = 1;
    q.batch = padded_batch(p.batch);
    // (a batch whose padded copies would pass the size limit stays on the kernel it has)
    if (check_shape(q.batch, p.a, p.b, p.c, p.d, p.x_dtype, p.w_dtype, p.y_dtype) != KSMM_OK) return false;
    memset(&t, 0, sizeof(t));
    // (the vector form of the generic kernel counts as a real kernel: variant 1)
    return table_run(q, true, false, &t) == KSMM_OK && (t.algo != KSMM_ALGO_GENERIC || t.variant == 1);
}

// Batch-size-last rows are `batch` elements long: when that is not a multiple of the 16-byte
// vector only the k-loop tiles, the split-K and the one-thread-per-output kernels take the problem.  With a workspace it runs on a
// copy whose rows are zero-filled to the next multiple of 16 columns (the vector of every type)
// and the result rows are cut back: two copies more, but on the kernel of the padded batch, where that
// is priced lower (route_pays).
bool find_padded(const Problem &p)
{
    if (!p.bs_last || p.batch % 16 == 0) return false;
    ksmm_tile t;
    memset(&t, 0, sizeof(t));
    if (table_run(p, true, false, &t) != KSMM_OK || t.algo != KSMM_ALGO_GENERIC || t.variant == 1)
        return false;
    Problem q = p;
    q.batch = padded_batch(p.batch);
    if (check_shape(q.batch, p.a, p.b, p.c, p.d, p.x_dtype, p.w_dtype, p.y_dtype) != KSMM_OK) return false;
    memset(&t, 0, sizeof(t));
    return table_run(q, true, false, &t) == KSMM_OK && (t.algo != KSMM_ALGO_GENERIC || t.variant == 1);
}

// What takes a problem as it is.  `direct`: the full-batch choice is a kernel of its own, not the
// one-thread-per-output one.
struct Pick {
    Choice c;     // AUTO: the full-batch choice
    bool direct;
    bool transposed, padded;  // the problem has that route
    float us;     // predicted time, < 0: no model of it
    bool own;     // it has the transposed route, and a whole-d tile that is priced below it: no copies, no workspace
};

// Full batches that no row of the table names.  The heuristics were made on the patterns of the table; the prices, fitted on
// batches up to 16384, find instances that they pass by: (12,64,256,1) fp32 at 25088 rows 221 us / 111, (12,256,64,1) feature-major
// 131 / 55, (3,128,128,2) fp16 at 17040 rows 27.7 / 11.2, (6,256,64,1) e4m3 at 19440 41.8 / 21.2.  How far below the
// heuristics' price an instance has to be priced is from 2400 drawn problems of 8192 .. 25088 columns, us of the priced one / of
// the heuristics' in the geometric mean over those that change: fp32 at 0.9 0.77 feature-major and 0.67 rows (117 problems, 2 of them
// more than 3 percent slower, by 1.06), the others at 0.85 0.57 .. 0.84 (195 problems, 11 slower, by 1.15 at most); at 0.9
// 23 of 267 are slower, at 0.97 56 of 469.  Beyond, the error of the prices that are extrapolated furthest grows; from 900 problems
// of 25089 .. 110000 columns whose choice would change: fp32 at 0.9 0.69 rows and 0.77 feature-major (285 problems, 5 slower), e4m3
// rows at 0.85 0.64 (209, 3 slower); fp16 rows at 0.85 0.95 (84, 23 slower, up to 1.54) and at 0.75 0.90 (24, 1 slower by 1.07);
// fp16 and e4m3 feature-major at 0.85 0.85 and 0.75 (321, 115 slower, up to 1.33), at 0.7 0.64 and 0.50 (135, 8 slower, up to 1.13).
// (e4m3 weights on fp16 inputs keep the heuristics' choice: what they lose to fp16 weights is what decode_pays goes by.)
float heuristic_margin(const Problem &p)
{
    if (p.x_dtype == KSMM_F32) return 0.9f;
    if (p.batch <= 25088 || (p.x_dtype == KSMM_FP8_E4M3 && !p.bs_last)) return 0.85f;
    return p.bs_last ? 0.7f : 0.75f;
}

// Whether the kernels that move aligned 16-byte vectors take a problem's tensors (null: they will be).
bool on_vectors(const Problem &p) { return (((uintptr_t)p.x | (uintptr_t)p.w | (uintptr_t)p.y) & 15) == 0; }

// Below TUNED_MIN_BATCH, and where the full-batch choice is the one-thread-per-output kernel, the
// cheapest instance by the model of ksmm_choose.hip; else the full-batch choice, a row of the table, or the heuristics' one
// unless an instance is priced well below it (heuristic_margin).  Tensors off the
// vector take the cheapest of the kernels that do not need it.  A function of the sizes, types and that
// alignment alone: each thread remembers its last answers (pricing every instance takes tens
// of microseconds, a launch five).
float route_us(const Problem &p);
Pick pick_of(const Problem &given, bool table)
{
    const bool aligned = on_vectors(given);
    Problem p = given;  // (the routes of a problem are those the workspace query sees)
    p.x = p.w = nullptr;
    p.y = nullptr;
    struct Entry {
        int64_t batch;
        int key[8];
        Pick pick;
    };
    // sets of four: with one entry a hash, two factors of a chain that share it cost 3 to 5 us a call
    constexpr unsigned SETS = 64, WAYS = 4;
    static thread_local Entry memo[SETS][WAYS];  // batch 0: empty
    static thread_local uint8_t oldest[SETS];
    const int key[8] = {p.a, p.b, p.c, p.d, p.x_dtype, p.w_dtype, p.y_dtype, p.bs_last * 4 + (table ? 2 : 0) + (aligned ? 1 : 0)};
    uint64_t h = (uint64_t)p.batch;
    for (int v : key) h = (h ^ (uint64_t)v) * 0x9E3779B97F4A7C15ull;
    const unsigned set = (h >> 40) % SETS;
    for (const Entry &e : memo[set])
        if (e.batch == p.batch && memcmp(e.key, key, sizeof(key)) == 0) return e.pick;
    ksmm_tile t;
    memset(&t, 0, sizeof(t));
    Pick k{{KSMM_ALGO_AUTO, -1, -1.f}, true, find_transposed(p), find_padded(p), -1.f, false};
    // in place of the full-batch choice, priced at k.us.  A kernel of its own that has no price is not known to
    // be slower: it stays.  The one-thread-per-output kernel has to be ahead by the error of its fit (0.3):
    // on 14900 measured problems that it takes, chosen / fastest is 1.059 in the geometric mean so, 1.062 without
    // the margin and 1.081 (up to 13.5) if it is never taken.
    auto replace = [&](const Choice &c, float margin) {
        if (c.algo == KSMM_ALGO_AUTO || (k.us < 0.f ? k.direct : c.us >= (k.direct ? margin : 1.3f) * k.us)) return;
        k.c = c;
        k.us = c.us;
    };
    if (!aligned) {
        k.direct = false;
        generic_run(p, 0, false, &t);
        k.us = predicted_us(p, t);
        replace(cheapest_instance(p, true), 1.f);
    } else if (table_run(p, table, false, &t) == KSMM_OK) {
        k.direct = t.algo != KSMM_ALGO_GENERIC || t.variant == 1;
        k.us = predicted_us(p, t);
        if (p.batch < TUNED_MIN_BATCH || !k.direct) replace(cheapest_instance(p, false), 1.f);
        else if (!(table && tuned_for(p)) && p.w_dtype == p.x_dtype) replace(cheapest_instance(p, false), heuristic_margin(p));
    }
    if (k.transposed && !aligned) {
        k.own = pick_of(p, table).own;
    } else if (k.transposed && k.c.algo == KSMM_ALGO_TILE && (k.c.variant >> 24) == 3 && bf_inst_whole(k.c.variant & 0xff)) {
        const float route = route_us(p);
        k.own = route >= 0.f && k.us <= route;
        k.direct |= k.own;
    }
    Entry &e = memo[set][oldest[set]++ % WAYS];
    e.batch = p.batch;
    memcpy(e.key, key, sizeof(key));
    e.pick = k;
    return k;
}

bool wants_transposed(const Problem &p)
{
    const Pick k = pick_of(p, true);
    return k.transposed && !k.own;
}
bool wants_padded(const Problem &p) { return pick_of(p, true).padded; }

int dispatch(const Problem &p, int algo, int variant, bool launch, ksmm_tile *tile)
{
    if (algo != KSMM_ALGO_AUTO) return family_run(p, algo, variant, launch, tile);
    const bool table = variant == -1;
    const Pick k = pick_of(p, table);
    if (k.c.algo != KSMM_ALGO_AUTO) {
        const int rc = family_run(p, k.c.algo, k.c.variant, launch, tile);
        if (rc != KSMM_ERR_BAD_ALGO) {
            // a problem without a kernel of its own at full batches is reported as the generic
            // family's, which takes the same instance by that number
            if (tile && !k.direct && tile->algo == KSMM_ALGO_TILE) {
                tile->algo = KSMM_ALGO_GENERIC;
                tile->variant += GENERIC_TILE;
            }
            return rc;
        }
    }
    return on_vectors(p) ? table_run(p, table, launch, tile) : generic_run(p, 0, launch, tile);
}

// The same problem in batch-size-last layout with padded rows (what both routes run in the middle).
Problem twin_of(const Problem &p)
{
    Problem q = p;
    q.x = nullptr;  // (copies in a workspace)
    q.y = nullptr;
    q.bs_last = 1;
    q.batch = padded_batch(p.batch);
    return q;
}

// Predicted time of the transposed or padded-rows route of a problem that has one (< 0: no model of it)
float route_us(const Problem &p)
{
    const Pick q = pick_of(twin_of(p), true);
    if (q.us < 0.f) return -1.f;
    const int64_t bp = padded_batch(p.batch);
    const float copies = copy_us((int64_t)p.a * p.c * p.d, p.batch, bp, (int)dtype_size(p.x_dtype), !p.bs_last) +
                         copy_us((int64_t)p.a * p.b * p.d, p.batch, bp, (int)dtype_size(p.y_dtype), !p.bs_last);
    return copies + q.us;
}

// Whether it beats the kernel that takes the problem as it is: small problems are done before the first copy would be.
bool route_pays(const Problem &p)
{
    const float now = pick_of(p, true).us, route = route_us(p);
    return now < 0.f || route < 0.f || route < now;
}

int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }

// Bytes of the weight gradient's partial sums
int64_t wgrad_partial_bytes(int64_t batch, int a, int b, int c, int d, int dtype, int bs_last)
{
    return align256(wgrad_partial_floats(batch, a, b, c, d, dtype, bs_last) * 4);
}

bool overlaps(const void *p, int64_t p_bytes, const void *q, int64_t q_bytes)
{
    const char *pb = (const char *)p, *qb = (const char *)q;
    return pb < qb + q_bytes && qb < pb + p_bytes;
}


int check_epilogue(const ksmm_epilogue *ep)
{
    if (!ep) return KSMM_OK;
    if (ep->act != KSMM_ACT_NONE && ep->act != KSMM_ACT_GELU) return KSMM_ERR_BAD_EPILOGUE;
    return KSMM_OK;
}

int factor_forward_impl(const void *x, const void *w, void *y, int64_t batch, int a, int b, int c, int d,
                        int x_dtype, int w_dtype, int y_dtype, int bs_last, float scale, int algo, int variant,
                        const ksmm_epilogue *ep, void *stream, const float *x_scale = nullptr)
{
    int rc = check_shape(batch, a, b, c, d, x_dtype, w_dtype, y_dtype);
    if (rc != KSMM_OK) return rc;
    if ((rc = check_epilogue(ep)) != KSMM_OK) return rc;
    if (!x || !w || !y) return KSMM_ERR_NULL_POINTER;
    const int64_t xbytes = (int64_t)a * c * d * batch * (int64_t)dtype_size(x_dtype);
    const int64_t ybytes = (int64_t)a * b * d * batch * (int64_t)dtype_size(y_dtype);
    if (overlaps(x, xbytes, y, ybytes)) return KSMM_ERR_ALIAS;
    Problem p{x, w, y, batch, a, b, c, d, x_dtype, w_dtype, y_dtype, bs_last ? 1 : 0, scale,
              (hipStream_t)stream};
    if (ep) {
        p.bias = ep->bias;
        p.act = ep->act;
    }
    p.x_scale = x_scale;
    // Every kernel but the split-K and the one-thread-per-output ones moves aligned 16-byte vectors:
    // tensors that do not start on a 16-byte boundary run on those (a forced family refuses them).
    // All of them read a bias at the alignment of its elements.
    if (algo != KSMM_ALGO_AUTO && !on_vectors(p))
        return algo == KSMM_ALGO_GENERIC && variant <= 0 ? generic_run(p, 0, true, nullptr) : KSMM_ERR_BAD_ALGO;
    return dispatch(p, algo, variant, true, nullptr);
}

int factor_forward_ws_impl(const void *x, const void *w, void *y, int64_t batch, int a, int b, int c, int d,
                           int x_dtype, int w_dtype, int y_dtype, int bs_last, float scale,
                           const ksmm_epilogue *ep, void *workspace, int64_t workspace_bytes, void *stream)
{
    const int64_t need = ksmm_factor_workspace(batch, a, b, c, d, x_dtype, w_dtype, y_dtype, bs_last);
    if (need < 0) return (int)need;
    if (need == 0)
        return factor_forward_impl(x, w, y, batch, a, b, c, d, x_dtype, w_dtype, y_dtype, bs_last, scale,
                                   KSMM_ALGO_AUTO, -1, ep, stream);
    if (!x || !w || !y) return KSMM_ERR_NULL_POINTER;
    if (!workspace || workspace_bytes < need) return KSMM_ERR_WORKSPACE;
    const int64_t in_size = (int64_t)a * c * d, out_size = (int64_t)a * b * d;
    const int64_t xbytes = in_size * batch * (int64_t)dtype_size(x_dtype);
    const int64_t ybytes = out_size * batch * (int64_t)dtype_size(y_dtype);
    if (overlaps(x, xbytes, y, ybytes) || overlaps(workspace, need, x, xbytes) || overlaps(workspace, need, y, ybytes))
        return KSMM_ERR_ALIAS;
    if (((uintptr_t)workspace & 15) != 0) return KSMM_ERR_WORKSPACE;
    Problem p{x, w, y, batch, a, b, c, d, x_dtype, w_dtype, y_dtype, bs_last ? 1 : 0, scale, (hipStream_t)stream};
    if (!route_pays(p))
        return factor_forward_impl(x, w, y, batch, a, b, c, d, x_dtype, w_dtype, y_dtype, bs_last, scale,
                                   KSMM_ALGO_AUTO, -1, ep, stream);
    if (bs_last) {
        // rows padded to the vector (see wants_padded)
        const int64_t bp = padded_batch(batch);
        char *xp = (char *)workspace;
        char *yp = xp + align256(in_size * bp * (int64_t)dtype_size(x_dtype));
        int rc = repitch_run(x, xp, in_size, batch, bp, (int)dtype_size(x_dtype), (hipStream_t)stream);
        if (rc != KSMM_OK) return rc;
        rc = factor_forward_impl(xp, w, yp, bp, a, b, c, d, x_dtype, w_dtype, y_dtype, 1, scale, KSMM_ALGO_AUTO, -1,
                                 ep, stream);
        if (rc != KSMM_OK) return rc;
        return repitch_run(yp, y, out_size, bp, batch, (int)dtype_size(y_dtype), (hipStream_t)stream);
    }
    // transposed copies with rows of bp columns (bp = batch when that is a multiple of 16)
    const int64_t bp = padded_batch(batch);
    char *xt = (char *)workspace;
    char *yt = xt + align256(in_size * bp * (int64_t)dtype_size(x_dtype));
    int rc = transpose_run(x, xt, batch, in_size, (int)dtype_size(x_dtype), (hipStream_t)stream, 0, bp);
    if (rc != KSMM_OK) return rc;
    rc = factor_forward_impl(xt, w, yt, bp, a, b, c, d, x_dtype, w_dtype, y_dtype, 1, scale, KSMM_ALGO_AUTO, -1,
                             ep, stream);
    if (rc != KSMM_OK) return rc;
    return transpose_run(yt, y, out_size, batch, (int)dtype_size(y_dtype), (hipStream_t)stream, bp, 0);
}

int check_chain(const ksmm_factor_desc *f, int n, int64_t batch, int x_dtype, int y_dtype)
{
    if (!f) return KSMM_ERR_NULL_POINTER;
    if (n < 1 || n > KSMM_MAX_FACTORS) return KSMM_ERR_BAD_CHAIN;
    for (int i = 0; i < n; ++i) {
        // the first factor reads x_dtype, later ones read the intermediate type y_dtype
        int rc = check_shape(batch, f[i].a, f[i].b, f[i].c, f[i].d, i == 0 ? x_dtype : y_dtype,
                             f[i].w_dtype, y_dtype);
        if (rc != KSMM_OK) return rc;
        if (i > 0 && (int64_t)f[i].a * f[i].c * f[i].d != (int64_t)f[i - 1].a * f[i - 1].b * f[i - 1].d)
            return KSMM_ERR_CHAIN_MISMATCH;
    }
    return KSMM_OK;
}

bool chain_route_pays(const ksmm_factor_desc *f, int n, const void *x, void *y, int64_t batch, int x_dtype, int y_dtype, int bs_last,
                      bool fuse);

// batch-size-first chain with at least one factor that needs the transposed route, or where one pair of copies for all of its
// factors is priced below their own tiles
bool chain_wants_transposed(const ksmm_factor_desc *f, int n, int64_t batch, int x_dtype, int y_dtype,
                            int bs_last)
{
    if (bs_last) return false;
    // a chain the fused kernel takes in batch-size-last layout: one pass over the data between two
    // transposes instead of one pass per factor
    if (chain16_run(f, n, nullptr, nullptr, padded_batch(batch), x_dtype, y_dtype, 1, false, nullptr, nullptr) == KSMM_OK)
        return true;
    // (a function of the sizes and types: what is asked for is what a call needs, wherever its tensors lie)
    ksmm_factor_desc sizes[KSMM_MAX_FACTORS];
    bool own = false;
    for (int i = 0; i < n; ++i) {
        sizes[i] = f[i];
        sizes[i].w = nullptr;
        const Pick k = pick_of(Problem{nullptr, nullptr, nullptr, batch, f[i].a, f[i].b, f[i].c, f[i].d, i == 0 ? x_dtype : y_dtype,
                                       f[i].w_dtype, y_dtype, 0, 1.f, nullptr}, true);
        if (k.transposed && !k.own) return true;
        own |= k.own;
    }
    return own && n > 1 && chain_route_pays(sizes, n, nullptr, nullptr, batch, x_dtype, y_dtype, 0, false);
}

// batch-size-last chain whose batch is not a multiple of the vector, with at least one factor
// that has a real kernel at the padded batch
bool chain_wants_padded(const ksmm_factor_desc *f, int n, int64_t batch, int x_dtype, int y_dtype, int bs_last)
{
    if (!bs_last || batch % 16 == 0) return false;
    for (int i = 0; i < n; ++i) {
        Problem p{nullptr, nullptr, nullptr, batch, f[i].a, f[i].b, f[i].c, f[i].d, i == 0 ? x_dtype : y_dtype,
                  f[i].w_dtype, y_dtype, 1, 1.f, nullptr};
        if (wants_padded(p)) return true;
    }
    return false;
}

// Predicted time of the fused radix-16 chain (< 0: it does not take the chain).  Measured in
// microseconds at batches 16 .. 25088: 2 factors of 256 features 5.4, 3 of 512 8.1, 3 of 1024 10.7 with
// e4m3 weights, 1.3 times that with fp16 ones, plus the input and output at 5 TB/s.
float chain16_us(const ksmm_factor_desc *f, int n, int64_t batch, int x_dtype, int y_dtype)
{
    if (chain16_run(f, n, nullptr, nullptr, batch, x_dtype, y_dtype, 1, false, nullptr, nullptr) != KSMM_OK) return -1.f;
    const double features = (double)f[0].a * f[0].c * f[0].d;
    const double base = (2.7 * n + (features > 512 ? 2.6 : 0.)) * (f[0].w_dtype == KSMM_F16 ? 1.3 : 1.);
    return (float)(base + features * batch * (double)(dtype_size(x_dtype) + dtype_size(y_dtype)) / 5e6);
}

// Predicted time of a chain factor by factor, as given (x and y: its tensors) or in batch-size-last
// layout with padded rows (< 0: a factor has no price)
float chain_us(const ksmm_factor_desc *f, int n, const void *x, void *y, int64_t batch, int x_dtype, int y_dtype, int bs_last, bool twin)
{
    float sum = 0.f;
    for (int i = 0; i < n; ++i) {
        Problem p{i == 0 ? x : nullptr, f[i].w, i == n - 1 ? y : nullptr, batch, f[i].a, f[i].b, f[i].c, f[i].d,
                  i == 0 ? x_dtype : y_dtype, f[i].w_dtype, y_dtype, bs_last, 1.f, nullptr};
        const Pick k = pick_of(twin ? twin_of(p) : p, true);
        if (k.us < 0.f) return -1.f;
        sum += k.us;
    }
    return sum;
}

// Whether the fused chain is the faster way through a batch-size-last chain that it takes: at full
// batches it saves the intermediates' traffic; on a few thousand columns a launch per factor is
// done first (2.4 us each on the wave kernels against 3 to 4 us a factor in the fused one).
bool fused_pays(const ksmm_factor_desc *f, int n, const void *x, void *y, int64_t batch, int x_dtype, int y_dtype)
{
    if (batch >= TUNED_MIN_BATCH) return true;
    const float fused = chain16_us(f, n, batch, x_dtype, y_dtype), each = chain_us(f, n, x, y, batch, x_dtype, y_dtype, 1, false);
    return fused < 0.f || each < 0.f || fused < each;
}

// Whether the fused chain of ksmm_chain16r.hip is the fastest way through a chain that it takes.  Measured on chains of
// 256, 512 and 1024 features, us of the routes below / this one: batch-size-first always (1024 features at 197, 2050, 9408 and
// 25088 rows: fp32 14 / 11, 21 / 12, 51 / 31, 119 / 66; fp16 14 / 7, 16 / 8, 39 / 16, 81 / 28; e4m3 21 / 8, 24 / 9, 29 / 16,
// 54 / 26).  Batch-size-last fp32 and fp16 as well (fp32 13 / 11.5, 29 / 15.5, 49 / 29, 107 / 58; at 4800 columns, where the second
// round of chunks is nearly empty, 24 / 21; fp16, whose routes below are the kernel for whole vectors, ksmm_chain16.hip, 4800 columns
// 16.4 / 11.3, 9408 18.7 / 16.9, 25088 33.2 / 29.7, with e4m3 weights 18.6 / 17.4 and 33.1 / 30.4).  On e4m3 inputs that kernel, with
// its longer chunks, is ahead once this one needs a second round (4800 columns 12.9 / 11.7, 8192 13.3 / 12.3, 9408 14.5 / 17.0,
// 25088 24.0 / 26.7); on other row lengths it needs padded copies.  Narrower chains leave most of a workgroup idle: one
// round only.
bool fused_rows_pay(const ksmm_factor_desc *f, int n, const void *x, void *y, int64_t batch, int x_dtype, int y_dtype, int bs_last)
{
    if (chain16r_run(f, n, x, y, batch, x_dtype, y_dtype, bs_last ? 1 : 0, false, nullptr, nullptr) != KSMM_OK) return false;
    const int64_t features = (int64_t)f[0].a * f[0].c * f[0].d, round = 256 * 16;
    if (features < 256) return batch <= round;
    if (!bs_last || x_dtype != KSMM_FP8_E4M3) return true;
    return batch <= 2 * round || chain16_run(f, n, x, y, batch, x_dtype, y_dtype, 1, false, nullptr, nullptr) != KSMM_OK;
}

// Whether a chain that has a transposed or padded-rows route should take it.
bool chain_route_pays(const ksmm_factor_desc *f, int n, const void *x, void *y, int64_t batch, int x_dtype, int y_dtype, int bs_last,
                      bool fuse)
{
    const float direct = chain_us(f, n, x, y, batch, x_dtype, y_dtype, bs_last, false);
    if (direct < 0.f) return true;
    const int64_t bp = padded_batch(batch);
    float middle = chain_us(f, n, x, y, batch, x_dtype, y_dtype, bs_last, true);
    const float fused = fuse ? chain16_us(f, n, bp, x_dtype, y_dtype) : -1.f;
    if (fused >= 0.f && (middle < 0.f || fused < middle)) middle = fused;
    if (middle < 0.f) return true;
    const ksmm_factor_desc &l = f[n - 1];
    return copy_us((int64_t)f[0].a * f[0].c * f[0].d, batch, bp, (int)dtype_size(x_dtype), !bs_last) +
               copy_us((int64_t)l.a * l.b * l.d, batch, bp, (int)dtype_size(y_dtype), !bs_last) + middle < direct;
}

// What a chain cannot do without (a chain with decoded weights uses more, see decode_pays)
int64_t chain_layout(const ksmm_factor_desc *factors, int n_factors, int64_t batch, int x_dtype, int y_dtype, int bs_last)
{
    int rc = check_chain(factors, n_factors, batch, x_dtype, y_dtype);
    if (rc != KSMM_OK) return rc;
    const int64_t nb = chain_wants_transposed(factors, n_factors, batch, x_dtype, y_dtype, bs_last) ||
                               chain_wants_padded(factors, n_factors, batch, x_dtype, y_dtype, bs_last)
                           ? padded_batch(batch) : 0;
    if (nb == 0) return ksmm_chain_workspace(factors, n_factors, batch, y_dtype);
    int64_t widest = 0;
    for (int i = 0; i < n_factors; ++i) {
        int64_t o = (int64_t)factors[i].a * factors[i].b * factors[i].d;
        if (o > widest) widest = o;
    }
    const int64_t in0 = (int64_t)factors[0].a * factors[0].c * factors[0].d;
    return align256(in0 * nb * (int64_t)dtype_size(x_dtype)) +
           2 * align256(widest * nb * (int64_t)dtype_size(y_dtype));
}

// Predicted time of a chain by the faster of its routes (< 0: no price); *copies: that is the one between copies
float chain_best_us(const ksmm_factor_desc *f, int n, int64_t batch, int x_dtype, int y_dtype, int bs_last, bool *copies)
{
    *copies = false;
    const float direct = chain_us(f, n, nullptr, nullptr, batch, x_dtype, y_dtype, bs_last, false);
    if (!(bs_last ? chain_wants_padded(f, n, batch, x_dtype, y_dtype, 1) : chain_wants_transposed(f, n, batch, x_dtype, y_dtype, 0))) return direct;
    const float middle = chain_us(f, n, nullptr, nullptr, batch, x_dtype, y_dtype, bs_last, true);
    if (middle < 0.f) return direct;
    const int64_t bp = padded_batch(batch);
    const ksmm_factor_desc &l = f[n - 1];
    const float route = middle + copy_us((int64_t)f[0].a * f[0].c * f[0].d, batch, bp, (int)dtype_size(x_dtype), !bs_last) +
                        copy_us((int64_t)l.a * l.b * l.d, batch, bp, (int)dtype_size(y_dtype), !bs_last);
    *copies = direct < 0.f || route < direct;
    return *copies ? route : direct;
}

// Factors of e4m3 weights on an fp16 input (all but the first of an e4m3 layer): the kernels that decode such weights
// on the way to LDS take up to twice the time of the fp16 ones, of which there are more.  Decoded once a call, in one
// launch for the chain and exactly, the weights run on those.  Whether that pays: `decoded` is the chain with such
// weights (w is not set).  The decoding is priced at a launch (4 us with its host time) and 3 bytes a weight, and has to be
// ahead by the error of the prices, unless it saves the copies of a route or a split-K kernel on thousands of rows, whose
// price is too low by up to 3: measured on the projections of feed-forward
// blocks of widths 192 .. 1024 at ten batches, what was predicted to take less than 0.855 of the time was 1.08 to 2.7 times
// faster, from there to 1 it was 0.88 to 1.4 times.  us a call without and with: (6,64,64,1)+(1,768,192,2) on
// 25088 columns 143 / 52, on rows 103 / 65, (3,64,256,1)+(1,64,64,3) on 4800 rows 36 / 15, (12,64,256,1)+(1,256,256,3) on
// 10070 rows 79 / 44, on 25088 125 / 101.
bool decode_pays(const ksmm_factor_desc *f, int n, int64_t batch, int x_dtype, int y_dtype, int bs_last, ksmm_factor_desc *decoded)
{
    if (batch < 512 || y_dtype != KSMM_F16) return false;
    int64_t weights = 0;
    bool split = false;
    for (int i = 0; i < n; ++i) {
        decoded[i] = f[i];
        if (f[i].w_dtype != KSMM_FP8_E4M3 || (i == 0 ? x_dtype : y_dtype) != KSMM_F16) continue;
        decoded[i].w_dtype = KSMM_F16;
        auto on_split = [&](int w_dtype) {
            const Choice c = pick_of(Problem{nullptr, nullptr, nullptr, batch, f[i].a, f[i].b, f[i].c, f[i].d, KSMM_F16, w_dtype, y_dtype,
                                             bs_last, 1.f, nullptr}, true).c;
            return c.algo == KSMM_ALGO_TILE && (c.variant >> 24) == 5;
        };
        split |= batch >= 4096 && on_split(KSMM_FP8_E4M3) && !on_split(KSMM_F16);
        weights += (int64_t)f[i].a * f[i].b * f[i].c * f[i].d;
    }
    if (weights == 0) return false;
    // (chains of one kernel read their weights once a workgroup)
    if (chain16r_run(f, n, nullptr, nullptr, batch, x_dtype, y_dtype, bs_last ? 1 : 0, false, nullptr, nullptr) == KSMM_OK) return false;
    // (short chains cannot win a launch back: no more than their own prices is looked up)
    const float direct = chain_us(f, n, nullptr, nullptr, batch, x_dtype, y_dtype, bs_last, false);
    if (direct >= 0.f && direct < 12.f) return false;
    bool copied, copied_then;
    const float now = chain_best_us(f, n, batch, x_dtype, y_dtype, bs_last, &copied);
    const float then = chain_best_us(decoded, n, batch, x_dtype, y_dtype, bs_last, &copied_then) + 4.f + (float)weights * 1.5e-6f;
    return now > 0.f && then > 4.f && then < ((split || copied) && !copied_then ? 1.f : 0.855f) * now;
}

// Whether two factors run in one launch (ksmm_pair.hip): where that is priced below the other routes by PAIR_AHEAD.  Of 16270 measured
// chains (see pair_us) it is so in 5790, which take 0.73 to 0.84 of the time of two launches by type and layout; 2.2 percent
// of them are more than 3 percent slower (9 percent of feature-major fp32 and e4m3 chains, whose two launches are priced too high by most,
// if those need to be ahead by 0.7 only).
// A call that goes to the GPU as it is made costs the host 6.1 us with one launch and 9.7 with two, for which the GPU waits: there, up
// to a time of HOST_US it may be priced up to a microsecond later.  (6,64,64,1)+(1,768,192,2) fp32 on 32 columns 8.9 us on the GPU
// for 8.0, but 8.8 a call for 9.6.  In a graph that waits for nobody, the GPU's time alone decides.
constexpr float PAIR_AHEAD = 0.5f, PAIR_AHEAD_LAST = 1.f /* fp32 and e4m3 */, HOST_US = 9.5f;
struct PairChoice {
    PairShape shape;
    bool on_gpu, on_call;  // in a graph, and as a call of its own
};
PairChoice pair_choice(const ksmm_factor_desc *f, int n, int64_t batch, int x_dtype, int y_dtype, int bs_last)
{
    PairChoice c{{1, 1}, false, false};
    float us = pair_us(f, n, batch, x_dtype, y_dtype, bs_last, &c.shape);
    if (us < 0.f) return c;
    bool copies;
    float best = chain_best_us(f, n, batch, x_dtype, y_dtype, bs_last, &copies);
    ksmm_factor_desc decoded[2];
    if (decode_pays(f, n, batch, x_dtype, y_dtype, bs_last, decoded)) best = fminf(best, chain_best_us(decoded, n, batch, x_dtype, y_dtype, bs_last, &copies) + 4.f);
    us += bs_last && f[0].w_dtype != KSMM_F16 ? PAIR_AHEAD_LAST : PAIR_AHEAD;
    c.on_gpu = us < best;
    c.on_call = us < best + fminf(fmaxf(HOST_US - best, 0.f), 1.f);
    return c;
}

// Whether a stream's launches go into a graph.  (The default stream's cannot, and asking about it fails while another one is captured.)
bool captured(hipStream_t stream)
{
    hipStreamCaptureStatus status;
    return stream && hipStreamIsCapturing(stream, &status) == hipSuccess && status == hipStreamCaptureStatusActive;
}

// A function of the sizes and types, and where these leave it open of whether the stream is captured; asked up to three times
// a call: each thread remembers its last answers (2 us otherwise, of a call of 10), in sets of four as pick_of does: two layers of
// a network that share an entry would ask anew each call.
bool pair_pays(const ksmm_factor_desc *f, int n, int64_t batch, int x_dtype, int y_dtype, int bs_last, hipStream_t stream, PairShape *shape)
{
    if (n != 2 || f[0].d != 1 || (f[0].b == 16 && f[0].c == 16)) return false;  // (radix-16 chains have kernels of their own)
    struct Entry {
        int64_t batch;  // 0: empty
        int key[13];
        PairChoice choice;
    };
    constexpr unsigned SETS = 64, WAYS = 4;
    static thread_local Entry memo[SETS][WAYS];
    static thread_local uint8_t oldest[SETS];
    const int key[13] = {f[0].a, f[0].b, f[0].c, f[0].d, f[0].w_dtype, f[1].a, f[1].b, f[1].c, f[1].d, f[1].w_dtype, x_dtype, y_dtype, bs_last != 0};
    uint64_t h = (uint64_t)batch;
    for (int v : key) h = (h ^ (uint64_t)v) * 0x9E3779B97F4A7C15ull;
    const unsigned set = (h >> 40) % SETS;
    const Entry *hit = nullptr;
    for (const Entry &e : memo[set])
        if (e.batch == batch && memcmp(e.key, key, sizeof(key)) == 0) hit = &e;
    if (!hit) {
        Entry &e = memo[set][oldest[set]++ % WAYS];
        e.batch = batch;
        memcpy(e.key, key, sizeof(key));
        e.choice = pair_choice(f, n, batch, x_dtype, y_dtype, bs_last);
        hit = &e;
    }
    *shape = hit->choice.shape;
    return hit->choice.on_gpu || (hit->choice.on_call && !captured(stream));
}

// Workspace of a chain with decoded weights: that of either chain, then (from *at) the fp16 weights
int64_t decode_layout(const ksmm_factor_desc *f, const ksmm_factor_desc *decoded, int n, int64_t batch, int x_dtype, int y_dtype,
                      int bs_last, int64_t *at)
{
    const int64_t one = chain_layout(f, n, batch, x_dtype, y_dtype, bs_last), two = chain_layout(decoded, n, batch, x_dtype, y_dtype, bs_last);
    *at = align256(one > two ? one : two);
    int64_t bytes = *at;
    for (int i = 0; i < n; ++i)
        if (decoded[i].w_dtype != f[i].w_dtype) bytes += align256((int64_t)f[i].a * f[i].b * f[i].c * f[i].d * 2);
    return bytes;
}

// The chain launcher behind ksmm_chain_forward, ksmm_chain_forward_ep and
// ksmm_chain_forward_static: `ep` (may be null) belongs to the last factor, `x_scale` (device
// memory, may be null) multiplies the first one's scale.
int chain_forward_impl(const ksmm_factor_desc *factors, int n_factors, const void *x, void *y, void *workspace,
                       int64_t workspace_bytes, int64_t batch, int x_dtype, int y_dtype, int bs_last, int fuse,
                       const ksmm_epilogue *ep, void *stream, const float *x_scale = nullptr)
{
    int rc = check_chain(factors, n_factors, batch, x_dtype, y_dtype);
    if (rc != KSMM_OK) return rc;
    if ((rc = check_epilogue(ep)) != KSMM_OK) return rc;
    if (!x || !y) return KSMM_ERR_NULL_POINTER;
    for (int i = 0; i < n_factors; ++i)
        if (!factors[i].w) return KSMM_ERR_NULL_POINTER;
    const ksmm_factor_desc &last = factors[n_factors - 1];
    const int64_t in0 = (int64_t)factors[0].a * factors[0].c * factors[0].d;
    const int64_t out_n = (int64_t)last.a * last.b * last.d;
    const int64_t xbytes = in0 * batch * (int64_t)dtype_size(x_dtype);
    const int64_t ybytes = out_n * batch * (int64_t)dtype_size(y_dtype);
    if (overlaps(x, xbytes, y, ybytes)) return KSMM_ERR_ALIAS;
    if (workspace && workspace_bytes > 0) {
        if (overlaps(workspace, workspace_bytes, x, xbytes) || overlaps(workspace, workspace_bytes, y, ybytes))
            return KSMM_ERR_ALIAS;
        if (((uintptr_t)workspace & 15) != 0) return KSMM_ERR_WORKSPACE;
    }
    PairShape shape;
    if (fuse && pair_pays(factors, n_factors, batch, x_dtype, y_dtype, bs_last, (hipStream_t)stream, &shape)) {
        // (with the workspace that the other routes ask for: a call that lacks it is refused whichever route is the faster)
        const int64_t asked = chain_layout(factors, n_factors, batch, x_dtype, y_dtype, bs_last);
        if (asked <= 0 || (workspace && workspace_bytes >= asked))
            return pair_run(factors, n_factors, x, y, batch, x_dtype, y_dtype, bs_last, shape, (hipStream_t)stream, ep, x_scale);
    }
    ksmm_factor_desc decoded[KSMM_MAX_FACTORS];
    if (workspace && decode_pays(factors, n_factors, batch, x_dtype, y_dtype, bs_last, decoded)) {
        int64_t at;
        if (workspace_bytes >= decode_layout(factors, decoded, n_factors, batch, x_dtype, y_dtype, bs_last, &at)) {
            DecodeJob jobs[KSMM_MAX_FACTORS];
            int n_jobs = 0;
            char *to = (char *)workspace + at;
            for (int i = 0; i < n_factors; ++i) {
                if (decoded[i].w_dtype == factors[i].w_dtype) continue;
                const int64_t n = (int64_t)factors[i].a * factors[i].b * factors[i].c * factors[i].d;
                jobs[n_jobs++] = DecodeJob{factors[i].w, to, n};
                decoded[i].w = to;
                to += align256(n * 2);
            }
            if ((rc = decode_run(jobs, n_jobs, (hipStream_t)stream)) != KSMM_OK) return rc;
            return chain_forward_impl(decoded, n_factors, x, y, workspace, at, batch, x_dtype, y_dtype, bs_last, fuse, ep, stream, x_scale);
        }
    }
    auto ep_of = [&](int i) { return i == n_factors - 1 ? ep : nullptr; };
    if (fuse && fused_rows_pay(factors, n_factors, x, y, batch, x_dtype, y_dtype, bs_last)) {
        const int64_t asked = chain_layout(factors, n_factors, batch, x_dtype, y_dtype, bs_last);
        if (asked <= 0 || (workspace && workspace_bytes >= asked)) {
            rc = chain16r_run(factors, n_factors, x, y, batch, x_dtype, y_dtype, bs_last ? 1 : 0, true, (hipStream_t)stream, ep, x_scale);
            if (rc != KSMM_ERR_BAD_ALGO) return rc;
        }
    }
    // The whole chain in batch-size-last layout on workspace buffers: input x0 (nb columns), two
    // ping-pong buffers of `one` bytes at pp; *result = where the last factor's output is.
    auto run_bs_last = [&](const void *x0, char *pp, int64_t one, int64_t nb, const void **result) -> int {
        int rc2 = KSMM_ERR_BAD_ALGO;
        if (fuse && fused_pays(factors, n_factors, x0, pp, nb, x_dtype, y_dtype))
            rc2 = chain16_run(factors, n_factors, x0, pp, nb, x_dtype, y_dtype, 1, true, (hipStream_t)stream, ep, x_scale);
        if (rc2 == KSMM_OK) {
            *result = pp;
            return KSMM_OK;
        }
        if (rc2 != KSMM_ERR_BAD_ALGO) return rc2;
        const void *cur = x0;
        int cur_dtype = x_dtype;
        for (int i = 0; i < n_factors; ++i) {
            void *dst = pp + (i & 1) * one;
            rc2 = factor_forward_impl(cur, factors[i].w, dst, nb, factors[i].a, factors[i].b, factors[i].c,
                                      factors[i].d, cur_dtype, factors[i].w_dtype, y_dtype, 1, factors[i].scale,
                                      KSMM_ALGO_AUTO, -1, ep_of(i), stream, i == 0 ? x_scale : nullptr);
            if (rc2 != KSMM_OK) return rc2;
            cur = dst;
            cur_dtype = y_dtype;
        }
        *result = cur;
        return KSMM_OK;
    };
    if (chain_wants_transposed(factors, n_factors, batch, x_dtype, y_dtype, bs_last)) {
        // transpose once, run the whole chain in batch-size-last layout, transpose back
        // (a workspace below what ksmm_chain_workspace_layout() asks for is an error, as it is for
        // ksmm_factor_forward_ws: the factor-by-factor route would land on the one-thread-per-output
        // kernel without a word)
        const int64_t need_t = chain_layout(factors, n_factors, batch, x_dtype, y_dtype, 0);
        if (!workspace || workspace_bytes < need_t) return KSMM_ERR_WORKSPACE;
        if (chain_route_pays(factors, n_factors, x, y, batch, x_dtype, y_dtype, 0, fuse != 0)) {
            const int64_t bp = padded_batch(batch);  // row length of the transposed copies
            const int64_t xt_bytes = align256(in0 * bp * (int64_t)dtype_size(x_dtype));
            char *xt = (char *)workspace;
            rc = transpose_run(x, xt, batch, in0, (int)dtype_size(x_dtype), (hipStream_t)stream, 0, bp);
            if (rc != KSMM_OK) return rc;
            const void *cur = nullptr;
            rc = run_bs_last(xt, xt + xt_bytes, (need_t - xt_bytes) / 2, bp, &cur);
            if (rc != KSMM_OK) return rc;
            return transpose_run(cur, y, out_n, batch, (int)dtype_size(y_dtype), (hipStream_t)stream, bp, 0);
        }
    } else if (chain_wants_padded(factors, n_factors, batch, x_dtype, y_dtype, bs_last)) {
        // pad the rows once, run the whole chain at the padded batch, cut the result rows back
        const int64_t need_p = chain_layout(factors, n_factors, batch, x_dtype, y_dtype, 1);
        if (!workspace || workspace_bytes < need_p) return KSMM_ERR_WORKSPACE;
        if (chain_route_pays(factors, n_factors, x, y, batch, x_dtype, y_dtype, 1, fuse != 0)) {
            const int64_t bp = padded_batch(batch);
            const int64_t xp_bytes = align256(in0 * bp * (int64_t)dtype_size(x_dtype));
            char *xp = (char *)workspace;
            rc = repitch_run(x, xp, in0, batch, bp, (int)dtype_size(x_dtype), (hipStream_t)stream);
            if (rc != KSMM_OK) return rc;
            const void *cur = nullptr;
            rc = run_bs_last(xp, xp + xp_bytes, (need_p - xp_bytes) / 2, bp, &cur);
            if (rc != KSMM_OK) return rc;
            return repitch_run(cur, y, out_n, bp, batch, (int)dtype_size(y_dtype), (hipStream_t)stream);
        }
    }
    if (fuse && (!bs_last || fused_pays(factors, n_factors, x, y, batch, x_dtype, y_dtype))) {
        // chains whose intermediates fit LDS run as one kernel (no workspace traffic)
        rc = chain16_run(factors, n_factors, x, y, batch, x_dtype, y_dtype, bs_last ? 1 : 0, true,
                         (hipStream_t)stream, ep, x_scale);
        if (rc != KSMM_ERR_BAD_ALGO) return rc;
    }
    const int64_t need = ksmm_chain_workspace(factors, n_factors, batch, y_dtype);
    if (n_factors > 1 && (!workspace || workspace_bytes < need)) return KSMM_ERR_WORKSPACE;
    char *buf[2] = {(char *)workspace, (char *)workspace + need / 2};
    const void *cur = x;
    int cur_dtype = x_dtype;
    for (int i = 0; i < n_factors; ++i) {
        void *dst = (i == n_factors - 1) ? y : (void *)buf[i & 1];
        rc = factor_forward_impl(cur, factors[i].w, dst, batch, factors[i].a, factors[i].b, factors[i].c,
                                 factors[i].d, cur_dtype, factors[i].w_dtype, y_dtype, bs_last, factors[i].scale,
                                 KSMM_ALGO_AUTO, -1, ep_of(i), stream, i == 0 ? x_scale : nullptr);
        if (rc != KSMM_OK) return rc;
        cur = dst;
        cur_dtype = y_dtype;
    }
    return KSMM_OK;
}

// Offsets in the workspace of a layer's backward pass
struct LayerBackward {
    int64_t dz, bias_sums;               // gradient of what the activation was applied to; partial sums of the bias's
    int64_t blocks[KSMM_MAX_FACTORS];    // transposed blocks of each factor
    int64_t sums[KSMM_MAX_FACTORS];      // partial sums of each weight gradient: all are added at the end
    int64_t grads[2];                    // gradient of factor i's input, 0 < i, at grads[i & 1]
    int64_t forward;                     // what the forward kernels of the transposed factors ask for
};

// bytes of it, or an error
int64_t layer_backward_layout(const ksmm_factor_desc *f, int n, int64_t batch, int dtype, int bs_last, int act, LayerBackward *l)
{
    if (dtype != KSMM_F32 && dtype != KSMM_F16) return KSMM_ERR_BAD_DTYPE;
    int rc = check_chain(f, n, batch, dtype, dtype);
    if (rc != KSMM_OK) return rc;
    const int64_t es = (int64_t)dtype_size(dtype), out = (int64_t)f[n - 1].a * f[n - 1].b * f[n - 1].d;
    int64_t at = 0, widest[2] = {0, 0}, forward = 0;
    auto take = [&](int64_t bytes) {
        const int64_t was = at;
        at += align256(bytes);
        return was;
    };
    l->dz = take(act != KSMM_ACT_NONE ? out * batch * es : 0);
    l->bias_sums = take(4 * act_bwd_partial_floats(batch, out, dtype, bs_last));
    for (int i = 0; i < n; ++i) {
        l->blocks[i] = take((int64_t)f[i].a * f[i].b * f[i].c * f[i].d * es);
        l->sums[i] = take(wgrad_partial_bytes(batch, f[i].a, f[i].b, f[i].c, f[i].d, dtype, bs_last));
        const int64_t need = ksmm_factor_workspace(batch, f[i].a, f[i].c, f[i].b, f[i].d, dtype, dtype, dtype, bs_last);
        if (need < 0) return need;
        if (need > forward) forward = need;
        const int64_t in = (int64_t)f[i].a * f[i].c * f[i].d;
        if (i > 0 && in > widest[i & 1]) widest[i & 1] = in;
    }
    l->grads[0] = take(widest[0] * batch * es);
    l->grads[1] = take(widest[1] * batch * es);
    l->forward = take(forward);
    return at;
}

// ---- scratch of ksmm_chain_forward_static ---------------------------------------------------
// The device address of the array is asked for once per device, with that device current, and
// kept; kernels and copies only ever see that address.
constexpr int MAX_DEVICES = 64;
std::atomic<void *> scratch_ptr[MAX_DEVICES];

int static_scratch(void **out)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return KSMM_ERR_LAUNCH;
    void *ptr = scratch_ptr[dev].load(std::memory_order_acquire);
    if (!ptr) {
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return KSMM_ERR_LAUNCH;
        scratch_ptr[dev].store(ptr, std::memory_order_release);  // racing callers store the same address
    }
    *out = ptr;
    return KSMM_OK;
}

}  // namespace

extern "C" {

int ksmm_version(void) { return KSMM_VERSION; }

const char *ksmm_strerror(int status)
{
    switch (status) {
    case KSMM_OK: return "ok";
    case KSMM_ERR_NULL_POINTER: return "null tensor pointer";
    case KSMM_ERR_BAD_PATTERN: return "pattern (a,b,c,d) must be four positive integers";
    case KSMM_ERR_BAD_BATCH: return "batch size must be positive";
    case KSMM_ERR_BAD_DTYPE: return "unsupported data type combination";
    case KSMM_ERR_TOO_LARGE: return "tensor too large (2^31 elements or more)";
    case KSMM_ERR_BAD_ALGO: return "kernel family/variant unknown or not applicable to this problem";
    case KSMM_ERR_LAUNCH: return "HIP kernel launch failed";
    case KSMM_ERR_CHAIN_MISMATCH: return "consecutive factors have incompatible sizes";
    case KSMM_ERR_WORKSPACE: return "workspace missing or too small";
    case KSMM_ERR_BAD_CHAIN: return "bad number of factors";
    case KSMM_ERR_ALIAS: return "output, input or workspace overlap";
    case KSMM_ERR_BAD_EPILOGUE: return "unknown activation in the epilogue";
    default: return "unknown ksmm status";
    }
}

int ksmm_validate(int64_t batch, int a, int b, int c, int d, int x_dtype, int w_dtype,
                  int y_dtype, int bs_last)
{
    (void)bs_last;
    return check_shape(batch, a, b, c, d, x_dtype, w_dtype, y_dtype);
}

int ksmm_query_tile(int64_t batch, int a, int b, int c, int d, int x_dtype, int w_dtype,
                    int y_dtype, int bs_last, int algo, ksmm_tile *out)
{
    if (!out) return KSMM_ERR_NULL_POINTER;
    int rc = check_shape(batch, a, b, c, d, x_dtype, w_dtype, y_dtype);
    if (rc != KSMM_OK) return rc;
    Problem p{nullptr, nullptr, nullptr, batch, a, b, c, d, x_dtype, w_dtype, y_dtype,
              bs_last ? 1 : 0, 1.f, nullptr};
    memset(out, 0, sizeof(*out));
    return dispatch(p, algo, -1, false, out);
}

int ksmm_query_tile_variant(int64_t batch, int a, int b, int c, int d, int x_dtype, int w_dtype,
                            int y_dtype, int bs_last, int algo, int variant, ksmm_tile *out)
{
    if (!out) return KSMM_ERR_NULL_POINTER;
    int rc = check_shape(batch, a, b, c, d, x_dtype, w_dtype, y_dtype);
    if (rc != KSMM_OK) return rc;
    Problem p{nullptr, nullptr, nullptr, batch, a, b, c, d, x_dtype, w_dtype, y_dtype,
              bs_last ? 1 : 0, 1.f, nullptr};
    memset(out, 0, sizeof(*out));
    return dispatch(p, algo, variant, false, out);
}

int ksmm_price(int64_t batch, int a, int b, int c, int d, int x_dtype, int w_dtype, int y_dtype, int bs_last,
               int algo, int variant, float *us)
{
    if (!us) return KSMM_ERR_NULL_POINTER;
    ksmm_tile t;
    const int rc = ksmm_query_tile_variant(batch, a, b, c, d, x_dtype, w_dtype, y_dtype, bs_last, algo, variant, &t);
    if (rc != KSMM_OK) return rc;
    if (t.algo == KSMM_ALGO_GENERIC && t.variant >= GENERIC_TILE) {  // a tile instance by the number it is reported under
        t.algo = KSMM_ALGO_TILE;
        t.variant -= GENERIC_TILE;
    }
    const Problem p{nullptr, nullptr, nullptr, batch, a, b, c, d, x_dtype, w_dtype, y_dtype, bs_last ? 1 : 0, 1.f, nullptr};
    *us = predicted_us(p, t);
    return KSMM_OK;
}

int ksmm_tuned_count(void) { return N_TUNED; }

int ksmm_tuned_row(int index, int row[10])
{
    if (!row) return KSMM_ERR_NULL_POINTER;
    if (index < 0 || index >= N_TUNED) return KSMM_ERR_BAD_ALGO;
    const TunedRow &r = tuned_rows[index];
    int variant = -1;  // the row's instance is gone from the library: the heuristics serve the pattern
    if (!resolve_variant(r.algo, r.id, r.param, r.combo, r.bs_last, &variant)) variant = -1;
    const int v[10] = {r.a, r.b, r.c, r.d, r.combo, r.bs_last, r.algo, (int)r.id, r.param, variant};
    for (int i = 0; i < 10; ++i) row[i] = v[i];
    return KSMM_OK;
}

int ksmm_variant_id(int algo, int variant, int x_dtype, int w_dtype, int y_dtype, int bs_last,
                    uint32_t *id, int *param)
{
    if (!id || !param) return KSMM_ERR_NULL_POINTER;
    const int combo = combo_of(x_dtype, w_dtype, y_dtype);
    if (combo < 0) return KSMM_ERR_BAD_DTYPE;
    return describe_variant(algo, variant, combo, bs_last ? 1 : 0, id, param) ? KSMM_OK : KSMM_ERR_BAD_ALGO;
}

int ksmm_variant_from_id(int algo, uint32_t id, int param, int x_dtype, int w_dtype, int y_dtype,
                         int bs_last, int *variant)
{
    if (!variant) return KSMM_ERR_NULL_POINTER;
    const int combo = combo_of(x_dtype, w_dtype, y_dtype);
    if (combo < 0) return KSMM_ERR_BAD_DTYPE;
    return resolve_variant(algo, id, param, combo, bs_last ? 1 : 0, variant) ? KSMM_OK : KSMM_ERR_BAD_ALGO;
}

int ksmm_factor_forward_algo(const void *x, const void *w, void *y, int64_t batch, int a,
                             int b, int c, int d, int x_dtype, int w_dtype, int y_dtype,
                             int bs_last, float scale, int algo, int variant, void *stream)
{
    return factor_forward_impl(x, w, y, batch, a, b, c, d, x_dtype, w_dtype, y_dtype, bs_last, scale, algo,
                               variant, nullptr, stream);
}

int ksmm_factor_forward(const void *x, const void *w, void *y, int64_t batch, int a, int b,
                        int c, int d, int x_dtype, int w_dtype, int y_dtype, int bs_last,
                        float scale, void *stream)
{
    return factor_forward_impl(x, w, y, batch, a, b, c, d, x_dtype, w_dtype, y_dtype, bs_last, scale,
                               KSMM_ALGO_AUTO, -1, nullptr, stream);
}

int64_t ksmm_factor_workspace(int64_t batch, int a, int b, int c, int d, int x_dtype, int w_dtype,
                              int y_dtype, int bs_last)
{
    int rc = check_shape(batch, a, b, c, d, x_dtype, w_dtype, y_dtype);
    if (rc != KSMM_OK) return rc;
    Problem p{nullptr, nullptr, nullptr, batch, a, b, c, d, x_dtype, w_dtype, y_dtype,
              bs_last ? 1 : 0, 1.f, nullptr};
    // both routes stage the input and the output: transposed, or with rows padded to the vector
    const int64_t nb = wants_transposed(p) || wants_padded(p) ? padded_batch(batch) : 0;
    if (nb == 0) return 0;
    return align256((int64_t)a * c * d * nb * (int64_t)dtype_size(x_dtype)) +
           align256((int64_t)a * b * d * nb * (int64_t)dtype_size(y_dtype));
}

int ksmm_factor_forward_ws(const void *x, const void *w, void *y, int64_t batch, int a, int b,
                           int c, int d, int x_dtype, int w_dtype, int y_dtype, int bs_last,
                           float scale, void *workspace, int64_t workspace_bytes, void *stream)
{
    return factor_forward_ws_impl(x, w, y, batch, a, b, c, d, x_dtype, w_dtype, y_dtype, bs_last, scale, nullptr,
                                  workspace, workspace_bytes, stream);
}

int ksmm_factor_forward_ep(const void *x, const void *w, void *y, int64_t batch, int a, int b,
                           int c, int d, int x_dtype, int w_dtype, int y_dtype, int bs_last,
                           float scale, const ksmm_epilogue *epilogue, void *workspace,
                           int64_t workspace_bytes, void *stream)
{
    return factor_forward_ws_impl(x, w, y, batch, a, b, c, d, x_dtype, w_dtype, y_dtype, bs_last, scale, epilogue,
                                  workspace, workspace_bytes, stream);
}

int64_t ksmm_chain_workspace(const ksmm_factor_desc *factors, int n_factors, int64_t batch,
                             int y_dtype)
{
    if (!factors) return KSMM_ERR_NULL_POINTER;
    if (n_factors < 1 || n_factors > KSMM_MAX_FACTORS) return KSMM_ERR_BAD_CHAIN;
    if (batch < 1) return KSMM_ERR_BAD_BATCH;
    if (!dtype_known(y_dtype)) return KSMM_ERR_BAD_DTYPE;
    int64_t widest = 0;
    for (int i = 0; i + 1 < n_factors; ++i) {
        if (factors[i].a < 1 || factors[i].b < 1 || factors[i].d < 1) return KSMM_ERR_BAD_PATTERN;
        int64_t o = (int64_t)factors[i].a * factors[i].b * factors[i].d;
        if (o > widest) widest = o;
    }
    // two buffers, each rounded up to 256 bytes so that both stay 256-byte aligned
    int64_t one = (widest * batch * (int64_t)dtype_size(y_dtype) + 255) / 256 * 256;
    return n_factors > 1 ? 2 * one : 0;
}

int64_t ksmm_chain_workspace_layout(const ksmm_factor_desc *factors, int n_factors, int64_t batch,
                                    int x_dtype, int y_dtype, int bs_last)
{
    const int64_t need = chain_layout(factors, n_factors, batch, x_dtype, y_dtype, bs_last);
    if (need < 0) return need;
    ksmm_factor_desc decoded[KSMM_MAX_FACTORS];
    if (!decode_pays(factors, n_factors, batch, x_dtype, y_dtype, bs_last, decoded)) return need;
    int64_t at;
    return decode_layout(factors, decoded, n_factors, batch, x_dtype, y_dtype, bs_last, &at);
}

int ksmm_chain_forward(const ksmm_factor_desc *factors, int n_factors, const void *x, void *y,
                       void *workspace, int64_t workspace_bytes, int64_t batch, int x_dtype,
                       int y_dtype, int bs_last, int fuse, void *stream)
{
    return chain_forward_impl(factors, n_factors, x, y, workspace, workspace_bytes, batch, x_dtype, y_dtype,
                              bs_last, fuse, nullptr, stream);
}

int ksmm_chain_forward_ep(const ksmm_factor_desc *factors, int n_factors, const void *x, void *y,
                          void *workspace, int64_t workspace_bytes, int64_t batch, int x_dtype,
                          int y_dtype, int bs_last, int fuse, const ksmm_epilogue *epilogue,
                          void *stream)
{
    return chain_forward_impl(factors, n_factors, x, y, workspace, workspace_bytes, batch, x_dtype, y_dtype,
                              bs_last, fuse, epilogue, stream);
}

int ksmm_chain_forward_fused(const ksmm_factor_desc *factors, int n_factors, const void *x, void *y, int64_t batch, int x_dtype,
                             int y_dtype, int bs_last, const ksmm_epilogue *epilogue, void *stream)
{
    int rc = check_chain(factors, n_factors, batch, x_dtype, y_dtype);
    if (rc != KSMM_OK) return rc;
    if ((rc = check_epilogue(epilogue)) != KSMM_OK) return rc;
    if (!x || !y) return KSMM_ERR_NULL_POINTER;
    for (int i = 0; i < n_factors; ++i)
        if (!factors[i].w) return KSMM_ERR_NULL_POINTER;
    const ksmm_factor_desc &l = factors[n_factors - 1];
    if (overlaps(x, (int64_t)factors[0].a * factors[0].c * factors[0].d * batch * (int64_t)dtype_size(x_dtype), y,
                 (int64_t)l.a * l.b * l.d * batch * (int64_t)dtype_size(y_dtype)))
        return KSMM_ERR_ALIAS;
    PairShape shape;
    if (pair_pays(factors, n_factors, batch, x_dtype, y_dtype, bs_last ? 1 : 0, (hipStream_t)stream, &shape))
        return pair_run(factors, n_factors, x, y, batch, x_dtype, y_dtype, bs_last ? 1 : 0, shape, (hipStream_t)stream, epilogue);
    if (!fused_rows_pay(factors, n_factors, x, y, batch, x_dtype, y_dtype, bs_last)) return KSMM_ERR_BAD_ALGO;
    return chain16r_run(factors, n_factors, x, y, batch, x_dtype, y_dtype, bs_last ? 1 : 0, true, (hipStream_t)stream, epilogue);
}

// workspace of the chain that quantises its input: codes | partial maxima | scale | the chain's own
static int64_t quant_layout(const ksmm_factor_desc *f, int64_t batch, int64_t *maxima)
{
    *maxima = align256((int64_t)f[0].a * f[0].c * f[0].d * batch);
    return *maxima + align256(quantize_scratch_bytes()) + 256;
}

int64_t ksmm_chain_quant_workspace(const ksmm_factor_desc *factors, int n_factors, int64_t batch, int x_dtype, int y_dtype,
                                   int bs_last)
{
    if (x_dtype != KSMM_F32 && x_dtype != KSMM_F16) return KSMM_ERR_BAD_DTYPE;
    const int64_t chain = ksmm_chain_workspace_layout(factors, n_factors, batch, KSMM_FP8_E4M3, y_dtype, bs_last);
    if (chain < 0) return chain;
    int64_t maxima;
    return quant_layout(factors, batch, &maxima) + chain;
}

int ksmm_chain_forward_quant(const ksmm_factor_desc *factors, int n_factors, const void *x, void *y, void *workspace,
                             int64_t workspace_bytes, int64_t batch, int x_dtype, int y_dtype, int bs_last, int fuse,
                             const ksmm_epilogue *epilogue, void *stream)
{
    // (more is asked for than a chain without decoded weights needs: with less it runs without them)
    const int64_t asked = ksmm_chain_quant_workspace(factors, n_factors, batch, x_dtype, y_dtype, bs_last);
    if (asked < 0) return (int)asked;
    int64_t maxima;
    const int64_t own = quant_layout(factors, batch, &maxima);
    int64_t need = own + chain_layout(factors, n_factors, batch, KSMM_FP8_E4M3, y_dtype, bs_last);
    int rc = check_epilogue(epilogue);
    if (rc != KSMM_OK) return rc;
    if (!x || !y) return KSMM_ERR_NULL_POINTER;
    for (int i = 0; i < n_factors; ++i)
        if (!factors[i].w) return KSMM_ERR_NULL_POINTER;
    if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 15) != 0) return KSMM_ERR_WORKSPACE;
    if (workspace_bytes >= asked) need = asked;
    const ksmm_factor_desc &last = factors[n_factors - 1];
    const int64_t n = (int64_t)factors[0].a * factors[0].c * factors[0].d * batch, xbytes = n * (int64_t)dtype_size(x_dtype);
    const int64_t ybytes = (int64_t)last.a * last.b * last.d * batch * (int64_t)dtype_size(y_dtype);
    if (overlaps(x, xbytes, y, ybytes) || overlaps(workspace, need, x, xbytes) || overlaps(workspace, need, y, ybytes))
        return KSMM_ERR_ALIAS;
    char *ws = (char *)workspace;
    float *scale = (float *)(ws + own - 256);
    rc = quantize_run(x, x_dtype, ws, scale, ws + maxima, n, (hipStream_t)stream);
    if (rc != KSMM_OK) return rc;
    return chain_forward_impl(factors, n_factors, ws, y, need > own ? ws + own : nullptr, need - own, batch, KSMM_FP8_E4M3, y_dtype,
                              bs_last, fuse, epilogue, stream, scale);
}

int64_t ksmm_factor_backward_workspace(int64_t batch, int a, int b, int c, int d, int dtype, int bs_last)
{
    int rc = check_shape(batch, a, b, c, d, dtype, dtype, dtype);
    if (rc != KSMM_OK) return rc;
    if (dtype != KSMM_F32 && dtype != KSMM_F16) return KSMM_ERR_BAD_DTYPE;
    const int64_t nnz = (int64_t)a * b * c * d;
    // transposed blocks (input gradient) | fp32 partial sums, one slice per batch split (weight
    // gradient) | what the forward kernels of the transposed factor ask for
    const int64_t fwd = ksmm_factor_workspace(batch, a, c, b, d, dtype, dtype, dtype, bs_last);
    if (fwd < 0) return fwd;
    return align256(nnz * (int64_t)dtype_size(dtype)) + wgrad_partial_bytes(batch, a, b, c, d, dtype, bs_last ? 1 : 0) + align256(fwd);
}

int ksmm_factor_backward_input(const void *dy, const void *w, void *dx, int64_t batch, int a, int b,
                               int c, int d, int dtype, int bs_last, float scale, void *workspace,
                               int64_t workspace_bytes, void *stream)
{
    const int64_t need = ksmm_factor_backward_workspace(batch, a, b, c, d, dtype, bs_last);
    if (need < 0) return (int)need;
    if (!dy || !w || !dx) return KSMM_ERR_NULL_POINTER;
    if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 15) != 0) return KSMM_ERR_WORKSPACE;
    const int64_t nnz = (int64_t)a * b * c * d;
    char *wt = (char *)workspace;
    char *fwd_ws = wt + align256(nnz * (int64_t)dtype_size(dtype)) + wgrad_partial_bytes(batch, a, b, c, d, dtype, bs_last ? 1 : 0);
    const TransposeJob job{w, wt, (int64_t)a * d, b, c};
    int rc = block_transpose_run(&job, 1, dtype, (hipStream_t)stream);
    if (rc != KSMM_OK) return rc;
    // dX = K^T dY: the factor with pattern (a, c, b, d) and transposed blocks
    return factor_forward_ws_impl(dy, wt, dx, batch, a, c, b, d, dtype, dtype, dtype, bs_last, scale, nullptr, fwd_ws,
                                  workspace_bytes - (fwd_ws - wt), stream);
}

int ksmm_factor_backward_weight(const void *dy, const void *x, void *dw, int64_t batch, int a, int b,
                                int c, int d, int dtype, int bs_last, float scale, void *workspace,
                                int64_t workspace_bytes, void *stream)
{
    const int64_t need = ksmm_factor_backward_workspace(batch, a, b, c, d, dtype, bs_last);
    if (need < 0) return (int)need;
    if (!dy || !x || !dw) return KSMM_ERR_NULL_POINTER;
    if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 15) != 0) return KSMM_ERR_WORKSPACE;
    const int64_t nnz = (int64_t)a * b * c * d;
    float *acc = (float *)((char *)workspace + align256(nnz * (int64_t)dtype_size(dtype)));
    FinishJob rest;
    const int rc = wgrad_run(dy, x, dw, acc, batch, a, b, c, d, dtype, bs_last ? 1 : 0, scale, (hipStream_t)stream, &rest);
    return rc == KSMM_OK ? finish_run(&rest, 1, dtype, (hipStream_t)stream) : rc;
}

int64_t ksmm_epilogue_backward_workspace(int64_t batch, int64_t features, int dtype, int bs_last)
{
    if (features < 1) return KSMM_ERR_BAD_PATTERN;
    if (batch < 1) return KSMM_ERR_BAD_BATCH;
    if (dtype != KSMM_F32 && dtype != KSMM_F16) return KSMM_ERR_BAD_DTYPE;
    if (batch > 0x7fffffffLL / features) return KSMM_ERR_TOO_LARGE;
    return align256(4 * act_bwd_partial_floats(batch, features, dtype, bs_last ? 1 : 0));
}

int ksmm_epilogue_backward(const void *dy, const void *z, void *dz, void *dbias, int64_t batch, int64_t features, int dtype,
                           int bs_last, int act, void *workspace, int64_t workspace_bytes, void *stream)
{
    const int64_t need = ksmm_epilogue_backward_workspace(batch, features, dtype, bs_last);
    if (need < 0) return (int)need;
    if (act != KSMM_ACT_NONE && act != KSMM_ACT_GELU) return KSMM_ERR_BAD_EPILOGUE;
    if (!dy || (act != KSMM_ACT_NONE && (!z || !dz))) return KSMM_ERR_NULL_POINTER;
    if (dbias && (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 15) != 0)) return KSMM_ERR_WORKSPACE;
    if (!dbias && act == KSMM_ACT_NONE) return KSMM_OK;
    FinishJob rest;
    const int rc = act_bwd_run(dy, z, dz, dbias, (float *)workspace, batch, features, dtype, bs_last ? 1 : 0, act, (hipStream_t)stream, &rest);
    return rc == KSMM_OK ? finish_run(&rest, 1, dtype, (hipStream_t)stream) : rc;
}

int64_t ksmm_layer_backward_workspace(const ksmm_factor_desc *factors, int n_factors, int64_t batch, int dtype, int bs_last,
                                      int act)
{
    LayerBackward l;
    return layer_backward_layout(factors, n_factors, batch, dtype, bs_last ? 1 : 0, act, &l);
}

int ksmm_layer_backward(const ksmm_factor_desc *factors, int n_factors, const void *const *inputs, const void *z, const void *dy,
                        void *dx, void *const *dw, void *dbias, void *workspace, int64_t workspace_bytes, int64_t batch, int dtype,
                        int bs_last, int act, void *stream)
{
    LayerBackward l;
    const int64_t need = layer_backward_layout(factors, n_factors, batch, dtype, bs_last ? 1 : 0, act, &l);
    if (need < 0) return (int)need;
    if (act != KSMM_ACT_NONE && act != KSMM_ACT_GELU) return KSMM_ERR_BAD_EPILOGUE;
    if (!inputs || !dw || !dy || (act != KSMM_ACT_NONE && !z)) return KSMM_ERR_NULL_POINTER;
    if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 15) != 0) return KSMM_ERR_WORKSPACE;
    int lowest = -1;  // the first factor that a gradient goes through or to
    for (int i = n_factors - 1; i >= 0; --i) {
        if (dw[i] && !inputs[i]) return KSMM_ERR_NULL_POINTER;
        if (dw[i] || dx) lowest = i;
    }
    if (dx) lowest = 0;
    char *ws = (char *)workspace;
    const hipStream_t s = (hipStream_t)stream;
    const ksmm_factor_desc &last = factors[n_factors - 1];
    const int64_t out_size = (int64_t)last.a * last.b * last.d;
    FinishJob rest[KSMM_MAX_FACTORS + 1];
    TransposeJob flips[KSMM_MAX_FACTORS];
    int jobs = 0, n_flips = 0, rc;
    const void *grad = dy;
    if (act != KSMM_ACT_NONE || dbias) {
        void *dz = act != KSMM_ACT_NONE ? ws + l.dz : nullptr;
        rc = act_bwd_run(dy, z, dz, dbias, (float *)(ws + l.bias_sums), batch, out_size, dtype, bs_last ? 1 : 0, act, s, &rest[jobs++]);
        if (rc != KSMM_OK) return rc;
        if (dz) grad = dz;
    }
    // factors whose input's gradient is needed: all behind the first one wanted, and that one for dx
    for (int i = lowest < 0 ? n_factors : dx ? 0 : lowest + 1; i < n_factors; ++i) {
        const ksmm_factor_desc &f = factors[i];
        if (!f.w) return KSMM_ERR_NULL_POINTER;
        flips[n_flips++] = TransposeJob{f.w, ws + l.blocks[i], (int64_t)f.a * f.d, f.b, f.c};
    }
    rc = block_transpose_run(flips, n_flips, dtype, s);
    if (rc != KSMM_OK) return rc;
    for (int i = n_factors - 1; i >= 0 && i >= lowest && lowest >= 0; --i) {
        const ksmm_factor_desc &f = factors[i];
        if (dw[i]) {
            rc = wgrad_run(grad, inputs[i], dw[i], (float *)(ws + l.sums[i]), batch, f.a, f.b, f.c, f.d, dtype, bs_last ? 1 : 0,
                           f.scale, s, &rest[jobs++]);
            if (rc != KSMM_OK) return rc;
        }
        if (i == lowest && !dx) break;
        void *to = i == 0 ? dx : ws + l.grads[i & 1];
        // dX = K^T dY: the factor with pattern (a, c, b, d) and transposed blocks
        rc = factor_forward_ws_impl(grad, ws + l.blocks[i], to, batch, f.a, f.c, f.b, f.d, dtype, dtype, dtype, bs_last, f.scale, nullptr,
                                    ws + l.forward, workspace_bytes - l.forward, stream);
        if (rc != KSMM_OK) return rc;
        grad = to;
    }
    return finish_run(rest, jobs, dtype, s);
}

int64_t ksmm_static_scratch_bytes(void) { return KSMM_STATIC_SCRATCH_BYTES; }

int ksmm_chain_forward_static(const ksmm_factor_desc *factors, int n_factors, const void *x, void *y,
                              int64_t batch, int x_dtype, int y_dtype, int bs_last, int fuse,
                              const ksmm_epilogue *epilogue, void *stream)
{
    // what the chain would ask a caller to lend (0 when it needs no scratch at all)
    const int64_t need = chain_layout(factors, n_factors, batch, x_dtype, y_dtype, bs_last);
    if (need < 0) return (int)need;
    if (need > KSMM_STATIC_SCRATCH_BYTES) return KSMM_ERR_WORKSPACE;
    void *buf = nullptr;
    if (need > 0) {
        const int rc = static_scratch(&buf);
        if (rc != KSMM_OK) return rc;
    }
    return chain_forward_impl(factors, n_factors, x, y, buf, need > 0 ? KSMM_STATIC_SCRATCH_BYTES : 0, batch,
                              x_dtype, y_dtype, bs_last, fuse, epilogue, stream);
}

}  // extern "C"
