// Fused radix-16 chains in either layout, in fp32 as well, for any batch: the chains of ksmm_chain16.hip
// (b = c = 16, power-of-two d, N = a*16*d <= 1024 features) on chunks of 16 or 32 batch rows.
//
// A workgroup (16 waves) holds the whole feature vector of a chunk in LDS, feature by feature: a row of
// 16 batch elements per feature and plane (NS planes of 16).  Every block reads and writes the same 16
// rows, so each factor is applied in place: wave w owns blocks w, w + 16, ..., whose weights stay in its
// registers.  Batch-size-first tensors are transposed on the way in and out in registers (four rows of
// one 16-byte vector each, one v_perm per output word), so x and y are touched once, in whole lines, and no
// transposed copy exists.
//
// LDS rows are 32 bytes (fp16: four 8-byte pieces of 4 batch elements) or 64 (fp32: four 16-byte ones).
// 256 bytes, all banks, hold 8 or 4 rows: the rows of such a line are permuted, and the pieces of a row, by
// `key`, the XOR of the row number's 4-bit fields, which takes 16 values on the rows r0 + i*d of a block for
// any power-of-two d.  So the 16 rows that a 16-lane group of accumulators writes lie in different banks, and so do
// the 4 rows that such a group reads.  That is not the whole of it: the counters show conflicts in 0.12 of the LDS-active
// cycles in fp32 and 0.43 in fp16, where staging and output (lanes 8 rows apart) hit a bank twice and the rest is not
// accounted for.  The map is linear over GF(2): the position of row0 ^ off is the XOR of both.
//
// MFMA roles: A = X^T (rows = batch elements; fp16: transpose loads), B = W^T (lanes = outputs): a lane
// holds 4 batch elements of one output, one piece.
//
// What bounds it: a small batch is one launch instead of one per factor, and then the latency of a chunk
// (weights, input, a barrier per factor, output), 6 us of it on the GPU; full batches the rounds of chunks, one
// workgroup a CU with the next chunk's input in flight (1024 features, 25088 rows, fp16: 28 us, 3.1 rounds of 32 rows,
// where the memory would take 18).  us a call before (a launch per factor, batch-size-first 16-bit chains between
// two transposes) and of a replay now, three factors of 1024 features, 197 / 9408 / 25088 rows: fp32 14 / 51 / 119 and
// 10.5 / 31 / 66, fp16 14 / 39 / 81 and 7.3 / 16 / 28, e4m3 21 / 29 / 54 and 8.2 / 16 / 26.  64 registers a wave, for two
// workgroups a CU, spill (fp16 80 us); fp32 with two planes does too.
//
// Reference counterpart: the Python loop over factors of KSLinear.forward_bs_first / forward_bs_last
// (src/ksmm_py/layer/kronecker_sparse/interface.py:193-211, 269-291).
#include <type_traits>

#include "ksmm_mfma.h"

namespace ksmm {

namespace {

constexpr int CR_THREADS = 1024, CR_WAVES = CR_THREADS / 64, CR_MAXB = 64 / CR_WAVES;

struct Chain16RArgs {
    const void *w[4];
    int log2d[4];
    float scale[4];
    const void *bias;  // of the last factor's outputs, or none
    int act;
    const float *x_scale;  // device: factor of scale[0] that only the GPU knows, or none
    int64_t batch;
    int n_feat;
};

typedef short4_t __attribute__((address_space(3))) * lds_tr_ptr;

// TC: what LDS holds and the MFMA multiplies
template <typename TC> struct cr;
template <> struct cr<half_t> {
    static constexpr int ROW = 32;  // bytes
    typedef half4_t piece_t;
    typedef half4_t operand_t;  // k = 4 (lane / 16) .. + 3
    __device__ static __forceinline__ int pos(int row, int piece)
    {
        const int k = row ^ (row >> 4) ^ (row >> 8);
        const int line = (row & ~7) | ((k ^ ((k >> 2) & 2)) & 7);
        return line * ROW + ((piece ^ ((k >> 2) & 2)) << 3);
    }
    // per-lane part of an operand's position, and the operand of the block at `base`
    __device__ static __forceinline__ int operand_pos(int q, int r, int ld) { return pos((4 * q + (r >> 2)) << ld, r & 3); }
    __device__ static __forceinline__ half4_t operand(const unsigned char *s, int base, int lane_pos, int, int)
    {
        return __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr)(s + (base ^ lane_pos))));
    }
    __device__ static __forceinline__ float4_t mfma(half4_t a, half4_t b)
    {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, float4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    }
};
template <> struct cr<float> {
    static constexpr int ROW = 64;
    typedef float4_t piece_t;
    typedef float4_t operand_t;  // k = lane / 16 + 4 e
    __device__ static __forceinline__ int pos(int row, int piece)
    {
        const int k = (row ^ (row >> 4) ^ (row >> 8)) & 15;
        return ((row & ~3) | ((k ^ (k >> 2)) & 3)) * ROW + ((piece ^ (k >> 2)) << 4);
    }
    __device__ static __forceinline__ int operand_pos(int q, int r, int ld) { return pos(q << ld, r >> 2) + 4 * (r & 3); }
    __device__ static __forceinline__ float4_t operand(const unsigned char *s, int base, int lane_pos, int p4, int p8)
    {
        // rows (q + 4 e) d: XOR with the positions of rows 4d and 8d
        const int at = base ^ lane_pos;
        return float4_t{*(const float *)(s + at), *(const float *)(s + (at ^ p4)), *(const float *)(s + (at ^ p8)),
                        *(const float *)(s + (at ^ p4 ^ p8))};
    }
    __device__ static __forceinline__ float4_t mfma(float4_t a, float4_t b)
    {
        float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], acc, 0, 0, 0);
        return acc;
    }
};

__device__ __forceinline__ half4_t four_halves(uint32_t v)
{
    const half2_t lo = fp8x2_to_half2(v), hi = fp8x2_hi_to_half2(v);
    return half4_t{lo[0], lo[1], hi[0], hi[1]};
}

// One staged vector square: four 16-byte vectors of x (batch-size-first: of four rows) and the pieces they give
template <typename TX> struct square;
template <> struct square<half_t> {
    static constexpr int N = 8;  // features per vector
    __device__ static __forceinline__ half4_t piece(const uint4_t (&v)[4], int e)
    {
        const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
        const uint2_t p = {__builtin_amdgcn_perm(v[1][e >> 1], v[0][e >> 1], sel), __builtin_amdgcn_perm(v[3][e >> 1], v[2][e >> 1], sel)};
        return __builtin_bit_cast(half4_t, p);
    }
};
template <> struct square<fp8_t> {
    static constexpr int N = 16;
    __device__ static __forceinline__ half4_t piece(const uint4_t (&v)[4], int e)
    {
        const int w = e >> 2;
        const uint32_t bytes = (e & 2) ? 0x07030602u : 0x05010400u;
        const uint32_t a = __builtin_amdgcn_perm(v[1][w], v[0][w], bytes), b = __builtin_amdgcn_perm(v[3][w], v[2][w], bytes);
        return four_halves(__builtin_amdgcn_perm(b, a, (e & 1) ? 0x07060302u : 0x05040100u));
    }
};
template <> struct square<float> {
    static constexpr int N = 4;
    __device__ static __forceinline__ float4_t piece(const uint4_t (&v)[4], int e)
    {
        return __builtin_bit_cast(float4_t, uint4_t{v[0][e], v[1][e], v[2][e], v[3][e]});
    }
};

// row j of the square whose pieces are p (16 bytes of one batch row of y)
__device__ __forceinline__ uint4_t row_of(const half4_t (&p)[8], int j)
{
    const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
    uint4_t o;
#pragma unroll
    for (int w = 0; w < 4; ++w)
        o[w] = __builtin_amdgcn_perm(__builtin_bit_cast(uint2_t, p[2 * w + 1])[j >> 1], __builtin_bit_cast(uint2_t, p[2 * w])[j >> 1], sel);
    return o;
}
__device__ __forceinline__ uint4_t row_of(const float4_t (&p)[4], int j)
{
    return __builtin_bit_cast(uint4_t, float4_t{p[0][j], p[1][j], p[2][j], p[3][j]});
}

__device__ __forceinline__ half4_t weight4(const half_t *w) { return half4_t{w[0], w[16], w[32], w[48]}; }
__device__ __forceinline__ half4_t weight4(const fp8_t *w)
{
    return four_halves(w[0].bits | (uint32_t)w[16].bits << 8 | (uint32_t)w[32].bits << 16 | (uint32_t)w[48].bits << 24);
}
// k = 4 (lane / 16) .. + 3 in fp16, lane / 16 + 4 e in fp32: w points to the lane's first
__device__ __forceinline__ float4_t weight4(const float *w) { return float4_t{w[0], w[64], w[128], w[192]}; }

template <typename TX, typename TW, int NF, bool BS_LAST, int NS>
__global__ __launch_bounds__(CR_THREADS) void ks_chain16r_kernel(const TX *__restrict__ x, void *__restrict__ y_, Chain16RArgs args)
{
    typedef typename std::conditional<sizeof(TX) == 4, float, half_t>::type TC;  // and y's type
    typedef cr<TC> C;
    typedef square<TX> SX;
    typedef typename C::piece_t piece_t;
    constexpr int COLS = 16 * NS, VX = 16 / (int)sizeof(TX), VY = 16 / (int)sizeof(TC);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    TC *__restrict__ y = (TC *)y_;
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, r = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n_feat = args.n_feat, n_blocks = n_feat / 16, plane = n_feat * C::ROW;
    const int64_t batch = args.batch, step = (int64_t)gridDim.x * COLS;
    float scale0 = args.scale[0];
    if (sizeof(TX) == 1 && args.x_scale) scale0 *= *args.x_scale;

    // ---- input of a chunk, in registers.  Batch-size-first: squares of four rows x one vector;
    // batch-size-last: vectors of a feature's row ----
    constexpr int SQUARES = BS_LAST ? 1 : (1024 / SX::N) * (COLS / 4) > CR_THREADS ? (1024 / SX::N) * (COLS / 4) / CR_THREADS : 1;
    constexpr int VPR = COLS / VX > 0 ? COLS / VX : 1;  // vectors per feature row
    constexpr int VECS = BS_LAST ? 1024 * VPR / CR_THREADS : 4 * SQUARES;
    uint4_t xreg[VECS];
    const int octets = n_feat / SX::N;
    auto load = [&](int64_t n0) {
        if constexpr (!BS_LAST) {
#pragma unroll
            for (int s = 0; s < SQUARES; ++s) {
                const int id = tid + s * CR_THREADS, g = id / octets, f = (id - g * octets) * SX::N;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int64_t n = n0 + 4 * g + j;
                    xreg[4 * s + j] = uint4_t{0u, 0u, 0u, 0u};
                    if (g < COLS / 4 && n < batch) xreg[4 * s + j] = *(const uint4_t *)(x + n * n_feat + f);
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < VECS; ++i) {
                const int id = tid + i * CR_THREADS, row = id / VPR;
                const int64_t n = n0 + (id % VPR) * VX;
                const TX *src = x + (int64_t)row * batch + n;
                xreg[i] = uint4_t{0u, 0u, 0u, 0u};
                if (row >= n_feat || n >= batch) continue;
                if (n + VX <= batch) {
                    __builtin_memcpy(&xreg[i], src, 16);  // (at element alignment: any row length)
                } else {
                    TX e[VX] = {};
#pragma unroll
                    for (int k = 0; k < VX; ++k)
                        if (n + k < batch) e[k] = src[k];
                    __builtin_memcpy(&xreg[i], e, 16);
                }
            }
        }
    };
    auto stage = [&]() {
        if constexpr (!BS_LAST) {
#pragma unroll
            for (int s = 0; s < SQUARES; ++s) {
                const int id = tid + s * CR_THREADS, g = id / octets, f = (id - g * octets) * SX::N;
                if (g >= COLS / 4) continue;
                const uint4_t v[4] = {xreg[4 * s], xreg[4 * s + 1], xreg[4 * s + 2], xreg[4 * s + 3]};
                const int at = C::pos(f, g & 3) + (g >> 2) * plane;  // (f is a multiple of N: the rows f + e differ in e's bits)
#pragma unroll
                for (int e = 0; e < SX::N; ++e) {
                    const int off = C::pos(e, 0);
                    *(piece_t *)(smem + (g >> 2) * plane + ((at - (g >> 2) * plane) ^ off)) = SX::piece(v, e);
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < VECS; ++i) {
                const int id = tid + i * CR_THREADS, row = id / VPR, c0 = (id % VPR) * VX;
                if (row >= n_feat) continue;
#pragma unroll
                for (int p = 0; p < VX / 4; ++p) {
                    const int pc = c0 / 4 + p;
                    piece_t v;
                    if constexpr (sizeof(TX) == 1) v = four_halves(xreg[i][p]);
                    else if constexpr (sizeof(TX) == 2) v = __builtin_bit_cast(half4_t, uint2_t{xreg[i][2 * p], xreg[i][2 * p + 1]});
                    else v = __builtin_bit_cast(float4_t, xreg[i]);
                    *(piece_t *)(smem + (pc >> 2) * plane + C::pos(row, pc & 3)) = v;
                }
            }
        }
    };
    // Batch-size-last, a chunk is a part of a 128-byte line whose rest belongs to its neighbours: on a full grid these
    // go to workgroups of one XCD (blockIdx.x % 8), as in ksmm_chain16.hip
    int first = blockIdx.x;
    if (BS_LAST && gridDim.x % 32 == 0) first = 4 * (8 * (first / 32) + first % 8) + (first / 8) % 4;
    int64_t n0 = (int64_t)first * COLS;
    load(n0);

    // ---- weights, and the per-lane parts of the positions: operand, row r*d piece q (result) ----
    typename C::operand_t wreg[NF][CR_MAXB];
    int v_in[NF], v_out[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
#pragma unroll
        for (int bi = 0; bi < CR_MAXB; ++bi) {
            const int g = min(wave + CR_WAVES * bi, n_blocks - 1);
            wreg[f][bi] = weight4((const TW *)args.w[f] + (size_t)g * 256 + (sizeof(TW) == 4 ? q : 4 * q) * 16 + r);
        }
        v_in[f] = C::operand_pos(q, r, args.log2d[f]);
        v_out[f] = C::pos(r << args.log2d[f], q);
    }

    for (; n0 < batch; n0 += step) {
        stage();
        __syncthreads();
        if (n0 + step < batch) load(n0 + step);
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            const int ld = args.log2d[f];
            const float scale = f == 0 ? scale0 : args.scale[f];
            const int p4 = C::pos(4 << ld, 0), p8 = C::pos(8 << ld, 0);
            int opaque = 0;
            asm volatile("" : "+s"(opaque));  // keeps the address arithmetic of all blocks in the loop
#pragma unroll
            for (int bi = 0; bi < CR_MAXB; ++bi) {
                const int g = wave + CR_WAVES * bi + opaque;
                if (g >= n_blocks) break;  // uniform
                const int row0 = ((g >> ld) << (ld + 4)) | (g & ((1 << ld) - 1)), base = C::pos(row0, 0);
                float4_t acc[NS];
#pragma unroll
                for (int s = 0; s < NS; ++s) acc[s] = C::mfma(C::operand(smem + s * plane, base, v_in[f], p4, p8), wreg[f][bi]);
                piece_t o[NS];
                if (f + 1 == NF && (args.bias != nullptr || args.act != KSMM_ACT_NONE)) {
                    const Epi ep{scale, args.act, args.bias, nullptr};
                    const float bv = epi_bias<TC>(ep, (size_t)(row0 + (r << ld)));
#pragma unroll
                    for (int s = 0; s < NS; ++s)
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[s][e] = (TC)epi_finish(ep, acc[s][e], bv);
                } else {
#pragma unroll
                    for (int s = 0; s < NS; ++s)
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[s][e] = (TC)(acc[s][e] * scale);
                }
#pragma unroll
                for (int s = 0; s < NS; ++s) *(piece_t *)(smem + s * plane + (base ^ v_out[f])) = o[s];
            }
            __syncthreads();
        }
        // ---- the chunk's result ----
        if constexpr (!BS_LAST) {
            constexpr int OUT = (1024 / VY) * (COLS / 4) / CR_THREADS > 0 ? (1024 / VY) * (COLS / 4) / CR_THREADS : 1;
            const int groups = n_feat / VY;
#pragma unroll
            for (int s = 0; s < OUT; ++s) {
                const int id = tid + s * CR_THREADS, g = id / groups, f = (id - g * groups) * VY;
                if (g >= COLS / 4) continue;
                piece_t p[VY];
                const int at = C::pos(f, g & 3);
#pragma unroll
                for (int e = 0; e < VY; ++e) p[e] = *(const piece_t *)(smem + (g >> 2) * plane + (at ^ C::pos(e, 0)));
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int64_t n = n0 + 4 * g + j;
                    if (n < batch) *(uint4_t *)(y + n * n_feat + f) = row_of(p, j);
                }
            }
        } else {
            constexpr int YPR = COLS / VY, OUT = 1024 * YPR / CR_THREADS;
#pragma unroll
            for (int i = 0; i < OUT; ++i) {
                const int id = tid + i * CR_THREADS, row = id / YPR, c0 = (id % YPR) * VY;
                const int64_t n = n0 + c0;
                if (row >= n_feat || n >= batch) continue;
                uint4_t v;
                if constexpr (sizeof(TC) == 2) {
                    const int pc = c0 / 4;
                    const unsigned char *s = smem + (pc >> 2) * plane;
                    const uint2_t lo = *(const uint2_t *)(s + C::pos(row, pc & 3)), hi = *(const uint2_t *)(s + C::pos(row, (pc & 3) + 1));
                    v = uint4_t{lo[0], lo[1], hi[0], hi[1]};
                } else {
                    v = *(const uint4_t *)(smem + (c0 >> 4) * plane + C::pos(row, (c0 >> 2) & 3));
                }
                TC *to = y + (int64_t)row * batch + n;
                if (n + VY <= batch) {
                    __builtin_memcpy(to, &v, 16);
                } else {
                    TC e[VY];
                    __builtin_memcpy(e, &v, 16);
#pragma unroll
                    for (int k = 0; k < VY; ++k)
                        if (n + k < batch) to[k] = e[k];
                }
            }
        }
        __syncthreads();  // the rows are read: the next chunk may be staged over them
    }
}

template <typename TX, typename TW, bool BS_LAST, int NS> const void *fn_of(int nf)
{
    switch (nf) {
    case 2: return (const void *)ks_chain16r_kernel<TX, TW, 2, BS_LAST, NS>;
    case 3: return (const void *)ks_chain16r_kernel<TX, TW, 3, BS_LAST, NS>;
    default: return (const void *)ks_chain16r_kernel<TX, TW, 4, BS_LAST, NS>;
    }
}
// (fp32 with two planes does not fit the registers)
template <typename TX, typename TW> const void *fn_of(int nf, bool bs_last, int ns)
{
    if constexpr (sizeof(TX) == 4) return bs_last ? fn_of<TX, TW, true, 1>(nf) : fn_of<TX, TW, false, 1>(nf);
    if (bs_last) return ns == 1 ? fn_of<TX, TW, true, 1>(nf) : fn_of<TX, TW, true, 2>(nf);
    return ns == 1 ? fn_of<TX, TW, false, 1>(nf) : fn_of<TX, TW, false, 2>(nf);
}

}  // namespace

// Returns KSMM_ERR_BAD_ALGO when the chain is not a radix-16 butterfly this kernel takes.
int chain16r_run(const ksmm_factor_desc *f, int n, const void *x, void *y, int64_t batch, int x_dtype, int y_dtype, int bs_last,
                 bool launch, hipStream_t stream, const ksmm_epilogue *ep, const float *x_scale)
{
    if (n < 2 || n > 4) return KSMM_ERR_BAD_ALGO;
    const int64_t n_feat = (int64_t)f[0].a * 16 * f[0].d;
    if (n_feat > 1024) return KSMM_ERR_BAD_ALGO;
    for (int i = 0; i < n; ++i) {
        if (f[i].b != 16 || f[i].c != 16 || (int64_t)f[i].a * 16 * f[i].d != n_feat) return KSMM_ERR_BAD_ALGO;
        if (f[i].d & (f[i].d - 1)) return KSMM_ERR_BAD_ALGO;
        if (f[i].w_dtype != f[0].w_dtype) return KSMM_ERR_BAD_ALGO;
    }
    const int combo = combo_of(x_dtype, f[0].w_dtype, y_dtype);
    if (combo < 0) return KSMM_ERR_BAD_ALGO;
    const bool aligned = (((uintptr_t)x | (uintptr_t)y) & 15) == 0;
    if (!bs_last && !aligned) return KSMM_ERR_BAD_ALGO;
    if (!launch) return KSMM_OK;
    // two planes a chunk where chunks of one would need a second round
    const int ns = combo != 0 && batch > 256 * 16 ? 2 : 1;
    // One workgroup a CU: with twice as many, the second half starts cold (weights, first input) behind the first.  us with
    // 512 / 256, 1024 features at 9409 and 25087 rows: batch-size-last fp16 27.4 / 19.9 and 44.9 / 42.3, e4m3 26.6 / 19.4
    // and 47.5 / 43.3, fp32 34.5 / 32.4 and 71.3 / 73.0, batch-size-first fp16 18.5 / 16.4 and 30.2 / 28.3; 256 features
    // 1.1 to 1.3 times as fast; the one loss is fp32 beyond 40000 rows of 1024 features, 130 / 133 at 50000.
    const int64_t chunks = (batch + 16 * ns - 1) / (16 * ns), most = 256;
    const void *fn = combo == 0   ? fn_of<float, float>(n, bs_last, ns)
                     : combo == 1 ? fn_of<half_t, half_t>(n, bs_last, ns)
                     : combo == 2 ? fn_of<fp8_t, fp8_t>(n, bs_last, ns)
                                  : fn_of<half_t, fp8_t>(n, bs_last, ns);
    Chain16RArgs args;
    for (int i = 0; i < 4; ++i) {
        const int j = i < n ? i : n - 1;
        args.w[i] = f[j].w;
        args.log2d[i] = __builtin_ctz((unsigned)f[j].d);
        args.scale[i] = f[j].scale;
    }
    args.bias = ep ? ep->bias : nullptr;
    args.act = ep ? ep->act : KSMM_ACT_NONE;
    args.x_scale = x_scale;
    args.batch = batch;
    args.n_feat = (int)n_feat;
    const int lds = (int)n_feat * ns * (combo == 0 ? 64 : 32);
    if (ensure_dynamic_lds(fn, lds) != KSMM_OK) return KSMM_ERR_LAUNCH;
    void *kargs[] = {(void *)&x, (void *)&y, (void *)&args};
    const hipError_t e = hipLaunchKernel(fn, dim3((unsigned)(chunks < most ? chunks : most)), dim3(CR_THREADS), kargs, lds, stream);
    return e == hipSuccess ? KSMM_OK : KSMM_ERR_LAUNCH;
}

}  // namespace ksmm
