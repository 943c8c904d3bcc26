// fox_batch.hip -- projections of a batched pass (a prompt's tokens, more
// than the FOX_GPU_MAX_TOKENS of the decode kernels), bit-identical to them,
// and of a few tokens where the one-launch kernels of fox_fused.hip do not
// apply (few_gemm: the K-quants) or are slower.
//
// batch_prep quantises the tokens once (optionally RMS-normalised first), a
// workgroup per token, and batch_gemm is an int8 MFMA matrix product over
// the 256-element weight blocks:
//   * the activations are the MFMA's A operand (16 tokens), the weight rows
//     its B operand (16 rows), so lane (j, g) holds row j's sums of tokens
//     4g .. 4g + 3: a lane needs the scales of one row only;
//   * a wave owns its rows' whole K range and adds each block's float term
//     as the block is done, in block order from 0.0f, which is the
//     reference's row loop (src/ternary.c:226-246, src/kernels.c:571-661):
//     no terms go through memory;
//   * the integer sums start from the bits of 1.5 * 2^23 (MAGIC), so an
//     accumulator's bits are the float 12582912 + S exactly (|S| < 2^22), and
//     fma(d, that, -12582912 d) is d * S rounded once (12582912 d is exact:
//     d has at most 17 significant bits), the reference's d * (float)S, one
//     instruction in place of a conversion and a product.  A row whose d is
//     infinite or NaN takes the conversion (wave-uniform test).
//
// The pass over a 1024-token prompt is bound by the matrix cores and the
// vector unit about equally on ternary weights (four MFMAs, 64 clocks,
// against 8 vector instructions per 16 x 16 x 256 tile and the split of the
// codes, 28 shared by the wave's token tiles) and by the vector unit on the
// K-quants (5 instructions per 32-element sub-block and output for Q4_K).
// Measured: two 4B-class layers over a 1024-token prompt 22.0 ms in passes of
// eight, 1.12 ms batched; two 8B-class layers over 77 tokens on 1024 cached
// rows 7.24 -> 0.71 ms.  A 1024-token gate/up (2 x 9728 x 2560, ternary) takes
// 100 us, a 77-token one of the 8B class (Q4_K, 2 x 14336 x 4096) 77 us.
#include "fox_gemv_dev.h"
#include "fox_math.h"

#include <cstring>
#include <type_traits>

#define BT_THREADS 256
#define MAGIC_BITS 0x4B400000           // 12582912.0f = 1.5 * 2^23
#define MAGIC_F 12582912.0f
#define B_TILE 4096                     // operand bytes of 16 tokens and one block

// 16-byte quads of per-token values per (16-token tile, block): TQ2_0 the
// negated block sums (plus MAGIC_BITS), Q4_K eight sub-block sums and the
// block scale as floats, Q6_K the block scale
__host__ __device__ constexpr int aux_quads(int fmt)
{
    return fmt == FMT_Q4K ? 36 : 4;
}

// ------------------------------------------------------------------ prep

// Where lane dl's dword (elements 4 dl .. 4 dl + 3 of a block) goes in the
// operand of a token tile and block, token 0's offset (a token is 16 bytes
// on): [step][g][16 tokens][16 bytes], what lane group g feeds to MFMA step
// `step` (mirroring the weight decodes below).  A wave's operand load is one
// contiguous 1 KB.
template <int FMT>
__device__ __forceinline__ int piece_off(int dl)
{
    const int e0 = 4 * dl;
    if (FMT == FMT_TQ2) {
        const int half = e0 >> 7, l = (e0 >> 5) & 3, o = e0 & 31;
        const int g = 2 * half + (o >> 4), u = (o & 15) >> 2;
        return (u * 4 + g) * 256 + l * 4;
    } else if (FMT == FMT_Q4K) {
        // sub-blocks 2p and 2p + 1 side by side, eight elements of each
        const int s = e0 >> 5, o = e0 & 31;
        return ((s >> 1) * 4 + (o >> 3)) * 256 + (s & 1) * 8 + (o & 4);
    } else {
        return (e0 >> 4) * 256 + (e0 & 15);
    }
}

// the same for up to eight tokens (few_gemm): the block's 2048 bytes hold, for
// each operand load, the 16 bytes of every lane side by side; token 0's offset
// (a token is 16 bytes on)
template <int FMT>
__device__ __forceinline__ int few_off(int dl)
{
    const int e0 = 4 * dl;
    if (FMT == FMT_Q4K) {
        // [sub-block quad][g][half][token]: eight elements of sub-blocks
        // 4 qd + half and 4 qd + 2 + half
        const int s = e0 >> 5, o = e0 & 31;
        return (((s >> 2) * 4 + (o >> 3)) * 16 + (s & 1) * 8) * 16 + ((s >> 1) & 1) * 8 + (o & 4);
    } else {
        return (e0 >> 4) * 128 + (e0 & 15);                // [16-element piece][token]
    }
}

// one dword of four quantised values, and the scale: the reference's
// per-element rule for an amax whose bits are am (the largest |x| bit
// pattern: NaN above inf) and m, the largest |x| that is not NaN
struct Quant {
    float inv, act;
    int mode;                  // 0 zeros, 1 quant_fast, 2 quant_one
};
__device__ __forceinline__ Quant quant_of(uint32_t am, float m)
{
    Quant q;
    if (am >= 0x03800000u && am < 0x7f800000u) {
        const float amax = __uint_as_float(am);
        q.inv = fox_div(127.0f, amax);
        q.act = fox_div(amax, 127.0f);
        q.mode = 1;
    } else if (m > 0.0f) {
        q.inv = fox_div(127.0f, m);
        q.act = fox_div(m, 127.0f);
        q.mode = 2;
    } else {
        q.inv = q.act = 0.0f;
        q.mode = 0;
    }
    return q;
}

__device__ __forceinline__ uint32_t quant4(const Quant &q, const float4 &x)
{
    if (q.mode == 1)
        return pack_lo_bytes(quant_fast(x.x, q.inv), quant_fast(x.y, q.inv),
                             quant_fast(x.z, q.inv), quant_fast(x.w, q.inv));
    if (q.mode == 2)
        return pack_lo_bytes(quant_one(x.x, q.inv), quant_one(x.y, q.inv), quant_one(x.z, q.inv),
                             quant_one(x.w, q.inv));
    return 0u;
}

__device__ __forceinline__ uint32_t abs_bits4(const float4 &x)
{
    const uint32_t a = max(__float_as_uint(x.x) & 0x7fffffffu, __float_as_uint(x.y) & 0x7fffffffu);
    const uint32_t b = max(__float_as_uint(x.z) & 0x7fffffffu, __float_as_uint(x.w) & 0x7fffffffu);
    return max(a, b);
}

// the largest |x| that is not NaN (src/gemv.c:20-23: `a > amax` from 0)
__device__ __forceinline__ float abs_max4(const float4 &x)
{
    const float v[4] = {fabsf(x.x), fabsf(x.y), fabsf(x.z), fabsf(x.w)};
    float m = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; e++) m = v[e] > m ? v[e] : m;
    return m;
}

__device__ __forceinline__ uint32_t wave_max_u(uint32_t v)
{
    return wave_reduce(v, 0u, [](uint32_t x, uint32_t y) { return x > y ? x : y; });
}

// Token blockIdx.x: RMSNorm (NORM; src/ops.c:7-22), int8 quantisation and the
// block sums.  512 threads; thread tid holds dwords tid + 512 r, so a wave
// holds whole blocks (block wave + 8 r).  The K-quants without a norm have
// nothing to share between blocks: there blockIdx.y takes 8 R blocks each.
// Eight tokens in a row run on one XCD (blockIdx % 8): they share the cache
// lines of the operand.
// q: [token / 16][block][4096], in piece_off order, or (few)
// [block][2048], in few_off order; aux: [token / 16][block][aux_quads][token % 16].
template <int FMT, bool NORM, int R>
__global__ __launch_bounds__(512) void batch_prep(const float *__restrict__ x,
                                                  const float *__restrict__ norm_w, int K,
                                                  size_t x_stride, float eps, int M, int few,
                                                  uint8_t *__restrict__ q,
                                                  uint32_t *__restrict__ aux,
                                                  float *__restrict__ scale)
{
    __shared__ double dred[8];
    __shared__ uint32_t ured[8];
    const int bx = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int t = few ? bx : (bx >> 6) * 64 + (bx & 7) * 8 + ((bx >> 3) & 7);
    if (t >= M) return;                                     // (uniform)
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b_first = FMT != FMT_TQ2 && !NORM ? (int)blockIdx.y * 8 * R : 0;
    const int nb = (K >> 8) - b_first, nd = nb * 64;
    const float *xt = x + (size_t)t * x_stride;
    const float4 *x4 = (const float4 *)xt + b_first * 64, *w4 = (const float4 *)norm_w;
    float4 xv[R], wv[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int m = min(tid + 512 * r, nd - 1);
        xv[r] = x4[m];
        if (NORM) wv[r] = w4[m];
    }
#pragma unroll
    for (int r = 0; r < R; r++)
        if (tid + 512 * r >= nd) xv[r] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (NORM) {
        double ss = 0.0;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const double x0 = xv[r].x, x1 = xv[r].y, x2 = xv[r].z, x3 = xv[r].w;
            ss = __builtin_fma(x0, x0, ss);
            ss = __builtin_fma(x1, x1, ss);
            ss = __builtin_fma(x2, x2, ss);
            ss = __builtin_fma(x3, x3, ss);
        }
        ss = wave_reduce(ss, 0.0, [](double a, double b) { return a + b; });
        if (lane == 0) dred[wave] = ss;
        __syncthreads();
        double tot = 0.0;
        for (int w = 0; w < 8; w++) tot += dred[w];
        // the scale from both ends of the interval that holds the
        // index-order sum (fox_fused.hip, rms_apply); undecided: that sum
        const double rel = (double)(K + 64) * 0x1p-52;
        const double sgn = (lane & 1) ? 1.0 : -1.0;
        const double y = 1.0 / __builtin_sqrt(tot * (1.0 + sgn * rel) / (double)K + (double)eps) *
                         (1.0 - sgn * 0x1p-50);
        const float f = (float)y;
        float rs = read_lane(f, 0);
        if (rs != read_lane(f, 1)) {
            double seq = 0.0;
            for (int i = 0; i < K; i++) seq += (double)xt[i] * (double)xt[i];
            rs = (float)(1.0 / __builtin_sqrt(seq / (double)K + (double)eps));
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            xv[r].x = xv[r].x * rs * wv[r].x;
            xv[r].y = xv[r].y * rs * wv[r].y;
            xv[r].z = xv[r].z * rs * wv[r].z;
            xv[r].w = xv[r].w * rs * wv[r].w;
            // (dwords past the end: 0 * rs * w may be NaN)
            if (tid + 512 * r >= nd) xv[r] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    }
    Quant qv;
    if (FMT == FMT_TQ2) {
        uint32_t am = 0;
#pragma unroll
        for (int r = 0; r < R; r++) am = max(am, abs_bits4(xv[r]));
        am = wave_max_u(am);
        if (lane == 0) ured[wave] = am;
        __syncthreads();
        am = 0;
        for (int w = 0; w < 8; w++) am = max(am, ured[w]);
        float m = 0.0f;
        if (am >= 0x7f800000u || am < 0x03800000u) {        // (uniform over the workgroup)
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float v = abs_max4(xv[r]);
                m = v > m ? v : m;
            }
            m = wave_max(m);
            __syncthreads();
            if (lane == 0) ured[wave] = __float_as_uint(m);
            __syncthreads();
            m = 0.0f;
            for (int w = 0; w < 8; w++) m = fmaxf(m, __uint_as_float(ured[w]));
        }
        qv = quant_of(am, m);
        if (tid == 0) scale[t] = qv.act;
    }
    const bool fw = FMT != FMT_TQ2 && few;
    const size_t bs = fw ? 2048 : B_TILE;
    uint8_t *qt = q + (fw ? (size_t)t * 16 + few_off<FMT>(lane)
                          : (size_t)(t >> 4) * (K >> 8) * B_TILE + (t & 15) * 16 + piece_off<FMT>(lane)) +
                  b_first * bs;
    uint32_t *at = aux + ((size_t)(t >> 4) * (K >> 8) + b_first) * (aux_quads(FMT) * 4) + (t & 15);
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int b = wave + 8 * r;
        if (b >= nb) break;                                 // (uniform)
        if (FMT != FMT_TQ2) {
            // one scale per block (src/kernels.c:722-754)
            const uint32_t am = wave_max_u(abs_bits4(xv[r]));
            const float m = am >= 0x7f800000u || am < 0x03800000u ? wave_max(abs_max4(xv[r])) : 0.0f;
            qv = quant_of(am, m);
        }
        const uint32_t qd = quant4(qv, xv[r]);
        *(uint32_t *)(qt + b * bs) = qd;
        uint32_t *ab = at + (size_t)b * (aux_quads(FMT) * 4);
        if (FMT == FMT_TQ2) {
            const int s = wave_sum_i(__builtin_amdgcn_sdot4((int)qd, 0x01010101, 0, false));
            if (lane == 0) ab[0] = (uint32_t)(MAGIC_BITS - s);
        } else {
            if (FMT == FMT_Q4K) {
                int s = __builtin_amdgcn_sdot4((int)qd, 0x01010101, 0, false);
                s += dpp_t<0xB1, 0xF>(0, s);
                s += dpp_t<0x4E, 0xF>(0, s);
                s += dpp_t<0x141, 0xF>(0, s);               // sums of 8 lanes: 32 elements
                if ((lane & 7) == 0) ab[(lane >> 3) * 16] = __float_as_uint((float)s);
            }
            if (lane == 0) ab[(aux_quads(FMT) * 4) - 16] = __float_as_uint(qv.act);
        }
    }
}

// ------------------------------------------------------------------ GEMM

struct BatchArgs {
    const uint8_t *w[MAX_SEGS];
    float *out[MAX_SEGS];
    size_t out_stride[MAX_SEGS];
    int n_rows[MAX_SEGS];
    int tile_start[MAX_SEGS + 1];
    int nseg, nb, M, n_tg, n_wg;
    unsigned flags;
    const uint8_t *q;
    const uint32_t *aux;
    const float *scale;
};

enum { BE_STORE = 0, BE_SILU = 1 };

// blocks per stage: as many as keep a stage's loads at four 16-byte pieces
// per thread (few tokens), fewer for the K-quants, whose raw blocks take
// more registers
__host__ __device__ constexpr int stage_blocks(int fmt, int C)
{
    return C >= 3 ? 1 : fmt == FMT_TQ2 ? 4 / C : fmt == FMT_Q4K ? 2 / C : 1;
}

__host__ __device__ constexpr int batch_chunk(int fmt)
{
    return fmt == FMT_TQ2 ? TQ2_CHUNK : fmt == FMT_Q4K ? Q4K_CHUNK : Q6K_CHUNK;
}

typedef float f4v __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

// a lane's bytes of one weight block (row j of a 16-row tile, group g)
template <int FMT>
struct RawBlock;
template <>
struct RawBlock<FMT_TQ2> {
    u4v qs;
    uint32_t d;
    __device__ __forceinline__ void load(const uint8_t *ch, int lane)
    {
        qs = *(const u4v *)(ch + 16 * lane);
        d = *(const unsigned short *)(ch + 1024 + 2 * (lane & 15));
    }
};
template <>
struct RawBlock<FMT_Q4K> {
    u4v q0, q1, h;
    __device__ __forceinline__ void load(const uint8_t *ch, int lane)
    {
        q0 = *(const u4v *)(ch + 32 * lane);
        q1 = *(const u4v *)(ch + 32 * lane + 16);
        h = *(const u4v *)(ch + 2048 + 16 * (lane & 15));
    }
};
// Q6_K: lane group g takes the 16 ql bytes 64 h + 16 g of half h of its row:
// low nibbles sub-group c = g / 2 of quarter 2 h + g % 2, high nibbles c + 2
// of the same quarter (a wave's load is a contiguous 64 bytes of 16 rows)
template <>
struct RawBlock<FMT_Q6K> {
    u4v l[2], hq[2], sc;
    uint32_t d;
    __device__ __forceinline__ void load(const uint8_t *ch, int lane)
    {
        const int i = lane & 15, g = lane >> 4;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            l[h] = *(const u4v *)(ch + 128 * i + 64 * h + 16 * g);
            hq[h] = *(const u4v *)(ch + 2048 + 64 * i + 32 * h + 16 * (g & 1));
        }
        sc = *(const u4v *)(ch + 3072 + 16 * i);
        d = *(const unsigned short *)(ch + 3328 + 2 * i);
    }
};

// the signed bytes 4 (q - 32) of half h (the 6-bit value shifted up, its top
// bit flipped; the factor is taken out of the integer sums): hi = 0 the low
// nibbles' sub-groups, 1 the high ones'
__device__ __forceinline__ v4i q6_bytes(const RawBlock<FMT_Q6K> &w, int h, int hi, int g)
{
    const int sh = 2 * (g >> 1) + 4 * hi;
    v4i r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t lo = (hi ? w.l[h][i] >> 2 : w.l[h][i] << 2) & 0x3c3c3c3cu;
        const uint32_t up = ((w.hq[h][i] >> sh) & 0x03030303u) << 6;
        r[i] = (int)((lo | up) ^ 0x80808080u);
    }
    return r;
}

// scale byte n of the row, signed
__device__ __forceinline__ int q6_scale(const u4v &sc, int n)
{
    return (int)(sc[n >> 2] << (24 - 8 * (n & 3))) >> 24;
}

__device__ __forceinline__ v4i mfma64(v4i a, v4i b, v4i c)
{
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

// any lane's value infinite or NaN (wave-uniform)
__device__ __forceinline__ bool any_nonfinite(float d)
{
    return __builtin_amdgcn_ballot_w64(!(fabsf(d) < INFINITY)) != 0;
}

// One block of R row tiles against C token tiles, its float terms added to
// acc.  bl: the block's operand in LDS (tile c at bl + c * B_TILE),
// ax: its aux (tile c at ax + c * aux_quads quads).
template <int FMT, int R, int C>
__device__ __forceinline__ void block_terms(const RawBlock<FMT> (&raw)[R], const uint8_t *bl,
                                            const u4v *ax, int lane, f4v (&acc)[R][C])
{
    const int g = lane >> 4;
    const uint8_t *bt = bl + lane * 16;
    if constexpr (FMT == FMT_TQ2) {
        v4i D[R][C], corr[C];
#pragma unroll
        for (int c = 0; c < C; c++) corr[c] = ((const v4i *)ax)[c * 4 + g];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            v4i w[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const uint32_t d = raw[r].qs[u];
                w[r] = v4i{(int)(d & 0x03030303u), (int)((d >> 2) & 0x03030303u),
                           (int)((d >> 4) & 0x03030303u), (int)((d >> 6) & 0x03030303u)};
            }
#pragma unroll
            for (int c = 0; c < C; c++) {
                const v4i a = *(const v4i *)(bt + c * B_TILE + u * 1024);
#pragma unroll
                for (int r = 0; r < R; r++) D[r][c] = mfma64(a, w[r], u == 0 ? corr[c] : D[r][c]);
            }
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            const float d = half_bits_to_float(raw[r].d);
            if (!any_nonfinite(d)) {
                const float nd = -MAGIC_F * d;
#pragma unroll
                for (int c = 0; c < C; c++)
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        acc[r][c][k] = acc[r][c][k] + __builtin_fmaf(d, __int_as_float(D[r][c][k]), nd);
            } else {
#pragma unroll
                for (int c = 0; c < C; c++)
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        acc[r][c][k] = acc[r][c][k] + d * (float)(D[r][c][k] - MAGIC_BITS);
            }
        }
    } else if constexpr (FMT == FMT_Q4K) {
        // d * sc and dmin * mn of the row's eight sub-blocks (exact: 11 + 6
        // bits), src/kernels.c:246-255, 585-599
        float A[R][8], B[R][8];
        bool odd = false;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t s0 = raw[r].h[1], s1 = raw[r].h[2], s2 = raw[r].h[3];
            const uint32_t sc[2] = {s0 & 0x3f3f3f3fu,
                                    (s2 & 0x0f0f0f0fu) | (((s0 >> 6) & 0x03030303u) << 4)};
            const uint32_t mn[2] = {s1 & 0x3f3f3f3fu,
                                    ((s2 >> 4) & 0x0f0f0f0fu) | (((s1 >> 6) & 0x03030303u) << 4)};
            const float d = half_bits_to_float(raw[r].h[0] & 0xffffu);
            const float dmin = half_bits_to_float(raw[r].h[0] >> 16);
            odd = odd || any_nonfinite(d);
#pragma unroll
            for (int s = 0; s < 8; s++) {
                A[r][s] = d * (float)((sc[s >> 2] >> (8 * (s & 3))) & 0xffu);
                B[r][s] = dmin * (float)((mn[s >> 2] >> (8 * (s & 3))) & 0xffu);
            }
        }
        const v4i magic = {MAGIC_BITS, MAGIC_BITS, MAGIC_BITS, MAGIC_BITS};
        auto run = [&](auto finite) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < 4; p++) {
                long wl[R], wh[R];
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const uint32_t a0 = p < 2 ? raw[r].q0[2 * p] : raw[r].q1[2 * p - 4];
                    const uint32_t a1 = p < 2 ? raw[r].q0[2 * p + 1] : raw[r].q1[2 * p - 3];
                    wl[r] = (long)((uint64_t)(a0 & 0x0f0f0f0fu) | (uint64_t)(a1 & 0x0f0f0f0fu) << 32);
                    wh[r] = (long)((uint64_t)((a0 >> 4) & 0x0f0f0f0fu) |
                                   (uint64_t)((a1 >> 4) & 0x0f0f0f0fu) << 32);
                }
#pragma unroll
                for (int c = 0; c < C; c++) {
                    typedef long l2v __attribute__((ext_vector_type(2)));
                    const l2v a = *(const l2v *)(bt + c * B_TILE + p * 1024);
                    const f4v as = ((const f4v *)ax)[c * 36 + 32 + g];
#pragma unroll
                    for (int hh = 0; hh < 2; hh++) {
                        const int s = 2 * p + hh;
                        const f4v sq = ((const f4v *)ax)[c * 36 + 4 * s + g];
#pragma unroll
                        for (int r = 0; r < R; r++) {
                            const v4i D = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                                a[hh], hh ? wh[r] : wl[r], magic, 0, 0, 0);
                            const float na = -MAGIC_F * A[r][s];
#pragma unroll
                            for (int k = 0; k < 4; k++) {
                                const float pr =
                                    decltype(finite)::value
                                        ? __builtin_fmaf(A[r][s], __int_as_float(D[k]), na)
                                        : A[r][s] * (float)(D[k] - MAGIC_BITS);
                                const float tv = pr - B[r][s] * sq[k];
                                acc[r][c][k] = acc[r][c][k] + as[k] * tv;
                            }
                        }
                    }
                }
            }
        };
        if (!odd) run(std::true_type{});
        else run(std::false_type{});
    } else {
        // Q6_K: an operand's four lane groups are four 16-element sub-groups
        // (group gg: quarter 2h + gg % 2, sub-group gg / 2, + 2 for the high
        // nibbles); one alone is the product with the other groups' weights
        // zeroed.
#pragma unroll
        for (int h = 0; h < 2; h++) {
            v4i w[R][2];
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int hi = 0; hi < 2; hi++) w[r][hi] = q6_bytes(raw[r], h, hi, g);
#pragma unroll
            for (int c = 0; c < C; c++) {
                v4i x[2];
                x[0] = *(const v4i *)(bt + c * B_TILE + h * 2048);
                x[1] = *(const v4i *)(bt + c * B_TILE + h * 2048 + 1024);
                const f4v as = ((const f4v *)ax)[c * 4 + g];
                asm volatile("" : "+v"(x[0]), "+v"(x[1]));    // (see below)
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const v4i zero = {0, 0, 0, 0};
                    v4i part[2] = {zero, zero};
#pragma unroll
                    for (int gg = 0; gg < 4; gg++) {
                        const int m = g == gg ? -1 : 0;
#pragma unroll
                        for (int hi = 0; hi < 2; hi++) {
                            const v4i wm = {w[r][hi][0] & m, w[r][hi][1] & m, w[r][hi][2] & m,
                                            w[r][hi][3] & m};
                            const v4i D = mfma64(x[hi], wm, zero);
                            const int sc = q6_scale(raw[r].sc, 8 * h + (gg & 1) + 2 * ((gg >> 1) + 2 * hi));
#pragma unroll
                            for (int k = 0; k < 4; k++) part[gg & 1][k] += __mul24(sc, D[k]);
                        }
                    }
                    const float d = half_bits_to_float(raw[r].d);
#pragma unroll
                    for (int s = 0; s < 2; s++)
#pragma unroll
                        for (int k = 0; k < 4; k++)
                            acc[r][c][k] = acc[r][c][k] + as[k] * d * (float)(part[s][k] >> 2);
                }
                // (left to itself the compiler issues every matrix product of
                // the block first and needs 256 more registers for them: the
                // two empty statements order this tile's before the next's)
#pragma unroll
                for (int r = 0; r < R; r++) asm volatile("" : "+v"(acc[r][c]));
            }
        }
    }
}

// Workgroup: 4 waves, each R 16-row tiles, all of them against the same C
// 16-token tiles.  Work item = (row group, token group); items run token
// groups first within contiguous ranges per XCD (blockIdx % 8), so that one
// XCD's L2 serves a row group's weights to all its token groups.
// BE_SILU: segment 0 is gate, segment 1 up; a wave's tiles are R / 2 gate
// tiles and the same up tiles, out = silu(gate) * up.
template <int FMT, int R, int C, int EPI>
__global__ __launch_bounds__(BT_THREADS, 2) void batch_gemm(BatchArgs a)
{
    constexpr int KB = stage_blocks(FMT, C), CH = batch_chunk(FMT), AQ = aux_quads(FMT);
    constexpr int BB = KB * C * B_TILE, NAX = KB * C * AQ;
    static_assert(NAX <= BT_THREADS, "one aux quad per thread and stage");
    static_assert(EPI != BE_SILU || R % 2 == 0, "gate and up tiles in pairs");
    __shared__ __align__(16) uint8_t Bs[2][BB];
    __shared__ u4v As[2][NAX];
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int per = (a.n_wg + 7) >> 3;
    const int item = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (item >= a.n_wg || (int)(blockIdx.x >> 3) >= per) return;    // (uniform)
    const int rg = item / a.n_tg, tg = item - rg * a.n_tg;
    const int nb = a.nb, ntt = (a.M + 15) >> 4;

    // this wave's tiles: weights, segment and tile within it (tiles past the
    // end repeat the last one and are not written)
    const uint8_t *wp[R];
    int seg[R], tl[R];
    bool live[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (EPI == BE_SILU) {
            const int p = (rg * 4 + wave) * (R / 2) + (r >> 1);
            seg[r] = r & 1;
            live[r] = p < a.tile_start[1];
            tl[r] = live[r] ? p : a.tile_start[1] - 1;
        } else {
            int t = (rg * 4 + wave) * R + r;
            live[r] = t < a.tile_start[a.nseg];
            t = live[r] ? t : a.tile_start[a.nseg] - 1;
            int s = 0;
            while (s + 1 < a.nseg && t >= a.tile_start[s + 1]) s++;
            seg[r] = s;
            tl[r] = t - a.tile_start[s];
        }
        wp[r] = a.w[seg[r]] + (size_t)tl[r] * nb * CH;
    }

    // staging: piece i = (block kb, tile c) of a stage, 4 KB, 16 bytes of it
    // per thread
    const uint8_t *qrow[C];
#pragma unroll
    for (int c = 0; c < C; c++)
        qrow[c] = a.q + (size_t)min(tg * C + c, ntt - 1) * nb * B_TILE + tid * 16;
    u4v br[KB * C], ar = {0, 0, 0, 0};
    auto fetch = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
#pragma unroll
            for (int c = 0; c < C; c++)
                br[kb * C + c] = *(const u4v *)(qrow[c] + (size_t)min(s * KB + kb, nb - 1) * B_TILE);
        const int ai = min(tid, NAX - 1), i = ai / AQ, kb = i / C, c = i - kb * C;
        ar = ((const u4v *)a.aux)[((size_t)min(tg * C + c, ntt - 1) * nb + min(s * KB + kb, nb - 1)) * AQ +
                                  (ai - i * AQ)];
    };
    auto stash = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < KB * C; i++)
            *(u4v *)(Bs[buf] + i * B_TILE + tid * 16) = br[i];
        if (tid < NAX) As[buf][tid] = ar;
    };
    RawBlock<FMT> cur[KB][R], nxt[KB][R];
    auto weights = [&](int s, RawBlock<FMT> (&dst)[KB][R]) __attribute__((always_inline)) {
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
#pragma unroll
            for (int r = 0; r < R; r++)
                dst[kb][r].load(wp[r] + (size_t)min(s * KB + kb, nb - 1) * CH, lane);
    };
    f4v acc[R][C];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int c = 0; c < C; c++) acc[r][c] = f4v{0.0f, 0.0f, 0.0f, 0.0f};

    const int ns = (nb + KB - 1) / KB;
    fetch(0);
    weights(0, cur);
    stash(0);
    __syncthreads();
    for (int s = 0; s < ns; s++) {
        const int buf = s & 1, sn = min(s + 1, ns - 1);
        fetch(sn);
        weights(sn, nxt);
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
            if (s * KB + kb < nb)                            // (uniform)
                block_terms<FMT, R, C>(cur[kb], Bs[buf] + kb * C * B_TILE,
                                       &As[buf][kb * C * AQ], lane, acc);
        // the other buffer was last read before the previous barrier
        stash(buf ^ 1);
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
#pragma unroll
            for (int r = 0; r < R; r++) cur[kb][r] = nxt[kb][r];
        __syncthreads();
    }

    // lane (j, g): row j of each tile, tokens 4g .. 4g + 3 of each token tile
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int t0 = (tg * C + c) * 16 + 4 * g;
        float sc[4];
#pragma unroll
        for (int k = 0; k < 4; k++) sc[k] = FMT == FMT_TQ2 ? a.scale[min(t0 + k, a.M - 1)] : 1.0f;
        if (EPI == BE_SILU) {
#pragma unroll
            for (int r = 0; r < R; r += 2) {
                const int row = tl[r] * 16 + j;
                if (!live[r] || row >= a.n_rows[0]) continue;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    if (t0 + k >= a.M) continue;
                    const float gt = FMT == FMT_TQ2 ? acc[r][c][k] * sc[k] : acc[r][c][k];
                    const float up = FMT == FMT_TQ2 ? acc[r + 1][c][k] * sc[k] : acc[r + 1][c][k];
                    const float sg = fox_div(gt, 1.0f + fox_expf(-gt));
                    a.out[0][(size_t)(t0 + k) * a.out_stride[0] + row] = sg * up;
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int row = tl[r] * 16 + j;
                if (!live[r] || row >= a.n_rows[seg[r]]) continue;
                float *o = a.out[seg[r]] + row;
                const size_t os = a.out_stride[seg[r]];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    if (t0 + k >= a.M) continue;
                    const float y = FMT == FMT_TQ2 ? acc[r][c][k] * sc[k] : acc[r][c][k];
                    float *p = o + (size_t)(t0 + k) * os;
                    *p = (a.flags & FOX_GPU_GEMV_ACCUMULATE) ? *p + y : y;
                }
            }
        }
    }
}

// ------------------------------------------------- few tokens, K-quants

// K-quant matrices against 2 .. 8 tokens: a workgroup per 16-row tile, its
// waves take the blocks in turn (block wave + KS r) and write each block's
// float terms to one of two LDS buffers, and 128 lanes (row, token) add them
// in block order after each round (one barrier a round).  The weights are
// the whole traffic, so what counts is bytes in flight and few instructions
// per block:
//   * the activations of a block are used once, so they go from L2 straight
//     to registers, in the operand's layout; their sums and scales are in
//     LDS (as register loads they cost a quarter of the vector memory time
//     and the fourth wave per SIMD);
//   * the MFMA's 16 operand rows are 8 tokens x 2: Q4_K's sub-blocks 2p and
//     2p + 1 (a lane's 8 low-nibble and 8 high-nibble weights; the other
//     half's activations zero), or Q6_K's quarters 2h and 2h + 1 (one
//     sub-group at a time, the other lane groups' activations zero), so a lane
//     forms the terms of its half only.
// Q4_K 14336 x 4096, 8 tokens, preparation included: 13.1 us (55.2 with
// act_prep and gemv_blocks); Q6_K 4096 x 14336: 17.8 (93).
template <int FMT>
struct FewTerms;                        // one lane's terms of a block, per token k
template <>
struct FewTerms<FMT_Q4K> { f4v t[4]; }; // sub-blocks 2p + half, p = 0 .. 3
typedef float f2v __attribute__((ext_vector_type(2)));
template <>
struct FewTerms<FMT_Q6K> { f2v t[4]; }; // quarters half, 2 + half

template <int FMT, int KS, int EPI>
__global__ __launch_bounds__(KS * 64, FMT == FMT_Q4K ? 4 : 3) void few_gemm(BatchArgs a)
{
    constexpr int CH = batch_chunk(FMT), AQ = aux_quads(FMT);
    typedef decltype(FewTerms<FMT>::t[0]) TV0;
    typedef std::remove_reference_t<TV0> TV;
    constexpr int NT = FMT == FMT_Q4K ? 4 : 2;             // terms per half
    __shared__ TV terms[2][KS][2][8][16];                  // [buffer][slot][half][token][row]
    extern __shared__ f4v axl[];                           // [block][AQ / 4][2]: aux of tokens 0 .. 7
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = a.nb;
    const int half = g >> 1, t4 = 4 * (g & 1);             // of this lane's sums: half, tokens t4 ..
    const int ih = j >> 3;                                 // of its operand row
    // (tokens past M: bytes that no token wrote, products that nothing reads)
    const uint8_t *qrow = a.q + (FMT == FMT_Q4K ? lane : g * 8 + (j & 7)) * 16;
    const int crow = tid & 15, ct = tid >> 4;              // of the combine: row, token (tid < 128)
    float y[EPI == BE_SILU ? 2 : 1];
    int tile = blockIdx.x, s = 0;
    if (EPI != BE_SILU) {
        while (s + 1 < a.nseg && tile >= a.tile_start[s + 1]) s++;
        tile -= a.tile_start[s];
    }
    const int ns = (nb + KS - 1) / KS;
    // (the first aux quads are requested before the weights and stored after
    // those are under way)
    const int nax = nb * (AQ / 2);
    f4v ax0[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int i = min(tid + k * KS * 64, nax - 1);
        ax0[k] = ((const f4v *)a.aux)[(i >> 1) * 4 + (i & 1)];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int it = 0; it < (EPI == BE_SILU ? 2 : 1); it++) {
        const uint8_t *wp = a.w[EPI == BE_SILU ? it : s] + (size_t)tile * nb * CH;
        struct Unit {
            RawBlock<FMT> w;
            u4v q[FMT == FMT_Q4K ? 2 : 4];
        };
        auto load = [&](int r, Unit &u) __attribute__((always_inline)) {
            const int b = min(r * KS + wave, nb - 1);
            u.w.load(wp + (size_t)b * CH, lane);
            // Q4_K: loads of 1 KB, two operands each; Q6_K: of 512 bytes (the
            // two halves' rows the same)
#pragma unroll
            for (int p = 0; p < (FMT == FMT_Q4K ? 2 : 4); p++)
                u.q[p] = *(const u4v *)(qrow + (size_t)b * 2048 + p * (FMT == FMT_Q4K ? 1024 : 512));
        };
        auto compute = [&](int r, const Unit &u, FewTerms<FMT> &o) __attribute__((always_inline)) {
            const f4v *ax = axl + min(r * KS + wave, nb - 1) * (AQ / 2) + (g & 1);
            const f4v as = ax[AQ / 2 - 2];
            if constexpr (FMT == FMT_Q4K) {
                const uint32_t s0 = u.w.h[1], s1 = u.w.h[2], s2 = u.w.h[3];
                // the scales and minima of sub-blocks half, half + 2 (bytes 0, 2)
                const int sh = 8 * half;
                const uint32_t sc[2] = {(s0 & 0x3f3f3f3fu) >> sh,
                                        ((s2 & 0x0f0f0f0fu) | (((s0 >> 6) & 0x03030303u) << 4)) >> sh};
                const uint32_t mn[2] = {(s1 & 0x3f3f3f3fu) >> sh,
                                        (((s2 >> 4) & 0x0f0f0f0fu) | (((s1 >> 6) & 0x03030303u) << 4)) >> sh};
                const float d = half_bits_to_float(u.w.h[0] & 0xffffu);
                const float dmin = half_bits_to_float(u.w.h[0] >> 16);
                const uint32_t m0 = ih ? 0u : ~0u, m1 = ~m0;
                const v4i magic = {MAGIC_BITS, MAGIC_BITS, MAGIC_BITS, MAGIC_BITS};
                auto run = [&](auto finite) __attribute__((always_inline)) {
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    const uint32_t a0 = p < 2 ? u.w.q0[2 * p] : u.w.q1[2 * p - 4];
                    const uint32_t a1 = p < 2 ? u.w.q0[2 * p + 1] : u.w.q1[2 * p - 3];
                    const v4i w = {(int)(a0 & 0x0f0f0f0fu), (int)(a1 & 0x0f0f0f0fu),
                                   (int)((a0 >> 4) & 0x0f0f0f0fu), (int)((a1 >> 4) & 0x0f0f0f0fu)};
                    const uint32_t x0 = u.q[p >> 1][2 * (p & 1)], x1 = u.q[p >> 1][2 * (p & 1) + 1];
                    const v4i x = {(int)(x0 & m0), (int)(x1 & m0), (int)(x0 & m1), (int)(x1 & m1)};
                    const v4i D = mfma64(x, w, magic);
                    const f4v sq = ax[2 * (2 * p + half)];
                    const float A = d * (float)((sc[p >> 1] >> (16 * (p & 1))) & 0xffu);
                    const float B = dmin * (float)((mn[p >> 1] >> (16 * (p & 1))) & 0xffu);
                    const float na = -MAGIC_F * A;
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const float pr = decltype(finite)::value
                                             ? __builtin_fmaf(A, __int_as_float(D[k]), na)
                                             : A * (float)(D[k] - MAGIC_BITS);
                        o.t[k][p] = as[k] * (pr - B * sq[k]);
                    }
                }
                };
                if (!any_nonfinite(d)) run(std::true_type{});
                else run(std::false_type{});
            } else {
                const float d = half_bits_to_float(u.w.d);
                f4v dd;
#pragma unroll
                for (int k = 0; k < 4; k++) dd[k] = as[k] * d;
                // sub-groups g / 2 = 0 and 1 of quarter 2h + ih
                const uint32_t m0 = g == ih ? ~0u : 0u, m1 = g == 2 + ih ? ~0u : 0u;
                const v4i zero = {0, 0, 0, 0};
                const u4v sc = {u.w.sc[0] >> 8 * half, u.w.sc[1] >> 8 * half, u.w.sc[2] >> 8 * half,
                                u.w.sc[3] >> 8 * half};
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    v4i part = zero;
#pragma unroll
                    for (int hi = 0; hi < 2; hi++) {
                        const v4i w = q6_bytes(u.w, h, hi, g);
                        const u4v q = u.q[2 * h + hi];
                        const v4i x0 = {(int)(q[0] & m0), (int)(q[1] & m0), (int)(q[2] & m0), (int)(q[3] & m0)};
                        const v4i x1 = {(int)(q[0] & m1), (int)(q[1] & m1), (int)(q[2] & m1), (int)(q[3] & m1)};
                        const v4i D0 = mfma64(x0, w, zero), D1 = mfma64(x1, w, zero);
                        // scales 8h + half + 4 hi (sub-group 2 hi) and + 2
                        const int c0 = q6_scale(sc, 8 * h + 4 * hi), c1 = q6_scale(sc, 8 * h + 4 * hi + 2);
#pragma unroll
                        for (int k = 0; k < 4; k++)
                            part[k] += __mul24(c0, D0[k]) + __mul24(c1, D1[k]);
                    }
#pragma unroll
                    for (int k = 0; k < 4; k++) o.t[k][h] = dd[k] * (float)(part[k] >> 2);
                }
            }
        };
        float acc = 0.0f;
        auto combine = [&](int r) __attribute__((always_inline)) {
            if (tid >= 128) return;
#pragma unroll
            for (int w = 0; w < KS; w++) {
                if (r * KS + w >= nb) break;               // (uniform)
                const TV h0 = terms[r & 1][w][0][ct][crow], h1 = terms[r & 1][w][1][ct][crow];
#pragma unroll
                for (int p = 0; p < NT; p++) {
                    acc = acc + h0[p];
                    acc = acc + h1[p];
                }
            }
        };
        auto round = [&](int r, Unit &u) __attribute__((always_inline)) {
            if (r < ns) {                                  // (uniform)
                FewTerms<FMT> o;
                compute(r, u, o);
#pragma unroll
                for (int k = 0; k < 4; k++) terms[r & 1][wave][half][t4 + k][j] = o.t[k];
            }
            load(r + 2, u);
            // (the loads stay here and in this order: a unit's wait then
            // leaves the unit after it in flight)
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            combine(r);
        };
        // two units in flight; a buffer is written again two rounds later,
        // past the barrier that its combine precedes
        Unit u0, u1;
        load(0, u0);
        __builtin_amdgcn_sched_barrier(0);
        load(1, u1);
        __builtin_amdgcn_sched_barrier(0);
        if (it == 0) {
#pragma unroll
            for (int k = 0; k < 2; k++)
                if (tid + k * KS * 64 < nax) axl[tid + k * KS * 64] = ax0[k];
            for (int i = tid + 2 * KS * 64; i < nax; i += KS * 64)
                axl[i] = ((const f4v *)a.aux)[(i >> 1) * 4 + (i & 1)];
            __syncthreads();
        }
        // (always both: a way out between them would leave the compiler
        // unsure at the loop's head how many loads follow the first unit's)
        for (int r = 0; r < ns; r += 2) {
            round(r, u0);
            round(r + 1, u1);
        }
        y[it] = acc;
        if (EPI == BE_SILU) __syncthreads();               // (the buffers start over)
    }
    if (tid >= 128 || ct >= a.M) return;
    const int row = tile * 16 + crow;
    if (row >= a.n_rows[s]) return;
    float *o = a.out[s] + (size_t)ct * a.out_stride[s] + row;
    if (EPI == BE_SILU) *o = fox_div(y[0], 1.0f + fox_expf(-y[0])) * y[EPI == BE_SILU];
    else *o = (a.flags & FOX_GPU_GEMV_ACCUMULATE) ? *o + y[0] : y[0];
}

// ------------------------------------------- few row tiles: blocks split

// batch_gemm's waves each walk the whole of K, so a matrix of few rows leaves
// the chip part empty and every block waits for its loads (Q6_K 4096 x 14336,
// 16 tokens: 59 us, here 26; Q4_K 4096 x 4096 19, here 10.5).  Here a
// workgroup is one row tile and one token tile, its KS waves take units of U
// blocks in turn, operands straight from L2 to registers, and pass the float
// terms through LDS to 256 lanes (token, row) that add them in block order, as
// in few_gemm.
template <int FMT>
struct SplitTerms;                      // one lane's terms of a unit, per token k
template <>
struct SplitTerms<FMT_TQ2> { static constexpr int U = 2, NV = 1; typedef f2v V; };   // two blocks
template <>
struct SplitTerms<FMT_Q4K> { static constexpr int U = 1, NV = 2; typedef f4v V; };   // sub-blocks 4v ..
template <>
struct SplitTerms<FMT_Q6K> { static constexpr int U = 1, NV = 1; typedef f4v V; };   // quarters

#define SPLIT_KS 4
template <int FMT, int EPI>
__global__ __launch_bounds__(256, FMT == FMT_Q4K ? 2 : 3) void split_gemm(BatchArgs a)
{
    typedef SplitTerms<FMT> ST;
    typedef typename ST::V V;
    constexpr int KS = SPLIT_KS, U = ST::U, NV = ST::NV, CH = batch_chunk(FMT), AQ = aux_quads(FMT);
    __shared__ V terms[2][KS][NV][16][16];                 // [buffer][slot][..][token][row]
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = a.nb, tt = blockIdx.y;
    const uint8_t *qp = a.q + (size_t)tt * nb * B_TILE + lane * 16;
    const f4v *axp = (const f4v *)a.aux + (size_t)tt * nb * AQ + g;
    const int crow = tid & 15, ct = tid >> 4;              // of the combine: row, token
    float y[EPI == BE_SILU ? 2 : 1];
    int tile = blockIdx.x, s = 0;
    if (EPI != BE_SILU) {
        while (s + 1 < a.nseg && tile >= a.tile_start[s + 1]) s++;
        tile -= a.tile_start[s];
    }
    const int nu = (nb + U - 1) / U, ns = (nu + KS - 1) / KS;
#pragma unroll
    for (int it = 0; it < (EPI == BE_SILU ? 2 : 1); it++) {
        const uint8_t *wp = a.w[EPI == BE_SILU ? it : s] + (size_t)tile * nb * CH;
        struct Unit {
            RawBlock<FMT> w[U];
            v4i x[U][4];
            f4v ax[U][FMT == FMT_Q4K ? 9 : 1];
        };
        auto load = [&](int r, Unit &u) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < U; i++) {
                const int b = min((r * KS + wave) * U + i, nb - 1);
                u.w[i].load(wp + (size_t)b * CH, lane);
#pragma unroll
                for (int p = 0; p < 4; p++) u.x[i][p] = *(const v4i *)(qp + (size_t)b * B_TILE + p * 1024);
#pragma unroll
                for (int p = 0; p < (FMT == FMT_Q4K ? 9 : 1); p++) u.ax[i][p] = axp[(size_t)b * AQ + 4 * p];
            }
        };
        auto compute = [&](const Unit &u, V (*o)[NV][16][16]) __attribute__((always_inline)) {
            V t[NV][4];
            if constexpr (FMT == FMT_TQ2) {
#pragma unroll
                for (int i = 0; i < U; i++) {
                    v4i D = __builtin_bit_cast(v4i, u.ax[i][0]);
#pragma unroll
                    for (int p = 0; p < 4; p++) {
                        const uint32_t d = u.w[i].qs[p];
                        const v4i w = {(int)(d & 0x03030303u), (int)((d >> 2) & 0x03030303u),
                                       (int)((d >> 4) & 0x03030303u), (int)((d >> 6) & 0x03030303u)};
                        D = mfma64(u.x[i][p], w, D);
                    }
                    const float d = half_bits_to_float(u.w[i].d);
                    if (!any_nonfinite(d)) {
                        const float nd = -MAGIC_F * d;
#pragma unroll
                        for (int k = 0; k < 4; k++) t[0][k][i] = __builtin_fmaf(d, __int_as_float(D[k]), nd);
                    } else {
#pragma unroll
                        for (int k = 0; k < 4; k++) t[0][k][i] = d * (float)(D[k] - MAGIC_BITS);
                    }
                }
            } else if constexpr (FMT == FMT_Q4K) {
                // (batch_gemm's terms, block_terms)
                const RawBlock<FMT> &raw = u.w[0];
                const uint32_t s0 = raw.h[1], s1 = raw.h[2], s2 = raw.h[3];
                const uint32_t sc[2] = {s0 & 0x3f3f3f3fu,
                                        (s2 & 0x0f0f0f0fu) | (((s0 >> 6) & 0x03030303u) << 4)};
                const uint32_t mn[2] = {s1 & 0x3f3f3f3fu,
                                        ((s2 >> 4) & 0x0f0f0f0fu) | (((s1 >> 6) & 0x03030303u) << 4)};
                const float d = half_bits_to_float(raw.h[0] & 0xffffu);
                const float dmin = half_bits_to_float(raw.h[0] >> 16);
                const v4i magic = {MAGIC_BITS, MAGIC_BITS, MAGIC_BITS, MAGIC_BITS};
                const f4v as = u.ax[0][8];
                auto run = [&](auto finite) __attribute__((always_inline)) {
#pragma unroll
                    for (int sb = 0; sb < 8; sb++) {
                        const int p = sb >> 1, hh = sb & 1;
                        const uint32_t a0 = (p < 2 ? raw.q0[2 * p] : raw.q1[2 * p - 4]) >> (4 * hh);
                        const uint32_t a1 = (p < 2 ? raw.q0[2 * p + 1] : raw.q1[2 * p - 3]) >> (4 * hh);
                        const long w = (long)((uint64_t)(a0 & 0x0f0f0f0fu) | (uint64_t)(a1 & 0x0f0f0f0fu) << 32);
                        const long x = (long)((uint64_t)(uint32_t)u.x[0][p][2 * hh] |
                                              (uint64_t)(uint32_t)u.x[0][p][2 * hh + 1] << 32);
                        const v4i D = __builtin_amdgcn_mfma_i32_16x16x32_i8(x, w, magic, 0, 0, 0);
                        const float A = d * (float)((sc[sb >> 2] >> (8 * (sb & 3))) & 0xffu);
                        const float B = dmin * (float)((mn[sb >> 2] >> (8 * (sb & 3))) & 0xffu);
                        const float na = -MAGIC_F * A;
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            const float pr = decltype(finite)::value
                                                 ? __builtin_fmaf(A, __int_as_float(D[k]), na)
                                                 : A * (float)(D[k] - MAGIC_BITS);
                            t[sb >> 2][k][sb & 3] = as[k] * (pr - B * u.ax[0][sb][k]);
                        }
                    }
                };
                if (!any_nonfinite(d)) run(std::true_type{});
                else run(std::false_type{});
            } else {
                const float d = half_bits_to_float(u.w[0].d);
                const v4i zero = {0, 0, 0, 0};
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    v4i part[2] = {zero, zero};
#pragma unroll
                    for (int hi = 0; hi < 2; hi++) {
                        const v4i w = q6_bytes(u.w[0], h, hi, g);
#pragma unroll
                        for (int gg = 0; gg < 4; gg++) {
                            const int m = g == gg ? -1 : 0;
                            const v4i wm = {w[0] & m, w[1] & m, w[2] & m, w[3] & m};
                            const v4i D = mfma64(u.x[0][2 * h + hi], wm, zero);
                            const int sc = q6_scale(u.w[0].sc, 8 * h + (gg & 1) + 2 * ((gg >> 1) + 2 * hi));
#pragma unroll
                            for (int k = 0; k < 4; k++) part[gg & 1][k] += __mul24(sc, D[k]);
                        }
                    }
#pragma unroll
                    for (int v = 0; v < 2; v++)
#pragma unroll
                        for (int k = 0; k < 4; k++)
                            t[0][k][2 * h + v] = u.ax[0][0][k] * d * (float)(part[v][k] >> 2);
                }
            }
#pragma unroll
            for (int v = 0; v < NV; v++)
#pragma unroll
                for (int k = 0; k < 4; k++) (*o)[v][4 * g + k][j] = t[v][k];
        };
        float acc = 0.0f;
        auto combine = [&](int r) __attribute__((always_inline)) {
#pragma unroll
            for (int w = 0; w < KS; w++) {
                const int b = (r * KS + w) * U;
                if (b >= nb) break;                        // (uniform)
#pragma unroll
                for (int v = 0; v < NV; v++) {
                    const V x = terms[r & 1][w][v][ct][crow];
                    if (FMT == FMT_TQ2) {
                        acc = acc + x[0];
                        if (b + 1 < nb) acc = acc + x[1];  // (uniform)
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; i++) acc = acc + x[i];
                    }
                }
            }
        };
        auto round = [&](int r, Unit &u) __attribute__((always_inline)) {
            if (r < ns) compute(u, &terms[r & 1][wave]);   // (uniform)
            load(r + 2, u);
            __builtin_amdgcn_sched_barrier(0);             // (as in few_gemm)
            __syncthreads();
            combine(r);
        };
        Unit u0, u1;
        load(0, u0);
        __builtin_amdgcn_sched_barrier(0);
        load(1, u1);
        __builtin_amdgcn_sched_barrier(0);
        for (int r = 0; r < ns; r += 2) {
            round(r, u0);
            round(r + 1, u1);
        }
        y[it] = acc;
        if (EPI == BE_SILU) __syncthreads();               // (the buffers start over)
    }
    const int t = tt * 16 + ct, row = tile * 16 + crow;
    if (t >= a.M || row >= a.n_rows[s]) return;
    if (FMT == FMT_TQ2) {
        const float sc = a.scale[t];
#pragma unroll
        for (int it = 0; it < (EPI == BE_SILU ? 2 : 1); it++) y[it] = y[it] * sc;
    }
    float *o = a.out[s] + (size_t)t * a.out_stride[s] + row;
    if (EPI == BE_SILU) *o = fox_div(y[0], 1.0f + fox_expf(-y[0])) * y[EPI == BE_SILU];
    else *o = (a.flags & FOX_GPU_GEMV_ACCUMULATE) ? *o + y[0] : y[0];
}

// ------------------------------------------------------------------ host

static size_t up256(size_t v) { return (v + 255) & ~(size_t)255; }

#define PREP_MAX_R 16                   // batch_prep: K <= 2048 * PREP_MAX_R

struct BatchWs {
    uint8_t *q;
    uint32_t *aux;
    float *scale;
};

// the prepared operand of M tokens of width K in the context's workspace
// (fixed: memory that holds it, in place of the context's)
static fox_gpu_status batch_carve(fox_gpu_ctx *ctx, int fmt, size_t K, size_t M, uint8_t *fixed,
                                  BatchWs *w)
{
    // (few_gemm's operand has room for eight tokens whatever M is)
    const size_t nq = M <= FOX_GPU_MAX_TOKENS && fmt != FMT_TQ2 ? FOX_GPU_MAX_TOKENS * K
                                                                : (M + 15) / 16 * 16 * K;
    const size_t na = up256((M + 15) / 16 * (K / 256) * (size_t)aux_quads(fmt) * 16);
    const size_t ns = up256(M * 4);
    if (!fixed) {
        fox_gpu_status st = fox_ws_reserve(ctx, nq + na + ns);
        if (st) return st;
        fixed = ctx->ws;
    }
    w->q = fixed;
    w->aux = (uint32_t *)(fixed + nq);
    w->scale = (float *)(fixed + nq + na);
    return FOX_GPU_OK;
}

template <int FMT, bool NORM>
static const void *prep_kernel(int r)
{
    return r <= 1 ? (const void *)batch_prep<FMT, NORM, 1> : r <= 2 ? (const void *)batch_prep<FMT, NORM, 2>
         : r <= 3 ? (const void *)batch_prep<FMT, NORM, 3> : r <= 4 ? (const void *)batch_prep<FMT, NORM, 4>
         : r <= 6 ? (const void *)batch_prep<FMT, NORM, 6> : r <= 8 ? (const void *)batch_prep<FMT, NORM, 8>
         : r <= 12 ? (const void *)batch_prep<FMT, NORM, 12> : (const void *)batch_prep<FMT, NORM, 16>;
}

// (the K-quants without a norm: blocks apart on grid y, one dword a thread)
template <int FMT>
static const void *prep_fmt(bool norm, int r)
{
    if (norm) return prep_kernel<FMT, true>(r);
    if constexpr (FMT == FMT_TQ2) return prep_kernel<FMT, false>(r);
    else return (const void *)batch_prep<FMT, false, 1>;
}

template <int FMT, int R, int EPI>
static const void *gemm_c(int C)
{
    return C == 1 ? (const void *)batch_gemm<FMT, R, 1, EPI> : C == 2 ? (const void *)batch_gemm<FMT, R, 2, EPI>
         : C == 3 ? (const void *)batch_gemm<FMT, R, 3, EPI> : (const void *)batch_gemm<FMT, R, 4, EPI>;
}

static const void *gemm_kernel(int fmt, int R, int C, int epi)
{
    if (fmt == FMT_TQ2) {
        if (epi == BE_SILU) return R == 4 ? gemm_c<FMT_TQ2, 4, BE_SILU>(C) : gemm_c<FMT_TQ2, 2, BE_SILU>(C);
        return R == 4 ? gemm_c<FMT_TQ2, 4, BE_STORE>(C) : R == 2 ? gemm_c<FMT_TQ2, 2, BE_STORE>(C)
                                                                 : gemm_c<FMT_TQ2, 1, BE_STORE>(C);
    }
    if (fmt == FMT_Q4K)
        return epi == BE_SILU ? gemm_c<FMT_Q4K, 2, BE_SILU>(C) : gemm_c<FMT_Q4K, 1, BE_STORE>(C);
    return gemm_c<FMT_Q6K, 1, BE_STORE>(C);
}

// eight waves per row tile where four would leave the chip part empty
static const void *few_kernel(int fmt, bool wide, int epi)
{
#define FOX_FEW(f, e) (wide ? (const void *)few_gemm<f, 8, e> : (const void *)few_gemm<f, 4, e>)
    if (fmt == FMT_Q4K) return epi == BE_SILU ? FOX_FEW(FMT_Q4K, BE_SILU) : FOX_FEW(FMT_Q4K, BE_STORE);
    return epi == BE_SILU ? FOX_FEW(FMT_Q6K, BE_SILU) : FOX_FEW(FMT_Q6K, BE_STORE);
#undef FOX_FEW
}

static const void *split_kernel(int fmt, int epi)
{
#define FOX_SPLIT(f) (epi == BE_SILU ? (const void *)split_gemm<f, BE_SILU> : (const void *)split_gemm<f, BE_STORE>)
    return fmt == FMT_TQ2 ? FOX_SPLIT(FMT_TQ2) : fmt == FMT_Q4K ? FOX_SPLIT(FMT_Q4K) : FOX_SPLIT(FMT_Q6K);
#undef FOX_SPLIT
}

// split_gemm where batch_gemm would have too few waves to hide its loads: by
// row tiles times token groups, a measured line per format (us, split / whole):
// ternary 160 tiles x 2 groups (K 9728) 20 / 29, 336 x 2 (K 4096) 22 / 18;
// Q4_K (K 4096) 256 x 2 27 / 36, 256 x 4 59 / 53, 896 x 1 23 / 20; Q6_K
// (K 14336) 256 x 2 66 / 130, 256 x 4 143 / 162.
static bool split_better(int fmt, int tiles, int mt, int n_cu)
{
    return tiles * ((mt + 3) / 4) < (fmt == FMT_TQ2 ? 2 : fmt == FMT_Q4K ? 3 : 5) * n_cu;
}

static fox_gpu_status batch_check(fox_gpu_ctx *ctx, size_t n, const fox_gpu_tensor *const *ws,
                                  const float *x, size_t x_stride, size_t M, float *const *outs,
                                  const size_t *out_strides)
{
    if (!ctx || !ws || !x || !outs || !out_strides || n == 0 || n > MAX_SEGS)
        return fox_fail(FOX_GPU_ERR_ARG, "batch: bad argument");
    if (M == 0 || M > FOX_GPU_BATCH_TOKENS)
        return fox_fail(FOX_GPU_ERR_ARG, "batch: %zu tokens; 1 to %d per call", M,
                        FOX_GPU_BATCH_TOKENS);
    for (size_t i = 0; i < n; i++) {
        if (!ws[i] || !outs[i]) return fox_fail(FOX_GPU_ERR_ARG, "batch: null matrix or output");
        if (ws[i]->type != ws[0]->type || ws[i]->ne0 != ws[0]->ne0)
            return fox_fail(FOX_GPU_ERR_ARG,
                            "batch: matrices of one call must share type and width");
        if (out_strides[i] < ws[i]->ne1)
            return fox_fail(FOX_GPU_ERR_ARG, "batch: output stride < rows");
        if (ws[i]->ne0 > (1u << 20) || ws[i]->ne1 > (1u << 30))
            return fox_fail(FOX_GPU_ERR_UNSUPPORTED, "batch: matrix too large");
    }
    if (x_stride < ws[0]->ne0) return fox_fail(FOX_GPU_ERR_ARG, "batch: input stride < K");
    return FOX_GPU_OK;
}

// prepare + GEMM; FOX_GPU_ERR_UNSUPPORTED (no error recorded) where the
// caller takes the calls of FOX_GPU_MAX_TOKENS tokens
static fox_gpu_status batch_run(fox_gpu_ctx *ctx, size_t n, const fox_gpu_tensor *const *ws,
                                const float *x, size_t x_stride, size_t M, const float *norm_w,
                                float eps, float *const *outs, const size_t *out_strides,
                                unsigned flags, int epi, uint8_t *fixed = nullptr)
{
    const int fmt = fmt_of(ws[0]->type);
    const size_t K = (size_t)ws[0]->ne0;
    if (fmt < 0 || K == 0 || K % 256 || K > 2048 * PREP_MAX_R || x_stride % 4 ||
        ((uintptr_t)x | (uintptr_t)norm_w) % 16)
        return FOX_GPU_ERR_UNSUPPORTED;
    // (Q6_K gate/up pairs: two such tiles per wave do not fit its registers)
    if (fmt == FMT_Q6K && epi == BE_SILU && M > FOX_GPU_MAX_TOKENS &&
        !split_better(fmt, (int)ws[0]->n_tiles, (int)((M + 15) / 16), ctx->n_cu))
        return FOX_GPU_ERR_UNSUPPORTED;
    BatchWs w;
    fox_gpu_status st = batch_carve(ctx, fmt, K, M, fixed, &w);
    if (st) return st;
    {
        const int r = (int)((K / 4 + 511) / 512);
        const bool norm = norm_w != nullptr;
        const bool blocks = fmt != FMT_TQ2 && !norm;       // (grid y: 8 blocks each)
        const void *k = fmt == FMT_TQ2 ? prep_fmt<FMT_TQ2>(norm, r)
                      : fmt == FMT_Q4K ? prep_fmt<FMT_Q4K>(norm, r) : prep_fmt<FMT_Q6K>(norm, r);
        int iK = (int)K, iM = (int)M, few = fmt != FMT_TQ2 && M <= FOX_GPU_MAX_TOKENS;
        void *args[] = {(void *)&x, (void *)&norm_w, (void *)&iK, (void *)&x_stride, (void *)&eps,
                        (void *)&iM, (void *)&few, (void *)&w.q, (void *)&w.aux, (void *)&w.scale};
        const dim3 grid(few ? (unsigned)M : (unsigned)((M + 63) / 64 * 64), blocks ? (unsigned)r : 1u);
        hipError_t e = hipLaunchKernel(k, grid, dim3(512), args, 0, ctx->stream);
        if (e != hipSuccess) return fox_hip_fail(e, "batch: prepare");
        FOX_LAUNCHED("batch: prepare");
    }
    BatchArgs a;
    memset(&a, 0, sizeof(a));
    a.nseg = (int)n;
    a.nb = (int)(K / 256);
    a.M = (int)M;
    a.flags = flags;
    a.q = w.q;
    a.aux = w.aux;
    a.scale = w.scale;
    int tiles = 0;
    for (size_t i = 0; i < n; i++) {
        a.w[i] = ws[i]->d;
        a.out[i] = outs[i];
        a.out_stride[i] = out_strides[i];
        a.n_rows[i] = (int)ws[i]->ne1;
        a.tile_start[i] = tiles;
        tiles += (int)ws[i]->n_tiles;
    }
    a.tile_start[n] = tiles;
    if (fmt != FMT_TQ2 && M <= FOX_GPU_MAX_TOKENS) {
        // K-quants, up to eight tokens: a workgroup per row tile
        const int nt = epi == BE_SILU ? a.tile_start[1] : tiles;
        const bool wide = nt < 2 * ctx->n_cu;
        const void *k = few_kernel(fmt, wide, epi);
        void *args[] = {(void *)&a};
        const size_t lds = K / 256 * (size_t)aux_quads(fmt) * 8;   // (at most 36 KB)
        hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e == hipSuccess)
            e = hipLaunchKernel(k, dim3((unsigned)nt), dim3(wide ? 512 : 256), args, lds, ctx->stream);
        if (e != hipSuccess) return fox_hip_fail(e, "batch: product");
        FOX_LAUNCHED("batch: product");
        return FOX_GPU_OK;
    }
    const int mt = (int)((M + 15) / 16);
    const int wt = epi == BE_SILU ? a.tile_start[1] : tiles;        // workgroup tiles
    if (split_better(fmt, wt, mt, ctx->n_cu)) {
        const void *k = split_kernel(fmt, epi);
        void *args[] = {(void *)&a};
        hipError_t e = hipLaunchKernel(k, dim3((unsigned)wt, (unsigned)mt), dim3(256), args, 0, ctx->stream);
        if (e != hipSuccess) return fox_hip_fail(e, "batch: product");
        FOX_LAUNCHED("batch: product");
        return FOX_GPU_OK;
    }
    // token groups of C 16-token tiles, as even as they come at C <= 4
    const int n_tg = (mt + 3) / 4, C = (mt + n_tg - 1) / n_tg;
    a.n_tg = (mt + C - 1) / C;
    // row tiles per wave: more share each token operand read from LDS (the
    // ternary kernel's LDS reads take as long as its MFMAs below four), as
    // long as every compute unit still gets two workgroups
    int R = epi == BE_SILU ? 2 : 1;
    if (fmt == FMT_TQ2) {
        const int want = 2 * ctx->n_cu;
        while (R < 4 && (tiles + 8 * R - 1) / (8 * R) * a.n_tg >= want) R *= 2;
    }
    a.n_wg = (tiles + 4 * R - 1) / (4 * R) * a.n_tg;
    const void *k = gemm_kernel(fmt, R, C, epi);
    void *args[] = {(void *)&a};
    hipError_t e = hipLaunchKernel(k, dim3((unsigned)((a.n_wg + 7) / 8 * 8)), dim3(BT_THREADS), args, 0,
                                   ctx->stream);
    if (e != hipSuccess) return fox_hip_fail(e, "batch: product");
    FOX_LAUNCHED("batch: product");
    return FOX_GPU_OK;
}

// fox_gpu_gemv's and fox_gpu_gemv_multi's products of 2 to FOX_GPU_MAX_TOKENS
// tokens that fox_fused_gemv leaves: the K-quants and some ternary ones
// (arguments checked by the caller; `fixed` holds FOX_NOALLOC_SCRATCH bytes,
// several times the operand of the widest row batch_run takes)
fox_gpu_status fox_few_gemv(fox_gpu_ctx *ctx, size_t n, const fox_gpu_tensor *const *ws,
                            const float *x, size_t x_stride, size_t M, float *const *outs,
                            const size_t *out_strides, unsigned flags, uint8_t *fixed)
{
    return batch_run(ctx, n, ws, x, x_stride, M, nullptr, 0.0f, outs, out_strides, flags, BE_STORE,
                     fixed);
}

extern "C" fox_gpu_status fox_gpu_batch_gemv(fox_gpu_ctx *ctx, size_t n,
                                             const fox_gpu_tensor *const *ws, const float *x,
                                             size_t x_stride, size_t M, float *const *outs,
                                             const size_t *out_strides, unsigned flags)
{
    fox_gpu_status st = batch_check(ctx, n, ws, x, x_stride, M, outs, out_strides);
    if (st) return st;
    if (fmt_of(ws[0]->type) < 0) {
        for (size_t i = 0; i < n && !st; i++)
            st = fox_float_gemv(ctx, ws[i], x, x_stride, M, outs[i], out_strides[i], flags);
        return st;
    }
    st = batch_run(ctx, n, ws, x, x_stride, M, nullptr, 0.0f, outs, out_strides, flags, BE_STORE);
    if (st != FOX_GPU_ERR_UNSUPPORTED) return st;
    for (size_t t = 0; t < M; t += FOX_GPU_MAX_TOKENS) {
        const size_t m = M - t < FOX_GPU_MAX_TOKENS ? M - t : FOX_GPU_MAX_TOKENS;
        float *o[MAX_SEGS];
        for (size_t i = 0; i < n; i++) o[i] = outs[i] + t * out_strides[i];
        st = fox_gemv_launch(ctx, n, ws, x + t * x_stride, x_stride, nullptr, nullptr, m, o,
                             out_strides, flags, nullptr);
        if (st) return st;
    }
    return FOX_GPU_OK;
}

extern "C" fox_gpu_status fox_gpu_batch_gemv_rmsnorm(fox_gpu_ctx *ctx, size_t n,
                                                     const fox_gpu_tensor *const *ws,
                                                     const float *x, size_t x_stride, size_t M,
                                                     const float *norm_w, float eps,
                                                     float *const *outs, const size_t *out_strides,
                                                     unsigned flags)
{
    fox_gpu_status st = batch_check(ctx, n, ws, x, x_stride, M, outs, out_strides);
    if (st) return st;
    if (!norm_w) return fox_fail(FOX_GPU_ERR_ARG, "batch: null norm weights");
    return batch_run(ctx, n, ws, x, x_stride, M, norm_w, eps, outs, out_strides, flags, BE_STORE);
}

extern "C" fox_gpu_status fox_gpu_batch_gate_up_silu(fox_gpu_ctx *ctx, const fox_gpu_tensor *w_gate,
                                                     const fox_gpu_tensor *w_up, const float *x,
                                                     size_t x_stride, size_t M,
                                                     const float *norm_w, float eps, float *h_out,
                                                     size_t h_stride)
{
    const fox_gpu_tensor *ws[2] = {w_gate, w_up};
    float *outs[2] = {h_out, h_out};
    size_t strides[2] = {h_stride, h_stride};
    if (w_gate && w_up && w_gate->type != w_up->type) return FOX_GPU_ERR_UNSUPPORTED;
    fox_gpu_status st = batch_check(ctx, 2, ws, x, x_stride, M, outs, strides);
    if (st) return st;
    if (!norm_w) return fox_fail(FOX_GPU_ERR_ARG, "batch: null norm weights");
    if (w_gate->ne1 != w_up->ne1)
        return fox_fail(FOX_GPU_ERR_ARG, "batch: gate and up must have the same rows");
    return batch_run(ctx, 2, ws, x, x_stride, M, norm_w, eps, outs, strides, 0, BE_SILU);
}
