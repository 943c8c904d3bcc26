// fox_battn.hip -- exact attention of a batched pass (many tokens), every sum
// in the reference's order (src/forward.c:222-257, src/ops.c:24-39), so
// bit-identical to the kernels of fox_ops.hip:
//   batt_qk   scores: a thread owns a register tile of (token, position)
//             pairs and adds their products in dimension order;
//   batt_sm   the exps and their sum: a wave per 16 (or 4) tokens of a head;
//   batt_av   values: a thread owns a register tile of (token, column) pairs
//             and adds a_j v_j in position order.
// With many tokens the independent sums fill the chip by themselves, so each
// runs one add at a time in its own register and the kernels are bound by
// the vector unit: a product and an add per term (the reference rounds both,
// so neither a fused multiply-add nor the matrix cores apply).  A 1024-token
// prompt of 32 heads of 128: scores 114 us and values 110 us per layer, where
// the vector unit needs 109 each (2.15 G terms, a product and an add each).
#include "fox_internal.h"
#include "fox_gemv_dev.h"
#include "fox_math.h"

#define BQ_POS 64                // positions of a scores tile (the softmax's maxima are per 64)
#define BQ_DQ 8                  // dimension quads staged at a time
#define BQ_STR 9                 // LDS row stride in quads (one quad of padding)

typedef float f4v __attribute__((ext_vector_type(4)));

// Scores of 16 TI tokens x 64 positions of one query head: 256 threads,
// thread (tx, ty) = (tid % 16, tid / 16) owns tokens ty * TI + i and positions
// tx + 16 k; the products are added a dimension at a time, both operands read
// from LDS as quads of four dimensions (TI + 4 reads per 32 TI vector
// instructions).  Positions at or past a token's end are not written and
// stay out of the maxima.
template <int TI>
__global__ __launch_bounds__(256) void batt_qk(const float *__restrict__ q, size_t q_stride,
                                               const float *__restrict__ kc, int n_head,
                                               int n_head_kv, int hd,
                                               const uint32_t *__restrict__ pos, int t_base,
                                               int n_ctx, size_t att_stride,
                                               float *__restrict__ att, float *__restrict__ tmax,
                                               int n_tiles, int M)
{
    constexpr int TT = 16 * TI;
    __shared__ f4v Qs[TT * BQ_STR], Ks[BQ_POS * BQ_STR];
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    const int tile = blockIdx.x, p0 = tile * BQ_POS, h = blockIdx.y, t0 = (int)blockIdx.z * TT;
    const int kvh = h / (n_head / n_head_kv), kvd = n_head_kv * hd, hd4 = hd >> 2;
    const size_t pz = (size_t)pos[0] + (size_t)t_base;
    auto upto_of = [&](int t) { return (int)min(pz + (size_t)t + 1, (size_t)n_ctx); };
    const int t_last = min(t0 + TT, M) - 1, upto_last = upto_of(t_last);
    if (p0 >= upto_last) return;                           // (uniform)
    const f4v *kb = (const f4v *)(kc + (size_t)p0 * kvd + (size_t)kvh * hd);
    const int rows = min(BQ_POS, upto_last - p0);
    float acc[TI][4];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int k = 0; k < 4; k++) acc[i][k] = 0.0f;
    // staging: quad idx = tid + 256 u of the chunk is row idx / 8, quad
    // idx % 8 (rows past the end repeat the last one)
    constexpr int NQ = TT * BQ_DQ / 256, NK = BQ_POS * BQ_DQ / 256;
    f4v qr[NQ], kr[NK];
    auto fetch = [&](int d0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < NQ; u++) {
            const int idx = tid + 256 * u, t = min(t0 + (idx >> 3), t_last);
            qr[u] = ((const f4v *)(q + (size_t)t * q_stride + (size_t)h * hd))[min(d0 + (idx & 7), hd4 - 1)];
        }
#pragma unroll
        for (int u = 0; u < NK; u++) {
            const int idx = tid + 256 * u;
            kr[u] = kb[(size_t)min(idx >> 3, rows - 1) * (kvd / 4) + min(d0 + (idx & 7), hd4 - 1)];
        }
    };
    fetch(0);
    for (int d0 = 0; d0 < hd4; d0 += BQ_DQ) {
        if (d0) __syncthreads();
#pragma unroll
        for (int u = 0; u < NQ; u++) {
            const int idx = tid + 256 * u;
            Qs[(idx >> 3) * BQ_STR + (idx & 7)] = qr[u];
        }
#pragma unroll
        for (int u = 0; u < NK; u++) {
            const int idx = tid + 256 * u;
            Ks[(idx >> 3) * BQ_STR + (idx & 7)] = kr[u];
        }
        __syncthreads();
        if (d0 + BQ_DQ < hd4) fetch(d0 + BQ_DQ);
        const int nd = min(BQ_DQ, hd4 - d0);
        auto step = [&](int d) __attribute__((always_inline)) {
            f4v kv[4];
#pragma unroll
            for (int k = 0; k < 4; k++) kv[k] = Ks[(tx + 16 * k) * BQ_STR + d];
#pragma unroll
            for (int i = 0; i < TI; i++) {
                const f4v qv = Qs[(ty * TI + i) * BQ_STR + d];
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int k = 0; k < 4; k++) acc[i][k] = acc[i][k] + qv[e] * kv[k][e];
            }
        };
        if (nd == BQ_DQ) {
#pragma unroll
            for (int d = 0; d < BQ_DQ; d++) step(d);
        } else {
            for (int d = 0; d < nd; d++) step(d);
        }
    }
    const float scale = fox_div(1.0f, fox_sqrtf((float)hd));
#pragma unroll
    for (int i = 0; i < TI; i++) {
        const int t = t0 + ty * TI + i;
        const int upto = t < M ? upto_of(t) : 0;
        float *row = att + ((size_t)t * n_head + h) * att_stride + p0;
        float m = -INFINITY;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float s = acc[i][k] * scale;
            const bool ok = p0 + tx + 16 * k < upto;
            if (ok) row[tx + 16 * k] = s;
            m = ok && s > m ? s : m;                       // (a NaN is never taken)
        }
        // over the 16 lanes of the token
        auto mx = [](float a, float b) { return b > a ? b : a; };
        m = mx(m, dpp_t<0xB1, 0xF>(m, m));
        m = mx(m, dpp_t<0x4E, 0xF>(m, m));
        m = mx(m, dpp_t<0x141, 0xF>(m, m));
        m = mx(m, dpp_t<0x140, 0xF>(m, m));
        if (tx == 0 && p0 < upto) tmax[((size_t)t * n_head + h) * n_tiles + tile] = m;
    }
}

// Softmax of ROWS tokens of one head per wave, no wave waiting for another:
// lane (r, c) = (lane / LPR, lane % LPR) computes four consecutive exps of row
// r a chunk (16 LPR bytes a row), e_j = expf(s_j - max) goes back over the
// scores and into the wave's LDS, and lane r of the first ROWS adds row r's
// chunk in position order.  1 / sum is left in the row's first tile maximum
// for batt_av, which forms a_j = e_j * (1 / sum) as it stages them.  Bound by
// the exps (about 240 clocks per wave and element); the chains cost CP adds
// per chunk of 256 exps, 16 with ROWS = 16.  ROWS = 4 where 16 would leave
// most SIMDs without a wave.  (A workgroup per row, attn_sm, took 133 us per
// layer for 1024 tokens of 32 heads.)
template <int ROWS>
__global__ __launch_bounds__(256) void batt_sm(float *__restrict__ att, size_t att_stride,
                                               float *__restrict__ tmax, int n_tiles, int n_head,
                                               const uint32_t *__restrict__ pos, int t_base,
                                               int n_ctx, int M)
{
    constexpr int LPR = 64 / ROWS, CP = 4 * LPR, RS = LPR + 1;
    __shared__ f4v E[4][ROWS * RS];
    __shared__ uint64_t tab[32];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (tid < 32) tab[tid] = fox_exp2_tab[tid];
    __syncthreads();
    // (row groups from the last, longest one on)
    const int h = blockIdx.x, g0 = ((M + ROWS - 1) / ROWS - 1 - ((int)blockIdx.y * 4 + wave)) * ROWS;
    if (g0 < 0) return;                                    // (uniform over the wave)
    const size_t pz = (size_t)pos[0] + (size_t)t_base;
    auto upto_of = [&](int t) { return (int)min(pz + (size_t)min(t, M - 1) + 1, (size_t)n_ctx); };
    const int r = lane / LPR, c = lane % LPR, t = min(g0 + r, M - 1);
    const int upto = upto_of(t);
    float *row = att + ((size_t)t * n_head + h) * att_stride;
    float *tm = tmax + ((size_t)t * n_head + h) * n_tiles;
    // src/ops.c:26-30: a NaN first score stays the maximum
    float m = -INFINITY;
    for (int i = c; i < (upto + BQ_POS - 1) / BQ_POS; i += LPR) {
        const float v = tm[i];
        m = v > m ? v : m;
    }
    auto mx = [](float a, float b) { return b > a ? b : a; };
    m = mx(m, dpp_t<0xB1, 0xF>(m, m));
    m = mx(m, dpp_t<0x4E, 0xF>(m, m));
    if (LPR == 16) {
        m = mx(m, dpp_t<0x141, 0xF>(m, m));
        m = mx(m, dpp_t<0x140, 0xF>(m, m));
    }
    const float s0 = row[0];
    if (s0 != s0) m = s0;
    const int nch = (upto_of(g0 + ROWS - 1) + CP - 1) / CP, full = upto_of(g0) / CP;
    const int up_ch = upto_of(g0 + (lane & (ROWS - 1)));   // of the row this lane sums
    auto load = [&](int k) { return ((const f4v *)row)[min(k * LPR + c, (upto - 1) >> 2)]; };
    f4v *Ew = E[wave];
    f4v nxt = load(0);
    float sum = 0.0f;
    for (int k = 0; k < nch; k++) {
        const f4v s = nxt;
        nxt = load(min(k + 1, nch - 1));
        const int j = k * CP + 4 * c;
        f4v e;
#pragma unroll
        for (int i = 0; i < 4; i++) e[i] = fox_expf_t(s[i] - m, tab);
        Ew[r * RS + c] = e;
        if (j < upto && g0 + r < M) ((f4v *)row)[k * LPR + c] = e;
        __builtin_amdgcn_wave_barrier();                   // (a wave's LDS accesses run in order)
        if (lane < ROWS) {
            const f4v *er = Ew + lane * RS;
            if (k < full) {                                // (uniform)
#pragma unroll
                for (int q = 0; q < LPR; q++) {
                    const f4v x = er[q];
#pragma unroll
                    for (int i = 0; i < 4; i++) sum = sum + x[i];
                }
            } else {
                for (int q = 0; q < LPR; q++) {
                    const f4v x = er[q];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float y = sum + x[i];
                        sum = k * CP + 4 * q + i < up_ch ? y : sum;
                    }
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    // src/ops.c:35-38: a_j = e_j * (1 / sum) when the sum is positive, else e_j
    if (lane < ROWS && g0 + lane < M)
        tmax[((size_t)(g0 + lane) * n_head + h) * n_tiles] = sum > 0.0f ? fox_div(1.0f, sum) : 1.0f;
}

// Values of one query head for CW columns and 256 * 4 / CW * TI tokens: thread
// (cx, ty) = (tid % (CW / 4), tid / (CW / 4)) owns columns cx + CW / 4 * k and
// tokens ty * TI + i.  Position quads are staged BV_Q at a time (the cache
// keeps a column's four positions side by side); a quad costs TI + 4 LDS
// reads and 32 TI vector instructions.  Positions at or past a token's end
// are not added (quads that reach one take the masked form).  att holds e_j,
// inv each (token, head)'s factor, inv_stride apart.
#define BV_Q 8
template <int CW, int TI>
__global__ __launch_bounds__(256) void batt_av(const float *__restrict__ att, size_t att_stride,
                                               const float *__restrict__ inv, int inv_stride,
                                               const float *__restrict__ vc, int n_head,
                                               int n_head_kv, int hd,
                                               const uint32_t *__restrict__ pos, int t_base,
                                               int n_ctx, float *__restrict__ out,
                                               size_t out_stride, int M)
{
    constexpr int NX = CW / 4, NY = 256 / NX, TT = NY * TI;
    constexpr int AS = BV_Q + 1;                           // (a quad of padding per token)
    constexpr int NV = CW * BV_Q / 256, NA = (TT * BV_Q + 255) / 256;
    __shared__ f4v Vs[2][BV_Q * CW], A[2][TT * AS];
    const int tid = threadIdx.x, cx = tid % NX, ty = tid / NX;
    const int h = blockIdx.x, c0 = (int)blockIdx.z * CW;
    // (token groups from the last, longest one on)
    const int t0 = (int)(gridDim.y - 1 - blockIdx.y) * TT;
    const int kvh = h / (n_head / n_head_kv), kvd = n_head_kv * hd;
    const size_t pz = (size_t)pos[0] + (size_t)t_base;
    auto upto_of = [&](int t) { return (int)min(pz + (size_t)t + 1, (size_t)n_ctx); };
    const int t_last = min(t0 + TT, M) - 1;
    const int nq_max = (upto_of(t_last) + 3) >> 2;         // quads of the longest token
    const int nq_full = upto_of(t0) >> 2;                  // quads whole for every token
    f4v vr[NV], ar[NA];
    float ai[NA];
#pragma unroll
    for (int u = 0; u < NA; u++) {
        const int idx = min(tid + 256 * u, TT * BV_Q - 1), t = min(t0 + idx / BV_Q, t_last);
        ai[u] = inv[((size_t)t * n_head + h) * inv_stride];
    }
    auto fetch = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < NV; u++) {
            const int idx = tid + 256 * u, qq = idx / CW, c = idx - qq * CW;
            vr[u] = ((const f4v *)vc)[(size_t)min(b * BV_Q + qq, nq_max - 1) * kvd + (size_t)kvh * hd +
                                      min(c0 + c, hd - 1)];
        }
#pragma unroll
        for (int u = 0; u < NA; u++) {
            const int idx = min(tid + 256 * u, TT * BV_Q - 1), t = min(t0 + idx / BV_Q, t_last);
            ar[u] = ((const f4v *)(att + ((size_t)t * n_head + h) * att_stride))
                [min(b * BV_Q + idx % BV_Q, nq_max - 1)];
        }
    };
    auto stash = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < NV; u++) Vs[buf][tid + 256 * u] = vr[u];
#pragma unroll
        for (int u = 0; u < NA; u++) {
            const int idx = tid + 256 * u;
            if (idx < TT * BV_Q) A[buf][idx / BV_Q * AS + idx % BV_Q] = ar[u] * ai[u];
        }
    };
    float acc[TI][4];
    int upto[TI];
#pragma unroll
    for (int i = 0; i < TI; i++) {
        upto[i] = upto_of(min(t0 + ty * TI + i, t_last));
#pragma unroll
        for (int k = 0; k < 4; k++) acc[i][k] = 0.0f;
    }
    const int nblk = (nq_max + BV_Q - 1) / BV_Q;
    fetch(0);
    stash(0);
    __syncthreads();
    for (int b = 0; b < nblk; b++) {
        const int buf = b & 1;
        fetch(min(b + 1, nblk - 1));
        if ((b + 1) * BV_Q <= nq_full) {                   // (uniform)
#pragma unroll
            for (int qq = 0; qq < BV_Q; qq++) {
                f4v v[4];
#pragma unroll
                for (int k = 0; k < 4; k++) v[k] = Vs[buf][qq * CW + cx + NX * k];
#pragma unroll
                for (int i = 0; i < TI; i++) {
                    const f4v a = A[buf][(ty * TI + i) * AS + qq];
#pragma unroll
                    for (int e = 0; e < 4; e++)
#pragma unroll
                        for (int k = 0; k < 4; k++) acc[i][k] = acc[i][k] + a[e] * v[k][e];
                }
            }
        } else {
            for (int qq = 0; qq < BV_Q; qq++) {
                f4v v[4];
#pragma unroll
                for (int k = 0; k < 4; k++) v[k] = Vs[buf][qq * CW + cx + NX * k];
#pragma unroll
                for (int i = 0; i < TI; i++) {
                    const f4v a = A[buf][(ty * TI + i) * AS + qq];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const bool in = (b * BV_Q + qq) * 4 + e < upto[i];
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            const float s = acc[i][k] + a[e] * v[k][e];
                            acc[i][k] = in ? s : acc[i][k];
                        }
                    }
                }
            }
        }
        stash(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < TI; i++) {
        const int t = t0 + ty * TI + i;
        if (t >= M) continue;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int c = c0 + cx + NX * k;
            if (c < hd) out[(size_t)t * out_stride + (size_t)h * hd + c] = acc[i][k];
        }
    }
}

// scores of one run of tokens at most this many bytes, or those of 64 tokens
// where these are more (64 heads over 32768 positions: 520 MB)
#define BATT_BYTES ((size_t)256 << 20)

extern "C" fox_gpu_status fox_gpu_batch_attention(fox_gpu_ctx *ctx, float *out, size_t out_stride,
                                                  const float *q, size_t q_stride,
                                                  const float *k_cache, const float *v_cache,
                                                  size_t n_head, size_t n_head_kv,
                                                  size_t head_dim, size_t M, const uint32_t *pos,
                                                  size_t n_ctx)
{
    if (!ctx || !out || !q || !k_cache || !v_cache || !pos || n_head == 0 || n_head_kv == 0 ||
        head_dim == 0 || M == 0 || n_ctx == 0)
        return fox_fail(FOX_GPU_ERR_ARG, "attention: bad argument");
    if (n_head % n_head_kv)
        return fox_fail(FOX_GPU_ERR_ARG, "attention: %zu heads over %zu kv heads", n_head, n_head_kv);
    if (n_head / n_head_kv > 8 || head_dim > 256 || head_dim % 4 || n_head > 65535)
        return fox_fail(FOX_GPU_ERR_UNSUPPORTED, "attention: at most 8 query heads per kv head, "
                        "head_dim a multiple of 4 up to 256");
    if (M > FOX_GPU_BATCH_TOKENS) return fox_fail(FOX_GPU_ERR_ARG, "attention: too many tokens");
    if (((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) % 16 || q_stride % 4)
        return fox_fail(FOX_GPU_ERR_ARG, "attention: q and the caches must be 16-byte aligned and "
                        "the q stride a multiple of 4");
    // (the decode kernels' limit, which keep a head's weights in LDS: a context
    // that takes a prompt here goes on there)
    if (n_ctx > 32768)
        return fox_fail(FOX_GPU_ERR_UNSUPPORTED, "attention: %zu positions; exact mode takes at "
                        "most 32768", n_ctx);
    const size_t att_stride = (n_ctx + 3) & ~(size_t)3;
    const int n_tiles = (int)((n_ctx + BQ_POS - 1) / BQ_POS);
    const size_t per_tok = n_head * (att_stride + (size_t)n_tiles) * sizeof(float);
    // tokens of one run: whole groups of 64
    size_t run = BATT_BYTES / per_tok / 64 * 64;
    if (run < 64) run = 64;
    if (run > M) run = M;
    fox_gpu_status st = fox_ws_reserve(ctx, run * per_tok);
    if (st) return st;
    float *att = (float *)ctx->ws, *tmax = att + run * n_head * att_stride;
    const int inh = (int)n_head, ikv = (int)n_head_kv, ihd = (int)head_dim, ictx = (int)n_ctx;
    for (size_t tb = 0; tb < M; tb += run) {
        const int m = (int)(M - tb < run ? M - tb : run), itb = (int)tb;
        const float *qr = q + tb * q_stride;
        float *orow = out + tb * out_stride;
        {
            // tokens per thread: four, or two where the tiles are then too few
            const size_t tiles4 = (size_t)((m + 63) / 64) * n_head * (size_t)n_tiles;
            const int ti = m > 32 && tiles4 >= 2 * (size_t)ctx->n_cu ? 4 : 2;
            const void *k = ti == 4 ? (const void *)batt_qk<4> : (const void *)batt_qk<2>;
            void *args[] = {(void *)&qr, (void *)&q_stride, (void *)&k_cache, (void *)&inh,
                            (void *)&ikv, (void *)&ihd, (void *)&pos, (void *)&itb, (void *)&ictx,
                            (void *)&att_stride, (void *)&att, (void *)&tmax, (void *)&n_tiles,
                            (void *)&m};
            hipError_t e = hipLaunchKernel(k, dim3((unsigned)n_tiles, (unsigned)n_head,
                                                   (unsigned)((m + 16 * ti - 1) / (16 * ti))),
                                           dim3(256), args, 0, ctx->stream);
            if (e != hipSuccess) return fox_hip_fail(e, "attention scores");
            FOX_LAUNCHED("attention scores");
        }
        {
            const bool r16 = (size_t)((m + 15) / 16) * n_head >= 4 * (size_t)ctx->n_cu;
            const int rows = r16 ? 16 : 4;
            const void *k = r16 ? (const void *)batt_sm<16> : (const void *)batt_sm<4>;
            void *args[] = {(void *)&att, (void *)&att_stride, (void *)&tmax, (void *)&n_tiles,
                            (void *)&inh, (void *)&pos, (void *)&itb, (void *)&ictx, (void *)&m};
            hipError_t e = hipLaunchKernel(k, dim3((unsigned)n_head, (unsigned)((m + 4 * rows - 1) / (4 * rows))),
                                           dim3(256), args, 0, ctx->stream);
            if (e != hipSuccess) return fox_hip_fail(e, "attention softmax");
            FOX_LAUNCHED("attention softmax");
        }
        {
            // tokens per thread: as many as leave every compute unit two
            // workgroups
            const int cw = head_dim <= 64 ? 64 : 128, ny = 1024 / cw;
            const int ncg = (int)((head_dim + cw - 1) / cw);
            int ti = 4;
            while (ti > 1 && (size_t)((m + ny * ti - 1) / (ny * ti)) * n_head * ncg < 2 * (size_t)ctx->n_cu)
                ti /= 2;
#define FOX_AV(w) (ti == 4 ? (const void *)batt_av<w, 4> : ti == 2 ? (const void *)batt_av<w, 2> \
                                                                 : (const void *)batt_av<w, 1>)
            const void *k = cw == 64 ? FOX_AV(64) : FOX_AV(128);
#undef FOX_AV
            void *args[] = {(void *)&att, (void *)&att_stride, (void *)&tmax, (void *)&n_tiles, (void *)&v_cache,
                            (void *)&inh,
                            (void *)&ikv, (void *)&ihd, (void *)&pos, (void *)&itb, (void *)&ictx,
                            (void *)&orow, (void *)&out_stride, (void *)&m};
            hipError_t e = hipLaunchKernel(k, dim3((unsigned)n_head, (unsigned)((m + ny * ti - 1) / (ny * ti)),
                                                   (unsigned)ncg),
                                           dim3(256), args, 0, ctx->stream);
            if (e != hipSuccess) return fox_hip_fail(e, "attention values");
            FOX_LAUNCHED("attention values");
        }
    }
    return FOX_GPU_OK;
}
