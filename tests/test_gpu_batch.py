"""Batched passes (fox_gpu_batch_*: up to 1024 tokens) bit-identical to the
oracle's single-token steps and to the decode kernels in passes of eight, at
the edges of their tiles: 16 tokens and rows, 64-position score tiles, groups
of four tiles, ragged last blocks."""
import numpy as np
import pytest

import rustfox_amd as rf
from rustfox_amd import synth
from test_gpu_gemv import TYPES, bits, nonfinite_rows, oracle_gemv, same_or_both_nan, weights

pytestmark = pytest.mark.gpu

EPS = 1e-5


@pytest.mark.parametrize("tname,K,Ns,M", [
    ("TQ1_0", 256, [16], 9), ("TQ2_0", 1280, [40, 23], 17), ("TQ2_0", 2560, [130], 64),
    ("TQ1_0", 768, [80, 16, 48], 33), ("TQ2_0", 512, [4100], 100), ("TQ2_0", 512, [9000], 200),
    ("Q4_K", 256, [16], 9), ("Q4_K", 768, [33, 50], 20), ("Q4_K", 1024, [70], 65),
    ("TQ2_0", 2304, [5000], 24), ("Q4_K", 2304, [9000], 150), ("Q6_K", 1024, [9000], 130),
    ("TQ1_0", 4352, [40], 16), ("Q4_K", 1280, [30], 16), ("Q6_K", 2304, [30], 17),
    ("Q6_K", 256, [16], 9), ("Q6_K", 768, [29], 31), ("Q6_K", 1280, [64, 100], 48),
    ("F16", 288, [50], 19), ("F32", 64, [9], 9),
])
def test_batch_gemv_bit_exact(gpu, oracle, tname, K, Ns, M):
    rng = np.random.default_rng(K + M)
    t = TYPES[tname]
    Ws = [weights(rng, t, N, K) for N in Ns]
    x = rng.standard_normal((M, K)).astype(np.float32)
    dx = gpu.array(x)
    ts = [gpu.tensor(t, K, N, w) for N, w in zip(Ns, Ws)]
    init = [rng.standard_normal((M, N)).astype(np.float32) for N in Ns]
    outs = [gpu.array(i) for i in init]
    gpu.batch_gemv(ts, dx, M, outs, flags=rf.GEMV_ACCUMULATE)
    for N, W, o, i in zip(Ns, Ws, outs, init):
        assert np.array_equal(bits(o.numpy()), bits(i + oracle_gemv(oracle, t, x, W, N, K))), N
    if K % 256 == 0:
        nw = rng.uniform(0.5, 1.5, K).astype(np.float32)
        outs = [gpu.empty(M * N, np.float32) for N in Ns]
        gpu.batch_gemv(ts, dx, M, outs, gpu.array(nw), EPS)
        xn = np.stack([oracle.rmsnorm(r, nw, EPS) for r in x])
        for N, W, o in zip(Ns, Ws, outs):
            want = oracle_gemv(oracle, t, xn, W, N, K)
            assert np.array_equal(bits(o.numpy()), bits(want).reshape(-1)), N


@pytest.mark.parametrize("tname", ["TQ2_0", "Q4_K", "Q6_K"])
@pytest.mark.parametrize("K", [2560, 6400, 8448, 12544, 20480, 32768])
def test_batch_preparation_of_wide_rows(gpu, oracle, tname, K):
    """One width of each of the preparation kernels' input registers above the
    first, up to the widest they take, with the norm and without."""
    rng = np.random.default_rng(K)
    t, N, M = TYPES[tname], 20, 9
    W = weights(rng, t, N, K)
    x = rng.standard_normal((M, K)).astype(np.float32)
    nw = rng.uniform(0.5, 1.5, K).astype(np.float32)
    w, dx, out = gpu.tensor(t, K, N, W), gpu.array(x), gpu.empty(M * N, np.float32)
    gpu.batch_gemv([w], dx, M, [out])
    assert np.array_equal(bits(out.numpy()), bits(oracle_gemv(oracle, t, x, W, N, K)).reshape(-1))
    gpu.batch_gemv([w], dx, M, [out], gpu.array(nw), EPS)
    xn = np.stack([oracle.rmsnorm(r, nw, EPS) for r in x])
    assert np.array_equal(bits(out.numpy()), bits(oracle_gemv(oracle, t, xn, W, N, K)).reshape(-1))


@pytest.mark.parametrize("tname", ["Q4_K", "Q6_K"])
@pytest.mark.parametrize("K,N,M", [(256, 16, 2), (1024, 40, 3), (2304, 8300, 8), (5376, 100, 5),
                                   (14336, 33, 7)])
def test_few_tokens_kquants_bit_exact(gpu, oracle, tname, K, N, M):
    """Two to eight tokens: fewer, as many and more blocks than a workgroup's
    four or eight waves, through fox_gpu_gemv and the normed batched call."""
    rng = np.random.default_rng(K + M)
    t = TYPES[tname]
    W = np.concatenate([weights(rng, t, min(N, 64), K)] * -(-N // 64))[:N * synth.row_bytes(t, K)]
    x = rng.standard_normal((M, K)).astype(np.float32)
    dw, dx = gpu.tensor(t, K, N, W), gpu.array(x)
    init = rng.standard_normal((M, N)).astype(np.float32)
    out = gpu.array(init)
    gpu.gemv(dw, dx, M, out, flags=rf.GEMV_ACCUMULATE)
    assert np.array_equal(bits(out.numpy()), bits(init + oracle_gemv(oracle, t, x, W, N, K)))
    nw = rng.uniform(0.5, 1.5, K).astype(np.float32)
    gpu.batch_gemv([dw], dx, M, [out], gpu.array(nw), EPS)
    xn = np.stack([oracle.rmsnorm(r, nw, EPS) for r in x])
    assert np.array_equal(bits(out.numpy()), bits(oracle_gemv(oracle, t, xn, W, N, K)))


@pytest.mark.parametrize("tname,K,ff,M", [("Q4_K", 1280, 9000, 8), ("Q6_K", 512, 50, 2), ("Q6_K", 256, 8300, 3), ("Q6_K", 768, 40, 30),
                                          ("Q6_K", 512, 21000, 12), ("TQ2_0", 1280, 8100, 12),
                                          ("TQ1_0", 512, 96, 9), ("TQ2_0", 2560, 700, 50),
                                          ("TQ2_0", 512, 8200, 65), ("Q4_K", 768, 40, 33)])
def test_batch_gate_up_bit_exact(gpu, oracle, tname, K, ff, M):
    rng = np.random.default_rng(K + ff + M)
    t = TYPES[tname]
    Wg, Wu = weights(rng, t, ff, K), weights(rng, t, ff, K)
    x = rng.standard_normal((M, K)).astype(np.float32)
    nw = rng.uniform(0.5, 1.5, K).astype(np.float32)
    h = gpu.empty(M * ff, np.float32)
    args = (gpu.tensor(t, K, ff, Wg), gpu.tensor(t, K, ff, Wu), gpu.array(x), M, gpu.array(nw), EPS, h)
    if tname == "Q6_K" and ff > 20000:
        # (two such tiles do not fit a wave's registers: the separate steps)
        with pytest.raises(rf.FoxError) as e:
            gpu.batch_gate_up_silu(*args)
        assert e.value.status == 5
        return
    gpu.batch_gate_up_silu(*args)
    got = h.numpy().reshape(M, ff)
    for r in range(M):
        xb = oracle.rmsnorm(x[r], nw, EPS)
        want = oracle.silu_mul(oracle.gemv(t, xb, Wg, ff, K), oracle.gemv(t, xb, Wu, ff, K))
        assert np.array_equal(bits(got[r]), bits(want)), f"token {r}"


@pytest.mark.parametrize("tname", ["TQ2_0", "Q4_K", "Q6_K"])
def test_batch_nonfinite_follows_the_reference(gpu, oracle, tname):
    """Rows with NaN, inf and tiny values, and a weight block whose scale is
    infinite or NaN (the conversion in place of the fused multiply-add), in
    the kernels of few row tiles."""
    rng = np.random.default_rng(5)
    K, N, t = 512, 20, TYPES[tname]
    W = weights(rng, t, N, K)
    rows = [np.asarray(r, np.float32) for r in nonfinite_rows(rng, K)]
    rows += [rng.standard_normal(K).astype(np.float32) for _ in range(9)]
    x = np.stack(rows)
    few = np.stack(rows[:7] + rows[-1:])
    for special in (None, np.inf, np.nan):
        w = W.copy()
        if special is not None:
            b = w.reshape(N * K // 256, -1)
            at = {"TQ2_0": 64, "Q4_K": 0, "Q6_K": 208}[tname]
            b[3, at:at + 2] = np.array([special], np.float16).view(np.uint8)
        out = gpu.empty(len(rows) * N, np.float32)
        gpu.batch_gemv([gpu.tensor(t, K, N, w)], gpu.array(x), len(rows), [out])
        got = out.numpy().reshape(len(rows), N)
        for r, xr in enumerate(rows):
            assert same_or_both_nan(got[r], oracle.gemv(t, xr, w, N, K)), (special, r)
        gpu.gemv(gpu.tensor(t, K, N, w), gpu.array(few), 8, out)
        got = out.numpy()[:8 * N].reshape(8, N)
        for r, xr in enumerate(few):
            assert same_or_both_nan(got[r], oracle.gemv(t, xr, w, N, K)), (special, r)


# shapes that leave split_gemm for batch_gemm on 256 compute units, by the row
# tiles per wave R and token tiles C of the kernel they take
@pytest.mark.parametrize("tname,K,Ns,M", [
    ("TQ2_0", 512, [8300], 9), ("TQ2_0", 1280, [9000], 24), ("TQ1_0", 768, [8000, 300], 32),   # R 1, C 1, 2, 2
    ("TQ2_0", 768, [4100], 65),                                                                # R 1, C 3
    ("TQ2_0", 256, [66000], 9), ("TQ2_0", 768, [4096], 1024), ("TQ2_0", 256, [66000], 23),     # R 2, C 1, 4, 2
    ("TQ2_0", 256, [33000], 77),                                                               # R 2, C 3
    ("TQ1_0", 512, [8192], 1024), ("TQ2_0", 256, [132000], 20), ("TQ2_0", 256, [70000], 77),   # R 4, C 4, 2, 3
    ("TQ2_0", 256, [132000], 9),                                                               # R 4, C 1
    ("Q4_K", 256, [12400], 9), ("Q4_K", 768, [13000], 24), ("Q4_K", 768, [9000], 65),          # C 1, 2, 3
    ("Q4_K", 512, [6100, 90], 128),                                                            # C 4
    ("Q6_K", 256, [20500], 9), ("Q6_K", 768, [20500], 24), ("Q6_K", 512, [10300], 77),         # C 1, 2, 3
    ("Q6_K", 512, [10300], 128),                                                               # C 4
])
def test_batch_gemm_equals_passes_of_eight(gpu, tname, K, Ns, M):
    rng = np.random.default_rng(K + M)
    t = TYPES[tname]
    ts = []
    for N in Ns:
        rows = weights(rng, t, 512, K).reshape(512, -1)
        ts.append(gpu.tensor(t, K, N, rows[rng.integers(0, 512, N)]))
    x = rng.standard_normal((M, K)).astype(np.float32)
    outs = [gpu.empty(M * N, np.float32) for N in Ns]
    gpu.batch_gemv(ts, gpu.array(x), M, outs)
    for w, N, o in zip(ts, Ns, outs):
        got = o.numpy().reshape(M, N)
        for m in range(0, M, 8):
            p = gpu.empty(min(8, M - m) * N, np.float32)
            gpu.gemv(w, gpu.array(x[m:m + 8]), min(8, M - m), p)
            assert np.array_equal(bits(got[m:m + 8]).reshape(-1), bits(p.numpy())), (N, m)


@pytest.mark.parametrize("tname,K,ff,M", [
    ("TQ2_0", 512, 8300, 9), ("TQ2_0", 1280, 8300, 24), ("TQ2_0", 768, 4200, 77),              # R 2, C 1, 2, 3
    ("TQ2_0", 512, 8300, 64),                                                                  # R 2, C 4
    ("TQ1_0", 256, 4096, 1024), ("TQ2_0", 256, 66000, 12), ("TQ2_0", 256, 66000, 41),          # R 4, C 4, 1, 3
    ("TQ2_0", 256, 66000, 20),                                                                 # R 4, C 2
    ("Q4_K", 256, 12400, 9), ("Q4_K", 768, 13000, 20), ("Q4_K", 768, 14336, 77),               # C 1, 2, 3
    ("Q4_K", 512, 6200, 100),                                                                  # C 4
])
def test_batch_gemm_gate_up_equals_passes_of_eight(gpu, tname, K, ff, M):
    rng = np.random.default_rng(K + ff + M)
    t = TYPES[tname]
    rows = weights(rng, t, 512, K).reshape(512, -1)
    wg, wu = (gpu.tensor(t, K, ff, rows[rng.integers(0, 512, ff)]) for _ in range(2))
    x = rng.standard_normal((M, K)).astype(np.float32)
    nw = gpu.array(rng.uniform(0.5, 1.5, K).astype(np.float32))
    h = gpu.empty(M * ff, np.float32)
    gpu.batch_gate_up_silu(wg, wu, gpu.array(x), M, nw, EPS, h)
    got = h.numpy().reshape(M, ff)
    for m in range(0, M, 8):
        n = min(8, M - m)
        p = gpu.empty(n * ff, np.float32)
        eight = gpu.gate_up_silu if t in (34, 35) or n == 1 else gpu.batch_gate_up_silu
        eight(wg, wu, gpu.array(x[m:m + 8]), n, nw, EPS, p)
        assert same_or_both_nan(got[m:m + 8].reshape(-1), p.numpy()), m


@pytest.mark.parametrize("tname,N,M", [("TQ2_0", 4100, 70), ("Q4_K", 9000, 70), ("Q6_K", 10300, 70),
                                       ("TQ2_0", 100, 70), ("Q4_K", 100, 70), ("Q4_K", 100, 7)])
def test_batch_nonfinite_scales_in_every_kernel(gpu, oracle, tname, N, M):
    """Weight blocks whose scale (Q4_K: or whose minimum's scale) is infinite or
    NaN among finite ones, and input rows with NaN, inf and tiny values, in
    batch_gemm (many rows), split_gemm and few_gemm."""
    rng = np.random.default_rng(N)
    K, base, t = 768, 20, TYPES[tname]
    rows = weights(rng, t, base, K).reshape(base, -1)
    fields = {"TQ2_0": [64], "Q4_K": [0, 2], "Q6_K": [208]}[tname]
    blocks = rows.reshape(base * K // 256, -1)
    for i, (at, v) in enumerate([(f, v) for f in fields for v in (np.inf, -np.inf, np.nan)]):
        blocks[5 * i + 3, at:at + 2] = np.array([v], np.float16).view(np.uint8)
    pick = rng.integers(0, base, N)
    x = np.concatenate([nonfinite_rows(rng, K)[:M - 1],
                        rng.standard_normal((M, K)).astype(np.float32)])[:M].astype(np.float32)
    out = gpu.empty(M * N, np.float32)
    w = gpu.tensor(t, K, N, rows[pick])
    if M <= 8:
        gpu.gemv(w, gpu.array(x), M, out)
    else:
        gpu.batch_gemv([w], gpu.array(x), M, [out])
    got = out.numpy().reshape(M, N)
    for r in range(M):
        want = oracle.gemv(t, x[r], rows.reshape(-1), base, K)
        assert same_or_both_nan(got[r], np.asarray(want)[pick]), r


@pytest.mark.parametrize("n_head,n_kv,hd,pos,M", [
    (4, 2, 128, 0, 9), (8, 1, 64, 0, 70), (6, 6, 48, 61, 67), (5, 1, 128, 700, 33),
    (4, 4, 256, 130, 20), (32, 8, 128, 0, 300), (2, 2, 20, 63, 65),
    # a wave per 16 tokens in the softmax, two and four tokens per value thread
    (32, 8, 128, 3, 512), (32, 4, 64, 90, 512), (32, 16, 64, 0, 1024),
])
def test_batch_attention_equals_the_decode_kernels(gpu, n_head, n_kv, hd, pos, M):
    rng = np.random.default_rng(n_head + hd + M)
    n_ctx, kvd = pos + M, n_kv * hd
    K, V = (rng.standard_normal((n_ctx, kvd)).astype(np.float32) for _ in range(2))
    # (a later token's row must not reach an earlier token's sums)
    V[-1, 0], K[-1, 0] = np.inf, np.nan
    kc = gpu.empty(n_ctx * kvd, np.float32)
    vc = gpu.empty((n_ctx + 3) // 4 * 4 * kvd, np.float32)
    gpu.kv_write(kc, vc, kvd, n_ctx, 0, gpu.array(K), gpu.array(V), n_ctx)
    q = rng.standard_normal((M, n_head * hd)).astype(np.float32)
    out = gpu.empty(M * n_head * hd, np.float32)
    gpu.batch_attention(out, gpu.array(q), kc, vc, n_head, n_kv, hd, M,
                        gpu.array(np.array([pos], np.uint32)), n_ctx)
    got = out.numpy().reshape(M, -1)
    for t in range(0, M, 8):
        m = min(8, M - t)
        o = gpu.empty(m * n_head * hd, np.float32)
        gpu.attention(o, gpu.array(q[t:t + m]), kc, vc, n_head, n_kv, hd, m,
                      gpu.array(np.array([pos + t], np.uint32)), n_ctx, rf.ATTN_EXACT)
        assert same_or_both_nan(got[t:t + m].reshape(-1), o.numpy()), f"tokens {t}.."


@pytest.mark.parametrize("name,over", [
    ("tiny-288", {}), ("tiny-512", {}),
    ("8b", dict(n_layer=1, n_vocab=512, n_embd=512, n_ff=768, n_head=8, n_head_kv=2, head_dim=64)),
])
def test_prompt_equals_passes_of_eight(tmp_path, name, over):
    """Prompts through batched passes (n_batch 32) and passes of eight: the
    same logits, last and all, on an empty and a filled cache, in both
    attention modes; an overrun leaves the position where passes of eight
    leave it."""
    s = synth.spec(name, n_ctx=160, **over)
    path = str(tmp_path / "m.gguf")
    synth.write_gguf(path, s)
    ids = synth.prompt_ids(150, s.n_vocab)
    with rf.Model(path) as m:
        a, b = m.context(160, n_batch=32), m.context(160, n_batch=8)
        for exact in (True, False):
            for c in (a, b):
                c.set_attention(exact)
                c.reset()
            for n0, n1 in ((0, 9), (9, 82), (82, 91), (91, 150)):
                x, y = a.eval(ids[n0:n1]).copy(), b.eval(ids[n0:n1])
                assert np.array_equal(bits(x), bits(y)), (exact, n0)
        for c in (a, b):
            c.set_attention(True)
            c.reset()
        assert np.array_equal(bits(a.eval_all(ids[:75])), bits(b.eval_all(ids[:75])))
        for c in (a, b):
            with pytest.raises(rf.FoxError):
                c.eval(np.concatenate([ids, ids])[:100])
            assert c.position == 75 + 80
        a.close()
        b.close()


@pytest.mark.parametrize("n_head,n_kv,hd,n_ctx,pos,M", [
    (32, 8, 128, 4196, 100, 1000), (12, 6, 96, 8300, 7000, 900), (32, 8, 64, 4200, 3176, 1024),
])
def test_batch_attention_in_several_runs(gpu, n_head, n_kv, hd, n_ctx, pos, M):
    """More tokens than one run's scores hold (448 and 640 here, the last run
    ragged): as the decode kernels give them."""
    rng = np.random.default_rng(M)
    kvd = n_kv * hd
    K, V = (rng.standard_normal((n_ctx, kvd)).astype(np.float32) for _ in range(2))
    kc = gpu.empty(n_ctx * kvd, np.float32)
    vc = gpu.empty((n_ctx + 3) // 4 * 4 * kvd, np.float32)
    gpu.kv_write(kc, vc, kvd, n_ctx, 0, gpu.array(K), gpu.array(V), n_ctx)
    q = rng.standard_normal((M, n_head * hd)).astype(np.float32)
    out = gpu.empty(M * n_head * hd, np.float32)
    gpu.batch_attention(out, gpu.array(q), kc, vc, n_head, n_kv, hd, M,
                        gpu.array(np.array([pos], np.uint32)), n_ctx)
    got = out.numpy().reshape(M, -1)
    for t in range(0, M, 8):
        m = min(8, M - t)
        o = gpu.empty(m * n_head * hd, np.float32)
        gpu.attention(o, gpu.array(q[t:t + m]), kc, vc, n_head, n_kv, hd, m,
                      gpu.array(np.array([pos + t], np.uint32)), n_ctx, rf.ATTN_EXACT)
        assert np.array_equal(bits(got[t:t + m]).reshape(-1), bits(o.numpy())), f"tokens {t}.."


@pytest.mark.parametrize("n_head,n_kv,hd,pos,M", [
    (40, 8, 128, 250, 2), (80, 16, 128, 61, 4), (80, 16, 128, 127, 3), (40, 8, 100, 511, 7),
    (32, 16, 128, 1020, 8), (64, 32, 64, 254, 5), (40, 8, 72, 0, 2),
])
def test_many_heads_equal_single_tokens(gpu, n_head, n_kv, hd, pos, M):
    """Two to eight tokens of many heads (attn_avt: more value workgroups than
    compute units): each token as a call of its own gives it."""
    rng = np.random.default_rng(n_head + hd + M)
    n_ctx, kvd = pos + M, n_kv * hd
    K, V = (rng.standard_normal((n_ctx, kvd)).astype(np.float32) for _ in range(2))
    V[-1, 0], V[-1, -1] = np.inf, np.nan           # (must not reach the tokens before)
    kc = gpu.empty(n_ctx * kvd, np.float32)
    vc = gpu.empty((n_ctx + 3) // 4 * 4 * kvd, np.float32)
    gpu.kv_write(kc, vc, kvd, n_ctx, 0, gpu.array(K), gpu.array(V), n_ctx)
    q = rng.standard_normal((M, n_head * hd)).astype(np.float32)
    out = gpu.empty(M * n_head * hd, np.float32)
    gpu.attention(out, gpu.array(q), kc, vc, n_head, n_kv, hd, M,
                  gpu.array(np.array([pos], np.uint32)), n_ctx, rf.ATTN_EXACT)
    got = out.numpy().reshape(M, -1)
    for t in range(M):
        o = gpu.empty(n_head * hd, np.float32)
        gpu.attention(o, gpu.array(q[t]), kc, vc, n_head, n_kv, hd, 1,
                      gpu.array(np.array([pos + t], np.uint32)), n_ctx, rf.ATTN_EXACT)
        assert same_or_both_nan(got[t], o.numpy()), f"token {t}"


def test_weights_past_32_bit_offsets(gpu):
    """Score rows of 5120 heads over a 32768-position cache: eight tokens' rows
    are more than 4 GB apart."""
    rng = np.random.default_rng(1)
    n_head, n_kv, hd, pos, M, n_ctx = 5120, 640, 4, 70, 8, 32768
    n, kvd = pos + M, n_kv * hd
    K, V = (rng.standard_normal((n, kvd)).astype(np.float32) for _ in range(2))
    kc, vc = (gpu.empty(n_ctx * kvd, np.float32) for _ in range(2))
    gpu.kv_write(kc, vc, kvd, n_ctx, 0, gpu.array(K), gpu.array(V), n)
    q = rng.standard_normal((M, n_head * hd)).astype(np.float32)
    out = gpu.empty(M * n_head * hd, np.float32)
    gpu.attention(out, gpu.array(q), kc, vc, n_head, n_kv, hd, M,
                  gpu.array(np.array([pos], np.uint32)), n_ctx, rf.ATTN_EXACT)
    got = out.numpy().reshape(M, -1)
    for t in range(M):
        o = gpu.empty(n_head * hd, np.float32)
        gpu.attention(o, gpu.array(q[t]), kc, vc, n_head, n_kv, hd, 1,
                      gpu.array(np.array([pos + t], np.uint32)), n_ctx, rf.ATTN_EXACT)
        assert np.array_equal(bits(got[t]), bits(o.numpy())), f"token {t}"


@pytest.mark.parametrize("kind,K,tiles,M", [
    ("gemv", 8192, 768, 7), ("gemv", 8192, 769, 7), ("gemv", 9216, 1280, 6), ("gemv", 9216, 1281, 6),
    ("gate_up", 5376, 768, 8), ("gate_up", 5376, 769, 8), ("gate_up", 7936, 512, 5),
    ("gate_up", 7936, 513, 5),
])
def test_wide_ternary_products_on_either_side_of_the_rule(gpu, kind, K, tiles, M):
    """Ternary products just below and above the row tiles from which they leave
    the one-launch kernel: as with that kernel's grid capped (a cap that binds
    nothing, but keeps it), which other tests compare with the oracle."""
    rng = np.random.default_rng(K + tiles)
    t, N = TYPES["TQ2_0"], 16 * tiles - 5
    rows = weights(rng, t, 1 << 10, K).reshape(1 << 10, -1)
    ws = [gpu.tensor(t, K, N, rows[rng.integers(0, 1 << 10, N)]) for _ in range(2 if kind == "gate_up" else 1)]
    x, nw = gpu.array(rng.standard_normal((M, K)).astype(np.float32)), gpu.array(np.ones(K, np.float32))
    got = []
    for cap in (0, 1 << 20):
        gpu.set_max_workgroups(cap)
        o = gpu.empty(M * N, np.float32)
        if kind == "gemv":
            gpu.gemv(ws[0], x, M, o)
        else:
            gpu.gate_up_silu(ws[0], ws[1], x, M, nw, EPS, o)
        got.append(bits(o.numpy()))
    gpu.set_max_workgroups(0)
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("n", [1025, 1200])
def test_a_prompt_of_two_batched_passes(tmp_path, n):
    """More than 1024 tokens: two batched passes in a row, the second on the
    first one's cache rows, against passes of eight."""
    s = synth.spec("tiny-512", n_layer=2, n_vocab=512, n_ctx=2048)
    path = str(tmp_path / "m.gguf")
    synth.write_gguf(path, s)
    ids = np.concatenate([synth.prompt_ids(400, s.n_vocab)] * 3)[:n]
    with rf.Model(path) as m:
        a, b = m.context(2048), m.context(2048, n_batch=8)
        assert np.array_equal(bits(a.eval(ids)), bits(b.eval(ids)))
        assert a.position == n
        assert np.array_equal(bits(a.eval(ids[:9])), bits(b.eval(ids[:9])))
        a.close()
        b.close()


def test_streamed_prompt_equals_resident(tmp_path):
    """A batched prompt over layers streamed through slots: the resident
    model's logits."""
    s = synth.spec("tiny-512", n_ctx=128)
    path = str(tmp_path / "m.gguf")
    synth.write_gguf(path, s)
    ids = synth.prompt_ids(100, s.n_vocab)
    with rf.Model(path) as m:
        c = m.context(128)
        want = c.eval(ids).copy()
        c.close()
    with rf.Model(path, mode=rf.WEIGHTS_STREAM) as m:
        c = m.context(128)
        assert np.array_equal(bits(c.eval(ids)), bits(want))
        c.close()


def test_a_refused_allocation_fails_no_later_call(gpu):
    """An allocation that the device refuses is that call's error only: the
    next launch does not report it again."""
    x = np.random.default_rng(2).standard_normal((9, 512)).astype(np.float32)
    W = weights(np.random.default_rng(3), TYPES["TQ2_0"], 40, 512)
    w, dx, out = gpu.tensor(TYPES["TQ2_0"], 512, 40, W), gpu.array(x), gpu.empty(9 * 40, np.float32)
    with pytest.raises(rf.FoxError) as e:
        gpu.empty(1 << 48, np.float32)
    assert e.value.status == 3
    gpu.batch_gemv([w], dx, 9, [out])
    assert np.isfinite(out.numpy()).all()


def test_few_tokens_on_a_long_cache_equal_passes_of_eight(tmp_path):
    """Batched passes whose attention runs in calls of eight tokens (few tokens
    on a long cache), and one on the same cache that is long enough not to."""
    s = synth.spec("8b", n_layer=2, n_vocab=512, n_embd=512, n_ff=768, n_head=8, n_head_kv=2, head_dim=64,
                   n_ctx=1600)
    path = str(tmp_path / "m.gguf")
    synth.write_gguf(path, s)
    rng = np.random.default_rng(7)
    with rf.Model(path) as m:
        a, b = m.context(1600), m.context(1600, n_batch=8)
        for l in range(2):
            k, v = (rng.standard_normal((1400, 128)).astype(np.float32) for _ in range(2))
            a.set_kv(l, 0, k, v)
            b.set_kv(l, 0, k, v)
        for pos, n in ((1400, 9), (1391, 16), (1203, 23), (1000, 100)):
            ids = synth.prompt_ids(n, s.n_vocab)
            for c in (a, b):
                c.set_position(pos)
            x, y = a.eval_all(ids), b.eval_all(ids)
            assert np.array_equal(bits(x), bits(y)), (pos, n)
        a.close()
        b.close()
