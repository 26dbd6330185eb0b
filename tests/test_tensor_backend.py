"""The op-level ITensorBackend of the hip backend (fh_op_*, forge_hip.tensor_backend).

CPU tests pin the oracle's restatement of the rest of CpuBackend (training ops) the
way the reference's own CpuBackendTests do: brute-force matmuls, the cross-entropy
hand literal, the AdamW first-step closed form, and finite-difference gradient checks
of every backward kernel against the oracle's forward (CpuBackendTests.cs:86-540,
TrainingTests.cs:40-51).  GPU tests are the reference's device-backend contract
(GpuBackendTests.cs:110-600, CudaBackendTests.cs:274-335) run through the C ABI: each
kernel against the oracle on the same inputs, with the reference's tolerances
(1e-4 forward, 1e-2 backward, exact for copies, gathers and masks), plus the
residency contract and the error paths.  Inputs come from the restated seeded
System.Random with the reference tests' seeds and Box-Muller helper (the stream
itself is parity unpinned vs .NET); index arrays use numpy generators.
"""
import numpy as np
import pytest

FWD, BWD = 1e-4, 1e-2


class NetRng:
    """Sequential NextDouble draws of new Random(seed) (restated generator)."""

    def __init__(self, oracle, seed, n=1 << 16):
        self.d = oracle.net_random_doubles(seed, n)
        self.i = 0

    def next_double(self):
        v = self.d[self.i]
        self.i += 1
        return v

    def rand(self, n, std=1.0):
        """GpuBackendTests.Rand: Box-Muller pairs (cos, sin) in double."""
        out = np.empty(n, np.float32)
        for i in range(0, n, 2):
            u1 = 1.0 - self.next_double()
            u2 = self.next_double()
            r = np.sqrt(-2.0 * np.log(u1))
            out[i] = np.float32(r * np.cos(2 * np.pi * u2) * std)
            if i + 1 < n:
                out[i + 1] = np.float32(r * np.sin(2 * np.pi * u2) * std)
        return out


def near_rel(actual, expected, tol):
    a = np.asarray(actual, np.float64)
    e = np.asarray(expected, np.float64)
    assert a.shape == e.shape
    if tol == 0:
        np.testing.assert_array_equal(np.asarray(actual), np.asarray(expected))
        return
    err = np.abs(a - e) / np.maximum(1.0, np.abs(e))
    assert not np.any(np.isnan(err)), "NaN"
    assert err.max(initial=0.0) <= tol, f"max rel/abs diff {err.max():.3g} > {tol}"


def naive_matmul(a, b, M, K, N, ta, tb):
    A = np.asarray(a, np.float64).reshape((K, M) if ta else (M, K))
    B = np.asarray(b, np.float64).reshape((N, K) if tb else (K, N))
    return ((A.T if ta else A) @ (B.T if tb else B)).reshape(-1)


def check_grad(analytic, param, loss, eps=1e-2, tol=2e-2):
    """Central differences of a float32 loss against the analytic gradient."""
    for i in range(param.size):
        old = param[i]
        param[i] = old + eps
        lp = loss()
        param[i] = old - eps
        lm = loss()
        param[i] = old
        num = (lp - lm) / (2 * eps)
        assert abs(num - analytic[i]) <= tol * max(1.0, abs(num)), (i, num, analytic[i])


# ---- CPU: the oracle's restatement pinned ----------------------------------------------

@pytest.mark.parametrize("mode,seed", [("nn", 1), ("nt", 2), ("tn", 3)])
def test_oracle_matmuls_match_naive(oracle, mode, seed):
    # CpuBackendTests.MatMulNN/NT/TN_Forward, plain and accumulating
    rng = NetRng(oracle, seed)
    M, K, N = 3, 5, 4
    a = rng.rand(M * K)
    b = rng.rand(K * N)
    y = np.zeros(M * N, np.float32)
    oracle.op_matmul(mode, a, b, y, M, K, N)
    ref = naive_matmul(a, b, M, K, N, mode == "tn", mode == "nt")
    near_rel(y, ref, 1e-4)
    y[:] = -1.5
    oracle.op_matmul(mode, a, b, y, M, K, N, accumulate=True)
    near_rel(y, ref - 1.5, 1e-4)
    # batched: slot s is the plain product of slot s's operands
    S = 3
    a3, b3 = rng.rand(S * M * K), rng.rand(S * K * N)
    y3 = np.zeros(S * M * N, np.float32)
    oracle.op_matmul(mode, a3, b3, y3, M, K, N, slots=S)
    for s in range(S):
        near_rel(y3[s * M * N:(s + 1) * M * N],
                 naive_matmul(a3[s * M * K:(s + 1) * M * K], b3[s * K * N:(s + 1) * K * N], M, K, N, mode == "tn",
                              mode == "nt"), 1e-4)


def test_oracle_rows_and_elementwise(oracle):
    # CpuBackendTests.Transpose_MatchesNaive, AddBiasSumRowsScaleAddInPlace
    rng = NetRng(oracle, 5)
    rows, cols = 3, 4
    y, bias = rng.rand(rows * cols), rng.rand(cols)
    want = y.reshape(rows, cols) + bias
    oracle.op_add_bias(y, bias, rows, cols)
    np.testing.assert_allclose(y.reshape(rows, cols), want, atol=1e-6)
    db = rng.rand(cols)
    prior = db.copy()
    oracle.op_sum_rows(y, db, rows, cols)
    np.testing.assert_allclose(db, prior + y.reshape(rows, cols).sum(0), atol=1e-5)
    z = rng.rand(rows * cols)
    zc = z.copy()
    oracle.op_scale(z, 2.5)
    np.testing.assert_allclose(z, zc * 2.5, atol=1e-5)
    oracle.op_add_in_place(z, zc)
    np.testing.assert_allclose(z, zc * 3.5, atol=1e-5)
    x = rng.rand(15)
    out = np.zeros(15, np.float32)
    oracle.op_transpose(x, out, 3, 5)
    np.testing.assert_array_equal(out.reshape(5, 3), x.reshape(3, 5).T)


def test_oracle_heads_block_mask_embedding(oracle):
    batch, T, H, hd = 3, 7, 2, 5
    D = H * hd
    src = np.arange(batch * T * 3 * D, dtype=np.float32)
    q = np.zeros(batch * H * T * hd, np.float32)
    oracle.op_pack_heads(src, 3 * D, q, batch, T, H, hd, D)
    s3 = src.reshape(batch, T, 3, H, hd)[:, :, 1]  # the K block: [batch, T, H, hd]
    np.testing.assert_array_equal(q.reshape(batch, H, T, hd), s3.transpose(0, 2, 1, 3))
    back = np.zeros_like(src)
    oracle.op_unpack_heads(q, back, 3 * D, batch, T, H, hd, D)
    np.testing.assert_array_equal(back.reshape(batch, T, 3, D)[:, :, 1], src.reshape(batch, T, 3, D)[:, :, 1])
    assert not back.reshape(batch, T, 3, D)[:, :, [0, 2]].any()
    # CopyBlock extract: a 7x23 block at (5, 11) of a [33, 65] into (3, 7) of a zeroed [12, 40]
    y = np.arange(33 * 65, dtype=np.float32)
    blk = np.zeros(12 * 40, np.float32)
    oracle.op_copy_block(y, 65, blk, 40, 5, 11, 3, 7, 7, 23)
    want = np.zeros((12, 40), np.float32)
    want[3:10, 7:30] = y.reshape(33, 65)[5:12, 11:34]
    np.testing.assert_array_equal(blk.reshape(12, 40), want)
    # CausalMask_SetsUpperTriangle over two packed blocks
    T = 4
    sc = np.ones(2 * T * T, np.float32)
    oracle.op_causal_mask(sc, T)
    tri = np.triu(np.ones((T, T), bool), 1)
    for blkn in range(2):
        m = sc[blkn * T * T:(blkn + 1) * T * T].reshape(T, T)
        assert np.all(np.isneginf(m[tri])) and np.all(m[~tri] == 1)
    # Embedding_Lookup
    table = np.arange(5 * 3, dtype=np.float32)
    out = np.zeros(4 * 3, np.float32)
    oracle.op_embedding_forward(table, [0, 2, 2, 4], out, 3)
    np.testing.assert_array_equal(out.reshape(4, 3), table.reshape(5, 3)[[0, 2, 2, 4]])


def test_oracle_layernorm_forward_statistics(oracle):
    # LayerNormForward with its cached statistics: out equals the inference
    # restatement bit for bit, mean and rstd are the row's mean and 1/sqrt(var+eps)
    rng = NetRng(oracle, 104)
    rows, cols, eps = 5, 48, 1e-5
    x, w, b = rng.rand(rows * cols), rng.rand(cols), rng.rand(cols)
    out, mean, rstd = np.zeros(rows * cols, np.float32), np.zeros(rows, np.float32), np.zeros(rows, np.float32)
    oracle.op_layernorm_forward(x, w, b, out, mean, rstd, rows, cols, eps)
    ref = oracle.layernorm(x.reshape(rows, cols), w, b, eps)
    np.testing.assert_array_equal(out.reshape(rows, cols), ref)
    X = x.reshape(rows, cols).astype(np.float64)
    np.testing.assert_allclose(mean, X.mean(1), atol=1e-6)
    np.testing.assert_allclose(rstd, 1 / np.sqrt(X.var(1) + eps), rtol=1e-5)


def test_oracle_cross_entropy_hand_literal(oracle):
    # CpuBackendTests.CrossEntropy_MatchesLogSoftmax
    T, V = 3, 4
    logits = np.array([1, 2, 0.5, -1, 0, 0, 0, 0, -2, 3, 1, 0], np.float32)
    targets = [1, 99, 0]
    probs = np.zeros(T * V, np.float32)
    loss = oracle.op_cross_entropy_forward(logits, targets, probs, T, V, 99)
    exp = 0.0
    for t in range(T):
        if targets[t] == 99:
            continue
        row = logits[t * V:(t + 1) * V].astype(np.float64)
        mx = row.max()
        exp += np.log(np.exp(row - mx).sum()) + mx - row[targets[t]]
    assert abs(loss - exp / 2) <= 1e-4
    np.testing.assert_allclose(probs.reshape(T, V).sum(1), 1.0, atol=1e-5)
    np.testing.assert_allclose(probs[V:2 * V], 0.25, atol=1e-6)


def test_oracle_cross_entropy_aliased_equals_separate(oracle):
    # CpuBackendTests.CrossEntropy_AliasedInPlaceMatchesSeparate
    rng = NetRng(oracle, 42)
    T, V = 3, 5
    logits = np.array([rng.next_double() * 4 - 2 for _ in range(T * V)], np.float32)
    targets = [2, 99, 0]
    pr = np.zeros_like(logits)
    lr_ = oracle.op_cross_entropy_forward(logits.copy(), targets, pr, T, V, 99)
    dr = np.zeros_like(logits)
    oracle.op_cross_entropy_backward(pr, targets, dr, T, V, 99)
    buf = logits.copy()
    l2 = oracle.op_cross_entropy_forward(buf, targets, buf, T, V, 99)
    assert l2 == lr_
    np.testing.assert_array_equal(buf, pr)
    oracle.op_cross_entropy_backward(buf, targets, buf, T, V, 99)
    np.testing.assert_array_equal(buf, dr)


def test_oracle_gradient_checks(oracle):
    # CpuBackendTests.*Backward_GradCheck: every backward kernel against central
    # differences of the oracle's own forward
    rng = NetRng(oracle, 42)
    M, K, N = 3, 4, 2
    a, b, dY = rng.rand(M * K), rng.rand(K * N), rng.rand(M * N)

    def mm_loss():
        y = np.zeros(M * N, np.float32)
        oracle.op_matmul("nn", a, b, y, M, K, N)
        return float(np.dot(y.astype(np.float64), dY))

    dA = np.zeros(M * K, np.float32)
    dB = np.zeros(K * N, np.float32)
    oracle.op_matmul("nt", dY, b, dA, M, N, K)
    oracle.op_matmul("tn", a, dY, dB, K, M, N)
    check_grad(dA, a, mm_loss)
    check_grad(dB, b, mm_loss)

    rows, cols = 3, 4
    x, w, bb, dO = rng.rand(rows * cols), rng.rand(cols), rng.rand(cols), rng.rand(rows * cols)
    mean, rstd = np.zeros(rows, np.float32), np.zeros(rows, np.float32)

    def ln_loss():
        out = np.zeros(rows * cols, np.float32)
        oracle.op_layernorm_forward(x, w, bb, out, mean, rstd, rows, cols, 1e-5)
        return float(np.dot(out.astype(np.float64), dO))

    ln_loss()
    dX, dW, dBb = np.zeros(rows * cols, np.float32), np.zeros(cols, np.float32), np.zeros(cols, np.float32)
    oracle.op_layernorm_backward(dO, x, w, mean, rstd, dX, dW, dBb, rows, cols)
    check_grad(dX, x, ln_loss)
    check_grad(dW, w, ln_loss)
    check_grad(dBb, bb, ln_loss)

    xs, dOs = rng.rand(rows * cols), rng.rand(rows * cols)

    def sm_loss():
        s = xs.copy()
        oracle.op_softmax_forward(s, rows, cols)
        return float(np.dot(s.astype(np.float64), dOs))

    s = xs.copy()
    oracle.op_softmax_forward(s, rows, cols)
    dXs = np.zeros_like(s)
    oracle.op_softmax_backward(dOs, s, dXs, rows, cols)
    check_grad(dXs, xs, sm_loss)

    xg, dOg = rng.rand(12), rng.rand(12)

    def gelu_loss():
        yv = np.zeros(12, np.float32)
        oracle.op_gelu_forward(xg, yv)
        return float(np.dot(yv.astype(np.float64), dOg))

    dXg = np.zeros(12, np.float32)
    oracle.op_gelu_backward(dOg, xg, dXg)
    check_grad(dXg, xg, gelu_loss)

    V, D = 5, 3
    table = rng.rand(V * D)
    idx = [0, 2, 2, 4]
    dOe = rng.rand(len(idx) * D)

    def emb_loss():
        out = np.zeros(len(idx) * D, np.float32)
        oracle.op_embedding_forward(table, idx, out, D)
        return float(np.dot(out.astype(np.float64), dOe))

    dT = np.zeros(V * D, np.float32)
    oracle.op_embedding_backward(dOe, idx, dT, D)
    check_grad(dT, table, emb_loss)
    np.testing.assert_allclose(dT[2 * D:3 * D], dOe[D:2 * D] + dOe[2 * D:3 * D], atol=1e-6)
    assert not dT[D:2 * D].any()

    T, Vc = 3, 4
    lg = rng.rand(T * Vc)
    tg = [1, 99, 0]

    def ce_loss():
        return oracle.op_cross_entropy_forward(lg, tg, np.zeros(T * Vc, np.float32), T, Vc, 99)

    pr = np.zeros(T * Vc, np.float32)
    oracle.op_cross_entropy_forward(lg, tg, pr, T, Vc, 99)
    dl = np.zeros(T * Vc, np.float32)
    oracle.op_cross_entropy_backward(pr, tg, dl, T, Vc, 99)
    check_grad(dl, lg, ce_loss)
    assert not dl[Vc:2 * Vc].any()


def test_oracle_adamw_first_step_and_decay(oracle):
    # TrainingTests.AdamW_FirstStepMovesByAboutLr: mhat = vhat = g after the bias
    # correction, so the first step moves w by lr * g / (|g| + eps) ~ lr
    w, g = np.array([1.0], np.float32), np.array([1.0], np.float32)
    m, v = np.zeros(1, np.float32), np.zeros(1, np.float32)
    oracle.op_adamw(w, g, m, v, 0.1, 0.9, 0.999, 1e-8, 0.0, 1, True)
    assert abs(w[0] - 0.9) <= 1e-4
    # the moments are (1 - beta) * g in float32: (1 - 0.9f) = 0.100000024f
    assert m[0] == np.float32(1) - np.float32(0.9) and v[0] == np.float32(1) - np.float32(0.999)
    # decoupled decay only for matrices: w -= lr*wd*w before the Adam step
    for matrix in (True, False):
        w2, m2, v2 = np.array([2.0], np.float32), np.zeros(1, np.float32), np.zeros(1, np.float32)
        oracle.op_adamw(w2, np.array([0.5], np.float32), m2, v2, 0.01, 0.9, 0.95, 1e-8, 0.1, 1, matrix)
        dec = 2.0 - (0.01 * 0.1 * 2.0 if matrix else 0.0)
        assert abs(w2[0] - (dec - 0.01 * 0.5 / (0.5 + 1e-8))) <= 1e-6


def test_oracle_sum_squares(oracle):
    x = np.random.default_rng(0).standard_normal(100003).astype(np.float32)
    assert abs(oracle.op_sum_squares(x) - float(np.dot(x.astype(np.float64), x))) <= 1e-9 * x.size


def test_python_tensor_mirror(fhp):
    # Tensor.cs: shape ctor zero-fills, data ctor checks the element count
    t = fhp.Tensor(2, 3)
    assert t.Shape == (2, 3) and t.Rank == 2 and t.Length == 6 and t.Cols == 3 and t.Rows == 2
    assert not t.Data.any()
    u = fhp.Tensor(np.arange(6), 3, 2)
    assert u.Data.dtype == np.float32 and u.Cols == 2
    with pytest.raises(ValueError):
        fhp.Tensor(np.arange(5), 3, 2)


# ---- GPU: the device-backend contract ------------------------------------------------------

@pytest.fixture(scope="module")
def tb(fhp):
    b = fhp.HipTensorBackend(0)
    yield b
    b.Dispose()


def dup(fhp, data, *shape):
    return fhp.Tensor(np.array(data, np.float32, copy=True), *shape)


@pytest.mark.gpu
def test_matmul_matches_cpu(fhp, oracle, tb):
    # GpuBackendTests.MatMul_MatchesCpu, plus a size that takes the MFMA GEMM
    rng = NetRng(oracle, 101, 1 << 20)
    for M, K, N in [(37, 53, 29), (128, 256, 192), (256, 512, 384)]:
        a, bN, bT, prior = rng.rand(M * K), rng.rand(K * N), rng.rand(N * K), rng.rand(M * N)
        for acc in (False, True):
            for mode, bb in (("nn", bN), ("nt", bT), ("tn", bN)):
                yc = prior.copy()
                oracle.op_matmul(mode, a, bb, yc, M, K, N, accumulate=acc)
                yg = dup(fhp, prior, M, N)
                fn = {"nn": tb.MatMulNN, "nt": tb.MatMulNT, "tn": tb.MatMulTN}[mode]
                ashape = (K, M) if mode == "tn" else (M, K)
                bshape = (N, K) if mode == "nt" else (K, N)
                fn(dup(fhp, a, *ashape), dup(fhp, bb, *bshape), yg, M, K, N, acc)
                tb.EnsureHostCurrent(yg)
                near_rel(yg.Data, yc, FWD)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["nn", "nt", "tn"])
@pytest.mark.parametrize("slots,M,K,N", [(1, 1, 1, 1), (2, 64, 32, 64), (3, 65, 33, 63), (1, 129, 31, 257),
                                         (5, 40, 331, 64), (1, 300, 2049, 130), (1, 1025, 768, 1100),
                                         (2, 200, 4096, 96)])
def test_split_matmul_tiles_and_remainders(fhp, tb, mode, slots, M, K, N):
    """Products around the split GEMM's tiles (64 and 128 rows and columns, 32 k), whole and split
    over K, plain and accumulated, against float64.  A sum is rounded 6 K / 16 times (a sixth of that in the
    64 x 64 tile), each time by an error that is uniform over an ulp, of at most 2^-23 of what the sum has come to,
    and the squares of that are half the last one's on average: (6 K / 16 / 2)^0.5 2^-23 / 12^0.5 = 2^-24 K^0.5 / 4
    in the 2-norm.  The last rounding and the split's left-out terms (three of 2^-26) take less than 2^-24 more."""
    g = np.random.default_rng(slots * 1000 + M + K + N)
    a = g.standard_normal((slots, K, M) if mode == "tn" else (slots, M, K)).astype(np.float32)
    b = g.standard_normal((slots, N, K) if mode == "nt" else (slots, K, N)).astype(np.float32)
    prior = g.standard_normal((slots, M, N)).astype(np.float32)
    A = a.astype(np.float64).transpose(0, 2, 1) if mode == "tn" else a.astype(np.float64)
    B = b.astype(np.float64).transpose(0, 2, 1) if mode == "nt" else b.astype(np.float64)
    want = A @ B
    fn = {"nn": tb.BatchedMatMulNN, "nt": tb.BatchedMatMulNT, "tn": tb.BatchedMatMulTN}[mode]
    for acc in (False, True):
        y = dup(fhp, prior, slots * M, N)
        fn(dup(fhp, a, slots * a.shape[1], a.shape[2]), dup(fhp, b, slots * b.shape[1], b.shape[2]), y, slots, M, K, N,
           acc)
        tb.EnsureHostCurrent(y)
        err = y.Data.reshape(want.shape) - want - (prior if acc else 0)
        size = np.linalg.norm(want) + (np.linalg.norm(prior) if acc else 0)
        assert np.linalg.norm(err) <= 2.0 ** -24 * (1 + np.sqrt(K) / 4) * size, np.linalg.norm(err) / size


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["nn", "nt", "tn"])
@pytest.mark.parametrize("slots,M,K,N", [(1, 300, 1, 517), (3, 65, 2, 64), (1, 63, 7, 130), (700, 8, 8, 8),
                                         (2, 200, 8, 90), (1, 70, 4, 70), (1, 70, 5, 70)])
def test_matmul_of_few_k_rounds_once(fhp, tb, mode, slots, M, K, N):
    """Up to 8 products to a sum: within half an ulp of float64; accumulated, within one of both terms."""
    g = np.random.default_rng(M + K)
    a = g.standard_normal((slots, K, M) if mode == "tn" else (slots, M, K)).astype(np.float32)
    b = g.standard_normal((slots, N, K) if mode == "nt" else (slots, K, N)).astype(np.float32)
    prior = g.standard_normal((slots, M, N)).astype(np.float32)
    want = (a.transpose(0, 2, 1) if mode == "tn" else a).astype(np.float64) @ \
        (b.transpose(0, 2, 1) if mode == "nt" else b).astype(np.float64)
    fn = {"nn": tb.BatchedMatMulNN, "nt": tb.BatchedMatMulNT, "tn": tb.BatchedMatMulTN}[mode]
    for acc in (False, True):
        y = dup(fhp, prior, slots * M, N)
        fn(dup(fhp, a, slots * a.shape[1], a.shape[2]), dup(fhp, b, slots * b.shape[1], b.shape[2]), y, slots, M, K, N,
           acc)
        tb.EnsureHostCurrent(y)
        err = np.abs(y.Data.reshape(want.shape) - want - (prior if acc else 0))
        if not acc:
            assert np.all(err <= 2.0 ** -24 * (1 + 1e-6) * np.abs(want))
        elif K == 1:
            assert np.all(err <= 2.0 ** -24 * (1 + 1e-6) * (2 * np.abs(want) + np.abs(prior)))
        else:  # the split GEMM where the result is wide: K roundings
            size = np.abs(a).max() * np.abs(b).max() * K + np.abs(prior)
            assert np.all(err <= 2.0 ** -24 * (K + 2) * size)


@pytest.mark.gpu
@pytest.mark.parametrize("mode,slots,M,K,N",
                         [(m, *s) for m in ("nn", "nt", "tn") for s in
                          [(1, (1 << 21) + 1, 17, 3), (1, 3, (1 << 21) + 7, 5), (1, 2, 18, (1 << 21) + 5),
                           (1, 2, 1, 1 << 22), (1, 1, 18, 1 << 22)]] + [("nn", 65535, 1, 13, 520)])
def test_matmul_of_millions(fhp, tb, mode, slots, M, K, N):
    """Each dimension past 2^21, the scalar kernel past 2^22 columns, and more than 2^19 tiles: against float64
    at rows, slots and columns of both ends."""
    g = np.random.default_rng(M % 97 + N % 89)

    def normal(*shape):  # a pattern whose length divides no dimension
        return np.resize(g.standard_normal(1000003).astype(np.float32), shape)

    a = normal(slots, K, M) if mode == "tn" else normal(slots, M, K)
    b = normal(slots, N, K) if mode == "nt" else normal(slots, K, N)
    prior = normal(slots, M, N)
    fn = {"nn": tb.BatchedMatMulNN, "nt": tb.BatchedMatMulNT, "tn": tb.BatchedMatMulTN}[mode]
    ta, tn = dup(fhp, a, slots * a.shape[1], a.shape[2]), dup(fhp, b, slots * b.shape[1], b.shape[2])
    ss = sorted({0, slots // 2, slots - 1})
    mm = sorted({*range(min(M, 40)), *range(max(0, M - 40), M)})
    nn = sorted({*range(min(N, 40)), *range(max(0, N - 40), N)})
    for acc in (False, True):
        y = dup(fhp, prior, slots * M, N)
        fn(ta, tn, y, slots, M, K, N, acc)
        tb.EnsureHostCurrent(y)
        got = y.Data.reshape(slots, M, N)
        for s in ss:
            A = (a[s].T if mode == "tn" else a[s])[mm].astype(np.float64)
            B = (b[s].T if mode == "nt" else b[s])[:, nn].astype(np.float64)
            P = prior[s][np.ix_(mm, nn)] if acc else 0
            err = got[s][np.ix_(mm, nn)] - A @ B - P
            size = np.linalg.norm(A @ B) + np.linalg.norm(P)
            assert np.linalg.norm(err) <= 2.0 ** -24 * (1 + np.sqrt(K) / 4) * size


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["nn", "nt", "tn"])
@pytest.mark.parametrize("acc", [False, True])
@pytest.mark.parametrize("M,K,N", [(150, 96, 140), (300, 2049, 130), (1025, 768, 1100), (70, 40, 70)])
def test_split_matmul_infinities_and_nan(fhp, tb, mode, acc, M, K, N):
    """Infinite, NaN and overflowing sums are those of fp32 arithmetic; other outputs stay exact to fp32:
    in one launch, split over K with the odd values in different parts of K, in tiles of 128 rows, and with a
    K that ends inside a stage."""
    g = np.random.default_rng(5)
    a = g.standard_normal((M, K)).astype(np.float32)
    b = g.standard_normal((K, N)).astype(np.float32)
    prior = g.standard_normal((M, N)).astype(np.float32)
    b[7] = 1.0  # exactly representable in bf16: its lower parts are zero
    a[3, 7] = np.inf
    a[5, 7], a[5, K - 1] = np.inf, -np.inf
    b[K - 1] = 2.0
    a[9, K - 2] = np.nan
    b[K // 2, 3] = -np.inf
    a[11, :] = 0.0
    a[11, 20], b[20, 4] = 3.4e38, 3.0  # overflows
    a[12, 21], b[21, :] = 3.4028235e38, 0.5  # rounds to infinity in bf16, is finite in fp32
    prior[14, 2] = np.inf
    with np.errstate(over="ignore", invalid="ignore"):
        # 0 * inf where a row of zeros meets b's infinity, as fp32 arithmetic has it
        want = (a.astype(np.float64) @ b.astype(np.float64) + (prior if acc else 0)).astype(np.float32)
    ta = dup(fhp, a.T.copy(), K, M) if mode == "tn" else dup(fhp, a, M, K)
    tn = dup(fhp, b.T.copy(), N, K) if mode == "nt" else dup(fhp, b, K, N)
    y = dup(fhp, prior, M, N)
    {"nn": tb.MatMulNN, "nt": tb.MatMulNT, "tn": tb.MatMulTN}[mode](ta, tn, y, M, K, N, accumulate=acc)
    tb.EnsureHostCurrent(y)
    got = y.Data.reshape(M, N)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    np.testing.assert_array_equal(got[inf], want[inf])
    ok = np.isfinite(want)
    assert np.all(np.isfinite(got[ok]))
    # sums of K standard products: K^0.5 of them in size, K^0.5 roundings of that (row 12's by 2^127)
    np.testing.assert_allclose(got[ok], want[ok], rtol=1e-5, atol=2.0 ** -24 * 8 * K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(64, 64, 64), (300, 2049, 130), (1025, 768, 1100)])
@pytest.mark.parametrize("exponent", [-60, -85, -108, -112, -118, -126])
def test_split_matmul_of_tiny_elements(fhp, tb, M, K, N, exponent):
    """Elements near the bottom of the normal range, on the left or the right, beside ordinary ones: the bound of
    ordinary elements, and a zero row stays zero.  (Products below 2^-126 are subnormal: multiples of 2^-149.)"""
    g = np.random.default_rng(K - exponent)
    a, b = g.standard_normal((M, K)).astype(np.float32), g.standard_normal((K, N)).astype(np.float32)
    tiny = np.float32(2.0) ** exponent
    for ta, tn in ((a * tiny, b), (a, b * tiny)):
        ta[5] = 0
        want = ta.astype(np.float64) @ tn.astype(np.float64)
        y = fhp.Tensor(M, N)
        tb.MatMulNN(dup(fhp, ta, M, K), dup(fhp, tn, K, N), y, M, K, N)
        tb.EnsureHostCurrent(y)
        got = y.Data.reshape(M, N)
        assert np.all(got[5] == 0)
        err = np.linalg.norm(got - want)
        assert err <= 2.0 ** -24 * (1 + np.sqrt(K) / 4) * np.linalg.norm(want) + np.sqrt(M * N * K) * 2.0 ** -149, err


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["nn", "nt", "tn"])
def test_split_matmul_of_nan_takes_a_few_times_a_finite_product(fhp, tb, mode):
    """Operands with NaN go through the fp32 matrix cores after the split: twice the time of a finite product.
    The bound leaves a factor of four for noise (a loop of scalar multiply-adds took 80 times)."""
    import time
    M, K, N = 2048, 768, 3072
    g = np.random.default_rng(6)
    a, b = g.standard_normal((M, K)).astype(np.float32), g.standard_normal((K, N)).astype(np.float32)
    fn = {"nn": tb.MatMulNN, "nt": tb.MatMulNT, "tn": tb.MatMulTN}[mode]
    y = fhp.Tensor(M, N)

    def best(first):
        a[0, 0] = first
        a[:, 5] = first
        ta = dup(fhp, a.T.copy(), K, M) if mode == "tn" else dup(fhp, a, M, K)
        tn = dup(fhp, b.T.copy(), N, K) if mode == "nt" else dup(fhp, b, K, N)
        times = []
        for _ in range(6):
            t = time.perf_counter()
            for _ in range(20):
                fn(ta, tn, y, M, K, N)
            tb.SumSquares(y)  # waits
            times.append(time.perf_counter() - t)
        return min(times)

    finite = best(1.0)
    assert best(np.nan) < 8 * finite


@pytest.mark.gpu
def test_elementwise_matches_cpu(fhp, oracle, tb):
    # GpuBackendTests.Elementwise_MatchesCpu
    rng = NetRng(oracle, 102)
    rows, cols = 33, 65
    y, bias = rng.rand(rows * cols), rng.rand(cols)
    yc, yg = y.copy(), dup(fhp, y, rows, cols)
    oracle.op_add_bias(yc, bias, rows, cols)
    tb.AddBias(yg, dup(fhp, bias, cols), rows, cols)
    tb.EnsureHostCurrent(yg)
    near_rel(yg.Data, yc, FWD)
    db0 = rng.rand(cols)
    dbc, dbg = db0.copy(), dup(fhp, db0, cols)
    oracle.op_sum_rows(y, dbc, rows, cols)
    tb.SumRows(dup(fhp, y, rows, cols), dbg, rows, cols)
    tb.EnsureHostCurrent(dbg)
    near_rel(dbg.Data, dbc, BWD)
    src = rng.rand(rows * cols)
    yc, yg = y.copy(), dup(fhp, y, rows, cols)
    oracle.op_add_in_place(yc, src)
    tb.AddInPlace(yg, dup(fhp, src, rows, cols))
    tb.EnsureHostCurrent(yg)
    near_rel(yg.Data, yc, FWD)
    yc, yg = y.copy(), dup(fhp, y, rows, cols)
    oracle.op_scale(yc, -1.75)
    tb.Scale(yg, -1.75)
    tb.EnsureHostCurrent(yg)
    near_rel(yg.Data, yc, FWD)
    trc, trg = np.zeros(cols * rows, np.float32), fhp.Tensor(cols, rows)
    oracle.op_transpose(y, trc, rows, cols)
    tb.Transpose(dup(fhp, y, rows, cols), trg, rows, cols)
    tb.EnsureHostCurrent(trg)
    near_rel(trg.Data, trc, 0)
    cpg = fhp.Tensor(rows, cols)
    tb.Copy(dup(fhp, y, rows, cols), cpg)
    tb.EnsureHostCurrent(cpg)
    near_rel(cpg.Data, y, 0)
    blkc, blkg = np.zeros(12 * 40, np.float32), fhp.Tensor(12, 40)
    oracle.op_copy_block(y, cols, blkc, 40, 5, 11, 3, 7, 7, 23)
    tb.CopyBlock(dup(fhp, y, rows, cols), blkg, 5, 11, 3, 7, 7, 23)
    tb.EnsureHostCurrent(blkg)
    near_rel(blkg.Data, blkc, 0)
    intoc, intog = y.copy(), dup(fhp, y, rows, cols)
    oracle.op_copy_block(blkc, 40, intoc, cols, 3, 7, 9, 30, 7, 23)
    tb.CopyBlock(dup(fhp, blkc, 12, 40), intog, 3, 7, 9, 30, 7, 23)
    tb.EnsureHostCurrent(intog)
    near_rel(intog.Data, intoc, 0)  # the partial write keeps the rest


@pytest.mark.gpu
def test_flat_dispatch_beyond_one_dimension(fhp, tb):
    # GpuBackendTests.FlatDispatch_BeyondOneDimensionalLimit: 5,000,123 elements
    n = 5_000_123
    r = np.random.default_rng(103)
    a, b = r.standard_normal(n).astype(np.float32), r.standard_normal(n).astype(np.float32)
    ag = dup(fhp, a, n)
    tb.AddInPlace(ag, dup(fhp, b, n))
    tb.EnsureHostCurrent(ag)
    near_rel(ag.Data, a + b, FWD)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(33, 64), (300, 768)])
def test_layernorm_matches_cpu(fhp, oracle, tb, rows, cols):
    # GpuBackendTests.LayerNorm_MatchesCpu (and a 300-row case: column sums over chunks)
    rng = NetRng(oracle, 104, 1 << 20)
    eps = 1e-5
    x, w, b = rng.rand(rows * cols), rng.rand(cols), rng.rand(cols)
    oc, mc, rc = np.zeros(rows * cols, np.float32), np.zeros(rows, np.float32), np.zeros(rows, np.float32)
    oracle.op_layernorm_forward(x, w, b, oc, mc, rc, rows, cols, eps)
    og, mg, rg = fhp.Tensor(rows, cols), fhp.Tensor(rows), fhp.Tensor(rows)
    tb.LayerNormForward(dup(fhp, x, rows, cols), dup(fhp, w, cols), dup(fhp, b, cols), og, mg, rg, rows, cols, eps)
    for t in (og, mg, rg):
        tb.EnsureHostCurrent(t)
    near_rel(og.Data, oc, FWD)
    near_rel(mg.Data, mc, FWD)
    near_rel(rg.Data, rc, FWD)
    dO, dw0, db0 = rng.rand(rows * cols), rng.rand(cols), rng.rand(cols)
    dxc, dwc, dbc = np.zeros(rows * cols, np.float32), dw0.copy(), db0.copy()
    oracle.op_layernorm_backward(dO, x, w, mc, rc, dxc, dwc, dbc, rows, cols)
    dxg, dwg, dbg = fhp.Tensor(rows, cols), dup(fhp, dw0, cols), dup(fhp, db0, cols)
    tb.LayerNormBackward(dup(fhp, dO, rows, cols), dup(fhp, x, rows, cols), dup(fhp, w, cols), dup(fhp, mc, rows),
                         dup(fhp, rc, rows), dxg, dwg, dbg, rows, cols)
    for t in (dxg, dwg, dbg):
        tb.EnsureHostCurrent(t)
    near_rel(dxg.Data, dxc, BWD)
    near_rel(dwg.Data, dwc, BWD)
    near_rel(dbg.Data, dbc, BWD)


@pytest.mark.gpu
def test_softmax_and_gelu_match_cpu(fhp, oracle, tb):
    # GpuBackendTests.Softmax_MatchesCpu, Gelu_MatchesCpu
    rng = NetRng(oracle, 105, 1 << 17)
    rows, cols = 29, 257
    x = rng.rand(rows * cols, 3.0)
    xc, xg = x.copy(), dup(fhp, x, rows, cols)
    oracle.op_softmax_forward(xc, rows, cols)
    tb.SoftmaxForward(xg, rows, cols)
    tb.EnsureHostCurrent(xg)
    near_rel(xg.Data, xc, FWD)
    dO = rng.rand(rows * cols)
    dxc, dxg = np.zeros(rows * cols, np.float32), fhp.Tensor(rows, cols)
    oracle.op_softmax_backward(dO, xc, dxc, rows, cols)
    tb.SoftmaxBackward(dup(fhp, dO, rows, cols), dup(fhp, xc, rows, cols), dxg, rows, cols)
    tb.EnsureHostCurrent(dxg)
    near_rel(dxg.Data, dxc, BWD)
    rng = NetRng(oracle, 106, 1 << 16)
    n = 10_003
    x = rng.rand(n, 2.0)
    oc, og = np.zeros(n, np.float32), fhp.Tensor(n)
    oracle.op_gelu_forward(x, oc)
    tb.GeluForward(dup(fhp, x, n), og)
    tb.EnsureHostCurrent(og)
    near_rel(og.Data, oc, FWD)
    dO = rng.rand(n)
    dc, dg = np.zeros(n, np.float32), fhp.Tensor(n)
    oracle.op_gelu_backward(dO, x, dc)
    tb.GeluBackward(dup(fhp, dO, n), dup(fhp, x, n), dg)
    tb.EnsureHostCurrent(dg)
    near_rel(dg.Data, dc, FWD)


@pytest.mark.gpu
def test_embedding_and_mask_match_cpu(fhp, oracle, tb):
    # GpuBackendTests.Embedding_MatchesCpu (heavy duplication) and CausalMask_MatchesCpu;
    # the scatter-add adds each id's rows in position order, so it equals the CPU loop
    rng = NetRng(oracle, 107)
    V, D, Tn = 51, 37, 96
    table = rng.rand(V * D)
    idx = np.random.default_rng(107).integers(0, V // 3, Tn).astype(np.int32)
    oc, og = np.zeros(Tn * D, np.float32), fhp.Tensor(Tn, D)
    oracle.op_embedding_forward(table, idx, oc, D)
    tb.EmbeddingForward(dup(fhp, table, V, D), idx, og, D)
    tb.EnsureHostCurrent(og)
    near_rel(og.Data, oc, 0)
    dO, dt0 = rng.rand(Tn * D), rng.rand(V * D)
    dtc, dtg = dt0.copy(), dup(fhp, dt0, V, D)
    oracle.op_embedding_backward(dO, idx, dtc, D)
    tb.EmbeddingBackward(dup(fhp, dO, Tn, D), idx, dtg, D)
    tb.EnsureHostCurrent(dtg)
    near_rel(dtg.Data, dtc, 0)
    rng = NetRng(oracle, 108)
    T = 47
    s = rng.rand(T * T * 3)
    sc, sg = s.copy(), dup(fhp, s, 3 * T, T)
    oracle.op_causal_mask(sc, T)
    tb.CausalMask(sg, T)
    tb.EnsureHostCurrent(sg)
    near_rel(sg.Data, sc, 0)
    with pytest.raises(fhp.ArgumentError, match="outside the table"):
        tb.EmbeddingForward(dup(fhp, table, V, D), [0, V], fhp.Tensor(2, D), D)


@pytest.mark.gpu
@pytest.mark.parametrize("aliased", [False, True])
def test_cross_entropy_matches_cpu(fhp, oracle, tb, aliased):
    # GpuBackendTests.CrossEntropy_MatchesCpu / CrossEntropy_AliasedInPlaceMatchesCpu
    rng = NetRng(oracle, 110 if aliased else 109, 1 << 17)
    T, V, ignore = 61, 389, -1
    logits = rng.rand(T * V, 2.0)
    targets = np.random.default_rng(109).integers(0, V, T).astype(np.int32)
    targets[7] = targets[58] = ignore
    pc = np.zeros(T * V, np.float32)
    lc = oracle.op_cross_entropy_forward(logits, targets, pc, T, V, ignore)
    dlc = np.zeros(T * V, np.float32)
    oracle.op_cross_entropy_backward(pc, targets, dlc, T, V, ignore)
    if aliased:
        buf = dup(fhp, logits, T, V)
        lg = tb.CrossEntropyForward(buf, targets, buf, T, V, ignore)
        tb.EnsureHostCurrent(buf)
        near_rel(buf.Data, pc, FWD)
        tb.CrossEntropyBackward(buf, targets, buf, T, V, ignore)
        tb.EnsureHostCurrent(buf)
        near_rel(buf.Data, dlc, BWD)
    else:
        pg = fhp.Tensor(T, V)
        lg = tb.CrossEntropyForward(dup(fhp, logits, T, V), targets, pg, T, V, ignore)
        tb.EnsureHostCurrent(pg)
        near_rel(pg.Data, pc, FWD)
        dlg = fhp.Tensor(T, V)
        tb.CrossEntropyBackward(dup(fhp, pc, T, V), targets, dlg, T, V, ignore)
        tb.EnsureHostCurrent(dlg)
        near_rel(dlg.Data, dlc, BWD)
        # all ignored: zero loss, zero gradient
        allign = np.full(T, ignore, np.int32)
        assert tb.CrossEntropyForward(dup(fhp, logits, T, V), allign, fhp.Tensor(T, V), T, V, ignore) == 0.0
        dz = dup(fhp, np.ones(T * V), T, V)
        tb.CrossEntropyBackward(dup(fhp, logits, T, V), allign, dz, T, V, ignore)
        tb.EnsureHostCurrent(dz)
        assert not dz.Data.any()
    near_rel(lg, lc, FWD)


@pytest.mark.gpu
def test_loss_accumulation_returns_combined_mean(fhp, tb):
    # CpuBackendTests.CrossEntropy_LossAccumulationReturnsCombinedMean on the device
    f = dup(fhp, [2, 0, -1, 0, 1, 2], 2, 3)
    s = dup(fhp, [-1, 3, 0], 1, 3)
    first = tb.CrossEntropyForward(f, [0, 2], fhp.Tensor(2, 3), 2, 3, -1)
    second = tb.CrossEntropyForward(s, [1], fhp.Tensor(1, 3), 1, 3, -1)
    tb.BeginLossAccumulation()
    assert tb.CrossEntropyForward(f, [0, 2], fhp.Tensor(2, 3), 2, 3, -1) == 0.0  # stays on the device
    tb.CrossEntropyForward(s, [1], fhp.Tensor(1, 3), 1, 3, -1)
    acc = tb.EndLossAccumulation()
    assert abs(acc - (first * 2 + second) / 3) <= 1e-6
    with pytest.raises(fhp.InvalidOperationError, match="not active"):
        tb.EndLossAccumulation()
    tb.BeginLossAccumulation()
    with pytest.raises(fhp.InvalidOperationError, match="already active"):
        tb.BeginLossAccumulation()
    assert tb.EndLossAccumulation() == 0.0


@pytest.mark.gpu
def test_batched_attention_kernels_match_cpu(fhp, oracle, tb):
    # GpuBackendTests.BatchedAttentionKernels_MatchCpu
    rng = NetRng(oracle, 113)
    batch, T, H, hd = 3, 7, 2, 5
    D = H * hd
    src = rng.rand(batch * T * 3 * D)
    pkc = np.zeros(batch * H * T * hd, np.float32)
    oracle.op_pack_heads(src, 3 * D, pkc, batch, T, H, hd, D)
    pkg = fhp.Tensor(batch * H * T, hd)
    tb.PackHeads(dup(fhp, src, batch * T, 3 * D), pkg, batch, T, H, hd, D)
    tb.EnsureHostCurrent(pkg)
    near_rel(pkg.Data, pkc, 0)
    unc = np.zeros(batch * T * 3 * D, np.float32)
    oracle.op_unpack_heads(pkc, unc, 3 * D, batch, T, H, hd, 2 * D)
    ung = fhp.Tensor(batch * T, 3 * D)
    tb.UnpackHeads(dup(fhp, pkc, batch * H * T, hd), ung, batch, T, H, hd, 2 * D)
    tb.EnsureHostCurrent(ung)
    near_rel(ung.Data, unc, 0)
    qkv = [np.zeros(batch * H * T * hd, np.float32) for _ in range(3)]
    for i in range(3):
        oracle.op_pack_heads(src, 3 * D, qkv[i], batch, T, H, hd, i * D)
    qg, kg, vg = (fhp.Tensor(batch * H * T, hd) for _ in range(3))
    tb.PackQkvHeads(dup(fhp, src, batch * T, 3 * D), qg, kg, vg, batch, T, H, hd)
    for t, want in zip((qg, kg, vg), qkv):
        tb.EnsureHostCurrent(t)
        near_rel(t.Data, want, 0)
    back = fhp.Tensor(batch * T, 3 * D)
    tb.UnpackQkvHeads(qg, kg, vg, back, batch, T, H, hd)
    tb.EnsureHostCurrent(back)
    near_rel(back.Data, src, 0)
    rows = batch * H * T
    scores, dO = rng.rand(rows * T), rng.rand(rows * T)
    scale = 0.375
    pc = scores.copy()
    oracle.op_scaled_causal_softmax_forward(pc, rows, T, scale)
    pg = dup(fhp, scores, rows, T)
    tb.ScaledCausalSoftmaxForward(pg, rows, T, scale)
    tb.EnsureHostCurrent(pg)
    near_rel(pg.Data, pc, FWD)
    dsc = np.zeros(rows * T, np.float32)
    oracle.op_scaled_softmax_backward(dO, pc, dsc, rows, T, scale)
    dsg = fhp.Tensor(rows, T)
    tb.ScaledSoftmaxBackward(dup(fhp, dO, rows, T), pg, dsg, rows, T, scale)
    tb.EnsureHostCurrent(dsg)
    near_rel(dsg.Data, dsc, BWD)
    slots, M, K, N = batch * H, T, hd, T
    a, bN, bT, prior = rng.rand(slots * M * K), rng.rand(slots * K * N), rng.rand(slots * N * K), rng.rand(slots * M * N)
    for acc in (False, True):
        for mode, bb, fn in (("nn", bN, tb.BatchedMatMulNN), ("nt", bT, tb.BatchedMatMulNT),
                             ("tn", bN, tb.BatchedMatMulTN)):
            yc = prior.copy()
            oracle.op_matmul(mode, a, bb, yc, M, K, N, accumulate=acc, slots=slots)
            yg = dup(fhp, prior, slots * M, N)
            fn(dup(fhp, a, slots * M, K), dup(fhp, bb, slots * K, N), yg, slots, M, K, N, acc)
            tb.EnsureHostCurrent(yg)
            near_rel(yg.Data, yc, FWD)


@pytest.mark.gpu
def test_residency_contract(fhp, tb):
    # GpuBackendTests.Residency_*, EnsureHostCurrent_RoundTripsDeviceResults
    x = dup(fhp, np.ones(8), 8)
    y = fhp.Tensor(8)
    tb.Copy(x, y)                 # x now has a device copy
    x.Data[:] = 5.0               # host write without InvalidateDeviceCache
    tb.Copy(x, y)
    tb.EnsureHostCurrent(y)
    assert np.all(y.Data == 1.0)  # the kernel saw the stale device copy
    tb.InvalidateDeviceCache(x)
    tb.Copy(x, y)
    assert np.all(y.Data == 1.0)  # no download yet: host copy of y is stale
    tb.EnsureHostCurrent(y)
    assert np.all(y.Data == 5.0)
    tb.Scale(y, 2.0)
    tb.EnsureHostCurrent(y)
    tb.EnsureHostCurrent(y)       # idempotent
    assert np.all(y.Data == 10.0)
    tb.Zero(y)
    assert not y.Data.any()
    tb.AddInPlace(y, x)
    tb.EnsureHostCurrent(y)
    assert np.all(y.Data == 5.0)


@pytest.mark.gpu
def test_adamw_and_sum_squares_match_cpu(fhp, oracle, tb):
    # CudaBackendTests.AdamWAndSumSquares_MatchCpu, GlobalSumSquares_MatchesCpuWithOneReadback
    rng = NetRng(oracle, 912)
    rows, cols = 17, 19

    def vals():
        return np.array([rng.next_double() * 2 - 1 for _ in range(rows * cols)], np.float32)

    w, g, m = vals(), vals(), vals()
    v = np.abs(vals())
    wc, mc, vc = w.copy(), m.copy(), v.copy()
    oracle.op_adamw(wc, g, mc, vc, 3e-4, 0.9, 0.95, 1e-8, 0.1, 37, True)
    wg, gg, mg, vg = (dup(fhp, a, rows, cols) for a in (w, g, m, v))
    tb.AdamWStep(wg, gg, mg, vg, 3e-4, 0.9, 0.95, 1e-8, 0.1, 37)
    for t in (wg, mg, vg):
        tb.EnsureHostCurrent(t)
    np.testing.assert_allclose(wg.Data, wc, atol=2e-5)
    np.testing.assert_allclose(mg.Data, mc, atol=2e-5)
    np.testing.assert_allclose(vg.Data, vc, atol=2e-5)
    # a vector (rank 1) gets no weight decay
    b0 = vals()[:cols]
    bc = b0.copy()
    oracle.op_adamw(bc, g[:cols].copy(), np.zeros(cols, np.float32), np.zeros(cols, np.float32), 1e-2, 0.9, 0.95,
                    1e-8, 0.5, 1, False)
    bg = dup(fhp, b0, cols)
    tb.AdamWStep(bg, dup(fhp, g[:cols], cols), fhp.Tensor(cols), fhp.Tensor(cols), 1e-2, 0.9, 0.95, 1e-8, 0.5, 1)
    tb.EnsureHostCurrent(bg)
    np.testing.assert_allclose(bg.Data, bc, atol=2e-6)
    assert abs(tb.SumSquares(gg) - oracle.op_sum_squares(g)) <= 2e-4 * max(1.0, oracle.op_sum_squares(g))
    r2 = NetRng(oracle, 914, 1 << 21)
    ts, expected = [], 0.0
    for n in (1, 257, 4097, 1_000_003):
        a = np.array(r2.d[r2.i:r2.i + n] * 2 - 1, np.float64) * 0.1
        r2.i += n
        a = a.astype(np.float32)
        expected += float(np.dot(a.astype(np.float64), a))
        ts.append(dup(fhp, a, n))
    actual = tb.GlobalSumSquares(ts)
    assert abs(actual - expected) / max(1.0, expected) < 2e-5
    assert tb.GlobalSumSquares([]) == 0.0


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(1, 1), (64, 63), (65, 64), (33, 65), (2049, 257), (700, 513), (2100, 769),
                                       (5, 1024), (300, 1025), (1, 4001), (32, 2000), (33, 2000)])
def test_column_reductions_chunks_and_widths(fhp, tb, rows, cols):
    """SumRows and LayerNormBackward (dx, dw, db) around their row chunks and row widths against
    float64.  A float32 sum of n terms in any order is off by at most n 2^-24 times the sum of their
    sizes; sums in several chains stay under a quarter of that.  dx has a few roundings per element."""
    g = np.random.default_rng(rows * 31 + cols)
    d, x = g.standard_normal((2, rows, cols)).astype(np.float32)
    w = (1 + 0.1 * g.standard_normal(cols)).astype(np.float32)
    prior = g.standard_normal((3, cols)).astype(np.float32)
    x64, d64 = x.astype(np.float64), d.astype(np.float64)
    mean = x64.mean(1).astype(np.float32)
    rstd = (1 / np.sqrt(x64.var(1) + 1e-5)).astype(np.float32)
    xh = (x64 - mean[:, None].astype(np.float64)) * rstd[:, None].astype(np.float64)
    sums = [dup(fhp, v, cols) for v in prior]
    dt, dx = dup(fhp, d, rows, cols), fhp.Tensor(rows, cols)
    tb.SumRows(dt, sums[0], rows, cols)
    tb.LayerNormBackward(dt, dup(fhp, x, rows, cols), dup(fhp, w, cols), dup(fhp, mean, rows), dup(fhp, rstd, rows), dx,
                         sums[1], sums[2], rows, cols)
    for t in sums + [dx]:
        tb.EnsureHostCurrent(t)
    for t, p, terms in zip(sums, prior.astype(np.float64), (d64, d64 * xh, d64)):
        bound = 2.0 ** -24 * (4 + rows / 4) * (np.abs(terms).sum(0) + np.abs(p))
        assert np.all(np.abs(t.Data - p - terms.sum(0)) <= bound)
    dxh = d64 * w
    want = rstd[:, None] * (dxh - dxh.mean(1, keepdims=True) - xh * (dxh * xh).mean(1, keepdims=True))
    size = np.abs(rstd[:, None]) * (np.abs(dxh) + np.abs(dxh).mean(1, keepdims=True) +
                                    np.abs(xh) * np.abs(dxh * xh).mean(1, keepdims=True))
    assert np.all(np.abs(dx.Data.reshape(rows, cols) - want) <= 2.0 ** -24 * (8 + cols / 16) * size)


@pytest.mark.gpu
def test_global_sum_squares_over_many_tensors(fhp, tb):
    """More tensors than one launch takes, an empty one among them, each end of the block counts: double sums."""
    g = np.random.default_rng(9)
    sizes = [1, 255, 8192, 8193, 0, 100003, 5000000] + [7 + i for i in range(130)]
    data = [g.standard_normal(n).astype(np.float32) for n in sizes]
    want = sum(float((v.astype(np.float64) ** 2).sum()) for v in data)
    got = tb.GlobalSumSquares([dup(fhp, v, len(v)) for v in data])
    assert abs(got - want) <= 1e-12 * want


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(1, 1), (5, 64), (7, 65), (130, 129), (9, 384), (6, 385), (4, 769), (5, 1024),
                                       (3, 1025)])
def test_row_kernels_widths(fhp, tb, rows, cols):
    """Softmax forward (plain and causal) and backward and LayerNorm forward at the edges of the row
    widths that pick a kernel, against float64.  expf, a sum over the row and a few products: 16 roundings
    and cols / 64 in a lane's chain; the backward's difference is against the size of its two terms."""
    g = np.random.default_rng(rows * 7 + cols)
    x, d = g.standard_normal((2, rows, cols)).astype(np.float32)
    ulp = 2.0 ** -24 * (16 + cols / 16)
    for causal in (False, True):
        z = x.astype(np.float64) * (0.3 if causal else 1.0)
        if causal:
            z = np.where(np.arange(cols)[None, :] <= (np.arange(rows) % cols)[:, None], z, -np.inf)
        p = np.exp(z - z.max(1, keepdims=True))
        p /= p.sum(1, keepdims=True)
        t = dup(fhp, x, rows, cols)
        if causal:
            tb.ScaledCausalSoftmaxForward(t, rows, cols, 0.3)
        else:
            tb.SoftmaxForward(t, rows, cols)
        tb.EnsureHostCurrent(t)
        got = t.Data.reshape(rows, cols).astype(np.float64)
        assert np.all(np.abs(got - p) <= (ulp + 2.0 ** -22 * np.abs(x)) * p)  # the scaled score's own rounding too
        dx = fhp.Tensor(rows, cols)
        tb.ScaledSoftmaxBackward(dup(fhp, d, rows, cols), t, dx, rows, cols, 0.3)
        tb.EnsureHostCurrent(dx)
        dot = (got * d).sum(1, keepdims=True)
        size = 0.3 * got * (np.abs(d) + np.abs(got * d).sum(1, keepdims=True))
        assert np.all(np.abs(dx.Data.reshape(rows, cols) - 0.3 * got * (d - dot)) <= ulp * size)
    w, b = (1 + 0.1 * g.standard_normal((2, cols))).astype(np.float32)
    out, mean, rstd = fhp.Tensor(rows, cols), fhp.Tensor(rows), fhp.Tensor(rows)
    tb.LayerNormForward(dup(fhp, x, rows, cols), dup(fhp, w, cols), dup(fhp, b, cols), out, mean, rstd, rows, cols, 1e-5)
    tb.EnsureHostCurrent(out)
    x64 = x.astype(np.float64)
    rs = 1 / np.sqrt(x64.var(1, keepdims=True) + 1e-5)
    want = (x64 - x64.mean(1, keepdims=True)) * rs * w + b
    size = (np.abs(x64) + np.abs(x64).mean(1, keepdims=True)) * rs * np.abs(w) + np.abs(b)
    assert np.all(np.abs(out.Data.reshape(rows, cols) - want) <= ulp * size)


@pytest.mark.gpu
@pytest.mark.parametrize("T,V", [(3, 1), (2100, 2), (700, 65), (9, 128), (4099, 10), (5, 769), (3, 1024), (3, 1025),
                                 (2, 1023), (5, 4096), (3, 4097), (4, 16385), (2, 32768), (2, 32769)])
def test_cross_entropy_vocabulary_widths(fhp, tb, T, V):
    """CrossEntropy forward (in place) and backward at the edges of the vocabularies that pick a kernel."""
    g = np.random.default_rng(T + V)
    x = (3 * g.standard_normal((T, V))).astype(np.float32)
    x[0, V // 2] = -np.inf if V > 1 else 0.0
    tg = g.integers(0, V, T).astype(np.int32)
    tg[-1] = -1  # ignored
    if V > 1 and tg[0] == V // 2:
        tg[0] = 0
    t = dup(fhp, x, T, V)
    loss = tb.CrossEntropyForward(t, tg, t, T, V, -1)
    z = x.astype(np.float64)
    p = np.exp(z - z.max(1, keepdims=True))
    s = p.sum(1, keepdims=True)
    p /= s
    on = tg >= 0
    nll = np.log(s[:, 0]) + z.max(1) - z[np.arange(T), np.maximum(tg, 0)]
    assert abs(loss - nll[on].mean()) <= 2.0 ** -24 * 32 * np.abs(nll[on]).mean() + 1e-6
    tb.EnsureHostCurrent(t)
    got = t.Data.reshape(T, V).astype(np.float64)
    assert np.all(np.abs(got - p) <= 2.0 ** -24 * (24 + V / 1024) * p + 2.0 ** -22 * p * np.abs(np.where(p > 0, z, 0)))
    tb.CrossEntropyBackward(t, tg, t, T, V, -1)
    tb.EnsureHostCurrent(t)
    one = np.zeros((T, V))
    one[np.arange(T)[on], tg[on]] = 1
    want = np.where(on[:, None], got - one, 0) / on.sum()
    assert np.all(np.abs(t.Data.reshape(T, V) - want) <= 2.0 ** -23 * (got + one) / on.sum())


@pytest.mark.gpu
@pytest.mark.parametrize("batch,T,H,hd,pad", [(1, 1, 1, 1, 0), (2, 5, 3, 6, 2), (3, 17, 2, 64, 0), (1, 300, 4, 20, 1),
                                              (2, 9, 5, 8, 4), (701, 1, 3, 8, 0), (40, 1, 5, 7, 3), (30000, 1, 3, 2, 0),
                                              (5, 4, 3, 256, 4), (3, 129, 3, 4, 0), (2, 256, 2, 1, 0), (2, 257, 2, 1, 0)])
def test_head_packing_widths(fhp, tb, batch, T, H, hd, pad):
    """Head packing in both directions, by 16-byte and by single loads (odd widths and offsets), exactly."""
    d = H * hd
    src = np.random.default_rng(T + hd).standard_normal((batch, T, d + 2 * pad)).astype(np.float32)
    want = src[:, :, pad:pad + d].reshape(batch, T, H, hd).transpose(0, 2, 1, 3)
    out = fhp.Tensor(batch * H * T, hd)
    tb.PackHeads(dup(fhp, src, batch * T, d + 2 * pad), out, batch, T, H, hd, pad)
    back = dup(fhp, 0 * src - 1, batch * T, d + 2 * pad)
    tb.UnpackHeads(out, back, batch, T, H, hd, pad)
    tb.EnsureHostCurrent(out)
    tb.EnsureHostCurrent(back)
    np.testing.assert_array_equal(out.Data.reshape(want.shape), want)
    full = -np.ones_like(src)
    full[:, :, pad:pad + d] = src[:, :, pad:pad + d]
    np.testing.assert_array_equal(back.Data.reshape(src.shape), full)


@pytest.mark.gpu
@pytest.mark.parametrize("n,D,vocab", [(1, 3, 5), (255, 64, 7), (257, 300, 2), (2048, 40, 1000), (8192, 8, 50),
                                       (8193, 8, 50)])
def test_embedding_backward_repeated_ids(fhp, tb, n, D, vocab):
    """Every position of a repeated id, in ascending order: the sums of a sequential float32 loop, exactly,
    grouped on the device and (past 8192 positions) on the host."""
    g = np.random.default_rng(n)
    ids = (g.random(n) ** 3 * vocab).astype(np.int32)
    dout = g.standard_normal((n, D)).astype(np.float32)
    want = g.standard_normal((vocab, D)).astype(np.float32)
    t = dup(fhp, want, vocab, D)
    for i, r in zip(ids, dout):
        want[i] += r
    tb.EmbeddingBackward(dup(fhp, dout, n, D), ids, t, D)
    tb.EnsureHostCurrent(t)
    np.testing.assert_array_equal(t.Data.reshape(vocab, D), want)


@pytest.mark.gpu
def test_index_uploads_run_ahead(fhp, tb):
    """More uploads than there are staging areas before anything waits, of changing sizes, from one host
    array that is overwritten after each call."""
    g = np.random.default_rng(3)
    table = g.standard_normal((100, 4)).astype(np.float32)
    t = dup(fhp, table, 100, 4)
    buf = np.empty(20000, np.int32)
    outs, want = [], []
    for i in range(40):
        n = (1 + 37 * i) if i % 7 else 20000
        ids = buf[:n]
        ids[:] = g.integers(0, 100, n)
        outs.append(fhp.Tensor(n, 4))
        want.append(table[ids])
        tb.EmbeddingForward(t, ids, outs[-1], 4)
    for o, w in zip(outs, want):
        tb.EnsureHostCurrent(o)
        np.testing.assert_array_equal(o.Data.reshape(w.shape), w)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(6, 12), (8, 12), (6, 15)])
def test_unpack_qkv_zeroes_what_it_does_not_fill(fhp, tb, rows, cols):
    """dst of exactly the three slices, with rows past them, and with wider rows: zeros around the slices."""
    g = np.random.default_rng(cols)
    B, T, H, hd = 2, 3, 2, 2
    qkv = [dup(fhp, g.standard_normal((B * H * T, hd)), B * H * T, hd) for _ in range(3)]
    dst = dup(fhp, np.full((rows, cols), 5.0), rows, cols)
    tb.UnpackQkvHeads(*qkv, dst, B, T, H, hd)
    tb.EnsureHostCurrent(dst)
    want = np.zeros((rows, cols), np.float32)
    for i, t in enumerate(qkv):
        want[:B * T, 4 * i:4 * i + 4] = t.Data.reshape(B, H, T, hd).transpose(0, 2, 1, 3).reshape(B * T, 4)
    np.testing.assert_array_equal(dst.Data.reshape(rows, cols), want)


@pytest.mark.gpu
def test_unpack_qkv_zeroes_before_calls_out_of_the_ordinary(fhp, tb):
    """dst zeroed where q is dst itself (its slice is then of zeros), and before sizes that are refused."""
    g = np.random.default_rng(3)
    B, T, H, hd = 2, 3, 2, 2
    k, v = (dup(fhp, g.standard_normal((B * H * T, hd)), B * H * T, hd) for _ in range(2))
    dst = dup(fhp, np.full((B * T, 12), 5.0), B * T, 12)
    tb.Scale(dst, 1.0)
    tb.UnpackQkvHeads(dst, k, v, dst, B, T, H, hd)
    tb.EnsureHostCurrent(dst)
    want = np.zeros((B * T, 12), np.float32)
    for i, t in ((1, k), (2, v)):
        want[:, 4 * i:4 * i + 4] = t.Data.reshape(B, H, T, hd).transpose(0, 2, 1, 3).reshape(B * T, 4)
    np.testing.assert_array_equal(dst.Data.reshape(B * T, 12), want)
    dst = dup(fhp, np.full((B * T, 12), 5.0), B * T, 12)
    with pytest.raises(Exception, match="head slices"):
        tb.UnpackQkvHeads(k, k, v, dst, -B, -T, H, hd)
    tb.EnsureHostCurrent(dst)
    assert np.all(dst.Data == 0)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 4, 1023, 1024, 100001])
def test_adamw_lengths(fhp, tb, n):
    """Lengths around the 16-byte groups: every element stepped once, against float64 (a few roundings)."""
    g = np.random.default_rng(n)
    w, gr, m = (g.standard_normal((3, n)) * 0.1).astype(np.float32)
    v = (g.random(n) * 1e-2 + 1e-4).astype(np.float32)
    t = [dup(fhp, a, 1, n) for a in (w, gr, m, v)]
    tb.AdamWStep(*t, 1e-2, 0.9, 0.99, 1e-8, 0.1, 3)
    for x in t:
        tb.EnsureHostCurrent(x)
    f = lambda x: float(np.float32(x))  # noqa: E731 - fp32 hyperparameters
    b1, b2, lr, wd = f(0.9), f(0.99), f(1e-2), f(0.1)
    m64 = b1 * m.astype(np.float64) + (1 - b1) * gr
    v64 = b2 * v.astype(np.float64) + (1 - b2) * gr.astype(np.float64) ** 2
    w64 = w.astype(np.float64) * (1 - lr * wd)
    up = lr * (m64 / (1 - b1 ** 3)) / (np.sqrt(v64 / (1 - b2 ** 3)) + f(1e-8))
    ulp = 2.0 ** -24
    assert np.all(np.abs(t[2].Data - m64) <= 8 * ulp * (np.abs(m) + np.abs(gr)))
    assert np.all(np.abs(t[3].Data - v64) <= 8 * ulp * (v + gr ** 2))
    # the bias corrections 1 - b^3 lose up to 4 bits in fp32
    assert np.all(np.abs(t[0].Data - (w64 - up)) <= 8 * ulp * np.abs(w) + 256 * ulp * (np.abs(up) + lr))


def _gelu64(x):
    """GELU (tanh form) and its derivative in float64; 1 + tanh u as 2 / (1 + e^-2u), which keeps the tail."""
    x = x.astype(np.float64)
    c = np.sqrt(2 / np.pi)
    g = 1 / (1 + np.exp(-2 * c * (x + 0.044715 * x ** 3)))
    return x * g, g + 2 * x * g * (1 - g) * c * (1 + 3 * 0.044715 * x * x)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 4, 1023, 1028, 300001])
@pytest.mark.parametrize("offset", [0, 1])
def test_elementwise_lengths_and_alignment(fhp, tb, n, offset):
    """Lengths around the 16-byte groups, pointers on and off 16 bytes: every element once, none past the end.

    GELU's gate is 1 / (1 + e^-2u): a relative error of e^-2u is that of 2u (4 roundings of up to 2|u| < 14 for
    |x| < 4) and a few ulp of exp, add and divide."""
    import ctypes
    from forge_hip import _native as N
    g = np.random.default_rng(n)
    x, d = np.clip(g.standard_normal((2, n + 2)), -4, 4).astype(np.float32)
    t = {k: dup(fhp, a, 1, n + 2) for k, a in dict(x=x, d=d, f=x * 0 + 7, b=x * 0 + 7, a=x).items()}
    at = {k: ctypes.c_void_p(tb._write(v, preserve=True).value + 4 * offset) for k, v in t.items()}
    L, ctx = N.lib(), tb._ctx
    N.check(L.fh_op_gelu_forward(ctx, at["x"], at["f"], n))
    N.check(L.fh_op_gelu_backward(ctx, at["d"], at["x"], at["b"], n))
    N.check(L.fh_op_add_in_place(ctx, at["a"], at["d"], n))
    for v in t.values():
        tb.EnsureHostCurrent(v)
    s = slice(offset, offset + n)
    f64, b64 = _gelu64(x[s])
    ulp = 2.0 ** -24
    assert np.all(np.abs(t["f"].Data[s] - f64) <= 80 * ulp * np.abs(f64) + 1e-30)
    # the derivative's terms reach 1.2 each and cancel
    assert np.all(np.abs(t["b"].Data[s] - d[s] * b64) <= 80 * ulp * np.abs(d[s]) * 1.2 + 1e-30)
    np.testing.assert_array_equal(t["a"].Data[s], x[s] + d[s])
    rest = np.r_[0:offset, offset + n:n + 2]
    assert np.all(t["f"].Data[rest] == 7) and np.all(t["b"].Data[rest] == 7)
    np.testing.assert_array_equal(t["a"].Data[rest], x[rest])


@pytest.mark.gpu
def test_gelu_of_infinities_and_nan(fhp, oracle, tb):
    """What 0.5 x (1 + tanh u) gives: NaN at -inf and NaN, inf at inf, signed zeros of the tails."""
    x = np.array([-np.inf, np.inf, np.nan, -100, 100, -1e15, 1e15, 0.0, -0.0], np.float32)
    xt, out, dx = dup(fhp, x, 1, 9), fhp.Tensor(1, 9), fhp.Tensor(1, 9)
    tb.GeluForward(xt, out)
    tb.GeluBackward(dup(fhp, np.ones(9, np.float32), 1, 9), xt, dx)
    tb.EnsureHostCurrent(out)
    tb.EnsureHostCurrent(dx)
    np.testing.assert_array_equal(out.Data, np.array([np.nan, np.inf, np.nan, 0, 100, 0, 1e15, 0, 0], np.float32))
    np.testing.assert_array_equal(dx.Data, np.array([np.nan, np.nan, np.nan, 0, 1, 0, 1, 0.5, 0.5], np.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 4), (5, 1023), (2, 1028), (9000, 8), (1100000, 1), (300, 31),
                                       (70001, 40), (5, 256), (5, 260), (100, 129)])
def test_add_bias_shapes(fhp, tb, rows, cols):
    """Rows by 16 bytes and by 4, a last strip in part, more rows than block rows: one addition each."""
    g = np.random.default_rng(rows + cols)
    y, b = g.standard_normal((rows, cols)).astype(np.float32), g.standard_normal(cols).astype(np.float32)
    t = dup(fhp, y, rows, cols)
    tb.AddBias(t, dup(fhp, b, cols), rows, cols)
    tb.EnsureHostCurrent(t)
    np.testing.assert_array_equal(t.Data.reshape(rows, cols), y + b)


@pytest.mark.gpu
@pytest.mark.parametrize("hd,extra", [(8, 0), (8, 4), (8, 3), (6, 0)])
def test_pack_qkv_in_one_launch(fhp, tb, hd, extra):
    """Widths by 16 bytes and not, rows wider than the three slices, and one tensor for two of them
    (the later slice stays, as in three packs)."""
    g = np.random.default_rng(hd + extra)
    B, T, H = 2, 37, 3
    d = H * hd
    src = g.standard_normal((B * T, 3 * d + extra)).astype(np.float32)
    want = [src[:, i * d:(i + 1) * d].reshape(B, T, H, hd).transpose(0, 2, 1, 3).reshape(-1, hd) for i in range(3)]
    ts = dup(fhp, src, B * T, 3 * d + extra)
    q, k, v = (fhp.Tensor(B * H * T, hd) for _ in range(3))
    tb.PackQkvHeads(ts, q, k, v, B, T, H, hd)
    for t, w in zip((q, k, v), want):
        tb.EnsureHostCurrent(t)
        np.testing.assert_array_equal(t.Data.reshape(w.shape), w)
    back = fhp.Tensor(B * T, 3 * d + extra)
    tb.UnpackQkvHeads(q, k, v, back, B, T, H, hd)
    tb.EnsureHostCurrent(back)
    np.testing.assert_array_equal(back.Data.reshape(src.shape)[:, :3 * d], src[:, :3 * d])
    assert np.all(back.Data.reshape(src.shape)[:, 3 * d:] == 0)
    tb.PackQkvHeads(ts, q, q, v, B, T, H, hd)
    tb.EnsureHostCurrent(q)
    np.testing.assert_array_equal(q.Data.reshape(want[1].shape), want[1])


def _pace(tb, f, ref):
    """Time of f over that of ref, each the best of several runs of 40 calls."""
    import time

    def best(g):
        times = []
        for _ in range(6):
            t = time.perf_counter()
            for _ in range(40):
                g()
            wait()
            times.append(time.perf_counter() - t)
        return min(times)

    import forge_hip
    one = forge_hip.Tensor(1)
    wait = lambda: tb.SumSquares(one)  # noqa: E731 - the next call that waits for the device
    best(ref)
    return best(f) / best(ref)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(1 << 20, 1), (1 << 20, 8), (1 << 18, 31)])
def test_add_bias_of_narrow_rows_keeps_pace(fhp, tb, rows, cols):
    """Against AddInPlace of as many elements, which moves half as much again: at most three times its time."""
    y, src, b = (dup(fhp, np.ones(n), *s) for n, s in ((rows * cols, (rows, cols)), (rows * cols, (rows, cols)),
                                                      (cols, (cols,))))
    assert _pace(tb, lambda: tb.AddBias(y, b, rows, cols), lambda: tb.AddInPlace(src, y)) < 3


@pytest.mark.gpu
@pytest.mark.parametrize("batch,T,H,hd", [(16384, 1, 4, 8), (4096, 1, 12, 64), (2000, 3, 8, 5)])
def test_head_packing_of_short_slots_keeps_pace(fhp, tb, batch, T, H, hd):
    """Against Copy of the packed tensor, which moves as much: at most three times its time."""
    n = batch * T * H * hd
    src = dup(fhp, np.ones(n), batch * T, H * hd)
    out, cp = fhp.Tensor(batch * H * T, hd), fhp.Tensor(batch * H * T, hd)
    assert _pace(tb, lambda: tb.PackHeads(src, out, batch, T, H, hd, 0), lambda: tb.Copy(out, cp)) < 3


@pytest.mark.gpu
@pytest.mark.parametrize("T,V", [(65536, 10), (65536, 100)])
def test_cross_entropy_of_narrow_vocabularies_keeps_pace(fhp, tb, T, V):
    """Forward (the loss summed on the device by one block) and backward against Copy of the logits, with the
    targets' upload in both: at most five times its time (1024 threads to a position: seven and more)."""
    lg, pr = dup(fhp, np.zeros(T * V), T, V), fhp.Tensor(T, V)
    tg = np.zeros(T, np.int32)
    tab, up = dup(fhp, np.zeros(4), 4, 1), fhp.Tensor(T, 1)

    def ref():
        tb.EmbeddingForward(tab, tg, up, 1)  # the same upload
        tb.Copy(lg, pr)

    tb.BeginLossAccumulation()
    fw = _pace(tb, lambda: tb.CrossEntropyForward(lg, tg, pr, T, V, -1), ref)
    tb.EndLossAccumulation()
    bw = _pace(tb, lambda: tb.CrossEntropyBackward(pr, tg, lg, T, V, -1), ref)
    print(fw, bw)
    assert fw < 5 and bw < 5


@pytest.mark.gpu
def test_cross_entropy_of_millions_of_positions(fhp, tb):
    """2^22 positions and more, narrow and (in place on 17 GB) wider than a wave's registers: uniform rows."""
    from forge_hip import _native as N
    import ctypes
    for T, V in ((5000001, 3), ((1 << 22) + 1, 1025)):
        buf = fhp.DeviceBuffer(tb.backend, 4 * T * V)
        N.check(N.lib().fh_op_zero(tb._ctx, buf.ptr, T * V))
        tg = np.zeros(T, np.int32)
        loss = ctypes.c_float()
        N.check(N.lib().fh_op_cross_entropy_forward(tb._ctx, buf.ptr, tg.ctypes.data, buf.ptr, T, V, -1,
                                                    ctypes.byref(loss)))
        assert abs(loss.value - np.log(V)) < 1e-5
        N.check(N.lib().fh_op_cross_entropy_backward(tb._ctx, buf.ptr, tg.ctypes.data, buf.ptr, T, V, -1))
        for row in (0, T // 2, T - 1):
            got = np.empty(V, np.float32)
            N.check(N.lib().fh_buffer_read(tb._ctx, got.ctypes.data, ctypes.c_void_p(buf.ptr.value + 4 * row * V),
                                           4 * V))
            want = np.full(V, 1 / V / T)
            want[0] -= 1 / T
            np.testing.assert_allclose(got, want, rtol=1e-5, atol=0)
        buf.free()
