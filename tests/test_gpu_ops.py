"""GPU parity of the operators (layernorm, softmax_rows, rope_apply,
window partition, add_bcast, gemm, mha) through the C ABI against the
oracle. Data movement and exact-integer products are bit-exact; float
arithmetic is held to rel-L2 <= 2e-5 (fp32 path) or 2e-2 (bf16 path)."""
import numpy as np
import pytest

from gpu_common import rel_l2, report

pytestmark = pytest.mark.gpu

FP32_TOL = 2e-5
BF16_TOL = 2e-2


@pytest.fixture(scope="module")
def hip():
    import sam3_hip
    return sam3_hip


@pytest.fixture(scope="module")
def be(hip):
    b = hip.Backend(precision="fp32")
    yield b
    b.free()


@pytest.fixture(scope="module")
def be16(hip):
    b = hip.Backend(precision="bf16")
    yield b
    b.free()


def model(hip, be, E=128):
    return hip.Model(be, embed=E, heads=E // 64)


def rng(seed):
    return np.random.default_rng(seed)


@pytest.mark.parametrize("C", [1024, 256, 100, 3000, 3072, 4096, 4608, 64, 32, 128])
def test_layernorm(hip, be, orc, C):
    m = model(hip, be)
    g = rng(C)
    X = (2 * g.standard_normal((37, C)) + 0.5).astype(np.float32)
    w = g.standard_normal(C).astype(np.float32)
    b = g.standard_normal(C).astype(np.float32)
    dX, dW, dB = be.upload(X), be.upload(w), be.upload(b)
    dY = be.alloc(X.nbytes)
    hip.layernorm(m, 37, C, dX, dY, dW, dB, 1e-5, hip.ACT_NONE)
    got = be.read(dY).reshape(37, C)
    assert report("layernorm C=%d" % C, got, orc.layernorm(X, w, b)) <= FP32_TOL
    # In place (Y aliases X), with GELU.
    hip.layernorm(m, 37, C, dX, dX, dW, dB, 1e-5, hip.ACT_GELU)
    got = be.read(dX).reshape(37, C)
    assert rel_l2(got, orc.layernorm(X, w, b, act=orc.ACT_GELU)) <= FP32_TOL


@pytest.mark.parametrize("L", [576, 5184, 40])
def test_softmax_rows(hip, be, orc, L):
    m = model(hip, be)
    S = (3 * rng(L).standard_normal((20, L))).astype(np.float32)
    dS = be.upload(S)
    hip.softmax_rows(m, dS, 20, L)
    got = be.read(dS).reshape(20, L)
    assert report("softmax_rows L=%d" % L, got, orc.softmax_rows(S)) <= FP32_TOL


def test_rope_apply_bit_exact(hip, be, orc):
    E, side = 256, 24
    m = model(hip, be, E)
    table = orc.rope_table(side)
    qkv = rng(0).standard_normal((2 * side * side, 3 * E)).astype(np.float32)
    m.m.qkv = be.upload(qkv)
    hip.rope_apply(m, be.upload(table), qkv.shape[0], side * side)
    got = be.read(m.m.qkv).reshape(qkv.shape)
    np.testing.assert_array_equal(got, orc.rope_apply(qkv, E, 64, side * side,
                                                      table))


@pytest.mark.parametrize("H,ws", [(72, 24), (10, 4)])
def test_window_partition_bit_exact(hip, be, orc, H, ws):
    C = 64
    m = model(hip, be)
    nwx = -(-H // ws)
    X = rng(H).standard_normal((H * H, C)).astype(np.float32)
    dX = be.upload(X)
    dW = be.alloc(nwx * nwx * ws * ws * C * 4)
    hip.window_partition(m, dX, dW, H, C, ws, nwx)
    Xw = be.read(dW).reshape(-1, C)
    np.testing.assert_array_equal(Xw, orc.window_partition(X, H, H, C, ws))
    Y = rng(H + 1).standard_normal((H * H, C)).astype(np.float32)
    dY = be.upload(Y)
    hip.window_unpartition_add(m, dY, dW, H, C, ws, nwx)
    np.testing.assert_array_equal(be.read(dY).reshape(-1, C),
                                  orc.window_unpartition_add(Y, Xw, H, H, C, ws))


def test_add_bcast_bit_exact(hip, be, orc):
    m = model(hip, be)
    a = rng(1).standard_normal(5184 * 3).astype(np.float32)
    b = rng(2).standard_normal(3 * 64).astype(np.float32)
    da, db = be.upload(a), be.upload(b)
    hip.add_bcast(m, da, da, db, a.size, b.size)
    np.testing.assert_array_equal(be.read(da), orc.add_bcast(a, b, b.size))


def _gemm_case(hip, be, orc, M, N, K, transb, nb=4, nb1=2, ints=False,
               act=0, residual=True, seed=0, bias=True):
    """Batched GEMM with padded leading dims and offsets on the GPU and in
    the oracle (sequential arithmetic); returns (gpu, oracle)."""
    m = model(hip, be)
    g = rng(seed)
    draw = (lambda n: g.integers(-3, 4, n).astype(np.float32)) if ints else \
        (lambda n: g.standard_normal(n).astype(np.float32))
    lda, ldc = K + 4, N + 4
    ldb = K + 8 if transb else N + 8
    brows = N if transb else K
    sa1, sb1, sc1 = M * lda, brows * ldb, M * ldc
    A = draw(8 + nb * sa1)
    B = draw(16 + nb * sb1)
    C0 = draw(4 + nb * sc1)
    bv = draw(N) if bias else None
    A_, B_, C_ = (be.upload(A), be.upload(B), be.upload(C0))
    bias_d = be.upload(bv) if bias else None
    hip.gemm(m, M, N, K, hip.bmat(A_, 8, lda, sa1 * nb1, sa1),
             hip.bmat(B_, 16, ldb, sb1 * nb1, sb1), transb,
             hip.bmat(C_, 4, ldc, sc1 * nb1, sc1), nb, nb1, bias_d,
             C_ if residual else None, 4, 0.5, act)
    got = be.read(C_)
    want = C0.copy()
    orc.gemm(orc.GEMM_SEQ, M, N, K, A, 8, lda, sa1 * nb1, sa1, B, 16, ldb,
             sb1 * nb1, sb1, transb, want, 4, ldc, sc1 * nb1, sc1, nb, nb1, bv,
             want if residual else None, 4, 0.5, act)
    return got, want


@pytest.mark.parametrize("transb", [0, 1])
@pytest.mark.parametrize("M,N,K", [(130, 70, 40), (64, 64, 64), (5, 3, 7)])
def test_gemm_exact_integers(hip, be, orc, transb, M, N, K):
    got, want = _gemm_case(hip, be, orc, M, N, K, transb, ints=True, act=2)
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("transb", [0, 1])
@pytest.mark.parametrize("act", [0, 1])
def test_gemm_f32(hip, be, orc, transb, act):
    got, want = _gemm_case(hip, be, orc, 200, 150, 300, transb, act=act, seed=3)
    assert report("gemm f32 transb=%d act=%d" % (transb, act), got, want) <= FP32_TOL


@pytest.mark.parametrize("transb", [0, 1])
def test_gemm_bf16(hip, be16, orc, transb):
    got, want = _gemm_case(hip, be16, orc, 200, 150, 300, transb, seed=4)
    assert report("gemm bf16 transb=%d" % transb, got, want) <= BF16_TOL


def to_bf16(x):
    """float32 -> bf16 bits, round to nearest even."""
    u = np.ascontiguousarray(x, np.float32).view(np.uint32)
    return ((u + ((u >> 16) & 1) + 0x7FFF) >> 16).astype(np.uint16)


def from_bf16(u):
    return (np.asarray(u, np.uint16).astype(np.uint32) << 16).view(np.float32)


@pytest.mark.parametrize("M,N,K,act,res,cbf", [
    (5184, 3072, 1024, 0, False, False),   # QKV projection
    (5184, 1024, 1024, 0, True, False),    # attention projection + residual
    (5184, 4096, 1024, 1, False, True),    # MLP fc1, GELU, bf16 hidden
    (5184, 1024, 4096, 0, True, False),    # MLP fc2 + residual
    (5000, 3000, 1024, 0, False, False),   # 256 x 256 tiles, ragged edges
    (5100, 3968, 1024, 1, False, True),    # 192 x 256 tiles, ragged edges
    (2100, 1000, 2048, 2, False, False),   # 192 x 128 tiles, ragged edges
    (2100, 1000, 2048, 1, False, True),    # the same, bf16 C
    (2100, 1000, 2048, 0, True, True),     # 128 x 64 tiles, bf16 C and residual
    (5184, 3072, 2048, 0, True, False),    # residual, long K: 256 x 256 tiles of k_gemm_nt
    (5184, 3072, 2048, 1, True, True),     # the same with GELU and bf16 C
    (3000, 700, 2048, 0, True, False),     # 128 x 64 tiles, residual, ragged
    (2500, 900, 1024, 1, True, False),     # GELU + residual, ragged
    (300, 200, 128, 1, True, False),       # ragged tiles on both sides
    (257, 129, 192, 2, True, True),
    (1, 1, 64, 0, False, False),
])
def test_gemm_nt_bf16(hip, be16, orc, M, N, K, act, res, cbf):
    """bf16 activations x bf16 weight rows (the NT kernel): the oracle's
    linear on the same bf16 values in float, sampled rows at full size."""
    m = model(hip, be16)
    g = rng(M + N + K)
    A = to_bf16(g.standard_normal((M, K), dtype=np.float32))
    W = to_bf16(g.uniform(-0.06, 0.06, (N, K)).astype(np.float32))
    bias = g.standard_normal(N, dtype=np.float32)
    C0 = g.standard_normal((M, N), dtype=np.float32)
    if cbf:
        C0 = from_bf16(to_bf16(C0))
    dA, dW = be16.upload_typed(A, hip.BF16), be16.upload_typed(W, hip.BF16)
    db = be16.upload(bias)
    dC = be16.upload_typed(to_bf16(C0), hip.BF16) if cbf else be16.upload(C0)
    hip.prof_reset()
    be16._b.profile = 1
    hip.linear(m, M, K, N, dA, 0, dW, db, dC, 0, act, int(res))
    be16._b.profile = 0
    assert "gemm_nt_bf16" in [r[0] for r in hip.prof_table()]
    got = be16.read(dC)
    got = (from_bf16(got) if cbf else got).reshape(M, N)
    rows = np.sort(rng(1).choice(M, min(M, 96), replace=False))
    want = orc.linear(from_bf16(A[rows]), from_bf16(W), bias, act=act,
                      cpu=False)
    if res:
        want = want + C0[rows]
    if cbf:
        want = from_bf16(to_bf16(want))
    tol = 1e-2 if cbf else 1e-5
    assert report("gemm_nt bf16 %dx%dx%d act=%d res=%d cbf=%d" %
                  (M, N, K, act, res, cbf), got[rows], want) <= tol


def test_profile_in_flow(hip, be16):
    """profile 2 brackets each launch with events without waiting: the
    results are those of an unprofiled run, and hipb_finish adds each
    launch's time to the per-kernel table (one entry per call)."""
    m = model(hip, be16)
    g = rng(5)
    M, N, K = 512, 384, 256
    A = be16.upload_typed(to_bf16(g.standard_normal((M, K), dtype=np.float32)), hip.BF16)
    W = be16.upload_typed(to_bf16(g.uniform(-0.06, 0.06, (N, K)).astype(np.float32)), hip.BF16)
    b = be16.upload(g.standard_normal(N, dtype=np.float32))
    C = be16.alloc(M * N * 4)
    hip.linear(m, M, K, N, A, 0, W, b, C, 0, 0, 0)
    plain = be16.read(C)
    hip.prof_reset()
    be16._b.profile = 2
    for _ in range(3):
        hip.linear(m, M, K, N, A, 0, W, b, C, 0, 0, 0)
    be16.finish()
    be16._b.profile = 0
    tab = {r[0]: r for r in hip.prof_table()}
    assert np.array_equal(be16.read(C), plain)
    row = tab["gemm_nt_bf16"]
    assert row[4] == 3 and row[1] > 0.0 and row[3] == 3 * 2.0 * M * N * K
    for d in (A, W, b, C):
        be16.release(d)


@pytest.mark.parametrize("M,N,K,act,res,cbf", [
    (5184, 4096, 1024, 1, False, True),    # fc1, GELU, bf16 hidden
    (5184, 1024, 4096, 0, True, False),    # fc2 + residual
])
def test_gemm_nt_every_row(hip, be16, orc, M, N, K, act, res, cbf):
    """The MLP's NT GEMMs at full size: every row against the oracle, and
    a second launch gives the same bits."""
    m = model(hip, be16)
    g = rng(M + 2 * N + K)
    A = to_bf16(g.standard_normal((M, K), dtype=np.float32))
    W = to_bf16(g.uniform(-0.06, 0.06, (N, K)).astype(np.float32))
    bias = g.standard_normal(N, dtype=np.float32)
    C0 = g.standard_normal((M, N), dtype=np.float32)
    if cbf:
        C0 = from_bf16(to_bf16(C0))
    dA, dW = be16.upload_typed(A, hip.BF16), be16.upload_typed(W, hip.BF16)
    db = be16.upload(bias)

    def run():
        dC = be16.upload_typed(to_bf16(C0), hip.BF16) if cbf else be16.upload(C0)
        hip.linear(m, M, K, N, dA, 0, dW, db, dC, 0, act, int(res))
        got = be16.read(dC)
        be16.release(dC)
        return (from_bf16(got) if cbf else got).reshape(M, N)

    print("gemm_nt every row %dx%dx%d" % (M, N, K), flush=True)
    first, second = run(), run()
    assert np.array_equal(first, second)
    want = orc.linear(from_bf16(A), from_bf16(W), bias, act=act, cpu=False)
    if res:
        want = want + C0
    if cbf:
        want = from_bf16(to_bf16(want))
    tol = 1e-2 if cbf else 1e-5
    assert report("gemm_nt every row %dx%dx%d" % (M, N, K), first, want) <= tol


def test_linear_fp16_weights(hip, orc):
    be = hip.Backend(precision="fp16")
    try:
        m = model(hip, be)
        g = rng(5)
        X = g.standard_normal((77, 96)).astype(np.float32)
        W = g.standard_normal((48, 96)).astype(np.float32)
        b = g.standard_normal(48).astype(np.float32)
        dW = be.upload_weight(W)
        assert dW.contents.dtype == hip.F16
        dX, db = be.upload(X), be.upload(b)
        dY = be.alloc(77 * 48 * 4)
        hip.linear(m, 77, 96, 48, dX, 0, dW, db, dY, 0, hip.ACT_RELU, 0)
        Wh = W.astype(np.float16).astype(np.float32)
        want = orc.linear(X, Wh, b, act=orc.ACT_RELU, cpu=False)
        assert report("linear fp16 weights", be.read(dY).reshape(77, 48),
                      want) <= FP32_TOL
    finally:
        be.free()


def test_gemm_operand_out_of_bounds_is_fatal(hip, be):
    m = model(hip, be)
    A = be.alloc(10 * 10 * 4)
    with pytest.raises(hip.Sam3HipError, match="operand A reaches element"):
        hip.gemm(m, 11, 10, 10, hip.mat(A, 0, 10), hip.mat(A, 0, 10), 1,
                 hip.mat(A, 0, 10), 1, 1)


# ---------------------------------------------------------------- decoder

def _dec(seed, P, Nq, Nk, dint, shared_k=False, shared_q=False):
    g = rng(seed)
    q = g.standard_normal(((1 if shared_q else P) * Nq, dint)).astype(np.float32)
    k = g.standard_normal(((1 if shared_k else P) * Nk, dint)).astype(np.float32)
    v = g.standard_normal(((1 if shared_k else P) * Nk, dint)).astype(np.float32)
    return (q, 0 if shared_q else Nq * dint, k, 0 if shared_k else Nk * dint,
            v, 0 if shared_k else Nk * dint)


@pytest.mark.parametrize("P,Nq,Nk,dint,shk,shq", [
    (64, 7, 4096, 128, False, False),    # token -> image, per-prompt keys
    (64, 8, 5184, 128, True, False),     # token -> image, shared keys
    (3, 9, 300, 128, False, False),      # more than 8 queries, short keys
    (64, 4096, 7, 128, False, False),    # image -> token, per-prompt queries
    (16, 5184, 8, 128, False, True),     # image -> token, shared queries
    (64, 8, 8, 256, False, False),       # token self-attention, c = 32
    (8, 2048, 65, 128, False, False),    # many keys, key range not split
    (2, 3, 261, 128, False, False),      # many keys, ragged last step
    (3, 20, 40, 128, False, False),      # 9..64 keys, generic few-keys
    (5, 17, 1, 128, False, False),       # one key: O = V
])
def test_mha(hip, be, orc, P, Nq, Nk, dint, shk, shq):
    m = model(hip, be)
    q, sq, k, sk, v, sv = _dec(P + Nq + Nk, P, Nq, Nk, dint, shk, shq)
    dq, dk, dv = be.upload(q), be.upload(k), be.upload(v)
    do = be.alloc(P * Nq * dint * 4)
    hip.mha(m, P, Nq, Nk, dint, dq, sq, dk, sk, dv, sv, do)
    got = be.read(do).reshape(P * Nq, dint)
    want = orc.mha(P, Nq, Nk, dint, q, sq, k, sk, v, sv)
    assert report("mha P=%d Nq=%d Nk=%d dint=%d" % (P, Nq, Nk, dint), got,
                  want) <= FP32_TOL
    for d in (dq, dk, dv, do):
        be.release(d)


def test_mha_unaligned_prompt_strides(hip, be, orc):
    """Per-prompt strides that are not a multiple of 4 floats take the
    generic few-keys kernel; with many keys they are a fatal error."""
    m = model(hip, be)
    P, Nq, Nk, dint = 3, 11, 7, 128
    g = rng(5)
    sq, sk = Nq * dint + 2, Nk * dint + 1
    q = g.standard_normal(P * sq).astype(np.float32)
    k = g.standard_normal(P * sk).astype(np.float32)
    v = g.standard_normal(P * sk).astype(np.float32)
    dq, dk, dv = be.upload(q), be.upload(k), be.upload(v)
    do = be.alloc(P * Nq * dint * 4)
    hip.mha(m, P, Nq, Nk, dint, dq, sq, dk, sk, dv, sk, do)
    got = be.read(do).reshape(P * Nq, dint)
    want = orc.mha(P, Nq, Nk, dint, q, sq, k, sk, v, sk)
    assert report("mha unaligned strides", got, want) <= FP32_TOL
    d = be.alloc(P * 100 * dint * 4 + 64)
    with pytest.raises(hip.Sam3HipError, match="multiples of 4"):
        hip.mha(m, P, 4, 100, dint, d, 0, d, 100 * dint + 2, d, 0, d)
    for x in (dq, dk, dv, do, d):
        be.release(x)


def test_mha_rejects_wide_heads_with_many_keys(hip, be):
    m = model(hip, be)
    d = be.alloc(100 * 256 * 4)
    with pytest.raises(hip.Sam3HipError, match="mha: unsupported shape"):
        hip.mha(m, 1, 4, 100, 256, d, 0, d, 0, d, 0, d)


@pytest.fixture(scope="module")
def be_half(hip):
    b = hip.Backend(precision="fp16")
    yield b
    b.free()


@pytest.mark.parametrize("M,N,K,transb", [
    (1, 1, 4, 1), (8, 256, 2048, 1), (33, 70, 300, 1), (32, 4096, 520, 1),  # f32 MFMA
    (5184, 128, 256, 1), (700, 1024, 68, 1),      # split while staged, 64 x 64 tiles
    (33000, 100, 36, 1), (16500, 256, 256, 0),    # 128 x 64 tiles; K x N operand
    (2500, 1030, 1024, 1),                        # packed, 64 x 64 tiles
    (5184, 1024, 260, 1), (5100, 4096, 132, 1),   # 128 x 64 and 256 x 128
    (5184, 3072, 512, 1), (9000, 1000, 516, 0),   # 256 x 256; K x N operand
    (4600, 2050, 64, 1),
])
@pytest.mark.parametrize("half", [False, True])
def test_gemm_split_paths(hip, be, be_half, M, N, K, transb, half):
    """The exact path's product kernels (f32 MFMA over split K, operands split
    while staged, operands packed) at ragged sizes against float64, float and
    half B, with bias and residual. A sum of K products of N(0, 1) values
    rounded at most K times to 2^-24 of its running size, errors of random
    sign: below sqrt(K) 2^-24 of the result (and one rounding for the
    epilogue)."""
    b = be_half if half else be
    m = model(hip, b)
    g = rng(M + N + K)
    A = g.standard_normal((M, K), dtype=np.float32)
    B = (g.standard_normal((N, K) if transb else (K, N), dtype=np.float32) * 0.05)
    if half:
        B = B.astype(np.float16).astype(np.float32)
    bias = g.standard_normal(N, dtype=np.float32)
    C0 = g.standard_normal((M, N), dtype=np.float32)
    dA, dB, dv, dC = b.upload(A), b.upload_weight(B), b.upload(bias), b.upload(C0)
    hip.gemm(m, M, N, K, hip.mat(dA, 0, K), hip.mat(dB, 0, K if transb else N),
             transb, hip.mat(dC, 0, N), 1, 1, dv, dC, 0, 0.5, hip.ACT_RELU)
    got = b.read(dC).reshape(M, N)
    rows = np.unique(np.concatenate([np.arange(min(M, 40)), [M - 1],
                                     g.integers(0, M, 60)]))
    p = A[rows].astype(np.float64) @ (B.T if transb else B).astype(np.float64)
    want = np.maximum(0.5 * p + bias, 0) + C0[rows]
    assert rel_l2(got[rows], want) <= (np.sqrt(K) + 2) * 2.0 ** -24
    for x in (dA, dB, dv, dC):
        b.release(x)


def test_gemm_split_packed_bits(hip, be):
    """Packing the operands first or splitting them while they are staged
    gives the same bits: the first 700 rows of a product that is packed, and
    the product of those rows alone, which is not."""
    m = model(hip, be)
    g = rng(7)
    A = g.standard_normal((5184, 1000), dtype=np.float32)
    B = g.standard_normal((1024, 1000), dtype=np.float32)
    dA, dB, dC = be.upload(A), be.upload(B), be.alloc(5184 * 1024 * 4)
    out = []
    for rows in (5184, 700):
        hip.linear(m, rows, 1000, 1024, dA, 0, dB, None, dC, 0)
        out.append(be.read(dC, 700 * 1024).copy())
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("M,N,K", [(700, 1024, 68), (5184, 1024, 260), (40, 64, 64)])
def test_gemm_split_non_finite(hip, be, orc, M, N, K):
    """Infinities, NaN and values that round past the largest bf16: every
    output is what the sequential float sum gives (finite rows untouched)."""
    m = model(hip, be)
    g = rng(M)
    A = g.standard_normal((M, K), dtype=np.float32)
    B = g.standard_normal((N, K), dtype=np.float32)
    A[3, 5], A[4, 6], A[5, 7] = np.inf, np.nan, np.float32(3.4e38)
    A[6, 1], A[6, 2] = np.inf, -np.inf
    B[9, 5] = 0.0
    B[11, 3] = -np.inf
    B[:, 7] = 0.25
    dA, dB, dC = be.upload(A), be.upload(B), be.alloc(M * N * 4)
    hip.gemm(m, M, N, K, hip.mat(dA, 0, K), hip.mat(dB, 0, K), 1,
             hip.mat(dC, 0, N))
    got = be.read(dC).reshape(M, N)
    want = np.zeros((16, N), np.float32)
    orc.gemm(orc.GEMM_SEQ, 16, N, K, A[:16].ravel().copy(), 0, K, 0, 0, B.ravel(), 0, K,
             0, 0, 1, want, 0, N, 0, 0, 1, 1)
    assert np.array_equal(np.isnan(got[:16]), np.isnan(want))
    assert np.array_equal(got[:16][np.isinf(want)], want[np.isinf(want)])
    fin = np.isfinite(want)
    assert np.array_equal(np.isfinite(got[:16]), fin)
    assert np.all(np.abs(got[:16][fin] - want[fin]) <= 1e-5 * np.abs(want[fin]) + 2e-4)


@pytest.mark.parametrize("M,N,K,act,abf,cbf", [
    (8, 256, 256, 0, False, False), (1, 4, 64, 1, False, False),
    (17, 33, 128, 2, True, True), (512, 256, 2048, 0, False, False),
    (512, 300, 576, 1, True, False), (40, 4000, 1088, 0, False, True),
])
def test_gemm_small_bf16(hip, be16, orc, M, N, K, act, abf, cbf):
    """The bf16 path's smallest products (16-column tiles, K over the waves),
    with bias and residual, against float64 of the bf16 operands: each element
    within one rounding of the f32 sum (K 2^-24 of the operands' magnitude)
    and, stored as bf16, one of the result (2^-9)."""
    m = model(hip, be16)
    g = rng(M + N + K + 5)
    A = g.standard_normal((M, K), dtype=np.float32)
    A16 = from_bf16(to_bf16(A))
    W = to_bf16(g.uniform(-0.06, 0.06, (N, K)).astype(np.float32))
    bias = g.standard_normal(N, dtype=np.float32)
    C0 = from_bf16(to_bf16(g.standard_normal((M, N), dtype=np.float32)))
    dA = be16.upload_typed(to_bf16(A), hip.BF16) if abf else be16.upload(A)
    dW, dv = be16.upload_typed(W, hip.BF16), be16.upload(bias)
    dC = be16.upload_typed(to_bf16(C0), hip.BF16) if cbf else be16.upload(C0)
    hip.linear(m, M, K, N, dA, 0, dW, dv, dC, 0, act, 1)
    got = be16.read_f32(dC, M * N).reshape(M, N).astype(np.float64)
    p = A16.astype(np.float64) @ from_bf16(W).T.astype(np.float64) + bias
    if act == 1:
        from scipy.special import erf
        p = 0.5 * p * (1 + erf(p / np.sqrt(2)))
    elif act == 2:
        p = np.maximum(p, 0)
    want = p + C0
    tol = K * 2.0 ** -24 * np.abs(A16).max() * 0.06 * 8 + 1e-6
    if cbf:
        tol = tol + 2.0 ** -8 * np.abs(want)
    assert np.all(np.abs(got - want) <= tol)


def us(be, call):
    """The fastest of five launches in a row, by events."""
    call()
    best = 1e9
    for _ in range(5):
        be.finish()
        be.timer_start()
        call()
        best = min(best, 1e3 * be.timer_stop())
    return best


@pytest.mark.parametrize("M,N,K,transb,nb", [(16, 16, 16, 0, 1000), (64, 64, 64, 0, 1000),
                                             (16, 64, 32, 0, 777)])
def test_gemm_many_tiny_products(hip, be, M, N, K, transb, nb):
    """A thousand products of a tile each cost at most four times one (they
    fit the chip at once), and are right."""
    m = model(hip, be)
    g = rng(M + nb)
    A = g.standard_normal((nb, M, K), dtype=np.float32)
    B = g.standard_normal((nb, K, N), dtype=np.float32)
    dA, dB, dC = be.upload(A), be.upload(B), be.alloc(nb * M * N * 4)

    def run(n):
        hip.gemm(m, M, N, K, hip.bmat(dA, 0, K, M * K, 0), hip.bmat(dB, 0, N, K * N, 0), transb,
                 hip.bmat(dC, 0, N, M * N, 0), n, 1)

    one, many = us(be, lambda: run(1)), us(be, lambda: run(nb))
    want = A.astype(np.float64) @ B.astype(np.float64)
    assert rel_l2(be.read(dC).reshape(nb, M, N), want) <= (np.sqrt(K) + 2) * 2.0 ** -24
    print("%d x %d x %d: one %.1f us, %d %.1f us" % (M, N, K, one, nb, many))
    assert many <= 4 * one


@pytest.mark.parametrize("n,K,nb", [(576, 64, 144), (196, 64, 256), (256, 128, 64)])
def test_gemm_batch_costs_what_its_size_does(hip, be, n, K, nb):
    """A batch of Q K^T sized products takes at most 1.8 times one product
    with as many operations and results, and each product's bits do not
    depend on how many the call holds."""
    m = model(hip, be)
    g = rng(n + nb)
    A = g.standard_normal((nb, n, K), dtype=np.float32)
    B = g.standard_normal((nb, n, K), dtype=np.float32)
    dA, dB, dC = be.upload(A), be.upload(B), be.alloc(nb * n * n * 4)

    def run(first, count):
        hip.gemm(m, n, n, K, hip.bmat(dA, first * n * K, K, n * K, 0),
                 hip.bmat(dB, first * n * K, K, n * K, 0), 1,
                 hip.bmat(dC, first * n * n, n, n * n, 0), count, 1)

    batch = us(be, lambda: run(0, nb))
    got = be.read(dC).reshape(nb, n, n)
    rows = g.integers(0, n, 20)
    want = A[:, rows].astype(np.float64) @ B.astype(np.float64).transpose(0, 2, 1)
    assert rel_l2(got[:, rows], want) <= (np.sqrt(K) + 2) * 2.0 ** -24
    for first in (0, 3, nb - 1):
        run(first, 1)
        assert np.array_equal(be.read(dC, n * n, off=4 * first * n * n).reshape(n, n), got[first])
    one = us(be, lambda: hip.gemm(m, nb * n, n, K, hip.mat(dA, 0, K), hip.mat(dB, 0, K), 1,
                                  hip.mat(dC, 0, n)))
    print("%d x %d x %d x %d: %.1f us, as one product %.1f us" % (nb, n, n, K, batch, one))
    assert batch <= 1.8 * one


def test_gemm_packed_row_chunks(hip, be):
    """A product whose rows are packed in two chunks (1280 rows of K = 65536
    fill the 512 MiB of pieces): rows around the seam and at the end against
    float64, with bias and residual."""
    M, N, K = 1400, 1024, 65536
    m = model(hip, be)
    g = rng(70)
    A = g.standard_normal((M, K), dtype=np.float32)
    B = g.standard_normal((N, K), dtype=np.float32)
    bias = g.standard_normal(N, dtype=np.float32)
    C0 = 100 * g.standard_normal((M, N), dtype=np.float32)
    dA, dB, dv, dC = be.upload(A), be.upload(B), be.upload(bias), be.upload(C0)
    try:
        hip.gemm(m, M, N, K, hip.mat(dA, 0, K), hip.mat(dB, 0, K), 1, hip.mat(dC, 0, N), 1, 1,
                 dv, dC, 0, 0.5)
        assert be._b.gemm_ws_bytes >= 864 << 20
        got = be.read(dC).reshape(M, N)
    finally:
        for x in (dA, dB, dv, dC):
            be.release(x)
    rows = np.array([0, 31, 1247, 1278, 1279, 1280, 1281, 1311, 1312, 1398, 1399])
    want = 0.5 * (A[rows].astype(np.float64) @ B.T.astype(np.float64)) + bias + C0[rows]
    assert rel_l2(got[rows] - C0[rows], want - C0[rows]) <= (np.sqrt(K) + 2) * 2.0 ** -24


def test_callers_capture(hip, be):
    """A large product and a large attention while the caller captures the
    stream: no workspace is used or grown; the product's replays have the eager
    call's bits, the attention's (f32 MFMA there) agree to rounding. Every
    replay is checked, eager work and a synchronisation between them."""
    import ctypes
    import os
    rt = ctypes.CDLL(os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib",
                                  "libamdhip64.so"))
    vp = ctypes.c_void_p
    m = hip.Model(be, embed=1024, heads=16)
    g = rng(71)
    M, N, K, T = 2500, 1030, 512, 1601
    A, B = (be.upload(g.standard_normal(s, dtype=np.float32)) for s in ((M, K), (N, K)))
    qkv = be.upload(g.standard_normal((T, 3072), dtype=np.float32))
    C, O = be.alloc(M * N * 4), be.alloc(T * 1024 * 4)

    def calls():
        hip.linear(m, M, K, N, A, 0, B, None, C, 0)
        hip.attn_fused(m, T, 16, 16, hip.bmat(qkv, 0, 3072, 0, 64),
                       hip.bmat(qkv, 1024, 3072, 0, 64), hip.bmat(qkv, 2048, 3072, 0, 64),
                       hip.bmat(O, 0, 1024, 0, 64))

    calls()
    want = be.read(C).copy(), be.read(O).copy()
    ws = be._b.gemm_ws_count, be._b.gemm_ws_bytes
    stream, graph, run = vp(be._b.stream), vp(), vp()
    assert rt.hipStreamBeginCapture(stream, 2) == 0   # relaxed
    try:
        calls()
    finally:
        assert rt.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert (be._b.gemm_ws_count, be._b.gemm_ws_bytes) == ws and not be._b.gemm_ws_held
    assert rt.hipGraphInstantiate(ctypes.byref(run), graph, None, None, 0) == 0
    try:
        for _ in range(4):
            for x in (C, O):
                be.write(x, 0, np.zeros(x.contents.bytes // 4, np.float32))
            assert rt.hipGraphLaunch(run, stream) == 0
            be.finish()
            assert np.array_equal(be.read(C), want[0])
            assert rel_l2(be.read(O), want[1]) <= 2e-6
            hip.add_bcast(m, C, C, C, M * N, M * N)
            be.finish()
    finally:
        rt.hipGraphExecDestroy(run)
        rt.hipGraphDestroy(graph)
