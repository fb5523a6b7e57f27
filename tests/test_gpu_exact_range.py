"""The exact path (precision=fp32) outside ordinary magnitudes: operands as
small as floats go, results beyond the largest float, and what a call costs
when its operands hold NaN.

The larger products and attentions run on operands split into bf16 pieces.
Scaling an operand by a power of two is exact, so each result here is that of
an ordinary problem times a known power of two, and the tolerance is the
ordinary one: sqrt(K) 2^-24 of the result for a sum of K products."""
import numpy as np
import pytest

from gpu_common import rel_l2, report

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import sam3_hip
    return sam3_hip


@pytest.fixture(scope="module")
def be(hip):
    b = hip.Backend(precision="fp32")
    yield b
    b.free()


def ms(be, call):
    """The fastest of five calls, by events."""
    call()
    best = 1e9
    for _ in range(5):
        be.finish()
        be.timer_start()
        call()
        best = min(best, be.timer_stop())
    return best


# Packed operands; split while staged (float and K x N operand); f32 MFMA.
GEMMS = [(2500, 1030, 512, 1), (700, 1024, 68, 1), (16500, 256, 256, 0), (33, 70, 300, 1)]


def product(hip, be, A, B, transb, C, alpha=1.0):
    M, K = A.shape
    N = B.shape[0] if transb else B.shape[1]
    m = hip.Model(be, embed=128, heads=2)
    dA, dB, dC = be.upload(A), be.upload(B), be.upload(C)
    try:
        hip.gemm(m, M, N, K, hip.mat(dA, 0, K), hip.mat(dB, 0, B.shape[1]), transb,
                 hip.mat(dC, 0, N), 1, 1, None, None, 0, alpha)
        return be.read(dC).reshape(M, N)
    finally:
        for x in (dA, dB, dC):
            be.release(x)
        m.free()


@pytest.mark.parametrize("M,N,K,transb", GEMMS)
def test_gemm_nan_costs_no_more_than_the_f32_units(hip, be, M, N, K, transb):
    """A product of NaN takes at most ten times the ordinary one (the f32
    matrix unit is a sixteenth of the bf16 one's rate, six products of which
    an ordinary one takes)."""
    m = hip.Model(be, embed=128, heads=2)
    g = np.random.default_rng(M)
    A = g.standard_normal((M, K), dtype=np.float32)
    B = g.standard_normal((N, K) if transb else (K, N), dtype=np.float32)
    dA, dB, dC = be.upload(A), be.upload(B), be.alloc(M * N * 4)
    t = []
    for bad in (False, True):
        if bad:
            A[:, K // 2] = np.nan
            be.write(dA, 0, A)
        t.append(ms(be, lambda: hip.gemm(m, M, N, K, hip.mat(dA, 0, K),
                                         hip.mat(dB, 0, K if transb else N), transb,
                                         hip.mat(dC, 0, N))))
    assert np.isnan(be.read(dC, M * N)).all()
    print("gemm %d x %d x %d: %.1f us, NaN %.1f us" % (M, N, K, 1e3 * t[0], 1e3 * t[1]))
    assert t[1] <= 10 * t[0]


@pytest.mark.parametrize("ea,eb", [
    (-118, 100),   # low pieces of A below bf16's range
    (-140, 110),   # A subnormal
    (110, -138),   # the other way round
    (-60, -60),    # small results
    (90, 30),      # results past the split's range, formed by the f32 unit
    (105, 10),     # an operand past it
])
@pytest.mark.parametrize("M,N,K,transb", GEMMS)
def test_gemm_magnitudes(hip, be, M, N, K, transb, ea, eb):
    """A 2^ea times B 2^eb: the ordinary product times 2^(ea + eb). Subnormal
    operands are first rounded to what the float type holds. A residual of the
    result's size, bias none."""
    g = np.random.default_rng(M + 200 + ea)
    A = np.ldexp(g.standard_normal((M, K), dtype=np.float32), ea).astype(np.float32)
    B = np.ldexp(g.standard_normal((N, K) if transb else (K, N), dtype=np.float32),
                 eb).astype(np.float32)
    got = product(hip, be, A, B, transb, np.zeros((M, N), np.float32))
    rows = np.unique(np.concatenate([np.arange(40) % M, [M - 1], g.integers(0, M, 60)]))
    want = np.ldexp(A[rows].astype(np.float64), -ea) @ np.ldexp(
        (B.T if transb else B).astype(np.float64), -eb)
    r = rel_l2(np.ldexp(got[rows].astype(np.float64), -ea - eb), want)
    print("2^%d x 2^%d, %d x %d x %d: rel-L2 %.2e" % (ea, eb, M, N, K, r))
    assert r <= (np.sqrt(K) + 2) * 2.0 ** -24


@pytest.mark.parametrize("M,N,K,transb", GEMMS)
def test_gemm_wide_rows(hip, be, M, N, K, transb):
    """Rows of A that span the float's range (2^-140 to 2^60, B the other way
    round, so that every product counts): each result within sqrt(K) 2^-24 of
    the size of its products."""
    g = np.random.default_rng(K)
    e = g.integers(-140, 60, K)
    A = np.ldexp(g.standard_normal((M, K), dtype=np.float32), e).astype(np.float32)
    B = g.standard_normal((N, K), dtype=np.float32)
    B = np.ldexp(B, np.minimum(-e - 20, 100)).astype(np.float32)
    got = product(hip, be, A, np.ascontiguousarray(B if transb else B.T), transb,
                  np.zeros((M, N), np.float32))
    a, b = A[:64].astype(np.float64), B.astype(np.float64)
    size = np.sqrt((a * a) @ (b * b).T)
    err = np.abs(got[:64] - a @ b.T) / size
    print("wide rows %d x %d x %d: %.2e" % (M, N, K, err.max()))
    assert np.sqrt((err ** 2).mean()) <= (np.sqrt(K) + 2) * 2.0 ** -24


def decoder(hip, be, G, P, emb, w, s0):
    """lowres of P prompts on a G x G image, and the time of its second
    upscaling (ms)."""
    model = hip.Model(be, embed=1024, heads=16)
    model.m.grid = G
    dec = hip.Decoder(model, w, P, img=14 * G)
    try:
        g = np.random.default_rng(3)
        dec.set_image(emb, s0, g.standard_normal((4 * G * G, 64)).astype(np.float32))
        pts = g.uniform(0, 14 * G, (P, 2)).astype(np.float32)
        dec.decode(pts)
        t = 1e9
        for _ in range(4):
            hip.prof_reset()
            be.set_profile(True)
            try:
                dec.decode(pts)
            finally:
                be.set_profile(False)
            t = min([t] + [r[1] for r in hip.prof_table() if r[0] == "upscale2"])
        return dec.lowres(P).copy(), t
    finally:
        dec.free()
        model.free()


@pytest.mark.parametrize("G,P", [(36, 4), (9, 3)])
def test_upscaling_nan_cost(hip, be, G, P):
    """A decode of a NaN image spends at most five times the ordinary time in
    the second upscaling: its products on the f32 unit beside the same GELUs."""
    g = np.random.default_rng(G)
    w = hip.random_decoder_weights(7)
    emb = g.standard_normal((G * G, 256)).astype(np.float32)
    s0 = g.standard_normal((16 * G * G, 32)).astype(np.float32)
    low, t = decoder(hip, be, G, P, emb, w, s0)
    assert np.isfinite(low).all()
    emb[G] = np.nan
    low, tn = decoder(hip, be, G, P, emb, w, s0)
    assert np.isnan(low).all()
    print("upscaling G=%d P=%d: %.1f us, NaN %.1f us" % (G, P, 1e3 * t, 1e3 * tn))
    assert tn <= 5 * t


def test_upscaling_small_weights(hip, be):
    """The second upscaling's weights times 2^-118, its bias and map zero: the
    logits are those of weights times 2^-60 (where GELU is linear too and the
    pieces are ordinary) times 2^-58, within the rounding of the 64 products."""
    G, P = 9, 2
    g = np.random.default_rng(5)
    emb = g.standard_normal((G * G, 256)).astype(np.float32)
    s0 = np.zeros((16 * G * G, 32), np.float32)
    out = []
    for e in (-60, -118):
        w = dict(hip.random_decoder_weights(7))
        w["up3w"] = np.ldexp(w["up3w"], e).astype(np.float32)
        w["up3b"] = np.zeros_like(w["up3b"])
        low, _ = decoder(hip, be, G, P, emb, w, s0)
        out.append(np.ldexp(low.astype(np.float64), -e))
    r = rel_l2(out[1], out[0])
    print("upscaling weights 2^-118: rel-L2 %.2e" % r)
    assert np.abs(out[0]).max() > 0 and r <= 8 * 2.0 ** -24


def attention(hip, be, Q, K, V, heads, hd, causal=False):
    """attend of Nq queries over Nk keys, and its time (ms)."""
    D = heads * hd
    m = hip.Model(be, embed=128, heads=2)
    dq, dk, dv = be.upload(Q), be.upload(K), be.upload(V)
    do = be.alloc(Q.size * 4)
    try:
        t = ms(be, lambda: hip.attend(m, Q.shape[0], K.shape[0], heads, hd, dq, D, dk, D, dv, D,
                                      do, D, causal, None, None, 0))
        return be.read(do).reshape(Q.shape), t
    finally:
        for x in (dq, dk, dv, do):
            be.release(x)
        m.free()


def normal(g, n, D, e=0):
    return np.ldexp(g.standard_normal((n, D), dtype=np.float32), e).astype(np.float32)


# Split operands, one split and several; the f32 MFMA kernel.
ATTENTIONS = [(1601, 1601, 16, 64, False), (1000, 2000, 6, 64, False), (1300, 1300, 16, 32, False),
              (1500, 1500, 12, 64, True), (201, 700, 8, 32, False)]


@pytest.mark.parametrize("nq,nk,heads,hd,causal", ATTENTIONS)
def test_attention_nan_cost(hip, be, nq, nk, heads, hd, causal):
    """An attention of NaN takes at most ten times the ordinary one."""
    g = np.random.default_rng(nq)
    q, k, v = (normal(g, n, heads * hd) for n in (nq, nk, nk))
    _, t = attention(hip, be, q, k, v, heads, hd, causal)
    k[0] = np.nan
    got, tn = attention(hip, be, q, k, v, heads, hd, causal)
    assert np.isnan(got).all()
    print("attention %d x %d, %d x %d: %.1f us, NaN %.1f us" % (nq, nk, heads, hd, 1e3 * t,
                                                                1e3 * tn))
    assert tn <= 10 * t


def softmax_rows64(q, k, v, heads, hd, causal, rows):
    """Sampled queries in 64 bits."""
    out = np.empty((len(rows), heads * hd))
    for h in range(heads):
        c = slice(h * hd, (h + 1) * hd)
        s = q[rows][:, c].astype(np.float64) @ k[:, c].astype(np.float64).T / np.sqrt(hd)
        if causal:
            s[np.arange(k.shape[0])[None] > rows[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, c] = p / p.sum(1, keepdims=True) @ v[:, c].astype(np.float64)
    return out


@pytest.mark.parametrize("eq,ek,ev", [
    (118, -118, 0),     # low pieces of K below bf16's range
    (-122, 122, 0),     # Q small, K past the range that splits
    (0, 0, -118),       # small values
    (110, -110, 100),   # Q and V past the split's range
])
@pytest.mark.parametrize("nq,nk,heads,hd,causal", ATTENTIONS)
def test_attention_magnitudes(hip, be, nq, nk, heads, hd, causal, eq, ek, ev):
    """Queries, keys and values times powers of two: the ordinary attention
    (queries times 2^(eq + ek), which the scores carry) times 2^ev. Scores are
    sums of hd products (their error, times the score's size of about 4, enters
    the weights) and outputs of nk: 4 sqrt(hd) + sqrt(nk) roundings."""
    g = np.random.default_rng(nq + 200 + ek)
    q, k, v = (normal(g, n, heads * hd, e) for n, e in ((nq, eq), (nk, ek), (nk, ev)))
    got, _ = attention(hip, be, q, k, v, heads, hd, causal)
    rows = np.unique(np.concatenate([np.arange(33), [nq - 1], g.integers(0, nq, 40)]))
    want = softmax_rows64(q, k, np.ldexp(v.astype(np.float64), -ev), heads, hd, causal, rows)
    r = rel_l2(np.ldexp(got[rows].astype(np.float64), -ev), want)
    print("attention 2^%d 2^%d 2^%d, %d x %d x %d: rel-L2 %.2e" % (eq, ek, ev, nq, nk, hd, r))
    assert r <= (4 * np.sqrt(hd) + np.sqrt(nk)) * 2.0 ** -24


@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("nq,nk,heads,hd,causal", ATTENTIONS)
def test_attention_scores_past_the_split_range(hip, be, nq, nk, heads, hd, causal, sign):
    """Scores of 2^88, all of one sign (below zero they must not turn into a
    mask): the softmax is one-hot, each output the value row of the largest
    score."""
    g = np.random.default_rng(nq)
    q = np.abs(normal(g, nq, heads * hd, 45)) + np.float32(2.0 ** 44)
    k = sign * (np.abs(normal(g, nk, heads * hd, 40)) + np.float32(2.0 ** 39))
    v = normal(g, nk, heads * hd)
    got, _ = attention(hip, be, q, k.astype(np.float32), v, heads, hd, causal)
    rows = np.arange(0, nq, 37)
    for h in range(heads):
        c = slice(h * hd, (h + 1) * hd)
        s = q[rows][:, c].astype(np.float64) @ k[:, c].astype(np.float64).T
        if causal:
            s[np.arange(nk)[None] > rows[:, None]] = -np.inf
        top = np.sort(s, 1)[:, -2:]
        # Clear of the scores' own rounding (hd terms of 2^-24 each).
        sure = np.diff(top)[:, 0] > hd * 2.0 ** -23 * np.abs(top[:, 1])
        assert sure.sum() > len(rows) // 2
        assert np.array_equal(got[rows][sure][:, c], v[s.argmax(1)][sure][:, c])
