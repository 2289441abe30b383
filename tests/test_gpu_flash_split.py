"""Attention on the bf16 matrix cores (three exact bf16 parts per value): what
the split does not cover is repeated on the fp32 MFMA with the same results as
binary32 arithmetic -- infinities, NaN, values of 2^104 and more, scores far
below zero -- and sparse masks whose 32-key blocks have no allowed key."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as o  # noqa: E402
from tests._gpu_helpers import dev, fp32_tol, host, normal  # noqa: E402

pytestmark = pytest.mark.gpu


def vedic():
    from logos_amd import vedic as v

    return v


def _nan_equal(got, want):
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])
    fin = np.isfinite(want)
    return fin


@pytest.mark.parametrize("seq", [40, 700])
def test_nonfinite_operands(seq):
    """One infinite V entry reaches every query that attends to its key (P > 0
    there), a NaN in Q or K its row or the rows that see it, and the rows
    before them are the finite call's."""
    v = vedic()
    rng = np.random.default_rng(seq)
    Q, K, V = (normal(rng, (seq, 64)) for _ in range(3))
    clean = host(v.flash_attention_fwd(dev(Q), dev(K), dev(V)))
    V2 = V.copy()
    V2[seq // 2, 5] = np.inf
    got = host(v.flash_attention_fwd(dev(Q), dev(K), dev(V2)))
    assert np.all(np.isinf(got[seq // 2:, 5]) | np.isnan(got[seq // 2:, 5]))
    err = np.abs(got[:seq // 2 // 32 * 32] - clean[:seq // 2 // 32 * 32])
    assert err.size == 0 or err.max() <= fp32_tol(64) * np.abs(clean).max()
    Q2 = Q.copy()
    Q2[seq // 3, 7] = np.nan
    got = host(v.flash_attention_fwd(dev(Q2), dev(K), dev(V)))
    assert np.all(np.isnan(got[seq // 3]))
    rest = np.delete(np.arange(seq), seq // 3)
    assert np.abs(got[rest] - clean[rest]).max() <= fp32_tol(64) * np.abs(clean).max()


@pytest.mark.parametrize("heads", [1, 3])
@pytest.mark.parametrize("scales", [(1.0, 1.0, 2.0 ** 110), (2.0 ** 60, 2.0 ** -60, 2.0 ** -130), (1e-30, 1e-30, 1.0),
                                    (2.0 ** -126, 2.0 ** 100, 1.0), (3.0, 3.0, 2.0 ** -146)])
def test_scales(heads, scales):
    """Q, K and V at extreme scales against float64."""
    v = vedic()
    rng = np.random.default_rng(17)
    seq, dh = 333, 64
    sq, sk, sv = (np.float32(x) for x in scales)
    Q, K, V = ([normal(rng, (seq, dh)) * s for _ in range(heads)] for s in (sq, sk, sv))
    outs = v.flash_attention_fwd_heads([dev(x) for x in Q], [dev(x) for x in K], [dev(x) for x in V])
    for i in range(heads):
        want = o.flash_attention_f64(Q[i], K[i], V[i], 0.125, 1, 0, 0, 1)
        # subnormal results: the partial of each of at most three key chunks and the
        # merged row are rounded to half of 2^-149
        assert np.abs(host(outs[i]) - want).max() <= fp32_tol(dh) * np.abs(want).max() + 4 * 2.0 ** -150


@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("k", [60, 84, 96, 104, 110, 118, 125])
def test_scores_from_far_apart_operands(dh, sign, k):
    """Q of about 2^-k against K of about 2^k, and the other way round: scores of
    order one, whose bits the parts of a tiny operand carry.  One head (its keys
    split over work items) and three."""
    v = vedic()
    rng = np.random.default_rng(k + 1000 * dh + sign)
    seq = 205
    for heads in (1, 3):
        Q, K, V = ([normal(rng, (seq, dh)) * np.float32(s) for _ in range(heads)]
                   for s in (2.0 ** (-sign * k), 2.0 ** (sign * k), 1.0))
        assert np.isfinite(Q).all() and np.isfinite(K).all()
        outs = v.flash_attention_fwd_heads([dev(x) for x in Q], [dev(x) for x in K], [dev(x) for x in V])
        for i in range(heads):
            want = o.flash_attention_f64(Q[i], K[i], V[i], dh ** -0.5, 1, 0, 0, 1)
            # (a score of up to 4: 4 sqrt(dh) roundings of its size)
            assert o.inf_rel_err(host(outs[i]), want) <= 16 * np.sqrt(dh) * o.U32, (heads, i)


@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("e", [90, 84, 78, 50])
def test_scores_past_the_split(dh, e):
    """Scores of size 2^e, some rows all negative: past 2^80 the scaled scores
    are infinite and the item is repeated, also where every one is -inf."""
    v = vedic()
    rng = np.random.default_rng(e + dh)
    seq = 150
    K, V = np.abs(normal(rng, (seq, dh))), normal(rng, (seq, dh))
    Q = np.abs(normal(rng, (seq, dh))) * np.float32(2.0 ** e)
    Q[::2] = -Q[::2]
    got = host(v.flash_attention_fwd(dev(Q), dev(K), dev(V)))
    # (scores this far apart leave one key per row; two whose scores lie within
    # the rounding of their sum would be a tie that binary32 cannot decide)
    s = (Q.astype(np.float64) @ K.astype(np.float64).T) * dh ** -0.5
    s[np.triu_indices(seq, 1)] = -np.inf
    top = np.sort(s, 1)[:, ::-1]
    clear = np.r_[True, top[1:, 0] - top[1:, 1] > fp32_tol(dh) * np.abs(top[1:, 1])]
    assert clear.sum() > 140
    want = o.flash_attention_f64(Q, K, V, dh ** -0.5, 1, 0, 0, 1)
    assert np.abs(got[clear] - want[clear]).max() <= fp32_tol(dh) * np.abs(want).max()


def test_infinite_score_that_cancels():
    """Partial sums of a score that leave the split's range and come back: -2^100
    from one group of 16 values, +2^100 from the next, the rest of order one."""
    v = vedic()
    rng = np.random.default_rng(31)
    seq, dh = 70, 64
    Q, K, V = (normal(rng, (seq, dh)) for _ in range(3))
    Q[:, 3] = Q[:, 20] = 2.0 ** 50
    K[:, 3], K[:, 20] = -2.0 ** 50, 2.0 ** 50
    Q[:, 4:20] = Q[:, :3] = Q[:, 21:] = 0  # (what else a partial sum of 2^100 holds would be rounded away)
    got = host(v.flash_attention_fwd(dev(Q), dev(K), dev(V)))
    want = o.flash_attention_f64(Q, K, V, 0.125, 1, 0, 0, 1)
    assert o.inf_rel_err(got, want) <= fp32_tol(dh)


@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("t", [60, 105, 112, 118, 124])
def test_tiny_probabilities(dh, t):
    """A key of probability 2^-t that holds the only values: its outputs keep
    the accuracy that the score's rounding leaves the probability."""
    v = vedic()
    rng = np.random.default_rng(t)
    seq = 100
    Q, K, V = np.zeros((seq, dh), np.float32), np.zeros((seq, dh), np.float32), np.zeros((seq, dh), np.float32)
    Q[:, 0] = 1 + 0.01 * rng.random(seq)
    K[7, 0] = -t * np.log(2.0) * dh ** 0.5
    V[7] = normal(rng, (dh,)) * np.float32(2.0 ** 76)
    got = host(v.flash_attention_fwd(dev(Q), dev(K), dev(V), causal=False)).astype(np.float64)
    want = o.flash_attention_f64(Q, K, V, dh ** -0.5, 0, 0, 0, 1)
    # the score t: 4 roundings (scale, Q, product, exponent) of t u each, and the sums of the row
    assert np.abs(got - want).max() <= (4 * t + 4 * np.sqrt(seq)) * o.U32 * np.abs(want).max()


def test_scores_far_below_zero():
    """Rows whose every score is about -2^101: below -1e29 the reference counts
    a score as masked."""
    v = vedic()
    rng = np.random.default_rng(19)
    seq, dh = 70, 64
    Q, K, V = np.abs(normal(rng, (seq, dh))), -np.abs(normal(rng, (seq, dh))), normal(rng, (seq, dh))
    Q[10:20] *= np.float32(2.0 ** 101)
    got = host(v.flash_attention_fwd(dev(Q), dev(K), dev(V)))
    want = o.flash_attention(Q, K, V, 0.125, 1, 0, 0, 1)
    assert np.all(got[10:20] == 0) and np.all(want[10:20] == 0)
    rest = np.r_[0:10, 20:seq]
    assert np.abs(got[rest] - want[rest]).max() <= 2 * fp32_tol(dh) * np.abs(want[rest]).max()


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("window,stride", [(0, 1000), (31, 33), (32, 64), (100, 129), (5, 32)])
def test_sparse_blocks(causal, window, stride):
    """Windows and strides around the 32-key block: whole blocks with no
    allowed key for a wave's 32 queries, and blocks with one."""
    v = vedic()
    rng = np.random.default_rng(window * 1000 + stride)
    seq, dh = 419, 64
    Q, K, V = (normal(rng, (seq, dh)) for _ in range(3))
    lse = torch.empty(seq, device="cuda")
    kw = dict(causal=bool(causal), shunyam=True, window=window, stride=stride)
    got = host(v.flash_attention_fwd(dev(Q), dev(K), dev(V), lse=lse, **kw))
    want = o.flash_attention_f64(Q, K, V, 0.125, causal, 1, window, stride)
    assert o.inf_rel_err(got, want) <= fp32_tol(dh)


def _backward(v, Q, K, V, dO, **kw):
    tQ, tK, tV = dev(Q), dev(K), dev(V)
    lse = torch.empty(Q.shape[0], device="cuda")
    out = v.flash_attention_fwd(tQ, tK, tV, lse=lse, **kw)
    return tuple(host(t) for t in v.flash_attention_bwd(tQ, tK, tV, out, dev(dO), lse, **kw))


@pytest.mark.parametrize("scales", [(1.0, 1.0, 1.0, 2.0 ** -60), (1.0, 1.0, 2.0 ** 50, 2.0 ** 40), (1e-20, 1e-20, 1.0, 1.0),
                                    (2.0 ** 30, 2.0 ** -30, 1.0, 1.0), (1.0, 1.0, 2.0 ** -70, 2.0 ** 20)])
def test_backward_scales(scales):
    """Operands and gradients at extreme scales: within the split's range, past
    its scaled sums (repeated on the fp32 MFMA) and below bf16's normal range."""
    v = vedic()
    rng = np.random.default_rng(23)
    seq, dh = 205, 64
    Q, K, V, dO = (normal(rng, (seq, dh)) * np.float32(s) for s in scales)
    got = _backward(v, Q, K, V, dO)
    want = o.flash_attention_bwd_f64(Q, K, V, dO, 0.125)
    for g, w, name in zip(got, want, ("dQ", "dK", "dV")):
        assert np.abs(g - w).max() <= fp32_tol(seq) * np.abs(w).max(), name


@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("grad", [-20, -60])
@pytest.mark.parametrize("k", [60, 84, 90, 96, 104, 110, 118, 125])
def test_backward_from_far_apart_operands(dh, sign, grad, k):
    """Q of about 2^-k against K of about 2^k, and the other way round: scores of
    order one, gradients small enough that no sum leaves the split's range."""
    v = vedic()
    rng = np.random.default_rng(k + 1000 * dh + sign)
    seq = 205
    Q, K, V, dO = (normal(rng, (seq, dh)) * np.float32(s) for s in (2.0 ** (-sign * k), 2.0 ** (sign * k), 1.0, 2.0 ** grad))
    got = _backward(v, Q, K, V, dO)
    want = o.flash_attention_bwd_f64(Q, K, V, dO, dh ** -0.5)
    for g, w, name in zip(got, want, ("dQ", "dK", "dV")):
        # (scores of up to 4: 4 sqrt(dh) roundings of their size, then sums of seq
        # terms; subnormal sums are rounded to 2^-149 at every term)
        bound = (16 * np.sqrt(dh) + 4 * np.sqrt(seq)) * o.U32 * np.abs(w).max() + seq * 2.0 ** -149
        assert np.abs(g - w).max() <= bound, name


@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("t", [60, 100, 105, 112, 118])
def test_backward_tiny_probabilities(dh, t):
    """dV of a key that every query gives a probability of about 2^-t / 100."""
    v = vedic()
    rng = np.random.default_rng(t)
    seq = 100
    Q, K = np.zeros((seq, dh), np.float32), np.zeros((seq, dh), np.float32)
    V, dO = normal(rng, (seq, dh)), normal(rng, (seq, dh))
    Q[:, 0] = 1 + 0.01 * rng.random(seq)
    K[7, 0] = -t * np.log(2.0) * dh ** 0.5
    got = _backward(v, Q, K, V, dO, causal=False)[2][7].astype(np.float64)
    want = o.flash_attention_bwd_f64(Q, K, V, dO, dh ** -0.5, 0)[2][7]
    # the score t: 4 roundings (scale, K, product, exponent) of t u each on every
    # term, and the sum of the seq terms
    size = (np.abs(dO).astype(np.float64).sum(0) * 2.0 ** -t / seq).max()
    assert np.abs(got - want).max() <= (4 * t + 4 * np.sqrt(seq)) * o.U32 * size


@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("std", [1.0, 6.0])
def test_passes_recompute_the_same_probabilities(dh, std):
    """P of one key, read out of each backward pass bit for bit: of the dK/dV pass
    by unit rows of dO (dV[key] = P), of the dQ pass by a unit value of V and O =
    0 (dS = P on that key, whose K has a 1).  A rounding of the scores that the
    two passes, and the forward that made lse, share cancels; one that differs
    is an error of P of its size."""
    v = vedic()
    rng = np.random.default_rng(41 + dh)
    seq, key, scale = 150, 37, 0.125
    Q, K = normal(rng, (seq, dh)) * np.float32(std), normal(rng, (seq, dh))
    K[:, dh - 1] = 0
    K[key, dh - 1] = 1
    lse = torch.empty(seq, device="cuda")
    v.flash_attention_fwd(dev(Q), dev(K), dev(K), lse=lse, scale=scale, causal=False)
    zero = np.zeros((seq, dh), np.float32)
    one, V = zero.copy(), zero.copy()
    one[np.arange(dh), np.arange(dh)] = 1.0  # dO of the first dh queries
    dV = host(v.flash_attention_bwd(dev(Q), dev(K), dev(zero), dev(zero), dev(one), lse, scale=scale, causal=False)[2])
    V[key, 0] = 1.0
    dO = zero.copy()
    dO[:, 0] = 1.0
    dQ = host(v.flash_attention_bwd(dev(Q), dev(K), dev(V), dev(zero), dev(dO), lse, scale=scale, causal=False)[0])
    assert np.all(dV[key, :] > 0)
    assert np.array_equal(dV[key, :], dQ[:dh, dh - 1] / np.float32(scale))


def test_backward_nonfinite():
    """A NaN in one dO row reaches every dK, dV row it attends to and its own
    dQ row; the other queries keep their finite dQ and the keys past its
    32-key block (whose masked weights of 0 meet the NaN) their dV."""
    v = vedic()
    rng = np.random.default_rng(29)
    seq, dh = 300, 64
    Q, K, V, dO = (normal(rng, (seq, dh)) for _ in range(4))
    clean = _backward(v, Q, K, V, dO)
    dO2 = dO.copy()
    dO2[200, 3] = np.nan
    dQ, dK, dV = _backward(v, Q, K, V, dO2)
    assert np.all(np.isnan(dQ[200])) and np.all(np.isnan(dV[:201, 3])) and np.all(np.isnan(dK[:201]))
    rest = np.delete(np.arange(seq), 200)
    assert np.abs(dQ[rest] - clean[0][rest]).max() <= fp32_tol(seq) * np.abs(clean[0]).max()
    assert np.abs(dV[224:] - clean[2][224:]).max() <= fp32_tol(seq) * np.abs(clean[2]).max()


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("window,stride", [(0, 1000), (31, 33), (100, 129)])
def test_backward_sparse_blocks(causal, window, stride):
    v = vedic()
    rng = np.random.default_rng(window * 1000 + stride + 1)
    seq, dh = 419, 64
    Q, K, V, dO = (normal(rng, (seq, dh)) for _ in range(4))
    got = _backward(v, Q, K, V, dO, causal=bool(causal), shunyam=True, window=window, stride=stride)
    want = o.flash_attention_bwd_f64(Q, K, V, dO, 0.125, causal, 1, window, stride)
    assert o.grad_rel_err(got, want) <= fp32_tol(seq)


@pytest.mark.parametrize("seq", [1, 31, 33, 129, 700])
@pytest.mark.parametrize("causal,sparse", [(1, 0), (0, 0), (1, 1), (0, 1)])
def test_forward_dh128(seq, causal, sparse):
    """Head dimension 128 around the 32-key block and the 128-query group, one
    head (its keys split over work items) and three: float64, and a head of
    2^110 (repeated on the fp32 MFMA) beside two ordinary ones."""
    v = vedic()
    rng = np.random.default_rng(seq)
    kw = dict(causal=bool(causal), shunyam=bool(sparse), window=40, stride=33)
    for heads in (1, 3):
        Q, K, V = ([normal(rng, (seq, 128)) for _ in range(heads)] for _ in range(3))
        V[-1] = V[-1] * np.float32(2.0 ** 110)
        outs = v.flash_attention_fwd_heads([dev(x) for x in Q], [dev(x) for x in K], [dev(x) for x in V], **kw)
        for i in range(heads):
            want = o.flash_attention_f64(Q[i], K[i], V[i], 128 ** -0.5, causal, sparse, 40, 33)
            assert o.inf_rel_err(host(outs[i]), want) <= fp32_tol(128), (heads, i)


@pytest.mark.parametrize("key", [0, 40, 299])
def test_forward_dh128_nonfinite(key):
    """An infinite V entry reaches the queries from its key on; the row groups
    of 32 before it keep the finite call's values."""
    v = vedic()
    rng = np.random.default_rng(key)
    Q, K, V = (normal(rng, (300, 128)) for _ in range(3))
    clean = host(v.flash_attention_fwd(dev(Q), dev(K), dev(V)))
    V[key, 100] = np.inf
    got = host(v.flash_attention_fwd(dev(Q), dev(K), dev(V)))
    assert not np.any(np.isfinite(got[key:, 100]))
    before = key // 32 * 32
    assert np.all(np.abs(got[:before] - clean[:before]) <= fp32_tol(128) * np.abs(clean).max())


@pytest.mark.parametrize("seq", [31, 33, 129, 300])
@pytest.mark.parametrize("causal,sparse", [(1, 0), (0, 0), (1, 1), (0, 1)])
@pytest.mark.parametrize("big", [False, True])
def test_backward_dh128(seq, causal, sparse, big):
    """Head dimension 128 around the 32-row block and the 128-row group; dO of
    2^60 leaves the split's scaled sums (repeated on the fp32 MFMA)."""
    v = vedic()
    rng = np.random.default_rng(seq + 1000 * big)
    kw = dict(causal=bool(causal), shunyam=bool(sparse), window=40, stride=33)
    Q, K, V, dO = (normal(rng, (seq, 128)) for _ in range(4))
    if big:
        dO = dO * np.float32(2.0 ** 60)
    got = _backward(v, Q, K, V, dO, **kw)
    want = o.flash_attention_bwd_f64(Q, K, V, dO, 128 ** -0.5, causal, sparse, 40, 33)
    assert o.grad_rel_err(got, want) <= fp32_tol(max(seq, 128))
