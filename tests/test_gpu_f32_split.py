"""fp32 products on the bf16 matrix cores (three exact bf16 parts per value):
every tile configuration at its edges, against the fp64 oracle under the
strict-fp32 bounds (4 sqrt(K) u componentwise); the ranges the split itself
does not cover (subnormal operands, values of 2^104 and more, infinities, NaN)."""
import zlib

import numpy as np
import pytest
import torch

from _gpu_helpers import check, dev, fp32_tol, host, normal
from oracle import oracle as o

pytestmark = pytest.mark.gpu
OPS = {"NN": o.NN, "NT": o.NT, "TN": o.TN}


def _operands(rng, layout, M, N, K):
    A = normal(rng, (K, M) if layout == o.TN else (M, K))
    B = normal(rng, (N, K) if layout == o.NT else (K, N), std=0.5)
    return A, B


# (M, N, K): 128 x 128 tiles (129 tiles and up, or 128 of them with a K that is
# split over workgroups, here 1160), 256 x 256 tiles, ragged edges, one step to several stage
# groups of the contraction
SHAPES = [(2049, 1025, 1), (2177, 1100, 16), (2100, 1160, 17), (1999, 2055, 33), (2048, 1024, 512), (1930, 1024, 1160),
          (3588, 3700, 40), (3841, 3585, 33), (3588, 3700, 72), (3841, 3585, 65)]


@pytest.mark.parametrize("opname", list(OPS))
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("pad", [0, 1, 4])
def test_tiles(opname, shape, pad):
    """Contiguous operands, pitches of no alignment and of 16-byte alignment;
    C beside its row padding; run twice, bit for bit."""
    from logos_amd import vedic

    layout = OPS[opname]
    M, N, K = shape
    rng = np.random.default_rng(zlib.crc32(f"f32s-{opname}-{shape}".encode()))
    A, B = _operands(rng, layout, M, N, K)
    a, b = (torch.zeros((x.shape[0], x.shape[1] + pad), device="cuda") for x in (A, B))
    a[:, :A.shape[1]], b[:, :B.shape[1]] = dev(A), dev(B)
    a, b = a[:, :A.shape[1]], b[:, :B.shape[1]]
    buf = torch.full((M, N + 3), 7.0, device="cuda")
    got = host(vedic.gemm(layout, a, b, buf[:, :N]))
    assert np.all(host(buf)[:, N:] == 7.0)
    check(got, layout, A, B, tol=fp32_tol(K), label=f"{opname} {shape} pad {pad}")
    assert np.array_equal(host(vedic.gemm(layout, a, b)), got)


@pytest.mark.parametrize("opname", list(OPS))
@pytest.mark.parametrize("shape", [(2049, 1032), (2100, 1161), (200, 330), (8, 4)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("K", [1, 2, 3, 4])
def test_few_steps(opname, shape, K):
    """One product is rounded once, two products at most three times: no part
    of a value may be dropped there.  From three on the split's bound is within
    binary32 summation's (K roundings, and 2^-24 of each product dropped)."""
    from logos_amd import vedic

    layout = OPS[opname]
    M, N = shape
    rng = np.random.default_rng(zlib.crc32(f"f32s-few-{opname}-{shape}-{K}".encode()))
    A, B = _operands(rng, layout, M, N, K)
    got = host(vedic.gemm(layout, dev(A), dev(B)))
    a, b = (A.T if layout == o.TN else A).astype(np.float64), (B.T if layout == o.NT else B).astype(np.float64)
    if K == 1:
        assert np.array_equal(got, (a @ b).astype(np.float32))
    bound = {1: 1, 2: 2, 3: 4, 4: 5}[K] * o.U32 * (np.abs(a) @ np.abs(b))
    assert np.all(np.abs(got - a @ b) <= bound)


@pytest.mark.parametrize("opname", list(OPS))
@pytest.mark.parametrize("shape", [(63, 65, 100), (200, 33, 300), (130, 700, 2000), (1, 64, 5), (40, 1, 1)],
                         ids=lambda s: "x".join(map(str, s)))
def test_small_unaligned(opname, shape):
    """Few output tiles with rows that are not 16-byte aligned (64 x 64 tiles,
    split over K where long), operands one element into wider buffers."""
    from logos_amd import vedic

    layout = OPS[opname]
    M, N, K = shape
    rng = np.random.default_rng(zlib.crc32(f"f32s-small-{opname}-{shape}".encode()))
    A, B = _operands(rng, layout, M, N, K)
    a, b = (torch.zeros((x.shape[0], x.shape[1] + 2), device="cuda") for x in (A, B))
    a[:, 1:-1], b[:, 1:-1] = dev(A), dev(B)
    C0 = normal(rng, (M, N))
    check(host(vedic.gemm(layout, a[:, 1:-1], b[:, 1:-1])), layout, A, B, tol=fp32_tol(K), label=f"{opname} {shape}")
    check(host(vedic.gemm(layout, a[:, 1:-1], b[:, 1:-1], dev(C0), alpha=0.5, beta=-2.0)), layout, A, B, tol=fp32_tol(K),
          alpha=0.5, beta=-2.0, C0=C0, label=f"{opname} {shape} alpha/beta")


@pytest.mark.parametrize("shape", [(2100, 1160, 50), (3841, 3585, 33), (3841, 3585, 81)], ids=lambda s: "x".join(map(str, s)))
def test_epilogues(shape):
    """Each fused epilogue on the 128 x 128 and 256 x 256 tiles."""
    from logos_amd import vedic

    M, N, K = shape
    rng = np.random.default_rng(zlib.crc32(f"f32s-epi-{shape}".encode()))
    A, B = _operands(rng, o.NN, M, N, K)
    a, b, bias, C0 = dev(A), dev(B), normal(rng, (N,), std=0.1), normal(rng, (M, N))
    tol = fp32_tol(K)
    pre = torch.empty((M, N), device="cuda")
    H = host(vedic.gemm_bias_gelu(a, b, dev(bias), preact=pre))
    check(H, o.NN, A, B, tol=tol, bias=bias, gelu=True, label="bias + gelu")
    check(host(pre), o.NN, A, B, tol=tol, bias=bias, label="pre-activation")
    assert np.array_equal(host(vedic.gemm_bias_gelu(a, b, dev(bias))), H)
    P = host(vedic.vedic_gemm_bias(a, b, dev(bias)))
    assert np.array_equal(P, host(pre))
    assert np.array_equal(host(vedic.gemm_bias_residual(a, b, dev(bias), dev(C0))), C0 + P)
    check(host(vedic.gemm(o.NN, a, b, dev(C0), beta=1.0)), o.NN, A, B, tol=tol, beta=1.0, C0=C0, label="accumulate")
    cs = torch.zeros(N, device="cuda")
    C = host(vedic.gemm(o.NN, a, b, alpha=0.5, colsum=cs))
    assert np.array_equal(C, host(vedic.gemm(o.NN, a, b)) * np.float32(0.5))
    want = C.astype(np.float64).sum(0)
    assert np.all(np.abs(host(cs) - want) <= M * o.U32 * np.abs(C.astype(np.float64)).sum(0))


def test_range_edges():
    """Subnormal operands against large ones, products that are subnormal,
    finite values of 2^104 up to the largest binary32, and results past 2^80:
    within the fp32 bound of the oracle."""
    from logos_amd import vedic

    M, N, K = 2100, 1160, 48
    rng = np.random.default_rng(5)
    A, B = normal(rng, (M, K)), normal(rng, (K, N))
    rows = {0: -140, 300: -110, 700: -70, 1100: 110, 1500: 126, 2000: 60}
    for r, e in rows.items():
        A[r] *= np.float32(2.0 ** (e / 2)) * np.float32(2.0 ** (e / 2))
    A[1700], B[:, 50] = A[1700] * np.float32(2.0 ** -100), B[:, 50] * np.float32(2.0 ** 90)
    A[1701, 0], B[0, 60] = np.float32(3.4028235e38), np.float32(0.25)
    ok = np.abs(A.astype(np.float64)) @ np.abs(B.astype(np.float64)) < 3e38
    got = host(vedic.gemm(o.NN, dev(A), dev(B))).astype(np.float64)
    want = A.astype(np.float64) @ B.astype(np.float64)
    bound = 4 * np.sqrt(K) * o.U32 * (np.abs(A.astype(np.float64)) @ np.abs(B.astype(np.float64))) + K * 2.0 ** -149
    assert ok.sum() > 0.99 * ok.size
    bad = ok & ~(np.abs(got - want) <= bound + 2 * o.U32 * np.abs(want))
    assert not bad.any(), f"{bad.sum()} entries, first {np.argwhere(bad)[:5]}"


@pytest.mark.parametrize("opname", list(OPS))
def test_nonfinite(opname):
    """Infinities and NaN in either operand: infinite and NaN outputs where
    binary32 arithmetic has them, finite outputs elsewhere within the bound."""
    from logos_amd import vedic

    layout = OPS[opname]
    M, N, K = 2100, 1160, 24
    rng = np.random.default_rng(6)
    A, B = normal(rng, (M, K)), normal(rng, (K, N))
    A[7, 3], A[900, 5], A[901, 5], A[902, 6] = np.inf, -np.inf, np.inf, np.nan
    A[901, 9] = -np.inf
    B[2, 1000], B[9, 1100], A[30] = np.inf, np.nan, 0.0
    a = dev(np.ascontiguousarray(A.T) if layout == o.TN else A)
    b = dev(np.ascontiguousarray(B.T) if layout == o.NT else B)
    got = host(vedic.gemm(layout, a, b)).astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = np.einsum("ik,kj->ij", A.astype(np.float64), B.astype(np.float64))
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])
    fin = np.isfinite(want)
    assert np.all(np.abs(got[fin] - want[fin]) <= 4 * np.sqrt(K) * o.U32 * K * 30)


# (M, N, K, element offset of the operands): 256 x 256 tiles; 128 x 128 tiles in
# slices of K, unsplit with a ragged last group, unaligned; 64 x 64 tiles in slices, unaligned
REPEAT = [(3841, 3585, 81, 0), (1930, 1024, 1160, 0), (2177, 1100, 300, 0), (2100, 1160, 47, 1), (130, 700, 2000, 1)]


@pytest.mark.parametrize("opname", list(OPS))
@pytest.mark.parametrize("shape", REPEAT, ids=lambda s: "x".join(map(str, s)))
def test_repeat(opname, shape):
    """Blocks repeated on the fp32 MFMA in every tile configuration, beside
    blocks that are not: an infinity and a NaN at steps past the middle (with
    slices only a later one repeats), a row of 2^110 and a column of 2^60
    against a row of 2^40 (a result past 2^80)."""
    from logos_amd import vedic

    layout = OPS[opname]
    M, N, K, off = shape
    rng = np.random.default_rng(zlib.crc32(f"f32s-repeat-{opname}-{shape}".encode()))
    A, B = normal(rng, (M, K)), normal(rng, (K, N))
    A[5, K - 2], A[M - 1, K // 2 + 1] = np.inf, np.nan
    A[M // 2] *= np.float32(2.0 ** 110)
    A[M // 2 + 1] *= np.float32(2.0 ** 40)
    B[:, N // 3] *= np.float32(2.0 ** 60)
    A[M // 2, :] *= np.float32(2.0 ** -55)
    A[M // 2, 0] = np.float32(2.0 ** 110)

    def put(X):
        t = torch.zeros((X.shape[0], X.shape[1] + 2 * off), device="cuda")
        t[:, off:off + X.shape[1]] = dev(np.ascontiguousarray(X))
        return t[:, off:off + X.shape[1]]

    C0 = normal(rng, (M, N))
    a, b = put(A.T if layout == o.TN else A), put(B.T if layout == o.NT else B)
    got = host(vedic.gemm(layout, a, b, dev(C0), beta=1.0)).astype(np.float64)
    with np.errstate(invalid="ignore"):
        A64, B64 = A.astype(np.float64), B.astype(np.float64)
        want = A64 @ B64 + C0
        size = np.abs(A64) @ np.abs(B64) + np.abs(C0)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    inf = np.isinf(want)
    assert inf.any() and np.array_equal(got[inf], want[inf])
    fin = ~nan & ~inf & (size < 3e38)
    assert fin.sum() > 0.99 * (fin.size - nan.sum() - inf.sum())
    assert np.all(np.abs(got[fin] - want[fin]) <= 4 * np.sqrt(K) * o.U32 * size[fin])
