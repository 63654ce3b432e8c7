"""The split (three bf16 pieces) GEMM at the edges of its tiles, against
float64, and on the values its pieces cannot hold, against the oracle.

Bound of a result: every fp32 rounding of the accumulator is at most 2^-24 of
the running sum of |a b|, six piece products per 16 of k and one more for each
K chunk; the three dropped piece products are at most 2^-24 |a b| together.
That finds a wrong element, not a lost piece, whose size is 2^-17 |a b|: the
bounds of split3_model do.
"""
import numpy as np
import pytest

import helpers
import oracle
import split3_model as sm
from neuralscript_amd import runtime, synth

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def product(A, B, variant, splits=None, act=0):
    """C = A . B through the entry point, A [M, K], B [K, N]."""
    (M, K), N = A.shape, B.shape[1]
    tA, tB = variant == "tn", variant == "nt"
    dA = runtime.DeviceArray.from_host(np.ascontiguousarray(A.T if tA else A))
    dB = runtime.DeviceArray.from_host(np.ascontiguousarray(B.T if tB else B))
    dC = runtime.DeviceArray(M * N)
    lda, ldb = M if tA else K, K if tB else N
    if splits is None:
        runtime.gemm(dA, dB, dC, M, N, K, lda, ldb, N, tA, tB, act)
    else:
        runtime.gemm_splitk(dA, dB, dC, M, N, K, lda, ldb, N, tA, tB, act, splits)
    return dC.to_host().reshape(M, N)


def operands(M, N, K, seed):
    return (synth.normal(seed, M * K).reshape(M, K), synth.normal(seed + 1, K * N).reshape(K, N))


# one element short of, at and past each tile (128 and 256 rows, 128 columns; the
# contiguous extent of an operand is a multiple of 4), K at the least the split
# kernel takes and inside a slab, more tiles than CUs
SHAPES = [(4, 4, 128), (124, 132, 132), (128, 128, 128), (132, 252, 140), (256, 256, 144), (260, 516, 196),
          (4096, 256, 160), (4100, 4100, 132), (8192, 2052, 128), (260, 132, 124)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("variant", ["nn", "nt", "tn"])
def test_split_product_against_float64(M, N, K, variant):
    print(f"split gemm {variant} M={M} N={N} K={K}", flush=True)
    A, B = operands(M, N, K, M + 3 * N + K)
    rows = np.unique(np.clip(np.array([0, 1, 31, 32, 127, 128, 255, 256, M // 2, M - 2, M - 1]), 0, M - 1))
    got = product(A, B, variant)[rows].astype(np.float64)
    a, b = A[rows].astype(np.float64), B.astype(np.float64)
    bound = (6 * (K // 16 + 1) + 4) * U * (np.abs(a) @ np.abs(b))
    assert np.all(np.abs(got - a @ b) <= bound)


# on the small kernel, on 256- and 128-row tiles, over K chunks
PRECISE = [(256, 512, 128, None), (40, 72, 2048, None), (2048, 2048, 256, None), (4096, 1028, 132, None),
           (1500, 516, 512, None), (1024, 1028, 4096, 0), (260, 132, 1032, 4)]


@pytest.mark.parametrize("M,N,K,splits", PRECISE)
@pytest.mark.parametrize("variant", ["nn", "nt", "tn"])
def test_every_piece_counts_on_normal_operands(M, N, K, splits, variant):
    print(f"precise gemm {variant} M={M} N={N} K={K}", flush=True)
    A, B = operands(M, N, K, 3 * M + N + K)
    got = product(A, B, variant, splits)
    assert sm.rel(got, A.astype(np.float64) @ B.astype(np.float64)) <= sm.normal_bound(K)


@pytest.mark.parametrize("M,N,K,splits", PRECISE)
@pytest.mark.parametrize("variant", ["nn", "nt", "tn"])
def test_every_piece_counts_in_products_of_one_term(M, N, K, splits, variant):
    """Row m of A holds one value, at k = m mod K, of 24 significant bits."""
    rng = np.random.default_rng(M + K)
    B = (1 + rng.random((K, N))).astype(np.float32) * rng.choice(np.float32([-1, 1]), (K, N))
    A, k, a = np.zeros((M, K), np.float32), np.arange(M) % K, (1 + rng.random(M)).astype(np.float32)
    a[0] = B[0, 0] = float.fromhex("0x1.00ff8p+0")  # where the dropped products weigh most
    A[np.arange(M), k] = a
    ref = a[:, None].astype(np.float64) * B[k]
    assert np.max(np.abs(product(A, B, variant, splits) / ref - 1)) <= sm.one_term_bound()


@pytest.mark.parametrize("M,N,K,splits", [(128, 128, 512, 3), (260, 132, 1032, 4), (512, 512, 4096, 0)])
@pytest.mark.parametrize("variant", ["nn", "nt", "tn"])
def test_split_k_product_against_float64(M, N, K, splits, variant):
    A, B = operands(M, N, K, 7 * M + N + K)
    got = product(A, B, variant, splits).astype(np.float64)
    a, b = A.astype(np.float64), B.astype(np.float64)
    bound = (6 * (K // 16 + 1) + 40) * U * (np.abs(a) @ np.abs(b))
    assert np.all(np.abs(got - a @ b) <= bound)


@pytest.mark.parametrize("M,N,K", [(132, 136, 140), (512, 8192, 128), (8192, 512, 128)])
@pytest.mark.parametrize("variant", ["nn", "nt", "tn"])
def test_values_without_three_pieces(M, N, K, variant):
    """Infinities, NaN and values that bf16 rounds to infinity: where the
    oracle's are; the rows beside them as if they were not there."""
    A, B = operands(M, N, K, 11 * M + K)
    A[1, 0], A[3, K - 1], A[5, 1] = np.inf, -np.inf, np.nan
    A[6, 0], A[6, 1] = np.inf, -np.inf
    A[8, 2], A[M - 1, K - 1] = 3.4e38, -3.39e38
    rows = [0, 1, 2, 3, 4, 5, 6, 7, 8, 9, M - 2, M - 1]
    with np.errstate(all="ignore"):
        ref = oracle.matmul(A[rows].ravel(), B.ravel(), len(rows), K, N).reshape(-1, N)
    got = product(A, B, variant)[rows]
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isposinf(got), np.isposinf(ref)) and np.array_equal(np.isneginf(got), np.isneginf(ref))
    ok = np.isfinite(ref)
    # (8, .) and (M - 1, .) carry sums of the order of 3e38
    small = ok & (np.abs(ref) < 1e30)
    helpers.assert_close(got[small], ref[small], f"beside special values {variant}")
    assert np.all(np.abs(got[ok] - ref[ok]) <= 1e-5 * np.abs(ref[ok]) + 1e-4)


@pytest.mark.parametrize("scale", [2.0 ** -100, 2.0 ** -115, 2.0 ** -126, 2.0 ** -135, 2.0 ** -140, 2.0 ** 70])
@pytest.mark.parametrize("variant", ["nn", "nt", "tn"])
def test_operands_of_any_magnitude(scale, variant):
    """Operands down to fp32's subnormals and up to sums past 2^80 keep the
    relative accuracy of their own bits."""
    M, N, K = 136, 260, 144
    A, B = operands(M, N, K, 77)
    A = (A * np.float32(scale)).astype(np.float32)  # subnormal operands keep the bits fp32 has there
    B = (B * np.float32(2.0 ** 20)).astype(np.float32)
    got = product(A, B, variant).astype(np.float64)
    a, b = A.astype(np.float64), B.astype(np.float64)
    bound = (K + 8) * U * (np.abs(a) @ np.abs(b)) + 2.0 ** -149 * K
    assert np.all(np.abs(got - a @ b) <= bound)


# the small kernel: one and two row blocks of 32, edges of its 32 columns,
# K of one wave's step, of every wave's first step and past the loads in flight
@pytest.mark.parametrize("M,N,K", [(1, 1, 4), (1, 10, 256), (31, 33, 16), (33, 31, 20), (64, 64, 132), (65, 97, 516),
                                   (256, 10, 256), (5, 40, 1100), (70, 32, 2052)])
@pytest.mark.parametrize("variant", ["nn", "nt", "tn"])
@pytest.mark.parametrize("act", [0, 6])
def test_small_product_against_float64(M, N, K, variant, act):
    print(f"small gemm {variant} M={M} N={N} K={K} act={act}", flush=True)
    A, B = operands(M, N, K, 5 * M + N + K)
    got = product(A, B, variant, act=act).astype(np.float64)
    a, b = A.astype(np.float64), B.astype(np.float64)
    ref = a @ b
    # eight partial sums of K / 8 steps each; GELU has a slope of at most 1.13
    bound = (K + 24) * U * (np.abs(a) @ np.abs(b))
    if act:
        from math import erf, sqrt
        ref = np.vectorize(lambda x: 0.5 * x * (1 + erf(x / sqrt(2))))(ref)
        bound = 1.13 * bound + 4 * U * np.abs(ref) + 1e-7
    assert np.all(np.abs(got - ref) <= bound)


@pytest.mark.parametrize("variant", ["nn", "nt", "tn"])
def test_small_product_of_special_values(variant):
    M, N, K = 40, 36, 136
    A, B = operands(M, N, K, 4)
    A[1, 0], A[3, K - 1], A[5, 1], A[7, 2] = np.inf, -np.inf, np.nan, 3.4e38
    with np.errstate(all="ignore"):
        ref = oracle.matmul(A.ravel(), B.ravel(), M, K, N).reshape(M, N)
    got = product(A, B, variant)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    calm = np.isfinite(ref) & (np.abs(ref) < 1e30)
    helpers.assert_close(got[calm], ref[calm], f"small gemm beside special values {variant}")


# products of few tiles and a long K by the kernel that can read them: the small
# kernel (aligned; it needs no chunks), and the fp32 kernel, which it must not
# leave with one chunk (K % 4 != 0, or both transposed)
@pytest.mark.parametrize("M,N,K,variant,chunks", [(33, 64, 1200, "nn", 1), (33, 64, 1201, "nn", 4),
                                                  (33, 64, 1201, "nt", 4), (33, 64, 1200, "tt", 4),
                                                  (33, 64, 1201, "tn", 1), (1501, 160, 1501, "nn", 5),
                                                  (33, 64, 511, "nn", 1), (33, 64, 512, "tt", 2)])
def test_chosen_chunks_of_long_products(M, N, K, variant, chunks):
    """The workspace shows the chunks that were written: `chunks` blocks of M x N
    floats, inside what nsh_op_gemm_splitk_workspace asked for."""
    print(f"split count {variant} M={M} N={N} K={K}", flush=True)
    A, B = operands(M, N, K, 13 * M + K)
    tA, tB = variant[0] == "t", variant[1] == "t"
    dA = runtime.DeviceArray.from_host(np.ascontiguousarray(A.T if tA else A))
    dB = runtime.DeviceArray.from_host(np.ascontiguousarray(B.T if tB else B))
    dC = runtime.DeviceArray(M * N)
    need = runtime.lib().nsh_op_gemm_splitk_workspace(M, N, K, 0) // 4
    ws = runtime.DeviceArray.from_host(np.full(need + 33 * M * N, np.nan, np.float32))
    runtime.check(runtime.lib().nsh_op_gemm_splitk(dA.ptr, dB.ptr, dC.ptr, M, N, K, M if tA else K, K if tB else N, N,
                                                   int(tA), int(tB), 0, 0, ws.ptr), "gemm_splitk")
    written = np.flatnonzero(~np.isnan(ws.to_host()))
    assert written.size == (chunks * M * N if chunks > 1 else 0)
    assert written.size == 0 or written[-1] < need
    a, b = A.astype(np.float64), B.astype(np.float64)
    bound = (K + 40) * U * (np.abs(a) @ np.abs(b))
    assert np.all(np.abs(dC.to_host().reshape(M, N).astype(np.float64) - a @ b) <= bound)


def test_split_without_a_workspace():
    """Refused where the shape asks for chunks, run unsplit where only the
    operands' alignment does."""
    for M, N, K, refused in [(33, 64, 1201, False), (512, 512, 4096, True)]:
        A, B = operands(M, N, K, K)
        dA, dB, dC = runtime.DeviceArray.from_host(A), runtime.DeviceArray.from_host(B), runtime.DeviceArray(M * N)
        rc = runtime.lib().nsh_op_gemm_splitk(dA.ptr, dB.ptr, dC.ptr, M, N, K, K, N, N, 0, 0, 0, 0, None)
        assert (rc != 0) == refused
        if not refused:
            a, b = A.astype(np.float64), B.astype(np.float64)
            assert np.all(np.abs(dC.to_host().reshape(M, N) - a @ b) <= (K + 8) * U * (np.abs(a) @ np.abs(b)))
