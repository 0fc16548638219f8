"""The product kernel's edges: float32 products formed from bf16 parts (csrc/split_bf16.hpp).

* Sizes around the tiles (64, 128, 256), the 32-deep stages and their 8-deep units, all four
  transposes and every alignment, against float64. Bound per element: each output sums
  6 ceil(K / 16) matrix-core steps, each rounding once relative to a partial sum of at most
  (|A||B|)_ij, and the parts left out and the closing additions are below 8 more such units:
  |dC| <= (6 ceil(K / 16) + 8) 2^-24 (|A||B|)_ij.
* Inputs whose parts overflow when scaled, infinities, NaN, results past 2^80: the float32 path
  that those outputs are formed again on (same classification as float64 rounded to float32).
* Tiny and denormal inputs, inputs of 2^87 to 2^103: no part is lost (the same bound).
* K of 1 and 2: the float32 cores' roundings.
* Sums over operands by sequence and in segments whose lengths are 16 mod 32 (half a stage), with
  K split inside a sequence or segment, and with infinities in them.
"""
import ctypes

import numpy as np
import pytest

from helpers import uniform

pytestmark = pytest.mark.gpu


def bound(A, B, K):
    return (6 * -(-K // 16) + 8) * 2.0 ** -24 * (np.abs(A) @ np.abs(B))


def check(C, A, B):
    A, B = A.astype(np.float64), B.astype(np.float64)
    assert C.shape == (A.shape[0], B.shape[1])
    assert np.all(np.abs(C - A @ B) <= bound(A, B, A.shape[1]) + 2.0 ** -149)


@pytest.mark.parametrize("M,N", [(2, 2), (33, 65), (64, 129), (65, 64), (127, 128), (129, 257), (257, 130), (300, 31),
                                 (1100, 2100)])
@pytest.mark.parametrize("K", [1, 7, 8, 9, 16, 31, 32, 33, 65, 100])
def test_edges(hip, M, N, K):
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    A, B = uniform(rng, (M, K)), uniform(rng, (K, N))
    for tA in (False, True):
        for tB in (False, True):
            C = hip.matmul(hip.tensor(A.T if tA else A), hip.tensor(B.T if tB else B), tA, tB).numpy()
            check(C, A, B)


@pytest.mark.parametrize("M,N,K", [(130, 70, 2500), (40, 300, 4111), (769, 770, 8200), (3000, 1400, 2049)])
def test_split_k_edges(hip, M, N, K):
    rng = np.random.default_rng(M + N + K)
    A, B = uniform(rng, (M, K)), uniform(rng, (K, N))
    check(hip.matmul(hip.tensor(A), hip.tensor(B)).numpy(), A, B)
    check(hip.matmul(hip.tensor(A), hip.tensor(B.T), False, True).numpy(), A, B)


def same_class(C, ref):
    """C finite, infinite (with the sign) and NaN exactly where ref is."""
    assert np.array_equal(np.isnan(C), np.isnan(ref))
    fin = np.isfinite(ref)
    assert np.array_equal(fin, np.isfinite(C))
    inf = np.isinf(ref)
    assert np.array_equal(np.sign(C[inf]), np.sign(ref[inf]))


@pytest.mark.parametrize("M,N,K", [(5, 6, 9), (130, 200, 100), (600, 1100, 70), (100, 90, 2600)])
@pytest.mark.parametrize("tA,tB", [(False, False), (True, False), (False, True), (True, True)])
def test_not_finite(hip, M, N, K, tA, tB):
    rng = np.random.default_rng(M + N + K)
    A, B = uniform(rng, (M, K), 0.5, 1.0), uniform(rng, (K, N), 0.5, 1.0)
    A[1, K // 2] = np.inf
    A[M - 1, 0] = np.nan
    B[K - 1, N - 1] = -np.inf
    B[0, 2] = np.inf
    with np.errstate(invalid="ignore"):
        ref = A.astype(np.float64) @ B.astype(np.float64)
    C = hip.matmul(hip.tensor(A.T if tA else A), hip.tensor(B.T if tB else B), tA, tB).numpy()
    same_class(C, ref)
    fin = np.isfinite(ref)
    assert np.all(np.abs(C[fin] - ref[fin]) <= 4 * K * 2.0 ** -24 * np.abs(ref[fin]))   # all terms positive


@pytest.mark.parametrize("sa,sb", [(1e34, 1e-6), (1e15, 1e15), (3e38, 1e-3), (2e18, 1e18)])
@pytest.mark.parametrize("M,N,K", [(70, 90, 50), (300, 1500, 33)])
def test_large_values(hip, sa, sb, M, N, K):
    """Inputs past 2^104 or results past 2^80 (up to 1e38): float32 sums of finite results."""
    rng = np.random.default_rng(K)
    A, B = uniform(rng, (M, K), -1, 1) * np.float32(sa), uniform(rng, (K, N), -1, 1) * np.float32(sb)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    C = hip.matmul(hip.tensor(A), hip.tensor(B)).numpy()
    assert np.isfinite(C).all()
    assert np.all(np.abs(C - ref) <= 2 * K * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)))


@pytest.mark.parametrize("sa,sb", [(1e-30, 1e10), (1e-37, 1.0), (1e-41, 1e20), (1e-44, 1e30), (1e-20, 1e-20)])
def test_tiny_values(hip, sa, sb):
    rng = np.random.default_rng(3)
    M, N, K = 130, 140, 77
    A = (uniform(rng, (M, K)).astype(np.float64) * sa).astype(np.float32)
    B = (uniform(rng, (K, N)).astype(np.float64) * sb).astype(np.float32)
    check(hip.matmul(hip.tensor(A), hip.tensor(B)).numpy(), A, B)


@pytest.mark.parametrize("M,N,K", [(5, 6, 3), (130, 140, 77), (300, 1500, 33), (100, 90, 2600)])
@pytest.mark.parametrize("large", ["A", "B"])
def test_large_values_within_the_scaled_range(hip, M, N, K, large):
    """One operand spread over 2^87 to 2^103, just below the inputs whose parts overflow when scaled, the other so
    small that results stay below 2^80: the bf16 parts, exact there too."""
    rng = np.random.default_rng(K)
    B = uniform(rng, (K, N)) * np.float32(2.0 ** -40)
    A = (2.0 ** rng.uniform(87, 103, (M, K)) * rng.choice([-1.0, 1.0], (M, K))).astype(np.float32)
    if large == "B":
        A, B = np.ascontiguousarray(B.T), np.ascontiguousarray(A.T)
    check(hip.matmul(hip.tensor(A), hip.tensor(B)).numpy(), A, B)
    check(hip.matmul(hip.tensor(A), hip.tensor(B.T), False, True).numpy(), A, B)


@pytest.mark.parametrize("M,N", [(3, 5), (64, 129), (300, 500), (1100, 2100)])
@pytest.mark.parametrize("tA,tB", [(False, False), (True, False), (False, True), (True, True)])
def test_one_and_two_products(hip, M, N, tA, tB):
    """K = 1: each product rounded once. K = 2: at most two roundings, of a product and of the sum."""
    rng = np.random.default_rng(M)
    for K in (1, 2):
        A, B = (rng.normal(0, 1, s).astype(np.float32) for s in ((M, K), (K, N)))
        C = hip.matmul(hip.tensor(A.T if tA else A), hip.tensor(B.T if tB else B), tA, tB).numpy()
        if K == 1:
            assert np.array_equal(C, A * B)
        else:
            A, B = A.astype(np.float64), B.astype(np.float64)
            assert np.all(np.abs(C - A @ B) <= 2 * 2.0 ** -24 * (np.abs(A) @ np.abs(B)))


class BySeq(ctypes.Structure):
    _fields_ = [("len", ctypes.c_size_t), ("step", ctypes.c_size_t)]


def _ptrs(ts):
    return (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])


@pytest.mark.parametrize("klen", [16, 48, 80, 176])
def test_segments_of_half_stages(hip, klen):
    lib, P, SZ = hip._lib, ctypes.c_void_p, ctypes.c_size_t
    lib.nnhip_gemm_tn_sum.argtypes = [P, P, SZ, P, SZ, SZ, SZ, ctypes.c_float, P, SZ, P]
    lib.nnhip_engine_stream.restype, lib.nnhip_engine_stream.argtypes = P, [P]
    M, N = 132, 260
    rng = np.random.default_rng(klen)
    A, B = [uniform(rng, (klen, M)) for _ in range(3)], [uniform(rng, (klen, N)) for _ in range(3)]
    a, b, c = [hip.tensor(x) for x in A], [hip.tensor(x) for x in B], hip.create_tensor(M, N)
    assert lib.nnhip_gemm_tn_sum(_ptrs(a), _ptrs(b), 3, c.data_ptr(), M, N, klen, 1.0, None, 0,
                                 lib.nnhip_engine_stream(hip._e)) == 0
    check(c.numpy(), np.concatenate(A).T, np.concatenate(B))


@pytest.mark.parametrize("T,nseq", [(16, 9), (48, 5), (80, 16)])
def test_by_sequence_of_half_stages(hip, T, nseq):
    """Weight gradients G X^T whose A and B are heads' rows of sequences 16 mod 32 long."""
    lib, P, SZ = hip._lib, ctypes.c_void_p, ctypes.c_size_t
    lib.nnhip_gemm_group_acc_seq.argtypes = [P, P, P, SZ, SZ, SZ, SZ, ctypes.c_int, ctypes.c_int, P, ctypes.c_int, P, P,
                                             P, SZ, P]
    lib.nnhip_engine_stream.restype, lib.nnhip_engine_stream.argtypes = P, [P]
    d, K = 128, T * nseq
    rng = np.random.default_rng(T)
    G, X = uniform(rng, (d, K)), uniform(rng, (d, K))
    seq = [hip.tensor(np.ascontiguousarray(x.reshape(d, nseq, T).transpose(1, 0, 2)).reshape(-1, T)) for x in (G, X)]
    c, rows = hip.tensor(np.zeros((d, d))), hip.tensor(np.zeros((d, 1)))
    lay = (BySeq * 1)(BySeq(T, d * T))
    assert lib.nnhip_gemm_group_acc_seq(_ptrs(seq[:1]), _ptrs(seq[1:]), _ptrs([c]), 1, d, d, K, 1, 1, _ptrs([rows]), 1,
                                        lay, lay, None, 0, lib.nnhip_engine_stream(hip._e)) == 0
    check(c.numpy(), G, X.T)
    ref = G.astype(np.float64).sum(1, keepdims=True)
    assert np.all(np.abs(rows.numpy() - ref) <= K * 2.0 ** -24 * np.abs(G).astype(np.float64).sum(1, keepdims=True))


def check_class(C, A, B):
    """check, and where the float64 result is not finite its class."""
    A, B = A.astype(np.float64), B.astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref = A @ B
    same_class(C, ref)
    fin = np.isfinite(ref)
    b = bound(np.where(np.isfinite(A), A, 0.0), np.where(np.isfinite(B), B, 0.0), A.shape[1])
    assert np.all(np.abs(C[fin] - ref[fin]) <= b[fin] + 2.0 ** -149)


@pytest.fixture
def lib(hip):
    l, P, SZ, F, I = hip._lib, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_float, ctypes.c_int
    l.nnhip_gemm_workspace_bytes.restype, l.nnhip_gemm_workspace_bytes.argtypes = SZ, [SZ] * 4
    l.nnhip_engine_stream.restype, l.nnhip_engine_stream.argtypes = P, [P]
    l.nnhip_gemm_tn_sum.argtypes = [P, P, SZ, P, SZ, SZ, SZ, F, P, SZ, P]
    l.nnhip_gemm_tn_sum_seq.argtypes = [P, P, SZ, P, SZ, SZ, SZ, F, BySeq, P, SZ, P]
    l.nnhip_gemm_epilogue_seq.argtypes = [P, P, P, SZ, SZ, SZ, F, P, I, BySeq, P, SZ, P]
    l.nnhip_gemm_group_acc_seq.argtypes = [P, P, P, SZ, SZ, SZ, SZ, I, I, P, I, P, P, P, SZ, P]
    return l


def by_seq(hip, X, T):
    """X (d, K) as heads' rows: per sequence of T columns its (d, T)."""
    d = X.shape[0]
    return hip.tensor(np.ascontiguousarray(X.reshape(d, -1, T).transpose(1, 0, 2)).reshape(-1, T))


@pytest.mark.parametrize("klen,split", [(48, False), (1040, True), (688, True)])
@pytest.mark.parametrize("bad", [False, True])
def test_segments(hip, lib, klen, split, bad):
    """Three segments, with K split across them, and with an infinity in one (the float32 path)."""
    M, N = 132, 260
    rng = np.random.default_rng(klen)
    A, B = [uniform(rng, (klen, M)) for _ in range(3)], [uniform(rng, (klen, N)) for _ in range(3)]
    if bad:
        A[1][klen - 1, 70], B[2][17, 200] = np.inf, np.nan
    a, b, c = [hip.tensor(x) for x in A], [hip.tensor(x) for x in B], hip.create_tensor(M, N)
    wsb = lib.nnhip_gemm_workspace_bytes(M, N, 3 * klen, 1) if split else 0
    assert (wsb > 0) == split
    ws = hip.create_tensor(1, max(wsb // 4, 1))
    assert lib.nnhip_gemm_tn_sum(_ptrs(a), _ptrs(b), 3, c.data_ptr(), M, N, klen, 1.0, ws.data_ptr() if wsb else None,
                                 wsb, lib.nnhip_engine_stream(hip._e)) == 0
    check_class(c.numpy(), np.concatenate(A).T, np.concatenate(B))


@pytest.mark.parametrize("T,nseq,split", [(48, 6, False), (16, 130, True), (48, 50, True), (80, 27, True)])
@pytest.mark.parametrize("bad", [False, True])
def test_by_sequence(hip, lib, T, nseq, split, bad):
    """Two weight gradients G X^T of rows by sequence with their row sums: K split inside a sequence (k slices are
    multiples of 32, sequences of 16), and an infinity."""
    d, K, n = 128, T * nseq, 2
    rng = np.random.default_rng(T)
    G, X = [uniform(rng, (d, K)) for _ in range(n)], [uniform(rng, (d, K)) for _ in range(n)]
    if bad:
        G[0][70, K - 3], X[1][5, T + 1] = np.inf, -np.inf
    g, x = [by_seq(hip, a, T) for a in G], [by_seq(hip, a, T) for a in X]
    c, rows = [hip.tensor(np.zeros((d, d))) for _ in range(n)], [hip.tensor(np.zeros((d, 1))) for _ in range(n)]
    lay = (BySeq * n)(*[BySeq(T, d * T)] * n)
    wsb = lib.nnhip_gemm_workspace_bytes(d, d, K, n) if split else 0
    assert (wsb > 0) == split
    ws = hip.create_tensor(1, max(wsb // 4, 1))
    assert lib.nnhip_gemm_group_acc_seq(_ptrs(g), _ptrs(x), _ptrs(c), n, d, d, K, 1, 1, _ptrs(rows), 1, lay, lay,
                                        ws.data_ptr() if wsb else None, wsb, lib.nnhip_engine_stream(hip._e)) == 0
    for i in range(n):
        check_class(c[i].numpy(), G[i], X[i].T)
        ref, r = G[i].astype(np.float64).sum(1, keepdims=True), rows[i].numpy()
        same_class(r, ref)
        fin = np.isfinite(ref)
        assert np.all(np.abs(r[fin] - ref[fin]) <= (K * 2.0 ** -24 * np.abs(G[i]).astype(np.float64).sum(1, keepdims=True))[fin])


@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("n", [1, 2])
def test_columns_by_sequence(hip, lib, n, bad):
    """B by sequence, untransposed: W X and a sum of two W^T X."""
    M, K, T, nseq = 128, 48, 128, 3
    rng = np.random.default_rng(n)
    A, B = [uniform(rng, (K, M)) for _ in range(n)], [uniform(rng, (K, T * nseq)) for _ in range(n)]
    if bad:
        A[0][40, 9], B[n - 1][3, T + 70] = np.nan, np.inf
    b, c, st = [by_seq(hip, x, T) for x in B], hip.create_tensor(M, T * nseq), lib.nnhip_engine_stream(hip._e)
    if n == 1:
        a = hip.tensor(A[0].T)
        rc = lib.nnhip_gemm_epilogue_seq(a.data_ptr(), b[0].data_ptr(), c.data_ptr(), M, T * nseq, K, 1.0, None, 0,
                                         BySeq(T, K * T), None, 0, st)
    else:
        a = [hip.tensor(x) for x in A]
        rc = lib.nnhip_gemm_tn_sum_seq(_ptrs(a), _ptrs(b), n, c.data_ptr(), M, T * nseq, K, 1.0, BySeq(T, K * T), None,
                                       0, st)
    assert rc == 0
    check_class(c.numpy(), np.concatenate(A).T, np.concatenate(B))
