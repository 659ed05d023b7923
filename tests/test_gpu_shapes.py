"""Kernel dispatch edges: widths and row counts around the tiles, panels and
blocks of the fast-order Gram, the padded updates, the small LU and the QR."""

import ctypes

import numpy as np
import pytest

from cacg_amd import problems as P

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


# a block of G is at most 8 x 10 tiles of 16; pairs of columns need two of them
GRAM = [(1, 1, 1, 0), (1, 5, 4, 1), (2, 4, 4, 1), (3, 1, 1, 1), (15, 16, 16, 1), (17, 17, 17, 3),
        (63, 21, 21, 3), (64, 40, 40, 5), (65, 33, 30, 2), (127, 2, 3, 7), (129, 96, 96, 12),
        (1000, 129, 160, 0), (999, 128, 129, 17), (513, 145, 20, 141), (8191, 8, 8, 1),
        (8192, 8, 8, 1), (8193, 60, 60, 10), (20001, 100, 100, 20), (4097, 128, 128, 32),
        (300, 256, 256, 32), (2, 1, 17, 1)]


@pytest.mark.parametrize("n,kl,kr1,kr2", GRAM)
def test_gram_fast_edges_exact_on_integers(gpu_lib, n, kl, kr1, kr2):
    rng = np.random.default_rng(n + kl + kr1 + kr2)
    L, R1, R2 = (rng.integers(-8, 9, size=(n, k)).astype(np.float64) for k in (kl, kr1, kr2))
    print(f"gram n={n} {kl} x ({kr1} + {kr2})", flush=True)
    out = gpu_lib.k_gram(L, R1, R2 if kr2 else None, mode="fast")
    G1, G2 = out if kr2 else (out, None)
    assert np.array_equal(G1, L.T @ R1)   # integers below 2^53: exact in any order
    if kr2:
        assert np.array_equal(G2, L.T @ R2)


@pytest.mark.parametrize("n,k", [(1, 2), (130, 17), (9000, 31), (5000, 60)])
def test_gram_f64f32_edges_exact_on_integers(gpu_lib, n, k):
    rng = np.random.default_rng(n + k)
    L = rng.integers(-8, 9, size=(n, k)).astype(np.float64)
    R = rng.integers(-8, 9, size=(n, k)).astype(np.float32)
    print(f"gram f64 x f32 n={n} k={k}", flush=True)
    assert np.array_equal(gpu_lib.k_gram_f64f32(L, R), L.T @ R.astype(np.float64))


@pytest.mark.parametrize("n", [1, 15, 16, 17, 1000, 16385])
@pytest.mark.parametrize("sm,m", [(1, 1), (3, 1), (7, 7), (10, 2), (15, 3), (17, 1), (60, 10),
                                  (63, 21), (100, 20), (127, 1), (24, 8), (31, 31)])
def test_padded_updates_exact_on_integers(gpu_lib, n, sm, m):
    rng = np.random.default_rng(n + 131 * sm + m)
    ints = lambda *s: rng.integers(-8, 9, size=s).astype(np.float64)  # noqa: E731
    S, Q, AQ, beta, alpha, X, R = (ints(n, sm), ints(n, sm), ints(n, sm), ints(sm, sm),
                                   ints(sm, m), ints(n, m), ints(n, m))
    print(f"updates n={n} sm={sm} m={m}", flush=True)
    assert np.array_equal(gpu_lib.k_qupdate(S, Q, beta, mode="fast"), S - Q @ beta)
    assert np.array_equal(gpu_lib.k_qupdate_s32(S.astype(np.float32), Q, beta), S - Q @ beta)
    Xn, Rn, norm2 = gpu_lib.k_xrupdate(Q, AQ, alpha, X, R, mode="fast")
    assert np.array_equal(Xn, X + Q @ alpha) and np.array_equal(Rn, R - AQ @ alpha)
    assert np.array_equal(norm2, ((R - AQ @ alpha) ** 2).sum(0))


def _spd(N, seed):
    M = np.random.default_rng(seed).standard_normal((N, N))
    return M @ M.T + N * np.eye(N)


@pytest.mark.parametrize("N,k", [(1, 1), (7, 7), (8, 16), (9, 32), (31, 33), (33, 5), (64, 64),
                                 (65, 32), (120, 33), (127, 1), (128, 128), (129, 3), (200, 40),
                                 (256, 32), (257, 257), (300, 1)])
def test_lu_panels_and_blocks_bitwise(gpu_lib, oracle_lib, N, k):
    """Fast and reference order, first call and kept factor, around the panel
    (8), the right-hand sides that ride along (32) and the block (128)."""
    from conftest import lu_restated
    A, rng = _spd(N, N + k), np.random.default_rng(k)
    rhs, rhs2 = rng.standard_normal((N, k)), rng.standard_normal((N, N))
    print(f"lu N={N} k={k}", flush=True)
    x, x2, flag = gpu_lib.k_lu_solve(A, rhs, mode="fast", rhs2=rhs2)
    assert flag == 0
    assert np.array_equal(x, lu_restated(A, rhs, "fast"))
    assert np.array_equal(x2, lu_restated(A, rhs2, "fast"))
    x, x2, flag = gpu_lib.k_lu_solve(A, rhs, mode="reference", rhs2=rhs2)
    assert flag == 0
    assert np.array_equal(x, oracle_lib.lu_solve(A, rhs))
    assert np.array_equal(x2, oracle_lib.lu_solve(A, rhs2))


@pytest.mark.parametrize("N,p", [(12, 0), (40, 17), (128, 127), (200, 130)])
def test_lu_flags_a_zero_pivot_anywhere(gpu_lib, N, p):
    A = np.eye(N)
    A[p, p] = 0.0
    print(f"lu zero pivot N={N} p={p}", flush=True)
    for mode in ("fast", "reference"):
        assert gpu_lib.k_lu_solve(A, np.ones((N, 2)), mode=mode)[1] == 1


@pytest.mark.parametrize("n,k,lda", [(300, 7, 7), (300, 8, 11), (1000, 9, 16), (2000, 33, 40),
                                     (5000, 65, 65), (5000, 127, 128)])
def test_tsqr_strided_input(gpu_lib, n, k, lda):
    """A with a row stride is read where it lies; bounds as for contiguous input:
    orthogonality 50 k u, residual 1e-13."""
    W = np.random.default_rng(n + k).standard_normal((n, lda))
    L = gpu_lib.lib()
    dA, dQ, dR = (gpu_lib.DeviceBuffer.from_array(W), gpu_lib.DeviceBuffer(8 * n * k),
                  gpu_lib.DeviceBuffer(8 * k * k))
    ws = gpu_lib.DeviceBuffer(8 * L.cacg_tsqr_workspace(k))
    flag = gpu_lib.DeviceBuffer.from_array(np.zeros(1, dtype=np.int32))
    print(f"tsqr n={n} k={k} lda={lda}", flush=True)
    assert L.cacg_k_tsqr(n, k, dA.ptr, lda, dQ.ptr, dR.ptr, ws.ptr, flag.ptr, None) == 0
    Q, R = dQ.download((n, k)), dR.download((k, k))
    assert int(flag.download(1, np.int32)[0]) == 0
    assert np.array_equal(dA.download((n, lda)), W)
    assert np.all(np.tril(R, -1) == 0.0) and np.all(np.diag(R) > 0)
    assert np.abs(Q.T @ Q - np.eye(k)).max() <= 50 * k * EPS / 2
    assert np.linalg.norm(Q @ R - W[:, :k]) <= 1e-13 * np.linalg.norm(W[:, :k])


# blocks of 1, 2, 4, 5 and 8 columns of L by the size of G; stages of 192, 96 or 48 rows, the
# last 8 or so of them checked row by row
GREF = [(1, 1, 1, 0), (191, 3, 3, 2), (192, 16, 15, 1), (193, 17, 33, 3), (1728, 20, 16, 4),
        (1727, 60, 60, 10), (1921, 33, 128, 16), (96, 128, 128, 0), (863, 112, 112, 14),
        (865, 127, 128, 0), (97, 128, 128, 16), (960, 125, 126, 18), (49, 160, 160, 20),
        (431, 161, 150, 17), (433, 168, 168, 1)]


@pytest.mark.parametrize("n,kl,kr1,kr2", GREF)
def test_gram_reference_edges_bitwise(gpu_lib, oracle_lib, n, kl, kr1, kr2):
    rng = np.random.default_rng(n + kl + kr1 + kr2)
    L, R1, R2 = (rng.standard_normal((n, k)) for k in (kl, kr1, kr2))
    print(f"reference gram n={n} {kl} x ({kr1} + {kr2})", flush=True)
    out = gpu_lib.k_gram(L, R1, R2 if kr2 else None, mode="reference")
    G1, G2 = out if kr2 else (out, None)
    assert np.array_equal(G1, oracle_lib.gram(L, R1))
    if kr2:
        assert np.array_equal(G2, oracle_lib.gram(L, R2))


@pytest.mark.parametrize("n,m,ld", [(15, 4, 4), (16, 5, 7), (17, 3, 3), (511, 6, 6), (512, 16, 16),
                                    (513, 7, 9), (1025, 9, 9)])
def test_colnorm2_reference_edges_bitwise(gpu_lib, oracle_lib, n, m, ld):
    R = np.random.default_rng(n + m).standard_normal((n, m))
    print(f"reference column norms n={n} m={m} ld={ld}", flush=True)
    want = np.array([oracle_lib.col_norm2sq(R, c) for c in range(m)])
    assert np.array_equal(gpu_lib.k_colnorm2_ref(R, ld), want)


class BSys(ctypes.Structure):
    _fields_ = ([(f, ctypes.c_int) for f in ("n", "m", "sm", "ntile", "nchunk", "pad_")] +
                [(f, ctypes.c_void_p) for f in ("rowptr", "col", "val", "val32", "B", "X", "R", "S",
                                                "Q", "AQ", "QtAQ", "QtAS", "beta", "lu", "QtR",
                                                "alpha", "gpart", "npart", "norm2", "flag")] +
                [(f, ctypes.c_double) for f in ("sa", "sb")])


# (n, m, sm) of systems that share a launch: one tile to 8 x 10, chunks of 1 to 2048 rows, steps
# in flight 12 to 32
BGRAM = [[(1, 1, 1)], [(127, 1, 4), (2048, 2, 8), (2049, 17, 17), (95, 32, 128)],
         [(6000, 3, 9), (4097, 5, 20), (255, 8, 32), (2175, 10, 40)],
         [(2047, 16, 64), (130, 32, 96), (2303, 30, 120), (383, 7, 112)], [(5000, 32, 128)]]


@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("systems", BGRAM)
def test_batched_gram_exact_on_integers(gpu_lib, systems, f32):
    lib, D, rng = gpu_lib.lib(), gpu_lib.DeviceBuffer.from_array, np.random.default_rng(len(systems))
    print(f"batched gram {systems} f32={f32}", flush=True)
    descs, host, keep = (BSys * len(systems))(), [], []
    for d, (n, m, sm) in zip(descs, systems):
        Q, AQ, S = (rng.integers(-8, 9, size=(n, sm)).astype(np.float64) for _ in range(3))
        R = rng.integers(-8, 9, size=(n, m)).astype(np.float64)
        d.n, d.m, d.sm, d.ntile, d.nchunk = n, m, sm, (n + 63) // 64, (n + 2047) // 2048
        bufs = dict(Q=D(Q), AQ=D(AQ), S=D(S.astype(np.float32) if f32 else S), R=D(R),
                    gpart=D(np.full(d.nchunk * sm * (sm + m), np.nan)),
                    QtAQ=D(np.full((sm, sm), np.nan)), QtAS=D(np.full((sm, sm), np.nan)),
                    QtR=D(np.full((sm, m), np.nan)))
        for f, b in bufs.items():
            setattr(d, f, b.ptr)
        host.append((Q, AQ, S, R))
        keep.append(bufs)
    dsys = D(np.frombuffer(bytes(descs), dtype=np.uint8))
    for which in (0, 1):
        kr = [sm + (m if which else 0) for _, m, sm in systems]
        chunks = [(i, c) for i, d in enumerate(descs) for c in range(d.nchunk)]
        blocks = [(i, e) for i, (_, _, sm) in enumerate(systems) for e in range((sm * kr[i] + 255) // 256)]
        groups = max(lib.cacg_bgram_groups(sm, k) for (_, _, sm), k in zip(systems, kr))
        dc, db = (D(np.array(v, dtype=np.int32)) for v in (chunks, blocks))
        assert lib.cacg_kb_gram(dsys.ptr, dc.ptr, len(chunks), groups, which, f32, None) == 0
        assert lib.cacg_kb_gram_reduce(dsys.ptr, db.ptr, len(blocks), which, None) == 0
        for (n, m, sm), (Q, AQ, S, R), b in zip(systems, host, keep):
            if which == 0:
                assert np.array_equal(b["QtAS"].download((sm, sm)), AQ.T @ S)
            else:
                assert np.array_equal(b["QtAQ"].download((sm, sm)), Q.T @ AQ)
                assert np.array_equal(b["QtR"].download((sm, m)), Q.T @ R)


@pytest.mark.parametrize("k", [2, 6, 10, 14, 18, 22, 30, 34, 66, 130])
def test_spmm_column_pairs_bitwise(gpu_lib, oracle_lib, k):
    """Even widths that are no multiple of 4 (two columns a lane), every epilogue; the FP32 forms
    against the row split, which sums the same products in the same order."""
    A = P.random_spd_like(P.laplacian_3d(9), seed=5)
    X, p1, p2 = (P.rhs_normal(A.n, k, sd) for sd in (1, 2, 3))
    print(f"spmm pairs k={k}", flush=True)
    AX, a, b = oracle_lib.spmm(A, X), 0.37, -0.21
    assert np.array_equal(gpu_lib.k_spmm(A, X), AX)
    assert np.array_equal(gpu_lib.k_spmm(A, X, "cheb", a, b, p1=p1, p2=p2), (a * AX + b * p1) - p2)
    assert np.array_equal(gpu_lib.k_spmm(A, X, "resid", p1=p1), p1 - AX)
    S1, S0 = gpu_lib.k_spmm(A, X, "cheb1", a, b, want_copy0=True)
    assert np.array_equal(S0, X) and np.array_equal(S1, a * AX + b * X)
    X32, q1, q2 = (v.astype(np.float32) for v in (X, p1, p2))
    for epi, kw in (("none", {}), ("cheb", dict(p1=q1, p2=q2))):
        want = gpu_lib.k_spmm_f32(A, X32, epi, 0.5, -0.25, long_min=1, **kw)
        assert np.array_equal(gpu_lib.k_spmm_f32(A, X32, epi, 0.5, -0.25, long_min=0, **kw), want)
    for w, g in zip(gpu_lib.k_cheb1_f32(A, X, 0.5, -0.25, long_min=1),
                    gpu_lib.k_cheb1_f32(A, X, 0.5, -0.25, long_min=0)):
        assert np.array_equal(g, w)


@pytest.mark.parametrize("edge,k", [(96, 3), (73, 12), (96, 16), (69, 104)])
def test_spmm_default_order_gives_the_same_bits(gpu_lib, edge, k):
    """Blocks just past the sizes from which the default order is chunks over a resident grid."""
    A = P.laplacian_3d(edge)
    X = P.rhs_uniform(A.n, k, 3)
    print(f"spmm default order {edge}^3 k={k}", flush=True)
    assert np.array_equal(gpu_lib.k_spmm(A, X), gpu_lib.k_spmm(A, X, sched=(4096, 0, 0)))


@pytest.mark.parametrize("n,sm,m", [(1, 1, 1), (300, 4, 1), (16384, 4, 1), (5000, 6, 2), (2000, 8, 8),
                                    (4097, 7, 3), (700, 5, 5), (20001, 8, 4), (333, 3, 8)])
def test_gram_with_solve_gives_the_bits_of_the_two_calls(gpu_lib, n, sm, m):
    lib, D, rng = gpu_lib.lib(), gpu_lib.DeviceBuffer.from_array, np.random.default_rng(n + sm)
    B = gpu_lib.DeviceBuffer
    Q, S = rng.standard_normal((n, sm)), rng.standard_normal((n, sm))
    R, AQ = rng.standard_normal((n, m)), Q * 2.0 + 0.1 * rng.standard_normal((n, sm))
    dQ, dAQ, dS, dS32, dR = D(Q), D(AQ), D(S), D(S.astype(np.float32)), D(R)
    ws = B(8 * lib.cacg_gram_workspace(sm, sm + m))
    print(f"gram + solve n={n} sm={sm} m={m}", flush=True)
    got, want = ({k: B(8 * sz) for k, sz in (("g1", sm * sm), ("g2", sm * m), ("x", sm * m), ("lu", sm * sm),
                                             ("as", sm * sm), ("b", sm * sm), ("as32", sm * sm),
                                             ("b32", sm * sm))} for _ in range(2))
    flag = D(np.zeros(1, dtype=np.int32))
    w = {k: b.ptr for k, b in want.items()}
    assert lib.cacg_k_gram_fast(n, dQ.ptr, sm, sm, dAQ.ptr, sm, sm, dR.ptr, m, m, w["g1"], w["g2"],
                                ws.ptr, None) == 0
    assert lib.cacg_k_lu_solve(sm, w["g1"], m, w["g2"], w["x"], w["lu"], flag.ptr, 1, 0, None) == 0
    assert lib.cacg_k_gram_fast(n, dAQ.ptr, sm, sm, dS.ptr, sm, sm, None, 1, 0, w["as"], None, ws.ptr,
                                None) == 0
    assert lib.cacg_k_lu_solve(sm, w["g1"], sm, w["as"], w["b"], w["lu"], flag.ptr, 1, 1, None) == 0
    assert lib.cacg_k_gram_fast_f64f32(n, dAQ.ptr, sm, sm, dS32.ptr, sm, sm, None, 1, 0, w["as32"], None,
                                       ws.ptr, None) == 0
    assert lib.cacg_k_lu_solve(sm, w["g1"], sm, w["as32"], w["b32"], w["lu"], flag.ptr, 1, 1, None) == 0
    g = {k: b.ptr for k, b in got.items()}
    flag2 = D(np.zeros(1, dtype=np.int32))
    assert lib.cacg_k_gram_alpha(n, sm, m, dQ.ptr, dAQ.ptr, dR.ptr, g["g1"], g["g2"], g["x"], g["lu"],
                                 flag2.ptr, ws.ptr, None) == 0
    assert lib.cacg_k_gram_beta(n, sm, dAQ.ptr, dS.ptr, None, g["as"], g["b"], g["lu"], ws.ptr, None) == 0
    assert lib.cacg_k_gram_beta(n, sm, dAQ.ptr, None, dS32.ptr, g["as32"], g["b32"], g["lu"], ws.ptr,
                                None) == 0
    for k, b in got.items():
        sz = (b.nbytes // 8,)
        assert np.array_equal(b.download(sz), want[k].download(sz), equal_nan=True), k
    assert flag2.download((1,), np.int32)[0] == flag.download((1,), np.int32)[0]


@pytest.mark.parametrize("sm,m", [(9, 1), (8, 9), (0, 1), (4, 0)])
def test_gram_with_solve_refuses_wider_blocks(gpu_lib, sm, m):
    assert gpu_lib.lib().cacg_gram_solve_supported(sm, m) == 0
    assert gpu_lib.lib().cacg_k_gram_alpha(10, sm, m, *([None] * 10)) != 0


@pytest.mark.parametrize("N,k", [(1, 3), (2, 1), (15, 4), (16, 5), (17, 16), (32, 17), (47, 3), (60, 60),
                                 (64, 1), (79, 10), (96, 33), (100, 20), (112, 7), (127, 16), (128, 130)])
def test_lu_reference_edges_bitwise(gpu_lib, oracle_lib, N, k):
    rng = np.random.default_rng(N + k)
    M = rng.standard_normal((N, N))
    A, rhs = M @ M.T + N * np.eye(N), rng.standard_normal((N, k))
    print(f"reference solve N={N} k={k}", flush=True)
    x, flag = gpu_lib.k_lu_solve(A, rhs, mode="reference")
    assert flag == 0 and np.array_equal(x, oracle_lib.lu_solve(A, rhs))


@pytest.mark.parametrize("n", [1, 16, 33, 5000, 40007])
@pytest.mark.parametrize("k,lda", [(1, 1), (2, 5), (15, 15), (17, 20), (32, 32), (63, 64), (80, 80),
                                   (97, 97), (112, 114), (128, 128)])
def test_triangular_row_product_exact_on_integers(gpu_lib, n, k, lda):
    lib, D, rng = gpu_lib.lib(), gpu_lib.DeviceBuffer.from_array, np.random.default_rng(n + k)
    A = rng.integers(-8, 9, size=(n, lda)).astype(np.float64)
    W = np.triu(rng.integers(-8, 9, size=(k, k))).astype(np.float64)
    dA, dW, Q = D(A), D(W), gpu_lib.DeviceBuffer(8 * n * k)
    print(f"triangular row product n={n} k={k} lda={lda}", flush=True)
    assert lib.cacg_k_trimul_neg(n, k, dA.ptr, lda, Q.ptr, dW.ptr, None) == 0
    assert np.array_equal(Q.download((n, k)), -(A[:, :k] @ W))
    if lda == k:   # in place
        assert lib.cacg_k_trimul_neg(n, k, dA.ptr, lda, dA.ptr, dW.ptr, None) == 0
        assert np.array_equal(dA.download((n, k)), -(A @ W))


@pytest.mark.parametrize("n,sm,m", [(16, 16, 4), (15, 32, 8), (17, 48, 12), (2048 * 16 + 5, 64, 16),
                                    (4000, 96, 12), (4099, 112, 28), (33000, 128, 16), (5000, 128, 32),
                                    (3000, 64, 32)])
def test_q_update_whole_and_last_tiles_exact_on_integers(gpu_lib, n, sm, m):
    rng = np.random.default_rng(n + sm)
    S, Q = (rng.integers(-8, 9, size=(n, sm)).astype(np.float64) for _ in range(2))
    beta, alpha = (rng.integers(-8, 9, size=(sm, k)).astype(np.float64) for k in (sm, m))
    X = rng.integers(-8, 9, size=(n, m)).astype(np.float64)
    print(f"q update n={n} sm={sm} m={m}", flush=True)
    assert np.array_equal(gpu_lib.k_qupdate(S, Q, beta, mode="fast"), S - Q @ beta)
    Qn, Xn = gpu_lib.k_qxupdate(S, Q, beta, alpha, X)
    assert np.array_equal(Qn, S - Q @ beta) and np.array_equal(Xn, X + Q @ alpha)
    Qb, Xb = gpu_lib.k_qxupdate_blk(S, Q, beta, alpha, X, 0)
    assert np.array_equal(Qb, Qn) and np.array_equal(Xb, Xn)


@pytest.mark.parametrize("sm", [4, 8, 12, 16, 20, 96, 100, 128])
@pytest.mark.parametrize("n", [17, 5000])
def test_q_update_without_s_exact_on_integers(gpu_lib, n, sm):
    lib, D, rng = gpu_lib.lib(), gpu_lib.DeviceBuffer.from_array, np.random.default_rng(n + sm)
    Q = rng.integers(-8, 9, size=(n, sm)).astype(np.float64)
    beta = rng.integers(-8, 9, size=(sm, sm)).astype(np.float64)
    dQ, db = D(Q), D(beta)
    print(f"q update without S n={n} sm={sm}", flush=True)
    assert lib.cacg_k_qupdate_zero(n, sm, dQ.ptr, db.ptr, None) == 0
    assert np.array_equal(dQ.download((n, sm)), -(Q @ beta))


@pytest.mark.parametrize("which,tm,tn", [(0, 1, 2), (1, 2, 1), (1, 1, 4), (2, 1, 1), (1, 9, 9), (0, 0, 0)])
def test_batched_gram_class_refuses_what_is_no_class(gpu_lib, which, tm, tn):
    assert gpu_lib.lib().cacg_kb_gram_class(None, None, 1, which, 0, tm, tn, None) != 0


@pytest.mark.parametrize("n,kl,kr1,kr2,ld2", [(130, 6, 6, 2, 9), (600011, 4, 4, 2, 16),
                                              (600011, 2, 2, 1, 12), (530001, 3, 5, 3, 8)])
def test_gram_fast_strided_second_block_exact_on_integers(gpu_lib, n, kl, kr1, kr2, ld2):
    """R2 as columns of a wider block, with chunks of few rows and of more than 1023."""
    lib, D, rng = gpu_lib.lib(), gpu_lib.DeviceBuffer.from_array, np.random.default_rng(n + kl)
    L, R1, R2 = (rng.integers(-8, 9, size=(n, k)).astype(np.float64) for k in (kl, kr1, ld2))
    dL, d1, d2 = D(L), D(R1), D(R2)
    g1, g2 = gpu_lib.DeviceBuffer(8 * kl * kr1), gpu_lib.DeviceBuffer(8 * kl * kr2)
    ws = gpu_lib.DeviceBuffer(8 * lib.cacg_gram_workspace(kl, kr1 + kr2))
    print(f"gram n={n} {kl} x ({kr1} + {kr2} of {ld2})", flush=True)
    assert lib.cacg_k_gram_fast(n, dL.ptr, kl, kl, d1.ptr, kr1, kr1, d2.ptr, ld2, kr2, g1.ptr, g2.ptr,
                                ws.ptr, None) == 0
    assert np.array_equal(g1.download((kl, kr1)), L.T @ R1)
    assert np.array_equal(g2.download((kl, kr2)), L.T @ R2[:, :kr2])


@pytest.mark.parametrize("n,kl,kr1,kr2", [(100003, 99, 99, 11), (150001, 61, 61, 7), (200003, 127, 127, 0),
                                          (120001, 81, 81, 0)])
def test_gram_many_stages_of_odd_widths_exact_on_integers(gpu_lib, n, kl, kr1, kr2):
    """Chunks of 18 to 29 whole stages and a part of one, pairs that start a column early: 2 x 2,
    1 x 4 and 1 x 3 tiles in 16 waves, 1 x 5 in 8."""
    test_gram_fast_edges_exact_on_integers(gpu_lib, n, kl, kr1, kr2)


@pytest.mark.parametrize("n,sm,m", [
    (131072, 6, 2), (131073, 6, 2), (131073, 3, 3), (131073, 10, 2), (262144, 5, 5), (262145, 5, 5),
    (1 << 20, 12, 1), ((1 << 20) + 1, 12, 1), (1 << 21, 9, 3), (1 << 21, 8, 8), (1024, 100, 20),
    (1025, 100, 20), (2304, 72, 12), (2305, 72, 12), (512, 127, 1), (513, 127, 1)])
def test_updates_at_the_lines_between_the_kernels_exact_on_integers(gpu_lib, n, sm, m):
    """Row counts on both sides of the lines where another kernel takes over."""
    test_padded_updates_exact_on_integers(gpu_lib, n, sm, m)


@pytest.mark.parametrize("n,k", [(600011, 60), (70001, 47), (40003, 100), (5000, 128), (9001, 33)])
def test_gram_f64f32_part_waves_exact_on_integers(gpu_lib, n, k):
    """Rows of L that end inside a wave's lanes: R1's vectors start at the next wave."""
    test_gram_f64f32_edges_exact_on_integers(gpu_lib, n, k)


@pytest.mark.parametrize("n,kl,kr1,kr2", [
    # the direct kernel and, past its rows, the tile kernel; several batches a wave, a ragged last chunk
    (262144, 32, 32, 31), (262145, 32, 32, 31), (250001, 3, 2, 1), (100003, 17, 30, 3),
    # few workgroups: halved blocks, some with a single column left over
    (200, 112, 112, 16), (300, 33, 33, 3), (2000, 100, 100, 20), (1000, 160, 160, 32), (900, 97, 97, 1),
    # chunks of 128 rows for large partials; whole 16-row stages a chunk at 128 columns
    (3073, 256, 256, 32), (5000, 192, 192, 32), (140000, 128, 128, 16)])
def test_gram_few_rows_exact_on_integers(gpu_lib, n, kl, kr1, kr2):
    test_gram_fast_edges_exact_on_integers(gpu_lib, n, kl, kr1, kr2)


@pytest.mark.parametrize("n,k", [(131072, 32), (131073, 32), (1000, 30), (64, 17), (2001, 25)])
def test_gram_f64f32_few_rows_exact_on_integers(gpu_lib, n, k):
    test_gram_f64f32_edges_exact_on_integers(gpu_lib, n, k)
