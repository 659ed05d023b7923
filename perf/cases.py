"""The work this library is asked for, as cases that can be timed and compared.

Each case names a kind of call and its sizes:

  solve            a whole device-resident solve (cacg_solver_solve_device), x0 = 0 to 1e-10
  reference        the drop-in's solve: host arrays in and out, the reference's summation order
  batch            many small systems through the batching engine, submission to last result
  basis            the Chebyshev basis of one outer iteration (s - 1 fused SpMM steps)
  aq               the A Q product of one outer iteration
  gram             [Q^T A Q | Q^T R] of one outer iteration, fast order
  gram_reference   the same sums in the reference's order
  update           Q = S - Q beta, X += Q alpha, R -= A Q alpha and the column norms, fast order
  coefficients     alpha = G^{-1} Q^T R, then beta = G^{-1} Q^T A S on the kept factor
  tsqr             the tall-skinny QR

listed() are fixed cases, draw() gives others of the same ranges, prepare() makes what a program
holds before the call, run() is one call, work() its least bytes and operations, exact() its result
in 64 bits from torch alone.
"""

import ctypes
import math
from types import SimpleNamespace

import numpy as np
import torch

import cacg_amd
from cacg_amd import batch as cbatch
from cacg_amd import problems

DEV = "cuda"
TOL = 1e-10
EPI_NONE, EPI_CHEB1, EPI_CHEB = 0, 2, 3


def listed():
    return [
        # one right-hand side on a small grid: every launch and synchronisation counts
        {"name": "solve-2d128-m1-s4", "kind": "solve", "grid": 2, "edge": 128, "m": 1, "s": 4,
         "bounds": "lanczos", "precision": "fp64"},
        # the benchmark's workload: 2.1M rows, 16 right-hand sides
        {"name": "solve-3d128-m16-s8", "kind": "solve", "grid": 3, "edge": 128, "m": 16, "s": 8,
         "bounds": "gerschgorin", "precision": "fp64"},
        # bcbcg_v1 as shipped: host arrays, the reference's summation order
        {"name": "reference-3d64-m16-s8", "kind": "reference", "grid": 3, "edge": 64, "m": 16,
         "s": 8},
        # a service's burst of small systems, FP32 basis with FP64 refinement
        {"name": "batch-64", "kind": "batch", "count": 64, "lmin": 32, "lmax": 256, "sizes": 3,
         "s": 4, "precision": "fp32"},
        # the bandwidth-bound part of the benchmark's iteration
        {"name": "basis-3d128-m16-s8", "kind": "basis", "grid": 3, "edge": 128, "m": 16, "s": 8,
         "matrix": "laplacian", "precision": "fp64"},
        {"name": "aq-3d128-k128", "kind": "aq", "grid": 3, "edge": 128, "k": 128,
         "matrix": "laplacian"},
        # the matrix-core part
        {"name": "gram-2097152-m16-s8", "kind": "gram", "n": 2097152, "m": 16, "s": 8},
        # ragged: 63^3 rows, a basis of 60 columns
        {"name": "update-250047-m10-s6", "kind": "update", "n": 250047, "m": 10, "s": 6},
        # the small dense solves, serial by nature: 128 unknowns, and the widest block
        {"name": "coefficients-m16-s8", "kind": "coefficients", "m": 16, "s": 8, "order": "fast"},
        {"name": "coefficients-m32-s8", "kind": "coefficients", "m": 32, "s": 8, "order": "fast"},
        # most of a reference-order iteration
        {"name": "gram-reference-262144-m16-s8", "kind": "gram_reference", "n": 262144, "m": 16,
         "s": 8},
        {"name": "tsqr-300000-k96", "kind": "tsqr", "n": 300000, "k": 96},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _block(rng, widest):
    """(m, s) with s m at most `widest`: 1 to 32 right-hand sides, basis length 2 to 8."""
    while True:
        m = rng.choice([1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32])
        s = rng.randint(2, 8)
        if m * s <= widest:
            return m, s


def draw(rng):
    kind = rng.choice(["solve", "solve", "reference", "batch", "basis", "aq", "gram",
                       "gram_reference", "update", "coefficients", "tsqr"])
    if kind in ("solve", "reference"):
        grid = rng.choice([2, 3])
        edge = _log_int(rng, 40, 256) if grid == 2 else _log_int(rng, 16, 96)
        if kind == "reference":
            edge = min(edge, 64) if grid == 3 else edge
        m = rng.choice([1, 2, 3, 4, 5, 8, 10, 16])
        s = rng.randint(3, 6)
        if kind == "reference":
            return {"kind": kind, "grid": grid, "edge": edge, "m": m, "s": s}
        return {"kind": kind, "grid": grid, "edge": edge, "m": m, "s": s,
                "bounds": rng.choice(["gerschgorin", "lanczos"]),
                "precision": rng.choice(["fp64", "fp64", "fp32"])}
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(16, 64), "lmin": 32,
                "lmax": _log_int(rng, 64, 256), "sizes": rng.randint(1, 9999),
                "s": rng.choice([3, 4]), "precision": rng.choice(["fp32", "fp64"])}
    if kind in ("basis", "aq"):
        grid = rng.choice([2, 3])
        edge = _log_int(rng, 64, 1024) if grid == 2 else _log_int(rng, 24, 128)
        matrix = rng.choice(["laplacian", "laplacian", "random"])
        m, s = _block(rng, 128)
        if kind == "aq":
            if rng.random() < 0.2:  # rows of very different lengths
                return {"kind": kind, "grid": 2, "edge": _log_int(rng, 64, 512), "k": m * s,
                        "matrix": "power"}
            return {"kind": kind, "grid": grid, "edge": edge, "k": m * s, "matrix": matrix}
        return {"kind": kind, "grid": grid, "edge": edge, "m": m, "s": max(s, 3),
                "matrix": matrix, "precision": rng.choice(["fp64", "fp64", "fp32"])}
    if kind == "coefficients":
        m, s = _block(rng, 256)
        return {"kind": kind, "m": m, "s": s, "order": rng.choice(["fast", "fast", "reference"])}
    if kind == "tsqr":
        return {"kind": kind, "n": _log_int(rng, 2000, 1000000), "k": rng.randint(4, 128)}
    m, s = _block(rng, 128)
    top = 300000 if kind == "gram_reference" else 2097152
    return {"kind": kind, "n": _log_int(rng, 4096, top), "m": m, "s": s}


# ---- preparation ---------------------------------------------------------------------


def _matrix(case, seed):
    edge = case["edge"]
    if case.get("matrix") == "power":
        return problems.power_law_spd(edge, 16, edge * edge // 64, 5)
    A = problems.laplacian_2d(edge) if case["grid"] == 2 else problems.laplacian_3d(edge)
    return problems.random_spd_like(A, seed) if case.get("matrix") == "random" else A


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float64)


def _empty(*shape, dtype=torch.float64):
    return torch.empty(*shape, device=DEV, dtype=dtype)


def _interval(A):
    """Gerschgorin interval of A."""
    rows = np.repeat(np.arange(A.n), np.diff(A.rowptr))
    diag = np.zeros(A.n)
    diag[rows[A.col == rows]] = A.val[A.col == rows]
    off = np.add.reduceat(np.abs(A.val), A.rowptr[:-1]) - np.abs(diag)
    return float((diag - off).min()), float((diag + off).max())


def _tsqr_input(case, seed):
    g = _gen(seed)
    k = case["k"]
    scale = torch.pow(10.0, torch.rand(k, generator=g, device=DEV, dtype=torch.float64) * 2 - 1)
    return _randn(g, case["n"], k) * scale


def _coeff_input(case, seed):
    """A Gram matrix of a random basis with columns of uneven length, and two right-hand sides."""
    n, m = case["m"] * case["s"], case["m"]
    g = torch.Generator().manual_seed(seed)
    V = torch.randn(4 * n, n, generator=g, dtype=torch.float64)
    V *= torch.pow(10.0, torch.rand(n, generator=g, dtype=torch.float64) * 2 - 1)
    G = (V.T @ V) / (4 * n)
    R = torch.randn(n, m, generator=g, dtype=torch.float64)
    B = torch.randn(n, n, generator=g, dtype=torch.float64)
    return G.contiguous(), R, B


def _gram_input(case, seed):
    g = _gen(seed)
    n, m, sm = case["n"], case["m"], case["m"] * case["s"]
    return _randn(g, n, sm), _randn(g, n, sm), _randn(g, n, m)


def _update_input(case, seed):
    """S, Q, A Q, beta, alpha, X, R; beta a contraction, as of a converging recurrence."""
    g = _gen(seed)
    n, m, sm = case["n"], case["m"], case["m"] * case["s"]
    beta = _randn(g, sm, sm) * (0.25 / math.sqrt(sm))
    alpha = _randn(g, sm, m) / math.sqrt(sm)
    return (_randn(g, n, sm), _randn(g, n, sm), _randn(g, n, sm), beta, alpha, _randn(g, n, m),
            _randn(g, n, m))


def _batch_systems(case):
    return problems.sample_batch_systems(case["count"], case["sizes"], case["lmin"], case["lmax"])


def _batch_rhs(case, seed):
    rng = np.random.default_rng(seed)
    return [rng.random((L * L, m)) for L, _, m in _batch_systems(case)]


def _rhs(case, seed):
    return np.random.default_rng(seed).random((case["edge"] ** case["grid"], case["m"]))


def prepare(case, seed):
    st = SimpleNamespace(kind=case["kind"], case=case, L=cacg_amd.lib())
    kind = case["kind"]
    if kind == "solve":
        A = _matrix(case, seed)
        st.solver = cacg_amd.Solver(A, case["m"], case["s"], tol=TOL, maxiter=1000, order="fast",
                                    bounds=case["bounds"], precision=case["precision"])
        st.B = torch.from_numpy(_rhs(case, seed)).to(DEV)
        st.X = torch.zeros_like(st.B)
        st.dB, st.dX = (SimpleNamespace(ptr=t.data_ptr()) for t in (st.B, st.X))
    elif kind == "reference":
        st.A = _matrix(case, seed)
        st.B = _rhs(case, seed)
        st.X0 = np.zeros_like(st.B)
        st.eps = TOL * float(np.linalg.norm(st.B[:, 0]))
    elif kind == "batch":
        st.systems = [(problems.laplacian_2d(L, shift), B) for (L, shift, _), B in
                      zip(_batch_systems(case), _batch_rhs(case, seed))]
        st.batch = cbatch.Batch(s=case["s"], precision=case["precision"], hbm_bytes=8 << 30)
    elif kind in ("basis", "aq"):
        A = _matrix(case, seed)
        st.A = cacg_amd.DeviceCSR(A)
        g = _gen(seed)
        if kind == "aq":
            st.X = _randn(g, A.n, case["k"])
            st.Y = torch.empty_like(st.X)
        else:
            lo, hi = _interval(A)
            st.a, st.b = 2.0 / (hi - lo), -(hi + lo) / (hi - lo)
            st.f32 = case["precision"] == "fp32"
            st.mat = st.A.s32 if st.f32 else st.A.s
            st.R = _randn(g, A.n, case["m"])
            st.S = _empty(case["s"], A.n, case["m"], dtype=torch.float32 if st.f32 else torch.float64)
    elif kind in ("gram", "gram_reference"):
        st.Q, st.AQ, st.R = _gram_input(case, seed)
        sm, m = st.Q.shape[1], st.R.shape[1]
        st.G1, st.G2 = _empty(sm, sm), _empty(sm, m)
        st.ws = _empty(st.L.cacg_gram_workspace(sm, sm + m))
    elif kind == "update":
        S, st.Q, st.AQ, st.beta, st.alpha, st.X, st.R = _update_input(case, seed)
        n, m, s = case["n"], case["m"], case["s"]
        st.split = bool(st.L.cacg_k_split_supported(m * s, m))
        st.blocks = st.split and m % 4 == 0
        st.S = S.reshape(n, s, m).permute(1, 0, 2).contiguous() if st.blocks else S
        st.norm2 = _empty(m)
        st.ws = _empty(st.L.cacg_xrupdate_workspace(m))
    elif kind == "coefficients":
        G, R, B = _coeff_input(case, seed)
        st.G, st.R, st.B = G.to(DEV), R.to(DEV), B.to(DEV)
        st.alpha, st.beta = torch.empty_like(st.R), torch.empty_like(st.B)
        st.factor = torch.empty_like(st.G)
        st.flag = torch.zeros(1, device=DEV, dtype=torch.int32)
    elif kind == "tsqr":
        st.A = _tsqr_input(case, seed)
        k = case["k"]
        st.Q, st.R = torch.empty_like(st.A), _empty(k, k)
        st.ws = _empty(st.L.cacg_tsqr_workspace(k))
        st.flag = torch.zeros(1, device=DEV, dtype=torch.int32)
    else:
        raise ValueError(kind)
    return st


# ---- one call ------------------------------------------------------------------------


def _ok(rc):
    if rc != 0:
        raise RuntimeError(f"call failed with code {rc}")


def _run_basis(st, stream):
    m, s, L, S = st.case["m"], st.case["s"], st.L, st.S
    mat, blk = ctypes.byref(st.mat), [S[j].data_ptr() for j in range(s)]
    a, b = st.a, st.b
    if st.f32:
        _ok(L.cacg_k_cheb1_f32(mat, m, st.R.data_ptr(), m, blk[1], m, blk[0], m, a, b, stream))
        for j in range(2, s):
            _ok(L.cacg_k_spmm_f32(mat, m, blk[j - 1], m, blk[j], m, EPI_CHEB, 2 * a, 2 * b,
                                  blk[j - 1], m, blk[j - 2], m, stream))
    else:
        _ok(L.cacg_k_spmm(mat, m, st.R.data_ptr(), m, blk[1], m, EPI_CHEB1, a, b, None, m, None, m,
                          blk[0], m, stream))
        for j in range(2, s):
            _ok(L.cacg_k_spmm(mat, m, blk[j - 1], m, blk[j], m, EPI_CHEB, 2 * a, 2 * b, blk[j - 1],
                              m, blk[j - 2], m, None, m, stream))
    return S


def _run_update(st, stream):
    n, m, L = st.case["n"], st.case["m"], st.L
    sm = m * st.case["s"]
    S, Q, AQ, beta, alpha, X, R, norm2, ws = (
        t.data_ptr() for t in (st.S, st.Q, st.AQ, st.beta, st.alpha, st.X, st.R, st.norm2, st.ws))
    if st.blocks:
        _ok(L.cacg_k_qxupdate_blk(n, sm, m, S, n * m, Q, beta, alpha, X, stream))
    elif st.split:
        _ok(L.cacg_k_qxupdate(n, sm, m, S, Q, beta, alpha, X, stream))
    if st.split:
        _ok(L.cacg_k_xrupdate_split(n, sm, m, None, AQ, alpha, None, R, norm2, ws, 2, stream))
    else:
        _ok(L.cacg_k_qupdate(n, sm, S, Q, beta, 1, stream))
        _ok(L.cacg_k_xrupdate(n, sm, m, Q, AQ, alpha, X, R, norm2, ws, 1, stream))
    return {"Q": st.Q, "X": st.X, "R": st.R, "norm2": st.norm2}


def run(st):
    case, kind = st.case, st.kind
    if kind == "solve":
        st.X.zero_()
        st.solver.solve(st.dB, st.dX)
        return st.X
    if kind == "reference":
        return cacg_amd.bcbcg(st.A, st.B, st.X0, case["s"], stop_mode=0, eps=st.eps, maxiter=1000,
                              order="reference")["X"]
    if kind == "batch":
        ids = [st.batch.submit(A, B, tol=TOL) for A, B in st.systems]
        out = st.batch.run()
        return [out[i]["X"] for i in ids]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "basis":
        return _run_basis(st, stream)
    if kind == "aq":
        k = case["k"]
        _ok(st.L.cacg_k_spmm(ctypes.byref(st.A.s), k, st.X.data_ptr(), k, st.Y.data_ptr(), k,
                             EPI_NONE, 0.0, 0.0, None, k, None, k, None, k, stream))
        return st.Y
    if kind == "update":
        return _run_update(st, stream)
    if kind == "coefficients":
        m, N = case["m"], case["m"] * case["s"]
        mode = cacg_amd.MODE[case["order"]]
        _ok(st.L.cacg_k_lu_solve(N, st.G.data_ptr(), m, st.R.data_ptr(), st.alpha.data_ptr(),
                                 st.factor.data_ptr(), st.flag.data_ptr(), mode, 0, stream))
        _ok(st.L.cacg_k_lu_solve(N, st.G.data_ptr(), N, st.B.data_ptr(), st.beta.data_ptr(),
                                 st.factor.data_ptr(), st.flag.data_ptr(), mode, 1, stream))
        return {"alpha": st.alpha, "beta": st.beta, "flag": st.flag}
    if kind == "tsqr":
        n, k = case["n"], case["k"]
        _ok(st.L.cacg_k_tsqr(n, k, st.A.data_ptr(), k, st.Q.data_ptr(), st.R.data_ptr(),
                             st.ws.data_ptr(), st.flag.data_ptr(), stream))
        return {"Q": st.Q, "R": st.R, "flag": st.flag}
    n, m = case["n"], case["m"]
    sm = m * case["s"]
    args = (n, st.Q.data_ptr(), sm, sm, st.AQ.data_ptr(), sm, sm, st.R.data_ptr(), m, m,
            st.G1.data_ptr(), st.G2.data_ptr())
    if kind == "gram":
        _ok(st.L.cacg_k_gram_fast(*args, st.ws.data_ptr(), stream))
    else:
        _ok(st.L.cacg_k_gram_ref(*args, stream))
    return {"QtAQ": st.G1, "QtR": st.G2}


# ---- least work ----------------------------------------------------------------------


def _iteration(n, nnz, m, s):
    """(bytes, flops) of one outer iteration: the matrix once per product, each block once per use."""
    sm = s * m
    by = (s * (12 * nnz + 4 * n) + 8 * n * (3 * m * (s - 1) + 2 * sm)      # basis, A Q
          + 8 * n * (2 * sm + m) + 16 * n * sm                             # both Gram blocks
          + 8 * n * (3 * sm + 2 * m) + 8 * n * (sm + 2 * m))               # Q and X, R
    fl = (2 * nnz * (m * (s - 1) + sm) + 2 * n * sm * (2 * sm + m) + 2 * n * sm * sm
          + 4 * n * sm * m + 4 * sm ** 3)
    return by, fl


def work(case):
    kind = case["kind"]
    if kind in ("solve", "reference"):
        d, e, m, s = case["grid"], case["edge"], case["m"], case["s"]
        n = e ** d
        by, fl = _iteration(n, (2 * d + 1) * n, m, s)
        # conjugate gradients from cold takes about 3 edge steps, s of them an iteration, fewer in
        # a block
        it = max(3.0, 3.0 * e / s / m ** 0.15)
        return {"bytes": it * by, "flops": it * fl}
    if kind == "batch":
        by = fl = 0.0
        for L, shift, m in _batch_systems(case):
            b, f = _iteration(L * L, 5 * L * L, m, case["s"])
            it = max(3.0, 20.0 / math.sqrt(shift + 10.0 / (L * L)) / case["s"] / m ** 0.15)
            by, fl = by + it * b, fl + it * f
        return {"bytes": by, "flops": fl}
    if kind in ("basis", "aq"):
        n = case["edge"] ** case["grid"]
        nnz = (2 * case["grid"] + 1) * n
        if kind == "aq":
            return {"bytes": 12 * nnz + 4 * n + 16 * n * case["k"], "flops": 2 * nnz * case["k"]}
        m, s = case["m"], case["s"]
        w = 4 if case["precision"] == "fp32" else 8
        return {"bytes": (s - 1) * ((4 + w) * nnz + 4 * n) + 8 * n * m + w * n * m * (3 * s - 4),
                "flops": 2 * (s - 1) * (nnz + 2 * n) * m}
    if kind == "coefficients":
        m, N = case["m"], case["m"] * case["s"]
        return {"bytes": 8 * (N * N + 2 * N * m + 2 * N * N),
                "flops": 2 * N ** 3 / 3 + 2 * N * N * (m + N)}
    if kind == "tsqr":
        n, k = case["n"], case["k"]
        return {"bytes": 16 * n * k + 8 * k * k, "flops": 4 * n * k * k}
    n, m = case["n"], case["m"]
    sm = m * case["s"]
    if kind == "update":
        return {"bytes": 8 * (4 * n * sm + 4 * n * m + sm * sm + sm * m),
                "flops": 2 * n * sm * (sm + 2 * m)}
    return {"bytes": 8 * (n * (2 * sm + m) + sm * (sm + m)), "flops": 2 * n * sm * (sm + m)}


# ---- the results in 64 bits ----------------------------------------------------------


def _poisson(grid, edge, B, shift=0.0):
    """(Laplacian + shift)^{-1} B by the sine transform that diagonalises it."""
    m = B.shape[1]
    k = torch.arange(1, edge + 1, dtype=torch.float64, device=B.device)
    F = torch.sin(torch.outer(k, k) * (math.pi / (edge + 1))) * math.sqrt(2.0 / (edge + 1))
    ev = 2.0 - 2.0 * torch.cos(k * (math.pi / (edge + 1)))
    lam = ev[:, None] + ev if grid == 2 else ev[:, None, None] + ev[:, None] + ev

    def transform(T):
        for _ in range(grid):  # each axis in turn to the front, transformed, then put last
            T = torch.tensordot(T, F, dims=([0], [0]))
        return T

    T = B.reshape(*([edge] * grid), m).movedim(-1, 0)
    out = [transform(transform(T[c]) / (lam + shift)).reshape(-1) for c in range(m)]
    return torch.stack(out, dim=1)


def _sparse(A):
    return torch.sparse_csr_tensor(torch.from_numpy(A.rowptr), torch.from_numpy(A.col),
                                   torch.from_numpy(A.val), size=(A.n, A.n)).to(DEV)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("solve", "reference"):
        return _poisson(case["grid"], case["edge"], torch.from_numpy(_rhs(case, seed)).to(DEV))
    if kind == "batch":
        return [_poisson(2, L, torch.from_numpy(B).to(DEV), shift)
                for (L, shift, _), B in zip(_batch_systems(case), _batch_rhs(case, seed))]
    if kind in ("basis", "aq"):
        A = _matrix(case, seed)
        M, g = _sparse(A), _gen(seed)
        if kind == "aq":
            return M @ _randn(g, A.n, case["k"])
        lo, hi = _interval(A)
        a, b = 2.0 / (hi - lo), -(hi + lo) / (hi - lo)
        S = [_randn(g, A.n, case["m"])]
        S.append(a * (M @ S[0]) + b * S[0])
        for _ in range(2, case["s"]):
            S.append(2 * a * (M @ S[-1]) + 2 * b * S[-1] - S[-2])
        S = torch.stack(S)
        return S.float() if case["precision"] == "fp32" else S
    if kind in ("gram", "gram_reference"):
        Q, AQ, R = _gram_input(case, seed)
        return {"QtAQ": Q.T @ AQ, "QtR": Q.T @ R}
    if kind == "update":
        S, Q, AQ, beta, alpha, X, R = _update_input(case, seed)
        m = case["m"]
        new = S - Q @ beta
        # with the split kernels X takes the old Q, one iteration late
        X = X + (Q if cacg_amd.lib().cacg_k_split_supported(m * case["s"], m) else new) @ alpha
        R = R - AQ @ alpha
        return {"Q": new, "X": X, "R": R, "norm2": (R * R).sum(0)}
    if kind == "coefficients":
        G, R, B = _coeff_input(case, seed)
        return {"alpha": torch.linalg.solve(G, R), "beta": torch.linalg.solve(G, B), "flag": None}
    if kind == "tsqr":
        Q, R = torch.linalg.qr(_tsqr_input(case, seed).cpu())
        d = torch.sign(torch.diagonal(R))
        return {"Q": Q * d, "R": R * d[:, None], "flag": None}
    return None
