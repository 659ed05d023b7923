"""A default route must not take longer than another one that the caller could name for the same
call.  Both run in turn; the factors leave room for noise, the cases once differed by 2 and more."""

import ctypes
import time

import numpy as np
import pytest

from cacg_amd import problems as P

pytestmark = pytest.mark.gpu


def best_seconds(lib_sync, *calls, launches=10, rounds=7):
    """The shortest time of `launches` launches of each call, the calls in turn."""
    best = [1e9] * len(calls)
    for _ in range(rounds):
        for i, call in enumerate(calls):
            lib_sync()
            t = time.perf_counter()
            for _ in range(launches):
                assert call() == 0
            lib_sync()
            best[i] = min(best[i], time.perf_counter() - t)
    return best


@pytest.mark.parametrize("k", [16, 128])
def test_default_spmm_order_on_uneven_rows(gpu_lib, k):
    """Rows of 1 to 250 nonzeros, none long enough to be split: the default order against bands."""
    n, rng = 1 << 18, np.random.default_rng(3)
    lens = np.minimum(250, np.maximum(1, (rng.pareto(1.2, n) * 3).astype(int)))
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    col = np.clip(np.repeat(np.arange(n), lens) + rng.integers(-2000, 2000, rp[-1]), 0, n - 1)
    A = gpu_lib.DeviceCSR(P.CSR(n=n, rowptr=rp, col=col.astype(np.int64), val=rng.random(rp[-1])))
    B, lib = gpu_lib.DeviceBuffer, gpu_lib.lib()
    X, Y = B.from_array(rng.random((n, k))), B(8 * n * k)
    bands = gpu_lib.SpmmSched(8192 if k <= 32 else 4096, 0, 0)
    run = lambda s: lib.cacg_k_spmm_x(ctypes.byref(A.s), k, X.ptr, k, Y.ptr, k, 0, 0.0, 0.0, None, k,  # noqa: E731
                                      None, k, None, k, s, None)
    print(f"spmm uneven rows k={k}", flush=True)
    default, named = best_seconds(lambda: Y.download(1), lambda: run(None),
                                  lambda: run(ctypes.byref(bands)))
    assert default < 1.3 * named, (default, named)


@pytest.mark.parametrize("sm", [1, 2, 3])
def test_fast_order_q_update_of_few_columns(gpu_lib, sm):
    """Against the reference order, whose kernel forms the same products one by one."""
    n, B, lib = 1 << 20, gpu_lib.DeviceBuffer, gpu_lib.lib()
    S, Q, beta = (B.from_array(np.ones(s)) for s in ((n, sm), (n, sm), (sm, sm)))
    run = lambda mode: lib.cacg_k_qupdate(n, sm, S.ptr, Q.ptr, beta.ptr, mode, None)  # noqa: E731
    print(f"q update sm={sm}", flush=True)
    fast, ref = best_seconds(lambda: Q.download(1), lambda: run(gpu_lib.MODE["fast"]),
                             lambda: run(gpu_lib.MODE["reference"]), launches=40)
    assert fast < 1.5 * ref, (fast, ref)
