"""FP64 logistic-regression gradient beyond 128 coefficients (the column-split
matrix-core kernel) against the closed form in numpy, at the edges of its tiles:
column slices of 16 x 4 / 8 tiles per wave, 16-row tiles, 16-point groups, and the
host entry against the sampler's lockstep transition."""
import ctypes as C

import numpy as np
import pytest

import cmdstan_amd as ca
from cmdstan_amd._lib import last_error, lib
from oracle import oracle as O
from tests.model_cases import logistic

pytestmark = pytest.mark.gpu


def _closed_form(d, q):
    eta = d["X"] @ q.T
    lp = (d["y"][:, None] * eta - np.logaddexp(0, eta)).sum(axis=0) - 0.5 * (q * q).sum(axis=1) / 6.25
    return lp, (d["X"].T @ (d["y"][:, None] - 1 / (1 + np.exp(-eta)))).T - q / 6.25


@pytest.mark.parametrize("N,D,n", [(1, 129, 1), (17, 255, 16), (1000, 256, 17), (333, 257, 3), (5000, 500, 64),
                                   (64, 512, 33), (130, 513, 1), (700, 1000, 5), (15, 1024, 130)])
def test_wide_gradient(N, D, n):
    d = logistic(seed=N + D, N=N, D=D)
    q = 0.3 * np.random.default_rng(D).standard_normal((n, D))
    lp, g = ca.Model("logistic_regression", d).log_prob_grad(q)
    lp0, g0 = _closed_form(d, q)
    # sums of N terms of size |x| <= 6: rounding below 1e-15 of the sum of magnitudes
    scale = np.abs(d["X"]).sum(axis=0).max() + 1.0
    assert np.abs(g - g0).max() <= 1e-13 * scale
    assert np.abs(lp - lp0).max() <= 1e-13 * (np.abs(d["X"] @ q.T).sum(axis=0).max() + N + 1.0)


def test_wide_gradient_scratch_limit():
    """More points than the allocation-free entry has partial sums for: one chunk per group, G written directly."""
    D, n = 600, 4096
    d = logistic(seed=5, N=90, D=D)
    q = 0.1 * np.random.default_rng(3).standard_normal((n, D))
    m = ca.Model("logistic_regression", d)
    hip = C.CDLL("libamdhip64.so.7")
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    hip.hipFree.argtypes = [C.c_void_p]
    bufs = []
    for nbytes in (q.nbytes, 8 * n, q.nbytes):
        p = C.c_void_p()
        assert hip.hipMalloc(C.byref(p), nbytes) == 0
        bufs.append(p)
    assert hip.hipMemcpy(bufs[0], q.ctypes.data_as(C.c_void_p), q.nbytes, 1) == 0
    assert lib().nuts_log_prob_grad_noalloc(m.h, 0, bufs[0], n, 1, bufs[1], bufs[2], None) == 0, last_error()
    assert hip.hipDeviceSynchronize() == 0
    lp, g = np.empty(n), np.empty((n, D))
    assert hip.hipMemcpy(lp.ctypes.data_as(C.c_void_p), bufs[1], lp.nbytes, 2) == 0
    assert hip.hipMemcpy(g.ctypes.data_as(C.c_void_p), bufs[2], g.nbytes, 2) == 0
    for p in bufs:
        hip.hipFree(p)
    lp0, g0 = _closed_form(d, q)
    assert np.abs(g - g0).max() <= 1e-13 * (np.abs(d["X"]).sum(axis=0).max() + 1.0)
    assert np.abs(lp - lp0).max() <= 1e-13 * (np.abs(d["X"] @ q.T).sum(axis=0).max() + 91.0)


@pytest.mark.parametrize("driver", ["fused", "lockstep", "lockstep_block"])
def test_wide_transition_replay(driver):
    d = logistic(seed=8, N=400, D=150)
    rng = np.random.default_rng(2)
    nch = 5
    q0 = 0.2 * rng.standard_normal((nch, 150))
    u, z = rng.random((nch, 2048)), rng.standard_normal((nch, 150))
    m, o = ca.Model("logistic_regression", d), O.Model("logistic_regression", d)
    q, info = m.transition_replay(q0, u, z, 0.05, driver=driver)
    for k in range(nch):
        qo, io = o.transition_replay(q0[k], u[k], z[k], 0.05, metric=1, minv=np.ones(150))
        assert (info[k]["depth"], info[k]["n_leapfrog"]) == (io["depth"], io["n_leapfrog"])
        assert np.allclose(q[k], qo, rtol=1e-10, atol=1e-12)


@pytest.mark.parametrize("N,D", [(10000, 500), (3000, 200)])
def test_wide_gradient_against_extended_precision(N, D):
    """The error against 80-bit sums is no larger than that of the same closed form in 64 bits."""
    d = logistic(seed=11, N=N, D=D)
    rng = np.random.default_rng(4)
    q = np.linalg.lstsq(d["X"], 3.0 * (d["y"] - 0.5), rcond=None)[0] + np.sqrt(5.0 / N) * rng.standard_normal((4, D))
    X, Q = d["X"].astype(np.longdouble), q.astype(np.longdouble)
    eta = X @ Q.T
    g_ext = (X.T @ (d["y"][:, None] - 1 / (1 + np.exp(-eta)))).T - Q / np.longdouble(6.25)
    _, g = ca.Model("logistic_regression", d).log_prob_grad(q)
    g64 = _closed_form(d, q)[1]
    err, err64 = (float(np.linalg.norm(v - g_ext) / np.linalg.norm(g_ext)) for v in (g, g64))
    print(f"error {err:.2e}, in 64 bits {err64:.2e}")
    assert err <= err64
