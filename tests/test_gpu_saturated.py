"""Log density where the observations saturate: log(1 + e^-|eta|) far below the rounding of 1.

The FP64 kernels sum these terms as the logarithm of a product; a product of rounded 1 + t loses
what of t lies below 2^-53.  The exact value here is a sum of log1p of 80-bit terms, and the linear
predictors are sums of positive terms, so their own rounding is known."""
import numpy as np
import pytest

import cmdstan_amd as ca

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53


def exact_terms(X, q, y):
    """sum_n log1p(e^-|eta_n|) of every point; every row is classified correctly."""
    eta = X.astype(np.longdouble) @ q.T.astype(np.longdouble)
    assert np.all((eta > 0) == (y[:, None] == 1))
    return np.log1p(np.exp(-np.abs(eta))).sum(axis=0)


@pytest.mark.parametrize("lo,hi", [(20.0, 60.0), (36.8, 60.0)])
@pytest.mark.parametrize("points", [3, 40])
@pytest.mark.parametrize("D", [1, 7, 100, 200])
def test_saturated_rows_glm(D, points, lo, hi):
    rng = np.random.default_rng(D + points)
    N = 3001
    q = 1e-3 * rng.uniform(0.9, 1.0, (points, D))
    X = rng.uniform(0.5, 1.0, (N, D))
    X *= (rng.uniform(lo, hi, N) / (X @ q.min(axis=0)))[:, None]
    y = rng.integers(0, 2, N)
    X *= np.where(y == 1, 1.0, -1.0)[:, None]
    m = ca.Model("logistic_regression", dict(N=N, D=D, X=X, y=y, prior_scale=1e8))
    lp, _ = m.log_prob_grad(q)
    want = -exact_terms(X, q, y) - 0.5e-16 * np.sum(q.astype(np.longdouble) ** 2, axis=1)
    # relative: the linear predictor's D roundings on at most 80, exp and log1p a few ulps, a
    # rounding or two per observation on the running product and sum
    tol = (D + 2) * 80 * EPS + 8 * EPS + 4 * N * EPS
    assert np.max(np.abs((lp - want) / want)) < tol


@pytest.mark.parametrize("points", [5, 70])
def test_saturated_rows_hier(points):
    N, K, G = 20000, 3, 4
    rng = np.random.default_rng(points)
    b = 0.01 * rng.uniform(0.999, 1.0, points)
    x = 36.8 / (K * b.min())  # e^-36.8 is below half an ulp of 1
    y = rng.integers(0, 2, N)
    X = x * np.where(y == 1, 1.0, -1.0)[:, None] * np.ones((N, K))
    m = ca.Model("hier_logistic_cp", dict(N=N, K=K, G=G, X=X, group=rng.integers(1, G + 1, N), y=y))
    q = np.zeros((points, m.dim))
    q[:, :K] = b[:, None]          # mu = beta: z = 0, and tau = e^0 = 1
    q[:, 2 * K:] = b[:, None]
    lp, _ = m.log_prob_grad(q, jacobian=False)
    base = ca.Model("hier_logistic_cp", dict(N=G, K=K, G=G, X=np.zeros((G, K)), group=np.arange(1, G + 1),
                                             y=np.zeros(G, dtype=np.int64)))
    prior = base.log_prob_grad(q, jacobian=False)[0] + G * np.log(np.longdouble(2))
    want = prior - exact_terms(X, q[:, 2 * K:3 * K], y)
    # absolute: the prior terms' magnitude is below 8 (two evaluations), the sum itself 2e-12
    tol = 64 * 8 * EPS
    assert tol < 0.1 * N * np.exp(-36.8)
    assert np.max(np.abs(lp - want)) < tol
