"""Two-pass reduced-precision gradient (D > 128): the reduction's column blocks at their edges, points and
rows inside a tile, against the closed form on BF16-representable X."""
import numpy as np
import pytest

import cmdstan_amd as ca
from tests.model_cases import logistic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("N,D,n", [(1, 129, 1), (200, 255, 3), (129, 256, 65), (300, 257, 2), (500, 512, 130), (65, 520, 17)])
def test_two_pass_columns(N, D, n, precision):
    eps = 2.0 ** -24
    d = logistic(seed=N + D, N=N, D=D)
    d["X"] = (d["X"].astype(np.float32).view(np.uint32) & 0xFFFF0000).view(np.float32).astype(np.float64)
    q = 0.1 * np.random.default_rng(D + n).standard_normal((n, D))
    lp, g = ca.Model("logistic_regression", d).log_prob_grad(q, precision=precision)
    eta = d["X"] @ q.T
    lp0 = (d["y"][:, None] * eta - np.logaddexp(0, eta)).sum(axis=0) - 0.5 * (q * q).sum(axis=1) / 6.25
    g0 = (d["X"].T @ (d["y"][:, None] - 1 / (1 + np.exp(-eta)))).T - q / 6.25
    # worst case: an eta of D products and sums (four roundings of a three-term operand), the
    # term's few operations, at most N sums in one FP32 chain
    deta = (D + 6) * eps * (np.abs(d["X"]) @ np.abs(q).T).max()
    assert np.abs(g - g0).max() <= (np.abs(d["X"]).sum(axis=0).max() + 1.0) * (0.25 * deta + (16 + N) * eps)
    assert np.abs(lp - lp0).max() <= N * (deta + 8 * eps * (1 + np.abs(eta).max()))
