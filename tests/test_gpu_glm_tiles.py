"""FP64 logistic-regression gradient up to 128 coefficients against the closed form in numpy, at the edges
of its tiles: every count of 16-column tiles and of four-column steps in the last, one to 129 points
(waves split over rows up to 16 points, over points above), rows that end inside a tile."""
import numpy as np
import pytest

import cmdstan_amd as ca
from tests.model_cases import logistic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [1, 3, 4, 5, 9, 16, 17, 31, 33, 40, 52, 64, 65, 79, 84, 96, 100, 109, 112, 113, 127, 128])
def test_glm_tiles(D):
    for N, n in ((1, 1), (15, 16), (63, 17), (65, 64), (1000, 65), (4097, 3), (333, 129)):
        d = logistic(seed=N + D, N=N, D=D)
        q = 0.3 * np.random.default_rng(D + n).standard_normal((n, D))
        lp, g = ca.Model("logistic_regression", d).log_prob_grad(q)
        eta = d["X"] @ q.T
        lp0 = (d["y"][:, None] * eta - np.logaddexp(0, eta)).sum(axis=0) - 0.5 * (q * q).sum(axis=1) / 6.25
        g0 = (d["X"].T @ (d["y"][:, None] - 1 / (1 + np.exp(-eta)))).T - q / 6.25
        # sums of N terms of size |x| <= 6: rounding below 1e-15 of the sum of magnitudes
        assert np.abs(g - g0).max() <= 1e-13 * (np.abs(d["X"]).sum(axis=0).max() + 1.0), (N, n)
        assert np.abs(lp - lp0).max() <= 1e-13 * (np.abs(eta).sum(axis=0).max() + N + 1.0), (N, n)


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("D", [1, 4, 15, 16, 17, 33, 48, 63, 65, 81, 100, 112, 113, 128])
def test_glm_tiles_fp32(D, precision, monkeypatch):
    """The single-pass FP32 kernel (path 0) on outcomes and BF16-representable X."""
    monkeypatch.setenv("CMDSTAN_AMD_GLM_PATH", "0")
    eps = 2.0 ** -24
    for N, n in ((1, 1), (31, 16), (33, 17), (65, 64), (1000, 65), (4097, 3), (333, 129)):
        d = logistic(seed=N + D, N=N, D=D)
        d["X"] = (d["X"].astype(np.float32).view(np.uint32) & 0xFFFF0000).view(np.float32).astype(np.float64)
        q = 0.3 * np.random.default_rng(D + n).standard_normal((n, D))
        lp, g = ca.Model("logistic_regression", d).log_prob_grad(q, precision=precision)
        eta = d["X"] @ q.T
        lp0 = (d["y"][:, None] * eta - np.logaddexp(0, eta)).sum(axis=0) - 0.5 * (q * q).sum(axis=1) / 6.25
        g0 = (d["X"].T @ (d["y"][:, None] - 1 / (1 + np.exp(-eta)))).T - q / 6.25
        # worst case: an eta of D rounded products and sums (q rounded too), the term's few
        # operations, at most 64 + N / 256 sums per FP32 chain
        deta = (D + 2) * eps * (np.abs(d["X"]) @ np.abs(q).T).max()
        assert np.abs(g - g0).max() <= (np.abs(d["X"]).sum(axis=0).max() + 1.0) * (0.25 * deta + (72 + N / 256) * eps), (N, n)
        assert np.abs(lp - lp0).max() <= N * (deta + 8 * eps * (1 + np.abs(eta).max())), (N, n)
