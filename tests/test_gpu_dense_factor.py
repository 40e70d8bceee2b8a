"""The blocked Cholesky factor and inverse of a given dense metric, at the edges of its 32-column
panels: one transition from the drawn momentum (p = L^-T z) against the oracle, and the refusal of a
metric that is not positive definite in its last direction only."""
import numpy as np
import pytest

import cmdstan_amd as ca
from oracle import oracle as O
from tests.model_cases import gauss

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [1, 2, 16, 31, 32, 33, 47, 64, 65, 97, 130, 161])
def test_dense_factor_transition(D):
    rng = np.random.default_rng(D)
    data = gauss(seed=D, D=D)
    A = rng.standard_normal((D, D))
    minv = A @ A.T / D + 0.5 * np.eye(D)
    q0 = data["mu"] + 0.5 * rng.standard_normal((3, D))
    u, z = rng.random((3, 512)), rng.standard_normal((3, D))
    eps = 0.5 * D ** -0.25
    gm, om = ca.Model("gauss", data), O.Model("gauss", data)
    q, info = gm.transition_replay(q0, u, z, eps, metric="dense_e", inv_metric=minv, max_depth=5)
    for k in range(3):
        qo, io = om.transition_replay(q0[k], u[k], z[k], eps, metric=2, minv=minv, max_depth=5)
        assert (info[k]["depth"], info[k]["n_leapfrog"]) == (io["depth"], io["n_leapfrog"])
        # condition numbers below 1e2 and 31 leapfrogs: 1e4 roundings
        assert np.allclose(q[k], qo, rtol=1e-11, atol=1e-11)
        assert abs(info[k]["energy"] - io["energy"]) <= 1e-10 * (1 + abs(io["energy"]))


@pytest.mark.parametrize("D", [1, 33, 96])
def test_dense_factor_not_positive_definite(D):
    m = ca.Model("gauss", gauss(seed=3, D=D))
    minv = np.eye(D)
    minv[-1, -1] = -1e-3
    with pytest.raises(ca.SamplerError, match="not positive definite"):
        m.transition_replay(np.zeros((2, D)), np.full((2, 64), 0.5), np.zeros((2, D)), 0.1, metric="dense_e",
                            inv_metric=minv)
