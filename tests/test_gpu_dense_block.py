"""Dense metric with a block per chain, against the oracle's transitions: rows per thread of the metric
products (1, 2, 3 or 4 by D) at the edges of their ranges, one chain per block up to many blocks."""
import numpy as np
import pytest

import cmdstan_amd as ca
from oracle import oracle as O
from tests.model_cases import logistic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,nch", [(1, 3), (2, 3), (15, 3), (256, 2), (257, 2), (512, 2), (513, 2), (768, 2), (769, 2),
                                   (1024, 2), (9, 600)])
def test_dense_block(D, nch):
    data = logistic(seed=D, N=60, D=D)
    gm, om = ca.Model("logistic_regression", data), O.Model("logistic_regression", data)
    rng = np.random.default_rng(D)
    A = rng.standard_normal((D, D)) / np.sqrt(D)
    minv = (A @ A.T * 0.3 + np.eye(D)).ravel()
    q0 = 0.1 * rng.standard_normal((nch, D))
    u, z = rng.random((nch, 256)), rng.standard_normal((nch, D))
    eps = 0.15 / np.sqrt(D)
    q, info = gm.transition_replay(q0, u, z, eps, metric="dense_e", inv_metric=minv, max_depth=3,
                                   driver="lockstep_block")
    for k in (range(nch) if nch < 10 else (0, 1, nch // 2, nch - 1)):
        qo, io = om.transition_replay(q0[k], u[k], z[k], eps, metric=O.METRICS["dense_e"], minv=minv, max_depth=3)
        assert (info[k]["depth"], info[k]["n_leapfrog"]) == (io["depth"], io["n_leapfrog"])
        # sums of at most 1024 products per leaf, 7 leaves: 1e-13 of the values; two orders kept for the inverse factor
        assert np.allclose(q[k], qo, rtol=1e-10, atol=1e-11)
