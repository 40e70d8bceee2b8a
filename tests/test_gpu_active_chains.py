"""Lockstep gradients of the waiting chains found from their request flags (at most 64 chains) and from
the compacted list (more), around that limit: trees of different depths leave chains waiting and done in
any mix.  The single transitions agree with the oracle's."""
import numpy as np
import pytest

import cmdstan_amd as ca
from oracle import oracle as O
from tests.model_cases import hier_logistic, logistic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("driver", ["lockstep", "lockstep_block"])
@pytest.mark.parametrize("name,data", [("logistic_regression", logistic(seed=3, N=150, D=5)),
                                       ("logistic_regression", logistic(seed=4, N=90, D=131)),
                                       ("hier_logistic_cp", hier_logistic(seed=5))],
                         ids=["d5", "wide", "hier"])
@pytest.mark.parametrize("nch", [1, 17, 64, 65])
def test_active_chains(name, data, nch, driver):
    m, o = ca.Model(name, data), O.Model(name, data)
    D = m.dim
    rng = np.random.default_rng(100 + nch)
    q0 = 0.3 * rng.standard_normal((nch, D))
    u, z = rng.random((nch, 2048)), rng.standard_normal((nch, D))
    q, info = m.transition_replay(q0, u, z, 0.06, max_depth=6, driver=driver)
    depths = set()
    for k in range(nch):
        qo, io = o.transition_replay(q0[k], u[k], z[k], 0.06, metric=1, minv=np.ones(D), max_depth=6)
        assert (info[k]["depth"], info[k]["n_leapfrog"]) == (io["depth"], io["n_leapfrog"])
        assert np.allclose(q[k], qo, rtol=1e-10, atol=1e-12)
        depths.add(io["n_leapfrog"])
    assert nch < 17 or len(depths) > 1
