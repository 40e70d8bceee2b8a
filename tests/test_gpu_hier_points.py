"""Hierarchical logistic gradient at the edges of its point tiles (16 points up to 32, 64 above), its
observation split (ragged groups around 128 staged rows, an empty group) and its covariate count (a
template parameter), against the oracle."""
import numpy as np
import pytest

import cmdstan_amd as ca
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _data(K, sizes, seed):
    rng = np.random.default_rng(seed)
    grp = np.repeat(np.arange(1, len(sizes) + 1), sizes)
    X = rng.standard_normal((len(grp), K))
    y = (rng.random(len(grp)) < 0.4).astype(np.int64)
    perm = rng.permutation(len(grp))
    return dict(N=len(grp), K=K, G=len(sizes), X=X[perm], y=y[perm], group=grp[perm])


@pytest.mark.parametrize("K,points", [(1, 1), (2, 15), (3, 16), (4, 17), (5, 32), (7, 33), (8, 63), (10, 64),
                                      (11, 65), (13, 2), (15, 130), (16, 31)])
def test_hier_points(K, points):
    data = _data(K, [1, 7, 0, 127, 128, 129, 31], seed=K)
    D = 2 * K + 7 * K
    rng = np.random.default_rng(points)
    q = 0.5 * rng.standard_normal((points, D))
    g, o = ca.Model("hier_logistic_cp", data), O.Model("hier_logistic_cp", data)
    for jac in (True, False):
        lp, gr = g.log_prob_grad(q, jacobian=jac)
        for k in range(points):
            lo, go = o.log_prob_grad(q[k], jac)
            assert abs(lp[k] - lo) <= 1e-12 * (1 + abs(lo))
            # 423 terms of size up to |x| / tau^3: 1e-12 of the largest component
            assert np.abs(gr[k] - go).max() <= 1e-12 * (1 + np.abs(go).max())
