"""The fused machine with the chains' vectors in LDS against the one in global memory: the same
operations in the same order, so one transition of the same chains has the same bits, whether
the batch is small enough for LDS or, with more chains than the LDS form takes, is not."""
import numpy as np
import pytest

import cmdstan_amd as ca
from tests.model_cases import CASES, gauss, hier_normal

pytestmark = pytest.mark.gpu

MANY = 2100  # more chains than 256 CUs hold at eight a CU


@pytest.mark.parametrize("name,data,metric", [
    ("bernoulli", CASES["bernoulli"], "diag_e"), ("eight_schools_cp", CASES["eight_schools_cp"], "unit_e"),
    ("gauss", gauss(D=3), "dense_e"), ("gauss", gauss(D=16), "diag_e"), ("gauss", gauss(D=64), "dense_e"),
    ("gauss", gauss(D=65), "dense_e"), ("gauss", gauss(D=130), "dense_e"), ("gauss", gauss(D=130), "unit_e"),
    ("hier_normal_nc", hier_normal(J=63), "diag_e")])
def test_lds_equals_global(name, data, metric):
    m = ca.Model(name, data)
    D = m.dim
    rng = np.random.default_rng(D)
    q0 = np.tile(0.3 * rng.standard_normal((7, D)), (MANY // 7, 1))
    u, z = np.tile(rng.random((7, 600)), (MANY // 7, 1)), np.tile(rng.standard_normal((7, D)), (MANY // 7, 1))
    A = rng.standard_normal((D, D))
    minv = A @ A.T / D + np.eye(D) if metric == "dense_e" else (np.ones(D) if metric == "unit_e" else 0.5 + rng.random(D))
    big, info = m.transition_replay(q0, u, z, 0.11, metric=metric, inv_metric=minv, max_depth=6)
    small, info7 = m.transition_replay(q0[:7], u[:7], z[:7], 0.11, metric=metric, inv_metric=minv, max_depth=6)
    assert np.array_equal(big[:7], small) and np.array_equal(big[-7:], small)
    assert info[:7] == info7
    assert max(i["n_leapfrog"] for i in info7) >= 3


def test_lds_launch_boundary_and_fp32():
    """Runs of several launches (256 gradients each) continue from the copied-back vectors, in both vector types."""
    m = ca.Model("hier_normal_nc", hier_normal(J=20))
    for precision in ("fp64", "fp32"):
        kw = dict(num_warmup=60, num_samples=40, seed=3, precision=precision)
        few = m.sample(num_chains=3, **kw)
        many = m.sample(num_chains=MANY, **kw)
        for k in range(3):
            assert np.array_equal(few.draws[k], many.draws[k])
