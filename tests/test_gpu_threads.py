"""Calls of several threads on one handle: the kept device buffers belong to one call at a time."""
import threading

import numpy as np
import pytest

import cmdstan_amd as ca
from tests.model_cases import hier_logistic, logistic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,data", [("logistic_regression", logistic(seed=2, N=3000, D=40)),
                                       ("logistic_regression", logistic(seed=2, N=500, D=200)),
                                       ("hier_logistic_cp", hier_logistic(seed=2))], ids=["glm", "wide", "hier"])
def test_threads_share_a_handle(name, data):
    m = ca.Model(name, data)
    rng = np.random.default_rng(1)
    qs = [0.2 * rng.standard_normal((n, m.dim)) for n in (1, 16, 33, 70)]
    want = [m.log_prob_grad(q) for q in qs]
    wrong = []

    def work(k):
        for _ in range(20):
            lp, g = m.log_prob_grad(qs[k])
            if not (np.array_equal(lp, want[k][0]) and np.array_equal(g, want[k][1])):
                wrong.append(k)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong
