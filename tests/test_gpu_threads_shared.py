"""Calls of several threads on one handle that build or share the handle's own state: the converted
copies of X and the tuning results of reduced-precision calls, a flow's activations."""
import threading

import numpy as np
import pytest

import cmdstan_amd as ca
from cmdstan_amd.sampler import Flow
from tests.model_cases import EIGHT, logistic

pytestmark = pytest.mark.gpu


def run_together(jobs, rounds):
    """Every job (a call and the result it has when run alone) in its own thread; the jobs that differ."""
    wrong, start = [], threading.Barrier(len(jobs))

    def work(k):
        try:
            call, want = jobs[k]
            start.wait()
            for _ in range(rounds):
                got = call()
                if not all(np.array_equal(a, b) for a, b in zip(got, want)):
                    wrong.append(k)
        except Exception as e:  # noqa: BLE001
            wrong.append((k, repr(e)))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    return wrong


@pytest.mark.parametrize("path", ["0", "1", "2"])
@pytest.mark.parametrize("D", [40, 200])
def test_precisions_share_a_handle(monkeypatch, path, D):
    monkeypatch.setenv("CMDSTAN_AMD_GLM_PATH", path)  # the kernel, so that a call alone gives the same sums
    data = logistic(seed=4, N=3000, D=D)
    alone = ca.Model("logistic_regression", data)
    m = ca.Model("logistic_regression", data)
    rng = np.random.default_rng(1)
    jobs = []
    for precision in ("fp32", "bf16", "fp32", "bf16", "fp64"):
        q = 0.2 * rng.standard_normal((int(rng.integers(1, 70)), D))
        jobs.append((lambda q=q, p=precision: m.log_prob_grad(q, precision=p), alone.log_prob_grad(q, precision=precision)))
    assert run_together(jobs, 10) == []


def test_sampling_shares_a_handle():
    m = ca.Model("eight_schools_cp", EIGHT)
    opts = dict(num_chains=3, num_samples=50, num_warmup=50)
    q = np.random.default_rng(2).standard_normal((5, m.dim))
    jobs = [(lambda s=s: m.sample(seed=s, **opts).draws, m.sample(seed=s, **opts).draws) for s in (1, 2)]
    jobs.append((lambda: m.log_prob_grad(q), m.log_prob_grad(q)))
    assert run_together(jobs, 5) == []


def test_threads_share_a_flow():
    D, n = 37, 20
    f = Flow(D, n_layers=4, hidden=16, max_rows=32)
    rng = np.random.default_rng(3)
    f.set_params(f.get_params() + 0.05 * rng.standard_normal(f.n_params).astype(np.float32))
    z, gx = rng.standard_normal((4, n, D)), rng.standard_normal((n, D))
    calls = [lambda: f.forward(z[0]), lambda: f.inverse(z[1]), lambda: (f.pullback_grad(z[2], gx),),
             lambda: f.loss_grad(z[3])]
    jobs = [(c, c()) for c in calls]
    assert run_together(jobs, 20) == []
