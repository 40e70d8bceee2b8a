"""Device memory that idle handles keep: bounded over all of them, given back on request and with them."""
import ctypes as C

import numpy as np
import pytest

import cmdstan_amd as ca
from cmdstan_amd._lib import lib
from tests.model_cases import EIGHT

pytestmark = pytest.mark.gpu

GIB = 2.0 ** 30


def free_bytes():
    hip = C.CDLL("libamdhip64.so.7")  # the runtime that the library links
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_idle_workspaces_are_bounded():
    q = np.zeros((5_000_000, 10))
    q[:, 1] = 0.5
    models = [ca.Model("eight_schools_cp", EIGHT) for _ in range(8)]
    want = models[0].log_prob_grad(q[:1])
    lib().nuts_release_workspaces()
    start = free_bytes()
    for m in models:  # some 0.9 GiB of workspace each
        lp, g = m.log_prob_grad(q)
        assert lp[-1] == want[0][0] and np.array_equal(g[-1], want[1][0])
    kept = start - free_bytes()
    assert 0.5 * GIB < kept < 4.25 * GIB
    assert lib().nuts_release_workspaces() > 0.5 * GIB
    assert start - free_bytes() < 0.25 * GIB
    assert lib().nuts_release_workspaces() == 0
