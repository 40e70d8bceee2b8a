"""A flow run whose plain phase fails: its rows are not the caller's, so the draws array stays as it was."""
import ctypes as C

import numpy as np
import pytest

import cmdstan_amd as ca
from cmdstan_amd._lib import DP, lib, nuts_config, nuts_output
from tests.model_cases import gauss

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flow", [1, 2])
@pytest.mark.parametrize("thin,saved", [(1, -1), (2, 1)])
def test_failed_plain_phase_leaves_the_draws_array(flow, thin, saved):
    D, chains, warm, pilot = 5, 2, 50, 20
    m = ca.Model("gauss", gauss(D=D))
    cfg = nuts_config()
    lib().nuts_config_default(C.byref(cfg))
    cfg.num_chains, cfg.num_samples, cfg.num_warmup, cfg.thin = chains, 2, warm, thin
    cfg.flow, cfg.flow_pilot, cfg.max_saved_params = flow, pilot, saved
    # room for every row of the earlier phase, so that a copy of it would stay inside
    draws = np.full(chains * (warm + pilot) * (7 + D), -12345.0)
    status = np.zeros(chains, dtype=np.int32)
    init = np.full((chains, D), 1e200)  # the log density is -inf: initialisation fails
    out = nuts_output()
    out.draws = draws.ctypes.data_as(DP)
    out.status = status.ctypes.data_as(C.POINTER(C.c_int))
    rc = lib().nuts_sample(m.h, C.byref(cfg), init.ctypes.data_as(DP), None, C.byref(out))
    assert rc != 0
    assert np.all(status == 1)  # initialisation failed
    assert np.all(draws == -12345.0)
