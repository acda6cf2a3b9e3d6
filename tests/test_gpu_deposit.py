"""The deposit's window sizes (1, 2 or 4 slots per thread by the particle
count, 1 through a permutation) at their edges, against the oracle."""
import numpy as np
import pytest

import oracle as O
import synergia2_amd as sc
from helpers import BETA, gaussian_parts, rel_l2
from test_gpu_parity import gpu_run, make_opts, oracle_kw, oracle_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sort_period", [0, 1])
@pytest.mark.parametrize("n", [2, 255, 256, 257, 513, 249_999, 250_000, 250_001, 749_999, 750_003])
def test_deposit_windows(gpu, n, sort_period):
    shape = (24, 20, 32)
    parts = gaussian_parts(n, (2e-3, 1e-4, 1.5e-3, 1e-4, 5e-3, 1e-4), seed=n)
    masks = np.ones(n, np.uint8)
    masks[3::11] = 0
    dt = 0.1 / (BETA * sc.C_LIGHT)
    print(f"case deposit windows {n} {sort_period}", flush=True)
    rc, out = oracle_run(oracle_kw(shape), parts, masks, 1e10, dt, want=("rho",))
    assert rc == 0, O.last_error()
    op, _ = gpu_run(make_opts(shape, sort_period=sort_period), parts, masks, 1e10, dt)
    assert rel_l2(op.debug(sc.DBG_RHO), out["rho"]) <= 1e-13
    op32, _ = gpu_run(make_opts(shape, sort_period=sort_period, precision=sc.FP32_GRID), parts,
                      masks, 1e10, dt)
    assert rel_l2(op32.debug(sc.DBG_RHO), out["rho"]) <= 2e-7
