"""The transform passes of other lengths than powers of two: every radix of
their plans, prime factors without one, the longest lines, odd numbers of
rows and columns (pairs with one member missing), against the oracle."""
import numpy as np
import pytest

import oracle as O
import synergia2_amd as sc
from helpers import BETA, gaussian_parts, rel_l2
from test_gpu_parity import gpu_run, make_opts, oracle_kw, oracle_run

pytestmark = pytest.mark.gpu

SHAPES = [
    (5, 6, 7),       # 10, 12, 14 in one pass each
    (15, 9, 13),     # 6*5, 6*3, 13*2
    (11, 21, 10),    # 11*2, 7*6, 5*4
    (27, 33, 25),    # 9*6, 11*6, 10*5
    (35, 39, 45),    # 10*7, 13*6, 10*9
    (75, 55, 49),    # 15*10, 11*10, 14*7
    (17, 34, 19),    # 17*2, 17*4, 19*2
    (4, 289, 5),     # Dx = 8, Dy = 17*17*2
    (512, 5, 4),     # Dx = 1024
    (6, 512, 5),     # Dy = 1024
    (5, 4, 509),     # Dz = 1018: the longest prime factor
    (487, 5, 4),
    (7, 509, 4),
]


@pytest.mark.parametrize("green", [sc.GREEN_LINEAR, sc.GREEN_POINTLIKE])
@pytest.mark.parametrize("shape", SHAPES)
def test_any_length(gpu, shape, green):
    n = 4001
    parts = gaussian_parts(n, (2e-3, 1e-4, 1.5e-3, 1e-4, 5e-3, 1e-4), seed=sum(shape))
    masks = np.ones(n, np.uint8)
    dt = 0.1 / (BETA * sc.C_LIGHT)
    print(f"case any length {shape} {green}", flush=True)
    gname = "linear" if green == sc.GREEN_LINEAR else "pointlike"
    rc, out = oracle_run(oracle_kw(shape, gname), parts, masks, 1e10, dt,
                         want=("rho", "phi", "ex", "ey", "ez"))
    assert rc == 0, O.last_error()
    op, _ = gpu_run(make_opts(shape, green), parts, masks, 1e10, dt)
    assert rel_l2(op.debug(sc.DBG_PHI), out["phi"]) <= 1e-12
    for tap, name in ((sc.DBG_EX, "ex"), (sc.DBG_EY, "ey"), (sc.DBG_EZ, "ez")):
        assert rel_l2(op.debug(tap), out[name]) <= 1e-12, name
    op32, _ = gpu_run(make_opts(shape, green, precision=sc.FP32_GRID), parts, masks, 1e10, dt)
    for tap, name in ((sc.DBG_EX, "ex"), (sc.DBG_EY, "ey"), (sc.DBG_EZ, "ez")):
        assert rel_l2(op32.debug(tap), out[name]) <= 2e-6, name
