"""The single-precision plans' composite radices 8 and 12 (lengths 24 = 8 3,
36 = 12 3, 40 = 8 5, 60 = 12 5), which no other shape has: Green's spectrum
element by element, and the field."""
import numpy as np
import pytest

import oracle as O
import synergia2_amd as sc
from helpers import BETA, gaussian_parts, oracle_run, rel_l2
from test_gpu_any_length_spectrum import spectrum
from test_gpu_parity import gpu_run, make_opts, oracle_kw

pytestmark = pytest.mark.gpu

SHAPES = [(12, 18, 20), (20, 30, 12), (30, 12, 18)]  # every length on every axis


@pytest.mark.parametrize("shape", SHAPES)
def test_composite_radices(gpu, shape):
    gx, gy, gz = shape
    print(f"case composite radices {shape}", flush=True)
    op, got = spectrum(shape, sc.GREEN_LINEAR, sc.FP32_GRID)
    g2 = O.green_fn2("linear", shape, op.debug(sc.DBG_DOMAIN)["h"])[:, :, :2 * gx]
    want = np.fft.rfftn(g2).real[:gz + 1, :gy + 1]
    # each element of three passes: a few 2^-24 of the largest value times the
    # root of the line length (at most 60); a wrong index or twiddle is O(1)
    assert np.abs(got - want).max() <= 3 * 4 * np.sqrt(60) * 2.0 ** -24 * np.abs(want).max()
    n = 4001
    parts = gaussian_parts(n, (2e-3, 1e-4, 1.5e-3, 1e-4, 5e-3, 1e-4), seed=sum(shape))
    masks = np.ones(n, np.uint8)
    dt = 0.1 / (BETA * sc.C_LIGHT)
    rc, out = oracle_run(oracle_kw(shape), parts, masks, 1e10, dt, want=("ex", "ey", "ez"))
    assert rc == 0, O.last_error()
    for precision, tol in ((sc.FP64, 1e-12), (sc.FP32_GRID, 2e-6)):
        op, _ = gpu_run(make_opts(shape, precision=precision), parts, masks, 1e10, dt)
        for tap, name in ((sc.DBG_EX, "ex"), (sc.DBG_EY, "ey"), (sc.DBG_EZ, "ez")):
            assert rel_l2(op.debug(tap), out[name]) <= tol, (precision, name)
