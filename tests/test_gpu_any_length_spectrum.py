"""The Green's spectrum of the passes for other lengths than powers of two,
column by column, where both column passes have an odd number of columns: the
last one has no partner in its complex line."""
import numpy as np
import pytest

import oracle as O
import synergia2_amd as sc
from helpers import BETA, gaussian_parts
from test_gpu_parity import gpu_run, make_opts

pytestmark = pytest.mark.gpu

DT = 0.1 / (BETA * sc.C_LIGHT)


def spectrum(shape, green, precision=sc.FP64):
    parts = gaussian_parts(2003, (2e-3, 1e-4, 1.5e-3, 1e-4, 5e-3, 1e-4), seed=sum(shape))
    op, _ = gpu_run(make_opts(shape, green, precision=precision), parts,
                    np.ones(2003, np.uint8), 1e10, DT)
    gx, gy, gz = shape
    return op, op.debug(sc.DBG_GHAT).reshape(gz + 1, gy + 1, gx + 1)


# shapes whose g2 has the plain index decomposition (nothing is added to the
# spectrum's symmetric values)
@pytest.mark.parametrize("green", ["linear", "pointlike"])
@pytest.mark.parametrize("shape", [(12, 10, 14), (12, 18, 20), (60, 54, 100)])
def test_spectrum_columns(gpu, shape, green):
    gx, gy, gz = shape
    assert (gz + 1) * (gx + 1) % 2 and (gy + 1) * (gx + 1) % 2
    print(f"case spectrum {shape} {green}", flush=True)
    op, got = spectrum(shape, sc.GREEN_LINEAR if green == "linear" else sc.GREEN_POINTLIKE)
    g2 = O.green_fn2(green, shape, op.debug(sc.DBG_DOMAIN)["h"])[:, :, :2 * gx]
    want = np.fft.rfftn(g2).real[:gz + 1, :gy + 1]
    # every element: both transforms leave a few 2^-53 of the largest value
    # times the square root of a line's length in each of three passes; a
    # partner read while it is overwritten leaves an error of its own size
    tol = 1e-13 * np.abs(want).max()
    assert np.abs(got - want).max() <= tol
    assert np.abs(got[gz, :, gx] - want[gz, :, gx]).max() <= tol  # last of the y pass
    assert np.abs(got[:, gy, gx] - want[:, gy, gx]).max() <= tol  # last of the z pass


@pytest.mark.parametrize("shape", [(12, 10, 14), (110, 110, 200)])
def test_spectrum_repeats(gpu, shape):
    """The same bits from every run (the second shape has more blocks than the
    chip holds at a time)."""
    runs = []
    for k in range(3):
        print(f"case spectrum repeats {shape} {k}", flush=True)
        runs.append(spectrum(shape, sc.GREEN_LINEAR)[1].copy())
    assert np.array_equal(runs[0], runs[1]) and np.array_equal(runs[0], runs[2])
