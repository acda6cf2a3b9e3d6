"""The precision form's density: each window's weights rounded to FP32 per node,
summed exactly, rounded once more.  No node carries an error that depends on
the order of the adds, so the density and a tracked bunch, through its reorders,
come out the same every run."""
import numpy as np
import pytest

import oracle as O
import synergia2_amd as sc
from helpers import BETA, GAMMA, gaussian_parts, oracle_run, rel_l2
from test_gpu_parity import gpu_run, make_opts, oracle_kw

pytestmark = pytest.mark.gpu

SHAPE = (32, 32, 64)
DT = 0.1 / (BETA * sc.C_LIGHT)


def parts_of(n):
    return gaussian_parts(n, (2e-3, 1e-4, 1.5e-3, 1e-4, 5e-3, 1e-4), seed=n)


# windows that end inside the bunch and (sort_period 3, second apply) windows of a
# storage that was shuffled since
@pytest.mark.parametrize("sort_period", [0, 1, 3])
@pytest.mark.parametrize("n", [4001, 249_999, 250_003, 750_003])
def test_density_rounding(gpu, n, sort_period):
    parts, masks = parts_of(n), np.ones(n, np.uint8)
    masks[3::11] = 0
    print(f"case density rounding {n} {sort_period}", flush=True)
    rc, out = oracle_run(oracle_kw(SHAPE), parts, masks, 1e10, DT, want=("rho",))
    assert rc == 0, O.last_error()
    op, b = gpu_run(make_opts(SHAPE, sort_period=sort_period, precision=sc.FP32_GRID), parts,
                    masks, 1e10, DT)
    if sort_period == 3:
        order = np.random.default_rng(n).permutation(n)
        b.set_host(np.ascontiguousarray(parts[:, order]), masks[order])
        op.apply_bunch(b, DT)
    got, want = op.debug(sc.DBG_RHO).ravel(), out["rho"].ravel()
    on = want > 0.0
    # half a unit in the last place of FP32 for the parts (all positive) and once
    # more for the sum, and FP64 sums of up to n weights
    assert np.abs(got[on] / want[on] - 1.0).max() <= 2.0 ** -23 * (1 + 1e-6) + 1e-12
    assert np.all(got[~on] == 0.0)


@pytest.mark.parametrize("sort_period", [0, 1])
@pytest.mark.parametrize("n", [100_003, 750_003])
def test_density_repeats(gpu, n, sort_period):
    """The same bits every run, but for the rare part whose FP64 sum in LDS falls
    on either side of a rounding boundary (odds of some 1e-8 per node)."""
    parts, masks = parts_of(n), np.ones(n, np.uint8)
    runs = []
    for r in range(3):
        print(f"case density repeats {n} {sort_period} run {r}", flush=True)
        op, _ = gpu_run(make_opts(SHAPE, sort_period=sort_period, precision=sc.FP32_GRID), parts,
                        masks, 1e10, DT)
        runs.append(op.debug(sc.DBG_RHO).copy())
    assert (runs[0] != runs[1]).sum() <= 2 and (runs[0] != runs[2]).sum() <= 2


def test_track_repeats_slot_for_slot(gpu):
    """Twelve steps with a reorder on every second one, twice: the field repeats
    far below one FP32 rounding (6e-8 of it; 1e-9 of x' here), the slots exactly."""
    n = 400_000
    parts, masks = parts_of(n), np.ones(n, np.uint8)
    runs = []
    for r in range(2):
        b = sc.Bunch(n, 1e11, gamma=GAMMA)
        b.set_host(parts, masks)
        op = sc.SpaceCharge3dOpenHockney(
            make_opts(SHAPE, sort_period=2, precision=sc.FP32_GRID))
        drift = sc.make_slices([(sc.MAP_DRIFT, 0.5, 0.0)], b.p, b.mass)
        for k in range(12):
            print(f"case track repeat {r} step {k}", flush=True)
            sc.apply_maps(b, drift)
            op.apply_bunch(b, 10 * DT)
        runs.append(b.host()[0])
    assert np.array_equal(runs[0][6], runs[1][6])
    for c in range(6):
        assert rel_l2(runs[0][c], runs[1][c]) <= 1e-10, c
