"""Drift / quadrupole maps on the device against the oracle, bit for bit, on
the bunches where the shared reciprocal square root of the fast form could
round differently or must hand over to the general form."""
import numpy as np
import pytest

import oracle as O
import synergia2_amd as sc
from helpers import GAMMA

pytestmark = pytest.mark.gpu

N = 20003
CELL = [(sc.MAP_DRIFT, 0.37, 0.0), (sc.MAP_QUADRUPOLE, 0.2, 0.6), (sc.MAP_DRIFT, 1.0, 0.0),
        (sc.MAP_QUADRUPOLE, 0.13, -0.6)]


def bunch_columns(kind, rng):
    """(7, N) columns; every kind mixes in exactly on-axis particles."""
    p = np.zeros((7, N))
    p[0], p[2] = 1e-3 * rng.standard_normal((2, N))
    p[4] = 1e-2 * rng.standard_normal(N)
    p[6] = np.arange(N)
    # slopes over nine decades: a = dp^2 - x'^2 - y'^2 next to 1, where the
    # square root and its reciprocal come closest to rounding ties
    slope = 10.0 ** rng.uniform(-9, -2, N)
    p[1], p[3] = slope * rng.standard_normal((2, N))
    if kind == "design momentum":
        p[3, ::2] = 0.0
    elif kind == "beam":
        p[5] = 1e-4 * rng.standard_normal(N)
    elif kind == "wide":  # out of the fast form's range in part: a from about 0 to 3
        p[1], p[3] = rng.uniform(-0.6, 0.6, (2, N))
        p[5] = rng.uniform(-0.5, 0.8, N)
    elif kind == "lost":  # no longer a beam: NaN, infinities, x'^2 + y'^2 > dp^2
        p[1, ::3] = 2.0
        p[3, 1::5] = np.inf
        p[0, 2::7] = np.nan
        p[5, 3::11] = -1.5
    p[1, :64] = p[3, :64] = 0.0
    p[0, :32] = p[2, :32] = 0.0
    return p


@pytest.mark.parametrize("kind", ["design momentum", "beam", "wide", "lost"])
@pytest.mark.parametrize("program", ["cell", "backwards", "skew", "zero length", "massless"])
def test_maps_bits(gpu, kind, program):
    rng = np.random.default_rng(len(kind) * 100 + len(program))
    mass = 0.0 if program == "massless" else sc.PROTON_MASS
    spec = [(k, -L, k1) for k, L, k1 in CELL] if program == "backwards" else list(CELL)
    if program == "zero length":
        spec.insert(1, (sc.MAP_DRIFT, 0.0, 0.0))
    b = sc.Bunch(N, 1e11, gamma=GAMMA)
    b.mass = mass
    p0 = bunch_columns(kind, rng)
    m0 = np.ones(N, np.uint8)
    m0[5::17] = 0
    b.set_host(p0, m0)
    arr, n = sc.make_slices(spec, b.p, mass)
    oarr = O.make_slices([(k, L, k1, 4, arr[i].ref_cdt) for i, (k, L, k1) in enumerate(spec)])
    if program == "skew":
        arr[1].k1s = oarr[1].k1s = 0.3
    sc.apply_maps(b, (arr, n))
    got, _ = b.host()
    want = np.ascontiguousarray(p0.copy())
    ob = O.make_bunch(want, m0.copy(), N, 1e11, 1, mass, b.gamma, b.beta, b.p)
    O.lib().orc_apply_maps(O.C.byref(ob), oarr, n)
    for c in range(7):
        assert np.array_equal(got[c], want[c], equal_nan=True), c
