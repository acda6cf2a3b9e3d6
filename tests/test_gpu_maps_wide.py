"""Maps of wavefronts that hold one particle out of the fast drift's range
(a = dp^2 - x'^2 - y'^2 outside [1/2, 2]): from the start, from a later slice
on, or with no finite path at all; bit for bit against the oracle, alone and
fused behind the kick."""
import numpy as np
import pytest

import oracle as O
import synergia2_amd as sc
from helpers import GAMMA
from test_gpu_maps import CELL

pytestmark = pytest.mark.gpu

N = 4099


def wide_columns(kind):
    rng = np.random.default_rng(len(kind))
    p = np.zeros((7, N))
    p[0], p[2] = 1e-3 * rng.standard_normal((2, N))
    p[1], p[3] = 1e-4 * rng.standard_normal((2, N))
    p[4] = 1e-2 * rng.standard_normal(N)
    p[5] = 1e-4 * rng.standard_normal(N)
    p[6] = np.arange(N)
    one = slice(17, None, 64)  # one lane of every wavefront
    if kind == "slope":
        p[1, one] = 0.8
    elif kind == "steep":  # a about 1e-12
        p[1, one] = np.sqrt((1.0 + p[5, one]) ** 2 - p[3, one] ** 2) * (1 - 5e-13)
    elif kind == "later":  # pushed out by the quadrupole slices
        p[0, one] = 6.0
    elif kind == "momentum":
        p[5, one] = 3.0
    elif kind == "slow":
        p[5, one] = -0.9
    elif kind == "no path":  # a < 0
        p[3, one] = 1.5
    elif kind == "backwards":
        p[5, one] = -1.5
    return p


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("kind", ["slope", "steep", "later", "momentum", "slow", "no path",
                                  "backwards"])
@pytest.mark.parametrize("skew", [0.0, 0.3])
def test_wide_bits(gpu, kind, skew, fused):
    p0, m0 = wide_columns(kind), np.ones(N, np.uint8)
    m0[5::29] = 0
    b = sc.Bunch(N, 1e11, gamma=GAMMA)
    b.set_host(p0, m0)
    arr, n = sc.make_slices(CELL, b.p, b.mass)
    oarr = O.make_slices([(k, L, k1, 4, arr[i].ref_cdt) for i, (k, L, k1) in enumerate(CELL)])
    arr[3].k1s = oarr[3].k1s = skew
    print(f"case wide maps {kind} {skew} {fused}", flush=True)
    if fused:  # behind a kick of nothing, storage order kept
        o = sc.default_options(16, 16, 16)
        o.kick_scale, o.sort_period = 0.0, 0
        sc.set_fixed_domain(o, (0.0, 0.0, 0.0), (0.02, 0.02, 0.1))
        op = sc.SpaceCharge3dOpenHockney(o)
        op.set_post_kick_maps((arr, n))
        op.apply_bunch(b, 1e-9)
    else:
        sc.apply_maps(b, (arr, n))
    got, _ = b.host()
    want = np.ascontiguousarray(p0.copy())
    ob = O.make_bunch(want, m0.copy(), N, 1e11, 1, b.mass, b.gamma, b.beta, b.p)
    O.lib().orc_apply_maps(O.C.byref(ob), oarr, n)
    for c in range(7):
        assert np.array_equal(got[c], want[c], equal_nan=True), c
