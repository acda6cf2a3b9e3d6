"""The first reorder (particle records from 250000 particles on) with the kick
that follows (two particles per lane from 1e6 on), and the cell
sort's tiles (1024, 2048 or 4096 items by the particle count) and
digit widths (up to 8 bits, 9 where that saves a pass) at their edges: the
permutation is the stable order of the keys, the keys the oracle's."""
import numpy as np
import pytest

import oracle as O
import synergia2_amd as sc
from helpers import BETA, gaussian_parts
from test_gpu_parity import check_kicked, gpu_run, make_opts, oracle_kw, oracle_run

pytestmark = pytest.mark.gpu


# 9, 14, 17 and 20 key bits
@pytest.mark.parametrize("shape", [(8, 8, 5), (24, 20, 32), (32, 32, 64), (64, 64, 128)])
@pytest.mark.parametrize("n", [1, 1023, 1025, 8191, 2_500_000, 2_500_001, 8_000_001])
def test_sort_permutation(gpu, shape, n):
    parts = gaussian_parts(n, (2e-3, 1e-4, 1.5e-3, 1e-4, 5e-3, 1e-4), seed=n)
    masks = np.ones(n, np.uint8)
    masks[2::13] = 0
    if n == 1:  # no extent of its own
        fixed = ((0.02, 0.02, 0.08), (0.0, 0.0, 0.0))
    else:
        fixed = None
    dt = 0.1 / (BETA * sc.C_LIGHT)
    print(f"case sort {shape} {n}", flush=True)
    op, _ = gpu_run(make_opts(shape, sort_period=0, fixed=fixed), parts, masks, 1e10, dt)
    keys, perm = op.debug(sc.DBG_KEYS, n), op.debug(sc.DBG_PERM, n)
    assert np.array_equal(perm, np.argsort(keys, kind="stable"))
    if 1 < n < 10_000:
        rc, out = oracle_run(oracle_kw(shape), parts, masks, 1e10, dt, want=("keys",))
        assert rc == 0, O.last_error()
        assert np.array_equal(keys, out["keys"])


@pytest.mark.parametrize("n", [249_999, 250_000, 250_003, 999_999, 1_000_003])
def test_first_reorder(gpu, n):
    shape = (24, 20, 32)
    parts = gaussian_parts(n, (2e-3, 1e-4, 1.5e-3, 1e-4, 5e-3, 1e-4), seed=n)
    masks = (np.arange(n) % 7).astype(np.uint8)  # 0 inactive, any other byte active
    dt = 0.1 / (BETA * sc.C_LIGHT)
    print(f"case first reorder {n}", flush=True)
    rc, out = oracle_run(oracle_kw(shape), parts, (masks != 0).astype(np.uint8), 1e10, dt,
                         want=("perm",))
    assert rc == 0, O.last_error()
    op, b = gpu_run(make_opts(shape, sort_period=1), parts, masks, 1e10, dt)
    perm = op.debug(sc.DBG_PERM, n)
    assert np.array_equal(perm, out["perm"])
    got, gmasks = b.host()
    assert np.array_equal(gmasks, masks[perm])
    for c in (0, 2, 4, 6):
        assert np.array_equal(got[c], parts[c][perm])
    check_kicked(got, gmasks, out["parts"], parts)
